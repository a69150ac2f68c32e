// RWKV-5.x / RWKV-6 forward for any T >= 1.
//
// Per layer: time mix
//   v5: lnmix_seq (LN1, token shift, static k/v/r(/g) mixes)
//   v6: mix1 (LN1, sx = prev - xx, xxx = xx + sx * maa_x) -> tanh(xxx @ W1) -> mix2 (five rank-32
//       products with W2 and the five data-dependent mixes) -> decay LoRA tanh(wx @ D1) @ D2
//   r, k, v (fp16, widened by the consumer), g = SiLU(.) through mm() below
//   wkv56 (per-head 64x64 state in registers for the whole T loop; decay exp(-exp(.)), GroupNorm
//   and the gate fused) -> output matrix with the residual add in its epilogue
// then the channel mix exactly as RWKV-4 (RWKV-6 mixes with kx = xx + (prev - xx) * maa).
// mm(): T == 1 -> streaming GEMV (vec_kernel: ry scaling and the row sums in its prologue,
// activation / residual in its epilogue); T > 1 -> mm8_prepare + MFMA GEMM with the same epilogues.
#include "mm_dispatch.h"
#include "rows.h"

namespace {

struct Mix1Args {
    int T, C;
    const rwkv_half *x, *ln_w, *ln_b, *sx, *maa_x;
    rwkv_half *xx, *sxd, *xxx, *state_out;   // state_out: the token-shift state (may be sx)
};

// One workgroup per row, NT threads: xx = LN1(x[t]); sxd = prev - xx; xxx = xx + sxd * maa_x (rows.h).  A thread's
// chunks of the row and of the previous row stay in registers from one round of loads, and the four sums of the two rows'
// statistics share their barriers.
template <int CH, int NT>
__global__ __launch_bounds__(NT) void v6_mix1_kernel(const rwkv_half *x0, const rwkv_half *ln_w, const rwkv_half *ln_b, const rwkv_half *maa_x,
                                                     const rwkv_half *sx, int C, int T, Mix1Args a) {
    __shared__ __align__(16) float red[24];
    __shared__ float hop[NT == 512 ? 256 * 6 : 1];
    const int t = blockIdx.x, nch = C >> 3;
    const int j8_0 = NT == 256 ? (int)threadIdx.x : (int)(threadIdx.x & 255) + 256 * CH * (int)(threadIdx.x >> 8);
    const rwkv_half *x = x0 + (size_t)t * C;
    const rwkv_half *xp = t > 0 ? x - C : x;
    // row 0's workgroup also forms the new token-shift state LN1(x[T-1]); its statistics ride in the same barriers
    const bool commit = t == 0;
    const rwkv_half *xl = commit ? x0 + (size_t)(T - 1) * C : x;
    h16x8 xv[CH], pxv[CH], lv[CH], wv[CH], bv[CH], mv[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int j8 = min(j8_0 + c * 256, nch - 1);   // chunks past the end repeat the last one (unused)
        xv[c] = *(const h16x8 *)(x + 8 * j8);
        pxv[c] = *(const h16x8 *)(xp + 8 * j8);
        lv[c] = *(const h16x8 *)(xl + 8 * j8);
        wv[c] = *(const h16x8 *)(ln_w + 8 * j8);
        bv[c] = *(const h16x8 *)(ln_b + 8 * j8);
        mv[c] = *(const h16x8 *)(maa_x + 8 * j8);
    }
    float sq[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // sum and sum of squares of the row, the previous row, the last row
    row_sums<6, NT>(sq, red, hop, [&](float (&v)[6], auto) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if (j8_0 + c * 256 < nch) {
                sum_and_squares8(xv[c], v[0], v[1]);
                sum_and_squares8(pxv[c], v[2], v[3]);
                if (commit) sum_and_squares8(lv[c], v[4], v[5]);
            }
    });
    const float mean = sq[0] / C, rstd = rsqrtf(fmaxf(sq[1] / C - mean * mean, 0.f) + LN_EPS);
    const float pmean = sq[2] / C, prstd = rsqrtf(fmaxf(sq[3] / C - pmean * pmean, 0.f) + LN_EPS);
    const float lmean = sq[4] / C, lrstd = rsqrtf(fmaxf(sq[5] / C - lmean * lmean, 0.f) + LN_EPS);
    float d[8];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int j8 = j8_0 + c * 256;
        if (j8 >= nch) break;
        less_mean8(xv[c], mean, d);
        const h16x8 xx = norm8(d, rstd, wv[c], bv[c]);
        h16x8 pv;
        if (t > 0) {
            less_mean8(pxv[c], pmean, d);
            pv = norm8(d, prstd, wv[c], bv[c]);
        } else {
            pv = *(const h16x8 *)(sx + 8 * j8);
        }
        const size_t o = (size_t)t * C + 8 * j8;
        *(h16x8 *)(a.xx + o) = xx;
        *(h16x8 *)(a.sxd + o) = pv - xx;
        *(h16x8 *)(a.xxx + o) = mix8(xx, pv, mv[c], true);
        // the new token-shift state: written by row 0's workgroup, the only one that reads the old state, each thread
        // exactly the chunk it has just read
        if (commit) {
            less_mean8(lv[c], lmean, d);
            *(h16x8 *)(a.state_out + 8 * j8) = norm8(d, lrstd, wv[c], bv[c]);
        }
    }
}
// 256 or 512 threads per row as in lnmix_seq_launch.  us, 256 rows of 4096 channels: 7.2 -> 5.4 with
// the element code of rows.h.
void v6_mix1_launch(const Mix1Args &a, hipStream_t st) {
    const bool few = a.T <= 512;
    const auto kernel = a.C <= 2048   ? v6_mix1_kernel<1, 256>
                        : a.C <= 4096 ? (few ? v6_mix1_kernel<1, 512> : v6_mix1_kernel<2, 256>)
                                      : (few ? v6_mix1_kernel<2, 512> : v6_mix1_kernel<4, 256>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)a.T), dim3(few && a.C > 2048 ? 512 : 256), 0, st, a.x, a.ln_w, a.ln_b, a.maa_x, a.sx, a.C, a.T, a);
}

struct Mix2Args {
    int T, C, R;                     // R = LoRA rank (32)
    const rwkv_half *t1;             // [T, 5R] tanh output
    const rwkv_half *w2;             // [5][R][C]
    const rwkv_half *xx, *sxd;       // [T, C]; sxd NULL (T == 1): prev - xx is formed here from `prev`
    const rwkv_half *prev;           // [C] token-shift state
    const rwkv_half *maa[5];         // w, k, v, r, g
    rwkv_half *out[5];               // [T, C] each
    // v6_mix2_mfma_kernel, uint8 matrices: ry[j] != NULL: out[j] is stored as fp16(mix * ry[j]), the input of matrix j's
    // product, and the sums of mix and mix * my[j] over each block of 256 channels go to p0[j] / p2[j] [T][npart]
    // (npart = the number of blocks rounded up to a multiple of four, the padding entries zero)
    const rwkv_half *ry[5], *my[5];
    float *p0[5], *p2[5];
    int npart;
};

// grid (ceil(T / MIX2_TT), C/256, 5): m_j[c] = sum_i t1[t, jR + i] * w2[j][i][c]; out_j = xx + sxd * (maa_j + m_j).
// One (channel, mix) per thread for a tile of MIX2_TT tokens (4, or 1 for a one-token call): the R coefficients of the channel are loaded once
// and reused for every token of the tile; the sum runs in index order.
template <int MIX2_TT>
__global__ __launch_bounds__(256) void v6_mix2_kernel(Mix2Args a) {
    __shared__ __align__(16) float st1[64][MIX2_TT];   // [i][token]: the tokens of one i are read with 16-byte LDS loads
    const int t0 = blockIdx.x * MIX2_TT, c = blockIdx.y * 256 + threadIdx.x, j = blockIdx.z, R = a.R, C = a.C;
    const int nt = min(MIX2_TT, a.T - t0);
    for (int i = threadIdx.x; i < nt * R; i += 256) {
        const int tt = i / R, r = i - tt * R;
        st1[r][tt] = h2f(a.t1[(size_t)(t0 + tt) * 5 * R + j * R + r]);
    }
    __syncthreads();
    if (c >= C) return;
    const rwkv_half maa = a.maa[j][c];
    const rwkv_half *w = a.w2 + (size_t)j * R * C + c;
    float m[MIX2_TT];
#pragma unroll
    for (int tt = 0; tt < MIX2_TT; ++tt) m[tt] = 0.f;
    for (int i0 = 0; i0 < R; i0 += 16) {
        rwkv_half wv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) wv[i] = w[(size_t)min(i0 + i, R - 1) * C];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (i0 + i < R) {
                const float wf = h2f(wv[i]);
#pragma unroll
                for (int tt = 0; tt < MIX2_TT; ++tt) m[tt] += st1[i0 + i][tt] * wf;
            }
    }
#pragma unroll
    for (int tt = 0; tt < MIX2_TT; ++tt) {
        if (tt >= nt) break;
        const int t = t0 + tt;
        const h16 xx = __builtin_bit_cast(h16, a.xx[(size_t)t * C + c]);
        const h16 sd = a.sxd ? __builtin_bit_cast(h16, a.sxd[(size_t)t * C + c]) : __builtin_bit_cast(h16, a.prev[c]) - xx;
        const h16 mm = __builtin_bit_cast(h16, maa) + (h16)m[tt];
        // one rounding after the difference, as in mix8; calls of one token round the product too where lnmix_kernel mixes
        a.out[j][(size_t)t * C + c] = __builtin_bit_cast(rwkv_half, __builtin_elementwise_fma(sd, mm, xx));
    }
}

// The same for sequence calls, on the matrix cores: 16 tokens x 64 channels per wave, four waves side by side, the R (8 to 64)
// coefficients of a mix as one or two v_mfma_f32_16x16x32_f16 per 16 channels (fp16 operands, fp32 sums; k's past R are zero in
// both).  w2 is [R][C], so a block's coefficients pass through LDS, two k's of a channel to a word (rows of 16 KS + 2 words: two
// lanes to a bank when written, none when read).  Row r of the MFMA of block b is channel 16 (r / 4) + 4 b + r % 4 of the wave's
// 64, so that a lane ends with 16 adjacent channels of one token and four lanes cover a 128-byte line.  All of a workgroup's
// loads are requested at the top.  grid (ceil(T / 16), ceil(C / 256), 5): all five mixes in one workgroup, which reads xx and sxd
// once, is 0.5 % of a call faster at 1000 tokens and 3 % slower up to 45.
// The form before multiplied on the vector units, 4 or 16 tokens x 4 channels per thread, and was bound by their issue.  us, 4096
// channels, rank 32, uint8 (scaled, with sums), 256 tokens: 15.9 -> 11.1; 6 % of a call of 513 tokens.
// C callers may put w2 and the maa vectors on any boundary: their loads are of a type that is aligned to its elements.
typedef h16x8 h16x8_a2 __attribute__((aligned(2)));
template <int KS>
__global__ __launch_bounds__(256) void v6_mix2_mfma_kernel(Mix2Args a) {
    constexpr int ROW = 32 * KS + 4;                                     // halves of a channel's row
    __shared__ __align__(16) h16 sw[256 * ROW];
    __shared__ float red[2][4][16];
    const int C = a.C, R = a.R, t0 = blockIdx.x * 16, j = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, q = lane >> 4;
    const int cb = blockIdx.y * 256;                                     // C % 64 == 0: a wave's channels are all there or none
    const bool live = cb + 64 * wave < C, scaled = a.ry[j] != nullptr;   // scaled: the same for the whole workgroup
    const int c = live ? cb + 64 * wave + 16 * q : 0;                    // this lane's first channel
    const int t = min(t0 + n, a.T - 1);
    const size_t o = (size_t)t * C + c;
    // coefficients: thread (pair kp of k's, group g of 8 channels) of this workgroup's 256
    const int kp = threadIdx.x & 7, g = threadIdx.x >> 3, cg = min(cb + 8 * g, C - 8);
    h16x8 wr[2 * KS][2], tf[KS], mv[2], rv[2] = {}, yv[2] = {}, xx[2], sd[2];
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = 2 * (kp + 8 * i) + h;                          // rows past R: loaded from row 0, zeroed below
            wr[i][h] = *(const h16x8_a2 *)(a.w2 + ((size_t)j * R + (k < R ? k : 0)) * C + cg);
        }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int k = 32 * s + 8 * q;
        tf[s] = *(const h16x8 *)(a.t1 + (size_t)t * 5 * R + j * R + (k < R ? k : 0));
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        xx[p] = *(const h16x8 *)(a.xx + o + 8 * p);
        sd[p] = *(const h16x8 *)(a.sxd + o + 8 * p);
        mv[p] = *(const h16x8_a2 *)(a.maa[j] + c + 8 * p);
        if (scaled) { rv[p] = *(const h16x8 *)(a.ry[j] + c + 8 * p); yv[p] = *(const h16x8 *)(a.my[j] + c + 8 * p); }
    }
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
        const bool in = 2 * (kp + 8 * i) < R;                            // R % 8 == 0
#pragma unroll
        for (int e = 0; e < 8; ++e) *(h16x2 *)(sw + (8 * g + e) * ROW + 2 * (kp + 8 * i)) = in ? h16x2{wr[i][0][e], wr[i][1][e]} : h16x2{};
    }
    __syncthreads();
    f32x4 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        const h16 *row = sw + (64 * wave + 16 * (n >> 2) + 4 * b + (n & 3)) * ROW + 8 * q;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const h16x4 lo = *(const h16x4 *)(row + 32 * s), hi = *(const h16x4 *)(row + 32 * s + 4);
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(h16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]},
                                                           32 * s + 8 * q < R ? tf[s] : h16x8{}, acc[b], 0, 0, 0);
        }
    }
    float a0 = 0.f, a2 = 0.f;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const f32x4 u = acc[2 * p], v = acc[2 * p + 1];
        const h16x8 m = {(h16)u[0], (h16)u[1], (h16)u[2], (h16)u[3], (h16)v[0], (h16)v[1], (h16)v[2], (h16)v[3]};
        h16x8 k = __builtin_elementwise_fma(sd[p], mv[p] + m, xx[p]);
        if (scaled) {
            a0 = sum8(k, a0);
            a2 = dot8(k, yv[p], a2);
            k = k * rv[p];
        }
        if (t0 + n < a.T && live) *(h16x8 *)(a.out[j] + o + 8 * p) = k;
    }
    if (!scaled) return;
    a0 += __shfl_xor(a0, 16, WAVE);
    a2 += __shfl_xor(a2, 16, WAVE);
    a0 += __shfl_xor(a0, 32, WAVE);
    a2 += __shfl_xor(a2, 32, WAVE);
    if (lane < 16) { red[0][wave][lane] = live ? a0 : 0.f; red[1][wave][lane] = live ? a2 : 0.f; }
    __syncthreads();
    const int tok = threadIdx.x & 15, which = threadIdx.x >> 4;
    if (which < 2 && t0 + tok < a.T) {
        float *p = (which ? a.p2[j] : a.p0[j]) + (size_t)(t0 + tok) * a.npart;
        const float(&r)[4][16] = red[which];
        p[blockIdx.y] = ((r[0][tok] + r[1][tok]) + r[2][tok]) + r[3][tok];
        if (blockIdx.y == 0)
            for (int i = gridDim.y; i < a.npart; ++i) p[i] = 0.f;
    }
}
// Calls of up to 16 tokens keep the sums in index order, so that a conversation's first tokens come out as they did: a deep
// model whose state is nearly empty makes percents of its logits from the last bit of a mix.  The matrix cores gain 2 % of a
// call there.  One channel a thread: 5.4 / 6.0 / 6.1 us for 2 / 8 / 16 tokens of 4096 channels, four adjacent ones 6.3 / 6.6 / 6.7.
void v6_mix2_launch(const Mix2Args &a, bool mfma, hipStream_t st) {
    const auto kernel = !mfma ? v6_mix2_kernel<4> : a.R <= 32 ? v6_mix2_mfma_kernel<1> : v6_mix2_mfma_kernel<2>;
    const int tt = mfma ? 16 : 4;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.T + tt - 1) / tt), (unsigned)((a.C + 255) / 256), 5), dim3(256), 0, st, a);
}

struct Ws56 {
    rwkv_half *x, *xx, *sxd, *xxx, *t1, *mix[5], *d1, *d2, *r, *k, *v, *g, *att, *vx, *xs, *xx_att, *xx_ffn;
    float *sums, *splitk, *y32;
    float *parts;            // partial row sums handed from the key product's epilogue to the value product
    float *att_parts[4];     // RWKV-6: totals scratch + partial row sums of the scaled key / value / receptance / gate inputs
    rwkv_half *xs_side[3];   // scaled-activation scratch of the products that run beside the first one [T, C]
    float *sums_side[3];
    size_t total;
};

// partial sums per row that v6_mix2_mfma_kernel writes: one per block of 256 channels, rounded up to a multiple of four
int mix_parts(int64_t C) { return (int)((((C + 255) / 256) + 3) & ~(int64_t)3); }

Ws56 carve56(void *base, int64_t T, int64_t C, int64_t F, int64_t lm, int64_t ld) {
    Ws56 w;
    unsigned char *p = (unsigned char *)base;
    auto take = [&](size_t bytes) { void *q = p; p += align256(bytes); return (rwkv_half *)q; };
    const size_t tc = (size_t)T * C * 2, tf = (size_t)T * F * 2;
    w.x = take(tc); w.xx = take(tc); w.sxd = take(tc); w.xxx = take(tc);
    w.t1 = take((size_t)T * 5 * lm * 2);
    for (int j = 0; j < 5; ++j) w.mix[j] = take(tc);
    w.d1 = take((size_t)T * ld * 2); w.d2 = take(tc);
    w.r = take(tc); w.k = take(tc); w.v = take(tc); w.g = take(tc); w.att = take(tc);
    w.vx = take(tf); w.xs = take(tf > tc ? tf : tc);
    w.xx_att = take((size_t)C * 2); w.xx_ffn = take((size_t)C * 2);
    w.sums = (float *)take((size_t)T * 2 * sizeof(float));
    for (int j = 0; j < 3; ++j) {
        w.xs_side[j] = take(T > 1 ? tc : 256);
        w.sums_side[j] = (float *)take((size_t)T * 2 * sizeof(float));
    }
    w.splitk = (float *)take(RWKV_SPLITK_WS_BYTES);
    w.y32 = (float *)take(wkv56_scratch_bytes(T, C));
    w.parts = (float *)take(T > 1 ? (size_t)T * 2 * emitted_parts((int)F, EMIT_MIN_TN) * sizeof(float) : 256);
    for (int j = 0; j < 4; ++j) w.att_parts[j] = (float *)take(T > 1 ? (size_t)T * (2 + 2 * mix_parts(C)) * sizeof(float) : 256);
    w.total = (size_t)(p - (unsigned char *)base);
    return w;
}

bool mat_ok56(const rwkv_mat &m, bool u8, int64_t N, int64_t M) {
    if (!m.w || m.N != N || m.M != M || m.ld < N || !aligned16(m.w)) return false;
    if (u8) return m.mx && m.rx && m.my && m.ry && !(m.ld & 15) && aligned16(m.my) && aligned16(m.ry);
    return !(m.ld & 7);
}

}  // namespace

static int v56_check(const rwkv_v56_model *m) {
    if (!m || !m->layers || !m->emb || !m->ln_out_w || !m->ln_out_b) return RWKV_E_NULL;
    const int64_t C = m->n_embd, F = m->n_ffn, V = m->vocab;
    const int ver = m->version_x10;
    if (ver != 50 && ver != 51 && ver != 52 && ver != 60) return RWKV_E_DTYPE;
    if (m->n_layer <= 0 || C <= 0 || F <= 0 || V <= 0 || (C & 63) || (F & 63) || C > 8 * DTHREADS ||
        F > 8 * VP * DTHREADS || m->n_head * 64 != C)
        return RWKV_E_SHAPE;
    if (ver == 60 && (m->lora_maa <= 0 || m->lora_maa > 64 || (m->lora_maa * 5) % 8 || m->lora_decay % 64 ||
                      m->lora_decay <= 0))
        return RWKV_E_SHAPE;
    if (m->weights_u8 < 0 || m->weights_u8 > 2) return RWKV_E_DTYPE;
    for (int i = 0; i < m->n_layer; ++i) {
        const rwkv_v56_layer &l = m->layers[i];
        const bool u8 = mat_is_u8(m->weights_u8, l.att_key);   // one weight type per layer
        if (!l.ln1_w || !l.ln1_b || !l.ln2_w || !l.ln2_b || !l.time_decay || !l.time_first || !l.lnx_w || !l.lnx_b ||
            !l.ffn_mix_k || !l.ffn_mix_r)
            return RWKV_E_NULL;
        const int nmix = ver == 60 ? 6 : (ver == 50 ? 3 : 4);
        for (int j = 0; j < nmix; ++j)
            if (!l.att_mix[j]) return RWKV_E_NULL;
        if (ver == 60 && (!l.tm_w1 || !l.tm_w2 || !l.td_w1 || !l.td_w2)) return RWKV_E_NULL;
        if (!mat_ok56(l.att_key, u8, C, C) || !mat_ok56(l.att_value, u8, C, C) ||
            !mat_ok56(l.att_receptance, u8, C, C) || !mat_ok56(l.att_output, u8, C, C) ||
            (ver != 50 && !mat_ok56(l.att_gate, u8, C, C)) || !mat_ok56(l.ffn_key, u8, C, F) ||
            !mat_ok56(l.ffn_receptance, u8, C, C) || !mat_ok56(l.ffn_value, u8, F, C))
            return RWKV_E_LAYOUT;
    }
    if (!mat_ok56(m->head, mat_is_u8(m->weights_u8, m->head), C, V)) return RWKV_E_LAYOUT;
    return RWKV_OK;
}

extern "C" size_t rwkv_v56_workspace(const rwkv_v56_model *m, int64_t T) {
    if (!m || T <= 0) return 0;
    const int lm = m->lora_maa > 0 ? m->lora_maa : 32, ld = m->lora_decay > 0 ? m->lora_decay : 64;
    return carve56((void *)256, T, m->n_embd, m->n_ffn, lm, ld).total;
}

extern "C" int rwkv_v56_forward(const rwkv_v56_model *m, const rwkv_v56_layer_state *states, const int32_t *tokens,
                                int64_t T, int full_output, float *logits, void *workspace, size_t workspace_bytes,
                                void *stream) {
    int rc = v56_check(m);
    if (rc) return rc;
    int lb, le;
    if (!layer_range(m->n_layer, m->layer_begin, m->layer_end, lb, le)) return RWKV_E_SHAPE;
    const bool with_head = le == m->n_layer;
    if (!states || !tokens || (with_head && !logits) || !workspace) return RWKV_E_NULL;
    if (T <= 0 || T > (1 << 20)) return RWKV_E_SHAPE;
    if (workspace_bytes < rwkv_v56_workspace(m, T) || (((uintptr_t)workspace) & 255)) return RWKV_E_WORKSPACE;
    for (int i = lb; i < le; ++i) {
        const rwkv_v56_layer_state &s = states[i];
        if (!s.att_xx || !s.att_kv || !s.ffn_xx) return RWKV_E_NULL;
        if (!aligned16(s.att_xx) || !aligned16(s.ffn_xx)) return RWKV_E_LAYOUT;
    }
    hipStream_t st = (hipStream_t)stream;
    const int C = m->n_embd, F = m->n_ffn, H = m->n_head, ver = m->version_x10;
    const bool v6 = ver == 60, gated = ver != 50;
    const int lm = m->lora_maa, ld = m->lora_decay;
    Ws56 ws = carve56(workspace, T, C, F, v6 ? lm : 32, v6 ? ld : 64);
    Ctx c{st, false, T, num_cu(), ws.xs, ws.sums, ws.sums + T, ws.splitk, 0};
    // Sequence calls whose square products have more than 128 output tiles (none of them would split K) run
    // independent products side by side on two extra streams, each with its own activation scratch.  Shorter
    // calls are faster one product after the other with split-K (measured at 256 tokens, n_embd 4096).
    SideStreams *ss = (T / 128) * (C / 128) > 128 ? side_streams(st) : nullptr;
    Ctx cs[2] = {c, c};
    if (ss)
        for (int j = 0; j < 2; ++j) {
            cs[j].st = ss->s[j]; cs[j].xs = ws.xs_side[j]; cs[j].s0 = ws.sums_side[j]; cs[j].s2 = ws.sums_side[j] + T;
            cs[j].splitk = nullptr;
        }

    if (lb == 0 && (rc = gather_emb_launch(T, C, m->vocab, tokens, m->emb, ws.x, st))) return rc;
    for (int i = lb; i < le; ++i) {
        const rwkv_v56_layer &l = m->layers[i];
        const rwkv_v56_layer_state &s = states[i];
        const bool u8 = mat_is_u8(m->weights_u8, l.att_key);
        // long calls: every product through the direct-to-LDS kernel, one after the other (its tiles take a whole
        // CU, so products side by side on several streams gain nothing)
        const bool dma_seq = T >= 512;
        const rwkv_half *kx, *vx, *rx, *gx = nullptr, *wx = nullptr;
        bool fuse_d1 = false, att_scaled = false;
        int att_np = 0;   // RWKV-6: > 0 = the mixes arrive scaled, with this many partial row sums each
        // receptance, key, value (and gate) as one grouped launch (see below)
        const bool grouped = T > 1 && (T >= 256 || (!ss && ((T + 127) / 128) * (C / 128) <= 128)) && !(C & 127);
        float *att_sums[4] = {ws.sums, ws.sums_side[0], ws.sums_side[1], ws.sums_side[2]};   // of kx, vx, rx, gx
        if (v6) {
            Mix2Args b{};
            if (T == 1) {
                // LN1 + xxx = xx + (prev - xx) * maa_x + the first LoRA product (tanh) in one launch
                LnMixArgs a{};
                a.x = ws.x; a.C = C; a.ln_w = l.ln1_w; a.ln_b = l.ln1_b; a.sx = s.att_xx; a.xx_tmp = ws.xx_att;
                a.mix[0] = l.att_mix[0]; a.mat[0] = MatDev{l.tm_w1, C, nullptr, nullptr, nullptr, nullptr};
                a.M[0] = 5 * lm; a.epi[0] = EPI_TANH; a.out[0] = ws.t1; a.maa_form = 1;
                lnmix1_small_launch(a, st);
                b.xx = ws.xx_att; b.sxd = nullptr; b.prev = s.att_xx;
            } else {
                Mix1Args a{(int)T, C, ws.x, l.ln1_w, l.ln1_b, s.att_xx, l.att_mix[0], ws.xx, ws.sxd, ws.xxx, s.att_xx};
                v6_mix1_launch(a, st);
                if ((rc = mm(c, lora_mat(l.tm_w1, C, 5 * lm), false, ws.xxx, ACT_TANH, nullptr, nullptr, 1.f, ws.t1))) return rc;
                b.xx = ws.xx; b.sxd = ws.sxd; b.prev = nullptr;
            }
            b.T = (int)T; b.C = C; b.R = lm; b.t1 = ws.t1; b.w2 = l.tm_w2;
            for (int j = 0; j < 5; ++j) { b.maa[j] = l.att_mix[1 + j]; b.out[j] = ws.mix[j]; }
            // uint8 matrices, the four products as one grouped direct-to-LDS launch: the mixing kernel writes their
            // inputs already scaled, with partial row sums that the grouped launch adds up -- no scaling pass
            const bool mfma = T > 16;
            if (mfma && u8 && grouped && handover_enabled()) {
                const rwkv_half *xin[4] = {ws.mix[3], ws.mix[1], ws.mix[2], ws.mix[4]};
                const rwkv_mat *mats[4] = {&l.att_receptance, &l.att_key, &l.att_value, &l.att_gate};
                void *outs[4] = {ws.r, ws.k, ws.v, ws.g};
                if (gemm_group_plan(true, 4, T, C, xin, mats, outs, true).kind == 2) {
                    att_np = mix_parts(C);
                    const rwkv_mat *mj[5] = {nullptr, &l.att_key, &l.att_value, &l.att_receptance, &l.att_gate};
                    b.npart = att_np;
                    for (int j = 1; j < 5; ++j) {
                        b.ry[j] = mj[j]->ry; b.my[j] = mj[j]->my;
                        b.p0[j] = ws.att_parts[j - 1] + 2 * T; b.p2[j] = b.p0[j] + (size_t)T * att_np;
                    }
                }
            }
            if (T == 1) hipLaunchKernelGGL(v6_mix2_kernel<1>, dim3(1, (unsigned)((C + 255) / 256), 5), dim3(256), 0, st, b);
            else v6_mix2_launch(b, mfma, st);
            wx = ws.mix[0]; kx = ws.mix[1]; vx = ws.mix[2]; rx = ws.mix[3]; gx = ws.mix[4];
            // one token: the first decay-LoRA stage rides at the end of the receptance / key / value / gate launch
            fuse_d1 = T == 1 && C <= 8 * 512;
            if (!fuse_d1 && (rc = mm(c, lora_mat(l.td_w1, C, ld), false, wx, ACT_TANH, nullptr, nullptr, 1.f, ws.d1))) return rc;
            if (T > 1 && (rc = mm(c, lora_mat(l.td_w2, ld, C), false, ws.d1, ACT_NONE, nullptr, nullptr, 1.f, ws.d2))) return rc;
        } else {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln1_w; a.ln_b = l.ln1_b; a.sx = s.att_xx;
            // sequence calls: row 0's workgroup commits the new state; one token: the r / k / v launch below does
            if (T == 1) a.xx_last = ws.xx_att; else a.state_out = s.att_xx;
            const int nj = gated ? 4 : 3;
            // sequence calls with uint8 matrices: the same launch scales each mix by its matrix's ry and sums the rows
            att_scaled = T > 1 && u8;
            const rwkv_mat *mt[4] = {&l.att_key, &l.att_value, &l.att_receptance, &l.att_gate};
            for (int j = 0; j < nj; ++j) {
                a.mix[j] = l.att_mix[j]; a.xs[j] = ws.mix[j];
                a.ry[j] = att_scaled ? mt[j]->ry : nullptr; a.my[j] = att_scaled ? mt[j]->my : nullptr;
                a.s0[j] = att_sums[j]; a.s2[j] = att_sums[j] + T;
            }
            if ((rc = lnmix_seq_launch(a, nj, st))) return rc;
            kx = ws.mix[0]; vx = ws.mix[1]; rx = ws.mix[2]; gx = gated ? ws.mix[3] : nullptr;
        }
        // one token: the first matrix call also commits the new token-shift state (all readers of the old one are done)
        if (T == 1 && C <= 8 * 512) {
            // one launch for the receptance, key, value (and gate) rows
            MultiVecArgs a{};
            a.N = C; a.M = C; a.nm = gated ? 4 : 3;
            a.vin[0] = rx; a.mat[0] = to_dev56(l.att_receptance); a.act[0] = VACT_F16; a.out[0] = ws.r;
            a.vin[1] = kx; a.mat[1] = to_dev56(l.att_key); a.act[1] = VACT_F16; a.out[1] = ws.k;
            a.vin[2] = vx; a.mat[2] = to_dev56(l.att_value); a.act[2] = VACT_F16; a.out[2] = ws.v;
            if (gated) { a.vin[3] = gx; a.mat[3] = to_dev56(l.att_gate); a.act[3] = VACT_SILU; a.out[3] = ws.g; }
            a.commit_src = ws.xx_att; a.commit_dst = s.att_xx; a.commit_n = C;
            if (fuse_d1) { a.xin = wx; a.xmat = l.td_w1; a.xm = ld; a.xout = ws.d1; }
            multi_vec_launch(u8, a, c.grid, st);
        } else {
            // One grouped launch at full depth for receptance, key, value (and gate): in short calls, where each
            // product alone would split K and need a reduction pass, and from 256 rows on, where the group goes
            // through the direct-to-LDS kernel (256 x 256 tiles, K split while the group has few tiles).
            if (grouped) {
                const int n = gated ? 4 : 3;
                const rwkv_half *xin[4] = {rx, kx, vx, gx};
                const rwkv_mat *mats[4] = {&l.att_receptance, &l.att_key, &l.att_value, &l.att_gate};
                void *outs[4] = {ws.r, ws.k, ws.v, ws.g};
                rwkv_half *xsc[4] = {ws.xs, ws.xs_side[0], ws.xs_side[1], ws.xs_side[2]};
                float *sm[4] = {ws.sums, ws.sums_side[0], ws.sums_side[1], ws.sums_side[2]};
                GemmEpi ep[4];
                for (int j = 0; j < 4; ++j) {
                    ep[j] = GemmEpi{};
                    ep[j].act = j == 3 ? ACT_SILU : ACT_NONE; ep[j].out_scale = 1.f; ep[j].out_dtype = RWKV_DT_F16;
                    ep[j].ldres = C; ep[j].ldgate = C;
                }
                float *smx[4] = {att_sums[2], att_sums[0], att_sums[1], att_sums[3]};
                float *smp[4] = {ws.att_parts[2], ws.att_parts[0], ws.att_parts[1], ws.att_parts[3]};
                if (att_np) rc = gemm_group_launch(u8, n, T, C, xin, mats, outs, ep, nullptr, smp, ws.splitk, st, att_np);
                else rc = gemm_group_launch(u8, n, T, C, xin, mats, outs, ep, att_scaled ? nullptr : xsc, att_scaled ? smx : sm,
                                            ws.splitk, st);
                if (rc) return rc;
            } else if (att_scaled) {
                if ((rc = mm_scaled(c, l.att_receptance, u8, rx, att_sums[2], att_sums[2] + T, ACT_NONE, nullptr, nullptr, 1.f, ws.r)) ||
                    (rc = mm_scaled(c, l.att_key, u8, kx, att_sums[0], att_sums[0] + T, ACT_NONE, nullptr, nullptr, 1.f, ws.k)) ||
                    (rc = mm_scaled(c, l.att_value, u8, vx, att_sums[1], att_sums[1] + T, ACT_NONE, nullptr, nullptr, 1.f, ws.v)))
                    return rc;
                if (gated && (rc = mm_scaled(c, l.att_gate, u8, gx, att_sums[3], att_sums[3] + T, ACT_SILU, nullptr, nullptr, 1.f, ws.g)))
                    return rc;
            } else {
            // receptance (then gate) on the caller's stream, key and value on the side streams
            ForkScope par(ss, st, 2, !dma_seq);
            Ctx cr = c;
            if (par) cr.splitk = nullptr;
            if ((rc = mm(cr, l.att_receptance, u8, rx, ACT_NONE, nullptr, nullptr, 1.f, ws.r, ws.xx_att, T == 1 ? s.att_xx : nullptr, C))) return rc;
            if ((rc = mm(par ? cs[0] : c, l.att_key, u8, kx, ACT_NONE, nullptr, nullptr, 1.f, ws.k))) return rc;
            if ((rc = mm(par ? cs[1] : c, l.att_value, u8, vx, ACT_NONE, nullptr, nullptr, 1.f, ws.v))) return rc;
            if (gated && (rc = mm(c, l.att_gate, u8, gx, ACT_SILU, nullptr, nullptr, 1.f, ws.g))) return rc;
            if (!par.join()) return (int)hipErrorUnknown;
            }
        }
        // one token of v6: the second decay LoRA product is done inside the WKV kernel
        const bool d2_fused = v6 && T == 1;
        if ((rc = wkv56_fused_launch(v6, (int)T, C, H, s.att_kv, ws.r, ws.k, ws.v,
                                     v6 ? (const void *)(d2_fused ? ws.d1 : ws.d2) : (const void *)l.time_decay, l.time_decay,
                                     l.time_first, l.lnx_w, l.lnx_b, gated ? ws.g : nullptr, ws.att, st,
                                     d2_fused ? l.td_w2 : nullptr, ld, ws.y32)))
            return rc;
        if ((rc = mm(c, l.att_output, u8, ws.att, ACT_RESIDUAL, ws.x, nullptr, 1.f, ws.x))) return rc;
        // ---- channel mix
        const float scale = (m->rescale_layer > 0 && (i + 1) % m->rescale_layer == 0) ? 0.5f : 1.f;
        if (T == 1) {
            // LN2 + token shift + receptance and key rows in one launch, then the value rows
            LnMixArgs a{};
            a.x = ws.x; a.C = C; a.ln_w = l.ln2_w; a.ln_b = l.ln2_b; a.sx = s.ffn_xx; a.xx_tmp = ws.xx_ffn;
            a.mix[0] = l.ffn_mix_r; a.mat[0] = to_dev56(l.ffn_receptance); a.M[0] = C; a.epi[0] = EPI_SIGMOID; a.out[0] = ws.r;
            a.mix[1] = l.ffn_mix_k; a.mat[1] = to_dev56(l.ffn_key); a.M[1] = F; a.epi[1] = EPI_RELU_SQ; a.out[1] = ws.vx;
            a.maa_form = v6 ? 1 : 0;
            lnmix2_launch(u8, a, c.grid, st);
            if ((rc = mm(c, l.ffn_value, u8, ws.vx, ACT_GATED_RESIDUAL, ws.x, ws.r, scale, ws.x, ws.xx_ffn, s.ffn_xx, C))) return rc;
            RWKV_LAUNCH_CHECK();
            continue;
        }
        // LN2 + token shift + the two mixes; for uint8 matrices the same launch scales each mix by its matrix's ry and
        // sums the rows, so the two products below need no scaling pass
        rwkv_half *fx[2] = {u8 ? ws.xs_side[0] : ws.mix[0], u8 ? ws.xs_side[1] : ws.mix[1]};
        float *fs[2] = {ws.sums_side[0], ws.sums_side[1]};
        {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln2_w; a.ln_b = l.ln2_b; a.sx = s.ffn_xx;
            a.xx_last = nullptr; a.state_out = s.ffn_xx; a.maa_form = v6 ? 1 : 0;
            a.mix[0] = l.ffn_mix_r; a.mix[1] = l.ffn_mix_k;
            const rwkv_mat *mt[2] = {&l.ffn_receptance, &l.ffn_key};
            for (int j = 0; j < 2; ++j) {
                a.ry[j] = u8 ? mt[j]->ry : nullptr; a.my[j] = u8 ? mt[j]->my : nullptr;
                a.xs[j] = fx[j]; a.s0[j] = fs[j]; a.s2[j] = fs[j] + T;
            }
            if ((rc = lnmix_seq_launch(a, 2, st))) return rc;
        }
        const rwkv_half *xrk[2] = {fx[0], fx[1]};
        const rwkv_mat *mrk[2] = {&l.ffn_receptance, &l.ffn_key};
        void *ork[2] = {ws.r, u8 ? ws.xs : ws.vx};
        GemmEpi erk[2] = {};
        erk[0].act = ACT_SIGMOID; erk[1].act = ACT_RELU_SQ;
        for (int j = 0; j < 2; ++j) { erk[j].out_scale = 1.f; erk[j].out_dtype = RWKV_DT_F16; }
        if ((T <= 128 && !(C & 127) && !(F & 127)) || gemm_group_pays(u8, 2, T, C, xrk, mrk, ork, erk, ws.splitk)) {
            // Receptance and key in one grouped launch: short calls, and where the cost model puts it first.  The key product
            // hands the value product its input scaled where it can.  8 layers, us, by the limit of 128 tokens before -> by
            // cost: RWKV-5.2, n_embd 2048, fp16, 140 tokens 891 -> 813, 333 1070 -> 1012; RWKV-6, 4096, uint8, 333 tokens 2929 ->
            // 2757, 200 and 1000 tokens, which stay two launches, 1951 and 5100 against 2032 and 5330 as one.
            int np = 0;
            if (u8)
                np = mm_pair_parts(gemm_group_plan(true, 2, T, C, xrk, mrk, ork, true), c, l.ffn_key, l.ffn_value, true, ACT_GATED_RESIDUAL,
                                   ws.x, ws.r, ws.x, ws.parts);
            if (np) {
                erk[1].emit_ry = l.ffn_value.ry; erk[1].emit_my = l.ffn_value.my;
                erk[1].emit_s0 = ws.parts; erk[1].emit_s2 = ws.parts + (size_t)T * np;
            } else {
                ork[1] = ws.vx;
            }
            if ((rc = gemm_group_launch(u8, 2, T, C, xrk, mrk, ork, erk, nullptr, fs, ws.splitk, st))) return rc;
            if ((rc = mm_pair_second(c, l.ffn_key, l.ffn_value, u8, ws.vx, ACT_GATED_RESIDUAL, ws.x, ws.r, scale, ws.x, ws.parts, np)))
                return rc;
        } else {
            // channel-mix receptance beside the key product (one after the other in long calls); the key product
            // hands the value product its input already scaled where both run through the direct-to-LDS kernel
            ForkScope par(ss, st, 1, !dma_seq);
            if ((rc = mm_scaled(par ? cs[0] : c, l.ffn_receptance, u8, fx[0], fs[0], fs[0] + T, ACT_SIGMOID, nullptr, nullptr,
                                1.f, ws.r)))
                return rc;
            Ctx ck = c;
            ck.small_tiles = par ? 1 : 0;
            int np = 0;
            if ((rc = mm_pair_first(ck, c, l.ffn_key, l.ffn_value, u8, fx[1], fs[1], fs[1] + T, ACT_RELU_SQ, ws.vx,
                                    ACT_GATED_RESIDUAL, ws.x, ws.r, ws.x, ws.parts, &np)))
                return rc;
            if (!par.join()) return (int)hipErrorUnknown;
            if ((rc = mm_pair_second(c, l.ffn_key, l.ffn_value, u8, ws.vx, ACT_GATED_RESIDUAL, ws.x, ws.r, scale, ws.x, ws.parts, np)))
                return rc;
        }
        RWKV_LAUNCH_CHECK();
    }
    // ---- head
    if (!with_head) return RWKV_OK;
    const bool u8 = mat_is_u8(m->weights_u8, m->head);
    const bool all_rows = full_output && T > 1;
    const int64_t TH = all_rows ? T : 1;
    const rwkv_half *xh = all_rows ? ws.x : ws.x + (size_t)(T - 1) * C;
    if (TH == 1) {
        lnhead_launch(u8, xh, C, m->ln_out_w, m->ln_out_b, to_dev56(m->head), m->vocab, logits, c.grid, st);
        RWKV_LAUNCH_CHECK();
        return RWKV_OK;
    }
    {
        SeqMixArgs a{};
        a.T = (int)TH; a.C = C; a.x = xh; a.ln_w = m->ln_out_w; a.ln_b = m->ln_out_b; a.sx = nullptr; a.xx_last = nullptr;
        a.mix[0] = nullptr; a.ry[0] = nullptr; a.my[0] = nullptr; a.xs[0] = ws.xx;
        if ((rc = lnmix_seq_launch(a, 1, st))) return rc;
    }
    const rwkv_half *A = ws.xx;
    GemmEpi e{};
    e.out_scale = 1.f; e.act = ACT_NONE; e.out_dtype = RWKV_DT_F32; e.splitk_ws = ws.splitk; e.splitk_bytes = RWKV_SPLITK_WS_BYTES;
    if (u8) {
        if ((rc = mm8_prepare_launch(TH, C, ws.xx, C, m->head.ry, m->head.my, ws.xs, ws.sums, ws.sums + T, st))) return rc;
        A = ws.xs;
        e.mx = m->head.mx; e.rx = m->head.rx; e.s0 = ws.sums; e.s2 = ws.sums + T;
    }
    return gemm_launch(u8, TH, C, m->vocab, A, C, m->head.w, m->head.ld, logits, m->vocab, e, st);
}
