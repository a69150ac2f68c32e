// RWKV-7 forward for any T >= 1 (fp16 weights, fp32 state and decay).
//
// Per layer: time mix
//   lnmix_seq (LN1, token shift, the six static mixes r, w, k, v, a, g)
//   r, k, v rows; LoRA pairs: w = tanh(xw @ W1) @ W2, a = (xa @ A1) @ A2, v-gate = (xv @ V1) @ V2,
//   g = sigmoid(xg @ G1) @ G2   -- mm(): streaming GEMV for one token, MFMA GEMM otherwise
//   prep7   per (token, head): a = sigmoid(a0 + .), kk = normalised k * k_k, k *= 1 + (a - 1) k_a,
//           v += (v_first - v) sigmoid(v0 + .), decay = exp(-e^-0.5 sigmoid(w0 + .)), bonus = sum r k r_k
//   wkv7    the state recurrence, a head's 64 value rows split over four workgroups
//   gn7     GroupNorm per head, + bonus * v, * g
//   output matrix with the residual add in its epilogue
// then the channel mix: LN2, one mix, relu(. @ K)^2 @ V with the residual add.
//
// One token (T == 1) runs five launches per layer instead:
//   att7_kernel    LN1 + token shift + the six mixes -> rows (Wr[c], Wk[c], Wv[c]) per wave, then the rows of
//                  the four first LoRA stages (tanh / none / none / sigmoid)
//   tmix7_kernel   per head: second LoRA stages, the preparation above, one step of the recurrence,
//                  GroupNorm, bonus and gate
//   vec_kernel     rows of Wo, x += out
//   lnmix_kernel   LN2 + token shift + mix -> rows of the channel-mix key matrix, relu^2
//   vec_kernel     rows of the channel-mix value matrix, x += out
#include <algorithm>
#include "mm_dispatch.h"

namespace {

constexpr int HS7 = 64;   // head size
constexpr int TS7 = 32;   // tokens staged in LDS per slab

struct Prep7Args {
    int T, C, H;
    const rwkv_half *r;
    rwkv_half *k, *v;                         // updated in place
    const rwkv_half *w_raw, *a_raw, *vg_raw;  // LoRA outputs [T, C]; vg_raw NULL in layer 0
    const rwkv_half *v_first;                 // [T, C] value of layer 0 (NULL in layer 0)
    const rwkv_half *w0, *a0, *v0, *k_k, *k_a, *r_k;
    rwkv_half *an, *b;                        // -kk and kk * a
    float *dec;                               // decay in (0, 1)
    float *rk;                                // [T, H] bonus factor, fp16-rounded
};

// Eight adjacent channels per lane (16-byte accesses), so the eight lanes of a row of eight own one head of one
// token: a workgroup has 256 of the C / 8 chunks of one row.  Every step rounds to fp16 where an fp16 tensor operation of the
// reference does; the two sums over a head run over a lane's eight channels in index order and then over the
// eight lanes in three DPP steps.
DEV float head8_sum(float v) {
    v += dpp_mov<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_mov<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp_mov<0x141>(v);   // row_half_mirror: the other quad of the eight
    return v;
}

__global__ __launch_bounds__(256) void prep7_kernel(int per_row, uint64_t factor, Prep7Args a) {
    const int cpr = a.C / 8;   // chunks per token row
    {
        // whole waves take part in the DPP sums: chunks past the end of the row repeat its last one and store nothing
        const int t = div_by(blockIdx.x, factor), i = ((int)blockIdx.x - t * per_row) * 256 + threadIdx.x;
        const bool live = i < cpr;
        const int c = min(i, cpr - 1) * 8;
        const size_t o = (size_t)t * a.C + c;
        const h16x8 r8 = *(const h16x8 *)(a.r + o), k8 = *(const h16x8 *)(a.k + o), v8 = *(const h16x8 *)(a.v + o);
        const h16x8 ar8 = *(const h16x8 *)(a.a_raw + o), wr8 = *(const h16x8 *)(a.w_raw + o);
        h16x8 vg8 = {}, vf8 = {}, v08 = {};
        if (a.vg_raw) { vg8 = *(const h16x8 *)(a.vg_raw + o); vf8 = *(const h16x8 *)(a.v_first + o); v08 = *(const h16x8 *)(a.v0 + c); }
        const h16x8 a08 = *(const h16x8 *)(a.a0 + c), kk8 = *(const h16x8 *)(a.k_k + c), ka8 = *(const h16x8 *)(a.k_a + c);
        const h16x8 w08 = *(const h16x8 *)(a.w0 + c), rk8 = *(const h16x8 *)(a.r_k + c);
        float av[8], kku[8], k2[8], ss = 0.f, rks = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float k = (float)k8[e];
            av[e] = round_h(sigmoidf_(round_h((float)a08[e] + (float)ar8[e])));
            kku[e] = round_h(k * (float)kk8[e]);
            ss += kku[e] * kku[e];
            k2[e] = round_h(k * round_h(1.f + round_h(round_h(av[e] - 1.f) * (float)ka8[e])));
            rks += round_h(round_h((float)r8[e] * k2[e]) * (float)rk8[e]);
        }
        const float nrm = fmaxf(round_h(sqrtf(head8_sum(ss))), 1e-12f);
        rks = head8_sum(rks);
        h16x8 ko, ano, bo, vo = v8;
        f32x4 d0, d1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float kk = round_h(kku[e] / nrm);
            if (a.vg_raw) {
                const float v = (float)v8[e];
                const float sg = round_h(sigmoidf_(round_h((float)v08[e] + (float)vg8[e])));
                vo[e] = (h16)(v + round_h(round_h((float)vf8[e] - v) * sg));
            }
            const float z = round_h((float)w08[e] + (float)wr8[e]);
            const float dec = __expf(-0.606531f * sigmoidf_(z));
            if (e < 4) d0[e] = dec; else d1[e - 4] = dec;
            ko[e] = (h16)k2[e];
            ano[e] = (h16)(-kk);
            bo[e] = (h16)(kk * av[e]);
        }
        if (live) {
            if (a.vg_raw) *(h16x8 *)(a.v + o) = vo;
            *(f32x4 *)(a.dec + o) = d0;
            *(f32x4 *)(a.dec + o + 4) = d1;
            *(h16x8 *)(a.k + o) = ko;
            *(h16x8 *)(a.an + o) = ano;
            *(h16x8 *)(a.b + o) = bo;
            if (!(c & (HS7 - 1))) a.rk[t * a.H + c / HS7] = round_h(rks);
        }
    }
}

struct Wkv7Args {
    int T, C;
    float *state;                       // [H][value i][key j]
    const void *r, *w, *k, *v, *a, *b;  // [T, C]
    void *y;                            // [T, C]
};

// A head's value rows never interact (sa_i, y_i and row i of the state depend on v_i only), so a head is
// split over four workgroups of 16 value rows.  Thread (value i, key group g): lane & 15 = g owns keys
// 4g..4g+3 of row i; sums over a row's 16 key groups are DPP row sums in registers, so the token loop has
// no barrier.  r, w, k, a, b of a slab of tokens are staged in LDS as fp32.
// The only loop-carried chain is state -> sa -> state.  The read-out is taken off it by expanding
//     y_i = sum_j S'_ij r_j = sum_j S_ij (w_j r_j) + v_i (k . r) + sa_i (b . r)
// so that both row sums of a token run on the OLD state side by side; k . r and b . r are per-token
// scalars computed while staging.
//   DT:     element type of r, k, v, a, b (and of w, y in the operator form): RWKV_DT_F16, RWKV_DT_F32 or RWKV_DT_BF16
//   MODEL:  w is the fp32 decay itself and y an fp32 scratch; otherwise w is the log-decay
//           (decay = exp(-exp(w))) and y has the input type
// Staging: thread (token tid / 8, channels 8 (tid % 8) ..+7) loads its share of the NEXT slab into
// registers before the token loop of the current one, so the loads' latency is hidden behind the loop.
// bf16 <-> fp32: the upper half of the fp32 pattern; stores round to nearest even (NaN stays NaN)
DEV float bf2f(uint16_t v) { return __builtin_bit_cast(float, (uint32_t)v << 16); }
DEV uint16_t f2bf(float f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

template <int DT>
struct Stage7 {
    float r[8], k[8], a[8], b[8], w[8], v[2];

    DEV void load8(const void *p, size_t o, float (&d)[8]) {
        if (DT == RWKV_DT_F16) {
            const h16x8 x = *(const h16x8 *)((const rwkv_half *)p + o);
#pragma unroll
            for (int e = 0; e < 8; ++e) d[e] = (float)x[e];
        } else if (DT == RWKV_DT_BF16) {
            const u32x4 x = *(const u32x4 *)((const uint16_t *)p + o);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d[2 * e] = __builtin_bit_cast(float, x[e] << 16);
                d[2 * e + 1] = __builtin_bit_cast(float, x[e] & 0xffff0000u);
            }
        } else {
            const f32x4 x0 = *(const f32x4 *)((const float *)p + o), x1 = *(const f32x4 *)((const float *)p + o + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { d[e] = x0[e]; d[4 + e] = x1[e]; }
        }
    }
};

template <int DT, bool MODEL>
__global__ __launch_bounds__(256) void wkv7_kernel(Wkv7Args a) {
    __shared__ __align__(16) float swr[TS7][HS7], sk[TS7][HS7], sw[TS7][HS7], sa[TS7][HS7], sb[TS7][HS7];
    __shared__ float sv[TS7][16], skr[TS7], sbr[TS7];
    const int T = a.T, C = a.C;
    const int h = blockIdx.x >> 2, vb = blockIdx.x & 3;
    const int lane = threadIdx.x & 63, g = lane & 15;
    const int il = (threadIdx.x >> 6) * 4 + (lane >> 4);
    const int i = vb * 16 + il;
    const int stt = threadIdx.x >> 3, sc = (threadIdx.x & 7) * 8;   // staging role
    float *S = a.state + (size_t)h * HS7 * HS7 + (size_t)i * HS7 + 4 * g;
    f32x4 s = *(const f32x4 *)S;
    Stage7<DT> st;
    auto fetch = [&](int t0) {
        const size_t o = (size_t)min(t0 + stt, T - 1) * C + h * HS7;   // rows past the end re-read the last one
        st.load8(a.r, o + sc, st.r);
        st.load8(a.k, o + sc, st.k);
        st.load8(a.a, o + sc, st.a);
        st.load8(a.b, o + sc, st.b);
        if (MODEL) {
            const f32x4 x0 = *(const f32x4 *)((const float *)a.w + o + sc), x1 = *(const f32x4 *)((const float *)a.w + o + sc + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { st.w[e] = x0[e]; st.w[4 + e] = x1[e]; }
        } else {
            st.load8(a.w, o + sc, st.w);
        }
        const size_t ov = o + vb * 16 + 2 * (threadIdx.x & 7);
        if (DT == RWKV_DT_F16) {
            const h16x2 x = *(const h16x2 *)((const rwkv_half *)a.v + ov);
            st.v[0] = (float)x[0]; st.v[1] = (float)x[1];
        } else if (DT == RWKV_DT_BF16) {
            const uint32_t x = *(const uint32_t *)((const uint16_t *)a.v + ov);
            st.v[0] = __builtin_bit_cast(float, x << 16); st.v[1] = __builtin_bit_cast(float, x & 0xffff0000u);
        } else {
            st.v[0] = ((const float *)a.v)[ov]; st.v[1] = ((const float *)a.v)[ov + 1];
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < T; t0 += TS7) {
        const int nt = min(TS7, T - t0);
        __syncthreads();  // previous slab fully consumed
        {
            float kr = 0.f, br = 0.f;
            f32x4 o4[5][2];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float w = MODEL ? st.w[e] : __expf(-__expf(st.w[e]));
                o4[0][e >> 2][e & 3] = w * st.r[e];
                o4[1][e >> 2][e & 3] = st.k[e];
                o4[2][e >> 2][e & 3] = w;
                o4[3][e >> 2][e & 3] = st.a[e];
                o4[4][e >> 2][e & 3] = st.b[e];
                kr += st.k[e] * st.r[e];
                br += st.b[e] * st.r[e];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                *(f32x4 *)&swr[stt][sc + 4 * u] = o4[0][u];
                *(f32x4 *)&sk[stt][sc + 4 * u] = o4[1][u];
                *(f32x4 *)&sw[stt][sc + 4 * u] = o4[2][u];
                *(f32x4 *)&sa[stt][sc + 4 * u] = o4[3][u];
                *(f32x4 *)&sb[stt][sc + 4 * u] = o4[4][u];
            }
            sv[stt][2 * (threadIdx.x & 7)] = st.v[0];
            sv[stt][2 * (threadIdx.x & 7) + 1] = st.v[1];
            // the 8 threads of a token are 8 consecutive lanes: three DPP steps
            kr += dpp_mov<0xB1>(kr); br += dpp_mov<0xB1>(br);
            kr += dpp_mov<0x4E>(kr); br += dpp_mov<0x4E>(br);
            kr += dpp_mov<0x141>(kr); br += dpp_mov<0x141>(br);
            if ((threadIdx.x & 7) == 0) { skr[stt] = kr; sbr[stt] = br; }
        }
        __syncthreads();
        fetch(t0 + TS7);
        struct Tok { float vi, kr, br; f32x4 wr4, k4, w4, a4, b4; };
        auto ldtok = [&](int tt) {
            Tok q;
            q.vi = sv[tt][il]; q.kr = skr[tt]; q.br = sbr[tt];
            q.wr4 = *(const f32x4 *)&swr[tt][4 * g];
            q.k4 = *(const f32x4 *)&sk[tt][4 * g];
            q.w4 = *(const f32x4 *)&sw[tt][4 * g];
            q.a4 = *(const f32x4 *)&sa[tt][4 * g];
            q.b4 = *(const f32x4 *)&sb[tt][4 * g];
            return q;
        };
        // state update of one token; returns this thread's share of the read-out sum, p = the summed sa term
        auto advance = [&](const Tok &q, float &p) {
            p = (q.a4[0] * s[0] + q.a4[1] * s[1]) + (q.a4[2] * s[2] + q.a4[3] * s[3]);
            const float yw = (q.wr4[0] * s[0] + q.wr4[1] * s[1]) + (q.wr4[2] * s[2] + q.wr4[3] * s[3]);
            f32x4 kv;
#pragma unroll
            for (int e = 0; e < 4; ++e) kv[e] = s[e] * q.w4[e] + q.k4[e] * q.vi;
            p = row16_sum(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = kv[e] + p * q.b4[e];
            return yw;
        };
        auto store = [&](const Tok &q, int tt, float yw, float p) {
            if (g == 0) {
                const float y = yw + q.vi * q.kr + p * q.br;
                const size_t o = (size_t)(t0 + tt) * C + h * HS7 + i;
                if (MODEL || DT == RWKV_DT_F32) ((float *)a.y)[o] = y;
                else if (DT == RWKV_DT_BF16) ((uint16_t *)a.y)[o] = f2bf(y);
                else ((rwkv_half *)a.y)[o] = f2h(y);
            }
        };
        // PASS tokens per pass (TS7 % PASS == 0): their LDS reads are issued together, so the read latency is paid once
        // per pass; in a full pass the read-out row sums, which are not on the state chain, run interleaved after the
        // state updates
        constexpr int PASS = 4;   // 8 was slower here (138 against 128 us per 1024 tokens): 23 operand registers per token
        for (int tt = 0; tt < nt; tt += PASS) {
            Tok q[PASS];
#pragma unroll
            for (int u = 0; u < PASS; ++u) q[u] = ldtok(tt + u);
            float yw[PASS], p[PASS];
            if (tt + PASS - 1 < nt) {
#pragma unroll
                for (int u = 0; u < PASS; ++u) yw[u] = advance(q[u], p[u]);
#pragma unroll
                for (int u = 0; u < PASS; ++u) yw[u] = row16_sum(yw[u]);
#pragma unroll
                for (int u = 0; u < PASS; ++u) store(q[u], tt + u, yw[u], p[u]);
            } else {
#pragma unroll
                for (int u = 0; u < PASS - 1; ++u)
                    if (tt + u < nt) {
                        yw[u] = row16_sum(advance(q[u], p[u]));
                        store(q[u], tt + u, yw[u], p[u]);
                    }
            }
        }
    }
    *(f32x4 *)S = s;
}

// ---- the recurrence over a long sequence, model path, in chunks of 16 tokens -----------------------------------
// With A_t the product of the decays of the chunk's tokens up to and including t, S (keys x values) the state the chunk
// starts from and u_t = the row sa of token t,
//     u_t = (a_t . A_{t-1}) S + sum_{s<t} (AK_ts v_s + AB_ts u_s),    y_t = (r_t . A_t) S + sum_{s<=t} (QK_ts v_s + QB_ts u_s)
//     S'  = A_16 S + sum_s (k_s . A_16/A_s) v_s^T + (b_s . A_16/A_s) u_s^T
// (AK_ts = sum_j a_tj k_sj A_{t-1,j}/A_sj, QK with r_t and A_t, AB and QB with b_s.)  u is a unit lower triangular system,
// so with Z = (I - AB)^-1 everything that needs no S can be formed for all chunks at once:
//     u = TA S + TK v,   TA = Z (a . A),  TK = Z AK;      y = Y1 S + Y2 v,   Y1 = r . A + QB TA,  Y2 = QK + QB TK.
// The decays of this model lie in (0.545, 1) (exp(-e^-0.5 sigmoid)), so A_16 >= 6e-5 and the quotients by A_s are safe
// in fp32 and as exact as the products they replace.
//   wkv7_chunk_kernel  one workgroup per (head, chunk): the preparation of prep7_kernel for its 16 tokens, then Y1, TA,
//                      Y2, TK and the decayed k and b.  The four matrices and the products with Z and QB are
//                      v_mfma_f32_16x16x4_f32 (fp32 operands and sums).
//   wkv7_apply_kernel  workgroup (head, 16 values), wave jb = keys 16 jb .. + 15: one 16 x 16 block of S in MFMA
//                      accumulators for the whole call.  Operands arrive in fragment order, PD chunks in flight; the
//                      four waves' shares of u and y meet in LDS, one barrier per chunk.
// Values that are not finite count as 0 in TK v and Y2 v, as in the chunks of RWKV-5/6 (wkv.hip); other operands that are
// not finite are kept from the tokens before them where the first kernel forms its products.
// 20 KB of fp32 operands pass from one to the other per head and chunk.  The first kernel moves them at 3.0 TB/s of a
// copy's 4.8: about 1000 vector instructions a wave, a third of them the five exact divisions per element, six barriers and
// the forward substitution of one wave beside three that wait.  Six workgroups a CU, by its 78 registers, against five by 30 KB
// of LDS, and no chunks past the last: 777 tokens 39.3 -> 37 us (and 32 since the vectors
// are requested together).  The second is a chain of one exchange per chunk (35 us, 0.72 a chunk).  A
// 4096-wide layer, both together: 260 tokens 321 -> 314.5 us, 777 561.5 -> 557, 1024 the same.  Per layer at 64 heads,
// preparation and recurrence, token by token -> chunks: 1024 tokens 152 -> 89 us, 777 tokens 116 -> 72, 256 tokens 42 -> 31,
// 100 tokens 21 -> 19; at 64 tokens the two launches take as long as prep7_kernel and wkv7_kernel: CHUNKED7.
constexpr int SEG7 = 1024;        // tokens per pair of launches: bounds the scratch between them
constexpr int CHUNKED7 = 96;      // calls of at least so many tokens run in chunks
// one chunk's operands, in floats: Y1, TA, decayed k, decayed b as [key block][lane][4]; (Y2, TK) as [key block][lane][2];
// A_16 [64]; the values (fp16) as [value block][lane][4].  Lane = token or key or value, + 16 q; inner index 4 q + e.
constexpr int C7_Y1 = 0, C7_TA = 1024, C7_K = 2048, C7_B = 3072, C7_2 = 4096, C7_A = C7_2 + 512, C7_V = C7_A + 64, C7_FLOATS = C7_V + 512;
constexpr int LR7 = 68;           // LDS row of 64 floats, padded: 16 rows hit 16 different bank groups
constexpr int LM7 = 20;           // LDS row of 16 floats, padded

__global__ __launch_bounds__(256) void wkv7_chunk_kernel(Prep7Args a, int t_begin, float *__restrict__ scratch) {
    __shared__ __align__(16) float la[CL][LR7], lr[CL][LR7], lk[CL][LR7], lb[CL][LR7];   // a . A, r . A, k / A, b / A
    // 22 KB in all, room for seven workgroups a CU (the registers leave six): A_16 in the pads of la, piece g in row g; the decays where the
    // matrices come, Z over the rows of AB that it has used, the values at last over Z and QB
    __shared__ __align__(16) float mat[4][CL][LM7];
    constexpr int AK = 0, QK = 1, AB = 2, QB = 3;
    float (*const lw)[HS7] = (float (*)[HS7])&mat[0][0][0];
    float (*const lz)[LM7] = mat[AB];
    h16 *const lv = (h16 *)&mat[AB][0][0];
    static_assert(CL * HS7 <= 4 * CL * LM7 && CL * HS7 * sizeof(h16) <= 2 * CL * LM7 * sizeof(float) && LR7 == HS7 + 4, "");
    const int H = a.H, C = a.C, T = a.T;
    const int h = blockIdx.x % H, c = blockIdx.x / H;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s = tid >> 4, g = tid & 15;                 // token of the chunk, channels 4 g .. + 3 of the head
    float *out = scratch + (size_t)blockIdx.x * C7_FLOATS;
    const int t = t_begin + c * CL + s;
    const bool live = t < T;                              // past the end: r = k = a = b = v = 0, w = 1
    const int ch = h * HS7 + 4 * g;
    const size_t o = (size_t)min(t, T - 1) * C + ch;
    // ---- preparation, rounding by rounding as in prep7_kernel
    const h16x4 r4 = *(const h16x4 *)(a.r + o), k4 = *(const h16x4 *)(a.k + o), v4 = *(const h16x4 *)(a.v + o);
    const h16x4 ar4 = *(const h16x4 *)(a.a_raw + o), wr4 = *(const h16x4 *)(a.w_raw + o);
    // The vectors, on any boundary of two bytes, are requested here too: read where they are used, in branches, eight of the reads were a trip
    // to memory each, one after the other: 777 tokens of 4096 channels 36.4 -> 32.3 us, 1024 46.3 -> 40.3, 300 17.8 -> 16.2.
    typedef h16x4 h16x4_any __attribute__((aligned(2)));
    auto vec4 = [&](const rwkv_half *p) -> h16x4 { return *(const h16x4_any *)(p + ch); };
    const h16x4 a04 = vec4(a.a0), kk4 = vec4(a.k_k), ka4 = vec4(a.k_a), rk4 = vec4(a.r_k), w04 = vec4(a.w0), v04 = vec4(a.vg_raw ? a.v0 : a.a0);
    h16x4 vg4 = {}, vf4 = {};
    if (a.vg_raw) { vg4 = *(const h16x4 *)(a.vg_raw + o); vf4 = *(const h16x4 *)(a.v_first + o); }
    float kku[4], av[4], k2[4], ss = 0.f, rks = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float k = (float)k4[e];
        av[e] = round_h(sigmoidf_(round_h((float)a04[e] + (float)ar4[e])));
        kku[e] = round_h(k * (float)kk4[e]);
        ss += kku[e] * kku[e];
        k2[e] = round_h(k * round_h(1.f + round_h(round_h(av[e] - 1.f) * (float)ka4[e])));
        rks += round_h(round_h((float)r4[e] * k2[e]) * (float)rk4[e]);
    }
    const float nrm = fmaxf(round_h(sqrtf(row16_sum(ss))), 1e-12f);
    rks = row16_sum(rks);
    f32x4 w, rr, kk2, aa, bb;
    h16x4 vo = v4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float kk = round_h(kku[e] / nrm);
        if (a.vg_raw) {
            const float v = (float)v4[e];
            const float sg = round_h(sigmoidf_(round_h((float)v04[e] + (float)vg4[e])));
            vo[e] = (h16)(v + round_h(round_h((float)vf4[e] - v) * sg));
        }
        w[e] = live ? __expf(-0.606531f * sigmoidf_(round_h((float)w04[e] + (float)wr4[e]))) : 1.f;
        rr[e] = live ? (float)r4[e] : 0.f;
        kk2[e] = live ? k2[e] : 0.f;
        aa[e] = live ? -kk : 0.f;
        bb[e] = live ? round_h(kk * av[e]) : 0.f;
    }
    if (live) {
        if (a.vg_raw) *(h16x4 *)(a.v + o) = vo;
        if (g == 0) a.rk[(size_t)t * H + h] = round_h(rks);
    }
    *(f32x4 *)&lw[s][4 * g] = w;
    __syncthreads();
    // ---- decays: before = A_{s-1}; a wave holds the tokens 4 wave .. + 3
    f32x4 before = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int m = 0; m < CL - 1; ++m) {
        if (m >= 4 * wave + 3) continue;
        const f32x4 wm = *(const f32x4 *)&lw[m][4 * g];
        before = m < 4 * wave || m < s ? before * wm : before;
    }
    const f32x4 upto = before * w;
    f32x4 inv;
#pragma unroll
    for (int e = 0; e < 4; ++e) inv[e] = 1.f / upto[e];
    *(f32x4 *)&la[s][4 * g] = aa * before;
    *(f32x4 *)&lr[s][4 * g] = rr * upto;
    *(f32x4 *)&lk[s][4 * g] = kk2 * inv;
    *(f32x4 *)&lb[s][4 * g] = bb * inv;
    if (s == CL - 1) {
        *(f32x4 *)(out + C7_A + 4 * g) = upto;
        *(f32x4 *)&la[g][HS7] = upto;
    }
    __syncthreads();
    // ---- wave 0: AK, 1: AB, 2: QK, 3: QB.  Row t in the first operand's lanes, s in the second's; D: column s = lane & 15,
    // rows t = 4 q + e
    const int n16 = lane & 15, q = lane >> 4;
    {
        const float (*left)[LR7] = wave < 2 ? la : lr, (*right)[LR7] = wave & 1 ? lb : lk;
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const f32x4 x = *(const f32x4 *)&left[n16][16 * b + 4 * q], y = *(const f32x4 *)&right[n16][16 * b + 4 * q];
#pragma unroll
            for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], d, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 4 * q + e;
            mat[wave >> 1 | (wave & 1) << 1][row][n16] = (wave < 2 ? n16 < row : n16 <= row) ? d[e] : 0.f;
        }
    }
    __syncthreads();
    // ---- Z = (I - AB)^-1 by forward substitution, a column per lane (the four lane groups of wave 0 do the same)
    if (wave == 0) {
        float z[CL];
#pragma unroll
        for (int row = 0; row < CL; ++row) {
            float p[2] = {row == n16 ? 1.f : 0.f, 0.f};
#pragma unroll
            for (int m4 = 0; m4 < row; m4 += 4) {
                const f32x4 x = *(const f32x4 *)&mat[AB][row][m4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m4 + e < row) p[e & 1] = __builtin_fmaf(x[e], z[m4 + e], p[e & 1]);
            }
            z[row] = p[0] + p[1];
            if (q == 0) lz[row][n16] = z[row];
        }
    }
    __syncthreads();
    // ---- wave b: columns 16 b .. of TA = Z (a . A) and Y1 = r . A + QB TA (a D register is the next product's second
    // operand); wave 1 also TK = Z AK and Y2 = QK + QB TK
    const f32x4 zf = *(const f32x4 *)&lz[n16][4 * q], qb = *(const f32x4 *)&mat[QB][n16][4 * q];
    f32x4 ta = {0.f, 0.f, 0.f, 0.f}, y1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        ta = __builtin_amdgcn_mfma_f32_16x16x4f32(zf[e], la[4 * q + e][16 * wave + n16], ta, 0, 0, 0);
        y1[e] = lr[4 * q + e][16 * wave + n16];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qb[e], ta[e], y1, 0, 0, 0);
    f32x4 tk = {0.f, 0.f, 0.f, 0.f}, y2 = tk;
    if (wave == 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            tk = __builtin_amdgcn_mfma_f32_16x16x4f32(zf[e], mat[AK][4 * q + e][n16], tk, 0, 0, 0);
            y2[e] = mat[QK][4 * q + e][n16];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) y2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qb[e], tk[e], y2, 0, 0, 0);
    }
    // A token that is not finite: the products above multiplied it by the zeros of Z and QB for the tokens before it.  Once
    // more without those.
    const f32x4 sum = (ta + y1) + (tk + y2);
    if (__builtin_amdgcn_ballot_w64(!__builtin_isfinite((sum[0] + sum[1]) + (sum[2] + sum[3])))) {
        // rows t of L times the rows m <= t of x, which lane (column, q) holds four of
        auto add = [&](f32x4 d, const float (*L)[LM7], f32x4 x) {
#pragma unroll
            for (int m = 0; m < CL; ++m) {
                const float xm = __shfl(x[m & 3], n16 + 16 * (m >> 2), WAVE);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m <= 4 * q + e) d[e] = __builtin_fmaf(L[4 * q + e][m], xm, d[e]);
            }
            return d;
        };
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 x, y;
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[e] = la[4 * q + e][16 * wave + n16]; y[e] = lr[4 * q + e][16 * wave + n16]; }
        ta = add(zero, lz, x);
        y1 = add(y, mat[QB], ta);
        if (wave == 1) {
#pragma unroll
            for (int e = 0; e < 4; ++e) { x[e] = mat[AK][4 * q + e][n16]; y[e] = mat[QK][4 * q + e][n16]; }
            tk = add(zero, lz, x);
            y2 = add(y, mat[QB], tk);
        }
    }
    __syncthreads();
    // ---- to fragment order through LDS
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        la[4 * q + e][16 * wave + n16] = ta[e];
        lr[4 * q + e][16 * wave + n16] = y1[e];
        if (wave == 1) { mat[AK][4 * q + e][n16] = tk[e]; mat[QK][4 * q + e][n16] = y2[e]; }
        lv[256 * (g >> 2) + 4 * (4 * (g & 3) + e + 16 * (s >> 2)) + (s & 3)] = live ? vo[e] : (h16)0.f;
    }
    const f32x4 rest = *(const f32x4 *)&la[g][HS7] * inv;                          // A_16 / A_s
    *(f32x4 *)&lk[s][4 * g] = kk2 * rest;
    *(f32x4 *)&lb[s][4 * g] = bb * rest;
    __syncthreads();
    *(f32x4 *)(out + C7_Y1 + 4 * tid) = *(const f32x4 *)&lr[n16][16 * wave + 4 * q];
    *(f32x4 *)(out + C7_TA + 4 * tid) = *(const f32x4 *)&la[n16][16 * wave + 4 * q];
    f32x4 kf, bf;
#pragma unroll
    for (int e = 0; e < 4; ++e) { kf[e] = lk[4 * q + e][16 * wave + n16]; bf[e] = lb[4 * q + e][16 * wave + n16]; }
    *(f32x4 *)(out + C7_K + 4 * tid) = kf;
    *(f32x4 *)(out + C7_B + 4 * tid) = bf;
    // wave jb of the second kernel takes the inner indices 4 q + jb of Y2 and TK
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    *(f32x2 *)(out + C7_2 + 2 * tid) = f32x2{mat[QK][n16][4 * q + wave], mat[AK][n16][4 * q + wave]};
    *(h16x4 *)((h16 *)(out + C7_V) + 4 * tid) = *(const h16x4 *)(lv + 4 * tid);
}

__global__ __launch_bounds__(256, 2) void wkv7_apply_kernel(int H, int C, float *state, float *y32, int t_begin, int nchunk, const float *scratch) {
    __shared__ f32x4 redu[2][4][64], redy[2][4][64];
    const int h = blockIdx.x % H, ib = blockIdx.x / H;
    const int lane = threadIdx.x & 63, jb = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15, q = lane >> 4;
    const int i = 16 * ib + n16;                            // value column of the accumulators
    float *S = state + (size_t)h * HS7 * HS7 + (size_t)i * HS7 + 16 * jb + 4 * q;   // [value][key]
    f32x4 st = *(const f32x4 *)S;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    struct Ops { f32x4 ta, y1, k, b, al; f32x2 two; h16x4 v; };
    const uint32_t o16 = (256 * jb + 4 * lane) * 4, o2 = (C7_2 + 128 * jb + 2 * lane) * 4, oa = (C7_A + 16 * jb + 4 * q) * 4,
                   ov = C7_V * 4 + (256 * ib + 4 * lane) * 2;
    auto load = [&](Ops &x, int c) {     // the base is the same for the whole wave, the offsets never change
        const char *in = (const char *)(scratch + ((size_t)min(c, nchunk - 1) * H + h) * C7_FLOATS);
        x.ta = *(const f32x4 *)(in + C7_TA * 4 + o16);
        x.two = *(const f32x2 *)(in + o2);
        x.v = *(const h16x4 *)(in + ov);
        x.y1 = *(const f32x4 *)(in + C7_Y1 * 4 + o16);
        x.al = *(const f32x4 *)(in + oa);
        x.k = *(const f32x4 *)(in + C7_K * 4 + o16);
        x.b = *(const f32x4 *)(in + C7_B * 4 + o16);
    };
    // register jb of a lane's y: token 4 q + jb; stored one chunk late, the first (empty) store to the 16 rows ahead of token 0
    float *yo = y32 + (size_t)(4 * q + jb) * C + h * HS7 + i, *ynext = yo + (size_t)(CL + t_begin) * C;
    // u first (the next state waits for it), the keys' update while its shares are on their way to LDS, y while they come
    // back; y's shares are exchanged with the next chunk's u
    f32x4 yp = {0.f, 0.f, 0.f, 0.f};
    bool broken = false;                                    // this wave's share of the values was not all finite
    auto step = [&](const Ops &x, int buf) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (float)x.v[e];
        const float v01 = jb == 0 ? v[0] : v[1], v23 = jb == 2 ? v[2] : v[3], vj = jb < 2 ? v01 : v23;
        const bool fin = __builtin_isfinite(vj);            // see wkv56_apply_kernel
        broken |= !fin;
        const float vf = fin ? vj : 0.f;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, old = st;
        f32x4 u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.two[1], vf, zero, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.ta[e], old[e], u, 0, 0, 0);
        redy[buf][jb][lane] = yp;
        st = old * x.al;
        __builtin_amdgcn_sched_barrier(0);
        st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[0], v[0], st, 0, 0, 0);
        st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[1], v[1], st, 0, 0, 0);
        redu[buf][jb][lane] = u;
        __builtin_amdgcn_sched_barrier(0);
        st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[2], v[2], st, 0, 0, 0);
        st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[3], v[3], st, 0, 0, 0);
        asm volatile("" ::: "memory");        // no write of the exchange behind the barrier
        __builtin_amdgcn_s_waitcnt(0xC07F);   // LDS only: __syncthreads() would also wait for the loads in flight
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");        // no read of the exchange ahead of it
        const f32x4 u0 = redu[buf][0][lane], u1 = redu[buf][1][lane], u2 = redu[buf][2][lane], u3 = redu[buf][3][lane];
        float part[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) part[w] = ((const float *)&redy[buf][w][lane])[jb];
        __builtin_amdgcn_sched_barrier(0);
        yp = __builtin_amdgcn_mfma_f32_16x16x4f32(x.two[0], vf, zero, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) yp = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y1[e], old[e], yp, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        u = (u0 + u1) + (u2 + u3);
#pragma unroll
        for (int e = 0; e < 4; ++e) st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.b[e], u[e], st, 0, 0, 0);
        *yo = (part[0] + part[1]) + (part[2] + part[3]);   // the chunk before
        yo = ynext;
        ynext += (size_t)CL * C;
    };
    // The order of the loads is the order of their use, which the fences keep: the compiler counts its waits over both
    // ways into the loop, and a later chunk's load ahead of an earlier one's would make it wait for both.
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    Ops ops[PD];
#pragma unroll
    for (int u = 0; u < PD; ++u) {
        load(ops[u], u);
        fence();
    }
    for (int c0 = 0; c0 < nchunk; c0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            if (c0 + u >= nchunk) break;
            step(ops[u], u & 1);
            fence();
            load(ops[u], c0 + u + PD);
            fence();
        }
    }
    __syncthreads();
    redy[0][jb][lane] = yp;
    __syncthreads();
    const float *p = (const float *)&redy[0][0][lane] + jb;
    *yo = (p[0] + p[256]) + (p[512] + p[768]);
    *(f32x4 *)S = st;
    if (any_wave(broken, (int *)redu)) {
        yo -= (size_t)(nchunk - 1) * CL * C;                // the same thread stored these
        for (int c = 0; c < nchunk; ++c, yo += (size_t)CL * C) {
            Ops x;
            load(x, c);
            int first = CL;
#pragma unroll
            for (int e = 3; e >= 0; --e)
                if (!__builtin_isfinite((float)x.v[e])) first = 4 * q + e;
            first = min(first, __shfl_xor(first, 16, WAVE));
            first = min(first, __shfl_xor(first, 32, WAVE));
            if (4 * q + jb >= first) *yo = NAN;
        }
    }
}

// GroupNorm over each head's 64 outputs (eps 64e-5) on the fp16-rounded read-out, + bonus * v, * g.  Four adjacent
// channels per lane (16-byte loads of y, 8-byte accesses to v, g and the output): a row of 16 lanes owns one head
// of one token, its two sums are DPP row sums; a workgroup has 256 of the C / 4 chunks of one row.
__global__ __launch_bounds__(256) void gn7_kernel(int per_row, uint64_t factor, int C, const float *__restrict__ y,
                                                  const rwkv_half *__restrict__ lnx_w,
                                                  const rwkv_half *__restrict__ lnx_b, const float *__restrict__ rk,
                                                  const rwkv_half *__restrict__ v, const rwkv_half *__restrict__ gate,
                                                  rwkv_half *__restrict__ out) {
    const int cpr = C / 4, H = C / HS7;   // cpr % 16 == 0: whole rows of lanes are live or idle together
    {
        const int t = div_by(blockIdx.x, factor), i = ((int)blockIdx.x - t * per_row) * 256 + threadIdx.x;
        const bool live = i < cpr;
        const int c = min(i, cpr - 1) * 4;
        const size_t o = (size_t)t * C + c;
        const f32x4 y4 = *(const f32x4 *)(y + o);
        const h16x4 w4 = *(const h16x4 *)(lnx_w + c), b4 = *(const h16x4 *)(lnx_b + c);
        const h16x4 v4 = *(const h16x4 *)(v + o), g4 = *(const h16x4 *)(gate + o);
        const float bonus = rk[t * H + c / HS7];
        float yv[4], sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { yv[e] = round_h(y4[e]); sum += yv[e]; }
        const float mean = row16_sum(sum) * (1.f / HS7);
        float sq = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float d = yv[e] - mean; sq += d * d; }
        const float rstd = rsqrtf(row16_sum(sq) * (1.f / HS7) + 64e-5f);
        h16x4 o4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float q = round_h((yv[e] - mean) * rstd * (float)w4[e] + (float)b4[e]);
            q = round_h(q + round_h(bonus * (float)v4[e]));
            o4[e] = (h16)(q * (float)g4[e]);
        }
        if (live) *(h16x4 *)(out + o) = o4;
    }
}

// ---- one-token kernels ---------------------------------------------------------------------
struct Att7Args {
    const rwkv_half *mix[6];   // r, w, k, v, a, g
    MatDev mat[3];             // receptance, key, value
    rwkv_half *xx_tmp;
    const rwkv_half *x, *ln_w, *ln_b, *sx;
    int C;
    RowSplit lsplit;           // of the rtot rows
    rwkv_half *out[3];         // r, k, v  [C]
    const rwkv_half *lora1;    // [rtot][C]
    int rtot, o_a, o_v, o_g;   // rows, first row of the a / v / g blocks
    rwkv_half *l1;             // [rtot] activated first-stage outputs
};

__global__ __launch_bounds__(DTHREADS) void att7_kernel(const rwkv_half *x, const rwkv_half *ln_w, const rwkv_half *ln_b, const rwkv_half *sx,
                                                        RWKV_SPLIT_ARGS, int C, Att7Args a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[(2 + 3 * 6) * DWAVES];
    __shared__ unsigned sync[2];
    h16 *xs[6];
    const rwkv_half *mix[6];
    MatDev nomat[6] = {};
#pragma unroll
    for (int j = 0; j < 6; ++j) { xs[j] = (h16 *)smem + j * C; mix[j] = a.mix[j]; }
    LnMixPro<false, 6> pro;
    auto pro_load = [&]() { pro.load(x, C, ln_w, ln_b, sx, mix, nomat); };
    auto pro_compute = [&]() { pro.compute(C, true, mix, xs, a.xx_tmp, red, sync, true); };
    auto rowf = [&](int c, int k, const uint8_t *&row, const h16 *&xv) {
        row = row_ptr<false>(a.mat[k], c);
        xv = xs[k == 0 ? 0 : (k == 1 ? 2 : 3)];
    };
    auto epi_load = [&](int) { return NoEpi{}; };
    auto epi = [&](int c, const float (&d)[3], const NoEpi &) {
#pragma unroll
        for (int k = 0; k < 3; ++k) a.out[k][c] = f2h(d[k]);
    };
    const int nseg = (C * 2) >> 4;
    stream_rows<false, 1, 3, 2, NoEpi, true>(RWKV_SPLIT, nseg, pro_waves(C >> 3), sync, pro_load, pro_compute, [] {}, rowf, epi_load, epi);
    // first LoRA stages: row g of the stacked matrix belongs to block j = w, a, v, g
    auto block_of = [&](int g) { return (g >= a.o_a ? 1 : 0) + (g >= a.o_v ? 1 : 0) + (g >= a.o_g ? 1 : 0); };
    auto rowf2 = [&](int g, int, const uint8_t *&row, const h16 *&xv) {
        row = (const uint8_t *)(a.lora1 + (size_t)g * C);
        const int j = block_of(g);
        const int mi = j == 0 ? 1 : (j == 1 ? 4 : (j == 2 ? 3 : 5));   // xw, xa, xv, xg
        xv = (const h16 *)smem + mi * C;
    };
    auto epi2 = [&](int g, const float (&d)[1], const NoEpi &) {
        const int j = block_of(g);
        float v = round_h(d[0]);
        v = j == 0 ? tanhf(v) : (j == 3 ? sigmoidf_(v) : v);
        a.l1[g] = f2h(v);
    };
    stream_rows<false, 1, 1, 2, NoEpi, false>(a.lsplit, nseg, 0, nullptr, [] {}, [] {}, [] {}, rowf2, epi_load, epi2);
}

// besides the leading arguments l1 [rtot], lora2 [C][rtot], state [H][64][64], the stacked rows' total, offsets and ranks
struct Tmix7Args {
    int C, first_layer;
    const rwkv_half *r, *k, *v, *v_first;   // [C]; v_first unused in layer 0 (there v is the layer-0 value itself)
    const rwkv_half *w0, *a0, *v0, *k_k, *k_a, *r_k, *lnx_w, *lnx_b;
    rwkv_half *out;            // [C]
    const rwkv_half *commit_src;   // scratch xx -> token-shift state, done by workgroup 0
    rwkv_half *commit_dst;
};

// One workgroup of 16 waves per head.  All operands are requested in the first instructions (one memory
// round trip): wave w takes 16 (channel, product) rows of the second LoRA stages -- product w / 4, lane =
// 16-byte segment of the row, so a row is one coalesced request -- the first four waves also the head's
// state, wave 0 also the head's vectors.  Then: row sums -> LDS; wave 0 prepares the step; threads 0..255
// (value rows il + 16 m, key group g = lane & 15, holding S[i][4g..4g+3] of their four rows) advance the
// state, the sums over a row's key groups being DPP row sums; wave 0 normalises and gates.
__global__ __launch_bounds__(1024) void tmix7_kernel(const rwkv_half *l1, const rwkv_half *lora2, float *state, int rtot, int o_a, int o_v, int o_g,
                                                    int d_w, int d_a, int d_v, int d_g, Tmix7Args a) {
    __shared__ float lo[4][HS7];
    __shared__ __align__(16) float sr[HS7], sk[HS7], sw[HS7], sa[HS7], sb[HS7];
    __shared__ float sv[HS7], sy[HS7], srk;
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int il = (tid >> 4) & 15, g = tid & 15;
    const int c = h * HS7 + lane;
    float *S = state + (size_t)h * HS7 * HS7;
    // ---- loads
    const int q = w >> 2;
    const int off = q == 0 ? 0 : (q == 1 ? o_a : (q == 2 ? o_v : o_g));
    const int d8 = (q == 0 ? d_w : (q == 1 ? d_a : (q == 2 ? d_v : d_g))) >> 3;   // d_v: 0 in the first layer
    const int seg = lane < d8 ? lane : 0;
    const h16x8 xv = *(const h16x8 *)(l1 + off + 8 * seg);
    u32x4 wv[16];
#pragma unroll
    for (int jj = 0; jj < 16; ++jj)
        wv[jj] = *(const u32x4 *)(lora2 + (size_t)(h * HS7 + (w & 3) * 16 + jj) * rtot + off + 8 * seg);
    f32x4 s[4] = {};
    if (w < 4)
#pragma unroll
        for (int m = 0; m < 4; ++m) s[m] = *(const f32x4 *)(S + (size_t)(il + 16 * m) * HS7 + 4 * g);
    float r = 0.f, k = 0.f, v = 0.f, vf = 0.f, a0 = 0.f, w0 = 0.f, v0 = 0.f, k_k = 0.f, k_a = 0.f, r_k = 0.f, lw = 0.f, lb = 0.f;
    if (w == 0) {
        r = h2f(a.r[c]); k = h2f(a.k[c]); v = h2f(a.v[c]);
        a0 = h2f(a.a0[c]); w0 = h2f(a.w0[c]); k_k = h2f(a.k_k[c]); k_a = h2f(a.k_a[c]); r_k = h2f(a.r_k[c]);
        lw = h2f(a.lnx_w[c]); lb = h2f(a.lnx_b[c]);
        if (!a.first_layer) { vf = h2f(a.v_first[c]); v0 = h2f(a.v0[c]); }
    }
    // ---- second LoRA stages
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
        const float p = wave_sum(lane < d8 ? dot8_f16(wv[jj], xv, 0.f) : 0.f);
        if (lane == 0) lo[q][(w & 3) * 16 + jj] = round_h(p);
    }
    __syncthreads();
    if (w == 0) {
        const float av = round_h(sigmoidf_(round_h(a0 + lo[1][lane])));
        const float kku = round_h(k * k_k);
        const float nrm = fmaxf(round_h(sqrtf(wave_sum(kku * kku))), 1e-12f);
        const float kk = round_h(kku / nrm);
        const float k2 = round_h(k * round_h(1.f + round_h(round_h(av - 1.f) * k_a)));
        if (!a.first_layer) {
            const float sg = round_h(sigmoidf_(round_h(v0 + lo[2][lane])));
            v = round_h(v + round_h(round_h(vf - v) * sg));
        }
        const float z = round_h(w0 + lo[0][lane]);
        sr[lane] = r; sk[lane] = k2; sv[lane] = v;
        sw[lane] = __expf(-0.606531f * sigmoidf_(z));
        sa[lane] = -kk;
        sb[lane] = round_h(kk * av);
        const float rk = wave_sum(round_h(round_h(r * k2) * r_k));
        if (lane == 0) srk = round_h(rk);
    }
    __syncthreads();
    if (w < 4) {
        const f32x4 r4 = *(const f32x4 *)&sr[4 * g], k4 = *(const f32x4 *)&sk[4 * g], w4 = *(const f32x4 *)&sw[4 * g];
        const f32x4 a4 = *(const f32x4 *)&sa[4 * g], b4 = *(const f32x4 *)&sb[4 * g];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int i = il + 16 * m;
            const float vi = sv[i];
            float p = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) p += a4[e] * s[m][e];
            const float sav = row16_sum(p);
            float y = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[m][e] = s[m][e] * w4[e] + k4[e] * vi + sav * b4[e];
                y += s[m][e] * r4[e];
            }
            y = row16_sum(y);
            if (g == 0) sy[i] = y;
            *(f32x4 *)(S + (size_t)i * HS7 + 4 * g) = s[m];
        }
    }
    __syncthreads();
    if (w == 0) {
        const float yv = round_h(sy[lane]);
        const float mean = wave_sum(yv) * (1.f / HS7);
        const float dv = yv - mean;
        const float var = wave_sum(dv * dv) * (1.f / HS7);
        float o = round_h(dv * rsqrtf(var + 64e-5f) * lw + lb);
        o = round_h(o + round_h(srk * sv[lane]));
        a.out[c] = f2h(o * lo[3][lane]);
    }
    if (blockIdx.x == 0 && a.commit_dst)
        for (int j8 = tid; j8 < (a.C >> 3); j8 += 1024)
            *(u32x4 *)(a.commit_dst + 8 * j8) = *(const u32x4 *)(a.commit_src + 8 * j8);
}

// ---- DeepEmbed channel mix (model.py:578-594): keys of token t scaled by ((xx_t @ s1) @ E_t) @ s2 + s0 -----------
// First stage, one workgroup per token: sv = xx_t @ s1 (32 sums over C, eight per wave), then ss = sv @ E_t with
// E_t = row token_t of the merged table viewed 32 x 32.  Both rounded to fp16 as the reference's fp16 tensors are.
__global__ __launch_bounds__(256) void de_ss_kernel(int T, int C, int vocab, const int32_t *__restrict__ tokens,
                                                    const rwkv_half *__restrict__ xx, const rwkv_half *__restrict__ s1,
                                                    const rwkv_half *__restrict__ emb, rwkv_half *__restrict__ ss) {
    __shared__ float sv[32];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const rwkv_half *x = xx + (size_t)t * C;
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    for (int c8 = lane; c8 < (C >> 3); c8 += 64) {
        const h16x8 xv = *(const h16x8 *)(x + 8 * c8);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const h16x8 wv = *(const h16x8 *)(s1 + (size_t)(wave * 8 + j) * C + 8 * c8);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[j] += (float)xv[e] * (float)wv[e];
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float v = wave_sum(acc[j]);
        if (lane == 0) sv[wave * 8 + j] = (float)(h16)v;
    }
    __syncthreads();
    if (threadIdx.x < 32) {
        const rwkv_half *E = emb + (size_t)min(max(tokens[t], 0), vocab - 1) * 1024;
        float a = 0.f;
        for (int i = 0; i < 32; ++i) a += sv[i] * (float)h2f(E[i * 32 + threadIdx.x]);
        ss[(size_t)t * 32 + threadIdx.x] = f2h(a);
    }
}

// Second stage: k[t][f] *= (ss_t @ s2)[f] + s0[f], every step rounded to fp16.  A workgroup takes 256 columns of
// eight tokens, so a column of s2 is fetched once per eight tokens.
__global__ __launch_bounds__(256) void de_gate_kernel(int T, int F, const rwkv_half *__restrict__ ss,
                                                      const rwkv_half *__restrict__ s2, const rwkv_half *__restrict__ s0,
                                                      rwkv_half *__restrict__ k) {
    __shared__ float ssl[8][32];
    const int t0 = blockIdx.x * 8, f = blockIdx.y * 256 + threadIdx.x;
    {
        const int tt = threadIdx.x >> 5, j = threadIdx.x & 31;
        ssl[tt][j] = t0 + tt < T ? h2f(ss[(size_t)(t0 + tt) * 32 + j]) : 0.f;
    }
    __syncthreads();
    if (f >= F) return;
    float col[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) col[j] = h2f(s2[(size_t)j * F + f]);
    const float b = h2f(s0[f]);
    for (int tt = 0; tt < 8 && t0 + tt < T; ++tt) {
        float a = 0.f;
#pragma unroll
        for (int j = 0; j < 32; ++j) a += ssl[tt][j] * col[j];
        const float g = (float)(h16)((float)(h16)a + b);
        rwkv_half *kp = k + (size_t)(t0 + tt) * F + f;
        *kp = f2h(h2f(*kp) * g);
    }
}

int de_gate_launch(const rwkv_v7_layer &l, int64_t T, int C, int F, int vocab, const int32_t *tokens, const rwkv_half *xx,
                   rwkv_half *ss, rwkv_half *k, hipStream_t st) {
    hipLaunchKernelGGL(de_ss_kernel, dim3((unsigned)T), dim3(256), 0, st, (int)T, C, vocab, tokens, xx, l.de_s1, l.de_emb, ss);
    hipLaunchKernelGGL(de_gate_kernel, dim3((unsigned)((T + 7) / 8), (unsigned)((F + 255) / 256)), dim3(256), 0, st, (int)T, F,
                       ss, l.de_s2, l.de_s0, k);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

struct Ws7 {
    rwkv_half *x, *mix[6], *l1, *lw, *la, *lv, *lg, *w_raw, *a_raw, *vg_raw, *g, *r, *k, *v, *v_first, *an, *b, *att, *vx,
        *xx_att, *xx_ffn, *de_ss;
    float *dec, *rk, *y32, *splitk, *chunks;
    size_t total;
};

Ws7 carve7(void *base, int64_t T, const rwkv_v7_model *m) {
    Ws7 w;
    unsigned char *p = (unsigned char *)base;
    auto take = [&](size_t bytes) { void *q = p; p += align256(bytes); return (rwkv_half *)q; };
    const size_t C = m->n_embd, F = m->n_ffn;
    const size_t tc = (size_t)T * C * 2;
    w.x = take(tc);
    for (int j = 0; j < 6; ++j) w.mix[j] = take(tc);
    w.l1 = take((size_t)(m->lora_w + m->lora_a + m->lora_v + m->lora_g) * 2);
    w.lw = take((size_t)T * m->lora_w * 2); w.la = take((size_t)T * m->lora_a * 2);
    w.lv = take((size_t)T * m->lora_v * 2); w.lg = take((size_t)T * m->lora_g * 2);
    w.w_raw = take(tc); w.a_raw = take(tc); w.vg_raw = take(tc); w.g = take(tc);
    w.r = take(tc); w.k = take(tc); w.v = take(tc); w.v_first = take(tc); w.att = take(tc);
    w.vx = take((size_t)T * F * 2);
    w.xx_att = take(C * 2); w.xx_ffn = take(C * 2);
    w.de_ss = take((size_t)T * 32 * 2);
    // what prep7_kernel leaves for wkv7_kernel; longer calls' operands are the chunks
    const bool chunked = T >= CHUNKED7;
    w.an = take(chunked ? 256 : tc); w.b = take(chunked ? 256 : tc);
    w.dec = (float *)take(chunked ? 256 : 2 * tc);
    w.rk = (float *)take((size_t)T * m->n_head * 4);
    w.y32 = (float *)take((size_t)(chunked ? (wkv_chunks(T) + 1) * CL : T) * C * 4);   // a row for every padded token, and 16 in front
    w.chunks = (float *)take(!chunked ? 256 : (size_t)wkv_chunks(std::min<int64_t>(T, SEG7)) * m->n_head * C7_FLOATS * 4);
    w.splitk = (float *)take(RWKV_SPLITK_WS_BYTES);
    w.total = (size_t)(p - (unsigned char *)base);
    return w;
}

bool mat_ok7(const rwkv_mat &m, int64_t N, int64_t M) {
    return m.w && m.N == N && m.M == M && m.ld >= N && !(m.ld & 7) && aligned16(m.w);
}

int wkv7_check(int64_t B, int64_t T, int64_t C, int64_t H) {
    if (B != 1 || T <= 0 || H <= 0 || C != H * HS7 || T > (1 << 24)) return RWKV_E_SHAPE;
    return RWKV_OK;
}

}  // namespace

extern "C" int rwkv_wkv7_forward(int64_t B, int64_t T, int64_t C, int64_t H, float *state, const void *r,
                                 const void *w, const void *k, const void *v, const void *a, const void *b,
                                 void *y, int dtype, void *stream) {
    if (!state || !r || !w || !k || !v || !a || !b || !y) return RWKV_E_NULL;
    int rc = wkv7_check(B, T, C, H);
    if (rc) return rc;
    if (dtype != RWKV_DT_F16 && dtype != RWKV_DT_F32 && dtype != RWKV_DT_BF16) return RWKV_E_DTYPE;
    if (!aligned16(state) || !aligned16(r) || !aligned16(w) || !aligned16(k) || !aligned16(a) || !aligned16(b) ||
        (((uintptr_t)v) & 3))
        return RWKV_E_LAYOUT;
    Wkv7Args q{(int)T, (int)C, state, r, w, k, v, a, b, y};
    const dim3 grid((unsigned)(4 * H)), block(256);
    if (dtype == RWKV_DT_F16) hipLaunchKernelGGL((wkv7_kernel<RWKV_DT_F16, false>), grid, block, 0, (hipStream_t)stream, q);
    else if (dtype == RWKV_DT_BF16) hipLaunchKernelGGL((wkv7_kernel<RWKV_DT_BF16, false>), grid, block, 0, (hipStream_t)stream, q);
    else hipLaunchKernelGGL((wkv7_kernel<RWKV_DT_F32, false>), grid, block, 0, (hipStream_t)stream, q);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

static int v7_check(const rwkv_v7_model *m) {
    if (!m || !m->layers || !m->emb || !m->ln_out_w || !m->ln_out_b) return RWKV_E_NULL;
    const int64_t C = m->n_embd, F = m->n_ffn, V = m->vocab;
    if (m->n_layer <= 0 || C <= 0 || F <= 0 || V <= 0 || (C & 63) || (F & 63) || C > 8 * DTHREADS ||
        F > 8 * VP * DTHREADS || m->n_head * HS7 != C)
        return RWKV_E_SHAPE;
    const int ranks[4] = {m->lora_w, m->lora_a, m->lora_v, m->lora_g};
    for (int j = 0; j < 4; ++j)
        if (ranks[j] <= 0 || (ranks[j] & 63) || ranks[j] > 8 * DTHREADS) return RWKV_E_SHAPE;
    for (int i = 0; i < m->n_layer; ++i) {
        const rwkv_v7_layer &l = m->layers[i];
        if (!l.ln1_w || !l.ln1_b || !l.ln2_w || !l.ln2_b || !l.w0 || !l.a0 || !l.lora1 || !l.lora2 || !l.k_k ||
            !l.k_a || !l.r_k || !l.lnx_w || !l.lnx_b || !l.ffn_x_k)
            return RWKV_E_NULL;
        if (i > 0 && !l.v0) return RWKV_E_NULL;
        if (!aligned16(l.lora1) || !aligned16(l.lora2)) return RWKV_E_LAYOUT;
        if (l.de_emb || l.de_s1 || l.de_s2 || l.de_s0) {   // the DeepEmbed tensors come all four or not at all
            if (!l.de_emb || !l.de_s1 || !l.de_s2 || !l.de_s0) return RWKV_E_NULL;
            if (!aligned16(l.de_s1)) return RWKV_E_LAYOUT;
        }
        for (int j = 0; j < 6; ++j)
            if (!l.x_mix[j]) return RWKV_E_NULL;
        if (!mat_ok7(l.att_receptance, C, C) || !mat_ok7(l.att_key, C, C) || !mat_ok7(l.att_value, C, C) ||
            !mat_ok7(l.att_output, C, C) || !mat_ok7(l.ffn_key, C, F) || !mat_ok7(l.ffn_value, F, C))
            return RWKV_E_LAYOUT;
    }
    if (!mat_ok7(m->head, C, V)) return RWKV_E_LAYOUT;
    return RWKV_OK;
}

extern "C" size_t rwkv_v7_workspace(const rwkv_v7_model *m, int64_t T) {
    if (!m || T <= 0) return 0;
    return carve7((void *)256, T, m).total;
}

extern "C" int rwkv_v7_forward(const rwkv_v7_model *m, const rwkv_v56_layer_state *states, const int32_t *tokens,
                               int64_t T, int full_output, float *logits, void *workspace, size_t workspace_bytes,
                               void *stream) {
    int rc = v7_check(m);
    if (rc) return rc;
    if (!states || !tokens || !logits || !workspace) return RWKV_E_NULL;
    if (T <= 0 || T > (1 << 20)) return RWKV_E_SHAPE;
    if (workspace_bytes < rwkv_v7_workspace(m, T) || (((uintptr_t)workspace) & 255)) return RWKV_E_WORKSPACE;
    for (int i = 0; i < m->n_layer; ++i) {
        const rwkv_v56_layer_state &s = states[i];
        if (!s.att_xx || !s.att_kv || !s.ffn_xx) return RWKV_E_NULL;
        if (!aligned16(s.att_xx) || !aligned16(s.ffn_xx) || !aligned16(s.att_kv)) return RWKV_E_LAYOUT;
    }
    hipStream_t st = (hipStream_t)stream;
    const int C = m->n_embd, H = m->n_head;
    Ws7 ws = carve7(workspace, T, m);
    // the fp16 path needs no scaled-activation scratch or row sums
    Ctx c{st, false, T, num_cu(), nullptr, nullptr, nullptr, ws.splitk, 0};

    const int max_rank = std::max(std::max(m->lora_w, m->lora_a), std::max(m->lora_v, m->lora_g));
    const int o_a = m->lora_w, o_v = o_a + m->lora_a, o_g = o_v + m->lora_v, rtot = o_g + m->lora_g;
    // block j of the stacked LoRA matrices as matrices of their own
    auto lora_first = [&](const rwkv_v7_layer &l, int off, int d) { return lora_mat(l.lora1 + (size_t)off * C, C, d); };
    auto lora_second = [&](const rwkv_v7_layer &l, int off, int d) {
        rwkv_mat q{};
        q.w = l.lora2 + off; q.ld = rtot; q.N = d; q.M = C;
        return q;
    };

    SideStreams *ss = T >= 256 ? side_streams(st) : nullptr;

    if ((rc = gather_emb_launch(T, C, m->vocab, tokens, m->emb, ws.x, st))) return rc;
    for (int i = 0; i < m->n_layer; ++i) {
        const rwkv_v7_layer &l = m->layers[i];
        const rwkv_v56_layer_state &s = states[i];
        // one token: the six mixed activation vectors must fit the default LDS window, a LoRA row one request per wave
        if (T == 1 && C <= 5120 && max_rank <= 512) {
            rwkv_half *v1 = i == 0 ? ws.v_first : ws.v;
            {
                Att7Args a{};
                a.x = ws.x; a.C = C; a.ln_w = l.ln1_w; a.ln_b = l.ln1_b; a.sx = s.att_xx; a.xx_tmp = ws.xx_att;
                for (int j = 0; j < 6; ++j) a.mix[j] = l.x_mix[j];
                a.mat[0] = to_dev56(l.att_receptance); a.mat[1] = to_dev56(l.att_key); a.mat[2] = to_dev56(l.att_value);
                a.out[0] = ws.r; a.out[1] = ws.k; a.out[2] = v1;
                a.lora1 = l.lora1; a.rtot = rtot; a.o_a = o_a; a.o_v = o_v; a.o_g = o_g; a.l1 = ws.l1;
                a.lsplit = wave_split(rtot, c.grid);
                const RowSplit sp = wave_split(C, c.grid);
                hipLaunchKernelGGL(att7_kernel, dim3(c.grid), dim3(DTHREADS), 6 * (size_t)C * 2, st, a.x, a.ln_w, a.ln_b, a.sx, RWKV_SPLIT_PASS(sp),
                                   C, a);
            }
            {
                Tmix7Args a{};
                a.C = C; a.first_layer = i == 0;
                a.r = ws.r; a.k = ws.k; a.v = v1; a.v_first = ws.v_first;
                a.w0 = l.w0; a.a0 = l.a0; a.v0 = l.v0; a.k_k = l.k_k; a.k_a = l.k_a; a.r_k = l.r_k;
                a.lnx_w = l.lnx_w; a.lnx_b = l.lnx_b; a.out = ws.att;
                a.commit_src = ws.xx_att; a.commit_dst = s.att_xx;
                hipLaunchKernelGGL(tmix7_kernel, dim3((unsigned)H), dim3(1024), 0, st, ws.l1, l.lora2, s.att_kv, rtot, o_a, o_v, o_g, (int)m->lora_w,
                                   (int)m->lora_a, i == 0 ? 0 : (int)m->lora_v, (int)m->lora_g, a);
            }
            if ((rc = mm(c, l.att_output, false, ws.att, ACT_RESIDUAL, ws.x, nullptr, 1.f, ws.x))) return rc;
            {
                LnMixArgs a{};
                a.x = ws.x; a.C = C; a.ln_w = l.ln2_w; a.ln_b = l.ln2_b; a.sx = s.ffn_xx; a.xx_tmp = ws.xx_ffn;
                a.mix[0] = l.ffn_x_k; a.mat[0] = to_dev56(l.ffn_key); a.M[0] = (int)l.ffn_key.M; a.epi[0] = EPI_RELU_SQ;
                a.out[0] = ws.vx; a.maa_form = 1;
                lnmix1_launch(false, a, c.grid, st);
            }
            if (l.de_emb && (rc = de_gate_launch(l, 1, C, m->n_ffn, m->vocab, tokens, ws.xx_ffn, ws.de_ss, ws.vx, st))) return rc;
            if ((rc = mm(c, l.ffn_value, false, ws.vx, ACT_RESIDUAL, ws.x, nullptr, 1.f, ws.x, ws.xx_ffn, s.ffn_xx, C))) return rc;
            RWKV_LAUNCH_CHECK();
            continue;
        }
        {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln1_w; a.ln_b = l.ln1_b; a.sx = s.att_xx;
            a.xx_last = nullptr; a.state_out = s.att_xx; a.maa_form = 1;   // row 0's workgroup commits the new state
            for (int j = 0; j < 6; ++j) { a.mix[j] = l.x_mix[j]; a.xs[j] = ws.mix[j]; }
            if ((rc = lnmix_seq_launch(a, 6, st))) return rc;
        }
        const rwkv_half *xr = ws.mix[0], *xw = ws.mix[1], *xk = ws.mix[2], *xv = ws.mix[3], *xa = ws.mix[4],
                        *xg = ws.mix[5];
        rwkv_half *v = i == 0 ? ws.v_first : ws.v;
        // The three C x C products and the LoRA chain are independent of each other.  From 256 rows on receptance,
        // key and value are one grouped launch of the direct-to-LDS kernel; where that group is more than one round
        // of large tiles (2048 tokens at n_embd 4096), the LoRA launches (which do split K: one user of the split-K
        // scratch at a time) run beside it on a side stream.  Measured with the LoRA stages grouped: 46.0K against
        // 45.7K tok/s in calls of 2048, but 42.3K against 43.3K in calls of 1024, where the group is one round and
        // the two streams only slow each other down.
        const bool dma_seq = true;
        ForkScope par(ss, st, 1, dma_seq && 3 * ((T + 255) / 256) * ((C + 255) / 256) >= 384);
        Ctx cm = c, cv = c, cl = c;
        if (par) cl.st = ss->s[0];
        if (dma_seq && !(C & 7)) {
            // receptance, key and value as one grouped launch
            const rwkv_half *xin[3] = {xr, xk, xv};
            const rwkv_mat *mats[3] = {&l.att_receptance, &l.att_key, &l.att_value};
            void *outs[3] = {ws.r, ws.k, v};
            GemmEpi ep[3] = {};
            for (int j = 0; j < 3; ++j) { ep[j].act = ACT_NONE; ep[j].out_scale = 1.f; ep[j].out_dtype = RWKV_DT_F16; }
            if ((rc = gemm_group_launch(false, 3, T, C, xin, mats, outs, ep, nullptr, nullptr, ws.splitk, st))) return rc;
        } else {
        if ((rc = mm(cm, l.att_receptance, false, xr, ACT_NONE, nullptr, nullptr, 1.f, ws.r))) return rc;
        if ((rc = mm(cm, l.att_key, false, xk, ACT_NONE, nullptr, nullptr, 1.f, ws.k))) return rc;
        if ((rc = mm(cv, l.att_value, false, xv, ACT_NONE, nullptr, nullptr, 1.f, v))) return rc;
        }
        // The LoRA products: the first stages (same input width, their own inputs, ranks and activations) as one
        // grouped launch, then the second stages -- those of equal rank as one grouped launch, the others one by one.
        // RWKV_V7_LORA_GROUPS=0 launches all eight one by one (tuning).
        {
            const bool has_v = i > 0;
            struct Stage { const rwkv_half *x; int off, d, act; rwkv_half *l1, *out; };
            const Stage sg[4] = {{xw, 0, m->lora_w, ACT_TANH, ws.lw, ws.w_raw},
                                 {xa, o_a, m->lora_a, ACT_NONE, ws.la, ws.a_raw},
                                 {xv, o_v, m->lora_v, ACT_NONE, ws.lv, ws.vg_raw},
                                 {xg, o_g, m->lora_g, ACT_SIGMOID, ws.lg, ws.g}};
            const char *env = getenv("RWKV_V7_LORA_GROUPS");
            const bool groups = !(env && *env == '0') && !(C & 7);
            bool first_done[4] = {false, false, false, false}, second_done[4] = {false, false, false, false};
            if (groups) {
                const rwkv_half *xin[4];
                rwkv_mat mt[4];
                const rwkv_mat *mp[4];
                void *outs[4];
                GemmEpi ep[4] = {};
                int n = 0, idx[4];
                for (int q = 0; q < 4; ++q) {
                    if (q == 2 && !has_v) continue;
                    xin[n] = sg[q].x; mt[n] = lora_first(l, sg[q].off, sg[q].d); mp[n] = &mt[n]; outs[n] = sg[q].l1;
                    ep[n].act = sg[q].act; ep[n].out_scale = 1.f; ep[n].out_dtype = RWKV_DT_F16;
                    idx[n++] = q;
                }
                if ((rc = gemm_group_launch(false, n, T, C, xin, mp, outs, ep, nullptr, nullptr, cl.splitk, cl.st))) return rc;
                for (int q = 0; q < n; ++q) first_done[idx[q]] = true;
                // second stages of the most common rank together
                int best = -1, best_n = 0;
                for (int q = 0; q < 4; ++q) {
                    if (q == 2 && !has_v) continue;
                    int cnt = 0;
                    for (int r = 0; r < 4; ++r) cnt += (r != 2 || has_v) && sg[r].d == sg[q].d;
                    if (cnt > best_n) { best_n = cnt; best = q; }
                }
                if (best_n >= 2 && !(sg[best].d % 64)) {
                    n = 0;
                    for (int q = 0; q < 4; ++q) {
                        if ((q == 2 && !has_v) || sg[q].d != sg[best].d) continue;
                        xin[n] = sg[q].l1; mt[n] = lora_second(l, sg[q].off, sg[q].d); mp[n] = &mt[n]; outs[n] = sg[q].out;
                        ep[n] = GemmEpi{};
                        ep[n].act = ACT_NONE; ep[n].out_scale = 1.f; ep[n].out_dtype = RWKV_DT_F16;
                        idx[n++] = q;
                    }
                    if ((rc = gemm_group_launch(false, n, T, sg[best].d, xin, mp, outs, ep, nullptr, nullptr, cl.splitk, cl.st))) return rc;
                    for (int q = 0; q < n; ++q) second_done[idx[q]] = true;
                }
            }
            for (int q = 0; q < 4; ++q) {
                if (q == 2 && !has_v) continue;
                if (!first_done[q] &&
                    (rc = mm(cl, lora_first(l, sg[q].off, sg[q].d), false, sg[q].x, sg[q].act, nullptr, nullptr, 1.f, sg[q].l1)))
                    return rc;
                if (!second_done[q] &&
                    (rc = mm(cl, lora_second(l, sg[q].off, sg[q].d), false, sg[q].l1, ACT_NONE, nullptr, nullptr, 1.f, sg[q].out)))
                    return rc;
            }
        }
        if (!par.join()) return (int)hipErrorUnknown;
        {
            Prep7Args a{};
            a.T = (int)T; a.C = C; a.H = H; a.r = ws.r; a.k = ws.k; a.v = v; a.w_raw = ws.w_raw; a.a_raw = ws.a_raw;
            a.vg_raw = i > 0 ? ws.vg_raw : nullptr; a.v_first = i > 0 ? ws.v_first : nullptr;
            a.w0 = l.w0; a.a0 = l.a0; a.v0 = l.v0; a.k_k = l.k_k; a.k_a = l.k_a; a.r_k = l.r_k;
            a.an = ws.an; a.b = ws.b; a.dec = ws.dec; a.rk = ws.rk;
            if (T >= CHUNKED7) {
                for (int64_t t0 = 0; t0 < T; t0 += SEG7) {
                    const int nchunk = (int)((std::min<int64_t>(T - t0, SEG7) + CL - 1) / CL);
                    hipLaunchKernelGGL(wkv7_chunk_kernel, dim3((unsigned)(H * nchunk)), dim3(256), 0, st, a, (int)t0, ws.chunks);
                    hipLaunchKernelGGL(wkv7_apply_kernel, dim3((unsigned)(4 * H)), dim3(256), 0, st, H, C, s.att_kv, ws.y32, (int)t0, nchunk, ws.chunks);
                }
            } else {
                const int per_row = (C / 8 + 255) / 256;
                hipLaunchKernelGGL(prep7_kernel, dim3((unsigned)(T * per_row)), dim3(256), 0, st, per_row, div_factor(per_row), a);
                Wkv7Args q{(int)T, C, s.att_kv, ws.r, ws.dec, ws.k, v, ws.an, ws.b, ws.y32};
                hipLaunchKernelGGL((wkv7_kernel<RWKV_DT_F16, true>), dim3((unsigned)(4 * H)), dim3(256), 0, st, q);
            }
        }
        const int per_row = (C / 4 + 255) / 256;
        hipLaunchKernelGGL(gn7_kernel, dim3((unsigned)(T * per_row)), dim3(256), 0, st, per_row, div_factor(per_row), C,
                           ws.y32 + (T >= CHUNKED7 ? (size_t)CL * C : 0), l.lnx_w, l.lnx_b, ws.rk, v, ws.g, ws.att);
        if ((rc = mm(c, l.att_output, false, ws.att, ACT_RESIDUAL, ws.x, nullptr, 1.f, ws.x))) return rc;
        // ---- channel mix
        {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln2_w; a.ln_b = l.ln2_b; a.sx = s.ffn_xx;
            a.xx_last = nullptr; a.state_out = s.ffn_xx; a.maa_form = 1;
            a.mix[0] = l.ffn_x_k; a.xs[0] = ws.mix[0];
            a.mix[1] = nullptr; a.xs[1] = ws.mix[1];   // DeepEmbed also reads the LayerNorm output itself
            if ((rc = lnmix_seq_launch(a, l.de_emb ? 2 : 1, st))) return rc;
        }
        if ((rc = mm(c, l.ffn_key, false, ws.mix[0], ACT_RELU_SQ, nullptr, nullptr, 1.f, ws.vx))) return rc;
        if (l.de_emb && (rc = de_gate_launch(l, T, C, m->n_ffn, m->vocab, tokens, ws.mix[1], ws.de_ss, ws.vx, st))) return rc;
        if ((rc = mm(c, l.ffn_value, false, ws.vx, ACT_RESIDUAL, ws.x, nullptr, 1.f, ws.x))) return rc;
        RWKV_LAUNCH_CHECK();
    }
    // ---- head
    const bool all_rows = full_output && T > 1;
    const int64_t TH = all_rows ? T : 1;
    const rwkv_half *xh = all_rows ? ws.x : ws.x + (size_t)(T - 1) * C;
    if (TH == 1) {
        lnhead_launch(false, xh, C, m->ln_out_w, m->ln_out_b, to_dev56(m->head), m->vocab, logits, c.grid, st);
        RWKV_LAUNCH_CHECK();
        return RWKV_OK;
    }
    {
        SeqMixArgs a{};
        a.T = (int)TH; a.C = C; a.x = xh; a.ln_w = m->ln_out_w; a.ln_b = m->ln_out_b; a.sx = nullptr; a.xx_last = nullptr;
        a.xs[0] = ws.mix[0];
        if ((rc = lnmix_seq_launch(a, 1, st))) return rc;
    }
    GemmEpi e{};
    e.out_scale = 1.f; e.act = ACT_NONE; e.out_dtype = RWKV_DT_F32; e.splitk_ws = ws.splitk; e.splitk_bytes = RWKV_SPLITK_WS_BYTES;
    return gemm_launch(false, TH, C, m->vocab, ws.mix[0], C, m->head.w, m->head.ld, logits, m->vocab, e, st);
}
