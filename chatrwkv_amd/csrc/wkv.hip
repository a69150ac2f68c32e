// WKV recurrences: RWKV-4 (per channel, running-maximum form) and RWKV-5/6 (per-head 64x64 state).
#include <algorithm>
#include <type_traits>
#include "gemv_core.h"
#include "kernels.h"

namespace {

// ---------------------------------------------------------------------------------------
// RWKV-4.  One lane per channel, fp32 state in registers for the whole T loop; a wave reads
// 64 consecutive channels of a token (coalesced).  k/v for the next UNR tokens are loaded
// before the dependent chain of exp/div consumes them, so memory latency is off the
// critical path.  One wave per workgroup spreads the C/64 waves over as many CUs as possible.
//   MODE 0: k, v, y fp32 (operator-level interface)
//   MODE 1: k, v fp16; y = fp16(r * fp16(wkv)) with r fp16 (already sigmoid'ed), fp16 out
//   MODE 2: as MODE 1 with k, v fp32
// ---------------------------------------------------------------------------------------
// Rows of a tensor from one that the whole wave shares on: element c of row t by buffer instructions, whose address is a scalar
// base, a scalar offset t C and the lane's own, so that a token costs a few scalar instructions.  One wave per SIMD is bound by
// how many instructions it issues.  Offsets are 32 bits: up to 24 rows of WKV4_C values.
constexpr int64_t WKV4_C = 1 << 24;
template <class E> struct Rows {
    __amdgpu_buffer_rsrc_t p;
    DEV Rows(const E *base) : p(__builtin_amdgcn_make_buffer_rsrc((void *)base, 0, -1, 0x00027000)) {}
    DEV float ld(int row, int c) const {
        if constexpr (sizeof(E) == 4) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(p, 4 * c, 4 * row, 0));
        else return h2f(__builtin_amdgcn_raw_buffer_load_b16(p, 2 * c, 2 * row, 0));
    }
    DEV void st(int row, int c, float v) const {
        if constexpr (sizeof(E) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), p, 4 * c, 4 * row, 0);
        else __builtin_amdgcn_raw_buffer_store_b16(f2h(v), p, 2 * c, 2 * row, 0);
    }
};
template <int MODE> struct Wkv4IO {
    using KV = std::conditional_t<MODE == 1, rwkv_half, float>;
    using Y = std::conditional_t<MODE == 0, float, rwkv_half>;
    const KV *k, *v;
    Y *y;
    const rwkv_half *r;
};

// Sums of two products as one product that is rounded and one that is not, spelled out: left to the compiler, which of the two
// that is depended on a token's place in its batch of eight, and with it the last bit of the state.
DEV float wkv4_sum(float e1, float a, float e2, float v) { return __builtin_fmaf(e1, a, e2 * v); }
DEV void wkv4_step(float kk, float vv, float u, float w, float &aa, float &bb, float &pp, float &out) {
    float ww = u + kk;
    float p = fmaxf(pp, ww);
    float e1 = __expf(pp - p), e2 = __expf(ww - p);
    out = wkv4_sum(e1, aa, e2, vv) / __builtin_fmaf(e1, bb, e2);
    ww = w + pp;
    p = fmaxf(ww, kk);
    e1 = __expf(ww - p);
    e2 = __expf(kk - p);
    aa = wkv4_sum(e1, aa, e2, vv);
    bb = __builtin_fmaf(e1, bb, e2);
    pp = p;
}

// The tokens [t0, t1) of channel c of the rows from `base` on, in turn: step(k, v, out), and out stored where OUT.  Two batches of
// eight tokens: one is in flight while the other goes through the chain.  Every load is issued (past the end the last token
// again): with the loads of a batch in front of its own steps, and those of the last T % 8 tokens in front of each, the chain
// waited for memory once per batch and token.
// Measured within a call, us, eight tokens' loads in front of their steps / two batches with 64-bit addresses per lane / now: 45
// tokens, 4096 channels 9.3 / 7.7 / 7.3; chunked, 1024 tokens, 4096 channels 6.3 + 17.3 / 7.2 + 13.9 / 6.4 + 13.9, 513 tokens, 768
// channels 4.7 + 10.5 / 4.4 + 8.1 / 4.0 + 7.8 (the second launch also folds its chunk's predecessors eight at a time, not one).
// Operands in the caches, 1024 tokens, 768 channels 96.6 / 106 / 101.
template <bool OUT, int MODE, class Step>
DEV void wkv4_tokens(const Wkv4IO<MODE> &io, size_t base, int c, int C, int t0, int t1, Step step) {
    constexpr int UNR = 8;
    constexpr bool R = OUT && MODE != 0;
    struct Batch { float k[UNR], v[UNR], r[UNR]; } b0, b1;
    size_t row = base + (size_t)t0 * C;
    int left = t1 - t0;       // tokens from `row` on
    auto load = [&](Batch &b, int at) {
        const Rows<typename Wkv4IO<MODE>::KV> k(io.k + row), v(io.v + row);
        const Rows<rwkv_half> r(io.r + row);
#pragma unroll
        for (int i = 0; i < UNR; ++i) {
            const int o = min(at + i, left - 1) * C;
            b.k[i] = k.ld(o, c);
            b.v[i] = v.ld(o, c);
            b.r[i] = R ? r.ld(o, c) : 0.f;
        }
    };
    load(b0, 0);
    for (; left > 0; left -= 2 * UNR, row += 2 * UNR * (size_t)C) {
        const Rows<typename Wkv4IO<MODE>::Y> y(io.y + row);
        auto one = [&](const Batch &b, int at, int i) {
            float out = 0.f;
            step(b.k[i], b.v[i], out);
            if (OUT) y.st((at + i) * C, c, MODE == 0 ? out : b.r[i] * round_h(out));
        };
        auto run = [&](const Batch &b, int at) {
            if (at + UNR <= left) {   // no branch between the tokens: the division of one runs beside the chain of the next
#pragma unroll
                for (int i = 0; i < UNR; ++i) one(b, at, i);
            } else {
#pragma unroll
                for (int i = 0; i < UNR - 1; ++i)
                    if (at + i < left) one(b, at, i);
            }
        };
        load(b1, UNR);
        run(b0, 0);
        load(b0, 2 * UNR);
        run(b1, UNR);
    }
}

template <int MODE>
__global__ __launch_bounds__(64) void wkv4_kernel(int T, int C, const float *__restrict__ w_, const float *__restrict__ u_,
                                                  Wkv4IO<MODE> io, float *__restrict__ aa_, float *__restrict__ bb_,
                                                  float *__restrict__ pp_) {
    const int c = blockIdx.x * 64 + threadIdx.x;
    const int b = blockIdx.y;
    if (c >= C) return;
    const int so = b * C + c;
    const float u = u_[c], w = w_[c];
    float aa = aa_[so], bb = bb_[so], pp = pp_[so];
    wkv4_tokens<true>(io, (size_t)b * T * C + blockIdx.x * 64, threadIdx.x, C, 0, T, [&](float kk, float vv, float &out) { wkv4_step(kk, vv, u, w, aa, bb, pp, out); });
    aa_[so] = aa; bb_[so] = bb; pp_[so] = pp;
}

// ---------------------------------------------------------------------------------------
// RWKV-4 over a long sequence: the recurrence is a scan with an associative combine, so T is cut into
// chunks that run in parallel.  A state (a, b, p) stands for the sums A = a e^p, B = b e^p; n steps of
// decay add n w to p, and two states merge under the larger exponent.
//   pass 1  (chunk j, channel c): state after the chunk's tokens starting from the empty state
//   pass 2  (chunk j, channel c): incoming state = fold of the call's initial state and the summaries of
//           chunks 0..j-1 (decay by one chunk length between them), then the ordinary per-token steps of
//           the chunk; the last chunk stores the final state.
// Twice the arithmetic of the sequential kernel on T/L times as many lanes.
// scratch: (nchunks + 1) x 3 x C floats; slot 0 holds a copy of the initial state (the final state is
// written over the caller's while other chunks may still read it).
// ---------------------------------------------------------------------------------------
DEV void wkv4_merge(float &a, float &b, float &p, float a2, float b2, float p2) {
    const float q = fmaxf(p, p2);
    const float e1 = __expf(p - q), e2 = __expf(p2 - q);
    a = wkv4_sum(e1, a, e2, a2);
    b = wkv4_sum(e1, b, e2, b2);
    p = q;
}

template <int MODE>
__global__ __launch_bounds__(64) void wkv4_chunk_summary_kernel(int T, int C, int L, const float *__restrict__ w_,
                                                                Wkv4IO<MODE> io, const float *__restrict__ aa_,
                                                                const float *__restrict__ bb_, const float *__restrict__ pp_,
                                                                float *__restrict__ scratch) {
    const int c = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y;
    if (c >= C) return;
    if (j == 0) {
        scratch[c] = aa_[c]; scratch[C + c] = bb_[c]; scratch[2 * C + c] = pp_[c];
    }
    const float w = w_[c];
    float aa = 0.f, bb = 0.f, pp = -1e38f;
    wkv4_tokens<false>(io, 0, c, C, j * L, min(T, (j + 1) * L), [&](float kk, float vv, float &) {
        const float ww = w + pp;
        const float p = fmaxf(ww, kk);
        const float e1 = __expf(ww - p), e2 = __expf(kk - p);
        aa = wkv4_sum(e1, aa, e2, vv);
        bb = __builtin_fmaf(e1, bb, e2);
        pp = p;
    });
    float *o = scratch + (size_t)(j + 1) * 3 * C;
    o[c] = aa; o[C + c] = bb; o[2 * C + c] = pp;
}

template <int MODE>
__global__ __launch_bounds__(64) void wkv4_chunk_apply_kernel(int T, int C, int L, const float *__restrict__ w_,
                                                              const float *__restrict__ u_, Wkv4IO<MODE> io,
                                                              float *__restrict__ aa_, float *__restrict__ bb_,
                                                              float *__restrict__ pp_, const float *__restrict__ scratch) {
    const int c = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y;
    if (c >= C) return;
    const float u = u_[c], w = w_[c];
    const int t0 = j * L, t1 = min(T, t0 + L);
    float aa = scratch[c], bb = scratch[C + c], pp = scratch[2 * C + c];
    const float wl = w * (float)L;
    constexpr int FOLD = 8;
    for (int i0 = 0; i0 < j; i0 += FOLD) {
        float a2[FOLD], b2[FOLD], p2[FOLD];
#pragma unroll
        for (int i = 0; i < FOLD; ++i) {
            const float *sm = scratch + (size_t)(min(i0 + i, j - 1) + 1) * 3 * C;
            a2[i] = sm[c]; b2[i] = sm[C + c]; p2[i] = sm[2 * C + c];
        }
#pragma unroll
        for (int i = 0; i < FOLD; ++i)
            if (i0 + i < j) {
                pp += wl;
                wkv4_merge(aa, bb, pp, a2[i], b2[i], p2[i]);
            }
    }
    wkv4_tokens<true>(io, 0, c, C, t0, t1, [&](float kk, float vv, float &out) { wkv4_step(kk, vv, u, w, aa, bb, pp, out); });
    if (t1 == T) { aa_[c] = aa; bb_[c] = bb; pp_[c] = pp; }
}

// Chunk length for a T-token call: about sqrt(T), a multiple of 8.
int wkv4_chunk_len(int T) {
    int L = 16;
    while (L * L < T && L < 128) L <<= 1;
    return L;
}

// ---------------------------------------------------------------------------------------
// RWKV-5 / RWKV-6.  One workgroup of 256 threads per head (N = 64).  Thread (i, q), i = value
// index 0..63, q = key quarter 0..3, keeps S[i][16q .. 16q+16) in registers for the whole call.
// Tokens are processed in slabs of TS: r, k, v, w of the slab are staged in LDS once (one
// barrier), every thread runs the TS steps on its slice reading r/k/w as wave-uniform LDS
// broadcasts, writes its partial y to LDS, and after a second barrier the four quarters are
// summed and stored coalesced.  PER_TOKEN_W: RWKV-6 (w[t][c]); otherwise RWKV-5 (w[c]).
//   y_i = sum_j r_j (u_j k_j v_i + S_ij) ;  S_ij = S_ij w_j + k_j v_i
// ---------------------------------------------------------------------------------------
constexpr int HS = 64;   // head size
constexpr int TS = 16;   // tokens per slab

// Operand forms of the fused model path:
//   IN_F16   r, k, v are fp16 (the fp16-rounded GEMM outputs, widened here) instead of fp32
//   WMODE 0  w[C] fp32, constant decay in (0,1)                         (RWKV-5)
//   WMODE 1  w[T, C] fp32, already exp(-exp(.))                          (RWKV-6 operator interface)
//   WMODE 2  w[T, C] fp16 LoRA output; decay = exp(-exp(t_decay[c] + w)) (RWKV-6 model path)
//   OUT_GN   instead of y fp32, write fp16( fp16(GroupNorm_head(y) * lnx_w + lnx_b) * gate )
//            (GroupNorm over the 64 channels of the head, eps 64e-5, biased variance; gate optional)
struct Wkv56Args {
    int T, C;
    float *state;
    int state_layout;
    const void *r, *k, *v, *w;
    const float *u, *t_decay;
    float *y;
    const float *lnx_w, *lnx_b;
    const rwkv_half *gate;
    rwkv_half *out;
    const rwkv_half *dw2;  // WMODE 3: second decay LoRA matrix, row c = ld coefficients of channel c
    int ld;                // WMODE 3: LoRA rank (multiple of 8); w = tanh(. @ D1) [T, ld] fp16
};

template <bool IN_F16, int WMODE, bool OUT_GN>
__global__ __launch_bounds__(256) void wkv56_kernel(Wkv56Args a) {
    __shared__ __align__(16) float sr[TS][HS], sk[TS][HS], sv[TS][HS], sw[TS][HS];
    __shared__ __align__(16) float su[HS];
    __shared__ float part[TS][4][HS];
    const int T = a.T, C = a.C;
    const int h = blockIdx.x;
    const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
    float *S = a.state + (size_t)h * HS * HS;
    float s[16];
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
        const int j = 16 * q + jj;
        s[jj] = a.state_layout == 0 ? S[i * HS + j] : S[j * HS + i];
    }
    float tdec = 0.f;
    if (WMODE >= 2) tdec = a.t_decay[h * HS + i];
    if (threadIdx.x < HS) {
        su[threadIdx.x] = a.u[h * HS + threadIdx.x];
        if (WMODE == 0) sw[0][threadIdx.x] = ((const float *)a.w)[h * HS + threadIdx.x];
    }
    auto ld = [&](const void *p, size_t o) -> float {
        return IN_F16 ? h2f(((const rwkv_half *)p)[o]) : ((const float *)p)[o];
    };
    for (int t0 = 0; t0 < T; t0 += TS) {
        const int nt = min(TS, T - t0);
        __syncthreads();  // previous slab fully consumed (and su / sw[0] visible)
        for (int e = threadIdx.x; e < nt * HS; e += 256) {
            const int tt = e >> 6, c = e & 63;
            const size_t o = (size_t)(t0 + tt) * C + h * HS + c;
            sr[tt][c] = ld(a.r, o); sk[tt][c] = ld(a.k, o); sv[tt][c] = ld(a.v, o);
            if (WMODE == 1) sw[tt][c] = ((const float *)a.w)[o];
            if (WMODE == 2) sw[tt][c] = expf(-expf(tdec + h2f(((const rwkv_half *)a.w)[o])));
            if (WMODE == 3) {
                // decay LoRA: the rank-ld product for this channel, rounded to fp16 like the matrix product it replaces
                const rwkv_half *wr = a.dw2 + (size_t)(h * HS + c) * a.ld;
                const rwkv_half *dv = (const rwkv_half *)a.w + (size_t)(t0 + tt) * a.ld;
                float acc = 0.f;
                for (int j8 = 0; j8 < (a.ld >> 3); ++j8)
                    acc = dot8_f16(*(const u32x4 *)(wr + 8 * j8), *(const h16x8 *)(dv + 8 * j8), acc);
                sw[tt][c] = expf(-expf(tdec + round_h(acc)));
            }
        }
        __syncthreads();
        for (int tt = 0; tt < nt; ++tt) {
            const float vi = sv[tt][i];
            const float *wrow = WMODE != 0 ? sw[tt] : sw[0];
            float y = 0.f;
#pragma unroll
            for (int jj = 0; jj < 16; jj += 4) {
                const int j = 16 * q + jj;
                const f32x4 r4 = *(const f32x4 *)&sr[tt][j];
                const f32x4 k4 = *(const f32x4 *)&sk[tt][j];
                const f32x4 w4 = *(const f32x4 *)&wrow[j];
                const f32x4 u4 = *(const f32x4 *)&su[j];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = k4[e] * vi;
                    y += r4[e] * (u4[e] * x + s[jj + e]);
                    s[jj + e] = s[jj + e] * w4[e] + x;
                }
            }
            part[tt][q][i] = y;
        }
        __syncthreads();
        // wave q finishes tokens q, q+4, ...: lane = channel, so the GroupNorm of a token's head is
        // a wave reduction
        for (int tt = q; tt < nt; tt += 4) {
            const int c = i;
            const float y = (part[tt][0][c] + part[tt][1][c]) + (part[tt][2][c] + part[tt][3][c]);
            const size_t o = (size_t)(t0 + tt) * C + h * HS + c;
            if (!OUT_GN) {
                a.y[o] = y;
            } else {
                const float mean = wave_sum(y) * (1.f / HS);
                const float d = y - mean;
                const float var = wave_sum(d * d) * (1.f / HS);
                float g = d * rsqrtf(var + 64e-5f) * a.lnx_w[h * HS + c] + a.lnx_b[h * HS + c];
                g = round_h(g);
                if (a.gate) g = g * h2f(a.gate[o]);
                a.out[o] = f2h(g);
            }
        }
    }
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
        const int j = 16 * q + jj;
        if (a.state_layout == 0) S[i * HS + j] = s[jj]; else S[j * HS + i] = s[jj];
    }
}

}  // namespace

extern "C" int rwkv_wkv4_forward(int64_t B, int64_t T, int64_t C, const float *w, const float *u, const void *k,
                                 const void *v, void *y, int kv_dtype, float *aa, float *bb, float *pp,
                                 void *stream) {
    if (!w || !u || !k || !v || !y || !aa || !bb || !pp) return RWKV_E_NULL;
    if (B <= 0 || T <= 0 || C <= 0 || B > 65535 || B * T * C > ((int64_t)1 << 40)) return RWKV_E_SHAPE;
    dim3 grid((unsigned)((C + 63) / 64), (unsigned)B);
    if (kv_dtype == RWKV_DT_F32) {
        Wkv4IO<0> io{(const float *)k, (const float *)v, (float *)y, nullptr};
        if (C <= WKV4_C) {
            hipLaunchKernelGGL(wkv4_kernel<0>, grid, dim3(64), 0, (hipStream_t)stream, (int)T, (int)C, w, u, io, aa, bb, pp);
        } else {   // a row at a time: no offsets between rows
            for (int64_t r = 0; r < B * T; ++r) {
                const int64_t at = r * C, s = r / T * C;
                hipLaunchKernelGGL(wkv4_kernel<0>, dim3(grid.x), dim3(64), 0, (hipStream_t)stream, 1, (int)C, w, u,
                                   (Wkv4IO<0>{io.k + at, io.v + at, io.y + at, nullptr}), aa + s, bb + s, pp + s);
            }
        }
    } else {
        return RWKV_E_DTYPE;
    }
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// fused variant used by the model path: k, v (fp16 or fp32) and fp16 r in; y = fp16(r * fp16(wkv)).
// ---------------------------------------------------------------------------------------
// RWKV-5 / RWKV-6 over a short sequence (32 tokens to WKV_CHUNKED - 1), model path.  A head's 64 value columns never interact (y_i and the
// column S[:, i] depend on v_i only), so a head is split over four workgroups of 16 value columns: 4 H
// workgroups instead of H.  Thread (value i, key group g): lane & 15 = g owns keys 4g..4g+3 of column i,
// lane >> 4 and the wave index give i.  The sum over the 16 key groups of a value is a DPP row sum in
// registers, so the token loop has no barrier and no LDS partials; r, k, w of a slab of tokens are staged
// in LDS once (two barriers per slab).  Raw y goes to an fp32 [T, C] scratch; GroupNorm and the gate need
// the whole head and run in wkv56_gn_kernel.
//   WMODE 0: w[C] fp32 constant decay (RWKV-5);  WMODE 2: fp16 LoRA output [T, C] + t_decay (RWKV-6)
// ---------------------------------------------------------------------------------------
constexpr int TS2 = 32;  // tokens per slab

template <int WMODE>
__global__ __launch_bounds__(256) void wkv56_split_kernel(Wkv56Args a) {
    __shared__ __align__(16) float sr[TS2][HS], sk[TS2][HS], sw[TS2][HS];
    __shared__ float sv[TS2][16];
    const int T = a.T, C = a.C;
    const int h = blockIdx.x >> 2, vb = blockIdx.x & 3;
    const int lane = threadIdx.x & 63, g = lane & 15;
    const int il = (threadIdx.x >> 6) * 4 + (lane >> 4);   // value column within the block of 16
    const int i = vb * 16 + il;
    // staging role: token threadIdx.x / 8 of the slab, channels 8 (threadIdx.x % 8) .. + 7 of the head.  The
    // NEXT slab is fetched into registers before the token loop of the current one, which hides the loads.
    const int stt = threadIdx.x >> 3, sp = threadIdx.x & 7, sc = sp * 8;
    float *S = a.state + (size_t)h * HS * HS;               // [key][value]
    float s[4], u4[4], wc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = 4 * g + e;
        s[e] = S[j * HS + i];
        u4[e] = a.u[h * HS + j];
        wc[e] = WMODE == 0 ? ((const float *)a.w)[h * HS + j] : 0.f;
    }
    float tdec[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) tdec[e] = WMODE == 2 ? a.t_decay[h * HS + sc + e] : 0.f;
    h16x8 pr, pk, pw = {};
    h16x2 pv;
    auto fetch = [&](int t0) {
        const size_t o = (size_t)min(t0 + stt, T - 1) * C + h * HS;   // rows past the end re-read the last one
        pr = *(const h16x8 *)((const rwkv_half *)a.r + o + sc);
        pk = *(const h16x8 *)((const rwkv_half *)a.k + o + sc);
        if (WMODE == 2) pw = *(const h16x8 *)((const rwkv_half *)a.w + o + sc);
        pv = *(const h16x2 *)((const rwkv_half *)a.v + o + vb * 16 + 2 * sp);
    };
    fetch(0);
    for (int t0 = 0; t0 < T; t0 += TS2) {
        const int nt = min(TS2, T - t0);
        __syncthreads();  // previous slab fully consumed
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x4 r4, k4, w4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r4[e] = (float)pr[4 * u + e];
                k4[e] = (float)pk[4 * u + e];
                w4[e] = WMODE == 2 ? expf(-expf(tdec[4 * u + e] + (float)pw[4 * u + e])) : 0.f;
            }
            *(f32x4 *)&sr[stt][sc + 4 * u] = r4;
            *(f32x4 *)&sk[stt][sc + 4 * u] = k4;
            if (WMODE == 2) *(f32x4 *)&sw[stt][sc + 4 * u] = w4;
        }
        sv[stt][2 * sp] = (float)pv[0];
        sv[stt][2 * sp + 1] = (float)pv[1];
        __syncthreads();
        fetch(t0 + TS2);
        struct Tok { float vi; f32x4 r4, k4, w4; };
        auto ldtok = [&](int tt) {
            Tok q;
            q.vi = sv[tt][il];
            q.r4 = *(const f32x4 *)&sr[tt][4 * g];
            q.k4 = *(const f32x4 *)&sk[tt][4 * g];
            q.w4 = WMODE == 2 ? *(const f32x4 *)&sw[tt][4 * g] : f32x4{};
            return q;
        };
        // this thread's share of y for one token (before the sum over the 16 key groups), and the state update
        auto partial = [&](const Tok &q) {
            float y = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = q.k4[e] * q.vi;
                y += q.r4[e] * (u4[e] * x + s[e]);
                s[e] = s[e] * (WMODE == 2 ? q.w4[e] : wc[e]) + x;
            }
            return y;
        };
        auto step = [&](const Tok &q, int tt) {
            const float y = row16_sum(partial(q));
            if (g == 0) a.y[(size_t)(t0 + tt) * C + h * HS + i] = y;
        };
        // eight tokens per pass (TS2 % 8 == 0): their LDS reads are issued together, so the read latency is paid once per
        // eight, and in a full pass the eight row sums (independent of the state chain) run interleaved
        for (int tt = 0; tt < nt; tt += 8) {
            Tok q[8];
#pragma unroll
            for (int p = 0; p < 8; ++p) q[p] = ldtok(tt + p);
            if (tt + 7 < nt) {
                float y[8];
#pragma unroll
                for (int p = 0; p < 8; ++p) y[p] = partial(q[p]);
#pragma unroll
                for (int p = 0; p < 8; ++p) y[p] = row16_sum(y[p]);
                if (g == 0) {
                    float *yo = a.y + (size_t)(t0 + tt) * C + h * HS + i;
#pragma unroll
                    for (int p = 0; p < 8; ++p) yo[p * (size_t)C] = y[p];
                }
            } else {
#pragma unroll
                for (int p = 0; p < 7; ++p)
                    if (tt + p < nt) step(q[p], tt + p);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) S[(4 * g + e) * HS + i] = s[e];
}

// ---------------------------------------------------------------------------------------
// RWKV-5 / RWKV-6 over a sequence, model path, in chunks of 16 tokens.  With A_t the product of the decays of the
// chunk's tokens before t, and S the state (keys x values) the chunk starts from,
//     y_t = (r_t . A_t) S + sum_{s <= t} P_ts v_s,      P_ts = sum_j r_tj k_sj prod_{s < m < t} w_mj   (P_tt: u_j for the product)
//     S'  = A_16 S + sum_s (k_s . prod_{s < m} w_m) v_s^T
// so all that stays sequential is one 16-token step of matrix products.  The recurrence token by token took 245 - 300
// cycles a token, a latency chain on one wave per SIMD.
//   wkv56_chunk_kernel   one workgroup per (head, chunk), all of them independent: r . A, P, the decayed keys, A_16.
//                        Thread (s, key group g) carries k_s times the running product over t, the factors in the
//                        order the recurrence applies them (no logarithms, no quotients: any decay in [0, 1]).
//   wkv56_apply_kernel   workgroup (head, 16 values), wave jb = keys 16 jb .. + 15, one 16 x 16 block of S in MFMA
//                        accumulators for the whole call, v_mfma_f32_16x16x4_f32 throughout (fp32 operands and sums).
//                        An accumulator register of S is the second operand of r . A times S as it stands: key
//                        16 jb + 4 q + e in lane group q is inner index q of step e.  The four waves' shares of y
//                        meet in LDS, one barrier per chunk, off the state's chain.  The first kernel leaves every
//                        operand in fragment order (five loads per wave and chunk) and pads the chunks to whole
//                        groups of PD, so that PD chunks are in flight with no load, store or wait under a branch.
// Raw y goes to an fp32 [T, C] scratch; GroupNorm and the gate need the whole head and follow in wkv56_gn_kernel.
// A matrix product multiplies a token's values by the zeros of P for the tokens before it too, which would make NaN of
// those where a value is not finite.  Such values count as 0 in P v (not in the state, which they break for good, and the
// later chunks with it) and their column of y is set to NaN from their token on once the call is through: a select per chunk.
// Calls longer than WKV_SEG tokens run in segments, which bounds the scratch between the two kernels.
// Measured per layer, 64 heads, RWKV-6 (recurrence token by token -> chunks, both without GroupNorm): 1024 tokens 111 ->
// 50 us, 256 tokens 29.6 -> 19.4; RWKV-5, 32 heads, 333 tokens 29.3 -> 18.1.  At 64 tokens the second launch costs what
// the chunks save (11.1 -> 12.9 us), at 96 it does not (14.4 -> 13.0): WKV_CHUNKED.
//   WMODE 0: w[C] fp32 constant decay (RWKV-5);  WMODE 2: fp16 LoRA output [T, C] + t_decay (RWKV-6)
// ---------------------------------------------------------------------------------------
constexpr int WKV_SPLIT = 32;                         // calls of at least so many tokens split a head over four workgroups
constexpr int WKV_SEG = 2048;                         // tokens per segment
constexpr int WKV_CHUNKED = 80;                       // calls of at least so many tokens run in chunks
// one chunk's operands, in floats: r . A and decayed keys as [key block][lane][4], P as [key block][lane], A_16 [64], and
// the values (fp16) as [value block][lane][4]
constexpr int CH_R = 0, CH_K = CL * HS, CH_P = 2 * CL * HS, CH_A = CH_P + CL * CL, CH_V = CH_A + HS, CH_FLOATS = CH_V + CL * HS / 2;

template <int WMODE>
__global__ __launch_bounds__(256) void wkv56_chunk_kernel(Wkv56Args a, int H, int t_begin, float *__restrict__ scratch) {
    __shared__ __align__(16) float sr[CL][HS], sw[CL][HS];   // sr: later the keys in fragment order
    __shared__ __align__(16) h16 vf[CL * HS];
    const int T = a.T, C = a.C;
    const int h = blockIdx.x % H, c = blockIdx.x / H;
    const int s = threadIdx.x >> 4, g = threadIdx.x & 15;   // token of the chunk, keys 4 g .. 4 g + 3
    float *out = scratch + (size_t)blockIdx.x * CH_FLOATS;
    const int t = t_begin + c * CL + s;
    const bool live = t < T;                                // past the end: r = k = 0, w = 1
    const size_t o = (size_t)min(t, T - 1) * C + h * HS + 4 * g;
    const h16x4 r8 = *(const h16x4 *)((const rwkv_half *)a.r + o), k8 = *(const h16x4 *)((const rwkv_half *)a.k + o);
    const h16x4 v8 = *(const h16x4 *)((const rwkv_half *)a.v + o);
    h16x4 x8 = {};
    if (WMODE == 2) x8 = *(const h16x4 *)((const rwkv_half *)a.w + o);
    f32x4 r4, k4, w4, u4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = h * HS + 4 * g + e;
        u4[e] = a.u[j];
        w4[e] = WMODE == 2 ? expf(-expf(a.t_decay[j] + (float)x8[e])) : ((const float *)a.w)[j];
        r4[e] = live ? (float)r8[e] : 0.f;
        k4[e] = live ? (float)k8[e] : 0.f;
        w4[e] = live ? w4[e] : 1.f;
    }
    *(f32x4 *)&sr[s][4 * g] = r4;
    *(f32x4 *)&sw[s][4 * g] = w4;
    __syncthreads();
    // x: the product of the decays before token s while m < s, then k_s times the decays after it; a wave holds the
    // tokens 4 wave .. + 3, so what a step needs is decided per wave except at those four
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 before = {1.f, 1.f, 1.f, 1.f}, x = before;
    float mine = 0.f;
#pragma unroll
    for (int m = 0; m < CL; ++m) {
        const f32x4 wm = *(const f32x4 *)&sw[m][4 * g];
        if (m < 4 * wave) {
            x *= wm;
        } else {
            const f32x4 rm = *(const f32x4 *)&sr[m][4 * g];
            const bool own = m == s, mixed = m < 4 * wave + 4;
            if (mixed) {
                before = own ? x : before;
                x = own ? k4 * u4 : x;
            }
            const float p = row16_sum((rm[0] * x[0] + rm[1] * x[1]) + (rm[2] * x[2] + rm[3] * x[3]));
            if (g == m) mine = s <= m ? p : 0.f;            // P[m][s]
            x = mixed && own ? k4 : x * wm;
        }
    }
    // fragment order: token or key in the lower lane bits, the inner index q above them, the step e innermost
    *(f32x4 *)(out + CH_R + 256 * (g >> 2) + 4 * (s + 16 * (g & 3))) = r4 * before;
    out[CH_P + 64 * (s >> 2) + g + 16 * (s & 3)] = mine;
    if (s == CL - 1) *(f32x4 *)(out + CH_A + 4 * g) = before * w4;
    __syncthreads();
    float *kf = &sr[0][0];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int f = 256 * (g >> 2) + 4 * (4 * (g & 3) + e + 16 * (s & 3)) + (s >> 2);
        kf[f] = x[e];
        vf[f] = live ? v8[e] : (h16)0.f;
    }
    __syncthreads();
    *(f32x4 *)(out + CH_K + 4 * threadIdx.x) = *(const f32x4 *)(kf + 4 * threadIdx.x);
    *(h16x4 *)((h16 *)(out + CH_V) + 4 * threadIdx.x) = *(const h16x4 *)(vf + 4 * threadIdx.x);
}

constexpr int GC = 4;   // chunks per exchange of y: one barrier each, and the sums of a group are read during the next
static int wkv56_chunks(int tokens) { return (tokens + CL * GC - 1) / (CL * GC) * GC; }   // whole groups
__global__ __launch_bounds__(256, 2) void wkv56_apply_kernel(Wkv56Args a, int H, int t_begin, int nchunk, const float *scratch) {
    __shared__ f32x4 red[2][GC][4][64];
    const int C = a.C;
    const int h = blockIdx.x % H, ib = blockIdx.x / H;
    const int lane = threadIdx.x & 63, jb = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15, q = lane >> 4;
    const int i = 16 * ib + n16;                            // value column of the accumulators
    float *S = a.state + (size_t)h * HS * HS;               // [key][value]
    f32x4 st;
#pragma unroll
    for (int e = 0; e < 4; ++e) st[e] = S[(16 * jb + 4 * q + e) * HS + i];
    struct Ops { f32x4 r, k, al; float p; h16x4 v; };
    auto load = [&](Ops &x, int c) {
        const float *in = scratch + ((size_t)min(c, nchunk - 1) * H + h) * CH_FLOATS;
        x.r = *(const f32x4 *)(in + CH_R + 256 * jb + 4 * lane);
        x.k = *(const f32x4 *)(in + CH_K + 256 * jb + 4 * lane);
        x.al = *(const f32x4 *)(in + CH_A + 16 * jb + 4 * q);
        x.p = in[CH_P + 64 * jb + lane];
        x.v = *(const h16x4 *)((const h16 *)(in + CH_V) + 256 * ib + 4 * lane);
    };
    float *yo = a.y + (size_t)(t_begin + 4 * q + jb) * C + h * HS + i;   // register jb of a lane's y: token 4 q + jb
    bool broken = false;                                    // this wave's share of the values was not all finite
    auto step = [&](const Ops &x, int buf, int u) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (float)x.v[e];
        const float v01 = jb == 0 ? v[0] : v[1], v23 = jb == 2 ? v[2] : v[3], vj = jb < 2 ? v01 : v23;
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
        const bool fin = __builtin_isfinite(vj);
        broken |= !fin;
        y = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p, fin ? vj : 0.f, y, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) y = __builtin_amdgcn_mfma_f32_16x16x4f32(x.r[e], st[e], y, 0, 0, 0);
        st *= x.al;
#pragma unroll
        for (int e = 0; e < 4; ++e) st = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[e], v[e], st, 0, 0, 0);
        red[buf][u][jb][lane] = y;
    };
    float part[GC][4];
    auto exchange = [&](int buf) {
        __builtin_amdgcn_s_waitcnt(0xC07F);   // LDS only: __syncthreads() would also wait for the loads in flight
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");        // no read of the exchange ahead of the barrier
#pragma unroll
        for (int u = 0; u < GC; ++u)
#pragma unroll
            for (int w = 0; w < 4; ++w) part[u][w] = ((const float *)&red[buf][u][w][lane])[jb];
    };
    auto store = [&]() {
#pragma unroll
        for (int u = 0; u < GC; ++u) {
            *yo = (part[u][0] + part[u][1]) + (part[u][2] + part[u][3]);
            yo += (size_t)CL * C;
        }
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
    static_assert(PD == 2 * GC, "two groups per turn of the loop");
    for (int c0 = 0; c0 < nchunk; c0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            step(ops[u], u / GC, u % GC);
            fence();
            load(ops[u], c0 + u + PD);
            fence();
            if (u == GC - 1) {
                if (c0) store();                  // the second group of the turn before
                exchange(0);
                fence();
                if (c0 + GC >= nchunk) break;
            }
        }
        if (c0 + GC >= nchunk) break;
        store();
        exchange(1);
        fence();
    }
    store();
#pragma unroll
    for (int e = 0; e < 4; ++e) S[(16 * jb + 4 * q + e) * HS + i] = st[e];
    if (any_wave(broken, (int *)red[nchunk / GC & 1])) {    // the buffer that was read before the last barrier
        yo -= (size_t)nchunk * CL * C;                      // the same thread stored these
        for (int c = 0; c < nchunk; ++c, yo += (size_t)CL * C) {
            Ops x;
            load(x, c);
            int first = CL;
#pragma unroll
            for (int e = 3; e >= 0; --e)
                if (!__builtin_isfinite((float)x.v[e])) first = 4 * e + q;
            first = min(first, __shfl_xor(first, 16, WAVE));
            first = min(first, __shfl_xor(first, 32, WAVE));
            if (4 * q + jb >= first) *yo = NAN;
        }
    }
}

// GroupNorm over each head's 64 outputs (eps 64e-5), affine, fp16 rounding, gate.  Four adjacent channels per lane
// (16-byte loads of y and of the affine vectors, 8-byte accesses to the gate and the output): a row of 16 lanes owns
// one head of one token, its two sums are DPP row sums; a workgroup has 256 of the C / 4 chunks of one row.
__global__ __launch_bounds__(256) void wkv56_gn_kernel(int per_row, uint64_t factor, int C, const float *__restrict__ y,
                                                       const float *__restrict__ lnx_w, const float *__restrict__ lnx_b,
                                                       const rwkv_half *__restrict__ gate, rwkv_half *__restrict__ out) {
    const int cpr = C / 4;   // a multiple of 16: whole rows of lanes are live or idle together
    {
        const int t = div_by(blockIdx.x, factor), i = ((int)blockIdx.x - t * per_row) * 256 + threadIdx.x;
        const bool live = i < cpr;
        const int c = min(i, cpr - 1) * 4;
        const size_t o = (size_t)t * C + c;
        const f32x4 y4 = *(const f32x4 *)(y + o), w4 = *(const f32x4 *)(lnx_w + c), b4 = *(const f32x4 *)(lnx_b + c);
        h16x4 g4 = {};
        if (gate) g4 = *(const h16x4 *)(gate + o);
        const float mean = row16_sum((y4[0] + y4[1]) + (y4[2] + y4[3])) * (1.f / HS);
        float sq = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float d = y4[e] - mean; sq += d * d; }
        const float rstd = rsqrtf(row16_sum(sq) * (1.f / HS) + 64e-5f);
        h16x4 o4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float gq = round_h((y4[e] - mean) * rstd * w4[e] + b4[e]);
            if (gate) gq = gq * (float)g4[e];
            o4[e] = (h16)gq;
        }
        if (live) *(h16x4 *)(out + o) = o4;
    }
}


size_t wkv56_scratch_bytes(int64_t T, int64_t C) {
    if (T < WKV_SPLIT) return 256;
    if (T < WKV_CHUNKED) return (size_t)T * C * sizeof(float);   // raw y
    return ((size_t)wkv_chunks(T) * CL * C + (size_t)wkv_chunks(std::min<int64_t>(T, WKV_SEG)) * (C / HS) * CH_FLOATS) * sizeof(float);
}

size_t wkv4_scratch_bytes(int64_t T, int64_t C) {
    if (T < 64) return 256;
    const int L = wkv4_chunk_len((int)T);
    return (size_t)((T + L - 1) / L + 1) * 3 * (size_t)C * sizeof(float);
}

template <int MODE>
static void wkv4_fused_run(int T, int C, const float *w, const float *u, Wkv4IO<MODE> io, float *aa, float *bb, float *pp,
                           float *scratch, hipStream_t st) {
    if (T >= 64 && scratch) {
        const int L = wkv4_chunk_len(T);
        const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((T + L - 1) / L));
        hipLaunchKernelGGL(wkv4_chunk_summary_kernel<MODE>, grid, dim3(64), 0, st, T, C, L, w, io, aa, bb, pp, scratch);
        hipLaunchKernelGGL(wkv4_chunk_apply_kernel<MODE>, grid, dim3(64), 0, st, T, C, L, w, u, io, aa, bb, pp, scratch);
    } else {
        hipLaunchKernelGGL(wkv4_kernel<MODE>, dim3((unsigned)((C + 63) / 64), 1), dim3(64), 0, st, T, C, w, u, io, aa, bb, pp);
    }
}

int wkv4_fused_launch(int T, int C, const float *w, const float *u, const void *k, const void *v, int kv_f32,
                      const rwkv_half *r, rwkv_half *y, float *aa, float *bb, float *pp, hipStream_t st, float *scratch) {
    if (kv_f32) {
        Wkv4IO<2> io{(const float *)k, (const float *)v, y, r};
        wkv4_fused_run<2>(T, C, w, u, io, aa, bb, pp, scratch, st);
    } else {
        Wkv4IO<1> io{(const rwkv_half *)k, (const rwkv_half *)v, y, r};
        wkv4_fused_run<1>(T, C, w, u, io, aa, bb, pp, scratch, st);
    }
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

static int wkv56_launch(bool v6, int64_t B, int64_t T, int64_t C, int64_t H, float *state, int state_layout,
                        const float *r, const float *k, const float *v, const float *w, const float *u, float *y,
                        void *stream) {
    if (!state || !r || !k || !v || !w || !u || !y) return RWKV_E_NULL;
    if (B != 1 || T <= 0 || H <= 0 || C != H * HS) return RWKV_E_SHAPE;
    if (state_layout != 0 && state_layout != 1) return RWKV_E_DTYPE;
    Wkv56Args a{};
    a.T = (int)T; a.C = (int)C; a.state = state; a.state_layout = state_layout;
    a.r = r; a.k = k; a.v = v; a.w = w; a.u = u; a.y = y;
    if (v6)
        hipLaunchKernelGGL((wkv56_kernel<false, 1, false>), dim3((unsigned)H), dim3(256), 0, (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL((wkv56_kernel<false, 0, false>), dim3((unsigned)H), dim3(256), 0, (hipStream_t)stream, a);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// Model path: fp16 r, k, v; state in list layout [h][key][value]; GroupNorm (+ gate) fused; fp16 out.
// v6: w = fp16 LoRA output [T, C], t_decay fp32 [C]; v5: w = fp32 decay [C], t_decay unused.
int wkv56_fused_launch(bool v6, int T, int C, int H, float *state, const rwkv_half *r, const rwkv_half *k,
                       const rwkv_half *v, const void *w, const float *t_decay, const float *u, const float *lnx_w,
                       const float *lnx_b, const rwkv_half *gate, rwkv_half *out, hipStream_t st,
                       const rwkv_half *dw2, int ld, float *y32) {
    if (C != H * HS) return RWKV_E_SHAPE;
    Wkv56Args a{};
    a.T = T; a.C = C; a.state = state; a.state_layout = 1;
    a.r = r; a.k = k; a.v = v; a.w = w; a.u = u; a.t_decay = t_decay;
    a.lnx_w = lnx_w; a.lnx_b = lnx_b; a.gate = gate; a.out = out; a.dw2 = dw2; a.ld = ld;
    if (T >= WKV_SPLIT && y32) {
        // raw y to the fp32 scratch, then GroupNorm + gate
        a.y = y32;
        if (T < WKV_CHUNKED) {
            if (v6) hipLaunchKernelGGL((wkv56_split_kernel<2>), dim3((unsigned)(4 * H)), dim3(256), 0, st, a);
            else hipLaunchKernelGGL((wkv56_split_kernel<0>), dim3((unsigned)(4 * H)), dim3(256), 0, st, a);
        }
        float *chunks = y32 + (size_t)wkv_chunks(T) * CL * C;   // y has a row for every padded token
        for (int t0 = 0; t0 < T && T >= WKV_CHUNKED; t0 += WKV_SEG) {
            const int nchunk = wkv56_chunks(std::min(T - t0, WKV_SEG));
            const dim3 grid((unsigned)(H * nchunk));
            if (v6) hipLaunchKernelGGL((wkv56_chunk_kernel<2>), grid, dim3(256), 0, st, a, H, t0, chunks);
            else hipLaunchKernelGGL((wkv56_chunk_kernel<0>), grid, dim3(256), 0, st, a, H, t0, chunks);
            hipLaunchKernelGGL(wkv56_apply_kernel, dim3((unsigned)(4 * H)), dim3(256), 0, st, a, H, t0, nchunk, chunks);
        }
        const int per_row = (C / 4 + 255) / 256;
        hipLaunchKernelGGL(wkv56_gn_kernel, dim3((unsigned)(T * per_row)), dim3(256), 0, st, per_row, div_factor(per_row), C, y32, lnx_w, lnx_b,
                           gate, out);
    } else if (v6 && dw2) {
        if (ld <= 0 || (ld & 7)) return RWKV_E_SHAPE;
        hipLaunchKernelGGL((wkv56_kernel<true, 3, true>), dim3((unsigned)H), dim3(256), 0, st, a);
    } else if (v6)
        hipLaunchKernelGGL((wkv56_kernel<true, 2, true>), dim3((unsigned)H), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((wkv56_kernel<true, 0, true>), dim3((unsigned)H), dim3(256), 0, st, a);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

extern "C" int rwkv_wkv5_forward(int64_t B, int64_t T, int64_t C, int64_t H, float *state, int state_layout,
                                 const float *r, const float *k, const float *v, const float *w, const float *u,
                                 float *y, void *stream) {
    return wkv56_launch(false, B, T, C, H, state, state_layout, r, k, v, w, u, y, stream);
}

extern "C" int rwkv_wkv6_forward(int64_t B, int64_t T, int64_t C, int64_t H, float *state, int state_layout,
                                 const float *r, const float *k, const float *v, const float *w, const float *u,
                                 float *y, void *stream) {
    return wkv56_launch(true, B, T, C, H, state, state_layout, r, k, v, w, u, y, stream);
}
