// LayerNorm, token shift and mixes of rows of fp16 channels: what the kernels of sequence calls share (internal).
#pragma once
#include <type_traits>
#include "common.h"

namespace {

// ---- LayerNorm and mix, eight channels at a time ----------------------------------------------------------------
// Long calls are bound by vector-instruction issue, so each step is the fewest instructions that form the same value:
// sums and x - mean read their fp16 operand in place (v_fma_mix_f32 with 1.0: one rounding, as a conversion and an addition),
// the affine and the mixes end in v_fma_mix{lo,hi}_f16, sums of products take two channels per v_dot2_f32_f16.  The compiler
// takes two to four instructions for each of these.
DEV h16x2 pair(h16x8 v, int p) { return h16x2{v[2 * p], v[2 * p + 1]}; }
DEV float dot8(h16x8 v, h16x8 w, float a) {
#pragma unroll
    for (int p = 0; p < 4; ++p) a = __builtin_amdgcn_fdot2(pair(v, p), pair(w, p), a, false);
    return a;
}
// a + v[0] + v[1] ... in that order: calls of a few tokens return the same bits whatever adds up a row (v_dot2 with ones takes
// half the instructions and rounds otherwise; a deep RWKV-6 model at the start of a conversation, whose state is nearly empty,
// turns a last bit into percents of its logits)
DEV float sum8(h16x8 v, float a) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(a) : "v"(pair(v, p)));
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(a) : "v"(pair(v, p)));
    }
    return a;
}
DEV void less_mean8(h16x8 v, float mean, float (&d)[8]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(d[2 * p]) : "v"(pair(v, p)), "v"(mean));
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d[2 * p + 1]) : "v"(pair(v, p)), "v"(mean));
    }
}
// a + d[0]^2 + d[1]^2 ..., in that order but for the first two of a chain that starts at zero (FIRST): d[1]^2, then d[0]^2
template <bool FIRST>
DEV float squares8(const float (&d)[8], float a) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float f = d[FIRST && e < 2 ? 1 - e : e];
        a = __builtin_fmaf(f, f, a);
    }
    return a;
}
// a + v[0] + v[1] ..., and b + v[0]^2 + v[1]^2 ... in that order
DEV void sum_and_squares8(h16x8 v, float &a, float &b) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(a) : "v"(pair(v, p)));
        asm("v_fma_mix_f32 %0, %1, %1, %0 op_sel_hi:[1,1,0]" : "+v"(b) : "v"(pair(v, p)));
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(a) : "v"(pair(v, p)));
        asm("v_fma_mix_f32 %0, %1, %1, %0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "+v"(b) : "v"(pair(v, p)));
    }
}
// fp16(fma(t, w, b)) of two channels
DEV h16x2 fma_pair(float t0, float t1, h16x2 w, h16x2 b) {
    h16x2 r;
    asm("v_fma_mixlo_f16 %0, %1, %3, %4 op_sel_hi:[0,1,1]\n\tv_fma_mixhi_f16 %0, %2, %3, %4 op_sel:[0,1,1] op_sel_hi:[0,1,1]"
        : "=&v"(r) : "v"(t0), "v"(t1), "v"(w), "v"(b));
    return r;
}
DEV h16x8 join8(const h16x2 (&q)[4]) { return h16x8{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y}; }
DEV h16x8 norm8(const float (&d)[8], float rstd, h16x8 w, h16x8 b) {
    h16x2 q[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) q[p] = fma_pair(d[2 * p] * rstd, d[2 * p + 1] * rstd, pair(w, p), pair(b, p));
    return join8(q);
}
// A token's mix of a channel: fp16(xx m + prev (1 - m)) (RWKV-4, 5), or fp16(xx + fp16(prev - xx) m) (RWKV-6, 7: maa_form).
// The first as fma(xx, m, prev (1 - m)): prev + (xx - prev) m takes two instructions instead of three, and makes NaN of an
// infinite prev beside a finite xx.  us within a prompt of 1024 rows of 4096 channels, that form and this: three scaled mixes
// 16.2 / 16.6, two 12.8 / 13.5.
DEV h16x8 mix8(h16x8 xx, h16x8 prev, h16x8 m, bool maa_form) {
    if (maa_form) return __builtin_elementwise_fma(prev - xx, m, xx);
    h16x2 q[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const h16x2 x2 = pair(xx, p), p2 = pair(prev, p), m2 = pair(m, p);
        float r0, r1;                // 1 - m, then its product with prev: + -0.0 leaves every product as it is
        asm("v_fma_mix_f32 %0, %1, -1.0, 1.0 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(m2));
        asm("v_fma_mix_f32 %0, %1, -1.0, 1.0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(m2));
        asm("v_fma_mix_f32 %0, %0, %1, %2 op_sel_hi:[0,1,0]" : "+v"(r0) : "v"(p2), "v"(-0.f));
        asm("v_fma_mix_f32 %0, %0, %1, %2 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(r1) : "v"(p2), "v"(-0.f));
        asm("v_fma_mixlo_f16 %0, %1, %2, %3 op_sel_hi:[1,1,0]\n\tv_fma_mixhi_f16 %0, %1, %2, %4 op_sel:[1,1,0] op_sel_hi:[1,1,0]"
            : "=&v"(q[p]) : "v"(x2), "v"(m2), "v"(r0), "v"(r1));
    }
    return join8(q);
}
DEV float row_mean(float sum, int C) { return sum / C; }
DEV float row_rstd(float squares, int C) { return rsqrtf(squares / C + LN_EPS); }

// K sums over a row whose 8-wide chunks are dealt to 256 threads, chunk v, v + 256, ... to thread v, each thread adding up
// its own in that order: add(v, first) adds this thread's chunks to v, first: v is zero (a true_type or false_type).  With 512 threads the second 256 hold the later half of
// those chunks and go on, through LDS, from where the first left off: the same additions in the same order, so the
// totals are the same bits with either number of threads.  v starts at zero; red: 4 K floats of these sums' own, 16-byte
// aligned; hop: K * 256 floats (512 threads only).
template <int K, int NT, class Add>
DEV void row_sums(float (&v)[K], float *red, float *hop, Add add) {
    static_assert(NT == 256 || NT == 512, "two threads per chain at most");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (NT == 512) {
        const int chain = threadIdx.x & 255;
        if (wave < 4) {
            add(v, std::true_type{});
#pragma unroll
            for (int k = 0; k < K; ++k) hop[k * 256 + chain] = v[k];
        }
        __syncthreads();
        if (wave >= 4)
#pragma unroll
            for (int k = 0; k < K; ++k) v[k] = hop[k * 256 + chain];
    }
    if (NT == 256 || wave >= 4) {
        add(v, std::integral_constant<bool, NT == 256>{});
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = wave_sum_lane63(v[k]);
        if ((threadIdx.x & 63) == 63)
#pragma unroll
            for (int k = 0; k < K; ++k) red[k * 4 + (wave & 3)] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const f32x4 r = *(const f32x4 *)(red + 4 * k);
        v[k] = ((r[0] + r[1]) + r[2]) + r[3];
    }
}

}  // namespace
