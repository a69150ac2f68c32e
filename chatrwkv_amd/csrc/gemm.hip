// Prefill contraction y[T, M] = xs[T, N] @ W on fp16 MFMA.
//
// W is read in the input-contiguous layout (row m = N consecutive uint8 or fp16).  For
// uint8 weights each 16-byte global load is widened in registers to the exact fp16 values
// (b + 0.5) -- v_perm_b32 builds 1024 + b, one packed fp16 add removes 1023.5 -- and stored to
// LDS, so the matrix cores see a plain fp16 x fp16 product with fp32 accumulation.  The
// activation operand is the caller's x pre-multiplied by ry (mm8_prepare below), and the
// rank-1 corrections enter in the epilogue:
//     y[t, m] = rx[m] * acc[t, m] + mx[m] * S0[t] + S2[t],   S0 = sum_j x[t, j],  S2 = sum_j x[t, j] my[j].
//
// Tiling: BT x BM outputs per workgroup of 64 WT WM threads (WT x WM waves, each owning a
// (BT/WT) x (BM/WM) block built from 32x32 MFMA tiles), K step 64, LDS double buffered; both LDS
// tiles are [row][64 halves] with the eight 16-byte chunks of a row XOR-swizzled by (row & 7) so
// that the ds_read_b128 of 32 consecutive rows spreads over all banks.  A wave block of
// 128 x 128 needs 8 fragment reads per 16 MFMAs, which keeps the LDS pipe at half its peak; the
// 64 x 64 block of the small-tile variant needs 4 reads per 4 MFMAs and is LDS-bound, so it is
// only used when a larger tile would leave most CUs idle.
// Workgroup ids are remapped so that the workgroups which share a weight tile (same m0,
// different t0) run on the same XCD and the tile is fetched into that XCD's L2 once.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include "kernels.h"
#include "tile_choice.h"
#include "../../include/rwkv_hip_bench.h"
#include <cstdlib>
#include <mutex>

namespace {

constexpr int BK = 64;  // halves per LDS row

// LDS address (in halves) of 16-byte chunk `chunk` (0..7) of tile row `row`.  Rows are 128 bytes.
// The chunk index is XORed with a per-row key chosen so that a ds_read_b128 / ds_write_b128 is
// conflict free both if the LDS serves 8 lanes x 16 B per cycle from 32 banks (8 consecutive
// rows must hit 8 different chunk slots) and if it serves 16 lanes from 64 banks (the 8 even and
// the 8 odd rows of 16 consecutive rows must each hit 8 different slots).
DEV int swz(int row, int chunk) { return row * BK + ((chunk ^ ((row & 7) ^ ((row >> 3) & 1))) << 3); }

// Epilogue of one output element: rank-1 corrections of the uint8 format, activation / residual, store.
// Explicit fused multiply-adds, the result rounded to fp32 in a register of its own: left to itself the compiler joins
// the second one with the rounding to fp16 that follows where nothing else reads it (v_fma_mixlo_f16, one rounding
// instead of two) and not where something does, and the kernels that end in this epilogue would round differently.
DEV float epi_affine(float v, float rxm, float mxm, float s0, float s2) {
    float r = __builtin_fmaf(rxm, v, __builtin_fmaf(mxm, s0, s2));
    asm("" : "+v"(r));
    return r;
}
// Activation, residual and output scale of K outputs.  v: the contraction after epi_affine; res / gate: the residual and
// gate inputs where ep.act uses them.  The branch on the activation (the same for a whole launch) stands outside the loops
// over the elements: inside them every element stepped over the code of the other activations, and a launch fetched its
// epilogue from 12 KB of instructions.
template <int K, class V>
DEV void epi_act(float (&v)[K], V res, V gate, const GemmEpi &ep) {
#pragma unroll
    for (int e = 0; e < K; ++e) v[e] = round_h(v[e]);
    switch (ep.act) {
        case ACT_SIGMOID:
#pragma unroll
            for (int e = 0; e < K; ++e) v[e] = sigmoidf_(v[e]);
            break;
        case ACT_RELU_SQ:
#pragma unroll
            for (int e = 0; e < K; ++e) { v[e] = fmaxf(v[e], 0.f); v[e] = v[e] * v[e]; }
            break;
        case ACT_SILU:
#pragma unroll
            for (int e = 0; e < K; ++e) v[e] = v[e] * sigmoidf_(v[e]);
            break;
        case ACT_TANH:
#pragma unroll
            for (int e = 0; e < K; ++e) v[e] = tanhf(v[e]);
            break;
        case ACT_GATED_RESIDUAL:
#pragma unroll
            for (int e = 0; e < K; ++e) v[e] = round_h((float)gate[e] * v[e]);
            [[fallthrough]];
        case ACT_RESIDUAL:
#pragma unroll
            for (int e = 0; e < K; ++e) v[e] = (float)res[e] + v[e];
            break;
        default: break;
    }
    if (ep.out_scale != 1.f) {
#pragma unroll
        for (int e = 0; e < K; ++e) v[e] = round_h(v[e]) * ep.out_scale;
    }
}
DEV void gemm_epilogue(float v, int t, int m, float rxm, float mxm, const GemmEpi &ep, void *Y, int64_t ldy) {
    if (ep.rx) v = epi_affine(v, rxm, mxm, ep.s0[t], ep.s2[t]);
    if (ep.raw_f32) {
        ((float *)Y)[(size_t)t * ldy + m] = v;
        return;
    }
    h16 res[1] = {}, gate[1] = {};
    if (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL) res[0] = __builtin_bit_cast(h16, ep.res[(size_t)t * ep.ldres + m]);
    if (ep.act == ACT_GATED_RESIDUAL) gate[0] = __builtin_bit_cast(h16, ep.gate[(size_t)t * ep.ldgate + m]);
    float o[1] = {v};
    epi_act<1, const h16 *>(o, res, gate, ep);
    if (ep.out_dtype == RWKV_DT_F32)
        ((float *)Y)[(size_t)t * ldy + m] = round_h(o[0]);
    else
        ((rwkv_half *)Y)[(size_t)t * ldy + m] = f2h(o[0]);
}

// Epilogue of a few consecutive outputs of one row, operands laid out as dma_ok asks.
// n (< 4 or 8 in the last group of a width that is no multiple of it): values that are there
template <class V, int K>
DEV V load_n(const rwkv_half *p, int n) {
    if (n >= K) return *(const V *)p;
    V v = {};
#pragma unroll
    for (int e = 0; e < K; ++e)
        if (e < n) v[e] = __builtin_bit_cast(h16, p[e]);
    return v;
}
// May these outputs be stored 16 bytes at a time?  (An output width of 50277 has rows that start anywhere.)
__host__ DEV bool wide_rows(int M, int64_t ldy, const void *Y) { return (((M | (int)ldy) & 7) | (int)((uintptr_t)Y & 15)) == 0; }
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// Four outputs: fp32 results, and widths or strides that allow no aligned 16-byte stores of fp16 (no residual, gate or
// emitted sums there).  Fp32 leaves 16 bytes at a time on whatever 4-byte boundary the row has.
DEV void affine4(f32x4 &v, int col, int M, float s0t, float s2t, const GemmEpi &ep) {
    const h16x4 rx4 = load_n<h16x4, 4>(ep.rx + col, M - col), mx4 = load_n<h16x4, 4>(ep.mx + col, M - col);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = epi_affine(v[e], (float)rx4[e], (float)mx4[e], s0t, s2t);
}
DEV void finish_row4(f32x4 v, int t, int col, int M, const GemmEpi &ep, void *Y, int64_t ldy) {
    const int n = M - col;
    const bool f32 = ep.raw_f32 || ep.out_dtype == RWKV_DT_F32;
    const size_t at = (size_t)t * ldy + col;
    if (!ep.raw_f32) {
        h16x4 res4 = {}, gate4 = {};
        if (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL) res4 = *(const h16x4 *)(ep.res + (size_t)t * ep.ldres + col);
        if (ep.act == ACT_GATED_RESIDUAL) gate4 = *(const h16x4 *)(ep.gate + (size_t)t * ep.ldgate + col);
        float o[4] = {v[0], v[1], v[2], v[3]};
        epi_act(o, res4, gate4, ep);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = round_h(o[e]);
    }
    if (f32 && n >= 4) {
        *(f32x4_a4 *)((float *)Y + at) = f32x4_a4{v[0], v[1], v[2], v[3]};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < n) {
            if (f32) ((float *)Y)[at + e] = v[e];
            else ((rwkv_half *)Y)[at + e] = f2h(v[e]);
        }
}
// Eight outputs; the vectors over the columns are the caller's, who may finish several rows with them.
DEV void affine8(float (&v)[8], h16x8 rx8, h16x8 mx8, float s0t, float s2t) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = epi_affine(v[e], (float)rx8[e], (float)mx8[e], s0t, s2t);
}
struct Emit8 { h16x8 ry, my; };
DEV Emit8 emit8(const GemmEpi &ep, int col, bool ok) {
    Emit8 e = {};
    if (ep.emit_ry && ok) { e.ry = *(const h16x8 *)(ep.emit_ry + col); e.my = *(const h16x8 *)(ep.emit_my + col); }
    return e;
}
__host__ DEV bool by_four(int M, int64_t ldy, const void *Y, const GemmEpi &ep) {
    return ep.raw_f32 || ep.out_dtype == RWKV_DT_F32 || !wide_rows(M, ldy, Y);
}
// What eight outputs of row t read besides the contraction: the residual and gate, and (uint8 weights) the row's sums.
// Requested for all rows of a thread before the first one is finished: with the loads inside the loop over the rows every
// row waited for its own, 4 to 16 times 0.5 - 1 us at the end of a launch.
struct EpiIn { h16x8 res, gate; float s0, s2; };
DEV EpiIn epi_in(const GemmEpi &ep, int t, int col, bool ok, bool sums) {
    EpiIn in = {};
    if (!ok) return in;
    if (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL) in.res = *(const h16x8 *)(ep.res + (size_t)t * ep.ldres + col);
    if (ep.act == ACT_GATED_RESIDUAL) in.gate = *(const h16x8 *)(ep.gate + (size_t)t * ep.ldgate + col);
    if (sums) { in.s0 = ep.s0[t]; in.s2 = ep.s2[t]; }
    return in;
}
// activation / residual and 16-byte store of fp16 outputs; a0 / a2: these outputs' share of the emitted row sums (EMIT:
// products that may emit them)
template <bool EMIT>
DEV void finish_row8(float (&v)[8], const EpiIn &in, int t, int col, const GemmEpi &ep, void *Y, int64_t ldy, const Emit8 &em, float &a0, float &a2) {
    epi_act(v, in.res, in.gate, ep);
    h16x8 y8;
    if (EMIT && ep.emit_ry) {
        // what the scaling pass of the next product would make of the fp16 output: fp16(y * ry), sum y, sum y * my
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float yf = (float)(h16)v[e];
            y8[e] = (h16)(yf * (float)em.ry[e]);
            a0 += yf;
            a2 += yf * (float)em.my[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) y8[e] = (h16)v[e];
    }
    *(h16x8 *)((rwkv_half *)Y + (size_t)t * ldy + col) = y8;
}
// Split-K second pass: sums the KS partial slabs [KS][T][M] in slab order (deterministic) and runs the epilogue.
// Four consecutive outputs per thread (M % 4 == 0).
__global__ __launch_bounds__(256) void splitk_epilogue_kernel(int T, int M, int KS, const float *__restrict__ part, void *Y,
                                                              int64_t ldy, GemmEpi ep) {
    const int64_t n4 = (int64_t)T * M / 4, n = (int64_t)T * M;
    const int m4 = M / 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        const int t = (int)(i / m4), m = (int)(i - (int64_t)t * m4) * 4;
        f32x4 v = *(const f32x4 *)(part + 4 * i);
        for (int k = 1; k < KS; ++k) v += *(const f32x4 *)(part + (size_t)k * n + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float rxm = 1.f, mxm = 0.f;
            if (ep.rx) { rxm = h2f(ep.rx[m + e]); mxm = h2f(ep.mx[m + e]); }
            gemm_epilogue(v[e], t, m + e, rxm, mxm, ep, Y, ldy);
        }
    }
}

// The same pass for the direct-to-LDS launches, whose operands are all laid out for 16-byte accesses (dma_ok):
// eight consecutive outputs per thread, all slab loads of a thread in flight together, 16-byte loads of the
// residual / gate rows and 16-byte stores.  Same slab order and the same arithmetic per element as above.
template <int KS>
DEV void slab_sum8(size_t n, const float *__restrict__ p, f32x4 &lo, f32x4 &hi) {
    lo = *(const f32x4 *)p;
    hi = *(const f32x4 *)(p + 4);
    f32x4 pl[KS], ph[KS];
#pragma unroll
    for (int k = 1; k < KS; ++k) {
        pl[k] = *(const f32x4 *)(p + k * n);
        ph[k] = *(const f32x4 *)(p + k * n + 4);
    }
#pragma unroll
    for (int k = 1; k < KS; ++k) { lo += pl[k]; hi += ph[k]; }
}
// Chunk i of eight outputs, i < n8; factor: div_factor of a row's chunks (n8 < 2^20: the slabs fit 64 MB).
DEV void splitk_chunk8(int i, int n8, int M, uint64_t factor, int ks, const float *__restrict__ part, void *Y, int64_t ldy, const GemmEpi &ep) {
    if (i >= n8) return;
    const size_t n = (size_t)n8 * 8;
    const bool four = by_four(M, ldy, Y, ep);
    {
        const int t = div_by((uint32_t)i, factor), col = (i - t * (M / 8)) * 8;
        EpiIn in = {};
        h16x8 rx8 = {}, mx8 = {};
        if (!four) in = epi_in(ep, t, col, true, false);
        if (ep.rx) {   // M % 8 == 0
            rx8 = *(const h16x8 *)(ep.rx + col);
            mx8 = *(const h16x8 *)(ep.mx + col);
            in.s0 = ep.s0[t];
            in.s2 = ep.s2[t];
        }
        f32x4 lo, hi;
        switch (ks) {
            case 2: slab_sum8<2>(n, part + 8 * (size_t)i, lo, hi); break;
            case 3: slab_sum8<3>(n, part + 8 * (size_t)i, lo, hi); break;
            case 4: slab_sum8<4>(n, part + 8 * (size_t)i, lo, hi); break;
            case 5: slab_sum8<5>(n, part + 8 * (size_t)i, lo, hi); break;
            case 6: slab_sum8<6>(n, part + 8 * (size_t)i, lo, hi); break;
            case 7: slab_sum8<7>(n, part + 8 * (size_t)i, lo, hi); break;
            default: slab_sum8<8>(n, part + 8 * (size_t)i, lo, hi); break;   // tile_choice.h: at most eight
        }
        float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if (ep.rx) affine8(v, rx8, mx8, in.s0, in.s2);
        if (four) {
#pragma unroll 1
            for (int g = 0; g < 2; ++g) finish_row4(g ? f32x4{v[4], v[5], v[6], v[7]} : f32x4{v[0], v[1], v[2], v[3]}, t, col + 4 * g, M, ep, Y, ldy);
            return;
        }
        float a0 = 0.f, a2 = 0.f;   // a product that emits row sums does not split K
        finish_row8<false>(v, in, t, col, ep, Y, ldy, Emit8{}, a0, a2);
    }
}

__global__ __launch_bounds__(256) void splitk_epilogue8_kernel(const float *__restrict__ part, uint64_t factor, int n8, int M, int KS, void *Y,
                                                               int64_t ldy, GemmEpi ep) {
    splitk_chunk8((int)blockIdx.x * 256 + threadIdx.x, n8, M, factor, KS, part, Y, ldy, ep);
}

template <bool W_U8, int BT, int BM, int WT, int WM, int PF, bool SPLIT>
DEV void gemm_body(int T, int N, int M, const h16 *__restrict__ A, int64_t lda, const void *__restrict__ Wv, int64_t ldw,
                   void *__restrict__ Y, int64_t ldy, const GemmEpi &ep, int nk_split, float *__restrict__ part) {
    constexpr int NT = 64 * WT * WM;                 // threads per workgroup
    constexpr int RA = NT / 8, RB8 = NT / 4;         // tile rows one pass of 16-byte loads covers (fp16 / uint8 rows)
    static_assert(BT % (32 * WT) == 0 && BM % (32 * WM) == 0 && BT % RA == 0 && BM % RB8 == 0, "tile");
    constexpr int MI = BT / (32 * WT), NI = BM / (32 * WM);  // 32x32 blocks per wave in each direction
    extern __shared__ __align__(16) unsigned char smem[];
    h16 *lA[2], *lB[2];
    lA[0] = (h16 *)smem;
    lB[0] = lA[0] + BT * BK;
    lA[1] = lB[0] + BM * BK;
    lB[1] = lA[1] + BT * BK;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / WM, wc = wave % WM;
    // workgroup -> tile: hardware deals consecutive workgroup ids round-robin to the 8 XCDs;
    // undo that so each XCD gets a contiguous range of tiles, which walk the T direction first.
    const int tiles_t = (T + BT - 1) / BT;
    int bid = blockIdx.x;
    if ((gridDim.x & 7) == 0) bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);
    const int t0 = (bid % tiles_t) * BT, m0 = (bid / tiles_t) * BM;
    if (m0 >= M) return;   // grouped launches size the grid for their widest member

    constexpr int A_LD = BT / RA;                    // 16-byte loads per thread for the A tile
    constexpr int B_LD = W_U8 ? BM / RB8 : BM / RA;  // 16-byte loads per thread for the W tile
    // PF k-tiles are in flight in registers (global latency under load is several k-tile times);
    // the LDS holds the tile being multiplied and the next one.
    u32x4 ra[PF][A_LD], rb[PF][B_LD];

    // split-K: blockIdx.y owns k-tiles [kbase, kbase + nk) and writes raw partial sums to its slab
    const int kbase = SPLIT ? blockIdx.y * nk_split : 0;
    auto load_tiles = [&](u32x4 (&qa)[A_LD], u32x4 (&qb)[B_LD], int kt) {
        const int k0 = (kbase + kt) * BK;
#pragma unroll
        for (int i = 0; i < A_LD; ++i) {
            const int row = (tid >> 3) + RA * i, ch = tid & 7;
            const int t = min(t0 + row, T - 1);
            qa[i] = *(const u32x4 *)(A + (size_t)t * lda + k0 + ch * 8);
        }
        if (W_U8) {
#pragma unroll
            for (int i = 0; i < B_LD; ++i) {
                const int row = (tid >> 2) + RB8 * i, ch = tid & 3;
                const int m = min(m0 + row, M - 1);
                qb[i] = *(const u32x4 *)((const uint8_t *)Wv + (size_t)m * ldw + k0 + ch * 16);  // a 64-byte half line: the other half is the next k-tile, kept in L1
            }
        } else {
#pragma unroll
            for (int i = 0; i < B_LD; ++i) {
                const int row = (tid >> 3) + RA * i, ch = tid & 7;
                const int m = min(m0 + row, M - 1);
                qb[i] = *(const u32x4 *)((const h16 *)Wv + (size_t)m * ldw + k0 + ch * 8);
            }
        }
    };
    auto store_tiles = [&](const u32x4 (&qa)[A_LD], const u32x4 (&qb)[B_LD], int buf) {
#pragma unroll
        for (int i = 0; i < A_LD; ++i) {
            const int row = (tid >> 3) + RA * i, ch = tid & 7;
            *(u32x4 *)(lA[buf] + swz(row, ch)) = qa[i];
        }
        if (W_U8) {
            const h16x2 off = {(h16)1023.5f, (h16)1023.5f};
#pragma unroll
            for (int i = 0; i < B_LD; ++i) {
                const int row = (tid >> 2) + RB8 * i, ch = tid & 3;
                u32x4 lo, hi;
                const uint32_t d[4] = {qb[i].x, qb[i].y, qb[i].z, qb[i].w};
                uint32_t o[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[2 * e] = __builtin_bit_cast(uint32_t, u8pair_lo_1024(d[e]) - off);
                    o[2 * e + 1] = __builtin_bit_cast(uint32_t, u8pair_hi_1024(d[e]) - off);
                }
                lo.x = o[0]; lo.y = o[1]; lo.z = o[2]; lo.w = o[3];
                hi.x = o[4]; hi.y = o[5]; hi.z = o[6]; hi.w = o[7];
                // rows r and r+2 share the XOR key's low bit: alternate which half goes first so the
                // 16 lanes of one write touch 16 different slots
                const int odd = (row >> 1) & 1;
                *(u32x4 *)(lB[buf] + swz(row, 2 * ch + odd)) = odd ? hi : lo;
                *(u32x4 *)(lB[buf] + swz(row, 2 * ch + 1 - odd)) = odd ? lo : hi;
            }
        } else {
#pragma unroll
            for (int i = 0; i < B_LD; ++i) {
                const int row = (tid >> 3) + RA * i, ch = tid & 7;
                *(u32x4 *)(lB[buf] + swz(row, ch)) = qb[i];
            }
        }
    };

    f32x16 acc[MI][NI];
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

    const int nk = SPLIT ? nk_split : N / BK;
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            h16x8 fa[MI], fb[NI];
            const int ch = 2 * ks + (lane >> 5);
#pragma unroll
            for (int a = 0; a < MI; ++a) {
                const int row = wr * (BT / WT) + a * 32 + (lane & 31);
                fa[a] = *(const h16x8 *)(lA[buf] + swz(row, ch));
            }
#pragma unroll
            for (int b = 0; b < NI; ++b) {
                const int row = wc * (BM / WM) + b * 32 + (lane & 31);
                fb[b] = *(const h16x8 *)(lB[buf] + swz(row, ch));
            }
#pragma unroll
            for (int a = 0; a < MI; ++a)
#pragma unroll
                for (int b = 0; b < NI; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[a], fb[b], acc[a][b], 0, 0, 0);
        }
    };
    // Tile kt lives in register slot kt % PF from PF iterations before it is multiplied until it is written
    // to LDS buffer kt & 1 at the end of iteration kt - 1.  Every global load is issued unconditionally (past
    // the end the last k-tile is read again and never used): the compiler places its waits from a static
    // count of the loads issued after the one it needs, and a load under a branch would make it assume the
    // fewest, i.e. drain the whole prefetch queue before every LDS store.
#pragma unroll
    for (int p = 0; p < PF; ++p) load_tiles(ra[p], rb[p], min(p, nk - 1));
    store_tiles(ra[0], rb[0], 0);
    __syncthreads();
    for (int kt0 = 0; kt0 < nk; kt0 += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int kt = kt0 + p;
            load_tiles(ra[p], rb[p], min(kt + PF, nk - 1));  // slot freed when tile kt went to LDS
            if (kt < nk) compute(kt & 1);
            if (kt + 1 < nk) store_tiles(ra[(p + 1) % PF], rb[(p + 1) % PF], (kt + 1) & 1);
            __syncthreads();
        }
    }

    // epilogue: lane holds column m = .. + (lane & 31) and rows 8*(e/4) + 4*(lane>>5) + e%4
    float *slab = SPLIT ? part + (size_t)blockIdx.y * T * M : nullptr;
#pragma clang loop unroll(full)
    for (int b = 0; b < NI; ++b) {
        const int m = m0 + wc * (BM / WM) + b * 32 + (lane & 31);
        const bool m_ok = m < M;
        float rxm = 1.f, mxm = 0.f;
        if (!SPLIT && ep.rx && m_ok) { rxm = h2f(ep.rx[m]); mxm = h2f(ep.mx[m]); }
#pragma clang loop unroll(full)
        for (int a = 0; a < MI; ++a) {
#pragma clang loop unroll(full)
            for (int e = 0; e < 16; ++e) {
                const int t = t0 + wr * (BT / WT) + a * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (m_ok && t < T) {
                    if (SPLIT) slab[(size_t)t * M + m] = acc[a][b][e];
                    else gemm_epilogue(acc[a][b][e], t, m, rxm, mxm, ep, Y, ldy);
                }
            }
        }
    }
}

template <bool W_U8, int BT, int BM, int WT, int WM, int PF, bool SPLIT>
__global__ __launch_bounds__(64 * WT * WM) void gemm_kernel(int T, int N, int M, const h16 *__restrict__ A, int64_t lda,
                                                   const void *__restrict__ Wv, int64_t ldw, void *__restrict__ Y,
                                                   int64_t ldy, GemmEpi ep, int nk_split, float *__restrict__ part) {
    gemm_body<W_U8, BT, BM, WT, WM, PF, SPLIT>(T, N, M, A, lda, Wv, ldw, Y, ldy, ep, nk_split, part);
}

// ---- operands straight from global memory into LDS ------------------------------------------------------------
// Tiles of 96 to 256 rows and columns, eight waves (2 x 4, with K over two groups 2 x 2 each), stages of one 64-deep k-tile.
// The loads are global_load_lds_dwordx4: one wave instruction copies 64 x 16 B into 1 KB of LDS without passing through
// registers, so no wave spends issue slots on ds_write or on holding prefetched tiles.  A uint8 weight tile stays
// uint8 in LDS (half the bytes of fp16) and becomes fp16 in the fragments on the way to the matrix cores.
// The MFMA is v_mfma_f32_16x16x32_f16.  A chip full of large tiles is bound by its clock under load, and this one does more for
// the power: loops of nothing but MFMAs on random operands sustain 1810 to 1870 TFLOP/s with it and 1600 to 1620 with v_mfma_f32_32x32x16_f16
// (whose accumulator it reads and writes half as often per product).  [1024 x 4096] x [4096 x 16384] 126 -> 115 us (uint8), 133 ->
// 119 (fp16).  It also makes sides that are any multiple of 32, see tile_price.
// LDS layout of a stage: 128-byte rows [row][8 chunks of 16 B], chunk c of row r at slot c ^ ((r >> 1) & 7); uint8 weight rows
// [row][4 chunks of 16 B], chunk c of row r at slot c ^ ((r >> 2) & 3): the fragment reads (16 rows x one chunk per 16 lanes) hit every
// bank once.  The swizzle is applied on the global side: the lane that fills slot p of row r loads chunk p ^ key(r).
// LDS reads are inline asm with hand-placed s_waitcnt: the compiler waits for lgkmcnt(0) wherever older and newer reads are
// both outstanding.
// Schedules of a k-tile, two MFMA steps of 32 k's; its one barrier stands where the reads of the tile are back and the next tile has
// landed:
//   HS = 2     (more than 64 rows a wave) each step in two halves of the row blocks.  A half's activation fragments are read two halves
//              ahead, the uint8 fragments of a step widened behind the MFMAs of the one before; the barrier follows the second half,
//              and with three stages the loads of tile kt + 2 are issued in three parts between the halves.
//   HS = 1     (64 rows a wave) a step's fragments are read while the other step multiplies; the barrier follows the first step, and
//              the loads of the tile NST ahead go into the stage that has just been read.
//   KG = 2     (128 x 128 with four stages, one workgroup to a CU, and the tiles with a side of 96) the waves are two groups of 2 x 2, group g takes step g: 64 x 64 a
//              wave instead of 64 x 32, two fifths fewer fragment bytes; all fragments of a tile are read while the one before
//              multiplies.  us, one step after the other / two groups / as HS = 1: uint8 [256 x 4096] x [4096 x 12288] 38.8 / 37.5 /
//              40.4, [1024 x 4096] x [4096 x 4096] 40.7 / 39.5 / 41.8; fp16 [333 x 2048] x [2048 x 8192] 21.6 / 21.5 / 23.5.
// What a launch of one 256 x 256 tile per CU spends outside its k-tiles, by time stamps (us, uint8, 1024 rows, 115 in all): 4 until the
// first wave and after the last, 2.5 until the first tile is there, 3 until the outputs are in LDS, 7 until they have left (32 MB at once).
// Four stages instead of three on the 128 x 128 tile [256 x 4096] x [4096 x 12288] 46.0 -> 40.2 us; slower where the tiles take
// several rounds, as only one workgroup then fits a CU.
template <bool W_U8, int TM, int TN, int NSTG> struct DmaCfg {
    static constexpr int NW = 8;                                                              // waves
    static constexpr int A = TM * BK * 2, W = W_U8 ? TN * BK : TN * BK * 2, STAGE = A + W;
    static constexpr int NST = NSTG ? NSTG : 3 * STAGE + (W_U8 ? 2 * TM * 4 + 2 * TN * 2 : 0) <= 160 * 1024 ? 3 : 2;
    static constexpr int AP = A / 1024, WP = W / 1024;                                        // 1 KB loads of a stage
    static constexpr int AL = (AP + NW - 1) / NW, WL = (WP + NW - 1) / NW, LOADS = AL + WL;   // per wave; past the end the last one again
    static constexpr int KG = NST == 4 ? 2 : 1;                                               // groups of waves that share K
    static constexpr bool SPLITS = TM != 96 && TN != 96;                                      // K split over workgroups: see tile_choice.h
    static constexpr int WR = 2, WC = NW / WR / KG;                                           // waves of a group: rows, columns
    static constexpr int MI = TM / (16 * WR), NI = TN / (16 * WC);                            // 16 x 16 blocks per wave
    static constexpr int HS = MI > 4 ? 2 : 1, H0 = HS == 2 ? (MI + 1) / 2 : MI;               // row blocks in one or two halves
    static constexpr int STG_STRIDE = TN + 4;   // epilogue staging, floats: 16 bytes apart, so 16 rows fill all banks
    static constexpr int HSTRIDE = TN + 8;      // the same for fp16 outputs
    static constexpr int FROWS = TM > 128 ? TM / 2 : TM;                                      // rows of a pass of the former
    static constexpr int CPR = TN > 128 ? 32 : 16;                                            // threads that finish a row, eight outputs each
    static constexpr size_t max3(size_t a, size_t b, size_t c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }
    static constexpr size_t BODY = max3((size_t)NST * STAGE, (size_t)KG * FROWS * STG_STRIDE * 4, (size_t)TM * HSTRIDE * 2);
    static constexpr size_t LDS = BODY + (W_U8 ? 2 * TM * 4 + 2 * TN * 2 : 0);   // uint8: past the stages the rows' sums s0, s2 and the columns' rx, mx
    static_assert(TM % (16 * WR) == 0 && TN % (16 * WC) == 0 && MI <= 8 && NI <= 4 && H0 <= 4 && 2 * TM <= 64 * NW, "waves");
    static_assert((NST - 1) * LOADS < 64 && LDS <= 160 * 1024 && TN > 64 && TN <= 256, "tile");
};
DEV void emit_parts(const GemmEpi &ep, int t, int m0, int M, int TN, float a0, float a2) {
    const int parts = emitted_parts(M, TN), i = m0 / TN;
    float *p0 = ep.emit_s0 + (size_t)t * parts, *p2 = ep.emit_s2 + (size_t)t * parts;
    p0[i] = a0;
    p2[i] = a2;
    if (m0 + TN >= M)
        for (int j = i + 1; j < parts; ++j) p0[j] = p2[j] = 0.f;
}
// This workgroup's place in a launch of `units` workgroups.  The hardware deals consecutive workgroup ids round-robin to the 8 XCDs;
// undone here, so that each XCD gets a contiguous range of the units: tiles that walk the T direction first and share weight tiles in
// its L2, each with all of its K splits.  Dealt as the hardware does wherever the tiles were no multiple of eight, every XCD read
// all of both operands: fp16, us, [300 x 3200] x [3200 x 3200] 20.5 -> 14.4, [333 x 1280] x [1280 x 3840] 14.1 -> 10.8.  With one split
// after the other instead of one tile after the other an XCD reads a part of every row of the weights: 1 to 2 % slower over 5000 launches.
DEV int xcd_unit(int units) {
    const int x = blockIdx.x & 7, each = units >> 3;
    return x * each + min(x, units & 7) + ((int)blockIdx.x >> 3);
}
// Its place.  The walk goes along T, so that an XCD reads all activations and its own part of the weights, unless the activations
// are the larger operand and more than its 4 MB of L2 hold: then along M.  us, uint8, T -> M: 64 x 64 tile, [2048 x 4096] x [4096 x
// 1024] 49.0 -> 29.1, [777 x 4096] x [4096 x 512] 16.1 -> 14.7; [2048 x 3072] x [3072 x 768] 64 x 128 tile 18.9 -> 17.6, 128 x 128
// in two splits 21.8 -> 20.9; activations that fit: [2048 x 768] x [768 x 768] 10.7 -> 11.2, [1400 x 1024] x [1024 x 1024] 11.7 -> 12.3.
bool walks_m(bool w_u8, int64_t T, int64_t N, int64_t M) { return T * 2 > M * (w_u8 ? 1 : 2) && T * N > (2 << 20); }
struct TileAt { int t0, m0; };
template <int TM, int TN>
DEV TileAt tile_at(int bid, int T, int M, int walk_m) {
    const int n = walk_m ? (M + TN - 1) / TN : (T + TM - 1) / TM, q = bid / n, r = bid - q * n;
    return {(walk_m ? q : r) * TM, (walk_m ? r : q) * TN};
}
// s_waitcnt immediates: vmcnt(n) alone, vmcnt(n) with lgkmcnt(0), lgkmcnt(n) alone
constexpr int vm_only(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int vm_lgkm0(int n) { return 0x0070 | (n & 15) | ((n >> 4) << 14); }
constexpr int lgkm_only(int n) { return 0xC07F | (n << 8); }

template <bool W_U8, bool SPLIT, int TM, int TN, int NSTG>
DEV void gemm_dma_body(int bid, int T, int N, int M, int walk_m, const h16 *__restrict__ A, int64_t lda, const void *__restrict__ Wv,
                       int64_t ldw, void *__restrict__ Y, int64_t ldy, const GemmEpi &ep, int nk_split,
                       float *__restrict__ part, int split) {
    using Cfg = DmaCfg<W_U8, TM, TN, NSTG>;
    constexpr int D_A = Cfg::A, D_STAGE = Cfg::STAGE, D_NST = Cfg::NST, AL = Cfg::AL, WL = Cfg::WL, MI = Cfg::MI, NI = Cfg::NI;
    constexpr int HS = Cfg::HS, H0 = Cfg::H0, KG = Cfg::KG, NW = Cfg::NW;
    extern __shared__ __align__(1024) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave / (Cfg::WR * Cfg::WC), wr = wave / Cfg::WC % Cfg::WR, wc = wave % Cfg::WC;
    const TileAt at = tile_at<TM, TN>(bid, T, M, walk_m);
    const int t0 = at.t0, m0 = at.m0;
    const int kbase = SPLIT ? split * nk_split : 0, nk = nk_split;

    // load sources; rows past the end re-read the last row (never stored)
    auto a_piece = [&](int i) { return min(wave * AL + i, Cfg::AP - 1); };
    auto w_piece = [&](int i) { return min(wave * WL + i, Cfg::WP - 1); };
    const h16 *ga[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
        const int r = a_piece(i) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        ga[i] = A + (size_t)min(t0 + r, T - 1) * lda + (size_t)kbase * BK + c * 8;
    }
    const unsigned char *gw[WL];   // byte pointers
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        if (W_U8) {
            const int r = w_piece(i) * 16 + (lane >> 2), c = (lane & 3) ^ ((r >> 2) & 3);
            gw[i] = (const unsigned char *)Wv + (size_t)min(m0 + r, M - 1) * ldw + (size_t)kbase * BK + c * 16;
        } else {
            const int r = w_piece(i) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
            gw[i] = (const unsigned char *)((const h16 *)Wv + (size_t)min(m0 + r, M - 1) * ldw + (size_t)kbase * BK + c * 8);
        }
    }
    typedef __attribute__((address_space(1))) const void *gptr;
    typedef __attribute__((address_space(3))) void *lptr;
    // part 0 / 1: the halves of this wave's A loads, part 2: its weight loads; -1: all of them
    auto issue = [&](int kt, int so, int part) {
        unsigned char *base = smem + so;
#pragma unroll
        for (int i = 0; i < AL; ++i)
            if (part < 0 || part == (i >= (AL + 1) / 2 ? 1 : 0))
                __builtin_amdgcn_global_load_lds((gptr)(ga[i] + kt * BK), (lptr)(base + a_piece(i) * 1024), 16, 0, 0);
        if (part < 0 || part == 2) {
#pragma unroll
            for (int i = 0; i < WL; ++i)
                __builtin_amdgcn_global_load_lds((gptr)(gw[i] + kt * BK * (W_U8 ? 1 : 2)), (lptr)(base + D_A + w_piece(i) * 1024), 16, 0, 0);
        }
    };

    f32x4 acc[MI][NI];
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int b = 0; b < NI; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Fragments: lane (row, q) takes the k's 16 q + 8 s .. + 7 of the k-tile in MFMA step s, for both operands, so that a uint8
    // weight fragment of both steps is one 16-byte read.  Two groups: group g takes the k's 32 g + 8 q .. + 7.
    // Addresses within a stage; the swizzle keys depend on the lane only.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const int row = lane & 15, q = lane >> 4;
    constexpr int STEPS = KG == 2 ? 1 : 2, WN = W_U8 ? 1 : STEPS;
    uint32_t vA[STEPS], vB[WN];
    auto half_chunk = [&](int s) { return ((KG == 2 ? 4 * grp + q : 2 * q + s) ^ ((row >> 1) & 7)) << 4; };
#pragma unroll
    for (int s = 0; s < STEPS; ++s) vA[s] = lds0 + (wr * 16 * MI + row) * 128 + half_chunk(s);
#pragma unroll
    for (int s = 0; s < WN; ++s)
        vB[s] = lds0 + D_A + (!W_U8 ? (wc * 16 * NI + row) * 128 + half_chunk(s)
                              : (wc * 16 * NI + row) * 64 + (((KG == 2 ? 2 * grp + (q >> 1) : q) ^ ((row >> 2) & 3)) << 4) + (KG == 2 ? (q & 1) * 8 : 0));
    h16x8 fa[2][H0];                             // [set][row block]
    u32x4 rawb[NI];                              // uint8 weights, both steps of a k-tile
    u32x2 rawg[2][NI];                           // the same with two groups: [set]
    h16x8 fb[2][NI];                             // [step], two groups: [set]
    auto ld_a = [&](int set, int so, int s, int half) {
        const uint32_t p = vA[s] + so;
#pragma unroll
        for (int i = 0; i < H0; ++i)
            if (half * H0 + i < MI) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][i]) : "v"(p), "n"((half * H0 + i) * 2048));
    };
    auto ld_w = [&](int so, int s) {   // uint8: both steps, whatever s is
        const uint32_t p = vB[W_U8 ? 0 : s] + so;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if constexpr (W_U8) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(rawb[i]) : "v"(p), "n"(i * 1024));
            else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[s][i]) : "v"(p), "n"(i * 2048));
        }
    };
    auto ld_group = [&](int set, int so) {
        const uint32_t p = vB[0] + so;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if constexpr (W_U8) asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(rawg[set][i]) : "v"(p), "n"(i * 1024));
            else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[set][i]) : "v"(p), "n"(i * 2048));
        }
        ld_a(set, so, 0, 0);
    };
    const h16x2 off = {(h16)1023.5f, (h16)1023.5f};
    auto widen8 = [&](uint32_t x, uint32_t y) {
        const h16x2 q0 = u8pair_lo_1024(x) - off, q1 = u8pair_hi_1024(x) - off, q2 = u8pair_lo_1024(y) - off, q3 = u8pair_hi_1024(y) - off;
        return h16x8{q0.x, q0.y, q1.x, q1.y, q2.x, q2.y, q3.x, q3.y};
    };
    auto widen = [&](int s) {
        if constexpr (W_U8) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
                fb[s][i] = KG == 2 ? widen8(rawg[s][i].x, rawg[s][i].y) : widen8(s ? rawb[i].z : rawb[i].x, s ? rawb[i].w : rawb[i].y);
        }
    };
    // weights first: a lane ends with four consecutive outputs of one row
    auto mfmas = [&](int set, int s, int half) {
#pragma unroll
        for (int a = 0; a < H0; ++a)
            if (half * H0 + a < MI) {
#pragma unroll
                for (int b = 0; b < NI; ++b)
                    acc[half * H0 + a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[s][b], fa[set][a], acc[half * H0 + a][b], 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto reads_done = [&]() {
        __builtin_amdgcn_s_waitcnt(lgkm_only(0));
        __builtin_amdgcn_sched_barrier(0);
    };

    // Every wave issues exactly LOADS loads per tile, so "vmcnt(LOADS n)" means "all but my newest n tiles have
    // landed".  Past the last tile the loads repeat it into a stage nobody reads any more, which keeps the counts static.
    // Three stages: while tile kt multiplies, tile kt + 1 has landed or is landing and the loads of tile kt + 2 are
    // issued in three parts between the MFMA steps, into the stage tile kt - 1 was read from (a burst of all of
    // them right after the barrier measured 2 % slower).  Two stages: tile kt + 2 can only go where tile kt is, so
    // its loads follow the barrier in one go.
    constexpr bool SPREAD = HS == 2 && D_NST >= 3;
    constexpr int PD = HS == 1 ? D_NST : SPREAD ? D_NST - 1 : 2;   // tiles in flight ahead of the one being multiplied
    // What the epilogue reads of the uint8 format is put into LDS while the first tiles are in flight: a row's sums and a column's
    // rx and mx, requested ahead of the tiles.
    float *const lsum = (float *)(smem + Cfg::BODY);
    h16 *const lcol = (h16 *)(lsum + 2 * TM);
    const bool parts = W_U8 && ep.parts > 1;
    float sum1 = 0.f;
    h16x4 col4 = {};
    if constexpr (W_U8 && !SPLIT) {
        if (tid < TN / 2) {
            const int c = tid % (TN / 4) * 4;
            if (m0 + c < M) col4 = load_n<h16x4, 4>((tid < TN / 4 ? ep.rx : ep.mx) + m0 + c, M - m0 - c);
        }
        if (!parts && tid < 2 * TM) sum1 = (tid < TM ? ep.s0 : ep.s2)[min(t0 + tid % TM, T - 1)];
        __builtin_amdgcn_sched_barrier(0);
    }
    issue(0, 0, -1);
    issue(min(1, nk - 1), D_STAGE, -1);
#pragma unroll
    for (int p = 2; p < PD; ++p) issue(min(p, nk - 1), p * D_STAGE, -1);
    if constexpr (W_U8 && !SPLIT) {
        __builtin_amdgcn_sched_barrier(0);
        if (tid < TN / 2) *(h16x4 *)(lcol + tid * 4) = col4;
        if (!parts && tid < 2 * TM) lsum[tid] = sum1;
    }
    // The input's row sums arrive as partial sums per column tile of the launch that produced it: this tile's rows
    // are added up here, in index order, while the first two tiles are in flight (the waits for these loads cover the
    // older tile loads too, so the counted waits below still hold).  Full depth: into LDS for the epilogue;
    // K split: the first column tile's first split writes the totals out for the second pass.
    if constexpr (W_U8) {
        if (parts && (!SPLIT || (m0 == 0 && split == 0))) {
            if (tid < 2 * TM) {
                const int row = tid % TM, which = tid / TM, t = min(t0 + row, T - 1);
                const float *p = (which ? ep.p2 : ep.p0) + (size_t)t * ep.parts;
                float tot = 0.f;
                for (int j = 0; j < ep.parts; j += 64) {   // parts % 4 == 0; up to 64 partial sums in flight per thread
                    f32x4 q[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) q[u] = j + 4 * u < ep.parts ? *(const f32x4 *)(p + j + 4 * u) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int u = 0; u < 16; ++u) tot = (((tot + q[u][0]) + q[u][1]) + q[u][2]) + q[u][3];
                }
                if constexpr (SPLIT) {
                    if (t0 + row < T) (which ? (float *)ep.s2 : (float *)ep.s0)[t] = tot;
                } else {
                    lsum[tid] = tot;
                }
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(vm_only((PD - 1) * Cfg::LOADS));   // tile 0 has landed
    __builtin_amdgcn_s_barrier();
    int so = 0, sp = (D_NST - 1) * D_STAGE;   // the stage being read and (three stages and more) the one read before it
    if constexpr (KG == 1) {
        ld_a(0, 0, 0, 0);
        ld_w(0, 0);
        ld_a(1, 0, HS == 1, HS == 2);
        if (!W_U8 && HS == 1) ld_w(0, 1);
        reads_done();
        widen(0);
    } else {
        ld_group(0, 0);
        reads_done();
    }
    if constexpr (KG == 2) {
        // all fragments of a k-tile are read while the one before multiplies
        auto tile = [&](int kt, int set) {
            const int sn = so + D_STAGE >= D_NST * D_STAGE ? 0 : so + D_STAGE;
            __builtin_amdgcn_s_waitcnt(vm_only((D_NST - 2) * Cfg::LOADS));   // my part of tile kt + 1 has landed
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            ld_group(set ^ 1, sn);
            issue(min(kt + PD, nk - 1), so, -1);
            widen(set);
            mfmas(set, set, 0);
            reads_done();
            so = sn;
        };
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            tile(kt, 0);
            tile(kt + 1, 1);
        }
        if (kt < nk) tile(kt, 0);
    } else if constexpr (HS == 2) {
        for (int kt = 0; kt < nk; ++kt) {
            const int sn = so + D_STAGE >= D_NST * D_STAGE ? 0 : so + D_STAGE;
            const int kl = min(kt + PD, nk - 1);
            mfmas(0, 0, 0);
            reads_done();
            widen(1);
            ld_a(0, so, 1, 0);
            if (!W_U8) ld_w(so, 1);
            if (SPREAD) issue(kl, sp, 0);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(1, 0, 1);
            reads_done();
            ld_a(1, so, 1, 1);
            if (SPREAD) issue(kl, sp, 1);
            __builtin_amdgcn_sched_barrier(0);
            // my part of tile kt + 1 has landed (newer: the A loads of tile kt + 2) and all my reads of tile kt are back
            __builtin_amdgcn_s_waitcnt(vm_lgkm0(SPREAD ? (PD - 2) * Cfg::LOADS + AL : 0));
            __builtin_amdgcn_s_barrier();
            if (!SPREAD) issue(kl, so, -1);
            mfmas(0, 1, 0);
            ld_a(0, sn, 0, 0);
            ld_w(sn, 0);
            if (SPREAD) issue(kl, sp, 2);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(1, 1, 1);
            reads_done();
            widen(0);
            ld_a(1, sn, 0, 1);
            __builtin_amdgcn_sched_barrier(0);
            sp = so;
            so = sn;
        }
    } else {
        for (int kt = 0; kt < nk; ++kt) {
            const int sn = so + D_STAGE >= D_NST * D_STAGE ? 0 : so + D_STAGE;
            const int kl = min(kt + PD, nk - 1);
            mfmas(0, 0, 0);
            widen(1);
            // my part of tile kt + 1 has landed and all my reads of tile kt are back
            __builtin_amdgcn_s_waitcnt(vm_lgkm0((D_NST - 2) * Cfg::LOADS));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            issue(kl, so, -1);
            ld_a(0, sn, 0, 0);
            ld_w(sn, 0);
            __builtin_amdgcn_sched_barrier(0);
            mfmas(1, 1, 0);
            reads_done();
            widen(0);
            ld_a(1, sn, 1, 0);
            if (!W_U8) ld_w(sn, 1);
            __builtin_amdgcn_sched_barrier(0);
            so = sn;
        }
    }
    // vmcnt(0) lgkmcnt(0): nothing may land in LDS after the workgroup has gone -- and nothing in registers: the last
    // iteration has read a fragment set that nobody multiplies.  The compiler does not know that an inline-asm
    // ds_read writes its output later: to it those registers are dead from here on, and it reused them for the
    // epilogue's column index and addresses ahead of this wait (a read that returned late then overwrote the
    // index: an access far outside the buffers).  So the wait comes first, fenced against the scheduler, and every
    // fragment register stays "in use" until it has passed.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int set = 0; set < 2; ++set)
#pragma unroll
        for (int a = 0; a < H0; ++a)
            if (set * H0 + a < MI || HS == 1) asm volatile("" ::"v"(fa[set][a]));
#pragma unroll
    for (int b = 0; b < NI; ++b) {
        if constexpr (W_U8 && KG == 2) asm volatile("" ::"v"(rawg[0][b]), "v"(rawg[1][b]));
        else if constexpr (W_U8) asm volatile("" ::"v"(rawb[b]));
        else asm volatile("" ::"v"(fb[0][b]), "v"(fb[1][b]));
    }
    __builtin_amdgcn_sched_barrier(0);

    constexpr int CPR = Cfg::CPR, RPI = 64 * NW / CPR;   // threads per row, rows per pass of the workgroup
    const int cq = tid % CPR, col = m0 + cq * 8;
    const bool in_tile = cq * 8 < TN, col_ok = in_tile && col < M;
    constexpr int SW = Cfg::STG_STRIDE;                  // row stride of fp32 in LDS, in floats
    float *const stg = (float *)smem;
    constexpr int ITS = TM / RPI, AHEAD_ROWS = KG == 2 ? ITS : ITS % 4 ? 2 : 4;      // rows of a thread; rows requested together
    static_assert(ITS % AHEAD_ROWS == 0 && TM % RPI == 0 && Cfg::FROWS % RPI == 0, "rows");
    // the sums of a row of the tile that the CPR threads finishing it hold, neighbours in one wave: every lane takes part
    auto emit_row = [&](int t, bool valid, float a0, float a2) {
        a0 = row16_sum(a0);
        a2 = row16_sum(a2);
        if constexpr (CPR == 32) { a0 += __shfl_xor(a0, 16, WAVE); a2 += __shfl_xor(a2, 16, WAVE); }
        if (valid && cq == 0) emit_parts(ep, t, m0, M, TN, a0, a2);
    };
    auto request = [&](EpiIn (&in)[AHEAD_ROWS], int it) {
#pragma unroll
        for (int i = 0; i < AHEAD_ROWS; ++i) {
            const int t = t0 + (it + i) * RPI + tid / CPR;
            in[i] = epi_in(ep, t, col, t < T && col_ok, false);
        }
    };

    if constexpr (KG == 2) {
        // the partial tiles of both groups meet in LDS and are added in group order
        static_assert(TM == Cfg::FROWS && TM * SW * 8 <= (int)Cfg::BODY && ITS == AHEAD_ROWS, "two groups");
        __syncthreads();   // every wave has read its last fragments
#pragma unroll
        for (int a = 0; a < MI; ++a)
#pragma unroll
            for (int b = 0; b < NI; ++b)
                *(f32x4 *)(stg + (grp * TM + wr * 16 * MI + a * 16 + row) * SW + wc * 16 * NI + b * 16 + 4 * q) = acc[a][b];
        auto sum4 = [&](int r, int c) { return *(const f32x4 *)(stg + r * SW + c) + *(const f32x4 *)(stg + (TM + r) * SW + c); };
        if constexpr (SPLIT) {
            __syncthreads();
            float *slab = part + (size_t)split * T * M;
#pragma unroll
            for (int it = 0; it < ITS; ++it) {
                const int r = it * RPI + tid / CPR, t = t0 + r;
                if (t < T && col_ok) *(f32x4 *)(slab + (size_t)t * M + col) = sum4(r, cq * 8);           // M % 4 == 0
                if (t < T && col_ok && col + 4 < M) *(f32x4 *)(slab + (size_t)t * M + col + 4) = sum4(r, cq * 8 + 4);
            }
        } else if (by_four(M, ldy, Y, ep)) {
            __syncthreads();
#pragma unroll 1
            for (int it = 0; it < ITS; ++it) {
                const int r = it * RPI + tid / CPR, t = t0 + r;
                if (t >= T) break;
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const int c = g * (TN / 2) + cq * 4;
                    if (!in_tile || m0 + c >= M) continue;
                    f32x4 v = sum4(r, c);
                    if constexpr (W_U8) affine4(v, m0 + c, M, lsum[r], lsum[TM + r], ep);
                    finish_row4(v, t, m0 + c, M, ep, Y, ldy);
                }
            }
        } else {
            const Emit8 em = emit8(ep, col, col_ok);
            EpiIn in[AHEAD_ROWS];
            request(in, 0);
            __syncthreads();
#pragma unroll 1
            for (int it = 0; it < ITS; ++it) {
                const EpiIn cur = in[0];
#pragma unroll
                for (int i = 0; i + 1 < AHEAD_ROWS; ++i) in[i] = in[i + 1];   // a loop that is not unrolled has no other index
                const int r = it * RPI + tid / CPR, t = t0 + r;
                const bool valid = t < T && col_ok;
                float a0 = 0.f, a2 = 0.f;
                if (valid) {
                    const f32x4 lo = sum4(r, cq * 8), hi = sum4(r, cq * 8 + 4);
                    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    if constexpr (W_U8) affine8(v, *(const h16x8 *)(lcol + cq * 8), *(const h16x8 *)(lcol + TN + cq * 8), lsum[r], lsum[TM + r]);
                    finish_row8<true>(v, cur, t, col, ep, Y, ldy, em, a0, a2);
                }
                if (ep.emit_ry) emit_row(t, valid, a0, a2);
            }
        }
        return;
    }
    const int roff = wr * 16 * MI;   // this wave's first row
    if constexpr (SPLIT) {
        // partial sums go to this split's fp32 slab; splitk_epilogue8_kernel adds the slabs and finishes
        float *slab = part + (size_t)split * T * M;
#pragma unroll
        for (int a = 0; a < MI; ++a) {
            const int t = t0 + roff + a * 16 + row;
#pragma unroll
            for (int b = 0; b < NI; ++b) {
                const int m = m0 + wc * 16 * NI + b * 16 + 4 * q;
                if (m < M && t < T) *(f32x4 *)(slab + (size_t)t * M + m) = acc[a][b];   // M % 4 == 0
            }
        }
    } else {
        __syncthreads();   // every wave has read its last fragments
        if (by_four(M, ldy, Y, ep)) {
            // fp32 outputs, and rows that start on no 16-byte boundary, leave four at a time: the accumulators pass through LDS (free
            // now), at most 128 tile rows at a time.  A 50277-wide head is such a product.
            constexpr int FROWS = Cfg::FROWS;
#pragma unroll 1
            for (int h = 0; h < TM / FROWS; ++h) {
                if (TM == FROWS || wr == h) {
#pragma unroll
                    for (int a = 0; a < MI; ++a)
#pragma unroll
                        for (int b = 0; b < NI; ++b)
                            *(f32x4 *)(stg + (roff - h * FROWS + a * 16 + row) * SW + wc * 16 * NI + b * 16 + 4 * q) = acc[a][b];
                }
                __syncthreads();
#pragma unroll 1
                for (int it = 0; it < FROWS / RPI; ++it) {
                    const int r = h * FROWS + it * RPI + tid / CPR, t = t0 + r;
                    if (t >= T) break;
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        const int c = g * (TN / 2) + cq * 4;
                        if (!in_tile || m0 + c >= M) continue;
                        f32x4 v = *(const f32x4 *)(stg + (r - h * FROWS) * SW + c);
                        if constexpr (W_U8) affine4(v, m0 + c, M, lsum[r], lsum[TM + r], ep);
                        finish_row4(v, t, m0 + c, M, ep, Y, ldy);
                    }
                }
                __syncthreads();
            }
            return;
        }
        // fp16 outputs: corrected and rounded where they are, which the other steps begin with anyway, so the whole tile fits LDS as
        // fp16; then each thread finishes eight consecutive outputs of a row, with 16-byte loads of the residual / gate rows and
        // 16-byte stores.  The activations stay in that loop, whose body is small enough for the instruction cache (written out for
        // 128 accumulators they were not: 28 us of a launch of 160).
        constexpr int HW = Cfg::HSTRIDE;                   // row stride in halves: 16 rows x 8 bytes fall on different banks
        h16 *const hstg = (h16 *)smem;
        h16x4 rx4[NI], mx4[NI];
        if constexpr (W_U8) {
#pragma unroll
            for (int b = 0; b < NI; ++b) {
                const int c = wc * 16 * NI + b * 16 + 4 * q;
                rx4[b] = *(const h16x4 *)(lcol + c);
                mx4[b] = *(const h16x4 *)(lcol + TN + c);
            }
        }
#pragma unroll
        for (int a = 0; a < MI; ++a) {
            const int r = roff + a * 16 + row;
            const float s0 = W_U8 ? lsum[r] : 0.f, s2 = W_U8 ? lsum[TM + r] : 0.f;
#pragma unroll
            for (int b = 0; b < NI; ++b) {
                h16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] = (h16)(W_U8 ? epi_affine(acc[a][b][e], (float)rx4[b][e], (float)mx4[b][e], s0, s2) : acc[a][b][e]);
                *(h16x4 *)(hstg + r * HW + wc * 16 * NI + b * 16 + 4 * q) = o;
            }
        }
        const Emit8 em = emit8(ep, col, col_ok);
#pragma unroll 1
        for (int it = 0; it < ITS; it += AHEAD_ROWS) {
            EpiIn in[AHEAD_ROWS];
            request(in, it);
            if (it == 0) __syncthreads();                  // the outputs are in LDS
            if (t0 + it * RPI >= T) break;
#pragma unroll
            for (int i = 0; i < AHEAD_ROWS; ++i) {
                const int r = (it + i) * RPI + tid / CPR, t = t0 + r;
                const bool valid = t < T && col_ok;
                float a0 = 0.f, a2 = 0.f;
                if (valid) {
                    const h16x8 y = *(const h16x8 *)(hstg + r * HW + cq * 8);
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = (float)y[e];
                    finish_row8<true>(v, in[i], t, col, ep, Y, ldy, em, a0, a2);
                }
                if (ep.emit_ry) emit_row(t, valid, a0, a2);
            }
        }
    }
}

// One to four contractions [T, N] x [N, M_i] in one launch: short calls, where each of them alone would split K and need
// a reduction pass.  Register-staged tiles: blockIdx.y picks the member, the grid is as wide as the widest one.
// Direct-to-LDS tiles: the units run over the tiles of all members, first[i] being member i's first, and the K splits.  (With a grid
// for the widest member the tiles of the narrow ones all fell on the first XCDs: four first LoRA stages of 128, 128,
// 128 and 512 outputs took two rounds on two XCDs with the others idle, 41 us instead of 23 with the 64 x 64 tile.)
struct GemmMember {
    const h16 *A;     // what the first loads need, 32 bytes
    const void *W;
    int64_t ldw;
    int M, walk_m;    // walk_m: consecutive tiles walk along M first (direct-to-LDS launches)
    void *Y;
    int64_t ldy;
    float *part;      // split-K slabs, [splits][T][M] (direct-to-LDS launches only)
    GemmEpi ep;
};
struct GemmMembers { GemmMember m[4]; };
struct GemmGroup : GemmMembers {
    int64_t lda;
    int first[4];     // members that are not there: INT_MAX
    int nk_split;
};

// register-staged 128 x 128 tiles: uint8 matrices whose mx or rx lie on no 16-byte boundary
__global__ __launch_bounds__(256) void gemm_group_kernel(int T, int N, GemmGroup g) {
    const int gi = blockIdx.y, M = g.m[gi].M;
    gemm_body<true, 128, 128, 2, 2, 4, false>(T, N, M, g.m[gi].A, g.lda, g.m[gi].W, g.m[gi].ldw, g.m[gi].Y, M, g.m[gi].ep, N / BK, nullptr);
}

// The member that a tile belongs to, and its tile of it.  first1 .. first3 are kernel arguments of their own ahead of the members:
// such ones are in scalar registers when a wave starts.  What the first loads need of a member is read at once: left alone, the compiler
// reads M, waits, and then reads the pointers.
DEV int group_member(int first1, int first2, int first3, int &tile) {
    const int gi = (tile >= first1) + (tile >= first2) + (tile >= first3);
    tile -= tile >= first3 ? first3 : tile >= first2 ? first2 : tile >= first1 ? first1 : 0;
    return gi;
}
struct GemmIn { const h16 *A; const void *W; int64_t ldw; int M, walk_m; };
DEV GemmIn gemm_in(const GemmMember &m) {
    GemmIn in = {m.A, m.W, m.ldw, m.M, m.walk_m};
    asm volatile("" ::"s"(in.A), "s"(in.W), "s"(in.ldw), "s"(in.M), "s"(in.walk_m));
    return in;
}
// fills `first` and the walks for tiles of tm x tn; returns the tiles of the launch
int64_t group_tiles(bool w_u8, GemmGroup &g, int n, int64_t T, int64_t N, int tm, int tn) {
    int64_t tiles = 0;
    for (int i = 0; i < n; ++i) g.m[i].walk_m = walks_m(w_u8, T, N, g.m[i].M);
    for (int i = 0; i < 4; ++i) {
        g.first[i] = i < n ? (int)tiles : 0x7fffffff;
        if (i < n) tiles += ((T + tm - 1) / tm) * ((g.m[i].M + tn - 1) / tn);
    }
    return tiles;
}

// the direct-to-LDS kernel
template <bool W_U8, bool SPLIT, int TM, int TN, int NSTG>
__global__ __launch_bounds__(512) void gemm_dma_kernel(int T, int N, int units, int splits, int first1, int first2, int first3, int nk_split,
                                                           int64_t lda, GemmMembers g) {
    const int unit = xcd_unit(units);
    int tile = SPLIT ? unit / splits : unit;
    const int split = SPLIT ? unit - tile * splits : 0;
    const GemmMember &m = g.m[group_member(first1, first2, first3, tile)];
    const GemmIn in = gemm_in(m);
    gemm_dma_body<W_U8, SPLIT, TM, TN, NSTG>(tile, T, N, in.M, in.walk_m, in.A, lda, in.W, in.ldw, m.Y, m.ldy, m.ep, nk_split, m.part,
                                                 split);
}

template <bool W_U8, int TM, int TN, int NSTG>
int launch_dma(GemmGroup &g, int n, int64_t T, int64_t N, int ks, hipStream_t st) {
    using Cfg = DmaCfg<W_U8, TM, TN, NSTG>;
    constexpr size_t lds = Cfg::LDS;
    if (ks > 1 && !Cfg::SPLITS) return RWKV_E_DTYPE;
    static PerDeviceOnce once;
    bool *attr_done = once.slot();
    if (!attr_done || !*attr_done) {
        hipError_t e = hipFuncSetAttribute((const void *)gemm_dma_kernel<W_U8, false, TM, TN, NSTG>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if constexpr (Cfg::SPLITS) {
            if (e == hipSuccess)
                e = hipFuncSetAttribute((const void *)gemm_dma_kernel<W_U8, true, TM, TN, NSTG>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)lds);
        }
        if (e != hipSuccess) return (int)e;
        if (attr_done) *attr_done = true;
    }
    const int units = (int)group_tiles(W_U8, g, n, T, N, TM, TN) * ks;
    const auto kernel = Cfg::SPLITS && ks > 1 ? gemm_dma_kernel<W_U8, Cfg::SPLITS, TM, TN, NSTG> : gemm_dma_kernel<W_U8, false, TM, TN, NSTG>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)units), dim3(64 * Cfg::NW), lds, st, (int)T, (int)N, units, ks, g.first[1], g.first[2], g.first[3], g.nk_split, g.lda,
                       (const GemmMembers &)g);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// ---- K over wave groups: products whose large tiles would leave the chip idle ---------------------------------
// [T, 768..4096] x [.., 768..4096] products of a few hundred rows have 12 to 100 tiles of 128 x 128: most CUs idle, or a
// K split whose fp32 slabs need a second launch; and calls of up to 128 rows are bound by how fast the weights arrive.
// Here the tile is 64 x 64 or 64 x 128 and a workgroup's eight waves are KG = 8 or 4 groups that share K: every wave
// computes a 64 x 64 block (the fewest fragment bytes per MFMA that eight waves allow) over its part of each stage, and the
// partial blocks are added in group order through LDS (deterministic).  A stage holds 128 or 256 k's, so that a uint8 weight
// row is one or two whole 128-byte lines: with 64 k's per stage half a line per request, at the same cost per request.
// Lane half h of a group takes 8 consecutive k's per MFMA step from KW / 2 h on, for both operands, so uint8 fragments are
// 16-byte reads of two steps' worth; a stage's first fragments are read while the stage before multiplies.
// What bounds it, loops taken apart: from about 190 workgroups on the weights (uint8 [45 x 4096] x [4096 x 12288] 4.1 TB/s in
// the loop, fp16 4.8), otherwise the requests that a CU has in flight (0.14 - 0.2 us per 64 k's of a 64 x 64 tile); + 5 - 7 us
// of launch, first stages and epilogue.  Rows past T are not worth skipping (buffer loads with bounds: 2 - 4 % slower).
// Measured, weights from HBM, us, against the same with K over four waves that each had stages of their own, and the
// 128 x 128 tiles: uint8 [256 x 4096] x [4096 x 4096] 17.3 -> 16.6, [45 x 4096] x [4096 x 12288] 20.3 (two K splits of 64 x 128
// tiles 19.4) -> 17.7, [128 x 4096] x [4096 x 12288] 31.8 (two splits 24.4) -> 25.3, [100 x 16384] x [16384 x 2048] 32.3 -> 20.6;
// fp16 [513 x 768] x [768 x 768] 7.8 -> 7.2, [333 x 2048] x [2048 x 2048] 10.4 -> 10.1, [128 x 4096] x [4096 x 768] 12.8 -> 10.5.
// 128 x 128 (KG = 2) and 128 x 256 (1) tiles of this form: 42.0 and 55.8 against 38.8 us on [1024 x 4096] x [4096 x 4096],
// not built.
template <bool W_U8, int TM, int TN> struct KgCfg {
    static constexpr int RA = TM / 64, RB = TN / 64, KG = 8 / (RA * RB);   // 64 x 64 blocks of the tile; groups that share K
    static constexpr int BKS = W_U8 && KG == 8 ? 256 : 128;                // k's of a stage
    static constexpr int KW = BKS / KG, US = KW / 16;                                  // k's and MFMA steps of a wave and stage
    static constexpr int ABYTES = BKS * 2, WBYTES = W_U8 ? BKS : BKS * 2;              // bytes of a row
    static constexpr int A = TM * ABYTES, W = TN * WBYTES, STAGE = A + W;
    static constexpr int AL = A / 8192, WL = W / 8192, LOADS = AL + WL;                // 1 KB loads per wave and stage
    static constexpr int SW = 68, REGION = 64 * SW * 4;                                // partial tile of a wave: row stride (floats), bytes
    static constexpr int NST = (160 * 1024 - 2 * TM * 4) / STAGE < 4 ? (160 * 1024 - 2 * TM * 4) / STAGE : 4;
    static constexpr size_t BODY = NST * STAGE > 8 * REGION ? NST * STAGE : 8 * REGION, LDS = BODY + (W_U8 ? 2 * TM * 4 : 0);
    static_assert((KG == 8 || KG == 4) && (US == 1 || US == 2) && NST >= 2 && LDS <= 160 * 1024 && (NST - 1) * LOADS < 64, "tile");
};
// slot of a 16-byte chunk in a row of RBYTES: conflict-free for 16 rows x one chunk (64 banks of 4 bytes)
template <int RBYTES> DEV int kg_key(int row) {
    constexpr int RPB = RBYTES < 256 ? 256 / RBYTES : 1, CH = RBYTES / 16 < 16 ? RBYTES / 16 : 16;
    return (row / RPB) & (CH - 1);
}
template <bool W_U8, bool SPLIT, int TM, int TN>
DEV void gemm_kg_body(int bid, int T, int N, int M, int walk_m, const h16 *__restrict__ A, int64_t lda, const void *__restrict__ Wv, int64_t ldw,
                      void *__restrict__ Y, int64_t ldy, const GemmEpi &ep, int nk_split, float *__restrict__ part, int split) {
    using Cfg = KgCfg<W_U8, TM, TN>;
    constexpr int NST = Cfg::NST, STAGE = Cfg::STAGE, AL = Cfg::AL, WL = Cfg::WL, BKS = Cfg::BKS, KW = Cfg::KW, US = Cfg::US;
    constexpr int AB = Cfg::ABYTES, WB = Cfg::WBYTES, RA = Cfg::RA, RB = Cfg::RB, SW = Cfg::SW;
    extern __shared__ __align__(1024) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = wave % (RA * RB), grp = wave / (RA * RB), wr = blk / RB, wc = blk % RB;
    const TileAt at = tile_at<TM, TN>(bid, T, M, walk_m);
    const int t0 = at.t0, m0 = at.m0;
    const int kbase = SPLIT ? split * nk_split * BK : 0, K = nk_split * BK;   // this workgroup's k's (a multiple of 64)
    const int nk = (K + BKS - 1) / BKS;

    // load sources; rows past the end re-read the last row (never stored).  Load i of a wave fills 1 KB: the rows
    // (wave AL + i) 1024 / AB and up; the lane that fills slot p of row r fetches chunk p ^ key(r).
    constexpr int ALR = AB / 16, WLR = WB / 16;   // lanes per row
    auto a_row = [&](int i) { return (wave * AL + i) * (64 / ALR) + lane / ALR; };
    auto w_row = [&](int i) { return (wave * WL + i) * (64 / WLR) + lane / WLR; };
    auto a_k = [&](int i) { return ((lane % ALR) ^ kg_key<AB>(a_row(i))) * 8; };
    auto w_k = [&](int i) { return ((lane % WLR) ^ kg_key<WB>(w_row(i))) * (W_U8 ? 16 : 8); };
    const unsigned char *ga[AL], *gw[WL];
#pragma unroll
    for (int i = 0; i < AL; ++i) ga[i] = (const unsigned char *)(A + (size_t)min(t0 + a_row(i), T - 1) * lda + kbase + a_k(i));
#pragma unroll
    for (int i = 0; i < WL; ++i)
        gw[i] = (const unsigned char *)Wv + ((size_t)min(m0 + w_row(i), M - 1) * ldw + kbase + w_k(i)) * (W_U8 ? 1 : 2);
    typedef __attribute__((address_space(1))) const void *gptr;
    typedef __attribute__((address_space(3))) void *lptr;
    auto issue = [&](int kt, int so) {   // a whole stage
        unsigned char *base = smem + so;
#pragma unroll
        for (int i = 0; i < AL; ++i) __builtin_amdgcn_global_load_lds((gptr)(ga[i] + kt * AB), (lptr)(base + (wave * AL + i) * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < WL; ++i) __builtin_amdgcn_global_load_lds((gptr)(gw[i] + kt * WB), (lptr)(base + Cfg::A + (wave * WL + i) * 1024), 16, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto issue_any = [&](int kt, int so) {
        if (kt * BKS + BKS <= K) { issue(kt, so); return; }
        // the last stage of a K that is no multiple of BKS: chunks past the end fetch k 0 .. 63 (never multiplied)
        unsigned char *base = smem + so;
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int k = a_k(i), d = kt * BKS + k < K ? kt * BKS : (k & 63) - k;
            __builtin_amdgcn_global_load_lds((gptr)(ga[i] + d * 2), (lptr)(base + (wave * AL + i) * 1024), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int k = w_k(i), d = kt * BKS + k < K ? kt * BKS : (k & 63) - k;
            __builtin_amdgcn_global_load_lds((gptr)(gw[i] + d * (W_U8 ? 1 : 2)), (lptr)(base + Cfg::A + (wave * WL + i) * 1024), 16, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x16 acc[2][2];   // [weight block][token block]
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[b][a][e] = 0.f;

    // fragments: lane (row, h) of group g takes k g KW + h KW / 2 + 8 s .. + 7 of the stage in step s, for both operands
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const int row = lane & 31, h = lane >> 5, k0 = grp * KW + h * (KW / 2);
    constexpr int WN = W_U8 ? 1 : US;   // weight reads per stage and block
    uint32_t vA[US], vW[WN];
#pragma unroll
    for (int j = 0; j < US; ++j) vA[j] = lds0 + (wr * 64 + row) * AB + (((k0 / 8 + j) ^ kg_key<AB>(row)) << 4);
#pragma unroll
    for (int j = 0; j < WN; ++j) vW[j] = lds0 + Cfg::A + (wc * 64 + row) * WB + (((W_U8 ? k0 / 16 : k0 / 8 + j) ^ kg_key<WB>(row)) << 4);
    h16x8 fa[2][US][2];    // [set][step][token block]
    u32x4 fw[2][WN][2];    // [set][read][weight block]
    auto ldstage = [&](int set, int so) {
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const uint32_t p = vW[j] + so;
            asm volatile("ds_read_b128 %0, %1" : "=v"(fw[set][j][0]) : "v"(p));
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fw[set][j][1]) : "v"(p), "n"(32 * WB));
        }
#pragma unroll
        for (int j = 0; j < US; ++j) {
            const uint32_t p = vA[j] + so;
            asm volatile("ds_read_b128 %0, %1" : "=v"(fa[set][j][0]) : "v"(p));
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][j][1]) : "v"(p), "n"(32 * AB));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const h16x2 off = {(h16)1023.5f, (h16)1023.5f};
    auto mul = [&](int set, int j) {
        h16x8 wf[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if constexpr (W_U8) {
                const uint32_t b0 = j ? fw[set][0][b].z : fw[set][0][b].x, b1 = j ? fw[set][0][b].w : fw[set][0][b].y;
                const h16x2 q0 = u8pair_lo_1024(b0) - off, q1 = u8pair_hi_1024(b0) - off;
                const h16x2 q2 = u8pair_lo_1024(b1) - off, q3 = u8pair_hi_1024(b1) - off;
                wf[b] = h16x8{q0.x, q0.y, q1.x, q1.y, q2.x, q2.y, q3.x, q3.y};
            } else {
                wf[b] = __builtin_bit_cast(h16x8, fw[set][j][b]);
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[b][a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[b], fa[set][j][a], acc[b][a], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto reads_done = [&]() {
        __builtin_amdgcn_s_waitcnt(lgkm_only(0));
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < NST; ++s)
        if (s < nk) issue_any(s, s * STAGE);
    bool lds_sums = false;
    float *lsum = (float *)(smem + Cfg::BODY);
    if constexpr (W_U8) {
        if (ep.parts > 1 && (!SPLIT || (m0 == 0 && split == 0))) {
            lds_sums = !SPLIT;
            if (tid < 2 * TM) {
                const int r = tid & (TM - 1), which = tid / TM, t = min(t0 + r, T - 1);
                const float *p = (which ? ep.p2 : ep.p0) + (size_t)t * ep.parts;
                float tot = 0.f;
                for (int j = 0; j < ep.parts; j += 64) {
                    f32x4 v[16];
#pragma unroll
                    for (int q = 0; q < 16; ++q) v[q] = j + 4 * q < ep.parts ? *(const f32x4 *)(p + j + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int q = 0; q < 16; ++q) tot = (((tot + v[q][0]) + v[q][1]) + v[q][2]) + v[q][3];
                }
                if constexpr (SPLIT) {
                    if (t0 + r < T) (which ? (float *)ep.s2 : (float *)ep.s0)[t] = tot;
                } else {
                    lsum[tid] = tot;
                }
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (nk >= NST) __builtin_amdgcn_s_waitcnt(vm_lgkm0((NST - 1) * Cfg::LOADS));   // my part of stage 0 has landed
    else __builtin_amdgcn_s_waitcnt(vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    int so = 0;
    ldstage(0, 0);
    reads_done();
    // One stage.  Past its barrier stage kt + 1 has landed for every wave and nobody reads stage kt any more, so stage kt + NST
    // goes where it was.  STEADY: that one is there and whole; the last stages take the form with the branches (four of them
    // per stage left the matrix cores idle for 170 clocks, as both waves of a SIMD stand at the same barrier).  With two
    // steps per stage the first one's products go ahead of the loads and reads, which then issue while the matrix cores work.
    auto stage = [&](auto steady, int kt, int set) {
        constexpr bool STEADY = decltype(steady)::value;
        const bool mine = STEADY || kt * BKS + grp * KW < K;   // the wave's k's of the last stage may be past the end
        const int sn = so + STAGE >= NST * STAGE ? 0 : so + STAGE;
        if (STEADY || kt + NST <= nk) __builtin_amdgcn_s_waitcnt(vm_only((NST - 2) * Cfg::LOADS));
        else __builtin_amdgcn_s_waitcnt(vm_only(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (US == 1) ldstage(set ^ 1, sn);
        if (mine) mul(set, 0);
        if constexpr (STEADY) issue(kt + NST, so);
        else if (kt + NST < nk) issue_any(kt + NST, so);
        if (US > 1) {
            ldstage(set ^ 1, sn);
            if (mine) mul(set, US - 1);
        }
        reads_done();
        so = sn;
    };
    int kt = 0;
    const int steady = max(K / BKS - NST, 0) & ~1;   // stage kt + NST is whole for kt < K / BKS - NST
    for (; kt < steady; kt += 2) {
        stage(std::true_type{}, kt, 0);
        stage(std::true_type{}, kt + 1, 1);
    }
    for (; kt < nk; kt += 2) {   // an odd number of stages ends with one in which nobody multiplies
        stage(std::false_type{}, kt, 0);
        stage(std::false_type{}, kt + 1, 1);
    }
    // nothing may land in LDS or in a fragment register after this point (see gemm_dma_body)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int set = 0; set < 2; ++set) {
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b) asm volatile("" ::"v"(fw[set][j][b]));
#pragma unroll
        for (int j = 0; j < US; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) asm volatile("" ::"v"(fa[set][j][a]));
    }
    __builtin_amdgcn_sched_barrier(0);
    float *mypart = (float *)(smem + wave * Cfg::REGION);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(f32x4 *)(mypart + (a * 32 + row) * SW + b * 32 + 8 * q + 4 * h) =
                    f32x4{acc[b][a][4 * q], acc[b][a][4 * q + 1], acc[b][a][4 * q + 2], acc[b][a][4 * q + 3]};
    // eight consecutive outputs of a row per thread and pass: the partial tiles of the groups are added in group order
    constexpr int CPR = TN / 8, RPI = 512 / CPR, ITS = TM / RPI, AHEAD_ROWS = ITS < 4 ? ITS : 4;
    auto tile_sum = [&](int r, int c, f32x4 &lo) {   // four values at tile row r, column c
        const float *p = (const float *)(smem + ((r >> 6) * RB + (c >> 6)) * Cfg::REGION) + (r & 63) * SW + (c & 63);
        lo = *(const f32x4 *)p;
#pragma unroll
        for (int k = 1; k < Cfg::KG; ++k) lo += *(const f32x4 *)(p + k * (RA * RB * Cfg::REGION / 4));
    };
    const int cq = tid % CPR, col = m0 + cq * 8;
    const bool col_ok = col < M;
    if constexpr (SPLIT) {
        __syncthreads();
        float *slab = part + (size_t)split * T * M;
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
            const int r = it * RPI + tid / CPR, t = t0 + r;
            f32x4 lo, hi;
            tile_sum(r, cq * 8, lo);
            tile_sum(r, cq * 8 + 4, hi);
            if (t < T && col < M) *(f32x4 *)(slab + (size_t)t * M + col) = lo;           // M % 4 == 0
            if (t < T && col + 4 < M) *(f32x4 *)(slab + (size_t)t * M + col + 4) = hi;
        }
    } else {
        if (by_four(M, ldy, Y, ep)) {   // a loop of its own, as in gemm_dma_body
            __syncthreads();
#pragma unroll 1
            for (int it = 0; it < ITS; ++it) {
                const int r = it * RPI + tid / CPR, t = t0 + r;
                if (t >= T) break;
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const int c = g * (TN / 2) + cq * 4;
                    if (m0 + c >= M) continue;
                    f32x4 v;
                    tile_sum(r, c, v);
                    if constexpr (W_U8) affine4(v, m0 + c, M, lds_sums ? lsum[r] : ep.s0[t], lds_sums ? lsum[TM + r] : ep.s2[t], ep);
                    finish_row4(v, t, m0 + c, M, ep, Y, ldy);
                }
            }
            return;
        }
        const bool emit = ep.emit_ry != nullptr;
        h16x8 rx8 = {}, mx8 = {};
        EpiIn in[AHEAD_ROWS] = {};
        if (W_U8 && col_ok) { rx8 = load_n<h16x8, 8>(ep.rx + col, M - col); mx8 = load_n<h16x8, 8>(ep.mx + col, M - col); }
        const Emit8 em = emit8(ep, col, col_ok);
#pragma unroll 1
        for (int it = 0; it < ITS; ++it) {
            const int r = it * RPI + tid / CPR, t = t0 + r;
            if (it % AHEAD_ROWS == 0) {
#pragma unroll
                for (int i = 0; i < AHEAD_ROWS; ++i) in[i] = epi_in(ep, t + i * RPI, col, t + i * RPI < T && col_ok, W_U8 && !lds_sums);
                if (it == 0) __syncthreads();   // the partial tiles are in LDS
            }
            const EpiIn cur = in[0];
#pragma unroll
            for (int i = 0; i + 1 < AHEAD_ROWS; ++i) in[i] = in[i + 1];
            const bool valid = t < T && col_ok;
            float a0 = 0.f, a2 = 0.f;
            if (valid) {
                f32x4 lo, hi;
                tile_sum(r, cq * 8, lo);
                tile_sum(r, cq * 8 + 4, hi);
                float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                if constexpr (W_U8) affine8(v, rx8, mx8, lds_sums ? lsum[r] : cur.s0, lds_sums ? lsum[TM + r] : cur.s2);
                finish_row8<true>(v, cur, t, col, ep, Y, ldy, em, a0, a2);
            }
            if (emit) {   // the CPR threads of a row are neighbours in one wave; every lane takes part
#pragma unroll
                for (int o = 1; o < CPR; o <<= 1) { a0 += __shfl_xor(a0, o, WAVE); a2 += __shfl_xor(a2, o, WAVE); }
                if (valid && cq == 0) emit_parts(ep, t, m0, M, TN, a0, a2);
            }
        }
    }
}

template <bool W_U8, bool SPLIT, int TM, int TN>
__global__ __launch_bounds__(512) void gemm_kg_kernel(int T, int N, int units, int splits, int first1, int first2, int first3, int nk_split, int64_t lda,
                                                      GemmMembers g) {
    const int unit = xcd_unit(units);
    int tile = SPLIT ? unit / splits : unit;
    const int split = SPLIT ? unit - tile * splits : 0;
    const GemmMember &m = g.m[group_member(first1, first2, first3, tile)];
    const GemmIn in = gemm_in(m);
    gemm_kg_body<W_U8, SPLIT, TM, TN>(tile, T, N, in.M, in.walk_m, in.A, lda, in.W, in.ldw, m.Y, m.ldy, m.ep, nk_split, m.part,
                                      split);
}

template <bool W_U8, int TM, int TN>
int launch_kg(GemmGroup &g, int n, int64_t T, int64_t N, int ks, hipStream_t st) {
    constexpr size_t lds = KgCfg<W_U8, TM, TN>::LDS;
    static PerDeviceOnce once;
    bool *attr_done = once.slot();
    if (!attr_done || !*attr_done) {
        hipError_t e = hipFuncSetAttribute((const void *)gemm_kg_kernel<W_U8, false, TM, TN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e == hipSuccess) e = hipFuncSetAttribute((const void *)gemm_kg_kernel<W_U8, true, TM, TN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        if (attr_done) *attr_done = true;
    }
    const int units = (int)group_tiles(W_U8, g, n, T, N, TM, TN) * ks;
    const auto kernel = ks > 1 ? gemm_kg_kernel<W_U8, true, TM, TN> : gemm_kg_kernel<W_U8, false, TM, TN>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)units), dim3(512), lds, st, (int)T, (int)N, units, ks, g.first[1], g.first[2], g.first[3], g.nk_split, g.lda,
                       (const GemmMembers &)g);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// ---- few rows: tiles of 32, 48 or 64 rows and 16 to 96 columns ----------------------------------------------------
// For calls of up to 128 rows (tiles of 16 and 32 columns) and 256.  Those of 17 to 64 rows are bound by how fast a CU takes its operands, 50 GB/s with a tile's activations at twice the bytes of its
// uint8 weights, so what counts is that every CU has the same share and no rows past the end: 12288 outputs are 192 tiles of 64 x 64
// and 256 of 48 x 48.  The form is that of gemm_kg_kernel (the waves share K, partial blocks meet in LDS and are added in group order)
// with v_mfma_f32_16x16x32_f16, whose blocks make sides of any multiple of 16: KG = 8 groups of one wave, or four of two waves side by
// side, and 32 k's a wave and stage, so that a stage is one MFMA step.  A stage's 1 KB loads are dealt to the waves, activations
// and weights alike; the last ones repeat where they do not divide.
template <bool W_U8, int TM, int TN> struct FewCfg {
    static constexpr int RB = TN == 16 || TN == 48 ? 1 : 2, KG = 8 / RB, BKS = 32 * KG;   // waves side by side, groups that share K, k's of a stage
    static constexpr int AB = BKS * 2, WB = BKS * (W_U8 ? 1 : 2);                         // bytes of a row
    static constexpr int A = TM * AB, STAGE = A + TN * WB, AP = A / 1024, PIECES = STAGE / 1024, LOADS = (PIECES + 7) / 8;
    static constexpr int NST = (160 * 1024 - 2 * TM * 4) / STAGE < 4 ? (160 * 1024 - 2 * TM * 4) / STAGE : 4;
    static constexpr int MI = TM / 16, NI = TN / (16 * RB);                               // 16 x 16 blocks of a wave
    static constexpr int SW = TN / RB + 4, REGION = TM * SW * 4;                          // partial tile of a wave: row stride (floats), bytes
    static constexpr int BODY = NST * STAGE > 8 * REGION ? NST * STAGE : 8 * REGION, LDS = BODY + (W_U8 ? 2 * TM * 4 : 0);
    static constexpr int CPR = TN <= 16 ? 2 : TN <= 32 ? 4 : TN <= 64 ? 8 : 16;           // threads that finish a row, eight outputs each
    static_assert(TM % 16 == 0 && TN % (16 * RB) == 0 && A % 1024 == 0 && STAGE % 1024 == 0 && NST >= 2 && LDS <= 160 * 1024, "tile");
};
template <bool W_U8, int TM, int TN>
__global__ __launch_bounds__(512) void gemm_few_kernel(int T, int units, int splits, int first1, int first2, int first3, int nk_split, int64_t lda,
                                                       GemmMembers g) {
    using Cfg = FewCfg<W_U8, TM, TN>;
    constexpr int NST = Cfg::NST, STAGE = Cfg::STAGE, LOADS = Cfg::LOADS, BKS = Cfg::BKS, AB = Cfg::AB, WB = Cfg::WB, MI = Cfg::MI, NI = Cfg::NI;
    constexpr int KG = Cfg::KG, RB = Cfg::RB, SW = Cfg::SW, REGION = Cfg::REGION, CPR = Cfg::CPR;
    extern __shared__ __align__(1024) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave / RB, wc = wave % RB;
    const int unit = xcd_unit(units);
    int tile = splits > 1 ? unit / splits : unit;
    const int split = splits > 1 ? unit - tile * splits : 0;
    const GemmMember &mb = g.m[group_member(first1, first2, first3, tile)];
    const GemmIn in = gemm_in(mb);
    const int M = in.M;
    const TileAt at = tile_at<TM, TN>(tile, T, M, in.walk_m);
    const int t0 = at.t0, m0 = at.m0;
    const int kbase = split * nk_split * BK, K = nk_split * BK, nk = (K + BKS - 1) / BKS;

    // load i of this wave: 1 KB of a stage, whole rows; rows past the end re-read the last row (never stored).  The lane that fills
    // slot p of row r fetches chunk p ^ key(r).
    const unsigned char *src[LOADS];
    int klane[LOADS], kb[LOADS];   // this lane's first k of a stage; bytes per k
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int p = min(wave + 8 * i, Cfg::PIECES - 1);
        if (p < Cfg::AP) {
            const int r = p * (1024 / AB) + lane / (AB / 16), c = (lane % (AB / 16)) ^ kg_key<AB>(r);
            klane[i] = c * 8;
            kb[i] = 2;
            src[i] = (const unsigned char *)(in.A + (size_t)min(t0 + r, T - 1) * lda + kbase + klane[i]);
        } else {
            const int r = (p - Cfg::AP) * (1024 / WB) + lane / (WB / 16), c = (lane % (WB / 16)) ^ kg_key<WB>(r);
            klane[i] = c * (W_U8 ? 16 : 8);
            kb[i] = W_U8 ? 1 : 2;
            src[i] = (const unsigned char *)in.W + ((size_t)min(m0 + r, M - 1) * in.ldw + kbase + klane[i]) * (W_U8 ? 1 : 2);
        }
    }
    typedef __attribute__((address_space(1))) const void *gptr;
    typedef __attribute__((address_space(3))) void *lptr;
    auto issue = [&](int kt, int so) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            __builtin_amdgcn_global_load_lds((gptr)(src[i] + kt * BKS * kb[i]), (lptr)(smem + so + min(wave + 8 * i, Cfg::PIECES - 1) * 1024), 16, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto issue_any = [&](int kt, int so) {
        if (kt * BKS + BKS <= K) { issue(kt, so); return; }
        // the last stage of a K that is no multiple of BKS: chunks past the end fetch k's 0 .. 63 (never multiplied)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int d = kt * BKS + klane[i] < K ? kt * BKS : (klane[i] & 63) - klane[i];
            __builtin_amdgcn_global_load_lds((gptr)(src[i] + d * kb[i]), (lptr)(smem + so + min(wave + 8 * i, Cfg::PIECES - 1) * 1024), 16, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    f32x4 acc[MI][NI];
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int b = 0; b < NI; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // fragments: lane (row, q) of group g takes the k's 32 g + 8 q .. + 7 of the stage, for both operands
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)smem;
    const int row = lane & 15, q = lane >> 4;
    uint32_t vA[MI], vW[NI];   // the swizzle keys of a block's rows depend on the block where a row is 256 bytes or more
#pragma unroll
    for (int a = 0; a < MI; ++a) vA[a] = lds0 + (a * 16 + row) * AB + (((4 * grp + q) ^ kg_key<AB>(a * 16 + row)) << 4);
#pragma unroll
    for (int b = 0; b < NI; ++b) {
        const int r = wc * 16 * NI + b * 16 + row;
        vW[b] = lds0 + Cfg::A + r * WB + (((W_U8 ? 2 * grp + (q >> 1) : 4 * grp + q) ^ kg_key<WB>(r)) << 4) + (W_U8 ? (q & 1) * 8 : 0);
    }
    h16x8 fa[2][MI], fb[2][NI];
    u32x2 raw[2][NI];
    auto ldstage = [&](int set, int so) {
#pragma unroll
        for (int b = 0; b < NI; ++b) {
            if constexpr (W_U8) asm volatile("ds_read_b64 %0, %1" : "=v"(raw[set][b]) : "v"(vW[b] + so));
            else asm volatile("ds_read_b128 %0, %1" : "=v"(fb[set][b]) : "v"(vW[b] + so));
        }
#pragma unroll
        for (int a = 0; a < MI; ++a) asm volatile("ds_read_b128 %0, %1" : "=v"(fa[set][a]) : "v"(vA[a] + so));
        __builtin_amdgcn_sched_barrier(0);
    };
    const h16x2 off = {(h16)1023.5f, (h16)1023.5f};
    auto mul = [&](int set) {
#pragma unroll
        for (int b = 0; b < NI; ++b) {
            h16x8 w;
            if constexpr (W_U8) {
                const u32x2 v = raw[set][b];
                const h16x2 q0 = u8pair_lo_1024(v.x) - off, q1 = u8pair_hi_1024(v.x) - off, q2 = u8pair_lo_1024(v.y) - off, q3 = u8pair_hi_1024(v.y) - off;
                w = h16x8{q0.x, q0.y, q1.x, q1.y, q2.x, q2.y, q3.x, q3.y};
            } else {
                w = fb[set][b];
            }
#pragma unroll
            for (int a = 0; a < MI; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, fa[set][a], acc[a][b], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto reads_done = [&]() {
        __builtin_amdgcn_s_waitcnt(lgkm_only(0));
        __builtin_amdgcn_sched_barrier(0);
    };
    const GemmEpi &ep = mb.ep;
#pragma unroll
    for (int s = 0; s < NST; ++s)
        if (s < nk) issue_any(s, s * STAGE);
    bool lds_sums = false;
    float *lsum = (float *)(smem + Cfg::BODY);
    if constexpr (W_U8) {
        if (ep.parts > 1 && (splits == 1 || (m0 == 0 && split == 0))) {   // as in gemm_dma_body
            lds_sums = splits == 1;
            if (tid < 2 * TM) {
                const int r = tid % TM, which = tid / TM, t = min(t0 + r, T - 1);
                const float *p = (which ? ep.p2 : ep.p0) + (size_t)t * ep.parts;
                float tot = 0.f;
                for (int j = 0; j < ep.parts; j += 64) {
                    f32x4 v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) v[u] = j + 4 * u < ep.parts ? *(const f32x4 *)(p + j + 4 * u) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int u = 0; u < 16; ++u) tot = (((tot + v[u][0]) + v[u][1]) + v[u][2]) + v[u][3];
                }
                if (splits > 1) {
                    if (t0 + r < T) (which ? (float *)ep.s2 : (float *)ep.s0)[t] = tot;
                } else {
                    lsum[tid] = tot;
                }
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (nk >= NST) __builtin_amdgcn_s_waitcnt(vm_lgkm0((NST - 1) * LOADS));   // my part of stage 0 has landed
    else __builtin_amdgcn_s_waitcnt(vm_lgkm0(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    int so = 0;
    ldstage(0, 0);
    reads_done();
    // One stage: past its barrier stage kt + 1 has landed for every wave and nobody reads stage kt any more, so stage kt + NST goes
    // where it was.  STEADY: that one is there and whole.
    auto stage = [&](auto steady, int kt, int set) {
        constexpr bool STEADY = decltype(steady)::value;
        const int sn = so + STAGE >= NST * STAGE ? 0 : so + STAGE;
        if (STEADY || kt + NST <= nk) __builtin_amdgcn_s_waitcnt(vm_only((NST - 2) * LOADS));
        else __builtin_amdgcn_s_waitcnt(vm_only(0));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        ldstage(set ^ 1, sn);
        if constexpr (STEADY) issue(kt + NST, so);
        else if (kt + NST < nk) issue_any(kt + NST, so);
        if (STEADY || kt * BKS + grp * 32 < K) mul(set);   // the wave's k's of the last stage may be past the end
        reads_done();
        so = sn;
    };
    int kt = 0;
    const int steady = max(K / BKS - NST, 0) & ~1;   // stage kt + NST is whole for kt < K / BKS - NST
    for (; kt < steady; kt += 2) {
        stage(std::true_type{}, kt, 0);
        stage(std::true_type{}, kt + 1, 1);
    }
    for (; kt < nk; kt += 2) {   // an odd number of stages ends with one in which nobody multiplies
        stage(std::false_type{}, kt, 0);
        stage(std::false_type{}, kt + 1, 1);
    }
    // nothing may land in LDS or in a fragment register after this point (see gemm_dma_body)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int set = 0; set < 2; ++set) {
#pragma unroll
        for (int b = 0; b < NI; ++b) {
            if constexpr (W_U8) asm volatile("" ::"v"(raw[set][b]));
            else asm volatile("" ::"v"(fb[set][b]));
        }
#pragma unroll
        for (int a = 0; a < MI; ++a) asm volatile("" ::"v"(fa[set][a]));
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();   // every wave has read its last fragments: the partial tiles go where the stages were
    float *mypart = (float *)(smem + wave * REGION);
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int b = 0; b < NI; ++b) *(f32x4 *)(mypart + (a * 16 + row) * SW + b * 16 + 4 * q) = acc[a][b];
    auto tile_sum = [&](int r, int c) {   // four values at tile row r, column c: the groups' in group order
        const int half = RB == 2 && c >= TN / 2 ? 1 : 0;
        const float *p = (const float *)(smem + half * REGION) + r * SW + c - half * (TN / 2);
        f32x4 v = *(const f32x4 *)p;
#pragma unroll
        for (int k = 1; k < KG; ++k) v += *(const f32x4 *)(p + k * (RB * REGION / 4));
        return v;
    };
    constexpr int RPI = 512 / CPR, ITS = (TM + RPI - 1) / RPI;   // rows of a pass, passes
    const int cq = tid % CPR, col = m0 + cq * 8;
    const bool in_tile = cq * 8 < TN, col_ok = in_tile && col < M;
    if (splits > 1) {
        __syncthreads();
        float *slab = mb.part + (size_t)split * T * M;
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
            const int r = it * RPI + tid / CPR, t = t0 + r;
            if (r >= TM || t >= T || !col_ok) continue;
            *(f32x4 *)(slab + (size_t)t * M + col) = tile_sum(r, cq * 8);                                   // M % 4 == 0
            if (col + 4 < M) *(f32x4 *)(slab + (size_t)t * M + col + 4) = tile_sum(r, cq * 8 + 4);
        }
        return;
    }
    if (by_four(M, mb.ldy, mb.Y, ep)) {   // a loop of its own, as in gemm_dma_body
        __syncthreads();
#pragma unroll 1
        for (int it = 0; it < ITS; ++it) {
            const int r = it * RPI + tid / CPR, t = t0 + r;
            if (r >= TM || t >= T) break;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int c = e * (TN / 2) + cq * 4;
                if (!in_tile || m0 + c >= M) continue;
                f32x4 v = tile_sum(r, c);
                if constexpr (W_U8) affine4(v, m0 + c, M, lds_sums ? lsum[r] : ep.s0[t], lds_sums ? lsum[TM + r] : ep.s2[t], ep);
                finish_row4(v, t, m0 + c, M, ep, mb.Y, mb.ldy);
            }
        }
        return;
    }
    h16x8 rx8 = {}, mx8 = {};
    EpiIn ein[ITS] = {};
    if (W_U8 && col_ok) { rx8 = load_n<h16x8, 8>(ep.rx + col, M - col); mx8 = load_n<h16x8, 8>(ep.mx + col, M - col); }
    const Emit8 em = emit8(ep, col, col_ok);
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
        const int r = it * RPI + tid / CPR, t = t0 + r;
        ein[it] = epi_in(ep, t, col, r < TM && t < T && col_ok, W_U8 && !lds_sums);
    }
    __syncthreads();   // the partial tiles are in LDS
#pragma unroll 1
    for (int it = 0; it < ITS; ++it) {
        const EpiIn cur = ein[0];
#pragma unroll
        for (int i = 0; i + 1 < ITS; ++i) ein[i] = ein[i + 1];
        const int r = it * RPI + tid / CPR, t = t0 + r;
        const bool valid = r < TM && t < T && col_ok;
        float a0 = 0.f, a2 = 0.f;
        if (valid) {
            const f32x4 lo = tile_sum(r, cq * 8), hi = tile_sum(r, cq * 8 + 4);
            float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if constexpr (W_U8) affine8(v, rx8, mx8, lds_sums ? lsum[r] : cur.s0, lds_sums ? lsum[TM + r] : cur.s2);
            finish_row8<true>(v, cur, t, col, ep, mb.Y, mb.ldy, em, a0, a2);
        }
        if (ep.emit_ry) {   // the CPR threads of a row are neighbours in one wave; every lane takes part
#pragma unroll
            for (int o = 1; o < CPR; o <<= 1) { a0 += __shfl_xor(a0, o, WAVE); a2 += __shfl_xor(a2, o, WAVE); }
            if (valid && cq == 0) emit_parts(ep, t, m0, M, TN, a0, a2);
        }
    }
}

template <bool W_U8, int TM, int TN>
int launch_few(GemmGroup &g, int n, int64_t T, int64_t N, int ks, hipStream_t st) {
    constexpr int lds = FewCfg<W_U8, TM, TN>::LDS;
    static PerDeviceOnce once;
    bool *attr_done = once.slot();
    if (!attr_done || !*attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)gemm_few_kernel<W_U8, TM, TN>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
        if (attr_done) *attr_done = true;
    }
    const int units = (int)group_tiles(W_U8, g, n, T, N, TM, TN) * ks;
    hipLaunchKernelGGL((gemm_few_kernel<W_U8, TM, TN>), dim3((unsigned)units), dim3(512), lds, st, (int)T, units, ks, g.first[1], g.first[2], g.first[3],
                       g.nk_split, g.lda, (const GemmMembers &)g);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// second pass of a split group launch: member blockIdx.y, as splitk_epilogue8_kernel
struct SplitFactors { uint64_t f[4]; };
__global__ __launch_bounds__(256) void splitk_group_epilogue8_kernel(int T, int KS, SplitFactors rows, GemmMembers g) {
    const GemmMember &m = g.m[blockIdx.y];
    splitk_chunk8((int)blockIdx.x * 256 + threadIdx.x, T * (m.M / 8), m.M, rows.f[blockIdx.y], KS, m.part, m.Y, m.ldy, m.ep);
}

struct PrepGroup {
    const rwkv_half *x[4], *ry[4], *my[4];
    rwkv_half *xs[4];
    float *s0[4], *s2[4];
};

// xs[t, j] = fp16(x[t, j] * ry[j]);  s0[t] = sum_j x[t, j];  s2[t] = sum_j x[t, j] * my[j].  One workgroup (four
// waves) per row: a 16384-wide row per wave left the memory system with four waves per CU to draw from.
__global__ __launch_bounds__(256) void mm8_prepare_kernel(int T, int N, const rwkv_half *__restrict__ x, int64_t ldx,
                                                          const rwkv_half *__restrict__ ry,
                                                          const rwkv_half *__restrict__ my, rwkv_half *__restrict__ xs,
                                                          float *__restrict__ s0, float *__restrict__ s2) {
    __shared__ float red[8];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    float a0 = 0.f, a2 = 0.f;
    for (int j = threadIdx.x * 8; j < N; j += 256 * 8) {
        const u32x4 xv = *(const u32x4 *)(x + (size_t)t * ldx + j);
        const u32x4 rv = *(const u32x4 *)(ry + j);
        const u32x4 mv = *(const u32x4 *)(my + j);
        const h16x8 xh = __builtin_bit_cast(h16x8, xv), rh = __builtin_bit_cast(h16x8, rv),
                    mh = __builtin_bit_cast(h16x8, mv);
        h16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xf = (float)xh[e];
            o[e] = (h16)(xf * (float)rh[e]);
            a0 += xf;
            a2 += xf * (float)mh[e];
        }
        *(u32x4 *)(xs + (size_t)t * N + j) = __builtin_bit_cast(u32x4, o);
    }
    a0 = wave_sum(a0);
    a2 = wave_sum(a2);
    if (lane == 0) { red[wid] = a0; red[4 + wid] = a2; }
    __syncthreads();
    if (threadIdx.x == 0) {
        s0[t] = (red[0] + red[1]) + (red[2] + red[3]);
        s2[t] = (red[4] + red[5]) + (red[6] + red[7]);
    }
}

// the same for up to four (x, matrix) pairs in one launch: blockIdx.y picks the pair
__global__ __launch_bounds__(256) void mm8_prepare_group_kernel(int T, int N, PrepGroup g) {
    const int gi = blockIdx.y;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= T) return;
    const rwkv_half *x = g.x[gi], *ry = g.ry[gi], *my = g.my[gi];
    rwkv_half *xs = g.xs[gi];
    float a0 = 0.f, a2 = 0.f;
    for (int j = lane * 8; j < N; j += 64 * 8) {
        const h16x8 xh = *(const h16x8 *)(x + (size_t)t * N + j), rh = *(const h16x8 *)(ry + j), mh = *(const h16x8 *)(my + j);
        h16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xf = (float)xh[e];
            o[e] = (h16)(xf * (float)rh[e]);
            a0 += xf;
            a2 += xf * (float)mh[e];
        }
        *(h16x8 *)(xs + (size_t)t * N + j) = o;
    }
    a0 = wave_sum(a0);
    a2 = wave_sum(a2);
    if (lane == 0) { g.s0[gi][t] = a0; g.s2[gi][t] = a2; }
}



// ---- calls of 2 .. 16 rows: every weight row streamed once ---------------------------------------------------
// A ragged last prompt chunk (rwkv/utils.py:98-101) or a short chat turn has a handful of tokens: with 128-row
// tiles the contraction kernels spend their time on empty rows and a call costs several one-token steps.  Here
// (uint8) a workgroup of 16 waves, one per CU, takes a consecutive share of the launch's row groups (16 output rows each, the
// groups of all members in one order) and splits K over its waves: wave w owns the 64-wide units w, w + 16, ...; per
// unit a lane loads 16 bytes of one weight row (lane = row + 16 q), widens them to the exact fp16 value b + 1/2 and
// multiplies them with its token's values (lane = token + 16 q, rows past T repeat the last one) by
// v_mfma_f32_16x16x32_f16, weights first, so that lane (token j, q) ends with rows 4 q .. 4 q + 3 of token j.
// The 16 partial blocks are added in wave order through LDS (deterministic) by four of the waves, which round and store.
// Bound by HBM: the next step's weights, of the next row group where this one's end, are requested before a step is
// multiplied, and the barrier of an exchange waits for LDS only, so a wave always has a step in flight.  (A workgroup
// per row group, two to a CU, had its start, its activations and its end between any two requests.)
//   NU > 0   rows of up to 16 NU units: a wave holds its share of the activations in registers for all row groups.
//   NU == 0  longer rows: the activations come from L2 with the weights.  Fragment order asks for 16 rows per 16 lanes,
//            which the CU takes at 16 bytes a clock (9 TB/s over the chip from L2, 15.5 where four lanes ask for 64
//            consecutive bytes): they are read eight lanes to a row and change order in LDS of the wave's own.
// us a launch, 8 rows, against a workgroup per row group with fragment-order loads throughout: 4096 wide, three members of 4096
// outputs 18.7 -> 16.8, [8 x 16384] x [16384 x 4096] 22.9 -> 21.4, three of 5120 at 5120 wide 45.3 -> 28.9, [8 x 20480] x
// [20480 x 5120] 51.9 -> 46.6 (320 row groups on 256 CUs).  The same sums in the same order.
struct SkinnyGroup {
    int64_t lda;
    GemmMember m[4];
};

template <int NU>
__global__ __launch_bounds__(1024) void skinny_u8_kernel(uint64_t factor, int share, int rest, int T, int N, int n, SkinnyGroup g) {
    constexpr bool HELD = NU > 0;
    constexpr int UB = NU == 1 ? 1 : NU == 4 ? 4 : 2;           // units of a step
    constexpr int NS = HELD ? NU / UB : 2;                      // steps of a row group; NU == 0: of a pass of its loop
    constexpr int NB = HELD ? 2 : 1;                            // exchange buffers: with two, one barrier per row group
    constexpr int RQ = 80;                                      // floats per q of a block: the readers' banks differ
    __shared__ __align__(16) float red[NB][16][4 * RQ];
    __shared__ __align__(16) h16 sx[HELD ? 1 : 16][HELD ? 8 : 16 * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & 15, q = lane >> 4;
    const int nunits = N / 64;
    const h16x2 off = {(h16)1023.5f, (h16)1023.5f};
    const RowSplit sp = {factor, share, rest};
    const int b0 = split_at(sp, blockIdx.x), b1 = split_at(sp, blockIdx.x + 1);
    auto fence = [] {                                           // loads are used in the order of their issue (v7.hip)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](u32x4 wv, h16x8 x0, h16x8 x1, f32x4 &acc) {
        const h16x2 a0 = u8pair_lo_1024(wv.x) - off, a1 = u8pair_hi_1024(wv.x) - off;
        const h16x2 a2 = u8pair_lo_1024(wv.y) - off, a3 = u8pair_hi_1024(wv.y) - off;
        const h16x2 c0 = u8pair_lo_1024(wv.z) - off, c1 = u8pair_hi_1024(wv.z) - off;
        const h16x2 c2 = u8pair_lo_1024(wv.w) - off, c3 = u8pair_hi_1024(wv.w) - off;
        const h16x8 wa = {a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y};
        const h16x8 wb = {c0.x, c0.y, c1.x, c1.y, c2.x, c2.y, c3.x, c3.y};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa, x0, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb, x1, acc, 0, 0, 0);
    };
    int base = 0, count = 0;                                    // row groups of the members before; done by this workgroup
    for (int gi = 0; gi < n; ++gi) {
        const GemmIn in = gemm_in(g.m[gi]);
        const int M = in.M, groups = (M + 15) >> 4;
        const int lo = max(b0, base) - base, hi = min(b1, base + groups) - base;
        base += groups;
        if (lo >= hi) continue;
        const GemmEpi &ep = g.m[gi].ep;
        const h16 *A = in.A;
        const unsigned char *W = (const unsigned char *)in.W;
        const int64_t ldw = in.ldw;
        // In place of a unit past the end of the row, and of every unit past the share's last row group, all lanes load the
        // first bytes of the matrix, which nothing uses: a branch around a load would make the waits for those before it longer.
        struct Step { u32x4 w[UB]; h16x8 x[HELD ? 1 : UB][2]; };
        auto load_w = [&](Step &s, int grp, int i0) {
            const bool there = grp < hi;
            const size_t row = (size_t)min(16 * grp + sub, M - 1) * ldw + 16 * q;
#pragma unroll
            for (int i = 0; i < UB; ++i) {
                const int u = wave + 16 * (i0 + i);
                s.w[i] = __builtin_nontemporal_load((const u32x4 *)(W + (there && u < nunits ? row + (size_t)u * 64 : 0)));
            }
        };
        struct Ops { rwkv_half rx, mx, res, gate; float s0, s2; };
        const int ft = (threadIdx.x & 255) >> 4, fm = threadIdx.x & 15;   // the output that a thread of the four waves finishes
        const bool has_res = ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL, has_gate = ep.act == ACT_GATED_RESIDUAL;
        auto load_ops = [&](int grp) {
            Ops o = {};
            const int t = min(ft, T - 1), m = min(16 * grp + fm, M - 1);
            o.rx = ep.rx[m]; o.mx = ep.mx[m]; o.s0 = ep.s0[t]; o.s2 = ep.s2[t];
            o.res = *(has_res ? ep.res + (size_t)t * ep.ldres + m : (const rwkv_half *)A);
            o.gate = *(has_gate ? ep.gate + (size_t)t * ep.ldgate + m : (const rwkv_half *)A);
            return o;
        };
        auto finish = [&](int grp, const f32x4 &acc, const Ops &o) {
            const int buf = count & (NB - 1);
            if (NB == 1 && count) {                              // the sums of the row group before have been read
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            *(f32x4 *)&red[buf][wave][RQ * q + 4 * sub] = acc;
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);                  // LDS only: __syncthreads() would also wait for the loads in flight
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if ((wave >> 2) == (count & 3)) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < 16; ++w) v += red[buf][w][RQ * (fm >> 2) + 4 * ft + (fm & 3)];
                const int m = 16 * grp + fm;
                if (m < M && ft < T) {
                    const size_t at = (size_t)ft * g.m[gi].ldy + m;
                    v = epi_affine(v, h2f(o.rx), h2f(o.mx), o.s0, o.s2);
                    if (ep.raw_f32) {
                        ((float *)g.m[gi].Y)[at] = v;
                    } else {
                        float r[1] = {v};
                        h16 res[1] = {__builtin_bit_cast(h16, o.res)}, gate[1] = {__builtin_bit_cast(h16, o.gate)};
                        epi_act<1, const h16 *>(r, res, gate, ep);
                        if (ep.out_dtype == RWKV_DT_F32) ((float *)g.m[gi].Y)[at] = round_h(r[0]);
                        else ((rwkv_half *)g.m[gi].Y)[at] = f2h(r[0]);
                    }
                }
                if (NB == 1) __builtin_amdgcn_s_waitcnt(0xC07F);
            }
            ++count;
        };
        Step st[2];
        if constexpr (HELD) {
            const h16 *arow = A + (size_t)min(sub, T - 1) * g.lda;
            h16x8 rx[NU][2];
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                const int u = wave + 16 * i;
                const h16 *p = arow + (size_t)min(u, nunits - 1) * 64;
                rx[i][0] = *(const h16x8 *)(p + 16 * q);
                rx[i][1] = *(const h16x8 *)(p + 16 * q + 8);
            }
            fence();
            load_w(st[0], lo, 0);
            fence();
            constexpr int PASS = NS == 1 ? 2 : 1;                // row groups per pass: the two steps' registers alternate
            for (int grp = lo; grp < hi; grp += PASS) {
#pragma unroll
                for (int p = 0; p < PASS; ++p) {
                    if (grp + p >= hi) break;
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                    const Ops o = load_ops(grp + p);
                    fence();
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        const int j = p * NS + k;
                        load_w(st[(j + 1) & 1], k + 1 < NS ? grp + p : grp + p + 1, k + 1 < NS ? (k + 1) * UB : 0);
                        fence();
#pragma unroll
                        for (int i = 0; i < UB; ++i)
                            if (wave + 16 * (k * UB + i) < nunits) multiply(st[j & 1].w[i], rx[k * UB + i][0], rx[k * UB + i][1], acc);
                        fence();
                    }
                    finish(grp + p, acc, o);
                }
            }
        } else {
            const int r8 = lane >> 3, seg = lane & 7;
            const size_t xa = (size_t)min(r8, T - 1) * g.lda + 8 * seg, xb = (size_t)min(r8 + 8, T - 1) * g.lda + 8 * seg;
            h16 *slot = sx[wave];
            h16 *wr = slot + 64 * r8 + 8 * (seg ^ r8);           // (r8 + 8) & 7 == r8
            const h16 *rd0 = slot + 64 * sub + 8 * (2 * q ^ (sub & 7)), *rd1 = slot + 64 * sub + 8 * ((2 * q + 1) ^ (sub & 7));
            auto load = [&](Step &s, int grp, int i0) {
#pragma unroll
                for (int i = 0; i < UB; ++i) {
                    const int u = wave + 16 * (i0 + i);
                    const bool ok = grp < hi && u < nunits;
                    s.x[i][0] = *(const h16x8 *)(A + (ok ? xa + (size_t)u * 64 : 0));
                    s.x[i][1] = *(const h16x8 *)(A + (ok ? xb + (size_t)u * 64 : 0));
                }
                load_w(s, grp, i0);
            };
            // units per wave, whole passes
            const int span = ((nunits + 15) / 16 + NS * UB - 1) / (NS * UB) * (NS * UB);
            load(st[0], lo, 0);
            fence();
            for (int grp = lo; grp < hi; ++grp) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                for (int i0 = 0; i0 < span; i0 += NS * UB) {
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        const int next = i0 + (k + 1) * UB;
                        load(st[(k + 1) & 1], next < span ? grp : grp + 1, next < span ? next : 0);
                        fence();
#pragma unroll
                        for (int i = 0; i < UB; ++i) {
                            if (wave + 16 * (i0 + k * UB + i) >= nunits) continue;
                            *(h16x8 *)wr = st[k & 1].x[i][0];
                            *(h16x8 *)(wr + 8 * 64) = st[k & 1].x[i][1];
                            const h16x8 x0 = *(const h16x8 *)rd0, x1 = *(const h16x8 *)rd1;
                            multiply(st[k & 1].w[i], x0, x1, acc);
                        }
                        fence();
                    }
                }
                finish(grp, acc, load_ops(grp));
            }
        }
    }
}

// fp16 weights: a workgroup per 16 output rows (two to a CU), the same split of K over its waves: wave w owns the 32-wide
// chunks w, w + 16, ...  NCI > 0: a wave owns at most NCI chunks and keeps their activation values in registers; NCI == 0: any
// row length, activations re-read from L2 for every row group.  The uint8 form above with units of two neighbouring chunks, a
// whole line of a row, is 5 to 15 % faster per call, but adds in another order, and a deep RWKV-7 model at the start of a
// conversation makes 8 % of that (2-norm of its state); with these chunks, half a line to a request, it is up to 4 % slower in
// calls of 2 tokens (RWKV-7, 4096 wide, us a layer: 142.9 / 148.6).
template <int NCI>
__global__ __launch_bounds__(1024) void skinny_f16_kernel(int T, int N, SkinnyGroup g) {
    __shared__ float red[16][64][4];
    const int gi = blockIdx.y;
    const GemmIn gin = gemm_in(g.m[gi]);
    const int M = gin.M;
    const h16 *__restrict__ A = gin.A;
    const unsigned char *__restrict__ W = (const unsigned char *)gin.W;
    const int64_t lda = g.lda, ldw = gin.ldw;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & 15, q = lane >> 4;
    const int nchunks = N / 32;
    const int ngroups = (M + 15) >> 4;
    const h16 *arow = A + (size_t)min(sub, T - 1) * lda;   // this lane's token
    constexpr int NB = NCI > 0 ? NCI : 4;            // chunks loaded before any is multiplied
    auto load_x = [&](int c) { return *(const h16x8 *)(arow + (size_t)c * 32 + 8 * q); };
    auto load_w = [&](const unsigned char *wrow, int c) {
        return __builtin_nontemporal_load((const u32x4 *)(wrow + ((size_t)c * 32 + 8 * q) * 2));
    };
    auto multiply = [&](u32x4 wv, h16x8 x, f32x4 &acc) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h16x8, wv), x, acc, 0, 0, 0);
    };
    // chunks past the end of the row repeat the last one and multiply zeros: no branch sits between the loads and
    // their use (loads would be sunk behind it, one chunk in flight at a time)
    h16x8 rx[NB];
    if (NCI > 0) {
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            rx[i] = load_x(min(wave + 16 * i, nchunks - 1));
            if (wave + 16 * i >= nchunks) rx[i] = h16x8{};
        }
    }
    for (int grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const int m0 = grp << 4;
        const unsigned char *wrow = W + (size_t)min(m0 + sub, M - 1) * ldw * 2;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (NCI > 0) {
            u32x4 wv[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) wv[i] = load_w(wrow, min(wave + 16 * i, nchunks - 1));
#pragma unroll
            for (int i = 0; i < NB; ++i) multiply(wv[i], rx[i], acc);
        } else {
            for (int c0 = wave; c0 < nchunks; c0 += 16 * NB) {
                u32x4 wv[NB];
                h16x8 x[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const int c = min(c0 + 16 * i, nchunks - 1);
                    wv[i] = load_w(wrow, c);
                    x[i] = load_x(c);
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (c0 + 16 * i >= nchunks) x[i] = h16x8{};
                    multiply(wv[i], x[i], acc);
                }
            }
        }
        __syncthreads();                                          // the previous group's sums have been read
        *(f32x4 *)&red[wave][lane][0] = acc;
        __syncthreads();
        if (threadIdx.x < 256) {
            const int l = threadIdx.x & 63, r = threadIdx.x >> 6;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < 16; ++w) v += red[w][l][r];
            const int m = m0 + 4 * (l >> 4) + r, t = l & 15;
            if (m < M && t < T) gemm_epilogue(v, t, m, 1.f, 0.f, g.m[gi].ep, g.m[gi].Y, g.m[gi].ldy);
        }
    }
}

constexpr int SKINNY_MAX_ROWS = 16;

// what these kernels assume of one product: whole units or chunks, 16-byte aligned rows for its 16-byte loads
bool skinny_ok(bool w_u8, int64_t T, int64_t N, const void *A, int64_t lda, const void *W, int64_t ldw, const GemmEpi &ep) {
    auto a16 = [](const void *p) { return (((uintptr_t)p) & 15) == 0; };
    if (T < 2 || T > SKINNY_MAX_ROWS || N < 64 || (N % 64)) return false;
    if ((lda & 7) || (ldw & (w_u8 ? 15 : 7)) || !a16(A) || !a16(W)) return false;
    if (w_u8 && (!ep.rx || !ep.mx || !ep.s0 || !ep.s2)) return false;
    if (!w_u8 && ep.rx) return false;
    const char *e = getenv("RWKV_NO_SKINNY");                     // tuning: send short calls through the tile kernels
    return !(e && *e == '1');
}

int skinny_launch(bool w_u8, int n, int64_t T, int64_t N, const SkinnyGroup &g, hipStream_t st) {
    int total = 0, maxg = 1;
    for (int i = 0; i < n; ++i) {
        total += (g.m[i].M + 15) / 16;
        maxg = std::max(maxg, (g.m[i].M + 15) / 16);
    }
    const int64_t per_wave = (N / (w_u8 ? 64 : 32) + 15) / 16;    // chunks a wave owns
    const int grid = std::min(total, num_cu());
    const RowSplit sp = row_split(total, grid);
#define RWKV_SKINNY(NC)                                                                                                              \
    do {                                                                                                                             \
        if (w_u8) hipLaunchKernelGGL((skinny_u8_kernel<NC>), dim3((unsigned)grid), dim3(1024), 0, st, sp.factor, sp.q, sp.r, (int)T, \
                                     (int)N, n, g);                                                                                  \
        else hipLaunchKernelGGL((skinny_f16_kernel<NC>), dim3((unsigned)std::min(maxg, 2 * num_cu()), (unsigned)n), dim3(1024), 0,   \
                                st, (int)T, (int)N, g);                                                                              \
    } while (0)
    if (per_wave <= 1) RWKV_SKINNY(1);
    else if (per_wave <= 2) RWKV_SKINNY(2);
    else if (per_wave <= 4) RWKV_SKINNY(4);
    else if (per_wave <= 8) RWKV_SKINNY(8);
    else RWKV_SKINNY(0);
#undef RWKV_SKINNY
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// ---- narrow outputs: [T, N] x [N, M] with M of a LoRA rank and fp16 weights ------------------------------------
// The first stage of a low-rank product (RWKV-6 mixing and decay LoRA, RWKV-7's four) has thousands of input columns
// and a few dozen to a few hundred outputs: a handful of 128 x 128 tiles, which the tile kernels can only spread
// over the chip by splitting K and adding the slabs in a second launch.  Here a workgroup of eight waves takes a
// 16 x 16 block of the output and splits K over its waves: wave w owns the 32-wide k-chunks w, w + 8, ...; it loads
// 16 bytes a lane of the weight rows and of the activation rows, sixteen chunks in flight (one round at 4096), and issues
// v_mfma_f32_16x16x32_f16 with the weights as the first operand, so that lane (token j, q) ends with outputs 4 q .. 4 q + 3
// of token j.  The eight partial blocks are added in wave order through LDS (deterministic) and 64 threads round, apply the
// activation and store 8 bytes each.  Operands come from L2: the weights once per 16 rows of the call, the activation once
// per 16 outputs, 256 KB a workgroup at 4096, at the rate its CU takes them: 16 bytes a clock in the order of the fragments
// (16 rows for 16 lanes), 64 where four neighbouring lanes ask for 64 bytes of a row.  So they are loaded that way and change
// order in 2 KB of LDS per wave.  [256 x 4096] x [4096 x 160]: 9.9 us in fragment order with the ten loads in flight that the
// compiler left, 6.8 now; K-split tiles and their second pass 21.
__global__ __launch_bounds__(512) void narrow_kernel(int T, int N, int M, const h16 *__restrict__ A, int64_t lda,
                                                     const h16 *__restrict__ W, int64_t ldw, rwkv_half *__restrict__ Y,
                                                     int64_t ldy, GemmEpi ep) {
    __shared__ f32x4 red[8][64];
    __shared__ __align__(16) h16 order[8][2][16 * 32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane & 15, q = lane >> 4;
    const int t0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
    // loaded: row lane / 4, piece lane & 3 of eight k's; multiplied: row sub, piece q.  Piece p of row r lies at p ^ (r / 4)
    const int lr = lane >> 2, lp = lane & 3;
    const h16 *arow = A + (size_t)min(t0 + lr, T - 1) * lda + 8 * lp;
    const h16 *wrow = W + (size_t)min(m0 + lr, M - 1) * ldw + 8 * lp;
    h16 *const in = &order[wave][0][32 * lr + 8 * (lp ^ (lr >> 2))];
    const h16 *const frag = &order[wave][0][32 * sub + 8 * (q ^ (sub >> 2))];
    const int nchunks = N / 32;
    constexpr int NB = 16;   // chunks in flight per wave: a 4096-wide row is one round
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // chunks past the end repeat the last one and multiply zeros (no branch between the loads and their use)
    for (int c0 = wave; c0 < nchunks; c0 += 8 * NB) {
        h16x8 wv[NB], xv[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int c = min(c0 + 8 * i, nchunks - 1);
            wv[i] = *(const h16x8 *)(wrow + (size_t)c * 32);
            xv[i] = *(const h16x8 *)(arow + (size_t)c * 32);
        }
        __builtin_amdgcn_sched_barrier(0);   // all of them before the first use
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            if (c0 + 8 * i >= nchunks) xv[i] = h16x8{};
            *(h16x8 *)in = wv[i];
            *(h16x8 *)(in + 16 * 32) = xv[i];
            const h16x8 wf = *(const h16x8 *)frag, xf = *(const h16x8 *)(frag + 16 * 32);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf, acc, 0, 0, 0);
        }
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
        f32x4 v = red[0][lane];
#pragma unroll
        for (int w = 1; w < 8; ++w) v += red[w][lane];
        const int t = t0 + sub, m = m0 + 4 * q;
        if (t < T && m < M) {   // M % 4 == 0
            float r[4] = {v[0], v[1], v[2], v[3]};
            epi_act(r, h16x4{}, h16x4{}, ep);
            h16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (h16)r[e];
            *(h16x4 *)((h16 *)Y + (size_t)t * ldy + m) = o;
        }
    }
}

// narrow_kernel's operands: fp16 weights, at most NARROW_MAX_M outputs, rows of whole 32-wide chunks laid out for
// 16-byte loads, an epilogue without residual or gate, fp16 out; as many workgroups as CUs, or twice that where the rows are
// long.  us a product, this kernel and the tiles: one round, [400 x 512] x [512 x 64] 5.3 / 5.9, [256 x 768] x [768 x 160]
// 5.4 / 6.4, [1024 x 4096] x [4096 x 64] 6.6 / 15.7; two rounds, [777 x 4096] x [4096 x 160] 15.1 / 15.8, [512 x 2560] x
// [2560 x 160] 10.4 / 12.8, [777 x 2048] x [2048 x 160] 11.1 / 10.8, [512 x 1024] x [1024 x 160] 8.6 / 8.0; three, [1024 x
// 2560] x [2560 x 160] 14.0 / 12.5.  RWKV_NO_NARROW=1 sends these through the tile kernels (tuning).
constexpr int NARROW_MAX_M = 192;
bool narrow_ok(bool w_u8, int64_t T, int64_t N, int64_t M, const void *A, int64_t lda, const void *W, int64_t ldw, const void *Y,
               int64_t ldy, const GemmEpi &ep) {
    auto a16 = [](const void *p) { return (((uintptr_t)p) & 15) == 0; };
    if (w_u8 || ep.rx || T <= SKINNY_MAX_ROWS || M > NARROW_MAX_M || (M & 3) || N < 512 || (N % 32)) return false;
    if (((T + 15) / 16) * ((M + 15) / 16) > (N < 2560 ? 1 : 2) * num_cu()) return false;
    if ((lda & 7) || (ldw & 7) || (ldy & 3) || !a16(A) || !a16(W) || (((uintptr_t)Y) & 7)) return false;
    if (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL || ep.raw_f32 || ep.out_dtype != RWKV_DT_F16) return false;
    const char *e = getenv("RWKV_NO_NARROW");
    return !(e && *e == '1');
}

}  // namespace

namespace {

template <bool W_U8, int BT, int BM, int WT, int WM, int PF>
int launch_cfg(int64_t T, int64_t N, int64_t M, const rwkv_half *A, int64_t lda, const void *W, int64_t ldw, void *Y,
               int64_t ldy, const GemmEpi &ep, hipStream_t st) {
    constexpr size_t lds = 2 * (size_t)(BT + BM) * BK * sizeof(h16);
    static PerDeviceOnce once;
    bool *attr_done = once.slot();
    if (lds > 64 * 1024 && (!attr_done || !*attr_done)) {
        hipError_t e = hipFuncSetAttribute((const void *)gemm_kernel<W_U8, BT, BM, WT, WM, PF, false>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        if (attr_done) *attr_done = true;
    }
    const int64_t tiles = ((T + BT - 1) / BT) * ((M + BM - 1) / BM);
    // Too few tiles to fill the chip (short prompts, narrow matrices): split the contraction over KS
    // workgroups per tile; partial sums go to fp32 slabs and a second pass reduces them in slab order.
    int ks = 1;
    const int nk = (int)(N / BK);
    // up to 128 tiles: split until every CU has a workgroup; up to 256 tiles (at most one workgroup per CU, which
    // leaves a CU's four waves waiting on their own loads): split in two, +12-18 % on 1024 x 4096 x 4096,
    // 1024 x 16384 x 4096 and 256 x 4096 x 16384
    const int want = tiles <= 128 ? 256 : 512;
    if (ep.splitk_ws && tiles <= 256 && lds <= 64 * 1024 && (M & 3) == 0) {
        // the smallest split that reaches that many workgroups (slab traffic grows with the split)
        for (int c = 2; c <= 8; c <<= 1) {
            if (nk % c || nk / c < 8) break;                                      // whole k-tiles, several per split
            if ((size_t)c * T * M * sizeof(float) > ep.splitk_bytes) break;       // slabs must fit
            ks = c;
            if (tiles * c >= want) break;
        }
    }
    if (ks > 1) {
        hipLaunchKernelGGL((gemm_kernel<W_U8, BT, BM, WT, WM, PF, true>), dim3((unsigned)tiles, (unsigned)ks), dim3(64 * WT * WM), lds, st,
                           (int)T, (int)N, (int)M, (const h16 *)A, lda, W, ldw, Y, ldy, ep, nk / ks, ep.splitk_ws);
        const int64_t n = T * M;
        const unsigned blocks = (unsigned)((n + 1023) / 1024 < 16384 ? (n + 1023) / 1024 : 16384);
        hipLaunchKernelGGL(splitk_epilogue_kernel, dim3(blocks), dim3(256), 0, st, (int)T, (int)M, ks, ep.splitk_ws, Y, ldy, ep);
    } else {
        hipLaunchKernelGGL((gemm_kernel<W_U8, BT, BM, WT, WM, PF, false>), dim3((unsigned)tiles), dim3(64 * WT * WM), lds, st, (int)T,
                           (int)N, (int)M, (const h16 *)A, lda, W, ldw, Y, ldy, ep, nk, (float *)nullptr);
    }
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// what the direct-to-LDS kernels assume: whole k-tiles, 16-byte rows and row starts for their loads, and for the eight-wide
// epilogue unless the outputs are stored plainly (four at a time then, any width, stride and boundary)
bool dma_ok(bool w_u8, int64_t N, int64_t M, const void *A, int64_t lda, const void *W, int64_t ldw, const void *Y, int64_t ldy,
            const GemmEpi &ep) {
    auto a16 = [](const void *p) { return (((uintptr_t)p) & 15) == 0; };
    if ((N % BK) || (lda & 7) || (ldw & (w_u8 ? 15 : 7))) return false;
    // output rows that are not made of aligned 16-byte pieces: plain stores only
    const bool wide = !(M & 7) && !(ldy & 7) && a16(Y);
    if (!wide && (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL || ep.emit_ry)) return false;
    if (!a16(A) || !a16(W)) return false;
    if (w_u8 && (!ep.rx || !ep.mx || !ep.s0 || !ep.s2 || !a16(ep.rx) || !a16(ep.mx))) return false;
    if (!w_u8 && ep.rx) return false;
    if (ep.act == ACT_RESIDUAL || ep.act == ACT_GATED_RESIDUAL)
        if (!ep.res || !a16(ep.res) || (ep.ldres & 7)) return false;
    if (ep.act == ACT_GATED_RESIDUAL)
        if (!ep.gate || !a16(ep.gate) || (ep.ldgate & 7)) return false;
    return true;
}

// The second pass of a direct-to-LDS launch with K split ks ways: eight outputs wide where M is a multiple.
int launch_splitk_epilogue(int ks, int64_t T, int64_t M, void *Y, int64_t ldy, const GemmEpi &ep, hipStream_t st) {
    const int64_t n = T * M;
    if (M & 7) {
        hipLaunchKernelGGL(splitk_epilogue_kernel, dim3((unsigned)std::min<int64_t>((n + 1023) / 1024, 16384)), dim3(256), 0, st, (int)T, (int)M, ks,
                           ep.splitk_ws, Y, ldy, ep);
    } else {
        hipLaunchKernelGGL(splitk_epilogue8_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, st, ep.splitk_ws, div_factor(M / 8),
                           (int)(n / 8), (int)M, ks, Y, ldy, ep);
    }
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

// A launch of tile `tile` with K split ks ways, its slabs in g.part.
template <bool W_U8>
int launch_tile(int tile, GemmGroup &g, int n, int64_t T, int64_t N, int ks, hipStream_t st) {
    switch (tile) {
        case TILE_256x256: return launch_dma<W_U8, 256, 256, 0>(g, n, T, N, ks, st);
        case TILE_S: return launch_dma<W_U8, 128, 128, 0>(g, n, T, N, ks, st);
        case TILE_S4: return launch_dma<W_U8, 128, 128, 4>(g, n, T, N, ks, st);
        case TILE_K8: return launch_kg<W_U8, 64, 64>(g, n, T, N, ks, st);
        case TILE_K4: return launch_kg<W_U8, 64, 128>(g, n, T, N, ks, st);
        case TILE_256x192: return launch_dma<W_U8, 256, 192, 0>(g, n, T, N, ks, st);
        case TILE_224x256: return launch_dma<W_U8, 224, 256, 0>(g, n, T, N, ks, st);
        case TILE_224x192: return launch_dma<W_U8, 224, 192, 0>(g, n, T, N, ks, st);
        case TILE_192x256: return launch_dma<W_U8, 192, 256, 0>(g, n, T, N, ks, st);
        case TILE_192x192: return launch_dma<W_U8, 192, 192, 0>(g, n, T, N, ks, st);
        case TILE_160x256: return launch_dma<W_U8, 160, 256, 0>(g, n, T, N, ks, st);
        case TILE_160x192: return launch_dma<W_U8, 160, 192, 0>(g, n, T, N, ks, st);
        case TILE_128x256: return launch_dma<W_U8, 128, 256, 0>(g, n, T, N, ks, st);
        case TILE_128x192: return launch_dma<W_U8, 128, 192, 0>(g, n, T, N, ks, st);
        case TILE_96x128: return launch_dma<W_U8, 96, 128, 4>(g, n, T, N, ks, st);
        case TILE_128x96: return launch_dma<W_U8, 128, 96, 4>(g, n, T, N, ks, st);
        case TILE_96x96: return launch_dma<W_U8, 96, 96, 4>(g, n, T, N, ks, st);
        case TILE_32x16: return launch_few<W_U8, 32, 16>(g, n, T, N, ks, st);
        case TILE_32x32: return launch_few<W_U8, 32, 32>(g, n, T, N, ks, st);
        case TILE_32x48: return launch_few<W_U8, 32, 48>(g, n, T, N, ks, st);
        case TILE_32x64: return launch_few<W_U8, 32, 64>(g, n, T, N, ks, st);
        case TILE_32x96: return launch_few<W_U8, 32, 96>(g, n, T, N, ks, st);
        case TILE_48x16: return launch_few<W_U8, 48, 16>(g, n, T, N, ks, st);
        case TILE_48x32: return launch_few<W_U8, 48, 32>(g, n, T, N, ks, st);
        case TILE_48x48: return launch_few<W_U8, 48, 48>(g, n, T, N, ks, st);
        case TILE_48x64: return launch_few<W_U8, 48, 64>(g, n, T, N, ks, st);
        case TILE_48x96: return launch_few<W_U8, 48, 96>(g, n, T, N, ks, st);
        case TILE_64x16: return launch_few<W_U8, 64, 16>(g, n, T, N, ks, st);
        case TILE_64x32: return launch_few<W_U8, 64, 32>(g, n, T, N, ks, st);
        case TILE_64x48: return launch_few<W_U8, 64, 48>(g, n, T, N, ks, st);
        case TILE_64x64: return launch_few<W_U8, 64, 64>(g, n, T, N, ks, st);
        case TILE_64x96: return launch_few<W_U8, 64, 96>(g, n, T, N, ks, st);
        default: return RWKV_E_DTYPE;
    }
}

constexpr int CFG_DMA = 16;   // + TILE_*
template <bool W_U8>
int launch_pick(int cfg, int ks, int64_t T, int64_t N, int64_t M, const rwkv_half *A, int64_t lda, const void *W, int64_t ldw,
                void *Y, int64_t ldy, const GemmEpi &ep, hipStream_t st) {
    switch (cfg) {
        case 3: return launch_cfg<W_U8, 128, 128, 2, 2, 4>(T, N, M, A, lda, W, ldw, Y, ldy, ep, st);
        case 9:
            if constexpr (W_U8) return launch_cfg<true, 256, 256, 4, 4, 2>(T, N, M, A, lda, W, ldw, Y, ldy, ep, st);
            return RWKV_E_DTYPE;
        default: break;
    }
    if (cfg < CFG_DMA || cfg >= CFG_DMA + TILES) return RWKV_E_DTYPE;
    if (!dma_ok(W_U8, N, M, A, lda, W, ldw, Y, ldy, ep)) return RWKV_E_LAYOUT;
    GemmGroup g{};
    g.m[0].A = (const h16 *)A; g.m[0].W = W; g.m[0].Y = Y; g.lda = lda; g.m[0].ldw = ldw; g.m[0].ldy = ldy; g.m[0].M = (int)M; g.m[0].ep = ep;
    g.nk_split = (int)(N / BK) / ks;
    g.m[0].part = ep.splitk_ws;
    const int rc = launch_tile<W_U8>(cfg - CFG_DMA, g, 1, T, N, ks, st);
    if (rc || ks == 1) return rc;
    return launch_splitk_epilogue(ks, T, M, Y, ldy, ep, st);
}

// Tile choice (RWKV_GEMM_CFG overrides it for tuning sweeps: 3 and 9 the register-staged tiles by their number here, 14 and 15 the
// direct-to-LDS 256 x 256 and 128 x 128 ones, 18 TILE_S4, 20 to 48 the others in the order of tile_choice.h, with the K split of least
// cost).
//   CFG_DMA +  operands laid out for 16-byte loads: the direct-to-LDS kernel with the tile and K split that the cost
//              model puts first (128 x 128 tiles at full depth when another product runs beside this one: a 256 x 256
//              tile's LDS leaves no room beside it on the CU, two small ones fit)
//   9          uint8 weights otherwise, where 256 x 256 tiles of the register-staged kernel fill the chip: one per CU
//              and round, the last round at least 70 % full
//   3          everything else: 128 x 128 tiles, 4 k-tiles of prefetch
int pick_cfg(int64_t T, int64_t N, int64_t M, bool w_u8, const GemmEpi &ep, bool dma, int *ks, float *us = nullptr) {
    const bool alone = !ep.small_tiles;
    *ks = 1;
    // The reduction pass takes eight outputs at a time, or four.  Not splitting widths that are no multiple of eight cost
    // [100 x 16384] x [16384 x 1004] 45.7 us against 28.2, [300 x 16384] x [16384 x 1004] 48.8 against 33.4.
    const size_t ws = !(M & 3) && ep.splitk_ws ? ep.splitk_bytes : 0;
    auto take = [&](const TilePick &p) {
        *ks = p.ks;
        if (us) *us = p.us;
        return CFG_DMA + p.tile;
    };
    auto with_split = [&](int tile) { return take(Launch(T, (int)(N / BK), 1, &M, ws).with(w_u8, tile)); };
    const char *e = getenv("RWKV_GEMM_CFG");
    if (e && *e) {
        const int cfg = atoi(e);
        return cfg == 14 ? with_split(TILE_256x256) : cfg == 15 ? with_split(TILE_S) : cfg == 18 ? with_split(TILE_S4)
             : cfg >= 20 && cfg < 20 + TILES - TILE_K8 ? with_split(cfg - 20 + TILE_K8) : cfg < CFG_DMA ? cfg : -1;
    }
    if (dma && !alone) return with_split(TILE_S);
    if (dma) return take(Launch(T, (int)(N / BK), 1, &M, ws).best(w_u8));
    if (!alone) return 3;
    const int64_t big = ((T + 255) / 256) * ((M + 255) / 256), rounds = (big + 255) / 256;
    return w_u8 && big * 10 >= rounds * 256 * 7 ? 9 : 3;   // fp16 weight tiles are twice the bytes: the large tile spills
}

}  // namespace

GemmPlan gemm_plan(bool w_u8, int64_t T, int64_t N, int64_t M, const rwkv_half *A, int64_t lda, const void *W,
                   int64_t ldw, const void *Y, int64_t ldy, const GemmEpi &ep) {
    if (skinny_ok(w_u8, T, N, A, lda, W, ldw, ep)) return GemmPlan{0, 0, 0, 1, 0.0};
    int ks;
    float us;
    const int cfg = pick_cfg(T, N, M, w_u8, ep, dma_ok(w_u8, N, M, A, lda, W, ldw, Y, ldy, ep), &ks, &us);
    if (cfg < CFG_DMA) return GemmPlan{1, 0, 0, 1, 0.0};
    const TileDim d = tile_dim[cfg - CFG_DMA];
    return GemmPlan{2, d.tm, d.tn, ks, us};
}

int gemm_launch(bool w_u8, int64_t T, int64_t N, int64_t M, const rwkv_half *A, int64_t lda, const void *W,
                int64_t ldw, void *Y, int64_t ldy, const GemmEpi &ep, hipStream_t st) {
    if (skinny_ok(w_u8, T, N, A, lda, W, ldw, ep)) {
        SkinnyGroup g{};
        g.m[0].A = (const h16 *)A; g.m[0].W = W; g.m[0].Y = Y; g.lda = lda; g.m[0].ldw = ldw; g.m[0].ldy = ldy; g.m[0].M = (int)M; g.m[0].ep = ep;
        return skinny_launch(w_u8, 1, T, N, g, st);
    }
    if (narrow_ok(w_u8, T, N, M, A, lda, W, ldw, Y, ldy, ep)) {
        hipLaunchKernelGGL(narrow_kernel, dim3((unsigned)((T + 15) / 16), (unsigned)((M + 15) / 16)), dim3(512), 0, st, (int)T, (int)N,
                           (int)M, (const h16 *)A, lda, (const h16 *)W, ldw, (rwkv_half *)Y, ldy, ep);
        RWKV_LAUNCH_CHECK();
        return RWKV_OK;
    }
    int ks;
    const int cfg = pick_cfg(T, N, M, w_u8, ep, dma_ok(w_u8, N, M, A, lda, W, ldw, Y, ldy, ep), &ks);
    return w_u8 ? launch_pick<true>(cfg, ks, T, N, M, A, lda, W, ldw, Y, ldy, ep, st)
                : launch_pick<false>(cfg, ks, T, N, M, A, lda, W, ldw, Y, ldy, ep, st);
}

int mm8_prepare_launch(int64_t T, int64_t N, const rwkv_half *x, int64_t ldx, const rwkv_half *ry,
                       const rwkv_half *my, rwkv_half *xs, float *s0, float *s2, hipStream_t st) {
    hipLaunchKernelGGL(mm8_prepare_kernel, dim3((unsigned)T), dim3(256), 0, st, (int)T, (int)N, x, ldx, ry, my, xs, s0, s2);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}


// n (2..4) products [T, N] x [N, M_i] of uint8 or fp16 weights with their own inputs, outputs and epilogues in one
// launch.  uint8 with xs != NULL: x[i] is the unscaled activation and xs[i] / sums[i] (2 T floats) are scratch;
// uint8 with xs == NULL: x[i] is already scaled by ry and sums[i] holds its row sums -- as 2 T totals, or with
// parts > 1 (a multiple of four; direct-to-LDS launches only, see gemm_group_plan) as 2 T floats of scratch
// followed by [T][parts] partial sums of x and [T][parts] of x * my, which the launch adds up in index order.
// Operands laid out for 16-byte loads: the direct-to-LDS kernel, tile size and K split (over splitk_ws,
// RWKV_SPLITK_WS_BYTES of scratch, or NULL) from the cost model; otherwise register-staged 128 x 128 tiles at full depth.
static TilePick group_tile(bool w_u8, int n, int64_t T, int64_t N, const rwkv_mat *const *mats, bool may_split) {
    int64_t outs[4];
    bool m8 = true;
    for (int i = 0; i < n; ++i) {
        outs[i] = mats[i]->M;
        m8 = m8 && !(mats[i]->M & 7);
    }
    return Launch(T, (int)(N / BK), n, outs, may_split && m8 ? RWKV_SPLITK_WS_BYTES : 0).best(w_u8);
}
GemmPlan gemm_group_plan(bool w_u8, int n, int64_t T, int64_t N, const rwkv_half *const *x, const rwkv_mat *const *mats,
                         void *const *Y, bool may_split) {
    GemmPlan p{1, 0, 0, 1, 0.0};
    if (n < 2 || n > 4 || (N % BK)) return p;
    const float one = 0.f;
    bool skinny = true;
    for (int i = 0; i < n; ++i) {
        GemmEpi e{};
        if (w_u8) { e.mx = mats[i]->mx; e.rx = mats[i]->rx; e.s0 = &one; e.s2 = &one; }
        e.out_dtype = RWKV_DT_F16;
        if (mats[i]->N != N || !dma_ok(w_u8, N, mats[i]->M, x[i], N, mats[i]->w, mats[i]->ld, Y[i], mats[i]->M, e)) return p;
        skinny = skinny && skinny_ok(w_u8, T, N, x[i], N, mats[i]->w, mats[i]->ld, e);
    }
    if (skinny) { p.kind = 0; return p; }
    const TilePick t = group_tile(w_u8, n, T, N, mats, may_split);
    return GemmPlan{2, tile_dim[t.tile].tm, tile_dim[t.tile].tn, t.ks, t.us};
}
bool gemm_group_pays(bool w_u8, int n, int64_t T, int64_t N, const rwkv_half *const *x, const rwkv_mat *const *mats,
                     void *const *Y, const GemmEpi *eps, float *splitk_ws) {
    const GemmPlan g = gemm_group_plan(w_u8, n, T, N, x, mats, Y, splitk_ws != nullptr);
    if (g.kind != 2) return false;
    const float one = 0.f;
    double us = 0.0;
    for (int i = 0; i < n; ++i) {
        GemmEpi e = eps[i];
        e.splitk_ws = splitk_ws; e.splitk_bytes = RWKV_SPLITK_WS_BYTES;
        if (w_u8) { e.mx = mats[i]->mx; e.rx = mats[i]->rx; e.s0 = &one; e.s2 = &one; }
        const GemmPlan p = gemm_plan(w_u8, T, N, mats[i]->M, x[i], N, mats[i]->w, mats[i]->ld, Y[i], mats[i]->M, e);
        if (p.kind != 2) return false;
        us += p.us;
    }
    return g.us < us;
}

int gemm_group_launch(bool w_u8, int n, int64_t T, int64_t N, const rwkv_half *const *x, const rwkv_mat *const *mats,
                      void *const *Y, const GemmEpi *eps, rwkv_half *const *xs, float *const *sums, float *splitk_ws,
                      hipStream_t st, int parts) {
    if (n < 2 || n > 4 || (N % BK)) return RWKV_E_SHAPE;
    if (parts > 1 && (xs || !w_u8 || (parts & 3))) return RWKV_E_SHAPE;
    GemmGroup g{};
    g.lda = N;
    const bool prep = w_u8 && xs;
    if (prep) {
        PrepGroup p{};
        for (int i = 0; i < n; ++i) {
            p.x[i] = x[i]; p.ry[i] = mats[i]->ry; p.my[i] = mats[i]->my; p.xs[i] = xs[i]; p.s0[i] = sums[i]; p.s2[i] = sums[i] + T;
        }
        hipLaunchKernelGGL(mm8_prepare_group_kernel, dim3((unsigned)((T + 3) / 4), (unsigned)n), dim3(256), 0, st, (int)T, (int)N, p);
    }
    int64_t tiles = 0, max_out = 0;   // tiles: register-staged fallback
    bool dma = true;
    for (int i = 0; i < n; ++i) {
        if (mats[i]->N != N) return RWKV_E_SHAPE;
        g.m[i].A = (const h16 *)(prep ? xs[i] : x[i]);
        g.m[i].W = mats[i]->w; g.m[i].ldw = mats[i]->ld; g.m[i].Y = Y[i]; g.m[i].ldy = mats[i]->M; g.m[i].M = (int)mats[i]->M;
        g.m[i].ep = eps[i];
        g.m[i].ep.ldres = g.m[i].ep.ldgate = mats[i]->M;
        if (w_u8) { g.m[i].ep.mx = mats[i]->mx; g.m[i].ep.rx = mats[i]->rx; g.m[i].ep.s0 = sums[i]; g.m[i].ep.s2 = sums[i] + T; }
        if (parts > 1) { g.m[i].ep.parts = parts; g.m[i].ep.p0 = sums[i] + 2 * T; g.m[i].ep.p2 = sums[i] + 2 * T + (size_t)T * parts; }
        tiles = std::max<int64_t>(tiles, ((T + 127) / 128) * ((mats[i]->M + 127) / 128));
        max_out = std::max<int64_t>(max_out, T * mats[i]->M);
        dma = dma && dma_ok(w_u8, N, mats[i]->M, g.m[i].A, N, g.m[i].W, g.m[i].ldw, g.m[i].Y, mats[i]->M, g.m[i].ep);
    }
    {
        bool skinny = true;
        for (int i = 0; i < n; ++i) skinny = skinny && skinny_ok(w_u8, T, N, g.m[i].A, N, g.m[i].W, g.m[i].ldw, g.m[i].ep);
        if (skinny) {
            if (parts > 1) return RWKV_E_LAYOUT;
            SkinnyGroup sg{};
            sg.lda = N;
            for (int i = 0; i < n; ++i) {
                sg.m[i].A = g.m[i].A; sg.m[i].W = g.m[i].W; sg.m[i].Y = g.m[i].Y; sg.m[i].ldw = g.m[i].ldw; sg.m[i].ldy = g.m[i].M; sg.m[i].M = g.m[i].M;
                sg.m[i].ep = g.m[i].ep;
            }
            return skinny_launch(w_u8, n, T, N, sg, st);
        }
    }
    if (dma) {
        // tile and K split of least cost, as for a single product
        const TilePick pick = group_tile(w_u8, n, T, N, mats, splitk_ws != nullptr);
        const int ks = pick.ks;
        g.nk_split = (int)(N / BK) / ks;
        if (ks > 1) {
            float *p = splitk_ws;
            for (int i = 0; i < n; ++i) { g.m[i].part = p; p += (size_t)ks * T * mats[i]->M; }
        }
        const int rc = w_u8 ? launch_tile<true>(pick.tile, g, n, T, N, ks, st) : launch_tile<false>(pick.tile, g, n, T, N, ks, st);
        if (rc) return rc;
        if (ks > 1) {
            SplitFactors rows{};
            for (int i = 0; i < n; ++i) rows.f[i] = div_factor(g.m[i].M / 8);
            hipLaunchKernelGGL(splitk_group_epilogue8_kernel, dim3((unsigned)((max_out + 2047) / 2048), (unsigned)n), dim3(256), 0, st, (int)T, ks, rows,
                               (const GemmMembers &)g);
        }
        RWKV_LAUNCH_CHECK();
        return RWKV_OK;
    }
    if (parts > 1 || !w_u8) return RWKV_E_LAYOUT;   // partial sums only through the direct-to-LDS kernel; fp16 operands all pass dma_ok
    constexpr size_t lds = 2 * (size_t)(128 + 128) * BK * sizeof(h16);
    const dim3 grid((unsigned)tiles, (unsigned)n);
    hipLaunchKernelGGL(gemm_group_kernel, grid, dim3(256), lds, st, (int)T, (int)N, g);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

extern "C" size_t rwkv_mm8_seq_workspace(int64_t B, int64_t N) {
    if (B <= 0 || N <= 0) return 0;
    return (((size_t)B * N * 2 + 255) & ~(size_t)255) + (((size_t)B * 8 + 255) & ~(size_t)255) + RWKV_SPLITK_WS_BYTES;
}

// rwkv_mm8_seq_f16 in its two launches: the activation-scaling pass (`reps` < 0), the contraction alone `reps`
// times on the already scaled rows (`reps` > 0), or one of each (`reps` == 0: the product)
static int mm8_seq_parts(int64_t B, int64_t N, int64_t M, const rwkv_half *x, int64_t x_stride, const uint8_t *w,
                         int64_t w_stride_n, int64_t w_stride_m, const rwkv_half *mx, const rwkv_half *rx,
                         const rwkv_half *my, const rwkv_half *ry, rwkv_half *y, int64_t y_stride, void *workspace,
                         size_t workspace_bytes, hipStream_t st, int reps) {
    if (!x || !w || !mx || !rx || !my || !ry || !y || !workspace) return RWKV_E_NULL;
    if (B <= 0 || N <= 0 || M <= 0 || (N % BK) != 0 || B > (1 << 24) || M > (1 << 24)) return RWKV_E_SHAPE;
    if (w_stride_n != 1 || w_stride_m < N || (w_stride_m & 15) || !aligned16(w)) return RWKV_E_LAYOUT;
    if (x_stride < N || (x_stride & 7) || !aligned16(x) || y_stride < M || !aligned16(my) || !aligned16(ry))
        return RWKV_E_LAYOUT;
    if (workspace_bytes < rwkv_mm8_seq_workspace(B, N) || !aligned16(workspace)) return RWKV_E_WORKSPACE;
    rwkv_half *xs = (rwkv_half *)workspace;
    const size_t xs_bytes = ((size_t)B * N * 2 + 255) & ~(size_t)255;
    float *s0 = (float *)((unsigned char *)workspace + xs_bytes);
    float *s2 = s0 + B;
    if (reps <= 0) {
        int rc = mm8_prepare_launch(B, N, x, x_stride, ry, my, xs, s0, s2, st);
        if (rc || reps < 0) return rc;
    }
    GemmEpi ep{};
    ep.mx = mx; ep.rx = rx; ep.s0 = s0; ep.s2 = s2; ep.act = ACT_NONE; ep.out_scale = 1.f; ep.out_dtype = RWKV_DT_F16;
    ep.splitk_ws = (float *)((unsigned char *)workspace + xs_bytes + (((size_t)B * 8 + 255) & ~(size_t)255));
    ep.splitk_bytes = RWKV_SPLITK_WS_BYTES;
    int rc = RWKV_OK;
    for (int r = 0; r < (reps > 0 ? reps : 1) && rc == RWKV_OK; ++r)
        rc = gemm_launch(true, B, N, M, xs, N, w, w_stride_m, y, y_stride, ep, st);
    return rc;
}

extern "C" int rwkv_mm8_seq_f16(int64_t B, int64_t N, int64_t M, const rwkv_half *x, int64_t x_stride,
                                const uint8_t *w, int64_t w_stride_n, int64_t w_stride_m, const rwkv_half *mx,
                                const rwkv_half *rx, const rwkv_half *my, const rwkv_half *ry, rwkv_half *y,
                                int64_t y_stride, void *workspace, size_t workspace_bytes, void *stream) {
    return mm8_seq_parts(B, N, M, x, x_stride, w, w_stride_n, w_stride_m, mx, rx, my, ry, y, y_stride, workspace,
                         workspace_bytes, (hipStream_t)stream, 0);
}

extern "C" int rwkv_mm8_seq_time_kernel(int64_t B, int64_t N, int64_t M, const rwkv_half *x, int64_t x_stride,
                                        const uint8_t *w, int64_t w_stride_n, int64_t w_stride_m,
                                        const rwkv_half *mx, const rwkv_half *rx, const rwkv_half *my,
                                        const rwkv_half *ry, rwkv_half *y, int64_t y_stride, void *workspace,
                                        size_t workspace_bytes, void *stream, int reps, float *ms_per_launch) {
    if (!ms_per_launch) return RWKV_E_NULL;
    if (reps <= 0) return RWKV_E_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    int rc = mm8_seq_parts(B, N, M, x, x_stride, w, w_stride_n, w_stride_m, mx, rx, my, ry, y, y_stride, workspace,
                           workspace_bytes, st, -1);
    if (rc) return rc;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return (int)hipErrorOutOfMemory;
    if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); return (int)hipErrorOutOfMemory; }
    (void)hipEventRecord(e0, st);
    rc = mm8_seq_parts(B, N, M, x, x_stride, w, w_stride_n, w_stride_m, mx, rx, my, ry, y, y_stride, workspace,
                       workspace_bytes, st, reps);
    (void)hipEventRecord(e1, st);
    hipError_t e = hipEventSynchronize(e1);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e != hipSuccess && rc == RWKV_OK) rc = (int)e;
    *ms_per_launch = ms / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

// ---- rwkv_mm8_seq_f16 without a caller workspace ------------------------------------------------------------
// The scratch of the product (the ry-scaled copy of x, its two row sums, split-K slabs) in a file-scope device
// array instead of a workspace argument.  The array's name is only a host-side handle: the device address of each
// GPU's copy comes from hipGetSymbolAddress, once per device, and that pointer is what the kernels get.
constexpr size_t STATIC_XS_BYTES = (size_t)8 << 20;       // B * N <= 4 Mi elements
constexpr size_t STATIC_SUMS_BYTES = (size_t)64 << 10;    // B <= 8192
constexpr size_t STATIC_SPLITK_BYTES = (size_t)16 << 20;  // the K split is limited to slabs that fit here
constexpr size_t STATIC_SCRATCH_BYTES = STATIC_XS_BYTES + STATIC_SUMS_BYTES + STATIC_SPLITK_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int STATIC_MAX_DEVICES = 64;
static void *g_scratch_ptr[STATIC_MAX_DEVICES];
static std::mutex g_scratch_mutex;

// device address of the current device's copy of `scratch` (looked up on the first call on that device)
static int static_scratch(unsigned char **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= STATIC_MAX_DEVICES) return RWKV_E_SHAPE;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return RWKV_E_NULL;
        g_scratch_ptr[dev] = p;
    }
    *out = (unsigned char *)g_scratch_ptr[dev];
    return RWKV_OK;
}

extern "C" size_t rwkv_mm8_seq_static_max_elems(void) { return STATIC_XS_BYTES / 2; }
extern "C" size_t rwkv_mm8_seq_static_max_rows(void) { return STATIC_SUMS_BYTES / 8; }

extern "C" int rwkv_mm8_seq_f16_static(int64_t B, int64_t N, int64_t M, const rwkv_half *x, int64_t x_stride,
                                       const uint8_t *w, int64_t w_stride_n, int64_t w_stride_m, const rwkv_half *mx,
                                       const rwkv_half *rx, const rwkv_half *my, const rwkv_half *ry, rwkv_half *y,
                                       int64_t y_stride, void *stream) {
    if (!x || !w || !mx || !rx || !my || !ry || !y) return RWKV_E_NULL;
    if (B <= 0 || N <= 0 || M <= 0 || (N % BK) != 0 || B > (1 << 24) || M > (1 << 24)) return RWKV_E_SHAPE;
    if (w_stride_n != 1 || w_stride_m < N || (w_stride_m & 15) || !aligned16(w)) return RWKV_E_LAYOUT;
    if (x_stride < N || (x_stride & 7) || !aligned16(x) || y_stride < M || !aligned16(my) || !aligned16(ry))
        return RWKV_E_LAYOUT;
    if ((size_t)B * (size_t)N * 2 > STATIC_XS_BYTES || (size_t)B * 8 > STATIC_SUMS_BYTES) return RWKV_E_SCRATCH;
    unsigned char *base = nullptr;
    int rc = static_scratch(&base);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    rwkv_half *xs = (rwkv_half *)base;
    float *s0 = (float *)(base + STATIC_XS_BYTES);
    float *s2 = s0 + B;
    // every row of xs / s0 / s2 and every slab element the product reads is written by this call first:
    // nothing in the array has to start at zero
    rc = mm8_prepare_launch(B, N, x, x_stride, ry, my, xs, s0, s2, st);
    if (rc) return rc;
    GemmEpi ep{};
    ep.mx = mx; ep.rx = rx; ep.s0 = s0; ep.s2 = s2; ep.act = ACT_NONE; ep.out_scale = 1.f; ep.out_dtype = RWKV_DT_F16;
    ep.splitk_ws = (float *)(base + STATIC_XS_BYTES + STATIC_SUMS_BYTES);
    ep.splitk_bytes = STATIC_SPLITK_BYTES;
    return gemm_launch(true, B, N, M, xs, N, w, w_stride_m, y, y_stride, ep, st);
}

extern "C" int rwkv_gemm_f16(int64_t B, int64_t N, int64_t M, const rwkv_half *a, int64_t a_stride,
                             const rwkv_half *b, int64_t b_stride_n, int64_t b_stride_m, void *c, int64_t c_stride,
                             int c_dtype, void *stream) {
    if (!a || !b || !c) return RWKV_E_NULL;
    if (B <= 0 || N <= 0 || M <= 0 || (N & 7) || B > (1 << 24) || M > (1 << 24)) return RWKV_E_SHAPE;
    if (c_dtype != RWKV_DT_F16 && c_dtype != RWKV_DT_F32) return RWKV_E_DTYPE;
    if (b_stride_n != 1 || b_stride_m < N || (b_stride_m & 7) || !aligned16(b)) return RWKV_E_LAYOUT;
    if (a_stride < N || (a_stride & 7) || !aligned16(a) || c_stride < M) return RWKV_E_LAYOUT;
    hipStream_t st = (hipStream_t)stream;
    if (B == 1) {
        if (N > 32768) return RWKV_E_SHAPE;
        return gemv_f16_launch(N, M, a, b, b_stride_m, c, c_dtype, st);
    }
    if (N % BK) return RWKV_E_SHAPE;
    GemmEpi ep{};
    ep.act = ACT_NONE; ep.out_scale = 1.f; ep.out_dtype = c_dtype; ep.raw_f32 = (c_dtype == RWKV_DT_F32);
    return gemm_launch(false, B, N, M, a, a_stride, b, b_stride_m, c, c_stride, ep, st);
}

extern "C" int rwkv_gemm_f16_batched(int64_t batch, int64_t B, int64_t N, int64_t M, const rwkv_half *a, int64_t a_stride,
                                     int64_t a_batch_stride, const rwkv_half *b, int64_t b_stride_n, int64_t b_stride_m,
                                     int64_t b_batch_stride, void *c, int64_t c_stride, int64_t c_batch_stride, int c_dtype,
                                     void *stream) {
    if (batch <= 0 || batch > (1 << 20)) return RWKV_E_SHAPE;
    if (!a || !b || !c) return RWKV_E_NULL;
    if (c_dtype != RWKV_DT_F16 && c_dtype != RWKV_DT_F32) return RWKV_E_DTYPE;
    // every product of the batch must itself be acceptable: 16-byte aligned operands
    if ((a_batch_stride & 7) || (b_batch_stride & 7) || a_batch_stride < 0 || b_batch_stride < 0 || c_batch_stride < 0)
        return RWKV_E_LAYOUT;
    const size_t csz = c_dtype == RWKV_DT_F16 ? 2 : 4;
    for (int64_t i = 0; i < batch; ++i) {
        const int rc = rwkv_gemm_f16(B, N, M, a + i * a_batch_stride, a_stride, b + i * b_batch_stride, b_stride_n, b_stride_m,
                                     (char *)c + (size_t)(i * c_batch_stride) * csz, c_stride, c_dtype, stream);
        if (rc) return rc;
    }
    return RWKV_OK;
}
