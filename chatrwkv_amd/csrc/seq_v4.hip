// RWKV-4 sequence mode (len(tokens) > 1): per layer
//   lnmix_seq (LN1, token shift, k/v/r mixes, ry scaling, row sums) -> 3 MFMA GEMMs (sigmoid fused for r)
//   -> WKV-4 over T (r gating fused) -> GEMM Wo (+ residual)
//   lnmix_seq (LN2, ...) -> GEMM Wr (sigmoid), GEMM Wk (relu^2) -> GEMM Wv (gate, residual, /2)
// With uint8 weights a scaling pass (mm8_prepare) sits in front of Wo; the input of Wv arrives scaled by that
// matrix's ry, with partial row sums, from the epilogue of the Wk product (long calls through the direct-to-LDS
// kernel; otherwise it has a scaling pass too).
// and LN_out + head on the last row (GEMV) or on every row (GEMM) for full_output.
#include <algorithm>
#include <cstdlib>
#include <mutex>
#include "kernels.h"
#include "rows.h"

namespace {

// ids outside [0, vocab) are clamped to the nearest valid row: a bad id never becomes an out-of-bounds read
__global__ __launch_bounds__(256) void gather_emb_kernel(int T, int C, int vocab, const int32_t *__restrict__ tokens,
                                                         const rwkv_half *__restrict__ emb,
                                                         rwkv_half *__restrict__ x) {
    const int t = blockIdx.x;
    const u32x4 *src = (const u32x4 *)(emb + (size_t)min(max(tokens[t], 0), vocab - 1) * C);
    u32x4 *dst = (u32x4 *)(x + (size_t)t * C);
    for (int i = threadIdx.x; i < (C >> 3); i += blockDim.x) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void copy16_kernel(int n16, const u32x4 *__restrict__ src, u32x4 *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n16) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void ln_f32_f16_kernel(int C, const float *__restrict__ x_, const float *__restrict__ w,
                                                         const float *__restrict__ b, rwkv_half *__restrict__ y_) {
    __shared__ float red[4];
    const float *x = x_ + (size_t)blockIdx.x * C;
    rwkv_half *y = y_ + (size_t)blockIdx.x * C;
    float s = 0.f;
    for (int j = threadIdx.x; j < C; j += blockDim.x) s += x[j];
    const float mean = block_sum(s, red) / C;
    float q = 0.f;
    for (int j = threadIdx.x; j < C; j += blockDim.x) { const float d = x[j] - mean; q += d * d; }
    const float rstd = rsqrtf(block_sum(q, red) / C + LN_EPS);
    for (int j = threadIdx.x; j < C; j += blockDim.x) y[j] = f2h((x[j] - mean) * rstd * w[j] + b[j]);
}

// LayerNorm, token shift and mixes of a row of C <= 8 NT CH channels, one workgroup per row.  Row t needs LN(x[t-1]) for the token
// shift: it is recomputed here from x[t-1] (same code, same data => same bits as row t-1 computes for itself), which keeps all
// rows independent.  A thread's chunks of the row, of the previous row and of the LayerNorm vectors are requested together at the
// top and kept in registers, the statistics of the two rows share their barriers, and so do the 2 NJ sums at the end: two global
// round trips and three rounds of barriers.  256 threads per row and 512 form every value with the same operations in the same
// order (row_sums), so both agree bit for bit.
// The first chunk's mix and scale vectors are requested at the top too, together, and the next chunk's ahead of this one's stores: a wait for a
// load is one for every older store as well.  Requested mix by mix they were two trips to memory and a store's way there for each mix, one
// after the other.
// Q: some of the mixes are scaled and summed.
template <int NJ, int CH, int NT, bool Q>
__global__ __launch_bounds__(NT) void lnmix_seq_fast_kernel(const rwkv_half *x0, const rwkv_half *ln_w, const rwkv_half *ln_b, const rwkv_half *sx,
                                                            rwkv_half *state_out, int C, int T, SeqMixArgs a) {
    constexpr int NSUM = 2 * NJ > 3 ? 2 * NJ : 3;
    __shared__ __align__(16) float red[24 + 8 * NJ];
    __shared__ float hop[NT == 512 ? 256 * NSUM : 1];
    const int t = blockIdx.x, nch = C >> 3;
    // this thread's chunk c: tid + 256 c, or with 512 threads the first CH and the last CH of a chain's 2 CH
    const int j8_0 = NT == 256 ? (int)threadIdx.x : (int)(threadIdx.x & 255) + 256 * CH * (int)(threadIdx.x >> 8);
    const rwkv_half *x = x0 + (size_t)t * C;
    const bool shift = sx != nullptr, prev_row = shift && t > 0;
    const rwkv_half *xp = prev_row ? x - C : x;
    // Row 0's workgroup also forms the new token-shift state LN(x[T-1]): its statistics ride in the same barriers
    const bool commit = state_out && t == 0;
    const rwkv_half *xl = commit ? x0 + (size_t)(T - 1) * C : x;
    h16x8 xv[CH], pxv[CH], lv[CH], wv[CH], bv[CH], mv[NJ], rv[Q ? NJ : 1], yv[Q ? NJ : 1];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int j8 = min(j8_0 + c * 256, nch - 1);   // chunks past the end repeat the last one (unused)
        xv[c] = *(const h16x8 *)(x + 8 * j8);
        pxv[c] = *(const h16x8 *)(xp + 8 * j8);
        lv[c] = *(const h16x8 *)(xl + 8 * j8);
        wv[c] = *(const h16x8 *)(ln_w + 8 * j8);
        bv[c] = *(const h16x8 *)(ln_b + 8 * j8);
    }
    const void *vec[3 * NJ];   // mix, ry, my
#pragma unroll
    for (int j = 0; j < NJ; ++j) { vec[3 * j] = a.mix[j]; vec[3 * j + 1] = a.ry[j]; vec[3 * j + 2] = a.my[j]; }
    auto request = [&](int c) {
        const int j8 = min(j8_0 + c * 256, nch - 1);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            mv[j] = load8(vec[3 * j] ? vec[3 * j] : ln_w, j8);
            if constexpr (Q) {
                rv[j] = load8(vec[3 * j + 1] ? vec[3 * j + 1] : ln_w, j8);
                yv[j] = load8(vec[3 * j + 1] ? vec[3 * j + 2] : ln_w, j8);
            }
        }
    };
    if constexpr (NJ <= 4) at_once(vec);
    request(0);
    float st[3] = {0.f, 0.f, 0.f};
    row_sums<3, NT>(st, red, hop, [&](float (&v)[3], auto) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if (j8_0 + c * 256 < nch) {
                v[0] = sum8(xv[c], v[0]);
                v[1] = sum8(pxv[c], v[1]);
                v[2] = sum8(lv[c], v[2]);
            }
    });
    const float mean = row_mean(st[0], C), pmean = row_mean(st[1], C), lmean = row_mean(st[2], C);
    float dx[CH][8], dp[CH][8];
    st[0] = st[1] = st[2] = 0.f;
    row_sums<3, NT>(st, red + 12, hop, [&](float (&v)[3], auto first) {
        constexpr bool FIRST = decltype(first)::value;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            less_mean8(xv[c], mean, dx[c]);
            less_mean8(pxv[c], pmean, dp[c]);
            if (j8_0 + c * 256 < nch) {
                v[0] = FIRST && c == 0 ? squares8<true>(dx[c], v[0]) : squares8<false>(dx[c], v[0]);
                v[1] = FIRST && c == 0 ? squares8<true>(dp[c], v[1]) : squares8<false>(dp[c], v[1]);
                if (commit) {   // the last row's statistics: only the workgroup that writes the new state needs them
                    float dl[8];
                    less_mean8(lv[c], lmean, dl);
                    v[2] = FIRST && c == 0 ? squares8<true>(dl, v[2]) : squares8<false>(dl, v[2]);
                }
            }
        }
    });
    const float rstd = row_rstd(st[0], C), prstd = row_rstd(st[1], C), lrstd = row_rstd(st[2], C);
    float acc[2 * NJ];
#pragma unroll
    for (int i = 0; i < 2 * NJ; ++i) acc[i] = 0.f;
    auto add_mix = [](float (&v)[2 * NJ], int j, h16x8 kx, h16x8 y8) {
        v[2 * j] = sum8(kx, v[2 * j]);
        v[2 * j + 1] = dot8(kx, y8, v[2 * j + 1]);
    };
    h16x8 kv[CH][NJ], sv[CH][NJ];   // 512 threads: the mixes and their my, added up when the first half's sums are there
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int j8 = j8_0 + c * 256;
        if (j8 >= nch) break;
        if (NT == 512) {   // a thread of one half has skipped the other half's sums
            less_mean8(xv[c], mean, dx[c]);
            less_mean8(pxv[c], pmean, dp[c]);
        }
        const h16x8 xx = norm8(dx[c], rstd, wv[c], bv[c]);
        h16x8 pv = xx;
        if (shift) {
            if (t > 0) pv = norm8(dp[c], prstd, wv[c], bv[c]);
            else pv = *(const h16x8 *)(sx + 8 * j8);
        }
        if (a.xx_last && t == T - 1) *(h16x8 *)(a.xx_last + 8 * j8) = xx;
        h16x8 o[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const h16x8 kx = vec[3 * j] ? mix8(xx, pv, mv[j], a.maa_form) : xx;
            o[j] = kx;
            if (Q && vec[3 * j + 1]) {
                o[j] = kx * rv[j];
                if constexpr (NT == 256) add_mix(acc, j, kx, yv[j]);
                else { kv[c][j] = kx; sv[c][j] = yv[j]; }
            }
        }
        if (c + 1 < CH) request(c + 1);
#pragma unroll
        for (int j = 0; j < NJ; ++j) *(h16x8 *)(a.xs[j] + (size_t)t * C + 8 * j8) = o[j];
        // Only row 0 reads the old state, so row 0's workgroup writes the new one, each thread exactly the chunk it
        // has just read: no second launch.
        if (commit) {
            float dl[8];
            less_mean8(lv[c], lmean, dl);
            *(h16x8 *)(state_out + 8 * j8) = norm8(dl, lrstd, wv[c], bv[c]);
        }
    }
    if constexpr (Q) {
        row_sums<2 * NJ, NT>(acc, red + 24, hop, [&](float (&v)[2 * NJ], auto) {
            if constexpr (NT > 256)
#pragma unroll
                for (int c = 0; c < CH; ++c)
                    if (j8_0 + c * 256 < nch)
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
                            if (vec[3 * j + 1]) add_mix(v, j, kv[c][j], sv[c][j]);
        });
        if (threadIdx.x == 0)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                if (vec[3 * j + 1]) { a.s0[j][t] = acc[2 * j]; a.s2[j][t] = acc[2 * j + 1]; }
    }
}

}  // namespace

template <int CH, int NT, bool Q>
static bool lnmix_seq_fast_launch(const SeqMixArgs &a, int nj, hipStream_t st) {
    const dim3 grid((unsigned)a.T), block(NT);
    switch (nj) {
        case 1: hipLaunchKernelGGL((lnmix_seq_fast_kernel<1, CH, NT, Q>), grid, block, 0, st, a.x, a.ln_w, a.ln_b, a.sx, a.state_out, a.C, a.T, a); break;
        case 2: hipLaunchKernelGGL((lnmix_seq_fast_kernel<2, CH, NT, Q>), grid, block, 0, st, a.x, a.ln_w, a.ln_b, a.sx, a.state_out, a.C, a.T, a); break;
        case 3: hipLaunchKernelGGL((lnmix_seq_fast_kernel<3, CH, NT, Q>), grid, block, 0, st, a.x, a.ln_w, a.ln_b, a.sx, a.state_out, a.C, a.T, a); break;
        case 4: hipLaunchKernelGGL((lnmix_seq_fast_kernel<4, CH, NT, Q>), grid, block, 0, st, a.x, a.ln_w, a.ln_b, a.sx, a.state_out, a.C, a.T, a); break;
        case 6: hipLaunchKernelGGL((lnmix_seq_fast_kernel<6, CH, NT, Q>), grid, block, 0, st, a.x, a.ln_w, a.ln_b, a.sx, a.state_out, a.C, a.T, a); break;
        default: return false;
    }
    return true;
}

template <bool Q>
static bool lnmix_seq_fast_width(const SeqMixArgs &a, int nj, hipStream_t st) {
    const bool few = a.T <= 512;
    if (a.C <= 2048) return lnmix_seq_fast_launch<1, 256, Q>(a, nj, st);
    if (a.C <= 4096) return few ? lnmix_seq_fast_launch<1, 512, Q>(a, nj, st) : lnmix_seq_fast_launch<2, 256, Q>(a, nj, st);
    return few ? lnmix_seq_fast_launch<2, 512, Q>(a, nj, st) : lnmix_seq_fast_launch<4, 256, Q>(a, nj, st);
}

int lnmix_seq_launch(const SeqMixArgs &a, int nj, hipStream_t st) {
    // A chain of additions has 1, 2 or 4 chunks of 8 channels (every model has at most 8192).
    // Calls of up to 512 rows have one or two rows per CU: there a row's own chain of barriers and instructions is the time,
    // so rows of more than 2048 channels get 512 threads instead of 256, with the same sums (row_sums).  4096 channels, us,
    // 256 -> 512 threads at 45 / 256 / 512 / 600 / 1024 rows: one mix 4.2 -> 3.4, 4.4 -> 3.6, 4.7 -> 4.8, 5.4 -> 5.7, 6.6 -> 7.1;
    // three mixes with scaling 6.7 -> 5.4, 7.4 -> 6.1, 8.4 -> 7.9, 9.4 -> 10.4, 11.7 -> 12.6; six mixes without 6.7 -> 5.5, 8.0 ->
    // 6.8, 9.1 -> 8.5, 10.0 -> 11.7, 12.8 -> 14.5 (5120 channels, three mixes: 512 rows 10.6 -> 10.2, 600 rows 11.8 -> 14.6).
    // These are launches one after the other on the same rows.  Within a call, whose products have used the caches since, us
    // before the element code of rows.h was written out (three to four instructions per step) and now: three scaled mixes of 4096
    // channels at 45 / 1024 rows 7.3 / 20.5 -> 5.9 / 16.1, two 6.3 / 16.5 -> 5.6 / 12.7; at 777 rows six 20.3 -> 16.7, one 9.5 ->
    // 7.0; four of 2048 channels at 333 rows 7.1 -> 5.3; three of 768 at 513 rows 6.7 -> 4.9.  With the vectors requested together, before ->
    // now: three scaled mixes of 4096 channels at 1024 / 2048 rows 16.5 / 26.3 -> 14.5 / 22.3, of 5120 at 1024 26.2 -> 21.7; six of 4096 at 300 / 777 /
    // 2048 9.7 / 16.9 / 30.2 -> 8.0 / 12.2 / 23.3; two scaled ones of 768 at 300 5.3 -> 4.5.  An empty launch is 3.2; at 1024 rows
    // it is the 130 KB per row through a CU's L1 and the 24 MB of stores.
    // Several rows per workgroup, sharing vectors and the previous row's statistics, measured with the element code before: slower
    // at every length (1024 rows 21.8 with two, 33 with four, 20.7 with one).
    if (a.C > 8192) return RWKV_E_SHAPE;
    bool scaled = false;
    for (int j = 0; j < nj; ++j) scaled = scaled || a.ry[j];
    if (!(scaled ? lnmix_seq_fast_width<true>(a, nj, st) : lnmix_seq_fast_width<false>(a, nj, st))) return RWKV_E_SHAPE;
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

int gather_emb_launch(int64_t T, int C, int vocab, const int32_t *tokens, const rwkv_half *emb, rwkv_half *x, hipStream_t st) {
    hipLaunchKernelGGL(gather_emb_kernel, dim3((unsigned)T), dim3(256), 0, st, (int)T, C, vocab, tokens, emb, x);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

int copy_h16_launch(int n, const rwkv_half *src, rwkv_half *dst, hipStream_t st) {
    const int n16 = n >> 3;
    hipLaunchKernelGGL(copy16_kernel, dim3((n16 + 255) / 256), dim3(256), 0, st, n16, (const u32x4 *)src, (u32x4 *)dst);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

namespace {

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct SeqWs {
    rwkv_half *x, *xs[3], *r, *rwkv, *vx, *xsv, *xx_att, *xx_ffn;
    void *k, *v;       // fp16 (uint8 weights) or fp32 (fp16 weights)
    float *sums;       // 8 * T floats
    float *parts;      // partial row sums handed from one product's epilogue to the next product: 2 * T * PARTS_MAX floats
    float *splitk;     // RWKV_SPLITK_WS_BYTES of split-K scratch for the contraction kernel
    float *wkv;        // chunk summaries of the WKV scan
    size_t total;
};

// most partial sums a row can have
int64_t parts_max(int64_t F) { return emitted_parts((int)F, EMIT_MIN_TN); }

SeqWs carve(void *base, int64_t T, int64_t C, int64_t F) {
    SeqWs w;
    unsigned char *p = (unsigned char *)base;
    auto take = [&](size_t bytes) { void *q = p; p += align256(bytes); return q; };
    const size_t tc = (size_t)T * C * 2, tf = (size_t)T * F * 2;
    w.x = (rwkv_half *)take(tc);
    for (int j = 0; j < 3; ++j) w.xs[j] = (rwkv_half *)take(tc);
    w.r = (rwkv_half *)take(tc);
    w.rwkv = (rwkv_half *)take(tc);
    w.k = take(2 * tc);
    w.v = take(2 * tc);
    w.vx = (rwkv_half *)take(tf);
    w.xsv = (rwkv_half *)take(tf);
    w.xx_att = (rwkv_half *)take((size_t)C * 2);
    w.xx_ffn = (rwkv_half *)take((size_t)C * 2);
    w.sums = (float *)take((size_t)T * 8 * sizeof(float));
    w.parts = (float *)take((size_t)T * 2 * parts_max(F) * sizeof(float));
    w.splitk = (float *)take(RWKV_SPLITK_WS_BYTES);
    w.wkv = (float *)take(wkv4_scratch_bytes(T, C));
    w.total = (size_t)(p - (unsigned char *)base);
    return w;
}

int run_gemm(const rwkv_mat &m, bool u8, int64_t T, const rwkv_half *A, const float *s0, const float *s2, void *Y,
             int64_t ldy, GemmEpi ep, hipStream_t st, float *splitk) {
    ep.splitk_ws = splitk;
    ep.splitk_bytes = RWKV_SPLITK_WS_BYTES;
    ep.mx = u8 ? m.mx : nullptr;
    ep.rx = u8 ? m.rx : nullptr;
    ep.s0 = s0;
    ep.s2 = s2;
    return gemm_launch(u8, T, m.N, m.M, A, m.N, m.w, m.ld, Y, ldy, ep, st);
}

// how run_gemm with the same arguments would be launched
GemmPlan plan_gemm(const rwkv_mat &m, bool u8, int64_t T, const rwkv_half *A, const float *s0, const float *s2, const void *Y,
                   int64_t ldy, GemmEpi ep, float *splitk) {
    ep.splitk_ws = splitk;
    ep.splitk_bytes = RWKV_SPLITK_WS_BYTES;
    ep.mx = u8 ? m.mx : nullptr;
    ep.rx = u8 ? m.rx : nullptr;
    ep.s0 = s0;
    ep.s2 = s2;
    return gemm_plan(u8, T, m.N, m.M, A, m.N, m.w, m.ld, Y, ldy, ep);
}

// RWKV_HANDOVER=0 keeps the separate scaling passes (for A/B timing)
bool handover_enabled() {
    const char *e = getenv("RWKV_HANDOVER");
    return !(e && *e == '0');
}

// Two side streams (default priority) for contractions that are independent of each other and too small
// to fill the chip alone: k / v / r of the time mix and r / k of the channel mix run side by side.
}  // namespace

namespace {
// The table of side-stream sets: one per (device, caller stream) pair, at most 32 at a time.  A set whose caller
// stream has been given back (rwkv_release_stream) is taken over, with its streams and events, by the next new pair
// on the same device.
struct SideSlot { int dev; hipStream_t caller; bool bound; SideStreams ss; };
constexpr int MAX_SIDE_SLOTS = 32;
SideSlot g_side_slots[MAX_SIDE_SLOTS];
int g_n_side_slots = 0;
std::mutex g_side_mu;
}  // namespace

SideStreams *side_streams(hipStream_t caller) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_side_mu);
    SideSlot *spare = nullptr;
    for (int i = 0; i < g_n_side_slots; ++i) {
        SideSlot &sl = g_side_slots[i];
        if (sl.dev != dev) continue;
        if (sl.bound && sl.caller == caller) return sl.ss.ok ? &sl.ss : nullptr;
        if (!sl.bound && sl.ss.ok && !spare) spare = &sl;
    }
    if (spare) {
        spare->caller = caller;
        spare->bound = true;
        return &spare->ss;
    }
    if (g_n_side_slots == MAX_SIDE_SLOTS) return nullptr;   // more caller streams than slots: those run without side streams
    SideSlot &sl = g_side_slots[g_n_side_slots++];
    sl.dev = dev;
    sl.caller = caller;
    sl.bound = true;
    SideStreams &ss = sl.ss;
    ss.ok = hipStreamCreateWithFlags(&ss.s[0], hipStreamNonBlocking) == hipSuccess &&
            hipStreamCreateWithFlags(&ss.s[1], hipStreamNonBlocking) == hipSuccess &&
            hipEventCreateWithFlags(&ss.fork, hipEventDisableTiming) == hipSuccess &&
            hipEventCreateWithFlags(&ss.join[0], hipEventDisableTiming) == hipSuccess &&
            hipEventCreateWithFlags(&ss.join[1], hipEventDisableTiming) == hipSuccess;
    return ss.ok ? &ss : nullptr;
}

extern "C" int rwkv_release_stream(void *stream) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    std::lock_guard<std::mutex> lock(g_side_mu);
    for (int i = 0; i < g_n_side_slots; ++i) {
        SideSlot &sl = g_side_slots[i];
        if (sl.dev == dev && sl.bound && sl.caller == (hipStream_t)stream) {
            sl.bound = false;
            sl.caller = nullptr;
        }
    }
    return RWKV_OK;
}

// after fork, work launched on side stream j sees everything queued on `st` so far
bool fork_streams(SideStreams *ss, hipStream_t st, int n) {
    if (hipEventRecord(ss->fork, st) != hipSuccess) return false;
    for (int j = 0; j < n; ++j)
        if (hipStreamWaitEvent(ss->s[j], ss->fork, 0) != hipSuccess) return false;
    return true;
}

// after join, work launched on `st` sees everything queued on the side streams
bool join_streams(SideStreams *ss, hipStream_t st, int n) {
    for (int j = 0; j < n; ++j) {
        if (hipEventRecord(ss->join[j], ss->s[j]) != hipSuccess) return false;
        if (hipStreamWaitEvent(st, ss->join[j], 0) != hipSuccess) return false;
    }
    return true;
}

extern "C" int rwkv_layernorm_f32_f16(int64_t T, int64_t C, const float *x, const float *w, const float *b,
                                      rwkv_half *y, void *stream) {
    if (!x || !w || !b || !y) return RWKV_E_NULL;
    if (T <= 0 || C <= 0 || T > 0x7fffffff) return RWKV_E_SHAPE;
    hipLaunchKernelGGL(ln_f32_f16_kernel, dim3((unsigned)T), dim3(256), 0, (hipStream_t)stream, (int)C, x, w, b, y);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

extern "C" size_t rwkv_v4_seq_workspace(const rwkv_v4_model *m, int64_t T, int full_output) {
    if (!m || T <= 0) return 0;
    (void)full_output;
    return carve((void *)256, T, m->n_embd, m->n_ffn).total;
}

extern "C" int rwkv_v4_forward_seq(const rwkv_v4_model *m, const rwkv_v4_layer_state *states, const int32_t *tokens,
                                   int64_t T, int full_output, float *logits, void *workspace,
                                   size_t workspace_bytes, void *stream) {
    int rc = v4_model_check(m);
    if (rc) return rc;
    int lb, le;
    if (!layer_range(m->n_layer, m->layer_begin, m->layer_end, lb, le)) return RWKV_E_SHAPE;
    const bool with_head = le == m->n_layer;
    if (!states || !tokens || (with_head && !logits) || !workspace) return RWKV_E_NULL;
    if (T <= 0 || T > (1 << 20)) return RWKV_E_SHAPE;
    if (workspace_bytes < rwkv_v4_seq_workspace(m, T, full_output) || (((uintptr_t)workspace) & 255))
        return RWKV_E_WORKSPACE;
    for (int i = lb; i < le; ++i) {
        const rwkv_v4_layer_state &s = states[i];
        if (!s.att_xx || !s.aa || !s.bb || !s.pp || !s.ffn_xx) return RWKV_E_NULL;
        if (!aligned16(s.att_xx) || !aligned16(s.ffn_xx)) return RWKV_E_LAYOUT;
    }
    hipStream_t st = (hipStream_t)stream;
    const int C = m->n_embd, F = m->n_ffn;
    SeqWs ws = carve(workspace, T, C, F);
    float *s0[3] = {ws.sums, ws.sums + 2 * T, ws.sums + 4 * T};
    float *s2[3] = {ws.sums + T, ws.sums + 3 * T, ws.sums + 5 * T};
    float *s0v = ws.sums + 6 * T, *s2v = ws.sums + 7 * T;

    if (lb == 0)
        hipLaunchKernelGGL(gather_emb_kernel, dim3((unsigned)T), dim3(256), 0, st, (int)T, C, (int)m->vocab, tokens, m->emb, ws.x);
    SideStreams *ss = T >= 256 ? side_streams(st) : nullptr;

    for (int i = lb; i < le; ++i) {
        const rwkv_v4_layer &l = m->layers[i];
        const rwkv_v4_layer_state &s = states[i];
        const bool u8 = mat_is_u8(m->weights_u8, l.att_key);
        // ---- time mix
        {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln1_w; a.ln_b = l.ln1_b; a.sx = s.att_xx;
            a.xx_last = nullptr; a.state_out = s.att_xx;
            const rwkv_half *mix[3] = {l.att_mix_k, l.att_mix_v, l.att_mix_r};
            const rwkv_mat *mt[3] = {&l.att_key, &l.att_value, &l.att_receptance};
            for (int j = 0; j < 3; ++j) {
                a.mix[j] = mix[j]; a.ry[j] = u8 ? mt[j]->ry : nullptr; a.my[j] = u8 ? mt[j]->my : nullptr;
                a.xs[j] = ws.xs[j]; a.s0[j] = s0[j]; a.s2[j] = s2[j];
            }
            if ((rc = lnmix_seq_launch(a, 3, st))) return rc;
        }
        GemmEpi e{};
        e.out_scale = 1.f;
        // k, v: uint8 weights return fp16 (widened by the consumer); fp16 weights return fp32 directly
        e.act = ACT_NONE; e.out_dtype = u8 ? RWKV_DT_F16 : RWKV_DT_F32; e.raw_f32 = u8 ? 0 : 1;
        {   // k, v, r as one grouped launch at every length (tile size and K split by cost)
            const rwkv_half *xin[3] = {ws.xs[0], ws.xs[1], ws.xs[2]};
            const rwkv_mat *mats[3] = {&l.att_key, &l.att_value, &l.att_receptance};
            void *outs[3] = {ws.k, ws.v, ws.r};
            GemmEpi ep[3] = {e, e, e};
            e.act = ACT_SIGMOID; e.out_dtype = RWKV_DT_F16; e.raw_f32 = 0;   // receptance, and every product after it
            ep[2] = e;
            if ((rc = gemm_group_launch(u8, 3, T, C, xin, mats, outs, ep, nullptr, s0, ws.splitk, st))) return rc;
        }
        if ((rc = wkv4_fused_launch((int)T, C, l.time_decay, l.time_first, ws.k, ws.v, u8 ? 0 : 1, ws.r, ws.rwkv, s.aa,
                                    s.bb, s.pp, st, ws.wkv)))
            return rc;
        const rwkv_half *a_out = ws.rwkv;
        if (u8) {
            if ((rc = mm8_prepare_launch(T, C, ws.rwkv, C, l.att_output.ry, l.att_output.my, ws.xs[0], s0[0], s2[0], st)))
                return rc;
            a_out = ws.xs[0];
        }
        e.act = ACT_RESIDUAL; e.res = ws.x; e.ldres = C;
        if ((rc = run_gemm(l.att_output, u8, T, a_out, s0[0], s2[0], ws.x, C, e, st, ws.splitk))) return rc;
        // ---- channel mix
        {
            SeqMixArgs a{};
            a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = l.ln2_w; a.ln_b = l.ln2_b; a.sx = s.ffn_xx;
            a.xx_last = nullptr; a.state_out = s.ffn_xx;
            const rwkv_half *mix[2] = {l.ffn_mix_r, l.ffn_mix_k};
            const rwkv_mat *mt[2] = {&l.ffn_receptance, &l.ffn_key};
            for (int j = 0; j < 2; ++j) {
                a.mix[j] = mix[j]; a.ry[j] = u8 ? mt[j]->ry : nullptr; a.my[j] = u8 ? mt[j]->my : nullptr;
                a.xs[j] = ws.xs[j]; a.s0[j] = s0[j]; a.s2[j] = s2[j];
            }
            if ((rc = lnmix_seq_launch(a, 2, st))) return rc;
        }
        e = GemmEpi{};
        e.out_scale = 1.f; e.out_dtype = RWKV_DT_F16;
        e.act = ACT_SIGMOID;
        int vparts = 0;   // > 0: the key product hands the value product its input with this many partial sums per row
        // the partial sums that a key launch of this plan hands over, 0: the value product's input has a scaling pass
        auto handed_over = [&](const GemmPlan &pk) {
            if (!handover_enabled() || pk.kind != 2 || pk.ks != 1) return 0;
            GemmEpi ev{};
            ev.out_scale = 1.f; ev.out_dtype = RWKV_DT_F16;
            ev.act = ACT_GATED_RESIDUAL; ev.gate = ws.r; ev.ldgate = C; ev.res = ws.x; ev.ldres = C;
            const GemmPlan pv = plan_gemm(l.ffn_value, true, T, ws.xsv, s0v, s2v, ws.x, C, ev, ws.splitk);
            return pv.kind == 2 && pk.tn >= EMIT_MIN_TN ? emitted_parts(F, pk.tn) : 0;
        };
        auto emit = [&](GemmEpi &k, int np) {
            if (!np) return;
            k.emit_ry = l.ffn_value.ry; k.emit_my = l.ffn_value.my;
            k.emit_s0 = ws.parts; k.emit_s2 = ws.parts + (size_t)T * np;
        };
        const rwkv_half *xrk[2] = {ws.xs[0], ws.xs[1]};
        const rwkv_mat *mrk[2] = {&l.ffn_receptance, &l.ffn_key};
        void *ork[2] = {ws.r, u8 ? ws.xsv : ws.vx};
        GemmEpi erk[2] = {e, e};
        erk[1].act = ACT_RELU_SQ;
        if ((T <= 128 && !(C & 127) && !(F & 127)) || gemm_group_pays(u8, 2, T, C, xrk, mrk, ork, erk, ws.splitk)) {
            // Receptance and key in one grouped launch: short calls, and where the cost model puts it first.  8 layers, us, by
            // the limit of 128 tokens before -> by cost: n_embd 768, fp16, 200 tokens 516 -> 455, 513 635 -> 609; 2048, uint8, 140
            // tokens 807 -> 726, 513 1388 -> 1305; 4096, uint8, 700 tokens 3814 -> 3396, 256 and 1000 tokens, which stay two launches,
            // 1647 and 4131 against 1686 and 4334 as one.  The key launch of a group hands over like one of its own (20 to 45 tokens
            // of 4096 channels, uint8: 957 -> 915).
            if (u8) vparts = handed_over(gemm_group_plan(true, 2, T, C, xrk, mrk, ork, true));
            emit(erk[1], vparts);
            if (!vparts) ork[1] = ws.vx;
            if ((rc = gemm_group_launch(u8, 2, T, C, xrk, mrk, ork, erk, nullptr, s0, ws.splitk, st))) return rc;
        } else {
        // The receptance product beside the key product where neither would split K.  From 512 tokens on one after the other: the
        // direct-to-LDS tiles take a whole CU, so products side by side gain nothing.
        ForkScope par2(ss, st, 1, T < 512 && (T / 128) * (C / 128) > 128);
        float *sk2 = par2 ? nullptr : ws.splitk;
        // uint8: the three-stage tile for both, so that one of each fits a CU (2 x 73 KB; the four-stage tile that the
        // receptance product gets by itself takes 97: 4.89 ms against 4.82 for 16 layers of n_embd 4096 at 257 tokens, 5.15
        // against 5.07 at 384).  Two fp16 tiles fit no CU with either: 4.85 four-stage, 4.91 three-stage at 257.
        e.small_tiles = par2 && u8 ? 1 : 0;
        if ((rc = run_gemm(l.ffn_receptance, u8, T, ws.xs[0], s0[0], s2[0], ws.r, C, e, par2 ? ss->s[0] : st, sk2))) return rc;
        e.act = ACT_RELU_SQ;
        e.small_tiles = par2 ? 1 : 0;   // the receptance product runs beside this one
        // Where the key product runs at full depth through the direct-to-LDS kernel and the value product through that
        // kernel too, the key product's epilogue writes relu(k)^2 already scaled for the value product, with the row
        // sums as one partial sum per column tile: no scaling pass, and the unscaled [T, F] activation is never stored.
        if (u8) vparts = handed_over(plan_gemm(l.ffn_key, true, T, ws.xs[1], s0[1], s2[1], ws.xsv, F, e, sk2));
        emit(e, vparts);
        if ((rc = run_gemm(l.ffn_key, u8, T, ws.xs[1], s0[1], s2[1], vparts ? ws.xsv : ws.vx, F, e, st, sk2))) return rc;
        e.small_tiles = 0;
        e.emit_ry = e.emit_my = nullptr; e.emit_s0 = e.emit_s2 = nullptr;
        if (!par2.join()) return (int)hipErrorUnknown;
        }
        const rwkv_half *a_v = ws.vx;
        if (vparts) {
            a_v = ws.xsv;
            e.parts = vparts; e.p0 = ws.parts; e.p2 = ws.parts + (size_t)T * vparts;
        } else if (u8) {
            if ((rc = mm8_prepare_launch(T, F, ws.vx, F, l.ffn_value.ry, l.ffn_value.my, ws.xsv, s0v, s2v, st))) return rc;
            a_v = ws.xsv;
        }
        e.act = ACT_GATED_RESIDUAL; e.gate = ws.r; e.ldgate = C; e.res = ws.x; e.ldres = C;
        e.out_scale = (m->rescale_layer > 0 && (i + 1) % m->rescale_layer == 0) ? 0.5f : 1.f;
        if ((rc = run_gemm(l.ffn_value, u8, T, a_v, s0v, s2v, ws.x, C, e, st, ws.splitk))) return rc;
        RWKV_LAUNCH_CHECK();
    }
    if (!with_head) return RWKV_OK;
    if (!full_output) return v4_head_launch(m, ws.x + (size_t)(T - 1) * C, logits, st);
    const bool u8 = mat_is_u8(m->weights_u8, m->head);
    {
        SeqMixArgs a{};
        a.T = (int)T; a.C = C; a.x = ws.x; a.ln_w = m->ln_out_w; a.ln_b = m->ln_out_b; a.sx = nullptr;
        a.xx_last = nullptr; a.mix[0] = nullptr;
        a.ry[0] = u8 ? m->head.ry : nullptr; a.my[0] = u8 ? m->head.my : nullptr;
        a.xs[0] = ws.xs[0]; a.s0[0] = s0[0]; a.s2[0] = s2[0];
        if ((rc = lnmix_seq_launch(a, 1, st))) return rc;
    }
    GemmEpi e{};
    e.out_scale = 1.f; e.act = ACT_NONE; e.out_dtype = RWKV_DT_F32;
    if ((rc = run_gemm(m->head, u8, T, ws.xs[0], s0[0], s2[0], logits, m->vocab, e, st, ws.splitk))) return rc;
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}
