// Sampling step after the head: token ban, presence / frequency penalties, softmax, nucleus (top-p) and
// top-k filter, temperature, one draw -- all on the device, so that a generation loop needs no
// device-to-host copy of the logits and no host synchronisation per token.
//
// One workgroup of 1024 threads keeps the vocabulary in registers: thread t holds the groups of four entries
// t, t + 1024, t + 2048, ... (at most 16 of them, V <= 65536), so every access is a coalesced 16-byte one and the
// entries 4096 c + 256 w .. + 255 of group row c belong to wave w.  (With a contiguous chunk of 64 entries per thread
// each load instruction touched 64 cache lines: the loads and stores alone took most of the kernel.)
// The nucleus cut is the largest value c with sum{p >= c} >= top_p -- the set the reference keeps (first sorted
// probability whose cumulative sum reaches top_p, ties kept) up to fp32 summation order -- and is searched on the bit
// pattern of c (positive floats order like their bit patterns): bisection over the registers until at most LIST_MAX
// entries lie between the bounds, then those entries move to LDS and each of the 16 waves tests a bound of its own,
// so a step divides the interval by 17, until no more than 64 are left, which are compared with each other.  The k-th largest value is found the same way on counts, starting at the
// nucleus cut.  The draw is an inverse-CDF walk in index order for a caller-supplied uniform number, over the sums of
// the 256 runs of 256 entries first.
// Bound by vector issue and barriers of the one CU it runs on.  Measured, V = 65536, logits N(0, 3), top_p 0.7,
// penalties: 36 us (one bit of the cut per pass over the registers and contiguous chunks: 265 us).
#include "kernels.h"

namespace {

constexpr int STHREADS = 1024, SWAVES = STHREADS / 64;
constexpr int ROWS_MAX = 16;                  // group rows: V <= 65536
constexpr int LIST_MAX = 1024;                // entries left when the search moves to LDS

struct SampleArgs {
    const float *logits;
    int V;
    float temperature, top_p;
    int top_k;
    const int32_t *ban;
    int n_ban;
    uint8_t *seen;
    float *occ;
    const float *weight;
    float presence, frequency, decay;
    const float *u;
    float *probs;
    int32_t *token;
};

// Workgroup totals of a sum and a count (counts <= 65536: exact in fp32).  Two buffers in turn, so one barrier a call:
// buffer k is written again only after the barrier of call k + 1, which every thread reaches after reading buffer k.
struct SumCount { float s, n; };
DEV SumCount block_total(float s, float n, f32x4 (&red)[2][SWAVES / 2], int &turn) {
    s = wave_sum(s);
    n = wave_sum(n);
    f32x4 *buf = red[turn];
    turn ^= 1;
    if ((threadIdx.x & 63) == 0) {
        ((float *)buf)[2 * (threadIdx.x >> 6)] = s;
        ((float *)buf)[2 * (threadIdx.x >> 6) + 1] = n;
    }
    __syncthreads();
    SumCount t = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SWAVES / 2; ++i) {
        const f32x4 v = buf[i];
        t.s = (t.s + v[0]) + v[2];
        t.n = (t.n + v[1]) + v[3];
    }
    return t;
}

DEV float block_max(float v, f32x4 (&red)[2][SWAVES / 2], int &turn) {
    v = wave_max(v);
    f32x4 *buf = red[turn];
    turn ^= 1;
    if ((threadIdx.x & 63) == 0) ((float *)buf)[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = ((float *)buf)[0];
#pragma unroll
    for (int i = 1; i < SWAVES; ++i) m = fmaxf(m, ((float *)buf)[i]);
    return m;
}

// inclusive sum over the lanes of a wave
DEV float wave_scan(float v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float up = __shfl_up(v, o, WAVE);
        if (lane >= o) v += up;
    }
    return v;
}

// POW: temperature other than 1 (its 64 copies stay out of the code of the usual case)
// SROWS: group rows, at least V / 4096.  Rows past the end hold zeros and are worked on like the others: with a test
// of V around each row the compiler made a copy of what follows for every number of rows.
template <int SROWS, bool POW>
__global__ __launch_bounds__(STHREADS) void sample_kernel(SampleArgs a) {
    __shared__ f32x4 red[2][SWAVES / 2];
    __shared__ float list[LIST_MAX];
    __shared__ __align__(16) float tail[64];
    __shared__ __align__(16) float seg[ROWS_MAX * SWAVES];   // sums of the runs of 256 entries, in index order
    __shared__ int pick_seg, pick_tok;
    __shared__ float pick_before, pick_target;
    const int V = a.V, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int EMAX = 4 * SROWS;         // entries per thread
    int turn = 0;
    float p[EMAX];
    // ---- adjusted logits (utils.py:103-106)
    uint32_t flag[SROWS];   // the four `seen` bytes of a group
    const int lim = (V - 4) & ~3;   // the last group that can be loaded whole
    if (V >= 4 && (((uintptr_t)a.logits) & 15) == 0 && (((uintptr_t)a.seen) & 3) == 0) {
#pragma unroll
        for (int c = 0; c < SROWS; ++c) {
            const int i = 4 * (c * STHREADS + tid);
            const f32x4 x = *(const f32x4 *)(a.logits + min(i, lim));
            flag[c] = 0;
            if (a.seen) flag[c] = *(const uint32_t *)(a.seen + min(i, lim));
#pragma unroll
            for (int e = 0; e < 4; ++e) p[4 * c + e] = i <= lim ? x[e] : -INFINITY;
            if (i > lim) flag[c] = 0;
        }
        // the group that ends inside (V % 4 entries)
        const int i = lim + 4;
        if (i < V && ((i >> 2) & (STHREADS - 1)) == tid) {
#pragma unroll
            for (int c = 0; c < SROWS; ++c)
                if (c == i / (4 * STHREADS)) {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (i + e < V) {
                            p[4 * c + e] = a.logits[i + e];
                            if (a.seen) flag[c] |= (uint32_t)a.seen[i + e] << (8 * e);
                        }
                }
        }
    } else {
#pragma unroll
        for (int c = 0; c < SROWS; ++c) {
            flag[c] = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 4 * (c * STHREADS + tid) + e;
                const float v = a.logits[min(i, V - 1)];
                p[4 * c + e] = i < V ? v : -INFINITY;
                if (a.seen) flag[c] |= (uint32_t)(i < V ? a.seen[min(i, V - 1)] : 0) << (8 * e);
            }
        }
    }
    unsigned long long seen_bits = 0;
#pragma unroll
    for (int c = 0; c < SROWS; ++c)
        if (flag[c]) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool on = (flag[c] >> (8 * e)) & 0xff;
                const float o = a.occ[min(4 * (c * STHREADS + tid) + e, V - 1)];
                seen_bits |= on ? 1ull << (4 * c + e) : 0ull;
                p[4 * c + e] -= on ? a.presence + o * a.frequency : 0.f;
            }
        }
    for (int b = 0; b < a.n_ban; ++b) {
        const int i = a.ban[b];
        if (((i >> 2) & (STHREADS - 1)) == tid) {
            const int k = (i >> 12) * 4 + (i & 3);
#pragma unroll
            for (int e = 0; e < EMAX; ++e)
                if (e == k) p[e] = -INFINITY;
        }
    }
    // ---- softmax (utils.py:59)
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < EMAX; ++e) mx = fmaxf(mx, p[e]);
    mx = block_max(mx, red, turn);
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < EMAX; ++e) { p[e] = (p[e] == -INFINITY) ? 0.f : exp_acc(p[e] - mx); s += p[e]; }
    const float inv = 1.f / block_total(s, 0.f, red, turn).s;
    float pmax = 0.f, total = 0.f;
#pragma unroll
    for (int e = 0; e < EMAX; ++e) { p[e] *= inv; pmax = fmaxf(pmax, p[e]); total += p[e]; }
    pmax = block_max(pmax, red, turn);
    total = block_total(total, 0.f, red, turn).s;

    const float top_p = a.temperature == 0.f ? 0.f : a.top_p;
    // sum and count of the entries >= c
    auto above = [&](float c) {
        float sc = 0.f;
        unsigned n = 0;
#pragma unroll
        for (int e = 0; e < EMAX; ++e) {
            const bool in = p[e] >= c;
            sc += in ? p[e] : 0.f;
            n += in ? 1u : 0u;
        }
        return block_total(sc, (float)n, red, turn);
    };
    // The largest bit pattern c in [lo, hi) for which enough({sum, count} of the entries >= c) holds: it holds at lo
    // and not at hi.  `guess` is the first bound tried.  at_lo / at_hi: the totals there.
    auto search = [&](unsigned lo, unsigned hi, unsigned guess, SumCount at_lo, bool counts) {
        auto enough = [&](SumCount t) { return counts ? t.n >= (float)a.top_k : t.s >= top_p; };
        SumCount at_hi = {0.f, 0.f};   // hi lies past the largest entry
        unsigned cand = guess;
        while (hi - lo > 1 && at_lo.n - at_hi.n > (float)LIST_MAX) {
            if (cand <= lo || cand >= hi) cand = lo + ((hi - lo) >> 1);
            const SumCount t = above(__uint_as_float(cand));
            if (enough(t)) { lo = cand; at_lo = t; } else { hi = cand; at_hi = t; }
            cand = 0;
        }
        if (hi - lo <= 1) return lo;
        const SumCount past_hi = at_hi;
        // the entries in [lo, hi) to LDS, in thread order (zeros, padding among them, decide nothing and stay out)
        const float flo = __uint_as_float(max(lo, 1u)), fhi = __uint_as_float(hi);
        int mine = 0;
#pragma unroll
        for (int e = 0; e < EMAX; ++e) mine += (p[e] >= flo && p[e] < fhi) ? 1 : 0;
        const float incl = wave_scan((float)mine);   // <= 1024: exact
        int n, at;
        {
            f32x4 *buf = red[turn];
            turn ^= 1;
            if (lane == 63) ((float *)buf)[wave] = incl;
            __syncthreads();
            float before = 0.f, all = 0.f;
#pragma unroll
            for (int w = 0; w < SWAVES; ++w) {
                const float v = ((float *)buf)[w];
                before += w < wave ? v : 0.f;
                all += v;
            }
            n = (int)all;
            at = (int)(before + incl) - mine;
        }
        // the same comparisons again, not 64 lane masks kept from above (they would not fit the scalar registers)
        float flo2 = flo, fhi2 = fhi;
        asm volatile("" : "+v"(flo2), "+v"(fhi2));
#pragma unroll
        for (int e = 0; e < EMAX; ++e)
            if (p[e] >= flo2 && p[e] < fhi2) list[min(at++, LIST_MAX - 1)] = p[e];
        __syncthreads();
        float left = (float)n;   // entries still between the bounds
        while (hi - lo > 1 && left > 64.f) {
            const unsigned step = (hi - lo) / (SWAVES + 1) + 1;
            const unsigned c = lo + step * (wave + 1);
            SumCount t = at_hi;      // the totals at hi and past it
            if (c < hi) {
                const float fc = __uint_as_float(c);
                float sc = 0.f, k = 0.f;
                for (int i = lane; i < n; i += 64) {
                    const float v = list[i];
                    if (v >= fc) { sc += v; k += 1.f; }
                }
                t.s = past_hi.s + wave_sum(sc);
                t.n = past_hi.n + wave_sum(k);
            }
            f32x4 *buf = red[turn];
            turn ^= 1;
            if (lane == 0) {
                ((float *)buf)[2 * wave] = t.s;
                ((float *)buf)[2 * wave + 1] = t.n;
            }
            __syncthreads();
            int good = 0;            // the bounds that hold are a leading run up to rounding: take the largest
            SumCount above_good = at_hi;
#pragma unroll
            for (int w = SWAVES - 1; w >= 0; --w) {
                const SumCount q = {((float *)buf)[2 * w], ((float *)buf)[2 * w + 1]};
                if (good == 0) {
                    if (lo + step * (w + 1) < hi && enough(q)) { good = w + 1; at_lo = q; }
                    else above_good = q;
                }
            }
            hi = min(hi, lo + step * (good + 1));
            lo = lo + step * good;
            at_hi = above_good;
            left = at_lo.n - at_hi.n;
        }
        if (hi - lo <= 1) return lo;
        // at most 64 are left: one to a lane, in list order; the largest of them at which the condition holds is the answer
        {
            const float l1 = __uint_as_float(max(lo, 1u)), h1 = __uint_as_float(hi);
            if (wave == 0) {
                int at64 = 0;
                for (int i0 = 0; i0 < n; i0 += 64) {
                    const float v = i0 + lane < n ? list[i0 + lane] : 0.f;
                    const bool in = v >= l1 && v < h1;
                    const unsigned long long m = __ballot(in);
                    if (in) tail[min(at64 + (int)__popcll(m & ((1ull << lane) - 1)), 63)] = v;
                    at64 += (int)__popcll(m);
                }
                if (lane >= at64) tail[lane] = 0.f;
            }
            __syncthreads();
            const float mine64 = tail[lane];
            SumCount t = at_hi;
#pragma unroll 2
            for (int i = 0; i < 64; i += 4) {
                const f32x4 v = *(const f32x4 *)&tail[i];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v[e] >= mine64) { t.s += v[e]; t.n += v[e] > 0.f ? 1.f : 0.f; }
            }
            const float best = wave_max(mine64 > 0.f && enough(t) ? mine64 : 0.f);
            __syncthreads();         // the lists may be written again
            if (best > 0.f) lo = __float_as_uint(best);
        }
        return lo;
    };

    // ---- nucleus cut (utils.py:55-58, 66-69): temperature 0 means top_p 0
    float cut = pmax;  // top_p <= 0, or no cumulative sum reaches top_p: the first sorted probability
    if (top_p >= 1.f && total >= top_p) cut = 0.f;   // everything: which of the last entries a sum of 1 can do without is rounding only
    // ---- top_k (utils.py:70-71): the k-th largest value, where that is more than the nucleus cut
#pragma unroll 1
    for (int counts = 0; counts < 2; ++counts) {     // one copy of the search's code
        unsigned lo = 0u, guess = 0u;
        SumCount at_lo = {total, (float)V};
        if (!counts) {
            if (!(top_p > 0.f && top_p < 1.f && total >= top_p)) continue;
            // entries below (total - top_p) / V cannot add up to what may be left out: the cut is hardly ever below that
            guess = __float_as_uint(fmaxf(0.5f * (total - top_p), 0.f) / (float)V);
        } else {
            if (!(a.top_k > 0 && a.top_k < V)) continue;
            at_lo = above(cut);
            if (!(at_lo.n > (float)a.top_k)) continue;
            lo = __float_as_uint(cut);
        }
        cut = __uint_as_float(search(lo, __float_as_uint(pmax) + 1, guess, at_lo, counts != 0));
    }
    // ---- filter, temperature (utils.py:69-73), sums of the runs
    const float invt = 1.f / a.temperature;
#pragma unroll
    for (int c = 0; c < SROWS; ++c) {
#pragma unroll
        for (int e = 4 * c; e < 4 * c + 4; ++e) {
            p[e] = (p[e] >= cut && p[e] > 0.f) ? p[e] : 0.f;
            if (POW && p[e] > 0.f) p[e] = powf(p[e], invt);
        }
        float run = (p[4 * c] + p[4 * c + 1]) + (p[4 * c + 2] + p[4 * c + 3]);
        if (__ballot(run > 0.f)) run = wave_sum(run);   // most runs hold nothing that is kept
        if (lane == 0) seg[c * SWAVES + wave] = run;
    }
    if (SROWS < ROWS_MAX && tid >= SROWS * SWAVES && tid < ROWS_MAX * SWAVES) seg[tid] = 0.f;
    if (a.probs && (((uintptr_t)a.probs) & 15) == 0) {
#pragma unroll
        for (int c = 0; c < SROWS; ++c) {
            const int i = 4 * (c * STHREADS + tid);
            if (i + 3 < V) *(f32x4 *)(a.probs + i) = f32x4{p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
            else if (i < V)
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (i + e < V) a.probs[i + e] = p[4 * c + e];
        }
    } else if (a.probs) {
#pragma unroll
        for (int e = 0; e < EMAX; ++e) {
            const int i = 4 * ((e >> 2) * STHREADS + tid) + (e & 3);
            if (i < V) a.probs[i] = p[e];
        }
    }
    __syncthreads();
    // ---- draw: first index whose running sum exceeds u * total; the last kept entry where rounding leaves none
    if (wave == 0) {
        const f32x4 g = *(const f32x4 *)&seg[4 * lane];
        const float mine = (g[0] + g[1]) + (g[2] + g[3]);
        const float incl = wave_scan(mine);
        const float target = (*a.u) * __shfl(incl, 63, WAVE);
        float run = incl - mine, before = 0.f;
        int first = 1 << 30, last = -1;
        float last_before = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (g[e] > 0.f) {
                if (first == (1 << 30) && run + g[e] > target) { first = 4 * lane + e; before = run; }
                last = 4 * lane + e;
                last_before = run;
            }
            run += g[e];
        }
        const unsigned long long hit = __ballot(first != (1 << 30)), kept = __ballot(last >= 0);
        const int from = hit ? __builtin_ctzll(hit) : (kept ? 63 - __builtin_clzll(kept) : 0);
        if (lane == from) {
            pick_seg = hit ? first : last;   // -1: nothing is kept
            pick_before = hit ? before : last_before;
            pick_target = target;
        }
    }
    __syncthreads();
    const int sg = pick_seg;
    if (sg >= 0 && wave == (sg & (SWAVES - 1))) {
        f32x4 q = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < SROWS; ++c)
            if (c == sg / SWAVES) q = f32x4{p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
        const float mine = (q[0] + q[1]) + (q[2] + q[3]), target = pick_target;
        float run = pick_before + (wave_scan(mine) - mine);
        int first = -1, last = -1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            run += q[e];
            if (q[e] > 0.f) {
                last = e;
                if (first < 0 && run > target) first = e;
            }
        }
        const unsigned long long hit = __ballot(first >= 0), kept = __ballot(last >= 0);
        const int from = hit ? __builtin_ctzll(hit) : (kept ? 63 - __builtin_clzll(kept) : 0);
        if (lane == from) pick_tok = 4 * (sg / SWAVES * STHREADS + tid) + max(hit ? first : last, 0);
    }
    __syncthreads();
    const int tok = sg >= 0 ? pick_tok : 0;
    if (tid == 0) *a.token = tok;
    // ---- occurrence table (utils.py:112-123): decay, then add the drawn token's weight
    if (a.seen && a.occ) {
        const bool owner = ((tok >> 2) & (STHREADS - 1)) == tid;
        const int tk = owner ? (tok >> 12) * 4 + (tok & 3) : -1;
        const float w = owner ? (a.weight ? a.weight[tok] : 1.f) : 0.f;
        if (owner && !((seen_bits >> tk) & 1)) {
            a.occ[tok] = w;
            a.seen[tok] = 1;
        }
        while (seen_bits) {
            const int k = __builtin_ctzll(seen_bits);
            seen_bits &= seen_bits - 1;
            const int i = 4 * ((k >> 2) * STHREADS + tid) + (k & 3);
            float o = a.occ[i] * a.decay;
            if (k == tk) o += w;
            a.occ[i] = o;
        }
    }
}

}  // namespace

// The temperature-0 draw without penalties or bans: the index of the largest logit, the lowest such index on
// ties (NaN entries are never chosen).  One workgroup; each thread scans a strided share of the vocabulary with
// eight loads in flight, then (value, index) pairs are reduced by wave shuffles and across the 16 waves in LDS.
template <bool F16>
__global__ __launch_bounds__(STHREADS) void greedy_kernel(const void *__restrict__ logits_, int V, int32_t *__restrict__ token) {
    const float *lf = (const float *)logits_;
    const rwkv_half *lh = (const rwkv_half *)logits_;
    __shared__ float rv[SWAVES];
    __shared__ int ri[SWAVES];
    float best = -__builtin_inff();
    int bi = 0x7fffffff;
    auto take = [&](float v, int i) {
        if (v > best || (v == best && i < bi)) { best = v; bi = i; }
    };
    for (int i0 = threadIdx.x; i0 < V; i0 += 8 * STHREADS) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u * STHREADS, V - 1);
            v[u] = F16 ? h2f(lh[i]) : lf[i];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + u * STHREADS < V) take(v[u], i0 + u * STHREADS);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) take(__shfl_xor(best, o, WAVE), __shfl_xor(bi, o, WAVE));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) { rv[wid] = best; ri[wid] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SWAVES; ++w) take(rv[w], ri[w]);
        *token = bi == 0x7fffffff ? 0 : bi;
    }
}

extern "C" int rwkv_greedy_token(const void *logits, int dtype, int64_t V, int32_t *token, void *stream) {
    if (!logits || !token) return RWKV_E_NULL;
    if (V <= 0 || V > 0x7fffffff) return RWKV_E_SHAPE;
    if (dtype == RWKV_DT_F32) hipLaunchKernelGGL(greedy_kernel<false>, dim3(1), dim3(STHREADS), 0, (hipStream_t)stream, logits, (int)V, token);
    else if (dtype == RWKV_DT_F16) hipLaunchKernelGGL(greedy_kernel<true>, dim3(1), dim3(STHREADS), 0, (hipStream_t)stream, logits, (int)V, token);
    else return RWKV_E_DTYPE;
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}

extern "C" int rwkv_sample_logits(const float *logits, int64_t V, float temperature, float top_p, int32_t top_k,
                                  const int32_t *token_ban, int32_t n_ban, uint8_t *seen, float *occurrence,
                                  const float *token_weight, float alpha_presence, float alpha_frequency,
                                  float alpha_decay, const float *u, float *probs, int32_t *token, void *stream) {
    if (!logits || !u || !token) return RWKV_E_NULL;
    if (V <= 0 || V > (int64_t)STHREADS * 4 * ROWS_MAX || n_ban < 0 || (n_ban > 0 && !token_ban)) return RWKV_E_SHAPE;
    if ((seen == nullptr) != (occurrence == nullptr)) return RWKV_E_NULL;
    if (!(temperature >= 0.f) || top_k < 0) return RWKV_E_SHAPE;
    SampleArgs a{logits, (int)V, temperature, top_p, top_k, token_ban, n_ban, seen, occurrence, token_weight,
                 alpha_presence, alpha_frequency, alpha_decay, u, probs, token};
    // group rows: 4 (small vocabularies), 13 (the 50277-entry ones) or 16
    const bool pow = temperature != 0.f && temperature != 1.f;
#define RWKV_SAMPLE(ROWS)                                                                                                      \
    do {                                                                                                                      \
        if (pow) hipLaunchKernelGGL((sample_kernel<ROWS, true>), dim3(1), dim3(STHREADS), 0, (hipStream_t)stream, a);         \
        else hipLaunchKernelGGL((sample_kernel<ROWS, false>), dim3(1), dim3(STHREADS), 0, (hipStream_t)stream, a);            \
    } while (0)
    if (V <= 4 * 4 * STHREADS) RWKV_SAMPLE(4);
    else if (V <= 13 * 4 * STHREADS) RWKV_SAMPLE(13);
    else RWKV_SAMPLE(16);
#undef RWKV_SAMPLE
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}
