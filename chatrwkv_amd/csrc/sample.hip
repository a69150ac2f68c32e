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
// so a step divides the interval by 17, until no more than 64 are left, which are compared with each other.  The k-th
// largest value is found the same way on counts, starting at the nucleus cut.  The draw is an inverse-CDF walk in index order for a caller-supplied uniform number, over the sums of
// the 256 runs of 256 entries first.
// Bound by vector issue and barriers of the one CU it runs on.  Measured, V = 65536, logits N(0, 3), top_p 0.7,
// penalties, draw after draw: 39 us (one bit of the cut per pass over the registers and contiguous chunks: 265 us).
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

// inclusive sum over the lanes of a wave: four steps within the rows of 16 lanes, the last lanes of the rows before (DPP)
template <int CTRL, int ROWS>
DEV float dpp_rows(float v) {   // 0 in the rows that are not written
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xf, true));
}
DEV float wave_scan(float v) {
    v += dpp_rows<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v += dpp_rows<0x112, 0xf>(v);
    v += dpp_rows<0x114, 0xf>(v);
    v += dpp_rows<0x118, 0xf>(v);
    v += dpp_rows<0x142, 0xa>(v);   // row_bcast 15 into rows 1 and 3
    v += dpp_rows<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
    return v;
}
DEV float last_lane(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63)); }

// Does a bound hold whose entries add up to t?  The nucleus cut asks for a sum, the k-th largest value (top_k >= 0) for a count.
DEV bool enough(SumCount t, float top_p, int top_k) { return top_k >= 0 ? t.n >= (float)top_k : t.s >= top_p; }

// The largest bit pattern c in [lo, hi) that holds, from the n <= LIST_MAX entries of [lo, hi) in LDS: it holds at lo (the
// entries from there on: at_lo) and not at hi (at_hi).
DEV unsigned search_list(const float *list, int n, unsigned lo, unsigned hi, SumCount at_lo, SumCount at_hi, float top_p, int top_k,
                         f32x4 (&tail)[16], f32x4 (&red)[2][SWAVES / 2], int &turn) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const SumCount past_hi = at_hi;
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
                if (lo + step * (w + 1) < hi && enough(q, top_p, top_k)) { good = w + 1; at_lo = q; }
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
                if (in) ((float *)tail)[min(at64 + (int)__popcll(m & ((1ull << lane) - 1)), 63)] = v;
                at64 += (int)__popcll(m);
            }
            if (lane >= at64) ((float *)tail)[lane] = 0.f;
        }
        __syncthreads();
        const float mine64 = ((float *)tail)[lane];
        SumCount t = at_hi;
#pragma unroll 2
        for (int i = 0; i < 16; ++i) {
            const f32x4 v = tail[i];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (v[e] >= mine64) { t.s += v[e]; t.n += v[e] > 0.f ? 1.f : 0.f; }
        }
        const float best = wave_max(mine64 > 0.f && enough(t, top_p, top_k) ? mine64 : 0.f);
        __syncthreads();         // the lists may be written again
        if (best > 0.f) lo = __float_as_uint(best);
    }
    return lo;
}

// POW: temperature other than 1 (its 64 copies stay out of the code of the usual case)
// SROWS: group rows, at least V / 4096.  Rows past the end hold zeros and are worked on like the others: with a test
// of V around each row the compiler made a copy of what follows for every number of rows.
template <int SROWS, bool POW>
__global__ __launch_bounds__(STHREADS) void sample_kernel(SampleArgs a) {
    __shared__ f32x4 red[2][SWAVES / 2];
    __shared__ float list[LIST_MAX];
    __shared__ f32x4 tail[16];
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
    for (int e = 0; e < EMAX; ++e) { p[e] = (p[e] == -INFINITY) ? 0.f : expf(p[e] - mx); s += p[e]; }
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
        SumCount at_hi = {0.f, 0.f};   // hi lies past the largest entry
        unsigned cand = guess;
        while (hi - lo > 1 && at_lo.n - at_hi.n > (float)LIST_MAX) {
            if (cand <= lo || cand >= hi) cand = lo + ((hi - lo) >> 1);
            const SumCount t = above(__uint_as_float(cand));
            if (enough(t, top_p, counts ? a.top_k : -1)) { lo = cand; at_lo = t; } else { hi = cand; at_hi = t; }
            cand = 0;
        }
        if (hi - lo <= 1) return lo;
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
        return search_list(list, n, lo, hi, at_lo, at_hi, top_p, counts ? a.top_k : -1, tail, red, turn);
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

// ---- the same draw over the chip -------------------------------------------------------------------------------
// One workgroup issues every instruction of a pass over 65536 entries 256 times per SIMD, half a microsecond each, and the
// exponential alone takes twenty.  With scratch from the caller the passes over the vocabulary run on one workgroup per
// SEG entries, in three launches:
//   adjust: bans and penalties, the segment's largest logit and sum of exponentials;
//   probs:  the probabilities (every workgroup forms the total) and their powers, for BOUNDS bounds half an octave apart below the largest
//           one the segment's sum and count of the entries that reach it, and the list, in index order, of the entries that
//           the nucleus can need: those below (1 - top_p) / 2 V cannot add up to what may be left out;
//   draw:   every workgroup finds the cut for itself -- the bounds leave half an octave, which goes to its 64th part that
//           holds the cut until no more than FEW entries are left, and these are sorted -- and draws; it writes the filtered
//           probabilities and the occurrence counts of its segment.
// Sums are added in a fixed order throughout.  Where the total is no positive number (a NaN, an infinity or nothing but masks
// among the logits) nothing is kept and id 0 is drawn, which is what the kernel above makes of such logits.
// Bound by the latency of the three launches.  Measured as above, V = 65536: 16.4 us a draw (2.9 + 4.4 + 7.7 and the gaps), 38 with one
// workgroup; with the lists in LDS and the bracket searched by search_list 25.8, 5 us of it in the search.
// The draw's workgroups each take in the candidates of all segments, 64 bytes a clock and less, and issue every comparison with
// them 16 waves deep.  So there are two lists: of N(0, 3) 40 % of the entries are candidates at top_p 0.7, and 10 % reach bound HIGH, which has the whole
// nucleus.  us a draw, one list / two: 65536 entries, top_p 0.7 17.0 / 16.4, 0.85 20.9 / 16.4 (with the sort below), top_k 50 25.5 / 19.9; 50277 from
// N(0, 0.3), which need the long one a trip to memory later, 39.9 / 36.9.
constexpr int SEG = 1024, SEGS_MAX = 64, BOUNDS = 32;
constexpr int FEW = 256;                      // entries of a bracket that are compared with each other at once
constexpr int HIGH = 25;                      // a bound 2^-13 below the largest probability
constexpr int PART = 2 * BOUNDS + 3;          // per segment: sums and counts at the bounds, sum of all, length of the list, its smallest entry

struct SampleWs {
    float *p;          // [segments][SEG] adjusted logits, then probabilities
    float *list;       // [segments][SEG] candidates in index order
    float *pow;        // [segments][SEG] the same to the power 1 / temperature, at temperatures other than 0 and 1
    uint16_t *idx;     // [segments][SEG] their places in the segment
    float *high, *high_pow;   // list, pow and idx of the entries that reach bound HIGH alone
    uint16_t *high_idx;
    float *soft;       // [segments][2] largest logit, sum of exponentials
    float *part;       // [segments][PART]
};

__global__ __launch_bounds__(256) void sample_adjust_kernel(SampleArgs a, SampleWs ws) {
    __shared__ float red[8];
    const int V = a.V, i0 = blockIdx.x * SEG + 4 * threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    at_once({a.logits, a.seen, a.occ, a.ban, ws.p, ws.soft});
    // everything is requested before anything is looked at, whether an entry has been seen or not
    f32x4 x, occ = {0.f, 0.f, 0.f, 0.f};
    uint32_t flag = 0;
    const int banned = lane < a.n_ban ? a.ban[lane] : 0;
    if (i0 + 3 < V && ((((uintptr_t)a.logits) | ((uintptr_t)a.occ)) & 15) == 0 && (((uintptr_t)a.seen) & 3) == 0) {
        x = *(const f32x4 *)(a.logits + i0);
        if (a.seen) {
            flag = *(const uint32_t *)(a.seen + i0);
            occ = *(const f32x4 *)(a.occ + i0);
        }
    } else {
        uint8_t f[4] = {};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = min(i0 + e, V - 1);
            x[e] = a.logits[i];
            if (a.seen) { f[e] = a.seen[i]; occ[e] = a.occ[i]; }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = i0 + e < V ? x[e] : -INFINITY;
            flag |= (i0 + e < V ? (uint32_t)f[e] : 0u) << (8 * e);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if ((flag >> (8 * e)) & 0xff) x[e] -= a.presence + occ[e] * a.frequency;
    for (int b = 0; b < a.n_ban; ++b) {
        const int k = (b < 64 ? __builtin_amdgcn_readlane(banned, b) : a.ban[b]) - i0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e == k) x[e] = -INFINITY;
    }
    *(f32x4 *)(ws.p + i0) = x;
    float m = wave_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) s += x[e] == -INFINITY ? 0.f : expf(x[e] - m);
    s = wave_sum(s);
    if (lane == 0) red[4 + wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        ws.soft[2 * blockIdx.x] = m;
        ws.soft[2 * blockIdx.x + 1] = (red[4] + red[5]) + (red[6] + red[7]);
    }
}

// The largest logit and the sum of the exponentials from the segments'; every lane gets both.
struct Soft { float mx, sum; };
typedef float f32x2 __attribute__((ext_vector_type(2)));
DEV Soft soft_total(f32x2 own, int segs) {   // own: those of segment `lane`
    const int lane = threadIdx.x & 63;
    const float m = lane < segs ? own[0] : -INFINITY, s = lane < segs ? own[1] : 0.f;
    const float mx = wave_max(m);
    return {mx, wave_sum(m == -INFINITY ? 0.f : s * expf(m - mx))};
}
DEV float list_floor(float top_p, int V) { return 0.5f * (1.f - top_p) / (float)V; }   // of the candidates
DEV float bound_at(float pmax, int k) { return __uint_as_float(__float_as_uint(pmax) - ((unsigned)(k + 1) << 22)); }

// Probabilities in units of 2^-62.  Those from 2^-39 on are whole numbers of them (a bound is at least 2^-32, a candidate 2^-27),
// and all together are about 1: their sums are exact, so the same in any order, and rounded once.
DEV unsigned long long fixed(float p) { return (unsigned long long)(p * 0x1p62f); }
DEV float from_fixed(unsigned long long s) { return (float)s * 0x1p-62f; }

// Sums over the 16 lanes of a row, in every one of them.
constexpr int COPIES = 16;
template <int CTRL> DEV unsigned dpp_u32(unsigned v) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true); }
template <int CTRL> DEV unsigned long long dpp_u64(unsigned long long v) {
    return (unsigned long long)dpp_u32<CTRL>((unsigned)(v >> 32)) << 32 | dpp_u32<CTRL>((unsigned)v);
}
DEV unsigned row16_total(unsigned v) {
    v += dpp_u32<0xB1>(v);    // quad_perm: neighbours, then pairs
    v += dpp_u32<0x4E>(v);
    v += dpp_u32<0x141>(v);   // row_half_mirror
    return v + dpp_u32<0x140>(v);   // row_mirror
}
DEV unsigned long long row16_total(unsigned long long v) {
    v += dpp_u64<0xB1>(v);
    v += dpp_u64<0x4E>(v);
    v += dpp_u64<0x141>(v);
    return v + dpp_u64<0x140>(v);
}

// POW: the candidates' powers are formed here, four entries a thread over the chip.  In sample_draw_kernel each of the up to 64
// workgroups formed those of all candidates, 64 a thread, half of a draw from flat logits.  us a draw, 50277 entries, top_p 0.85,
// temperature 0.8, one workgroup / powers there / here: N(0, 0.3) 81 / 95 / 45, N(0, 3) 68 / 38 / 24.
template <bool POW>
__global__ __launch_bounds__(256) void sample_probs_kernel(SampleArgs a, SampleWs ws) {
    __shared__ unsigned long long bin_s[BOUNDS];   // sums in fixed point
    __shared__ unsigned bin_n[BOUNDS];
    __shared__ float red[4][2], least[4];
    __shared__ int highs[4];
    if (threadIdx.x < BOUNDS) { bin_s[threadIdx.x] = 0; bin_n[threadIdx.x] = 0; }
    const int i0 = blockIdx.x * SEG + 4 * threadIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int segs = (a.V + SEG - 1) / SEG;
    f32x4 p = *(const f32x4 *)(ws.p + i0);
    const Soft st = soft_total(*(const f32x2 *)(ws.soft + 2 * min(lane, segs - 1)), segs);
    const float inv = 1.f / st.sum;   // of the largest entry: its exponential is 1
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = p[e] == -INFINITY ? 0.f : expf(p[e] - st.mx) * inv;
    *(f32x4 *)(ws.p + i0) = p;
    const float top_p = a.temperature == 0.f ? 0.f : a.top_p;
    const float floor_ = top_p > 0.f ? list_floor(top_p, a.V) : inv;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const unsigned k = (__float_as_uint(inv) - __float_as_uint(p[e])) >> 22;   // the first bound that the entry reaches is k or k - 1
        const unsigned bin = k < BOUNDS + 1 ? (k > 0 && p[e] >= bound_at(inv, k - 1) ? k - 1 : k) : BOUNDS;
        if (bin < BOUNDS) {
            atomicAdd(&bin_s[bin], fixed(p[e]));
            atomicAdd(&bin_n[bin], 1u);
        }
    }
    const float total = wave_sum((p[0] + p[1]) + (p[2] + p[3]));
    unsigned long long in[4], in_high[4];
    int before = 0, n_wave = 0, before_high = 0, n_high = 0;
    float small = INFINITY;
    const float high = top_p > 0.f ? bound_at(inv, HIGH) : INFINITY;   // temperature 0: `list` has the largest entries alone
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        in[e] = __ballot(p[e] >= floor_);
        small = p[e] >= floor_ ? fminf(small, p[e]) : small;
        before += (int)__popcll(in[e] & ((1ull << lane) - 1));
        n_wave += (int)__popcll(in[e]);
        in_high[e] = __ballot(p[e] >= high);
        before_high += (int)__popcll(in_high[e] & ((1ull << lane) - 1));
        n_high += (int)__popcll(in_high[e]);
    }
    small = -wave_max(-small);
    if (lane == 0) { red[wave][0] = total; red[wave][1] = (float)n_wave; least[wave] = small; highs[wave] = n_high; }
    __syncthreads();
    int at = blockIdx.x * SEG + before, at_high = blockIdx.x * SEG + before_high;
#pragma unroll
    for (int w = 0; w < 3; ++w)
        if (w < wave) { at += (int)red[w][1]; at_high += highs[w]; }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const bool one = (in[e] >> lane) & 1, two = (in_high[e] >> lane) & 1;
        float power = 0.f;
        if (POW && (one || two)) power = powf(p[e], 1.f / a.temperature);
        if (one) {
            ws.list[at] = p[e];
            if (POW) ws.pow[at] = power;
            ws.idx[at++] = (uint16_t)(4 * threadIdx.x + e);
        }
        if (two) {
            ws.high[at_high] = p[e];
            if (POW) ws.high_pow[at_high] = power;
            ws.high_idx[at_high++] = (uint16_t)(4 * threadIdx.x + e);
        }
    }
    float *part = ws.part + blockIdx.x * PART;
    if (threadIdx.x == 2) part[2 * BOUNDS + 2] = fminf(fminf(least[0], least[1]), fminf(least[2], least[3]));
    if (threadIdx.x < 2) part[2 * BOUNDS + threadIdx.x] = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
    if (wave == 1 && lane < BOUNDS) {   // an entry of bin k reaches the bounds from k on
        unsigned long long sum = 0;
        unsigned n = 0;
#pragma unroll
        for (int k = 0; k < BOUNDS; ++k) {
            sum += k <= lane ? bin_s[k] : 0;
            n += k <= lane ? bin_n[k] : 0;
        }
        part[lane] = from_fixed(sum);
        part[BOUNDS + lane] = (float)n;
    }
}

template <bool POW>
__global__ __launch_bounds__(STHREADS) void sample_draw_kernel(SampleArgs a, SampleWs ws) {
    __shared__ f32x4 red[2][SWAVES / 2];
    __shared__ float seg_sum[SEGS_MAX];
    __shared__ unsigned long long part_s[64 * COPIES], total_s[64];
    __shared__ unsigned part_n[64 * COPIES], total_n[64];
    __shared__ __align__(16) float cols[2 * BOUNDS][SWAVES + 4], few[FEW], sorted[FEW];
    __shared__ int pick, n_few[2];
    const int V = a.V, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), segs = (V + SEG - 1) / SEG;
    const int own = blockIdx.x * SEG + tid;                 // this thread's entry
    at_once({a.seen, a.occ, a.u, a.weight, a.probs, ws.p, ws.high, ws.soft, ws.part});
    // All that does not depend on the cut is requested first and together.  Read where it is used, it was eight trips to memory one
    // after the other, the four parts below among them: 20.7 us a draw, 18.7 now.
    const float p_own = ws.p[own];
    uint8_t seen_own = 0;
    float occ_own = 0.f;
    if (a.seen) {
        seen_own = a.seen[min(own, V - 1)];
        occ_own = a.occ[min(own, V - 1)];
    }
    const float target_u = *a.u;
    const f32x2 soft_own = *(const f32x2 *)(ws.soft + 2 * min(lane, segs - 1));
    float col[SEGS_MAX / SWAVES];
#pragma unroll
    for (int j = 0; j < SEGS_MAX / SWAVES; ++j) col[j] = ws.part[min(wave * (SEGS_MAX / SWAVES) + j, segs - 1) * PART + lane];
    const float *const rest = ws.part + min(lane, segs - 1) * PART + 2 * BOUNDS;   // sum of all, candidates, the smallest of segment `lane`
    const float all_own = rest[0], len_own = rest[1], small_own = rest[2], high_own = rest[HIGH - BOUNDS];
    const float top_p = a.temperature == 0.f ? 0.f : a.top_p;
    // 16 threads a segment hold its list: thread r the entries 64 j + 4 r .. + 3.  The first rounds of the short one are requested
    // before the lengths are known and which list it is to be
    constexpr int EARLY = 2;
    const int sg = tid >> 4, r = tid & 15;
    f32x4 v[SEG / 64];
#pragma unroll
    for (int j = 0; j < EARLY; ++j) v[j] = *(const f32x4 *)(ws.high + min(sg, segs - 1) * SEG + 64 * j + 4 * r);
    if (tid < 2) n_few[tid] = 0;
    if (tid < FEW) few[tid] = 0.f;
    // ---- totals of the segments
    {
        float c = 0.f;
#pragma unroll
        for (int j = 0; j < SEGS_MAX / SWAVES; ++j) {
            if (wave * (SEGS_MAX / SWAVES) + j < segs) c += col[j];
        }
        cols[lane][wave] = c;
    }
    const Soft st = soft_total(soft_own, segs);
    const float pmax = 1.f / st.sum;
    const float all = wave_sum(lane < segs ? all_own : 0.f);
    // token, and the occurrence table: decay, then add the drawn token's weight
    auto store = [&](int tok) {
        if (blockIdx.x == 0 && tid == 0) *a.token = tok;
        if (a.seen && own < V && (seen_own || own == tok)) {
            const float w = own == tok ? (a.weight ? a.weight[tok] : 1.f) : 0.f;
            float o = w;
            if (seen_own) {
                o = occ_own * a.decay;
                if (own == tok) o += w;
            } else {
                a.seen[own] = 1;
            }
            a.occ[own] = o;
        }
    };
    // all: NaN where soft_total left out the NaN of a segment that is masked otherwise
    if (!(st.sum > 0.f && st.sum < INFINITY && all > 0.f)) {
        if (a.probs && own < V) a.probs[own] = 0.f;
        store(0);
        return;
    }
    __syncthreads();
    // ---- which half octave holds the cut: lane k has the sum and the count at bound k
    SumCount at_k = {0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SWAVES; w += 4) {
        const f32x4 x = *(const f32x4 *)&cols[lane & (BOUNDS - 1)][w], y = *(const f32x4 *)&cols[BOUNDS + (lane & (BOUNDS - 1))][w];
        at_k.s += (x[0] + x[1]) + (x[2] + x[3]);
        at_k.n += (y[0] + y[1]) + (y[2] + y[3]);
    }
    // ---- where the nucleus ends at bound HIGH or above it, or is the largest entry alone, the short list has all of it
    const bool nucleus = top_p > 0.f && all >= top_p;
    const bool high = top_p > 0.f && (!nucleus || __ballot(lane <= HIGH && enough(at_k, top_p, -1)) != 0);
    const float *const list = high ? ws.high : ws.list, *const powers = high ? ws.high_pow : ws.pow;
    const uint16_t *const idx = high ? ws.high_idx : ws.idx;
    const float n = wave_sum(lane < segs ? len_own : 0.f);  // candidates
    const float len = lane < segs ? (high ? high_own : len_own) : 0.f;
    const int n_seg = (int)__shfl(len, sg, WAVE), rounds = ((int)wave_max(len) + 63) >> 6;   // rounds: those that any segment has
#pragma unroll
    for (int j = 0; j < SEG / 64; ++j)
        if (j < rounds && (j >= EARLY || !high)) v[j] = *(const f32x4 *)(list + min(sg, segs - 1) * SEG + 64 * j + 4 * r);
#pragma unroll
    for (int j = 0; j < SEG / 64; ++j)
        if (j < rounds) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = 64 * j + 4 * r + e < n_seg ? v[j][e] : 0.f;
        }
    // calls f for every candidate that this thread holds (zeros fill the last round)
    auto each = [&](auto f) {
#pragma unroll
        for (int j = 0; j < SEG / 64; ++j)
            if (j < rounds) {
#pragma unroll
                for (int e = 0; e < 4; ++e) f(v[j][e]);
            }
    };
    int turn = 0;
    auto above = [&](float c) {   // c > 0
        float sc = 0.f;
        unsigned k = 0;
        each([&](float x) {
            const bool in = x >= c;
            sc += in ? x : 0.f;
            k += in ? 1u : 0u;
        });
        return block_total(sc, (float)k, red, turn);
    };
    float cut = pmax;   // as in the kernel above
#pragma unroll 1
    for (int counts = 0; counts < 2; ++counts) {
        const int want = counts ? a.top_k : -1;
        unsigned lo, hi = __float_as_uint(pmax) + 1;
        SumCount at_lo, at_hi = {0.f, 0.f};
        if (!counts) {
            if (!nucleus) continue;
            lo = __float_as_uint(list_floor(top_p, V));
            at_lo = {all, n};
        } else {
            if (!(a.top_k > 0 && a.top_k < V)) continue;
            at_lo = above(cut);
            if (!(at_lo.n > (float)a.top_k)) continue;
            lo = __float_as_uint(cut);
        }
        const unsigned long long holds = __ballot(lane < BOUNDS && enough(at_k, top_p, want));
        const int k = holds ? __builtin_ctzll(holds) : BOUNDS;
        if (k < BOUNDS && __float_as_uint(bound_at(pmax, k)) > lo) {
            lo = __float_as_uint(bound_at(pmax, k));
            at_lo = {__shfl(at_k.s, k, WAVE), __shfl(at_k.n, k, WAVE)};
        }
        if (k > 0) {
            hi = __float_as_uint(bound_at(pmax, k - 1));
            at_hi = {__shfl(at_k.s, k - 1, WAVE), __shfl(at_k.n, k - 1, WAVE)};
        }
        if (!counts && at_lo.n == n && n - at_hi.n > (float)FEW)   // all candidates reach lo: begin at the smallest of them
            lo = max(lo, __float_as_uint(-wave_max(lane < segs ? -small_own : -INFINITY)));
        while (hi - lo > 1 && at_lo.n - at_hi.n > (float)FEW) {
            // Sums and counts of up to 64 equal parts of the interval.  us a draw, one workgroup / bisection down to 1024 entries and a
            // list of these / this: 65536 equal logits, top_p 0.7 67 / 68 / 34, 50277 of them 58 / 67 / 33; 50277 from N(0, 3),
            // top_p 0.999 40.6 / 49.3 / 41.1 (58.5 from 0 up instead of list_floor: three parts take all additions).  Logits closer to
            // each other than that fell into two or three parts, whose additions wait for each other: so the interval begins at the
            // smallest candidate, and a part has COPIES sums, each for four lanes of a wave.  50277 from N(0, 0.003), top_p 0.7, one workgroup /
            // neither / the former / both 51 / 117 / 57.5 / 50.7, N(0, 0.03) 46.4 / 61.7 / 54.9 / 49.7, N(0, 0.3) 42.0 / 42.0 / 42.3 /
            // 43.5, equal ones 58 / 33 / 19 / 19, N(0, 3) 32.0 / 16.2 / 16.3 / 16.4.
            const int shift = max(26 - __builtin_clz(hi - lo - 1), 0);
            const float flo = __uint_as_float(max(lo, 1u)), fhi = __uint_as_float(hi);
            static_assert(64 * COPIES == STHREADS, "a thread clears and adds up a copy");
            part_s[tid] = 0;
            part_n[tid] = 0;
            __syncthreads();
            each([&](float x) {
                const bool in = x >= flo && x < fhi;
                const unsigned long long m = __ballot(in);
                if (!m) return;
                const unsigned first = (unsigned)__builtin_amdgcn_readlane(__builtin_bit_cast(int, x), __builtin_ctzll(m));
                const bool ties = __ballot(in && __float_as_uint(x) != first) == 0;   // else an addition each
                const int n = ties ? (int)__popcll(m) : 1;
                if (ties ? lane == 0 : in) {
                    const float y = ties ? __uint_as_float(first) : x;
                    const unsigned part = ((__float_as_uint(y) - lo) >> shift) * COPIES + (lane & (COPIES - 1));
                    atomicAdd(&part_s[part], (unsigned long long)n * fixed(y));
                    atomicAdd(&part_n[part], (unsigned)n);
                }
            });
            __syncthreads();
            {
                const unsigned long long s = row16_total(part_s[tid]);
                const unsigned n = row16_total(part_n[tid]);
                if ((tid & (COPIES - 1)) == 0) { total_s[tid / COPIES] = s; total_n[tid / COPIES] = n; }
            }
            __syncthreads();
            // lane i: the part i from above, and the sum and the count from its lower end on
            const SumCount t = {at_hi.s + wave_scan(from_fixed(total_s[63 - lane])), at_hi.n + wave_scan((float)total_n[63 - lane])};
            const unsigned long long good = __ballot(enough(t, top_p, want));
            const int i = good ? __builtin_ctzll(good) : 63;
            if (good) at_lo = {__shfl(t.s, i, WAVE), __shfl(t.n, i, WAVE)};
            if (i > 0) at_hi = {__shfl(t.s, i - 1, WAVE), __shfl(t.n, i - 1, WAVE)};
            hi = min(hi, lo + ((unsigned)(64 - i) << shift));
            lo += (unsigned)(63 - i) << shift;
            __syncthreads();   // the parts have been read
        }
        if (hi - lo > 1) {
            // the entries of the interval, at most FEW, in any order at first
            unsigned ulo = max(lo, 1u);
            const unsigned span = hi - ulo;   // positive floats order like their bits, and 0 falls out
            auto inside = [&](float x) { return __float_as_uint(x) - ulo < span; };
            int mine = 0;
            each([&](float x) { mine += inside(x) ? 1 : 0; });
            const float upto = wave_scan((float)mine);
            const int of_wave = (int)last_lane(upto);
            if (of_wave) {
                int at = 0;
                if (lane == 0) at = atomicAdd(&n_few[counts], of_wave);
                at = __builtin_amdgcn_readfirstlane(at) + (int)upto - mine;
                asm volatile("" : "+v"(ulo));   // 64 masks kept from the count would not fit the scalar registers
#pragma unroll
                for (int j = 0; j < SEG / 64; ++j)
                    if (j < rounds && (inside(v[j][0]) || inside(v[j][1]) || inside(v[j][2]) || inside(v[j][3]))) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (inside(v[j][e])) few[min(at++, FEW - 1)] = v[j][e];
                    }
            }
            __syncthreads();
            // sorted by counting the larger ones (four threads an entry), then added from the largest down
            const int m = min(n_few[counts], FEW), own_few = tid >> 2, q4 = tid & 3;
            if (16 * wave < m) {
                // A place is the number of larger entries and of equal ones ahead of it: y >= x is y > x - 1 in bits, for the groups of
                // four ahead of its own.  Two instructions a comparison; places from m on hold zeros, which are never larger.
                typedef int i32x4 __attribute__((ext_vector_type(4)));
                const int x = __float_as_int(few[own_few]), group = own_few & ~3;
                int rank = 0;
#pragma unroll 4
                for (int i = 4 * q4; i < m; i += 16) {
                    const i32x4 y = *(const i32x4 *)&few[i];
                    const int than = i < group ? x - 1 : x;
#pragma unroll
                    for (int e = 0; e < 4; ++e) rank += y[e] > than ? 1 : 0;
                }
                if (group % 16 == 4 * q4) {
#pragma unroll
                    for (int e = 0; e < 3; ++e) rank += e < own_few - group && __float_as_int(few[group + e]) == x ? 1 : 0;
                }
                rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xf, 0xf, true);
                rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xf, 0xf, true);
                if (q4 == 0 && own_few < m) sorted[rank] = __int_as_float(x);
            }
            __syncthreads();
            const f32x4 y = *(const f32x4 *)&sorted[4 * lane];
            float in4[4], four = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                in4[e] = 4 * lane + e < m ? y[e] : 0.f;
                four += in4[e];
            }
            float sum = at_hi.s + (wave_scan(four) - four), at = -1.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum += in4[e];
                if (at < 0.f && in4[e] > 0.f && enough(SumCount{sum, at_hi.n + (float)(4 * lane + e + 1)}, top_p, want)) at = in4[e];
            }
            const unsigned long long good = __ballot(at > 0.f);
            if (good) lo = (unsigned)__builtin_amdgcn_readlane(__builtin_bit_cast(int, at), __builtin_ctzll(good));
            if (!counts && tid < FEW) few[tid] = 0.f;   // read ahead of the last barrier, written past the next one
        }
        cut = __uint_as_float(lo);
    }
    // ---- filter, temperature, sums of the segments
    auto keep = [&](float x) { return x >= cut && x > 0.f; };
    {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < SEG / 64; ++j)
            if (j < rounds) {
                f32x4 q = v[j];
                if (POW) q = *(const f32x4 *)(powers + min(sg, segs - 1) * SEG + 64 * j + 4 * r);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum += keep(v[j][e]) ? q[e] : 0.f;
            }
        sum = row16_sum(sum);
        if (r == 0) seg_sum[sg] = sum;
    }
    if (!POW && a.probs && own < V) a.probs[own] = keep(p_own) ? p_own : 0.f;
    __syncthreads();
    // ---- draw: first index whose running sum exceeds u * total; the last kept entry where rounding leaves none
    if (wave == 0) {
        const float mine = seg_sum[lane], upto = wave_scan(mine), target = target_u * last_lane(upto);
        const unsigned long long hit = __ballot(mine > 0.f && upto > target), some = __ballot(mine > 0.f);
        const int from = hit ? __builtin_ctzll(hit) : (some ? 63 - __builtin_clzll(some) : 0);
        float run = __shfl(upto - mine, from, WAVE);
        const int end = (int)__shfl(len, from, WAVE);
        int found = -1, last = 0;                 // places in the segment
        for (int i0 = 0; i0 < end && found < 0; i0 += 256) {   // four entries a lane
            const int i = i0 + 4 * lane;
            f32x4 q = *(const f32x4 *)(list + from * SEG + i), w = q;
            if (POW) w = *(const f32x4 *)(powers + from * SEG + i);
            const uint2 id = *(const uint2 *)(idx + from * SEG + i);
            const int ids[4] = {(int)(id.x & 0xffff), (int)(id.x >> 16), (int)(id.y & 0xffff), (int)(id.y >> 16)};
#pragma unroll
            for (int e = 0; e < 4; ++e) q[e] = i + e < end && keep(q[e]) ? w[e] : 0.f;
            const float mine4 = (q[0] + q[1]) + (q[2] + q[3]), up = wave_scan(mine4);
            float at = run + (up - mine4);
            int f = -1, l = -1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                at += q[e];
                if (q[e] > 0.f) {
                    l = ids[e];
                    if (f < 0 && at > target) f = ids[e];
                }
            }
            const unsigned long long over = __ballot(f >= 0), any = __ballot(l >= 0);
            if (hit && over) found = __shfl(f, __builtin_ctzll(over), WAVE);
            if (any) last = __shfl(l, 63 - __builtin_clzll(any), WAVE);
            run += last_lane(up);
        }
        if (lane == 0) pick = some ? from * SEG + (found >= 0 ? found : last) : 0;
    }
    __syncthreads();
    store(pick);
    if (POW && a.probs && own < V) a.probs[own] = keep(p_own) ? powf(p_own, 1.f / a.temperature) : 0.f;
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

static int sample_args(SampleArgs &a, const float *logits, int64_t V, float temperature, float top_p, int32_t top_k,
                       const int32_t *token_ban, int32_t n_ban, uint8_t *seen, float *occurrence, const float *token_weight,
                       float alpha_presence, float alpha_frequency, float alpha_decay, const float *u, float *probs, int32_t *token) {
    if (!logits || !u || !token) return RWKV_E_NULL;
    if (V <= 0 || V > (int64_t)STHREADS * 4 * ROWS_MAX || n_ban < 0 || (n_ban > 0 && !token_ban)) return RWKV_E_SHAPE;
    if ((seen == nullptr) != (occurrence == nullptr)) return RWKV_E_NULL;
    if (!(temperature >= 0.f) || top_k < 0) return RWKV_E_SHAPE;
    a = SampleArgs{logits, (int)V, temperature, top_p, top_k, token_ban, n_ban, seen, occurrence, token_weight,
                   alpha_presence, alpha_frequency, alpha_decay, u, probs, token};
    return RWKV_OK;
}

extern "C" int rwkv_sample_logits(const float *logits, int64_t V, float temperature, float top_p, int32_t top_k,
                                  const int32_t *token_ban, int32_t n_ban, uint8_t *seen, float *occurrence,
                                  const float *token_weight, float alpha_presence, float alpha_frequency,
                                  float alpha_decay, const float *u, float *probs, int32_t *token, void *stream) {
    SampleArgs a;
    const int rc = sample_args(a, logits, V, temperature, top_p, top_k, token_ban, n_ban, seen, occurrence, token_weight,
                               alpha_presence, alpha_frequency, alpha_decay, u, probs, token);
    if (rc) return rc;
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

static size_t sample_ws(SampleWs &ws, void *base, int64_t V) {
    const size_t segs = (size_t)((V + SEG - 1) / SEG), n = segs * SEG;
    ws.p = (float *)base;
    ws.list = ws.p + n;
    ws.pow = ws.list + n;
    ws.high = ws.pow + n;
    ws.high_pow = ws.high + n;
    ws.idx = (uint16_t *)(ws.high_pow + n);
    ws.high_idx = ws.idx + n;
    ws.soft = (float *)(ws.high_idx + n);
    ws.part = ws.soft + 2 * segs;
    return (5 * n + segs * (PART + 2)) * sizeof(float) + 2 * n * sizeof(uint16_t);
}

extern "C" size_t rwkv_sample_workspace(int64_t V) {
    SampleWs ws;
    return V > 0 && V <= SEG * SEGS_MAX ? sample_ws(ws, nullptr, V) : 0;
}

extern "C" int rwkv_sample_logits_ws(const float *logits, int64_t V, float temperature, float top_p, int32_t top_k,
                                     const int32_t *token_ban, int32_t n_ban, uint8_t *seen, float *occurrence,
                                     const float *token_weight, float alpha_presence, float alpha_frequency, float alpha_decay,
                                     const float *u, float *probs, int32_t *token, void *workspace, size_t workspace_bytes,
                                     void *stream) {
    SampleArgs a;
    const int rc = sample_args(a, logits, V, temperature, top_p, top_k, token_ban, n_ban, seen, occurrence, token_weight,
                               alpha_presence, alpha_frequency, alpha_decay, u, probs, token);
    if (rc) return rc;
    if (!workspace) return RWKV_E_NULL;
    if (workspace_bytes < rwkv_sample_workspace(V) || !aligned16(workspace)) return RWKV_E_WORKSPACE;
    // One workgroup: vocabularies that are four entries a thread there, and cuts that leave (almost) everything.
    if (V <= 4 * 4 * STHREADS || (temperature != 0.f && !(top_p <= 0.999f)))
        return rwkv_sample_logits(logits, V, temperature, top_p, top_k, token_ban, n_ban, seen, occurrence, token_weight, alpha_presence,
                                  alpha_frequency, alpha_decay, u, probs, token, stream);
    hipStream_t st = (hipStream_t)stream;
    SampleWs ws;
    sample_ws(ws, workspace, V);
    const dim3 grid((unsigned)((V + SEG - 1) / SEG));
    const bool pow = temperature != 0.f && temperature != 1.f;
    hipLaunchKernelGGL(sample_adjust_kernel, grid, dim3(256), 0, st, a, ws);
    if (pow) {
        hipLaunchKernelGGL(sample_probs_kernel<true>, grid, dim3(256), 0, st, a, ws);
        hipLaunchKernelGGL(sample_draw_kernel<true>, grid, dim3(STHREADS), 0, st, a, ws);
    } else {
        hipLaunchKernelGGL(sample_probs_kernel<false>, grid, dim3(256), 0, st, a, ws);
        hipLaunchKernelGGL(sample_draw_kernel<false>, grid, dim3(STHREADS), 0, st, a, ws);
    }
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
}
