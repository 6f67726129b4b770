// The FULL path's selection: rows that keep the head of the descending order
// (top-k, or top-p over the whole vocabulary; select_eligible). k_full_pass has
// counted the row into bins (select_bins.h); then
//
//   k_full_gather  (chunks x rows)  picks the bin the head reaches down to,
//                                   reads the row again (from the caches while
//                                   the batch fits them) and collects the
//                                   elements of the bins down to it; for top-p
//                                   it sums the exact p of all the others
//   k_full_head    (groups x rows)  sorts what was collected and finishes the
//                                   row: p, cut, min-p, total, draw
//                                   (sample.rs:279-358); a head of up to
//                                   SEL_FIN_CAP elements in one workgroup's
//                                   LDS, a longer one a group at a time
//                                   (full_head.h)
//   k_full_rest    (rows)           sorts whole the rows that this does not
//                                   decide
//
// Before, k_full_rest sorted every such row: four radix passes over the
// vocabulary on one CU. A call over one row of 248 320 at top-p 0.95 went from
// 1347 to 35 us, 24 unaligned rows of 151 935 at top-p 0.9 from 899 to 47-50 us,
// 16 rows of 248 320 at top-k 100 from 928 to 40 us. What bounds it now: four
// launches and, in each, one chain of dependent steps (about 10, 9, 10 and 2 us
// at one row); the logits' two reads are a small part.
//
// Measured and not kept: the finish in the gather's last chunk to arrive (the
// stores' wait, the arrival and the loads behind it took 3-4 us more than the
// next launch does); the finish inside k_full_rest (its old passes then spill
// 271 registers and the 256-row ties batch goes from 385 to 600 us).
//
// The top-p cut needs the mass of the whole row, in the reference's order of
// addition. The collected elements come first in that order and every p is the
// reference's f32 value, so the running sums along them are exact (or
// replayed), and the target top_p * mass lies in an interval of a few parts in
// 10^11 around the sum of all p in any order (sel_target_interval): the cut is
// taken when its two ends agree on it.
#pragma once
#include "full_kernels.h"

namespace rl {

constexpr uint32_t SEL_THREADS = 1024;
constexpr uint32_t SEL_WAVES = SEL_THREADS / WAVE;
constexpr uint32_t SEL_FIN_CAP = SEL_GROUP;          // elements finished in LDS
constexpr uint32_t SEL_U = 2;                        // float4 per thread per step of the gather
constexpr uint32_t SEL_STEP = SEL_THREADS * SEL_U;   // float4 per step
constexpr uint32_t SORT_BUCKETS = 4096;
constexpr uint32_t SORT_CROWD = 192;                 // a bucket above this is sorted by the network

// ------------------------------------------------------ block helpers ---
template <uint32_t NT>
__device__ __forceinline__ uint32_t block_sum_u32(uint32_t v, RL_LDS uint32_t *red) {
    v = wave_sum_u32(v);
    __syncthreads();
    if (lane_id() == 0) red[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint32_t t = 0;
    for (uint32_t w = 0; w < NT / WAVE; ++w) t += red[w];
    return t;
}

template <uint32_t NT>
__device__ __forceinline__ int64_t block_max_i64(int64_t v, RL_LDS int64_t *red) {
    v = (int64_t)wave_fold_u64((uint64_t)v, [](uint64_t a, uint64_t b) { return (int64_t)a > (int64_t)b ? a : b; });
    __syncthreads();
    if (lane_id() == 0) red[threadIdx.x / WAVE] = v;
    __syncthreads();
    int64_t t = red[0];
    for (uint32_t w = 1; w < NT / WAVE; ++w) t = red[w] > t ? red[w] : t;
    return t;
}

// Exclusive prefix of v over the workgroup's threads in thread order; *total
// gets the sum. For doubles it is only used where every partial sum is exact.
template <uint32_t NT, class T>
__device__ __forceinline__ T block_exclusive(T v, RL_LDS T *red, T *total) {
    const uint32_t lane = lane_id(), wave = threadIdx.x / WAVE;
    T incl;
    if constexpr (std::is_same<T, double>::value) {
        incl = wave_incl_f64(v);
    } else {
        static_assert(std::is_same<T, uint32_t>::value, "u32 or f64");
        incl = wave_incl_u32(v);
    }
    __syncthreads();
    if (lane == WAVE - 1) red[wave] = incl;
    __syncthreads();
    T before = 0, all = 0;
    for (uint32_t w = 0; w < NT / WAVE; ++w) {
        if (w < wave) before += red[w];
        all += red[w];
    }
    *total = all;
    return before + incl - v;
}

// Where every partial sum of the probabilities is exact: the first j in
// [lo, hi) with base + p[lo] + ... + p[j] >= target, and that sum in *at; or
// hi, with the sum of them all in *at. Any order of addition gives these exact
// sums, so a block scan serves. Whole workgroup.
template <uint32_t NT>
__device__ __forceinline__ uint32_t exact_first_reaching(const float *probs, uint32_t lo, uint32_t hi, double base,
                                                         double target, RL_LDS double *red, RL_LDS uint32_t *hit,
                                                         RL_LDS double *hit_sum, double *at, const HotRange &hr) {
    for (uint32_t b = lo; b < hi; b += NT * CI) {
        const uint32_t j0 = b + threadIdx.x * CI;
        float pv[CI];
        double mine = 0.0;
#pragma unroll
        for (uint32_t i = 0; i < CI; ++i) {
            uint32_t w = hr.word;
            if (j0 + i < hi && !hr.has(j0 + i)) w = ((const RL_GLB uint32_t *)probs)[j0 + i];
            pv[i] = j0 + i < hi ? __uint_as_float(w) : 0.0f;
            mine += (double)pv[i];
        }
        if (threadIdx.x == 0) *hit = 0xFFFFFFFFu;
        double step_total;
        double c = base + block_exclusive<NT, double>(mine, red, &step_total);
        uint32_t my_hit = 0xFFFFFFFFu;
        double my_sum = 0.0;
#pragma unroll
        for (uint32_t i = 0; i < CI; ++i) {
            if (my_hit == 0xFFFFFFFFu && j0 + i < hi) {
                c += (double)pv[i];
                if (c >= target) {
                    my_hit = j0 + i;
                    my_sum = c;
                }
            }
        }
        if (my_hit != 0xFFFFFFFFu) atomicMin((uint32_t *)hit, my_hit);
        __syncthreads();
        const uint32_t h = *hit;
        if (h != 0xFFFFFFFFu) {
            if (my_hit == h) *hit_sum = my_sum;
            __syncthreads();
            *at = *hit_sum;
            __syncthreads();
            return h;
        }
        base += step_total;
        __syncthreads();
    }
    *at = base;
    return hi;
}

// A thread's share of the candidate list's statistics (those kept in LDS
// beside the segments): p at index j seen by add.
struct PStats {
    int emin = 1 << 20;
    uint32_t bad = 0, count = 0, last_in = 0, first_out = 0xFFFFFFFFu;
    __device__ __forceinline__ void add(float p, uint32_t j, float min_p) {
        if (!(p <= 3.40282347e38f)) {
            bad = 1;  // NaN or +inf
        } else if (p > 0.0f) {
            emin = min(emin, f32_exponent(p));
        }
        if (p >= min_p) {
            ++count;
            last_in = max(last_in, j + 1);
        } else {
            first_out = min(first_out, j);
        }
    }
    // Folds the wave's shares into L's (lane 0 adds them with LDS atomics,
    // after L's were set by stats_reset and a barrier).
    template <class Lds>
    __device__ __forceinline__ void merge(RL_LDS Lds *L) {
        emin = (int)wave_fold_u32((uint32_t)emin, [](uint32_t a, uint32_t b) { return (int)a < (int)b ? a : b; });
        bad = wave_fold_u32(bad, [](uint32_t a, uint32_t b) { return a | b; });
        count = wave_sum_u32(count);
        last_in = wave_fold_u32(last_in, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
        first_out = wave_fold_u32(first_out, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
        if (lane_id() == 0) {
            atomicMin((int *)&L->st_emin, emin);
            atomicOr((uint32_t *)&L->st_bad, bad);
            atomicAdd((uint32_t *)&L->st_count, count);
            atomicMax((uint32_t *)&L->st_last_in, last_in);
            atomicMin((uint32_t *)&L->st_first_out, first_out);
        }
    }
};

// The list statistics before any merge (one thread).
template <class Lds>
__device__ __forceinline__ void stats_reset(RL_LDS Lds *L) {
    L->st_emin = 1 << 20;
    L->st_bad = 0;
    L->st_count = 0;
    L->st_last_in = 0;
    L->st_first_out = 0xFFFFFFFFu;
}

// ---------------------------------------------------------- the sort ---
struct SortLds {
    uint32_t start[SORT_BUCKETS + 1];  // per bucket: its elements, then where it starts
    float lo[SEL_WAVES], hi[SEL_WAVES];
    uint32_t sum[SEL_WAVES], most[SEL_WAVES];
};

// Sorts n composites (n <= E * SEL_THREADS), descending, into v (LDS, room for
// the next power of two from n): x[q] is element q * SEL_THREADS + tid. Whole
// workgroup; ends with a barrier.
//
// The logits are spread linearly over SORT_BUCKETS buckets between the largest
// and the smallest, each element takes a slot of its bucket from an LDS
// counter, and its place is the bucket's start plus the number of the bucket's
// composites above it. A head's logits thin out smoothly towards the top, so a
// bucket holds a few elements: a handful of LDS accesses an element and six
// barriers, against 78 stages of a sorting network at 4096. (Spread by key
// instead, whose octaves around zero are as wide as those of the large logits,
// heads that reach below zero crowded: 932 elements took 7.4 us.) A crowded
// bucket (ties, an outlier far above the rest) sends the sort to the network.
template <uint32_t E>
__device__ __forceinline__ void bucket_sort(const uint64_t (&x)[E], uint32_t n, RL_LDS uint64_t *v,
                                            RL_LDS SortLds *L) {
    constexpr uint32_t PER = SORT_BUCKETS / SEL_THREADS;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    float lo = __builtin_inff(), hi = -__builtin_inff();  // finite: no logit is NaN or +inf here
#pragma unroll
    for (uint32_t q = 0; q < E; ++q)
        if (q * SEL_THREADS + tid < n) {
            const float l = key_value(comp_key(x[q]));
            if (l > -__builtin_inff()) lo = fminf(lo, l);
            hi = fmaxf(hi, l);
        }
    hi = wave_maxnum_f32(hi);
    lo = -wave_maxnum_f32(-lo);
    if (lane == 0) {
        L->lo[wave] = lo;
        L->hi[wave] = hi;
    }
    for (uint32_t i = tid; i < SORT_BUCKETS; i += SEL_THREADS) L->start[i] = 0;
    __syncthreads();
    for (uint32_t w = 0; w < SEL_WAVES; ++w) {
        lo = fminf(lo, L->lo[w]);
        hi = fmaxf(hi, L->hi[w]);
    }
    // The bucket of a logit: its distance from the largest times the buckets
    // per unit, cut at the last (which takes -inf too). It never falls as the
    // logit falls: each step is one rounding of a monotone function. Equal
    // logits (-0 and +0 as well) share a bucket.
    const float scale = fminf((float)SORT_BUCKETS / (hi - lo), 3.0e38f);
    auto bucket = [&](uint64_t c) {
        return (uint32_t)fminf((hi - key_value(comp_key(c))) * scale, (float)(SORT_BUCKETS - 1));
    };
    uint32_t at[E];
#pragma unroll
    for (uint32_t q = 0; q < E; ++q)
        if (q * SEL_THREADS + tid < n) at[q] = atomicAdd((uint32_t *)&L->start[bucket(x[q])], 1u);
    __syncthreads();
    // The buckets' starts, and the fullest.
    uint32_t c[PER], mine = 0, most = 0;
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        c[i] = L->start[tid * PER + i];
        mine += c[i];
        most = max(most, c[i]);
    }
    const uint32_t incl = wave_incl_u32(mine);
    most = wave_fold_u32(most, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
    if (lane == WAVE - 1) {
        L->sum[wave] = incl;
        L->most[wave] = most;
    }
    __syncthreads();
    uint32_t run = incl - mine;
    for (uint32_t w = 0; w < SEL_WAVES; ++w) {
        if (w < wave) run += L->sum[w];
        most = max(most, L->most[w]);
    }
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        L->start[tid * PER + i] = run;
        run += c[i];
    }
    if (tid == SEL_THREADS - 1) L->start[SORT_BUCKETS] = run;
    __syncthreads();
    if (most > SORT_CROWD) {
        uint32_t n2 = 1;
        while (n2 < n) n2 <<= 1;
#pragma unroll
        for (uint32_t q = 0; q < E; ++q) {
            const uint32_t i = q * SEL_THREADS + tid;
            if (i < n2) v[i] = i < n ? x[q] : 0ull;
        }
        __syncthreads();
        lds_bitonic_desc(v, n2, SEL_THREADS);
        return;
    }
#pragma unroll
    for (uint32_t q = 0; q < E; ++q)
        if (q * SEL_THREADS + tid < n) v[L->start[bucket(x[q])] + at[q]] = x[q];
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < E; ++q)
        if (q * SEL_THREADS + tid < n) {
            const uint32_t b = bucket(x[q]);
            const uint32_t j0 = L->start[b], j1 = L->start[b + 1];
            uint32_t r = j0;
            for (uint32_t j = j0; j < j1; ++j) r += v[j] > x[q] ? 1u : 0u;
            at[q] = r;
        }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < E; ++q)
        if (q * SEL_THREADS + tid < n) v[at[q]] = x[q];
    __syncthreads();
}

// Sorts n <= SORT_FEW composites, descending, into v: x is element tid. Whole
// workgroup; ends with a barrier. An element's place is the number of those
// above it: n reads of LDS at one address, with none of the buckets' six
// barriers and clearing (1 x 248320 at top-p 0.95, a head of 97: 37.7 -> 36.3 us
// a call with the finish's one candidate a thread).
constexpr uint32_t SORT_FEW = 256;
__device__ __forceinline__ void count_sort(uint64_t x, uint32_t n, RL_LDS uint64_t *v) {
    const uint32_t tid = threadIdx.x;
    if (tid < n) v[tid] = x;
    __syncthreads();
    uint32_t r = 0;
    if (tid < n) {
#pragma unroll 4
        for (uint32_t j = 0; j < n; ++j) r += v[j] > x ? 1u : 0u;
    }
    __syncthreads();
    if (tid < n) v[r] = x;
    __syncthreads();
}

// --------------------------------------------------------- the finish ---
constexpr uint32_t DRAW_BLOCK = 32;

struct FinishLds {
    uint64_t v[SEL_FIN_CAP];                  // the elements, sorted
    __attribute__((aligned(16))) uint32_t p[SEL_FIN_CAP + DRAW_BLOCK];  // their p, then q (f32 words)
    SortLds sort;
    uint64_t exp_tab[32];
    double red_d[SEL_WAVES];
    uint32_t red_u[SEL_WAVES];
    uint32_t pre[FULL_CHUNKS + 1];            // elements in the chunks before
    uint32_t sh_hit, sh_in, sh_out;
    double sh_at;
};

// The draw (sample.rs:349-358) over the m terms q[0..m) in LDS: the index of
// the first whose running f32 sum exceeds u, or m - 1. q is 16-byte aligned and
// holds zeros from m to the next multiple of DRAW_BLOCK. One wave, every lane
// alike: the sum is one chain of additions, so the rest is kept off it: the
// next block's reads are in flight, and only a block's last sum is compared
// (the sums never fall).
__device__ __forceinline__ uint32_t draw_walk(RL_LDS const uint32_t *q, uint32_t m, float u) {
    typedef float vf4 __attribute__((ext_vector_type(4)));
    vf4 nx[DRAW_BLOCK / 4];
#pragma unroll
    for (uint32_t i = 0; i < DRAW_BLOCK / 4; ++i) nx[i] = *(RL_LDS const vf4 *)&q[4 * i];
    float run = 0.0f;
    for (uint32_t j = 0; j < m; j += DRAW_BLOCK) {
        vf4 x[DRAW_BLOCK / 4];
#pragma unroll
        for (uint32_t i = 0; i < DRAW_BLOCK / 4; ++i) x[i] = nx[i];
        const uint32_t jn = j + DRAW_BLOCK < m ? j + DRAW_BLOCK : j;
#pragma unroll
        for (uint32_t i = 0; i < DRAW_BLOCK / 4; ++i) nx[i] = *(RL_LDS const vf4 *)&q[jn + 4 * i];
        float c = run;
#pragma unroll
        for (uint32_t i = 0; i < DRAW_BLOCK; ++i) c += x[i / 4][i & 3u];
        if (c > u) {
            c = run;
            uint32_t hit = DRAW_BLOCK;
#pragma unroll
            for (uint32_t i = 0; i < DRAW_BLOCK; ++i) {
                c += x[i / 4][i & 3u];
                if (hit == DRAW_BLOCK && c > u) hit = i;
            }
            return min(j + hit, m - 1);
        }
        run = c;
    }
    return m - 1;
}

// The finish of a row of n <= SEL_FIN_CAP collected elements by one
// workgroup: L->v holds them sorted, tail is the sum of every other p (0 for
// top-k). Returns false (nothing written) when the row is not decided here.
__device__ __forceinline__ bool finish_selected(const RowIO &a, uint32_t row, const rl_sampling &s, float M, uint32_t n,
                                                double tail, RL_LDS FinishLds *L) {
    constexpr uint32_t PER = SEL_FIN_CAP / SEL_THREADS;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t V = a.vocab, k = full_k(s, V);
    const bool by_k = k < V;
    const uint32_t kk = by_k ? k : n;  // the candidates
    if (n < kk) return false;
    const LdsExpTable etab{(RL_LDS uint64_t *)L->exp_tab};
    const TempScale tscale(s.temperature);
    const bool min_on = s.min_p > 0.0f;
    // Thread t holds the candidates per t ..: p, what min-p and the sums'
    // exactness depend on, and their f64 sum. One each up to 1024 of them: their
    // p are one chain of latencies then, not PER.
    const uint32_t per = kk <= SEL_THREADS ? 1u : PER;
    float p[PER];
    const float u = ((const RL_GLB float *)a.uniforms)[row];
    int emin = 1 << 20;
    bool bad = false;
    double mine = 0.0;
    if (tid == 0) {
        L->sh_hit = 0xFFFFFFFFu;
        L->sh_in = 0;
        L->sh_out = 0xFFFFFFFFu;
    }
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        p[i] = 0.0f;
        if (i >= per) continue;
        const uint32_t j = tid * per + i;
        if (j < kk) {
            p[i] = expf_libm_t(tscale(key_value(comp_key(L->v[j])) - M), etab);
            if (!(p[i] <= 3.40282347e38f)) bad = true;
            else if (p[i] > 0.0f) emin = min(emin, f32_exponent(p[i]));
            mine += (double)p[i];
        }
        L->p[j] = __float_as_uint(p[i]);
    }
    // The smallest exponent, or INT_MIN for a NaN or infinite p.
    emin = bad ? (int)0x80000000u : emin;
    emin = wave_min_i32(emin);
    if (lane == 0) L->red_u[wave] = (uint32_t)emin;
    double list;
    const double before = block_exclusive<SEL_THREADS, double>(mine, (RL_LDS double *)L->red_d, &list);
    for (uint32_t w = 0; w < SEL_WAVES; ++w) emin = min(emin, (int)L->red_u[w]);
    if (emin == (int)0x80000000u) return false;
    // Every p a multiple of 2^(emin - 23) and their sum below 2^53 of those:
    // every partial sum is exact in any order. Else the sums are replayed
    // in order, every wave alike.
    const bool exact = emin > 1000 || list < mul_pow2(1.0 - 0x1p-30, 30 + emin);
    RL_LDS const uint32_t *pw = (RL_LDS const uint32_t *)L->p;
    // The first of the first n sums to reach `stop`, or n, and that sum: one
    // wave's work (by every wave alike, four to a SIMD, 26 x 7552 at temperature
    // 0.52, top-k 1904, took 119 us a call, 79 so; wave_walk's passes took 20
    // less, and their code cost a head of 100 that never runs it 0.3).
    auto replay = [&](uint32_t n, double stop, double *sum) {
        if (wave == 0) {
            double c = 0.0;
            const uint32_t j = seq_walk<53>(pw, n, [stop](double x) { return x >= stop; }, c);
            if (lane == 0) {
                L->sh_at = c;
                L->sh_hit = j;
            }
        }
        __syncthreads();
        const uint32_t j = L->sh_hit;
        *sum = L->sh_at;
        __syncthreads();
        return j;
    };
    uint32_t m = kk;
    double total = list;
    bool have_total = exact;
    if (s.top_p < 1.0f) {
        double t_lo, t_hi;
        if (by_k) {
            if (__builtin_expect(!exact, 0)) replay(kk, __builtin_inf(), &list);
            t_lo = t_hi = (double)s.top_p * list;  // the candidates' mass, in order
        } else {
            sel_target_interval(tail + list, V, s.top_p, &t_lo, &t_hi);
        }
        uint32_t j;
        if (__builtin_expect(exact, 1)) {
            double c = before;
            uint32_t hit = 0xFFFFFFFFu;
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) {
                c += (double)p[i];
                if (hit == 0xFFFFFFFFu && i < per && tid * per + i < kk && c >= t_lo) {
                    hit = tid * per + i;
                    mine = c;
                }
            }
            // The first in the workgroup: the first lane of the first wave
            // that has one (later threads' sums only grow).
            const uint64_t hm = ballot(hit != 0xFFFFFFFFu);
            if (hm != 0 && lane == (uint32_t)__builtin_ctzll(hm)) atomicMin((uint32_t *)&L->sh_hit, hit);
            __syncthreads();
            j = L->sh_hit;
            if (j == hit && hit != 0xFFFFFFFFu) L->sh_at = mine;
            __syncthreads();
            total = L->sh_at;
        } else {
            j = replay(kk, t_lo, &total);
            if (j >= kk) j = 0xFFFFFFFFu;
        }
        if (j == 0xFFFFFFFFu) {
            if (!by_k) return false;  // the head does not reach the target
            total = list;             // a mass the running sum never reaches: no cut
        } else {
            if (!(total >= t_hi)) return false;  // the cut could fall on either side
            m = j + 1;
        }
        have_total = true;
    }
    if (min_on) {
        // Survivors are the first m with p >= min_p, a prefix (p falls along
        // the order; checked, not assumed).
        uint32_t in = 0, out = 0xFFFFFFFFu;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t j = tid * per + i;
            if (i < per && j < m) {
                if (p[i] >= s.min_p) in = j + 1;
                else out = min(out, j);
            }
        }
        in = wave_fold_u32(in, [](uint32_t x, uint32_t y) { return x > y ? x : y; });
        out = wave_fold_u32(out, [](uint32_t x, uint32_t y) { return x < y ? x : y; });
        if (lane == 0) {
            atomicMax((uint32_t *)&L->sh_in, in);
            atomicMin((uint32_t *)&L->sh_out, out);
        }
        __syncthreads();
        in = L->sh_in;
        if (in > L->sh_out) return false;
        const uint32_t w = in > 1 ? in : 1u;
        if (w != m) have_total = false;
        m = w;
    }
    if (!have_total) {
        if (__builtin_expect(exact, 1)) {
            double part = 0.0;
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) part += i < per && tid * per + i < m ? (double)p[i] : 0.0;
            block_exclusive<SEL_THREADS, double>(part, (RL_LDS double *)L->red_d, &total);
        } else {
            replay(m, __builtin_inf(), &total);
        }
    }
    const float inv = (float)(1.0 / total);
    if (!(inv <= 3.40282347e38f)) return false;
    __syncthreads();  // every replay's reads of p are done
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i)
        if (i < per) L->p[tid * per + i] = tid * per + i < m ? __float_as_uint(p[i] * inv) : 0u;
    __syncthreads();
    if (wave == 0) {
        // The draw, while the other waves write the candidates.
        const uint32_t pick = draw_walk(pw, m, u);
        if (lane == 0) {
            a.out_token[row] = comp_id(L->v[pick]);
            a.out_kept[row] = m;
            a.out_used[row] = 1;
        }
    } else if (a.out_ids) {
        for (uint32_t j = tid - WAVE; j < m; j += SEL_THREADS - WAVE) {
            a.out_ids[(uint64_t)row * a.cand_stride + j] = comp_id(L->v[j]);
            a.out_probs[(uint64_t)row * a.cand_stride + j] = __uint_as_float(L->p[j]);
        }
    }
    return true;
}

// A short head (k_full_head, one workgroup): the chunks' elements and tails,
// the sort and the finish. Returns false when the row is not decided.
__device__ __forceinline__ bool finish_short(const RowIO &a, const SelScratch &f, uint32_t slot, uint32_t row,
                                             const rl_sampling &s, const FullRow &st, RL_LDS FinishLds *L) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t C = f.gather_chunks, n4 = a.vocab / 4;
    const bool okc = lane < C;
    const uint32_t nc = okc ? f.sel_n[slot * FULL_CHUNKS + lane] : 0u;
    const double tail = wave_total_f64(okc ? f.sel_tail[slot * FULL_CHUNKS + lane] : 0.0);
    const uint32_t incl = wave_incl_u32(nc);
    const uint32_t n = read_lane_u32(incl, WAVE - 1);
    if (tid < 32) L->exp_tab[tid] = EXP2_32_TAB[tid];
    if (wave == 0) L->pre[lane] = incl - nc;  // lanes from C on: n
    __syncthreads();
    if (!(tail >= 0.0) || n > SEL_FIN_CAP) return false;  // a NaN logit
    constexpr uint32_t E = SEL_FIN_CAP / SEL_THREADS;
    uint64_t x[E];
#pragma unroll
    for (uint32_t q = 0; q < E; ++q) {
        const uint32_t i = q * SEL_THREADS + tid;
        x[q] = 0;
        if (i < n) {
            uint32_t c = 0;  // the last chunk that starts at or before i
#pragma unroll
            for (uint32_t h = FULL_CHUNKS / 2; h > 0; h >>= 1)
                if (c + h < C && L->pre[c + h] <= i) c += h;
            const uint64_t at = (uint64_t)slot * a.vocab + 4 * chunk_lo(n4, c, C) + (i - L->pre[c]);
            x[q] = composite(f.keyA[at], f.idA[at]);
        }
    }
    if (n <= SORT_FEW)
        count_sort(x[0], n, (RL_LDS uint64_t *)L->v);
    else
        bucket_sort<E>(x, n, (RL_LDS uint64_t *)L->v, (RL_LDS SortLds *)&L->sort);
    return finish_selected(a, row, s, st.M, n, tail, L);
}

// ------------------------------------------------- the gather kernel ---
struct GatherLds {
    uint32_t bm[SEL_CHUNK_MAX / 32 + 1];  // window ids in this chunk, one bit per element
    uint32_t pos[SEL_BINS];               // a long head: elements in the bins before each
    uint32_t cnt[SEL_GROUPS];             // this step's elements per group
    uint32_t base[SEL_GROUPS];            // where they go
    uint32_t off[SEL_GROUPS];             // where each group starts
    uint64_t exp_tab[32];
    double red_d[SEL_WAVES];
    uint32_t red_u[SEL_WAVES];
    uint32_t last, count, groups, most, n;
};

// Picks the last bin to collect (whole workgroup): the bin in which the k-th
// element lies, or, for top-p, the one in which the mass (an estimate, so with
// a tenth of what is left out to spare) passes top_p of the whole. c, m: the
// counts and masses of the bins SEL_PER tid ..; M: the row's maximum. Sets
// st.thr, st.count and st.groups and, for a long head, L->pos and L->off; or
// leaves the row to k_full_rest whole (st.thr SEL_NONE): a bin too full to be
// sorted in LDS (many tied logits), a long head on the bf16 grid with few
// workgroups for it (SEL_GRID_SHARE), ties or every id in a small vocabulary
// (SEL_SMALL_VOCAB), or no mass to go by. Such a row has paid for its bins and
// two launches: 151936 ids, 40 % of them tied, at top-p 0.9 take 324 us at one
// row and 428 at 256, against 315 and 381 sorted at once; constant logits 190
// and 295 against 186 and 251.
constexpr uint32_t SEL_PER = 3;
static_assert(SEL_PER * SEL_THREADS >= SEL_BINS && SEL_BINS % SEL_PER == 0, "the bins over the threads");

__device__ __forceinline__ void pick_bins(const uint32_t (&c)[SEL_PER], const uint32_t (&m)[SEL_PER], uint32_t V,
                                          const rl_sampling &s, bool grid, bool pen, uint32_t head_wgs,
                                          FullRow &st, RL_LDS GatherLds *L) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const float c2 = (float)(1.4426950408889634 / (double)s.temperature);
    const uint32_t k = full_k(s, V);
    const bool by_k = k < V;
    // A bin's mass is its sum of parts of the p at its upper edge.
    double y[SEL_PER], ysum = 0.0;
    uint32_t csum = 0;
#pragma unroll
    for (uint32_t i = 0; i < SEL_PER; ++i) {
        const float z = fminf((sel_edge(tid * SEL_PER + i, st.R) - st.M) * c2, 0.0f);
        y[i] = by_k ? (double)c[i] : c[i] ? (double)((float)m[i] * __builtin_amdgcn_exp2f(z)) : 0.0;
        ysum += y[i];
        csum += c[i];
    }
    const uint32_t ci = wave_incl_u32(csum);
    const double yi = wave_incl_f64(ysum);
    if (lane == WAVE - 1) {
        L->red_u[wave] = ci;
        L->red_d[wave] = yi;
    }
    if (tid == 0) {
        L->last = 0;
        L->count = 0;
        L->groups = 0;
        L->most = 0;
    }
    if (tid < SEL_GROUPS) L->off[tid] = 0xFFFFFFFFu;
    __syncthreads();
    uint32_t c0 = ci - csum;
    double y0 = 0.0, yt = 0.0;
    for (uint32_t w = 0; w < SEL_WAVES; ++w) {
        if (w < wave) {
            c0 += L->red_u[w];
            y0 += L->red_d[w];
        }
        yt += L->red_d[w];
    }
    const double y1 = y0 + yi;
    y0 = y1 - ysum;
    const double tp = (double)s.top_p;
    // A top_p <= 0 is met by the first candidate.
    const double want = by_k ? (double)k : fmax(tp + 0.1 * (1.0 - tp), 0.1) * yt;
    if (y0 < want && y1 >= want) {
        double t = y0;
        uint32_t n = c0, bins = 0;  // this thread's bins up to the one that reaches it
#pragma unroll
        for (uint32_t i = 0; i < SEL_PER; ++i)
            if (i == 0 || t < want) {
                t += y[i];
                n += c[i];
                bins = i + 1;
            }
        // More than one thread only where the masses' rounding makes it so.
        atomicMax((uint32_t *)&L->last, tid * SEL_PER + bins);
        atomicMax((uint32_t *)&L->count, n);
    }
    __syncthreads();
    const uint32_t last = L->last, count = L->count;
    if (last == 0) return;
    const bool small = V < SEL_SMALL_VOCAB, big = count > SEL_FIN_CAP;
    if (big && grid && (pen ? SEL_GRID_SHARE_PEN : SEL_GRID_SHARE) * (count / head_wgs) > 2 * V) return;
    if (small && count == V) return;
    if (big || small) {
        uint32_t most = 0;
#pragma unroll
        for (uint32_t i = 0; i < SEL_PER; ++i) most = max(most, tid * SEL_PER + i < last ? c[i] : 0u);
        most = wave_fold_u32(most, [](uint32_t p, uint32_t q) { return p > q ? p : q; });
        if (lane == 0) atomicMax((uint32_t *)&L->most, most);
        __syncthreads();
        if (L->most > (small ? SEL_SMALL_TIES : SEL_GROUP)) return;
    }
    if (big) {
        uint32_t run = c0;
#pragma unroll
        for (uint32_t i = 0; i < SEL_PER; ++i) {
            const uint32_t b = tid * SEL_PER + i;
            if (b < SEL_BINS) L->pos[b] = run;
            if (b < last && c[i] != 0) {
                if ((run >> SEL_GROUP_LOG) < SEL_GROUPS) atomicMin((uint32_t *)&L->off[run >> SEL_GROUP_LOG], run);
                atomicMax((uint32_t *)&L->groups, (run >> SEL_GROUP_LOG) + 1);
            }
            run += c[i];
        }
        __syncthreads();
        if (L->groups > SEL_GROUPS) return;
    }
    st.thr = last - 1;
    st.count = count;
    st.groups = L->groups;
}

// grid (chunks, slots), SEL_THREADS: the selection rows. A short head (at most
// SEL_FIN_CAP elements): each chunk's elements go, in any order, to its own
// stretch of keyA/idA. A longer one: every element goes to its group's
// stretch, whose places the chunks draw from the row's counters a step at a
// time. Every chunk picks the bin for itself (a read of the row's bins from
// the cache and two scans, while its logits are in flight) rather than wait
// for the pass to have one workgroup do it after all the others.
template <bool VEC>
__global__ __launch_bounds__(SEL_THREADS) void k_full_gather(RowIO a, SelScratch f) {
    __shared__ GatherLds L_;
    RL_LDS GatherLds *L = (RL_LDS GatherLds *)&L_;
    const uint32_t slot = blockIdx.y, chunk = blockIdx.x;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t row = a.rows ? a.rows[slot] : a.row0 + slot;
    const uint32_t V = a.vocab, C = f.gather_chunks, C1 = f.pass_chunks;
    const float *rowp = a.logits + (uint64_t)row * a.stride;
    const uint32_t n4 = V / 4;
    const uint32_t q0 = chunk_lo(n4, chunk, C), q1 = chunk_lo(n4, chunk + 1, C);
    const uint32_t e0 = 4 * q0, e1 = chunk == C - 1 ? V : 4 * q1;
    const uint64_t base = (uint64_t)slot * V;
    // Loads in the order of their use: settings, window ids (clamped to the
    // call's stride), the pass's records and bins, then the first step.
    const uint32_t head_w = row_words(a, row);
    constexpr uint32_t WIN_PER = 2;
    static_assert(WIN_PER * SEL_THREADS >= 2048, "a window's ids fit the threads");
    uint32_t wid[WIN_PER];
    {
        const bool have_win = a.windows && a.wlen && a.wstride > 0;
        const uint32_t *win = have_win ? a.windows + (uint64_t)row * a.wstride
                                       : reinterpret_cast<const uint32_t *>(a.settings + row);
        const uint32_t wn = !have_win ? 1u : min(a.wstride, WIN_PER * SEL_THREADS);
#pragma unroll
        for (uint32_t k = 0; k < WIN_PER; ++k) {
            const uint32_t i = k * SEL_THREADS + tid;
            wid[k] = ((const RL_GLB uint32_t *)win)[i < wn ? i : wn - 1];
        }
    }
    const uint32_t lc = min(lane, C1 - 1);
    const float pm = ((const RL_GLB float *)f.part_max)[slot * C1 + lc];
    const float R = ((const RL_GLB float *)&f.row[slot].R)[0];
    const uint32_t binned = ((const RL_GLB uint32_t *)&f.row[slot].binned)[0];
    uint32_t c[SEL_PER], m[SEL_PER];
#pragma unroll
    for (uint32_t i = 0; i < SEL_PER; ++i) {
        const uint32_t b = min(tid * SEL_PER + i, SEL_BINS - 1);
        c[i] = ((const RL_GLB uint32_t *)f.sel_cnt)[(uint64_t)slot * SEL_BINS + b];
        m[i] = ((const RL_GLB uint32_t *)f.sel_mass)[(uint64_t)slot * SEL_BINS + b];
    }
    const uint64_t tab = EXP2_32_TAB[tid & 31u];
    f32x4 nx[SEL_U];
    // A chunk holds a float4 (sel_gather_chunks): q1 - 1 is one of its own.
    auto fetch = [&](uint32_t b) {
#pragma unroll
        for (uint32_t u = 0; u < SEL_U; ++u) {
            const uint32_t q = b + u * SEL_THREADS + tid;
            nx[u] = load4<VEC>(rowp, q < q1 ? q : q1 - 1);
        }
    };
    fetch(q0);
    const uint32_t e_odd = 4 * n4 + tid;  // the row's last vocab % 4, with the last chunk's last step
    const float x_odd = ((const RL_GLB float *)rowp)[min(e_odd, V - 1)];
    __builtin_amdgcn_sched_barrier(0);
    rl_sampling s;
    uint32_t wl;
    row_head(a, head_w, s, wl);
    if (!select_eligible(s, V)) return;
    const bool pen = penalises(s) && wl > 0;
    const bool by_k = full_k(s, V) < V;
    if (tid < 32) L->exp_tab[tid] = tab;
    if (tid == 0) L->n = 0;
    if (tid < SEL_GROUPS) L->cnt[tid] = 0;
    if (pen) {
        for (uint32_t i = tid; i < (e1 - e0 + 31) / 32; i += SEL_THREADS) L->bm[i] = 0;
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < WIN_PER; ++k) {
            const uint32_t id = wid[k];
            if (k * SEL_THREADS + tid < wl && id >= e0 && id < e1)
                atomicOr((uint32_t *)&L->bm[(id - e0) >> 5], 1u << ((id - e0) & 31));
        }
    }
    FullRow st{};
    st.M = uniform_f32(wave_maxnum_f32(pm));
    st.thr = SEL_NONE;
    st.R = uniform_f32(R);
    st.binned = uniform_u32(binned);  // and R: what the other chunks may yet read stays as it is
    const bool finite = st.M > -__builtin_inff() && st.M < __builtin_inff();
    st.done = finite ? 0u : 1u;
#pragma unroll
    for (uint32_t i = 0; i < SEL_PER; ++i)
        if (tid * SEL_PER + i >= SEL_BINS) c[i] = m[i] = 0;
    if (finite) pick_bins(c, m, V, s, st.binned == 2, pen, f.head_wgs, st, L);
    if (chunk == 0) {
        if (tid == 0) {
            f.row[slot] = st;
            // sample.rs:270-277: argmax, no draw; the first +inf, or 0 when
            // nothing is above -inf.
            if (!finite) {
                uint32_t first = 0xFFFFFFFFu;
                for (uint32_t i = 0; i < C1; ++i) first = min(first, (uint32_t)f.part_am[slot * C1 + i]);
                write_single(a, row, st.M == __builtin_inff() ? first : 0u);
            }
        }
        if (st.thr != SEL_NONE && st.count > SEL_FIN_CAP && tid <= st.groups)
            f.sel_off[(uint64_t)slot * (SEL_GROUPS + 1) + tid] = tid < st.groups ? L->off[tid] : st.count;
    }
    if (st.thr == SEL_NONE) return;
    const bool big = st.count > SEL_FIN_CAP;
    __syncthreads();  // the bitmap, the tables and the picked bins are in place
    const LdsExpTable etab{(RL_LDS uint64_t *)L->exp_tab};
    const TempScale tscale(s.temperature);
    double S = 0.0;
    bool nan = false;
    constexpr uint32_t NE = 4 * SEL_U + 1;  // a thread's elements of a step, and one of the row's last vocab % 4
    for (uint32_t b = q0; b < q1; b += SEL_STEP) {
        float x[NE];
#pragma unroll
        for (uint32_t u = 0; u < SEL_U; ++u)
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) x[4 * u + i] = nx[u][i];
        x[NE - 1] = x_odd;
        const bool odd = chunk == C - 1 && b + SEL_STEP >= q1 && e_odd < V;
        if (b + SEL_STEP < q1) fetch(b + SEL_STEP);
        auto id_of = [&](uint32_t i) {
            return i + 1 < NE ? 4 * (b + (i / 4) * SEL_THREADS + tid) + (i & 3u) : e_odd;
        };
        uint32_t to[NE];  // a long head: group << 16 | place among the step's elements of the group
        uint32_t took = 0;
#pragma unroll
        for (uint32_t i = 0; i < NE; ++i) {
            const bool in = i + 1 < NE ? b + (i / 4) * SEL_THREADS + tid < q1 : odd;
            if (!in) continue;
            const uint32_t e = id_of(i);
            float v = x[i];
            if (pen && ((L->bm[(e - e0) >> 5] >> ((e - e0) & 31)) & 1u)) v = penalize(v, s.repeat_penalty);
            x[i] = v;
            nan = nan || v != v;
            const uint32_t bin = sel_bin(v, st.R);
            if (bin <= st.thr) {
                if (big) {
                    const uint32_t g = L->pos[bin] >> SEL_GROUP_LOG;
                    to[i] = (g << 16) | atomicAdd((uint32_t *)&L->cnt[g], 1u);
                    took |= 1u << i;
                } else {
                    const uint32_t at = e0 + atomicAdd((uint32_t *)&L->n, 1u);
                    f.keyA[base + at] = total_key(v);
                    f.idA[base + at] = e;
                }
            } else if (!by_k) {
                S += (double)expf_libm_t(tscale(v - st.M), etab);
            }
        }
        if (big) {
            __syncthreads();
            if (tid < st.groups) {
                const uint32_t n = L->cnt[tid];
                L->base[tid] = n == 0 ? 0u
                                      : L->off[tid] + __hip_atomic_fetch_add(f.sel_fill + (uint64_t)slot * SEL_GROUPS + tid,
                                                                             n, __ATOMIC_RELAXED,
                                                                             __HIP_MEMORY_SCOPE_AGENT);
                L->cnt[tid] = 0;
            }
            __syncthreads();
#pragma unroll
            for (uint32_t i = 0; i < NE; ++i)
                if ((took >> i) & 1u) {
                    const uint32_t at = L->base[to[i] >> 16] + (to[i] & 0xFFFFu);
                    if (at < V) {
                        f.keyA[base + at] = total_key(x[i]);
                        f.idA[base + at] = id_of(i);
                    }
                }
        }
    }
    S = wave_total_f64(ballot(nan) != 0 ? __builtin_nan("") : S);
    if (lane == 0) L->red_d[wave] = S;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (uint32_t w = 0; w < SEL_WAVES; ++w) t += L->red_d[w];
        f.sel_tail[slot * FULL_CHUNKS + chunk] = t;
        f.sel_n[slot * FULL_CHUNKS + chunk] = L->n;
    }
}

}  // namespace rl
