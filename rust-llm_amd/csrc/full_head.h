// The FULL path's selection, second half: k_full_head sorts the heads that
// k_full_gather collected (full_select.h) and finishes their rows.
//
// A short head is one workgroup's work in LDS (finish_short): reading,
// sorting, cutting and drawing 930 elements takes about 10 us, the barriers and
// the draw's chain of additions most of it. A long head is sorted in groups of
// some 4096 elements, spread over the row's workgroups; the last of them to
// finish goes through the whole list. Heads of tens of thousands of elements
// are what flat rows (a high temperature, top_p 0.99) leave.
#pragma once
#include "full_select.h"

namespace rl {

struct HeadLds {
    union {
        uint64_t group[SEL_GROUP_CAP];  // a group's elements
        ChunkLds cr;                    // the list's replays
    } u;
    SortLds sort;
    uint64_t exp_tab[32];
    double red_d[SEL_WAVES];
    double seg_sum[SEL_GROUPS];  // each group's sum of p
    uint32_t goff[SEL_GROUPS + 1];
    // The list's statistics (PStats).
    int st_emin;
    uint32_t st_bad, st_count, st_last_in, st_first_out;
    uint32_t sh_last, sh_hit;
    double sh_hit_sum;
};

// Sorts the collected groups blockIdx.x, blockIdx.x + gridDim.x, ... of a long
// head: each group's elements into the reference's order, ids to fid and p to
// fp at the group's place in the list (the first k candidates), with
// device-scope stores for the workgroup that finishes the row, and its share of
// the list's statistics to f.sel_rec.
__device__ __forceinline__ void sort_groups(const SelScratch &f, uint32_t slot, RL_LDS HeadLds *L, const FullRow &st,
                                            uint32_t V, uint32_t k, float min_p, const TempScale &tscale,
                                            const LdsExpTable &etab, uint32_t *fid, float *fp) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    constexpr uint32_t E = SEL_GROUP_CAP / SEL_THREADS;
    for (uint32_t g = blockIdx.x; g < st.groups; g += gridDim.x) {
        const uint32_t lo = L->goff[g], n = L->goff[g + 1] - lo;
        const uint64_t src = (uint64_t)slot * V + lo;
        uint64_t x[E];
#pragma unroll
        for (uint32_t q = 0; q < E; ++q) {
            const uint32_t i = q * SEL_THREADS + tid;
            x[q] = i < n ? composite(f.keyA[src + i], f.idA[src + i]) : 0ull;
        }
        bucket_sort<E>(x, n, (RL_LDS uint64_t *)L->u.group, (RL_LDS SortLds *)&L->sort);
        if (tid == 0) stats_reset(L);
        PStats ps;
        double sum = 0.0;
        for (uint32_t i = tid; i < n && lo + i < k; i += SEL_THREADS) {
            const uint64_t c = L->u.group[i];
            const float p = expf_libm_t(tscale(key_value(comp_key(c)) - st.M), etab);
            __hip_atomic_store(fid + lo + i, comp_id(c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store((uint32_t *)fp + lo + i, __float_as_uint(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sum += (double)p;
            ps.add(p, lo + i, min_p);
        }
        sum = wave_total_f64(sum);
        if (lane == 0) L->red_d[wave] = sum;
        __syncthreads();
        ps.merge(L);
        __syncthreads();
        if (tid < 4) {
            double t = 0.0;
            for (uint32_t w = 0; w < SEL_WAVES; ++w) t += L->red_d[w];
            const uint64_t r = tid == 0   ? (uint64_t)__double_as_longlong(t)
                               : tid == 1 ? ((uint64_t)L->st_bad << 32) | (uint32_t)L->st_emin
                               : tid == 2 ? ((uint64_t)L->st_count << 32) | L->st_last_in
                                          : (uint64_t)L->st_first_out;
            __hip_atomic_store(f.sel_rec + ((uint64_t)slot * SEL_GROUPS + g) * 4 + tid, r, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
    }
}

// The finish of a long head by the row's last workgroup: fid, fp hold its
// first k candidates in order, CS groups' records their statistics, tail the
// sum of every other p (0 for top-k). Returns false (no output final) when the
// row is not decided here.
__device__ __forceinline__ bool finish_long(const RowIO &a, const SelScratch &f, uint32_t slot, uint32_t row,
                                            const rl_sampling &s, const FullRow &st, uint32_t k, double tail,
                                            RL_LDS HeadLds *L, uint32_t *fid, float *fp) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t V = a.vocab;
    const bool by_k = full_k(s, V) < V;
    const bool out = a.out_ids != nullptr;
    // The groups that hold candidates, and their records, a group a lane.
    uint32_t CS = 0;
    while (CS < st.groups && L->goff[CS] < k) ++CS;
    auto group_start = [&](uint32_t c) { return min(L->goff[c], k); };
    if (tid == 0) stats_reset(L);
    __syncthreads();
    PStats ps;
    if (wave == 0 && lane < CS) {
        const uint64_t *rec = f.sel_rec + ((uint64_t)slot * SEL_GROUPS + lane) * 4;
        const uint64_t r1 = rec[1], r2 = rec[2];
        L->seg_sum[lane] = __longlong_as_double((long long)rec[0]);
        ps.emin = (int)(uint32_t)r1;
        ps.bad = (uint32_t)(r1 >> 32);
        ps.last_in = (uint32_t)r2;
        ps.count = (uint32_t)(r2 >> 32);
        ps.first_out = (uint32_t)rec[3];
    }
    if (wave == 0) ps.merge(L);
    __syncthreads();
    if (L->st_bad) return false;
    const int emin = L->st_emin;
    const uint32_t count = L->st_count, last_in = L->st_last_in, first_out = L->st_first_out;
    const bool min_on = s.min_p > 0.0f;
    if (min_on && last_in > first_out) return false;  // the survivors of min-p are not a prefix
    double list = 0.0;
    for (uint32_t c = 0; c < CS; ++c) list += L->seg_sum[c];
    // As in finish_selected: every partial sum exact, or replayed in order.
    const bool exact = emin > 1000 || list < mul_pow2(1.0 - 0x1p-30, 30 + emin);
    const uint32_t *fpw = (const uint32_t *)fp;
    const auto as_f32 = [](uint32_t b) { return __uint_as_float(b); };
    RL_LDS ChunkLds *cr = (RL_LDS ChunkLds *)&L->u.cr;
    uint32_t m = k;
    bool have_total = false;
    double total = 0.0;
    if (s.top_p < 1.0f) {
        double t_lo, t_hi;
        if (by_k) {
            if (!exact) chunk_replay<53, SEL_THREADS>(fpw, as_f32, k, [](double) { return false; }, cr, &list);
            t_lo = t_hi = (double)s.top_p * list;
        } else {
            sel_target_interval(tail + list, V, s.top_p, &t_lo, &t_hi);
        }
        uint32_t j = k;
        if (exact) {
            double b = 0.0;
            uint32_t c = 0;
            while (c < CS && !(b + L->seg_sum[c] >= t_lo)) b += L->seg_sum[c++];
            if (c < CS)
                j = exact_first_reaching<SEL_THREADS>(fp, group_start(c), group_start(c + 1), b, t_lo, L->red_d,
                                                      &L->sh_hit, &L->sh_hit_sum, &total, HotRange());
        } else {
            j = chunk_replay<53, SEL_THREADS>(fpw, as_f32, k, [t_lo](double c) { return c >= t_lo; }, cr, &total);
        }
        if (j >= k) {
            if (!by_k) return false;  // the head does not reach the target
            total = list;             // a mass the running sum never reaches: no cut
        } else {
            if (!(total >= t_hi)) return false;  // the cut could fall on either side
            m = j + 1;
        }
        have_total = true;
    }
    if (min_on) {
        uint32_t w = min(m, count);
        w = w > 1 ? w : 1u;
        if (w != m) have_total = false;
        m = w;
    }
    if (!have_total) {
        if (exact) {
            // The groups before the m-th candidate, and the part of its own.
            total = 0.0;
            uint32_t c = 0;
            while (c < CS && group_start(c + 1) <= m) total += L->seg_sum[c++];
            if (c < CS && group_start(c) < m) {
                const double b = total;
                exact_first_reaching<SEL_THREADS>(fp, group_start(c), m, b, __builtin_inf(), L->red_d, &L->sh_hit,
                                                  &L->sh_hit_sum, &total, HotRange());
            }
        } else {
            chunk_replay<53, SEL_THREADS>(fpw, as_f32, m, [](double) { return false; }, cr, &total);
        }
    }
    const float inv = (float)(1.0 / total);
    if (!(inv <= 3.40282347e38f)) return false;
    // The draw (sample.rs:349-358), storing q over p for the rounds it stages
    // when the caller wants the candidates; then q over the rest of the kept
    // prefix (sample.rs:344-347).
    const float u = a.uniforms[row];
    double unused;
    uint32_t qdone = 0;
    const uint32_t j = chunk_replay<24, SEL_THREADS>(
        fpw, [inv](uint32_t b) { return __uint_as_float(b) * inv; }, m, [u](double c) { return c > (double)u; }, cr,
        &unused, out ? (uint32_t *)fp : nullptr, &qdone);
    __syncthreads();  // every read of p by the draw precedes the writes of q
    if (tid == 0) {
        a.out_token[row] = fid[j < m ? j : m - 1];
        a.out_kept[row] = m;
        a.out_used[row] = 1;
    }
    if (out)
        for (uint32_t i = qdone + tid; i < m; i += SEL_THREADS) fp[i] = fp[i] * inv;
    return true;
}

// grid (groups, slots), SEL_THREADS: the rows whose heads were collected. A
// short head is the first workgroup's; a long one is sorted by all of the
// row's, the last of which finishes it. Also clears the bins of every row that
// was counted into them, for the next call.
__global__ __launch_bounds__(SEL_THREADS) void k_full_head(RowIO a, SelScratch f) {
    __shared__ union {
        HeadLds h;
        FinishLds fin;
    } L_;
    RL_LDS HeadLds *L = (RL_LDS HeadLds *)&L_.h;
    const uint32_t slot = blockIdx.y;
    const FullRow st = f.row[slot];
    const uint32_t tid = threadIdx.x, lane = lane_id();
    if (st.binned && blockIdx.x == 0) {
        for (uint32_t i = tid; i < SEL_BINS; i += SEL_THREADS) {
            f.sel_cnt[(uint64_t)slot * SEL_BINS + i] = 0;
            f.sel_mass[(uint64_t)slot * SEL_BINS + i] = 0;
        }
        if (tid < SEL_GROUPS) f.sel_fill[(uint64_t)slot * SEL_GROUPS + tid] = 0;
    }
    if (st.done || st.thr == SEL_NONE) return;
    const bool big = st.count > SEL_FIN_CAP;
    if (!big && blockIdx.x != 0) return;
    const uint32_t row = a.rows ? a.rows[slot] : a.row0 + slot;
    const rl_sampling s = a.settings[row];
    if (!big) {
        const bool fin = finish_short(a, f, slot, row, s, st, (RL_LDS FinishLds *)&L_.fin);
        if (tid == 0 && fin) f.row[slot].done = 1;
        return;
    }
    const uint32_t V = a.vocab;
    uint32_t *fid = a.out_ids ? a.out_ids + (uint64_t)row * a.cand_stride : f.idB + (uint64_t)slot * V;
    float *fp = a.out_ids ? a.out_probs + (uint64_t)row * a.cand_stride : f.probs + (uint64_t)slot * V;
    const uint32_t k = min(full_k(s, V), st.count);
    if (tid <= st.groups) L->goff[tid] = f.sel_off[(uint64_t)slot * (SEL_GROUPS + 1) + tid];
    copy_exp_table((RL_LDS uint64_t *)L->exp_tab);  // ends with a barrier
    sort_groups(f, slot, L, st, V, k, s.min_p, TempScale(s.temperature), LdsExpTable{(RL_LDS uint64_t *)L->exp_tab}, fid,
                fp);
    __builtin_amdgcn_s_waitcnt(WAITCNT_VM0);  // this wave's stores have completed
    __syncthreads();                          // and every other wave's
    if (tid == 0) L->sh_last = atomicAdd(&f.arrive[slot], 1u) == gridDim.x - 1 ? 1u : 0u;
    __syncthreads();
    if (!L->sh_last) return;
    if (tid == 0) f.arrive[slot] = 0;
    // What the other workgroups stored is read from here on.
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const double tail = wave_total_f64(lane < f.gather_chunks ? f.sel_tail[slot * FULL_CHUNKS + lane] : 0.0);
    if (!(tail >= 0.0)) return;  // a NaN logit
    const bool fin = finish_long(a, f, slot, row, s, st, k, tail, L, fid, fp);
    if (tid == 0 && fin) f.row[slot].done = 1;
}

}  // namespace rl
