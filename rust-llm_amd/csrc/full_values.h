// The FULL path's value path: nearly flat rows on the bf16 grid, whose values
// k_full_pass counted (value_bins.h). k_full_rest calls finish_values for them.
//
// The reference orders such a row's candidates by value, then id
// (sample.rs:279-305). Equal values have equal p, so the row is a short list of
// runs (one a value that occurs, and one an element without a bin), and every
// sum the reference forms over the candidates is a sum over runs of equal
// terms: the mass, the cut and the total by a block scan while the sums are
// exact, else, like the draw, by run_walk, which replays the reference's
// additions a run at a time (rl_seqsum.h). The ids matter only at the end: the
// drawn candidate is the n-th occurrence of its value, found by the chunks'
// counts and one read of its chunk.
//
// What bounds it: one workgroup's chain of dependent steps, with little for its
// other CUs to take over. Sorting these rows (256 x 151936, 40 % of a row tied)
// took 364 us in k_full_rest after a pass of 32; counting takes 54 after a pass
// of 41 (its LDS atomics), and the call 385 -> 93 us.
#pragma once
#include "full_head.h"

namespace rl {

constexpr uint32_t VAL_EXC = 1024;                  // elements without a bin of a row
constexpr uint32_t VAL_RUNS = VAL_BINS + VAL_EXC;
constexpr uint32_t VAL_PER = VAL_RUNS / SEL_THREADS;  // runs a thread
static_assert(VAL_PER * SEL_THREADS == VAL_RUNS && VAL_BINS == 4 * SEL_THREADS, "the runs over the threads");
constexpr uint32_t VAL_BLOCK = 16 * WAVE;           // elements of a wave's step through a chunk
constexpr uint32_t VAL_BLOCKS = 65536 / VAL_BLOCK;

struct ValLds {
    uint64_t exc[VAL_EXC];         // the elements without a bin, sorted
    uint32_t term[VAL_RUNS];       // per run: the f32 term's bits (p, then q); first, per place: the bins taken before it
    uint32_t n[VAL_RUNS];          // its occurrences
    uint32_t key[VAL_RUNS];        // its value's total-order key
    uint32_t bm[65536 / 32 + 1];   // window ids in the drawn candidate's chunk
    uint32_t blk[VAL_BLOCKS];      // occurrences per block of that chunk
    uint32_t pre[FULL_CHUNKS];     // elements without a bin in the chunks before
    uint64_t exp_tab[32];
    double red_d[SEL_WAVES];
    uint32_t red_u[SEL_WAVES];
    int st_emin;
    uint32_t st_bad, st_count, st_last_in, st_first_out;
    uint32_t sh_hit, sh_m, sh_run, sh_off, sh_chunk, sh_nth;
    double sh_at;
};

// One wave adds the R runs of equal terms (n[r] terms with the bits term[r]) to
// a running sum from 0 in order, every lane alike, in f64 (run_walk) or, for
// the draw, in f32 (run_draw: term[0] >= 2^-60, sums below 2^60, a run a lane).
// Lane l counts the steps of runs pos + l WK .. on the grid of the sum's segment, ties
// resolved as in wave_walk; the first lane whose runs leave the segment or meet
// pred goes through them one by one, and the run that does so is crossed in
// closed form. Returns the first term whose partial sum meets pred (its place
// among all terms), with that sum in s, or 0xFFFFFFFF with the total in s.
template <uint32_t WK, class Pred>
__device__ __forceinline__ uint32_t run_walk(RL_LDS const uint32_t *term, RL_LDS const uint32_t *n, uint32_t R,
                                             Pred pred, double &s) {
    constexpr int P = 53;
    const uint32_t lane = lane_id();
    uint32_t before = 0;  // terms added so far
    for (uint32_t pos = 0; pos < R;) {
        uint32_t x[WK], c[WK], mine_n = 0;
#pragma unroll
        for (uint32_t i = 0; i < WK; ++i) {
            const uint32_t r = pos + lane * WK + i;
            x[i] = r < R ? term[r] : 0u;
            c[i] = r < R ? n[r] : 0u;
            mine_n += c[i];
        }
        uint32_t l = 0;       // the lane to go through
        const uint32_t upto_n = wave_incl_u32(mine_n);
        if (s > 0.0) {
            const SumSegF g = segf_of<P>(s);
            const double scale = mul_pow2(1.0, -g.uexp);
            StepRun r = run_identity();
#pragma unroll
            for (uint32_t i = 0; i < WK; ++i)
                if (c[i] != 0) run_add_equal(r, x[i], c[i], scale);
            r.base = r.base < STEP_CAP ? r.base : STEP_CAP;
            const uint64_t T = ballot(r.tie != 0), O = ballot(run_par(r) != 0);
            uint32_t dep;
            const uint32_t k = parity_in(T, O, lane, &dep);
            const uint32_t pl = dep ? (parity_of(g.n) ^ k) : k;
            const double mine = r.base + (r.tie ? (double)((pl ^ r.c) & 1u) : 0.0);
            const double ahead = wave_excl_f64(mine);  // exact below the room, where it is used
            const double upto = ahead + mine;
            const bool ev = !(upto < g.lim - g.n) || pred(mul_pow2(g.n + upto, g.uexp));
            const uint64_t evm = ballot(ev);
            if (evm == 0) {
                s = mul_pow2(g.n + read_lane_f64(upto, WAVE - 1), g.uexp);
                before += read_lane_u32(upto_n, WAVE - 1);
                pos += WAVE * WK;
                continue;
            }
            l = (uint32_t)__builtin_ctzll(evm);
            s = mul_pow2(g.n + read_lane_f64(ahead, l), g.uexp);
        }
        before += read_lane_u32(upto_n - mine_n, l);
        pos += l * WK;
#pragma unroll
        for (uint32_t i = 0; i < WK; ++i) {
            if (pos >= R) continue;
            const uint32_t cnt = read_lane_u32(c[i], l);
            const uint32_t j = equal_run_walk<P>(s, read_lane_u32(x[i], l), cnt, pred);
            if (j < cnt) return before + j;
            before += cnt;
            ++pos;
        }
    }
    return 0xFFFFFFFFu;
}

// Returns the run whose terms' partial sum first exceeds u, *off the term in it;
// or R. Written for few instructions, since the code runs once a launch and is
// fetched cold: with the first runs and four runs a lane written out, the draw
// took 21 us in f64 and no less in these 32-bit operations; with one run a lane
// and loops left rolled, here and above, the 256-row call went from 100 to 93 us.
__device__ __forceinline__ uint32_t run_draw(RL_LDS const uint32_t *term, RL_LDS const uint32_t *n, uint32_t R, float u,
                                             uint32_t *off) {
    const uint32_t lane = lane_id();
    const auto pred = [u](float x) { return x > u; };
    float s = 0.0f;
    for (uint32_t pos = 0; pos < R;) {
        const uint32_t rr = min(pos + lane, R - 1);
        const uint32_t x = term[rr], c = pos + lane < R ? n[rr] : 0u;
        uint32_t l = 0;  // the lane whose run holds an event
        if (s > 0.0f) {
            const Seg32 g = seg32_of(s);
            Run32 r{0, 0, 0, 0};
            if (c != 0) run32_add_equal(r, __uint_as_float(x), c, g.scale);
            const uint64_t T = ballot(r.tie != 0);
            uint32_t mine = min(r.base, STEP32_CAP);
            if (T != 0) {
                const uint64_t O = ballot(run32_par(r) != 0);
                uint32_t dep;
                const uint32_t k = parity_in(T, O, lane, &dep);
                mine += r.tie ? ((dep ? g.n ^ k : k) ^ r.c) & 1u : 0u;
            }
            const uint32_t upto = wave_incl_u32(mine);  // at most 64 (STEP32_CAP + 1): no wrap-around
            const uint64_t ev = ballot(upto >= (1u << 24) - g.n || pred((float)(g.n + upto) * g.step));
            l = ev ? (uint32_t)__builtin_ctzll(ev) : WAVE;
            const uint32_t at = read_lane_u32(upto, min(l, WAVE - 1)) - (ev ? read_lane_u32(mine, l) : 0u);
            s = (float)(g.n + at) * g.step;
        }
        pos += l;
        if (l == WAVE || pos >= R) continue;
        const uint32_t cnt = read_lane_u32(c, l);
        const uint32_t j = equal_run_walk32(s, __uint_as_float(read_lane_u32(x, l)), cnt, pred);
        if (j < cnt) {
            *off = j;
            return pos;
        }
        ++pos;
    }
    return R;
}

// Finishes a row from its values' counts (st.values: their window). One
// workgroup. Returns whether the row is final; if not, *M is its maximum and it
// is sorted whole: a NaN, an element list that did not fit, or p or q that the
// walks here do not take.
__device__ __forceinline__ bool finish_values(const RowIO &a, const FullScratch &f, uint32_t slot, uint32_t row,
                                              const rl_sampling &s, uint32_t lo, uint32_t wl, RL_LDS ValLds *L,
                                              float *M_out) {
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t V = a.vocab, C = a.chunks;
    const bool okc = lane < C;
    // The chunks' counts (two a word) of the four bins at the places 4 tid ..
    // 4 tid + 3 of the order, and each chunk's record, a chunk a lane.
    const uint32_t b0 = tid < VAL_SPAN / 4 ? VAL_SPAN - 4 - 4 * tid : 4 * tid;
    uint32_t c[4] = {0, 0, 0, 0};
#pragma unroll 8
    for (uint32_t ch = 0; ch < C; ++ch) {
        const RL_GLB uint32_t *t = (const RL_GLB uint32_t *)chunk_counts(f, V, slot, ch) + b0 / 2;
        const uint32_t w0 = t[0], w1 = t[1];
        c[0] += w0 & 0xFFFFu;
        c[1] += w0 >> 16;
        c[2] += w1 & 0xFFFFu;
        c[3] += w1 >> 16;
    }
    if (tid < VAL_SPAN / 4) {  // positive bins: the largest first
        const uint32_t x0 = c[0], x1 = c[1];
        c[0] = c[3];
        c[1] = c[2];
        c[2] = x1;
        c[3] = x0;
    }
    const float Mr = okc ? f.part_max[slot * C + lane] : -__builtin_inff();
    const uint64_t rec = okc ? f.part_am[slot * C + lane] : 0xFFFFFFFFull;
    const uint32_t nc = (uint32_t)(rec >> 32);
    const float M = uniform_f32(wave_maxnum_f32(Mr));
    *M_out = M;
    if (!(M > -__builtin_inff() && M < __builtin_inff())) {
        // sample.rs:270-277: argmax, no draw; the first +inf, or 0 when
        // nothing is above -inf.
        const uint32_t fi = wave_fold_u32((uint32_t)rec, [](uint32_t x, uint32_t y) { return x < y ? x : y; });
        if (tid == 0) write_single(a, row, M == __builtin_inff() ? fi : 0u);
        return true;
    }
    if (ballot(nc == LIST_OVER) != 0) return false;
    const uint32_t incl = wave_incl_u32(nc), E = read_lane_u32(incl, WAVE - 1);
    if (E > VAL_EXC) return false;

    // ---- the elements without a bin, sorted ----
    if (wave == 0) L->pre[lane] = incl - nc;
    if (tid < 32) L->exp_tab[tid] = EXP2_32_TAB[tid];
    if (tid == 0) {
        stats_reset(L);
        L->sh_hit = 0xFFFFFFFFu;
        L->sh_m = V;
    }
    __syncthreads();
    bool nan = false;
    for (uint32_t ch = wave; ch < C; ch += SEL_WAVES) {
        const uint64_t *src = f.surv + (uint64_t)slot * SURV_CAP + ch * (SURV_CAP / C);
        const uint32_t nch = read_lane_u32(nc, ch), at = L->pre[ch];
        for (uint32_t i = lane; i < nch; i += WAVE) {
            const uint64_t x = src[i];
            const float v = key_value(comp_key(x));
            nan = nan || v != v;
            L->exc[at + i] = x;
        }
    }
    if (nan) L->st_bad = 1;
    __syncthreads();
    if (L->st_bad) return false;
    // Each takes the place that the number of elements above it gives.
    const uint64_t own = tid < E ? L->exc[tid] : 0ull;
    uint32_t place = 0;
#pragma unroll 4
    for (uint32_t i = 0; i < E; ++i) place += L->exc[i] > own ? 1u : 0u;
    __syncthreads();
    if (tid < E) L->exc[place] = own;

    // ---- the runs in the reference's order ----
    const auto place_key = [lo](uint32_t o) { return total_key(__uint_as_float(val_bits(val_order(o), lo))); };
    uint32_t taken = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) taken += c[i] != 0 ? 1u : 0u;
    uint32_t nbins;
    uint32_t at = block_exclusive<SEL_THREADS, uint32_t>(taken, (RL_LDS uint32_t *)L->red_u, &nbins);
    const uint32_t R = nbins + E;
    // Elements without a bin above each bin's value (none equals it): four
    // searches side by side.
    uint32_t key[4], above[4] = {0, 0, 0, 0};
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) key[i] = place_key(4 * tid + i);
    uint32_t h0 = E ? 1u << (31 - __builtin_clz(E)) : 0u;
    for (uint32_t h = h0; h > 0; h >>= 1) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t e = above[i] + h;
            const uint32_t k = comp_key(L->exc[min(e, E) - 1]);
            above[i] = e <= E && k > key[i] ? e : above[i];
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        L->term[4 * tid + i] = at;
        if (c[i] != 0) {
            L->n[at + above[i]] = c[i];
            L->key[at + above[i]] = key[i];
            ++at;
        }
    }
    __syncthreads();
    uint32_t mine_exc = 0xFFFFFFFFu;  // the run of the element exc[tid]
    if (tid < E) {
        const uint32_t key = comp_key(L->exc[tid]);
        uint32_t b = 0;  // places whose values are above it
        for (uint32_t h = VAL_BINS / 2; h > 0; h >>= 1)
            if (place_key(b + h - 1) > key) b += h;
        // b <= VAL_BINS - 1: at the last place, -inf, nothing but a NaN below it is missed.
        mine_exc = L->term[b] + tid;
        L->n[mine_exc] = 1;
        L->key[mine_exc] = key;
    }
    __syncthreads();

    // ---- p, and what the sums' exactness and min-p depend on ----
    // Thread t's runs are r0 .. r1 - 1, in loops that are not unrolled (run_draw).
    const LdsExpTable etab{(RL_LDS uint64_t *)L->exp_tab};
    const TempScale tscale(s.temperature);
    const uint32_t per = (R + SEL_THREADS - 1) / SEL_THREADS;
    const uint32_t r0 = min(tid * per, R), r1 = min(r0 + per, R);
    double mass_t = 0.0;
    uint32_t n_t = 0;
    PStats ps;
#pragma unroll 1
    for (uint32_t r = r0; r < r1; ++r) {
        const float p = expf_libm_t(tscale(key_value(L->key[r]) - M), etab);
        const uint32_t n = L->n[r];
        L->term[r] = __float_as_uint(p);
        ps.add(p, r, s.min_p);
        if (p >= s.min_p) ps.count += n - 1;
        mass_t += (double)p * (double)n;
        n_t += n;
    }
    ps.merge(L);
    double mass;
    const double mass_before = block_exclusive<SEL_THREADS, double>(mass_t, (RL_LDS double *)L->red_d, &mass);
    uint32_t all;
    const uint32_t n_before = block_exclusive<SEL_THREADS, uint32_t>(n_t, (RL_LDS uint32_t *)L->red_u, &all);
    const int emin = L->st_emin;
    // The survivors of min-p are a prefix (p falls along the order; checked).
    if (L->st_bad || L->st_last_in > L->st_first_out || all != V) return false;
    // As in k_full_rest: every partial sum exact in any order, or replayed.
    const bool exact = emin > 1000 || mass < mul_pow2(1.0 - 0x1p-30, 30 + emin);
    RL_LDS const uint32_t *term = (RL_LDS const uint32_t *)L->term;
    RL_LDS const uint32_t *occ = (RL_LDS const uint32_t *)L->n;
    constexpr uint32_t WK = 2;
    const auto never = [](double) { return false; };

    // ---- the top-p cut (sample.rs:307-324) ----
    uint32_t m = V;
    double total = mass;
    if (exact) {
        const double target = (double)s.top_p * mass;
        double b = mass_before;
        uint32_t nb = n_before, hit = 0xFFFFFFFFu;
        // Only the thread in whose runs the sum reaches it goes through them.
        if (b + mass_t >= target && (b < target || tid == 0))
#pragma unroll 1
            for (uint32_t r = r0; r < r1; ++r) {
                const double x = (double)__uint_as_float(L->term[r]);
                const uint32_t n = L->n[r];
                if (b + x * (double)n >= target) {
                    hit = r;
                    // The first of the run's terms to reach it.
                    uint32_t k = 1;
                    if (x > 0.0) {
                        const double d = (target - b) / x;
                        k = d >= (double)n ? n : d > 1.0 ? (uint32_t)d : 1u;
                    }
                    while (k > 1 && b + x * (double)(k - 1) >= target) --k;
                    while (k < n && b + x * (double)k < target) ++k;
                    nb += k;
                    b += x * (double)k;
                    break;
                }
                b += x * (double)n;
                nb += n;
            }
        if (hit != 0xFFFFFFFFu) atomicMin((uint32_t *)&L->sh_hit, hit);
        __syncthreads();
        if (hit != 0xFFFFFFFFu && L->sh_hit == hit) {
            L->sh_m = nb;
            L->sh_at = b;
        }
        __syncthreads();
        m = L->sh_m;  // V where no sum reaches it
        if (L->sh_hit != 0xFFFFFFFFu) total = L->sh_at;
    } else {
        if (wave == 0) {
            double sum = 0.0, at_cut = 0.0;
            run_walk<WK>(term, occ, R, never, sum);
            const double target = (double)s.top_p * sum;
            // A target <= 0 is met by the first term.
            uint32_t j = 0;
            if (0.0 >= target) at_cut = (double)__uint_as_float(term[0]);
            else j = run_walk<WK>(term, occ, R, [target](double x) { return x >= target; }, at_cut);
            if (lane == 0) {
                L->sh_m = j == 0xFFFFFFFFu ? V : j + 1;
                L->sh_at = at_cut;
            }
        }
        __syncthreads();
        m = L->sh_m;
        total = L->sh_at;
    }

    // ---- min-p (sample.rs:326-340) ----
    const uint32_t w = min(m, L->st_count);
    const bool recount = w != m;
    m = w > 1 ? w : 1u;
    // The runs past the m-th candidate end there, for the walks below.
    uint32_t nb = n_before;
    double part = 0.0;
#pragma unroll 1
    for (uint32_t r = r0; r < r1; ++r) {
        const uint32_t n = L->n[r], k = nb < m ? min(n, m - nb) : 0u;
        if (k != n) L->n[r] = k;
        part += (double)__uint_as_float(L->term[r]) * (double)k;
        if (k != 0 && nb + n >= m) L->sh_run = r + 1;  // the runs kept
        nb += n;
    }
    if (recount && exact) block_exclusive<SEL_THREADS, double>(part, (RL_LDS double *)L->red_d, &total);
    __syncthreads();
    const uint32_t Rm = L->sh_run;
    if (recount && !exact) {
        if (wave == 0) {
            double sum = 0.0;
            run_walk<WK>(term, occ, Rm, never, sum);
            if (lane == 0) L->sh_at = sum;
        }
        __syncthreads();
        total = L->sh_at;
    }
    const float inv = (float)(1.0 / total);
    if (!(inv <= 3.40282347e38f)) return false;
    for (uint32_t r = tid; r < Rm; r += SEL_THREADS) L->term[r] = __float_as_uint(__uint_as_float(L->term[r]) * inv);
    __syncthreads();

    // ---- the draw (sample.rs:349-358) ----
    if (wave == 0) {
        const float u = a.uniforms[row];
        uint32_t off = 0;
        uint32_t r = 0.0f > u ? 0u : run_draw(term, occ, Rm, u, &off);
        if (r == Rm) {  // a shortfall takes the last candidate
            r = Rm - 1;
            off = occ[r] - 1;
        }
        if (lane == 0) {
            L->sh_run = r;
            L->sh_off = off;
        }
    }
    __syncthreads();
    const uint32_t run = L->sh_run, off = L->sh_off;
    if (tid == 0) {
        a.out_kept[row] = m;
        a.out_used[row] = 1;
    }
    const uint32_t word = __float_as_uint(key_value(L->key[run]));
    const uint32_t bin = val_bin(word, lo);
    if (bin == VAL_NONE) {
        if (mine_exc == run) a.out_token[row] = comp_id(L->exc[tid]);
        return true;
    }

    // ---- the off-th occurrence of the value in id order ----
    if (wave == 0) {
        const uint32_t h = okc ? (chunk_counts(f, V, slot, lane)[bin / 2] >> (16 * (bin & 1u))) & 0xFFFFu : 0u;
        const uint32_t hi = wave_incl_u32(h);
        const uint32_t ch = (uint32_t)__builtin_ctzll(ballot(hi > off));  // the counts sum to more than off
        if (lane == ch) {
            L->sh_chunk = ch;
            L->sh_nth = off - (hi - h);
        }
    }
    __syncthreads();
    const uint32_t chunk = L->sh_chunk, nth = L->sh_nth, n4 = V / 4;
    const uint32_t e0 = 4 * chunk_lo(n4, chunk, C), e1 = chunk == C - 1 ? V : 4 * chunk_lo(n4, chunk + 1, C);
    const float *rowp = a.logits + (uint64_t)row * a.stride;
    const bool pen = penalises(s) && wl > 0;
    if (pen) {
        const uint32_t *win = a.windows + (uint64_t)row * a.wstride;
        for (uint32_t i = tid; i < (e1 - e0 + 31) / 32; i += SEL_THREADS) L->bm[i] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < wl; i += SEL_THREADS) {
            const uint32_t id = win[i];
            if (id >= e0 && id < e1) atomicOr((uint32_t *)&L->bm[(id - e0) >> 5], 1u << ((id - e0) & 31));
        }
        __syncthreads();
    }
    constexpr uint32_t U = VAL_BLOCK / WAVE;
    auto fetch = [&](uint32_t blk, float (&x)[U]) {
#pragma unroll
        for (uint32_t i = 0; i < U; ++i)
            x[i] = ((const RL_GLB float *)rowp)[min(e0 + blk * VAL_BLOCK + i * WAVE + lane, e1 - 1)];
    };
    auto matches = [&](uint32_t blk, const float (&x)[U], uint32_t i) {
        const uint32_t o = blk * VAL_BLOCK + i * WAVE + lane;  // id e0 + o
        if (o >= e1 - e0) return false;
        const float v = pen && ((L->bm[o >> 5] >> (o & 31)) & 1u) ? penalize(x[i], s.repeat_penalty) : x[i];
        return __float_as_uint(v) == word;
    };
    const uint32_t blocks = (e1 - e0 + VAL_BLOCK - 1) / VAL_BLOCK;
    for (uint32_t blk = wave; blk < blocks; blk += SEL_WAVES) {
        float x[U];
        fetch(blk, x);
        uint32_t k = 0;
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) k += (uint32_t)__popcll(ballot(matches(blk, x, i)));
        if (lane == 0) L->blk[blk] = k;
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t h = lane < blocks ? L->blk[lane] : 0u;
        const uint32_t hi = wave_incl_u32(h);
        const uint64_t past = ballot(hi > nth);
        const uint32_t blk = past ? (uint32_t)__builtin_ctzll(past) : blocks - 1;
        uint32_t left = nth - read_lane_u32(hi - h, blk);
        float x[U];
        fetch(blk, x);
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) {
            const bool is = matches(blk, x, i);
            const uint64_t k = ballot(is);
            if (is && lanes_below(k) == left) a.out_token[row] = e0 + blk * VAL_BLOCK + i * WAVE + lane;
            left -= (uint32_t)__popcll(k);  // wraps once the occurrence is past
        }
    }
    return true;
}

}  // namespace rl
