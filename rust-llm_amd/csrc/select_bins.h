// The selection path's bins: which part of a row k_full_gather collects.
//
// A row that keeps the head of the descending order (top-k, or top-p over the
// whole vocabulary) needs only that head sorted. k_full_pass counts its
// penalised logits into SEL_BINS bins that fall along the order (bin 0 holds
// the largest), and every chunk of k_full_gather picks the bin down to which the
// head reaches. A bin only decides which elements are collected: the row is then
// finished from the exact values, or left to k_full_rest.
//
// The bins are spaced in the distance of a logit from a reference value R (the
// maximum of the row's first SEL_SAMPLE logits, so that every chunk has it
// without hearing of the others): 64 to an octave of |R - v| between 2^-10 and
// 2^8, on either side of R, the ends taking what lies beyond. So a bin is
// about 1.1-1.6 % of the distance from R wide, wherever the row's logits lie
// and however far they spread: a few per cent of a logit where a trained
// head's candidates end, and at most about one part in sixty of a row spread
// like a normal distribution.
//
// Plain C++ (no device dependency), so that a host-built test can check that
// the bins fall along the order.
#pragma once
#include <stdint.h>
#include <string.h>

#ifndef RL_HD
#ifdef __HIPCC__
#define RL_HD __host__ __device__
#else
#define RL_HD
#endif
#endif

namespace rl {

constexpr uint32_t SEL_OCTAVES = 18;
constexpr uint32_t SEL_SIDE = 64 * SEL_OCTAVES;  // bins on either side of R
constexpr uint32_t SEL_BINS = 2 * SEL_SIDE;
constexpr uint32_t SEL_SAMPLE = 1024;            // logits R is taken from
constexpr uint32_t SEL_NONE = 0xFFFFFFFFu;       // FullRow::thr of a row that is not collected
// Collected elements are sorted a group at a time: a group is the bins whose
// first element's rank shares its upper bits, at most SEL_GROUP elements and
// the rest of a last bin. No bin of a collected head holds more than SEL_GROUP:
// a fuller one could reach past the next group, which no bin would then start.
constexpr uint32_t SEL_GROUP_LOG = 12;
constexpr uint32_t SEL_GROUP = 1u << SEL_GROUP_LOG;
constexpr uint32_t SEL_GROUP_CAP = 2 * SEL_GROUP;  // most elements of a group (no bin above SEL_GROUP)
constexpr uint32_t SEL_GROUPS = 64;                // most groups of a row
// A head on the bf16 grid that is too long for one workgroup's LDS is collected
// when this many times its elements, shared by the row's workgroups of
// k_full_head, are no more than twice the vocabulary. Its few distinct values crowd
// the sort's buckets, so a group takes a sorting network's time (75-85 us
// against 20), while k_full_rest sorts such a row in two passes instead of four:
// 151936 N(0, 2^2) ids at top-p 0.9, nine groups a row, take 303 us collected at
// 64 rows (four workgroups a row) against 510 sorted whole, and 832 against 543
// at 256 (one); nearly flat ones, 34 groups, 238 against 439 at 8 rows, but 691
// against 450 at 64 and 2110 against 481 at 256. Rows off the grid gain to the
// end (256 nearly flat rows 830 against 982). Penalised logits leave the grid,
// and the whole sort then takes its four passes too (256 nearly flat rows 1065
// against 2115 collected, N(0, 2^2) 1066 against 840).
constexpr uint32_t SEL_GRID_SHARE = 12, SEL_GRID_SHARE_PEN = 3;
// Below this vocabulary, where the whole sort takes 45-100 us, a head with a bin
// of more than SEL_SMALL_TIES is left to it: the bin's ties crowd the sort's
// buckets (4 x 2854 ids, 40 % tied, at top-p 0.95: 54 us sorted, 82 collected);
// and so is a head of every id (37 x 15680: 116 us sorted, 174 collected).
constexpr uint32_t SEL_SMALL_VOCAB = 16384, SEL_SMALL_TIES = 512;
// k_full_gather reads a row in chunks of whole float4, each of at least one and
// of at most SEL_CHUNK_MAX elements (a window bitmap of 8 KiB; the last chunk
// takes the row's vocab % 4 besides).
constexpr uint32_t SEL_CHUNK_MAX = 65536;
constexpr uint32_t SEL_MIN_VOCAB = 4;

// Whether a row takes the selection path (full_select.h): it keeps the head of
// the descending order, by top-k (top_k < V), or by top-p alone over the whole
// vocabulary (with min-p on it tries the min-p path). The host's rule; a
// vocabulary without a float4 to read launches no selection kernel, and its
// rows are left to k_full_rest.
inline bool sel_takes(float temperature, uint64_t top_k, float top_p, float min_p, uint32_t V) {
    const bool by_k = top_k != 0 && top_k < V;
    return V >= SEL_MIN_VOCAB && temperature > 0.0f && (by_k || (top_p < 1.0f && !(min_p > 0.0f)));
}

// The gather's chunks a row when `want` are wished for (vocab >= SEL_MIN_VOCAB):
// each of at least a float4 for each of a workgroup's `threads`, or one chunk,
// and as many as SEL_CHUNK_MAX asks for.
RL_HD inline uint32_t sel_gather_chunks(uint32_t vocab, uint32_t want, uint32_t threads) {
    const uint32_t most = vocab / (4 * threads), least = (vocab + SEL_CHUNK_MAX - 1) / SEL_CHUNK_MAX;
    const uint32_t c = want < most ? want : most;
    return c > least ? c : least;
}

// Chunk c of n items split into `chunks`: [chunk_lo(c), chunk_lo(c + 1)).
// Callers split a row's float4 (n <= 2^19, the vocabulary being at most 2^21)
// into at most FULL_CHUNKS, so n * c fits 32 bits.
RL_HD inline uint32_t chunk_lo(uint32_t n, uint32_t c, uint32_t chunks) { return n * c / chunks; }

RL_HD inline uint32_t sel_bits(float v) {
#ifdef __HIP_DEVICE_COMPILE__
    return __float_as_uint(v);
#else
    uint32_t b;
    memcpy(&b, &v, 4);
    return b;
#endif
}
RL_HD inline float sel_float(uint32_t b) {
#ifdef __HIP_DEVICE_COMPILE__
    return __uint_as_float(b);
#else
    float v;
    memcpy(&v, &b, 4);
    return v;
#endif
}

// The bits of the distance at which side bin 0 starts, and of one bin.
constexpr int32_t SEL_LO = (127 - 10) << 6;
constexpr uint32_t SEL_STEP_BITS = 17;

// The bin of logit v (not NaN) for the reference r (finite, not -0): never falls as v
// falls, since r - v is one rounding of a decreasing function and the bins
// follow its bits (the octave and the six bits below it: bits 17..30).
RL_HD inline uint32_t sel_bin(float v, float r) {
    const uint32_t b = sel_bits(r - v);
    int32_t j = (int32_t)((b & 0x7FFFFFFFu) >> SEL_STEP_BITS) - SEL_LO;
    j = j < 0 ? 0 : j;
    j = j > (int32_t)SEL_SIDE - 1 ? (int32_t)SEL_SIDE - 1 : j;
    return (b >> 31) ? SEL_SIDE - 1 - (uint32_t)j : SEL_SIDE + (uint32_t)j;
}

// The largest logit a bin holds, as far as the bins' spacing says (the end
// bins reach further).
RL_HD inline float sel_edge(uint32_t bin, float r) {
    return bin < SEL_SIDE ? r + sel_float((uint32_t)(SEL_LO + (int32_t)(SEL_SIDE - bin)) << SEL_STEP_BITS)
           : bin == SEL_SIDE ? r
                             : r - sel_float((uint32_t)(SEL_LO + (int32_t)(bin - SEL_SIDE)) << SEL_STEP_BITS);
}

// A bin's mass is summed as whole parts of the p at its edge, 1 / SEL_MASS_ONE
// each: LDS adds integers at the rate of stores and floats several times
// slower (the one-row pass took 18 us with f32 sums against 11 with these).
// SEL_MASS_ONE parts of 2^21 logits fit 32 bits.
constexpr float SEL_MASS_ONE = 1024.0f;

// The bin of v, and in *below how far v lies below its edge (for v beyond the
// end bins' spacing, below the edge its own spacing would have).
RL_HD inline uint32_t sel_bin(float v, float r, float *below) {
    const float d = r - v;
    const uint32_t b = sel_bits(d);
    const uint32_t cut = (b & 0x7FFFFFFFu) >> SEL_STEP_BITS << SEL_STEP_BITS;
    *below = (b >> 31) ? sel_float(cut + (1u << SEL_STEP_BITS)) + d : d - sel_float(cut);
    return sel_bin(v, r);
}

// The interval that holds the reference's top-p target, top_p * S_ref, from a
// sum S of the row's V terms p_j in f64 in any order. The terms are the
// reference's own f32 values, all non-negative, so S and the sequential S_ref
// are each within gamma_(V - 1) of the exact sum (V - 1 additions, whatever
// their order), and the target adds one rounding.
RL_HD inline void sel_target_interval(double S, uint32_t V, float top_p, double *t_lo, double *t_hi) {
    const double rel = (2.0 * (double)V + 64.0) * 0x1p-53;
    const double t = (double)top_p * S;
    const double w = (t < 0.0 ? -t : t) * rel;
    *t_lo = t - w;
    *t_hi = t + w;
}

}  // namespace rl
