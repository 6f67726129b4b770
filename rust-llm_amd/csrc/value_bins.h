// The value path's bins: one for each value that a row on the bf16 grid can
// hold in a window of sixteen octaves.
//
// A nearly flat row of a head computed in bf16 has some thousand distinct
// logits. What such a row's sampling needs of them (its mass, its top-p cut,
// its draw) follows from how often each value occurs, so k_full_pass counts the
// values instead of listing candidates, and k_full_rest finishes the row from
// the counts (full_values.h) without sorting the vocabulary.
//
// The window is given by lo, the upper 15 magnitude bits of its start. Every
// value whose low 16 bits are zero and whose magnitude lies in the window has a
// bin, and so have the two zeros and -inf. Anything else (a penalised logit off
// the grid, a magnitude outside the window, a NaN) has none and is listed by
// itself. A bin is its magnitude's distance from the window's start, the
// negative values after the positive ones (few operations for the pass);
// val_order turns it into its place along the descending total order.
//
// Plain C++ (no device dependency), so that a host-built test can check that
// the bins are the values and fall along the order.
#pragma once
#include <stdint.h>

#include "select_bins.h"

namespace rl {

constexpr uint32_t VAL_SPAN = 16u << 7;   // a magnitude's exponent and seven significand bits, over sixteen octaves
constexpr uint32_t VAL_BINS = 2 * VAL_SPAN;
constexpr uint32_t VAL_NONE = 0xFFFFFFFFu;

// The window for rows whose largest magnitude has the bits `most` (finite): up
// to the octave above it, so that a maximum taken from a sample serves.
// Never 0, and below the infinities.
RL_HD inline uint32_t val_window(uint32_t most) {
    const int32_t e = (int32_t)((most & 0x7FFFFFFFu) >> 23) - 14;
    const uint32_t first = e < 1 ? 1u : e > 239 ? 239u : (uint32_t)e;
    return first << 7;
}

// The places in the window that are values': its two smallest magnitudes and
// its largest have no bin, since the zeros (bins 1 and 0) and -inf (the last
// bin) take theirs.
constexpr uint32_t VAL_FIRST = 2, VAL_LAST = VAL_SPAN - 2;

// The magnitude's distance from the window's start for the value with bits b;
// VAL_SPAN or more when it lies before it, past it or off the grid (the low 16
// bits then end up above the others).
RL_HD inline uint32_t val_dist(uint32_t b, uint32_t lo) { return (((b >> 16) | (b << 16)) & ~0x8000u) - lo; }

// The bin of the value with bits b, or VAL_NONE.
RL_HD inline uint32_t val_bin(uint32_t b, uint32_t lo) {
    const uint32_t d = val_dist(b, lo);
    if (d - VAL_FIRST <= VAL_LAST - VAL_FIRST) return d + ((b >> 31) ? VAL_SPAN : 0u);
    if ((b & 0x7FFFFFFFu) == 0) return 1u - (b >> 31);
    return b == 0xFF800000u ? VAL_BINS - 1 : VAL_NONE;
}

// A bin's place along the descending order, and the bin of a place.
RL_HD inline uint32_t val_order(uint32_t bin) { return bin < VAL_SPAN ? VAL_SPAN - 1u - bin : bin; }

// The bits of the value of a bin that a value can take.
RL_HD inline uint32_t val_bits(uint32_t bin, uint32_t lo) {
    if (bin < VAL_FIRST) return bin ? 0u : 0x80000000u;
    if (bin == VAL_BINS - 1) return 0xFF800000u;
    return bin < VAL_SPAN ? (lo + bin) << 16 : 0x80000000u | ((lo + bin - VAL_SPAN) << 16);
}

}  // namespace rl
