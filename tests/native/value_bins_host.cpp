// Test harness (host only; test infrastructure): the value path's bins
// (rust-llm_amd/csrc/value_bins.h) built by the host compiler.
#include "value_bins.h"

extern "C" {

uint32_t val_window(uint32_t most) { return rl::val_window(most); }

void val_bins(const uint32_t *bits, uint32_t lo, uint64_t n, uint32_t *bin, uint32_t *back) {
    for (uint64_t i = 0; i < n; ++i) {
        bin[i] = rl::val_bin(bits[i], lo);
        back[i] = bin[i] == rl::VAL_NONE ? 0u : rl::val_bits(bin[i], lo);
    }
}

// The bits of the values at every place of the order that a value can take.
uint32_t val_all(uint32_t lo, uint32_t *bits) {
    uint32_t n = 0;
    for (uint32_t o = 0; o < rl::VAL_BINS; ++o) {
        const uint32_t bin = rl::val_order(o), b = rl::val_bits(bin, lo);
        if (rl::val_bin(b, lo) == bin) bits[n++] = b;
    }
    return n;
}

uint32_t val_bin_count() { return rl::VAL_BINS; }

}
