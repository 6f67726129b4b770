// Test harness (host only; test infrastructure): the selection path's bins and
// top-p interval (rust-llm_amd/csrc/select_bins.h) built by the host compiler.
#include "select_bins.h"

extern "C" {

void sel_bins(const float *v, float r, uint64_t n, uint32_t *bin, float *below, float *edge) {
    for (uint64_t i = 0; i < n; ++i) {
        bin[i] = rl::sel_bin(v[i], r, &below[i]);
        edge[i] = rl::sel_edge(bin[i], r);
    }
}

uint32_t sel_bin_count() { return rl::SEL_BINS; }

void sel_interval(double s, uint32_t vocab, float top_p, double *lo, double *hi) {
    rl::sel_target_interval(s, vocab, top_p, lo, hi);
}

}
