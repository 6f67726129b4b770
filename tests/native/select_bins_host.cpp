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

uint32_t sel_takes_row(float temperature, uint64_t top_k, float top_p, float min_p, uint32_t vocab) {
    return rl::sel_takes(temperature, top_k, top_p, min_p, vocab);
}

// The gather's chunks for `vocab`, the fewest float4 of one of them, and the
// most elements of one.
uint32_t sel_chunks(uint32_t vocab, uint32_t want, uint32_t *fewest4, uint32_t *most) {
    const uint32_t n4 = vocab / 4, C = rl::sel_gather_chunks(vocab, want, 1024);
    *fewest4 = 0xFFFFFFFFu;
    *most = 0;
    for (uint32_t c = 0; c < C; ++c) {
        const uint32_t q0 = rl::chunk_lo(n4, c, C), q1 = rl::chunk_lo(n4, c + 1, C);
        const uint32_t n = (c == C - 1 ? vocab : 4 * q1) - 4 * q0;
        if (q1 - q0 < *fewest4) *fewest4 = q1 - q0;
        if (n > *most) *most = n;
    }
    return C;
}

void sel_interval(double s, uint32_t vocab, float top_p, double *lo, double *hi) {
    rl::sel_target_interval(s, vocab, top_p, lo, hi);
}

}
