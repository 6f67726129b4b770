"""The selection path's bins (select_bins.h, the kernels' own header built for
the host): a row's head is collected by bin, so the bins must fall along the
order for every pair of logits, and the top-p interval must hold the
reference's target for a sum of p in any order (sample.rs:307-324)."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libselect_bins.so")


@pytest.fixture(scope="module")
def lib():
    L = ctypes.CDLL(LIB)
    p = ctypes.c_void_p
    L.sel_bins.argtypes = [p, ctypes.c_float, ctypes.c_uint64, p, p, p]
    L.sel_interval.argtypes = [ctypes.c_double, ctypes.c_uint32, ctypes.c_float, p, p]
    L.sel_takes_row.argtypes = [ctypes.c_float, ctypes.c_uint64, ctypes.c_float, ctypes.c_float, ctypes.c_uint32]
    L.sel_chunks.argtypes = [ctypes.c_uint32, ctypes.c_uint32, p, p]
    return L


def bins(L, v, r):
    v = np.ascontiguousarray(v, np.float32)
    b, below, edge = np.empty(v.size, np.uint32), np.empty(v.size, np.float32), np.empty(v.size, np.float32)
    L.sel_bins(v.ctypes.data, r, v.size, b.ctypes.data, below.ctypes.data, edge.ctypes.data)
    return b, below, edge


@pytest.mark.parametrize("r", [0.0, 1.0, 3.25, -7.5, 12.0, 1e-30, 4096.0, -3e38, 3e38, 1e-45])
def test_bins_never_fall_as_the_logit_falls(lib, r):
    rng = np.random.default_rng(11)
    r = float(np.float32(r))
    any_bits = rng.integers(0, 2**32, 200_000, dtype=np.uint64).astype(np.uint32).view(np.float32)
    near = (r + rng.normal(0, 1, 100_000) * 10.0 ** rng.uniform(-6, 2.5, 100_000)).astype(np.float32)
    special = np.array([np.inf, -np.inf, 0.0, -0.0, 3.4028235e38, -3.4028235e38, r], np.float32)
    v = np.concatenate([any_bits, near, special])
    v = np.sort(v[~np.isnan(v)])[::-1]
    b, _, _ = bins(lib, v, r)
    assert np.all(np.diff(b.astype(np.int64)) >= 0)
    assert b.max() < lib.sel_bin_count()


def test_a_bin_is_narrow_and_its_edge_lies_above_it(lib):
    rng = np.random.default_rng(12)
    r = 4.0
    v = (r + rng.choice([-1, 1], 200_000) * 2.0 ** rng.uniform(-9.5, 7.5, 200_000)).astype(np.float32)
    b, below, edge = bins(lib, v, r)
    d = np.abs(v.astype(np.float64) - r)
    tol = 4e-7 * (abs(r) + d)
    assert np.all(edge.astype(np.float64) - v >= -tol)
    assert np.all(edge.astype(np.float64) - v <= d / 64 + tol)
    assert np.all(np.abs(below - (edge.astype(np.float64) - v)) <= tol)


def test_the_interval_holds_the_target_for_sums_in_any_order(lib):
    rng = np.random.default_rng(13)
    lo, hi = ctypes.c_double(), ctypes.c_double()
    for n, spread in ((65, 1.0), (5003, 30.0), (248320, 0.01), (248320, 12.0), (1 << 18, 80.0)):
        p = np.sort(np.exp(-rng.random(n) * spread).astype(np.float32))[::-1]
        seq = 0.0
        for x in p.tolist():
            seq += x
        for order in (np.arange(n)[::-1], rng.permutation(n)):
            s = float(np.cumsum(p[order], dtype=np.float64)[-1])
            for top_p in (0.0, 0.1, 0.95, 0.9999, -0.5):
                lib.sel_interval(s, n, top_p, ctypes.byref(lo), ctypes.byref(hi))
                t = float(np.float32(top_p)) * seq
                assert lo.value <= t <= hi.value
                assert hi.value - lo.value <= 1e-9 * max(abs(t), 1e-300) or t == 0.0


def test_every_chunk_of_a_row_it_takes_can_be_read(lib):
    """A chunk clamps its reads to its own last float4, so it must have one;
    its window bitmap holds SEL_CHUNK_MAX elements and the row's vocab % 4."""
    fewest, most = ctypes.c_uint32(), ctypes.c_uint32()
    rng = np.random.default_rng(14)
    vocabs = list(range(1, 9000)) + [2**21 - d for d in range(5)] + rng.integers(9000, 2**21, 3000).tolist()
    vocabs += [65536 * m + d for m in range(1, 32) for d in range(-5, 6)]
    for V in vocabs:
        takes = [lib.sel_takes_row(1.0, 0, 0.9, 0.0, V), lib.sel_takes_row(1.0, 65, 1.0, 0.0, V),
                 lib.sel_takes_row(0.5, 1, 0.9, 0.1, V)]
        assert takes == [V >= 4, V > 65, V >= 4], V
        if not any(takes):
            continue
        for want in (64, 32, 5, 1):
            c = lib.sel_chunks(V, want, ctypes.byref(fewest), ctypes.byref(most))
            assert 1 <= c <= 64 and fewest.value >= 1 and most.value <= 65536 + 3, (V, want, c)


def test_rows_it_does_not_take(lib):
    nan = float("nan")
    for t, k, top_p, min_p in ((0.0, 0, 0.9, 0.0), (-1.0, 100, 0.9, 0.0), (nan, 100, 0.9, 0.0), (1.0, 0, 1.0, 0.0),
                               (1.0, 0, nan, 0.0), (1.0, 5000, 1.0, 0.0), (1.0, 2**40, 1.5, 0.0), (1.0, 0, 0.9, 0.05)):
        assert lib.sel_takes_row(t, k, top_p, min_p, 5000) == 0, (t, k, top_p, min_p)
    assert lib.sel_takes_row(1.0, 0, 0.9, nan, 5000) == 1  # min_p > 0 does not hold
