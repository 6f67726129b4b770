"""The value path's bins (value_bins.h, the kernels' own header built for the
host): a bin is one value, the bins fall along the descending total order, and
no bin is taken by a value off the bf16 grid, a NaN or +inf."""
import ctypes
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libvalue_bins.so")


@pytest.fixture(scope="module")
def lib():
    L = ctypes.CDLL(LIB)
    p = ctypes.c_void_p
    L.val_bins.argtypes = [p, ctypes.c_uint32, ctypes.c_uint64, p, p]
    L.val_all.argtypes = [ctypes.c_uint32, p]
    return L


@pytest.mark.parametrize("most", [0.03125, 1.0, 12.0, 3.0e38, 1e-30, 1e-40, 0.0, -7.5])
def test_a_bin_is_a_value_of_the_grid(lib, most):
    lo = lib.val_window(int(np.float32(most).view(np.uint32)))
    bits = (np.arange(65536, dtype=np.uint32) << np.uint32(16))
    bits = np.concatenate([bits, bits | np.uint32(1), bits | np.uint32(0x8000)])
    b, back = np.empty_like(bits), np.empty_like(bits)
    lib.val_bins(bits.ctypes.data, lo, bits.size, b.ctypes.data, back.ctypes.data)
    has = b != 0xFFFFFFFF
    assert np.array_equal(back[has], bits[has])
    assert np.unique(b[has]).size == has.sum() == lib.val_bin_count() - 3
    v = bits.view(np.float32)
    assert not np.any(has & (np.isnan(v) | (v == np.inf) | ((bits & 0xFFFF) != 0)))
    assert has[0] and has[0x8000] and has[0xFF80]  # the zeros and -inf
    mag = np.abs(v)
    m = abs(float(np.float32(most)))
    if m >= 2.0 ** -112 and m < 1e38:  # the window clear of the exponents' ends
        inside = ((bits & 0xFFFF) == 0) & (mag < 2 * m) & (mag >= m * 2.0 ** -13) & np.isfinite(v)
        assert np.all(has[inside])


@pytest.mark.parametrize("most", [0.03125, 3.0e38, 0.0])
def test_bins_fall_along_the_total_order(lib, most):
    lo = lib.val_window(int(np.float32(most).view(np.uint32)))
    bits = np.empty(lib.val_bin_count(), np.uint32)
    n = lib.val_all(lo, bits.ctypes.data)
    assert n == bits.size - 3  # the window's largest magnitudes and one smallest
    bits = bits[:n]
    key = np.where(bits >> 31, ~bits, bits | np.uint32(0x80000000)).astype(np.int64)
    assert np.all(np.diff(key) < 0)
