"""The min-p path's rows with more survivors than a wave holds: at the sizes
where the workgroup's finish changes its sort (a survivor a thread up to 256)
and its walks (64 terms in a wave's lanes, four a test), with and without
top-p, against the oracle."""
import numpy as np
import pytest

import rl_sampler as R
from test_gpu_long_windows import assert_rows_match, run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_top", [65, 95, 96, 97, 255, 256, 257, 511, 513, 1023])
def test_finish_of_a_block(device, n_top):
    print("survivors", n_top, flush=True)
    rng = np.random.default_rng(n_top)
    V, rows = 9001, 6
    x = np.full((rows, V), -90.0, np.float32)
    for r in range(rows):
        x[r, rng.permutation(V)[:n_top]] = rng.normal(0.0, 0.7, n_top).astype(np.float32).clip(-2, 2)
    x[3, x[3] > -3] = 0.5  # tied survivors: id order
    settings = [R.sampling(1.0, 0, 0.9, 0.01, 1.0, 0, 1), R.sampling(1.3, 0, 1.0, 0.01, 1.0, 0, 2),
                R.sampling(1.0, 0, 0.9999, 0.01, 1.0, 0, 3), R.sampling(1.0, 0, 0.5, 0.01, 1.0, 0, 4),
                R.sampling(0.9, 0, 0.0, 0.005, 1.0, 0, 5), R.sampling(1.1, 0, 0.97, 0.02, 1.0, 0, 6)]
    u = rng.random(rows).astype(np.float32)
    u[1] = np.float32(1.0 - 2.0 ** -24)
    got, want = run_case(device, x, settings, np.zeros((rows, 64), np.uint32), np.zeros(rows, np.uint32), u, "own",
                         max_window=64)
    assert_rows_match("survivors %d" % n_top, got, want, settings)


@pytest.mark.parametrize("n_top", [20, 65, 130, 300])
def test_uniforms_outside_the_draw(device, n_top):
    """The draw is the reference's comparison whatever the uniform: below 0 the
    first candidate, at 1 and above (and for NaN) the last."""
    print("uniforms outside", n_top, flush=True)
    rng = np.random.default_rng(7 * n_top)
    V, u = 9001, np.array([-0.5, -1e-30, -0.0, 0.0, 1.0, 3.0, np.nan, -np.inf], np.float32)
    rows = u.size
    x = np.full((rows, V), -90.0, np.float32)
    for r in range(rows):
        x[r, rng.permutation(V)[:n_top]] = rng.normal(0.0, 0.7, n_top).astype(np.float32).clip(-2, 2)
    for st in (R.sampling(1.0, 0, 0.9999, 0.01, 1.0, 0, 1), R.sampling(1.0, 0, 1.0, 0.01, 1.0, 0, 2),
               R.sampling(1.0, 0, 0.9, 0.0, 1.0, 0, 3), R.sampling(1.0, 70, 0.95, 0.0, 1.0, 0, 4)):
        got, want = run_case(device, x, [st] * rows, np.zeros((rows, 64), np.uint32), np.zeros(rows, np.uint32), u,
                             "own", max_window=64)
        assert_rows_match("%d survivors" % n_top, got, want, [st] * rows)
