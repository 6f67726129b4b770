"""Short heads of the selection path around the sizes where their finish
changes: 256 collected elements (sorted by counting, or by buckets) and 1024
candidates (one a thread, or four), against the oracle."""
import numpy as np
import pytest

import rl_sampler as R
from test_gpu_long_windows import assert_rows_match, run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [66, 248, 252, 255, 256, 257, 1023, 1024, 1025])
def test_heads_around_a_change_of_sort(device, k):
    print("short head", k, flush=True)
    rng = np.random.default_rng(k)
    V, rows = 20003, 5
    x = rng.normal(0.0, 2.0, (rows, V)).astype(np.float32)
    # A gap below the k best of some rows: the head collected is then k elements.
    for r in (0, 1, 2):
        x[r] = -40.0 - np.abs(x[r])
        x[r, rng.permutation(V)[:k]] = rng.normal(0.0, 1.0, k).astype(np.float32)
    x[2, x[2] > -10] = 1.25  # tied
    settings = [R.sampling(1.0, k, 1.0, 0.0, 1.0, 0, 1), R.sampling(0.8, k, 0.95, 0.0, 1.0, 0, 2),
                R.sampling(1.0, k, 0.9, 0.0, 1.0, 0, 3), R.sampling(1.3, k, 0.999, 0.001, 1.0, 0, 4),
                R.sampling(0.1, k, 0.99, 0.0, 1.0, 0, 5)]
    u = rng.random(rows).astype(np.float32)
    u[0] = np.float32(1.0 - 2.0 ** -24)
    got, want = run_case(device, x, settings, np.zeros((rows, 64), np.uint32), np.zeros(rows, np.uint32), u, "own",
                         max_window=64)
    assert_rows_match("short head %d" % k, got, want, settings)
