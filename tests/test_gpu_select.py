"""The selection path on the GPU (top-k above 64, and top-p over the whole
vocabulary) against the oracle, bit for bit: heads of a few elements, around
the 4096 that one workgroup finishes, and of many groups; rows it hands to the
whole-row sort (ties, NaN, a top-p near 1); odd and unaligned rows; rows of it
beside rows of the other paths in one call; calls repeated on one context."""
import numpy as np
import pytest

import rl_sampler as R
from test_gpu_long_windows import assert_rows_match, run_case
from test_gpu_values import to_grid

pytestmark = pytest.mark.gpu


def logits_of(kind, rng, rows, V):
    x = rng.normal(0.0, 2.0, (rows, V))
    if kind == "zipf":
        x = rng.normal(0.0, 3.0, (rows, V)) - 1.1 * np.log(rng.permutation(V) + 1.0)
    elif kind == "offset":     # every logit in one octave
        x += 24.0
    elif kind == "flat":
        x *= 0.005
    elif kind == "bf16":
        x = (x.astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    elif kind == "masked":     # most ids ruled out
        x[:, rng.random(V) < 0.9] = -np.inf
    elif kind == "outlier":    # one logit far above the rest crowds the sort's buckets
        x[:, V // 3] = 3e4
    elif kind == "tied":       # one value for all but a few
        x[:, :] = 1.5
        x[:, :: 97] = rng.normal(0.0, 1.0, x[:, :: 97].shape)
    elif kind == "specials":
        x[0, 5] = np.nan
        x[1, V - 1] = np.inf
        x[2, :] = -np.inf
        x[3, V // 2] = -np.nan
        x[4, :] = np.nan
        x[5, :] = -np.inf
        x[5, 7] = -3.0
        x[6, :2000] = -np.inf  # the sample of the reference value
        x[7, :] = 0.0
        x[7, ::2] = -0.0
    return x.astype(np.float32)


SETTINGS = [
    R.sampling(0.8, 65, 0.95, 0.0, 1.0, 0, 1),
    R.sampling(1.0, 100, 1.0, 0.0, 1.3, 64, 2),
    R.sampling(1.2, 4095, 0.999, 0.0, 1.1, 64, 3),
    R.sampling(3.0, 4096, 0.9, 0.0, 1.0, 0, 4),
    R.sampling(2.0, 4097, 1.0, 0.001, 1.0, 0, 5),
    R.sampling(2.0, 9000, 0.97, 0.0, 0.8, 64, 6),
    R.sampling(1.0, 100, 0.9, 0.2, 1.0, 0, 7),
    R.sampling(0.05, 300, 0.95, 0.0, 1.0, 0, 8),       # p far below the sums' exact range
    R.sampling(0.7, 0, 0.8, 0.0, 1.1, 64, 9),
    R.sampling(1.0, 0, 0.95, 0.0, 1.0, 0, 10),
    R.sampling(1.5, 0, 0.99, 0.0, 1.2, 64, 11),
    R.sampling(0.01, 0, 0.9, 0.0, 1.0, 0, 12),
    R.sampling(4.0, 0, 0.9, 0.0, 1.0, 0, 13),
    R.sampling(1.0, 0, 0.99999, 0.0, 1.0, 0, 14),
    R.sampling(1.0, 0, 0.0, 0.0, 1.0, 0, 15),
    R.sampling(1.0, 0, 1e-30, 0.0, 1.0, 0, 16),
]


def settings_for(V, rows):
    out = []
    for r in range(rows):
        s = SETTINGS[r % len(SETTINGS)]
        if s.top_k >= V:
            s = R.sampling(s.temperature, V - 1, s.top_p, s.min_p, s.repeat_penalty, s.repeat_last_n, s.seed)
        out.append(s)
    return out


def check(device, label, logits, settings, rng):
    rows, V = logits.shape
    win = rng.integers(0, V + 5, (rows, 64)).astype(np.uint32)
    top = np.argsort(np.nan_to_num(logits, nan=-1e30), axis=1)[:, -24:]
    win[:, 8:32] = top  # ids the penalty moves
    wlen = rng.integers(0, 65, rows).astype(np.uint32)
    u = rng.random(rows).astype(np.float32)
    u[0] = np.float32(1.0 - 2.0 ** -24)
    got, want = run_case(device, logits, settings, win, wlen, u, "own", max_window=64)
    assert_rows_match(label, got, want, settings)


@pytest.mark.parametrize("kind", ["normal", "zipf", "offset", "flat", "bf16", "masked", "outlier", "tied", "specials"])
@pytest.mark.parametrize("V", [4099, 50004])
def test_heads_match_the_oracle(device, kind, V):
    print("select", kind, V, flush=True)
    rng = np.random.default_rng([ord(c) for c in kind] + [V])
    logits = logits_of(kind, rng, len(SETTINGS), V)
    check(device, kind, logits, settings_for(V, len(SETTINGS)), rng)


@pytest.mark.parametrize("V", [66, 257, 1023, 8193, 151937])
def test_vocabulary_edges(device, V):
    print("select vocabulary", V, flush=True)
    rng = np.random.default_rng(V)
    rows = 8
    logits = logits_of("zipf", rng, rows, V)
    st = settings_for(V, 16)
    check(device, "V %d top-k" % V, logits, st[:rows], rng)
    check(device, "V %d top-p" % V, logits, st[8:8 + rows], rng)


@pytest.mark.parametrize("V", [1, 2, 3, 4, 5, 7, 8, 9])
def test_smallest_vocabularies(device, V):
    """Below four ids a row has no float4 to gather (it is sorted whole); from
    four on it is gathered from one or two, top-p alone, one row and several."""
    for rows in (1, 6):
        print("select smallest", V, rows, flush=True)
        rng = np.random.default_rng(20 + V + rows)
        logits = rng.normal(0.0, 1.0, (rows, V)).astype(np.float32)
        st = [R.sampling(0.9, 0, tp, 0.0, 1.1, 64, r) for r, tp in enumerate((0.9, 0.5, 0.99, 0.0, 0.999, 0.3))][:rows]
        win = rng.integers(0, V + 2, (rows, 64)).astype(np.uint32)
        got, want = run_case(device, logits, st, win, np.full(rows, 3, np.uint32),
                             rng.random(rows).astype(np.float32), "own", max_window=64)
        assert_rows_match("V %d" % V, got, want, st)


@pytest.mark.parametrize("rows", [1, 3, 70, 300])
def test_rows_beside_other_paths(device, rows):
    print("select mixed", rows, flush=True)
    rng = np.random.default_rng(rows)
    V = 9001
    logits = logits_of("zipf", rng, rows, V)
    st = settings_for(V, rows)
    for r in range(rows):
        if r % 5 == 3:
            st[r] = R.sampling(1.0, 0, 0.95, 0.05, 1.0, 0, r)     # min-p
        elif r % 11 == 7:
            st[r] = R.sampling(0.6, 20, 0.95, 0.0, 1.0, 0, r)     # stream
        elif r % 13 == 5:
            st[r] = R.sampling(1.0, 0, 1.0, 0.0, 1.0, 0, r)       # id order
    check(device, "mixed %d" % rows, logits, st, rng)


def test_a_context_is_reused(device):
    """Bins and counters return to zero: calls over other logits on one
    context, without candidates, equal the same calls on a new one."""
    import torch
    V, rows = 30011, 6
    st = settings_for(V, 16)[5:11]
    ctx = R.DeviceSampler(rows, V, max_window=64)
    ctx.configure(st)
    for i, kind in enumerate(["zipf", "normal", "specials", "flat", "zipf", "normal"]):
        rng = np.random.default_rng(100 + i)
        x = logits_of(kind, rng, max(rows, 8), V)[:rows]
        u = torch.from_numpy(rng.random(rows).astype(np.float32)).to(device)
        d = torch.from_numpy(x).to(device)
        res = []
        for c in (ctx, None):
            if c is None:
                c = R.DeviceSampler(rows, V, max_window=64)
                c.configure(st)
            tok = torch.empty(rows, dtype=torch.int32, device=device)
            kept, used = torch.empty_like(tok), torch.empty(rows, dtype=torch.uint8, device=device)
            c.sample_rows(d, rows, V, tok, kept, used, uniforms=u)
            torch.cuda.synchronize()
            res.append((tok.tolist(), kept.tolist(), used.tolist()))
        assert res[0] == res[1], (kind, res)


@pytest.mark.parametrize("top_p,penalty", [(0.9, 1.0), (0.5, 1.0), (0.9, 1.1), (-0.5, 1.0)])
def test_long_heads_on_the_grid_at_many_rows(device, top_p, penalty):
    """One workgroup a row: heads of bf16 logits past three groups of 4096 are
    sorted whole, shorter ones and penalised ones collected; a top_p below 0
    keeps the first candidate."""
    print("select grid", top_p, penalty, flush=True)
    rng = np.random.default_rng(31)
    V, rows = 20004, 256
    x = np.repeat(to_grid(rng.normal(0.0, 0.01, (4, V))), rows // 4, axis=0)
    x[:: 3, ::2] = 0.015625  # every second id tied, in and above the head
    st = [R.sampling(1.0, 0, top_p, 0.0, penalty, 64, r) for r in range(rows)]
    check(device, "grid", x, st, rng)


def test_heads_that_leave_nothing_out(device):
    """top-k one below the vocabulary and top-p next to 1: the bins reach the
    row's end, with ties there and without."""
    print("select whole rows", flush=True)
    rng = np.random.default_rng(32)
    for V in (3001, 50004):
        x = rng.normal(0.0, 2.0, (6, V)).astype(np.float32)
        x[1::2, rng.random(V) < 0.02] = -9.0
        x[4, :] = 0.5
        st = [R.sampling(1.0, V - 1, 1.0, 0.0, 1.1, 64, 1), R.sampling(1.0, V - 1, 0.9, 0.0, 1.0, 0, 2),
              R.sampling(1.0, 0, 0.9999999, 0.0, 1.0, 0, 3), R.sampling(2.0, V - 2, 1.0, 0.001, 1.0, 0, 4),
              R.sampling(1.0, V - 1, 1.0, 0.0, 1.0, 0, 5), R.sampling(0.1, 0, 0.9999999, 0.0, 1.0, 0, 6)]
        check(device, "whole %d" % V, x, st, rng)


def test_largest_vocabularies(device):
    """Eight rows of 2^21 - 1 ids, which the gather reads in chunks of 65536 (and
    three): short heads, a penalised window at the chunks' edges, and heads on
    either side of the 64 groups that are collected."""
    print("select largest", flush=True)
    rng = np.random.default_rng(33)
    V, rows = 2**21 - 1, 8
    x = rng.normal(0.0, 2.0, (rows, V)).astype(np.float32)
    edges = np.concatenate([np.arange(c * 65536 - 2, c * 65536 + 2) for c in range(1, 16)] + [[V - 4, V - 3, V - 2, V - 1]])
    x[:, edges] = rng.uniform(9.0, 14.0, (rows, edges.size))
    for r, n in ((4, 261000), (5, 263500)):   # 255 and 257 ids a bin, far above the others
        x[r] -= 3000.0
        x[r, rng.permutation(V)[:n]] = 20.0 - 2.0 ** rng.uniform(-8.0, 7.9, n)
    win = np.resize(edges, (rows, 64)).astype(np.uint32)
    st = [R.sampling(0.8, 100, 0.95, 0.0, 1.1, 64, 1), R.sampling(0.7, 0, 0.9, 0.0, 1.2, 64, 2),
          R.sampling(1.0, 0, 0.5, 0.0, 1.0, 0, 3), R.sampling(1.0, 65, 1.0, 0.0, 1.3, 64, 4),
          R.sampling(50.0, 261000, 0.999, 0.0, 1.0, 0, 5), R.sampling(50.0, 263500, 0.999, 0.0, 1.0, 0, 6),
          R.sampling(1.0, 4000, 0.99, 0.0, 1.1, 64, 7), R.sampling(1.0, 0, 0.3, 0.0, 0.9, 64, 8)]
    got, want = run_case(device, x, st, win, np.full(rows, 64, np.uint32), rng.random(rows).astype(np.float32), "own",
                         max_window=64)
    assert_rows_match("largest", got, want, st)


def test_many_rows_of_the_largest_vocabulary(device):
    """256 rows of 2^21 ids: the pass's largest chunks (two a row), whose window
    bitmap and bins take nearly all of a compute unit's LDS."""
    import torch
    import oracle as O
    from conftest import as_oracle_settings
    print("select many large rows", flush=True)
    rng = np.random.default_rng(34)
    V, rows = 2**21, 256
    x = rng.normal(0.0, 2.0, (2, V)).astype(np.float32)
    x[:, rng.permutation(V)[:64]] = rng.uniform(9.0, 14.0, (2, 64))
    win = rng.integers(0, V, (2, 64)).astype(np.uint32)
    win[:, :32] = np.argsort(x, axis=1)[:, -32:]
    wlen, u = np.full(2, 64, np.uint32), np.array([0.3, 0.9], np.float32)
    st = [R.sampling(0.8, 100, 0.95, 0.0, 1.1, 64, 1), R.sampling(0.7, 0, 0.9, 0.0, 1.2, 64, 2)]
    want = O.pick_rows(x, [as_oracle_settings(s) for s in st], win, wlen, u, cand_cap=100)
    ctx = R.DeviceSampler(rows, V, max_window=64)
    ctx.configure(st * (rows // 2))
    rep = lambda a: torch.from_numpy(a).to(device).repeat(rows // 2, *([1] * (a.ndim - 1)))
    tok = torch.zeros(rows, dtype=torch.int32, device=device)
    kept, used = torch.zeros_like(tok), torch.zeros(rows, dtype=torch.uint8, device=device)
    ctx.sample_rows(rep(x), rows, V, tok, kept, used, windows=rep(win.view(np.int32)), window_stride=64,
                    window_len=rep(wlen.view(np.int32)), uniforms=rep(u))
    torch.cuda.synchronize()
    for got, name in ((tok, "token"), (kept, "kept"), (used, "used")):
        assert np.array_equal(got.cpu().numpy().reshape(-1, 2).astype(np.int64),
                              np.repeat(want[name][None].astype(np.int64), rows // 2, axis=0)), name
    ctx.close()
