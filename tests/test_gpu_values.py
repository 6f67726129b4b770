"""The value path on the GPU (nearly flat min-p rows on the bf16 grid, no
candidates taken) against the oracle: tokens and kept counts of rows with ties,
with no ties, of one value, with zeros and ruled-out ids, whose sums are exact
and not, with penalised ids off the grid, and of the rows it leaves to the
whole-row sort; the smallest and largest vocabularies; uniforms over the whole
draw."""
import numpy as np
import pytest

import oracle as O
import rl_sampler as R
from conftest import as_oracle_settings

pytestmark = pytest.mark.gpu

KINDS = ["ties", "grid", "one", "two", "zeros", "masked", "wide", "mixed", "small", "specials"]


def to_grid(x):
    return (x.astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)


def logits_of(kind, rng, rows, V):
    x = rng.normal(0.0, 0.01, (rows, V))
    if kind == "wide":         # p far apart: sums that are not exact
        x = rng.normal(0.0, 1.5, (rows, V))
    elif kind == "one":
        x[:, :] = -0.75
    elif kind == "two":
        x = np.where(rng.random((rows, V)) < 0.5, 1.0, 1.0078125)
    x = to_grid(x)
    if kind in ("ties", "masked"):
        x[rng.random((rows, V)) < 0.4] = -0.0234375
    if kind == "zeros":
        x[rng.random((rows, V)) < 0.3] = 0.0
        x[rng.random((rows, V)) < 0.3] = -0.0
    if kind == "masked":       # past the sample: ids ruled out
        x[:, 300:][rng.random((rows, V - 300)) < 0.5] = -np.inf
    if kind == "mixed":        # elements off the grid past the sample, a few to too many
        for r in range(rows):
            n = [1, 63, 64, 65, 500, 1024, 1025, V - 300][r % 8]
            at = 300 + rng.permutation(V - 300)[:n]
            x[r, at] = rng.normal(0.0, 0.01, n).astype(np.float32)
    if kind == "small":        # magnitudes below the window
        x[:, 300::50] *= np.float32(2.0 ** -30)
    if kind == "specials":
        x[0, V - 1] = np.nan
        x[1, V - 2] = np.inf
        x[2, 5] = -np.nan
        x[3, 7] = np.inf
        x[4, V // 2] = 3e30
        x[5, 0] = -np.inf
    return x


SETTINGS = [
    R.sampling(1.0, 0, 0.99, 0.02, 1.0, 0, 1),
    R.sampling(1.0, 0, 0.99, 0.02, 1.1, 64, 2),
    R.sampling(0.7, 0, 0.5, 0.05, 1.3, 64, 3),
    R.sampling(2.0, 0, 0.999, 1e-7, 0.8, 64, 4),
    R.sampling(1.0, 0, 0.0, 0.02, 1.0, 0, 5),
    R.sampling(1.0, 0, 0.9999999, 1e-7, 1.1, 64, 6),
    R.sampling(1.0, 0, 0.95, 0.9995, 1.0, 0, 7),
    R.sampling(0.9, 0, 0.9, 1e-7, 1.0, 0, 8),
]


def sample(ctx, device, x, win, wlen, u, stride=None):
    import torch
    rows, V = x.shape
    stride = V if stride is None else stride
    buf = np.zeros((rows, stride), np.float32)
    buf[:, :V] = x
    tok = torch.zeros(rows, dtype=torch.int32, device=device)
    kept, used = torch.zeros_like(tok), torch.zeros(rows, dtype=torch.uint8, device=device)
    ctx.sample_rows(torch.from_numpy(buf.reshape(-1)).to(device), rows, stride, tok, kept, used,
                    windows=torch.from_numpy(win.view(np.int32)).to(device), window_stride=win.shape[1],
                    window_len=torch.from_numpy(wlen.view(np.int32)).to(device),
                    uniforms=torch.from_numpy(u).to(device))
    torch.cuda.synchronize()
    return tok.cpu().numpy().view(np.uint32), kept.cpu().numpy().view(np.uint32), used.cpu().numpy()


def check(ctx, device, label, x, settings, win, wlen, u, stride=None):
    ctx.configure(settings)
    got = sample(ctx, device, x, win, wlen, u, stride)
    want = O.pick_rows(x, [as_oracle_settings(s) for s in settings], win, wlen, u, cand_cap=x.shape[1])
    for i, name in enumerate(("token", "kept", "used")):
        bad = np.nonzero(got[i] != want[name])[0]
        assert bad.size == 0, (label, name, bad, [settings[r] for r in bad[:3]], got[i][bad[:3]], want[name][bad[:3]])


@pytest.mark.parametrize("V", [4096, 4099, 50004])
@pytest.mark.parametrize("kind", KINDS)
def test_rows_match_the_oracle(device, kind, V):
    print("values", kind, V, flush=True)
    rng = np.random.default_rng([ord(c) for c in kind] + [V])
    rows = len(SETTINGS)
    x = logits_of(kind, rng, rows, V)
    ctx = R.DeviceSampler(rows, V, max_window=64)
    win = rng.integers(0, V + 5, (rows, 64)).astype(np.uint32)
    win[:, :8] = win[:, 8:16]  # repeated ids
    wlen = np.full(rows, 64, np.uint32)
    wlen[-1] = 0
    for u in ([0.0, 2.0 ** -24, 0.25, 0.5], [0.75, 0.999, 1.0 - 2.0 ** -24, 0.1], rng.random(4)):
        check(ctx, device, kind, x, SETTINGS, win, wlen, np.resize(u, rows).astype(np.float32))


@pytest.mark.parametrize("V,rows,wl", [(262144, 1, 64), (151936, 2, 2048), (151935, 3, 500), (32000, 70, 64)])
def test_sizes(device, V, rows, wl):
    print("values size", V, rows, wl, flush=True)
    rng = np.random.default_rng(V + rows)
    x = logits_of("ties", rng, rows, V)
    settings = [SETTINGS[r % 4] for r in range(rows)]
    settings = [R.sampling(s.temperature, 0, s.top_p, s.min_p, s.repeat_penalty, wl if s.repeat_last_n else 0, r)
                for r, s in enumerate(settings)]
    ctx = R.DeviceSampler(rows, V, max_window=wl)
    win = rng.integers(0, V, (rows, wl)).astype(np.uint32)
    for stride in (V, -(-V // 64) * 64):
        check(ctx, device, "size", x, settings, win, np.full(rows, wl, np.uint32),
              rng.random(rows).astype(np.float32), stride)


def test_the_draw_at_every_part_of_the_row(device):
    """One row, 256 uniforms: the occurrence drawn within its value's run."""
    print("values draw", flush=True)
    rng = np.random.default_rng(5)
    V, rows = 32003, 256
    x = np.repeat(logits_of("ties", rng, 1, V), rows, axis=0)
    ctx = R.DeviceSampler(rows, V, max_window=64)
    win = np.repeat(rng.integers(0, V, (1, 64)).astype(np.uint32), rows, axis=0)
    u = ((np.arange(rows) + rng.random(rows)) / rows).astype(np.float32)
    u[:40] = (2.0 ** -rng.uniform(1, 16, 40)).astype(np.float32)
    check(ctx, device, "draw", x, [SETTINGS[1]] * rows, win, np.full(rows, 64, np.uint32), u)


def test_samples_that_mislead(device):
    """The rule looks at 64 ids, eight at each of eight places: rows flat there
    and peaked elsewhere, peaked there and flat elsewhere, ruled out there, tied
    there, and with few to too many ids off the grid elsewhere."""
    print("values misled", flush=True)
    rng = np.random.default_rng(12)
    V, rows = 20004, 13
    at = ((np.arange(64) // 8) * (V // 8) + V // 16 + (np.arange(64) & 7))
    x = logits_of("ties", rng, rows, V)
    x[0] = to_grid(rng.normal(0.0, 3.0, V))
    x[1] = rng.normal(0.0, 3.0, V).astype(np.float32)
    x[2] = rng.normal(0.0, 0.01, V).astype(np.float32)
    x[:3, at] = -0.0234375
    x[3, at] = to_grid(rng.normal(0.0, 3.0, 64))
    x[4, at] = -np.inf
    x[5, at[3:]] = -np.inf
    x[6, at[8:]] = -np.inf
    x[7, at] = -3.0
    others = np.setdiff1d(np.arange(V), at)
    for r, n in enumerate((500, 1023, 1024, 1025, V // 2)):
        x[8 + r, rng.permutation(others)[:n]] = rng.normal(0.0, 0.01, n).astype(np.float32)
    ctx = R.DeviceSampler(rows, V, max_window=64)
    win = rng.integers(0, V, (rows, 64)).astype(np.uint32)
    for st in SETTINGS[:3]:
        check(ctx, device, "misled", x, [st] * rows, win, np.full(rows, 64, np.uint32),
              rng.random(rows).astype(np.float32))


def test_beside_other_paths(device):
    """Value rows, min-p rows, selection rows and stream rows in one call, twice."""
    print("values mixed", flush=True)
    rng = np.random.default_rng(9)
    V, rows = 20004, 40
    x = logits_of("ties", rng, rows, V)
    settings = [SETTINGS[r % len(SETTINGS)] for r in range(rows)]
    for r in range(0, rows, 3):
        x[r] = rng.normal(0.0, 3.0, V)
        settings[r] = [R.sampling(1.0, 0, 0.9, 0.05, 1.0, 0, r), R.sampling(0.8, 100, 0.95, 0.0, 1.1, 64, r),
                       R.sampling(0.6, 20, 0.95, 0.0, 1.0, 0, r)][r // 3 % 3]
    ctx = R.DeviceSampler(rows, V, max_window=64)
    win = rng.integers(0, V, (rows, 64)).astype(np.uint32)
    for _ in range(2):
        check(ctx, device, "mixed", x, settings, win, np.full(rows, 64, np.uint32), rng.random(rows).astype(np.float32))


@pytest.mark.parametrize("V", [2096800, 2096895, 2096900, 2**21])
def test_chunk_counts_at_their_limit(device, V):
    """One row in 32 chunks: counts of up to 65531 equal values a chunk, two a
    word, below 2096896 ids, and the sort above; the value that fills the chunks
    is the one counted in registers, and is not."""
    print("values limit", V, flush=True)
    rng = np.random.default_rng(V)
    at = ((np.arange(64) // 8) * (V // 8) + V // 16 + (np.arange(64) & 7))
    win = rng.integers(0, V, (1, 64)).astype(np.uint32)
    ctx = R.DeviceSampler(1, V, max_window=64)
    for sampled, step in ((0.5, 64), (0.50390625, 1 << 20)):
        x = np.full((1, V), 0.5, np.float32)
        x[0, ::step] = 0.498046875
        x[0, at] = sampled
        for u in (0.001, 0.5, 0.999):
            check(ctx, device, "limit", x, [SETTINGS[1]], win, np.full(1, 64, np.uint32), np.array([u], np.float32))
