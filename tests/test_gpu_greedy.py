"""Argmax in one launch (k_greedy): the workgroup of a row's last chunk collects what the others
report. Ids equal the reference's (first index of the greatest value, a NaN at index 0 stays),
whether it waits for them or, with a wait limit of 0 polls, reads the row for itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from gpu_util import run_rows  # noqa: E402

# (rows, n): one chunk, a chunk and one element, chunks of 2048 and of 8192, rows in eights (one
# XCD each) and not, the edge of two chunk sizes (rows * ceil(n / 8192) = 512)
SIZES = [(1, 1), (1, 2048), (3, 2049), (8, 128256), (7, 50257), (2, 262144), (63, 65536), (64, 65536),
         (130, 40001)]


@pytest.mark.parametrize("form", ["plain", "penalties", "mask", "unaligned"])
@pytest.mark.parametrize("rows,n", SIZES)
def test_argmax_of_every_shape(oracle, rows, n, form):
    from geistlib_amd import HipSampler, SampleParams
    print(f"greedy rows={rows} n={n} {form}", flush=True)
    g = np.random.default_rng(rows * 13 + n)
    # few distinct values: the greatest is there many times and the first of them counts
    x = (np.round(g.standard_normal((rows, n)) * 4) / 4).astype(np.float32)
    x[rows // 2] = -np.inf
    if rows > 2:
        x[1, 0] = np.nan
        x[2] = np.nan
        x[2, n // 2] = -5.0
    if rows > 3:
        x[3] = 0.0
        x[3, : n // 2] = -0.0
    hist = hl = allowed = None
    kw = {}
    seen = x
    if form == "penalties":
        hist = g.integers(0, n, (rows, 257)).astype(np.int32)
        hl = np.full(rows, 257, dtype=np.int32)
        hl[0] = 0
        kw = dict(rep=1.3, freq=0.4, pres=0.2)
        seen = np.stack([oracle.penalties(x[r], hist[r, :hl[r]], 1.3, 0.4, 0.2) for r in range(rows)])
    if form == "mask":
        allowed = g.random((rows, n)) < 0.5
        allowed[:, 0] = True
        seen = np.where(allowed, x, -np.inf).astype(np.float32)
    want = [oracle.argmax(np.ascontiguousarray(seen[r])) for r in range(rows)]
    layout = dict(pad=3, lead=1) if form == "unaligned" else {}
    s = HipSampler(max_rows=rows, max_vocab=max(n, 16))
    try:
        for limit in (None, 0, None):
            s.set_wait_limit(65536 if limit is None else limit)
            got = run_rows(s, torch, x, None, SampleParams.make(temperature=0.0, **kw), history=hist,
                           history_len=hl, allowed=allowed, **layout)
            assert got.tolist() == want, limit
    finally:
        s.close()


@pytest.mark.parametrize("static", [False, True])
def test_recorded_argmax_replays(oracle, static):
    from test_gpu_graph_replay import test_recorded_call_replays
    test_recorded_call_replays(oracle, static, 16, 50000, dict(temperature=0.0))
