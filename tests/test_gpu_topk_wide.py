"""Top-k for a k of hundreds (k_tmax_scan, then k_topk_wide) against the oracle: token ids bit for
bit, at the edges of its lists and ranks, on ragged, masked, penalised and soft-capped rows and on the
rows it has to hand to the whole-row selection."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpu_util import compare_ids, run_rows  # noqa: E402


@pytest.fixture(scope="module")
def hs():
    from geistlib_amd import HipSampler
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a device; the sampling path has no CPU fallback")
    s = HipSampler(max_rows=16, max_vocab=262144)
    yield s
    s.close()


def rows_of(g, n):
    """Ordinary rows and, from row 4 on, what the bound does not fit: sorted, runs of equal values,
    all equal, fewer finite logits than k, leaders in one thread's elements, NaN and infinities."""
    x = (g.standard_normal((14, n)) * 2).astype(np.float32)
    x[1] = (g.standard_t(3, n) * 2.5).astype(np.float32)
    x[2, g.integers(0, n, 5)] += 10
    x[3] -= 40                                   # all negative
    x[4] = -np.sort(-x[4])
    x[5] = np.round(x[5] * 2) / 2
    x[6] = 0.5
    x[7] = -np.inf
    x[7, g.integers(0, n, 40)] = g.standard_normal(40).astype(np.float32)
    at = min(n, 4096) // 2
    x[8, at:at + 700] += 20
    x[9, ::3] = np.nan
    x[10, :3] = [np.inf, 1e30, -np.inf]
    x[11, n - 200:] = 30.0
    x[12] = np.round(x[12] * 64) / 64
    x[13, : n // 2] = x[13, 0]
    return x


@pytest.mark.parametrize("n,k", [(32000, 129), (32001, 300), (50257, 65), (65536, 1024), (65535, 1000),
                                 (128256, 200), (262144, 256), (262143, 257), (8192 * 17, 1025),
                                 (20000, 313), (16383, 56)])
@pytest.mark.parametrize("form", ["plain", "pen", "mask", "cap", "all"])
def test_top_k_of_hundreds_matches_oracle(hs, oracle, n, k, form):
    print(f"wide n={n} k={k} {form}", flush=True)
    from geistlib_amd import SampleParams
    g = np.random.default_rng(n + k)
    x = rows_of(g, n)
    rows = x.shape[0]
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    pen, cap, mask = form in ("pen", "all"), form in ("cap", "all"), form in ("mask", "all")
    kw = dict(temperature=0.9, top_k=k, top_p=0.97)
    pk, hist, hl, allowed = {}, None, None, None
    if pen:
        pk = dict(rep=1.2, freq=0.3, pres=0.1)
        hist = g.integers(0, n, (rows, 3000)).astype(np.int32)
        hist[:, : k // 3] = np.argsort(-np.nan_to_num(x), axis=1)[:, : k // 3]
        hist[0, :3] = [-1, n, int(np.argmax(x[0]))]
        hl = np.full(rows, 3000, dtype=np.int32)
        hl[1], hl[2] = 0, 2500
    if cap:
        pk["softcap"] = 20.0
    if mask:
        allowed = g.random((rows, n)) < 0.6
        allowed[7] = True
    got = run_rows(hs, torch, x, u, SampleParams.make(**kw, **pk), hist, hl, allowed=allowed,
                   lead=1 if n % 2 else 0)
    want, infos = [], []
    for r in range(rows):
        row = x[r]
        if pen:
            row = oracle.penalties(row, hist[r, : hl[r]], 1.2, 0.3, 0.1)
        if cap:
            row = oracle.softcap(row, 20.0)
        if mask:
            row = np.where(allowed[r], row, np.float32(-np.inf))
        t, i = oracle.chain_u(row, float(u[r]), **kw)
        want.append(t)
        infos.append(i)
    assert compare_ids(got, want, infos, f"wide n={n} k={k} {form}") <= 1


@pytest.mark.parametrize("k", [2, 40, 64])
@pytest.mark.parametrize("pen", [False, True])
def test_large_batches_select_from_the_thread_maxima(oracle, k, pen):
    """From 2^24 logits on, plain rows of any k: the call says that the thread maxima served it."""
    from geistlib_amd import HipSampler, SampleParams
    n, rows = 262144, 64
    g = np.random.default_rng(k + pen)
    x = np.tile((g.standard_normal((16, n)) * 2).astype(np.float32), (4, 1))
    x[1] = -np.sort(-x[1])
    x[2] = np.round(x[2])
    x[3] = 1.5
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    kw = dict(temperature=0.7, top_k=k, top_p=0.9)
    hist = g.integers(0, n, (rows, 700)).astype(np.int32)
    hist[:, :20] = np.argsort(-x[5])[:20]
    hl = np.full(rows, 700, dtype=np.int32)
    s = HipSampler(max_rows=rows, max_vocab=n)
    s.one_launch_topk(False)
    got = run_rows(s, torch, x, u, SampleParams.make(**kw, **(dict(rep=1.1, freq=0.5, pres=0.2) if pen else {})),
                   hist if pen else None, hl if pen else None)
    paths = s.topk_paths(rows).tolist()
    s.close()
    check = list(range(0, 20)) + [rows - 1]
    want = [oracle.chain_u(oracle.penalties(x[r], hist[r], 1.1, 0.5, 0.2) if pen else x[r], float(u[r]), **kw)
            for r in check]
    compare_ids([got[r] for r in check], [t for t, _ in want], [i for _, i in want], f"large k={k} {pen}")
    assert set(paths) <= {1, 2} and paths.count(1) >= rows - 8, paths
