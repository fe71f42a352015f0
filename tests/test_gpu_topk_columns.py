"""Top-k rows whose leaders share columns of the maxima: k_topk_wide's bound of up to 256 ranks is taken
from the largest maximum of each of 1024 threads, eight maxima apart, so with leaders at the same place
of every fourth chunk up to eight times the rank reach it. Token ids against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from gpu_util import compare_ids, run_rows  # noqa: E402


@pytest.mark.parametrize("k", [65, 150, 200, 256])
@pytest.mark.parametrize("pen", [False, True])
def test_leaders_in_shared_columns(oracle, k, pen):
    print(f"columns k={k} pen={pen}", flush=True)
    from geistlib_amd import HipSampler, SampleParams
    n, rows = 262144, 4
    g = np.random.default_rng(k + pen)
    x = (g.standard_normal((rows, n)) * 2).astype(np.float32)
    chunks = np.arange(2, 32, 4) * 8192                       # eight chunks, four apart
    place = 4 * g.permutation(256)                            # of 4 j 256 + 4 thread + component
    one = (chunks[:, None] + place[None, :k]).ravel()         # a leader to each maximum: 8 k of them
    x[0, one] = 12 + g.random(one.size).astype(np.float32)
    few = (chunks[:, None] + place[None, :k // 4]).ravel()    # ... twice the rank
    x[1, few] = 12 + g.random(few.size).astype(np.float32)
    every = (few[:, None, None] + 1024 * np.arange(8)[None, :, None] + np.arange(4)).ravel()
    x[2, every] = 12 + g.random(every.size).astype(np.float32)   # all 32 of each: beyond the list
    x[3, one] = 12.5                                          # ... and all equal
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    kw = dict(temperature=0.9, top_k=k, top_p=0.97)
    pk, hist, hl = {}, None, None
    if pen:
        pk = dict(rep=1.2, freq=0.3, pres=0.1)
        hist = np.concatenate([g.permutation(one)[:60][None].repeat(rows, 0),
                               g.integers(0, n, (rows, 200))], 1).astype(np.int32)
        hl = np.full(rows, hist.shape[1], dtype=np.int32)
    s = HipSampler(max_rows=rows, max_vocab=n)
    got = run_rows(s, torch, x, u, SampleParams.make(**kw, **pk), hist, hl)
    s.close()
    want = [oracle.chain_u(oracle.penalties(x[r], hist[r], 1.2, 0.3, 0.1) if pen else x[r], float(u[r]), **kw)
            for r in range(rows)]
    assert compare_ids(got, [t for t, _ in want], [i for _, i in want], f"columns k={k}") <= 1


@pytest.mark.parametrize("rows,n,first", [(128, 131072, 0), (255, 131072, 0), (256, 131072, 1),
                                          (127, 131076, 0), (128, 131076, 1)])
@pytest.mark.parametrize("pen", [False, True])
def test_the_first_path_follows_from_the_batch(rows, n, first, pen):
    """Candidates handed on by the scan (0) or the thread maxima (1): the same ids either way, those of
    the rows in calls of a few."""
    print(f"first path {rows} x {n} pen={pen}", flush=True)
    from geistlib_amd import HipSampler, SampleParams
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + n + pen)
    x = torch.randn((rows, n), device="cuda", generator=gen) * 2
    hist = torch.randint(0, n, (rows, 300), device="cuda", generator=gen, dtype=torch.int32)
    hl = torch.full((rows,), 300, device="cuda", dtype=torch.int32)
    u = torch.rand((rows,), device="cuda", generator=gen)
    prm = SampleParams.make(temperature=0.7, top_k=40, top_p=0.9, **(dict(rep=1.1, freq=0.5, pres=0.3) if pen else {}))
    out, few = (torch.full((rows,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
    s = HipSampler(max_rows=rows, max_vocab=n)
    s.one_launch_topk(False)
    s.sample(HipSampler.rows(x, hist, hl), prm, u, out)
    paths = s.topk_paths(rows).tolist()
    for at in range(0, rows, 16):
        to = slice(at, at + 16)
        s.sample(HipSampler.rows(x[to], hist[to], hl[to]), prm, u[to].contiguous(), few[to])
    s.sync()
    s.close()
    assert out.tolist() == few.tolist()
    assert paths.count(first) > rows // 2, paths    # (a few leave it: their leaders crowd)
