"""Min-p of a few percent: the exp-sum pass lists the rows in chunks of 2048 (small batches) or 8192, and
rows whose list overflows are walked in full. Token ids against the oracle on either side of the
limits, with penalties, soft-cap and mask."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from gpu_util import compare_ids, run_rows  # noqa: E402


@pytest.mark.parametrize("rows,n", [(1, 2047), (3, 2049), (2, 50257), (4, 130000), (11, 131072), (11, 131073), (34, 65536), (34, 65537),
                                    (10, 262144)])
@pytest.mark.parametrize("form", ["plain", "pen", "cap", "all"])
def test_min_p_batches_in_either_chunks(oracle, rows, n, form):
    print(f"min-p {rows} x {n} {form}", flush=True)
    from geistlib_amd import HipSampler, SampleParams
    g = np.random.default_rng(rows + n)
    x = (g.standard_normal((rows, n)) * 2).astype(np.float32)
    x[rows - 1] = 0.25                                   # every element listed: beyond the list from 16384 on
    x[0, g.integers(0, n, 5)] += 10
    if rows > 2:
        x[1] = np.round(x[1] * 4) / 4
        x[2, ::3] = -np.inf
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    pen, cap, mask = form in ("pen", "all"), form in ("cap", "all"), form == "all"
    kw = dict(temperature=0.9, top_p=0.9, min_p=0.04)
    pk, hist, hl, allowed = {}, None, None, None
    if pen:
        pk = dict(rep=1.2, freq=0.3, pres=0.1)
        hist = g.integers(0, n, (rows, 900)).astype(np.int32)
        hl = np.full(rows, 900, dtype=np.int32)
    if cap:
        pk["softcap"] = 20.0
    if mask:
        allowed = g.random((rows, n)) < 0.6
    s = HipSampler(max_rows=rows, max_vocab=n)
    got = run_rows(s, torch, x, u, SampleParams.make(**kw, **pk), hist, hl, allowed=allowed)
    s.close()
    check = sorted(set(list(range(min(rows, 4))) + [rows - 2, rows - 1]) & set(range(rows)))
    want = []
    for r in check:
        row = oracle.penalties(x[r], hist[r], 1.2, 0.3, 0.1) if pen else x[r]
        row = oracle.softcap(row, 20.0) if cap else row
        row = np.where(allowed[r], row, np.float32(-np.inf)) if mask else row
        want.append(oracle.chain_u(row, float(u[r]), **kw))
    assert compare_ids([got[r] for r in check], [t for t, _ in want], [i for _, i in want], form) <= 1
