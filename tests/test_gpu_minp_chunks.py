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


@pytest.mark.parametrize("rows", [6, 60])       # chunks of 2048, chunks of 8192
@pytest.mark.parametrize("form", ["plain", "pen", "cap"])
def test_min_p_candidates_crowded_into_one_run_of_2048_are_listed(oracle, rows, form):
    """Up to 2048 candidates among 2048 neighbouring ids are listed, whichever chunks the batch is cut
    into; twice 1500 among the same 8192 ids are walked in full, twice 1100 among different ones
    listed. Ids against the oracle, the rows' paths by the call's own account."""
    print(f"min-p crowded runs, {rows} rows, {form}", flush=True)
    from geistlib_amd import HipSampler, SampleParams
    n = 40000
    g = np.random.default_rng(53 + rows)
    x = (g.standard_normal((rows, n)) * 2).astype(np.float32)
    runs = [[(6144, 1025)], [(3000, 1500)], [(8192, 2048)], [(2048, 1100), (20480, 1100)],
            [(16384, 1500), (18432, 1500)], [(39000, 5)]]
    for r, row in enumerate(runs):              # (all others lie more than -log(min_p) below)
        top = x[r].max()
        for at, m in row:
            x[r, at:at + m] = top + 8 - 0.5 * g.random(m).astype(np.float32)
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    kw = dict(temperature=1.0, top_p=0.95, min_p=0.05)
    pk, hist, hl = {}, None, None
    if form == "pen":
        pk = dict(rep=1.2, freq=0.3, pres=0.1)
        hist = g.integers(0, n, (rows, 900)).astype(np.int32)
        hl = np.full(rows, 900, dtype=np.int32)
    elif form == "cap":
        pk = dict(softcap=20.0)
    s = HipSampler(max_rows=rows, max_vocab=n)
    for call in range(2):                       # (the second finds what the first left behind)
        got = run_rows(s, torch, x, u, SampleParams.make(**kw, **pk), hist, hl)
        paths = s.row_paths(rows)[:6].tolist()
        want = []
        for r in range(6):
            row = oracle.penalties(x[r], hist[r], 1.2, 0.3, 0.1) if form == "pen" else x[r]
            row = oracle.softcap(row, 20.0) if form == "cap" else row
            want.append(oracle.chain_u(row, float(u[r]), **kw))
        assert compare_ids(got[:6], [t for t, _ in want], [i for _, i in want], form) == 0
        assert paths[:4] == [2, 2, 2, 2] and paths[5] == 2, paths
        assert paths[4] in (3, 4), paths
    s.close()
