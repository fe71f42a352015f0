"""The whole-row walk of the top-p / min-p modes spread over the workgroups of the row's chunks
(geist_hip_sampler_set_whole_row_walk): the same tokens as the oracle's sorted walk
(sampler.c:246-304) in every mode of sending it -- always, never, and following the rows that
turn up --, with penalties, soft-cap and mask, on rows of equal values, and when the waits
between its steps run out and a row's first workgroup has to walk it alone."""
import numpy as np
import pytest

from gpu_util import compare_ids, crowded_rows, run_rows

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ADAPTIVE, SPREAD, ONE = 0, 1, 2


@pytest.fixture(scope="module")
def P():
    from geistlib_amd import SampleParams
    return SampleParams.make


def want_of(oracle, x, u, **kw):
    res = [oracle.chain_u(x[r], float(u[r]), **kw) for r in range(x.shape[0])]
    return [t for t, _ in res], [i for _, i in res]


@pytest.mark.parametrize("n", [128256, 50001, 20000, 8192, 151936])
def test_spread_walk_gives_the_oracles_tokens(oracle, P, n):
    from geistlib_amd import HipSampler
    print(f"spread walk n={n}", flush=True)
    g = np.random.default_rng(n)
    rows = 6
    hs = HipSampler(max_rows=8, max_vocab=n)
    try:
        hs.set_whole_row_walk(SPREAD)
        for kw in (dict(temperature=1.0, top_p=0.9), dict(temperature=0.8, top_p=0.95, min_p=1e-4),
                   dict(temperature=1.3, min_p=1e-5), dict(temperature=1.0, top_p=0.5)):
            x = crowded_rows(g, rows, n)
            u = g.random(rows).astype(np.float32)
            u[4] = 0.0
            u[5] = np.float32(1.0 - 2.0 ** -24)
            got = run_rows(hs, torch, x, u, P(**kw))
            paths = hs.row_paths(rows).tolist()
            want, infos = want_of(oracle, x, u, **kw)
            near = compare_ids(got, want, infos, f"spread walk n={n} {kw}")
            assert near <= 1
            # (short rows, whose crowd fits a list, and draws beside the crowd without a nucleus, need no
            # such walk)
            assert set(paths) <= {2, 4, 5}, (paths, kw)
            if n >= 50000 and "top_p" in kw:
                assert paths == [4] * rows, (paths, kw)
    finally:
        hs.close()


def test_spread_walk_with_penalties_cap_and_mask(oracle, P):
    from geistlib_amd import HipSampler
    n, rows = 70001, 5
    g = np.random.default_rng(7)
    x = crowded_rows(g, rows, n)
    u = g.random(rows).astype(np.float32)
    hist = g.integers(0, n, (rows, 300)).astype(np.int32)
    hlen = np.array([300, 0, 17, 300, 128], dtype=np.int32)
    allowed = g.random((rows, n)) < 0.8
    allowed[3] = True
    rep, freq, pres, cap = 1.3, 0.05, 0.1, 4.0
    hs = HipSampler(max_rows=8, max_vocab=n)
    try:
        hs.set_whole_row_walk(SPREAD)
        for lead, pad in ((0, 0), (1, 2)):
            for kw in (dict(temperature=1.0, top_p=0.9), dict(temperature=0.8, top_p=0.95, min_p=1e-4)):
                got = run_rows(hs, torch, x, u, P(rep=rep, freq=freq, pres=pres, softcap=cap, **kw),
                               history=hist, history_len=hlen, lead=lead, pad=pad, allowed=allowed)
                paths = hs.row_paths(rows).tolist()
                want, infos = [], []
                for r in range(rows):
                    row = oracle.penalties(x[r], hist[r, :hlen[r]], rep, freq, pres)
                    row = oracle.softcap(row, cap)
                    row[~allowed[r]] = -np.inf
                    t, i = oracle.chain_u(row, float(u[r]), **kw)
                    want.append(t)
                    infos.append(i)
                near = compare_ids(got, want, infos, f"spread walk, transforms, {kw} lead {lead}")
                assert near <= 1
                assert paths == [4] * rows, paths
    finally:
        hs.close()


def test_modes_agree_and_the_adaptive_one_follows_the_rows(oracle, P):
    """One workgroup, spread, adaptive: the same ids. In the adaptive mode the first call with
    such rows is served by one workgroup per row (path 3) and says so; the following calls are
    spread (path 4), until 64 calls in a row have had no such row. The other rows are served
    through the mass histogram (path 5) in all of them."""
    from geistlib_amd import HipSampler
    n, rows = 100000, 8
    g = np.random.default_rng(3)
    kw = dict(temperature=1.0, top_p=0.9, precedence=0)
    hs = HipSampler(max_rows=8, max_vocab=n)
    try:
        flat = [crowded_rows(g, rows, n) for _ in range(3)]
        peaked = (g.standard_normal((rows, n)) * 8).astype(np.float32)
        u = g.random(rows).astype(np.float32)
        ids = {}
        for mode in (ONE, SPREAD):
            hs.set_whole_row_walk(mode)
            ids[mode] = [run_rows(hs, torch, x, u, P(**kw)).tolist() for x in flat]
            assert hs.row_paths(rows).tolist() == [3 if mode == ONE else 4] * rows
        assert ids[ONE] == ids[SPREAD]
        for x, got in zip(flat, ids[SPREAD]):
            res = [oracle.top_p_u(x[r], 0.9, 1.0, float(u[r])) for r in range(rows)]
            assert compare_ids(np.array(got), [t for t, _ in res], [i for _, i in res], "modes") <= 1
        hs.set_whole_row_walk(ADAPTIVE)
        seen = []
        for x in [peaked] * 65 + [flat[0], flat[1], flat[2], peaked, flat[0]] + [peaked] * 65 + [flat[1], flat[2]]:
            got = run_rows(hs, torch, x, u, P(**kw)).tolist()
            seen.append(sorted(set(hs.row_paths(rows).tolist())))
            if x is not peaked:
                k = [i for i, f in enumerate(flat) if f is x][0]
                assert got == ids[ONE][k]
        # a call counts for the 64 that follow it
        assert seen == [[5]] * 65 + [[3], [4], [4], [5], [4]] + [[5]] * 65 + [[3], [4]], seen
    finally:
        hs.close()


def test_waits_that_run_out(oracle, P):
    """With a wait limit of zero no workgroup waits for a step's result: the workgroups that did
    not arrive last leave, the row's first one walks the row alone, and the following call (with
    the default limit again) finds its workspace cleared."""
    from geistlib_amd import HipSampler
    n, rows = 60000, 8
    g = np.random.default_rng(11)
    kw = dict(temperature=1.0, top_p=0.9)
    hs = HipSampler(max_rows=8, max_vocab=n)
    try:
        hs.set_whole_row_walk(SPREAD)
        x = crowded_rows(g, rows, n)
        u = g.random(rows).astype(np.float32)
        want, infos = want_of(oracle, x, u, **kw)
        hs.set_wait_limit(0)
        for _ in range(2):
            got = run_rows(hs, torch, x, u, P(**kw))
            assert compare_ids(got, want, infos, "no waiting") <= 1
            assert set(hs.row_paths(rows).tolist()) <= {3, 4}
        hs.set_wait_limit(65536)
        for _ in range(2):
            got = run_rows(hs, torch, x, u, P(**kw))
            assert compare_ids(got, want, infos, "after the waits that ran out") <= 1
            assert hs.row_paths(rows).tolist() == [4] * rows
    finally:
        hs.close()


def window_rows(g, rows, n):
    """Nuclei from a few entries to most of the row, and crowds where ranges of bins end or overflow."""
    x = (g.standard_normal((rows, n)) * g.choice([0.5, 1.5, 2.0, 3.0], (rows, 1))).astype(np.float32)
    x[1, : n // 2] = x[1].max() - 1.0 + 1e-3 * g.random(n // 2).astype(np.float32)  # one bin, over one chunk's stage
    x[2] = np.round(x[2] * 16) / 16                     # runs of equal values, a few hundred each
    x[3, 0], x[3, n - 1] = x[3].max() + 6.0, x[3].max() + 5.5   # first and last element lead
    return x


# 24 x 2047..50257: the plan found by the window pass itself; 96 rows: with a row-final kernel in front;
# 260 x 66000: several chunks to a workgroup
@pytest.mark.parametrize("rows,n", [(8, 2047), (8, 2048), (24, 2049), (5, 8193), (24, 50257), (96, 33001),
                                    (96, 32768), (260, 66000)])
@pytest.mark.parametrize("kw", [dict(top_p=0.95), dict(top_p=0.5, min_p=1e-3), dict(min_p=1e-4),
                                dict(top_p=0.999)])
def test_edge_and_draw_found_in_narrow_ranges(oracle, P, rows, n, kw):
    """The token of rows served through the histogram of the masses: every size at which the launch
    changes, draws at both ends, against the oracle's sorted walk. At most one row may lie within the
    contract's 1e-6 of a slot's edge. The rows without crowds are served there (path 5), or in larger
    batches by the shortcut or the min-p list in front; never by the whole-row walk."""
    from geistlib_amd import HipSampler
    print(f"window rows={rows} n={n} {kw}", flush=True)
    g = np.random.default_rng(rows * 100003 + n)
    base = window_rows(g, 6, n)
    x = np.ascontiguousarray(base[np.arange(rows) % 6])
    ub = g.random(6).astype(np.float32)
    ub[0], ub[5] = 0.0, np.float32(1.0 - 2.0 ** -24)
    u = ub[np.arange(rows) % 6]
    want, infos = want_of(oracle, base, ub, temperature=1.0, **kw)
    hs = HipSampler(max_rows=rows, max_vocab=n)
    try:
        for call in range(2):                           # (the second may spread its whole-row walks)
            got = run_rows(hs, torch, x, u, P(temperature=1.0, **kw))
            assert compare_ids(got[:6], want[:len(got[:6])], infos[:len(got[:6])], f"{rows}x{n} {kw}") <= 1
            assert all(got[r] == got[r % 6] for r in range(rows))
            small = rows * -(-n // 2048) <= 1024 and call == 0
            paths = hs.row_paths(rows).tolist()
            assert {paths[r] for r in range(rows) if r % 6 not in (1, 2)} <= ({5} if small else {1, 2, 5}), paths
    finally:
        hs.close()


def runs_of_equal_values(g, rows, n):
    """Rows whose edge or draw falls in a crowd of more entries than a workgroup has threads, all of it
    within the 16384 places of a row's list."""
    x = (g.standard_normal((rows, n)) * 2).astype(np.float32)
    top = x.max()
    x[0] = np.round(x[0] * 4) / 4                                         # quantised
    x[1, g.permutation(n)[:1000]] = top + 3                               # one value, all over the row
    x[2, n // 3 : n // 3 + 5000] = top + 2                                # one value, more than a workgroup's stage
    x[3] = np.round(x[3] * 8) / 8
    x[4, g.permutation(n)[:700]] = np.float32(top + 3) + np.float32(2.0 ** -20) * np.arange(700, dtype=np.float32)
    x[5, g.permutation(n)[:900]] = np.float32(top + 3) + np.float32(2.0 ** -20) * (np.arange(900) % 2).astype(np.float32)
    return x


@pytest.mark.parametrize("rows,n", [(8, 12000), (24, 50257), (96, 33001), (260, 66000)])
@pytest.mark.parametrize("kw", [dict(top_p=0.9), dict(top_p=0.5, min_p=1e-3), dict(top_p=0.03)])
def test_runs_of_equal_values_need_no_whole_row_walk(oracle, P, rows, n, kw):
    """Quantised logits, runs of one value and of neighbouring ones, at every form of the window's
    launch: the oracle's token, without a walk over the whole row."""
    from geistlib_amd import HipSampler
    print(f"equal values rows={rows} n={n} {kw}", flush=True)
    g = np.random.default_rng(rows + n)
    base = runs_of_equal_values(g, 6, n)
    x = np.ascontiguousarray(base[np.arange(rows) % 6])
    u = g.random(rows).astype(np.float32)
    u[0:2], u[2:4] = 0.0, np.float32(1.0 - 2.0 ** -24)
    check = min(rows, 36)
    want, infos = want_of(oracle, x[:check], u, temperature=1.0, **kw)
    hs = HipSampler(max_rows=rows, max_vocab=n)
    try:
        for _ in range(2):
            got = run_rows(hs, torch, x, u, P(temperature=1.0, **kw))
            assert compare_ids(got[:check], want, infos, f"{rows}x{n} {kw}") <= 1
            paths = hs.row_paths(rows).tolist()
            assert set(paths) <= ({5} if rows * -(-n // 2048) <= 1024 else {1, 2, 5}), paths
    finally:
        hs.close()


@pytest.mark.parametrize("rows,n", [(24, 50257), (260, 66001)])
def test_narrow_ranges_with_penalties_cap_and_mask(oracle, P, rows, n):
    """The window pass with everything it has to apply to the logits once more, in its small-batch form and
    with several chunks to a workgroup, whose history table is rebuilt from chunk to chunk; rows off a
    16-byte boundary, draws of their own for every row. Wide nuclei, so none is left to the shortcut."""
    from geistlib_amd import HipSampler
    print(f"window, transforms, rows={rows} n={n}", flush=True)
    g = np.random.default_rng(n)
    base = (g.standard_normal((5, n)) * 1.5).astype(np.float32)
    base[4] = np.round(base[4] * 4) / 4
    hist = g.integers(0, n, (rows, 400)).astype(np.int32)
    hist[:, 100:200] = base[np.arange(rows) % 5].argsort(axis=1)[:, -100:]   # the likeliest tokens among them
    hlen = g.integers(0, 401, rows).astype(np.int32)
    hlen[0], hlen[1] = 0, 400
    allowed = g.random((rows, n)) < 0.8
    allowed[3] = True
    x = np.ascontiguousarray(base[np.arange(rows) % 5])
    u = g.random(rows).astype(np.float32)
    rep, freq, pres, cap = 1.3, 0.05, 0.1, 6.0
    check = list(range(15)) + list(range(rows - 5, rows))
    hs = HipSampler(max_rows=rows, max_vocab=n)
    try:
        for lead, pad in ((0, 0), (1, 2)):
            for kw in (dict(temperature=1.0, top_p=0.9), dict(temperature=0.8, top_p=0.95, min_p=1e-4)):
                got = run_rows(hs, torch, x, u, P(rep=rep, freq=freq, pres=pres, softcap=cap, **kw),
                               history=hist, history_len=hlen, lead=lead, pad=pad, allowed=allowed)
                paths = hs.row_paths(rows).tolist()
                want, infos = [], []
                for r in check:
                    row = oracle.softcap(oracle.penalties(x[r], hist[r, :hlen[r]], rep, freq, pres), cap)
                    row[~allowed[r]] = -np.inf
                    t, i = oracle.chain_u(row, float(u[r]), **kw)
                    want.append(t)
                    infos.append(i)
                near = compare_ids(got[check], want, infos, f"window, transforms, {kw} lead {lead}")
                assert near <= 1
                assert set(paths) <= ({5} if rows < 100 or "min_p" not in kw else {2, 5}), paths
    finally:
        hs.close()


def test_flat_rows_of_a_large_vocabulary_need_no_whole_row_walk(oracle, P):
    """Ranges of some 9000 entries each around the middle of a flat row, with and without overlap."""
    from geistlib_amd import HipSampler
    rows, n = 6, 262144
    g = np.random.default_rng(5)
    x = (g.standard_normal((rows, n)) * 0.5).astype(np.float32)
    u = np.linspace(0.05, 0.95, rows).astype(np.float32)
    kw = dict(temperature=1.0, top_p=0.5)
    want, infos = want_of(oracle, x, u, **kw)
    for max_rows in (rows, 64):
        hs = HipSampler(max_rows=max_rows, max_vocab=n)
        try:
            got = run_rows(hs, torch, np.ascontiguousarray(x[np.arange(max_rows) % rows]),
                           u[np.arange(max_rows) % rows], P(**kw))
            assert compare_ids(got[:rows], want, infos, f"flat rows, {max_rows}") <= 1
            assert hs.row_paths(max_rows).tolist() == [5] * max_rows
        finally:
            hs.close()
