"""Temperature draws and min-p batches on either side of the sizes at which soft-caps, masks, penalties
and rows in eights send them another way: token ids against the oracle, and the same twice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from gpu_util import compare_ids, run_rows  # noqa: E402

TEMPERATURE = [(2, 180001, "cap"), (3, 172032, "cap"), (12, 262144, "cap"), (20, 188210, "cap pen"),
               (64, 32000, "cap"), (8, 262144, "mask"), (21, 131072, "mask"), (22, 131072, "mask"),
               (22, 131071, "mask pen"), (23, 131071, "mask pen"), (40, 65536, "mask"),
               (64, 32760, "mask"), (39, 65536, ""), (40, 65536, ""), (48, 64001, "pen")]
MIN_P = [(5, 165888, "pen"), (6, 149504, ""), (6, 151553, ""), (8, 151936, ""),      # 32768 and 46080 polls
         (24, 151552, "cap"), (24, 153600, "cap"), (24, 163840, "cap"), (24, 165889, "cap"),
         (16, 229376, "cap"), (16, 229377, "cap"), (56, 112640, "cap pen"), (32, 131072, "cap pen"),
         (32, 131073, "cap pen"), (48, 131072, "cap pen"), (51, 122880, "cap pen"), (51, 124928, "cap pen"),
         (50, 139264, "cap"), (50, 139265, "cap")]


@pytest.mark.parametrize("rows,n,form,options",
                         [(*c, dict(temperature=0.9)) for c in TEMPERATURE] +
                         [(*c, dict(temperature=0.9, top_p=0.95, min_p=0.05)) for c in MIN_P])
def test_ids_on_either_side_of_the_limits(oracle, rows, n, form, options):
    print(f"routes {rows} x {n} {form} {options}", flush=True)
    from geistlib_amd import HipSampler, SampleParams
    g = np.random.default_rng(rows + n)
    x = np.tile((g.standard_normal((4, n)) * 2).astype(np.float32), ((rows + 3) // 4, 1))[:rows]
    x[rows - 1, g.integers(0, n, 5)] += 6
    u = (g.integers(0, 1 << 24, rows) / np.float32(1 << 24)).astype(np.float32)
    pk, hist, hl, allowed = {}, None, None, None
    if "pen" in form:
        pk = dict(rep=1.2, freq=0.3, pres=0.1)
        hist = g.integers(0, n, (rows, 600)).astype(np.int32)
        hl = np.full(rows, 600, dtype=np.int32)
    if "cap" in form:
        pk["softcap"] = 20.0
    if "mask" in form:
        allowed = g.random((rows, n)) < 0.6
    s = HipSampler(max_rows=rows, max_vocab=n)
    got, again = (run_rows(s, torch, x, u, SampleParams.make(**options, **pk), hist, hl, allowed=allowed)
                  for _ in range(2))
    s.close()
    assert got.tolist() == again.tolist()
    check = sorted({0, 1, rows // 2, rows - 2, rows - 1})
    want = []
    for r in check:
        row = oracle.penalties(x[r], hist[r], 1.2, 0.3, 0.1) if "pen" in form else x[r]
        row = oracle.softcap(row, 20.0) if "cap" in form else row
        row = np.where(allowed[r], row, np.float32(-np.inf)) if "mask" in form else row
        want.append(oracle.chain_u(row, float(u[r]), **options))
    assert compare_ids([got[r] for r in check], [t for t, _ in want], [i for _, i in want], form) == 0
