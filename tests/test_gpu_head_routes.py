"""Q4_K and Q6_K tables on either side of the sizes at which another kernel takes them: each table row's
logit is its own, so parts of a table, small enough for the general route, give the same bits as the
whole; and the batches of tables too large for slices, over several blocks, those of the kernel that
reads the table as it lies in the file."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BYTES = {"q4k": 144, "q6k": 210}


@pytest.fixture(scope="module")
def hs():
    from geistlib_amd import HipSampler
    s = HipSampler(max_rows=16, max_vocab=262144)
    yield s
    s.close()


def table(kind, n_out, n_in, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    t = torch.randint(0, 256, (n_out * (n_in // 256), BYTES[kind]), device="cuda", generator=gen,
                      dtype=torch.uint8)
    scales = slice(208, 210) if kind == "q6k" else slice(0, 4)
    t[:, scales] = torch.tensor([0x6D, 0x0C] * ((scales.stop - scales.start) // 2), dtype=torch.uint8,
                                device="cuda")
    return t.view(n_out, -1)


def logits(hs, kind, w, n_in, x):
    """Of the packed copy: one row by the decode kernel, several by the batch's."""
    n_out, m = w.shape[0], x.shape[0]
    size, pack = ((hs.q6k_packed_bytes, hs.q6k_pack) if kind == "q6k" else
                  (hs.q4k_packed_bytes, hs.q4k_pack))
    packed = torch.zeros((size(n_out, n_in),), dtype=torch.uint8, device="cuda")
    pack(w, n_in, packed)
    y = torch.full((m + 1, n_out), 7.0, dtype=torch.float32, device="cuda")
    if m > 1:
        (hs.q6k_packed_linear_x86 if kind == "q6k" else hs.q4k_packed_linear_x86)(
            packed, n_out, n_in, x, y[:m])
    else:
        (hs.q6k_packed_gemv_x86 if kind == "q6k" else hs.q4k_packed_gemv_x86)(
            packed, n_out, n_in, x, y[:m])
    hs.sync()
    assert (y[m] == 7.0).all()                   # nothing beyond the batch
    return y[:m].view(torch.int32)


@pytest.mark.parametrize("kind,m,blocks,groups", [
    ("q4k", 1, 21, 1800), ("q4k", 1, 22, 1792), ("q4k", 1, 22, 1793), ("q4k", 1, 27, 1860),
    ("q4k", 1, 27, 1861), ("q4k", 1, 28, 1536), ("q4k", 1, 28, 1537), ("q4k", 1, 28, 1664),
    ("q4k", 1, 28, 1665), ("q4k", 1, 33, 1888), ("q4k", 1, 33, 1889),
    ("q4k", 3, 23, 800), ("q4k", 3, 24, 768), ("q4k", 3, 24, 769), ("q4k", 3, 32, 1024),
    ("q4k", 3, 24, 1025),
    ("q6k", 1, 16, 1810), ("q6k", 1, 17, 1804), ("q6k", 1, 17, 1805), ("q6k", 1, 31, 1872),
    ("q6k", 1, 32, 1792), ("q6k", 1, 32, 1793), ("q6k", 1, 33, 1873),
])
@pytest.mark.parametrize("ragged", [0, 24, 56])
def test_parts_of_a_table_give_the_bits_of_the_whole(hs, kind, m, blocks, groups, ragged):
    print(f"{kind} {m} rows, {groups} groups - {ragged}, {blocks} blocks", flush=True)
    n_out, n_in = groups * 64 - ragged, blocks * 256
    w = table(kind, n_out, n_in, groups + blocks)
    g = np.random.default_rng(blocks)
    x = torch.from_numpy((g.standard_normal((m, n_in)) * 2).astype(np.float32)).cuda()
    whole = logits(hs, kind, w, n_in, x)
    part = 400 * 64
    for at in range(0, n_out, part):
        few = logits(hs, kind, w[at:at + part].contiguous(), n_in, x)
        assert torch.equal(few, whole[:, at:at + part]), at


@pytest.mark.parametrize("n_in", [512, 1536])
@pytest.mark.parametrize("groups", [2049, 3001, 4097])
@pytest.mark.parametrize("ragged", [0, 5])
def test_q6k_batches_too_large_for_slices(hs, groups, n_in, ragged):
    print(f"q6k batches, {groups} groups - {ragged}, {n_in}", flush=True)
    n_out = groups * 64 - ragged
    w = table("q6k", n_out, n_in, groups + n_in)
    g = np.random.default_rng(groups)
    for m in range(2, 9):
        x = torch.from_numpy((g.standard_normal((m, n_in)) * 3).astype(np.float32)).cuda()
        file = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
        hs.q6k_linear_x86(w, n_in, x, file)
        assert torch.equal(logits(hs, "q6k", w, n_in, x), file.view(torch.int32)), m
