"""Sketch head with candidates crowded into few groups: whether the head has to decline is worked out on
the host from the rough scores, and wherever it does not, it answers as the oracle does."""
import numpy as np
import pytest

from test_gpu_spec_head import result_of, table

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hs():
    from geistlib_amd import HipSampler
    s = HipSampler(max_rows=1, max_vocab=66001)
    yield s
    s.close()


def ordered_keys(x):
    b = x.view(np.uint32)
    return np.where(b >> 31, ~b, b | np.uint32(0x80000000)).astype(np.uint32)


def listed(rough, topk):
    """Groups of 32 and rows that reach the topk-th largest group maximum, cut to 16 bits."""
    keys = ordered_keys(rough)
    padded = np.zeros((len(keys) + 31) // 32 * 32, dtype=np.uint32)
    padded[:len(keys)] = keys
    gmax = padded.reshape(-1, 32).max(1)
    bound = np.sort(gmax)[-topk] & np.uint32(0xffff0000)
    return int((gmax >= bound).sum()), int((keys >= bound).sum())


SHAPES = [(20000, 5120, 256), (66001, 1280, 1024), (8192, 1280, 16), (66000, 4096, 300)]


def crowded(vocab, d_model, topk, share):
    """A table with share x topk neighbouring rows along one direction, and activations along it by
    several strengths."""
    g = np.random.default_rng(vocab + topk)
    w16 = table(g, vocab, d_model)
    lean = (0.02 * g.standard_normal(d_model)).astype(np.float32)
    at = 32 * 7 + 5
    n = int(share * topk)
    w16[at:at + n] = (w16[at:at + n].astype(np.float32) + lean).astype(np.float16)
    return w16, [(s, (g.standard_normal(d_model) + s * lean).astype(np.float32))
                 for s in (5.0, 10.0, 20.0, 60.0)]


@pytest.mark.parametrize("vocab,d_model,topk", SHAPES)
@pytest.mark.parametrize("share", [0.5, 3])
def test_crowded_candidates_are_answered_unless_the_list_is_full(hs, oracle, vocab, d_model, topk, share):
    print(f"spec crowded vocab={vocab} d_model={d_model} topk={topk} share={share}", flush=True)
    w16, rows = crowded(vocab, d_model, topk, share)
    want_sh = oracle.spec_head_build(w16.view(np.uint16), topk=topk)
    sh = hs.spec_head_build(torch.from_numpy(w16.view(np.int16)).cuda(), topk=topk)
    res = torch.zeros(6, dtype=torch.int32, device="cuda")
    answered = 0
    for strength, h in rows:
        want = want_sh.try_row(h)
        groups, n = listed(want["rough"], topk)
        hs.spec_head_try(sh, torch.from_numpy(h).cuda(), res)
        hs.sync()
        got = result_of(res)
        full = groups > 2 * topk or n > 2 * topk
        assert bool(got.answered) == (not full), (strength, groups, n)
        assert got.n_listed == (groups if groups > 2 * topk else n), strength
        if full:
            assert got.token == -1
            continue
        answered += 1
        assert (got.token, got.cutoff, got.n_finalists) == (want["token"], want["cutoff"], topk)
    assert answered == 4 if share < 1 else answered < 4   # (the host counts agree, row by row)
    hs.spec_head_destroy(sh)
