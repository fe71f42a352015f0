"""The output head in front of the sampler on the device -- RMS norm and the tied F16 lm_head
(src/archs/transformer/forward/head.c:94-129 of the reference) -- through the C ABI against the
oracle, which is itself pinned bit for bit to the reference's compiled kernel
(tests/test_lm_head_oracle.py). Every float must agree in every bit."""
import numpy as np
import pytest

from gpu_util import fuzz_seeds, to_dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hs():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from geistlib_amd import HipSampler
    s = HipSampler(max_rows=32, max_vocab=40000)
    yield s
    s.close()


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def call_us(call, calls):
    """Microseconds of a call among others, the least of three runs."""
    call()
    best = float("inf")
    for _ in range(3):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(calls):
            call()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / calls)
    return best


def run_gemv(hs, w16, x):
    d_w = to_dev(w16.view(np.int16), torch)
    d_x = to_dev(x, torch)
    y = torch.full((x.shape[0], w16.shape[0]), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_gemv(d_w, d_x, y)
    hs.sync()
    return y.cpu().numpy()


@pytest.mark.parametrize("n_out,n_in,m", [(1000, 2560, 1), (130, 64, 1), (129, 128, 3),
                                          (4097, 1536, 2), (300, 8, 1), (300, 16, 5), (257, 24, 4),
                                          (31, 2568, 8), (640, 4096, 16), (500, 2560, 17),
                                          (50, 72, 16), (33, 40, 9), (1, 2560, 1)])
def test_f16_gemv_rows_bit_exact(hs, oracle, n_out, n_in, m):
    print(f"gemv n_out={n_out} n_in={n_in} m={m}", flush=True)
    g = np.random.default_rng(n_out * 7 + n_in + m)
    w16 = (g.standard_normal((n_out, n_in)) * g.choice([0.02, 1.0])).astype(np.float16).view(np.uint16)
    x = (g.standard_normal((m, n_in)) * g.choice([0.1, 1.0, 30.0], (m, 1))).astype(np.float32)
    got = run_gemv(hs, w16, x)
    want = oracle.f16_gemv(w16, x)
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


def test_f16_gemv_special_values(hs, oracle):
    """Subnormal and extreme binary16 weights, zeros of both signs, a row of zeros with negative
    activations (the sign of a zero result is part of the result)."""
    n_out, n_in = 64, 96
    g = np.random.default_rng(3)
    w = g.standard_normal((n_out, n_in)).astype(np.float16)
    w[0, :] = 0.0
    w[1, :] = -0.0
    w[2, :] = np.float16(6e-8)                     # smallest subnormals
    w[3, :] = np.float16(65504.0)
    w[4, ::2] = np.float16(-65504.0)
    w[5, :] = np.float16(2.0 ** -14)
    w16 = w.view(np.uint16)
    x = np.stack([g.standard_normal(n_in), -np.abs(g.standard_normal(n_in)),
                  np.full(n_in, 1e-30), np.full(n_in, 3e30)]).astype(np.float32)
    got = run_gemv(hs, w16, x)
    want = oracle.f16_gemv(w16, x)
    same = (bits(got) == bits(want)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), np.argwhere(~same)[:5]


def test_f16_gemv_strides_and_errors(hs, oracle):
    from geistlib_amd.binding import GeistHipError
    g = np.random.default_rng(4)
    n_out, n_in, m = 200, 256, 3
    w16 = g.standard_normal((n_out, n_in)).astype(np.float16).view(np.uint16)
    xbuf = np.full((m, n_in + 5), 1e30, dtype=np.float32)
    xbuf[:, :n_in] = g.standard_normal((m, n_in))
    d_x = to_dev(xbuf, torch)[:, :n_in]
    ybuf = torch.full((m, n_out + 3), -1.0, dtype=torch.float32, device="cuda")
    hs.f16_gemv(to_dev(w16.view(np.int16), torch), d_x, ybuf[:, :n_out])
    hs.sync()
    got = ybuf.cpu().numpy()
    assert (bits(got[:, :n_out]) == bits(oracle.f16_gemv(w16, xbuf[:, :n_in]))).all()
    assert (got[:, n_out:] == -1.0).all()
    bad = torch.zeros((4, 20), dtype=torch.float16, device="cuda")        # n_in % 8 != 0
    with pytest.raises(GeistHipError):
        hs.f16_gemv(bad, torch.zeros((1, 20), device="cuda"), torch.zeros((1, 4), device="cuda"))


@pytest.mark.parametrize("rows,n", [(3, 1), (2, 255), (2, 256), (2, 257), (2, 1024), (2, 1025),
                                    (512, 1030), (513, 1030), (513, 4095), (513, 4096), (513, 4097),
                                    (2, 4097), (700, 40)])
def test_rmsnorm_rows_at_the_edges_of_the_workgroup_sizes(hs, oracle, rows, n):
    """Rows on both sides of what 64, 256 and 1024 threads hold, and of the number of rows that
    chooses between the latter two: every bit as the oracle has it."""
    g = np.random.default_rng(rows + n)
    x = (g.standard_normal((rows, n)) * 3).astype(np.float32)
    w = (1 + 0.1 * g.standard_normal(n)).astype(np.float32)
    y = torch.full((rows, n), 7.0, dtype=torch.float32, device="cuda")
    hs.rmsnorm(to_dev(x, torch), to_dev(w, torch), 1e-6, y)
    hs.sync()
    assert (bits(y.cpu().numpy()) == bits(oracle.rmsnorm(x, w, 1e-6))).all()


def test_rmsnorm_of_many_short_rows_is_a_launch(hs):
    """4096 rows of 256 elements take what 512 take (3.5 times that with 1024 threads a row)."""
    w = torch.ones(256, device="cuda")
    x = [torch.randn((rows, 256), device="cuda") for rows in (512, 4096)]
    y = [torch.empty_like(t) for t in x]
    us = [call_us(lambda: hs.rmsnorm(a, w, 1e-6, b), 200) for a, b in zip(x, y)]
    assert us[1] < 2 * us[0], us


@pytest.mark.parametrize("rows,n", [(1, 2560), (5, 1536), (17, 4096), (3, 7), (2, 300)])
def test_rmsnorm_rows_bit_exact(hs, oracle, rows, n):
    g = np.random.default_rng(rows * 100 + n)
    x = (g.standard_normal((rows, n)) * g.choice([1e-3, 1.0, 50.0], (rows, 1))).astype(np.float32)
    w = (1.0 + 0.2 * g.standard_normal(n)).astype(np.float32)
    for eps in (1e-6, 1e-5):
        d_x = to_dev(x, torch)
        y = torch.empty_like(d_x)
        hs.rmsnorm(d_x, to_dev(w, torch), eps, y)
        hs.sync()
        assert (bits(y.cpu().numpy()) == bits(oracle.rmsnorm(x, w, eps))).all()
        hs.rmsnorm(d_x, to_dev(w, torch), eps, d_x)                        # in place
        hs.sync()
        assert (bits(d_x.cpu().numpy()) == bits(oracle.rmsnorm(x, w, eps))).all()


def test_head_to_token_without_leaving_the_device(hs, oracle):
    """head.c:94-188 end to end: norm -> lm_head -> sampler, logits never on the host. Equal to
    the oracle's chain on the oracle's logits, token for token."""
    from geistlib_amd import HipSampler, SampleParams
    g = np.random.default_rng(12)
    vocab, d_model, k = 32000, 2560, 6
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    hidden = (g.standard_normal((k, d_model)) * 3).astype(np.float32)
    norm_w = (1.0 + 0.1 * g.standard_normal(d_model)).astype(np.float32)
    u = g.random(k).astype(np.float32)
    d_h = to_dev(hidden, torch)
    hs.rmsnorm(d_h, to_dev(norm_w, torch), 1e-6, d_h)
    logits = torch.empty((k, vocab), dtype=torch.float32, device="cuda")
    hs.f16_gemv(to_dev(w16.view(np.int16), torch), d_h, logits)
    out = torch.empty(k, dtype=torch.int32, device="cuda")
    prm = dict(temperature=0.8, top_k=40, top_p=0.95)
    hs.sample(HipSampler.rows(logits), SampleParams.make(**prm), to_dev(u, torch), out)
    hs.sync()
    want_logits = oracle.f16_gemv(w16, oracle.rmsnorm(hidden, norm_w, 1e-6))
    assert (bits(logits.cpu().numpy()) == bits(want_logits)).all()
    want = [oracle.chain_u(want_logits[r], float(u[r]), **prm)[0] for r in range(k)]
    assert out.cpu().tolist() == want


@pytest.mark.parametrize("rows", [1, 2, 5])
@pytest.mark.parametrize("vocab,d_model", [(32000, 2560), (20001, 136), (8192, 64), (8193, 1536)])
def test_project_sample_rows_equals_the_separate_steps(hs, oracle, rows, vocab, d_model):
    """geist_hip_project_sample_rows: for one or two rows the norm runs inside the projection and,
    on the top-k path without soft-cap, the projection's epilogue replaces the sampler's scan.
    Logits bit-identical to the oracle's, tokens those of the oracle's chain."""
    from geistlib_amd import SampleParams
    print(f"project rows={rows} vocab={vocab} d_model={d_model}", flush=True)
    g = np.random.default_rng(rows * 1000 + vocab + d_model)
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    hidden = (g.standard_normal((rows, d_model)) * 3).astype(np.float32)
    norm_w = (1.0 + 0.1 * g.standard_normal(d_model)).astype(np.float32)
    u = g.random(rows).astype(np.float32)
    normed_want = oracle.rmsnorm(hidden, norm_w, 1e-6)
    # one row: the x86 decode kernel; more: the portable kernel that backend runs for batches
    want_logits = (oracle.f16_gemv(w16, normed_want) if rows == 1
                   else oracle.f16_linear_f64(w16, normed_want))
    d_w, d_h, d_nw, d_u = (to_dev(w16.view(np.int16), torch), to_dev(hidden, torch),
                           to_dev(norm_w, torch), to_dev(u, torch))
    normed = torch.empty((rows, d_model), dtype=torch.float32, device="cuda")
    for prm in (dict(temperature=0.8, top_k=40, top_p=0.95), dict(temperature=0.7, top_k=5),
                dict(temperature=0.0), dict(temperature=1.0), dict(temperature=0.9, top_p=0.9),
                dict(temperature=0.8, top_k=40, softcap=20.0), dict(temperature=0.8, top_k=300)):
        logits = torch.full((rows, vocab), 7.0, dtype=torch.float32, device="cuda")
        out = torch.full((rows,), -3, dtype=torch.int32, device="cuda")
        hs.project_sample(d_h, d_nw, 1e-6, d_w, logits, SampleParams.make(**prm), d_u, out,
                          normed=normed)
        hs.sync()
        assert (bits(logits.cpu().numpy()) == bits(want_logits)).all(), prm
        kw = {k: v for k, v in prm.items() if k != "softcap"}
        want = []
        for r in range(rows):
            row = want_logits[r]
            if prm.get("softcap") and prm["temperature"] > 0:
                row = oracle.softcap(row, prm["softcap"])
            want.append(oracle.argmax(row) if prm["temperature"] <= 0
                        else oracle.chain_u(row, float(u[r]), **kw)[0])
        assert out.cpu().tolist() == want, prm
    assert (d_h.cpu().numpy() == hidden).all()


def test_project_sample_rows_with_the_device_rng(hs, oracle):
    from geistlib_amd import SampleParams
    from geistlib_amd.workloads import xorshift_units
    g = np.random.default_rng(2)
    vocab, d_model, rows = 30000, 512, 2
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    hidden = (g.standard_normal((rows, d_model)) * 3).astype(np.float32)
    norm_w = np.ones(d_model, dtype=np.float32)
    st = torch.tensor([0xABCDEF], dtype=torch.int64, device="cuda")
    logits = torch.empty((rows, vocab), dtype=torch.float32, device="cuda")
    out = torch.empty(rows, dtype=torch.int32, device="cuda")
    hs.project_sample(to_dev(hidden, torch), to_dev(norm_w, torch), 1e-5,
                      to_dev(w16.view(np.int16), torch), logits,
                      SampleParams.make(temperature=0.8, top_k=40), None, out, rng_states=st,
                      normed=torch.empty((rows, d_model), dtype=torch.float32, device="cuda"))
    hs.sync()
    u, after = xorshift_units(0xABCDEF, rows)
    want_logits = oracle.f16_linear_f64(w16, oracle.rmsnorm(hidden, norm_w, 1e-5))
    want = [oracle.top_k_u(want_logits[r], 40, 0.8, float(u[r]))[0] for r in range(rows)]
    assert out.cpu().tolist() == want
    assert int(st.cpu().numpy().view(np.uint64)[0]) == after


@pytest.mark.parametrize("n_out,n_in,m", [(1000, 2560, 1), (130, 128, 1), (129, 256, 3),
                                          (4097, 1536, 2), (300, 16, 1), (300, 32, 5), (257, 48, 4),
                                          (640, 4096, 8), (500, 2560, 11), (33, 144, 2)])
def test_q8w_quantise_and_gemv_bit_exact(hs, oracle, n_out, n_in, m):
    """geist_hip_f16_to_q8w and geist_hip_q8w_gemv_rows against the oracle's restatement of
    f16_to_q8w / q8w_gemv_m1 (kernel_f16_gemv.c:66-127): int8 values, scales and results equal in
    every bit."""
    print(f"q8w n_out={n_out} n_in={n_in} m={m}", flush=True)
    g = np.random.default_rng(n_out + 3 * n_in + m)
    w16 = (g.standard_normal((n_out, n_in)) * g.choice([0.02, 1.0])).astype(np.float16)
    w16[0, :] = 0
    x = (g.standard_normal((m, n_in)) * g.choice([0.1, 1.0, 30.0], (m, 1))).astype(np.float32)
    d_w = to_dev(w16.view(np.int16), torch)
    d_wq = torch.empty((n_out, n_in), dtype=torch.int8, device="cuda")
    d_sc = torch.empty(n_out, dtype=torch.float32, device="cuda")
    hs.f16_to_q8w(d_w, d_wq, d_sc)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.q8w_gemv(d_wq, d_sc, to_dev(x, torch), y)
    hs.sync()
    wq, sc = oracle.f16_to_q8w(w16.view(np.uint16))
    assert (d_wq.cpu().numpy() == wq).all()
    assert (bits(d_sc.cpu().numpy()) == bits(sc)).all()
    want = oracle.q8w_gemv(wq, sc, x)
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


@pytest.mark.parametrize("n_out,n_in", [(1, 16), (63, 240), (64, 256), (65, 272), (130, 1040), (257, 752),
                                        (200, 1536)])
@pytest.mark.parametrize("m,tiny", [(3, False), (4, True), (5, False), (7, True), (8, False), (13, False)])
def test_q8w_gemv_of_several_rows(hs, oracle, n_out, n_in, m, tiny):
    """Batches of three and more rows, by chains on the matrix cores: remainders of a workgroup's 64 table
    rows, of a stage's 256 columns and of four activation rows, and sums among the subnormals. Every
    chain is the oracle's, so every result is equal in every bit."""
    print(f"q8w rows n_out={n_out} n_in={n_in} m={m} tiny={tiny}", flush=True)
    g = np.random.default_rng(n_out * 31 + n_in + m)
    wq = g.integers(-127, 128, (n_out, n_in)).astype(np.int8)
    sc = g.random(n_out).astype(np.float32)
    x = g.standard_normal((m, n_in)).astype(np.float32)
    if tiny:
        x *= np.float32(1e-40)
        sc[:] = 1.0
    y = torch.empty((m, n_out + 3), dtype=torch.float32, device="cuda")
    hs.q8w_gemv(to_dev(wq, torch), to_dev(sc, torch), to_dev(x, torch), y[:, :n_out])
    hs.sync()
    assert np.array_equal(y[:, :n_out].cpu().numpy().view(np.uint32), oracle.q8w_gemv(wq, sc, x).view(np.uint32))


@pytest.mark.parametrize("rows,vocab,d_model", [(1, 40000, 256), (1, 20000, 2560), (2, 9000, 512),
                                                (3, 8200, 128), (9, 5000, 64)])
def test_project_sample_rows_q8w_equals_the_separate_steps(hs, oracle, rows, vocab, d_model):
    """geist_hip_project_sample_rows_q8w: the int8 table in the fused tail. Logits bit-identical
    to the oracle's rmsnorm + q8w_gemv_m1, tokens those of the oracle's chain on them."""
    from geistlib_amd import SampleParams
    print(f"project q8w rows={rows} vocab={vocab} d_model={d_model}", flush=True)
    g = np.random.default_rng(rows * 77 + vocab + d_model)
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    wq, sc = oracle.f16_to_q8w(w16)
    hidden = (g.standard_normal((rows, d_model)) * 3).astype(np.float32)
    norm_w = (1.0 + 0.1 * g.standard_normal(d_model)).astype(np.float32)
    u = g.random(rows).astype(np.float32)
    want_logits = oracle.q8w_gemv(wq, sc, oracle.rmsnorm(hidden, norm_w, 1e-6))
    d_wq, d_sc, d_h, d_nw, d_u = (to_dev(wq, torch), to_dev(sc, torch), to_dev(hidden, torch),
                                  to_dev(norm_w, torch), to_dev(u, torch))
    normed = torch.empty((rows, d_model), dtype=torch.float32, device="cuda")
    for prm in (dict(temperature=0.8, top_k=40, top_p=0.95), dict(temperature=0.0),
                dict(temperature=0.9, top_p=0.9), dict(temperature=0.8, top_k=40, softcap=20.0),
                dict(temperature=0.8, top_k=300)):
        logits = torch.full((rows, vocab), 7.0, dtype=torch.float32, device="cuda")
        out = torch.full((rows,), -3, dtype=torch.int32, device="cuda")
        hs.project_sample_q8w(d_h, d_nw, 1e-6, d_wq, d_sc, logits, SampleParams.make(**prm), d_u,
                              out, normed=normed)
        hs.sync()
        assert (bits(logits.cpu().numpy()) == bits(want_logits)).all(), prm
        kw = {k: v for k, v in prm.items() if k != "softcap"}
        want = []
        for r in range(rows):
            row = want_logits[r]
            if prm.get("softcap") and prm["temperature"] > 0:
                row = oracle.softcap(row, prm["softcap"])
            want.append(oracle.argmax(row) if prm["temperature"] <= 0
                        else oracle.chain_u(row, float(u[r]), **kw)[0])
        assert out.cpu().tolist() == want, prm


def test_project_sample_rows_q8w_rejects_what_it_cannot_take(hs):
    from geistlib_amd import SampleParams
    from geistlib_amd.binding import GeistHipError
    vocab, d_model = 4096, 72                      # a multiple of 8, not of 16
    wq = torch.zeros((vocab, d_model), dtype=torch.int8, device="cuda")
    sc = torch.ones(vocab, dtype=torch.float32, device="cuda")
    h = torch.ones((1, d_model), dtype=torch.float32, device="cuda")
    nw = torch.ones(d_model, dtype=torch.float32, device="cuda")
    logits = torch.empty((1, vocab), dtype=torch.float32, device="cuda")
    out = torch.empty(1, dtype=torch.int32, device="cuda")
    with pytest.raises(GeistHipError):
        hs.project_sample_q8w(h, nw, 1e-6, wq, sc, logits, SampleParams.make(temperature=0.0),
                              None, out, normed=torch.empty_like(h))
    with pytest.raises(GeistHipError):
        hs.project_sample_q8w(h, nw, 1e-6, wq, None, logits, SampleParams.make(temperature=0.0),
                              None, out, normed=torch.empty_like(h))


@pytest.mark.parametrize("n_out,n_in,m", [(1000, 2560, 1), (130, 128, 1), (129, 256, 3),
                                          (4097, 1536, 2), (300, 8, 1), (300, 40, 5), (257, 72, 4),
                                          (640, 4096, 8), (500, 2560, 11), (20000, 2560, 8)])
def test_f16_linear_in_double_bit_exact(hs, oracle, n_out, n_in, m):
    """geist_hip_f16_linear_rows against cpu_scalar_w_quant_mN (weight_resolve.c:215-241): the
    double sum in index order, rounded once -- equal in every bit, also where the sum lies at a
    binary32 rounding boundary (integer inputs make many sums land exactly on one)."""
    print(f"f16 linear f64 n_out={n_out} n_in={n_in} m={m}", flush=True)
    g = np.random.default_rng(n_out + 5 * n_in + m)
    w16 = (g.standard_normal((n_out, n_in)) * g.choice([0.02, 1.0])).astype(np.float16)
    x = (g.standard_normal((m, n_in)) * g.choice([0.1, 1.0, 30.0], (m, 1))).astype(np.float32)
    if n_out > 256:
        # rows whose sums are exact halves of a binary32 step: every order must agree there too
        w16[:128] = g.integers(-4, 5, (128, n_in)).astype(np.float16)
        x[0] = g.integers(-3, 4, n_in).astype(np.float32)
        x[0, 0] += np.float32(2.0 ** -20)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


@pytest.mark.parametrize("m", [1, 3, 7])
def test_f16_linear_in_double_at_the_ends_of_the_range(hs, oracle, m):
    """Sums that overflow binary32, sums in its subnormal range, zero rows, weights that are
    binary16 subnormals and infinities: every bit as the oracle has it (NaN where it has NaN)."""
    g = np.random.default_rng(m)
    n_out, n_in = 700, 512
    w16 = (g.standard_normal((n_out, n_in)) * 0.05).astype(np.float16)
    w16[0] = 0
    w16[1] = np.float16(6.0e-8)                       # the smallest binary16 subnormals
    w16[2] = np.float16(65504.0)                      # the largest binary16
    w16[3, 5] = np.float16(np.inf)
    w16[4, 7] = np.float16(-np.inf)
    w16[4, 9] = np.float16(np.inf)                    # inf - inf
    x = (g.standard_normal((m, n_in)) * 3).astype(np.float32)
    x[0] = np.float32(1.0e-38)                        # subnormal results against rows of 0.05
    if m > 1:
        x[1] = np.float32(3.0e38)                     # overflows against every row of one sign
        x[1, ::2] *= -1
        x[1, :4] = np.float32(3.0e38)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    got = y.cpu().numpy()
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all()
    assert (bits(got)[~nan] == bits(want)[~nan]).all(), np.argwhere(bits(got) != bits(want))[:5]
    assert np.isinf(want).any() and nan.any() and (np.abs(want[0, 5:]) < 1.2e-38).any()


def sums_at_the_end_of_binary32(n_in, rng):
    """Activations against weights of 1 (or -1) whose sums lie around 2^128 - 2^103, where binary32
    ends: the exact sum below it and the sum in index order above it (17 additions that each round
    up by half a step of the double sum), the other way round, and well on either side."""
    top = np.float32(np.finfo(np.float32).max)
    x = np.zeros((6, n_in), dtype=np.float32)
    step = np.float32(2.0 ** 74)
    up, down = step * np.float32(1 + 2.0 ** -10), step * np.float32(1 - 2.0 ** -10)
    near = np.float32((2.0 ** 24 - 1) * 2.0 ** 79)          # 2^103 - 2^79
    x[0, :2], x[0, 2:19] = (top, near), up                  # exact: finite; in order: infinite
    x[1, :2], x[1, 2:40] = (top, near), down                # exact: infinite; in order: finite
    x[2, :2] = top, near                                    # finite either way
    x[3, :3] = top, near, np.float32(2.0 ** 80)             # infinite either way
    x[4] = rng.standard_normal(n_in) * 3e38 / np.sqrt(n_in) # about one row in three infinite
    x[5, :2] = top, top
    return x


def test_f16_linear_in_double_sums_at_the_end_of_binary32(hs, oracle):
    """Where the order of the additions decides whether a sum is the largest binary32 or infinite,
    the order is the reference's."""
    g = np.random.default_rng(77)
    n_out, n_in = 300, 64
    w16 = g.choice([-1.0, 1.0], (n_out, n_in)).astype(np.float16)
    w16[:8], w16[8:16] = 1.0, -1.0
    x = sums_at_the_end_of_binary32(n_in, g)
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    assert np.isinf(want[0, :16]).all() and np.isfinite(want[1, :16]).all()
    for m0, m1 in ((0, 6), (0, 1), (1, 2)):
        y = torch.full((m1 - m0, n_out), 7.0, dtype=torch.float32, device="cuda")
        hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x[m0:m1], torch), y)
        hs.sync()
        got = y.cpu().numpy()
        assert (bits(got) == bits(want[m0:m1])).all(), np.argwhere(bits(got) != bits(want[m0:m1]))[:8]


def f16_linear_us(hs, w16, x):
    y = torch.empty((x.shape[0], w16.shape[0]), dtype=torch.float32, device="cuda")
    return call_us(lambda: hs.f16_linear(w16, x, y), 20)


@pytest.mark.parametrize("m", [1, 5, 8, 16, 19])
def test_f16_linear_in_double_with_activations_that_are_not_finite(hs, oracle, m):
    """A NaN, an infinity, infinities of either sign, all of them, among rows that are finite: each
    output as the oracle has it, against weights that are zero, NaN and infinite among others."""
    g = np.random.default_rng(60 + m)
    n_out, n_in = 900, 264
    w16 = (g.standard_normal((n_out, n_in)) * 0.05).astype(np.float16)
    w16[0] = 0
    w16[1, 3], w16[2, 5], w16[3, 7] = np.nan, np.inf, -np.inf
    w16[4:200, 9] = 0
    w16[200:300] *= 100
    x = (g.standard_normal((m, n_in)) * 3).astype(np.float32)
    broken = ([(17, np.nan)], [(9, np.inf)], [(9, -np.inf)], [(9, np.inf), (100, -np.inf)],
              [(5, np.inf), (100, np.inf), (200, np.inf)], [(9, np.inf), (17, np.nan)], [(0, np.nan)])
    for r in range(m):
        if m == 1 or r % 2:
            for at, v in broken[(r // 2) % len(broken)]:
                x[r, at] = v
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    got = y.cpu().numpy()
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all(), np.argwhere(np.isnan(got) != nan)[:5]
    assert (bits(got)[~nan] == bits(want)[~nan]).all(), np.argwhere(bits(got) != bits(want))[:5]


def test_f16_linear_in_double_takes_rows_that_are_not_finite_in_its_stride(hs):
    """One broken row of a batch does not hold the others up: with a NaN nothing is looked at
    again (1.0 times the time of finite rows), with an infinity each output of the row once (2.4
    times). Sent through the sums in index order they took 37 times as long."""
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    w = torch.empty((64000, 2048), dtype=torch.float16, device="cuda").normal_(0, 0.05, generator=g)
    w, x = w.view(torch.int16), torch.randn((8, 2048), device="cuda", generator=g)
    finite = f16_linear_us(hs, w, x)
    for value, most in ((float("nan"), 2.0), (float("inf"), 6.0)):
        x[3, 100] = value
        assert f16_linear_us(hs, w, x) < most * finite, value


@pytest.mark.parametrize("m,n_in", [(2, 520), (8, 256), (16, 72), (6, 3528)])
def test_f16_linear_in_double_with_large_weights(hs, oracle, m, n_in):
    """Weights around the ends of what the leading digit and the conversion hold (64, 127, 2^7),
    alone in their rows and in each column of a group of sixteen, and rows of a large norm."""
    g = np.random.default_rng(90 + m)
    ends = np.array([62.5, 63.0, 63.47, 63.5, 63.97, 64.0, 64.5, 65.0, 65.47, 65.5, 66.0, 126.9,
                     127.0, 127.44, 127.5, 127.94, 128.0, 128.5, 129.0, 255.9, 1000.0, 65504.0])
    ends = np.concatenate([ends, -ends])
    n_out = 3 * len(ends) + 200
    w16 = (g.standard_normal((n_out, n_in)) * 0.05).astype(np.float16)
    for i, e in enumerate(ends):
        w16[i, g.integers(0, n_in)] = e
        w16[len(ends) + i, i % 16 + 16 * g.integers(0, n_in // 16)] = e
        w16[2 * len(ends) + i, ::3] = e
    w16[-200:] = (g.standard_normal((200, n_in)) * g.choice([3.0, 10.0, 30.0], (200, 1))).astype(np.float16)
    x = (g.standard_normal((m, n_in)) * 3).astype(np.float32)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


def test_f16_linear_in_double_takes_rows_of_a_large_norm_in_its_stride(hs):
    """It is a single weight's magnitude that the digits are bound by, not a row's norm: a table
    of standard deviation 4 takes what one of 0.05 takes (8 times as long when rows of a norm
    above 126 were left to the second kernel)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    x = torch.randn((8, 2048), device="cuda", generator=g)
    us = []
    for std in (0.05, 4.0):
        w = torch.empty((64000, 2048), dtype=torch.float16, device="cuda").normal_(0, std, generator=g)
        us.append(f16_linear_us(hs, w.view(torch.int16), x))
    assert us[1] < 2 * us[0], us


@pytest.mark.parametrize("n_out,n_in,m", [
    (50001, 72, 8), (50001, 256, 3), (33000, 264, 16), (33000, 72, 9),   # LDS-resident
    (49500, 3400, 5), (49500, 3656, 8), (49300, 5128, 2), (33000, 1672, 16),   # through LDS
    (40, 3392, 8), (40, 3400, 8), (40, 1664, 16), (40, 1672, 16), (40, 5120, 4), (40, 5128, 4)])
def test_f16_linear_in_double_beyond_a_wavefronts_first_tile(hs, oracle, n_out, n_in, m):
    """Tables that give some wavefronts a second tile of sixteen rows (49152 rows on 256 compute
    units, 32768 of more than 8 activation rows): weights of the next tile asked for across the end of
    one, activations in LDS or passing through it in an even (54, 27) and odd (58) number of stages;
    and the widest rows that LDS holds, with the next wider ones. Rows of both tiles are compared."""
    print(f"f16 linear second tile {n_out} x {n_in}, {m} rows", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n_out + n_in + m)
    w = torch.empty((n_out, n_in), dtype=torch.float16, device="cuda").normal_(0, 0.05, generator=g)
    x = torch.randn((m, n_in), device="cuda", generator=g) * 3
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(w.view(torch.int16), x, y)
    hs.sync()
    rows = np.unique(np.concatenate([np.arange(min(n_out, 40)), np.arange(max(0, n_out - 400), n_out),
                                     np.random.default_rng(m).integers(0, n_out, 300)]))
    at = torch.from_numpy(rows).cuda()
    want = oracle.f16_linear_f64(w[at].cpu().numpy().view(np.uint16), x.cpu().numpy())
    got = y[:, at].cpu().numpy()
    assert (bits(got) == bits(want)).all(), rows[np.argwhere(bits(got) != bits(want))[:5, 1]]
    # the rest of the outputs, all below 256: within a step of binary32 (2^-16) of a plain product in
    # double; a lost or doubled tile is off by the outputs themselves
    plain = x.double() @ w.double().T
    assert plain.abs().max().item() < 256 and (y.double() - plain).abs().max().item() < 2.0 ** -16


@pytest.mark.parametrize("rows,vocab,d_model", [(9, 33000, 72), (16, 900, 1672), (19, 700, 1672),
                                                (8, 1000, 3400), (3, 500, 5128), (7, 130, 8)])
def test_project_sample_of_many_hidden_rows(hs, oracle, rows, vocab, d_model):
    """The norm in the launch that cuts the activations: more than 8 rows, more than 16 (two passes),
    row lengths on both sides of what LDS holds. Normed rows and logits bit for bit, greedy tokens."""
    from geistlib_amd import SampleParams
    print(f"project rows={rows} vocab={vocab} d_model={d_model}", flush=True)
    g = np.random.default_rng(rows + vocab + d_model)
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    hidden = (g.standard_normal((rows, d_model)) * 3).astype(np.float32)
    norm_w = (1.0 + 0.1 * g.standard_normal(d_model)).astype(np.float32)
    normed = torch.full((rows, d_model), 7.0, dtype=torch.float32, device="cuda")
    logits = torch.full((rows, vocab), 7.0, dtype=torch.float32, device="cuda")
    out = torch.full((rows,), -3, dtype=torch.int32, device="cuda")
    hs.project_sample(to_dev(hidden, torch), to_dev(norm_w, torch), 1e-6,
                      to_dev(w16.view(np.int16), torch), logits, SampleParams.make(temperature=0.0),
                      None, out, normed=normed)
    hs.sync()
    normed_want = oracle.rmsnorm(hidden, norm_w, 1e-6)
    want = oracle.f16_linear_f64(w16, normed_want)
    assert (bits(normed.cpu().numpy()) == bits(normed_want)).all()
    assert (bits(logits.cpu().numpy()) == bits(want)).all()
    assert out.cpu().tolist() == [oracle.argmax(row) for row in want]


def few_bits(kind, shape, g):
    """Activations of few significant bits: small integers, bfloat16 values."""
    if kind == "int8":
        return torch.randint(-127, 128, shape, device="cuda", generator=g).float()
    return (torch.randn(shape, device="cuda", generator=g) * 3).bfloat16().float()


@pytest.mark.parametrize("kind,m,n_in", [("int8", 8, 1024), ("int8", 2, 520), ("int8", 16, 2568),
                                         ("bfloat16", 8, 1024), ("bfloat16", 3, 2560)])
def test_f16_linear_in_double_with_activations_of_few_bits(hs, oracle, kind, m, n_in):
    """Many sums lie right on a rounding boundary, and most are exact whatever the order: every bit
    as the oracle has it, also where a few large weights make the additions round."""
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n_in)
    x = few_bits(kind, (m, n_in), g)
    w = torch.empty((3000, n_in), dtype=torch.float16, device="cuda").normal_(0, 0.05, generator=g)
    w[1000:1100] *= 1000                               # sums of more than 53 bits
    w[1000:1100, ::2] *= 2.0 ** -12
    w[1100:1200] = 0
    y = torch.full((m, 3000), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(w.view(torch.int16), x, y)
    hs.sync()
    want = oracle.f16_linear_f64(w.cpu().numpy().view(np.uint16), x.cpu().numpy())
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


def test_f16_linear_in_double_takes_activations_of_few_bits_in_its_stride(hs):
    """8 rows of integers against 64000 x 2048 take 1.6 times what general rows take (9 times when
    each sum on a boundary was added once more in index order)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    w = torch.empty((64000, 2048), dtype=torch.float16, device="cuda").normal_(0, 0.05, generator=g)
    us = [f16_linear_us(hs, w.view(torch.int16), x)
          for x in (torch.randn((8, 2048), device="cuda", generator=g), few_bits("int8", (8, 2048), g))]
    assert us[1] < 4 * us[0], us


def sums_open_to_the_end(n_in):
    """An activation row whose sum over weights of 1 or -1 lies on a rounding boundary but for terms
    that its additions round away: 2^30 + 1 + 2^-24 - 2^30 and a few of 2^-60."""
    x = np.zeros(n_in, dtype=np.float32)
    x[[0, 1, 2, n_in - 2]] = 2.0 ** 30, 1.0, 2.0 ** -24, -2.0 ** 30
    x[[3, n_in - 1]] = 2.0 ** -60, 2.0 ** -62
    return x


@pytest.mark.parametrize("n_out,n_in,m", [(2100, 520, 16), (2100, 512, 16), (3, 8, 1), (20, 2568, 2),
                                          (1100, 1032, 16)])
def test_f16_linear_in_double_with_every_sum_in_index_order(hs, oracle, n_out, n_in, m):
    """Every output is left to the sum in index order: more than the list for that holds (2100 x
    16), fewer, and rows of up to 512 columns, which are not listed."""
    g = np.random.default_rng(n_out + n_in)
    w16 = g.choice([-1.0, 1.0], (n_out, n_in)).astype(np.float16)
    w16[: n_out // 2] = 1.0
    x = np.tile(sums_open_to_the_end(n_in), (m, 1)) * (2.0 ** np.arange(m))[:, None].astype(np.float32)
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


def test_f16_linear_in_double_scratch_is_one_list(hs):
    """The scratch of a table of 400000 rows: 16 entries of eight bytes a row, one list of them."""
    from geistlib_amd import HipSampler
    w = torch.zeros((400000, 8), dtype=torch.int16, device="cuda")
    x = torch.zeros((2, 8), device="cuda")
    y = torch.empty((2, 400000), device="cuda")
    hs.f16_linear(w[:100], x, y[:, :100])              # (the kernels are loaded)
    s = HipSampler(max_rows=2, max_vocab=1000)
    s.f16_linear(w[:8], x, y[:, :8])
    s.sync()
    free = torch.cuda.mem_get_info()[0]
    s.f16_linear(w, x, y)
    s.sync()
    used = free - torch.cuda.mem_get_info()[0]
    s.close()
    assert used < 1.25 * 400000 * 16 * 8, used


@pytest.mark.parametrize("m", [2, 9, 19])
def test_f16_linear_in_double_with_row_strides(hs, oracle, m):
    """Padded rows on both sides (row strides above the row lengths), 19 rows in two passes of the
    matrix-core kernel; the padding of the output is left alone."""
    g = np.random.default_rng(40 + m)
    n_out, n_in = 3000, 1536
    w16 = (g.standard_normal((n_out, n_in)) * 0.05).astype(np.float16)
    xbuf = (g.standard_normal((m, n_in + 24)) * 2).astype(np.float32)
    d_x = to_dev(xbuf, torch)
    y = torch.full((m, n_out + 8), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), d_x[:, :n_in], y[:, :n_out])
    hs.sync()
    got = y.cpu().numpy()
    want = oracle.f16_linear_f64(w16.view(np.uint16), xbuf[:, :n_in])
    assert (bits(got[:, :n_out]) == bits(want)).all()
    assert (got[:, n_out:] == 7.0).all()


def test_project_sample_rows_in_the_portable_backends_arithmetic(hs, oracle):
    """geist_hip_sampler_set_projection(PORTABLE): one row goes through the double-accumulation
    kernel too, as on the reference's cpu_scalar backend."""
    from geistlib_amd import SampleParams
    g = np.random.default_rng(61)
    vocab, d_model = 30000, 1536
    w16 = (g.standard_normal((vocab, d_model)) * 0.05).astype(np.float16).view(np.uint16)
    hidden = (g.standard_normal((1, d_model)) * 3).astype(np.float32)
    norm_w = (1.0 + 0.1 * g.standard_normal(d_model)).astype(np.float32)
    u = g.random(1).astype(np.float32)
    normed_want = oracle.rmsnorm(hidden, norm_w, 1e-6)
    logits = torch.empty((1, vocab), dtype=torch.float32, device="cuda")
    out = torch.empty(1, dtype=torch.int32, device="cuda")
    args = (to_dev(hidden, torch), to_dev(norm_w, torch), 1e-6, to_dev(w16.view(np.int16), torch),
            logits, SampleParams.make(temperature=0.8, top_k=40), to_dev(u, torch), out)
    normed = torch.empty((1, d_model), dtype=torch.float32, device="cuda")
    try:
        hs.set_projection(True)
        hs.project_sample(*args, normed=normed)
        hs.sync()
        want = oracle.f16_linear_f64(w16, normed_want)
        assert (bits(logits.cpu().numpy()) == bits(want)).all()
        assert out.cpu().tolist() == [oracle.top_k_u(want[0], 40, 0.8, float(u[0]))[0]]
    finally:
        hs.set_projection(False)
    hs.project_sample(*args, normed=normed)
    hs.sync()
    assert (bits(logits.cpu().numpy()) == bits(oracle.f16_gemv(w16, normed_want))).all()


@pytest.mark.parametrize("seed", fuzz_seeds(4))
def test_random_projection_shapes(hs, oracle, seed):
    """Norm, F16 and int8 projections, the quantiser and the projection in double on random
    shapes, scales and row counts, each against the oracle in every bit. Integer-valued and
    cancelling data put the sums in double on rounding boundaries of binary32."""
    g = np.random.default_rng(9000 + seed)
    for case in range(5):
        n_out = int(g.integers(1, 5000))
        n_in = 16 * int(g.integers(1, 257)) + (8 if g.random() < 0.3 else 0)
        m = int(g.integers(1, 21))
        kind = int(g.integers(0, 3))
        print(f"projection seed {seed} case {case}: n_out={n_out} n_in={n_in} m={m} kind={kind}",
              flush=True)
        w = (g.standard_normal((n_out, n_in)) * g.choice([1e-3, 0.05, 1.0, 30.0])).astype(np.float16)
        x = (g.standard_normal((m, n_in)) * g.choice([1e-3, 1.0, 100.0], (m, 1))).astype(np.float32)
        if kind == 1:
            w = g.integers(-6, 7, (n_out, n_in)).astype(np.float16)
            x = g.integers(-5, 6, (m, n_in)).astype(np.float32)
            x[:, 0] += np.float32(2.0 ** -int(g.integers(10, 30)))
        if kind == 2:
            w[:, 1::2] = -w[:, ::2]
            x[:, 1::2] = x[:, ::2] * np.float32(1 + 2.0 ** -12)
        w16 = w.view(np.uint16)
        d_w, d_x = to_dev(w.view(np.int16), torch), to_dev(x, torch)
        y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
        hs.f16_gemv(d_w, d_x, y)
        hs.sync()
        assert (bits(y.cpu().numpy()) == bits(oracle.f16_gemv(w16, x))).all()
        y.fill_(7.0)
        hs.f16_linear(d_w, d_x, y)
        hs.sync()
        assert (bits(y.cpu().numpy()) == bits(oracle.f16_linear_f64(w16, x))).all()
        if n_in % 16 == 0:
            wq = torch.empty((n_out, n_in), dtype=torch.int8, device="cuda")
            sc = torch.empty(n_out, dtype=torch.float32, device="cuda")
            hs.f16_to_q8w(d_w, wq, sc)
            hs.sync()
            wq_want, sc_want = oracle.f16_to_q8w(w16)
            assert (wq.cpu().numpy() == wq_want).all()
            assert (bits(sc.cpu().numpy()) == bits(sc_want)).all()
            y.fill_(7.0)
            hs.q8w_gemv(wq, sc, d_x, y)
            hs.sync()
            assert (bits(y.cpu().numpy()) == bits(oracle.q8w_gemv(wq_want, sc_want, x))).all()
        norm_w = g.standard_normal(n_in).astype(np.float32)
        eps = float(g.choice([1e-5, 1e-6, 0.0]))
        normed = torch.empty((m, n_in), dtype=torch.float32, device="cuda")
        hs.rmsnorm(d_x, to_dev(norm_w, torch), eps, normed)
        hs.sync()
        assert (bits(normed.cpu().numpy()) == bits(oracle.rmsnorm(x, norm_w, eps))).all()


@pytest.mark.parametrize("m", [1, 2, 5, 9, 14])
def test_f16_linear_in_double_on_order_sensitive_rows(hs, oracle, m):
    """Rows whose last quarter cancels a huge first quarter: the small terms in between are added
    to a sum 2^24 times their size, so the binary32 result depends on the ORDER of the additions in
    double (numpy's own float64 product rounds some of these outputs to another value). The
    device kernels add in another order and re-add, in index order, what their bound cannot
    decide: every bit equals the oracle, which equals the reference's cpu_scalar_w_quant_mN
    compiled from its tree (tests/test_lm_head_oracle.py)."""
    g = np.random.default_rng(900 + m)
    n_out, n_in = 3000, 1024
    q = n_in // 4
    w = (g.standard_normal((n_out, n_in)) * 4).astype(np.float16)
    x = (g.standard_normal((m, n_in)) * 100).astype(np.float32)
    x[:, :q] *= np.float32(2.0 ** 24)
    w[:, 3 * q: 4 * q] = -w[:, :q]
    x[:, 3 * q: 4 * q] = x[:, :q]
    y = torch.full((m, n_out), float("nan"), dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = np.atleast_2d(oracle.f16_linear_f64(w.view(np.uint16), x if m > 1 else x[0]))
    got = y.cpu().numpy()
    other = (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)
    assert (other != want).any()          # the case does hang on the order
    assert (got.view(np.uint32) == want.view(np.uint32)).all(), int((got != want).sum())


@pytest.mark.parametrize("n_out,n_in,m,scale", [
    (1, 8, 2, 0.05), (15, 56, 4, 0.05), (17, 64, 5, 0.05), (33, 72, 8, 0.05), (4113, 256, 9, 0.05),
    (50, 3520, 8, 0.05), (50, 1768, 13, 0.05), (31, 264, 16, 40.0), (64, 4096, 3, 2.5), (9, 65544, 2, 0.05)])
def test_f16_linear_digit_edges(hs, oracle, n_out, n_in, m, scale):
    """The int8-digit kernel at the edges of its tiles (16 weight rows, 64 columns, 4 / 8 / 16
    activation rows), of what LDS holds of the activations (3392 columns of 8 rows, 1664 of 16), of
    the weights' range (rows of magnitudes beyond 127, or of ||w|| that could hold one) and of the
    integer sums (65536 columns): equal to the oracle in every bit."""
    print(f"f16 digits n_out={n_out} n_in={n_in} m={m} scale={scale}", flush=True)
    g = np.random.default_rng(n_out + n_in + m)
    w16 = (g.standard_normal((n_out, n_in)) * scale).astype(np.float16)
    w16[0, :8] = [127.0, -127.5, 0.5, -0.5, 6e-8, -6e-8, 0.25, -0.0]
    w16[-1] = g.choice(np.array([2.0 ** -24, -2.0 ** -14, 0.498, -0.4990234375], np.float16), n_in)
    x = g.standard_normal((m, n_in)).astype(np.float32)
    x *= np.exp2(g.integers(-40, 3, x.shape)).astype(np.float32)   # remainders beyond six digits
    x[0] = np.where(g.random(n_in) < 0.5, np.float32(1.0), np.float32(-1.0))   # partial sums near 0
    y = torch.full((m, n_out), 7.0, dtype=torch.float32, device="cuda")
    hs.f16_linear(to_dev(w16.view(np.int16), torch), to_dev(x, torch), y)
    hs.sync()
    want = oracle.f16_linear_f64(w16.view(np.uint16), x)
    got = y.cpu().numpy()
    assert (bits(got) == bits(want)).all(), np.argwhere(bits(got) != bits(want))[:5]


@pytest.mark.parametrize("n", [1, 1023, 1025, 4095, 4097, 6000])
def test_rmsnorm_at_the_edges_of_what_a_workgroup_holds(hs, oracle, n):
    """A workgroup of 1024 threads holds four elements each; beyond 4096 it reads the row again."""
    g = np.random.default_rng(n)
    x = (g.standard_normal((3, n)) * 3).astype(np.float32)
    w = (1.0 + 0.2 * g.standard_normal(n)).astype(np.float32)
    d_x = to_dev(x, torch)
    for y in (torch.empty_like(d_x), d_x):                                 # and in place
        hs.rmsnorm(d_x, to_dev(w, torch), 1e-6, y)
        hs.sync()
        assert (bits(y.cpu().numpy()) == bits(oracle.rmsnorm(x, w, 1e-6))).all()


@pytest.mark.parametrize("table", ["q6k", "q4k"])
@pytest.mark.parametrize("d_model", [256, 1024, 1792, 4096, 4352, 6144])
def test_norm_and_quantiser_in_one_launch(hs, oracle, table, d_model):
    """The norm that quantises on the way (four super-blocks at a time, from 4096 elements on
    reading back) against the norm and the quantiser as launches of their own: bit for bit."""
    from geistlib_amd import SampleParams
    from oracle_lib import random_q4k_table, random_q6k_table
    g = np.random.default_rng(d_model)
    vocab = 72
    w = (random_q6k_table if table == "q6k" else random_q4k_table)(g, vocab, d_model)
    size, pack, run, linear = ((hs.q6k_packed_bytes, hs.q6k_pack, hs.project_sample_q6k_packed,
                                hs.q6k_packed_linear_x86) if table == "q6k" else
                               (hs.q4k_packed_bytes, hs.q4k_pack, hs.project_sample_q4k_packed,
                                hs.q4k_packed_linear_x86))
    packed = torch.empty(size(vocab, d_model), dtype=torch.uint8, device="cuda")
    pack(to_dev(w, torch), d_model, packed)
    norm_w = (1.0 + 0.2 * g.standard_normal(d_model)).astype(np.float32)
    for rows in (1, 3, 4):
        h = (g.standard_normal((rows, d_model)) * 3).astype(np.float32)
        logits = torch.empty((rows, vocab), device="cuda")
        normed = torch.empty((rows, d_model), device="cuda")
        out = torch.empty(rows, dtype=torch.int32, device="cuda")
        run(to_dev(h, torch), to_dev(norm_w, torch), 1e-6, packed, vocab, logits,
            SampleParams.make(temperature=0.0), None, out, normed)
        want = torch.empty((rows, vocab), device="cuda")
        linear(packed, vocab, d_model, normed, want)
        hs.sync()
        assert (bits(normed.cpu().numpy()) == bits(oracle.rmsnorm(h, norm_w, 1e-6))).all()
        assert (bits(logits.cpu().numpy()) == bits(want.cpu().numpy())).all(), rows
