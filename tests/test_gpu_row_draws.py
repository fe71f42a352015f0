"""Draws from the rows' own generators that a scan takes for the launches behind it, and recorded
calls whose workgroups wait for one another or take draws: tokens against the same call on units
computed on the host, generator states by their number, over several calls or replays."""
import numpy as np
import pytest

from gpu_util import to_dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

T = dict(temperature=0.9)
K40 = dict(temperature=0.7, top_k=40, top_p=0.9)
PEN = dict(rep=1.2, freq=0.3, pres=0.1)
CASES = [
    (80, 32000, T, ""), (80, 32000, {**T, **PEN}, ""),      # two launches, chunks of 2048
    (25, 131072, T, ""), (64, 128256, {**T, **PEN}, ""),    # ... of 8192
    (80, 32000, T, "fast"), (64, 128256, T, "fast"),        # ... without a meeting
    (80, 32000, {**T, **PEN}, "fast"),
    (40, 32000, K40, "two"), (12, 131072, {**K40, **PEN}, "two"),   # k_cand_scan, k_final_cand
    (64, 262144, K40, ""), (256, 131072, K40, ""),           # large: k_tmax_scan, k_topk_wide
    (16, 50001, K40, ""),                                   # k_tmax_scan, k_final_topk
    (4, 50001, dict(temperature=0.9, top_k=150), ""),       # k_tmax_scan, k_topk_wide
    (24, 50257, dict(temperature=1.0, top_p=0.95), ""),     # exp-sum pass, k_window
    (80, 70000, dict(temperature=1.0, top_p=0.95), ""),     # ... with the row-final kernel between
    (6, 40000, {**T, "min_p": 0.05}, ""), (80, 70000, {**T, **PEN, "min_p": 0.05}, ""),
]


def setup_case(rows, n, options, form, seed):
    from geistlib_amd import HipSampler, SampleParams
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x = torch.randn((rows, n), device="cuda", generator=gen) * 2
    hist = hl = None
    if "rep" in options:
        hist = torch.randint(0, n, (rows, 300), device="cuda", generator=gen, dtype=torch.int32)
        hl = torch.full((rows,), 300, device="cuda", dtype=torch.int32)
    hs = HipSampler(rows, n)
    hs.set_sums(fast=form == "fast")
    if form == "two":
        hs.one_launch_topk(False)
    prm = SampleParams.make(**options)
    hs.prepare(prm, n)
    seeds = [(r + seed) * 0x9E3779B97F4A7C15 % 2 ** 64 for r in range(1, rows + 1)]
    states = to_dev(np.array(seeds, dtype=np.uint64).view(np.int64), torch)
    out, want = (torch.full((rows,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
    return hs, HipSampler.rows(x, hist, hl), prm, seeds, states, out, want, (x, hist, hl)


def next_units(seeds):
    from geistlib_amd.workloads import xorshift_units
    drawn = [xorshift_units(s, 1) for s in seeds]
    return (to_dev(np.array([d[0][0] for d in drawn], dtype=np.float32), torch),
            [int(d[1]) for d in drawn])


def states_of(states):
    return states.cpu().numpy().view(np.uint64).tolist()


@pytest.mark.parametrize("rows,n,options,form", CASES)
def test_draws_taken_by_a_scan(rows, n, options, form):
    print(f"scan draws {rows} x {n} {options} {form}", flush=True)
    hs, view, prm, seeds, states, out, want, keep = setup_case(rows, n, options, form, rows + n)
    try:
        for step in range(4):
            if step == 2:
                hs.set_wait_limit(0)
            hs.sample_rng(view, prm, states, False, out)
            units, seeds = next_units(seeds)
            hs.sample(view, prm, units, want)
            hs.sync()
            assert out.tolist() == want.tolist(), step
            assert states_of(states) == seeds, step
    finally:
        hs.close()


@pytest.mark.parametrize("rows,n,options,form", [
    (9, 70001, T, ""), (24, 32000, {**T, **PEN}, ""),       # the last chunk draws
    (80, 32000, T, ""), (80, 32000, T, "fast"), (40, 32000, K40, "two"), (64, 262144, K40, ""),
    (24, 50257, dict(temperature=1.0, top_p=0.95), ""), (6, 40000, {**T, "min_p": 0.05}, ""),
    (9, 70001, dict(temperature=0.0), ""), (8, 32000, dict(temperature=0.0, **PEN), ""),
])
@pytest.mark.parametrize("own", [True, False])
def test_recorded_calls_draw_on_every_replay(rows, n, options, form, own):
    print(f"recorded {rows} x {n} {options} {form} own={own}", flush=True)
    greedy = options["temperature"] == 0.0
    hs, view, prm, seeds, states, out, want, (x, *_) = setup_case(rows, n, options, form, rows + n + own)
    units, _ = next_units(seeds)
    d_u = units.clone()

    def call(to):
        hs.sample_rng(view, prm, states, False, to) if own else hs.sample(view, prm, d_u, to)

    try:
        call(out)                                  # eager first: the eager arrays are in use
        hs.sync()
        if own and not greedy:
            _, seeds = next_units(seeds)
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            hs.set_stream(torch.cuda.current_stream().cuda_stream)
            call(out)
        torch.cuda.synchronize()
        hs.set_stream(None)
        for replay in range(4):
            x.copy_(x.roll(1, 0) * 0.97)           # other rows each time
            units, after = next_units(seeds)
            if greedy or not own:
                after = seeds
            d_u.copy_(units)
            out.fill_(-7)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            hs.sample(view, prm, units, want)      # the program's own eager call between replays
            hs.sync()
            assert out.tolist() == want.tolist(), replay
            seeds = after
            assert states_of(states) == seeds, replay
    finally:
        torch.cuda.synchronize()
        hs.close()
