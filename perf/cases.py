"""The work this library is called for, as measurable cases: a decode step's draw from logits that
are already on the device (one row up to a batch of 256), the verification of drafted tokens, and
the tail of a forward pass (output norm, lm_head over each table format, draw).

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` one more of the same
ranges; `prepare` makes what a program holds before a call, `run` is one call through the public
entry points, `work` the bytes and operations it cannot do without, `tolerance` how far two correct
implementations may differ.
"""
import math

import torch

from geistlib_amd import HipSampler, SampleParams

RMS_EPS = 1e-6
SKETCH_WIDTHS = {1536: 768, 2048: 1024, 2560: 640, 3072: 768}   # d_model -> kept dimensions
TABLE_BYTES_PER_BLOCK = {"f16": 512, "q8w": 256, "q6k": 210, "q4k": 144}   # per 256 weights
MOST_LOGITS = 256 * 262144
MOST_VERIFY_LOGITS = 32 * 9 * 128256
MOST_TABLE = {"f16": 128256 * 2560, "q8w": 128256 * 2560, "q6k": 262144 * 1536,
              "q4k": 262144 * 1536}


def _sample(name, rows, vocab, logits, temperature, top_k=0, top_p=1.0, min_p=0.0, history=0,
            softcap=0.0, mask=False, device_rng=False):
    case = {"kind": "sample", "rows": rows, "vocab": vocab, "logits": logits,
            "temperature": temperature, "top_k": top_k, "top_p": top_p, "min_p": min_p,
            "history": history, "softcap": softcap, "mask": mask, "device_rng": device_rng}
    return {"name": name, **case} if name else case


def _verify(name, seqs, drafts, vocab, temperature, point_mass):
    case = {"kind": "verify", "seqs": seqs, "drafts": drafts, "vocab": vocab,
            "temperature": temperature, "point_mass": point_mass}
    return {"name": name, **case} if name else case


def _head(name, table, rows, vocab, d_model, temperature, top_k=0, top_p=1.0, softcap=0.0):
    case = {"kind": "head", "table": table, "rows": rows, "vocab": vocab, "d_model": d_model,
            "temperature": temperature, "top_k": top_k, "top_p": top_p, "softcap": softcap}
    return {"name": name, **case} if name else case


def _sketch(name, vocab, d_model):
    case = {"kind": "sketch", "vocab": vocab, "d_model": d_model}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one session, a vocabulary of 32000, plain temperature (the default of a session): the
        # smallest call, where the launch and the chain of waits are the cost
        _sample("token_1x32000", 1, 32000, "normal", 0.8, device_rng=True),
        # one session's decode step with every filter and penalties over 2048 tokens of context
        _sample("step_1x128256", 1, 128256, "boosted", 0.7, top_k=40, top_p=0.9, history=2048,
                device_rng=True),
        # a serving batch with the same options: the library's headline configuration
        _sample("batch_64x128256", 64, 128256, "boosted", 0.7, top_k=40, top_p=0.9, history=2048),
        # the largest batch and vocabulary, heavy-tailed logits, top-k 64 into top-p
        _sample("batch_256x262144", 256, 262144, "student", 0.6, top_k=64, top_p=0.9),
        # nucleus and min-p over the whole vocabulary with penalties: every logit is weighed
        _sample("minp_128x151936", 128, 151936, "normal", 1.0, top_p=0.95, min_p=0.05,
                history=2048),
        # nucleus sampling at temperature 1 over a vocabulary of odd size (rows that are not 16-byte
        # aligned), rows from sharply peaked to nearly flat as a mixed batch has them
        _sample("topp_24x50257", 24, 50257, "mixed", 1.0, top_p=0.95),
        # speculative decoding: 8 drafted tokens for each of 32 sequences, rejection sampling
        # against the draft model's probabilities
        _verify("verify_32x8x128256", 32, 8, 128256, 1.0, False),
        # tail of one session's decode step over the tied table in int8 form
        _head("head_q8w_1x128256", "q8w", 1, 128256, 2560, 0.7, top_k=40, top_p=0.9),
        # greedy verify pass over the F16 table: 8 hidden rows at once
        _head("head_f16_8x128256", "f16", 8, 128256, 2560, 0.0),
        # tail of one session's decode step over a Q6_K table with a soft-cap
        _head("head_q6k_1x262144", "q6k", 1, 262144, 1536, 0.7, top_k=40, top_p=0.9, softcap=30.0),
        # verify pass of 8 rows over a Q4_K table with a soft-cap
        _head("head_q4k_8x262144", "q4k", 8, 262144, 1536, 0.7, top_k=40, top_p=0.9, softcap=30.0),
        # greedy decode step through the sketch of the F16 table
        _sketch("sketch_1x128256", 128256, 2560),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_vocab(rng, low, high):
    v = _log_int(rng, low, high)
    return v if rng.random() < 0.5 else max(low, v // 64 * 64)


def draw(rng):
    pick = rng.random()
    if pick < 0.5:
        vocab = _draw_vocab(rng, 32000, 262144)
        rows = _log_int(rng, 1, 256)
        rows = max(1, min(rows, MOST_LOGITS // vocab))
        mode = rng.choice(["greedy", "temperature", "topk", "topk", "topp", "minp"])
        return _sample(
            None, rows, vocab, rng.choice(["normal", "boosted", "student", "mixed"]),
            0.0 if mode == "greedy" else round(rng.uniform(0.5, 1.2), 2),
            top_k=_log_int(rng, 5, 200) if mode == "topk" else 0,
            top_p=round(rng.uniform(0.7, 0.98), 2) if mode in ("topk", "topp", "minp") else 1.0,
            min_p=round(rng.uniform(0.02, 0.1), 3) if mode == "minp" else 0.0,
            history=_log_int(rng, 64, 4096) if rng.random() < 0.5 else 0,
            softcap=30.0 if rng.random() < 0.2 else 0.0, mask=rng.random() < 0.15,
            device_rng=mode != "greedy" and rng.random() < 0.5)
    if pick < 0.65:
        vocab = _draw_vocab(rng, 32000, 151936)
        drafts = rng.randint(1, 8)
        seqs = max(1, min(_log_int(rng, 1, 32), MOST_VERIFY_LOGITS // (vocab * (drafts + 1))))
        return _verify(None, seqs, drafts, vocab, round(rng.uniform(0.6, 1.2), 2),
                       rng.random() < 0.3)
    if pick < 0.92:
        table = rng.choice(["f16", "q8w", "q6k", "q4k"])
        d_model = 256 * rng.randint(4, 12)
        vocab = _log_int(rng, 32000, min(262144, MOST_TABLE[table] // d_model))
        vocab = vocab // 8 * 8 if rng.random() < 0.8 else vocab
        return _head(None, table, rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 7, 8]), vocab, d_model,
                     rng.choice([0.0, 0.7, 1.0]), top_k=rng.choice([0, 40, 64]),
                     top_p=rng.choice([1.0, 0.9]), softcap=rng.choice([0.0, 30.0]))
    d_model = rng.choice(sorted(SKETCH_WIDTHS))
    most = min(199999, MOST_TABLE["f16"] // d_model)
    return _sketch(None, _log_int(rng, 65536, most) // 8 * 8, d_model)


def _logits(case, dev, g):
    rows, vocab = case["rows"], case["vocab"]
    x = torch.randn((rows, vocab), device=dev, generator=g)
    kind = case["logits"]
    if kind == "student":       # nu = 3
        chi = sum(torch.randn((rows, vocab), device=dev, generator=g) ** 2 for _ in range(3))
        return x / torch.sqrt(chi / 3.0) * 2.5
    x *= 2.0
    if kind == "boosted":       # a handful of likely tokens
        at = torch.randint(0, vocab, (rows, 5), device=dev, generator=g)
        x.scatter_add_(1, at, torch.full((rows, 5), 10.0, device=dev))
    elif kind == "mixed":       # likely tokens that fall off with their rank, from a row's own peak
        peak = 10.0 + 12.0 * torch.rand((rows, 1), device=dev, generator=g)
        lead = peak - 1.8 * torch.log(torch.arange(1, 513, device=dev, dtype=torch.float32))
        at = torch.argsort(torch.rand((rows, 8192), device=dev, generator=g), dim=1)
        x.scatter_(1, at[:, :512] * (vocab // 8192), lead)
    return x


def _history(case, dev, g):
    """Token ids of the context, Zipf-distributed as running text is."""
    rows, vocab, n = case["rows"], case["vocab"], case["history"]
    cdf = torch.arange(1, vocab + 1, device=dev, dtype=torch.float64).pow(-1.1).cumsum(0)
    at = torch.rand((rows, n), device=dev, generator=g, dtype=torch.float64) * cdf[-1]
    ids = torch.searchsorted(cdf, at).clamp_(max=vocab - 1).to(torch.int32)
    return ids, torch.full((rows,), n, dtype=torch.int32, device=dev)


def _params(case):
    penalised = case.get("history", 0) > 0
    return SampleParams.make(temperature=case["temperature"], top_k=case["top_k"],
                             top_p=case["top_p"], min_p=case.get("min_p", 0.0),
                             rep=1.1 if penalised else 1.0, freq=0.5 if penalised else 0.0,
                             pres=0.3 if penalised else 0.0, softcap=case["softcap"])


def _prepare_sample(case, dev, g):
    rows, vocab = case["rows"], case["vocab"]
    s = {"sampler": HipSampler(max_rows=rows, max_vocab=vocab), "params": _params(case)}
    s["sampler"].prepare(s["params"], vocab)
    s["logits"] = _logits(case, dev, g)
    history = _history(case, dev, g) if case["history"] else (None, None)
    mask = None
    if case["mask"]:            # a grammar that allows about half of the vocabulary
        mask = torch.randint(-2 ** 31, 2 ** 31, (1, (vocab + 31) // 32), device=dev, generator=g)
        mask = mask.to(torch.int32)
    s["keep"] = (history, mask)
    s["rows"] = HipSampler.rows(s["logits"], history[0], history[1], allowed=mask)
    s["uniforms"] = torch.rand((rows,), device=dev, generator=g)
    s["out"] = torch.empty((rows,), dtype=torch.int32, device=dev)
    if case["device_rng"]:      # every row its session's own generator
        s["states"] = torch.randint(1, 2 ** 62, (rows,), device=dev, generator=g)
    return s


def _prepare_verify(case, dev, g):
    n, drafts, vocab = case["seqs"], case["drafts"], case["vocab"]
    target = torch.randn((n, drafts + 1, vocab), device=dev, generator=g) * 2
    noisy = target[:, :drafts] + torch.randn((n, drafts, vocab), device=dev, generator=g) * 0.5
    q = torch.softmax(noisy / case["temperature"], dim=-1)
    draft = torch.searchsorted(q.cumsum(-1, dtype=torch.float64),
                               torch.rand((n, drafts, 1), device=dev, generator=g).double() * 0.999)
    return {"sampler": HipSampler(max_rows=n * (drafts + 1), max_vocab=vocab), "target": target,
            "q": None if case["point_mass"] else q,
            "draft": draft[..., 0].clamp_(max=vocab - 1).to(torch.int32).contiguous(),
            "uniforms": torch.rand((n, drafts + 1), device=dev, generator=g),
            "temperature": case["temperature"],
            "tokens": torch.full((n, drafts + 1), -1, dtype=torch.int32, device=dev),
            "accepted": torch.full((n,), -1, dtype=torch.int32, device=dev)}


def _f16_table(vocab, d_model, dev, g):
    t = torch.empty((vocab, d_model), dtype=torch.float16, device=dev)
    return t.normal_(0.0, 0.05, generator=g)


def _block_table(kind, vocab, d_model, dev, g):
    """Super-blocks as a model file holds them, scaled so that logits are a few units wide."""
    nb, size = d_model // 256, TABLE_BYTES_PER_BLOCK[kind]
    t = torch.randint(-2 ** 31, 2 ** 31, ((vocab * nb * size + 3) // 4,), device=dev, generator=g,
                      dtype=torch.int32)
    t = t.view(torch.uint8)[:vocab * nb * size].view(vocab, nb, size)
    if kind == "q6k":
        t[:, :, 192:208] &= 0x0F
        t[:, :, 208], t[:, :, 209] = 0x6D, 0x0C
    else:
        t[:, :, 0], t[:, :, 1] = 0x6D, 0x0C
        t[:, :, 2], t[:, :, 3] = 0x6D, 0x18
    return t.reshape(vocab, nb * size)


def _hidden(rows, d_model, dev, g):
    x = torch.randn((rows, d_model), device=dev, generator=g) * 3
    return x, 1.0 + 0.1 * torch.randn((d_model,), device=dev, generator=g)


def _prepare_head(case, dev, g):
    rows, vocab, d_model, kind = case["rows"], case["vocab"], case["d_model"], case["table"]
    hs = HipSampler(max_rows=rows, max_vocab=vocab)
    s = {"sampler": hs, "params": _params(case), "table_kind": kind, "vocab": vocab}
    hs.prepare(s["params"], vocab)
    if kind == "f16":
        s["table"] = _f16_table(vocab, d_model, dev, g)
    elif kind == "q8w":
        f16 = _f16_table(vocab, d_model, dev, g)
        s["table"] = torch.empty((vocab, d_model), dtype=torch.int8, device=dev)
        s["scales"] = torch.empty((vocab,), dtype=torch.float32, device=dev)
        hs.f16_to_q8w(f16, s["table"], s["scales"])
    else:
        blocks = _block_table(kind, vocab, d_model, dev, g)
        size, pack = ((hs.q6k_packed_bytes, hs.q6k_pack) if kind == "q6k" else
                      (hs.q4k_packed_bytes, hs.q4k_pack))
        s["table"] = torch.empty((size(vocab, d_model),), dtype=torch.uint8, device=dev)
        pack(blocks, d_model, s["table"])
    s["hidden"], s["norm_w"] = _hidden(rows, d_model, dev, g)
    s["normed"] = torch.empty_like(s["hidden"])
    s["logits"] = torch.empty((rows, vocab), dtype=torch.float32, device=dev)
    s["uniforms"] = torch.rand((rows,), device=dev, generator=g)
    s["out"] = torch.empty((rows,), dtype=torch.int32, device=dev)
    return s


class _SketchHead:
    """A built sketch head and its sampler, given back together."""

    def __init__(self, sampler, table):
        self.sampler, self.handle = sampler, sampler.spec_head_build(table)

    def __del__(self):
        self.sampler.spec_head_destroy(self.handle)


def _prepare_sketch(case, dev, g):
    hs = HipSampler(max_rows=1, max_vocab=case["vocab"])
    table = _f16_table(case["vocab"], case["d_model"], dev, g)
    s = {"sampler": hs, "head": _SketchHead(hs, table), "table": table}
    s["hidden"], s["norm_w"] = _hidden(1, case["d_model"], dev, g)
    s["normed"] = torch.empty_like(s["hidden"])
    s["result"] = torch.zeros((6,), dtype=torch.int32, device=dev)
    return s


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    s = {"sample": _prepare_sample, "verify": _prepare_verify, "head": _prepare_head,
         "sketch": _prepare_sketch}[case["kind"]](case, dev, g)
    s["kind"] = case["kind"]
    return s


def run(state):
    s, hs = state, state["sampler"]
    if s["kind"] == "sample":
        if "states" in s:
            hs.sample_rng(s["rows"], s["params"], s["states"], False, s["out"])
            return s["out"], s["states"]
        hs.sample(s["rows"], s["params"], s["uniforms"], s["out"])
        return s["out"]
    if s["kind"] == "verify":
        hs.spec_verify(s["target"], s["q"], s["draft"], s["uniforms"], s["temperature"],
                       s["tokens"], s["accepted"])
        return s["tokens"], s["accepted"]
    if s["kind"] == "sketch":
        hs.spec_head_try_hidden(s["head"].handle, s["hidden"], s["norm_w"], RMS_EPS, s["normed"],
                                s["result"])
        r = s["result"]         # r[3] counts the rows looked at on the way, a diagnostic
        return r[:3], r[4:].view(torch.float32), s["normed"]
    args = (s["hidden"], s["norm_w"], RMS_EPS, s["table"])
    tail = (s["logits"], s["params"], s["uniforms"], s["out"], s["normed"])
    if s["table_kind"] == "f16":
        hs.project_sample(*args, *tail)
    elif s["table_kind"] == "q8w":
        hs.project_sample_q8w(*args, s["scales"], *tail)
    elif s["table_kind"] == "q6k":
        hs.project_sample_q6k_packed(*args, s["vocab"], *tail)
    else:
        hs.project_sample_q4k_packed(*args, s["vocab"], *tail)
    return s["out"], s["logits"], s["normed"]


def work(case):
    vocab = case["vocab"]
    if case["kind"] == "sample":
        n = case["rows"] * vocab
        extra = case["rows"] * (8 + 4 * case["history"] + 16 * case["device_rng"])
        extra += case["mask"] * vocab // 8
        return {"bytes": 4 * n + extra, "flops": 2 * n}
    if case["kind"] == "verify":
        rows = case["seqs"] * (case["drafts"] + 1)
        q_rows = 0 if case["point_mass"] else case["seqs"]    # of the position that is rejected
        return {"bytes": 4 * vocab * (rows + q_rows) + 12 * rows, "flops": 2 * rows * vocab}
    d_model = case["d_model"]
    if case["kind"] == "sketch":
        width = SKETCH_WIDTHS[d_model]
        return {"bytes": vocab * (width + 4) + 1024 * 2 * d_model + 12 * d_model,
                "flops": 2 * vocab * width + 2 * 1024 * d_model}
    rows = case["rows"]
    table = vocab * d_model // 256 * TABLE_BYTES_PER_BLOCK[case["table"]]
    table += 4 * vocab if case["table"] == "q8w" else 0
    return {"bytes": table + 4 * rows * (vocab + 2 * d_model) + 4 * d_model,
            "flops": 2 * rows * vocab * d_model}


def tolerance(case):
    """Tokens, acceptance counts and generator states are whole numbers, and the logits and normed
    rows are those of a fixed order of summation, bit for bit."""
    return "exact"
