"""The work a user of the sampler has it do, as measurable cases: one call per pass (or the draft
chain's two), inputs and context in hand, through the package's public entry points.

A generation server holds the logits of the requests it decodes in HBM, one row per request, and asks
for one token per row and step (`Context.sample_batch`); a speculative decoder checks its k drafts on
k + 1 rows at once (`Context.verify`); a drafter takes the argmax and the embedding of its pick
(`argmax_rows` or `head_argmax`, then `embed_rows`); requests that ask for log-probabilities add
`logprobs`; the output head is `matvec`. Inputs, like the benchmark's workloads, are normal logits
with a Zipf bump over a random permutation of the vocabulary and Zipf histories over the same ranks.

Left out of the outputs, as a program leaves them out: the status word's bits above its low byte,
which only say which path settled a row; kept_count of a call without kept lists, which may be a lower
bound; and the device address that the draft pick also writes (the embedding read from it is there).
"""
import math

import numpy as np
import torch

from artemis_amd import WTYPE, Context, PackedSampling, Sampling, row_bytes, states_tensor

VOCAB = 248_320  # the benchmark's vocabulary
BLOCK = {"F32": (1, 4), "BF16": (1, 2), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}
SIGMA, BUMP = 2.5, 8.0
CAP = 256  # kept-list entries per row where a case asks for kept lists


def listed():
    return [
        # One request decoded greedily (temperature 0): the smallest call of a decode loop.
        dict(name="greedy_row", kind="sample", rows=1, vocab=VOCAB, hist=0, settings="greedy", kept=0),
        # One request with the package's default settings (T 0.6, top-k 20, top-p 0.95).
        dict(name="default_row", kind="sample", rows=1, vocab=VOCAB, hist=0, settings="default", kept=0),
        # One chat request deep into its answer: penalties over 4,096 ids, top-k, top-p and min-p.
        dict(name="penalised_row", kind="sample", rows=1, vocab=VOCAB, hist=4096, settings="penalised", kept=0),
        # One speculative step: five drafts checked on six rows, nucleus sampling.
        dict(name="verify_burst", kind="verify", k=5, vocab=VOCAB, hist=0, settings="nucleus"),
        # A full serving batch, every request with its own settings and a 2,048-id history.
        dict(name="serve_256", kind="sample", rows=256, vocab=VOCAB, hist=2048, settings="mixed", kept=0),
        # A small batch of odd width whose caller wants the kept sets and their probabilities.
        dict(name="kept_ragged_24", kind="sample", rows=24, vocab=100_003, hist=300, settings="mixed", kept=CAP),
        # A batch of plain sampling: temperature 1, no filter.
        dict(name="plain_256", kind="sample", rows=256, vocab=VOCAB, hist=0, settings="plain", kept=0),
        # Log-probabilities (the token's and the 20 best) of a full batch.
        dict(name="logprobs_256", kind="logprobs", rows=256, vocab=VOCAB, top=20),
        # ... and of one request's row.
        dict(name="logprobs_row", kind="logprobs", rows=1, vocab=VOCAB, top=20),
        # The output head's logits for one token, six-bit weights.
        dict(name="head_q6k", kind="matvec", wtype="Q6_K", rows=VOCAB, k=2048),
        # A greedy draft step: the head with its argmax fused, four-bit weights, and the pick's embedding.
        dict(name="draft_head_q4k", kind="draft", wtype="Q4_K", rows=VOCAB, k=2048),
        # A greedy draft step from logits that are there already: the argmax and the pick's embedding.
        dict(name="draft_argmax", kind="argmax", wtype="Q6_K", rows=1, vocab=VOCAB, k=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "verify", "logprobs", "matvec", "draft", "argmax"])
    vocab = rng.choice([VOCAB, _log_int(rng, 1000, VOCAB) | 1, _log_int(rng, 1000, VOCAB) // 4 * 4])
    if kind == "sample":
        settings = rng.choice(["greedy", "default", "penalised", "nucleus", "mixed", "mixed", "plain"])
        hist = 0 if settings == "plain" else rng.choice([0, _log_int(rng, 1, 6000)])
        kept = CAP if settings in ("default", "penalised", "mixed") and rng.random() < 0.3 else 0
        rows = _log_int(rng, 1, 256)
        return dict(kind=kind, rows=rows, vocab=vocab, hist=hist, settings=settings, kept=kept)
    if kind == "verify":
        return dict(kind=kind, k=rng.randint(1, 15), vocab=vocab, hist=rng.choice([0, _log_int(rng, 1, 6000)]),
                    settings=rng.choice(["nucleus", "default", "penalised", "greedy"]))
    if kind == "logprobs":
        return dict(kind=kind, rows=_log_int(rng, 1, 256), vocab=vocab, top=rng.choice([0, 1, 5, 20]))
    wtype = rng.choice(list(BLOCK))
    k = rng.choice([512, 1024, 1536, 2048, 2560, 4096])
    if kind == "argmax":
        return dict(kind=kind, wtype=wtype, rows=_log_int(rng, 1, 16), vocab=vocab, k=k)
    per, size = BLOCK[wtype]
    most = min(VOCAB, 417_000_000 // (k // per * size))
    return dict(kind=kind, wtype=wtype, rows=_log_int(rng, 256, most), k=k)


# ---- inputs -------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _logits(g, rows, vocab, hist):
    """[rows, vocab] f32 logits with a Zipf(1.1) bump, and (offsets, ids) of Zipf(1.2) histories of
    hist ids a row over the same ranks (None, None for none)."""
    dev = torch.device("cuda")
    x = torch.randn(rows, vocab, device=dev, generator=g) * SIGMA
    rank = torch.arange(1, vocab + 1, dtype=torch.float64, device=dev)
    bump = (BUMP * rank ** -1.1).float()
    cdf = torch.cumsum(rank ** -1.2, 0)
    ids = torch.empty(rows, hist, dtype=torch.int32, device=dev)
    for r in range(rows):
        perm = torch.randperm(vocab, device=dev, generator=g)
        x[r, perm] += bump
        if hist:
            u = torch.rand(hist, dtype=torch.float64, device=dev, generator=g) * cdf[-1]
            ids[r] = perm[torch.searchsorted(cdf, u).clamp_(max=vocab - 1)].int()
    if not hist:
        return x, None, None
    off = torch.arange(rows + 1, dtype=torch.int32, device=dev) * hist
    return x, off, ids.reshape(-1)


def _settings(case, seed):
    """A row's Sampling by name; `mixed` rows differ as the benchmark's full batch does."""
    rows = case.get("rows", 1) if case["kind"] == "sample" else 1
    name = case["settings"]
    one = {
        "greedy": Sampling(0.0, 0, 1.0, 0.0, 0.5 if case["hist"] else 0.0),
        "default": Sampling(0.6, 20, 0.95, 0.0, 0.5 if case["hist"] else 0.0),
        "penalised": Sampling(0.7, 40, 0.9, 0.05, 0.5, 0.3, 1.05),
        "nucleus": Sampling(0.6, 0, 0.95, 0.0, 0.5 if case["hist"] else 0.0),
        "plain": Sampling(1.0, 0, 1.0, 0.0),
    }
    if name != "mixed":
        return [one[name]] * rows
    rng = np.random.default_rng(seed)
    f = lambda v: float(np.float32(v))  # noqa: E731
    return [Sampling(f(rng.uniform(0.3, 1.0)), int(rng.choice([0, 20, 50])), f(rng.uniform(0.8, 1.0)),
                     f(rng.uniform(0.0, 0.1)), 0.5, f(0.3), f(1.05)) for _ in range(rows)]


def _f16_at(blocks, at, lo, hi, g):
    """Writes a random f16 scale in [lo, hi) at byte `at` of every block ([blocks, bytes] u8)."""
    d = (torch.rand(blocks.shape[0], device="cuda", generator=g) * (hi - lo) + lo).half()
    blocks[:, at:at + 2] = d.view(torch.uint8).view(-1, 2)


def _weights(g, wtype, rows, k):
    """[rows * row_bytes] u8: a table of weights of about 0.02 in size, as a trained layer's are."""
    dev = torch.device("cuda")
    if wtype == "F32":
        return (torch.randn(rows, k, device=dev, generator=g) * 0.02).view(torch.uint8).reshape(-1)
    if wtype == "BF16":
        return (torch.randn(rows, k, device=dev, generator=g) * 0.02).bfloat16().view(torch.uint8).reshape(-1)
    per, size = BLOCK[wtype]
    b = torch.randint(0, 256, (rows * (k // per), size), dtype=torch.uint8, device=dev, generator=g)
    if wtype == "Q8_0":
        _f16_at(b, 0, 1e-4, 4e-4, g)
    elif wtype == "Q6_K":
        _f16_at(b, 208, 1e-5, 4e-5, g)
    else:
        _f16_at(b, 0, 2e-5, 1e-4, g)
        _f16_at(b, 2, 2e-4, 1e-3, g)
    return b.reshape(-1)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case)
    dev = torch.device("cuda")
    if kind == "sample":
        s["x"], s["off"], s["ids"] = _logits(g, case["rows"], case["vocab"], case["hist"])
        s["params"] = PackedSampling(_settings(case, seed))
        s["rng"] = states_tensor(range(seed, seed + case["rows"]), dev)
        s["ctx"] = Context(max_rows=case["rows"], max_vocab=case["vocab"])
        s["out"] = s["ctx"].outputs(case["rows"], case["kept"])
        for t in s["out"]:
            t.zero_()  # a row writes the entries of its kept set only
        s["code"] = s["out"][1].view(torch.uint8).view(-1, 4)[:, 0]
    elif kind == "verify":
        s["x"], _, s["ids"] = _logits(g, case["k"] + 1, case["vocab"], case["hist"])
        if s["ids"] is not None:
            s["ids"] = s["ids"][:case["hist"]].contiguous()
        top = s["x"].argmax(dim=1).int()[:case["k"]]
        other = torch.randint(0, case["vocab"], (case["k"],), dtype=torch.int32, device=dev, generator=g)
        s["drafts"] = torch.where(torch.rand(case["k"], device=dev, generator=g) < 0.7, top, other).contiguous()
        s["stop"] = torch.randint(0, case["vocab"], (2,), dtype=torch.int32, device=dev, generator=g)
        s["params"] = _settings(case, seed)[0]
        s["rng"] = states_tensor([seed], dev)
        s["ctx"] = Context(max_rows=16, max_vocab=case["vocab"])
    elif kind == "logprobs":
        s["x"], _, _ = _logits(g, case["rows"], case["vocab"], 0)
        likely = s["x"].argmax(dim=1).int()
        other = torch.randint(0, case["vocab"], (case["rows"],), dtype=torch.int32, device=dev, generator=g)
        s["tok"] = torch.where(torch.rand(case["rows"], device=dev, generator=g) < 0.5, likely, other).contiguous()
        s["ctx"] = Context(max_rows=case["rows"], max_vocab=case["vocab"])
    elif kind in ("matvec", "draft"):
        s["w"] = _weights(g, case["wtype"], case["rows"], case["k"])
        s["h"] = torch.randn(case["k"], device=dev, generator=g)
        s["code"], s["rb"] = WTYPE[case["wtype"]], row_bytes(WTYPE[case["wtype"]], case["k"])
        s["ctx"] = Context(max_rows=16, max_vocab=4096)
        s["y"] = torch.empty(case["rows"], device=dev)
        s["id"] = torch.empty(1, dtype=torch.int32, device=dev)
        s["addr"] = torch.empty(1, dtype=torch.int64, device=dev)
    else:
        s["x"], _, _ = _logits(g, case["rows"], case["vocab"], 0)
        s["w"] = _weights(g, case["wtype"], case["vocab"], case["k"])
        s["code"], s["rb"] = WTYPE[case["wtype"]], row_bytes(WTYPE[case["wtype"]], case["k"])
        s["ctx"] = Context(max_rows=16, max_vocab=case["vocab"])
        s["id"] = torch.empty(case["rows"], dtype=torch.int32, device=dev)
        s["addr"] = torch.empty(case["rows"], dtype=torch.int64, device=dev)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "sample":
        tok, _, count, ids, probs = ctx.sample_batch(s["x"], s["params"], s["rng"], s["off"], s["ids"],
                                                     kept_cap=s["kept"], out=s["out"])
        res = dict(tokens=tok, status=s["code"], rng=s["rng"])
        if s["kept"]:
            res.update(kept_count=count, kept_ids=ids, kept_probs=probs)
        return res
    if kind == "verify":
        picks, result = ctx.verify(s["x"], s["drafts"], s["params"], s["rng"], s["ids"], s["stop"])
        return dict(picks=picks, result=result, rng=s["rng"])
    if kind == "logprobs":
        lp, ids, lps, st = ctx.logprobs(s["x"], s["tok"], s["top"])
        return dict(logprob=lp, top_ids=ids, top_logprobs=lps, status=st)
    if kind == "matvec":
        return ctx.matvec(s["w"], s["code"], s["rows"], s["k"], s["h"], s["y"])
    if kind == "draft":
        ctx.head_argmax(s["w"], s["code"], s["rows"], s["k"], s["h"], s["id"], s["addr"], s["w"].data_ptr(), s["rb"],
                        logits=s["y"])
        return dict(logits=s["y"], draft=s["id"], embedding=ctx.embed_rows(s["addr"], s["code"], s["k"]))
    ctx.argmax_rows(s["x"], s["id"], s["addr"], s["w"].data_ptr(), s["rb"])
    return dict(draft=s["id"], embedding=ctx.embed_rows(s["addr"], s["code"], s["k"]))


def work(case):
    kind = case["kind"]
    if kind == "sample":
        n = case["rows"] * case["vocab"]
        out = 40 + (12 * 64 if case["kept"] else 0)
        return dict(bytes=4 * n + 4 * case["rows"] * case["hist"] + case["rows"] * (32 + out), flops=n)
    if kind == "verify":
        n = (case["k"] + 1) * case["vocab"]
        return dict(bytes=4 * n + 4 * case["hist"] + 8 * case["k"] + 100, flops=n)
    if kind == "logprobs":
        n = case["rows"] * case["vocab"]
        return dict(bytes=4 * n + case["rows"] * (12 + 8 * case["top"]), flops=n)
    per, size = BLOCK[case["wtype"]]
    rb = case["k"] // per * size
    if kind == "argmax":
        n = case["rows"] * case["vocab"]
        return dict(bytes=4 * n + case["rows"] * (rb + 4 * case["k"] + 12), flops=n)
    b = case["rows"] * (rb + 4) + 4 * case["k"] + (rb + 4 * case["k"] + 12 if kind == "draft" else 0)
    return dict(bytes=b, flops=2 * case["rows"] * case["k"])


def tolerance(case):
    # Log-probabilities are f64 sums rounded once to f32, kept probabilities f64 quotients of the same
    # terms: another correct order moves the first by an ulp here and there and the second by 1e-11.
    if case["kind"] == "logprobs":
        return {"rel": 1e-7, "max": 1e-6}
    if case["kind"] == "sample" and case["kept"]:
        return {"rel": 1e-10, "max": 1e-8}
    # Tokens, streams, logits and embeddings are promised bit for bit.
    return "exact"


# ---- the same in 64 bits ------------------------------------------------------------------------

def _dequant(w, wtype, rows, k):
    """f64 [rows, k] of a table's bytes ([rows * row_bytes] u8), by the block layouts' definition."""
    if wtype == "F32":
        return w.view(torch.float32).view(rows, k).double()
    if wtype == "BF16":
        return w.view(torch.bfloat16).view(rows, k).double()
    per, size = BLOCK[wtype]
    b = w.view(-1, size)
    h = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if wtype == "Q8_0":
        return (h(0) * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, k)
    if wtype == "Q6_K":
        ql, qh = b[:, :128].view(-1, 2, 2, 32).int(), b[:, 128:192].view(-1, 2, 1, 32).int()
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        parts = []
        for m in range(4):
            lo = (ql[:, :, m & 1] >> (4 * (m >> 1))) & 15
            parts.append((lo | (((qh[:, :, 0] >> (2 * m)) & 3) << 4)) - 32)
        q = torch.stack(parts, 2).double().view(-1, 16, 16)
        return (h(208).unsqueeze(2) * sc.unsqueeze(2) * q).reshape(rows, k)
    s = b[:, 4:16].int()
    scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double()
    least = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
    qs = b[:, size - 128:].view(-1, 4, 1, 32).int()
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if wtype == "Q5_K":
        bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
        q = q + (((b[:, 16:48].int().unsqueeze(1) >> bit) & 1) << 4)
    return ((h(0) * scale).unsqueeze(2) * q.double() - (h(2) * least).unsqueeze(2)).reshape(rows, k)


def _head64(s):
    y = torch.empty(s["rows"], dtype=torch.float64, device="cuda")
    step = 1 << 14
    for r in range(0, s["rows"], step):
        m = min(step, s["rows"] - r)
        y[r:r + m] = _dequant(s["w"][r * s["rb"]:(r + m) * s["rb"]], s["wtype"], m, s["k"]) @ s["h"].double()
    return y


def _kept64(s, settings):
    """The kept set's probabilities of every row, [rows, CAP] f64 (0 past the set)."""
    out = np.zeros((s["rows"], CAP))
    for r, p in enumerate(settings):
        x = s["x"][r].cpu().numpy()
        if s["ids"] is not None:
            ids, c = np.unique(s["ids"].view(s["rows"], -1)[r].cpu().numpy(), return_counts=True)
            v, f = x[ids], np.float32
            if p.repetition_penalty != 1.0:
                v = np.where(v > 0, v / f(p.repetition_penalty), v * f(p.repetition_penalty))
            x[ids] = v - (c.astype(f) * f(p.frequency_penalty) + f(p.presence_penalty))
        v = -np.sort(-x).astype(np.float64)
        if 0 < p.top_k < len(v):
            v = v[:p.top_k]
        top = v[0]
        keep = len(v)
        if p.top_p < 1.0:
            w = np.exp(v - top)
            keep = min(keep, int(np.searchsorted(np.cumsum(w) / w.sum(), float(np.float32(p.top_p)))) + 1)
        v = v[:keep]
        if p.min_p > 0.0:
            v = v[v >= top + math.log(float(np.float32(p.min_p)))]
        w = np.exp((v - top) / float(np.float32(p.temp)))
        w = (w / w.sum())[:CAP]
        out[r, :len(w)] = w
    return torch.from_numpy(out)


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "sample":
        res = dict(tokens=None, status=None, rng=None)
        if case["settings"] == "greedy" and not case["hist"]:
            res["tokens"] = s["x"].argmax(dim=1).int()
        if case["kept"]:
            res.update(kept_count=None, kept_ids=None, kept_probs=_kept64(s, _settings(case, seed)))
        return res if any(v is not None for v in res.values()) else None
    if kind == "verify":
        return None
    if kind == "logprobs":
        n = min(case["top"], 20, case["vocab"])
        lp = torch.empty(case["rows"], dtype=torch.float64)
        ids = torch.full((case["rows"], max(case["top"], 1)), -1, dtype=torch.int32)
        lps = torch.full((case["rows"], max(case["top"], 1)), float("nan"), dtype=torch.float64)
        for r in range(case["rows"]):
            x = s["x"][r].double()
            lse = torch.logsumexp(x, 0)
            lp[r] = x[s["tok"][r].long()] - lse
            if n:
                v, i = torch.sort(x, descending=True, stable=True)  # ties to the lower id
                ids[r, :n], lps[r, :n] = i[:n].int().cpu(), (v[:n] - lse).cpu()
        return dict(logprob=lp, top_ids=ids, top_logprobs=lps, status=None)
    if kind == "matvec":
        return _head64(s)
    if kind == "draft":
        # The pick is the argmax of the 32-bit logits, which 64-bit ones need not share; its embedding too.
        return dict(logits=_head64(s), draft=None, embedding=None)
    ids = s["x"].argmax(dim=1)
    row = torch.stack([s["w"][i * s["rb"]:(i + 1) * s["rb"]] for i in ids.tolist()])
    return dict(draft=ids.int(), embedding=_dequant(row.reshape(-1), case["wtype"], case["rows"], case["k"]))
