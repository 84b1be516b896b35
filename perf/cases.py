"""Performance cases of the speculative-verification hot path on one MI355X.

Each case is one call (or one whole verify round) through the package's public entry
points, on inputs of the kind the engine hands them:

* ``attend``: one layer's attention over a paged KV pool -- per-row decode, a verify
  window stored and attended in one call, pipelined rows at their loop-depth planes, and
  prompts (whole or a chunk after a cached prefix);
* ``accept``: the stochastic verify round, from target logits to committed tokens;
* ``draft``: one draft offset (argmax, distributions and draws);
* ``round``: a whole verify round of a small mixed batch.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges;
``prepare`` makes a case's inputs from a seed, ``run`` is the timed pass, ``work`` what it
cannot do without, ``exact`` the same outputs in float64 by plain torch.
"""

import importlib.util
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The framework: the directory vllm-rlt_amd, imported as ``vllm_rlt_amd``."""
    if "vllm_rlt_amd" not in sys.modules:
        path = os.path.join(_ROOT, "vllm-rlt_amd")
        spec = importlib.util.spec_from_file_location(
            "vllm_rlt_amd", os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        module = importlib.util.module_from_spec(spec)
        sys.modules["vllm_rlt_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["vllm_rlt_amd"]


_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_FP8 = torch.float8_e4m3fn
_DEV = "cuda"


# ------------------------------------------------------------------------------- cases

def _attend(name, form, batch, ctx, q_len, heads, dim, kv="same", dtype="bf16", window=0,
            layers=2):
    """``ctx`` and ``q_len``: (lowest, highest) per sequence, uniform; ``ctx`` counts the
    window rows.  ``kv``: "same" (the pool in q's type), "fp8" (per-tensor scales) or
    "fp8_vector" (one scale per token and kv head)."""
    return {"name": name, "kind": "attend", "form": form, "batch": batch, "ctx_lo": ctx[0],
            "ctx_hi": ctx[1], "q_lo": q_len[0], "q_hi": q_len[1], "heads": heads[0],
            "kv_heads": heads[1], "dim": dim, "kv": kv, "dtype": dtype, "window": window,
            "layers": layers}


def _accept(name, n, w1, vocab, temperature, top_p, top_k, logits="fp32"):
    """``top_p`` / ``top_k``: "none" or "all" (every request the same) or "mixed"."""
    return {"name": name, "kind": "accept", "n": n, "w1": w1, "vocab": vocab,
            "temperature": temperature, "top_p": top_p, "top_k": top_k, "logits": logits}


def listed():
    return [
        # one request generating token by token: one attention launch of one layer
        _attend("decode_1", "decode", 1, (700, 700), (1, 1), (16, 16), 128),
        # the decode batch: 16 / 16 heads, contexts up to 4096
        _attend("decode_64", "decode", 64, (512, 4096), (1, 1), (16, 16), 128),
        # the verify window of 4 drafts, stored and attended, GQA 4, contexts up to 8192
        _attend("verify_32", "store", 32, (1024, 8192), (5, 5), (16, 4), 128),
        # wide heads of an odd count and a head size that is no power of two
        _attend("verify_wide_16", "store", 16, (2048, 2048), (5, 5), (55, 55), 96),
        # long contexts in fp8, each window row at its loop-depth plane
        _attend("verify_planes_fp8_64", "planes", 64, (16384, 32768), (5, 5), (16, 8), 128,
                kv="fp8", layers=1),
        # whole prompts into an empty cache
        _attend("prompts_8", "store", 8, (2048, 2048), (2048, 2048), (16, 4), 128),
        # ragged prompt chunks behind a cached prefix, fp8 pool with a scale per vector
        _attend("chunks_fp8_6", "store", 6, (700, 3000), (300, 640), (16, 8), 128,
                kv="fp8_vector"),
        # the verify round: T = 0.7, top-p 0.9, 32 requests of 4 drafts
        _accept("accept_32", 32, 4, 49152, 0.7, "all", "none"),
        # a large batch sampled without truncation
        _accept("accept_plain_128", 128, 4, 65536, 1.0, "none", "none"),
        # a large vocabulary, bf16 logits, each request with its own top-k and top-p
        _accept("accept_mixed_16", 16, 4, 151936, 0.8, "mixed", "mixed", logits="bf16"),
        # one draft offset of the same requests as accept_32
        {"name": "draft_32", "kind": "draft", "rows": 32, "random": 32, "vocab": 49152,
         "temperature": 0.7, "top_p": "all", "top_k": "none", "logits": "fp32"},
        # one whole round of a few requests, one of them greedy
        {"name": "round_4", "kind": "round", "n": 4, "random": 3, "w1": 4, "vocab": 49152,
         "ctx_lo": 512, "ctx_hi": 2048, "heads": 16, "kv_heads": 4, "dim": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges; none costs more than the largest listed one."""
    kind = rng.choice(("decode", "decode", "verify", "verify", "planes", "prompt", "prompt",
                       "accept", "accept", "accept", "draft", "draft", "round"))
    if kind in ("accept", "draft", "round"):
        vocab = _log(rng, 8000, 152000)
        top_p, top_k = rng.choice((("none", "none"), ("all", "none"), ("mixed", "none"),
                                   ("none", "all"), ("mixed", "mixed")))
        temperature = rng.choice((0.7, 0.8, 1.0))
        logits = rng.choice(("fp32", "fp32", "bf16"))
        if kind == "accept":
            w1 = rng.randint(1, 8)
            n = min(_log(rng, 1, 128), 42_000_000 // (vocab * (w1 + 1)))
            return {k: v for k, v in _accept("", max(1, n), w1, vocab, temperature, top_p, top_k,
                                             logits).items() if k != "name"}
        if kind == "draft":
            rows = min(_log(rng, 1, 256), 42_000_000 // vocab)
            return {"kind": "draft", "rows": rows, "random": rng.randint((rows + 1) // 2, rows),
                    "vocab": vocab, "temperature": temperature, "top_p": top_p, "top_k": top_k,
                    "logits": logits}
        n = rng.randint(1, 8)
        hi = _log(rng, 128, 4096)
        return {"kind": "round", "n": n, "random": rng.randint(1, n), "w1": rng.randint(1, 6),
                "vocab": vocab, "ctx_lo": max(8, hi // 4), "ctx_hi": hi, "heads": 16,
                "kv_heads": rng.choice((4, 8, 16)), "dim": rng.choice((64, 96, 128))}
    heads = rng.choice(((16, 16), (16, 4), (16, 8), (32, 8), (55, 55)))
    dim = rng.choice((64, 96, 128, 128))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    kv = rng.choice(("same", "same", "fp8", "fp8_vector"))
    size = (heads[1] * dim * (2 if kv == "same" else 1))  # bytes of one position's keys
    if kind == "prompt":
        q_hi = _log(rng, 64, 4096)
        ctx_hi = q_hi + rng.choice((0, rng.randint(1, 4096)))
        rows = min(16384, int(3.4e10 / (heads[0] * dim * ctx_hi)))
        batch = max(1, min(rng.randint(1, 12), rows // q_hi))
        q_lo = q_hi if rng.random() < 0.3 else max(33, q_hi // 2)
        case = _attend("", "store", batch, (max(q_hi, (q_hi + ctx_hi) // 2), ctx_hi),
                       (q_lo, q_hi), heads, dim, kv, dtype)
    elif kind == "planes":
        ctx_hi = _log(rng, 512, 32768)
        batch = max(1, min(_log(rng, 2, 64), int(8e9 / (8 * size * ctx_hi))))
        w = rng.randint(2, 8)
        case = _attend("", "planes", batch, (max(16, ctx_hi // 2), ctx_hi), (w, w), heads, dim,
                       kv, dtype, layers=1)
    else:
        ctx_hi = _log(rng, 64, 16384)
        batch = max(1, min(_log(rng, 1, 96), int(1.5e9 / (2 * size * ctx_hi))))
        ctx = (max(16, ctx_hi // rng.choice((1, 4, 8))), ctx_hi)
        if kind == "decode":
            window = rng.choice((0, 0, 0, 1024))
            case = _attend("", "decode", batch, ctx, (1, 1), heads, dim, kv, dtype, window)
        else:
            w = rng.randint(2, 9)
            case = _attend("", "store", batch, ctx, (rng.choice((1, w)), w), heads, dim, kv,
                           dtype)
    del case["name"]
    return case


# ------------------------------------------------------------------------------ inputs

_BLOCK = 16
_PLANES = 4
_SCALE = 5.0 / 448.0  # a per-tensor scale that covers N(0, 1) values


def _rand_codes(shape, g):
    """fp8 codes of N(0, 1) values over _SCALE, filled in pieces."""
    out = torch.empty(shape, dtype=_FP8, device=_DEV)
    flat = out.view(-1)
    step = 1 << 28
    for i in range(0, flat.numel(), step):
        m = min(step, flat.numel() - i)
        x = torch.randn(m, generator=g, device=_DEV, dtype=torch.float16)
        flat[i:i + m] = x.mul_(1.0 / _SCALE).clamp_(-448, 448).to(_FP8)
    return out


def _pool(case, blocks, g):
    """Key and value pools [block, layer, token, kv_head, dim], one layer's views, and the
    scales of an fp8 pool."""
    shape = (blocks, case["layers"], _BLOCK, case["kv_heads"], case["dim"])
    if case["kv"] == "same":
        dt = _DTYPES[case["dtype"]]
        k, v = (torch.randn(shape, generator=g, device=_DEV, dtype=dt) for _ in range(2))
        ks = vs = None
    else:
        k, v = _rand_codes(shape, g), _rand_codes(shape, g)
        if case["kv"] == "fp8":
            ks, vs = (torch.tensor(_SCALE * s, device=_DEV) for s in (1.0, 0.9))
        else:
            ks, vs = ((torch.rand(shape[:-1], generator=g, device=_DEV) * 0.5 + 0.75).mul_(
                _SCALE)[:, -1] for _ in range(2))
    return k[:, -1], v[:, -1], ks, vs


def _attend_inputs(case, seed):
    h = torch.Generator().manual_seed(seed)
    g = torch.Generator(device=_DEV).manual_seed(seed)
    n, bs = case["batch"], _BLOCK
    dt = _DTYPES[case["dtype"]]
    # the window lengths belong to the case (outputs keep their shapes), the rest to the seed
    q_len = torch.randint(case["q_lo"], case["q_hi"] + 1, (n,),
                          generator=torch.Generator().manual_seed(n))
    q_len[0] = case["q_hi"]
    ctx = torch.maximum(torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (n,), generator=h),
                        q_len)
    width = -(-max(case["ctx_hi"], case["q_hi"]) // bs)
    s = {"case": case}
    if case["form"] == "planes":
        # window row j of a request reads the table of plane (d0 + j) mod planes; rows of
        # one plane are one packed sequence with their own lengths
        w = case["q_hi"]
        d0 = torch.randint(0, _PLANES, (n,), generator=h)
        tables = torch.randperm(n * _PLANES * width, generator=h).int().view(n, _PLANES, width)
        cu, seq, rows, max_q = [0], [], [], 0
        for i in range(n):
            for p in range(_PLANES):
                mine = [j for j in range(w) if (int(d0[i]) + j) % _PLANES == p]
                if mine:
                    seq.append((i, p, int(ctx[i]) - w + mine[-1] + 1))
                    rows += [int(ctx[i]) - w + j + 1 for j in mine]
                    cu.append(len(rows))
                    max_q = max(max_q, len(mine))
        s["tables"] = torch.stack([tables[i, p] for i, p, _ in seq]).to(_DEV)
        s["lengths"] = torch.tensor([c for _, _, c in seq], dtype=torch.int32, device=_DEV)
        s["row_lengths"] = torch.tensor(rows, dtype=torch.int32, device=_DEV)
        total, blocks = len(rows), n * _PLANES * width
    else:
        cu = [0] + torch.cumsum(q_len, 0).tolist()
        tables = torch.randperm(n * width, generator=h).int().view(n, width)
        s["tables"], s["lengths"] = tables.to(_DEV), ctx.int().to(_DEV)
        s["row_lengths"] = None
        total, blocks, max_q = cu[-1], n * width, int(q_len.max())
    s["cu"], s["max_q"] = torch.tensor(cu, dtype=torch.int32, device=_DEV), max_q
    s["k"], s["v"], s["ks"], s["vs"] = _pool(case, blocks, g)
    s["q"] = torch.randn(total, case["heads"], case["dim"], generator=g, device=_DEV, dtype=dt)
    if case["form"] == "store":
        shape = (total, case["kv_heads"], case["dim"])
        s["k_new"], s["v_new"] = (torch.randn(shape, generator=g, device=_DEV, dtype=dt)
                                  for _ in range(2))
    return s


def _filters(case, rows_of, rows, h):
    """Per-row temperature, top-k and top-p of a request's own settings (``rows_of`` rows
    each), and the host plan (max_top_k, apply_top_p)."""
    n = -(-rows // rows_of)
    temp = torch.full((n,), float(case["temperature"]))
    top_k = torch.full((n,), -1, dtype=torch.int64)
    top_p = torch.ones(n)
    if case["top_p"] == "all":
        top_p.fill_(0.9)
    elif case["top_p"] == "mixed":
        top_p = torch.tensor([1.0, 0.8, 0.9, 0.95])[torch.randint(0, 4, (n,), generator=h)]
    if case["top_k"] == "all":
        top_k.fill_(50)
    elif case["top_k"] == "mixed":
        top_k = torch.tensor([-1, 20, 50, 200])[torch.randint(0, 4, (n,), generator=h)]
    if case["top_p"] == "mixed" or case["top_k"] == "mixed":
        temp = temp * (0.8 + 0.4 * torch.rand(n, generator=h))
    return {"temp": temp.repeat_interleave(rows_of)[:rows].contiguous().to(_DEV),
            "top_k": top_k.repeat_interleave(rows_of)[:rows].contiguous().to(_DEV),
            "top_p": top_p.repeat_interleave(rows_of)[:rows].contiguous().to(_DEV),
            "max_top_k": max(0, int(top_k.max())), "apply_top_p": bool((top_p < 1).any())}


def _distributions(logits, temp, top_k, top_p, dtype):
    """softmax(logits / T) over the strict top-k, then top-p, tokens of each row (ties in
    column order), in ``dtype``, a few rows at a time."""
    out = torch.empty(logits.shape, dtype=dtype, device=logits.device)
    step = max(1, 4_000_000 // logits.shape[1])
    for i in range(0, logits.shape[0], step):
        part = slice(i, min(i + step, logits.shape[0]))
        x, order = (logits[part].to(dtype) / temp[part].to(dtype).unsqueeze(1)).sort(
            dim=1, descending=True, stable=True)
        at = torch.arange(x.shape[1], device=x.device).unsqueeze(0)
        k = top_k[part].unsqueeze(1)
        x = x.masked_fill((k > 0) & (at >= k), -torch.inf)
        mass = x.softmax(1)
        before = mass.cumsum(1) - mass
        p = top_p[part].to(dtype).unsqueeze(1)
        # the first token always survives
        x = x.masked_fill((p < 1) & (before > p) & (at > 0), -torch.inf)
        out[part] = torch.zeros_like(x).scatter_(1, order, x.softmax(1))
    return out


def _accept_inputs(case, seed, n, random):
    """Logits of n requests, and the drafts and uniforms of the first ``random`` ones."""
    h = torch.Generator().manual_seed(seed)
    g = torch.Generator(device=_DEV).manual_seed(seed)
    w1, vocab = case["w1"], case["vocab"]
    s = {"case": case, **_filters(case, w1 + 1, random * (w1 + 1), h)}
    draft = torch.randn(n, w1, vocab, generator=g, device=_DEV) * 3.0
    target = torch.cat([draft, draft[:, :1].flip(2)], 1)
    target += torch.randn(target.shape, generator=g, device=_DEV)
    s["logits"] = target.to(_DTYPES[case["logits"]])
    pick = lambda t: t.view(random, w1 + 1)[:, :w1].reshape(-1)  # noqa: E731
    rows = draft[:random].reshape(-1, vocab).to(_DTYPES[case["logits"]]).float()
    q = _distributions(rows, pick(s["temp"]), pick(s["top_k"]), pick(s["top_p"]), torch.float32)
    s["tokens"] = torch.empty(n, w1, dtype=torch.int64, device=_DEV)
    s["tokens"][:random] = torch.multinomial(q, 1, generator=g).view(random, w1)
    s["tokens"][random:] = draft[random:].argmax(2)
    s["q"] = q.view(random, w1, vocab)
    s["drafts"] = torch.randint(max(1, w1 - 1), w1 + 1, (n,), generator=h).to(_DEV)
    s["u_accept"] = torch.rand(random, w1, generator=g, device=_DEV)
    s["u_final"] = torch.rand(random, generator=g, device=_DEV)
    return s


def _round_case(case, part):
    """The attention or the acceptance of a round, as a case of its own."""
    if part == "attend":
        w = case["w1"] + 1
        lo = max(case["ctx_lo"], w)
        return _attend("", "store", case["n"], (lo, max(lo, case["ctx_hi"])), (w, w),
                       (case["heads"], case["kv_heads"]), case["dim"])
    return _accept("", case["random"], case["w1"], case["vocab"], 0.7, "all", "none")


def prepare(case, seed):
    _package()
    if case["kind"] == "attend":
        s = _attend_inputs(case, seed)
        s["kernel"] = _package().create_backend("auto", _DEV, _DTYPES[case["dtype"]], case["dim"],
                                                _BLOCK)
        return s
    if case["kind"] == "accept":
        return _accept_inputs(case, seed, case["n"], case["n"])
    if case["kind"] == "draft":
        h = torch.Generator().manual_seed(seed)
        g = torch.Generator(device=_DEV).manual_seed(seed)
        r = case["random"]
        logits = torch.randn(case["rows"], case["vocab"], generator=g, device=_DEV) * 3.0
        return {"case": case, **_filters(case, 1, r, h),
                "logits": logits.to(_DTYPES[case["logits"]]),
                "rows": torch.randperm(case["rows"], generator=h)[:r].sort()[0].to(_DEV),
                "u": torch.rand(r, generator=g, device=_DEV)}
    s = _accept_inputs(_round_case(case, "accept"), seed, case["n"], case["random"])
    a = _attend_inputs(_round_case(case, "attend"), seed + 1)
    n, r, w = case["n"], case["random"], case["w1"] + 1
    requests = torch.arange(r, device=_DEV)
    return {"case": case, "accept": s, "attend": a,
            "kernel": _package().create_backend("auto", _DEV, torch.bfloat16, case["dim"], _BLOCK),
            "requests": requests, "rows": torch.arange(r * w, device=_DEV),
            "ranks": requests.repeat_interleave(w),
            "offsets": torch.arange(w, device=_DEV).repeat(r),
            "starts": a["lengths"].long() - w, "inputs": torch.zeros_like(a["lengths"]).long()}


# -------------------------------------------------------------------------------- pass

def _bits(pool):
    """A pool's stored bits (one layer's view)."""
    return pool.view(torch.uint8 if pool.element_size() == 1 else torch.int16)


def _attend_run(s, kernel):
    form, window = s["case"]["form"], s["case"]["window"]
    if form == "decode":
        if window:
            return kernel.windowed(s["q"], s["k"], s["v"], s["tables"], s["lengths"], window,
                                   s["ks"], s["vs"])
        return kernel(s["q"], s["k"], s["v"], s["tables"], s["lengths"], s["ks"], s["vs"])
    if form == "planes":
        return kernel.prefill(s["q"], s["k"], s["v"], s["tables"], s["lengths"], s["cu"],
                              s["max_q"], s["ks"], s["vs"], row_lengths=s["row_lengths"])
    out = {"out": kernel.prefill_store(s["q"], s["k_new"], s["v_new"], s["k"], s["v"],
                                       s["tables"], s["lengths"], s["cu"], s["max_q"], s["ks"],
                                       s["vs"]),
           "keys": _bits(s["k"]), "values": _bits(s["v"])}
    if s["case"]["kv"] == "fp8_vector":
        out["key_scales"], out["value_scales"] = s["ks"], s["vs"]
    return out


def _accept_run(s, logits):
    r = s["q"].shape[0]
    targets, p, res = _package().verify_accept(
        logits, s["temp"], s["top_k"], s["top_p"], s["tokens"][:r], s["drafts"][:r], s["q"],
        s["u_accept"], s["u_final"], max_top_k=s["max_top_k"], apply_top_p=s["apply_top_p"])
    return targets, p, res


def run(state):
    s, pkg = state, sys.modules["vllm_rlt_amd"]
    kind = s["case"]["kind"]
    if kind == "attend":
        return _attend_run(s, s["kernel"])
    if kind == "accept":
        targets, p, res = _accept_run(s, s["logits"])
        return {"targets": targets, "p": p, "result": tuple(res)}
    if kind == "draft":
        proposed, q = pkg.propose_drafts(s["logits"], s["rows"], s["temp"], s["top_k"],
                                         s["top_p"], s["u"], max_top_k=s["max_top_k"],
                                         apply_top_p=s["apply_top_p"])
        return {"proposed": proposed, "q": q}
    a, c = s["attend"], s["accept"]
    out = _attend_run(a, s["kernel"])
    targets, accepted, following = pkg.greedy_accept_batched(c["tokens"], c["drafts"], c["logits"])
    _, p, res = _accept_run(c, c["logits"][:s["case"]["random"]])
    merged = pkg.merge_random_round(targets.view(-1), accepted, following, s["starts"],
                                    s["inputs"], res, s["requests"], s["rows"], s["ranks"],
                                    s["offsets"])
    return {"attend": out, "targets": targets, "p": p, "result": tuple(res),
            "merged": tuple(merged)}


# -------------------------------------------------------------------- work and tolerance

def _attend_work(case):
    q = (case["q_lo"] + case["q_hi"]) / 2
    ctx = max((case["ctx_lo"] + case["ctx_hi"]) / 2, q)
    if case["window"]:
        ctx = min(ctx, case["window"])
    seqs = case["batch"] * (min(_PLANES, case["q_hi"]) if case["form"] == "planes" else 1)
    rows = case["batch"] * q
    elt = 2 if case["kv"] == "same" else 1
    kv = 2 * case["kv_heads"] * case["dim"]  # elements of a position
    kept = ctx - q if case["form"] == "store" else ctx  # positions read from the pool
    nbytes = seqs * kept * kv * elt + 2 * rows * case["heads"] * case["dim"] * 2
    nbytes += seqs * ctx / _BLOCK * 4
    if case["kv"] == "fp8_vector":
        nbytes += seqs * kept * 2 * case["kv_heads"] * 4
    if case["form"] == "store":
        nbytes += rows * kv * (2 + elt)
    seen = ctx - (q - 1) / 2 if case["form"] == "store" else ctx  # keys a row sees, on average
    return nbytes, 4 * rows * case["heads"] * case["dim"] * seen


def _accept_work(case, n, random):
    rows, w1, vocab = random * (case["w1"] + 1), case["w1"], case["vocab"]
    elt = 4 if case["logits"] == "fp32" else 2
    nbytes = n * (w1 + 1) * vocab * elt + rows * vocab * 4 + random * w1 * vocab * 4
    return nbytes, 6 * rows * vocab


def work(case):
    if case["kind"] == "attend":
        b, f = _attend_work(case)
    elif case["kind"] == "accept":
        b, f = _accept_work(case, case["n"], case["n"])
    elif case["kind"] == "draft":
        elt = 4 if case["logits"] == "fp32" else 2
        b = case["vocab"] * (case["rows"] * elt + case["random"] * 4)
        f = 6 * case["random"] * case["vocab"]
    else:
        b, f = _attend_work(_round_case(case, "attend"))
        b2, f2 = _accept_work(_round_case(case, "accept"), case["n"], case["random"])
        b, f = b + b2, f + f2
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Attention in 16 bits: the output's and the weights' rounding (2^-9 in bf16, 2^-12
    in fp16; 2.1e-3 off float64 in bf16).  Distributions: 32-bit masses (6e-8 off float64),
    and now and then a token more or less at a top-p cut (its probability over the row's
    norm)."""
    if case["kind"] == "attend":
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 2e-3, "max": 0.1}
    if case["kind"] == "round":
        return {"rel": 8e-3, "max": 0.5}
    filtered = case["top_p"] != "none"
    return {"rel": 2e-3 if filtered else 1e-6, "max": 0.5 if filtered else 1e-5}


# ------------------------------------------------------------------------------- exact

def _attend_exact(s):
    """The attention output in float64 over the pool with the window rows stored (the
    stored bits of an fp8 pool are its quantizer's, so they are taken as stored values
    after quantizing here)."""
    case = s["case"]
    bs, hkv, dim = _BLOCK, case["kv_heads"], case["dim"]
    group = case["heads"] // hkv
    out = torch.empty_like(s["q"], dtype=torch.float64)
    lengths, tables = s["lengths"].tolist(), s["tables"].long()
    cu = s["cu"].tolist() if case["form"] != "decode" else list(range(len(lengths) + 1))
    limits = s["row_lengths"].tolist() if s["row_lengths"] is not None else None

    def quantized(x, scale):
        x = x.float()
        if case["kv"] == "fp8_vector":
            scale = (x.abs().amax(-1, keepdim=True) * (1.0 / 448.0)).clamp_min(
                torch.finfo(torch.float32).tiny)
        return (x / scale).clamp(-448, 448).to(_FP8).double() * scale.double()

    def gathered(pool, scale, new, seq, length):
        ids = tables[seq, : -(-length // bs)]
        x = pool.view(torch.uint8)[ids].view(_FP8).double() if pool.dtype == _FP8 else \
            pool[ids].double()
        if scale is not None:
            x = x * (scale[ids].double().unsqueeze(-1) if scale.ndim else scale.double())
        x = x.reshape(-1, hkv, dim)[:length]
        if new is not None:
            rows = new[cu[seq]:cu[seq + 1]]
            x[length - rows.shape[0]:] = rows.double() if pool.dtype != _FP8 else \
                quantized(rows, scale)
        return x

    for i, length in enumerate(lengths):
        a, b = cu[i], cu[i + 1]
        keys = gathered(s["k"], s["ks"], s.get("k_new"), i, length)
        values = gathered(s["v"], s["vs"], s.get("v_new"), i, length)
        if limits is not None:
            seen = torch.tensor(limits[a:b], device=_DEV)
        else:
            seen = torch.arange(length - (b - a) + 1, length + 1, device=_DEV)
        at = torch.arange(length, device=_DEV).unsqueeze(0)
        hidden = at >= seen.unsqueeze(1)
        if case["window"]:
            hidden |= at < seen.unsqueeze(1) - case["window"]
        for h in range(hkv):
            heads = slice(h * group, (h + 1) * group)
            q = s["q"][a:b, heads].double().reshape(-1, dim)
            score = (q @ keys[:, h].t().contiguous()) * dim ** -0.5
            score = score.masked_fill_(hidden.repeat_interleave(group, 0), -torch.inf)
            out[a:b, heads] = (score.softmax(1) @ values[:, h].contiguous()).view(
                b - a, group, dim)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "attend":
        out = _attend_exact(s)
        return {"out": out} if case["form"] == "store" else out
    if case["kind"] == "draft":
        return {"q": _distributions(s["logits"][s["rows"]], s["temp"], s["top_k"], s["top_p"],
                                    torch.float64)}
    c = s if case["kind"] == "accept" else s["accept"]
    r, w, vocab = c["q"].shape[0], case["w1"] + 1, case["vocab"]
    p = _distributions(c["logits"][:r].reshape(r * w, vocab), c["temp"], c["top_k"], c["top_p"],
                       torch.float64).view(r, w, vocab)
    found = {"p": p}
    if case["kind"] == "round":
        found["attend"] = {"out": _attend_exact(s["attend"])}
    return found
