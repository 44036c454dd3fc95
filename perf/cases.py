"""The calls that a decode or scoring loop makes of this package, as cases to be timed.

Each case is a dict of plain values.  `prepare` makes what a serving program holds
before the call (logits, hidden states, the LM head's weight, settings) on the GPU
from the seed, `run` is one pass through the public entry points, `work` the bytes
and operations a pass cannot do without, `exact` the same outputs in 64 bits.

Kinds: "sample" (one sampling step over [B, V] logits), "argmax" (greedy decode),
"rejection" (stochastic draft verification), "tree" (one EAGLE3 draft tree), "head"
(LM head + argmax, with or without the logits that a sampled step reads) and
"score" (LM head + log-likelihood of given targets).
"""
import math

import torch

import llima_amd

HEADS = (32000, 32768, 50257, 100352, 128256, 151936, 152064, 202048, 256000, 262144)


def listed():
    return [
        # One chat stream: a step's row through repetition, T, top-k and top-p (Qwen2.5 head).
        dict(name="sample_one_row", kind="sample", B=1, V=151936, dtype="f32", H=64, sigma=3.0,
             style="top_k", T=0.7, top_k=40, top_p=0.9, min_p=0.0, rep=1.1, pres=0.0, freq=0.0),
        # The headline decode batch: every stage on, a 2048-id history (Llama-3 head).
        dict(name="sample_batch", kind="sample", B=64, V=128256, dtype="f32", H=2048, sigma=4.0,
             style="top_k", T=0.8, top_k=50, top_p=0.95, min_p=0.05, rep=1.15, pres=0.5, freq=0.3),
        # A large serving batch of bf16 logits over the widest head (Gemma).
        dict(name="sample_large_bf16", kind="sample", B=256, V=262144, dtype="bf16", H=512,
             sigma=5.0, style="top_k", T=1.0, top_k=64, top_p=0.95, min_p=0.0, rep=1.05, pres=0.0,
             freq=0.0),
        # The common API default: nucleus sampling alone.
        dict(name="sample_top_p", kind="sample", B=64, V=128256, dtype="f32", H=0, sigma=4.0,
             style="top_p", T=1.0, top_k=0, top_p=0.9, min_p=0.0, rep=1.0, pres=0.0, freq=0.0),
        # Requests with settings of their own: half of the rows with top-k, half with top-p alone.
        dict(name="sample_mixed_rows", kind="sample", B=64, V=128256, dtype="f32", H=0, sigma=4.0,
             style="mixed", T=1.0, top_k=50, top_p=0.9, min_p=0.0, rep=1.0, pres=0.0, freq=0.0),
        # Structured output: a grammar allows about 2 % of the ids.
        dict(name="sample_grammar", kind="sample", B=32, V=151936, dtype="f32", H=0, sigma=3.0,
             style="grammar", allowed=0.02, T=1.0, top_k=0, top_p=0.9, min_p=0.0, rep=1.0,
             pres=0.0, freq=0.0),
        # Greedy decode of a large batch over bf16 logits.
        dict(name="argmax_bf16", kind="argmax", B=256, V=262144, dtype="bf16"),
        # Speculative decoding: 7 drafts a sequence checked by rejection sampling.
        dict(name="verify_rejection", kind="rejection", B=16, D=7, V=128256),
        # One EAGLE3 draft tree at the reference's shape.
        dict(name="draft_tree", kind="tree", K=5, depth=4, total=15, Vd=32000, V=128256),
        # One stream's decode step: the LM head read once for one row.
        dict(name="head_one_row", kind="head", B=1, H=4096, V=128256, packed=False, logits=False),
        # A decode batch through the weight packed at load time, with the logits a sampled step reads.
        dict(name="head_packed_b128", kind="head", B=128, H=4096, V=128256, packed=True,
             logits=True),
        # Log-likelihoods of a 512-token prompt chunk from its hidden states.
        dict(name="head_score_512", kind="score", B=512, H=4096, V=128256, packed=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, hi):
    """A head width of a served model, or any width up to hi."""
    if rng.random() < 0.4:
        return rng.choice([v for v in HEADS if v <= hi])
    return min(hi, _log(rng, 16000, hi))


def draw(rng):
    kind = rng.choice(["sample", "sample", "sample", "sample", "sample", "sample", "argmax",
                       "rejection", "tree", "head", "head", "score"])
    if kind == "sample":
        style = rng.choice(["top_k", "top_k", "top_k", "top_p", "mixed", "grammar"])
        bf16 = rng.random() < 0.4
        V = _vocab(rng, 262144)
        B = _log(rng, 1, 256 if style == "top_k" else 96)
        pen = style in ("top_k", "top_p") and rng.random() < 0.5
        c = dict(kind="sample", B=B, V=V, dtype="bf16" if bf16 else "f32",
                 H=_log(rng, 16, 4096) if pen else 0, sigma=round(rng.uniform(3.0, 5.0), 2),
                 style=style, T=round(rng.uniform(0.6, 1.2), 2),
                 top_k=rng.randint(10, 100) if style in ("top_k", "mixed") else 0,
                 top_p=round(rng.uniform(0.8, 0.97), 3),
                 min_p=rng.choice([0.0, 0.0, 0.02, 0.05]),
                 rep=round(rng.uniform(1.0, 1.3), 2) if pen else 1.0,
                 pres=rng.choice([0.0, 0.5]) if pen else 0.0,
                 freq=rng.choice([0.0, 0.3]) if pen else 0.0)
        if style == "grammar":
            c["allowed"] = rng.choice([0.005, 0.02, 0.1, 0.5])
        return c
    if kind == "argmax":
        return dict(kind="argmax", B=_log(rng, 1, 256), V=_vocab(rng, 262144),
                    dtype=rng.choice(["bf16", "f32"]))
    if kind == "rejection":
        return dict(kind="rejection", B=_log(rng, 1, 24), D=rng.randint(1, 8),
                    V=_vocab(rng, 151936))
    if kind == "tree":
        K, depth = rng.randint(3, 10), rng.randint(2, 6)
        return dict(kind="tree", K=K, depth=depth,
                    total=rng.randint(K, min(32, K + (depth - 1) * K * K)),
                    Vd=_log(rng, 8000, 64000), V=128256)
    packed = rng.random() < 0.5
    step = 256 if packed else 64
    H = step * rng.randint(1024 // step, 8192 // step)
    V = _vocab(rng, min(262144, 128256 * 4096 // H))
    if kind == "head":
        return dict(kind="head", B=_log(rng, 1, 256), H=H, V=V, packed=packed,
                    logits=rng.random() < 0.5)
    return dict(kind="score", B=_log(rng, 4, 512), H=H, V=V, packed=packed)


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device="cuda")


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _logits(c, g):
    """N(0, sigma^2) rows; bf16 rows soft-capped at 30, as the heads that emit bf16 do."""
    x = _normal(g, c["B"], c["V"]).mul_(c.get("sigma", 4.0))
    if c["dtype"] == "bf16":
        x = (30.0 * torch.tanh(x / 30.0)).to(torch.bfloat16)
    return x


def _zipf_history(c, g):
    """[B, H] ids from a Zipf(1.1) law over ranks, ranks mapped to ids by a permutation."""
    V = c["V"]
    cdf = torch.arange(1, V + 1, device="cuda", dtype=torch.float64).pow_(-1.1).cumsum_(0)
    ranks = torch.searchsorted(cdf / cdf[-1], torch.rand(c["B"], c["H"], generator=g, device="cuda",
                                                         dtype=torch.float64))
    perm = torch.randperm(V, generator=g, device="cuda")
    return perm[ranks.clamp_(max=V - 1)].to(torch.int32)


def _grammar(c, g, x):
    """The packed mask of a grammar: runs of 64 allowed ids (independent bits where half
    of the ids are allowed), and a forbidden id that outranks the row in most rows."""
    B, V = c["B"], c["V"]
    nw = (V + 31) // 32
    if c["allowed"] >= 0.5:
        m = torch.randint(-2**31, 2**31, (B, nw), generator=g, device="cuda").to(torch.int32)
    else:
        n = V // 64
        runs = max(1, int(c["allowed"] * n))
        blk = _rand(g, B, n).topk(runs, dim=1).indices
        m = torch.zeros(B, nw, dtype=torch.int32, device="cuda")
        m.scatter_(1, 2 * blk, -1)
        m.scatter_(1, 2 * blk + 1, -1)
    j = torch.randint(0, V, (B,), generator=g, device="cuda")
    rows = torch.arange(B, device="cuda")
    banned = ((m[rows, j >> 5] >> (j & 31).to(torch.int32)) & 1) == 0
    top = (x.amax(dim=1).float() + 5.0).to(x.dtype)
    x[rows, j] = torch.where(banned, top, x[rows, j])
    return m


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "sample":
        x = _logits(c, g)
        s = dict(kind=kind, logits=x, u=_rand(g, c["B"]), history=None, mask=None)
        if c["H"]:
            s["history"] = _zipf_history(c, g)
        if c["style"] == "grammar":
            s["mask"] = _grammar(c, g, x)
        cfg = dict(temperature=c["T"], top_k=c["top_k"], top_p=c["top_p"], min_p=c["min_p"],
                   repetition_penalty=c["rep"], presence_penalty=c["pres"],
                   frequency_penalty=c["freq"])
        if c["style"] == "mixed":
            even = (torch.arange(c["B"], device="cuda") % 2) == 0
            cfg["top_k"] = torch.where(even, c["top_k"], 0).to(torch.int32)
            cfg["top_p"] = torch.where(even, 0.95, c["top_p"]).to(torch.float32)
        s["cfg"] = llima_amd.SamplerConfig(**cfg)
        return s
    if kind == "argmax":
        return dict(kind=kind, logits=_logits(c, g))
    if kind == "rejection":
        B, D, V = c["B"], c["D"], c["V"]
        t = _normal(g, B, D + 1, V).mul_(4.0)
        d = _normal(g, B, D, V).mul_(1.5).add_(t[:, :D])
        ids = torch.multinomial(torch.softmax(d.reshape(B * D, V), 1), 1, generator=g)
        return dict(kind=kind, target=t, draft=d, ids=ids.reshape(B, D).to(torch.int32),
                    ua=_rand(g, B, D), ur=_rand(g, B))
    if kind == "tree":
        K, depth, Vd, V = c["K"], c["depth"], c["Vd"], c["V"]
        bf = torch.bfloat16
        root = _normal(g, Vd).mul_(3.0).to(bf)
        levels = [_normal(g, K, Vd).mul_(3.0).to(bf) for _ in range(depth - 1)]
        at = torch.randperm(V, generator=g, device="cuda")[:Vd].sort().values
        d2t = (at - torch.arange(Vd, device="cuda")).to(torch.int32)
        return dict(kind=kind, tree=llima_amd.Eagle3DraftTree(d2t, topk=K, depth=depth), root=root,
                    levels=levels, total=c["total"], token=int(seed) % V)
    # The LM head: rows whose winner stands out, as a trained model's do.
    B, H, V = c["B"], c["H"], c["V"]
    w = _normal(g, V, H, dtype=torch.bfloat16).mul_(H ** -0.5)
    t = torch.randint(0, V, (B,), generator=g, device="cuda", dtype=torch.int64)
    x = _normal(g, B, H) + (4.0 + 12.0 * _rand(g, B, 1)) * w[t].float()
    s = dict(kind=kind, hidden=x.to(torch.bfloat16), weight=llima_amd.lm_head_pack(w) if c["packed"] else w)
    if kind == "head":
        s["logits"] = c["logits"]
    else:  # most targets are the likely token, some any other
        other = torch.randint(0, V, (B,), generator=g, device="cuda", dtype=torch.int64)
        s["target"] = torch.where(_rand(g, B) < 0.7, t, other).to(torch.int32)
    return s


def run(s):
    kind = s["kind"]
    if kind == "sample":
        return llima_amd.sample(s["logits"], s["u"], s["cfg"], history=s["history"],
                                bitmask=s["mask"])
    if kind == "argmax":
        return llima_amd.argmax(s["logits"])
    if kind == "rejection":
        return llima_amd.verify_rejection(s["target"], s["draft"], s["ids"], s["ua"], s["ur"])
    if kind == "tree":
        tree = s["tree"]
        out = dict(begin=tree.begin(s["root"]))
        out["grow"] = [tree.grow(x) for x in s["levels"]]
        out["scores"] = tree.node_scores()
        out.update(tree.finish(s["total"], s["token"]))
        # the paths in the fixed-size buffer that a verification step of one shape takes
        r, n = out["retrieve"], s["total"] + 1
        out["retrieve"] = torch.nn.functional.pad(r, (0, n - r.shape[1], 0, n - r.shape[0]), value=-1)
        return out
    if kind == "head":
        if s["logits"]:
            return llima_amd.lm_head_argmax(s["hidden"], s["weight"], return_logits=True,
                                            logits_out="bf16")
        return llima_amd.lm_head_argmax(s["hidden"], s["weight"])
    return llima_amd.lm_head_score(s["hidden"], s["weight"], s["target"])


def work(case):
    c, kind = case, case["kind"]
    if kind in ("sample", "argmax"):
        n = c["B"] * c["V"]
        b = n * (2 if c["dtype"] == "bf16" else 4) + 12 * c["B"]
        if kind == "sample":
            b += 4 * c["B"] * c["H"]
            if c["style"] == "grammar":
                b += 4 * c["B"] * ((c["V"] + 31) // 32)
        return dict(bytes=b, flops=n)
    if kind == "rejection":
        n = c["B"] * (2 * c["D"] + 1) * c["V"]
        return dict(bytes=4 * n + 4 * c["B"] * (3 * c["D"] + 3), flops=2 * n)
    if kind == "tree":
        n = (1 + (c["depth"] - 1) * c["K"]) * c["Vd"]
        return dict(bytes=2 * n + 8 * (c["total"] + 1) ** 2, flops=2 * n)
    B, H, V = c["B"], c["H"], c["V"]
    b = 2 * V * H + 2 * B * H + 16 * B
    if kind == "head" and c["logits"]:
        b += 2 * B * V
    return dict(bytes=b, flops=2 * B * H * V)


def tolerance(case):
    # Selection is defined on exact integer weights: ids and probabilities are the same bits.
    if case["kind"] in ("sample", "argmax", "rejection"):
        return "exact"
    # Node scores are float32 log-probabilities: sums of K terms in another order.
    if case["kind"] == "tree":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    # bf16 logits of fp32 sums: another order of the sums moves one logit in some thousands
    # by one bf16 step (2^-8 of it), and with it now and then the winner of two close logits.
    if case["kind"] == "head":
        return {"rel": 4e-4, "max": 8e-3, "differ": 0.01}
    return {"rel": 4e-4, "max": 1e-2, "differ": 0.01}


# ------------------------------------------------------------------ 64 bits


def _exact_sample(c, s):
    """The sampler's stages in float64: penalties, mask, T, top-k, top-p, min-p, the draw."""
    ids, probs = [], []
    B, V = c["B"], c["V"]
    dev = s["logits"].device

    def rows(v, dtype=torch.float64):
        t = v if isinstance(v, torch.Tensor) else torch.full((B,), v, device=dev)
        return t.to(dtype)

    T, P = rows(s["cfg"].temperature), rows(s["cfg"].top_p)
    K = rows(s["cfg"].top_k, torch.int64)
    for r0 in range(0, B, 16):
        x = s["logits"][r0:r0 + 16].double()
        n = x.shape[0]
        if s["mask"] is not None:
            at = torch.arange(V, device=dev)
            word = s["mask"][r0:r0 + n][:, at >> 5]
            x.masked_fill_(((word >> (at & 31).to(torch.int32)) & 1) == 0, -math.inf)
        if s["history"] is not None:
            h = s["history"][r0:r0 + n].long()
            cnt = torch.zeros_like(x).scatter_add_(1, h, torch.ones_like(h, dtype=x.dtype))
            pen = torch.where(x < 0, x * c["rep"], x / c["rep"]) - c["freq"] * cnt - c["pres"]
            x = torch.where(cnt > 0, pen, x)
        x /= T[r0:r0 + n, None]
        srt = x.sort(dim=1, descending=True).values
        k = K[r0:r0 + n]
        kth = srt.gather(1, (torch.where((k > 0) & (k < V), k, V) - 1)[:, None])
        top = srt[:, :1]
        w = torch.exp(srt - top) * (srt >= kth)
        above = w.cumsum(1) - w
        first = torch.ones_like(srt, dtype=torch.bool)
        first[:, 1:] = srt[:, 1:] != srt[:, :-1]
        p = P[r0:r0 + n, None]
        ok = first & ((above < p * w.sum(1, keepdim=True)) | (p >= 1.0))
        cut = torch.where(ok, srt, math.inf).amin(1, keepdim=True)
        e = torch.exp(x - top)
        e *= (x >= torch.maximum(cut, kth)) & (e >= min(c["min_p"], 1.0))
        cum = e.cumsum(1)
        z = cum[:, -1:]
        i = torch.searchsorted(cum, s["u"][r0:r0 + n, None].double() * z, right=True).clamp_(max=V - 1)
        ids.append(i[:, 0].to(torch.int32))
        probs.append((e.gather(1, i) / z)[:, 0])
    return torch.cat(ids), torch.cat(probs)


def _exact_tree(c, s):
    """Node scores: the log-softmax of each row's top K, added to the score of its parent row."""
    K = c["K"]
    cur = torch.log_softmax(s["root"].double().topk(K).values, 0)
    flat = [cur]
    for x in s["levels"]:
        cand = (torch.log_softmax(x.double().topk(K).values, 1) + cur[:, None]).reshape(-1)
        flat.append(cand)
        cur = cand.topk(K).values
    return torch.cat(flat)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "rejection":  # whole numbers alone
        return None
    weight = None
    if kind in ("head", "score"):  # the plain weight, whichever layout the case uses
        s = prepare(dict(c, packed=False), seed)
        weight = s["weight"].double()
        logits = s["hidden"].double() @ weight.t()
        if kind == "head":
            v, i = logits.max(1)
            return (i.to(torch.int32), v, logits) if c["logits"] else (i.to(torch.int32), v)
        t = s["target"].long()[:, None]
        lp = torch.log_softmax(logits, 1).gather(1, t)[:, 0]
        return lp, logits.argmax(1) == t[:, 0]
    s = prepare(c, seed)
    if kind == "argmax":
        v, i = s["logits"].double().max(1)
        return i.to(torch.int32), v
    if kind == "sample":
        return _exact_sample(c, s)
    out = dict(begin=None, grow=[(None, None, None) for _ in s["levels"]], scores=_exact_tree(c, s),
               tokens=None, tree_mask=None, position_ids=None, retrieve=None)
    return out
