"""The calls this package is measured by: what a serving program asks of it.

Four kinds of call, all through the public entry points:

  decode   ``mla_decode`` over a paged (or dense) 16-bit latent cache at the
           DeepSeek dims (512 + 64), one or several query tokens a sequence;
  fp8      the same over an E4M3 cache with its scales;
  generic  ``mla_decode`` at other head dims or in fp32;
  layer    one decode step of the whole ``MLA`` layer.

``listed`` holds one call for each way the package is used, from a single
short sequence to a full batch of long ones; ``draw`` spreads over the same
ranges. Queries, caches and hidden states are N(0, 1), weights N(0, 0.02),
block tables are shuffled and the lengths of a batch are spread evenly over
[lo, hi] in a shuffled order, so a case's work does not depend on the seed.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.abspath("triton-mla_amd")  # the package's folder in the tree under test
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def _decode(name, batch, heads, lo, hi, dtype="bf16", page=64, q_len=1, dv=512, dr=64, fp8="", lse=False):
    """page 0: a dense cache; fp8: "" or the granularity of the scales."""
    kind = "fp8" if fp8 else "generic" if (dv, dr) != (512, 64) or dtype == "fp32" else "decode"
    return {"name": name, "kind": kind, "batch": batch, "heads": heads, "lo": lo, "hi": hi, "dtype": dtype,
            "page": page, "q_len": q_len, "dv": dv, "dr": dr, "fp8": fp8, "lse": lse}


def _layer(name, batch, heads, hidden, lo, hi, page=64, dtype="bf16"):
    return {"name": name, "kind": "layer", "batch": batch, "heads": heads, "hidden": hidden, "lo": lo, "hi": hi,
            "page": page, "dtype": dtype}


def listed():
    return [
        # One user's short chat: the time of a token is launches and latency.
        _decode("b1_h128_1k", 1, 128, 1024, 1024),
        # A small batch of short contexts: still latency, several sequences.
        _decode("b8_h128_1k", 8, 128, 1024, 1024),
        # The headline: a full batch at 8K tokens with all 128 heads on the GPU.
        _decode("b32_h128_8k", 32, 128, 8192, 8192),
        # Continuous batching: 64 sequences of 1K to 32K tokens, 128 heads.
        _decode("ragged_b64_h128", 64, 128, 1083, 32645),
        # The same batch on one rank of eight (16 heads): the cache's bytes.
        # The log-sum-exp is asked for, as a context-parallel merge needs it.
        _decode("ragged_b64_h16", 64, 16, 1083, 32645, lse=True),
        # Few long sequences on one rank of two (64 heads), in fp16.
        _decode("b8_h64_16k_fp16", 8, 64, 12001, 16384, dtype="fp16"),
        # Speculative decoding: a draft token verified beside the next one.
        _decode("spec2_b16_h128", 16, 128, 1021, 8191, q_len=2),
        # An fp8 cache on one rank of eight, one scale a page.
        _decode("fp8_ragged_b64_h16", 64, 16, 1083, 32645, fp8="page"),
        # An fp8 cache under all 128 heads at the headline's size.
        _decode("fp8_b32_h128_8k", 32, 128, 8192, 8192, fp8="page"),
        # A smaller latent than DeepSeek's (256 + 32), full batch.
        _decode("dims256_32_b32_h128", 32, 128, 4099, 8192, dv=256, dr=32),
        # Checking a model in float32 (a dense cache, as the tests hold one).
        _decode("fp32_b16_h16_8k", 16, 16, 5003, 8192, dtype="fp32", page=0),
        # One whole attention layer of DeepSeek-V3 in a serving step.
        _layer("layer_v3_b16_16k", 16, 128, 7168, 16384, 16384),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "spec", "fp8", "fp8", "generic", "generic", "fp32", "layer"])
    batch = _log_int(rng, 1, 64)
    hi = _log_int(rng, 200, 32768)
    lo = max(1, int(hi * rng.choice([0.03, 0.3, 0.7, 1.0])))
    heads = rng.choice([8, 16, 20, 32, 40, 64, 96, 128])
    page = rng.choice([0, 16, 64, 64, 64, 128])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "layer":
        cap = 262144
        batch, hi, lo = _fit(batch, hi, lo, cap)
        heads, hidden = rng.choice([(128, 7168), (128, 5120), (64, 7168), (16, 2048)])
        return _layer("", batch, heads, hidden, lo, hi, page=page or 64, dtype=dtype)
    if kind == "spec":
        q_len = rng.choice([2, 3, 4, 8])
        batch, hi, lo = _fit(batch, hi, lo, 900000 * 128 // (heads * q_len * 2))
        return _decode("", batch, heads, max(lo, q_len), max(hi, q_len), dtype, page, q_len)
    if kind == "fp8":
        # (one or four 32-head blocks a workgroup, or 16-head groups: the
        # forms the package's fp8 workloads run)
        heads = rng.choice([8, 16, 16, 20, 32, 128])
        batch, hi, lo = _fit(batch, hi, lo, 600000)
        return _decode("", batch, heads, lo, hi, dtype, page or 64, fp8=rng.choice(["page", "page", "token"]),
                       lse=rng.random() < 0.3)
    if kind == "generic":
        dv, dr = rng.choice([(64, 32), (128, 64), (256, 32), (256, 64), (512, 32)])
        batch, hi, lo = _fit(batch, hi, lo, 200000)
        return _decode("", batch, heads, lo, hi, dtype, page, dv=dv, dr=dr)
    if kind == "fp32":
        dv, dr = rng.choice([(512, 64), (512, 64), (128, 64)])
        heads = min(heads, 32)
        batch, hi, lo = _fit(batch, hi, lo, 100000 * 16 // max(heads, 16))
        return _decode("", batch, heads, lo, hi, "fp32", page, dv=dv, dr=dr)
    batch, hi, lo = _fit(batch, hi, lo, 900000)
    return _decode("", batch, heads, lo, hi, dtype, page, lse=rng.random() < 0.3)


def _fit(batch, hi, lo, cap):
    """A batch of at most cap cached tokens."""
    batch = max(1, min(batch, cap // hi))
    hi = min(hi, cap)
    return batch, hi, min(lo, hi)


def _lengths(case):
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    return [lo + round((hi - lo) * (i + 0.5) / b) for i in range(b)]


def _cache(case, width, generator, spare=0):
    """Lengths, block table (None: dense) and a latent cache with room for
    ``spare`` more tokens a sequence."""
    lens = _lengths(case)
    order = torch.randperm(case["batch"], generator=torch.Generator().manual_seed(generator.initial_seed()))
    lens = [lens[int(i)] for i in order]
    seqlens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    dtype = DTYPES[case["dtype"]]
    page = case["page"]
    if page == 0:
        kv = torch.randn(case["batch"], case["hi"] + spare, width, generator=generator, device="cuda", dtype=dtype)
        return seqlens, None, kv
    pages = [-(-(n + spare) // page) for n in lens]
    total, most = sum(pages), max(pages)
    perm = torch.randperm(total, generator=generator, device="cuda").to(torch.int32)
    table = torch.zeros(case["batch"], most, dtype=torch.int32, device="cuda")
    start = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[start:start + n]
        start += n
    kv = torch.randn(total, page, width, generator=generator, device="cuda", dtype=dtype)
    return seqlens, table, kv


def prepare(case, seed):
    import triton_mla

    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "layer":
        cfg = triton_mla.MLAConfig(hidden_size=case["hidden"], num_heads=case["heads"])
        with torch.device("cuda"), torch.no_grad():
            model = triton_mla.MLA(cfg).to(dtype)
            for name, p in model.named_parameters():
                if "norm" not in name:  # the norms' gains stay 1
                    p.normal_(0.0, 0.02, generator=g)
        seqlens, table, kv = _cache(case, cfg.kv_cache_dim, g, spare=1)
        x = torch.randn(case["batch"], case["hidden"], generator=g, device="cuda", dtype=dtype)
        return {"model": model, "x": x, "kv": kv, "seqlens": seqlens, "table": table}
    width = case["dv"] + case["dr"]
    seqlens, table, kv = _cache(case, width, g)
    shape = (case["batch"], case["heads"], width)
    if case["q_len"] > 1:
        shape = (case["batch"], case["q_len"], case["heads"], width)
    q = torch.randn(*shape, generator=g, device="cuda", dtype=dtype)
    scale = None
    if case["fp8"]:
        kv, scale = triton_mla.quantize_kv_fp8(kv, case["fp8"])
    softmax = 192 ** -0.5 if (case["dv"], case["dr"]) == (512, 64) else width ** -0.5
    return {"q": q, "kv": kv, "seqlens": seqlens, "table": table, "kv_scale": scale, "dv": case["dv"],
            "softmax_scale": softmax, "lse": case["lse"]}


def run(state):
    import triton_mla

    if "model" in state:
        with torch.no_grad():
            out, seqlens = state["model"](state["x"], state["kv"], state["seqlens"], state["table"])
        return {"out": out, "seqlens": seqlens, "cache": state["kv"]}
    res = triton_mla.mla_decode(state["q"], state["kv"], state["seqlens"], state["table"], head_dim_v=state["dv"],
                                softmax_scale=state["softmax_scale"], return_lse=state["lse"],
                                kv_scale=state["kv_scale"])
    return {"out": res[0], "lse": res[1]} if state["lse"] else {"out": res}


def work(case):
    tokens = sum(_lengths(case))
    b, h = case["batch"], case["heads"]
    elt = BYTES[case["dtype"]]
    if case["kind"] == "layer":
        hidden = case["hidden"]
        weights = hidden * (1536 + 576) + 1536 * h * 192 + 512 * h * 256 + h * 128 * hidden
        tokens += b
        return {"bytes": elt * (weights + tokens * 576 + b * 576 + 2 * b * hidden),
                "flops": 2 * b * weights + 2 * h * tokens * (576 + 512)}
    width = case["dv"] + case["dr"]
    rows = b * h * case["q_len"]
    cache = tokens * width * elt
    if case["fp8"]:
        cache = tokens * width + 4 * (tokens if case["fp8"] == "token" else tokens // case["page"])
    out = rows * (case["dv"] * elt + (4 if case["lse"] else 0))
    return {"bytes": cache + rows * width * elt + out,
            "flops": 2 * h * case["q_len"] * tokens * (width + case["dv"])}


def tolerance(case):
    """About four times the distance from ``exact``: probabilities, split
    partials and results rounded to the element type (2.5e-3 in bf16, 3e-4 in
    fp16), the layer's chain of roundings (4.3e-3), float32 sums in another
    order (1e-6 to 3e-6)."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    rel = 2e-2 if case["kind"] == "layer" else 1e-2
    return {"rel": rel / 8 if case["dtype"] == "fp16" else rel}


def _attend(q, kv, seqlens, table, dv, scale, kv_scale=None):
    """Softmax attention in float64, one sequence at a time: q [B, T, H, D]."""
    out = torch.zeros(*q.shape[:3], dv, dtype=torch.float64, device=q.device)
    lse = torch.full(q.shape[:3], -math.inf, dtype=torch.float64, device=q.device)
    t_len = q.shape[1]
    for b, n in enumerate(seqlens.tolist()):
        if table is None:
            rows = kv[b, :n].double()
        else:
            ids = table[b, :-(-n // kv.shape[1])].long()
            rows = kv[ids].double()
            if kv_scale is not None:
                s = kv_scale[ids].double()
                rows = rows * (s[:, None, None] if s.dim() == 1 else s[..., None])
            rows = rows.reshape(-1, rows.shape[-1])[:n]
        keys = rows.transpose(0, 1).contiguous()
        for t in range(t_len):
            seen = n - (t_len - 1 - t)
            logits = (q[b, t].double() @ keys[:, :seen].contiguous()) * scale
            lse[b, t] = torch.logsumexp(logits, dim=-1)
            out[b, t] = torch.softmax(logits, dim=-1) @ rows[:seen, :dv].contiguous()
    return out, lse


def _rope(x, positions, theta):
    dim = x.shape[-1]
    freq = theta ** (torch.arange(0, dim, 2, dtype=torch.float64, device=x.device) / dim)
    angles = positions.double()[..., None] / freq
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * angles.cos() - b * angles.sin(), b * angles.cos() + a * angles.sin()], dim=-1)


def _norm(x, eps):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps)


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] != "layer":
        q = state["q"] if state["q"].dim() == 4 else state["q"].unsqueeze(1)
        out, lse = _attend(q, state["kv"], state["seqlens"], state["table"], state["dv"], state["softmax_scale"],
                           state["kv_scale"])
        if case["q_len"] == 1:
            out, lse = out.squeeze(1), lse.squeeze(1)
        return {"out": out, "lse": lse} if case["lse"] else {"out": out}
    model, kv, pos = state["model"], state["kv"], state["seqlens"]
    cfg = model.cfg
    weight = {name: p.detach().double() for name, p in model.named_parameters()}
    x = state["x"].double()
    h = cfg.num_heads
    q_lat = _norm(x @ weight["wq_a.weight"].t(), cfg.rms_norm_eps)
    q = (q_lat @ weight["wq_b.weight"].t()).unflatten(-1, (h, 192))
    latent = x @ weight["wkv_a.weight"].t()
    row = torch.cat([_norm(latent[:, :512], cfg.rms_norm_eps), _rope(latent[:, 512:], pos, cfg.rope_theta)], dim=-1)
    w = weight["wkv_b.weight"].unflatten(0, (h, 256))
    absorbed = torch.stack([q[:, i, :128] @ w[i, :128] for i in range(h)], dim=1)
    q = torch.cat([absorbed, _rope(q[..., 128:], pos[:, None], cfg.rope_theta)], dim=-1)
    # attention over the cached rows and the new one
    out = torch.empty(x.shape[0], h, 512, dtype=torch.float64, device=x.device)
    for b, n in enumerate(pos.tolist()):
        ids = state["table"][b, :-(-n // kv.shape[1])].long()
        rows = torch.cat([kv[ids].reshape(-1, 576)[:n].double(), row[b:b + 1]])
        probs = torch.softmax((q[b] @ rows.t().contiguous()) * 192 ** -0.5, dim=-1)
        out[b] = probs @ rows[:, :512].contiguous()
    heads = torch.stack([out[:, i] @ w[i, 128:].t().contiguous() for i in range(h)], dim=1)
    page = state["table"].gather(1, (pos.long() // kv.shape[1])[:, None])[:, 0].long()
    cache = kv.double()
    cache[page, pos.long() % kv.shape[1]] = row
    return {"out": heads.flatten(1) @ weight["wo.weight"].t(), "seqlens": pos + 1, "cache": cache}
