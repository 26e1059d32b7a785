"""The calls whose speed is followed, and how their results are checked.

Each case is one call (or the few calls that go together) a serving program makes through
the package's public entry points: the drafter's cross-attention over the three K/V
layouts, the target's verify attention, tree drafting, the context writer, the sampler,
the several-jump draft's state kernels and a whole pass of the drafter network. ``listed``
names the cases, ``draw`` gives others of the same ranges, ``prepare`` makes what a program
holds before the call, ``run`` is one pass, ``work`` what a pass cannot do without,
``exact`` the same results from plain torch in float64.
"""

from __future__ import annotations

import math

import torch

from flashmap_amd import drafter, ops
from flashmap_amd.verify_attention import SplitKVVerify

DEV = "cuda"
EPS = 1e-6
K_ROWS = 16  # draft slots per block
PAGE = 16


def listed() -> list[dict]:
    return [
        # One user on the transformers path: a single sequence, contiguous cache, the
        # Qwen3-8B-shaped drafter layer. Latency and launches are all it is.
        {"name": "contig_b1", "kind": "attend", "layout": "contig", "fp8": False, "batch": 1, "hq": 32, "hkv": 8,
         "head_dim": 128, "lo": 2048, "hi": 2048, "cand": 1},
        # A lightly loaded vLLM server: a handful of requests of ragged, odd lengths.
        {"name": "paged_b4_ragged", "kind": "attend", "layout": "paged", "fp8": False, "batch": 4, "hq": 32, "hkv": 8,
         "head_dim": 128, "lo": 77, "hi": 3001, "cand": 1},
        # A full vLLM batch, contexts of 256 to 8192: the project's headline call.
        {"name": "paged_b64", "kind": "attend", "layout": "paged", "fp8": False, "batch": 64, "hq": 32, "hkv": 8,
         "head_dim": 128, "lo": 256, "hi": 8192, "cand": 1},
        # Few requests with long contexts.
        {"name": "paged_b8_32k", "kind": "attend", "layout": "paged", "fp8": False, "batch": 8, "hq": 32, "hkv": 8,
         "head_dim": 128, "lo": 32768, "hi": 32768, "cand": 1},
        # The 27B-class drafter: five query heads per KV head.
        {"name": "paged_gqa5_b32", "kind": "attend", "layout": "paged", "fp8": False, "batch": 32, "hq": 40, "hkv": 8,
         "head_dim": 128, "lo": 1024, "hi": 8192, "cand": 1},
        # The full batch on an e4m3 cache (bf16 queries, quantized per head in the call).
        {"name": "paged_fp8_b64", "kind": "attend", "layout": "paged", "fp8": True, "batch": 64, "hq": 32, "hkv": 8,
         "head_dim": 128, "lo": 256, "hi": 8192, "cand": 1},
        # SGLang tree drafting: 8 candidate blocks per request on the 8B drafter's own
        # heads (16 query, 16 KV), token-paged pool.
        {"name": "tree_b4_n8", "kind": "attend", "layout": "token", "fp8": False, "batch": 4, "hq": 16, "hkv": 16,
         "head_dim": 128, "lo": 1024, "hi": 8192, "cand": 8},
        # SGLang's target verification of a 17-token chain per request, full batch.
        {"name": "verify_b64", "kind": "verify", "batch": 64, "hq": 32, "hkv": 8, "head_dim": 128, "lo": 256,
         "hi": 8192, "length": 17},
        # A prompt's context rows into every layer's pages: the K/V of 6 layers at once.
        {"name": "write_prefill", "kind": "write", "fp8": False, "tokens": 8192, "layers": 6, "heads": 16,
         "head_dim": 128},
        # SGLang's sampler over the draft logits of a full batch, half the requests greedy.
        {"name": "sample_b64", "kind": "sample", "rows": 1024, "vocab": 151936, "greedy_share": 0.5},
        # Between the jumps of a two-jump draft: the vocabulary-sized state moves to the
        # jump head's distribution and is embedded for the next jump.
        {"name": "jump_state_b64", "kind": "state", "rows": 1024, "vocab": 151936},
        # One pass of the whole released 8B drafter network for one user.
        {"name": "drafter_b1", "kind": "network", "batch": 1, "context": 2047},
    ]


def _between(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["attend", "attend", "attend", "attend", "tree", "verify", "write", "sample", "state", "network"])
    if kind in ("attend", "tree"):
        layout = "token" if kind == "tree" else rng.choice(["contig", "paged", "paged", "token"])
        fp8 = layout == "paged" and rng.random() < 0.4
        hq, hkv = rng.choice([(16, 16), (32, 8), (32, 8), (40, 8), (64, 8)])
        head_dim = 64 if rng.random() < 0.15 else 128
        cand = rng.choice([2, 3, 4, 8, 16]) if kind == "tree" else 1
        batch = _between(rng, 1, 8) if kind == "tree" else _between(rng, 1, 64)
        # At most the full batch's bytes of K/V, and not more work than the largest case.
        top = min(32768, (1 << 30) // (batch * hkv * head_dim * 4),
                  10 ** 11 // (4 * cand * K_ROWS * hq * head_dim * batch))
        hi = _between(rng, 64, top)
        return {"kind": "attend", "layout": layout, "fp8": fp8, "batch": batch, "hq": hq, "hkv": hkv,
                "head_dim": head_dim, "lo": rng.randint(max(1, hi // 32), hi), "hi": hi, "cand": cand}
    if kind == "verify":
        batch = _between(rng, 1, 64)
        hq, hkv = rng.choice([(16, 16), (32, 8), (40, 8)])
        hi = _between(rng, 64, min(16384, 4194304 // (batch * hkv)))
        return {"kind": "verify", "batch": batch, "hq": hq, "hkv": hkv, "head_dim": 128,
                "lo": rng.randint(max(1, hi // 32), hi), "hi": hi, "length": rng.randint(2, 24)}
    if kind == "write":
        return {"kind": "write", "fp8": rng.random() < 0.5, "tokens": _between(rng, 16, 8192),
                "layers": rng.randint(1, 6), "heads": rng.choice([8, 16]), "head_dim": rng.choice([64, 128, 128])}
    if kind == "sample":
        return {"kind": "sample", "rows": 16 * _between(rng, 1, 64), "vocab": rng.randint(32000, 151936),
                "greedy_share": rng.choice([0.0, 0.5, 1.0])}
    if kind == "state":
        return {"kind": "state", "rows": 16 * _between(rng, 1, 64), "vocab": rng.randint(16384, 151936)}
    return {"kind": "network", "batch": _between(rng, 1, 4), "context": _between(rng, 64, 4096)}


# ------------------------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _lens(case: dict, seed: int) -> list[int]:
    g = torch.Generator().manual_seed(seed)
    return [int(n) for n in torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g)]


def _normal(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _e4m3(shape, g):
    """Unit normals in e4m3 (made in slices: the float32 copies stay small)."""
    out = torch.empty(shape, dtype=torch.float8_e4m3fn, device=DEV)
    for part in out.split(max(1, (1 << 26) // max(1, math.prod(shape[1:])))):
        part.copy_(torch.randn(part.shape, generator=g, device=DEV))
    return out


def _prologue(case: dict, positions: torch.Tensor, g) -> tuple[torch.Tensor, torch.Tensor]:
    """Query-norm weights and the rotary table ``(rows, D / 2, [cos, sin])``."""
    d = case["head_dim"]
    weight = 0.75 + 0.5 * torch.rand(d, generator=g, device=DEV)
    inv = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV).float() / d)
    angles = torch.arange(int(positions.max()) + 2, device=DEV).float()[:, None] * inv
    return weight, torch.stack([angles.cos(), angles.sin()], dim=-1).contiguous()


def _attend_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    batch, hq, hkv, d, rows = case["batch"], case["hq"], case["hkv"], case["head_dim"], case["cand"] * K_ROWS
    lens = _lens(case, seed)
    lens_d = torch.tensor(lens, dtype=torch.int32, device=DEV)
    # Every candidate's block stands at the positions after the context.
    pos = (lens_d[:, None].long() + torch.arange(K_ROWS, device=DEV).repeat(case["cand"])).reshape(-1)
    weight, table = _prologue(case, pos, g)
    s = {"case": case, "lens": lens, "lens_d": lens_d, "pos": pos, "weight": weight, "table": table, "scale": d ** -0.5,
         "q": _normal(g, batch, rows, hq, d)}
    if case["layout"] == "contig":
        s["k"], s["v"] = _normal(g, batch, hkv, max(lens), d), _normal(g, batch, hkv, max(lens), d)
    elif case["layout"] == "paged":
        pages = [-(-n // PAGE) for n in lens]
        perm = torch.randperm(sum(pages), generator=g, device=DEV).int()
        bt = torch.zeros(batch, max(pages), dtype=torch.int32, device=DEV)
        o = 0
        for b, n in enumerate(pages):
            bt[b, :n] = perm[o:o + n]
            o += n
        s["bt"] = bt
        shape = (sum(pages), hkv, PAGE, 2 * d)
        s["cache"] = _e4m3(shape, g) if case["fp8"] else _normal(g, *shape)
    else:
        perm = torch.randperm(sum(lens), generator=g, device=DEV).int()
        pt = torch.zeros(batch, max(lens), dtype=torch.int32, device=DEV)
        o = 0
        for b, n in enumerate(lens):
            pt[b, :n] = perm[o:o + n]
            o += n
        s["pt"] = pt
        s["k"], s["v"] = _normal(g, sum(lens), hkv, d), _normal(g, sum(lens), hkv, d)
    return s


def _verify_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    hq, hkv, d, lens = case["hq"], case["hkv"], case["head_dim"], _lens(case, seed)
    tokens = case["batch"] * case["length"]
    indptr = torch.zeros(case["batch"] + 1, dtype=torch.int32)
    indptr[1:] = torch.tensor(lens).cumsum(0)
    return {"case": case, "lens": lens, "indptr": indptr.to(DEV),
            "indices": torch.randperm(sum(lens), generator=g, device=DEV),
            "qo_indptr": torch.arange(0, tokens + 1, case["length"], dtype=torch.int32, device=DEV),
            "q": _normal(g, tokens, hq, d), "k": _normal(g, tokens, hkv, d), "v": _normal(g, tokens, hkv, d),
            "o": torch.empty(tokens, hq, d, dtype=torch.bfloat16, device=DEV),
            "pool_k": _normal(g, sum(lens), hkv, d), "pool_v": _normal(g, sum(lens), hkv, d), "scale": d ** -0.5}


def _write_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    n, layers, heads, d = case["tokens"], case["layers"], case["heads"], case["head_dim"]
    first = seed % 3001  # the rows continue a request that already holds some
    pos = torch.arange(first, first + n, device=DEV)
    _, table = _prologue(case, pos, g)
    pages = -(-n // PAGE) + 3
    slots = torch.randperm(pages, generator=g, device=DEV)[torch.arange(n, device=DEV) // PAGE] * PAGE
    dtype = torch.uint8 if case["fp8"] else torch.bfloat16
    caches = [torch.zeros(pages, heads, PAGE, 2 * d, dtype=dtype, device=DEV) for _ in range(layers)]
    return {"case": case, "kv": _normal(g, n, layers, 2, heads, d), "pos": pos, "table": table,
            "slots": slots + torch.arange(n, device=DEV) % PAGE, "caches": caches,
            "norm": 0.75 + 0.5 * torch.rand(layers, d, generator=g, device=DEV),
            "scales": 0.02 + 0.02 * torch.rand(layers, 2, generator=g, device=DEV)}


def _sample_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    rows, vocab = case["rows"], case["vocab"]
    # A language model's logits: a wide bulk and a few likely tokens far above it.
    logits = _normal(g, rows, vocab) * 2.5
    likely = torch.randint(0, vocab, (rows, 24), generator=g, device=DEV)
    logits.scatter_(1, likely, (8 + 14 * torch.rand(rows, 24, generator=g, device=DEV)).bfloat16())
    greedy = torch.zeros(rows, dtype=torch.bool, device=DEV)
    greedy[:int(rows * case["greedy_share"])] = True
    temps = 0.6 + 0.6 * torch.rand(rows, generator=g, device=DEV)
    return {"case": case, "logits": logits, "greedy": greedy[torch.randperm(rows, generator=g, device=DEV)],
            "temps": temps, "seed": torch.tensor(seed + 1, dtype=torch.int64, device=DEV)}


def _state_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    rows, vocab = case["rows"], case["vocab"]
    padded = -(-vocab // 4) * 4  # as the draft step lays its state and its operand out
    state = torch.randn(rows, padded, generator=g, device=DEV)[:, :vocab]
    logits = torch.randn(rows, padded, generator=g, device=DEV, dtype=torch.bfloat16)[:, :vocab] * 2.5
    start, end, _ = drafter.drafter_config().jump_grids["2"]
    return {"case": case, "state": state, "logits": logits, "start": start, "end": end,
            "evidence": end / max(1.0 - end, 1e-3) ** 2,
            "operand": torch.empty(2 * rows, padded, dtype=torch.bfloat16, device=DEV)[:, :vocab]}


def _network_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    batch, ctx = case["batch"], case["context"]
    with torch.device(DEV):
        torch.cuda.manual_seed(seed)
        model = drafter.FlashMapDraftModel().to(torch.bfloat16)
    cfg = model.config
    cache = drafter.FlashMapCache(cfg, batch, ctx + K_ROWS, device=DEV, dtype=torch.bfloat16)
    cache.kv.normal_(generator=g)
    pos = (ctx + 1 + torch.arange(K_ROWS, device=DEV)).expand(batch, K_ROWS)
    return {"case": case, "model": model, "context": cache.context(ctx + 1), "pos": pos,
            "x": _normal(g, batch, K_ROWS, cfg.target_hidden_size),
            "lm_head": _normal(g, 32000, cfg.target_hidden_size) / 64}


_INPUTS = {"attend": _attend_inputs, "verify": _verify_inputs, "write": _write_inputs, "sample": _sample_inputs,
           "state": _state_inputs, "network": _network_inputs}


def prepare(case: dict, seed: int) -> dict:
    s = _INPUTS[case["kind"]](case, seed)
    if case["kind"] == "attend":
        s["prologue"] = ops.Prologue(s["weight"], ops.rope_from_table(s["table"]), s["pos"], EPS)
        s["plan"] = ops.attention_plan(s["lens_d"])  # one per step, shared by its layers
        batch, rows = case["batch"], case["cand"] * K_ROWS
        if case["layout"] == "paged":
            s["q"] = s["q"].view(batch * rows, case["hq"], case["head_dim"])
            s["cu"] = torch.arange(0, batch * rows + 1, rows, dtype=torch.int32, device=DEV)
    elif case["kind"] == "verify":
        s["verify"] = SplitKVVerify()
    elif case["kind"] == "write":
        c = s["caches"][0]
        s["rope"] = ops.rope_from_table(s["table"])
        s["ptrs"] = torch.tensor([c.data_ptr() for c in s["caches"]], dtype=torch.int64, device=DEV)
        s["strides"] = (c.stride(0), c.stride(1), c.stride(2), case["head_dim"])
    return s


# --------------------------------------------------------------------------------- a pass


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "attend":
        kw = {"prologue": s["prologue"], "plan": s["plan"]}
        if case["layout"] == "contig":
            return ops.block_attention_contig(s["q"], s["k"], s["v"], s["scale"], s["lens_d"], **kw)
        if case["layout"] == "paged":
            attend = ops.block_attention_paged_fp8 if case["fp8"] else ops.block_attention_paged
            return attend(s["q"], s["cache"], s["cu"], s["lens_d"], s["bt"], case["cand"] * K_ROWS, case["hi"],
                          s["scale"], **kw)
        return ops.block_attention_token_paged(s["q"], s["k"], s["v"], s["lens_d"], s["pt"], s["scale"], **kw)
    if kind == "verify":
        handled = s["verify"](s["q"], s["k"], s["v"], s["o"], s["pool_k"], s["pool_v"], s["qo_indptr"], s["indptr"],
                              s["indices"], None, True, None, case["length"], sm_scale=s["scale"])
        if not handled:
            raise RuntimeError("the verify batch was declined")
        return s["o"]
    if kind == "write":
        args = (s["kv"], s["pos"], s["slots"], s["norm"], s["rope"], s["ptrs"], s["strides"], PAGE, EPS)
        if case["fp8"]:
            ops.write_context_kv_fp8(*args, s["scales"])
        else:
            ops.write_context_kv(*args)
        return s["caches"]
    if kind == "sample":
        return ops.sample_rows(s["logits"], s["temps"], s["greedy"], s["seed"])
    if kind == "state":
        ops.state_update(s["state"], s["logits"], s["start"], s["end"])
        return s["state"], ops.state_embed_rows(s["state"], s["evidence"], out=s["operand"])
    with torch.no_grad():
        hidden = s["model"](s["x"], 0.0, 1.0, s["pos"], s["context"])
        return hidden, hidden @ s["lm_head"].T


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("attend", "verify"):
        d, hq, hkv, batch = case["head_dim"], case["hq"], case["hkv"], case["batch"]
        positions = batch * (case["lo"] + case["hi"]) // 2
        rows = case["length"] if kind == "verify" else case["cand"] * K_ROWS
        es = 1 if case.get("fp8") else 2
        total = positions * hkv * d * 2 * es + 2 * batch * rows * hq * d * 2
        flops = 4 * rows * hq * d * positions
        if kind == "verify":
            total += 2 * batch * rows * hkv * d * 2 + 8 * positions
            flops += 4 * batch * rows * rows * hq * d
        else:
            total += batch * rows * d * 4 + (0 if case["layout"] == "contig" else
                                             4 * positions // (PAGE if case["layout"] == "paged" else 1))
        return {"bytes": total, "flops": flops}
    if kind == "write":
        values = case["tokens"] * case["layers"] * 2 * case["heads"] * case["head_dim"]
        return {"bytes": values * (3 if case["fp8"] else 4) + case["tokens"] * (16 + 4 * case["head_dim"]),
                "flops": 8 * values}
    n = case.get("rows", 0) * case.get("vocab", 0)
    if kind == "sample":
        return {"bytes": 2 * n + 8 * case["rows"], "flops": 0}
    if kind == "state":  # logits and state in; state, posterior and bf16 state out
        return {"bytes": n * (2 + 4 + 4 + 2 + 2), "flops": 16 * n}
    cfg = drafter.drafter_config()
    dim, target = cfg.hidden_size, cfg.target_hidden_size
    # per layer: self q/k/v/o, cross q/o, the MLP (the context's keys and values are given)
    weights = 2 * target * dim + cfg.num_hidden_layers * (6 * dim * dim + 2 * dim * cfg.intermediate_size) \
        + 32000 * target
    tokens, ctx = case["batch"] * K_ROWS, case["batch"] * (case["context"] + 1)
    return {"bytes": 2 * weights + cfg.num_hidden_layers * ctx * dim * 4 + 2 * tokens * (2 * target + 32000),
            "flops": 2 * tokens * weights + cfg.num_hidden_layers * 4 * dim * tokens * (case["context"] + 1 + K_ROWS)}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("attend", "verify"):
        # bf16 probabilities and outputs (2.3e-3 from float64; 2.6e-3 on e4m3 caches)
        return {"rel": 1e-2, "max": 0.1}
    if kind == "write":
        return {"rel": 4e-3, "max": 0.02, "differ": 0.01}
    if kind == "sample":
        return "exact"  # tokens of a fixed random stream
    if kind == "state":
        return {"rel": 1e-3, "max": 0.02}  # the bf16 operand: rounding ties
    return {"rel": 3e-2, "max": 0.4}  # six bf16 layers (6e-3 to 8e-3 from float64)


# ------------------------------------------------------------------------- in 64 bits


def _norm_rope64(x, weight, table, pos):
    """RMSNorm (its scale and its result rounded to the input's bf16, as the model's
    definition has it) and interleaved RoPE of ``x (..., T, heads, D)``, ``pos (T,)``."""
    x = x.double()
    scale = weight.double() * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    y = (x * scale.bfloat16().double()).bfloat16().double()
    cos, sin = (table[pos].double()[..., i][..., None, :] for i in (0, 1))
    e, o = y[..., 0::2], y[..., 1::2]
    return torch.stack([e * cos - o * sin, o * cos + e * sin], dim=-1).flatten(-2)


def _softmax_attend64(q, k, v, scale, mask=None):
    """``q (T, hq, D)`` onto ``k, v (hkv, L, D)``, all float64; ``(T, hq, D)``."""
    hkv = k.shape[0]
    t, hq, d = q.shape
    rows = q.transpose(0, 1).reshape(hkv, (hq // hkv) * t, d)
    s = torch.matmul(rows, k.transpose(1, 2).contiguous()) * scale
    if mask is not None:
        s = s.masked_fill(~mask.repeat(hq // hkv, 1), -math.inf)
    out = torch.matmul(s.softmax(-1), v)
    return out.view(hq, t, d).transpose(0, 1)


def _exact_attend(case, seed):
    s = _attend_inputs(case, seed)
    batch, rows, d = case["batch"], case["cand"] * K_ROWS, case["head_dim"]
    out = []
    for b, n in enumerate(s["lens"]):
        q = _norm_rope64(s["q"][b], s["weight"], s["table"], s["pos"].view(batch, rows)[b]).bfloat16()
        if case["fp8"]:  # the rows of each head quantized with their own scale
            scale = q.float().abs().amax((0, 2), keepdim=True).clamp_min(1e-12) / 448.0
            q = (q.float() / scale).to(torch.float8_e4m3fn).double() * scale.double()
        if case["layout"] == "contig":
            k, v = s["k"][b, :, :n], s["v"][b, :, :n]
        elif case["layout"] == "paged":
            at = torch.arange(n, device=DEV)
            cache = s["cache"].view(torch.uint8) if case["fp8"] else s["cache"]
            kv = cache[s["bt"][b, at // PAGE].long(), :, at % PAGE]
            kv = (kv.view(torch.float8_e4m3fn) if case["fp8"] else kv).transpose(0, 1)
            k, v = kv[..., :d], kv[..., d:]
        else:
            at = s["pt"][b, :n].long()
            k, v = s["k"][at].transpose(0, 1), s["v"][at].transpose(0, 1)
        out.append(_softmax_attend64(q.double(), k.double(), v.double(), s["scale"]))
    out = torch.stack(out)
    return out.reshape(batch * rows, case["hq"], d) if case["layout"] == "paged" else out


def _exact_verify(case, seed):
    s = _verify_inputs(case, seed)
    t, out, first = case["length"], [], 0
    for b, n in enumerate(s["lens"]):
        at, own = s["indices"][first:first + n], slice(b * t, (b + 1) * t)
        first += n
        k = torch.cat([s["pool_k"][at], s["k"][own]]).transpose(0, 1).double()
        v = torch.cat([s["pool_v"][at], s["v"][own]]).transpose(0, 1).double()
        seen = torch.ones(t, n + t, dtype=torch.bool, device=DEV).tril(n)
        out.append(_softmax_attend64(s["q"][own].double(), k, v, s["scale"], seen))
    return torch.cat(out)


def _exact_write(case, seed):
    if case["fp8"]:
        return None  # bytes
    s = _write_inputs(case, seed)
    d = case["head_dim"]
    out = []
    for i, cache in enumerate(s["caches"]):
        rows = cache.double().transpose(1, 2)  # (pages, page, heads, 2 D)
        keys = _norm_rope64(s["kv"][:, i, 0], s["norm"][i], s["table"], s["pos"])
        rows[s["slots"] // PAGE, s["slots"] % PAGE] = torch.cat([keys, s["kv"][:, i, 1].double()], dim=-1)
        out.append(rows.transpose(1, 2))
    return out


def _exact_state(case, seed):
    s = _state_inputs(case, seed)
    post = torch.empty(2 * case["rows"], case["vocab"], dtype=torch.float64, device=DEV)
    state = torch.empty(case["rows"], case["vocab"], dtype=torch.float64, device=DEV)
    for i in range(0, case["rows"], 64):
        part = slice(i, min(i + 64, case["rows"]))
        moved = ((1 - s["end"]) * s["state"][part].double()
                 + (s["end"] - s["start"]) * s["logits"][part].double().softmax(-1)) / (1 - s["start"])
        state[part] = moved
        post[part] = (s["evidence"] * moved).softmax(-1)
        post[case["rows"] + part.start:case["rows"] + part.stop] = moved
    return state, post


def _exact_network(case, seed):
    s = _network_inputs(case, seed)
    model, cfg = s["model"], s["model"].config
    w = {n: p.detach().double() for n, p in model.named_parameters()}
    d, heads = model.head_dim, cfg.num_attention_heads
    inv = 1.0 / cfg.rope_theta ** (torch.arange(0, d, 2, device=DEV).double() / d)
    angles = s["pos"][0].double()[:, None] * inv
    table, at = torch.stack([angles.cos(), angles.sin()], dim=-1), torch.arange(K_ROWS, device=DEV)

    def linear(x, name):
        y = x @ w[name + ".weight"].T
        return y + w[name + ".bias"] if name + ".bias" in w else y

    def normed(x, name):  # (T, dim) -> heads, normed and rotated
        x = x.view(K_ROWS, heads, d)
        y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.qk_norm_eps) * w[name + ".weight"]
        cos, sin = (table[at][..., i][:, None] for i in (0, 1))
        e, o = y[..., 0::2], y[..., 1::2]
        return torch.stack([e * cos - o * sin, o * cos + e * sin], dim=-1).flatten(-2)

    def layer_norm(x, scale, shift):
        y = (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + cfg.layer_norm_eps)
        return y * (1 + scale) + shift

    silu, gelu = torch.nn.functional.silu, torch.nn.functional.gelu
    cond = 0
    for t, name in ((0.0, "time_embed"), (1.0, "jump_embed")):
        half = cfg.time_embed_dim // 2
        freqs = torch.exp(-math.log(10000.0) * torch.arange(half, device=DEV).double() / half)
        a = t * cfg.time_scale * freqs
        cond = cond + linear(silu(linear(torch.cat([a.cos(), a.sin()]), name + ".linear_1")), name + ".linear_2")
    mods = lambda name: linear(silu(cond), name + ".linear").chunk(3)  # noqa: E731
    out = []
    for b in range(case["batch"]):
        x = linear(s["x"][b].double(), "x_embed")
        for i, (keys, values) in enumerate(s["context"]):
            p = f"layers.{i}."
            scale, shift, gate = mods(p + "self_attn_adaln")
            h = layer_norm(x, scale, shift)
            q, k = (normed(linear(h, f"{p}self_attn.{n}_proj"), f"{p}self_attn.{n}_norm") for n in "qk")
            v = linear(h, p + "self_attn.v_proj").view(K_ROWS, heads, d)
            y = _softmax_attend64(q, k.transpose(0, 1), v.transpose(0, 1), d ** -0.5)
            x = x + gate * linear(y.reshape(K_ROWS, -1), p + "self_attn.o_proj")
            scale, shift, gate = mods(p + "cross_attn_adaln")
            q = normed(linear(layer_norm(x, scale, shift), p + "cross_attn.q_proj"), p + "cross_attn.q_norm")
            y = _softmax_attend64(q, keys[b].double(), values[b].double(), d ** -0.5)
            x = x + gate * linear(y.reshape(K_ROWS, -1), p + "cross_attn.o_proj")
            scale, shift, gate = mods(p + "mlp_adaln")
            x = x + gate * linear(gelu(linear(layer_norm(x, scale, shift), p + "mlp.fc1")), p + "mlp.fc2")
        scale, shift, _ = mods("final_adaln")
        out.append(linear(layer_norm(x, scale, shift), "head"))
    hidden = torch.stack(out)
    return hidden, hidden @ s["lm_head"].double().T


_EXACT = {"attend": _exact_attend, "verify": _exact_verify, "write": _exact_write, "state": _exact_state,
          "network": _exact_network}


def exact(case: dict, seed: int):
    """What ``run`` gives for these inputs, from plain torch in float64; None for the
    sampler (token ids of a float32 stream) and for e4m3 bytes."""
    return _EXACT[case["kind"]](case, seed) if case["kind"] in _EXACT else None
