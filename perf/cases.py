"""The calls whose speed this framework is judged by, one pass each.

Every case is a layer, a block or a whole model as a program that serves the hybrid
block stack calls it through ``hybrid_llm_amd.ops`` or ``HybridDecoder``: the MoE
layer, banded attention, the gated delta rule, the dense projections, the
compressed-memory mixers, the vocabulary head with its draw, the prefill of a block
and whole decode steps.  A prefill is measured through one block, not twelve twice
over: a change of rounding in one layer makes later routers take other experts at
near-ties, and logits after 24 of them differ by a quarter between two orders of the
same sums.  Sizes are those of the configurations in ``hybrid_llm_amd.config`` (C1,
C5), of the op shapes ``bench.py`` reports and of ragged prompts in between.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges; a case is
a dict of plain values.  ``prepare`` makes what a program holds before the call,
``run`` is one call, ``exact`` the same in 64 bits without this package's code.
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch
import torch.nn.functional as F

from hybrid_llm_amd import ops
from hybrid_llm_amd.config import C1, C5, alternating, init_weights
from hybrid_llm_amd.engine import HybridDecoder

DEV = "cuda"
BF16 = torch.bfloat16

# index heads x head width, compression ratio, top-k (0 = dense) and d_model of the
# two compressed-memory mixers; local window and decode memory slots are shared
CMP = {"csa": (16, 128, 4, 32), "hca": (1, 1024, 32, 0)}
CMP_D, CMP_WINDOW, CMP_SLOTS = 1024, 128, 256

# (N, K) of the C5 projections over a prompt or a decode batch (q/k/v stacked, output,
# GDN input) and of C1's q/k/v
PROJECTIONS = ((3072, 1024), (1024, 1024), (4112, 1024), (768, 256))


def listed():
    return [
        # one token of one sequence through C1's MoE layer: a chat's next token
        {"name": "moe_one_token", "family": "moe", "tokens": 1, "d_model": 256, "experts": 8,
         "top_k": 2, "hidden": 512},
        # a decode batch of 64 sequences through the 24-expert MoE layer
        {"name": "moe_decode_64", "family": "moe", "tokens": 64, "d_model": 1024, "experts": 24,
         "top_k": 2, "hidden": 2048},
        # a 4096-token prompt through the same layer
        {"name": "moe_prompt_4096", "family": "moe", "tokens": 4096, "d_model": 1024,
         "experts": 24, "top_k": 2, "hidden": 2048},
        # banded attention over four long prompts
        {"name": "attn_prompt_4x8192", "family": "attn", "batch": 4, "tokens": 8192, "heads": 16,
         "head_dim": 64, "window": 512},
        # one new token each of 64 sequences against full 2048-token windows
        {"name": "attn_decode_64", "family": "attn_decode", "batch": 64, "heads": 16,
         "head_dim": 64, "window": 2048},
        # the gated delta rule over eight long prompts, 128-wide heads
        {"name": "gdn_prompt_8x4096", "family": "gdn", "batch": 8, "tokens": 4096, "heads": 16,
         "width": 128, "reset": False},
        # the same layer over one user's prompt of odd length, C5's 64-wide heads
        {"name": "gdn_prompt_1x1003", "family": "gdn", "batch": 1, "tokens": 1003, "heads": 16,
         "width": 64, "reset": False},
        # C5's q/k/v projection over a 4096-token prompt
        {"name": "qkv_prompt_4096", "family": "linear", "rows": 4096, "n": 3072, "k": 1024,
         "epilogue": "bf16"},
        # both branches of the CSA mixer over one 4096-token prompt
        {"name": "csa_prompt_4096", "family": "cmp_prompt", "kind": "csa", "batch": 1,
         "tokens": 4096},
        # the vocabulary head of a decode batch: logits, greedy ids, nucleus draw
        {"name": "head_64", "family": "head", "rows": 64, "vocab": 32000, "d_model": 1024,
         "temperature": 0.8, "top_p": 0.9, "top_k": 0},
        # prefill of eight 512-token prompts through a GDN block of C5 (projection, delta
        # rule, MoE), from token ids to the last positions' logits
        {"name": "block_prompt_8x512", "family": "block_prompt", "model": "c5", "kind": "gdn",
         "batch": 8, "tokens": 512},
        # whole-model decode step of 64 sequences with full windows
        {"name": "model_step_64", "family": "model_step", "model": "c5", "layers": 12,
         "batch": 64},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(("moe", "moe", "attn", "attn_decode", "gdn", "gdn", "gdn_step", "linear",
                         "cmp_prompt", "cmp_step", "head", "block_prompt", "block_prompt",
                         "model_step"))
    c = {"family": family}
    if family == "moe":
        big = rng.random() < 0.75
        c.update(tokens=_log(rng, 1, 4096), d_model=1024 if big else 256,
                 experts=24 if big else 8, top_k=2, hidden=2048 if big else 512)
    elif family == "attn":
        hd = rng.choice((64, 64, 128))
        c.update(batch=rng.randint(1, 4), tokens=_log(rng, 16, 8192), heads=1024 // hd,
                 head_dim=hd, window=rng.choice((128, 512, 2048)))
        if c["window"] == 2048:
            c["batch"] = 1
    elif family == "attn_decode":
        hd = rng.choice((64, 64, 128))
        c.update(batch=_log(rng, 1, 64), heads=1024 // hd, head_dim=hd,
                 window=rng.choice((128, 512, 2048)))
    elif family == "gdn":
        c.update(batch=rng.randint(1, 8), tokens=_log(rng, 24, 4096), heads=rng.choice((4, 16)),
                 width=rng.choice((64, 128)), reset=rng.random() < 0.25)
    elif family == "gdn_step":
        c.update(batch=_log(rng, 1, 64), heads=16, width=rng.choice((64, 128)))
    elif family == "linear":
        n, k = rng.choice(PROJECTIONS)
        c.update(rows=_log(rng, 1, 4096), n=n, k=k,
                 epilogue=rng.choice(("bf16", "f32", "residual", "gated")))
    elif family == "cmp_prompt":
        c.update(kind=rng.choice(("csa", "hca")), batch=1, tokens=_log(rng, 64, 4096))
    elif family == "cmp_step":
        c.update(kind=rng.choice(("csa", "hca")), batch=_log(rng, 1, 64))
    elif family == "head":
        c.update(rows=_log(rng, 1, 64), vocab=rng.choice((8192, 32000)),
                 d_model=rng.choice((256, 1024)), temperature=round(rng.uniform(0.5, 1.2), 3),
                 top_p=round(rng.uniform(0.5, 0.98), 3), top_k=rng.choice((0, 0, 40)))
    elif family == "block_prompt":
        c.update(model=rng.choice(("c1", "c5", "c5")), kind=rng.choice(("attn", "gdn")),
                 batch=rng.randint(1, 8), tokens=_log(rng, 24, 1024))
    else:
        c["model"] = rng.choice(("c1", "c5"))
        c["layers"] = 4 if c["model"] == "c1" else rng.choice((2, 4))
        c["batch"] = _log(rng, 1, 64)
    return c


# ----------------------------------------------------------------------- inputs
def _config(c):
    base = C1 if c["model"] == "c1" else C5
    if c["family"] == "block_prompt":
        return replace(base, layer_kinds=(c["kind"],), num_loops=1)
    return replace(base, layer_kinds=alternating(c["layers"]))


def prepare(c, seed):
    """Inputs, weights and engines of one case, made on the GPU from the seed."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def randn(*shape, std=1.0):
        return torch.empty(shape, device=DEV).normal_(0.0, std, generator=g)

    def rand(*shape):
        return torch.rand(shape, device=DEV, generator=g)

    s = {"case": c}
    f = c["family"]
    if f == "moe":
        T, D, E, H = c["tokens"], c["d_model"], c["experts"], c["hidden"]
        s["x"] = randn(T, D).to(BF16)
        s["w_router"] = randn(E, D, std=0.02)
        s["w_gate_up"] = ops.pack_weights(randn(E, 2 * H, D, std=0.02).to(BF16))
        s["w_down"] = ops.pack_weights(randn(E, D, H, std=0.02).to(BF16))
    elif f == "attn":
        shape = (c["batch"], c["tokens"], c["heads"], c["head_dim"])
        s["q"], s["k"], s["v"] = (randn(*shape).to(BF16) for _ in range(3))
    elif f == "attn_decode":
        B, H, hd, W = c["batch"], c["heads"], c["head_dim"], c["window"]
        s["qkv"] = randn(B, 3, H, hd).to(BF16)
        s["k_cache"], s["v_cache"] = (randn(B, H, W, hd).to(BF16) for _ in range(2))
        s["pos"] = torch.randint(W, 4 * W, (B,), device=DEV, dtype=torch.int32, generator=g)
    elif f in ("gdn", "gdn_step"):
        B, H, d = c["batch"], c["heads"], c["width"]
        lead = (B, c["tokens"], H) if f == "gdn" else (B, H)
        s["q"], s["k"] = (F.normalize(randn(*lead, d), dim=-1).to(BF16) for _ in range(2))
        s["v"] = randn(*lead, d).to(BF16)
        s["beta"] = torch.sigmoid(randn(*lead))
        s["g"] = torch.exp(-F.softplus(randn(*lead)))
        s["state"] = randn(B, H, d, d, std=0.1)
        if f == "gdn_step":
            s["gate"] = torch.sigmoid(randn(*lead, d)).to(BF16)
        else:
            s["reset"] = (rand(B, c["tokens"]) < 1 / 256).to(torch.int32) if c["reset"] else None
    elif f == "linear":
        s["x"] = randn(c["rows"], c["k"]).to(BF16)
        s["w"] = ops.pack_weights(randn(c["n"], c["k"], std=0.02).to(BF16))
        if c["epilogue"] in ("residual", "gated"):
            s["out"] = randn(c["rows"], c["n"])
        if c["epilogue"] == "gated":
            s["aux"] = torch.sigmoid(randn(c["rows"], c["n"]))
    elif f in ("cmp_prompt", "cmp_step"):
        H, Dh, ratio, top_k = CMP[c["kind"]]
        Kw, W, C, D, B = H * Dh, CMP_WINDOW, CMP_SLOTS, CMP_D, c["batch"]
        rows = B * c["tokens"] if f == "cmp_prompt" else B
        qkv = randn(rows, 2 * Kw + D).to(BF16)
        s["q"], s["k"], s["v"] = qkv[:, :Kw], qkv[:, Kw:2 * Kw], qkv[:, 2 * Kw:]
        s["out"] = torch.empty(rows, 2 * D, dtype=BF16, device=DEV)
        if f == "cmp_prompt":
            n = c["tokens"] // ratio
            kv = randn(B * n, Kw + D).to(BF16)
            s["mk"], s["mv"] = kv[:, :Kw], kv[:, Kw:]
            s["ws_local"] = ops.cmp_workspace(rows, H, W, 0, DEV)
            s["ws_memory"] = ops.cmp_workspace(rows, H, max(n, 1), top_k, DEV)
        else:
            s["ring_k"], s["ring_v"] = randn(B, W, Kw).to(BF16), randn(B, W, D).to(BF16)
            s["mk"], s["mv"] = randn(B, C, Kw).to(BF16), randn(B, C, D).to(BF16)
            s["tag"] = torch.arange(1, C + 1, device=DEV, dtype=torch.int32).repeat(B, 1)
            s["pos"] = torch.randint(2 * C * ratio, 4 * C * ratio, (B,), device=DEV,
                                     dtype=torch.int32, generator=g)
            s["ws_local"] = ops.cmp_workspace(B, H, W, 0, DEV, decode=True)
            s["ws_memory"] = ops.cmp_workspace(B, H, C, top_k, DEV, decode=True)
    elif f == "head":
        s["h"] = randn(c["rows"], c["d_model"]).to(BF16)
        # logits of a spread that a nucleus of some hundred ids meets
        s["w"] = ops.pack_weights(randn(c["vocab"], c["d_model"],
                                        std=3 / math.sqrt(c["d_model"])).to(BF16))
        s["u"] = rand(c["rows"])
    else:
        cfg = _config(c)
        weights = init_weights(cfg, seed=int(seed), device=DEV)
        step = f == "model_step"
        eng = HybridDecoder(cfg, weights, c["batch"], device=DEV,
                            sampling=(0.8, 0.9, 0) if step else None)
        del weights
        shape = (c["batch"],) if step else (c["batch"], c["tokens"])
        s["tokens"] = torch.randint(0, cfg.vocab, shape, device=DEV, dtype=torch.int32,
                                    generator=g)
        s["engine"] = eng
        if step:
            eng.set_uniforms(rand(c["batch"]))
            eng.pos.fill_(cfg.window)
            for st in eng.state.values():
                for name, t in st.items():
                    t.normal_(0.0, 0.1 if name == "S" else 1.0, generator=g)
            eng.capture()
    return s


# ----------------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    f = c["family"]
    if f == "moe":
        return ops.moe_forward(s["x"], s["w_router"], s["w_gate_up"], s["w_down"], c["top_k"],
                               layout=ops.LAYOUT_PACKED)
    if f == "attn":
        return ops.banded_attn_prefill(s["q"], s["k"], s["v"], c["window"])
    if f == "attn_decode":
        q, k, v = s["qkv"].unbind(1)
        out = ops.banded_attn_decode(q, k, v, s["k_cache"], s["v_cache"], s["pos"])
        return {"out": out, "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if f == "gdn":
        out = ops.gdn_prefill(s["q"], s["k"], s["v"], s["beta"], s["g"], s["state"],
                              reset=s["reset"])
        return {"out": out, "state": s["state"]}
    if f == "gdn_step":
        out = ops.gdn_step(s["q"], s["k"], s["v"], s["beta"], s["g"], s["state"], gate=s["gate"])
        return {"out": out, "state": s["state"]}
    if f == "linear":
        epi = {"bf16": ops.EPI_STORE_BF16, "f32": ops.EPI_STORE_F32,
               "residual": ops.EPI_RESID_ADD, "gated": ops.EPI_RESID_GATED}[c["epilogue"]]
        return ops.linear(s["x"], s["w"], out=s.get("out"), epilogue=epi, aux=s.get("aux"),
                          layout=ops.LAYOUT_PACKED)
    if f == "cmp_prompt":
        H, Dh, ratio, top_k = CMP[c["kind"]]
        D, out = CMP_D, s["out"]
        ops.cmp_local_prefill(s["q"], s["k"], s["v"], c["batch"], c["tokens"], H, Dh, CMP_WINDOW,
                              out=out[:, :D], workspace=s["ws_local"])
        ops.cmp_memory_prefill(s["q"], s["mk"], s["mv"], c["batch"], c["tokens"], ratio, H, Dh,
                               top_k, out=out[:, D:], workspace=s["ws_memory"])
        return out
    if f == "cmp_step":
        H, Dh, ratio, top_k = CMP[c["kind"]]
        D, out = CMP_D, s["out"]
        ops.cmp_local_decode(s["q"], s["k"], s["v"], s["ring_k"], s["ring_v"], s["pos"], H, Dh,
                             out=out[:, :D], workspace=s["ws_local"])
        ops.cmp_memory_decode(s["q"], s["mk"], s["mv"], s["tag"], s["pos"], H, Dh, top_k,
                              out=out[:, D:], workspace=s["ws_memory"])
        return {"out": out, "ring_k": s["ring_k"], "ring_v": s["ring_v"]}
    if f == "head":
        logits = ops.linear(s["h"], s["w"], epilogue=ops.EPI_STORE_F32, layout=ops.LAYOUT_PACKED)
        return {"logits": logits, "greedy": ops.argmax(logits),
                "drawn": ops.sample_top_p(logits, c["temperature"], c["top_p"], s["u"],
                                          top_k=c["top_k"])}
    eng = s["engine"]
    if f == "block_prompt":
        return {"logits": eng.prefill(s["tokens"]), "state": eng.state[(0, 0)]}
    return {"logits": eng.step(s["tokens"]), "greedy": eng.buf["next"],
            "drawn": eng.buf["sampled"]}


# ----------------------------------------------------------------------- necessary work
def _moe_work(T, D, E, H, k):
    """Weights of the experts that T tokens reach, router, rows in and out."""
    reached = E * (1 - (1 - k / E) ** T)
    return (reached * 3 * H * D * 2 + E * D * 4 + 2 * T * D * 2 + T * k * 8,
            2 * T * D * E + 2 * T * k * 3 * H * D)


def _pairs(T, W):
    """Query-key pairs of a causal band."""
    return sum(min(t + 1, W) for t in range(T))


def work(c):
    f = c["family"]
    if f == "moe":
        b, fl = _moe_work(c["tokens"], c["d_model"], c["experts"], c["hidden"], c["top_k"])
    elif f == "attn":
        B, T, H, hd = c["batch"], c["tokens"], c["heads"], c["head_dim"]
        b, fl = 4 * B * T * H * hd * 2, 4 * hd * B * H * _pairs(T, c["window"])
    elif f == "attn_decode":
        B, H, hd, W = c["batch"], c["heads"], c["head_dim"], c["window"]
        b, fl = 2 * B * H * W * hd * 2 + 6 * B * H * hd * 2, 4 * B * H * W * hd
    elif f in ("gdn", "gdn_step"):
        B, H, d = c["batch"], c["heads"], c["width"]
        rows = B * H * c.get("tokens", 1)
        b = rows * ((4 if f == "gdn" else 5) * d * 2 + 8) + 2 * B * H * d * d * 4
        fl = 6 * rows * d * d
    elif f == "linear":
        M, N, K = c["rows"], c["n"], c["k"]
        out = {"bf16": 2, "f32": 4, "residual": 8, "gated": 12}[c["epilogue"]]
        b, fl = M * K * 2 + N * K * 2 + M * N * out, 2 * M * N * K
    elif f == "cmp_prompt":
        H, Dh, ratio, top_k = CMP[c["kind"]]
        B, T, Kw, n = c["batch"], c["tokens"], H * Dh, c["tokens"] // ratio
        seen = sum(min(n, (t + 1) // ratio) for t in range(T))
        used = H * sum(min(top_k, (t + 1) // ratio) for t in range(T)) if top_k else seen
        b = B * (T * (2 * Kw + 3 * CMP_D) + n * (Kw + CMP_D)) * 2
        fl = 2 * B * (_pairs(T, CMP_WINDOW) * (Kw + CMP_D) + seen * Kw + used * CMP_D)
    elif f == "cmp_step":
        H, Dh, _, _ = CMP[c["kind"]]
        B, Kw, slots = c["batch"], H * Dh, CMP_WINDOW + CMP_SLOTS
        b = B * (slots * (Kw + CMP_D) + 2 * Kw + 3 * CMP_D) * 2
        fl = 2 * B * slots * (Kw + CMP_D)
    elif f == "head":
        M, V, D = c["rows"], c["vocab"], c["d_model"]
        b, fl = V * D * 2 + M * D * 2 + M * V * 4, 2 * M * V * D
    else:
        cfg = _config(c)
        B, T = c["batch"], c.get("tokens", 1)
        R, D, hw = B * T, cfg.d_model, cfg.attn_heads * cfg.attn_head_dim
        Hg, dk, dv = cfg.gdn_heads, cfg.gdn_dk, cfg.gdn_dv
        proj = 2 * Hg * dk + 2 * Hg * dv + Hg
        mb, mf = _moe_work(R, D, cfg.n_experts, cfg.expert_hidden, cfg.top_k)
        pairs = B * (_pairs(T, cfg.window) if T > 1 else cfg.window)
        b, fl = cfg.vocab * D * 2 + B * cfg.vocab * 4, 2 * B * cfg.vocab * D
        for kind in cfg.layer_kinds:
            b, fl = b + cfg.num_loops * mb, fl + cfg.num_loops * mf
            if kind == "attn":
                b += cfg.num_loops * (4 * D * hw * 2 + 2 * B * min(pairs // B, cfg.window) * hw * 2)
                fl += cfg.num_loops * (2 * R * 4 * D * hw + 4 * hw * pairs)
            else:
                b += cfg.num_loops * ((proj + Hg * dv) * D * 2 + 2 * B * Hg * dk * dv * 4)
                fl += cfg.num_loops * (2 * R * D * (proj + Hg * dv) + 6 * R * Hg * dk * dv)
    return {"bytes": b, "flops": fl}


def tolerance(c):
    """bf16 outputs round to 2^-9 of a value and are computed from operands (attention
    weights, SwiGLU products) rounded alike; fp32 sums of another order differ by about
    1e-6.  A row whose expert or summary choice ties within rounding may take the other."""
    f = c["family"]
    if f == "linear" and c["epilogue"] != "bf16":
        return {"rel": 1e-5, "max": 1e-3}
    if f == "head":
        return {"rel": 1e-5, "max": 1e-3}
    if f == "model_step":
        # every layer's rounding travels through all that follow, and through the routers
        return {"rel": 0.03, "max": 0.99, "differ": 0.01}
    if f == "block_prompt":
        # the mixer's, the MoE's and the head's roundings together: 3e-3 measured with the
        # model width's sums in another order, more where a row takes another expert
        return {"rel": 0.02, "max": 0.9}
    return {"rel": 1e-2, "max": 0.3}


# ----------------------------------------------------------------------- 64 bits
def _exact_moe(x, x_router, w_router, w_gate_up, w_down, k):
    """Gates [T, k] and the routed SwiGLU experts' sum for fp64 rows x."""
    top, idx = (x_router @ w_router.double().t()).topk(k, dim=-1)
    gates = top.softmax(-1)
    out = torch.zeros_like(x)
    for e in range(w_router.shape[0]):
        t, j = (idx == e).nonzero(as_tuple=True)
        a, b = (x[t] @ w_gate_up[e].double().t()).chunk(2, -1)
        out.index_add_(0, t, gates[t, j, None] * ((F.silu(a) * b) @ w_down[e].double().t()))
    return gates, out


def _exact_attn(q, k, v, W):
    """Banded causal attention of [B, T, H, hd] in blocks of queries."""
    B, T, H, hd = q.shape
    out = torch.empty(B, T, H, hd, dtype=torch.float64, device=DEV)
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    for t0 in range(0, T, 512):
        t1, j0 = min(T, t0 + 512), max(0, t0 - W + 1)
        gap = torch.arange(t0, t1, device=DEV)[:, None] - torch.arange(j0, t1, device=DEV)[None]
        p = q[:, :, t0:t1].double() @ k[:, :, j0:t1].double().transpose(-1, -2) / hd ** 0.5
        p = p.masked_fill((gap < 0) | (gap >= W), -math.inf).softmax(-1)
        out[:, t0:t1] = (p @ v[:, :, j0:t1].double()).transpose(1, 2)
    return out


def _gdn_token(S, q, k, v, beta, g):
    seen = (S * k[..., None]).sum(-2)
    S = g[..., None, None] * S + k[..., None] * (beta[..., None] * (v - seen))[..., None, :]
    return S, (S * q[..., None]).sum(-2)


def _exact_gdn(q, k, v, beta, g, S, reset=None):
    """The delta rule token by token: outputs [B, T, H, dv] and the last state."""
    out = torch.empty(v.shape, dtype=torch.float64, device=DEV)
    for t in range(v.shape[1]):
        if reset is not None:
            S = S * (reset[:, t] == 0)[:, None, None, None]
        S, out[:, t] = _gdn_token(S, *(a[:, t].double() for a in (q, k, v, beta, g)))
    return out, S


def _exact_block(c, seed):
    """Embedding, one mixer, one MoE and the tied head, from an empty state."""
    cfg, B, T = _config(c), c["batch"], c["tokens"]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    tokens = torch.randint(0, cfg.vocab, (B, T), device=DEV, dtype=torch.int32, generator=g)
    w = {n.removeprefix("L0."): t.double()
         for n, t in init_weights(cfg, seed=int(seed), device=DEV).items()}

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.eps) * w[name]

    x = w["embed"][tokens.long()]
    h = norm(x, "mix_norm")
    if c["kind"] == "attn":
        H, hd, W = cfg.attn_heads, cfg.attn_head_dim, cfg.window
        q, k, v = ((h @ w[n].t()).view(B, T, H, hd) for n in ("wq", "wk", "wv"))
        x = x + _exact_attn(q, k, v, W).reshape(B, T, -1) @ w["wo"].t()
        rows = torch.arange(max(0, T - W), T, device=DEV)
        state = {"k": k, "v": v}
        for n, t in state.items():
            ring = torch.zeros(B, H, W, hd, dtype=torch.float64, device=DEV)
            ring[:, :, rows % W] = t[:, rows].transpose(1, 2)
            state[n] = ring
    else:
        H, dk, dv, K = cfg.gdn_heads, cfg.gdn_dk, cfg.gdn_dv, cfg.conv_kernel
        q, k = (F.normalize((h @ w[n].t()).view(B, T, H, dk), dim=-1) for n in ("wq", "wk"))
        v, gate = ((h @ w[n].t()).view(B, T, H, dv) for n in ("wv", "wg"))
        beta = torch.sigmoid(h @ w["wb"].t() + w["bb"])
        S = torch.zeros(B, H, dk, dv, dtype=torch.float64, device=DEV)
        o, S = _exact_gdn(q, k, v, beta, torch.sigmoid(w["decay"]).expand(B, T, H), S)
        past = F.pad(h, (0, 0, K - 1, 0))
        conv = sum(past[:, j:j + T] * w["conv"][:, j] for j in range(K))
        y = (o * torch.sigmoid(gate)).reshape(B, T, -1) @ w["wout"].t()
        x = x + y * torch.sigmoid(conv)
        state = {"S": S, "hist": past[:, T:]}
    h = norm(x, "ffn_norm").view(B * T, -1)
    up = torch.cat([w["w_gate"], w["w_up"]], 1)
    _, y = _exact_moe(h, norm(h, "router_norm"), w["w_router"], up, w["w_down"], cfg.top_k)
    last = norm((x.view(B * T, -1) + y).view(B, T, -1)[:, -1], "final_norm")
    return {"logits": last @ w["embed"].t(), "state": state}


def exact(c, seed):
    """What run(prepare(c, seed)) returns in 64-bit arithmetic on the same inputs.  None
    for whole models: their expert choices are taken on 16-bit activations, so another
    precision takes other experts and its logits are no reference for these."""
    f = c["family"]
    if f == "model_step":
        return None
    if f == "block_prompt":
        return _exact_block(c, seed)
    s = prepare(c, seed)
    if f == "moe":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        T, D, E, H, k = c["tokens"], c["d_model"], c["experts"], c["hidden"], c["top_k"]
        # the same draws as prepare(), before the weights were laid out for the kernels
        torch.empty(T, D, device=DEV).normal_(0.0, 1.0, generator=g)
        torch.empty(E, D, device=DEV).normal_(0.0, 0.02, generator=g)
        gu = torch.empty(E, 2 * H, D, device=DEV).normal_(0.0, 0.02, generator=g).to(BF16)
        dn = torch.empty(E, D, H, device=DEV).normal_(0.0, 0.02, generator=g).to(BF16)
        x = s["x"].double()
        gates, out = _exact_moe(x, x, s["w_router"], gu, dn, k)
        return {"idx": None, "gates": gates, "out": out,
                "perm": dict.fromkeys(("counts", "offsets", "sorted_routes", "route_pos"))}
    if f == "attn":
        return _exact_attn(s["q"], s["k"], s["v"], c["window"])
    if f == "attn_decode":
        W = c["window"]
        q, k, v = (t.double() for t in s["qkv"].unbind(1))
        kc, vc = s["k_cache"].double(), s["v_cache"].double()
        row = torch.arange(c["batch"], device=DEV)
        kc[row, :, (s["pos"] % W).long()] = k
        vc[row, :, (s["pos"] % W).long()] = v
        p = ((kc * q[:, :, None]).sum(-1) / c["head_dim"] ** 0.5).softmax(-1)
        return {"out": (p[..., None] * vc).sum(2), "k_cache": kc, "v_cache": vc}
    if f in ("gdn", "gdn_step"):
        S = s["state"].double()
        if f == "gdn_step":
            S, o = _gdn_token(S, *(s[n].double() for n in ("q", "k", "v", "beta", "g")))
            return {"out": o * s["gate"].double(), "state": S}
        out, S = _exact_gdn(s["q"], s["k"], s["v"], s["beta"], s["g"], S, s["reset"])
        return {"out": out, "state": S}
    if f == "linear":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        torch.empty(c["rows"], c["k"], device=DEV).normal_(0.0, 1.0, generator=g)
        w = torch.empty(c["n"], c["k"], device=DEV).normal_(0.0, 0.02, generator=g).to(BF16)
        y = s["x"].double() @ w.double().t()
        y = y * s["aux"].double() if "aux" in s else y
        return s["out"].double() + y if "out" in s else y
    if f == "cmp_prompt":
        H, Dh, ratio, top_k = CMP[c["kind"]]
        B, T, W, n = c["batch"], c["tokens"], CMP_WINDOW, c["tokens"] // ratio
        t = torch.arange(T, device=DEV)[:, None]
        gap = t - torch.arange(T, device=DEV)[None]
        block = torch.arange(n, device=DEV)[None]

        def branch(k, v, seen, top):
            q = s["q"].double().view(B, T, H, Dh).transpose(1, 2)
            k = k.double().view(B, -1, H, Dh).transpose(1, 2)
            p = (q @ k.transpose(-1, -2) / Dh ** 0.5).masked_fill(~seen, -math.inf)
            if top and top < p.shape[-1]:
                p = p.masked_fill(p < p.topk(top, dim=-1).values[..., -1:], -math.inf)
            p = p.softmax(-1).nan_to_num(0.0).mean(1)
            return (p @ v.double().view(B, -1, CMP_D)).view(B * T, CMP_D)

        local = branch(s["k"], s["v"], (gap >= 0) & (gap < W), 0)
        memory = (branch(s["mk"], s["mv"], (block + 1) * ratio <= t + 1, top_k) if n
                  else torch.zeros_like(local))
        return torch.cat([local, memory], 1)
    if f == "cmp_step":
        H, Dh, _, top_k = CMP[c["kind"]]
        B, W, row = c["batch"], CMP_WINDOW, torch.arange(c["batch"], device=DEV)
        ring_k, ring_v = s["ring_k"].double(), s["ring_v"].double()
        ring_k[row, (s["pos"] % W).long()] = s["k"].double()
        ring_v[row, (s["pos"] % W).long()] = s["v"].double()

        def branch(k, v, top):
            q = s["q"].double().view(B, 1, H, Dh)
            p = (k.view(B, -1, H, Dh) * q).sum(-1).transpose(1, 2) / Dh ** 0.5
            if top and top < p.shape[-1]:
                p = p.masked_fill(p < p.topk(top, dim=-1).values[..., -1:], -math.inf)
            return (p.softmax(-1).mean(1)[..., None] * v).sum(1)

        out = torch.cat([branch(ring_k, ring_v, 0),
                         branch(s["mk"].double(), s["mv"].double(), top_k)], 1)
        return {"out": out, "ring_k": ring_k, "ring_v": ring_v}
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    torch.empty(c["rows"], c["d_model"], device=DEV).normal_(0.0, 1.0, generator=g)
    w = torch.empty(c["vocab"], c["d_model"], device=DEV)
    w = w.normal_(0.0, 3 / math.sqrt(c["d_model"]), generator=g).to(BF16)
    return {"logits": s["h"].double() @ w.double().t(), "greedy": None, "drawn": None}
