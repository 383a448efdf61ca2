"""Timed cases of the operator layer: what a serving or fine-tuning program has it do.

A case is a dict of plain values. `prepare` makes its weights, inputs and handles on the GPU, `run` is one pass
through the package's public modules, `exact` is the same pass in plain float64 torch, `work` counts the bytes and
floating-point operations of a pass, and `tolerance` says how far two correct implementations may lie apart.

The kinds, with the shapes of workloads.py (C1: a tiny fp32 layer, C2/C3: 8B-shape dense layer, C4: 30B-A3B-shape
MoE layer, C5: the vision block) and the sizes on both sides of them:

  decode         one token per sequence through a decoder layer over ragged KV caches, replayed as a HIP graph
  prefill        a prompt through a decoder layer (dense or MoE)
  model_prefill  a prompt with an image's 3D positions through a small stack of layers, final norm and lm_head
  vision_tower   images of different sizes packed through the vision tower
  train_text     forward and backward of a decoder layer (fp32 tiny layer, bf16 8B-shape layer)
  train_vision   forward and backward of a vision block
  train_moe      forward and backward of the sparse MoE block
  train_head     forward and backward of final norm, lm_head and the cross-entropy loss
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from qwen3_5_vl_cuda_custom_amd import kernels as K
from qwen3_5_vl_cuda_custom_amd import workloads as W
from qwen3_5_vl_cuda_custom_amd.configs import Qwen3VLConfig, TextConfig, VisionConfig
from qwen3_5_vl_cuda_custom_amd.models import CudaQwen3VLDenseModel, CudaVisionTower
from qwen3_5_vl_cuda_custom_amd.modules import (CudaLinear, CudaRMSNorm, CudaSparseMoE, CudaVisionBlock, PagedKVCache,
                                                StaticKVCache)
from qwen3_5_vl_cuda_custom_amd.modules.graph import StepGraph

DEV = "cuda"
VOCAB = 151936
LAYERS = {"tiny": W.C1, "dense": W.C2, "moe": W.C4}


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # A training step of the tiny fp32 parity layer: every call is small, launches and host work are the time.
        {"name": "train_text_tiny_fp32", "kind": "train_text", "layer": "tiny", "dtype": "float32", "batch": 1,
         "seq": 128},
        # One user's chat turn: a single sequence, one token at a time; the weights are all the traffic.
        {"name": "decode_b1", "kind": "decode", "layer": "dense", "batch": 1, "max_len": 1500, "page_rows": 0},
        # A full serving batch with ragged histories of 1k to 8k tokens.
        {"name": "decode_b32", "kind": "decode", "layer": "dense", "batch": 32, "max_len": 8192, "page_rows": 0},
        # A half-full MoE serving batch over a paged cache.
        {"name": "decode_moe_b16_paged", "kind": "decode", "layer": "moe", "batch": 16, "max_len": 4096,
         "page_rows": 64},
        # Long-prompt prefill, the headline shape.
        {"name": "prefill_s4096", "kind": "prefill", "layer": "dense", "batch": 1, "seq": 4096},
        # The same through an MoE layer.
        {"name": "prefill_moe_s4096", "kind": "prefill", "layer": "moe", "batch": 1, "seq": 4096},
        # Time to first token of an image question of odd length: layers, final norm and every position's logits.
        {"name": "model_prefill_s777", "kind": "model_prefill", "layers": 2, "batch": 1, "seq": 777, "grid": 14},
        # Three images of different sizes encoded together.
        {"name": "vision_tower_3_images", "kind": "vision_tower", "grids": "28x28,20x36,46x30"},
        # Fine-tuning a dense layer on a 2k-token sequence.
        {"name": "train_text_s2048", "kind": "train_text", "layer": "dense", "dtype": "bfloat16", "batch": 1,
         "seq": 2048},
        # Fine-tuning a vision block on four 448x448 images.
        {"name": "train_vision_4x784", "kind": "train_vision", "batch": 4, "grid_h": 28, "grid_w": 28},
        # Fine-tuning a sparse MoE block.
        {"name": "train_moe_s2048", "kind": "train_moe", "batch": 1, "seq": 2048},
        # The next-token loss of a 1,024-token sequence over the full vocabulary (1,023 targets, padding ignored).
        {"name": "train_head_n1023", "kind": "train_head", "rows": 1023},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "model_prefill", "vision_tower", "train_text",
                       "train_text", "train_vision", "train_moe", "train_head"])
    if kind == "decode":
        return {"kind": kind, "layer": rng.choice(["dense", "moe"]), "batch": _log_int(rng, 1, 32),
                "max_len": _log_int(rng, 256, 8192), "page_rows": rng.choice([0, 0, 32, 64, 128])}
    if kind == "prefill":
        batch = rng.choice([1, 1, 2, 3])
        return {"kind": kind, "layer": rng.choice(["dense", "moe"]), "batch": batch,
                "seq": _log_int(rng, 40, 4096 // batch)}
    if kind == "model_prefill":
        return {"kind": kind, "layers": rng.choice([1, 2]), "batch": 1, "seq": _log_int(rng, 120, 900),
                "grid": rng.choice([4, 7, 8, 10])}
    if kind == "vision_tower":
        sides = range(12, 44, 2)
        return {"kind": kind, "grids": ",".join(f"{rng.choice(sides)}x{rng.choice(sides)}"
                                                for _ in range(rng.choice([1, 2])))}
    if kind == "train_text":
        if rng.random() < 0.4:
            return {"kind": kind, "layer": "tiny", "dtype": rng.choice(["float32", "bfloat16"]), "batch":
                    rng.choice([1, 2, 4]), "seq": _log_int(rng, 16, 512)}
        batch = rng.choice([1, 1, 2])
        return {"kind": kind, "layer": "dense", "dtype": "bfloat16", "batch": batch,
                "seq": _log_int(rng, 64, 2048 // batch)}
    if kind == "train_vision":
        return {"kind": kind, "batch": rng.choice([1, 2, 3, 4]), "grid_h": rng.choice(range(8, 30, 2)),
                "grid_w": rng.choice(range(8, 30, 2))}
    if kind == "train_moe":
        return {"kind": kind, "batch": rng.choice([1, 2]), "seq": _log_int(rng, 64, 1024)}
    return {"kind": kind, "rows": _log_int(rng, 16, 1023)}


# ------------------------------------------------------------------ inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g: torch.Generator, *shape, dtype=torch.bfloat16) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _norms_around_one(module: torch.nn.Module, seed: int) -> None:
    """Norm weights as a trained checkpoint has them, near one but not equal to it (and biases near zero)."""
    g = _gen(seed)
    for m in module.modules():
        if type(m).__name__ in ("CudaRMSNorm", "CudaLayerNorm"):
            m.weight.data.copy_(1.0 + 0.1 * torch.randn(m.weight.shape, generator=g, device=DEV))
            if getattr(m, "bias", None) is not None:
                m.bias.data.copy_(0.1 * torch.randn(m.bias.shape, generator=g, device=DEV))


def _text_layer(case: dict, dtype, seed: int):
    layer = W.make_text_layer(LAYERS[case["layer"]], dtype, DEV, seed=seed)
    _norms_around_one(layer, seed + 5)
    return layer


def _lengths(case: dict, seed: int) -> list[int]:
    """Cache lengths of a batch: the longest sequence max_len, the others from an eighth of it up."""
    r = random.Random(seed)
    n = case["max_len"]
    return [n] + [r.randint(max(1, n // 8), n) for _ in range(case["batch"] - 1)]


def _grids(case: dict) -> list[tuple[int, int, int]]:
    return [(1, *map(int, g.split("x"))) for g in case["grids"].split(",")]


def _image_positions(case: dict) -> torch.Tensor:
    """(3, B, S) positions of a prompt with one grid x grid image a third of the way in."""
    S, g = case["seq"], case["grid"]
    before = (S - g * g) // 3
    rows = torch.arange(g).repeat_interleave(g)
    cols = torch.arange(g).repeat(g)
    pre = torch.arange(before).expand(3, before)
    img = torch.stack([torch.zeros_like(rows), rows, cols]) + before
    post = (torch.arange(S - before - g * g) + before + g).expand(3, -1)
    return torch.cat([pre, img, post], dim=1).unsqueeze(1).expand(3, case["batch"], S).contiguous()


def _make_decode(case: dict, seed: int) -> dict:
    cfg, B = LAYERS[case["layer"]], case["batch"]
    layer = _text_layer(case, torch.bfloat16, seed)
    lens, g = _lengths(case, seed), _gen(seed + 1)
    if case["page_rows"]:
        per_seq = -(-(case["max_len"] + 1) // case["page_rows"])
        cache = PagedKVCache(B, cfg.kv_heads, cfg.head_dim, num_pages=B * per_seq, max_pages=per_seq,
                             page_rows=case["page_rows"], dtype=torch.bfloat16, device=DEV, lens=lens)
        cache.prepare_append(1)
        kv = (cache.k_pages, cache.v_pages)
    else:
        cache = StaticKVCache(B, cfg.kv_heads, case["max_len"] + 1, cfg.head_dim, dtype=torch.bfloat16, device=DEV,
                              lens=lens)
        kv = (cache.k, cache.v)
    for t in kv:
        t.normal_(0.0, 1.0, generator=g)
    x = _randn(g, B, 1, cfg.hidden)
    pos = torch.tensor(lens, device=DEV).view(1, B, 1).expand(3, B, 1).contiguous()
    return {"layer": layer, "cache": cache, "kv": kv, "x": x, "pos": pos, "lens": lens,
            "lens0": cache.lens.clone(), "rope": W.make_rope(cfg, DEV)}


def _model_cfg(case: dict) -> Qwen3VLConfig:
    c = W.C2
    return Qwen3VLConfig(family="dense", vision=VisionConfig(num_layers=1, deepstack_layers=()),
                         text=TextConfig(hidden_size=c.hidden, intermediate_size=c.intermediate,
                                         num_layers=case["layers"], num_heads=c.heads, num_kv_heads=c.kv_heads,
                                         head_dim=c.head_dim, vocab_size=VOCAB, rope_theta=c.theta,
                                         mrope_section=list(c.mrope_section)))


def _on_gpu(make, dtype=torch.bfloat16):
    old = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device(DEV):
            return make().to(DEV)
    finally:
        torch.set_default_dtype(old)


def _make(case: dict, seed: int) -> dict:
    """Weights and inputs, before any handle is made of them (also what `exact` reads)."""
    kind, g = case["kind"], _gen(seed + 2)
    if kind == "decode":
        return _make_decode(case, seed)
    if kind in ("prefill", "train_text"):
        cfg = LAYERS[case["layer"]]
        dtype = getattr(torch, case.get("dtype", "bfloat16"))
        layer = _text_layer(case, dtype, seed)
        x, pos = W.text_inputs(cfg, case["batch"], case["seq"], dtype, DEV, seed=seed)
        return {"layer": layer, "x": x, "pos": pos, "rope": W.make_rope(cfg, DEV),
                "dy": _randn(g, *x.shape, dtype=dtype)}
    if kind == "model_prefill":
        model = _on_gpu(lambda: CudaQwen3VLDenseModel(_model_cfg(case))).eval().requires_grad_(False)
        W.init_normal_(model, seed)
        _norms_around_one(model, seed + 5)
        return {"model": model, "x": _randn(g, case["batch"], case["seq"], W.C2.hidden),
                "pos": _image_positions(case).to(DEV)}
    if kind == "vision_tower":
        tower = _on_gpu(lambda: CudaVisionTower(VisionConfig())).eval().requires_grad_(False)
        W.init_normal_(tower, seed, include_bias=True)
        _norms_around_one(tower, seed + 5)
        n = sum(h * w for _, h, w in _grids(case))
        px = torch.rand(n, 3 * 2 * 16 * 16, generator=g, device=DEV) * 2 - 1
        return {"tower": tower, "x": px.to(torch.bfloat16), "grids": _grids(case)}
    if kind == "train_vision":
        blk = W.make_vision_block(W.C5, torch.bfloat16, DEV, seed=seed)
        _norms_around_one(blk, seed + 5)
        grid = (case["grid_h"], case["grid_w"])
        n = grid[0] * grid[1]
        cos, sin = (t.float().contiguous() for t in _vision_cos_sin([(1, *grid)], W.C5.head_dim))
        return {"layer": blk, "x": _randn(g, case["batch"], n, W.C5.hidden), "cos": cos, "sin": sin,
                "dy": _randn(g, case["batch"], n, W.C5.hidden)}
    if kind == "train_moe":
        c = W.C4
        moe = _on_gpu(lambda: CudaSparseMoE(c.hidden, c.moe_intermediate, c.num_experts, c.top_k))
        W.init_normal_(moe, seed)
        x = _randn(g, case["batch"], case["seq"], c.hidden)
        return {"layer": moe, "x": x, "dy": _randn(g, *x.shape)}
    if kind == "train_head":
        norm, head = (_on_gpu(f) for f in (lambda: CudaRMSNorm(W.C2.hidden),
                                           lambda: CudaLinear(W.C2.hidden, VOCAB, bias=False)))
        both = torch.nn.ModuleDict({"norm": norm, "head": head})
        W.init_normal_(both, seed)
        _norms_around_one(both, seed + 5)
        tgt = torch.randint(0, VOCAB, (case["rows"],), generator=g, device=DEV)
        tgt[torch.rand(case["rows"], generator=g, device=DEV) < 0.1] = -100
        return {"layer": both, "x": _randn(g, case["rows"], W.C2.hidden), "tgt": tgt}
    raise ValueError(kind)


def prepare(case: dict, seed: int) -> dict:
    s = _make(case, seed)
    s["kind"] = kind = case["kind"]
    if kind == "decode":
        cache, binding = s["cache"], s["rope"].bind(s["pos"].to(torch.int32))
        host = cache.host_state()

        def step():  # one token per sequence after the same histories: the lengths are put back first
            cache.lens.copy_(s["lens0"])
            cache.set_host_state(host)
            return s["layer"](s["x"], binding, kv_cache=cache)[0]

        with torch.no_grad():
            s["graph"] = StepGraph(step)
        cache.set_host_state(host)
    elif kind.startswith("train"):
        s["layer"].requires_grad_(True)
        s["x"].requires_grad_(True)
        s["params"] = [s["x"], *s["layer"].parameters()]
    return s


def run(s: dict):
    kind = s["kind"]
    if kind == "decode":
        y = s["graph"].replay()
        return {"y": y, "k": s["kv"][0], "v": s["kv"][1], "lens": s["cache"].lens}
    if kind == "prefill":
        with torch.no_grad():
            y, logits, (k, v) = s["layer"](s["x"], s["rope"].bind(s["pos"]))
        return {"y": y, "k": k, "v": v, **({} if logits is None else {"logits": logits})}
    if kind == "model_prefill":
        with torch.no_grad():
            return {"logits": s["model"](inputs_embeds=s["x"], position_ids=s["pos"])}
    if kind == "vision_tower":
        with torch.no_grad():
            merged, last, deepstack = s["tower"](s["x"], s["grids"])
        return {"merged": merged, "last": last, "deepstack": deepstack}
    with torch.enable_grad():
        if kind == "train_head":
            logits = s["layer"]["head"](s["layer"]["norm"](s["x"]))
            y = K.cross_entropy(logits, s["tgt"])
            grads = torch.autograd.grad(y, s["params"])
        else:
            if kind == "train_text":
                y = s["layer"](s["x"], s["rope"].bind(s["pos"]))[0]
            elif kind == "train_vision":
                y = s["layer"](s["x"], s["cos"], s["sin"])
            else:
                y = s["layer"](s["x"])[0]
            grads = torch.autograd.grad(y, s["params"], s["dy"])
    return {"y": y.detach(), "grads": list(grads)}


# ------------------------------------------------------------------ the same in float64
def _d(t: torch.Tensor) -> torch.Tensor:
    return t.detach().double()


def _rms(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _ln(x, w, b, eps):
    return F.layer_norm(x, (x.shape[-1],), w, b, eps)


def _rotate(x, cos, sin):
    """Rotate-half of x (B, H, S, D) by cos/sin broadcastable to (B, 1, S, D / 2)."""
    x1, x2 = x.chunk(2, dim=-1)
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1)


def _mrope(cfg, rope, pos):
    """cos, sin (B, 1, S, D / 2): column c of the half takes its angle from the axis of its section."""
    axis = torch.cat([torch.full((n,), i % 3) for i, n in enumerate(cfg.mrope_section)]).to(DEV)
    p = pos.double()[axis].permute(1, 2, 0)  # (B, S, D / 2)
    ang = (p * rope.inv_freq.double()).unsqueeze(1)
    return ang.cos(), ang.sin()


def _attend(q, k, v, scale, causal):
    """softmax(scale QK^T) V, (B, H, S, D) with grouped KV heads, one KV head at a time."""
    G, outs = q.shape[1] // k.shape[1], []
    S, T = q.shape[2], k.shape[2]
    mask = torch.ones(S, T, dtype=torch.bool, device=q.device).tril() if causal else None
    for h in range(k.shape[1]):
        a = (q[:, h * G:(h + 1) * G] * scale) @ k[:, h:h + 1].transpose(-1, -2).contiguous()
        if mask is not None:
            a = a.masked_fill(~mask, -math.inf)
        outs.append(a.softmax(-1) @ v[:, h:h + 1])
    return torch.cat(outs, dim=1)


def _qkv(cfg, p, x, rope, pos, pre="self_attn."):
    B, S, _ = x.shape
    q, k, v = ((x @ p[pre + n + "_proj.weight"].t()).view(B, S, -1, cfg.head_dim) for n in "qkv")
    cos, sin = _mrope(cfg, rope, pos)
    q = _rotate(_rms(q, p[pre + "q_norm.weight"], cfg.eps).transpose(1, 2), cos, sin)
    k = _rotate(_rms(k, p[pre + "k_norm.weight"], cfg.eps).transpose(1, 2), cos, sin)
    return q, k, v.transpose(1, 2)


def _moe(cfg, x, gate, gate_up, down):
    """(y, logits) of the routed experts; the routing reads the logits as the block returns them (in x's bf16)."""
    xf = x.reshape(-1, x.shape[-1])
    exact_logits = xf @ gate.t()
    logits = exact_logits + (exact_logits.detach().to(torch.bfloat16).double() - exact_logits.detach())
    probs = logits.softmax(-1)
    order = probs.detach().sort(dim=-1, descending=True, stable=True).indices[:, :cfg.top_k]
    w = probs.gather(1, order)
    w = w / w.sum(-1, keepdim=True)
    y = torch.zeros_like(xf)
    for e in range(cfg.num_experts):
        tok, slot = (order == e).nonzero(as_tuple=True)
        if tok.numel():
            g, u = (xf[tok] @ gate_up[e].t()).chunk(2, dim=-1)
            y = y.index_add(0, tok, (F.silu(g) * u @ down[e].t()) * w[tok, slot, None])
    return y.view_as(x), exact_logits


def _mlp(p, x, pre="mlp."):
    return (F.silu(x @ p[pre + "gate_proj.weight"].t()) * (x @ p[pre + "up_proj.weight"].t())) \
        @ p[pre + "down_proj.weight"].t()


def _after_attention(cfg, p, x, o, pre=""):
    B, S, _ = x.shape
    h = x + o.transpose(1, 2).reshape(B, S, -1) @ p[pre + "self_attn.o_proj.weight"].t()
    n = _rms(h, p[pre + "post_attention_layernorm.weight"], cfg.eps)
    if cfg.use_moe:
        y, logits = _moe(cfg, n, p[pre + "mlp.gate_weight"], p[pre + "mlp.gate_up_proj"], p[pre + "mlp.down_proj"])
        return h + y, logits
    return h + _mlp(p, n, pre + "mlp."), None


def _exact_layer(cfg, p, x, rope, pos, pre=""):
    q, k, v = _qkv(cfg, p, _rms(x, p[pre + "input_layernorm.weight"], cfg.eps), rope, pos, pre + "self_attn.")
    y, logits = _after_attention(cfg, p, x, _attend(q, k, v, cfg.head_dim ** -0.5, True), pre)
    return y, logits, k, v


def _exact_decode(case, s):
    cfg, p, x = LAYERS[case["layer"]], {n: _d(t) for n, t in s["layer"].named_parameters()}, _d(s["x"])
    q, k, v = _qkv(cfg, p, _rms(x, p["input_layernorm.weight"], cfg.eps), s["rope"], s["pos"])
    kc, vc = _d(s["kv"][0]), _d(s["kv"][1])
    P, outs = case["page_rows"], []
    for b, n in enumerate(s["lens"]):
        if P:
            pages = s["cache"].block_table[b, :n // P + 1].long()
            kc[pages[-1], :, n % P], vc[pages[-1], :, n % P] = k[b, :, 0], v[b, :, 0]
            rows = [t[pages].permute(1, 0, 2, 3).reshape(cfg.kv_heads, -1, cfg.head_dim) for t in (kc, vc)]
        else:
            kc[b, :, n], vc[b, :, n] = k[b, :, 0], v[b, :, 0]
            rows = [kc[b], vc[b]]
        outs.append(_attend(q[b:b + 1], rows[0][None, :, :n + 1], rows[1][None, :, :n + 1], cfg.head_dim ** -0.5,
                            False))
    y, _ = _after_attention(cfg, p, x, torch.cat(outs))
    return {"y": y, "k": kc, "v": vc, "lens": None}


def _vision_coords(grids, merge=2):
    """(row, col) of every patch, in merge-block order."""
    out = []
    for _, h, w in grids:
        r = torch.arange(h, device=DEV).view(h // merge, 1, merge, 1).expand(h // merge, w // merge, merge, merge)
        c = torch.arange(w, device=DEV).view(1, w // merge, 1, merge).expand(h // merge, w // merge, merge, merge)
        out.append(torch.stack([r.reshape(-1), c.reshape(-1)], dim=-1))
    return torch.cat(out)


def _vision_cos_sin(grids, head_dim, theta=1e4):
    rot = head_dim // 2
    inv = 1.0 / theta ** (torch.arange(0, rot, 2, dtype=torch.float64, device=DEV) / rot)
    ang = (_vision_coords(grids).double().unsqueeze(-1) * inv).flatten(1)
    ang = torch.cat([ang, ang], dim=-1)
    return ang.cos(), ang.sin()


def _exact_vision_block(p, x, cos, sin, seqs, heads, eps, pre=""):
    """x (B, S, h); seqs: the token ranges that attend within themselves."""
    B, S, h = x.shape
    D = h // heads
    n = _ln(x, p[pre + "norm1.weight"], p[pre + "norm1.bias"], eps)
    qkv = (n @ p[pre + "attn.qkv.weight"].t() + p[pre + "attn.qkv.bias"]).view(B, S, 3, heads, D)
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    c, s_ = cos[:, :D // 2], sin[:, :D // 2]
    q, k = _rotate(q, c, s_), _rotate(k, c, s_)
    o = torch.cat([_attend(q[:, :, a:b], k[:, :, a:b], v[:, :, a:b], D ** -0.5, False) for a, b in seqs], dim=2)
    x = x + o.transpose(1, 2).reshape(B, S, h) @ p[pre + "attn.proj.weight"].t() + p[pre + "attn.proj.bias"]
    n = _ln(x, p[pre + "norm2.weight"], p[pre + "norm2.bias"], eps)
    a = F.gelu(n @ p[pre + "mlp.linear_fc1.weight"].t() + p[pre + "mlp.linear_fc1.bias"], approximate="tanh")
    return x + a @ p[pre + "mlp.linear_fc2.weight"].t() + p[pre + "mlp.linear_fc2.bias"]


def _exact_merger(p, x, pre, post):
    w, b = p[pre + "norm.weight"], p[pre + "norm.bias"]
    n = _ln(x.reshape(-1, w.numel()), w, b, 1e-6) if post else _ln(x, w, b, 1e-6).reshape(-1, 4 * x.shape[-1])
    a = F.gelu(n @ p[pre + "linear_fc1.weight"].t() + p[pre + "linear_fc1.bias"], approximate="tanh")
    return a @ p[pre + "linear_fc2.weight"].t() + p[pre + "linear_fc2.bias"]


def _exact_pos_embed(table, grids):
    side = int(math.isqrt(table.shape[0]))
    out, at = [], _vision_coords(grids)
    first = 0
    for _, h, w in grids:
        rc = at[first:first + h * w]
        first += h * w
        r = torch.linspace(0, side - 1, h, dtype=torch.float64, device=DEV)[rc[:, 0]]
        c = torch.linspace(0, side - 1, w, dtype=torch.float64, device=DEV)[rc[:, 1]]
        r0, c0 = r.floor().long(), c.floor().long()
        r1, c1 = (r0 + 1).clamp(max=side - 1), (c0 + 1).clamp(max=side - 1)
        fr, fc = (r - r0).unsqueeze(1), (c - c0).unsqueeze(1)
        out.append(table[r0 * side + c0] * (1 - fr) * (1 - fc) + table[r0 * side + c1] * (1 - fr) * fc
                   + table[r1 * side + c0] * fr * (1 - fc) + table[r1 * side + c1] * fr * fc)
    return torch.cat(out)


def _exact_tower(s):
    tower = s["tower"]
    cfg, grids = tower.cfg, s["grids"]
    p = {n: _d(t) for n, t in tower.named_parameters()}
    x = _d(s["x"]) @ p["patch_embed.weight"].reshape(cfg.hidden_size, -1).t() + p["patch_embed.bias"]
    x = (x + _exact_pos_embed(p["pos_embed.emb.weight"], grids)).unsqueeze(0)
    cos, sin = _vision_cos_sin(grids, tower.head_dim, cfg.rope_theta)
    ends = torch.tensor([0] + [h * w for _, h, w in grids]).cumsum(0).tolist()
    seqs, deepstack = list(zip(ends[:-1], ends[1:])), []
    for i in range(cfg.num_layers):
        x = _exact_vision_block(p, x, cos, sin, seqs, cfg.num_heads, cfg.rms_norm_eps, f"blocks.{i}.")
        if i in cfg.deepstack_layers:
            deepstack.append(_exact_merger(p, x[0], f"deepstack_mergers.{cfg.deepstack_layers.index(i)}.", True))
    return {"merged": _exact_merger(p, x[0], "merger.", False), "last": x[0], "deepstack": deepstack}


def exact(case: dict, seed: int):
    s, kind = _make(case, seed), case["kind"]
    if not kind.startswith("train"):
        with torch.no_grad():
            if kind == "decode":
                return _exact_decode(case, s)
            if kind == "vision_tower":
                return _exact_tower(s)
            if kind == "prefill":
                p = {n: _d(t) for n, t in s["layer"].named_parameters()}
                y, logits, k, v = _exact_layer(LAYERS[case["layer"]], p, _d(s["x"]), s["rope"], s["pos"])
                return {"y": y, "k": k, "v": v, **({} if logits is None else {"logits": logits})}
            p, x = {n: _d(t) for n, t in s["model"].named_parameters()}, _d(s["x"])
            for i in range(case["layers"]):
                x = _exact_layer(W.C2, p, x, s["model"].rotary, s["pos"], f"layers.{i}.")[0]
            return {"logits": _rms(x, p["norm.weight"], W.C2.eps) @ p["lm_head.weight"].t()}
    p = {n: _d(t).requires_grad_(True) for n, t in s["layer"].named_parameters()}
    x = _d(s["x"]).requires_grad_(True)
    with torch.enable_grad():
        if kind == "train_moe":
            # every expert's matrices as leaves of their own: indexing one leaf would copy all of it per expert
            gu, dn = ([t.detach().clone().requires_grad_(True) for t in p[n].detach().unbind(0)]
                      for n in ("gate_up_proj", "down_proj"))
            y = _moe(W.C4, x, p["gate_weight"], gu, dn)[0]
            got = torch.autograd.grad(y, [x, p["gate_weight"], *gu, *dn], _d(s["dy"]), allow_unused=True)
            got = [torch.zeros_like(t) if g is None else g
                   for g, t in zip(got, [x, p["gate_weight"], *gu, *dn])]
            E = W.C4.num_experts
            grads = {"gate_weight": got[1], "gate_up_proj": torch.stack(got[2:2 + E]),
                     "down_proj": torch.stack(got[2 + E:])}
            return {"y": y.detach(), "grads": [got[0]] + [grads[n] for n in p]}
        if kind == "train_head":
            logits = _rms(x, p["norm.weight"], s["layer"]["norm"].eps) @ p["head.weight"].t()
            y = F.cross_entropy(logits, s["tgt"], ignore_index=-100)
            return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *p.values()]))}
        if kind == "train_vision":
            n = x.shape[1]
            y = _exact_vision_block(p, x, s["cos"].double(), s["sin"].double(), [(0, n)], W.C5.heads, W.C5.eps)
        else:
            y = _exact_layer(LAYERS[case["layer"]], p, x, s["rope"], s["pos"])[0]
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *p.values()], _d(s["dy"])))}


# ------------------------------------------------------------------ work and tolerance
def _layer_params(cfg) -> int:
    attn = cfg.hidden * cfg.head_dim * (2 * cfg.heads + 2 * cfg.kv_heads)
    if cfg.use_moe:
        return attn + cfg.num_experts * (cfg.hidden + 3 * cfg.hidden * cfg.moe_intermediate)
    return attn + 3 * cfg.hidden * cfg.intermediate


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "decode":
        cfg, B = LAYERS[case["layer"]], case["batch"]
        keys = sum(_lengths(case, 0)) + B
        params = _layer_params(cfg)
        if cfg.use_moe:  # the experts that B tokens reach, if each picks top_k of them at random
            hit = cfg.num_experts * (1 - (1 - cfg.top_k / cfg.num_experts) ** B)
            params -= round((cfg.num_experts - hit) * 3 * cfg.hidden * cfg.moe_intermediate)
        return {"bytes": 2 * params + 4 * cfg.kv_heads * cfg.head_dim * keys + 4 * B * cfg.hidden,
                "flops": B * cfg.gemm_flops_per_token() + 4 * cfg.head_dim * cfg.heads * keys}
    if kind in ("prefill", "train_text"):
        cfg, B, S = LAYERS[case["layer"]], case["batch"], case["seq"]
        es = 4 if case.get("dtype") == "float32" else 2
        T, params = B * S, _layer_params(cfg)
        flops = T * cfg.gemm_flops_per_token() + cfg.causal_attn_flops(S, B)
        if kind == "prefill":
            return {"bytes": es * (params + 2 * T * cfg.hidden + 2 * T * cfg.kv_heads * cfg.head_dim), "flops": flops}
        # backward: two products per forward product, and the attention's scores once more
        flops = 3 * T * cfg.gemm_flops_per_token() + round(3.5 * cfg.causal_attn_flops(S, B))
        return {"bytes": es * (2 * params + 4 * T * cfg.hidden), "flops": flops}
    if kind == "model_prefill":
        cfg, T = W.C2, case["batch"] * case["seq"]
        head = cfg.hidden * VOCAB
        return {"bytes": 2 * (case["layers"] * _layer_params(cfg) + head + T * (cfg.hidden + VOCAB)),
                "flops": case["layers"] * (T * cfg.gemm_flops_per_token()
                                           + cfg.causal_attn_flops(case["seq"], case["batch"])) + 2 * T * head}
    if kind in ("vision_tower", "train_vision"):
        c = W.C5
        if kind == "train_vision":
            n, B = case["grid_h"] * case["grid_w"], case["batch"]
            params, seqs, T = 4 * c.hidden ** 2 + 2 * c.hidden * c.intermediate, [n] * B, n * B
            flops = 6 * T * params + round(3.5 * sum(4 * c.hidden * m * m for m in seqs))
            return {"bytes": 2 * (2 * params + 4 * T * c.hidden), "flops": flops}
        v, seqs = VisionConfig(), [h * w for _, h, w in _grids(case)]
        T, patch = sum(seqs), 3 * 2 * 16 * 16
        block = 4 * v.hidden_size ** 2 + 2 * v.hidden_size * v.intermediate_size
        merged = 4 * v.hidden_size
        merger = merged * merged + merged * v.out_hidden_size
        n_merge = 1 + len(v.deepstack_layers)
        return {"bytes": 2 * (v.num_layers * block + n_merge * merger + patch * v.hidden_size + T * patch
                              + T * v.hidden_size + n_merge * T // 4 * v.out_hidden_size),
                "flops": 2 * T * (v.num_layers * block + patch * v.hidden_size) + n_merge * 2 * (T // 4) * merger
                + v.num_layers * sum(4 * v.hidden_size * m * m for m in seqs)}
    if kind == "train_moe":
        c, T = W.C4, case["batch"] * case["seq"]
        params = c.num_experts * (c.hidden + 3 * c.hidden * c.moe_intermediate)
        return {"bytes": 2 * (2 * params + 4 * T * c.hidden),
                "flops": 6 * T * c.hidden * (3 * c.moe_intermediate * c.top_k + c.num_experts)}
    N, h = case["rows"], W.C2.hidden
    return {"bytes": 2 * (2 * h * VOCAB + 2 * N * h), "flops": 6 * N * h * VOCAB}


def tolerance(case: dict) -> dict:
    """About four times the distance to float64 measured for each kind (in bf16 that is the rounding of its stored
    intermediates, in fp32 the order of its sums); the tower's 27 layers reach 0.013."""
    if case.get("dtype") == "float32":
        return {"rel": 1e-5}
    return {"rel": {"decode": 0.015, "prefill": 0.02, "model_prefill": 0.025, "vision_tower": 0.03,
                    "train_text": 0.03, "train_vision": 0.02, "train_moe": 0.02, "train_head": 0.012}[case["kind"]]}
