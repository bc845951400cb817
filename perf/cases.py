"""The calls that the speed of this framework is judged by.

A case is one pass of the fused 2D-RoPE attention as a vision transformer
calls it: the forward alone (serving), or the forward and its gradients
(training), through ``sdpa_triton_fa_rope`` or the ``RoPEAttention`` layer.
``listed`` names twelve of them, from one image served alone to the largest
training batches; ``draw`` gives further ones of the same ranges:

* token grids of 4x4 to 64x64 patches, with and without the CLS token;
* head_dim 32, 64 and 128;
* bf16, fp16 and fp32 tensors, and fp32 tensors under bf16 autocast;
* q, k, v contiguous, or strided views of one qkv projection's output (and
  then dO a transposed view too, as the output projection's backward gives it);
* 1 to 512 images a pass.
"""
import math

import torch

from triton_fused_rope_flash_attn_amd import CosSinTable, RoPEAttention, sdpa_triton_fa_rope

ROPE_BASE = 100.0
DEVICE = "cuda"

# kind: "attn" (the op) or "layer" (qkv projection, op, output projection);
# mode: "train" (forward and gradients) or "infer" (forward without autograd);
# dtype: "bf16", "fp16", "fp32" or "amp" (fp32 tensors, bf16 autocast);
# views: q, k, v are views of one [B, N, 3, H, D] buffer;
# scale: factor on the N(0, 1) entries of q, k and v.
_DEFAULT = dict(kind="attn", mode="train", B=1, H=12, side=14, cls=True, D=64, dtype="bf16", views=False, scale=1.0)


def _case(name, **kw):
    return dict(_DEFAULT, name=name, **kw)


def listed():
    return [
        # One image served alone: the latency of a 14x14-patch forward of 12 heads.
        _case("serve_one", mode="infer", B=1, views=True),
        # The smallest training step in plain fp32 (a debugging or reference run).
        _case("train_fp32_small", B=2, H=8, dtype="fp32"),
        # A small training batch per GPU, as in fine-tuning (the README's example call).
        _case("train_small", B=8),
        # Serving a few high-resolution images in fp16: 32x32 patches, 16 heads.
        _case("serve_dense_fp16", mode="infer", B=4, H=16, side=32, dtype="fp16", views=True),
        # Attention within 8x8 windows with narrow heads: many short planes.
        _case("train_windows", B=512, H=8, side=8, cls=False, D=32, views=True),
        # Mixed precision by autocast over fp32 tensors: the usual training loop.
        _case("train_amp", B=64, dtype="amp"),
        # A whole attention layer of a small model (width 384, 6 heads) in training.
        _case("layer_small", kind="layer", B=64, H=6, views=True),
        # The training batches of a base model (14x14 patches + CLS): the headline workload.
        _case("train_base", B=256),
        # ... and of a large one without CLS token (16x16 patches).
        _case("train_large", B=128, H=16, side=16, cls=False),
        # Fine-tuning at a higher resolution: 24x24 patches + CLS.
        _case("train_finetune", B=32, side=24, views=True),
        # Dense prediction on a 64x64 grid: the longest sequences.
        _case("train_long", B=4, side=64, cls=False),
        # High resolution with wide heads, inputs of twice the unit scale.
        _case("train_hires", B=32, side=32, D=128, scale=2.0),
    ]


# What no drawn case may exceed: the listed cases' largest operation count and traffic.
_MOST_FLOPS = 7.0e11
_MOST_BYTES = 9.0e8


def draw(rng):
    c = dict(_DEFAULT)
    c["kind"] = "layer" if rng.random() < 0.12 else "attn"
    c["mode"] = "infer" if rng.random() < 0.35 else "train"
    c["D"] = rng.choice([32, 64, 64, 64, 64, 128, 128])
    c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp16", "fp16", "amp", "fp32"])
    c["H"] = rng.choice([3, 4, 6, 8, 12, 12, 16, 16])
    c["side"] = int(round(math.exp(rng.uniform(math.log(4), math.log(64)))))
    c["cls"] = rng.random() < 0.6
    c["views"] = c["kind"] == "layer" or rng.random() < 0.5
    c["scale"] = 2.0 if c["kind"] == "attn" and c["D"] == 128 and rng.random() < 0.3 else 1.0
    # the batch: log-uniform up to what the limits allow (fp32 products cost several times bf16's)
    one = work(dict(c, B=1))
    most_flops = _MOST_FLOPS / (8 if c["dtype"] == "fp32" else 1)
    most = max(1, min(512, int(most_flops // one["flops"]), int(_MOST_BYTES // one["bytes"])))
    c["B"] = max(1, min(most, int(round(math.exp(rng.uniform(0.0, math.log(most)))))))
    return c


def _n(case):
    return case["side"] ** 2 + int(case["cls"])


def _dtype(case):
    return {"bf16": torch.bfloat16, "fp16": torch.float16}.get(case["dtype"], torch.float32)


def _inputs(case, seed):
    """The tensors of a pass, in the order and layout that the caller holds them."""
    B, H, N, D = case["B"], case["H"], _n(case), case["D"]
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(*shape, factor=1.0):
        return (torch.randn(shape, generator=g, device=DEVICE) * factor).to(_dtype(case))

    if case["kind"] == "layer":
        C = H * D
        return {
            "x": randn(B, N, C),
            "dout": randn(B, N, C),
            "qkv.weight": randn(3 * C, C, factor=C ** -0.5),
            "qkv.bias": randn(3 * C, factor=0.02),
            "proj.weight": randn(C, C, factor=C ** -0.5),
            "proj.bias": randn(C, factor=0.02),
        }
    if case["views"]:
        q, k, v = randn(B, N, 3, H, D, factor=case["scale"]).permute(2, 0, 3, 1, 4).unbind(0)
        do = randn(B, N, H, D).transpose(1, 2)
    else:
        q, k, v = (randn(B, H, N, D, factor=case["scale"]) for _ in range(3))
        do = randn(B, H, N, D)
    return {"q": q, "k": k, "v": v, "do": do}


def prepare(case, seed):
    t = _inputs(case, seed)
    train = case["mode"] == "train"
    state = {"case": dict(case), "train": train}
    if case["kind"] == "layer":
        layer = RoPEAttention(case["H"] * case["D"], case["H"], H_img=case["side"], has_cls=case["cls"],
                              rope_base=ROPE_BASE, device=DEVICE, dtype=_dtype(case))
        with torch.no_grad():
            for name, p in layer.named_parameters():
                p.copy_(t[name])
        state["layer"], state["x"] = layer, t["x"].requires_grad_(train)
        if train:
            state["dout"] = t["dout"]
        return state
    state["table"] = CosSinTable(ROPE_BASE, case["side"], case["D"], device=DEVICE)
    for name in ("q", "k", "v"):
        state[name] = t[name].detach().requires_grad_(train)
    if train:
        state["do"] = t["do"]
    return state


def run(state):
    case = state["case"]
    with torch.autocast("cuda", torch.bfloat16, enabled=case["dtype"] == "amp"):
        if case["kind"] == "layer":
            layer, x = state["layer"], state["x"]
            if not state["train"]:
                with torch.no_grad():
                    return (layer(x),)
            out = layer(x)
            leaves, dout = (x, *layer.parameters()), state["dout"]
        else:
            args, kw = (state["q"], state["k"], state["v"], state["table"]), dict(H_img=case["side"], has_cls=case["cls"])
            if not state["train"]:
                with torch.no_grad():
                    return (sdpa_triton_fa_rope(*args, **kw),)
            out = sdpa_triton_fa_rope(*args, **kw)
            leaves, dout = args[:3], state["do"]
    return (out.detach(), *torch.autograd.grad(out, leaves, dout.to(out.dtype)))


def work(case):
    B, H, N, D = case["B"], case["H"], _n(case), case["D"]
    e = 2 if case["dtype"] in ("bf16", "fp16") else 4
    train = case["mode"] == "train"
    rows, C = B * N, H * D
    flops = (14 if train else 4) * B * H * N * N * D
    if case["kind"] == "layer":
        weights = 4 * C * C + 4 * C
        return {"bytes": ((4 if train else 2) * rows * C + (2 if train else 1) * weights) * e,
                "flops": flops + (3 if train else 1) * 2 * rows * C * 4 * C}
    return {"bytes": (8 if train else 4) * rows * C * e, "flops": flops}


def tolerance(case):
    # About four times the largest error against 64 bits seen over these ranges: the rounding
    # of operands and stored results to the type (bf16 4.7e-3, fp16 9.6e-4), and for fp32
    # tensors without autocast that of the split products (1.6e-5).  A layer adds its
    # projections' rounding (7.3e-3 under autocast).
    rel = {"bf16": 1.6e-2, "amp": 1.6e-2, "fp16": 3.6e-3, "fp32": 6e-5}[case["dtype"]]
    return {"rel": 1.6 * rel if case["kind"] == "layer" else rel}


# ---------------------------------------------------------------------------
# the same passes in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _rotation(case):
    """cos, sin [N, D/2] in 64 bits: the grid's row angles in the first half, the column's in the second."""
    side, P = case["side"], case["D"] // 4
    freq = ROPE_BASE ** (-torch.arange(P, dtype=torch.float64, device=DEVICE) / P)
    at = torch.arange(side * side, device=DEVICE)
    ang = torch.cat([(at // side).double()[:, None] * freq, (at % side).double()[:, None] * freq], dim=1)
    if case["cls"]:
        ang = torch.cat([torch.zeros_like(ang[:1]), ang])
    return ang.cos(), ang.sin()


def _rotate(x, cos, sin):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], dim=-1).flatten(-2)


def _attention(q, k, v, do, cos, sin):
    """o and, with do, dq, dk, dv of [P, N, D] planes in 64 bits."""
    scale = q.shape[-1] ** -0.5
    qh, kh = _rotate(q, cos, sin), _rotate(k, cos, sin)
    p = torch.softmax(torch.bmm(qh, kh.transpose(1, 2).contiguous()) * scale, dim=-1)
    o = torch.bmm(p, v)
    if do is None:
        return (o,)
    pt = p.transpose(1, 2).contiguous()
    dv = torch.bmm(pt, do)
    del pt
    ds = torch.bmm(do, v.transpose(1, 2).contiguous())
    ds = p * (ds - (do * o).sum(-1, keepdim=True)) * scale
    dq = _rotate(torch.bmm(ds, kh), cos, -sin)
    dk = _rotate(torch.bmm(ds.transpose(1, 2).contiguous(), qh), cos, -sin)
    return o, dq, dk, dv


def _attention_in_parts(q, k, v, do, case):
    B, H, N, D = q.shape
    cos, sin = _rotation(case)
    flat = [None if t is None else t.reshape(B * H, N, D) for t in (q, k, v, do)]
    step = max(1, int(6e7) // (N * N))
    parts = []
    for i in range(0, B * H, step):
        parts.append(_attention(*[None if t is None else t[i:i + step].double() for t in flat], cos, sin))
    return tuple(torch.cat(ts).reshape(B, H, N, D) for ts in zip(*parts))


def exact(case, seed):
    if work(case)["flops"] > 1.0e12:
        return None
    t = _inputs(case, seed)
    train = case["mode"] == "train"
    if case["kind"] == "attn":
        return _attention_in_parts(t["q"], t["k"], t["v"], t["do"] if train else None, case)
    B, H, N, D = case["B"], case["H"], _n(case), case["D"]
    C = H * D
    t = {name: x.double() for name, x in t.items()}
    x, dout = t["x"].reshape(B * N, C), t["dout"].reshape(B * N, C)
    qkv = torch.addmm(t["qkv.bias"], x, t["qkv.weight"].t().contiguous())
    q, k, v = qkv.reshape(B, N, 3, H, D).permute(2, 0, 3, 1, 4).unbind(0)
    da = (dout @ t["proj.weight"]).reshape(B, N, H, D).transpose(1, 2)
    got = _attention_in_parts(q, k, v, da if train else None, case)
    o = got[0].transpose(1, 2).reshape(B * N, C)
    out = torch.addmm(t["proj.bias"], o, t["proj.weight"].t().contiguous()).reshape(B, N, C)
    if not train:
        return (out,)
    dqkv = torch.stack(got[1:]).permute(1, 3, 0, 2, 4).reshape(B * N, 3 * C)   # [3, B, H, N, D] -> rows of qkv
    dt = dqkv.t().contiguous()
    dx = (dqkv @ t["qkv.weight"]).reshape(B, N, C)
    return out, dx, dt @ x, dqkv.sum(0), dout.t().contiguous() @ o, dout.sum(0)
