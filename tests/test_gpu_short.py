"""GPU: the short-plane kernels (csrc/short.hip) against the fp32 oracle."""
from __future__ import annotations

import pytest
import torch

from oracle import torch_ref
from tests.cases import ROPE_BASE, TOL_MEAN
from tests.test_gpu_parity import _compare
from triton_fused_rope_flash_attn_amd import CosSinTable, RoPEAttention, _lib, sdpa_triton_fa_rope

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "amp": torch.float32}


def _nan(*shape, dtype=torch.float32):
    return torch.full(shape, float("nan"), dtype=dtype, device=DEV)


# both sides of the 32-row blocks, the 64-row tiles, the staged 64 / 128 / 256
# rows and the longest plane: N = 4 (less than a subtile), 10, 36, 49, 64, 65, 82,
# 121, 122, 145, 197, 225, 226, 256; few planes, so that every rule takes them
@pytest.mark.parametrize("side,has_cls", [(2, False), (3, True), (6, False), (7, False), (8, False), (8, True), (9, True),
                                          (11, False), (11, True), (12, True), (14, True), (15, False), (15, True),
                                          (16, False)])
@pytest.mark.parametrize("D,io", [(64, "bf16"), (32, "fp16"), (32, "amp"), (64, "fp32"), (64, "amp"), (32, "fp32")])
def test_short_planes(side, has_cls, D, io):
    B, H = 2, 3
    N = side * side + int(has_cls)
    dt = DT[io]
    print(f"short planes N={N} D={D} {io}", flush=True)
    g = torch.Generator().manual_seed(61)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    # views of one projection buffer; dO a transposed view
    q, k, v = torch.randn(B, N, 3, H, D, generator=g).to(dt).to(DEV).permute(2, 0, 3, 1, 4).unbind(0)
    do = torch.randn(B, N, H, D, generator=g).to(dt).to(DEV).transpose(1, 2)
    comp = _lib.BF16 if io == "amp" else _lib.DTYPE_CODE[dt]
    desc = _lib.make_desc(B, H, N, D, N - int(has_cls), has_cls, _lib.DTYPE_CODE[dt], comp, D ** -0.5)
    rope = table.packed()
    # (the one-pass kernel keeps the backward of up to 32 rows in 16-bit compute at head_dim 64)
    assert _lib.tile_config(desc, 2)[0] == 3
    assert (_lib.tile_config(desc, 3)[0] == 5) == (D == 32 or io == "fp32" or N > 32)

    def run():
        o, dq, dk, dv = (_nan(B, H, N, D, dtype=dt) for _ in range(4))
        lse = _nan(B, H, N)
        _lib.attn_fwd(desc, q, k, v, rope, o, lse)
        _lib.attn_bwd(desc, q, k, v, o, do, lse, rope, dq, dk, dv, _nan(max(_lib.bwd_workspace_elems(desc), 1)))
        torch.cuda.synchronize()
        return o, lse, dq, dk, dv

    got = run()
    ref = torch_ref.forward_backward(*(t.float() for t in (q, k, v, do)), *table.tables(), has_cls)
    lse = torch_ref.logsumexp_rows(q.float(), k.float(), *table.tables(), has_cls)
    if io == "fp32":
        _compare(f"short-fp32-N{N}-D{D}", (got[0], *got[2:]), ref, tol_max=1e-4, tol_mean=1e-5)
    else:
        # fp32 tensors computed in bf16 are held to bf16's bound, the mean to twice it: the
        # oracle's inputs are not bf16 there, so up to four operands of a product
        # (dO, V, K-hat, dS) are off by 2^-9 each, and the gradients of a plane of a few
        # keys have a mean size of 0.3 (4 * 2^-9 * 0.3 = 2.3e-3)
        amp = io == "amp"
        _compare(f"short-{io}-N{N}-D{D}", (got[0], *got[2:]), ref, tol_mean=2e-3 if amp else TOL_MEAN,
                 out_dtype=torch.bfloat16 if amp else dt)
    # a logit of size s is off by about 2^-8 s (bf16 operands)
    assert (got[1] - lse).abs().max().item() < (1e-4 if io == "fp32" else 2e-2)
    assert all(torch.equal(a, b) for a, b in zip(got, run()))


@pytest.mark.parametrize("side,has_cls,dt,B", [(11, False, "bf16", 2), (14, True, "bf16", 2), (16, True, "bf16", 2),
                                               (16, False, "fp16", 2), (15, False, "fp16", 2), (32, True, "bf16", 1),
                                               (14, True, "bf16", 44)])   # 264 items of 128 rows: the 256-row ones
def test_wide_planes_of_small_calls(side, has_cls, dt, B):
    """head_dim 128 forward: 128-row items (one subtile per wave) while they fit one
    per CU.  Rows past the last item (N = 257: the folded row), planes shorter
    than an item, and a call past the limit."""
    H, D = 3, 128
    N = side * side + int(has_cls)
    dt = DT[dt]
    code = _lib.DTYPE_CODE[dt]
    desc = _lib.make_desc(B, H, N, D, side * side, has_cls, code, code, D ** -0.5)
    assert _lib.tile_config(desc, 2)[:2] == (0, 128 if B < 44 else 256)
    print(f"wide planes N={N} B={B} {dt}", flush=True)
    g = torch.Generator().manual_seed(62)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    q, k, v, do = (torch.randn(B, H, N, D, generator=g).to(dt).to(DEV) for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    o = sdpa_triton_fa_rope(*leaves, table, H_img=side, has_cls=has_cls)
    got = (o.detach(), *torch.autograd.grad(o, leaves, do))
    ref = torch_ref.forward_backward(*(t.detach().float() for t in (q, k, v)), do.float(), *table.tables(), has_cls)
    _compare(f"wide-N{N}-B{B}", got, ref, out_dtype=dt)


def _overlapping_rows(B, H, N, D, dt, gen, stride):
    """dO with one row stride for all rows: 0 (one row for every token, as the
    backward of a sum over the tokens gives it) or less than D (rows overlap)."""
    base = torch.randn(B, H, (N - 1) * stride + D, generator=gen).to(dt).to(DEV)
    return base.as_strided((B, H, N, D), (*base.stride()[:2], stride, 1))


# rows past the plane's end in the last 32-row block: 27 (N = 37), none (64), 31
# (65), 27 (197); few planes, so that the short kernels take them
@pytest.mark.parametrize("side,has_cls", [(6, True), (8, False), (8, True), (14, True)])
@pytest.mark.parametrize("D,io", [(64, "bf16"), (32, "fp16"), (32, "amp"), (64, "fp32"), (64, "amp"), (32, "fp32")])
@pytest.mark.parametrize("stride", [0, 16])
def test_short_planes_overlapping_dout_rows(side, has_cls, D, io, stride):
    B, H, N = 2, 3, side * side + int(has_cls)
    dt = DT[io]
    print(f"short planes, dO row stride {stride}, N={N} D={D} {io}", flush=True)
    g = torch.Generator().manual_seed(63)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    q, k, v = (torch.randn(B, H, N, D, generator=g).to(dt).to(DEV).requires_grad_() for _ in range(3))
    do = _overlapping_rows(B, H, N, D, dt, g, stride)
    with torch.autocast("cuda", torch.bfloat16, enabled=io == "amp"):
        o = sdpa_triton_fa_rope(q, k, v, table, H_img=side, has_cls=has_cls)
    got = (o.detach(), *torch.autograd.grad(o, (q, k, v), do))
    ref = torch_ref.forward_backward(*(t.detach().float() for t in (q, k, v)), do.float().contiguous(), *table.tables(),
                                     has_cls)
    tag = f"short-{io}-N{N}-D{D}-dOstride{stride}"
    if io == "fp32":
        # the split products' error grows with the entries: the bound for entries of unit size, times the largest
        big = max(1.0, ref[3].abs().max().item())
        _compare(tag, got, ref, tol_max=1e-4 * big, tol_mean=1e-5 * big)
    else:
        # (the gradients' bounds grow with their size: twice the error of storing them in the compute type)
        _compare(tag, got, ref, tol_mean=2e-3 if io == "amp" else TOL_MEAN, out_dtype=torch.bfloat16 if io == "amp" else dt)


def test_token_sum_pooling():
    """The backward of a sum over the tokens, whose gradient has a row stride of 0,
    through the layer's packed op, against the same gradient in memory of its own."""
    torch.manual_seed(64)
    layer = RoPEAttention(192, 3, H_img=6, device=DEV, dtype=torch.bfloat16)
    layer.proj = torch.nn.Identity()
    x = torch.randn(2, 37, 192, device=DEV).bfloat16().requires_grad_()
    w = torch.randn(2, 192, device=DEV).bfloat16()
    out = layer(x)
    leaves = (x, layer.qkv.weight)
    got = torch.autograd.grad(out.sum(1), leaves, w, retain_graph=True)
    want = torch.autograd.grad(out, leaves, w[:, None, :].repeat(1, 37, 1))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("D,io", [(64, "bf16"), (32, "bf16"), (32, "fp16"), (32, "amp"), (64, "fp32"), (32, "fp32")])
@pytest.mark.parametrize("what", ["q", "k"])
@pytest.mark.parametrize("side", [6, 14])
def test_short_planes_nan_reaches_every_gradient(side, what, D, io):
    """A NaN in one query (or key) makes that query's (every query's) probabilities
    NaN, and with them every key's dV; the other plane stays finite."""
    N = side * side
    g = torch.Generator(device=DEV).manual_seed(65)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    t = dict(zip("qkv", (torch.randn(1, 2, N, D, generator=g, device=DEV).to(DT[io]) for _ in range(3))))
    t[what][0, 0, 5, 3] = float("nan")
    leaves = [t[c].requires_grad_() for c in "qkv"]
    with torch.autocast("cuda", torch.bfloat16, enabled=io == "amp"):
        o = sdpa_triton_fa_rope(*leaves, table, H_img=side, has_cls=False)
    dq, dk, dv = torch.autograd.grad(o, leaves, torch.randn(1, 2, N, D, generator=g, device=DEV).to(DT[io]))
    assert dv[0, 0].isnan().all() and dk[0, 0].isnan().all()
    assert dq[0, 0, 5].isnan().all() if what == "q" else dq[0, 0].isnan().all()
    assert all(torch.isfinite(x[0, 1]).all() for x in (o, dq, dk, dv))


def test_more_planes_than_a_launch_of_tiles_holds():
    """2^24 planes of one row (1 GB a tensor): the softmax over one key is 1, so O = V."""
    B, D = 2 ** 24, 32
    print(f"{B} planes of one row", flush=True)
    g = torch.Generator(device=DEV).manual_seed(66)
    q, k, v = (torch.randn(B, 1, 1, D, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(3))
    table = CosSinTable(ROPE_BASE, 1, D, device=DEV)
    o, lse, _ = torch.ops.farope.attn_fwd(q, k, v, table.packed(), 1, False, D ** -0.5, _lib.BF16)
    assert torch.equal(o, v)
    # K-hat * c2 is rounded to bf16, by at most 2^-9 of each term of the logit (twice that
    # leaves room for the fp32 arithmetic)
    terms = q.float() * k.float() * D ** -0.5
    assert ((lse - terms.sum(-1)).abs() <= 2.0 ** -8 * terms.abs().sum(-1) + 1e-6).all()
