"""GPU: the layer's packed-layout ops against the same layer over strided views."""
from __future__ import annotations

import pytest
import torch

from triton_fused_rope_flash_attn_amd import RoPEAttention, sdpa_triton_fa_rope

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pass(layer, x, dout, autocast):
    x = x.clone().requires_grad_()
    with torch.autocast("cuda", torch.bfloat16, enabled=autocast):
        out = layer(x)
    return (out.detach(), *torch.autograd.grad(out, (x, *layer.parameters()), dout.to(out.dtype)))


# every backward family: short, one-pass, split (N = 257), streamed, stored dS
# (D = 128 bf16, with the residual), split at D = 256 and fp32
@pytest.mark.parametrize("B,side,has_cls,heads,D,dtype,autocast", [
    (2, 14, True, 6, 64, torch.bfloat16, False), (40, 14, True, 6, 64, torch.bfloat16, False),
    (2, 16, True, 3, 64, torch.float16, False), (2, 20, False, 3, 64, torch.bfloat16, False),
    (2, 8, False, 4, 32, torch.bfloat16, False), (2, 14, True, 2, 128, torch.bfloat16, False),
    (1, 9, True, 2, 256, torch.bfloat16, False), (2, 7, True, 3, 64, torch.float32, False),
    (2, 17, True, 3, 64, torch.float32, True),
])
def test_packed_layer_equals_views(B, side, has_cls, heads, D, dtype, autocast):
    C, N = heads * D, side * side + int(has_cls)
    torch.manual_seed(71)
    a = RoPEAttention(C, heads, H_img=side, has_cls=has_cls, device=DEV, dtype=dtype)
    b = RoPEAttention(C, heads, H_img=side, has_cls=has_cls, device=DEV, dtype=dtype,
                      attn=lambda *args, **kw: sdpa_triton_fa_rope(*args, **kw))
    b.load_state_dict(a.state_dict())
    x, dout = (torch.randn(B, N, C, device=DEV).to(dtype) for _ in range(2))
    for name, p, q in zip(("out", "dx", "dWqkv", "dbqkv", "dWproj", "dbproj"), _pass(a, x, dout, autocast),
                          _pass(b, x, dout, autocast)):
        # the attention's values are the same bit for bit; the projections' products may
        # add in another order where an operand's layout differs
        assert p.shape == q.shape and p.dtype == q.dtype
        rel = ((p.float() - q.float()).norm() / q.float().norm()).item()
        assert rel < (1e-5 if p.dtype == torch.float32 and not autocast else 2e-3), f"{name}: {rel:.2e}"
    with torch.no_grad():
        assert torch.equal(a(x), b(x)) or autocast


def test_packed_layer_compiles():
    import torch._dynamo

    torch._dynamo.reset()
    layer = RoPEAttention(192, 3, H_img=6, device=DEV, dtype=torch.bfloat16)
    x, dout = (torch.randn(2, 37, 192, device=DEV).to(torch.bfloat16) for _ in range(2))
    want = _pass(layer, x, dout, False)
    compiled = torch.compile(layer, fullgraph=True, backend="aot_eager")
    got = _pass(compiled, x, dout, False)
    assert all(torch.equal(p, q) for p, q in zip(got, want))
    torch._dynamo.reset()


def test_packed_op_passes_opcheck_and_refusals():
    layer = RoPEAttention(192, 3, H_img=6, device=DEV, dtype=torch.bfloat16)
    qkv = torch.randn(2, 37, 576, device=DEV).to(torch.bfloat16).requires_grad_()
    args = (layer.rope.packed(), 3, 36, True, 0.125, 2)
    torch.library.opcheck(torch.ops.farope.attn_qkv_fwd.default, (qkv, *args))
    with pytest.raises(ValueError, match="qkv must be"):
        torch.ops.farope.attn_qkv_fwd(qkv[..., :-1], *args)
    with pytest.raises(ValueError, match="packed RoPE table"):
        torch.ops.farope.attn_qkv_fwd(qkv, args[0][:-1], *args[1:])
    with pytest.raises(RuntimeError, match="ROCm GPUs only"):
        torch.ops.farope.attn_qkv_fwd(qkv.detach().cpu(), *args)
    o = torch.ops.farope.attn_qkv_fwd(qkv, *args)[0]
    (g,) = torch.autograd.grad(o, qkv, torch.ones_like(o), create_graph=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(g.float().sum(), qkv)
