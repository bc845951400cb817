"""GPU: the native kernels and autograd of the torch ops (csrc/torch_ops.cpp) behave
as the Python definitions they replace: saved-tensor hooks, refusals, streams."""
from __future__ import annotations

import pytest
import torch

from triton_fused_rope_flash_attn_amd import CosSinTable, TritonAttention, _lib, sdpa_triton_fa_rope

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIDE, D = 6, 64
N = SIDE * SIDE + 1


@pytest.fixture()
def case():
    g = torch.Generator(device=DEV).manual_seed(51)
    table = CosSinTable(100.0, SIDE, D, device=DEV)
    return table, *(torch.randn(2, 3, N, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4))


def _pass(table, q, k, v, do, fn=sdpa_triton_fa_rope):
    leaves = [t.detach().clone().requires_grad_() for t in (q, k, v)]
    o = fn(*leaves, table)
    return (o.detach(), *torch.autograd.grad(o, leaves, do))


def test_library_is_loaded():
    assert _lib.ops_error() is None


def test_both_entry_points_and_checkpoint_agree(case):
    from torch.utils.checkpoint import checkpoint

    want = _pass(*case)
    for fn in (lambda q, k, v, t: TritonAttention.apply(q, k, v, t, SIDE, True),
               lambda q, k, v, t: checkpoint(lambda a, b, c: sdpa_triton_fa_rope(a, b, c, t), q, k, v, use_reentrant=False)):
        assert all(torch.equal(a, b) for a, b in zip(_pass(*case, fn=fn), want))


def test_saved_tensor_hooks_see_every_saved_tensor(case):
    table, q, k, v, do = case
    want, packed, unpacked = _pass(*case), [], []
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(x) or x.cpu(),
                                                  lambda x: unpacked.append(x) or x.to(DEV)):
        o = sdpa_triton_fa_rope(*leaves, table)
    got = torch.autograd.grad(o, leaves, do)
    assert len(packed) == len(unpacked) == 7   # q, k, v, o, lse, table, residual
    assert all(torch.equal(a, b) for a, b in zip(got, want[1:]))


def test_refusals(case):
    table, q, k, v, do = case
    a = q.clone().requires_grad_()
    (g,) = torch.autograd.grad(sdpa_triton_fa_rope(a, k, v, table), a, do, create_graph=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(g.float().sum(), a)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda x: sdpa_triton_fa_rope(x, k, v, table).sum())(q)
    rope = table.packed()
    args = (rope, N - 1, True, 0.125, _lib.BF16)
    with pytest.raises(ValueError, match="same shape"):
        torch.ops.farope.attn_fwd(q, k[:1], v, *args)
    with pytest.raises(TypeError, match="share one dtype"):
        torch.ops.farope.attn_fwd(q, k.float(), v, *args)
    with pytest.raises(RuntimeError, match="same device"):
        torch.ops.farope.attn_fwd(q, k.cpu(), v, *args)
    with pytest.raises(ValueError, match="packed RoPE table"):
        torch.ops.farope.attn_fwd(q, k, v, rope[:-1], *args[1:])
    o, lse, res = torch.ops.farope.attn_fwd(q, k, v, *args)
    with pytest.raises(ValueError, match="LSE must be contiguous"):
        torch.ops.farope.attn_bwd(do, q, k, v, o, lse[:, :1], *args, res)
    with pytest.raises(ValueError, match="dO and O"):
        torch.ops.farope.attn_bwd(do[:1], q, k, v, o, lse, *args, res)


def test_other_stream_and_dout_dtype(case):
    table, q, k, v, do = case
    want = _pass(*case)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _pass(*case)
    s.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    args = (table.packed(), N - 1, True, D ** -0.5, _lib.BF16)
    o, lse, res = torch.ops.farope.attn_fwd(q, k, v, *args)
    grads = torch.ops.farope.attn_bwd(do.float(), q, k, v, o, lse, *args, res)
    assert all(torch.equal(a, b) for a, b in zip(grads, want[1:]))
