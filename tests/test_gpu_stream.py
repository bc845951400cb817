"""GPU: the streamed tiles (csrc/fwd_stream.hip, csrc/bwd_stream.hip) against the
fp32 oracle, and against the general kernels on the same values."""
from __future__ import annotations

import math

import pytest
import torch

from oracle import torch_ref
from tests.cases import ROPE_BASE
from tests.test_gpu_parity import _compare
from triton_fused_rope_flash_attn_amd import CosSinTable, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _nan(*shape, dtype=torch.float32):
    return torch.full(shape, float("nan"), dtype=dtype, device=DEV)


def _run(q, k, v, do, table, has_cls, ws=True):
    """(O, LSE, dQ, dK, dV) through the C ABI, every output and workspace filled
    with NaN first (a value read before it is written shows)."""
    B, H, N, D = q.shape
    code = _lib.DTYPE_CODE[q.dtype]
    desc = _lib.make_desc(B, H, N, D, N - int(has_cls), has_cls, code, code, 1 / math.sqrt(D))
    o, dq, dk, dv = (_nan(B, H, N, D, dtype=q.dtype) for _ in range(4))
    lse = _nan(B, H, N)
    fws = _nan(max(_lib.fwd_workspace_elems(desc), 1))
    bws = _nan(max(_lib.bwd_workspace_elems(desc), 1))
    rope = table.packed()
    _lib.attn_fwd(desc, q, k, v, rope, o, lse, None, fws if ws else None)
    _lib.attn_bwd(desc, q, k, v, o, do, lse, rope, dq, dk, dv, bws)
    torch.cuda.synchronize()
    return o, lse, dq, dk, dv


def _views(B, H, N, D, dt, gen, pad=0):
    """q, k, v as views of one projection buffer and dO as a transposed view; pad:
    extra elements per row that break the 16-byte alignment of the rows."""
    qkv = torch.randn(B, N, 3, H, D + pad, generator=gen).to(dt).to(DEV)[..., :D]
    q, k, v = qkv.permute(2, 0, 3, 1, 4).unbind(0)
    return q, k, v, torch.randn(B, N, H, D + pad, generator=gen).to(dt).to(DEV)[..., :D].transpose(1, 2)


# rows past the last 128-row tile, 64-row stage, 32-row block and 16-row half:
# N = 289 (33 rows of a tile, one row of the block's second half), 290, 324
# (68), 361 (105), 400 (16), 577 (65), 1024 (none), 1025 (one row); at D 32 from
# N = 257 on
@pytest.mark.parametrize("B,H", [(2, 3), (44, 6)])   # 64-row and 128-row tiles
@pytest.mark.parametrize("side,has_cls,D,dt", [
    (17, False, 64, "bf16"), (17, True, 64, "fp16"), (18, False, 64, "bf16"), (19, False, 64, "bf16"),
    (20, False, 64, "fp16"), (24, True, 64, "bf16"), (32, False, 64, "bf16"), (32, True, 64, "bf16"),
    (16, True, 32, "bf16"), (17, True, 32, "fp16"), (24, False, 32, "bf16"), (31, True, 32, "bf16"),
    (17, True, 128, "fp16"), (20, False, 128, "fp16"), (21, True, 128, "fp16"), (24, True, 128, "fp16"),
])
def test_streamed_tiles(side, has_cls, D, dt, B, H):
    N = side * side + int(has_cls)
    if B > 2 and N > 600:
        pytest.skip("the 128-row tiles' remainders are covered by the shorter planes")
    code = {"bf16": _lib.BF16, "fp16": _lib.F16}[dt]
    desc = _lib.make_desc(B, H, N, D, N - int(has_cls), has_cls, code, code, 0.1)
    assert _lib.tile_config(desc, 2)[:2] == (2, 64 if B == 2 else 128)
    assert _lib.tile_config(desc, 3)[:2] == (4, 64 if B == 2 or D == 128 else 128)
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16}[dt]
    print(f"streamed N={N} D={D} {dt}", flush=True)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    q, k, v, do = _views(B, H, N, D, dt, torch.Generator().manual_seed(41))
    got = _run(q, k, v, do, table, has_cls)
    ref = torch_ref.forward_backward(*(t.float() for t in (q, k, v, do)), *table.tables(), has_cls)
    _compare(f"streamed-N{N}-D{D}", (got[0], *got[2:]), ref, out_dtype=dt)
    lse = torch_ref.logsumexp_rows(q.float(), k.float(), *table.tables(), has_cls)
    assert torch.isfinite(got[1]).all()
    # the logits' operands are rounded to the type: a logit of size s is off by about 2^-8 s (bf16)
    assert (got[1] - lse).abs().max().item() < 2e-2
    again = _run(q, k, v, do, table, has_cls)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def _rel(x, y):
    return ((x.float() - y.float()).norm() / y.float().norm()).item()


# Two bf16 results of one quantity: in each, the probabilities (or dS) and the
# stored values are rounded by at most 2^-9 of themselves, and the errors of the
# sum's terms are independent, like the terms: 4 * 2^-9 in the 2-norm.
BF16_PATHS = 2.0 ** -7


def test_streamed_tiles_agree_with_general_kernels():
    """The same values with rows off the 16-byte grid take the general kernels."""
    B, H, side, D = 2, 2, 21, 64
    N = side * side + 1
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    odd = _views(B, H, N, D, torch.bfloat16, torch.Generator().manual_seed(42), pad=1)
    even = tuple(t.contiguous() for t in odd)
    a, b = _run(*even, table, True), _run(*odd, table, True)
    for name, x, y in zip(("O", "LSE", "dQ", "dK", "dV"), a, b):
        print(f"streamed vs general {name}: {_rel(x, y):.2e}", flush=True)
        # (LSE: the same rounded operands, fp32 sums in another order)
        assert _rel(x, y) < (1e-6 if name == "LSE" else BF16_PATHS), name


def test_streamed_tiles_large_logits():
    """Rows whose running maximum grows past the rescale threshold in a later
    block (logits of std 16: P far above 2^8 of the first block's maximum)."""
    B, H, side, D = 1, 2, 20, 64
    N = side * side
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    q, k, v, do = (t * s for t, s in zip(_views(B, H, N, D, torch.bfloat16, torch.Generator().manual_seed(43)), (4, 4, 1, 1)))
    got = _run(q, k, v, do, table, False)
    plain = _run(q, k, v, do, table, False, ws=False)   # fwd_kernel: other tiles, the same operands
    for name, x, y in zip(("O", "LSE", "dQ", "dK", "dV"), got, plain):
        assert torch.isfinite(x).all(), name
        assert _rel(x, y) < (1e-6 if name == "LSE" else BF16_PATHS), f"{name}: {_rel(x, y):.2e}"


# dO with one row stride for all rows: 0 (one row for every token, as the backward
# of a sum over the tokens gives it) or less than D (rows overlap); both tile sizes;
# N = 289, 324, 400, 577, 1025: 31, 28, 16, 31, 31 rows past the plane's end in the
# last 32-row block, and 290 and 257 in D 32
@pytest.mark.parametrize("stride", [0, 16])
@pytest.mark.parametrize("side,has_cls,D,dt,B", [
    (17, False, 64, "bf16", 2), (18, False, 64, "fp16", 2), (24, True, 64, "bf16", 2), (32, True, 64, "bf16", 1),
    (24, True, 64, "bf16", 44), (16, True, 32, "bf16", 2), (17, True, 32, "fp16", 2), (16, True, 32, "bf16", 100),
    (17, False, 128, "fp16", 2), (20, False, 128, "fp16", 2), (24, True, 128, "fp16", 2),
])
def test_streamed_tiles_overlapping_dout_rows(side, has_cls, D, dt, B, stride):
    H, N = 3, side * side + int(has_cls)
    dt = {"bf16": torch.bfloat16, "fp16": torch.float16}[dt]
    print(f"streamed, dO row stride {stride}, N={N} D={D} B={B} {dt}", flush=True)
    g = torch.Generator().manual_seed(44)
    table = CosSinTable(ROPE_BASE, side, D, device=DEV)
    q, k, v, _ = _views(B, H, N, D, dt, g)
    base = torch.randn(B, H, (N - 1) * stride + D, generator=g).to(dt).to(DEV)
    do = base.as_strided((B, H, N, D), (*base.stride()[:2], stride, 1))
    got = _run(q, k, v, do, table, has_cls)
    ref = torch_ref.forward_backward(*(t.float().contiguous() for t in (q, k, v, do)), *table.tables(), has_cls)
    _compare(f"streamed-N{N}-D{D}-dOstride{stride}", (got[0], *got[2:]), ref, out_dtype=dt)
