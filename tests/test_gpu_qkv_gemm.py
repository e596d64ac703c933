"""The one-launch prefill QKV (cbk_packed_gemm_qkv) against the three GEMMs, the column restore and
the rotation it replaces.

Where neither path splits K, V and unrotated Q and K are the same bits; rotated values may differ by
one rounding (the kernel may fuse a multiply and an add that torch rounds apart), and a K split
changes the order of the fp32 sums: then the bar is one output ulp of the largest value (2^-10 for
fp16, 2^-7 for bf16) for the GEMM's rounding and one for the rotation's."""
import numpy as np
import pytest
import torch

from crispybits_kernels import _C, fused_qkv, ops, permute_for_rope
from crispybits_kernels.io import from_packed_dict
from crispybits_kernels.reference import pack_linear_dict

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 1e-5}


def weight(n, k, bits, dtype, gs, seed, bias=False):
    g = torch.Generator().manual_seed(seed)
    b = torch.randn(n, generator=g) if bias else None
    return from_packed_dict(pack_linear_dict(torch.randn(n, k, generator=g) * 0.05, bits, gs, b, dtype), "cuda", dtype)


def tables(m, hd, dtype):
    a = torch.rand(m, hd, generator=torch.Generator().manual_seed(9)) * 6.28
    return a.cos().to(dtype).cuda(), a.sin().to(dtype).cuda()


def three_gemms(x, q, k, v, rope):
    """fused_qkv with the one-launch entry hidden: the sequence that any backend has."""
    names = ("packed_gemm", "packed_gemv", "fused_qkv", "fused_gate_up", "sm_count", "tile_n", "max_rho")
    backend = type("ThreeGemms", (), {n: staticmethod(getattr(_C, n)) for n in names})
    prev = ops._C
    ops.set_backend(backend)
    try:
        return fused_qkv(x, q, k, v, rope=rope)
    finally:
        ops.set_backend(prev)


def check(x, q, k, v, rope, ulps=2.0):
    one, three = fused_qkv(x, q, k, v, rope=rope), three_gemms(x, q, k, v, rope)
    for a, b in zip(one, three):
        assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous()
        err = (a.float() - b.float()).abs().max() / b.float().abs().max()
        assert err <= ulps * ULP[x.dtype], float(err)
    return one, three


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [(3, 3, 3), (4, 2, 3)])
@pytest.mark.parametrize("M,K,nq,nkv,hd,gs,rope", [
    (17, 512, 256, 128, 128, 128, torch.float32), (33, 4096, 384, 128, 128, 128, "x"),
    (77, 1000, 320, 160, 32, 32, "x"), (70, 2304, 48, 24, 12, 96, torch.float32), (130, 768, 640, 640, 64, 128, None),
    (300, 4128, 200, 40, 20, 64, "x")])
def test_qkv_gemm(hip, dtype, bits, M, K, nq, nkv, hd, gs, rope):
    q, k, v = (weight(n, K, b, dtype, gs, i, bias=i != 1) for i, (n, b) in enumerate(zip((nq, nkv, nkv), bits)))
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()
    qp, kp = permute_for_rope(q, hd), permute_for_rope(k, hd)
    tab = None if rope is None else (*tables(M, hd, dtype if rope == "x" else rope), hd)
    check(x, qp, kp, v, tab)
    one, three = check(x, q, k, v, None, ulps=1.0)         # rows in order, no rotation
    if K <= 1024:                                          # no K split in either: the same bits
        assert all(torch.equal(a, b) for a, b in zip(one, three))


@pytest.mark.parametrize("case", ["fp32", "unaligned", "fp64 tables", "broadcast tables"])
def test_qkv_gemm_other_calls(hip, case):
    """Calls the launch does not take run as before; tables broadcast over rows are taken."""
    M, K, hd = 40, 256, 32
    dtype = torch.float32 if case == "fp32" else torch.float16
    q, k, v = (weight(64, K, 4, dtype, 128, i) for i in range(3))
    q, k = permute_for_rope(q, hd), permute_for_rope(k, hd)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()
    if case == "unaligned":
        x = torch.empty(M * K + 1, dtype=dtype, device="cuda")[1:].view(M, K).copy_(x)
    cos, sin = tables(1 if case.startswith("broadcast") else M, hd, torch.float64 if case == "fp64 tables" else dtype)
    check(x, q, k, v, (cos, sin, hd))


def test_qkv_gemm_large_batch(hip):
    """128-row tiles, unsplit, with a batched [B, T, K] activation."""
    q, k, v = (weight(n, 1024, 3, torch.float16, 128, i) for i, n in enumerate((1024, 256, 256)))
    q, k = permute_for_rope(q, 128), permute_for_rope(k, 128)
    x = torch.randn(2, 1030, 1024, generator=torch.Generator().manual_seed(3)).half().cuda()
    cos, sin = tables(1030, 128, torch.float16)
    one, three = check(x, q, k, v, (cos.expand(2, -1, -1), sin.expand(2, -1, -1), 128))
    assert one[0].shape == (2, 1030, 1024)
    assert torch.equal(one[2], three[2])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,gs", [(1, 512, 128), (2, 512, 64), (3, 1024, 128), (16, 512, 128), (5, 500, 32)])
def test_decode_tables_in_x_dtype(hip, dtype, M, K, gs):
    """RoPE tables in x's dtype are read as they are: the bits of the same tables in fp32, on each
    decode kernel and with a K split."""
    hd = 32
    q, k, v = (weight(64, K, 3, dtype, gs, i) for i in range(3))
    q, k = permute_for_rope(q, hd), permute_for_rope(k, hd)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()
    cos, sin = tables(M, hd, dtype)
    for split_k in (None, 2):
        a = fused_qkv(x, q, k, v, split_k, rope=(cos, sin, hd))
        b = fused_qkv(x, q, k, v, split_k, rope=(cos.float(), sin.float(), hd))
        assert all(torch.equal(s, t) for s, t in zip(a, b))
    cols = torch.cat([cos, sin], dim=1)                    # tables that are views of one tensor
    a = fused_qkv(x, q, k, v, rope=(cols[:, :hd], cols[:, hd:], hd))
    assert all(torch.equal(s, t) for s, t in zip(a, fused_qkv(x, q, k, v, rope=(cos, sin, hd))))
