"""The 16-bit prefill GEMM's 64- and 128-row tiles, unsplit and with K split over workgroups, in
the plain, gate-up and QKV modes, against the oracle.  Each case asserts the plan it is there for
(cbk_gemm_plan), and has what each of them could go wrong on: K % 128 != 0, groups other than 128
codes, zero points the packed-fp16 dequantization does not take, odd N, partial tiles in M and N.
The 32-row tiles take the smaller shapes of the other prefill tests.

The bars: one output rounding (2^-11 fp16, 2^-8 bf16) of the largest output plus 1e-4 for the fp32
sums; three roundings for gate-up (each factor's, relative, and the product's), and two for the
rotated columns of QKV (the projection's value, then the rotation's)."""
import ctypes

import pytest
import torch

import cabi
from crispybits_kernels import fused_gate_up, fused_qkv, packed_linear, permute_for_rope
from crispybits_kernels.io import from_packed_dict
from crispybits_kernels.reference import pack_linear_dict
from oracle import emulator as E

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 2.0 ** -11 + 1e-4, torch.bfloat16: 2.0 ** -8 + 1e-4}
GEMV, QKV, GATEUP = 0, 1, 2
#: dtype, bits, group size, zero points off the integers for half the rows
VARIANTS = [(torch.float16, 3, 128, False), (torch.float16, 4, 96, True), (torch.bfloat16, 2, 32, False),
            (torch.bfloat16, 4, 256, True), (torch.float16, 2, 64, False), (torch.bfloat16, 3, 128, False)]


def make(N, K, variant, seed, bits=None):
    dtype, b, gs, fractional = variant
    bits = bits or b
    g = torch.Generator().manual_seed(seed)
    d = pack_linear_dict(torch.randn(N, K, generator=g) * 0.05, bits, gs, None, dtype)
    if fractional:
        z = d["zeros"].clone()
        z[: N // 2] += 0.375
        d["zeros"] = z
    W = E.gemm_weight64(d["packed"].numpy(), d["scales"].to(dtype).double().numpy(),
                        d["zeros"].to(dtype).double().numpy(), bits, K, gs, dtype, True)
    return from_packed_dict(d, "cuda", dtype), torch.from_numpy(W).cuda()


def randx(M, K, dtype):
    return torch.randn(M, K, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()


def plan(M, n, K, mode):
    """Rows of a tile, and whether K is split."""
    out = (ctypes.c_int32 * 3)()
    n = n if isinstance(n, tuple) else (n, 0, 0)
    assert cabi.lib.cbk_gemm_plan(M, *n, K, mode, out) == 0, cabi.last_error()
    return out[0], out[1] > 1


def off(y, ref):
    return float((y.double() - ref).abs().max() / ref.abs().max())


@pytest.mark.parametrize("variant", VARIANTS, ids=str)
@pytest.mark.parametrize("M,N,K,tiles", [(401, 2501, 408, (64, False)), (100, 3001, 3000, (64, True)),
                                         (401, 5001, 400, (128, False)), (801, 2500, 640, (128, False)),
                                         (401, 2500, 6024, (128, True))])
def test_plain(hip, M, N, K, tiles, variant):
    assert plan(M, N, K, GEMV) == tiles
    w, W = make(N, K, variant, 1)
    x = randx(M, K, variant[0])
    y = packed_linear(x, w, act="relu")
    assert off(y, (x.double() @ W.T).relu()) < BAR[variant[0]]
    assert torch.equal(packed_linear(x, w, act="relu"), y)


@pytest.mark.parametrize("variant", VARIANTS, ids=str)
@pytest.mark.parametrize("M,N,K,tiles", [(100, 4101, 408, (64, False)), (65, 2001, 3016, (64, True)),
                                         (131, 6001, 392, (128, False)), (131, 3001, 6008, (128, True))])
def test_gate_up(hip, M, N, K, tiles, variant):
    assert plan(M, N, K, GATEUP) == tiles
    dtype = variant[0]
    (g, G), (u, U) = (make(N, K, variant, s) for s in (1, 2))
    x = randx(M, K, dtype)
    gv, uv = x.double() @ G.T, x.double() @ U.T
    ref = (gv * torch.sigmoid(gv)).to(dtype).double() * uv.to(dtype).double()
    y = fused_gate_up(x, g, u)
    assert off(y, ref) < 3 * BAR[dtype]
    assert torch.equal(fused_gate_up(x, g, u), y)


@pytest.mark.parametrize("variant", VARIANTS, ids=str)
@pytest.mark.parametrize("M,nq,nkv,K,hd,tiles", [(300, 2560, 640, 408, 64, (64, False)), (801, 256, 64, 3016, 32, (64, True)),
                                                 (600, 2560, 640, 520, 128, (128, False)),
                                                 (130, 4096, 1024, 6008, 128, (128, True)),
                                                 (1001, 1500, 380, 392, 20, (128, False))])
def test_qkv(hip, M, nq, nkv, K, hd, tiles, variant):
    assert plan(M, (nq, nkv, nkv), K, QKV) == tiles
    dtype = variant[0]
    (q, Q), (k, KW), (v, V) = (make(n, K, variant, i, b) for i, (n, b) in enumerate(((nq, 4), (nkv, 2), (nkv, 3))))
    x = randx(M, K, dtype)
    ang = torch.rand(M, hd, generator=torch.Generator().manual_seed(9)) * 6.28
    cos, sin = ang.cos().to(dtype).cuda(), ang.sin().to(dtype).cuda()
    outs = fused_qkv(x, permute_for_rope(q, hd), permute_for_rope(k, hd), v, rope=(cos, sin, hd))
    for o, W in zip(outs, (Q, KW)):
        y = (x.double() @ W.T).view(M, -1, hd)
        half = torch.cat([-y[..., hd // 2:], y[..., :hd // 2]], dim=-1)
        ref = (y * cos.double()[:, None] + half * sin.double()[:, None]).reshape(M, -1)
        # a column's two products carry a rounding of y each: sqrt(2) of the largest at the most
        assert off(o, ref) < 2.5 * BAR[dtype]
    assert off(outs[2], x.double() @ V.T) < BAR[dtype]
