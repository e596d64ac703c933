"""Batched decode with groups finer than 128 codes on the streaming kernel's sub-unit builds
(multiples of 64, and of 32), against the oracle.  The shapes lie on both sides of the line
below which a call stays on the fp32 matrix-core kernel (K against rows and batch).

The bars: one output rounding (2^-11 fp16, 2^-8 bf16) of the largest output plus 1e-4 for the fp32
sums and the operands' staging; fp32 1e-6, four times the kernel's error against 64 bits."""
import numpy as np
import pytest
import torch

import cabi
from crispybits_kernels import PackedLinearWeight, _C, fused_gate_up, fused_qkv, packed_linear, permute_for_rope
from crispybits_kernels.io import from_packed_dict
from crispybits_kernels.reference import pack_linear_dict
from oracle import emulator as E

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 2.0 ** -11 + 1e-4, torch.bfloat16: 2.0 ** -8 + 1e-4, torch.float32: 1e-6}


def make(N, K, bits, dtype, gs, seed=1, bias=False, fractional=False):
    g = torch.Generator().manual_seed(seed)
    b = torch.randn(N, generator=g) if bias else None
    d = pack_linear_dict(torch.randn(N, K, generator=g) * 0.05, bits, gs, b, dtype)
    if fractional:
        d["zeros"] = d["zeros"] + 0.375
    W = E.dequant64(d["packed"].numpy(), d["scales"].to(dtype).double().numpy(),
                    d["zeros"].to(dtype).double().numpy(), bits, K, gs)
    return from_packed_dict(d, "cuda", dtype), W, 0.0 if b is None else b.to(dtype).double().numpy()


def randx(M, K, dtype, seed=3):
    return torch.randn(M, K, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def off(y, ref):
    return float(np.abs(y.float().cpu().double().numpy() - ref).max() / np.abs(ref).max())


@pytest.mark.parametrize("dtype,M", [(torch.float16, 3), (torch.float16, 16), (torch.bfloat16, 5),
                                     (torch.bfloat16, 16), (torch.float32, 2), (torch.float32, 8)])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("N,K,gs", [(1100, 2048, 64), (2100, 1000, 64), (515, 4128, 32), (3300, 640, 96),
                                    (22001, 96, 32), (520, 4104, 192), (200, 11008, 64), (1100, 2080, 160),
                                    (300, 512, 64), (4500, 1160, 64), (4500, 3112, 96), (2100, 1568, 32)])
def test_fine_groups(hip, dtype, M, bits, N, K, gs):
    w, W, b = make(N, K, bits, dtype, gs, bias=True)
    x = randx(M, K, dtype)
    ref = E.act64(x.double().cpu().numpy() @ W.T + b, 2)
    for split_k in (None, 3):
        y = packed_linear(x, w, split_k, act="silu")
        assert off(y, ref) < BAR[dtype]
        assert torch.equal(packed_linear(x, w, split_k, act="silu"), y)


def plan(dtype, M, K, gs, out, bits, kind="gemv"):
    """Kernel family and K splits of a decode call."""
    return _C.decode_plan(dtype, M, K, gs, out, bits, kind, 1, 1)[:2]


@pytest.mark.parametrize("dtype,M,K,gs,N,family", [
    (torch.float16, 3, 1024, 64, 2064, "bstream"), (torch.float16, 3, 1016, 64, 2064, "generic"),
    (torch.float16, 10, 2560, 32, 2048, "bstream"), (torch.float16, 10, 2552, 32, 2048, "generic"),
    (torch.float16, 9, 2048, 64, 2064, "bstream"), (torch.float16, 9, 1024, 64, 3072, "generic"),
    (torch.bfloat16, 16, 1024, 32, 4112, "bstream"), (torch.bfloat16, 16, 1024, 96, 4112, "generic"),
    (torch.bfloat16, 16, 3072, 64, 4096, "bstream"), (torch.bfloat16, 16, 3064, 64, 4096, "generic"),
    (torch.float32, 2, 1536, 64, 2064, "bstream"), (torch.float32, 2, 1528, 64, 2064, "generic"),
    (torch.float32, 8, 2560, 32, 11008, "bstream"), (torch.float32, 8, 2552, 32, 11008, "generic"),
    (torch.float32, 9, 4096, 32, 11008, "generic"), (torch.float16, 5, 4097, 64, 4096, "generic")])
def test_fine_groups_line(hip, dtype, M, K, gs, N, family):
    """Both sides of the line between the sub-unit builds and the fp32 matrix-core kernel: low where
    the streaming plan has no splits, which batch 9 and 10 with V <= 4096 rows, or gate-up there, do."""
    assert plan(dtype, M, K, gs, N, 4)[0] == family
    if K == 1024 and N < 4096:
        assert plan(dtype, M, K, gs, N // 2, 4, "gate_up")[0] == "generic"


@pytest.mark.parametrize("dtype,M", [(torch.float16, 6), (torch.bfloat16, 16), (torch.float32, 2), (torch.float32, 8)])
@pytest.mark.parametrize("gs,K", [(32, 3112), (64, 4096), (96, 11008), (64, 1056)])
def test_fine_groups_fused(hip, dtype, M, gs, K):
    """Fused QKV (a width per projection and one for all, with and without RoPE) and gate-up on the
    sub-unit builds, their splits combined in the dispatch; at K = 1056 on the fp32 matrix-core kernel."""
    x = randx(M, K, dtype)
    xd = x.double().cpu().numpy()
    hd = 64
    ws = [make(n, K, b, dtype, gs, i) for i, (n, b) in enumerate(((1024, 4), (512, 2), (512, 3), (512, 4), (512, 4)))]
    ang = torch.rand(M, hd, generator=torch.Generator().manual_seed(9)) * 6.28
    cos, sin = ang.cos().to(dtype).cuda(), ang.sin().to(dtype).cuda()
    cd, sd = cos.double().cpu().numpy(), sin.double().cpu().numpy()

    def rotated(y):
        y = y.reshape(M, -1, hd)
        half = np.concatenate([-y[..., hd // 2:], y[..., :hd // 2]], axis=-1)
        return (y * cd[:, None] + half * sd[:, None]).reshape(M, -1)

    family = "bstream" if K > 2048 else "generic"
    for pick in ((0, 1, 2), (0, 3, 4)):
        (q, Q, _), (k, KW, _), (v, V, _) = (ws[i] for i in pick)
        bits = tuple(ws[i][0].bits for i in pick)
        fam, splits = plan(dtype, M, K, gs, (1024, 512, 512), bits if len(set(bits)) > 1 else bits[0], "qkv")
        assert fam == family and (splits > 1 or family == "generic")
        refs = [xd @ w.T for w in (Q, KW, V)]
        for o, ref in zip(fused_qkv(x, q, k, v), refs):
            assert off(o, ref) < BAR[dtype]
        refs[:2] = [rotated(y) for y in refs[:2]]
        qp, kp = permute_for_rope(q, hd), permute_for_rope(k, hd)
        outs = fused_qkv(x, qp, kp, v, rope=(cos, sin, hd))
        for o, ref in zip(outs, refs):
            assert off(o, ref) < BAR[dtype]
        assert all(torch.equal(a, b) for a, b in zip(fused_qkv(x, qp, kp, v, rope=(cos, sin, hd)), outs))
    g, G, _ = make(1001, K, 3, dtype, gs, 5, fractional=True)
    u, U, _ = make(1001, K, 3, dtype, gs, 6, fractional=True)
    assert plan(dtype, M, K, gs, 1001, 3, "gate_up")[0] == family
    y = fused_gate_up(x, g, u)
    assert off(y, E.silu64(xd @ G.T) * (xd @ U.T)) < BAR[dtype]
    assert torch.equal(fused_gate_up(x, g, u), y)


def test_fine_groups_at_the_scratch_limit(hip):
    """A call without a partial buffer takes a plan that needs none, and so does a no-allocation call
    that asks for no split, so that such calls share nothing and may overlap: accepted, the same
    bits on both, within the bar of the oracle or the buffered call."""
    M, gs = 16, 64
    n, k = 72, 32768                                       # a plan with splits, few rows
    assert cabi.lib.cbk_gemv_partial_floats(0, M, n, k, gs, 1) > 0
    w, W, _ = make(n, k, 2, torch.float16, gs)
    x = randx(M, k, torch.float16)
    out = torch.empty(M, n, dtype=torch.float16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    ref = x.double().cpu().numpy() @ W.T
    rc = cabi.lib.cbk_packed_gemv(x.data_ptr(), 0, M, k, w.packed.data_ptr(), w.scales.data_ptr(),
                                  w.zeros.data_ptr(), None, n, 2, gs, 1, 1, 0, None, None, out.data_ptr(), 0, stream)
    assert rc == 0, cabi.last_error()
    torch.cuda.synchronize()
    assert off(out, ref) < BAR[torch.float16]
    assert not torch.equal(out, packed_linear(x, w))       # that call has splits: another order
    unbuffered = out.clone()
    out.zero_()
    rc = cabi.lib.cbk_packed_gemv_noalloc(x.data_ptr(), 0, M, k, w.packed.data_ptr(), w.scales.data_ptr(),
                                          w.zeros.data_ptr(), None, n, 2, gs, 1, 1, 0, out.data_ptr(), 0, stream)
    assert rc == 0, cabi.last_error()
    torch.cuda.synchronize()
    assert torch.equal(out, unbuffered)
    # past the scratch (P x 16 x 40000 floats): against the buffered call, random codes
    n, k = 40000, 8192
    assert cabi.lib.cbk_gemv_partial_floats(0, M, n, k, gs, 1) > 1 << 21
    g = torch.Generator(device="cuda").manual_seed(1)
    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 16), generator=g, device="cuda", dtype=torch.int32)
    scales = (torch.rand(n, k // gs, generator=g, device="cuda") + 0.5).half() / 64
    zeros = torch.full_like(scales, 2.0)
    x = randx(M, k, torch.float16)
    y = packed_linear(x, PackedLinearWeight(packed, scales, zeros, 2, gs, k, n))
    out = torch.empty(M, n, dtype=torch.float16, device="cuda")
    rc = cabi.lib.cbk_packed_gemv_noalloc(x.data_ptr(), 0, M, k, packed.data_ptr(), scales.data_ptr(),
                                          zeros.data_ptr(), None, n, 2, gs, 1, 1, 0, out.data_ptr(), 0, stream)
    assert rc == 0, cabi.last_error()
    torch.cuda.synchronize()
    assert off(out, y.double().cpu().numpy()) < 2 * BAR[torch.float16]      # two results, a rounding each


def activations(M, K, dtype, dist, seed=3):
    """Normal values at several magnitudes, with a few large channels ("outlier") and spread over
    2^-12 .. 2^4 ("wide")."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g, dtype=torch.float64)
    if dist == "outlier":
        x[:, torch.randperm(K, generator=g)[:4]] *= 1e3
    elif dist == "wide":
        x *= torch.exp2(torch.randint(-12, 5, (M, K), generator=g).double())
    else:
        x *= dist
    return x.to(dtype).cuda()


@pytest.mark.parametrize("bits,gs,M", [(2, 32, 5), (3, 64, 5), (4, 64, 16), (3, 96, 3)])
@pytest.mark.parametrize("dist", [1.0, 3e-3, 1e-3, 3e-4, 1e-4, 1e-5, "outlier", "wide"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fine_groups_magnitudes(hip, dtype, dist, bits, gs, M):
    """The 16-bit builds keep the precision of fp32 products at any magnitude of x: against 64 bits,
    no more than 1 % over the error of rounding the exact result to the type once (in quadrature,
    3e-5 of other error for fp16).  fp16 operands staged times the slot scale 2^-e are 2 to 30 times
    over from an rms of 1e-3 down, and with 1024 left in the decoded pairs it is 5 %."""
    N, K = 1024, 11008
    w, W, _ = make(N, K, bits, dtype, gs)
    x = activations(M, K, dtype, dist)
    ref = torch.from_numpy(x.double().cpu().numpy() @ W.T)
    once = (ref.to(dtype).double() - ref).norm()
    assert (packed_linear(x, w).double().cpu() - ref).norm() < 1.01 * once


def same_specials(y, z, bar):
    """The infinities and NaNs of z, and finite values within the bar of z's largest."""
    assert torch.equal(y.isnan(), z.isnan())
    assert torch.equal(y.isinf(), z.isinf()) and torch.equal(y[y.isinf()], z[z.isinf()])
    f = z.isfinite()
    assert f.any()
    assert (y[f].double() - z[f].double()).abs().max() <= 2 * bar * z[f].double().abs().max()


@pytest.mark.parametrize("kind", ["x inf", "x -inf and nan", "x large", "scale inf", "zero inf"])
@pytest.mark.parametrize("gs,M,K", [(64, 5, 4096), (32, 8, 3080), (96, 4, 11008)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_fine_groups_not_finite(hip, dtype, kind, gs, M, K):
    """Infinities and NaNs, and activations near the top of the type's range, come out as the fp32
    matrix-core kernel gives them, which forms (q - z) s first: infinities of one sign stay
    infinities, sums that fit stay finite, other rows stay as they are.  That kernel takes the
    same call with x off 16-byte alignment."""
    ws = [make(n, K, b, dtype, gs, i)[0] for i, (n, b) in enumerate(((1024, 4), (512, 2), (512, 3), (512, 3)))]
    x = randx(M, K, dtype)
    if kind == "x inf":
        x[1, 77] = float("inf")
        x[M - 1, K - 1] = float("inf")
    elif kind == "x -inf and nan":
        x[0, 5] = -float("inf")
        x[M - 1, 700] = float("nan")
        x[2, 9], x[2, 2100] = float("inf"), -float("inf")
    elif kind == "x large":
        # outputs of rms 0.05 sqrt(K) times this, 5e37, so six of them fit fp32; z sum x over a
        # sub-unit, 7.5 sqrt(32) times this, does not
        x[1] *= 1e3 if dtype == torch.float16 else 1e39 / K ** 0.5
    else:
        for w in ws:
            t = w.scales if kind == "scale inf" else w.zeros
            t[3, K // gs // 2] = float("inf")
            t[17, 0] = float("inf")
    off1 = torch.empty(M * K + 1, dtype=dtype, device="cuda")[1:].view(M, K).copy_(x)
    bar = BAR[dtype]
    assert plan(dtype, M, K, gs, 1024, 4)[0] == "bstream"
    y, z = packed_linear(x, ws[0]), packed_linear(off1, ws[0])
    same_specials(y, z, bar)
    assert z.isinf().any() or kind != "x inf"
    for qkv in (ws[:3], (ws[3], ws[2], ws[3])):            # a width per projection, and one for all
        for a, b in zip(fused_qkv(x, *qkv), fused_qkv(off1, *qkv)):
            same_specials(a, b, bar)
    if kind != "x large":                                  # (the product of two large factors)
        same_specials(fused_gate_up(x, ws[2], ws[3]), fused_gate_up(off1, ws[2], ws[3]), 3 * bar)


@pytest.mark.parametrize("gs", [32, 64])
def test_fine_groups_fp16_error(hip, gs):
    """The 16-bit builds keep the precision of fp32 products: against 64 bits, no more than 1 % over
    the error of rounding the exact result to fp16 once (in quadrature, 3e-5 of other error).  With
    1024 left in the decoded pairs it is 5 % over."""
    M, N, K = 5, 4096, 11008
    w, W, _ = make(N, K, 2, torch.float16, gs)
    x = randx(M, K, torch.float16)
    ref = torch.from_numpy(x.double().cpu().numpy() @ W.T)
    once = (ref.half().double() - ref).norm()
    assert (packed_linear(x, w).double().cpu() - ref).norm() < 1.01 * once
