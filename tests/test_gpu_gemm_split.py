"""The 16-bit prefill GEMM below a full chip: 32-row tiles with K split over workgroups whose
partial tiles are combined in the dispatch (test_gpu_gemm_tiles.py has the higher tiles).

The shapes have few tiles, so that the plan splits K (cbk_gemm_partial_floats > 0 says so), with
splits that start inside a scale window, a ragged K in the last split, partial tiles in M and N, and
zero points the packed-fp16 dequantization does not take.  The bar against the oracle is one output
rounding (half an ulp, 2^-11 for fp16 and 2^-8 for bf16, of the largest output) plus the fp32 sums,
K 2^-24 of the sum of magnitudes -- below 1e-4 of the largest output at these sizes."""
import ctypes
import os
import subprocess
import sys

if __name__ == "__main__":                                 # the test that needs a process of its own
    _HERE = os.path.dirname(os.path.abspath(__file__))
    sys.path[:0] = [os.path.dirname(_HERE), os.path.join(os.path.dirname(_HERE), "llm_quantization-kernel_amd")]

import numpy as np
import pytest
import torch

import cabi
from crispybits_kernels import _C, fused_gate_up, fused_qkv, packed_linear, permute_for_rope
from crispybits_kernels.io import from_packed_dict
from crispybits_kernels.reference import pack_linear_dict
from oracle import emulator as E

pytestmark = pytest.mark.gpu

BAR = {torch.float16: 2.0 ** -11 + 1e-4, torch.bfloat16: 2.0 ** -8 + 1e-4}
CODE = {torch.float16: 0, torch.bfloat16: 1}


def make(N, K, bits, dtype, gs, seed, bias=False, fractional=False):
    g = torch.Generator().manual_seed(seed)
    b = torch.randn(N, generator=g) if bias else None
    d = pack_linear_dict(torch.randn(N, K, generator=g) * 0.05, bits, gs, b, dtype)
    if fractional:
        z = d["zeros"].clone()
        z[: N // 2] += 0.375
        d["zeros"] = z
    W = E.gemm_weight64(d["packed"].numpy(), d["scales"].to(dtype).double().numpy(),
                        d["zeros"].to(dtype).double().numpy(), bits, K, gs, dtype, True)
    return from_packed_dict(d, "cuda", dtype), W, None if b is None else b.to(dtype).double().numpy()


def randx(M, K, dtype, seed=3):
    return torch.randn(M, K, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def off(y, ref):
    return float(np.abs(y.float().cpu().double().numpy() - ref).max() / np.abs(ref).max())


def splits(M, N, K, dtype, gate_up=False):
    return cabi.lib.cbk_gemm_partial_floats(CODE[dtype], M, N, K, int(gate_up)) > 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("M,N,K,gs", [(17, 100, 4096, 128), (32, 136, 4200, 96), (33, 256, 5128, 32),
                                      (64, 128, 11008, 128), (65, 96, 2816, 64), (100, 300, 4328, 256),
                                      (128, 260, 8192, 128), (257, 128, 6400, 512), (300, 1000, 3592, 128),
                                      (33, 257, 5128, 32), (20, 129, 4136, 64)])
def test_split_gemm(hip, dtype, bits, M, N, K, gs):
    assert splits(M, N, K, dtype)
    w, W, b = make(N, K, bits, dtype, gs, 1, bias=True)
    x = randx(M, K, dtype)
    ref = E.act64(x.double().cpu().numpy() @ W.T + b, 1)
    y = packed_linear(x, w, act="relu")
    assert off(y, ref) < BAR[dtype]
    for _ in range(3):                                     # the counters are back at zero, the order is fixed
        assert torch.equal(packed_linear(x, w, act="relu"), y)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,gs", [(17, 100, 4096, 128), (40, 130, 4200, 64), (130, 64, 8200, 128)])
def test_split_gate_up(hip, dtype, M, N, K, gs):
    assert splits(M, N, K, dtype, True)
    g, G, _ = make(N, K, 3, dtype, gs, 1)
    u, U, _ = make(N, K, 3, dtype, gs, 2)
    x = randx(M, K, dtype)
    xd = x.double().cpu().numpy()
    ref = E.round_to(E.silu64(xd @ G.T), dtype) * E.round_to(xd @ U.T, dtype)
    # three roundings: each factor's, relative, and the product's
    assert off(fused_gate_up(x, g, u), ref) < 3 * BAR[dtype]


@pytest.mark.parametrize("M,N,K", [(20, 200, 4096), (50, 128, 5000), (129, 128, 4096)])
def test_split_gemm_fractional_zeros(hip, M, N, K):
    w, W, _ = make(N, K, 4, torch.float16, 128, 1, fractional=True)
    x = randx(M, K, torch.float16)
    assert off(packed_linear(x, w), x.double().cpu().numpy() @ W.T) < BAR[torch.float16]


def test_unsplit_without_a_buffer(hip):
    """cbk_packed_gemm has no partial buffer: the same call runs unsplit, the sums in another order."""
    M, N, K = 48, 256, 4096
    w, W, _ = make(N, K, 4, torch.float16, 128, 1)
    x = randx(M, K, torch.float16)
    out = torch.empty(M, N, dtype=torch.float16, device="cuda")
    rc = cabi.lib.cbk_packed_gemm(x.data_ptr(), 0, M, K, w.packed.data_ptr(), w.scales.data_ptr(),
                                  w.zeros.data_ptr(), None, N, 4, 128, 0, 1, out.data_ptr(), 0,
                                  torch.cuda.current_stream().cuda_stream)
    assert rc == 0, cabi.last_error()
    torch.cuda.synchronize()
    assert off(out, x.double().cpu().numpy() @ W.T) < BAR[torch.float16]


def test_split_gemm_streams_and_replays(hip):
    """A split call on another stream, and captured: every replay, between eager calls, gives the
    bits of the eager call on the first stream (with counters or, in a process that has used every
    window, by the combine launch: the same split order)."""
    w, W, _ = make(512, 4096, 3, torch.float16, 128, 1)
    x = randx(40, 4096, torch.float16)
    y = packed_linear(x, w)
    assert off(y, x.double().cpu().numpy() @ W.T) < BAR[torch.float16]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ys = packed_linear(x, w)
    s.synchronize()
    assert torch.equal(ys, y)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = packed_linear(x, w)
    for _ in range(4):
        yg.zero_()
        g.replay()
        assert torch.equal(packed_linear(x, w), y)
        torch.cuda.synchronize()
        assert torch.equal(yg, y)


def test_split_gemm_without_counter_windows(hip):
    """With every counter window of the prefill GEMMs held by a stream, a further stream's split
    call adds its partials in a combine launch: the same bits in each mode, a launch more.  Decode
    windows are others, so a decode call there still combines in its one launch.  In a process of
    its own, whose windows are all free at the start."""
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "windows ok" in r.stdout, r.stdout + r.stderr


def _use_up_the_windows():
    M, K = 40, 4096
    calls = {}
    for dtype in (torch.float16, torch.bfloat16):
        x = randx(M, K, dtype)
        w = [make(n, K, 3, dtype, 128, i, bias=i == 0)[0] for i, n in enumerate((512, 256, 256, 512))]
        assert splits(M, 512, K, dtype) and splits(M, 512, K, dtype, True)
        q, k = permute_for_rope(w[0], 64), permute_for_rope(w[1], 64)
        rope = (x[:, :64].contiguous(), x[:, 64:128].contiguous(), 64)
        calls[f"plain {dtype}"] = lambda x=x, w=w: (packed_linear(x, w[0], act="silu"),)
        calls[f"gate-up {dtype}"] = lambda x=x, w=w: (fused_gate_up(x, w[3], w[0]),)
        calls[f"qkv {dtype}"] = lambda x=x, q=q, k=k, v=w[2], rope=rope: fused_qkv(x, q, k, v, rope=rope)
    wd = make(512, 11008, 3, torch.float16, 128, 1)[0]
    xd = randx(8, 11008, torch.float16)
    assert _C.decode_plan(torch.float16, 8, 11008, 128, 512, 3, "gemv", 1, 1)[1] > 1

    def run(call):
        """The call's outputs and launches."""
        assert cabi.lib.cbk_timer_start(16) == 0
        out = call()
        torch.cuda.synchronize()
        n = ctypes.c_int()
        assert cabi.lib.cbk_timer_stop(None, ctypes.byref(n), None, 0) == 0, cabi.last_error()
        return out, n.value

    ref = {name: run(call) for name, call in calls.items()}
    yd, nd = run(lambda: (packed_linear(xd, wd),))
    assert nd == 1 and all(n == 1 for _, n in ref.values()), (nd, {k: n for k, (_, n) in ref.items()})
    rt = ctypes.CDLL("libamdhip64.so.7")      # torch's instance, by its soname
    first = next(iter(calls.values()))
    streams = []
    for _ in range(300):                                    # more than there are windows
        h = ctypes.c_void_p()
        assert rt.hipStreamCreate(ctypes.byref(h)) == 0
        streams.append(torch.cuda.ExternalStream(h.value))
        with torch.cuda.stream(streams[-1]):
            assert torch.equal(first()[0], next(iter(ref.values()))[0][0])
    with torch.cuda.stream(streams[-1]):
        for name, call in calls.items():
            out, n = run(call)
            assert n == 2, (name, n)
            assert all(torch.equal(a, b) for a, b in zip(out, ref[name][0])), name
        out, n = run(lambda: (packed_linear(xd, wd),))
        assert n == 1 and torch.equal(out[0], yd[0]), n
    print("windows ok", flush=True)


def test_split_calls_on_forked_capture_streams(hip):
    """Split calls on streams forked into one capture become parallel branches of its graph, so each
    branch needs arrival counters of its own: every replay, between eager calls, gives the eager
    bits, for prefill GEMMs and decode calls alike."""
    shapes = [(512, 40, 4096), (256, 8, 11008), (384, 40, 4096), (320, 8, 11008), (512, 33, 5120), (384, 8, 11008)]
    calls = []
    for i, (N, M, K) in enumerate(shapes):                 # a prefill and a decode call for each branch
        if M > 16:
            assert splits(M, N, K, torch.float16)
        else:
            assert _C.decode_plan(torch.float16, M, K, 128, N, 3, "gemv", 1, 1)[1] > 1
        calls.append((randx(M, K, torch.float16, i), make(N, K, 3, torch.float16, 128, i)[0]))
    eager = [packed_linear(x, w) for x, w in calls]
    torch.cuda.synchronize()
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        main = torch.cuda.current_stream()
        outs = []
        for i, st in enumerate((main, *sides)):
            if st is not main:
                st.wait_stream(main)
            with torch.cuda.stream(st):
                outs += [[packed_linear(x, w) for _ in range(4)] for x, w in calls[2 * i:2 * i + 2]]
        for st in sides:
            main.wait_stream(st)
    for _ in range(5):
        for o in outs:
            for t in o:
                t.zero_()
        g.replay()
        again = [packed_linear(x, w) for x, w in calls]
        torch.cuda.synchronize()
        for o, y, z in zip(outs, eager, again):
            assert torch.equal(z, y)
            for t in o:
                assert torch.equal(t, y)


if __name__ == "__main__":
    _use_up_the_windows()
