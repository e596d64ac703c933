"""The workloads whose speed counts for this framework, as a user's program calls them.

A case is a plain dict; ``listed()`` names the fixed ones, ``draw(rng)`` gives more of the same
ranges.  ``prepare`` makes inputs, packed weights and (for a decode step) the captured graph on the
GPU from a seed, ``run`` is one pass through the public entry points, ``exact`` the same results in
64 bits by plain torch, ``work`` the bytes and operations one pass cannot do without.

Kinds:
  linear    ``packed_linear``: one projection, decode (up to 16 rows) and prefill
  qkv       ``fused_qkv`` with rotate-half RoPE: the attention input projections
  gate_up   ``fused_gate_up``: the gated MLP's first half
  mlp       ``FusedLlamaMLP``: gate, up and down as the installed module runs them
  step      the linears of a few decoder blocks at one decode step, replayed from a HIP graph as a
            serving loop does (each block: fused QKV with RoPE, o, fused gate-up, down)
  quantize  ``reference.quantize_pack``: the weight format's producer

Sizes are those of the Llama-2-7B and OPT-2.7B shapes that the benchmark and the tests use, of its
split-policy sweep, and ragged ones.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "llm_quantization-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HEAD_DIM = 128
HIDDEN, INTER = 4096, 11008
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
ESIZE = {"fp16": 2, "bf16": 2, "fp32": 4}
#: The largest listed case's products; a drawn case has no more.
MOST_MNK = 2048 * HIDDEN * 2 * INTER


# ----------------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call of a decode step: the attention's output projection for one token
        dict(name="o_m1", kind="linear", m=1, k=4096, n=4096, bits=4, group=128, dtype="fp16"),
        # the linears of one decode step of a mixed-width model, from a captured graph: more weight
        # bytes than the last-level cache holds, so every launch streams from HBM
        dict(name="step_m1", kind="step", m=1, blocks=8, group=128, dtype="fp16"),
        # a small decode batch on grouped-query attention, bf16 as most checkpoints have it
        dict(name="qkv_gqa_m4_bf16", kind="qkv", m=4, k=4096, nq=4096, nkv=1024, bq=4, bk=4, bv=4, group=128,
             dtype="bf16"),
        # a fuller decode batch on the widest layer
        dict(name="gate_up_m16", kind="gate_up", m=16, k=4096, n=11008, bits=3, group=128, dtype="fp16"),
        # OPT's first MLP linear: bias and ReLU in the epilogue, the finer group, an odd batch
        dict(name="fc1_relu_m5_g64", kind="linear", m=5, k=2560, n=10240, bits=4, group=64, dtype="fp16", bias=True,
             act="relu"),
        # full precision activations, as a model loaded in float32 has them
        dict(name="up_m8_fp32", kind="linear", m=8, k=4096, n=11008, bits=3, group=128, dtype="fp32"),
        # a serving batch above the decode threshold, on the longest K
        dict(name="down_m32", kind="linear", m=32, k=11008, n=4096, bits=4, group=128, dtype="fp16"),
        # a short prompt of odd length; widths drawn per projection
        dict(name="qkv_m77", kind="qkv", m=77, k=4096, nq=4096, nkv=4096, bq=4, bk=3, bv=3, group=128, dtype="fp16"),
        # a chunk of a prompt on a 13B-sized layer
        dict(name="up_m256_bf16", kind="linear", m=256, k=5120, n=13824, bits=4, group=128, dtype="bf16"),
        # the whole MLP module on a medium prompt
        dict(name="mlp_m512", kind="mlp", m=512, k=4096, n=11008, bits=3, group=128, dtype="fp16"),
        # a long prompt on the widest layer: the largest call
        dict(name="gate_up_m2048", kind="gate_up", m=2048, k=4096, n=11008, bits=3, group=128, dtype="fp16"),
        # preparing a model: one weight into the packed format
        dict(name="quantize_w3", kind="quantize", n=11008, k=4096, bits=3, group=128, dtype="fp16"),
    ]


_KN = [(4096, 4096), (4096, 11008), (11008, 4096), (2560, 2560), (2560, 10240), (10240, 2560), (5120, 5120),
       (5120, 13824), (13824, 5120), (4096, 14336), (14336, 4096), (2048, 8192), (4096, 1024)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _ragged(rng):
    """(K, N) off the usual sizes: K any multiple of 8, N any number."""
    return 8 * _log_int(rng, 32, 1376), _log_int(rng, 256, 14336)


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["qkv"] * 2 + ["gate_up"] * 2 + ["mlp", "step", "quantize"])
    group = rng.choice([128, 128, 128, 64, 32])
    bits = rng.choice([2, 3, 4])
    dtype = rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"])
    if kind == "step":
        return dict(kind=kind, m=rng.randint(1, 4), blocks=rng.randint(2, 7), group=128,
                    dtype=rng.choice(["fp16", "bf16"]))
    K, N = rng.choice(_KN) if rng.random() < 0.6 else _ragged(rng)
    if kind == "quantize":
        return dict(kind=kind, n=N, k=K, bits=bits, group=group, dtype=dtype)
    most = min(2048, 256 if dtype == "fp32" else 2048)
    if kind == "linear":
        m = _log_int(rng, 1, min(most, MOST_MNK // (K * N)))
        return dict(kind=kind, m=m, k=K, n=N, bits=bits, group=group, dtype=dtype, bias=rng.random() < 0.3,
                    act=rng.choice(["", "", "relu", "silu"]))
    if kind == "qkv":
        heads = rng.choice([8, 16, 20, 32, 40])
        nq = heads * HEAD_DIM
        nkv = rng.choice([heads, heads // 4]) * HEAD_DIM
        K = nq if rng.random() < 0.7 else K
        b = [rng.choice([2, 3, 4]) for _ in range(3)] if rng.random() < 0.5 else [bits] * 3
        m = _log_int(rng, 1, min(most, MOST_MNK // (K * (nq + 2 * nkv))))
        return dict(kind=kind, m=m, k=K, nq=nq, nkv=nkv, bq=b[0], bk=b[1], bv=b[2], group=group, dtype=dtype)
    if kind == "mlp":
        N -= N % 8                    # the module's down projection reads it as its K
    rows = (3 if kind == "mlp" else 2) * N
    m = _log_int(rng, 1, min(most, MOST_MNK // (K * rows)))
    return dict(kind=kind, m=m, k=K, n=N, bits=bits, group=group, dtype=dtype)


# ----------------------------------------------------------------------------- inputs

def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + what) & 0x7FFFFFFFFFFF)


def _activations(seed, what, m, k, dtype):
    """Normal values with the few large channels that a language model's hidden states have."""
    g = _gen(seed, what)
    x = torch.randn(m, k, generator=g, device="cuda")
    x *= torch.where(torch.rand(k, generator=g, device="cuda") < 1 / 256, 8.0, 1.0)
    return x.to(dtype)


def _codes(seed, what, n, k, bits, group, dtype):
    """Codes [n, k], scales and zeros [n, ceil(k / group)] of a normal weight quantized by groups."""
    w = torch.randn(n, k, generator=_gen(seed, what), device="cuda") * 0.02
    groups = -(-k // group)
    if groups * group != k:
        w = torch.cat([w, w[:, -1:].expand(n, groups * group - k)], dim=1)
    w = w.view(n, groups, group)
    lo, hi = w.amin(-1), w.amax(-1)
    qmax = float(2 ** bits - 1)
    s = ((hi - lo) / qmax).clamp_min(1e-8)
    z = torch.round(-lo / s).clamp(0, qmax)
    q = torch.clamp(torch.round(w / s[..., None]) + z[..., None], 0, qmax)
    return q.view(n, -1)[:, :k].to(torch.int32), s.to(dtype), z.to(dtype)


def _packed(q, bits):
    """Codes [n, k] -> int32 words [n, ceil(k / 32) * bits]: 32 codes to `bits` words, low bits first."""
    n, k = q.shape
    chunks = -(-k // 32)
    if chunks * 32 != k:
        q = torch.nn.functional.pad(q, (0, chunks * 32 - k))
    q = q.view(n, chunks, 32)
    out = torch.zeros(n, chunks, bits, dtype=torch.int32, device=q.device)
    for j in range(32):
        word, at = divmod(j * bits, 32)
        out[:, :, word] |= q[:, :, j] << at
        if at + bits > 32:
            out[:, :, word + 1] |= q[:, :, j] >> (32 - at)
    return out.view(n, chunks * bits)


def _weight(seed, what, n, k, bits, group, dtype, bias=None):
    from crispybits_kernels import PackedLinearWeight
    q, s, z = _codes(seed, what, n, k, bits, group, dtype)
    return PackedLinearWeight(_packed(q, bits), s, z, bits, group, k, n, bias)


def _weight64(seed, what, n, k, bits, group, dtype):
    q, s, z = _codes(seed, what, n, k, bits, group, dtype)
    at = torch.arange(k, device="cuda") // group
    return (q.double() - z.double()[:, at]) * s.double()[:, at]


def _bias(seed, n, dtype):
    return (torch.randn(n, generator=_gen(seed, 90), device="cuda") * 0.1).to(dtype)


def _tables(seed, m, dtype):
    """cos and sin [m, head_dim] at consecutive positions, in the model's type as a model hands them over."""
    start = (int(seed) * 37) % 1024
    pos = torch.arange(start, start + m, device="cuda").float()
    inv = 10000.0 ** (-torch.arange(0, HEAD_DIM, 2, device="cuda").float() / HEAD_DIM)
    angle = torch.cat([pos[:, None] * inv, pos[:, None] * inv], dim=1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


def _step_widths(blocks):
    """Widths block by block, 3 bits in the mean."""
    return [(3, 4, 2)[i % 3] for i in range(blocks)]


def _step_linears():
    return [("q", HIDDEN, HIDDEN), ("k", HIDDEN, HIDDEN), ("v", HIDDEN, HIDDEN), ("o", HIDDEN, HIDDEN),
            ("gate", INTER, HIDDEN), ("up", INTER, HIDDEN), ("down", HIDDEN, INTER)]


# ----------------------------------------------------------------------------- passes

def prepare(case, seed):
    import crispybits_kernels as ck
    from crispybits_kernels.ops import PackedLinear
    kind, dtype, group = case["kind"], DTYPES[case["dtype"]], case["group"]
    st = {"kind": kind, "act": case.get("act") or None}
    if kind == "quantize":
        st["w"] = (torch.randn(case["n"], case["k"], generator=_gen(seed, 1), device="cuda") * 0.02).to(dtype)
        st.update(bits=case["bits"], group=group)
        return st
    m = case["m"]
    if kind == "step":
        x, h = _activations(seed, 0, m, HIDDEN, dtype), _activations(seed, 1, m, INTER, dtype)
        rope = (*_tables(seed, m, dtype), HEAD_DIM)
        blocks = []
        for i, bits in enumerate(_step_widths(case["blocks"])):
            ws = {nm: _weight(seed, 10 * i + 100 + j, n, k, bits, group, dtype)
                  for j, (nm, n, k) in enumerate(_step_linears())}
            ws["q"], ws["k"] = (ck.permute_for_rope(ws[nm], HEAD_DIM) for nm in "qk")
            blocks.append(ws)

        def step():
            out = []
            for b in blocks:
                out += ck.fused_qkv(x, b["q"], b["k"], b["v"], rope=rope)
                out += [ck.packed_linear(x, b["o"]), ck.fused_gate_up(x, b["gate"], b["up"]),
                        ck.packed_linear(h, b["down"])]
            return out

        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
        st.update(graph=graph, out=out, keep=(x, h, rope, blocks))
        return st
    st["x"] = _activations(seed, 0, m, case["k"], dtype)
    if kind == "linear":
        bias = _bias(seed, case["n"], dtype) if case.get("bias") else None
        st["w"] = _weight(seed, 1, case["n"], case["k"], case["bits"], group, dtype, bias)
    elif kind == "qkv":
        q, k, v = (_weight(seed, 1 + i, n, case["k"], b, group, dtype) for i, (n, b) in enumerate(
            ((case["nq"], case["bq"]), (case["nkv"], case["bk"]), (case["nkv"], case["bv"]))))
        st["w"] = (ck.permute_for_rope(q, HEAD_DIM), ck.permute_for_rope(k, HEAD_DIM), v)
        st["rope"] = (*_tables(seed, m, dtype), HEAD_DIM)
    elif kind == "gate_up":
        st["w"] = tuple(_weight(seed, 1 + i, case["n"], case["k"], case["bits"], group, dtype) for i in range(2))
    elif kind == "mlp":
        sizes = ((case["n"], case["k"]), (case["n"], case["k"]), (case["k"], case["n"]))
        st["module"] = ck.FusedLlamaMLP(*(PackedLinear(_weight(seed, 1 + i, n, k, case["bits"], group, dtype))
                                          for i, (n, k) in enumerate(sizes)))
    else:
        raise ValueError(kind)
    return st


def run(st):
    import crispybits_kernels as ck
    kind = st["kind"]
    if kind == "linear":
        return ck.packed_linear(st["x"], st["w"], act=st["act"])
    if kind == "qkv":
        return ck.fused_qkv(st["x"], *st["w"], rope=st["rope"])
    if kind == "gate_up":
        return ck.fused_gate_up(st["x"], *st["w"])
    if kind == "mlp":
        with torch.no_grad():
            return st["module"](st["x"])
    if kind == "step":
        st["graph"].replay()
        return st["out"]
    from crispybits_kernels.reference import quantize_pack
    return quantize_pack(st["w"], st["bits"], st["group"], st["w"].dtype)


# ----------------------------------------------------------------------------- what a pass needs

def _linear_work(m, n, k, bits, group, dtype, x=True):
    e = ESIZE[dtype]
    return {"bytes": n * -(-k // 32) * bits * 4 + 2 * n * -(-k // group) * e + (m * k * e if x else 0) + m * n * e,
            "flops": 2 * m * n * k}


def work(case):
    kind, d, g = case["kind"], case["dtype"], case["group"]
    if kind == "quantize":
        n, k = case["n"], case["k"]
        return {"bytes": n * k * ESIZE[d] + n * -(-k // 32) * case["bits"] * 4 + 2 * n * -(-k // g) * ESIZE[d],
                "flops": 4 * n * k}
    m = case["m"]
    if kind == "linear":
        parts = [_linear_work(m, case["n"], case["k"], case["bits"], g, d)]
        if case.get("bias"):
            parts.append({"bytes": case["n"] * ESIZE[d], "flops": 0})
    elif kind == "qkv":
        parts = [_linear_work(m, case["nq"], case["k"], case["bq"], g, d),
                 _linear_work(m, case["nkv"], case["k"], case["bk"], g, d, x=False),
                 _linear_work(m, case["nkv"], case["k"], case["bv"], g, d, x=False),
                 {"bytes": 2 * m * HEAD_DIM * ESIZE[d], "flops": 0}]
    elif kind in ("gate_up", "mlp"):
        gate = _linear_work(m, case["n"], case["k"], case["bits"], g, d)
        up = _linear_work(m, case["n"], case["k"], case["bits"], g, d, x=False)
        up["bytes"] -= m * case["n"] * ESIZE[d]           # the product is one output
        parts = [gate, up]
        if kind == "mlp":                                  # x, the weights and the module's output
            down = _linear_work(m, case["k"], case["n"], case["bits"], g, d, x=False)
            parts[0]["bytes"] -= m * case["n"] * ESIZE[d]
            parts.append(down)
    else:
        parts = [{"bytes": m * (HIDDEN + INTER + 2 * HEAD_DIM) * ESIZE[d], "flops": 0}]
        for bits in _step_widths(case["blocks"]):
            parts += [_linear_work(m, n, k, bits, g, d, x=False) for _, n, k in _step_linears()]
            parts.append({"bytes": -m * INTER * ESIZE[d], "flops": 0})
    return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}


def tolerance(case):
    """About four times the distance between the kernels' results and the 64-bit ones: one output
    rounding, and above the decode range the weight's rounding to the activation type (an MLP
    carries its hidden values' rounding into the second half)."""
    if case["kind"] == "quantize":
        return "exact"
    return {"fp16": {"rel": 2e-3, "max": 2e-2}, "bf16": {"rel": 1.5e-2, "max": 1.5e-1},
            "fp32": {"rel": 4e-6, "max": 4e-5}}[case["dtype"]]


# ----------------------------------------------------------------------------- in 64 bits

def _silu64(v):
    return v * torch.sigmoid(v)


def _rope64(y, cos, sin):
    m, n = y.shape
    y = y.view(m, n // HEAD_DIM, HEAD_DIM)
    half = torch.cat([-y[..., HEAD_DIM // 2:], y[..., :HEAD_DIM // 2]], dim=-1)
    return (y * cos.double()[:, None] + half * sin.double()[:, None]).reshape(m, n)


def exact(case, seed):
    kind, dtype, g = case["kind"], DTYPES[case["dtype"]], case["group"]
    if kind == "quantize":
        n, k, bits = case["n"], case["k"], case["bits"]
        w = (torch.randn(n, k, generator=_gen(seed, 1), device="cuda") * 0.02).to(dtype).double()
        groups = -(-k // g)
        if groups * g != k:
            w = torch.cat([w, w[:, -1:].expand(n, groups * g - k)], dim=1)
        w = w.view(n, groups, g)
        lo, hi = w.amin(-1), w.amax(-1)
        s = ((hi - lo) / (2 ** bits - 1)).clamp_min(1e-8)
        return None, s, torch.round(-lo / s).clamp(0, 2 ** bits - 1)
    m = case["m"]
    if kind == "step":
        x, h = (_activations(seed, i, m, k, dtype).double() for i, k in enumerate((HIDDEN, INTER)))
        cos, sin = _tables(seed, m, dtype)
        out = []
        for i, bits in enumerate(_step_widths(case["blocks"])):
            def times(v, j):
                _, n, k = _step_linears()[j]
                return v @ _weight64(seed, 10 * i + 100 + j, n, k, bits, g, dtype).T
            out += [_rope64(times(x, 0), cos, sin), _rope64(times(x, 1), cos, sin), times(x, 2), times(x, 3),
                    _silu64(times(x, 4)) * times(x, 5), times(h, 6)]
        return out
    x = _activations(seed, 0, m, case["k"], dtype).double()

    def linear(v, what, n, k, bits):
        return v @ _weight64(seed, what, n, k, bits, g, dtype).T

    if kind == "linear":
        y = linear(x, 1, case["n"], case["k"], case["bits"])
        if case.get("bias"):
            y = y + _bias(seed, case["n"], dtype).double()
        act = case.get("act")
        return y.relu() if act == "relu" else _silu64(y) if act == "silu" else y
    if kind == "qkv":
        cos, sin = _tables(seed, m, dtype)
        return (_rope64(linear(x, 1, case["nq"], case["k"], case["bq"]), cos, sin),
                _rope64(linear(x, 2, case["nkv"], case["k"], case["bk"]), cos, sin),
                linear(x, 3, case["nkv"], case["k"], case["bv"]))
    hidden = (_silu64(linear(x, 1, case["n"], case["k"], case["bits"]))
              * linear(x, 2, case["n"], case["k"], case["bits"]))
    return hidden if kind == "gate_up" else linear(hidden, 3, case["k"], case["n"], case["bits"])
