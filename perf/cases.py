"""The work a program built on this framework has it do, as cases that can be
timed: FP8 linear layers (training steps and inference calls), grouped MoE
layers, token dispatch and bare quantization, each through its public entry
point.

A case is a dict of plain values; ``op`` says which entry point it calls:

  linear     ops.gemm_fp8 on high-precision operands; with ``grad`` also both
             gradients (a training step of the layer), as autograd gives them
  linear_w8  ops.gemm_fp8 without gradients on a weight quantized once
             (create_quantized_weight), as an inference server keeps it
  moe        ops.grouped_gemm_fp8, a training step of the expert layer
  moe_w8     ops.grouped_gemm_fp8 without gradients on expert weights
             quantized once
  dispatch   ops.moe_permute + ops.moe_unpermute, forward and backward
  quant      ops.quantize_fp8 / quantize_fp8_with_trans, and dequantize_fp8 of
             the result (activation offload, exchange buffers, checkpoints)
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "primus-turbo_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import primus_turbo.pytorch as turbo  # noqa: E402
from primus_turbo.pytorch.core.low_precision import (  # noqa: E402
    Float8QuantConfig,
    Format,
    ScaleDtype,
    ScalingGranularity,
)
from primus_turbo.pytorch.core.quantized_tensor import (  # noqa: E402
    QuantizedTensorPair,
    create_quantized_weight,
)

DEV = "cuda"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
_FP8_MAX = {torch.float8_e4m3fn: 448.0, torch.float8_e5m2: 57344.0}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _linear(name, gran, M, N, K, fmt="E4M3", dtype="bf16", trans_b=True, op="linear"):
    return {"name": name, "op": op, "gran": gran, "fmt": fmt, "M": M, "N": N, "K": K, "dtype": dtype,
            "trans_b": trans_b}


def listed():
    return [
        # decoding: 32 sequences in flight, one token each, against a projection
        # of a served model; latency and launches are what counts
        _linear("decode_tensorwise_32x7168x2048", "TENSORWISE", 32, 7168, 2048, op="linear_w8"),
        # a small layer's training step (the tests' and the benchmark's smallest
        # configuration), both operands row-major [M, K] x [K, N]
        _linear("step_tensorwise_512x1024x1024", "TENSORWISE", 512, 1024, 1024, trans_b=False),
        # a mid-size fp16 layer: fewer output tiles than the chip has compute units
        _linear("step_tensorwise_2048x2048x2048_fp16", "TENSORWISE", 2048, 2048, 2048, dtype="fp16"),
        # ragged: token and feature counts that no tile divides (the last
        # micro-batch of a packed data set, an odd vocabulary shard)
        _linear("step_blockwise_1000x4000x3080", "BLOCKWISE", 1000, 4000, 3080),
        # attention-output-sized projection, blockwise scaled
        _linear("step_blockwise_4096x7168x2048", "BLOCKWISE", 4096, 7168, 2048),
        # the benchmark's flagship: dense MLP up-projection, blockwise scaled
        _linear("step_blockwise_4096x18432x7168", "BLOCKWISE", 4096, 18432, 7168),
        # MLP up-projection with per-row scales
        _linear("step_rowwise_8192x14336x4096", "ROWWISE", 8192, 14336, 4096),
        # the largest: a 70B-class MLP up-projection, MX blocks, e5m2 gradients
        _linear("step_mx_hybrid_8192x28672x8192", "MX_BLOCKWISE", 8192, 28672, 8192, fmt="HYBRID"),
        # expert layer of a large MoE on one rank: 32 experts, skewed loads, four
        # of them idle
        {"name": "step_moe_blockwise_65536_32x2048x7168", "op": "moe", "gran": "BLOCKWISE", "fmt": "E4M3",
         "rows": 65536, "G": 32, "N": 2048, "K": 7168, "dtype": "bf16", "trans_b": True, "idle": 4},
        # the same experts while serving: 64 sequences, top-8, about 16 rows an expert
        {"name": "decode_moe_tensorwise_512_32x2048x7168", "op": "moe_w8", "gran": "TENSORWISE", "fmt": "E4M3",
         "rows": 512, "G": 32, "N": 2048, "K": 7168, "dtype": "bf16", "trans_b": True, "idle": 0},
        # token dispatch of that layer: 8192 tokens to 8 of 32 experts and back
        {"name": "dispatch_8192x7168_top8_of_32", "op": "dispatch", "tokens": 8192, "hidden": 7168, "topk": 8,
         "experts": 32, "dtype": "bf16"},
        # bare quantization with a token count that no block divides, both
        # directions, and back
        {"name": "quant_blockwise_5000x6144", "op": "quant", "gran": "BLOCKWISE", "M": 5000, "N": 6144,
         "fmt": "E4M3", "dtype": "bf16"},
    ]


_MOST_FLOPS = 3 * 2.0 * 8192 * 28672 * 8192
_GRANS = ("TENSORWISE", "ROWWISE", "BLOCKWISE", "MX_BLOCKWISE")


def _log(rng, lo, hi, mult=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(mult, int(v / mult + 0.5) * mult)


def draw(rng):
    while True:
        op = rng.choice(("linear", "linear", "linear", "linear_w8", "moe", "moe", "moe_w8", "dispatch", "quant"))
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
        if op == "linear":
            gran = rng.choice(_GRANS)
            fmt = rng.choice(("E4M3", "HYBRID"))
            # features come in multiples of 8 (32 for MX); half of the time whole tiles
            m = 32 if gran == "MX_BLOCKWISE" else 8
            mult = 128 if rng.random() < 0.5 else m
            trans_b = gran in ("MX_BLOCKWISE",) or rng.random() < 0.8
            c = {"op": op, "gran": gran, "fmt": fmt, "M": _log(rng, 256, 16384, 256 if rng.random() < 0.5 else 1),
                 "N": _log(rng, 512, 28672, mult), "K": _log(rng, 512, 28672, mult), "dtype": dtype,
                 "trans_b": trans_b}
        elif op == "linear_w8":
            c = {"op": op, "gran": "TENSORWISE", "fmt": "E4M3", "M": _log(rng, 1, 512),
                 "N": _log(rng, 512, 28672, 128), "K": _log(rng, 512, 16384, 128), "dtype": dtype, "trans_b": True}
        elif op in ("moe", "moe_w8"):
            gran = "TENSORWISE" if op == "moe_w8" else rng.choice(("BLOCKWISE", "BLOCKWISE", "TENSORWISE"))
            G = rng.choice((4, 8, 16, 32, 64))
            c = {"op": op, "gran": gran, "fmt": "E4M3",
                 "rows": _log(rng, 64, 2048) if op == "moe_w8" else _log(rng, 2048, 65536), "G": G,
                 "N": _log(rng, 512, 4096, 128), "K": _log(rng, 512, 7168, 128), "dtype": dtype, "trans_b": True,
                 "idle": rng.choice((0, 0, 1, G // 8))}
        elif op == "dispatch":
            experts = rng.choice((8, 16, 32, 64))
            c = {"op": op, "tokens": _log(rng, 64, 16384), "hidden": _log(rng, 512, 7168, 64),
                 "topk": rng.choice((1, 2, 4, 8)), "experts": experts, "dtype": dtype}
        else:
            c = {"op": op, "gran": rng.choice(_GRANS), "M": _log(rng, 16, 32768), "N": _log(rng, 512, 16384, 32),
                 "fmt": rng.choice(("E4M3", "HYBRID")), "dtype": dtype}
        if op in ("dispatch", "quant") or work(c)["flops"] <= _MOST_FLOPS:
            return c


def work(case):
    op = case["op"]
    if op in ("linear", "linear_w8"):
        M, N, K = case["M"], case["N"], case["K"]
        if op == "linear_w8":
            return {"bytes": 2 * M * K + N * K + 2 * M * N, "flops": 2.0 * M * N * K}
        # a, w and the output's gradient in; output and both gradients out
        return {"bytes": 2 * (2 * M * K + 2 * N * K + 2 * M * N), "flops": 3 * 2.0 * M * N * K}
    if op in ("moe", "moe_w8"):
        M, N, K, G = case["rows"], case["N"], case["K"], case["G"]
        if op == "moe_w8":
            return {"bytes": 2 * M * K + (G - case["idle"]) * N * K + 2 * M * N, "flops": 2.0 * M * N * K}
        return {"bytes": 2 * (2 * M * K + 2 * G * N * K + 2 * M * N), "flops": 3 * 2.0 * M * N * K}
    if op == "dispatch":
        T, P, H = case["tokens"], case["tokens"] * case["topk"], case["hidden"]
        # forward: tokens -> rows -> tokens; backward the same the other way
        return {"bytes": 2 * H * (4 * T + 4 * P), "flops": 2.0 * 2 * P * H}
    M, N = case["M"], case["N"]
    both = case["gran"] in ("BLOCKWISE", "MX_BLOCKWISE")
    # read x, write q (both directions where the granularity has them); read q, write y
    return {"bytes": M * N * (2 + (2 if both else 1) + 1 + 2), "flops": 4.0 * M * N}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _config(case):
    gran = ScalingGranularity[case["gran"]]
    more = {}
    if gran == ScalingGranularity.BLOCKWISE:
        more = {"block_size": 128}
    elif gran == ScalingGranularity.MX_BLOCKWISE:
        more = {"block_size": 32, "scale_dtype": ScaleDtype.E8M0}
    return Float8QuantConfig(granularity=gran, format=Format[case["fmt"]], **more)


def _activations(shape, dt, g, gran):
    """N(0, 1) with 0.1% outliers x50, as activations have them; MX layers get
    values spread over many binades instead."""
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    if gran == "MX_BLOCKWISE":
        s = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
        return (torch.sign(s) * torch.exp(1.5 * x)).to(dt)
    hit = torch.rand(shape, generator=g, device=DEV) < 1e-3
    return torch.where(hit, 50.0 * x, x).to(dt)


def _weights(shape, dt, g):
    return (0.02 * torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)).to(dt)


def _grads(shape, dt, g):
    return (1e-2 * torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)).to(dt)


def _loads(total, G, idle, seed):
    """Rows per expert: weights r^-1.1 over the experts in use, shuffled."""
    g = torch.Generator().manual_seed(int(seed))
    n = max(1, G - idle)
    w = torch.arange(1, n + 1, dtype=torch.float64) ** -1.1
    cnt = torch.floor(total * w / w.sum()).to(torch.int64)
    cnt[0] += total - int(cnt.sum())
    lens = torch.zeros(G, dtype=torch.int64)
    lens[:n] = cnt
    return lens[torch.randperm(G, generator=g)]


def _inputs(case, seed):
    """The high-precision tensors of a case, from the seed alone."""
    g, op = _gen(seed), case["op"]
    dt = _DT[case["dtype"]]
    if op in ("linear", "linear_w8"):
        M, N, K = case["M"], case["N"], case["K"]
        d = {"a": _activations((M, K), dt, g, case["gran"]),
             "w": _weights((N, K) if case["trans_b"] else (K, N), dt, g)}
        if op == "linear":
            d["g"] = _grads((M, N), dt, g)
        return d
    if op in ("moe", "moe_w8"):
        M, N, K, G = case["rows"], case["N"], case["K"], case["G"]
        d = {"a": _activations((M, K), dt, g, case["gran"]), "w": _weights((G, N, K), dt, g),
             "lens": _loads(M, G, case["idle"], seed).to(DEV)}
        if op == "moe":
            d["g"] = _grads((M, N), dt, g)
        return d
    if op == "dispatch":
        T, H, E = case["tokens"], case["hidden"], case["experts"]
        scores = torch.rand((T, E), generator=g, device=DEV)
        probs, idx = torch.topk(scores, case["topk"], dim=1)
        return {"x": _activations((T, H), dt, g, ""), "idx": idx, "probs": probs.contiguous(),
                "g": _grads((T, H), dt, g)}
    return {"x": _activations((case["M"], case["N"]), dt, g, case["gran"])}


def prepare(case, seed):
    op, d = case["op"], _inputs(case, seed)
    state = {"case": case, **d}
    if op in ("linear", "linear_w8", "moe", "moe_w8"):
        state["config"] = _config(case)
    if op in ("linear", "moe"):
        state["a"].requires_grad_(True)
        state["w"].requires_grad_(True)
    elif op in ("linear_w8", "moe_w8"):
        fp8 = torch.float8_e4m3fn
        w, w_t = create_quantized_weight(d["w"], fp8, state["config"], need_weight_transpose_cache=True)
        state["w"] = QuantizedTensorPair(w, w_t)
    elif op == "dispatch":
        state["x"].requires_grad_(True)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    op = case["op"]
    if op == "linear":
        out = turbo.ops.gemm_fp8(state["a"], state["w"], trans_b=case["trans_b"], config=state["config"])
        ga, gw = torch.autograd.grad(out, (state["a"], state["w"]), state["g"])
        return {"out": out.detach(), "grad_a": ga, "grad_w": gw}
    if op == "linear_w8":
        with torch.no_grad():
            return turbo.ops.gemm_fp8(state["a"], state["w"], trans_b=True, config=state["config"])
    if op == "moe":
        out = turbo.ops.grouped_gemm_fp8(state["a"], state["w"], state["lens"], trans_b=True,
                                         config=state["config"])
        ga, gw = torch.autograd.grad(out, (state["a"], state["w"]), state["g"])
        return {"out": out.detach(), "grad_a": ga, "grad_w": gw}
    if op == "moe_w8":
        with torch.no_grad():
            return turbo.ops.grouped_gemm_fp8(state["a"], state["w"], state["lens"], trans_b=True,
                                              config=state["config"])
    if op == "dispatch":
        x = state["x"]
        rows, row_id_map, per_expert, _, n, _, row_probs = turbo.ops.moe_permute(
            x, state["idx"], num_local_experts=case["experts"], num_topk=case["topk"],
            num_permuted_tokens=case["tokens"] * case["topk"], probs=state["probs"])
        back, _ = turbo.ops.moe_unpermute(rows, row_id_map, n, restore_shape=x.shape,
                                          num_local_experts=case["experts"])
        (gx,) = torch.autograd.grad(back, x, state["g"])
        return {"rows": rows.detach(), "per_expert": per_expert, "row_probs": row_probs, "back": back.detach(),
                "grad_x": gx}
    gran, fmt = ScalingGranularity[case["gran"]], _fp8(case)
    x, dt = state["x"], _DT[case["dtype"]]
    if case["gran"] in ("BLOCKWISE", "MX_BLOCKWISE"):
        bs = 128 if case["gran"] == "BLOCKWISE" else 32
        q, s, q_col, s_col = turbo.ops.quantize_fp8_with_trans(x, fmt, gran, block_size=bs)
        y = turbo.ops.dequantize_fp8(q, dt, gran, block_size=bs, axis=1, scale_inv=s)
        return {"q": q, "s": s.view(torch.uint8), "q_col": q_col, "s_col": s_col.view(torch.uint8), "y": y}
    axis = None if case["gran"] == "TENSORWISE" else 1
    q, s = turbo.ops.quantize_fp8(x, fmt, gran, axis=axis)
    y = turbo.ops.dequantize_fp8(q, dt, gran, axis=axis, scale_inv=s)
    return {"q": q, "s": s.view(1).view(torch.uint8) if s.dim() == 0 else s.view(torch.uint8), "y": y}


# ---------------------------------------------------------------------------
# what a correct answer is
# ---------------------------------------------------------------------------
def tolerance(case):
    if case["op"] == "quant":
        return "exact"
    # fp8 operands are exact data and the sums are fp32: what differs between
    # correct implementations is the rounding of the result to 16 bits (measured
    # against 64 bits: 1.7e-3 for bf16, 2.1e-4 for fp16)
    return {"rel": 7e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}


def _fp8(case, fwd=True):
    if case["fmt"] == "HYBRID" and not fwd:
        return torch.float8_e5m2
    return torch.float8_e4m3fn


def _scaled_cast(x, amax, eps, fmt):
    """fp8 bytes and fp32 inverse scales for amax broadcast over x (fp32): the
    quotients are rounded once (an fp64 quotient of fp32 values rounds to the
    correctly rounded fp32 one)."""
    m = _FP8_MAX[fmt]
    s = (m / amax.clamp(min=eps).double()).float()
    inv = (1.0 / s.double()).float()
    return (x * s).clamp(-m, m).to(fmt), inv


def _pad_to(x, rows, cols):
    M, N = x.shape
    out = torch.zeros((-(-M // rows) * rows, -(-N // cols) * cols), dtype=x.dtype, device=x.device)
    out[:M, :N] = x
    return out


def _block(x, fmt, br, bc, eps):
    """Per-(br x bc)-block quantization of a matrix, as fp64 values."""
    M, N = x.shape
    p = _pad_to(x.float(), br, bc)
    v = p.view(p.shape[0] // br, br, p.shape[1] // bc, bc)
    q, inv = _scaled_cast(v, v.abs().amax(dim=(1, 3), keepdim=True), eps, fmt)
    return (q.double() * inv.double()).view(p.shape)[:M, :N]


def _mx(x, fmt, br, bc):
    """MX quantization with one power of two per (br x bc) block, as fp64
    values: the smallest exponent at which the block's maximum does not
    overflow the format."""
    M, N = x.shape
    p = _pad_to(x.float(), br, bc)
    v = p.view(p.shape[0] // br, br, p.shape[1] // bc, bc)
    amax = v.abs().amax(dim=(1, 3), keepdim=True).double()
    m = _FP8_MAX[fmt]
    _, e2 = torch.frexp(amax)
    e = e2 - 1 - (8 if fmt == torch.float8_e4m3fn else 15)
    e = torch.where(torch.ldexp(amax, -e) > m, e + 1, e).clamp(-127, 127)
    e = torch.where(amax > 0, e, torch.full_like(e, -127))
    q = torch.ldexp(v.double(), -e).clamp(-m, m).float().to(fmt)
    out = torch.ldexp(q.double(), e) * (amax > 0)
    return out.view(p.shape)[:M, :N]


def _tensor(x, fmt):
    q, inv = _scaled_cast(x.float(), x.float().abs().amax(), 1e-12, fmt)
    return q.double() * inv.double()


def _row(x, fmt, axis):
    q, inv = _scaled_cast(x.float(), x.float().abs().amax(dim=axis, keepdim=True), 1e-12, fmt)
    return q, inv


def _value(q, inv):
    return q.double() * inv.double()


def _again(q, inv, dt, fmt, axis):
    """The rowwise layers' second copy: dequantized to the input type and
    quantized along the other axis."""
    return _value(*_row((q.float() * inv).to(dt), fmt, axis))


def _layer_operands(case, a, w, g):
    """fp64 operands of the three products of a layer, w as [N, K]:
    (a for out, w for out, g for grad_a, w for grad_a, g for grad_w, a for grad_w)."""
    gran, f, b = case["gran"], _fp8(case), _fp8(case, fwd=False)
    dt = _DT[case["dtype"]]
    if gran == "TENSORWISE":
        qa, qw = _tensor(a, f), _tensor(w, f)
        qg = None if g is None else _tensor(g, b)
        return qa, qw, qg, qw, qg, qa
    if gran == "ROWWISE":
        qa, qw = _row(a, f, 1), _row(w, f, 1)
        if g is None:
            return _value(*qa), _value(*qw), None, None, None, None
        return (_value(*qa), _value(*qw), _value(*_row(g, b, 1)), _again(*qw, dt, f, 0),
                _value(*_row(g, b, 0)), _again(*qa, dt, f, 0))
    if gran == "BLOCKWISE":
        qw = _block(w, f, 128, 128, 1e-4)
        return (_block(a, f, 1, 128, 1e-4), qw, None if g is None else _block(g, b, 1, 128, 1e-4), qw,
                None if g is None else _block(g, b, 128, 1, 1e-4), _block(a, f, 128, 1, 1e-4))
    qw = _mx(w, f, 32, 32)
    return (_mx(a, f, 1, 32), qw, _mx(g, b, 1, 32), qw, _mx(g, b, 32, 1), _mx(a, f, 32, 1))


def exact(case, seed):
    """run()'s answer in 64 bits: quantized as the formats define it, multiplied
    and summed in fp64."""
    d, op = _inputs(case, seed), case["op"]
    if op in ("linear", "linear_w8"):
        w = d["w"] if case["trans_b"] else d["w"].t().contiguous()
        a0, w0, g1, w1, g2, a2 = _layer_operands(case, d["a"], w, d.get("g"))
        out = a0 @ w0.t()
        if op == "linear_w8":
            return out
        gw = g2.t() @ a2
        return {"out": out, "grad_a": g1 @ w1, "grad_w": gw if case["trans_b"] else gw.t().contiguous()}
    if op in ("moe", "moe_w8"):
        lens = d["lens"].tolist()
        f, b = _fp8(case), _fp8(case, fwd=False)
        a, g, w = d["a"], d.get("g"), d["w"]
        if case["gran"] == "TENSORWISE":
            qa, qw = _tensor(a, f), _tensor(w, f)
            qg = None if g is None else _tensor(g, b)
        out, ga, gw, at = [], [], [], 0
        for e, n in enumerate(lens):
            s = slice(at, at + n)
            at += n
            if case["gran"] == "TENSORWISE":
                ops = (qa[s], qw[e], None if g is None else qg[s], qw[e], None if g is None else qg[s], qa[s])
            elif n:
                ops = _layer_operands(case, a[s], w[e], None if g is None else g[s])
            else:
                z = torch.zeros((0, w.shape[2]), dtype=torch.float64, device=DEV)
                h = torch.zeros((0, w.shape[1]), dtype=torch.float64, device=DEV)
                ops = (z, w[e].double(), h, w[e].double(), h, z)
            out.append(ops[0] @ ops[1].t())
            if op == "moe":
                ga.append(ops[2] @ ops[3])
                gw.append(ops[4].t() @ ops[5])
        if op == "moe_w8":
            return torch.cat(out)
        return {"out": torch.cat(out), "grad_a": torch.cat(ga), "grad_w": torch.stack(gw)}
    if op == "dispatch":
        T, k, E = case["tokens"], case["topk"], case["experts"]
        idx = d["idx"].reshape(-1)
        # expert-major rows, tokens in order within an expert
        token = torch.arange(T, device=DEV).repeat_interleave(k)
        order = torch.argsort(idx * T + token)
        row = token[order]
        rows = d["x"][row].double()
        back = torch.zeros((T, case["hidden"]), dtype=torch.float64, device=DEV).index_add_(0, row, rows)
        # the gradient's way back through rows of the input's type
        gx = torch.zeros_like(back).index_add_(0, row, d["g"][row].double())
        return {"rows": rows, "per_expert": None, "row_probs": d["probs"].reshape(-1)[order].double(),
                "back": back, "grad_x": gx}
    x, f, dt = d["x"], _fp8(case), _DT[case["dtype"]]
    if case["gran"] == "MX_BLOCKWISE":
        return {"q": None, "s": None, "q_col": None, "s_col": None, "y": _pad_to(_mx(x, f, 1, 32).to(dt).double(), 1, 128)}
    if case["gran"] == "BLOCKWISE":
        return {"q": None, "s": None, "q_col": None, "s_col": None, "y": _block(x, f, 1, 128, 1e-4).to(dt).double()}
    if case["gran"] == "ROWWISE":
        return {"q": None, "s": None, "y": _value(*_row(x, f, 1))}
    return {"q": None, "s": None, "y": _tensor(x, f)}
