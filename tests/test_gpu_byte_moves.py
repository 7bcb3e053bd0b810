"""Byte transposes and dequantization at the sizes where their tiles, access
widths and row chunks change (GPU)."""

import pytest
import torch

from primus_turbo.pytorch.kernels.grouped_gemm.grouped_gemm_fp8_impl import grouped_gemm_fp8_variable_k_impl
from primus_turbo.pytorch.kernels.quantization.quantization_impl import transpose_fp8
from primus_turbo.pytorch.core.low_precision import ScalingGranularity, ScalingRecipe
from primus_turbo.pytorch.ops.quantization import dequantize_fp8, quantize_fp8

pytestmark = pytest.mark.gpu
E4 = torch.float8_e4m3fn


def _bytes(shape, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, 256, shape, generator=g, dtype=torch.uint8)


@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("M", [1, 16, 127, 128, 136, 250, 257])
@pytest.mark.parametrize("N", [1, 8, 120, 128, 130, 272])
def test_transpose_widths(B, M, N):
    x = _bytes((B, M, N), M * 1000 + N)
    y = transpose_fp8(x.cuda().view(E4)).view(torch.uint8).cpu()
    assert torch.equal(y, x.transpose(1, 2).contiguous())


@pytest.mark.parametrize("off", [1, 8])
def test_transpose_of_a_shifted_buffer(off):
    """A base pointer that is not 16-byte aligned takes the narrower accesses."""
    x = _bytes((off + 256 * 128,), off)
    v = x.cuda()[off:].view(256, 128)
    assert torch.equal(transpose_fp8(v.view(E4)).view(torch.uint8).cpu(), x[off:].view(256, 128).t().contiguous())


@pytest.mark.parametrize("cols", [(128, 256), (136, 72), (130, 257)])
def test_segment_transpose_through_variable_k(cols):
    """Small integers: the products are exact, so the whole result is."""
    lens = torch.tensor([0, 1, 127, 128, 129, 0, 300])
    M = int(lens.sum())
    g = torch.Generator().manual_seed(7)
    a = torch.randint(-4, 5, (M, cols[0]), generator=g).float()
    b = torch.randint(-4, 5, (M, cols[1]), generator=g).float()
    offs = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)])
    one = torch.ones((), device="cuda")
    out = grouped_gemm_fp8_variable_k_impl(a.to(E4).cuda(), b.to(E4).cuda(), one, one, lens.cuda(), offs.cuda(), True,
                                           False, False, torch.float32, ScalingGranularity.TENSORWISE.value)
    for i in range(lens.numel()):
        s = slice(int(offs[i]), int(offs[i + 1]))
        assert torch.equal(out[i].cpu(), a[s].t() @ b[s])


# rows of whole 8-element chunks take the vector kernel, others the scalar one
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 8), (5, 128), (257, 264), (300, 100), (3, 1001)])
def test_dequant_routes_agree_with_the_definition(shape, out_dtype):
    g = torch.Generator().manual_seed(shape[1])
    x = (torch.randn(shape, generator=g) * 3).to(torch.bfloat16).cuda()

    def want(q, s):
        return (q.float().cpu() * s.float().cpu()).to(out_dtype)

    q, s = quantize_fp8(x, E4, ScalingGranularity.TENSORWISE)
    assert torch.equal(dequantize_fp8(q, out_dtype, ScalingGranularity.TENSORWISE, scale_inv=s).cpu(), want(q, s))
    for axis in (0, 1):
        q, s = quantize_fp8(x, E4, ScalingGranularity.ROWWISE, axis=axis)
        y = dequantize_fp8(q, out_dtype, ScalingGranularity.ROWWISE, axis=axis, scale_inv=s)
        assert torch.equal(y.cpu(), want(q, s))
        q, s = quantize_fp8(x, E4, ScalingGranularity.BLOCKWISE, axis=axis, block_size=128)
        y = dequantize_fp8(q, out_dtype, ScalingGranularity.BLOCKWISE, axis=axis, block_size=128, scale_inv=s)
        wide = s.repeat_interleave(128, dim=axis)[: shape[0], : shape[1]]
        assert torch.equal(y.cpu(), want(q, wide))
    recipe = ScalingRecipe(use_2d_block=True)
    x3 = torch.stack([x, x * 2])
    q, s = quantize_fp8(x3, E4, ScalingGranularity.BLOCKWISE, block_size=128, scaling_recipe=recipe)
    y = dequantize_fp8(q, out_dtype, ScalingGranularity.BLOCKWISE, block_size=128, scale_inv=s, scaling_recipe=recipe)
    wide = s.repeat_interleave(128, 1).repeat_interleave(128, 2)[:, : shape[0], : shape[1]]
    assert torch.equal(y.cpu(), want(q, wide))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fmt", [E4, torch.float8_e5m2])
@pytest.mark.parametrize("shape", [(16, 16), (128, 128), (144, 272), (1040, 528), (4096, 512)])
def test_rowwise_columns_transposed(shape, fmt, dtype):
    """The column quantization that writes transposed bytes, from high-precision
    rows and from fp8 rows, against the definition (quotients rounded once)."""
    from primus_turbo.pytorch.kernels.quantization.quantization_impl import quantize_fp8_rowwise_cols_t_impl

    g = torch.Generator().manual_seed(shape[0])
    x = (torch.randn(shape, generator=g) * torch.logspace(-6, 3, shape[1])).to(dtype)
    x[:, 1] = 0
    x[0, 2], x[1, 2], x[0, 3] = float("inf"), -float("inf"), float("nan")
    top = torch.finfo(fmt).max

    def want(v):
        a = v.float().abs().nan_to_num(nan=0.0, posinf=float("inf")).amax(0)
        s = (top / a.clamp(min=1e-12).double()).float()
        p = v.float() * s
        q = torch.where(p.isnan(), torch.full_like(p, top), p).clamp(-top, top).to(fmt)
        return q.t().contiguous().view(torch.uint8), (1.0 / s.double()).float()

    q, s = quantize_fp8_rowwise_cols_t_impl(x.cuda(), fmt)
    wq, ws = want(x)
    assert torch.equal(q.view(torch.uint8).cpu(), wq) and torch.equal(s.cpu(), ws)
    plain = quantize_fp8(x.cuda(), fmt, ScalingGranularity.ROWWISE, axis=0)
    assert torch.equal(plain[0].view(torch.uint8).cpu(), wq.t()) and torch.equal(plain[1].cpu().view(-1), ws)
    # fp8 rows with a scale each: as their dequantization to dtype
    x = torch.nan_to_num(x.float(), nan=1.0, posinf=2.0, neginf=-2.0).to(dtype)
    r, rs = quantize_fp8(x.cuda(), fmt, ScalingGranularity.ROWWISE, axis=1)
    q, s = quantize_fp8_rowwise_cols_t_impl(r, fmt, rs, dtype)
    wq, ws = want((r.float().cpu() * rs.cpu()).to(dtype))
    assert torch.equal(q.view(torch.uint8).cpu(), wq) and torch.equal(s.cpu(), ws)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt", [E4, torch.float8_e5m2])
def test_rowwise_columns_of_special_rows(fmt, dtype):
    """The column maximum is rounded once, after the maximum: every byte pattern,
    products past the type's largest value and below its smallest, and row scales
    that are zero, infinite or NaN give what quantizing the dequantized rows gives."""
    from primus_turbo.pytorch.kernels.quantization.quantization_impl import quantize_fp8_rowwise_cols_t_impl

    r = _bytes((208, 528), 5).view(fmt)
    rs = torch.logspace(-42, 36, 208)
    rs[3], rs[70], rs[131] = 0.0, float("inf"), float("nan")
    keep = torch.arange(528) % 3 > 0  # a third of the columns has every special value
    clean = torch.randn((208, 528), generator=torch.Generator().manual_seed(6)).to(fmt)
    r = torch.where(keep[None], clean.view(torch.uint8), r.view(torch.uint8)).cuda().view(fmt)
    for scales in (rs, torch.logspace(-9, 2, 208)):
        sc = scales.cuda()[:, None].contiguous()
        q, s = quantize_fp8_rowwise_cols_t_impl(r, fmt, sc, dtype)
        wq, ws = quantize_fp8_rowwise_cols_t_impl((r.float() * sc).to(dtype), fmt)
        assert torch.equal(s.view(torch.int32), ws.view(torch.int32))
        assert torch.equal(q.view(torch.uint8), wq.view(torch.uint8))


@pytest.mark.parametrize("trans_b", [True, False])
def test_rowwise_layer_takes_a_gradient_at_an_odd_offset(trans_b):
    """A contiguous gradient whose storage starts off a 16-byte boundary gives the
    bits that an aligned copy of it gives."""
    from primus_turbo.pytorch.core.low_precision import Float8QuantConfig
    from primus_turbo.pytorch.ops import gemm_fp8

    M, N, K = 144, 272, 128
    g = torch.Generator().manual_seed(9)
    a = torch.randn((M, K), generator=g).bfloat16().cuda().requires_grad_()
    b = torch.randn((N, K) if trans_b else (K, N), generator=g).bfloat16().cuda().requires_grad_()
    config = Float8QuantConfig(granularity=ScalingGranularity.ROWWISE)
    grad = torch.randn(M * N + 1, generator=g).bfloat16().cuda()[1:].view(M, N)
    assert grad.data_ptr() % 16
    got = torch.autograd.grad(gemm_fp8(a, b, trans_b=trans_b, config=config), (a, b), grad)
    want = torch.autograd.grad(gemm_fp8(a, b, trans_b=trans_b, config=config), (a, b), grad.clone())
    assert all(torch.equal(x, y) for x, y in zip(got, want))
