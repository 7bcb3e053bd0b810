"""The 256 x 256-tile GEMM's main loops at K extents around their prologue (one,
two and three K blocks, cut last blocks) and tiles cut in either dimension, bit
for bit against the small-tile kernel (same K and scaling order)."""

import pytest
import torch

from test_gpu_gemm_small import _cd, _scales, _strided_args

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scales", ["TENSORWISE", "ROWWISE", "BLOCK_1Dx2D", "BLOCK_2Dx1D", "BLOCK_1Dx1D", "MX_KMAJOR"])
@pytest.mark.parametrize("K", [16, 128, 144, 256, 272, 384, 400, 512, 1152])
@pytest.mark.parametrize("mn", [(256, 512), (129, 257), (300, 136)])
def test_large_tile_loop_edges(scales, K, mn):
    from primus_turbo.pytorch.kernels.gemm.gemm_fp8_impl import gemm_fp8_nt

    if scales.startswith("MX") and K % 128:
        pytest.skip("MX takes whole K blocks")
    M, N = mn
    kb = _cd(K, 128)
    if scales == "BLOCK_2Dx1D":  # C^T of the forward: the weight on the A side
        qa, qb, g, nt = _strided_args(M, N, K, "BLOCK_1Dx2D", 60)
        nt = dict(a_scale=_scales((_cd(M, 128), kb), 61), sa_strides=(kb, 1), a_scale_2d=True,
                  b_scale=_scales((N, kb), 62), sb_strides=(kb, 1))
    else:
        qa, qb, g, nt = _strided_args(M, N, K, scales, 60)
    large = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt, large_tiles_only=True)
    small = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt)
    again = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt, large_tiles_only=True)
    torch.cuda.synchronize()
    assert torch.equal(large.view(torch.int16), small.view(torch.int16))
    assert torch.equal(large.view(torch.int16), again.view(torch.int16))


@pytest.mark.parametrize("gran", ["TENSORWISE", "ROWWISE", "BLOCKWISE", "MX_BLOCKWISE"])
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("mnk", [(33, 264, 160), (256, 512, 384)])
def test_forward_without_gradients_is_the_same(gran, trans_b, mnk):
    """A call that no gradient can follow makes no backward copies: the same
    output, for high-precision operands and for a weight quantized once."""
    import primus_turbo.pytorch as turbo
    from primus_turbo.pytorch.core.low_precision import Float8QuantConfig, ScaleDtype, ScalingGranularity
    from primus_turbo.pytorch.core.quantized_tensor import QuantizedTensor, create_quantized_weight

    if gran == "MX_BLOCKWISE" and not trans_b:
        pytest.skip("MX takes the NT layout")
    more = {"BLOCKWISE": dict(block_size=128), "MX_BLOCKWISE": dict(block_size=32, scale_dtype=ScaleDtype.E8M0)}
    cfg = Float8QuantConfig(granularity=ScalingGranularity[gran], **more.get(gran, {}))
    M, N, K = mnk
    g = torch.Generator().manual_seed(5)
    a = torch.randn((M, K), generator=g).bfloat16().cuda()
    w = torch.randn((N, K) if trans_b else (K, N), generator=g).bfloat16().cuda()
    want = turbo.ops.gemm_fp8(a.clone().requires_grad_(), w, trans_b=trans_b, config=cfg)
    with torch.no_grad():
        assert torch.equal(turbo.ops.gemm_fp8(a, w, trans_b=trans_b, config=cfg), want)
    assert torch.equal(turbo.ops.gemm_fp8(a, w, trans_b=trans_b, config=cfg), want)
    if trans_b or gran in ("TENSORWISE", "BLOCKWISE"):
        qw = create_quantized_weight(w, torch.float8_e4m3fn, cfg)[0]
        assert isinstance(qw, QuantizedTensor)
        assert torch.equal(turbo.ops.gemm_fp8(a, qw, trans_b=trans_b, config=cfg), want)


@pytest.mark.parametrize("scales,mnk", [("BLOCK_1Dx2D", (1000, 3080, 4000)), ("BLOCK_1Dx1D", (1000, 3080, 4016)),
                                        ("TENSORWISE", (1500, 4000, 4048)), ("ROWWISE", (1000, 4000, 3984)),
                                        ("BLOCK_1Dx1D", (1024, 4096, 2048)), ("BLOCK_1Dx1D", (1536, 4096, 1936))])
def test_k_split_of_cut_extents(scales, mnk):
    """K splits whose last block is cut, and the shorter ones that 1-D by 1-D
    scales take: the whole-K kernel's result to within the fp32 summation order, and
    the same bits again.  Two fp32 sums that differ in their last bits round to bf16
    values at most one unit apart, 2^-7 of the value; where terms cancel, the sums'
    own difference (the terms' magnitude times a few thousand roundings of 2^-24)
    stays below 2^-14 of the largest result."""
    from primus_turbo.pytorch.kernels.gemm.gemm_fp8_impl import gemm_fp8_nt

    M, N, K = mnk
    qa, qb, g, nt = _strided_args(M, N, K, scales, 70)
    out = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt)
    again = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt)
    ref = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt, large_tiles_only=True)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    o, r = out.double(), ref.double()
    assert bool(((o - r).abs() <= 2.0**-7 * r.abs() + 2.0**-14 * r.abs().max()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(40, 24), (130, 1000), (257, 136), (300, 1001), (128, 256)])
def test_padded_quantized_rows(shape, dtype):
    """Rows padded to 16 hold the unpadded bytes and zeros; rows of whole 8-element
    chunks (not 16) give what the oracle's definition gives."""
    import numpy as np

    from helpers import u8
    from oracle import oracle as O
    from primus_turbo.pytorch.kernels.quantization.quantization_impl import (
        quant_fp8_blockwise_dual_impl,
        quant_fp8_blockwise_for_weight_impl,
    )

    M, N = shape
    x = (torch.randn(shape, generator=torch.Generator().manual_seed(N)) * 3).to(dtype)
    x[0, 0], x[1, 1] = float("inf"), float("nan")
    want = O.quant_block_dual(x, 0)
    wq, ws = O.quant_block_weight(x, 0)
    for pad in (False, True):
        qr, sr, qc, sc = quant_fp8_blockwise_dual_impl(x.cuda(), torch.float8_e4m3fn, 128, row_pad16=pad)
        assert np.array_equal(u8(qr)[:, :N], want[0]) and not u8(qr)[:, N:].any()
        assert np.array_equal(u8(qc), want[2])
        assert np.array_equal(sr.cpu().numpy(), want[1]) and np.array_equal(sc.cpu().numpy(), want[3])
        q, s, qt = quant_fp8_blockwise_for_weight_impl(x.cuda(), torch.float8_e4m3fn, 128, with_transpose=True, pad16=pad)
        assert np.array_equal(u8(q)[:, :N], wq) and not u8(q)[:, N:].any() and np.array_equal(s.cpu().numpy(), ws)
        assert np.array_equal(u8(qt)[:, :M], wq.T) and not u8(qt)[:, M:].any()


@pytest.mark.parametrize("K", [2048, 4016])
def test_split_without_its_workspace_runs_whole(K):
    """A problem that splits only for its 1-D by 1-D scales or with a cut K takes a
    call without the partial tiles' workspace, bit for bit the unsplit kernel."""
    from primus_turbo.pytorch import _C
    from primus_turbo.pytorch.kernels.gemm.gemm_fp8_impl import gemm_fp8_nt

    M, N = 1024, 4096
    qa, qb, g, nt = _strided_args(M, N, K, "BLOCK_1Dx1D", 70)
    ref = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt, large_tiles_only=True)
    real = _C.workspace
    try:
        _C.workspace = lambda n, device: None
        got = gemm_fp8_nt(qa, qb, torch.bfloat16, g, **nt)
    finally:
        _C.workspace = real
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
