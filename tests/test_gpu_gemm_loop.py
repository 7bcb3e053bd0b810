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
