"""Prompts' products with float32 results and a bias: which go into the tiles, and their results against 64 bits."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K,tiles", [(1000, 6160, 2048, True), (1500, 7172, 1088, None), (2048, 4100, 1024, None), (600, 6160, 2048, False),
                                        (1000, 6162, 2048, False), (1000, 6160, 2080, False)])
def test_products_with_a_bias(M, N, K, tiles):
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    ops._even_columns = lambda *a: 0
    if tiles is not None:
        assert ops._bias_tiles(M, N, K) is tiles
    else:
        ops._bias_tiles = lambda *a: True                        # (edges of rows, columns and chunks, whatever the rate)
    g = torch.Generator(device=DEV).manual_seed(N)
    x, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    bias = torch.randn(N, generator=g, device=DEV)
    got = ops.linear(x, ops.prepare_weight(w), bias, out_f32=True)
    want = x.double() @ w.double().T + bias.double()
    # float32 sums of K products in any order, one more for the bias
    bar = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + bias.double().abs())
    assert got.shape == (M, N) and got.is_contiguous() and ((got.double() - want).abs() <= bar).all()
