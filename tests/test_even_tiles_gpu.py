"""Products of prompts in tiles that go round the CUs once, at the edges of tiles, chunks and the ring, against sums in 64 bits."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# every width of a tile; rows and columns that end a tile and pass it; one chunk of 64, an odd number, fewer and more than the ring's
@pytest.mark.parametrize("columns", [96, 128, 160, 192, 224])
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (128, 512, 192), (129, 516, 128), (300, 268, 448), (1025, 100, 1024), (527, 1000, 320)])
def test_sums(columns, M, N, K):
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    bias = torch.randn(N, generator=g, device=DEV)
    weight = ops.prepare_weight(w)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bar = K * 2.0 ** -24 * size + 1e-30                      # float sums of K products, rounded once a term at most
    got = ops.linear_even(x, weight, bias, columns, True).double()
    assert ((got - want - bias.double()).abs() <= bar + 2.0 ** -24 * got.abs()).all()
    got = ops.linear_even(x, weight, None, columns).double()
    assert ((got - want).abs() <= bar + 2.0 ** -8 * want.abs()).all()


def test_which_products_take_them():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    c = ops._even_columns
    assert c(2048, 3584, 3584) == 224 and c(2048, 2560, 2048) == 160 and c(527, 4608, 3584) == 96 and c(2048, 2048, 2048) == 128
    assert c(2048, 4608, 3584) == 0 and c(1500, 4096, 4096) == 0             # two rounds; 224 columns on 0.89 of the CUs
    assert c(527, 2048, 4096) == 0 and c(527, 2048, 2048) == 96              # idle CUs with longer rows
    assert c(2048, 2048, 8192) == 0 and c(2048, 2048, 2080) == 0 and c(2048, 508, 2048) == 0 and c(2048, 2050, 2048) == 0
    K, N, M = 512, 640, 700
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    weight, b = ops.prepare_weight(w), torch.randn(N, device=DEV)
    assert torch.equal(ops.linear(x, weight, b), ops.linear_even(x, weight, b, 96))
    assert torch.equal(ops.linear(x, weight, b, True), ops.linear_even(x, weight, b, 96, True))
    # rows that do not start at a multiple of 16 bytes, and matrices without the tiled copy, stay with the library
    odd = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)[1:].view(x.shape).copy_(x)
    calls = []
    ops.linear_even = lambda *a: calls.append(a)
    want = x.double() @ w.double().T
    for got in (ops.linear(odd, weight, None), ops.linear(x, w, None)):
        assert calls == [] and (got.double() - want).norm() <= 2.0 ** -8 * want.norm()


def test_idle_cus():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    c = ops._even_columns
    # few CUs: prompts that wait for the host, or short rows; longer ones from 0.425 of them on
    assert c(448, 2048, 2048) == 96 and c(449, 2048, 2048) == 0 and c(512, 2048, 1024) == 96 and c(512, 2048, 1088) == 0
    assert c(640, 2048, 1536) == 96 and c(640, 1536, 1536) == 0 and c(2048, 512, 2048) == 0 and c(512, 2560, 2048) == 0
    # three quarters of them with rows of more than 2,048 values: in tiles of 96 columns, not of 128
    assert c(512, 4608, 3584) == 96 and c(700, 4096, 4096) == 0 and c(1536, 2048, 2112) == 0 and c(1536, 2048, 2048) == 128
    assert c(1537, 2048, 4096) == 128
