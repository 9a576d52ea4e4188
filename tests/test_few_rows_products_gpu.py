"""The few-rows products in every form of a workgroup (half a tile of W, one, two) at the edges of rows, tiles and k-steps, against
sums in 64 bits."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one k-step, an odd one beside none, one or many pairs (fewer and more than the eight wavefronts, and than the loads of one trip);
# one row, 8, the first of 9 to 16, 16; tiles of few columns, of a half, of one more than a half, many
@pytest.mark.parametrize("M,N,K", [(1, 8, 32), (8, 9, 96), (9, 16, 32), (16, 24, 96), (3, 40, 544), (8, 64, 2048), (5, 50, 2080),
                                   (1, 2048, 4128), (2, 300, 11008), (9, 200, 4128), (16, 2056, 544), (12, 33, 1056)])
@pytest.mark.parametrize("tiles", [0, 1, 2])
def test_every_form_of_a_workgroup(M, N, K, tiles):
    ops = HipOps(torch.bfloat16, DEV)
    ops._tiles_a_workgroup = lambda *a: tiles
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    bias, gain = torch.randn(N, generator=g, device=DEV), 1 + 0.1 * torch.randn(N, generator=g, device=DEV)
    weight = ops.prepare_weight(w)
    exact = x.double() @ w.double().T
    # sums of K float32 products in any order, each sum rounded once a matrix instruction and once a wavefront: K roundings at most
    bar = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    plain = ops.linear_skinny(x, weight, bias, True)
    assert ((plain.double() - exact - bias.double()).abs() <= bar + 2.0 ** -24 * plain.double().abs()).all()
    rounded = ops.linear_skinny(x, weight, None)
    assert ((rounded.double() - exact).abs() <= bar + 2.0 ** -8 * exact.abs()).all()
    # added to a stream, whose rows and sums of squares come with it
    stream = torch.randn(M, N, generator=g, device=DEV)
    resid = stream.clone()
    rows = ops.add_rmsnorm(resid, ops.linear(x, weight, bias, defer=True), gain, 1e-6, fuse=True)
    assert ((resid.double() - stream.double() - exact - bias.double()).abs() <= bar + 2.0 ** -23 * (resid.double().abs() + exact.abs())).all()
    assert torch.allclose(rows.parts.sum(0)[:M], (resid.double() ** 2).sum(1).float(), rtol=1e-5)
    assert not rows.parts[:, M:].any()
    assert torch.equal(rows.plain_x(), (resid * gain).bfloat16())


# rows of up to one load of x and of two; half tiles (th None) and lower ones
@pytest.mark.parametrize("M", [8, 16])
@pytest.mark.parametrize("th", [None, 8])
@pytest.mark.parametrize("K,plain,added", [(896, (8.0e-8, 8.3e-8), (8.0e-8, 8.3e-8)), (11008, (1.65e-7, 2.3e-7), (1.4e-7, 1.75e-7)),
                                           (27648, (2.6e-7, 3.7e-7), (2.0e-7, 2.7e-7))])
def test_running_sums_are_no_longer_than_they_were(M, th, K, plain, added):
    """Errors of results, and of deltas in a float stream, against 64 bits: no larger than with a workgroup of eight wavefronts, or of sixteen for
    deltas of 2,048 values and more, whose odd and even k-steps were summed apart at up to eight rows (measured so 3 to 10 % below the bars)."""
    ops, N = HipOps(torch.bfloat16, DEV), 2048
    errors = []
    for seed in range(4):
        g = torch.Generator(device=DEV).manual_seed(seed)
        x, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
        ops.lower_tiles = th is not None
        weight, want = ops.prepare_weight(w, residual_delta=True, _th=th), x.double() @ w.double().T
        stream = torch.zeros(M, N, device=DEV)
        ops.add_rmsnorm(stream, ops.linear(x, weight, None, defer=True), torch.ones(N, device=DEV), 1e-6, fuse=True)
        errors.append([float((got.double() - want).norm() / want.norm()) for got in (ops.linear_skinny(x, weight, None, True), stream)])
    for got, bar in zip(zip(*errors), (plain, added)):
        assert sum(got) / len(got) <= bar[M > 8]


def test_halves_go_round_the_cus_once():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    assert [ops._tiles_a_workgroup(4, N, 2048, 16, False) for N in (64, 2048, 2049, 3584)] == [0, 0, 1, 1]
    assert ops._tiles_a_workgroup(4, 2048, 2048, 16, True) == 1 and ops._tiles_a_workgroup(4, 2048, 2048, 10, False) == 1


def test_three_halves_on_a_cu_for_two_tiles():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    form = lambda M, N, K, whole=False, plain=True: ops._tiles_a_workgroup(M, N, K, 16, whole, plain)
    assert [form(4, N, 1024) for N in (4096, 4097, 6144, 6145)] == [1, 0, 0, 1]
    assert form(5, 5120, 1024) == 1 and form(4, 5120, 992) == 1 and form(4, 5120, 1024, True) == 1 and form(4, 5120, 1024, False, False) == 1
    # the products, and a delta of as many columns, whose sums of squares are one a whole tile
    M, N, K = 3, 4136, 1056
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    ops.lower_tiles = False
    weight, want = ops.prepare_weight(w, residual_delta=True), x.double() @ w.double().T
    bar = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    assert ((ops.linear(x, weight, None, True).double() - want).abs() <= bar).all()
    stream = torch.zeros(M, N, device=DEV)
    rows = ops.add_rmsnorm(stream, ops.linear(x, weight, None, defer=True), torch.ones(N, device=DEV), 1e-6, fuse=True)
    assert ((stream.double() - want).abs() <= bar).all() and rows.parts.shape[0] == -(-N // 16)
