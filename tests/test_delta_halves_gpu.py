"""Deltas of few columns in halves of tiles: which matrices, and the trips to memory of 8 to 11 pairs of k-steps a wavefront."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_no_copy_in_lower_tiles_where_halves_go_round():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    make = lambda N: ops.prepare_weight(torch.zeros(N, 64, dtype=torch.bfloat16, device=DEV), residual_delta=True)
    assert make(896).lower is None and make(2048).lower is None and make(2049).th == ops.producer_tile_height(2049)[0]
    assert make(5120).th == 10


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("K", [2048, 2080, 4096, 4640, 4864, 5120, 5152])       # 4, 5, 8, 9.1, 9.5, 10 and 10.1 pairs a wavefront
def test_trips_of_halves(M, K):
    ops, N = HipOps(torch.bfloat16, DEV), 120
    g = torch.Generator(device=DEV).manual_seed(K + M)
    x, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    weight, want = ops.prepare_weight(w, residual_delta=True), x.double() @ w.double().T
    bar = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30            # every product exact, K roundings at most
    stream = torch.zeros(M, N, device=DEV)
    rows = ops.add_rmsnorm(stream, ops.linear(x, weight, None, defer=True), torch.ones(N, device=DEV), 1e-6, fuse=True)
    assert ((stream.double() - want).abs() <= bar).all() and not rows.parts[:, M:].any()
    assert ((ops.linear_skinny(x, weight, None, True).double() - want).abs() <= bar).all()
