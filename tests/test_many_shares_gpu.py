"""Residual deltas of prompts in four to eight shares of K: the choice at the edges of its range, and the sums."""
import pytest
import torch

from servelab_amd.kernels import HipOps
from servelab_amd.kernels.values import PartialSums

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Rows:
    w = True


def test_which_sizes_take_how_many():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    plan = lambda M, N, K: ops._shares_by_estimate(M, N, K, Rows)
    assert plan(2048, 2048, 11008) == (4, True) and plan(2048, 1536, 8960) == (5, True) and plan(1792, 3584, 18944) == (2, True)
    assert plan(1536, 2048, 11008) is None and plan(2049, 2048, 11008) is None                  # rows of other rules, of no rule
    assert plan(2048, 2048, 8128) is None and plan(2048, 2050, 11008) is None and plan(2048, 8448, 11008) is None
    assert plan(2048, 4352, 8192) is None                                                       # 136 tiles: no second share


def test_two_shares_on_few_cus_stay_with_the_library():
    ops = HipOps(torch.bfloat16, DEV)
    ops._num_cus = 256
    plan = lambda M, N, K: ops._shares_by_estimate(M, N, K, Rows)
    # 192 tiles of 256 rows, 182, 196; 234 of 192 rows
    assert plan(1930, 3072, 8192) is None and plan(1792, 3328, 8192) is None and plan(1792, 3584, 8192) == (2, True)
    assert plan(1537, 3328, 8192) == (2, True)


@pytest.mark.parametrize("M,N,K", [(1537, 260, 8192), (2048, 1024, 8256)])       # part-filled tiles; chunks that do not divide by the shares
def test_the_sums_of_the_shares(M, N, K):
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    ops._shares_plan = lambda *a: None
    ops.BLOCK_MIN_ELEMENTS = 0
    delta = ops.linear(x, ops.prepare_weight(w), None, defer=True)
    assert isinstance(delta, PartialSums) and delta.parts.shape[0] == ops._shares_by_estimate(M, N, K, Rows)[0] >= 2
    # float sums of K terms: K 2^-24 of their absolute sum
    assert ((delta.parts.double().sum(0) - x.double() @ w.double().T).abs() <= K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
