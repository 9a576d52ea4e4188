"""Gated products of a prompt in tiles of 256 or 192 rows of x by 256 rows of W, and the shares of K of a long-row product
of many rows, at the sizes where their edges lie, against float64."""
import pytest
import torch

from servelab_amd.kernels import HipOps
from servelab_amd.kernels.ops import PartialSums

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def act64(z, name):
    if name == "relu":
        return z.clamp(min=0)
    return torch.nn.functional.silu(z) if name == "silu" else torch.nn.functional.gelu(z, approximate="tanh")


# one row of x, a tile less and more by one; half a block's tile of W, a column tile with one matrix-instruction tile, one and
# three chunks of K
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (191, 272, 192), (193, 256, 64), (255, 528, 128), (257, 1040, 192), (385, 32, 64)])
@pytest.mark.parametrize("act", ["silu", "relu", "gelu_tanh"])
@pytest.mark.parametrize("rows", [192, 256])
def test_gated_tiles(M, N, K, act, rows):
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g) if act != "relu" else None
    z = x.double() @ w.double().T + (0 if b is None else b.double())
    z = z.view(M, N // 16, 2, 8)
    want = (act64(z[:, :, 0], act) * z[:, :, 1]).reshape(M, N // 2)
    code = {"silu": 1, "relu": 2, "gelu_tanh": 4}[act]
    got = ops.linear_gated_block(x.to(DEV), ops.prepare_weight(w.to(DEV)), None if b is None else b.to(DEV), rows, code)
    # one rounding to bfloat16 (2^-9 of the value) and float sums of K terms: K 2^-24 of their absolute sum, twice
    # (gate and up), times the other factor
    size = (x.double().abs() @ w.double().abs().T + (0 if b is None else b.double().abs())).max().item()
    bar = 2.0 ** -8 * want.abs() + 4 * K * 2.0 ** -24 * size * z.abs().max().item() + 1e-30
    assert ((got.double().cpu() - want).abs() <= bar).all()


def test_routes_of_prompts_products():
    ops = HipOps(torch.bfloat16, DEV)
    gated = ops._gated_rows
    assert ops._num_cus == 256
    # rows of up to 1,024 values: always, in the tiles that take fewer or shorter rounds
    assert [gated(M, 8192, 1024) for M in (255, 256, 1536, 1537, 2048, 2049, 2560, 2561)] == [None, 192, 192, 256, 256, 192, 192, None]
    assert [gated(M, 9728, 896) for M in (256, 1152, 1153, 1536, 1537)] == [192, 192, 256, 256, 192]
    assert gated(256, 4096, 64) == 192 and gated(256, 4095, 1024) is None and gated(1536, 8192, 1000) is None
    # up to 1,536: one round, 0.7 of it useful
    assert [gated(M, 17920, 1536) for M in (491, 492, 576, 577, 655, 656, 768, 769)] == [None, 192, 192, None, None, 256, 256, None]
    assert gated(1536, 8192, 1536) == 192 and gated(1536, 8192, 1600) is None and gated(1536, 8192, 1056) is None
    # longer rows: several rounds, the last one more than half filled, and no tile of the library's that divides N
    assert [gated(M, 37888, 3584) for M in (1536, 1792, 1793, 2048, 2049)] == [None, None, 256, 256, None]
    assert [gated(M, 27392, 2560) for M in (1536, 1537, 1792, 1793)] == [None, 256, 256, None]
    assert gated(2048, 35840, 3584) is None and gated(2048, 24576, 3072) is None               # 160 times 224, 128 times 192
    assert gated(2048, 9216, 3584) is None and gated(1536, 8192, 1664) is None and gated(2048, 37888, 5184) is None
    x = torch.randn(1200, 1024, device=DEV).bfloat16()
    w = (torch.randn(8192, 1024, device=DEV) * 0.03).bfloat16()
    weight = ops.prepare_weight(w)
    fused = ops.linear_gated_block(x, weight, None, 192, 1)
    assert torch.equal(ops.gated_linear(x, weight, 8), fused)
    # rows that do not start at a multiple of 16 bytes stay with the library, which takes them
    odd = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)[1:].view(x.shape).copy_(x)
    assert (ops.gated_linear(odd, weight, 8).float() - fused.float()).abs().max() <= 2.0 ** -7 * fused.abs().max()
    # a residual delta of 1,537 and more rows: two or three shares
    K, N, M = 8192, 1024, 1600
    w = (torch.randn(N, K, device=DEV) * 0.02).bfloat16()
    weight, x = ops.prepare_weight(w), torch.randn(M, K, device=DEV).bfloat16()
    class Rows:
        w = True
    shares = lambda M, N, K: ops._shares_plan(M, N, K, Rows)
    assert shares(1792, 3584, 18944) is None and shares(1793, 3584, 18944) == (2, True)       # 0.77 and 0.875 of the CUs
    assert shares(1793, 3328, 8192) is None and shares(1537, 3072, 8192) == (3, True) and shares(1793, 3072, 8192) is None
    assert shares(1537, 2560, 9728) == (3, True) and shares(2048, 2048, 11008) is None        # four shares
    ops._num_cus = 64
    assert ops._shares_plan(M, N, K, weight) == (2, True) and ops._shares_plan(1536, N, K, weight) is None
    assert ops._shares_plan(2049, N, K, weight) is None and ops._shares_plan(M, 2 * N, K, weight) is None
    delta = ops.linear(x, weight, None, defer=True)
    assert isinstance(delta, PartialSums) and delta.parts.shape == (2, M, N)
    want = x.double() @ w.double().T
    # float sums of K terms: K 2^-24 of their absolute sum
    assert ((delta.parts.double().sum(0) - want).abs() <= K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
    assert not isinstance(ops.linear(x, weight, None), PartialSums)


def test_shapes_tuned_for_the_library_stay_with_it(tmp_path):
    """The ones whose library product was timed, here or by an earlier process; not those that went to a kernel of this table while
    the tuning was open, nor other numbers of rows."""
    ops, later = HipOps(torch.bfloat16, DEV), HipOps(torch.bfloat16, DEV)
    weight = ops.prepare_weight((torch.randn(8192, 1024, device=DEV) * 0.03).bfloat16())
    x = torch.randn(1700, 1024, device=DEV).bfloat16()
    calls = []
    for table in (ops, later):
        table.linear_gated_block = lambda *a, own=table.linear_gated_block: calls.append(a[0].shape[0]) or own(*a)
    try:
        with ops.library_tuning(1, str(tmp_path / "tuned.csv")):
            ops.gated_linear(x, weight, 8)
            assert ops._block_plan(300, 8192, 1024, weight)
            ops.gated_linear(x[:300], weight, 8)
        with later.library_tuning(1, str(tmp_path / "tuned.csv")):
            pass
        assert calls == []
        for table in (ops, later):
            assert (1700, 8192, 1024) in table._tuned and (320, 8192, 1024) not in table._tuned
            table.gated_linear(x, weight, 8)
            assert calls == []
            table.gated_linear(x[:1650], weight, 8)
            assert calls.pop() == 1650
    finally:
        torch.cuda.tunable.enable(False)
