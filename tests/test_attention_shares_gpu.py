"""Attention of a few single tokens that the output projection merges from its shares, against the kernels it stands for."""
import pytest
import torch

from servelab_amd.kernels import HipOps
from servelab_amd.kernels.values import AttentionShares, Deferred
from test_kernels_gpu import make_attention_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one row in 2, 3, 5 .. 8 shares, several rows, a context shorter than its shares,
# rows of 1, 16 and 64 k-steps for sixteen wavefronts, columns of the last tile part-filled, lower tiles
@pytest.mark.parametrize("nh,nkv,D,N,ctx,shares", [(14, 2, 64, 896, [300], 5), (1, 1, 32, 16, [70], 2), (16, 2, 128, 2048, [900], 8),
                                                   (14, 2, 64, 904, [300, 40], 3), (4, 4, 128, 528, [5, 260, 200, 130], 4),
                                                   (32, 8, 64, 1000, [90] * 8, 2), (12, 2, 128, 1536, [500], 6), (8, 1, 64, 512, [33, 700], 8)])
def test_projection_merges_the_shares(nh, nkv, D, N, ctx, shares):
    ops = HipOps(torch.bfloat16, DEV)
    K, T = nh * D, len(ctx)
    qkv, kc, vc, tables, batch = make_attention_case(torch.bfloat16, nh, nkv, D, 16, [(n, 1) for n in ctx], seed=N)[:5]
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    weight = ops.prepare_weight(w, residual_delta=True, **({"_th": 10} if N == 1000 else {}))
    gain, stream, bias = 1 + 0.1 * torch.randn(N, device=DEV), torch.randn(T, N, device=DEV), torch.randn(N, device=DEV)
    ops._decode_launches = lambda n, *a: [(0, n, False, shares)]
    ops.SHARES_MAX_VALUES = 1 << 30

    def run():
        resid = stream.clone()
        delta = ops.attend_and_project(qkv, nh, nkv, D, kc, vc, 16, tables, batch, D ** -0.5, None, weight, bias, defer=True)
        whole = ops.materialize(delta)
        return delta, whole, resid, ops.add_rmsnorm(resid, delta, gain, 1e-6, fuse=True)
    delta, whole, resid, rows = run()
    assert isinstance(delta, Deferred) and isinstance(delta.x, AttentionShares) and delta.x.o.shape == (T, nh, shares, D)
    ops.merge_shares = False
    plain, whole2, resid2, rows2 = run()
    assert not isinstance(plain.x, AttentionShares)
    assert torch.equal(whole, whole2)                                  # (merged by the same kernel)
    # the merged values are rounded to bfloat16 in both, from sums in another order: a value may differ by its last place
    x = plain.x.rows() if hasattr(plain.x, "rows") else plain.x
    bar = 2.0 ** -8 * (x.double().abs() @ w.double().abs().T) * 2.0 ** -3 + 2.0 ** -16
    assert ((resid.double() - resid2.double()).abs() <= bar).all()
    exact = stream.double() + x.double() @ w.double().T + bias.double()
    assert (resid.double() - exact).norm() <= 2.0 ** -9 * (exact - stream.double()).norm()
    near = (rows.plain_x().float() - rows2.plain_x().float()).abs()
    assert (near <= 2.0 ** -7 * rows2.plain_x().float().abs() + 2 * bar.float()).all()
    assert torch.allclose(rows.parts.sum(0)[:T], (resid.double() ** 2).sum(1).float(), rtol=1e-5)


def test_which_steps_leave_their_shares():
    ops = HipOps(torch.bfloat16, DEV)
    nh, nkv, D = 14, 2, 64
    weight = ops.prepare_weight((torch.randn(896, 896, device=DEV) * 0.03).bfloat16())

    def taken(ctx, **changes):
        qkv, kc, vc, tables, batch = make_attention_case(torch.bfloat16, nh, nkv, D, 16, [(n, 1) for n in ctx], seed=1)[:5]
        for name, value in changes.items():
            setattr(ops, name, value)
        return ops._shares_for_projection(len(ctx), nh, nkv, D, tables, 16, batch, None, weight)
    assert 2 <= taken([300]) <= 8 and taken([100]) == 0               # (merged in the workgroup)
    assert taken([300] * 9) == 0                                       # more rows than it takes
    assert taken([4000]) == 0                                          # more shares than it takes
    assert taken([300], SHARES_MAX_K=512) == 0
    assert taken([300], SHARES_MAX_K=2048, SHARES_MAX_VALUES=896) == 0
    assert taken([300], SHARES_MAX_VALUES=8192, merge_shares=False) == 0
