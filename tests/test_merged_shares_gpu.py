"""The kernels that merge shares of keys, on both sides of each of their numbers of shares, against sums in 64 bits."""
import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps
from servelab_amd.kernels.values import AttentionShares, Deferred
from test_float32_forms_gpu import emu_batch
from test_kernels_gpu import make_attention_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shares", [1, 4, 5, 16, 17, 64, 65, 256])
@pytest.mark.parametrize("nh,D", [(3, 64), (2, 128), (1, 96)])
def test_shares_of_bfloat16_attention(shares, nh, D):
    ops, T = HipOps(torch.bfloat16, DEV), 5
    g = torch.Generator(device=DEV).manual_seed(shares + D)
    o = torch.randn(T, nh, shares, D, generator=g, device=DEV)
    ml = torch.rand(T, nh, shares, 2, generator=g, device=DEV) * 3 + 0.5                     # a maximum in powers of two, a sum
    if shares > 2:
        ml[1, 0, 1] = torch.tensor([float("-inf"), 0.0])                                     # a share without keys
        ml[2, 0, :-1, 0], ml[2, 0, :-1, 1] = float("-inf"), 0.0                              # the last alone has some
    w = torch.exp2(ml[..., 0].double() - ml[..., 0].double().amax(-1, keepdim=True))
    want = ((w[..., None] * o.double()).sum(2) / (w * ml[..., 1].double()).sum(2)[..., None]).view(T, nh * D)
    got = ops.combine_shares(AttentionShares(o, ml)).double()
    # float sums of `shares` terms, a division, and a rounding to bfloat16
    size = ((w[..., None] * o.double().abs()).sum(2) / (w * ml[..., 1].double()).sum(2)[..., None]).view(T, nh * D)
    assert ((got - want).abs() <= (shares + 8) * 2.0 ** -23 * size + 2.0 ** -8 * want.abs()).all()


# a sequence of one key, of fewer than shares and of many; heads that end a wavefront's 64 channels and pass them
@pytest.mark.parametrize("shares", [2, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("D", [64, 96, 128])
def test_shares_of_float32_attention(shares, D):
    nh, nkv, page = 4, 2, 16
    ops, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    ops.GENERAL_ATTENTION_WAVES = shares * 3 * nkv                                           # (three tokens, a wavefront a kv head and share)
    qkv, kc, vc, tables, batch = make_attention_case(torch.float32, nh, nkv, D, page, [(1, 1), (40, 1), (1500, 1)])[:5]
    got = ops.paged_attention(qkv, nh, nkv, D, kc, vc, page, tables, batch, D ** -0.5, None)
    want = emu.paged_attention(qkv.cpu(), nh, nkv, D, kc.cpu(), vc.cpu(), page, tables.cpu(), emu_batch(batch), D ** -0.5, None)
    # float32 scores of D products on both sides, and sums of weights that add up to one
    assert float((got.cpu() - want).abs().max()) <= 4e-6 * max(1.0, float(want.abs().max()))


# rows of one load of x and of two, the most there are; half a tile a workgroup, a whole one, a lower one; a single k-step, an odd number of them
@pytest.mark.parametrize("T", [1, 8, 9, 16])
@pytest.mark.parametrize("nh,D,N", [(1, 32, 40), (5, 32, 2048), (8, 64, 300), (3, 64, 4112), (4, 128, 3600)])
def test_the_output_projection_merges_them(T, nh, D, N):
    ops, shares, K = HipOps(torch.bfloat16, DEV), 3, nh * D
    g = torch.Generator(device=DEV).manual_seed(T + N)
    o = torch.randn(T, nh, shares, D, generator=g, device=DEV)
    ml = torch.rand(T, nh, shares, 2, generator=g, device=DEV) * 3 + 0.5
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    gain, stream = torch.ones(N, device=DEV), torch.randn(T, N, generator=g, device=DEV)
    for weight in (ops.prepare_weight(w), ops.prepare_weight(w, residual_delta=True, _th=10)):
        resid = stream.clone()
        rows = ops.add_rmsnorm(resid, Deferred(AttentionShares(o, ml), weight, None), gain, 1e-6, fuse=True)
        x = ops.combine_shares(AttentionShares(o, ml)).double()
        # the merged rows are bfloat16 in both, rounded alike but for sums in another order: at most one of 2^-8 of a value
        size = x.abs() @ w.double().abs().T
        assert ((resid.double() - stream.double() - x @ w.double().T).abs() <= 2.0 ** -8 * size + 1e-6).all()
        assert float((resid.double() - stream.double() - x @ w.double().T).norm() / (x @ w.double().T).norm()) <= 2.0 ** -10
        assert torch.allclose(rows.parts.sum(0)[:T], (resid.double() ** 2).sum(1).float(), rtol=1e-5) and not rows.parts[:, T:].any()
        assert torch.equal(rows.plain_x(), resid.bfloat16())
