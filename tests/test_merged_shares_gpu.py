"""The kernels that merge shares of keys, on both sides of each of their numbers of shares, against sums in 64 bits."""
import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps
from servelab_amd.kernels.values import AttentionShares
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
