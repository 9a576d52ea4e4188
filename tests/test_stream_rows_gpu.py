"""Norms on a sublayer's output and the stream convolution of single tokens where the number of values a thread keeps and the
channels a block takes change, against float64."""
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def normed(y, eps, gain):
    return y / torch.sqrt((y * y).mean(-1, keepdim=True) + eps) * gain


# one, two, four, eight values a thread of 256 and of 512, one more than whole, more than eight
@pytest.mark.parametrize("H", [64, 257, 512, 513, 1030, 2047, 2049, 4096, 4100])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norms_on_outputs(H, dtype):
    ops, T = HipOps(dtype, DEV), 3
    g = torch.Generator().manual_seed(H)
    x, y = torch.randn(T, H, generator=g), torch.randn(T, H, generator=g).to(dtype)
    wy, w = torch.randn(H, generator=g), torch.randn(H, generator=g)
    # sums of H float terms, one rounding of the rows
    bar = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    r = x.clone().to(DEV)
    out = ops.add_postnorm(r, y.to(DEV), wy.to(DEV), 1e-6, 0.5)
    want = x.double() + 0.5 * normed(y.double(), 1e-6, wy.double())
    assert (r.cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()
    assert (out.cpu().double() - want).abs().max() <= bar * want.abs().max()
    r = x.clone().to(DEV)
    out = ops.add_normed_rmsnorm(r, y.to(DEV), wy.to(DEV), 1e-6, w.to(DEV), 1e-5)
    want = x.double() + normed(y.double(), 1e-6, wy.double())
    assert (r.cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()
    rows = normed(want, 1e-5, w.double())
    assert (out.cpu().double() - rows).abs().max() <= bar * rows.abs().max()


# a block a slice of channels; as many tokens as leave a block two slices, or all of them; a last slice that is not full
@pytest.mark.parametrize("T,C,taps", [(2, 3584, 4), (200, 3584, 2), (600, 3000, 4), (1100, 520, 6), (3, 100, 1)])
@pytest.mark.parametrize("with_output", [True, False])
def test_single_tokens_through_the_stream_convolution(T, C, taps, with_output):
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(T)
    x, y, wy = torch.randn(T, C, generator=g), torch.randn(T, C, generator=g).bfloat16(), torch.randn(C, generator=g)
    w, state = torch.randn(taps, C, generator=g), torch.randn(T, taps * C, generator=g)
    fresh = torch.arange(T) % 3 == 1
    i32 = lambda v: torch.as_tensor(v, dtype=torch.int32, device=DEV)
    batch = SimpleNamespace(cu_q=i32(range(T + 1)), positions=i32((~fresh).int() * 5), tok_seq=i32(range(T)), state_slots=i32(range(T)),
                            num_seqs=T, num_tokens=T, max_q_len=1)
    r, s = x.clone().to(DEV), state.clone().to(DEV)
    kw = dict(y=y.to(DEV), y_weight=wy.to(DEV), y_eps=1e-6) if with_output else {}
    out = ops.stream_conv(r, w.to(DEV), s, 0, batch, True, **kw)
    v = x.double() + (normed(y.double(), 1e-6, wy.double()) if with_output else 0)
    past = state[:, :(taps - 1) * C].view(T, taps - 1, C).double() * (~fresh)[:, None, None]
    want = v + (past * w[:-1].double()).sum(1) + w[-1].double() * v
    assert (r.cpu().double() - v).abs().max() <= 1e-5 * v.abs().max()
    assert (out.cpu().double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    kept = torch.cat([past, v[:, None]], 1)[:, 1:].flatten(1)
    got = s.cpu().double()
    assert (got[:, :(taps - 1) * C] - kept).abs().max() <= 1e-5 * v.abs().max() if taps > 1 else True
    assert torch.equal(s.cpu()[:, (taps - 1) * C:], state[:, (taps - 1) * C:])
