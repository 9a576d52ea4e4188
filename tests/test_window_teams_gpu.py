"""Prompts through the matrix-core window attention whose workgroups are two teams of wavefronts (every other block of 32 keys) or pairs
of them (halves of the channels), or one team where heads are wide or workgroups many: one block, two, an odd number, a last round for one team alone; caps;
channels that no half divides."""
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps
from test_window_kernels_gpu import dev, fill_pages, paged
from test_window_step_gpu import exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,Dk,Dv,in_keys", [(4, 2, 32, 16, False), (3, 1, 64, 80, False), (8, 2, 128, 128, False), (3, 1, 64, 48, True),
                                              (2, 1, 96, 80, True), (4, 1, 576, 512, True), (3, 1, 256, 256, True), (4, 2, 128, 256, False), (3, 1, 192, 272, False),
                                              (2, 1, 896, 64, False), (3, 1, 512, 384, False), (4, 2, 640, 512, False)])
@pytest.mark.parametrize("window,keep,chunk,softcap", [(None, 0, None, None), (37, 5, None, None), (None, 0, 48, 15.0), (None, 3, 64, None)])
@pytest.mark.parametrize("few", [True, False])
def test_prompts(H, G, Dk, Dv, in_keys, window, keep, chunk, softcap, few):
    ops, page = HipOps(torch.bfloat16, "cuda:0"), 16
    ops._window_few = lambda *a: few                                                     # (both forms, whatever the rule takes)
    g = torch.Generator().manual_seed(Dk + H)
    seqs = [(0, 32), (0, 33), (64, 1), (40, 75), (0, 1), (150, 9)]                       # (cached tokens, tokens of this step)
    lens = [a + b for a, b in seqs]
    tables, kc, vc = paged(lens, page, G, Dk, 0 if in_keys else Dv, torch.bfloat16, g)
    keys = [torch.randn(n, G, Dk, generator=g).bfloat16() for n in lens]
    values = [k[..., :Dv] for k in keys] if in_keys else [torch.randn(n, G, Dv, generator=g).bfloat16() for n in lens]
    fill_pages(tables, kc, vc, keys, None if in_keys else values, page)
    T = sum(b for _, b in seqs)
    q, sinks, slopes = torch.randn(T, H * Dk, generator=g).bfloat16(), torch.randn(H, generator=g), torch.rand(H, generator=g) * 0.1
    gates = torch.randn(T, H * Dv, generator=g)
    cu, pos, want = [0], [], []
    for s, (a, b) in enumerate(seqs):
        for i in range(b):
            o, _ = exact(q[cu[-1] + i].view(H, Dk), keys[s], values[s], a + i, Dk ** -0.5, window, keep, chunk, softcap, slopes, sinks)
            want.append(o * torch.sigmoid(gates[cu[-1] + i].double()).view(H, Dv))
        pos += list(range(a, a + b))
        cu.append(cu[-1] + b)
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    batch = SimpleNamespace(cu_q=i32(cu), positions=i32(pos), num_seqs=len(seqs), num_tokens=T, max_q_len=75, max_ctx_len=max(lens))
    got = ops.window_attention(dev(q), 0, H, G, Dk, Dv, dev(kc), None if in_keys else dev(vc), page, dev(tables), batch, Dk ** -0.5, window, keep,
                               dev(slopes), dev(sinks), softcap=softcap, chunk=chunk, channel_gate=dev(gates)).view(T, H, Dv).double().cpu()
    want = torch.stack(want)
    # results of a few units rounded to bfloat16 (2^-9 of the value); scores, weights and sums are float32
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -12 * want.abs().max() + 1e-5).all(), float((got - want).abs().max())
