"""Window attention of steps of one token a sequence on the matrix cores, against sums in 64 bits: windows, chunks and kept first tokens
whose borders lie in blocks of 32 keys, slots that hold NaN where no key is seen, shares without a block."""
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps
from test_window_kernels_gpu import dev, fill_pages, paged

pytestmark = pytest.mark.gpu


def exact(q, keys, values, pos, scale, window, keep, chunk, softcap, slopes, sinks):
    g = q.shape[0] // keys.shape[1]
    s = torch.einsum("hd,jhd->hj", q.double(), keys.double().repeat_interleave(g, 1)) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    j = torch.arange(keys.shape[0])
    if slopes is not None:
        s = s - slopes.double()[:, None] * (pos - j).double()
    seen = (j <= pos) & (((pos - j < (window or pos + 1)) & ((j // chunk == pos // chunk) if chunk else (j >= 0))) | (j < keep))
    s = s.masked_fill(~seen, float("-inf"))
    if sinks is not None:
        s = torch.cat([s, sinks.double()[:, None]], 1)
    p = torch.softmax(s, -1)[:, :keys.shape[0]]
    return torch.einsum("hj,jhd->hd", p, values.double().repeat_interleave(g, 1)), seen


# one column, groups that fill a tile of 16 columns, pass it, and fill two; channels of one tile and of many; workgroups of four wavefronts and of
# two (beyond 256 channels of values with pages of their own); widths whose steps take the kernel of prompts
@pytest.mark.parametrize("H,G,Dk,Dv,in_keys", [(2, 2, 32, 16, False), (8, 2, 128, 128, False), (16, 1, 64, 80, False), (20, 1, 96, 64, False),
                                              (3, 1, 64, 48, True), (32, 1, 576, 512, True), (17, 1, 96, 96, False), (8, 2, 128, 256, False),
                                              (17, 1, 192, 272, False), (2, 1, 896, 64, False), (17, 1, 512, 384, False), (4, 2, 640, 512, False),
                                              (20, 1, 256, 256, True)])
@pytest.mark.parametrize("window,keep,chunk,page,shares", [(None, 0, None, 16, 32), (9, 3, None, 16, 32), (40, 33, None, 32, 3), (None, 0, 48, 16, 5),
                                                          (1, 1, None, 64, 32), (700, 4, 512, 16, 1), (None, 0, None, 16, 1)])
@pytest.mark.parametrize("step", [True, False])
def test_steps_of_one_token(H, G, Dk, Dv, in_keys, window, keep, chunk, page, shares, step):
    ops = HipOps(torch.bfloat16, "cuda:0")
    ops.WINDOW_MFMA_MAX_SHARES = shares
    ops._window_takes_step = lambda *a: step                                       # (the kernel for steps, shares of the one for prompts)
    gen = torch.Generator().manual_seed(Dk + keep)
    # the first token, the ends of a page and of a block, a context of more blocks than a lane asks table entries for
    lens = [1, 16, 32, 33, 75, 4700 if shares == 1 else 1100]
    tables, kc, vc = paged(lens, page, G, Dk, 0 if in_keys else Dv, torch.bfloat16, gen)
    keys = [torch.randn(n, G, Dk, generator=gen).bfloat16() for n in lens]
    values = [k[..., :Dv] for k in keys] if in_keys else [torch.randn(n, G, Dv, generator=gen).bfloat16() for n in lens]
    fill_pages(tables, kc, vc, keys, None if in_keys else values, page)
    S = len(lens)
    q = torch.randn(S, H * Dk + 8, generator=gen).bfloat16()
    rich = shares != 32 or window is None
    slopes = torch.rand(H, generator=gen) * 0.1 if rich else None
    sinks = torch.randn(H, generator=gen) if rich else None
    gates = torch.randn(S, H * Dv, generator=gen) if shares == 3 else None
    softcap = 20.0 if shares == 5 else None
    want = []
    for s, n in enumerate(lens):
        o, seen = exact(q[s, 8:].view(H, Dk), keys[s], values[s], n - 1, Dk ** -0.5, window, keep, chunk, softcap, slopes, sinks)
        want.append(o * torch.sigmoid(gates[s].double()).view(H, Dv) if gates is not None else o)
        for p in range(-(-n // page)):                               # what no query sees: NaN, and not in the table where a page is
            places = [j for j in range(p * page, min((p + 1) * page, n)) if not seen[j]]
            for j in places:
                kc[int(tables[s, p]), :, j % page] = float("nan")
                vc[int(tables[s, p]), :, :, j % page] = float("nan")
            if len(places) == min((p + 1) * page, n) - p * page:
                tables[s, p] = 0
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    batch = SimpleNamespace(cu_q=i32(list(range(S + 1))), positions=i32([n - 1 for n in lens]), num_seqs=S, num_tokens=S, max_q_len=1,
                            max_ctx_len=max(lens))
    args = (dev(q), 8, H, G, Dk, Dv, dev(kc), None if in_keys else dev(vc), page, dev(tables), batch, Dk ** -0.5, window, keep,
            None if slopes is None else dev(slopes), None if sinks is None else dev(sinks))
    more = dict(softcap=softcap, chunk=chunk, channel_gate=None if gates is None else dev(gates))
    got = ops.window_attention(*args, **more).view(S, H, Dv).double().cpu()
    want = torch.stack(want)
    assert torch.isfinite(got).all()
    # results of a few units rounded to bfloat16 (2^-9 of the value); scores, weights and sums are float32
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -12 * want.abs().max() + 1e-5).all(), float((got - want).abs().max())


@pytest.mark.parametrize("H,G,Dk,Dv,in_keys", [(20, 1, 64, 80, False), (8, 2, 128, 128, False), (3, 1, 64, 48, True), (17, 1, 512, 384, False)])
@pytest.mark.parametrize("shares", [1, 3, 32])
def test_a_sequence_without_a_token(H, G, Dk, Dv, in_keys, shares):
    """Two tokens of three sequences: the kernel of prompts, over shares of the keys."""
    ops, page, lens = HipOps(torch.bfloat16, "cuda:0"), 16, [300, 40, 75]
    ops.WINDOW_MFMA_MAX_SHARES = shares
    gen = torch.Generator().manual_seed(Dk)
    tables, kc, vc = paged(lens, page, G, Dk, 0 if in_keys else Dv, torch.bfloat16, gen)
    keys = [torch.randn(n, G, Dk, generator=gen).bfloat16() for n in lens]
    values = [k[..., :Dv] for k in keys] if in_keys else [torch.randn(n, G, Dv, generator=gen).bfloat16() for n in lens]
    fill_pages(tables, kc, vc, keys, None if in_keys else values, page)
    q, sinks = torch.randn(2, H * Dk, generator=gen).bfloat16(), torch.randn(H, generator=gen)
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    batch = SimpleNamespace(cu_q=i32([0, 1, 1, 2]), positions=i32([299, 74]), num_seqs=3, num_tokens=2, max_q_len=1, max_ctx_len=300)
    got = ops.window_attention(dev(q), 0, H, G, Dk, Dv, dev(kc), None if in_keys else dev(vc), page, dev(tables), batch, Dk ** -0.5, None, 0, None,
                               dev(sinks)).view(2, H, Dv).double().cpu()
    want = torch.stack([exact(q[i].view(H, Dk), keys[s], values[s], lens[s] - 1, Dk ** -0.5, None, 0, None, None, None, sinks)[0]
                        for i, s in enumerate((0, 2))])
    # results of a few units rounded to bfloat16 (2^-9 of the value); scores, weights and sums are float32
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -12 * want.abs().max() + 1e-5).all(), float((got - want).abs().max())


@pytest.mark.parametrize("shares", [1, 2, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("Dv", [16, 64, 80])
def test_merging_of_shares(shares, Dv):
    """Every number of shares the merging kernel is built for and one more, over the float kernel's shares (some without a key)."""
    ops, H, page = HipOps(torch.float32, "cuda:0"), 2, 16
    ops.WINDOW_MAX_SHARES, ops.WINDOW_SHARE_KEYS = shares, 1
    gen = torch.Generator().manual_seed(shares)
    lens = [300, 5]
    tables, kc, vc = paged(lens, page, 1, 24, Dv, torch.float32, gen)
    keys, values = ([torch.randn(n, 1, d, generator=gen) for n in lens] for d in (24, Dv))
    fill_pages(tables, kc, vc, keys, values, page)
    q, sinks = torch.randn(2, H * 24, generator=gen), torch.randn(H, generator=gen)
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    batch = SimpleNamespace(cu_q=i32([0, 1, 2]), positions=i32([299, 4]), num_seqs=2, num_tokens=2, max_q_len=1, max_ctx_len=300)
    got = ops.window_attention(dev(q), 0, H, 1, 24, Dv, dev(kc), dev(vc), page, dev(tables), batch, 0.2, None, 0, None, dev(sinks)).view(2, H, Dv)
    want = torch.stack([exact(q[s].view(H, 24), keys[s], values[s], n - 1, 0.2, None, 0, None, None, None, sinks)[0] for s, n in enumerate(lens)])
    assert (got.double().cpu() - want).abs().max() <= 4e-6 * max(1.0, float(want.abs().max()))          # float32 sums of 300 terms
