"""The matrix-core window attention where its blocks of 32 keys hold keys that no query of the step sees: before a
window, between the kept first tokens and the window, behind the last token.  Their slots hold NaN here, and pages without
a seen key are not in the block table; several sequences and kv heads of different lengths share the launch."""
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps
from test_window_kernels_gpu import dev, fill_pages, paged, plain_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,Dk,Dv,in_keys", [(4, 2, 32, 16, False), (3, 1, 64, 48, True), (4, 4, 128, 128, False),
                                              (5, 1, 576, 512, True)])
@pytest.mark.parametrize("window,keep", [(None, 0), (9, 3), (40, 0), (33, 50), (1, 1)])
@pytest.mark.parametrize("page", [16, 32])
def test_blocks_with_unseen_keys(H, G, Dk, Dv, in_keys, window, keep, page):
    ops = HipOps(torch.bfloat16, "cuda:0")
    g = torch.Generator().manual_seed(Dk + keep)
    seqs = [(0, 71), (150, 20), (0, 33), (97, 2)]              # (cached tokens, tokens of this step)
    lens = [a + b for a, b in seqs]
    tables, kc, vc = paged(lens, page, G, Dk, 0 if in_keys else Dv, torch.bfloat16, g)
    keys = [torch.randn(n, G, Dk, generator=g).bfloat16() for n in lens]
    values = [k[..., :Dv] for k in keys] if in_keys else [torch.randn(n, G, Dv, generator=g).bfloat16() for n in lens]
    fill_pages(tables, kc, vc, keys, None if in_keys else values, page)
    T = sum(b for _, b in seqs)
    q = torch.randn(T, H * Dk, generator=g).bfloat16()
    cu, pos, want = [0], [], []
    for s, (a, b) in enumerate(seqs):
        want.append(plain_attention(q[cu[-1]:cu[-1] + b].view(b, H, Dk), keys[s], values[s], list(range(a, a + b)),
                                    Dk ** -0.5, window, keep, None, None, None))
        pos += list(range(a, a + b))
        cu.append(cu[-1] + b)
        unseen = [j for j in range(lens[s]) if window and j >= keep and j <= a - window]
        for j in unseen:
            kc[int(tables[s, j // page]), :, j % page] = float("nan")
            vc[int(tables[s, j // page]), :, :, j % page] = float("nan")
        for p in range(-(-lens[s] // page)):
            if all(j in unseen for j in range(p * page, min((p + 1) * page, lens[s]))):
                tables[s, p] = 0
    batch = SimpleNamespace(cu_q=dev(torch.tensor(cu, dtype=torch.int32)), positions=dev(torch.tensor(pos, dtype=torch.int32)),
                            num_seqs=len(seqs), num_tokens=T, max_q_len=max(b for _, b in seqs), max_ctx_len=max(lens))
    out = ops.window_attention(dev(q), 0, H, G, Dk, Dv, dev(kc), None if in_keys else dev(vc), page, dev(tables), batch,
                               Dk ** -0.5, window, keep, None, None, None, 0)
    assert ("window_attention_mfma", Dk, Dv, in_keys) in ops._lib
    want = torch.cat(want)
    # results of size up to a few units rounded to bfloat16 (2^-9 of the value); scores, weights and sums are float32
    assert (out.view(T, H, Dv).double().cpu() - want).abs().max() <= 2.0 ** -8 * want.abs().max() + 1e-4


# the order in which a launch takes its tiles: sequences of one length, nearly equal ones over fewer and more than eight
# (sequence, kv head) pairs, unequal ones; several tiles of 64 columns a sequence, the last one partly filled
@pytest.mark.parametrize("lens", [(70, 70, 70), (75, 60, 71), (90, 3, 1), (1, 1, 1)])
@pytest.mark.parametrize("H,G", [(4, 1), (4, 4)])
def test_orders_of_the_tiles(H, G, lens):
    ops = HipOps(torch.bfloat16, "cuda:0")
    g = torch.Generator().manual_seed(H + G)
    D, page = 64, 16
    cached = [5, 0, 40]
    whole = [a + b for a, b in zip(cached, lens)]
    tables, kc, vc = paged(whole, page, G, D, D, torch.bfloat16, g)
    keys, values = ([torch.randn(n, G, D, generator=g).bfloat16() for n in whole] for _ in range(2))
    fill_pages(tables, kc, vc, keys, values, page)
    q = torch.randn(sum(lens), H * D, generator=g).bfloat16()
    cu, pos, want = [0], [], []
    for s, (a, b) in enumerate(zip(cached, lens)):
        rows = list(range(a, a + b))
        want.append(plain_attention(q[cu[-1]:cu[-1] + b].view(b, H, D), keys[s], values[s], rows, D ** -0.5, None, 0, None, None, None))
        pos += rows
        cu.append(cu[-1] + b)
    batch = SimpleNamespace(cu_q=dev(torch.tensor(cu, dtype=torch.int32)), positions=dev(torch.tensor(pos, dtype=torch.int32)),
                            num_seqs=len(lens), num_tokens=cu[-1], max_q_len=max(lens), max_ctx_len=max(whole))
    out = ops.window_attention(dev(q), 0, H, G, D, D, dev(kc), dev(vc), page, dev(tables), batch, D ** -0.5, None, 0, None,
                               None, None, 0)
    want = torch.cat(want)
    # (as above)
    assert (out.view(-1, H, D).double().cpu() - want).abs().max() <= 2.0 ** -8 * want.abs().max() + 1e-4
