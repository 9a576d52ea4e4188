"""float32 prompts whose two teams of wavefronts take every other block of 32 keys: one block, two, an odd number; prompts of one team: many,
and of one block; NaN where no query sees a key, pages without a seen key not in the block table."""
import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps
from test_float32_forms_gpu import emu_batch
from test_kernels_gpu import make_attention_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("nh,nkv,D", [(6, 1, 128), (14, 2, 64)])
@pytest.mark.parametrize("page,window", [(16, None), (16, 21), (32, 50)])
@pytest.mark.parametrize("seqs", [[(32, 32), (64, 33), (97, 64), (31, 9), (200, 6)], [(70, 70 - i % 3) for i in range(48)], [(32, 32), (20, 9), (31, 31)],
                                  [(32, 32)] + [(5, 5)] * 9], ids=["unequal", "many", "one block", "one block, unequal"])
def test_blocks_of_teams(nh, nkv, D, page, window, seqs):
    """``seqs``: (context after the step, tokens of it)."""
    ops, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    qkv, kc, vc, tables, batch = make_attention_case(torch.float32, nh, nkv, D, page, seqs)[:5]
    want = emu.paged_attention(qkv.cpu(), nh, nkv, D, kc.cpu(), vc.cpu(), page, tables.cpu(), emu_batch(batch), D ** -0.5, window)
    for s, (ctx, n) in enumerate(seqs):
        for p in range(-(-ctx // page)):
            unseen = [j for j in range(p * page, (p + 1) * page) if j >= ctx or (window and j <= ctx - n - window)]
            pg = int(tables[s, p])
            for j in unseen:
                kc[pg, :, j % page] = float("nan")
                vc[pg, :, :, j % page] = float("nan")
            if len(unseen) == page:
                tables[s, p] = 0
    got = ops.paged_attention(qkv, nh, nkv, D, kc, vc, page, tables, batch, D ** -0.5, window)
    # float32 scores of 128 products and sums over at most 200 keys on both sides
    assert float((got.cpu() - want).abs().max()) <= 2e-6 * max(1.0, float(want.abs().max()))
