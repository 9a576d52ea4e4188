"""The matrix recurrences at the sizes of real heads, against the plain torch functions (tests/emulated_ops.py)."""
import types

import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def sequences(q_lens, starts, slots, device):
    cu, pos, seq = [0], [], []
    for i, (n, s) in enumerate(zip(q_lens, starts)):
        cu.append(cu[-1] + n)
        pos += list(range(s, s + n))
        seq += [i] * n
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=device)
    return types.SimpleNamespace(cu_q=i32(cu), positions=i32(pos), tok_seq=i32(seq), state_slots=i32(slots),
                                 num_seqs=len(q_lens), num_tokens=cu[-1], max_q_len=max(q_lens))


def close(a, b, tol):
    a, b = a.float().cpu(), b.float().cpu()
    assert torch.isfinite(a).all()
    assert (a - b).abs().max() <= tol * max(1.0, float(b.abs().max())), float((a - b).abs().max())


def test_normalisers_of_a_full_decode_batch():
    """A launch of many more blocks than the chip holds at once: every block needs the normaliser and the running maximum as
    they were before the step, also those that start when others have ended."""
    S, H, D, Dv = 64, 8, 128, 256
    hip, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    g = torch.Generator().manual_seed(3)
    buf = torch.randn(S, 2 * H * D + H * Dv + 2 * H, generator=g)
    state = torch.randn(S, H * D * Dv + H * D + H, generator=g) * 0.3
    args = ([1] * S, [5] * S, list(range(S)))
    cols = (0, H * D, 2 * H * D, 2 * H * D + H * Dv, 2 * H * D + H * Dv + H)
    s1, s2 = state.clone().to(DEV), state.clone()
    o1 = hip.mlstm_scan(buf.to(DEV), *cols, H, D, Dv, 4.0, D ** -0.5, s1, sequences(*args, DEV), True)
    batch = sequences(*args, "cpu")
    batch.q_lens, batch.starts = args[0], args[1]
    o2 = emu.mlstm_scan(buf, *cols, H, D, Dv, 4.0, D ** -0.5, s2, batch, True)
    # 128 products of a head's read-out, over a divisor that is at least 1e-6 and mostly near one
    close(o1, o2, 2e-5)
    close(s1, s2, 2e-5)
