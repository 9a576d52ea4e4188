"""The recurrences of a step of one token a sequence, against the plain functions and against the kernel that walks tokens."""
import pytest
import torch

import test_matrix_scan_gpu as scans
from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps
from test_matrix_scan_gpu import close, scan_case, sequences

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# heads of 16, 8, 32 and 64 lanes a column, of channels that no load of four divides and that no lane's eight do; value channels that no
# workgroup divides; few blocks and many
@pytest.mark.parametrize("S,H,G,D,Dv", [(3, 2, 2, 128, 256), (2, 3, 3, 20, 24), (5, 2, 2, 72, 15), (2, 1, 1, 200, 33), (2, 2, 1, 256, 16),
                                        (1, 4, 2, 64, 40), (3, 2, 2, 50, 7), (2, 1, 1, 512, 9), (40, 8, 8, 128, 130), (70, 16, 8, 60, 64), (10, 8, 8, 128, 250)])
@pytest.mark.parametrize("mode", ["decay", "delta", "delta, decay a head", "state space", "forget", "lstm"])
def test_steps_of_one_token(mode, S, H, G, D, Dv, monkeypatch):
    if mode in ("forget", "lstm"):
        G = H
    monkeypatch.setattr(scans, "Q_LENS", [1] * S)
    call, size, _ = scan_case(mode, H, G, D, Dv, False)
    starts, slots = [0 if i % 3 == 1 else 5 + i for i in range(S)], [(7 * i + 3) % (S + 2) for i in range(S)]
    slots = slots if len(set(slots)) == S else list(range(S))
    g = torch.Generator().manual_seed(S)
    state = torch.randn(S + 2, size + 8, generator=g) * 0.3
    for i in range(S):
        if starts[i] == 0:
            state[slots[i]] = float("nan")                           # what a fresh sequence's slot holds is left out
    hip, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    dev, cpu = sequences([1] * S, starts, slots, DEV), sequences([1] * S, starts, slots, "cpu")
    cpu.q_lens, cpu.starts = [1] * S, starts
    s1, s2, s3 = state.clone().to(DEV), state.clone(), state.clone().to(DEV)
    got, want = call(hip, s1, dev, DEV), call(emu, s2, cpu, "cpu")
    dev.max_q_len = 2                                                # (a bound: the kernel that walks tokens)
    walked = call(hip, s3, dev, DEV)
    # up to 512 products a read-out (of the matrix LSTM over a divisor near one) in another order
    close(got, want, 5e-5 if mode == "lstm" else 2e-5)
    close(got, walked, 5e-5 if mode == "lstm" else 2e-5)
    used = torch.tensor(slots)
    close(s1.cpu()[used][:, :size], s3.cpu()[used][:, :size], 2e-6)  # (no sum but the delta's: the same factors)
    rest = [i for i in range(S + 2) if i not in slots]
    assert torch.equal(s1.cpu()[rest], state[rest]) and torch.equal(torch.nan_to_num(s1.cpu()[:, size:]), torch.nan_to_num(state[:, size:]))
