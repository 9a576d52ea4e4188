"""The matrix-core window attention at wide heads whose values have pages of their own: every width it takes compiles into a workgroup that
fits a CU (a static assertion of the source), and its kernels keep what a block needs in registers; shares of steps."""
import os
import re
import subprocess
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps, build


def spilled(source, *defines):
    """Vector registers that each kernel of the library spills."""
    flags = [f for f in build.BASE_FLAGS if f not in ("-shared", "-fPIC")]
    out = subprocess.run([build.hipcc()] + flags + ["-D" + d for d in defines] + ["--cuda-device-only", "-S", "-o", os.devnull,
                          "-Rpass-analysis=kernel-resource-usage", os.path.join(build.CSRC, source)],
                         check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True).stdout
    names = re.findall(r"Function Name: (\S+)", out)
    counts = [int(n) for n in re.findall(r"VGPRs Spill: (\d+)", out)]
    assert len(names) == len(counts) > 0
    return dict(zip(names, counts))


# either side of the lines between two teams and one, and between places kept and worked out anew; the widest of each sort.  (Up to 25 spilled
# registers the narrow forms are still the faster ones, from 35 on they are not.)
@pytest.mark.skipif(not os.path.exists(build.hipcc()), reason="no hipcc")
@pytest.mark.parametrize("Dk,Dv", [(512, 256), (192, 512), (704, 256), (1024, 96), (896, 16), (256, 512), (512, 384), (1024, 112), (512, 512),
                                   (544, 512), (640, 512), (1024, 512)])
def test_registers(Dk, Dv):
    found = spilled("window_attention_mfma.hip", f"SL_DK={Dk}", f"SL_DV={Dv}", "SL_VK=0")
    assert max(found.values()) <= 25, found


class Recorded(HipOps):
    """The table's host side without a device: what it would launch is written down."""

    def __init__(self):
        self.act_dtype, self.device, self._num_cus, self.use_mfma_attention = torch.bfloat16, torch.device("cpu"), 256, True
        self._fn, self._lib, self.shares = {"sl_window_attention_mfma@64.64.0": None}, {}, []

    def _window_step_blocks(self, *a):
        return 4

    def _window_mfma_lib(self, *a):
        return "window_attention_mfma"

    def _check(self, *a, **k):
        pass

    def _call(self, stem, name, *a):
        self.shares.append(a[-3])


@pytest.mark.parametrize("S,shares", [(0, 32), (1, 32), (8, 16), (200, 1)])
def test_shares_of_a_step(S, shares):
    """A workgroup for every CU at most; a step without sequences is a call like any other."""
    ops = Recorded()
    batch = SimpleNamespace(cu_q=None, positions=None, num_seqs=S, num_tokens=S, max_q_len=1, max_ctx_len=4096)
    pages = torch.zeros(1, 2, 16, 64, dtype=torch.bfloat16)
    out = ops.window_attention(torch.zeros(S, 256, dtype=torch.bfloat16), 0, 4, 2, 64, 64, pages, pages, 16,
                               torch.zeros(S, 256, dtype=torch.int32), batch, 1.0, None)
    assert out.shape == (S, 256) and ops.shares == [shares]
