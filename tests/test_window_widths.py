"""The matrix-core window attention at wide heads whose values have pages of their own: every width it takes compiles into a workgroup that
fits a CU (a static assertion of the source), and its kernels keep what a block needs in registers; shares of steps."""
import os
import re
import subprocess
from types import SimpleNamespace

import pytest
import torch

from servelab_amd.kernels import HipOps, build


def spilled(source, *defines, what="VGPRs Spill"):
    """Vector registers that each kernel of the library spills (or another of the compiler's figures)."""
    flags = [f for f in build.BASE_FLAGS if f not in ("-shared", "-fPIC")]
    out = subprocess.run([build.hipcc()] + flags + ["-D" + d for d in defines] + ["--cuda-device-only", "-S", "-o", os.devnull,
                          "-Rpass-analysis=kernel-resource-usage", os.path.join(build.CSRC, source)],
                         check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True).stdout
    names = re.findall(r"Function Name: (\S+)", out)
    counts = [int(n) for n in re.findall(re.escape(what) + r": (\d+)", out)]
    assert len(names) == len(counts) > 0
    return dict(zip(names, counts))


# either side of the lines between two teams and one, between places kept and worked out anew, and between one form and two, of a latent between
# teams and pairs; the widest of each sort.  (Up to 25 spilled
# registers the narrow forms are still the faster ones, from 35 on they are not.)
@pytest.mark.skipif(not os.path.exists(build.hipcc()), reason="no hipcc")
@pytest.mark.parametrize("Dk,Dv,in_keys", [(512, 256, 0), (192, 512, 0), (704, 256, 0), (1024, 96, 0), (896, 16, 0), (256, 512, 0), (512, 384, 0), (1024, 112, 0),
                                           (512, 512, 0), (544, 512, 0), (640, 512, 0), (1024, 512, 0), (128, 128, 0), (320, 256, 0), (64, 512, 0), (544, 32, 0),
                                           (128, 128, 1), (288, 288, 1), (320, 256, 1), (544, 32, 1), (320, 272, 1), (576, 512, 1), (1024, 512, 1)])
def test_registers(Dk, Dv, in_keys):
    found = spilled("window_attention_mfma.hip", f"SL_DK={Dk}", f"SL_DV={Dv}", f"SL_VK={in_keys}")
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


def prompts(lens, heads, kv_heads, Dk, Dv, in_keys, cached=0):
    context = max(lens) + cached
    return Recorded()._window_few(sum(lens), len(lens), max(lens), context, context, heads, kv_heads, Dk, Dv, in_keys)


# (us measured with eight wavefronts a workgroup / with four beside each)
@pytest.mark.parametrize("lens,heads,kv_heads,Dk,Dv,in_keys,few", [
    ([1024], 16, 2, 128, 128, False, True), ([300] * 4, 16, 2, 128, 128, False, True),                    # 34 / 43, 16 / 18
    ([200] * 16, 32, 8, 128, 128, False, False), ([100] * 64, 16, 2, 128, 128, False, False),             # 37 / 30, 32 / 25
    ([50] * 64, 8, 8, 64, 64, False, False), ([1000] * 4, 8, 8, 64, 64, False, True),                     # 8.9 / 8.1, 28 / 34
    ([1024], 16, 1, 96, 64, True, True), ([500] * 16, 16, 1, 96, 64, True, False),                        # 37 / 48, 63 / 52
    ([2000] + [1] * 31, 32, 8, 64, 64, False, False), ([300] + [1] * 31, 16, 2, 128, 128, False, True),   # 122 / 101, 29 / 33
    ([2048], 16, 2, 192, 128, False, True), ([4096], 16, 2, 192, 128, False, False), ([300] * 4, 16, 2, 192, 128, False, True)])   # 78 / 93, 256 / 202, 17 / 20
def test_wavefronts_of_a_prompt_s_workgroups(lens, heads, kv_heads, Dk, Dv, in_keys, few):
    assert prompts(lens, heads, kv_heads, Dk, Dv, in_keys) is few


# (us measured in the kernel for steps / in shares of the one for prompts beside each)
@pytest.mark.parametrize("S,keys,heads,kv_heads,Dk,Dv,in_keys,step", [
    (1, 1000, 16, 1, 96, 64, True, True), (16, 300, 16, 1, 96, 64, True, True), (64, 2000, 16, 1, 96, 64, True, False),     # 7.9 / 9.3, 7.8 / 8.9, 37 / 28
    (1, 8000, 16, 1, 96, 64, True, False), (64, 300, 40, 2, 192, 128, True, False),                                         # 21 / 17, 25 / 18
    (256, 500, 16, 1, 576, 512, True, True), (1, 8000, 128, 1, 576, 512, True, True),                                       # 53 / 58, 0.8 of it
    (64, 2000, 40, 2, 576, 512, True, False), (128, 500, 40, 2, 576, 512, True, False), (64, 2000, 16, 2, 128, 128, False, True)])   # 201 / 120, 101 / 59
def test_kernel_of_a_step(S, keys, heads, kv_heads, Dk, Dv, in_keys, step):
    assert Recorded()._window_takes_step(S, keys, heads, kv_heads, Dk, Dv, in_keys) is step
