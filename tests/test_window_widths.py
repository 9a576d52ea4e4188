"""The matrix-core window attention at wide heads whose values have pages of their own: every width it takes compiles into a workgroup that
fits a CU (a static assertion of the source), and its kernels keep what a block needs in registers."""
import os
import re
import subprocess

import pytest

from servelab_amd.kernels import build


def spilled(Dk, Dv):
    """Vector registers that each kernel of the library spills."""
    flags = [f for f in build.BASE_FLAGS if f not in ("-shared", "-fPIC")]
    out = subprocess.run([build.hipcc()] + flags + [f"-DSL_DK={Dk}", f"-DSL_DV={Dv}", "-DSL_VK=0", "--cuda-device-only", "-S", "-o", os.devnull,
                          "-Rpass-analysis=kernel-resource-usage", os.path.join(build.CSRC, "window_attention_mfma.hip")],
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
    found = spilled(Dk, Dv)
    assert max(found.values()) <= 25, found
