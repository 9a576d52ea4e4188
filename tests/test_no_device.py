"""Entries that ask how many CUs there are, where that cannot be asked: an error comes back, as from any launch."""
import os
import subprocess
import sys

import pytest

from servelab_amd.kernels import build

CALL = """
import ctypes, sys
lib = ctypes.CDLL(sys.argv[1])
count = ctypes.c_int(0)
if lib.hipGetDeviceCount(ctypes.byref(count)) == 0 and count.value > 0:
    sys.exit("a device is visible: nothing is called")
lib.sl_gemm_f32_mfma.restype = ctypes.c_char_p
at = [ctypes.c_void_p(4096 * i) for i in range(1, 5)]
print(lib.sl_gemm_f32_mfma(at[0], at[1], None, at[2], 849, 1536, 512, 1, at[3], None))
"""


@pytest.mark.skipif(build.find_built(build.unit("gemm", "float32")) is None, reason="kernels are not built")
def test_float32_product_without_a_device():
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")
    run = subprocess.run([sys.executable, "-c", CALL, build.find_built(build.unit("gemm", "float32"))], env=env,
                         capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.returncode, run.stderr)
    assert run.stdout.startswith("b'") and "device" in run.stdout
