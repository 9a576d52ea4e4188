"""Norms that hold a row in registers: the widest rows a thread takes fit the registers of its wavefront; the walk over a recurrence's tokens
leaves room for two workgroups on a CU."""
import os

import pytest

from servelab_amd.kernels import build
from test_window_widths import spilled


@pytest.mark.skipif(not os.path.exists(build.hipcc()), reason="no hipcc")
@pytest.mark.parametrize("dtype", [(), ("SL_F32=1",)])
def test_rows_in_registers(dtype):
    found = {name: n for name, n in spilled("norm.hip", *dtype).items() if "vec_kernel" in name or "streams_norm" in name}
    # (two, for two workgroups a CU: 65 us where without them one workgroup takes 71)
    assert len(found) > 20 and max(found.values()) <= 2, found


@pytest.mark.skipif(not os.path.exists(build.hipcc()), reason="no hipcc")
def test_two_walks_on_a_cu():
    found = {name: n for name, n in spilled("recurrent.hip", what="Occupancy [waves/SIMD]").items() if "matrix_scan_kernel" in name}
    assert len(found) == 6 and min(found.values()) >= 4, found       # (of eight wavefronts each, on four SIMDs)
