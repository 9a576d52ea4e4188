"""Kernels whose loads go straight into LDS (lds_loads.h): no read of LDS may still be under way when a wavefront comes to a
barrier, since behind it another one's loads may land where that read goes.  The compiler waits for a read where its value is
used, which it may move behind the barrier; this reads the assembly of this repository's kernels."""
import os
import re
import subprocess

import pytest

from servelab_amd.kernels import build

SOURCES = sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip")
                 and '#include "lds_loads.h"' in open(os.path.join(build.CSRC, f)).read())


def pending_at_barriers(kernel):
    """For each barrier how many reads of LDS issued before it, in the order of the text, have not been waited for."""
    pending, found = 0, []
    for line in (x.strip() for x in kernel.split("\n")):
        if line.startswith("ds_read"):
            pending += 1
        elif line.startswith("s_waitcnt"):
            left = re.search(r"lgkmcnt\((\d+)\)", line)
            pending = min(pending, int(left[1])) if left else pending
        elif line.startswith("s_barrier"):
            found.append(pending)
    return found


def test_reader_of_assembly():
    assert pending_at_barriers("ds_read_b128 v1\nds_read_b64 v2\ns_waitcnt vmcnt(0)\ns_barrier\ns_waitcnt lgkmcnt(1)\ns_barrier\n"
                               "s_waitcnt vmcnt(0) lgkmcnt(0)\ns_barrier") == [2, 1, 0]


@pytest.mark.skipif(not os.path.exists(build.hipcc()), reason="no hipcc")
@pytest.mark.parametrize("source", SOURCES)
def test_no_read_of_lds_crosses_a_barrier(source, tmp_path):
    out = tmp_path / "kernels.s"
    flags = [f for f in build.BASE_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build.hipcc()] + flags + ["--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, source)],
                   check=True, stderr=subprocess.DEVNULL)
    text, checked = out.read_text(), 0
    for start in re.finditer(r"^(_Z\w+):", text, re.M):
        kernel = text[start.end():text.find(".Lfunc_end", start.end())]
        if "global_load_lds" in kernel:
            checked += 1
            found = pending_at_barriers(kernel)
            assert found and max(found) == 0, (start[1], found)
    assert checked
