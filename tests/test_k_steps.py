"""Which k-steps of a weight, or pairs of them, the wavefronts of a few-rows product read, and which they ask for ahead of attention's
shares (csrc/k_steps.h, gemm_few.h), on the host."""
import os
import shutil
import subprocess

import pytest

from servelab_amd.kernels import build

PROGRAM = """
#include <cstdio>
#include <initializer_list>
#include "k_steps.h"
int main() {
  for (int waves : {8, 16})
    for (int steps = 0; steps <= 600; ++steps)           // (none: the pairs of a single k-step)
      for (int wave = 0; wave < waves; ++wave) {
        const int first = first_k_step(steps, wave, waves), behind = first_k_step(steps, wave + 1, waves);
        std::printf("%d %d %d %d %d", waves, steps, wave, first, behind);
        ask_ahead<4>(first, behind, [](int u, int k) { std::printf(" %d %d", u, k); });
        std::puts("");
      }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_wavefronts_ask_for_their_own_k_steps(tmp_path):
    source, program = tmp_path / "steps.cpp", tmp_path / "steps"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", build.CSRC, "-o", str(program), str(source)], check=True)
    covered = {}
    for line in subprocess.run([str(program)], capture_output=True, text=True, check=True).stdout.splitlines():
        waves, steps, wave, first, behind, *ahead = map(int, line.split())
        assert covered.get((waves, steps), 0) == first                 # one wavefront begins where the one before it ends
        covered[waves, steps] = behind
        # four of its own k-steps, or none
        assert list(zip(ahead[::2], ahead[1::2])) == [(u, min(first + u, behind - 1)) for u in range(4 if first < behind else 0)]
    assert len(covered) == 1202 and all(behind == steps for (_, steps), behind in covered.items())

