"""The counters of the dataflow factorisation, compiled for the host: one that
several work-groups write must not go back when their stores arrive in another
order than the work-groups' own (the task of block column j + 1 may publish
before that of column j; a waiter for the larger value would never end)."""
from __future__ import annotations

import itertools
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "exageostat_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = """
#include "flow.hpp"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  int f = 0;
  for (int i = 1; i < argc; ++i) exa::PUBLISH(&f, std::atoi(argv[i]));
  std::printf("%d", f);
}
"""


@pytest.mark.skipif(not shutil.which(HIPCC), reason="needs hipcc")
def test_diagonal_counter_keeps_the_largest(tmp_path):
    """The function with which chol_flow.hip publishes the diagonal's counter,
    called with its values in every order."""
    with open(os.path.join(CSRC, "chol_flow.hip")) as f:
        used = re.findall(r"(\w+)\(a\.flags \+ kDiag, j", f.read())
    assert len(used) == 1
    src = tmp_path / "counter.hip"
    src.write_text(PROGRAM.replace("PUBLISH", used[0]))
    exe = str(tmp_path / "counter")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", CSRC, str(src), "-o", exe], check=True, capture_output=True)
    for order in itertools.permutations([1, 2, 3]):
        out = subprocess.run([exe] + [str(v) for v in order], check=True, capture_output=True, text=True).stdout
        assert int(out) == 3, order
