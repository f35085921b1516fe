"""The rule that gives a prompt attention call its kernel (csrc/prefill_plan.h), compiled for the
host: the GPU test's cases run the kernel that they name, no call that 128-row blocks only pad
takes them, and the calls that were measured slower with them don't either."""

import os
import shutil
import subprocess

import pytest

from test_gpu_prefill_wide import CASES
from torch2iron_amd.build import CSRC

MAIN = """
#include <stdio.h>
#include "prefill_plan.h"
int main() {
  for (int b, t, p, h, q; scanf("%d %d %d %d %d", &b, &t, &p, &h, &q) == 5;)
    printf("%d\\n", (int)t2i_host::prefill_wide(b, t, p, h, q));
}
"""


@pytest.fixture(scope="module")
def wide(tmp_path_factory):
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(d / "plan")], check=True)

    def run(calls):
        out = subprocess.run([str(d / "plan")], check=True, text=True, capture_output=True,
                             input="".join("%d %d %d %d %d\n" % c for c in calls)).stdout.split()
        assert len(out) == len(calls)
        return [v == "1" for v in out]

    return run


def test_gpu_test_cases_run_the_kernel_they_name(wide):
    assert wide([c[1:] for c in CASES]) == [c[0] for c in CASES]
    assert {c[5] for c in CASES if c[0]} == {1, 2, 4, 8} == {c[5] for c in CASES if not c[0]}


def test_padding_keeps_the_small_blocks(wide):
    """As many blocks of 128 rows as of 64: the second half of each would be padding."""
    calls = [(b, t, p, h, q) for q in (1, 2, 4, 8) for t in (1, 64 // q - 1, 64 // q) if t > 0
             for b in (1, 16, 64, 512, 4096) for h in (1, 8) for p in (0, 64, 500, 6000, 30000)]
    assert not any(wide(calls))


# (B, rows, first position, kv heads, q heads a kv head): us with 64-row and with 128-row blocks
SLOWER = {(312, 1, 0, 8, 1): (12.0, 19.7), (112, 32, 200, 8, 1): (22.8, 30.0), (56, 129, 0, 8, 1): (18.6, 22.5),
          (38, 320, 0, 8, 1): (27.8, 33.4), (31, 65, 200, 8, 2): (18.5, 20.3), (62, 16, 2000, 8, 2): (94.6, 116.9),
          (156, 33, 0, 8, 4): (30.4, 35.1), (312, 17, 0, 4, 8): (28.4, 34.4), (1, 2000, 0, 8, 2): (49.3, 58.5),
          (64, 20, 500, 8, 2): (25.6, 31.3)}
FASTER = {(1, 1999, 6001, 8, 4): (386, 278), (16, 250, 500, 8, 2): (45.4, 35.5), (16, 512, 0, 8, 2): (42.0, 39.7),
          (31, 64, 2000, 4, 8): (156, 97.4), (156, 64, 2000, 4, 8): (984, 609)}


def test_measured_calls(wide):
    assert not any(wide(list(SLOWER))) and all(wide(list(FASTER)))
