"""The rule that gives a product of more than 64 rows its kernel (csrc/prompt_plan.h), compiled
for the host as the library has it and as a tuning build has it: which form the GPU tests' shapes
run, and that no shape is given a kernel whose tiles do not divide it or that lacks what its
caller asks for (given row sums, output sums, the fused q|k|v epilogue)."""

import os
import shutil
import subprocess

import pytest

from test_gpu_prompt_ring import SHAPES
from torch2iron_amd.build import CSRC

FORMS = {"32x64, 4 slices": (2, 2, 2, 4), "64x128, 2 slices": (4, 2, 4, 2), "64x128, pairs": (4, 2, 4, 1),
         "128x256": (8, 2, 8, 1)}
NONE, TILES64, RING = 0, 1, 2
MAIN = """
#include <stdio.h>
#include "prompt_plan.h"
int main() {
  for (int m, k, n; scanf("%d %d %d", &m, &k, &n) == 3;) {
    const t2i_host::PromptPlan p = t2i_host::plan_prompt(m, k, n);
    printf("%d %d %d %d %d %d %d\\n", (int)p.kind, p.cfg[0], p.cfg[1], p.cfg[2], p.cfg[3],
           t2i_host::prompt_form_serves(p, n, false), t2i_host::prompt_form_serves(p, n, true));
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    """(shapes, T2I_PROMPT or None for the library's own rule) -> [(kind, form, serves plain, serves batch)]"""
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    for name, flags in (("plan", []), ("tuning", ["-DT2I_TUNING"])):
        subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", *flags, str(d / "main.cpp"), "-o", str(d / name)], check=True)

    def run(shapes, override=None):
        env = dict(os.environ)
        env.pop("T2I_PROMPT", None)
        if override is not None:
            env["T2I_PROMPT"] = override
        out = subprocess.run([str(d / ("plan" if override is None else "tuning"))], check=True, text=True, env=env,
                             capture_output=True, input="".join(f"{m} {k} {n}\n" for m, k, n in shapes)).stdout
        rows = [tuple(int(v) for v in line.split()) for line in out.splitlines()]
        assert len(rows) == len(shapes)
        return [(r[0], r[1:5], bool(r[5]), bool(r[6])) for r in rows]

    return run


ROWS = [1, 16, 64, 65, 79, 97, 128, 197, 256, 331, 390, 450, 500, 511, 512, 513, 633, 900, 2048, 4001, 8192]
GRID = [(m, 128 * g, n) for m in ROWS for g in (1, 2, 3, 8, 15, 16, 24, 48)
        for n in (16, 64, 96, 128, 192, 384, 1024, 2048, 3072, 4096, 6144, 12288, 32768)]


def test_gpu_test_shapes_run_the_forms_they_name(ask):
    got = ask([s[1:] for s in SHAPES])
    for (form, *shape), (kind, cfg, _, _) in zip(SHAPES, got):
        assert (kind, cfg) == (RING, FORMS[form]), shape
    assert {s[0] for s in SHAPES} == set(FORMS)


def test_every_plan_serves_its_calls(ask):
    for (m, k, n), (kind, cfg, plain, batch) in zip(GRID, ask(GRID)):
        if m <= 64 or (m >= 512 and n % 128):
            assert kind == NONE, (m, k, n)
        elif m >= 512:
            assert kind != NONE and plain and batch, (m, k, n, cfg)
        else:
            assert kind == NONE or (kind == RING and plain), (m, k, n, cfg)
        assert kind != RING or n % (16 * cfg[1] * cfg[2]) == 0


@pytest.mark.parametrize("override", ["2,2,2,4", "8,2,8,1", "4,2,4,1", "tiles", "0,0,0,0", "4,-2,4,1", "4,2,0,1"])
def test_tuning_override_keeps_the_bounds(ask, override):
    for (m, k, n), (kind, cfg, plain, batch) in zip(GRID, ask(GRID, override)):
        if m <= 64 or (m >= 512 and n % 128):
            assert kind == NONE, (m, k, n)
            continue
        assert plain or kind == NONE, (m, k, n, cfg)
        if kind == RING:
            assert ",".join(map(str, cfg)) == override and n % (16 * cfg[1] * cfg[2]) == 0
            assert batch == (16 * cfg[1] * cfg[2] % 128 == 0)     # else the launcher refuses a batch's call
        else:
            assert kind == (TILES64 if m >= 512 else NONE)
