"""The rule that gives a product of more than 64 rows its kernel (csrc/prompt_plan.h), compiled
for the host as the library has it and as a tuning build has it: which form the GPU tests' shapes
run, and that no shape is given a kernel whose tiles do not divide it or that lacks what its
caller asks for (given row sums, output sums, the fused q|k|v epilogue)."""

import os
import shutil
import subprocess

import pytest

from test_gpu_prompt_ring import SHAPES, SUMS_SHAPES
from torch2iron_amd.build import CSRC

NONE, TILES64, RING = 0, 1, 2
FORMS = {"decode tiles": (NONE, (0, 0, 0, 0)), "64x128 kernel": (TILES64, (0, 0, 0, 0)),
         "64x128, 2 slices": (RING, (4, 2, 4, 2)), "64x128, pairs": (RING, (4, 2, 4, 1)), "128x256": (RING, (8, 2, 8, 1))}
MAIN = """
#include <stdio.h>
#include "prompt_plan.h"
int main() {
  for (int m, k, n, sums; scanf("%d %d %d %d", &m, &k, &n, &sums) == 4;) {
    const t2i_host::PromptPlan p = t2i_host::plan_prompt(m, k, n, sums);
    printf("%d %d %d %d %d %d\\n", (int)p.kind, p.cfg[0], p.cfg[1], p.cfg[2], p.cfg[3],
           t2i_host::prompt_form_serves(p, n, sums));
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    """(shapes, given sums, T2I_PROMPT or None for the library's own rule) -> [(kind, form, serves)]"""
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    for name, flags in (("plan", []), ("tuning", ["-DT2I_TUNING"])):
        subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", *flags, str(d / "main.cpp"), "-o", str(d / name)], check=True)

    def run(shapes, sums=False, override=None):
        env = dict(os.environ)
        env.pop("T2I_PROMPT", None)
        if override is not None:
            env["T2I_PROMPT"] = override
        out = subprocess.run([str(d / ("plan" if override is None else "tuning"))], check=True, text=True, env=env,
                             capture_output=True, input="".join(f"{m} {k} {n} {int(sums)}\n" for m, k, n in shapes)).stdout
        rows = [tuple(int(v) for v in line.split()) for line in out.splitlines()]
        assert len(rows) == len(shapes)
        return [(r[0], r[1:5], bool(r[5])) for r in rows]

    return run


ROWS = [1, 16, 64, 65, 79, 97, 128, 197, 256, 331, 390, 450, 500, 511, 512, 513, 633, 900, 2048, 4001, 8192]
GRID = [(m, 128 * g, n) for m in ROWS for g in (1, 2, 3, 8, 15, 16, 24, 48)
        for n in (16, 64, 96, 128, 192, 384, 1024, 2048, 3072, 4096, 6144, 12288, 32768)]


def test_gpu_test_shapes_run_the_forms_they_name(ask):
    for shapes, sums in ((SHAPES, False), (SUMS_SHAPES, True)):
        for (form, *shape), (kind, cfg, _) in zip(shapes, ask([s[1:] for s in shapes], sums)):
            assert (kind, cfg) == FORMS[form], (shape, sums)
    assert {s[0] for s in SHAPES} == set(FORMS)


@pytest.mark.parametrize("sums", [False, True])
def test_every_plan_serves_its_calls(ask, sums):
    for (m, k, n), (kind, cfg, serves) in zip(GRID, ask(GRID, sums)):
        if m <= 64 or n % 128:
            assert kind == NONE, (m, k, n)
        else:
            assert serves or (kind == NONE and m < 512), (m, k, n, cfg)
        assert kind != TILES64 or m >= 512
        assert kind != RING or n % (16 * cfg[1] * cfg[2]) == 0


@pytest.mark.parametrize("sums", [False, True])
@pytest.mark.parametrize("override", ["8,2,8,1", "4,2,4,1", "2,2,2,4", "tiles", "0,0,0,0", "4,-2,4,1", "4,2,0,1"])
def test_tuning_override_keeps_the_bounds(ask, override, sums):
    for (m, k, n), (kind, cfg, serves) in zip(GRID, ask(GRID, sums, override)):
        if m <= 64 or n % 128:
            assert kind == NONE, (m, k, n)
        elif kind == RING:
            assert serves and ",".join(map(str, cfg)) == override and n % (16 * cfg[1] * cfg[2]) == 0
        else:
            assert kind == (TILES64 if m >= 512 else NONE)


# rows, K, N, given sums: the form that was measured slower than the kernel before the ring kernel's,
# us with that kernel and with the form (as the rule before this one chose); then products where the
# form is the faster one
SLOWER = {(8192, 1024, 4096, True): ("128x256", 99.4, 107.1), (1536, 2048, 2048, True): ("64x128, pairs", 24.7, 27.5),
          (6000, 6144, 2048, True): ("64x128, pairs", 190.7, 208.6), (1300, 2048, 12288, True): ("64x128, pairs", 94.2, 103.8),
          (768, 2048, 4096, True): ("64x128, pairs", 25.1, 27.4), (3000, 3072, 1024, True): ("64x128, pairs", 34.6, 37.4)}
FASTER = {(8192, 2048, 12288, False): ("128x256", 584, 438), (4001, 6144, 2048, False): ("128x256", 145.6, 103.5),
          (8192, 1024, 4096, False): ("128x256", 107.0, 104.2), (331, 2048, 12288, False): ("128x256", 52.2, 32.9),
          (8192, 2048, 1024, True): ("128x256", 48.5, 42.5), (8192, 6144, 2048, True): ("128x256", 245, 199)}


def test_measured_products(ask):
    for (m, k, n, sums), (form, _, _) in SLOWER.items():
        assert ask([(m, k, n)], sums)[0][:2] != FORMS[form], (m, k, n)
    for (m, k, n, sums), (form, _, _) in FASTER.items():
        assert ask([(m, k, n)], sums)[0][:2] == FORMS[form], (m, k, n)
