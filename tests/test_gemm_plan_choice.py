"""CPU-only: which tiles the size rule of csrc/gemm_plan.h picks where a wrong pick was measured, asked of the header itself."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

ALONG = [(2183, 64, 2624), (700, 192, 2624), (312, 64, 1280)]
ACROSS = [(192, 768, 3072), (256, 768, 3072), (982, 256, 3456)]

PROGRAM = r"""
#include "gemm_plan.h"
#include <stdio.h>
#include <stdlib.h>
int main(int argc, char** argv) {
    for (int i = 2; i + 2 < argc; i += 3) {
        const GemmPlan p = gemm_plan(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), 2, (size_t)-1, 256, ALIGNED, ANY_KERNEL, 0, false,
                                     atoi(argv[1]) != 0);
        printf("%d %d\n", p.cfg, p.splits);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which(HIPCC) is None:
        pytest.skip("no hipcc")
    path = tmp_path_factory.mktemp("plan")
    (path / "plan.hip").write_text(PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "pre-tjax_amd", "csrc"),
                    str(path / "plan.hip"), "-o", str(path / "plan")], check=True, capture_output=True)

    def ask(*sizes, along):
        out = subprocess.run([str(path / "plan"), str(int(along))] + [str(x) for s in sizes for x in s], check=True, capture_output=True, text=True).stdout
        return [tuple(int(x) for x in line.split()) for line in out.splitlines()]
    return ask


def test_small_tiles_of_a_long_contraction(plans):
    """Operands along the contraction: whole 32x32 tiles are 10 to 20 % faster than 64x64 tiles in parts (us in the header); across it the
    parts are, by 10 %."""
    for size, (cfg, splits) in zip(ALONG, plans(*ALONG, along=True)):
        assert cfg == 0 and splits <= 2, (size, cfg, splits)
    for size, (cfg, splits) in zip(ACROSS, plans(*ACROSS, along=False)):
        assert cfg == 9 and splits > 2, (size, cfg, splits)


def test_tiles_of_one_round(plans):
    """32x64, 64x64 with eight wavefronts and 64x128 with two K groups where they were the best."""
    for along in (False, True):
        assert plans((512, 768, 768), (1024, 768, 768), (1536, 768, 2304), along=along) == [(8, 1), (9, 1), (10, 1)]
