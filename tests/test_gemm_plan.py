"""The split GEMM's plan and slice workspace (picolm_qwen_amd/csrc/pqa_gemm_plan.h), built
on the CPU with g++: the workspace holds what the plan's K slices take, and that of a long
prompt holds those of every shorter one, in both modes of the K/V projection."""
import os
import subprocess

import pytest

pytest.importorskip("numpy")
from proj_cases import GEMM_CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "pqa_gemm_plan.h"

int main(int argc, char** argv) {
    if (argc == 4) {  // the plan of one product on 256 CUs
        const pqa::GemmPlan p = pqa::gemm_f16x3_plan(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]), 256);
        std::printf("%d %d %d\n", p.mi, p.nj, p.slices);
        return 0;
    }
    // columns of q, columns of k and v together, K
    const int shapes[][3] = {{4096, 2048, 2560}, {2560, 0, 4096}, {2048, 512, 2048}, {896, 256, 896},
                             {896, 0, 896},      {4096, 4096, 4096}, {8192, 2048, 8192}, {512, 128, 8192},
                             {4, 4, 32},         {128, 128, 64}};
    const int cus[] = {256, 64, 8};
    for (const auto& s : shapes)
        for (int cu : cus) {
            size_t before = 0;
            for (int m = 1; m <= 3000; m++) {
                const size_t room = pqa::gemm_slice_floats(m, s[0] + s[1], cu);
                if (room < before) {
                    std::printf("%d rows of %d columns on %d CUs: less workspace than a row fewer\n", m, s[0] + s[1], cu);
                    return 1;
                }
                before = room;
                for (int n : {s[0], s[0] + s[1]}) {
                    const pqa::GemmPlan p = pqa::gemm_f16x3_plan(m, n, s[2], cu);
                    if (p.slices < 1 || p.slices > s[2] / pqa::kGemmBK ||
                        (p.slices > 1 && (size_t)p.slices * m * n > room)) {
                        std::printf("%d x %d x %d on %d CUs: %d slices\n", m, n, s[2], cu, p.slices);
                        return 1;
                    }
                }
            }
        }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "plan_check.cpp", d / "plan_check"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "picolm_qwen_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True, capture_output=True, text=True)
    return str(exe)


def test_slices_fit_a_workspace_that_grows_with_the_prompt(program):
    out = subprocess.run([program], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


def test_gemm_cases_reach_every_tile(program):
    # the shapes that the GPU test of the split GEMM runs take the plans it says, and every tile is among them with
    # and without slices
    def up32(n):
        return (n + 31) // 32 * 32

    seen = set()
    for n_tok, dim, nh, out_rows, *plans in GEMM_CASES:
        shapes = ((nh * 64, up32(dim)), (nh * 64 + 128, up32(dim)), (out_rows, nh * 64))
        for (n, k), plan in zip(shapes, plans):
            got = subprocess.run([program, str(n_tok), str(n), str(k)], capture_output=True, text=True, check=True).stdout
            assert tuple(map(int, got.split())) == plan, (n_tok, n, k)
            seen.add((plan[:2], plan[2] > 1))
    assert seen == {(t, s) for t in ((4, 3), (4, 2), (2, 2), (2, 1), (1, 1)) for s in (False, True)}
