"""How the bf16 GEMMs cut a product (csrc/gemm_plan.hpp), compiled for the CPU."""
import os
import random
import subprocess

import pytest

from tests import test_gpu_gemm

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxinfer_amd", "csrc")
FMT = {"Q8_0": 1, "Q4_K": 2, "Q6_K": 3, "FP8": 4, "MLX": 6, "Q8": 7, "Q4_0": 8, "Q5_K": 9, "MXFP4": 10, "NVFP4": 11}

# reads lines of format, rows, columns, tokens; prints row tiles (0: gemm.hip's kernel) and slices of either kernel
PROGRAM = r"""
#include "gemm_plan.hpp"
#include <cstdio>
int main() {
    int f;
    unsigned n_out, n_in, t;
    while (std::scanf("%d %u %u %u", &f, &n_out, &n_in, &t) == 4) {
        const oxhip::ShortPlan p = oxhip::short_plan(f, n_out, n_in, t);
        std::printf("%u %u %u %d\n", p.rt, p.slices, oxhip::gemm_plan(f, n_out, n_in, (t + 15) / 16).slices, p.rt ? oxhip::short_form(f, t <= 32 ? 2 : (t + 15) / 16, p.rt) : 1);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("gemm_plan")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)

    def plans(calls):
        """[(format, rows, columns, tokens)] -> [(row tiles, slices, slices of gemm.hip's kernel, whether the form is built)]"""
        text = "\n".join("%d %d %d %d" % (FMT[f], n_out, n_in, t) for f, n_out, n_in, t in calls)
        r = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True)
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return plans


def test_rounds_that_are_nearly_empty_are_not_taken(plans):
    """Sizes where gemm_short.hip's fewest row tiles need a round more than they fill (257 to 400 workgroups on 256 CUs, one to a CU), or
    where its waves have more steps than gemm.hip's K slices leave: from HBM 1.12 to 2.2 times gemm.hip's time there."""
    slow = [("MLX", 18944, 4096, 64), ("Q4_K", 25600, 5120, 64), ("Q8_0", 17408, 5120, 64), ("Q6_K", 18944, 4096, 64), ("FP8", 18944, 4096, 64), ("Q8_0", 7168, 14336, 64),
            ("Q5_K", 7168, 14336, 64), ("FP8", 7168, 14336, 64), ("Q6_K", 7168, 18432, 64), ("Q8", 14336, 4096, 64), ("Q8", 7168, 18432, 64), ("Q8", 5120, 12288, 64),
            ("MLX", 128256, 2048, 64), ("Q8_0", 151936, 2560, 24), ("NVFP4", 250000, 256, 24)]
    for call, (rt, slices, four, _) in zip(slow, plans(slow)):
        assert rt == 0, (call, rt, slices)
    for call in (("MLX", 17408, 4096, 24), ("Q4_K", 18944, 4096, 24)):  # (three row tiles: two workgroups share a CU)
        assert plans([call])[0][:2] == (3, 1), call


def test_every_plan_can_run(plans):
    rng = random.Random(5)
    calls = [(rng.choice(list(FMT)), rng.choice([1, 16, 17, int(2 ** (18 * rng.random()))]), 256 * rng.randint(1, rng.choice([8, 80, 500])), rng.randint(1, 64)) for _ in range(20000)]
    for call, (rt, slices, four, built) in zip(calls, plans(calls)):
        steps = (call[2] + 127) // 128
        assert 0 <= rt <= 4 and built, call
        assert 1 <= slices <= 4 and (slices == 1 or steps >= 16 * slices), call
        assert 1 <= four <= 16 and (four - 1) * -(-steps // four) < steps, call


def test_the_gpu_tests_sizes_reach_every_form(plans):
    """tests/test_gpu_gemm.py's sizes for up to 64 tokens: in every format each number of row tiles at two, three and four token tiles, one, three
    and four slices, and gemm.hip's kernel whole; with slices in the formats that take it so."""
    for fmt in FMT:
        calls = [(fmt, n_out, n_in, t) for n_out, n_in in test_gpu_gemm.SHORT_SIZES for t in test_gpu_gemm.SHORT_TOKENS if not (fmt == "FP8" and t <= 32)]
        got = plans(calls)
        forms = {(max(2, (c[3] + 15) // 16), p[0]) for c, p in zip(calls, got)}
        want = {(ntt, rt) for ntt in (2, 3, 4) for rt in (1, 2, 3, 4)}
        want -= {(4, 4)} if fmt == "Q8" else {(2, rt) for rt in (1, 2, 3, 4)} if fmt == "FP8" else set()
        assert forms >= want, (fmt, want - forms)
        assert {1, 3, 4} <= {p[1] for p in got if p[0]} or fmt in ("Q8", "Q8_0", "FP8"), (fmt, got)
        four = {p[2] > 1 for p in got if p[0] == 0}
        assert False in four and (True in four or fmt in ("MXFP4", "NVFP4")), (fmt, four)
