"""How the launches of an MoE prefill pass are cut into workgroups (csrc/moe_plan.hpp), compiled for the CPU."""
import os
import subprocess

import pytest

from tests import test_gpu_moe

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxinfer_amd", "csrc")
FMT = {"Q8_0": 1, "Q4_K": 2, "mlx": 6, "Q4_0": 8, "MXFP4": 10}

# reads lines of format, h, inter, experts, routed rows; prints the gate / up launch's and the down launch's plan
PROGRAM = r"""
#include "moe_plan.hpp"
#include <cstdio>
using namespace oxhip;
int main() {
    int f;
    unsigned h, inter, n_exp, pairs;
    while (std::scanf("%d %u %u %u %u", &f, &h, &inter, &n_exp, &pairs) == 5) {
        const uint32_t most = (uint32_t)moe_most_chunks(pairs, n_exp), chunks = moe_expected_chunks(pairs, n_exp);
        const MoePlan g = moe_plan(f, 2 * inter, h, inter, most, chunks), d = moe_plan(f, h, inter, 0, most, chunks);
        std::printf("%u %u %u %u %u %u %u %u\n", g.rt, g.kw, g.nrep, g.nx, d.rt, d.kw, d.nrep, d.nx);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("moe_plan")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)

    def plans(passes):
        """[(format, h, inter, experts, routed rows)] -> [((rt, kw, nrep, nx) of the gate / up launch, of the down launch)]"""
        text = "\n".join("%d %d %d %d %d" % (FMT[p[0]], *p[1:]) for p in passes)
        r = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True)
        got = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
        return [(v[:4], v[4:]) for v in got]
    return plans


@pytest.mark.parametrize("fmt", list(FMT))
def test_the_gpu_tests_sizes_reach_every_form(plans, fmt):
    """tests/test_gpu_moe.py's sizes: K over one, two and four waves, and but for Q8_0 three row tiles per wave in either launch and two,
    three and four runs of row tiles per workgroup, groups and runs that end past the matrix among them."""
    rows = test_gpu_moe.CHUNK_ROWS
    gate, down, past = set(), set(), set()
    for h, inter, copies in test_gpu_moe.CHUNK_SIZES:
        if fmt == "Q4_K":
            inter = (inter + 255) // 256 * 256
        (g, d), = plans([(fmt, h, inter, len(rows) * copies, sum(rows) * copies)])
        gate.add(g[:2])
        down.add((d[0], d[2]))
        if g[0] == 3 and g[3] * 12 > inter // 16:
            past.add("gate")
        if d[2] > 1 and d[3] * d[2] * 16 > h // 16:
            past.add("down")
    assert {(2, 1), (2, 2), (2, 4)} <= gate and (2, 1) in down
    if fmt != "Q8_0":
        assert (3, 1) in gate and {(3, 1), (2, 2), (2, 3), (2, 4)} <= down, (gate, down)
        assert past == {"gate", "down"}, past


def test_every_plan_covers_the_matrix_with_forms_that_are_built(plans):
    passes = [(f, h, inter, n_exp, n_exp * rows + 1) for f in FMT for h in (128, 1280, 2048, 4096) for inter in (128, 384, 768, 1408, 4096) for n_exp in (1, 8, 60, 128) for rows in (6, 18, 100)]
    for p, (g, d) in zip(passes, plans(passes)):
        for (rt, kw, nrep, nx), tiles, gate in ((g, p[2] // 16, True), (d, p[1] // 16, False)):
            per = (8 // kw) * rt // (2 if gate else 1)
            assert rt in ((2,) if p[0] == "Q8_0" else (2, 3)) and kw in (1, 2, 4) and 1 <= nrep <= (1 if gate or p[0] == "Q8_0" else 4), p
            assert (kw == 1 or rt == 2) and (nrep == 1 or (rt == 2 and kw == 1)), p
            assert nx * nrep * per >= tiles > (nx - 1) * nrep * per, p
