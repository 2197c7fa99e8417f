"""The sizes of the amgpcg launches (amgpcg_plan.hpp, host only, compiled here):
what every workgroup adds of the launch before it stays bounded on large grids,
is no work that outgrows the grid's own, and fits the room kept for it."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "uaamg_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include "amgpcg_plan.hpp"
int main() {
    for (int n = 2; n <= 40000; n = n < 3000 ? n + 1 : n + 371) {
        const uaamg::AgPlan p = uaamg::ag_plan(n);
        std::printf("%d %d %d %d %d %d %ld %ld %ld\n", n, p.nm, p.nu, (int)p.fold, p.sum_m, p.sum_z, p.blocks_m, p.doubles, uaamg::ag_partials_room(n));
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "m"), str(d / "m.cpp")], check=True)
    out = subprocess.run([str(d / "m")], check=True, capture_output=True, text=True).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def test_finish_of_the_dot_products_is_bounded(plans):
    for n, nm, nu, fold, sum_m, sum_z, blocks_m, _, _ in plans:
        assert sum_m <= 2048 and sum_z <= 2048, n
        # the operator adds sum_z doubles per workgroup, level 0's down launch
        # sum_m: at most a few times the grid's cells, on every size
        assert blocks_m * sum_z <= 4 * n * n + 4096 and nu * sum_m <= 4 * n * n + 4096, n


def test_partials_fit(plans):
    for n, nm, nu, fold, *_, doubles, room in plans:
        assert nm + nu + (512 if fold else 0) <= doubles <= room, n


def test_folded_only_when_many(plans):
    assert {n for n, _, _, fold, *_ in plans if fold} == {n for n, *_ in plans if n > 1024}
