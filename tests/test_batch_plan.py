"""Which systems of a batch teams take (batch_plan.hpp), on the host: teams where
a few systems would hold up the launch, none where the systems fill the chip by
themselves, and the other workgroups left to the other systems."""
import os
import subprocess

import numpy as np
import pytest

from unap_amd import meshgen

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LEVELS = 18  # of a box with random numbering

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include "batch_plan.hpp"
using namespace unap_hip;
// cus, forced size, count, then rows a level and cost of each system, largest first
int main() {
    int cus, forced, n;
    if (std::scanf("%d %d %d", &cus, &forced, &n) != 3) return 1;
    std::vector<TeamSystem> s(n);
    for (auto& v : s)
        if (std::scanf("%d %lf", &v.rows, &v.cost) != 2) return 1;
    std::vector<int> order(n);
    std::iota(order.begin(), order.end(), 0);
    const TeamPlan p = planTeams(s, order, cus, forced);
    std::printf("%d %d %d", p.size, p.wide, p.teams);
    for (int i : p.order) std::printf(" %d", i);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "unap_amd", "csrc"), "-o", str(d / "plan"),
                    str(d / "plan.cpp")], check=True)

    def call(cells, cus=256, forced=0, levels=LEVELS):
        cells = sorted(cells, reverse=True)
        text = f"{cus} {forced} {len(cells)}\n" + "\n".join(f"{n // levels} {float(7.0 * n * n ** (1 / 3))!r}" for n in cells)
        out = subprocess.run([str(d / "plan")], input=text, check=True, capture_output=True, text=True).stdout.split()
        size, wide, teams = map(int, out[:3])
        order = list(map(int, out[3:]))
        assert sorted(order) == list(range(len(cells)))
        assert order[:wide] == sorted(order[:wide]) and order[wide:] == sorted(order[wide:])  # largest first
        assert (size == 1 and wide == teams == 0) if wide == 0 else (1 <= teams <= wide and teams * size <= max(cus, size))
        return size, wide, teams

    return call


def _boxes(count, lo, hi):
    return [x * y * z for x, y, z, _, _ in meshgen.batch_specs(count, lo, hi)]


def test_systems_that_fill_the_chip_are_solved_alone(plan):
    for cells in (_boxes(600, 28, 32), _boxes(2000, 8, 48), _boxes(3000, 8, 32), _boxes(64, 8, 24), [4096] * 5000):
        assert plan(cells) == (1, 0, 0)


def test_a_few_large_systems_leave_the_others_their_workgroups(plan):
    assert plan([48 ** 3] + _boxes(1000, 8, 12)) == (8, 1, 1)
    assert plan([40 ** 3] * 4 + _boxes(800, 8, 16)) == (8, 4, 4)
    size, wide, teams = plan(_boxes(512, 8, 48))
    assert size > 1 and size * teams < 256  # the others start at once


def test_large_systems_hold_most_workgroups(plan):
    size, wide, teams = plan(_boxes(96, 8, 48))
    assert size == 8 and teams == 32


def test_deep_schedules_are_solved_alone(plan):
    assert plan([48 ** 3] * 3, levels=400) == (1, 0, 0)


@pytest.mark.parametrize("cus", [1, 3, 4, 8, 32, 256])
def test_any_chip(plan, cus):
    rng = np.random.default_rng(cus)
    for _ in range(10):
        cells = np.exp(rng.uniform(np.log(1), np.log(2e5), int(rng.integers(1, 400)))).astype(int)
        for forced in (0, 1, 2, 3, 8):
            size, wide, _ = plan(cells, cus, forced)
            assert size == 1 or not forced or size == forced


def test_one_system(plan):
    assert plan([1]) == plan([512]) == (1, 0, 0)
    assert plan([110592]) == (8, 1, 1)
