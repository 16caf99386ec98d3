"""Tiles of two products dealt to the XCDs (csrc/xcd_runs.h), on the host: every tile once, by count where that is the rule, in runs of equal
work else, and none longer than an XCD holds where that matters."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
#include <cstdio>
#include "xcd_runs.h"
int main()
{
    long long a, b;
    int ka, kb, most;
    while (scanf("%lld %d %lld %d", &a, &ka, &b, &kb) == 4) {
        const mch::XcdRuns r = mch::xcd_runs(a, ka, b, kb, 84, &most);
        for (int x = 0; x < 9; x++) printf("%d ", r.first[x]);
        printf("%d\\n", most);
    }
}
"""


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    d = tmp_path_factory.mktemp("xcd_runs")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "mycaffe_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "main")], check=True)

    def run(cases):
        text = "\n".join("%d %d %d %d" % c for c in cases)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return run


def test_runs(runs):
    rng = np.random.default_rng(1)
    cases = [(188, 179, 564, 34), (315, 652, 441, 451), (314, 3118, 390, 2507), (9, 727, 69, 84), (1, 100, 0, 90), (0, 100, 1, 90), (256, 1024, 1024, 256), (56, 3181, 700, 256),
             (1 << 19, 70000, 1 << 19, 90)]
    for _ in range(3000):
        short = int(2 ** rng.uniform(0, 14))
        cases.append((int(2 ** rng.uniform(0, 11)), short + int(2 ** rng.uniform(0, 14)), int(2 ** rng.uniform(0, 11)), short))
    for (a, ka, b, kb), (*first, most) in zip(cases, runs(cases)):
        case, ca, cb = (a, ka, b, kb, first), ka + 84, kb + 84
        count = np.diff(first)
        assert first[0] == 0 and first[8] == a + b and (count >= 0).all() and most == count.max(), case
        if a + b <= 8 * 32 or (a + b <= 8 * 96 and 5 * ca < 7 * cb):
            assert most <= -(-(a + b) // 8), case            # by count
        elif a + b <= 8 * 96 and kb <= 64:
            assert most <= 96, case                           # what an XCD holds
        else:
            cost = np.minimum(first, a) * ca + np.maximum(np.array(first) - a, 0) * cb
            assert np.abs(np.diff(cost) - cost[8] / 8).max() <= ca + 1, case   # equal work, to a tile
