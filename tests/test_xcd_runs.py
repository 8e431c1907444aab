"""The force blocks of a batch on the eight XCDs: every XCD's sequence of workgroups is
longest first, whatever the sizes of the chunk groups, and a group's blocks stay on one
XCD but for the few that even out the runs."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "isspa-force-cuda_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include "xcd_runs.hpp"
struct B { int x, y, z; };
int main()
{
    std::vector<std::pair<long long, B>> t;
    long long w;
    B b;
    while (std::scanf("%lld %d %d %d", &w, &b.x, &b.y, &b.z) == 4) t.push_back({w, b});
    isspa::groups_to_xcds(t);
    for (int i = 0; i < (int)t.size(); ++i) {
        const auto &e = t[isspa::xcd_run_entry(i, (int)t.size())];
        std::printf("%lld %d %d %d\n", e.first, e.second.x, e.second.y, e.second.z);
    }
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("xcd")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)

    def run(table):
        text = "\n".join(" ".join(map(str, row)) for row in table)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True)
        return np.array([line.split() for line in out.stdout.splitlines()], dtype=int).reshape(-1, 4)

    return run


# (windows, receiver blocks, groups, points a share) of each kind of window
UMBRELLA = [(10, 1, 1, 10), (34, 1, 2, 55), (12, 4, 69, 16)]


@pytest.mark.parametrize("kinds", [
    UMBRELLA, [(18, 1, 1, 17), (38, 1, 4, 46), (15, 4, 107, 17)], [(3, 18, 6, 20)],
    [(9, 18, 1, 183)], [(2, 1, 1, 10)], [(1, 1, 1, 3), (1, 313, 2, 40)], [(256, 18, 7, 196)],
    [(7, 5, 3, 9), (5, 2, 11, 9), (31, 1, 1, 30)]])
def test_runs_are_longest_first(deal, kinds):
    table, w = [], 0
    for n, rblocks, groups, work in kinds:
        for _ in range(n):
            table += [(work, w, b, g) for g in range(groups) for b in range(rblocks)]
            w += 1
    table.sort(key=lambda e: -e[0])
    got = deal(table)
    assert sorted(map(tuple, got)) == sorted(table)
    apart = 0
    for x in range(8):
        assert np.all(np.diff(got[x::8, 0]) <= 0), f"XCD {x}: {got[x::8, 0]}"
    homes = {}
    for i, (_, win, _, g) in enumerate(got):
        homes.setdefault((win, g), []).append(i % 8)
    for v in homes.values():
        apart += len(v) - max(v.count(x) for x in set(v))
    # the longest group may leave a run over by all but one of its blocks
    longest = max(k[1] for k in kinds)
    assert apart <= 7 * longest
