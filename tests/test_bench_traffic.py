"""The k_force traffic that bench.py reports belongs to the kernel's present blocks
(CPU only): 64 receivers and four chunks a block, and one partial entry for them."""
import json
import math
import os
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402

N_ATOMS, N_POINTS = 19998, 399960
TRAFFIC = os.path.join(ROOT, "profiles", bench.FORCE_TRAFFIC_JSON)


def _points():
    with open(TRAFFIC) as fh:
        tr = json.load(fh)
    return tr, tr["points"]


@pytest.mark.parametrize("n,chunks,blocks", [
    (44, 68, 68), (64, 1, 1), (65, 5, 6), (128, 7, 8), (129, 7, 6), (1100, 8, 36),
    (19998, 207, 313 * 52)])
def test_force_grid(n, chunks, blocks):
    assert bench.force_grid(n, chunks) == 256 * blocks


def test_profile_matches_the_blocks():
    tr, pts = _points()
    entry_kib = 48 * N_ATOMS / 1024            # 6 FP64 partials per atom and group of chunks
    assert len(pts) >= 2 and tr["write_scale"] == 1.0 and 1.99 < tr["fetch_scale"] < 2.01
    for p in pts:
        groups = math.ceil(p["chunks"] / 4)
        assert p["grid"] == bench.force_grid(N_ATOMS, p["chunks"])
        assert abs(p["write_kib"] - entry_kib * groups) <= 64, p
        # the records and aux entries at least once
        assert p["fetch_kib"] * tr["fetch_scale"] * 1024 >= 80 * N_POINTS, p


def test_reported_traffic():
    tr, pts = _points()
    for p in pts:
        b, note, src = bench.traffic_at(p["chunks"], TRAFFIC)
        assert abs(b - p["traffic_bytes"]) <= 1024 and src == tr["summary"]
    # the counts that the tuner picks are covered: 0.5 to 2 times 207 and 414
    for c in (104, 207, 414, 827):
        assert bench.traffic_at(c, TRAFFIC)[0] is not None
    # one entry for four chunks: less than 2/3 of one for every chunk
    assert bench.traffic_at(414, TRAFFIC)[0] < 48 * N_ATOMS * 414 * 2 / 3
