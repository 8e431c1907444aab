"""The autotuner on models whose force call takes the small-window launch at some
tilings (no GPU): isspa_model_profile then reports that launch as the force stage
and the passes inside it as 0."""
import math

import pytest

from isspa_amd import autotune


@pytest.mark.parametrize("n", [1, 44, 64, 65, 128, 129, 1100, 4510, 19998])
def test_force_blocks_follow_the_grid(n):
    """The force pass launches ceil(n / 64) blocks for each group of chunks; four
    chunks are four groups with four shares of a chunk a block, two with two."""
    shares = 4 if n <= 64 else 2 if n <= 128 else 1
    assert 4 * autotune.force_blocks(n) == math.ceil(n / 64) * shares
    if n == 19998:
        # whole groups of four chunks: the grid of the candidate counts
        for c in autotune.round_aligned(n * 20, autotune.force_blocks(n), 208)[:-1]:
            if c % 4 == 0 and c != 208:
                rounds = math.ceil(n / 64) * (c // 4) * 4 / 8192
                assert rounds == int(rounds) or rounds % 1 >= 0.85


class _Model:
    """Stage times as a function of the tiling: one launch where the chunks are
    at most `limit`, the separate passes above."""

    class _Sys:
        n_atoms, n_points = 44, 4400

    windows = None
    system = _Sys()

    def __init__(self, limit, launch_ms):
        self.limit, self.launch_ms = limit, launch_ms
        self.t, self.waves = (0, 0), 32768

    def set_tiling(self, s, c):
        self.t = (s, c)

    def set_target_waves(self, w):
        self.waves = w

    def tiling(self):
        return self.t if self.t != (0, 0) else (4, 64)

    def profile(self, reps):
        s, c = self.tiling()
        if c <= self.limit:
            # splits and chunks nearer to 8 and 32 are faster
            return {"points": 0.0, "field": 0.0, "epilogue": 0.0, "reduce": 1.0,
                    "force": self.launch_ms + 0.1 * abs(s - 8) + 0.01 * abs(c - 32)}
        return {"points": 3.0, "field": 4.0, "epilogue": 3.0, "force": 4.0, "reduce": 1.0}

    def pass_ms(self):
        return sum(self.profile(1).values())


@pytest.mark.parametrize("limit,launch_ms", [(10 ** 6, 9.0), (64, 9.0), (48, 13.5)])
def test_whole_calls_are_compared(limit, launch_ms):
    """The separate passes take 15 ms a call, points included, the one launch 10
    (or 14.5) and more: a candidate that runs as one launch is not ranked by
    stages that it does not run, and the points are part of what it replaces."""
    g = _Model(limit, launch_ms)
    r = autotune.tune(g, reps=1)
    assert r.ms == pytest.approx(g.pass_ms())
    assert all(ms > launch_ms for kind, _, ms in r.table
               if kind not in ("field-splits", "force-chunks"))
    # the field splits are chosen by calls that run them
    splits = [(ms, v) for kind, v, ms in r.table if kind == "field-splits"]
    if limit >= 64:
        assert all(ms > launch_ms for ms, _ in splits)
        assert min(splits)[1] == min(((abs(v[0] - 8), v) for _, v in splits))[1]
    assert r.ms < 15.0


def test_separate_passes_rank_by_their_own_stages():
    g = _Model(0, 9.0)
    r = autotune.tune(g, reps=1)
    got = {kind: ms for kind, _, ms in r.table}
    assert got["field-splits"] == 7.0 and got["force-chunks"] == 5.0
    assert got["tiling"] == 15.0
