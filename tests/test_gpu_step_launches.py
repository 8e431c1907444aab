"""The engine step's points and epilogue launches: points drawn by four lanes
each (point counts that fill no wave and no block, several windows), bonded and
restraint blocks before the field pass or behind the epilogue, on both sides of
256 blocks, and minimum-image flags over atom counts around a round of loads.

Points equal the oracle's bit for bit, forces the separate calls' bit for bit,
replays of a captured step and its centres of mass the eager ones."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import batch, synth
from isspa_amd.engine import GpuSystem

pytestmark = pytest.mark.gpu


def _check(s, step=3):
    g, h = GpuSystem(s, "cuda:0"), GpuSystem(s, "cuda:0")
    print(f"{s.n_atoms} atoms, {s.n_points} points, box {s.lbox}", flush=True)
    g.set_step(step)
    h.set_step(step)
    f = g.forces().clone()
    h.zero_forces()
    if h.bonded is not None:
        h.bonded_force()
    h.isspa_force(step=step)
    h.nonbond_force()
    if h.us is not None:
        h.us_force()
    torch.cuda.synchronize()
    assert torch.equal(f, h.f)
    assert torch.equal(g.field()["pts"], h.field()["pts"])
    pts = g.field()["pts"].cpu().numpy()
    g.set_step(step)
    h.set_step(step)
    g.step(4)
    h.capture(2)
    for _ in range(2):
        h.replay(1)
        torch.cuda.synchronize()
    assert torch.equal(g.x, h.x) and torch.equal(g.v, h.v)
    if h.us is not None:
        assert torch.equal(g.com(), h.com())
    g.close()
    h.close()
    return pts


@pytest.mark.parametrize("chains,n_mc,lbox", [
    (12, 1, 400.0), (13, 7, 400.0), (14, 3, 60.0), (93, 2, 400.0), (94, 1, 120.0), (187, 1, 400.0)])
def test_points_and_flags(chains, n_mc, lbox):
    grid = int(np.ceil(chains ** (1 / 3) - 1e-9))
    s = synth.make_lattice(chains, 16.0 * grid, grid, lbox, seed=5)
    s.lbox, s.n_mc, s.seed = lbox, n_mc, 91
    pts = _check(s)
    assert np.array_equal(pts[:, :3], po.mc_points(s, step=3)[:, :3].astype(np.float32))


@pytest.mark.parametrize("chains,n_mc", [(100, 25), (100, 27), (100, 28), (100, 30)])
def test_riders_around_256_blocks(chains, n_mc):
    """215 to 258 epilogue blocks with 17 or more bonded blocks behind them."""
    s = synth.make_lattice(chains, 80.0, 5, 400.0, seed=5)
    s.n_mc, s.seed = n_mc, 91
    _check(s)


@pytest.mark.parametrize("pairs,small,big", [(0, 3, 2), (2, 40, 4), (40, 16, 8), (0, 40, 16)])
def test_riders_with_restraints(pairs, small, big):
    """Restraint blocks behind the epilogue, or, with many windows, before; the
    last batch has more than 4,096 atoms, its all-pairs blocks ride all the same."""
    _check(batch.merge_windows(batch.umbrella_windows(pairs, small, big, n_mc=20)))
