"""The small-window launch (points, field, epilogue and force in one block) on
both sides of its limits and at its edges: window sizes around 64, 128, 192 and
256 atoms (it takes windows up to 256 atoms if one has at most 144), chunk groups of one point, of a whole
number of waves and one more, and of the largest 256 points; every split count
from one to more than a pass holds; boxes with and without images.

The forces equal the sum of the separate passes' components (the component
kernel, which never takes this launch) to FP32 rounding and the FP64 oracle to
1e-5 relative RMS; the MC points equal the separate passes' bit for bit; the
engine equals the separate calls bit for bit."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import batch, synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _check(s, tiling, step=4):
    g = GpuSystem(s, "cuda:0", us=False)
    if tiling:
        g.set_tiling(*tiling)
    print(f"N={s.n_atoms} nMC={s.n_mc} box={s.lbox} tiling {g.tiling()}", flush=True)
    g.zero_forces()
    tot = g.isspa_force(step=step).clone()
    pts = g.field()["pts"].clone()
    comp = g.isspa_components(step=step)
    assert torch.equal(pts, g.field()["pts"])
    part = comp["lj"] + comp["pol"] + comp["cdd"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), part.cpu().numpy()) <= 2e-6
    ref = po.isspa_total(s, step=step)["total"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), ref) <= 1e-5
    g.set_step(step)
    f = g.forces().clone()
    g.zero_forces()
    if g.bonded is not None:
        g.bonded_force()
    g.isspa_force(step=step)
    g.nonbond_force()
    torch.cuda.synchronize()
    assert torch.equal(f, g.f)
    g.close()


def _atoms(n, n_mc, lbox=200.0):
    """n atoms of a lattice of chains (the last chain cut)."""
    import dataclasses
    chains = -(-n // 22)
    s = synth.make_lattice(chains, 48.0, 3, lbox, seed=80 + chains)
    keep = lambda a: a[:n].copy()  # noqa: E731
    pre = s.nexcl_prefix[:n].copy()
    it = dataclasses.replace(s.isspa, isspa_type=keep(s.isspa.isspa_type))
    s = dataclasses.replace(
        s, xyzq=keep(s.xyzq), vel=keep(s.vel), true_mass=keep(s.true_mass), ityp=keep(s.ityp),
        nexcl_prefix=pre, excl_list=s.excl_list[:pre[-1]].copy(), isspa=it,
        bond_atoms=s.bond_atoms[:0], angle_atoms=s.angle_atoms[:0], dih_atoms=s.dih_atoms[:0],
        dih_types=s.dih_types[:0])
    s.lbox, s.n_mc, s.seed = lbox, n_mc, 99
    return s


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257])
@pytest.mark.parametrize("lbox", [200.0, 50.0])
def test_window_sizes(n, lbox):
    _check(_atoms(n, 3, lbox), None)


@pytest.mark.parametrize("n,n_mc,tiling", [
    (44, 1, (4, 44)), (44, 3, (1, 132)), (44, 16, (3, 11)), (44, 13, (44, 9)), (44, 29, (5, 5)),
    (64, 4, (9, 1)), (64, 5, (9, 1)), (100, 5, (8, 4)), (100, 5, (12, 3)), (200, 3, (2, 10)),
    (200, 3, (7, 9)), (256, 1, (32, 4)), (256, 1, (64, 1)), (256, 1, (256, 256))])
def test_groups_and_splits(n, n_mc, tiling):
    _check(_atoms(n, n_mc), tiling)


@pytest.mark.parametrize("n,n_mc,tiling", [
    (64, 8, (8, 8)), (57, 9, (1, 57)), (242, 20, (4, 22)), (242, 19, (13, 242)), (130, 1, (9, 61))])
def test_sixteen_waves(n, n_mc, tiling):
    """Field items of a group on both sides of a pass of eight waves (512): the
    block has sixteen above it, with receiver groups of one wave, a share pair
    and more units than waves."""
    _check(_atoms(n, n_mc), tiling)


@pytest.mark.parametrize("n", [143, 144, 145, 192, 193, 255, 256, 257])
@pytest.mark.parametrize("n_mc,tiling", [(3, None), (1, (5, 9)), (2, (32, 40))])
def test_two_windows(n, n_mc, tiling):
    """A window and a small one, which bring both into the launch up to 256
    atoms: forces against the component pass and the oracle, and against the
    window alone at the same tiling, which above 144 atoms takes the separate
    launches: the same bit for bit."""
    w = _atoms(n, n_mc)
    m = batch.merge_windows([w, _atoms(22, n_mc)], [0, 1])
    # (the cut chain's exclusions reach past its window: no all-pairs term)
    g = GpuSystem(m, "cuda:0", us=False, nonbond=False)
    if tiling:
        g.set_tiling(*tiling)
    print(f"{n} and 22 atoms, nMC={n_mc}, tiling {g.tiling()}", flush=True)
    g.zero_forces()
    tot = g.isspa_force(step=4).clone()
    comp = g.isspa_components(step=4)
    part = comp["lj"] + comp["pol"] + comp["cdd"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), part.cpu().numpy()) <= 2e-6
    if tiling:
        h = GpuSystem(w, "cuda:0", us=False, nonbond=False)
        h.set_tiling(*tiling)
        h.zero_forces()
        assert torch.equal(h.isspa_force(step=4)[:, :3], tot[:n, :3])
        h.close()
    ref = po.isspa_total(w, step=4)["total"]
    assert max_abs_rel_rms(tot[:n, :3].double().cpu().numpy(), ref) <= 1e-5
    g.close()


@pytest.mark.parametrize("pairs,small,big", [(3, 2, 1), (0, 1, 2), (5, 0, 0)])
def test_batch_engine(pairs, small, big):
    """A batch that takes the launch: engine steps equal graph replays, and its
    forces the separate calls, restraints riding along."""
    m = batch.merge_windows(batch.umbrella_windows(pairs, small, big, n_mc=7))
    g, h = GpuSystem(m, "cuda:0"), GpuSystem(m, "cuda:0")
    print(f"{m.n_atoms} atoms in {len(m.windows)} windows", flush=True)
    g.set_step(0)
    h.set_step(0)
    f = g.forces().clone()
    h.zero_forces()
    if h.bonded is not None:
        h.bonded_force()
    h.isspa_force(step=0)
    h.nonbond_force()
    h.us_force()
    torch.cuda.synchronize()
    assert torch.equal(f, h.f)
    g.step(6)
    h.capture(2)
    for k in range(3):
        h.replay(1)
        torch.cuda.synchronize()
    assert torch.equal(g.x, h.x) and torch.equal(g.v, h.v) and torch.equal(g.f, h.f)
    assert torch.equal(g.com(), h.com())
    g.close()
    h.close()
