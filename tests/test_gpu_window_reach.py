"""The small-window launch with three and four receiver groups (two shares a wave),
in boxes that need images and boxes that do not, with blocks of eight and of sixteen
waves and groups of up to 512, 1,024 and more (point, field split) pairs.

Every case asserts, from the stages that isspa_model_profile reports, that the
launch is taken.  Its forces equal, bit for bit, those of the window alone at the
same tiling (above 144 atoms the separate passes), match the component pass to FP32
rounding and the FP64 oracle to 1e-5 relative RMS; the engine, whose all-pairs and
bonded blocks ride on the launch, equals the separate calls bit for bit."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import batch, synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _window(chains, n_mc, lbox):
    s = synth.make_lattice(chains, 44.0, 3, lbox, seed=60 + chains)
    s.n_mc, s.seed, s.temperature_k, s.pnu = n_mc, 99, 298.0, 0.01
    return s


def _one_launch(g):
    return g.profile(1)["points"] == 0.0


# chains, nMC, (splits, chunks): the largest group's (point, split) pairs and the
# waves of a block
CASES = [
    (7, 2, (8, 103)),     # 154 atoms: 512 pairs, 8 waves
    (7, 4, (9, 52)),      # 576, 16 waves
    (11, 4, (16, 61)),    # 242 atoms: 1,024, 16 waves
    (11, 4, (32, 61)),    # 1,984, two passes
    (9, 4, (61, 50)),     # 198 atoms: 3,200, four passes
    (8, 20, (8, 1174)),   # 176 atoms, 304 blocks: 512, 8 waves
    (10, 20, (16, 1100)),  # 220 atoms: 1,024, 8 waves, two passes
    (9, 20, (24, 990)),   # 1,408, 8 waves, three passes
]


def _small(n_mc, lbox):
    """The window beside: a chain, or two atoms where many points make it many blocks."""
    if n_mc < 20:
        return _window(1, n_mc, lbox)
    s = synth.two_atom_lj(sep=6.0, lbox=lbox)
    s.n_mc, s.seed, s.temperature_k, s.pnu = n_mc, 99, 298.0, 0.01
    return s


@pytest.mark.parametrize("chains,n_mc,tiling", CASES)
@pytest.mark.parametrize("lbox", [200.0, 50.0])
def test_receiver_groups(chains, n_mc, tiling, lbox):
    w = _window(chains, n_mc, lbox)
    n = w.n_atoms
    # the box decides whether the windows take their images
    far = float(np.ptp(w.xyzq[:, :3], axis=0).max() + w.isspa.rmax.max()) >= lbox / 2
    assert far == (lbox == 50.0)
    g = GpuSystem(batch.merge_windows([w, _small(n_mc, lbox)], [0, 1]), "cuda:0", us=False)
    g.set_tiling(*tiling)
    print(f"{g.system.n_atoms} atoms, {n} in the first window, nMC={n_mc}, box {lbox}, tiling {g.tiling()}", flush=True)
    assert _one_launch(g)
    g.zero_forces()
    tot = g.isspa_force(step=4).clone()
    pts = g.field()["pts"].clone()
    h = GpuSystem(w, "cuda:0", us=False)
    h.set_tiling(*tiling)
    assert not _one_launch(h)
    h.zero_forces()
    assert torch.equal(h.isspa_force(step=4)[:, :3], tot[:n, :3])
    h.close()
    comp = g.isspa_components(step=4)
    assert torch.equal(pts, g.field()["pts"])
    part = comp["lj"] + comp["pol"] + comp["cdd"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), part.cpu().numpy()) <= 2e-6
    ref = po.isspa_total(w, step=4)["total"]
    assert max_abs_rel_rms(tot[:n, :3].double().cpu().numpy(), ref) <= 1e-5
    g.set_step(4)
    f = g.forces().clone()
    g.zero_forces()
    g.bonded_force()
    g.isspa_force(step=4)
    g.nonbond_force()
    torch.cuda.synchronize()
    assert torch.equal(f, g.f)
    g.close()


@pytest.mark.parametrize("chains,n_mc,tiling", [
    (2, 12, (8, 9)), (2, 12, (9, 9)), (6, 5, (16, 42)), (6, 5, (33, 42)), (3, 21, (4, 13))])
def test_small_windows_alone(chains, n_mc, tiling):
    """Windows of 44, 66 and 132 atoms in a box that needs images: 512, 576, 960 and
    2,112 pairs a group, and groups of 214 points."""
    w = _window(chains, n_mc, 50.0)
    g = GpuSystem(w, "cuda:0", us=False)
    g.set_tiling(*tiling)
    print(f"{w.n_atoms} atoms, nMC={n_mc}, tiling {g.tiling()}", flush=True)
    assert _one_launch(g)
    g.zero_forces()
    tot = g.isspa_force(step=4).clone()
    comp = g.isspa_components(step=4)
    part = comp["lj"] + comp["pol"] + comp["cdd"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), part.cpu().numpy()) <= 2e-6
    ref = po.isspa_total(w, step=4)["total"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), ref) <= 1e-5
    g.close()
