"""All-pairs blocks of 64 receivers with a partner chunk a wave: atom counts
around a wave and a block, chunk counts that leave waves without a chunk, boxes
that need images, need none and are infinite (no images at all), several
windows.  Total and components against the FP64 oracle (1e-5 relative RMS)
and each other (1e-6); a second call equals the first bit for bit."""
import dataclasses

import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import batch, synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _atoms(n, lbox):
    """the first n atoms of a lattice of chains"""
    chains = -(-n // 22)
    grid = int(np.ceil(chains ** (1 / 3) - 1e-9))
    s = synth.make_lattice(chains, 16.0 * grid, grid, 400.0, seed=60 + chains)
    keep = lambda a: a[:n].copy()  # noqa: E731
    pre = s.nexcl_prefix[:n].copy()
    it = dataclasses.replace(s.isspa, isspa_type=keep(s.isspa.isspa_type))
    s = dataclasses.replace(
        s, xyzq=keep(s.xyzq), vel=keep(s.vel), true_mass=keep(s.true_mass), ityp=keep(s.ityp),
        nexcl_prefix=pre, excl_list=s.excl_list[:pre[-1]].copy(), isspa=it,
        bond_atoms=s.bond_atoms[:0], angle_atoms=s.angle_atoms[:0], dih_atoms=s.dih_atoms[:0],
        dih_types=s.dih_types[:0])
    s.lbox = lbox if lbox else float(np.ptp(s.xyzq[:, :3], axis=0).max()) + 4.0
    return s


def _check(s):
    print(f"N={s.n_atoms} box={s.lbox}", flush=True)
    g = GpuSystem(s, "cuda:0", isspa=False, bonded=False, us=False)
    tot = []
    for _ in range(2):
        g.zero_forces()
        g.nonbond_force()
        tot.append(g.f[:, :3].clone())
    assert torch.equal(tot[0], tot[1])
    t = tot[0].double().cpu().numpy()
    comp = {k: v.cpu().numpy() for k, v in g.nonbond_components().items()}
    g.close()
    return t, comp


@pytest.mark.parametrize("n", [2, 22, 63, 64, 65, 129, 255, 256, 257, 500, 1023, 2222])
@pytest.mark.parametrize("lbox", [400.0, 0.0, float("inf")])
def test_atom_counts(n, lbox):
    s = _atoms(n, lbox)
    t, comp = _check(s)
    ref = po.nonbond(dataclasses.replace(s, lbox=1.0e6) if np.isinf(lbox) else s)
    assert max_abs_rel_rms(t, ref["total"]) <= 1e-5
    assert max_abs_rel_rms(t, comp["lj"] + comp["coul"] + comp["pair"]) <= 1e-6


@pytest.mark.parametrize("windows", [(5, 3, 1), (40, 30, 8)])
def test_windows(windows):
    """each window's forces are those of the window alone, to FP64 regrouping"""
    ws = batch.umbrella_windows(*windows)
    t, comp = _check(batch.merge_windows(ws))
    assert max_abs_rel_rms(t, comp["lj"] + comp["coul"] + comp["pair"]) <= 1e-6
    a = 0
    for w in ws[:: max(1, len(ws) // 6)]:
        a = sum(v.n_atoms for v in ws[: next(k for k, v in enumerate(ws) if v is w)])
        assert max_abs_rel_rms(t[a:a + w.n_atoms], po.nonbond(w)["total"]) <= 1e-5
