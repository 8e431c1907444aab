"""The minimum image at its decision: separations of exactly half a box, one
float above and one below it, on every axis and with both signs, in boxes of
many sizes, against the FP64 oracle, which decides on the same FP32 values.  A
wrong image turns the pair's force round, so 1e-5 relative RMS finds one."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lbox", [1.0, 18.0, 33.3, 64.0, 200.0, 1000.0, 65536.5])
def test_half_box_separations(lbox):
    h = np.float32(0.5) * np.float32(lbox)
    for axis in range(3):
        for sep in (h, np.nextafter(h, np.float32(0)), np.nextafter(h, np.float32(np.inf))):
            for sign in (1, -1):
                s = synth.two_atom_lj(3.0, lbox=lbox)
                s.us = None
                # the first atom at the origin, so that the FP32 difference is the separation
                s.xyzq[:, :3] = 0.0
                s.xyzq[1, :3] = np.float32(0.1) * h
                s.xyzq[1, axis] = sign * sep
                s.xyzq[:, 3] = (3.0, -5.0)
                s.n_mc = 4
                print(f"box {lbox} axis {axis} separation {sign * sep!r}", flush=True)
                g = GpuSystem(s, "cuda:0", us=False)
                nb, ref = g.nonbond_components(), po.nonbond(s)
                for k in ("coul", "pair"):
                    assert max_abs_rel_rms(nb[k].cpu().numpy(), ref[k]) <= 1e-5, k
                g.zero_forces()
                tot = g.nonbond_force()[:, :3].double().cpu().numpy()
                assert max_abs_rel_rms(tot, ref["lj"] + ref["coul"] + ref["pair"]) <= 1e-5
                g.close()


def test_solvent_force_in_a_tight_box():
    """Every axis wraps for many pairs: 66 atoms in a box of 33 A."""
    s = synth.make_lattice(3, 33.0, 2, 33.0, seed=9)
    s.n_mc, s.seed = 7, 5
    g = GpuSystem(s, "cuda:0", us=False)
    comp, ref = g.isspa_components(step=1), po.isspa_total(s, step=1)
    for k in ("lj", "pol", "cdd"):
        assert max_abs_rel_rms(comp[k].cpu().numpy(), ref[k]) <= 1e-5, k
    torch.cuda.synchronize()
    g.close()
