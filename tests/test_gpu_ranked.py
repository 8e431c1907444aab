"""Waves ranked by progress in the field and force passes: launches on both
sides of the block counts where ranking begins (512), covers every block (up to
1,536) and covers the last blocks only, with spans of one record, of a few and
of several tiles, so quarters are empty, one record or cut tiles.

Forces against the component pass (FP32 rounding) and the FP64 oracle; a second
pass equals the first bit for bit."""
import pytest
import torch

import pyoracle as po
from isspa_amd import synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lbox", [300.0, 110.0])
@pytest.mark.parametrize("tiling", [(4, 4), (66, 184), (72, 188), (200, 556), (204, 560),
                                    (330, 900), (660, 1980)])
def test_ranked_launches(tiling, lbox):
    s = synth.make_lattice(30, 26.0, 4, lbox, seed=31)
    s.lbox, s.n_mc, s.seed = lbox, 3, 17
    g = GpuSystem(s, "cuda:0", us=False)
    g.set_tiling(*tiling)
    print(f"N={s.n_atoms} nMC={s.n_mc} box={lbox} tiling {g.tiling()}", flush=True)
    g.zero_forces()
    tot = g.isspa_force(step=2).clone()
    g.zero_forces()
    assert torch.equal(g.isspa_force(step=2), tot)
    comp = g.isspa_components(step=2)
    part = comp["lj"] + comp["pol"] + comp["cdd"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), part.cpu().numpy()) <= 2e-6
    ref = po.isspa_total(s, step=2)["total"]
    assert max_abs_rel_rms(tot[:, :3].double().cpu().numpy(), ref) <= 1e-5
    g.close()
