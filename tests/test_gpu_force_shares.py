"""The force pass's chunk groups at their edges: windows on both sides of the
64- and 128-atom share rules and of a 64-receiver block, with chunk counts that
fill a block's four shares and that leave one, two or three of them empty.

Tolerance: the FP64 oracle at 1e-5 relative RMS, as for every force pass; the
engine equals the separate calls, and isspa_force_keep the plain call, bit for
bit."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _system(chains):
    s = synth.make_lattice(chains, 48.0, 3, 200.0, seed=60 + chains)
    s.n_mc, s.seed = 3, 4321
    return s


@pytest.mark.parametrize("chains", [2, 5, 6, 12])  # 44, 110, 132 and 264 atoms
@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5, 7, 9, 33])
def test_chunk_groups_match_oracle(chains, chunks):
    s = _system(chains)
    g = GpuSystem(s, "cuda:0", us=False)
    g.set_tiling(3, chunks)
    print(f"N={s.n_atoms} tiling {g.tiling()}", flush=True)
    ref = po.isspa_total(s, step=2)
    comp = g.isspa_components(step=2)
    for k in ("lj", "pol", "cdd"):
        assert max_abs_rel_rms(comp[k].cpu().numpy(), ref[k]) <= 1e-5, k
    g.set_step(2)
    got = g.forces().clone()
    g.zero_forces()
    g.bonded_force()
    alone = torch.empty_like(g.f)
    g.isspa_force_keep(g.f, alone, step=2)
    g.nonbond_force()
    torch.cuda.synchronize()
    assert torch.equal(got, g.f)
    plain = torch.zeros_like(g.f)
    g.isspa_force(step=2, f=plain)
    assert torch.equal(plain, alone)
    assert max_abs_rel_rms(plain[:, :3].double().cpu().numpy(), ref["total"]) <= 1e-5
    g.close()
