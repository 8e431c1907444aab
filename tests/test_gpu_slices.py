"""The per-atom sums at the edges of their slices and batches: entry counts one
below, at and one above a slice round, a batch and several batches, atom counts
around a block of 16, and the engine's step counter across steps, graphs and
set_step.

The IS-SPA force against the FP64 oracle (1e-5 relative RMS) and, bit for bit,
the engine against the separate calls."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import synth
from isspa_amd.engine import GpuSystem
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _system(chains, n_mc, lbox=200.0):
    grid = int(np.ceil(chains ** (1 / 3) - 1e-9))
    s = synth.make_lattice(chains, 16.0 * grid, grid, lbox, seed=30 + chains)
    s.n_mc, s.seed = n_mc, 17
    synth.maxwell_velocities(s, seed=3)
    return s


# entries per atom: the chunk count at 22 atoms, a quarter of it (rounded up) at 286
@pytest.mark.parametrize("chains,n_mc,chunks", [(1, 24, c) for c in (1, 15, 16, 17, 63, 64, 65, 95, 96, 97,
                                                                      127, 128, 129, 257, 528)] +
                         [(13, 1, c) for c in (61, 64, 65, 260)])
def test_entry_counts(chains, n_mc, chunks):
    s = _system(chains, n_mc)
    g = GpuSystem(s, "cuda:0", us=False)
    g.set_tiling(2, chunks)
    print(f"N={s.n_atoms} tiling {g.tiling()}", flush=True)
    g.set_step(6)
    got = g.forces().clone()
    g.zero_forces()
    g.bonded_force()
    f = torch.zeros_like(g.f)
    g.isspa_force(step=6, f=f)
    g.isspa_force(step=6)
    g.nonbond_force()
    torch.cuda.synchronize()
    assert torch.equal(got, g.f)
    ref = po.isspa_total(s, step=6)["total"]
    assert max_abs_rel_rms(f[:, :3].double().cpu().numpy(), ref) <= 1e-5
    g.close()


@pytest.mark.parametrize("chains,n_mc", [(1, 3), (13, 2)])  # the small-window launch, and the separate passes
@pytest.mark.parametrize("per_graph", [1, 2, 3])
def test_step_counter(chains, n_mc, per_graph):
    """Graph replays, eager steps and separate calls with explicit step numbers
    draw the same points and collisions."""
    a, b, c = (GpuSystem(_system(chains, n_mc), "cuda:0", us=False) for _ in range(3))
    print(f"N={a.system.n_atoms}, {per_graph} steps a graph", flush=True)
    a.set_step(40)
    a.capture(per_graph)
    b.set_step(40)
    for k in range(2):
        a.replay(1)
        torch.cuda.synchronize()
        if k == 0:
            b.forces()  # a force evaluation does not move the step on
        b.step(per_graph)
        for j in range(per_graph):
            step = 40 + k * per_graph + j
            c.zero_forces()
            c.bonded_force()
            c.isspa_force(step=step)
            c.nonbond_force()
            c.leapfrog(step=step)
        torch.cuda.synchronize()
        for u, v, w in ((a.x, b.x, c.x), (a.v, b.v, c.v), (a.f, b.f, c.f)):
            assert torch.equal(u, v) and torch.equal(u, w)
    for g in (a, b, c):
        g.close()
