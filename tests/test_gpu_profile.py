"""isspa_model_profile times the launches that the force calls make: the separate
passes, or, where a model's windows take the small-window launch, that launch and
the reduction."""
import pytest

from isspa_amd import synth
from isspa_amd.engine import GpuSystem

pytestmark = pytest.mark.gpu


def _system(chains, n_mc):
    s = synth.make_lattice(chains, 80.0, 4, 200.0, seed=7) if chains > 1 else synth.make_chain()
    s.n_mc, s.seed = n_mc, 5
    return s


@pytest.mark.parametrize("chains,n_mc,tiling,one_launch", [
    (1, 4, None, True), (2, 100, None, True), (6, 20, None, True),
    (2, 100, (5, 2200), False),   # 2,200 chunks of two points: too many blocks
    (2, 100, (5, 4), False),      # chunks of 1,100 points: too large for a block
    (7, 20, None, False), (50, 20, None, False)])
def test_profile_times_what_runs(chains, n_mc, tiling, one_launch):
    g = GpuSystem(_system(chains, n_mc), "cuda:0", us=False)
    if tiling:
        g.set_tiling(*tiling)
    p = g.profile(2)
    print(f"{chains} chains, nMC={n_mc}, tiling {g.tiling()}: {p}", flush=True)
    passes = ("points", "field", "epilogue")
    if one_launch:
        assert all(p[k] == 0.0 for k in passes)
    else:
        assert all(p[k] > 0.0 for k in passes)
    assert p["force"] > 0.0 and p["reduce"] > 0.0
    # and leaves the next evaluation as it was
    f = g.forces().clone()
    g.profile(1)
    assert (g.forces() == f).all()
    g.close()
