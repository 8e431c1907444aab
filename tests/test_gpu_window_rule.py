"""Which batches take the small-window launch.  Windows of at most 144 atoms alone
take it and larger ones alone do not; with both, the longest chains decide
(window_pays): a small window must not carry a batch of large ones into the slower
route.  The route is the one that isspa_model_profile reports, and both give the
same forces bit for bit."""
import math
import random

import pytest
import torch

from isspa_amd import batch, synth
from isspa_amd.engine import GpuSystem

pytestmark = pytest.mark.gpu


def _windows(sizes, n_mc):
    """Windows of 2 atoms (size 0) or of so many chains of 22."""
    ws = []
    for k, c in enumerate(sizes):
        s = synth.two_atom_lj(sep=6.0, lbox=200.0) if c == 0 else \
            synth.make_lattice(c, 40.0, 3, 200.0, seed=50 + k)
        s.n_mc, s.temperature_k, s.pnu, s.seed = n_mc, 298.0, 0.01, 12348
        ws.append(s)
    return ws


def _atoms(sizes):
    return [22 * c or 2 for c in sizes]


def _one_launch(g):
    p = g.profile(1)
    assert (p["field"] == 0.0) == (p["points"] == 0.0) == (p["epilogue"] == 0.0)
    return p["field"] == 0.0


def _tile(ns, n_mc, splits, chunks):
    """Windows at an explicit tiling, as the library cuts them."""
    out = []
    for n in ns:
        P = n * n_mc
        aps = -(-n // min(splits, n))
        ppc = -(-P // min(chunks, P))
        shares = 4 if n <= 64 else 2 if n <= 128 else 1
        c = -(-P // ppc)
        out.append((n, P, aps, -(-n // aps), ppc, shares, -(-c // (4 // shares))))
    return out


def _expected(ns, n_mc, splits, chunks):
    w = _tile(ns, n_mc, splits, chunks)
    blocks = sum(t[6] for t in w)
    pts = [min(P, 4 // sh * ppc) for _, P, _, _, ppc, sh, _ in w]
    if max(ns) > 256 or max(pts) > 256 or blocks > 512:
        return False
    if max(ns) <= 144 or min(ns) > 144:
        return max(ns) <= 144
    items = max(t[3] * math.ceil(p / 64) * 64 for t, p in zip(w, pts))
    nt = 1024 if items > 512 and blocks <= 256 else 512
    chain = longest = entries = 0.0
    for (n, P, aps, s, ppc, sh, _), p in zip(w, pts):
        passes = math.ceil(s / (nt // (math.ceil(p / 64) * 64)))
        share = math.ceil(ppc / sh)
        chain = max(chain, passes * aps + 0.6 * (1 if n <= 128 else 2) * share)
        longest = max(longest, share)
        entries = max(entries, s // (4 if s % 4 == 0 else 2 if s % 2 == 0 else 1))
    return chain <= 20 + 0.6 * longest + 0.8 * entries + 8e-6 * sum(n * P for n, P, *_ in w)


@pytest.mark.parametrize("sizes,n_mc,one_launch", [
    ([10] * 4 + [0] * 4, 10, False),      # solvent force 28.4 us, 32.7 as one launch
    ([10] * 8 + [1] * 8, 5, False),       # 29.8, 32.2
    ([9] * 6 + [0], 20, False),           # 36.4, 41.6
    ([10] * 4 + [1] * 20, 10, True),      # 35.8, 30.3
    ([10] * 2 + [1] * 8 + [0] * 32, 20, True),
    ([10] + [1] * 40 + [0] * 39, 20, True),  # step 35.9 us separate, 32.1 as one launch
    ([10] + [1] * 12 + [0] * 4, 10, False),  # 35.3, 37.2
    ([6] * 3 + [0], 10, True),
    ([7, 8], 10, False)])
def test_where_the_work_is(sizes, n_mc, one_launch):
    g = GpuSystem(batch.merge_windows(_windows(sizes, n_mc)), "cuda:0", us=False)
    print(f"{sizes} nMC={n_mc} tiling {g.tiling()}", flush=True)
    assert _one_launch(g) == one_launch
    g.close()


def test_rule_over_tilings_and_equal_forces():
    """Explicit tilings: the route follows the rule, and the forces of every window
    are those of the window alone at the same tiling, by whichever route."""
    rng = random.Random(4)
    seen = set()
    for _ in range(24):
        sizes = [rng.choice([7, 8, 9, 10, 11]) for _ in range(rng.choice([1, 2, 3]))] + \
                [rng.choice([0, 1, 2, 4, 6]) for _ in range(rng.choice([1, 2, 4]))]
        n_mc, tiling = rng.choice([2, 5, 11]), (rng.choice([2, 4, 7, 12]),
                                                       rng.choice([12, 30, 61, 120]))
        ws = _windows(sizes, n_mc)
        m = batch.merge_windows(ws)
        g = GpuSystem(m, "cuda:0", us=False)
        g.set_tiling(*tiling)
        want = _expected(_atoms(sizes), n_mc, *tiling)
        print(f"{sizes} nMC={n_mc} tiling {tiling}: {'one launch' if want else 'separate'}",
              flush=True)
        assert _one_launch(g) == want
        seen.add(want)
        g.zero_forces()
        f = g.isspa_force(step=3).clone()
        for w, (a, b) in enumerate(batch.window_slices(m)):
            h = GpuSystem(batch.merge_windows([ws[w]], [w]), "cuda:0", us=False)
            h.set_tiling(*tiling)
            h.zero_forces()
            assert torch.equal(h.isspa_force(step=3), f[a:b]), (sizes, w)
            h.close()
        g.close()
    assert seen == {True, False}
