"""The differentiable model's fixed-order reductions at the edges of their
splits: chunk counts around the slices and batches of the per-atom sums, and
atom counts around one range of the per-type sums.

Tolerances: forces against the FP64 oracle as in test_gpu_diff.py (1e-5
relative RMS); the per-type sums against numpy's sum of the same FP64 terms,
n 2^-52 of the sum of their magnitudes."""
import numpy as np
import pytest
import torch

import pyoracle as po
from isspa_amd import synth
from isspa_amd.diff import DiffForces, DiffParams
from isspa_amd.system import max_abs_rel_rms

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.as_tensor(np.asarray(a, np.float64), device="cuda:0")


def _system(chains, n_mc):
    grid = int(np.ceil(chains ** (1 / 3) - 1e-9))
    s = synth.make_lattice(chains, 16.0 * grid, grid, 400.0, seed=7)
    s.n_mc, s.seed = n_mc, 78
    return s


@pytest.mark.parametrize("chunks", [1, 7, 8, 9, 31, 32, 33, 47, 48, 49, 66])
def test_chunk_counts(chunks):
    s = _system(3, 1)
    prm = DiffParams.from_system(s)
    m = DiffForces(s, prm, step=2)
    m.set_tiling(3, chunks)
    q, th = _t(prm.q), _t(prm.theta)
    pts = po.mc_points(s, step=2)
    print(f"chunks {chunks}", flush=True)
    err = max_abs_rel_rms(m.forces(q, th).cpu().numpy(), po.diff_forward(s, prm, pts)["total"])
    assert err <= 1e-5, err
    lam = np.random.default_rng(3).normal(size=(s.n_atoms, 3))
    gq, gt = m.vjp(q, th, _t(lam))
    rq, rt = po.diff_vjp(s, prm, pts, lam)
    assert max_abs_rel_rms(gq.cpu().numpy(), rq) <= 1e-4
    assert max_abs_rel_rms(gt.cpu().numpy(), rt) <= 1e-4


@pytest.mark.parametrize("chains", [1, 93, 94, 187])
def test_type_sums_over_atom_ranges(chains):
    """22, 2,046, 2,068 and 4,114 atoms: one, one, two and three ranges."""
    s = _system(chains, 1)
    prm = DiffParams.from_system(s)
    m = DiffForces(s, prm)
    print(f"{s.n_atoms} atoms", flush=True)
    lam = np.random.default_rng(4).normal(size=(s.n_atoms, 3))
    _, gt, ga = m.vjp(_t(prm.q), _t(prm.theta), _t(lam), per_atom=True)
    gt, ga = gt.cpu().numpy(), ga.cpu().numpy()
    for t in range(prm.n_types):
        mine = ga[s.isspa.isspa_type == t]
        tol = max(1, len(mine)) * 2.0 ** -52 * np.abs(mine).sum(axis=0)
        assert np.all(np.abs(gt[t] - mine.sum(axis=0)) <= tol), t


@pytest.mark.parametrize("chains,n_mc,splits,chunks", [
    (3, 1, 1, 1), (3, 1, 2, 66), (3, 2, 6, 5), (3, 2, 8, 132), (3, 1, 66, 3), (12, 2, 4, 24),
    (12, 2, 264, 420), (12, 5, 132, 1300)])
def test_adjoint_split_groups(chains, n_mc, splits, chunks):
    """One, two and four splits a block, points that fill no block, spans of
    one atom or record, and launches of up to 512, 1,536 and more blocks."""
    s = _system(chains, n_mc)
    prm = DiffParams.from_system(s)
    m = DiffForces(s, prm, step=2)
    m.set_tiling(splits, chunks)
    print(f"{s.n_atoms} atoms, {splits} splits, {chunks} chunks", flush=True)
    lam = np.random.default_rng(5).normal(size=(s.n_atoms, 3))
    gq, gt = m.vjp(_t(prm.q), _t(prm.theta), _t(lam))
    rq, rt = po.diff_vjp(s, prm, po.mc_points(s, step=2), lam)
    assert max_abs_rel_rms(gq.cpu().numpy(), rq) <= 1e-4
    assert max_abs_rel_rms(gt.cpu().numpy(), rt) <= 1e-4
