"""Dense eigensolve of spaces beyond one wavefront (gep_large.hip) against LAPACK on the engine's own H and S.

Bars fixed beforehand: the energy as in every parity test (1e-8 Eh), c^T S c = 1 to 1e-10 and the residual
|H c - E S c| to 1e-9 of the largest element of H (Lanczos stops at a residual of a few rounding units)."""
import dataclasses

import numpy as np
import pytest
import scipy.linalg

import xmvb_amd as vb

pytestmark = pytest.mark.gpu


def first_structures(topo, n, empty=False):
    """The space of the first n structures (empty: the last of them without determinants)."""
    keep = topo.term_structure < (n - 1 if empty else n)
    det = np.repeat(np.arange(topo.n_determinants), np.diff(topo.term_offsets))
    count = np.bincount(det[keep], minlength=topo.n_determinants)
    live = count > 0
    return dataclasses.replace(
        topo, raw_structures=topo.raw_structures[:n], det_alpha=topo.det_alpha[live], det_beta=topo.det_beta[live],
        term_offsets=np.concatenate([[0], np.cumsum(count[live])]).astype(np.int64),
        term_structure=topo.term_structure[keep].copy(), term_coefficient=topo.term_coefficient[keep].copy())


def check(sp, topo, ctx):
    prob = vb.Problem.from_synthetic(ctx, sp, topo)
    e, g = prob.evaluate(sp.C)
    mid = prob.intermediates()
    prob.close()
    H, S, c = (mid["H"] + mid["H"].T) / 2, (mid["S"] + mid["S"].T) / 2, mid["coef"]
    ref = scipy.linalg.eigh(H, S, subset_by_index=[0, 0], eigvals_only=True)[0]
    residual = np.abs(H @ c - e * (S @ c)).max() / np.abs(H).max()
    print(f"n_str={topo.n_structures} dE={e - ref:.1e} norm {c @ S @ c - 1:.1e} residual {residual:.1e}", flush=True)
    assert abs(e - ref) <= 1e-8
    assert abs(c @ S @ c - 1) <= 1e-10
    assert residual <= 1e-9
    assert np.isfinite(g).all()
    return e, g


@pytest.mark.parametrize("n_act,mult,sizes", [
    (6, 1, (65, 96, 97, 128, 129, 175)),
    (7, 2, (190, 191, 192, 193, 255, 256, 257, 448, 449, 784)),  # Cholesky in LDS to 190, blocked from 256
    (8, 1, (1024, 1025)),  # Lanczos to 1024
])
def test_lowest_root_at_every_form_of_the_solver(n_act, mult, sizes):
    sp = vb.synthetic_problem(17 + n_act, 24, n_act, 40)
    topo = vb.Topology.build("FULL", n_act, n_act, mult)
    ctx = vb.Context(0)
    for n in sizes:
        check(sp, first_structures(topo, n), ctx)
    ctx.close()


@pytest.mark.parametrize("n", [65, 257])
def test_more_problems_than_the_blocked_form_takes(n):
    """Nine problems per launch: one workgroup each through the whole solve."""
    topo = first_structures(vb.Topology.build("FULL", 7, 7, 2), n)
    sps = [vb.synthetic_problem(200 + k, 24, 7, 40) for k in range(9)]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 9)
    for k, sp in enumerate(sps):
        pool.load_synthetic(k, sp)
    e, g = pool.evaluate(list(range(9)), [sp.C for sp in sps])
    for k in (0, 8):
        e1, g1 = check(sps[k], topo, ctx)
        assert abs(e[k] - e1) <= 1e-8 and np.abs(g[k] - g1).max() <= 1e-7
    pool.close()
    ctx.close()


@pytest.mark.parametrize("n", [100, 300])
def test_a_singular_metric_is_refused(n):
    topo = first_structures(vb.Topology.build("FULL", 7, 7, 2), n, empty=True)
    ctx = vb.Context(0)
    sp = vb.synthetic_problem(3, 24, 7, 40)
    prob = vb.Problem.from_synthetic(ctx, sp, topo)
    with pytest.raises(vb.VbeError):
        prob.evaluate(sp.C)
    prob.close()
    ctx.close()
