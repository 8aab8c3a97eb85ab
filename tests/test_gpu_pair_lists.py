"""Ordered lists of deferred and rank-deficient pairs at the edges of the one-launch compaction (kernels.hip).

Two fragments without overlap give many rank-deficient blocks (nullity 1 and more); an entry that is missing,
doubled or out of place changes the energy. Bars of every parity test: 1e-8 Eh and 1e-7 in the gradient."""
import numpy as np
import pytest

import oracle
import xmvb_amd as vb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_act,mult", [
    (2, 1), (4, 1), (6, 1),  # 3 to 210 pairs: part of one sweep
    (9, 2),                  # 8,001 pairs: just below one sweep of 8,192
    (10, 3),                 # 22,155 pairs, three sweeps
    (10, 1),                 # 31,878 pairs, four sweeps, two listed per flagged spin-flip couple
    (11, 4),                 # 54,615 pairs: three launches
])
def test_lists_of_rank_deficient_blocks(n_act, mult):
    n_bf, n_aux = 24, 40
    sp = vb.synthetic_problem(5 + n_act, n_bf, n_act, n_aux)
    half, first = n_bf // 2, n_act // 2
    S, C = sp.S.copy(), sp.C.copy()
    S[:half, half:] = 0.0
    S[half:, :half] = 0.0
    C[:first, half:] = 0.0
    C[first:, :half] = 0.0
    sp = vb.SyntheticProblem(n_bf, n_act, n_aux, np.asfortranarray(S), sp.h, sp.B, C)
    topo = vb.Topology.build("COV", n_act, n_act, mult)
    ref = oracle.evaluate(n_bf, n_aux, topo, sp.S, sp.h, sp.B, sp.C)
    ctx = vb.Context(0)
    ctx.set_pair_condition_limit(9.9e4)  # the pair kernels whatever the size
    prob = vb.Problem.from_synthetic(ctx, sp, topo)
    e, g = prob.evaluate(sp.C)
    e2, g2 = prob.evaluate(sp.C)
    singular = prob.singular_pairs()
    prob.close()
    ctx.close()
    print(f"n_det={topo.n_determinants} singular {singular} dE={abs(e - ref['energy']):.1e} "
          f"dg={np.abs(g - ref['grad']).max():.1e}", flush=True)
    assert n_act == 2 or singular > 0
    assert abs(e - ref["energy"]) <= 1e-8
    assert np.abs(g - ref["grad"]).max() <= 1e-7
    assert e == e2 and np.array_equal(g, g2)
