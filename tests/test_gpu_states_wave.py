"""Selected states of small spaces on one wavefront (gep_wave.hip) against LAPACK on the engine's own H and S.

Bars fixed beforehand, those of every parity test: 1e-8 Eh for each state and for the weighted average."""
import numpy as np
import pytest
import scipy.linalg

import xmvb_amd as vb
from test_gpu_eigen_large import first_structures

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 17, 42, 63, 64])
def test_selected_states_of_small_spaces(n):
    topo = first_structures(vb.Topology.build("FULL", 5, 5, 2), n)
    sp = vb.synthetic_problem(77, 20, 5, 30)
    for states in ([1], [0, 1], [n - 1], [0, n // 2, n - 1] if n > 2 else [1, 0]):
        weights = np.arange(1.0, len(states) + 1)
        ctx = vb.Context(0)
        ctx.set_states(states, weights)
        prob = vb.Problem.from_synthetic(ctx, sp, topo)
        e, g = prob.evaluate(sp.C)
        found, mid = prob.state_energies(), prob.intermediates()
        prob.close()
        ctx.close()
        H, S = (mid["H"] + mid["H"].T) / 2, (mid["S"] + mid["S"].T) / 2
        ref = scipy.linalg.eigh(H, S, eigvals_only=True)[states]
        c = mid["coef"]
        print(f"n_str={n} {states} {np.abs(found - ref).max():.1e} norm {c @ S @ c - 1:.1e}", flush=True)
        assert np.abs(found - ref).max() <= 1e-8
        assert abs(e - (weights / weights.sum()) @ ref) <= 1e-8
        assert abs(c @ S @ c - 1) <= 1e-10
        assert np.isfinite(g).all()
