"""The string form (strings.hip) against the pair kernels and the FP64 oracle, through the C ABI.

A context with its own pair condition limit keeps the pair kernels, so the same problem evaluated with
the default limit and with another one compares the two forms, at the bars of every parity test: 1e-8 Eh
and 1e-7 in the gradient (the pair form amplifies the rounding of a block by its condition, up to 1e5)."""
import numpy as np
import pytest

import oracle
import xmvb_amd as vb

pytestmark = pytest.mark.gpu

E_TOL, G_TOL = 1e-8, 1e-7


def evaluate(sp, topo, C=None, pairs=False, states=None):
    ctx = vb.Context(0)
    if pairs:
        ctx.set_pair_condition_limit(9.9e4)
    if states:
        ctx.set_states(*states)
    prob = vb.Problem.from_synthetic(ctx, sp, topo)
    e, g = prob.evaluate(sp.C if C is None else C)
    singular = prob.singular_pairs()
    mid = prob.intermediates()
    prob.close()
    ctx.close()
    return e, g, singular, mid


@pytest.mark.parametrize("kw,n_act,n_el,mult", [
    ("COV", 10, 10, 1), ("COV", 10, 10, 3), ("COV", 11, 11, 2), ("COV", 12, 12, 1), ("COV", 13, 13, 2),
    ("FULL", 5, 5, 2),          # 100 determinants: the pair kernels alone
    ("FULL", 6, 6, 1), ("FULL", 7, 7, 2),  # many determinants per string, equal and unequal spins
    ("COV,ION(1)", 8, 8, 1),    # spin-flip couples and doubly occupied orbitals
    ("COV", 8, 6, 1),           # empty orbitals
    ("COV", 7, 9, 2),           # more electrons than orbitals
])
def test_string_form_matches_pair_kernels(kw, n_act, n_el, mult):
    print(f"case strings {kw} n_act={n_act} n_el={n_el} mult={mult}", flush=True)
    topo = vb.Topology.build(kw, n_act, n_el, mult)
    sp = vb.synthetic_problem(31 + n_act, 30, n_act, 45)
    C = sp.C.copy()
    C[:-1] += 0.4 * sp.C[1:]
    e, g, s, mid = evaluate(sp, topo, C)
    e2, g2, s2, mid2 = evaluate(sp, topo, C, pairs=True)
    print(f"dE={abs(e - e2):.2e} dg={np.abs(g - g2).max():.2e} singular {s} {s2}", flush=True)
    assert abs(e - e2) <= E_TOL
    assert np.abs(g - g2).max() <= G_TOL
    assert s == s2
    for k in ("H", "S"):
        assert np.abs(mid[k] - mid2[k]).max() <= 1e-10 * np.abs(mid2[k]).max()


def test_rank_deficient_blocks_are_counted_and_differentiated():
    """Two fragments without overlap: blocks of nullity 1 to 3; the string form takes their
    values from the complete-pivoting kernel and differentiates the minors directly."""
    n_bf, n_act = 24, 10
    sp = vb.synthetic_problem(5, n_bf, n_act, 40)
    half = n_bf // 2
    S = sp.S.copy()
    S[:half, half:] = 0.0
    S[half:, :half] = 0.0
    C = sp.C.copy()
    C[:5, half:] = 0.0
    C[5:, :half] = 0.0
    sp = vb.SyntheticProblem(n_bf, n_act, 40, np.asfortranarray(S), sp.h, sp.B, C)
    topo = vb.Topology.build("COV", n_act, n_act, 1)
    e, g, s, _ = evaluate(sp, topo)
    e2, g2, s2, _ = evaluate(sp, topo, pairs=True)
    ref = oracle.evaluate(n_bf, 40, topo, sp.S, sp.h, sp.B, sp.C)
    print(f"singular {s} {s2} dE={abs(e - ref['energy']):.2e} dg={np.abs(g - ref['grad']).max():.2e}", flush=True)
    assert s == s2 > 0
    assert abs(e - ref["energy"]) <= 1e-8 and abs(e - e2) <= E_TOL
    assert np.abs(g - ref["grad"]).max() <= 1e-7 and np.abs(g - g2).max() <= G_TOL


def test_ill_conditioned_orbitals_keep_the_pair_kernels_in_a_mixed_launch():
    """One launch of three slots: well separated orbitals (string form) around a slot whose first
    two orbitals nearly coincide (|S_act^-1| far above the limit), each equal to the slot alone."""
    topo = vb.Topology.build("COV", 10, 10, 1)
    sps = [vb.synthetic_problem(60 + k, 32, 10, 48) for k in range(3)]
    C = [sp.C.copy() for sp in sps]
    C[1][1] = C[1][0] + 0.05 * C[1][1]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 3)
    for k, sp in enumerate(sps):
        pool.load_synthetic(k, sp)
    e, g = pool.evaluate([0, 1, 2], C)
    for k, sp in enumerate(sps):
        ref = oracle.evaluate(32, 48, topo, sp.S, sp.h, sp.B, C[k])
        print(f"slot {k} dE={abs(e[k] - ref['energy']):.2e} dg={np.abs(g[k] - ref['grad']).max():.2e}", flush=True)
        assert abs(e[k] - ref["energy"]) <= 1e-8
        assert np.abs(g[k] - ref["grad"]).max() <= (1e-6 if k == 1 else 1e-7)
    # the slot alone, energy and gradient apart: the pair kernels follow the string form's first try
    prob = vb.Problem.from_synthetic(ctx, sps[1], topo)
    e1 = prob.evaluate_forward(C[1])
    g1 = prob.complete_gradient()
    assert abs(e1 - e[1]) <= 1e-8 and np.abs(g1 - g[1]).max() <= 1e-6
    e0, g0 = prob.evaluate(sps[1].C)  # and back
    ref = oracle.evaluate(32, 48, topo, sps[1].S, sps[1].h, sps[1].B, sps[1].C)
    assert abs(e0 - ref["energy"]) <= 1e-8 and np.abs(g0 - ref["grad"]).max() <= 1e-7
    prob.close()
    pool.close()
    ctx.close()


@pytest.mark.parametrize("n_act,n_el,mult", [(9, 9, 2), (14, 2, 1)])
def test_batches_of_smaller_spaces(n_act, n_el, mult):
    """126 determinants with unequal spins, and one electron of each spin (no double replacements): from
    sixteen problems per launch on."""
    topo = vb.Topology.build("COV", n_act, n_el, mult)
    sps = [vb.synthetic_problem(90 + k, 28, n_act, 40) for k in range(16)]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 16)
    for k, sp in enumerate(sps):
        pool.load_synthetic(k, sp)
    e, g = pool.evaluate(list(range(16)), [sp.C for sp in sps])
    for k in (0, 7, 15):
        e2, g2, _, _ = evaluate(sps[k], topo, pairs=True)
        assert abs(e[k] - e2) <= E_TOL and np.abs(g[k] - g2).max() <= G_TOL
    pool.close()
    ctx.close()


def test_bits_do_not_depend_on_the_batch():
    """The products' tile form and every launch shape follow the batch, the sums do not."""
    topo = vb.Topology.build("COV", 10, 10, 1)
    sps = [vb.synthetic_problem(80 + k, 24, 10, 30) for k in range(2)]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 40)
    for k in range(40):
        pool.load_synthetic(k, sps[k % 2])
    e, g = pool.evaluate(list(range(40)), [sps[k % 2].C for k in range(40)])
    e1, g1 = pool.evaluate([0], [sps[0].C])
    assert all(np.array_equal(g[k], g[k % 2]) for k in range(40))
    assert abs(e[0] - e1[0]) <= 1e-12 and np.abs(g[0] - g1[0]).max() <= 1e-12
    pool.close()
    ctx.close()


@pytest.mark.parametrize("states", [((0, 1, 2),), ((1,),), ((0, 3), (0.75, 0.25))])
@pytest.mark.parametrize("kw,n_act,mult", [("COV", 8, 1), ("COV", 10, 1), ("COV", 10, 3)])
def test_selected_states(kw, n_act, mult, states):
    topo = vb.Topology.build(kw, n_act, n_act, mult)
    sp = vb.synthetic_problem(11, 26, n_act, 40)
    e, g, _, _ = evaluate(sp, topo, states=states)
    e2, g2, _, _ = evaluate(sp, topo, states=states, pairs=True)
    idx = states[0]
    w = np.array(states[1] if len(states) > 1 else [1.0 / len(idx)] * len(idx))
    ref = oracle.evaluate(26, 40, topo, sp.S, sp.h, sp.B, sp.C, states=idx, weights=w)
    assert abs(e - e2) <= E_TOL and abs(e - ref["energy"]) <= 1e-8
    assert np.abs(g - g2).max() <= G_TOL and np.abs(g - ref["grad"]).max() <= 1e-7
