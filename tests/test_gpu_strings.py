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
    """Two fragments without overlap: blocks of nullity 1 to 3, in more pairs than the string form lists: the slot
    takes the pair kernels."""
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


def test_equal_slots_of_a_batch_have_equal_bits():
    """(A slot alone and in a batch: bit for bit where the launch shape is pinned, test_gpu_determinism.py; otherwise
    the list kernels' and the lane kernels' sums follow the batch.)"""
    topo = vb.Topology.build("COV", 10, 10, 1)
    sps = [vb.synthetic_problem(80 + k, 24, 10, 30) for k in range(2)]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 40)
    for k in range(40):
        pool.load_synthetic(k, sps[k % 2])
    e, g = pool.evaluate(list(range(40)), [sps[k % 2].C for k in range(40)])
    assert all(e[k] == e[k % 2] and np.array_equal(g[k], g[k % 2]) for k in range(40))
    pool.close()
    ctx.close()


def nearly_singular_orbitals(sp, sigma):
    """Orbital 0 mixed with orbital 6 so that the block between the strings 0-5 and 2-7 has the smallest singular
    value sigma (the strings differ in two orbitals: the mixture that makes it singular is small)."""
    x, y = range(6), range(2, 8)

    def block(t):
        C = sp.C.copy()
        C[0] = C[0] + t * C[6]
        C /= np.sqrt(np.einsum("im,mn,in->i", C, sp.S, C))[:, None]
        return C, (C @ sp.S @ C.T)[np.ix_(x, y)]

    grid = np.linspace(-2.0, 2.0, 4001)
    det = np.array([np.linalg.det(block(t)[1]) for t in grid])
    roots = np.nonzero(det[:-1] * det[1:] < 0)[0]
    k = roots[np.argmin(np.abs(grid[roots]))]
    lo, hi = grid[k], grid[k + 1]
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        if np.linalg.det(block(mid)[1]) * det[k] > 0:
            lo = mid
        else:
            hi = mid
    step = 1e-3
    slope = np.linalg.svd(block(lo + step)[1], compute_uv=False)[-1] / step
    C, X = block(lo + sigma / slope)
    return C, np.linalg.svd(X, compute_uv=False)[-1]


@pytest.mark.parametrize("sigma", [1e-4, 1e-6, 1e-8, 1e-10, 1e-13])
def test_nearly_singular_blocks_agree_with_the_pair_kernels(sigma):
    """The inverse of such a block loses digits (at 1e-8 the pair kernels' gradient is off by 7e-8, at 1e-10 by 8e-4), so its
    pairs stay with the list kernels in both forms: the forms agree to 1e-9 of the gradient whatever the block."""
    topo = vb.Topology.build("COV", 12, 12, 1)
    sp = vb.synthetic_problem(9, 40, 12, 60)
    C, found = nearly_singular_orbitals(sp, sigma)
    assert found <= 3.0 * sigma + 1e-14
    e, g, s, _ = evaluate(sp, topo, C)
    e2, g2, s2, _ = evaluate(sp, topo, C, pairs=True)
    print(f"sigma {found:.2e} dE={abs(e - e2):.1e} dg={np.linalg.norm(g - g2) / np.linalg.norm(g2):.1e} singular {s} {s2}", flush=True)
    assert s == s2
    assert abs(e - e2) <= 1e-9 and np.linalg.norm(g - g2) <= 1e-9 * np.linalg.norm(g2)


@pytest.mark.parametrize("kw,n_act,mult,seed", [("COV", 11, 2, 8), ("COV", 12, 1, 8), ("COV", 13, 2, 5), ("FULL", 7, 2, 3)])
def test_forms_agree_on_random_orbitals(kw, n_act, mult, seed):
    topo = vb.Topology.build(kw, n_act, n_act, mult)
    for k in range(4):
        sp = vb.synthetic_problem(1000 * seed + k, 40, n_act, 60)
        C = sp.C.copy()
        C[:-1] += 0.3 * sp.C[1:]
        e, g, s, _ = evaluate(sp, topo, C)
        e2, g2, s2, _ = evaluate(sp, topo, C, pairs=True)
        print(f"dE={abs(e - e2):.1e} dg={np.linalg.norm(g - g2) / np.linalg.norm(g2):.1e} singular {s} {s2}", flush=True)
        assert s == s2
        assert abs(e - e2) <= 1e-9 and np.linalg.norm(g - g2) <= 1e-9 * np.linalg.norm(g2)


def test_small_problems_alone_follow_the_pair_kernels():
    """One problem of 252 determinants is faster on the pair kernels; an optimisation amplifies even the rounding
    between the forms (up to 730 times in five iterations), so its iterates are theirs to the last bit."""
    topo = vb.Topology.build("COV", 10, 10, 1)
    sp = vb.synthetic_problem(17, 40, 10, 60)
    runs = []
    for limit in (None, 9.9e4):
        ctx = vb.Context(0)
        if limit:
            ctx.set_pair_condition_limit(limit)
        prob = vb.Problem.from_synthetic(ctx, sp, topo)
        r = prob.optimize(sp.C, max_iterations=5)
        e, g = prob.evaluate(sp.C)
        runs.append((e, g, r["energy"], r["C"], r["grad"], r["trace"]))
        prob.close()
        ctx.close()
    assert all(np.array_equal(a, b) for a, b in zip(*runs))


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
