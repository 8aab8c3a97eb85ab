"""The string form (strings.hip) against the pair kernels and the FP64 oracle, through the C ABI.

A context with its own pair condition limit keeps the pair kernels, so the same problem evaluated with
the default limit and with another one compares the two forms. Each test asserts the form that ran."""
import math

import numpy as np
import pytest
import torch

import oracle
import xmvb_amd as vb

pytestmark = pytest.mark.gpu

E_TOL, G_TOL = 1e-8, 1e-7


STRING_WORK = 3.0e8  # the dispatch's line: n_det^2 (m_a m_b)^2 over the launch


def string_problems(topo):
    """The fewest problems per launch that the string form serves."""
    return math.ceil(STRING_WORK / (topo.n_determinants * topo.n_alpha * topo.n_beta) ** 2)


def evaluate(sp, topo, C=None, pairs=False, states=None):
    """(energy, gradient, singular pairs, intermediates, form) of one problem."""
    ctx = vb.Context(0)
    if pairs:
        ctx.set_pair_condition_limit(9.9e4)
    if states:
        ctx.set_states(*states)
    prob = vb.Problem.from_synthetic(ctx, sp, topo)
    e, g = prob.evaluate(sp.C if C is None else C)
    singular = prob.singular_pairs()
    mid = prob.intermediates()
    form = prob.string_form()
    prob.close()
    ctx.close()
    return e, g, singular, mid, form


def evaluate_in_strings(sp, topo, C, states=None):
    """(energy, gradient) of the problem in a launch of copies that takes the string form."""
    count = string_problems(topo)
    ctx = vb.Context(0)
    if states:
        ctx.set_states(*states)
    pool = vb.Pool(ctx, topo, count)
    for k in range(count):
        pool.load_synthetic(k, sp)
    e, g = pool.evaluate(list(range(count)), [C] * count)
    assert pool.string_form()[0] == count
    assert all(e[k] == e[0] and np.array_equal(g[k], g[0]) for k in range(count))
    pool.close()
    ctx.close()
    return e[0], g[0]


@pytest.mark.parametrize("kw,n_act,n_el,mult", [
    ("COV", 9, 9, 2), ("COV", 10, 10, 1), ("COV", 10, 10, 3), ("COV", 11, 11, 2), ("COV", 12, 12, 1), ("COV", 13, 13, 2),
    ("FULL", 6, 6, 1), ("FULL", 7, 7, 2),  # many determinants per string, equal and unequal spins
    ("COV,ION(1)", 8, 8, 1),    # spin-flip couples and doubly occupied orbitals
    ("COV", 8, 6, 1), ("COV", 10, 4, 1),  # empty orbitals
    ("COV", 10, 4, 3),          # one beta electron: no double replacements
    ("COV", 7, 9, 2),           # more electrons than orbitals
])
def test_string_form_matches_pair_kernels(kw, n_act, n_el, mult):
    topo = vb.Topology.build(kw, n_act, n_el, mult)
    print(f"case strings {kw} n_act={n_act} n_el={n_el} mult={mult} n_det={topo.n_determinants} x {string_problems(topo)}", flush=True)
    sp = vb.synthetic_problem(31 + n_act, 30, n_act, 45)
    C = sp.C.copy()
    C[:-1] += 0.4 * sp.C[1:]
    e, g = evaluate_in_strings(sp, topo, C)
    e2, g2, _, _, form = evaluate(sp, topo, C, pairs=True)
    assert form == (0, 0)
    print(f"dE={abs(e - e2):.2e} dg={np.abs(g - g2).max():.2e}", flush=True)
    assert abs(e - e2) <= E_TOL
    assert np.abs(g - g2).max() <= G_TOL


def test_structure_matrices_and_counts_match():
    topo = vb.Topology.build("COV", 12, 12, 1)
    sp = vb.synthetic_problem(43, 30, 12, 45)
    e, g, s, mid, form = evaluate(sp, topo)
    e2, g2, s2, mid2, form2 = evaluate(sp, topo, pairs=True)
    assert form[0] == 1 and form2 == (0, 0)
    assert s == s2
    for k in ("H", "S"):
        assert np.abs(mid[k] - mid2[k]).max() <= 1e-10 * np.abs(mid2[k]).max()


def orthogonal_orbital(sp):
    """Orbital 11 made orthogonal to 0-5: every block between the string 0-5 and one with 11 has a zero row."""
    C = sp.C.copy()
    P = C[:6]
    C[11] -= (C[11] @ sp.S @ P.T) @ np.linalg.solve(P @ sp.S @ P.T, P)
    return C


def test_slots_with_many_rank_deficient_blocks_take_the_pair_kernels():
    topo = vb.Topology.build("COV", 12, 12, 1)
    sp = vb.synthetic_problem(5, 24, 12, 40)
    C = orthogonal_orbital(sp)
    e, g, s, _, form = evaluate(sp, topo, C)
    ref = oracle.evaluate(24, 40, topo, sp.S, sp.h, sp.B, C)
    print(f"singular {s} dE={abs(e - ref['energy']):.2e} dg={np.abs(g - ref['grad']).max():.2e}", flush=True)
    assert form == (0, 0) and s > 256
    assert abs(e - ref["energy"]) <= 1e-8 and np.abs(g - ref["grad"]).max() <= 1e-7


def test_ill_conditioned_orbitals_keep_the_pair_kernels_in_a_mixed_launch():
    """One launch of nine slots: well separated orbitals (string form) around slots whose first
    two orbitals nearly coincide (|S_act^-1| far above the limit)."""
    topo = vb.Topology.build("COV", 10, 10, 1)
    sps = [vb.synthetic_problem(60 + k, 32, 10, 48) for k in range(3)]
    C = [sp.C.copy() for sp in sps]
    C[1][1] = C[1][0] + 0.05 * C[1][1]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, 9)
    for k in range(9):
        pool.load_synthetic(k, sps[k % 3])
    e, g = pool.evaluate(list(range(9)), [C[k % 3] for k in range(9)])
    assert pool.string_form()[0] == 6
    for k in range(9):
        sp = sps[k % 3]
        ref = oracle.evaluate(32, 48, topo, sp.S, sp.h, sp.B, C[k % 3])
        print(f"slot {k} dE={abs(e[k] - ref['energy']):.2e} dg={np.abs(g[k] - ref['grad']).max():.2e}", flush=True)
        assert abs(e[k] - ref["energy"]) <= 1e-8
        assert np.abs(g[k] - ref["grad"]).max() <= (1e-6 if k % 3 == 1 else 1e-7)
    pool.close()
    ctx.close()


class Waited:
    """One 12-orbital problem through every way to evaluate it: each launch takes the kernels that the launches before
    needed and is repeated where its slots needed the others."""

    def __init__(self, call):
        self.topo = vb.Topology.build("COV", 12, 12, 1)
        self.sp = vb.synthetic_problem(77, 30, 12, 45)
        self.call = call
        self.ctx = vb.Context(0)
        if call in ("pool", "submit", "scheduler"):
            self.pool = vb.Pool(self.ctx, self.topo, 1)
            self.pool.load_synthetic(0, self.sp)
        else:
            self.prob = vb.Problem.from_synthetic(self.ctx, self.sp, self.topo)

    def __call__(self, C):
        if self.call == "evaluate":
            return *self.prob.evaluate(C), self.prob.string_form()[0]
        if self.call == "two_phase":
            e = self.prob.evaluate_forward(C)
            return e, self.prob.complete_gradient(), self.prob.string_form()[0]
        if self.call == "submit":  # the repetition happens at the poll or at the wait
            ticket = self.pool.submit([0], [C])
            self.polled = not getattr(self, "polled", False)
            while self.polled and not self.pool.poll(ticket):
                pass
            e, g = self.pool.wait(ticket)
            return e[0], g[0], self.pool.string_form()[0]
        if self.call == "scheduler":
            g = np.full(C.shape, np.nan)
            sched = vb.Scheduler(self.ctx)
            sched.submit(self.pool, 0, C, g)
            done = []
            while not done:
                done = sched.collect(wait_us=100000)
            sched.close()
            return done[0]["energy"], g, self.pool.string_form()[0]
        c = torch.from_numpy(np.ascontiguousarray(C)).to("cuda:0")
        g = torch.full_like(c, float("nan"))
        torch.cuda.synchronize()
        if self.call == "pool":
            e = self.pool.evaluate_device([0], c.data_ptr(), g.data_ptr())[0]
            form = self.pool.string_form()[0]
        else:
            call = self.prob.evaluate_device_noalloc if self.call == "noalloc" else self.prob.evaluate_device
            e = call(c.data_ptr(), g.data_ptr())
            form = self.prob.string_form()[0]
        return e, g.cpu().numpy().reshape(C.shape), form

    def close(self):
        (self.pool if hasattr(self, "pool") else self.prob).close()
        self.ctx.close()


@pytest.mark.parametrize("call", ["evaluate", "two_phase", "device", "noalloc", "pool", "submit", "scheduler"])
@pytest.mark.parametrize("order", ["ggi", "ggrg", "gggnig", "iiiiiiggi", "rrrrrgg"])
def test_launches_repeat_with_the_kernels_they_lack(call, order):
    """g: well separated orbitals (string form, after two of them alone); i: ill-conditioned S_act; r: too many rank
    deficient blocks; n: a nearly singular block (listed pairs). Five
    launches without a string slot leave the string kernels out until one has one."""
    w = Waited(call)
    C = {"g": w.sp.C, "i": w.sp.C.copy(), "r": orthogonal_orbital(w.sp), "n": nearly_singular_orbitals(w.sp, 1e-8)[0]}
    C["i"][1] = C["i"][0] + 0.05 * C["i"][1]
    ref = {k: evaluate(w.sp, w.topo, C[k], pairs=True)[:2] for k in set(order)}
    for at, k in enumerate(order):
        print(f"{call} {order} {at} {k}", flush=True)
        e, g, form = w(C[k])
        assert form == (1 if k in "gn" else 0)
        assert abs(e - ref[k][0]) <= 1e-9
        assert np.linalg.norm(g - ref[k][1]) <= 1e-9 * np.linalg.norm(ref[k][1])
    w.close()


@pytest.mark.parametrize("target,form", [(15.0, 1), (17.0, 0)])
def test_conditioning_of_the_active_overlap_near_the_limit(target, form):
    """Orbital 1 drawn towards orbital 0 until max|S_act^-1| is just below and above the limit of 16."""
    topo = vb.Topology.build("COV", 12, 12, 1)
    sp = vb.synthetic_problem(21, 36, 12, 50)

    def orbitals(t):
        C = sp.C.copy()
        C[1] = t * C[0] + (1.0 - t) * C[1]
        C /= np.sqrt(np.einsum("im,mn,in->i", C, sp.S, C))[:, None]
        return C, np.abs(np.linalg.inv(C @ sp.S @ C.T)).max()

    lo, hi = 0.0, 0.99
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if orbitals(mid)[1] < target else (lo, mid)
    C = orbitals(lo)[0]
    e, g, _, _, got = evaluate(sp, topo, C)
    e2, g2, _, _, _ = evaluate(sp, topo, C, pairs=True)
    print(f"limit {target} dE={abs(e - e2):.1e} dg={np.linalg.norm(g - g2) / np.linalg.norm(g2):.1e} listed {got[1]}", flush=True)
    assert got[0] == form
    assert abs(e - e2) <= 1e-9 and np.linalg.norm(g - g2) <= 1e-9 * np.linalg.norm(g2)


@pytest.mark.parametrize("n_act,mult", [(9, 2), (10, 1)])
def test_forms_agree_at_the_batch_size_that_changes_them(n_act, mult):
    topo = vb.Topology.build("COV", n_act, n_act, mult)
    count = string_problems(topo)
    sps = [vb.synthetic_problem(90 + k, 28, n_act, 40) for k in range(4)]
    ctx = vb.Context(0)
    pool = vb.Pool(ctx, topo, count)
    for k in range(count):
        pool.load_synthetic(k, sps[k % 4])
    e, g = pool.evaluate(list(range(count)), [sps[k % 4].C for k in range(count)])
    assert pool.string_form()[0] == count
    e2, g2 = pool.evaluate(list(range(count - 1)), [sps[k % 4].C for k in range(count - 1)])
    assert pool.string_form()[0] == 0
    for k in range(4):
        assert abs(e[k] - e2[k]) <= 1e-9 and np.linalg.norm(g[k] - g2[k]) <= 1e-9 * np.linalg.norm(g2[k])
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
    e, g, s, _, form = evaluate(sp, topo, C)
    e2, g2, s2, _, _ = evaluate(sp, topo, C, pairs=True)
    assert form[0] == 1 and form[1] > 0
    print(f"listed {form[1]} sigma {found:.2e} dE={abs(e - e2):.1e} dg={np.linalg.norm(g - g2) / np.linalg.norm(g2):.1e} singular {s} {s2}", flush=True)
    assert s == s2
    assert abs(e - e2) <= 1e-9 and np.linalg.norm(g - g2) <= 1e-9 * np.linalg.norm(g2)


@pytest.mark.parametrize("n_act,mult,seed", [(12, 1, 8), (13, 2, 5)])
def test_forms_agree_on_random_orbitals(n_act, mult, seed):
    topo = vb.Topology.build("COV", n_act, n_act, mult)
    for k in range(4):
        sp = vb.synthetic_problem(1000 * seed + k, 40, n_act, 60)
        C = sp.C.copy()
        C[:-1] += 0.3 * sp.C[1:]
        e, g, s, _, form = evaluate(sp, topo, C)
        e2, g2, s2, _, _ = evaluate(sp, topo, C, pairs=True)
        print(f"dE={abs(e - e2):.1e} dg={np.linalg.norm(g - g2) / np.linalg.norm(g2):.1e} singular {s} {s2} listed {form[1]}", flush=True)
        assert form[0] == 1 and s == s2
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
@pytest.mark.parametrize("kw,n_act,mult", [("COV", 10, 1), ("COV", 10, 3)])
def test_selected_states(kw, n_act, mult, states):
    topo = vb.Topology.build(kw, n_act, n_act, mult)
    sp = vb.synthetic_problem(11, 26, n_act, 40)
    e, g = evaluate_in_strings(sp, topo, sp.C, states)
    e2, g2, _, _, _ = evaluate(sp, topo, states=states, pairs=True)
    idx = states[0]
    w = np.array(states[1] if len(states) > 1 else [1.0 / len(idx)] * len(idx))
    ref = oracle.evaluate(26, 40, topo, sp.S, sp.h, sp.B, sp.C, states=idx, weights=w)
    assert abs(e - e2) <= E_TOL and abs(e - ref["energy"]) <= 1e-8
    assert np.abs(g - g2).max() <= G_TOL and np.abs(g - ref["grad"]).max() <= 1e-7


def test_string_arrays_give_way_to_slots():
    """Two slots of 12 orbitals (24 MB of string arrays each) under budgets that leave out the arrays of one and of both:
    the slots load as they would without the string form, and the pair kernels serve what has none."""
    topo = vb.Topology.build("COV", 12, 12, 1)
    sps = [vb.synthetic_problem(70 + k, 30, 12, 45) for k in range(2)]

    def run(budget):
        ctx = vb.Context(0, budget)
        pool = vb.Pool(ctx, topo, 2)
        for k, sp in enumerate(sps):
            pool.load_synthetic(k, sp)
        used = ctx.memory()[0]
        assert used == pool.device_bytes()
        forms, values = [], []
        for k, sp in enumerate(sps):
            e, g = pool.evaluate([k], [sp.C])
            values.append((e[0], g[0]))
            forms.append(pool.string_form()[0])
        pool.close()
        ctx.close()
        return used, forms, values

    full, forms, ref = run(0)
    assert forms == [1, 1]
    slack = 4 << 20  # staging of the evaluations
    one, forms, values = run(full - 1)
    arrays = full - one
    assert arrays > 4 * slack and forms == [1, 0]
    for budget, want in ((full - arrays + slack, [1, 0]), (full - 2 * arrays + slack, [0, 0])):
        used, forms, got = run(budget)
        assert used <= budget and forms == want
        values += got
    for at, (e, g) in enumerate(values):
        assert abs(e - ref[at % 2][0]) <= 1e-9
        assert np.linalg.norm(g - ref[at % 2][1]) <= 1e-9 * np.linalg.norm(ref[at % 2][1])
