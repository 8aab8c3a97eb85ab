"""Timed cases of the VBSCF energy+gradient engine.

Each case is one call that a program makes through the public entry points of `xmvb_amd`: a single
evaluation with host orbitals, the two-phase line-search contract, a batch over resident pool slots
(device or host orbitals), or a short P-LBFGS run. Inputs follow the recipe of the package's
synthetic problems (overlap I + 0.1 A A^T / n, random core Hamiltonian and RI factors, random
orbitals), with neighbouring orbitals mixed by `mix`, since the orbitals of bonded centres overlap.
"""
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xmvb-cpp_amd"))
import xmvb_amd as vb  # noqa: E402

DISTINCT = 8  # distinct molecules of a pool; further slots are other orbitals of the same molecules


def _case(kind, n_act, n_bf, n_aux, count=1, structures="COV", mult=1, mix=0.0, split=False, n_bf_min=0, ri=0,
          states=1, eigensolver=0, iterations=0):
    """kind: evaluate | two_phase | pool_device | pool_host | optimize. Pools with n_bf_min spread their
    slots' n_bf over [n_bf_min, n_bf] with n_aux = 3 n_bf. split: each orbital is expanded on its own
    share of the basis only (support masks)."""
    return dict(kind=kind, n_act=n_act, n_bf=n_bf, n_aux=n_aux, count=count, structures=structures, mult=mult, mix=mix,
                split=split, n_bf_min=n_bf_min, ri=ri, states=states, eigensolver=eigensolver, iterations=iterations)


def listed():
    cases = [
        # the two-orbital deck (H2 in a 10-function basis, one orbital per atom): smallest call there is
        ("h2_deck_single", _case("evaluate", 2, 10, 54, structures="FULL", split=True)),
        # a small molecule evaluated alone: launch latency
        ("cov4_single", _case("evaluate", 4, 46, 138, mix=0.5)),
        # a covalent + ionic set (175 structures, 400 determinants): the eigensolver beyond one wavefront
        ("full6_single", _case("evaluate", 6, 61, 183, structures="FULL", mix=0.4)),
        # one served launch: a scan of a small molecule, host orbitals in, gradients out
        ("cov6_scan64", _case("pool_host", 6, 83, 249, count=64, mix=0.5)),
        # many resident problems of uneven size, compensated FP32 RI factors
        ("cov8_ragged96_fp32c", _case("pool_host", 8, 200, 600, count=96, mix=0.3, n_bf_min=40, ri=2)),
        # open shell (no spin-flip partners), a line-search trial and the gradient at the accepted point
        ("doublet9_two_phase", _case("two_phase", 9, 97, 291, mult=2, mix=0.4)),
        # the medium problem alone, as an outside optimiser calls it
        ("cov10_single", _case("evaluate", 10, 120, 360, mix=0.5)),
        # the average of three states
        ("cov10_three_states", _case("evaluate", 10, 151, 453, states=3)),
        # the medium problem on the device optimiser, its first iterations
        ("cov10_optimize", _case("optimize", 10, 120, 360, iterations=5)),
        # the headline: a resident batch of medium problems, orbitals and gradients in device memory
        ("cov10_batch192", _case("pool_device", 10, 120, 360, count=192)),
        # uneven 12-orbital problems, host orbitals in, gradients out
        ("cov12_ragged32", _case("pool_host", 12, 200, 600, count=32, mix=0.3, n_bf_min=40)),
        # the large single problem: 429 structures, 3432 determinants
        ("cov14_single", _case("evaluate", 14, 400, 1200)),
    ]
    return [dict(name=name, **c) for name, c in cases]


def draw(rng):
    kind = rng.choice(["evaluate", "evaluate", "two_phase", "pool_device", "pool_host", "pool_host"])
    mix = rng.uniform(0.0, 0.6)
    if kind in ("evaluate", "two_phase"):
        n_act = rng.choice([2, 3, 4, 5, 6, 7, 8, 9, 10, 10, 11, 12, 13])
        mult = 1 if n_act % 2 == 0 else 2
        if n_act >= 4 and n_act % 2 == 0 and n_act <= 10 and rng.random() < 0.25:
            mult = 3
        n_bf = round(math.exp(rng.uniform(math.log(max(12, 3 * n_act)), math.log(300))))
        full = n_act <= 6 and mult < 3 and rng.random() < 0.4
        states = 2 if kind == "evaluate" and n_act >= 6 and rng.random() < 0.2 else 1
        return _case(kind, n_act, n_bf, n_bf * rng.choice([2, 3, 4]), structures="FULL" if full else "COV", mult=mult,
                     mix=mix, split=n_act <= 4 and rng.random() < 0.3, states=states,
                     eigensolver=1 if states == 1 and n_act >= 8 and rng.random() < 0.15 else 0)
    n_act = rng.choice([4, 6, 7, 8, 9, 10, 10, 12])
    mult = 1 if n_act % 2 == 0 else 2
    n_bf = rng.randint(40, 200)
    most = {4: 256, 6: 256, 7: 192, 8: 192, 9: 128, 10: 128, 12: 32}[n_act]
    count = round(math.exp(rng.uniform(math.log(2), math.log(most))))
    ragged = kind == "pool_host" and rng.random() < 0.6
    return _case(kind, n_act, n_bf, 3 * n_bf, count=count, mult=mult, mix=mix, n_bf_min=40 if ragged else 0,
                 ri=rng.choice([0, 0, 2]))


# ---- inputs -------------------------------------------------------------------------------------

def _molecule(rng, n_bf, n_aux):
    a = rng.standard_normal((n_bf, n_bf))
    S = np.eye(n_bf) + (0.1 / n_bf) * (a @ a.T)
    h = rng.standard_normal((n_bf, n_bf)) * math.sqrt(0.5)
    h = 0.5 * (h + h.T) - 2.0 * np.eye(n_bf)
    B = rng.standard_normal((n_bf * (n_bf + 1) // 2, n_aux))  # packed pair hi(hi+1)/2 + lo, auxiliary index fastest
    B *= math.sqrt(0.5 / n_bf)
    B[[i * (i + 3) // 2 for i in range(n_bf)]] *= math.sqrt(2.0)
    return dict(n_bf=n_bf, n_aux=n_aux, S=S, h=h, B=B)


def _orbitals(rng, case, n_bf):
    n = case["n_act"]
    C = rng.standard_normal((n, n_bf)) / math.sqrt(n_bf)
    C = C + case["mix"] * np.vstack([C[1:], np.zeros((1, n_bf))])
    if case["split"]:
        C = C * _support(case, n_bf)
    return np.ascontiguousarray(C)


def _support(case, n_bf):
    return (np.arange(n_bf)[None, :] * case["n_act"] // n_bf == np.arange(case["n_act"])[:, None]).astype(np.uint8)


def _inputs(case, seed):
    """(molecules, molecule of each slot, orbitals of each slot)."""
    rng = np.random.default_rng(seed)
    kinds = min(case["count"], DISTINCT)
    if case["n_bf_min"]:
        sizes = [int(x) for x in np.linspace(case["n_bf_min"], case["n_bf"], kinds).round()]
        mols = [_molecule(rng, n, 3 * n) for n in sizes]
    else:
        mols = [_molecule(rng, case["n_bf"], case["n_aux"]) for _ in range(kinds)]
    which = [int(k) for k in rng.permutation(case["count"]) % kinds]
    return mols, which, [_orbitals(rng, case, mols[k]["n_bf"]) for k in which]


# ---- one pass -----------------------------------------------------------------------------------

def prepare(case, seed):
    mols, which, orbitals = _inputs(case, seed)
    ctx = vb.Context(0)
    if case["ri"]:
        ctx.set_ri_precision(case["ri"])
    if case["eigensolver"]:
        ctx.set_eigensolver(case["eigensolver"])
    if case["states"] > 1:
        ctx.set_states(tuple(range(case["states"])))
    topo = vb.Topology.build(case["structures"], case["n_act"], case["n_act"], case["mult"])
    state = dict(kind=case["kind"], ctx=ctx, iterations=case["iterations"], support=None)
    if case["kind"] in ("evaluate", "two_phase", "optimize"):
        m = mols[0]
        state["problem"] = vb.Problem(ctx, m["n_bf"], m["n_aux"], topo, m["S"], m["h"], m["B"])
        state["C"] = orbitals[0]
        if case["split"]:
            state["support"] = _support(case, m["n_bf"])
        return state
    pool = vb.Pool(ctx, topo, case["count"])
    for slot, k in enumerate(which):
        m = mols[k]
        pool.load(slot, m["n_bf"], m["n_aux"], m["S"], m["h"], m["B"])
    state.update(pool=pool, slots=list(range(case["count"])))
    if case["kind"] == "pool_device":
        state["C"] = torch.from_numpy(np.concatenate([c.ravel() for c in orbitals])).to("cuda:0")
        state["grad"] = torch.zeros_like(state["C"])
        torch.cuda.synchronize()  # the engine's own streams read C
    else:
        state["C"] = orbitals
    return state


def run(state):
    kind = state["kind"]
    if kind == "evaluate":
        return state["problem"].evaluate(state["C"], state["support"])
    if kind == "two_phase":
        energy = state["problem"].evaluate_forward(state["C"], state["support"])
        return energy, state["problem"].complete_gradient()
    if kind == "optimize":
        r = state["problem"].optimize(state["C"], max_iterations=state["iterations"])
        return r["energy"], r["gradient_norm"], r["C"], r["grad"], r["trace"]
    if kind == "pool_device":
        energies = state["pool"].evaluate_device(state["slots"], state["C"].data_ptr(), state["grad"].data_ptr())
        return energies, state["grad"]
    energies, grads = state["pool"].evaluate(state["slots"], state["C"])
    return energies, np.concatenate([g.ravel() for g in grads])


# ---- what a pass cannot do without ----------------------------------------------------------------

def _spins(case):
    beta = (case["n_act"] - case["mult"] + 1) // 2
    return case["n_act"] - beta, beta


def _n_determinants(case):
    n = case["n_act"]
    ma, mb = _spins(case)
    return math.comb(n, ma) * (math.comb(n, mb) if case["structures"] == "FULL" else 1)


def work(case):
    """Bytes: S, h, the RI factors and the orbitals read once, the gradient written once. Flops: the
    one-index transform and the pair factors of the RI integrals, the packed kernel, and the
    m_a^2 m_b^2 opposite-spin products of every unordered determinant pair."""
    n, (ma, mb), nd = case["n_act"], _spins(case), _n_determinants(case)
    kinds = min(case["count"], DISTINCT)
    sizes = [(int(x), 3 * int(x)) for x in np.linspace(case["n_bf_min"], case["n_bf"], kinds).round()] \
        if case["n_bf_min"] else [(case["n_bf"], case["n_aux"])]
    bytes_, flops = 0.0, 0.0
    for nbf, naux in sizes:
        npair, np_ = nbf * (nbf + 1) // 2, n * (n + 1) // 2
        bytes_ += naux * npair * (5 if case["ri"] == 2 else 8) + 2 * 8 * nbf * nbf + 2 * 8 * n * nbf
        flops += 2.0 * naux * nbf * nbf * n + 2.0 * naux * nbf * np_ + naux * np_ * (np_ + 1)
        flops += 2.0 * (ma * mb) ** 2 * nd * (nd + 1) / 2
    calls = case["count"] / len(sizes) * max(1, case["iterations"] + 1)
    return {"bytes": bytes_ * calls, "flops": flops * calls}


# ---- the same in plain torch, 64 bits -------------------------------------------------------------

def _matchings(open_orbitals, n_open):
    """Non-crossing pairings of open_orbitals that leave n_open unpaired, none of them under an arc."""
    if not open_orbitals:
        return [[]] if n_open == 0 else []
    first, rest = open_orbitals[0], open_orbitals[1:]
    out = [m for m in _matchings(rest, n_open - 1)] if n_open > 0 else []
    for k in range(0, len(rest), 2):
        for inside in _matchings(rest[:k], 0):
            for outside in _matchings(rest[k + 1:], n_open):
                out.append([(first, rest[k])] + inside + outside)
    return out


def _sign(creators):
    """Parity of sorting the creators (spin, orbital): alpha before beta, orbitals ascending."""
    inversions = sum(a > b for a, b in itertools.combinations(creators, 2))
    return -1.0 if inversions % 2 else 1.0


def _structure_space(n, mult, full):
    """Determinants (alpha tuple, beta tuple) and T (n_det x n_str), a basis of the structure space."""
    open_spin = mult - 1
    columns, index = [], {}
    for doubly in range(0, (n - open_spin) // 2 + 1 if full else 1):
        for occ2 in itertools.combinations(range(n), doubly):
            left = [p for p in range(n) if p not in occ2]
            for singly in itertools.combinations(left, n - 2 * doubly):
                for bonds in _matchings(list(singly), open_spin):
                    bonded = {p for bond in bonds for p in bond}
                    column = {}
                    for flips in itertools.product((0, 1), repeat=len(bonds)):
                        creators = [c for p in occ2 for c in ((0, p), (1, p))]
                        for (i, j), f in zip(bonds, flips):
                            creators += [(0, j), (1, i)] if f else [(0, i), (1, j)]
                        creators += [(0, p) for p in singly if p not in bonded]
                        det = (tuple(sorted(p for s, p in creators if s == 0)),
                               tuple(sorted(p for s, p in creators if s == 1)))
                        at = index.setdefault(det, len(index))
                        column[at] = column.get(at, 0.0) + _sign(creators)
                    columns.append(column)
    T = np.zeros((len(index), len(columns)))
    for s, column in enumerate(columns):
        for at, v in column.items():
            T[at, s] = v
    return list(index), T


def _pair_values(S, h, g, rows, cols, dets):
    """H and S between determinants rows[k] and cols[k]: transition densities from the inverse overlap blocks."""
    n = S.shape[0]
    det, dens = 1.0, []
    for occ in dets:
        if occ.shape[1] == 0:
            dens.append(torch.zeros(len(rows), n * n, dtype=S.dtype, device=S.device))
            continue
        R, L = occ[rows], occ[cols]
        X = S[R[:, :, None], L[:, None, :]]
        det = det * torch.linalg.det(X)
        at = (R[:, :, None] * n + L[:, None, :]).reshape(len(rows), -1)
        D = torch.linalg.inv(X).transpose(1, 2).reshape(len(rows), -1)
        dens.append(torch.zeros(len(rows), n * n, dtype=S.dtype, device=S.device).scatter(1, at, D))
    G, A = g.reshape(n * n, n * n), (g - g.permute(0, 3, 2, 1)).reshape(n * n, n * n)
    phi = (dens[0] + dens[1]) @ h.reshape(-1) + ((dens[0] @ G) * dens[1]).sum(1)
    for D in dens:
        phi = phi + 0.5 * ((D @ A) * D).sum(1)
    return det * phi, det * torch.ones_like(phi)


def _strings(n, m):
    strings = list(itertools.combinations(range(n), m))
    return strings, {s: i for i, s in enumerate(strings)}


def _minors(R, m):
    """All m x m minors of R, by expansion along the first row."""
    n, M = R.shape[0], torch.ones(1, 1, dtype=R.dtype, device=R.device)
    for k in range(1, m + 1):
        strings, _ = _strings(n, k)
        _, below = _strings(n, k - 1)
        first, rest = [s[0] for s in strings], [below[s[1:]] for s in strings]
        out = 0.0
        for j in range(k):
            col, others = [s[j] for s in strings], [below[s[:j] + s[j + 1:]] for s in strings]
            out = out + (-1) ** j * R[first][:, col] * M[rest][:, others]
        M = out
    return M


def _replacements(n, m, dev):
    """(p, q) -> (string with q in place of p or -, sign) of every m-string, q == p included."""
    strings, index = _strings(n, m)
    source, sign = np.zeros((n, n, len(strings)), np.int64), np.zeros((n, n, len(strings)))
    for i, s in enumerate(strings):
        for p in s:
            for q in range(n):
                if q == p or q not in s:
                    left = [x for x in s if x != p]
                    at = sum(x < q for x in left)
                    source[p, q, i] = index[tuple(left[:at] + [q] + left[at:])]
                    sign[p, q, i] = (-1.0) ** (s.index(p) + at)
    return torch.from_numpy(source).to(dev), torch.from_numpy(sign).to(dev)


def _energy_of(S, h, L, dets, a, n, spins):
    """<v|H|v> and <v|v> of v = sum_d a_d |d>, expanded over the determinants of orthonormal orbitals
    (S = R^T R); no overlap block is inverted, so its derivative keeps its digits at any block."""
    R = torch.linalg.cholesky(S).T
    Ri = torch.linalg.inv(R)
    h, L = Ri.T @ h @ Ri, torch.einsum("pi,pqA,qj->ijA", Ri, L, Ri).reshape(n * n, -1)
    g = (L @ L.T).reshape(n, n, n, n)
    index = [_strings(n, m)[1] for m in spins]
    at = [torch.tensor([index[s][d[s]] for d in dets], device=S.device) for s in (0, 1)]
    M = [_minors(R, m) for m in spins]
    C = torch.zeros(len(index[0]), len(index[1]), dtype=S.dtype, device=S.device).index_put(tuple(at), a)
    v = M[0] @ C @ M[1].T
    (ra, sa), (rb, sb) = (_replacements(n, m, S.device) for m in spins)
    D = torch.stack([sa[p, q][:, None] * v[ra[p, q]] + sb[p, q] * v[:, rb[p, q]] for p in range(n) for q in range(n)])
    D = D.reshape(n * n, -1)
    P = (D @ D.T).reshape(n, n, n, n)
    one = h - 0.5 * torch.einsum("pqqs->ps", g)
    H = ((D @ v.reshape(-1)).reshape(n, n) * one).sum() + 0.5 * (g.transpose(0, 1) * P).sum()
    return H, (v * v).sum()


def _evaluate_exact(case, mol, C, dets, T):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    n, nbf = case["n_act"], mol["n_bf"]
    S_ao, h_ao = (torch.from_numpy(mol[k]).to(dev) for k in ("S", "h"))
    B = mol.setdefault("on_device", torch.from_numpy(mol["B"]).to(dev))
    hi, lo = (torch.from_numpy(x).to(dev) for x in np.tril_indices(nbf))
    raw = torch.from_numpy(C).to(dev).requires_grad_(True)
    mask = torch.from_numpy(_support(case, nbf)).to(dev) if case["split"] else 1.0
    c = raw * mask
    c = c / torch.sqrt(((c @ S_ao) * c).sum(1, keepdim=True))
    S, h = c @ S_ao @ c.T, c @ h_ao @ c.T
    off = (hi != lo).to(S.dtype)
    half = []
    for p in range(n):  # L[p, q, A] = sum c_p(mu) c_q(nu) B[mu nu, A] over the packed pairs
        w = torch.stack([c[p][hi] * c[q][lo] + off * c[p][lo] * c[q][hi] for q in range(n)])
        half.append(w @ B)
    L = torch.stack(half).reshape(n * n, -1)
    g = (L @ L.T).reshape(n, n, n, n)

    occ = [torch.tensor([d[s] for d in dets], device=dev).reshape(len(dets), -1) for s in (0, 1)]
    nd = len(dets)
    rows, cols = (torch.from_numpy(x).to(dev) for x in np.tril_indices(nd))
    step = max(1, 2 ** 25 // (n * n))
    Hd, Sd = (torch.zeros(nd, nd, dtype=S.dtype, device=dev) for _ in range(2))
    with torch.no_grad():
        for k in range(0, len(rows), step):
            r, q = rows[k:k + step], cols[k:k + step]
            H_rq, S_rq = _pair_values(S, h, g, r, q, occ)
            Hd[r, q], Hd[q, r], Sd[r, q], Sd[q, r] = H_rq, H_rq, S_rq, S_rq
        Td = torch.from_numpy(T).to(dev)
        Hs, Ss = (Td.T @ M @ Td for M in (Hd, Sd))
        Li = torch.linalg.inv(torch.linalg.cholesky(Ss.cpu()))
        lam, U = torch.linalg.eigh(Li @ Hs.cpu() @ Li.T)
        ns = case["states"]
        a = Td @ (Li.T @ U[:, :ns]).to(dev)
        lam = lam[:ns].to(dev)
        energy = float(lam.mean())
    spins = _spins(case)
    total = 0.0
    for k in range(ns):
        H, norm = _energy_of(S, h, L.reshape(n, n, -1), dets, a[:, k], n, spins)
        total = total + (H - lam[k] * norm) / ns
    total.backward()
    return energy, raw.grad.cpu().numpy()


def exact(case, seed):
    if case["kind"] == "optimize":
        return None  # its iterates are the algorithm's own; the evaluations in them are the other cases'
    if case["eigensolver"] == 1:
        return None  # converged to the caller's tolerance, not to the root of 64-bit arithmetic
    mols, which, orbitals = _inputs(case, seed)
    dets, T = _structure_space(case["n_act"], case["mult"], case["structures"] == "FULL")
    out = [_evaluate_exact(case, mols[k], C, dets, T) for k, C in zip(which, orbitals)]
    if case["kind"] in ("evaluate", "two_phase"):
        return out[0]
    grads = np.concatenate([g.ravel() for _, g in out])
    return np.array([e for e, _ in out]), torch.from_numpy(grads) if case["kind"] == "pool_device" else grads
