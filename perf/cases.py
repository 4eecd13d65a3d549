"""The performance cases of the HEOM solver: what a user's program has it compute.

Every case builds its hierarchy (ADO tuples and edges), site Hamiltonian and bath
prefactors here from a seed, hands them to heom_amd.Handle as a caller with instance
arrays of its own does, and runs one pass through the handle's public methods.  `exact`
evaluates the same equations in 64 bits with plain torch.

Kinds of cases (the "kind" entry) and what a pass is:

* propagate  RK4 population dynamics, populations observed on the device, and at the end
             the norm of every ADO (the reference's hierarchy_norm observation, by which a
             user judges the depth);
* ensemble   a static-disorder ensemble in one batch: per realisation a population
             hierarchy and three absorption hierarchies (dipole tensor components) with
             the ground state; reset, then populations and absorption traces;
* tss        iterations of the thermal state search, the top read back between blocks,
             and the ADO norms of the result;
* adjoint    a fit's gradient: forward sweep with observations, backward sweep;
* field      a run resumed from a checkpoint under a time-dependent field: the state goes
             up, the tops of every step, the state and the ADO norms come back.
"""
from __future__ import annotations

import functools
import itertools
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "dm-heom_amd"))
import heom_amd  # noqa: E402

HBAR = 1.05457148e-34  # J s, the solver's value
K_B = 1.3806504e-23    # J / K
INVCM = 1.98644543e-23  # J per cm^-1
FS = 1e-15
LLC_BYTES = 256 << 20  # last-level cache of the card


# ---- cases ---------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: seven sites, one mode each, depth 3 (120 ADOs), a first look
        # at a system; launches and their latency are what it costs
        dict(name="pop_7s7m_d3", kind="propagate", sites=7, modes_per_site=1, depth=3, precision="fp64",
             complex_h=False, graphs=False, steps=100, observe=10),
        # a dimer with three modes per site and a deep hierarchy (5,005 ADOs of 2 x 2, a
        # complex Hamiltonian, six terms per element), stepped through a captured graph
        dict(name="pop_2s6m_d9_complex", kind="propagate", sites=2, modes_per_site=3, depth=9, precision="fp64",
             complex_h=True, graphs=True, steps=100, observe=10),
        # the headline workload of bench.py: 8 sites, 16 modes, depth 8, 735,471 ADOs
        dict(name="pop_8s16m_d8_fp64", kind="propagate", sites=8, modes_per_site=2, depth=8, precision="fp64",
             complex_h=False, graphs=False, steps=16, observe=8),
        # the same with FP32 storage
        dict(name="pop_8s16m_d8_fp32", kind="propagate", sites=8, modes_per_site=2, depth=8, precision="fp32",
             complex_h=False, graphs=False, steps=16, observe=8),
        # the large system of bench.py: 24 sites, depth 4, 20,475 ADOs of 24 x 24
        dict(name="pop_24s24m_d4_fp64", kind="propagate", sites=24, modes_per_site=1, depth=4, precision="fp64",
             complex_h=False, graphs=False, steps=20, observe=10),
        dict(name="pop_24s24m_d4_fp32", kind="propagate", sites=24, modes_per_site=1, depth=4, precision="fp32",
             complex_h=False, graphs=False, steps=20, observe=10),
        # a quarter of the static-disorder ensemble of bench.py (depths 3 to 6), FP64
        dict(name="ensemble_7s_128_fp64", kind="ensemble", sites=7, members=128, min_depth=3, max_depth=6,
             precision="fp64", steps=32, observe=8),
        # the whole of it (2,048 hierarchies, about 1.4 million ADOs) with FP32 storage
        dict(name="ensemble_7s_512_fp32", kind="ensemble", sites=7, members=512, min_depth=3, max_depth=6,
             precision="fp32", steps=32, observe=8),
        # thermal states: 8 sites, 16 modes, depth 6 (74,613 ADOs), and a large system
        dict(name="tss_8s16m_d6", kind="tss", sites=8, modes_per_site=2, depth=6, iterations=40, observe=20),
        dict(name="tss_24s24m_d3", kind="tss", sites=24, modes_per_site=1, depth=3, iterations=20, observe=10),
        # one gradient of a fit: 8 sites, 8 modes, depth 6 (3,003 ADOs), 100 of its steps
        dict(name="adjoint_8s8m_d6", kind="adjoint", sites=8, modes_per_site=1, depth=6, steps=100, observe=1),
        # pump-probe on five sites with a ground state and two modes per site (complex
        # stage Hamiltonians, N = 6, 3,003 ADOs), from a checkpoint to the next
        dict(name="field_5s10m_d5", kind="field", sites=5, modes_per_site=2, depth=5, steps=50, observe=1),
    ]


def _count(width, depth):
    return math.comb(width + depth, depth)


def draw(rng):
    kind = rng.choice(["propagate", "propagate", "propagate", "wide", "ensemble", "tss", "tss", "adjoint", "field"])

    def hierarchy(sites, most, least=1, ks=(1, 2, 3)):
        """modes per site and a depth whose state has about a log-uniform share of `most` elements"""
        k = rng.choice([x for x in ks if sites * x <= 32])
        want = math.exp(rng.uniform(math.log(least), math.log(most))) / (sites * sites)
        depth = 1
        while depth < 12 and _count(sites * k, depth + 1) <= want:
            depth += 1
        return k, depth

    if kind == "ensemble":
        lo = rng.randint(2, 4)
        return dict(kind=kind, sites=rng.choice([5, 6, 7, 7]), members=int(round(2 ** rng.uniform(2, 8))), min_depth=lo,
                    max_depth=lo + rng.randint(1, 2), precision=rng.choice(["fp64", "fp32"]), steps=16, observe=8)
    if kind == "tss":
        sites = rng.choice([2, 3, 5, 7, 8, 9, 13, 17, 24])
        k, depth = hierarchy(sites, 4.8e6, 2.0e4, (1, 2))
        return dict(kind=kind, sites=sites, modes_per_site=k, depth=depth, iterations=20, observe=10)
    if kind == "adjoint":
        sites = rng.randint(2, 8)
        k, depth = hierarchy(sites, 2.0e5, 2.0e3, (1, 2))
        return dict(kind=kind, sites=sites, modes_per_site=k, depth=depth, steps=40, observe=rng.choice([1, 2, 5]))
    if kind == "field":
        sites = rng.randint(2, 7)
        k, depth = hierarchy(sites, 5.0e5, 2.0e3, (1, 2))
        return dict(kind=kind, sites=sites, modes_per_site=k, depth=depth, steps=rng.randint(10, 40),
                    observe=rng.choice([1, 5]))
    sites = rng.randint(9, 26) if kind == "wide" else rng.randint(2, 8)
    if kind == "wide":
        k, depth = hierarchy(sites, 1.2e7, 5.0e4, (1,))
    else:
        k, depth = hierarchy(sites, 4.8e7, 1.0e3)
    return dict(kind="propagate", sites=sites, modes_per_site=k, depth=depth, precision=rng.choice(["fp64", "fp32"]),
                complex_h=rng.random() < 0.3, graphs=rng.random() < 0.5, steps=20, observe=rng.choice([5, 10, 20]))


# ---- hierarchies and baths --------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _graph(width, depth):
    """All tuples of `width` non-negative numbers with a sum <= depth, by their sum, the
    all-zero tuple first, with the index of every neighbour (-1: none)."""
    rows = np.zeros((1, 0), dtype=np.int32)
    for _ in range(width):  # append one entry at a time, every value that still fits
        room = depth - rows.sum(axis=1)
        rep = np.repeat(np.arange(rows.shape[0]), room + 1)
        last = np.arange(rep.size) - np.repeat(np.cumsum(room + 1) - (room + 1), room + 1)
        rows = np.concatenate([rows[rep], last[:, None].astype(np.int32)], axis=1)
    tier = rows.sum(axis=1)
    rows = np.ascontiguousarray(rows[np.argsort(tier, kind="stable")])
    tier = rows.sum(axis=1)
    # a linear hash modulo 2^64: adding weight[m] to a tuple's key raises its entry m by one
    weight = np.random.default_rng(64).integers(0, 2 ** 64, width, dtype=np.uint64)
    key = (rows.astype(np.uint64) * weight).sum(axis=1, dtype=np.uint64)
    by_key = np.argsort(key)
    inner = np.flatnonzero(tier < depth)
    plus = np.full(rows.shape, -1, dtype=np.int32)
    minus = np.full(rows.shape, -1, dtype=np.int32)
    sorted_key = key[by_key]
    for m in range(width):
        up = by_key[np.searchsorted(sorted_key, key[inner] + weight[m])]
        plus[inner, m] = up
        minus[up, m] = inner
    return rows, plus, minus


def _modes(lam, rate, count, temperature):
    """Drude-Lorentz correlation function in `count` exponentials (the Drude pole and the
    first Matsubara poles): rates nu_k, coefficients c_k, Delta and Phi in SI units."""
    beta_hbar = HBAR / (K_B * temperature)
    nus = [rate] + [2.0 * math.pi * k / beta_hbar for k in range(1, count)]
    corr = sum(2.0 * rate ** 2 / (nu ** 2 - rate ** 2) for nu in nus[1:])
    cs = [2.0 * lam / beta_hbar * (1.0 - corr)]
    cs += [4.0 * lam * rate / beta_hbar * nu / (nu ** 2 - rate ** 2) for nu in nus[1:]]
    delta = (2.0 * lam / (beta_hbar * rate) - sum(c / nu for c, nu in zip(cs, nus))) / HBAR
    return nus, cs, delta, rate * lam / HBAR


def _complex_pairs(x):
    x = np.asarray(x, dtype=np.complex128)
    return np.ascontiguousarray(np.stack([x.real, x.imag], axis=-1).reshape(-1))


def _system(rng, sites, k, depth, complex_h=False, ground=False, disorder=None):
    """Instance arrays of a seeded system: site energies 12,000 to 12,600 cm^-1 (or the
    given base plus N(0, 50^2)) relative to their mean, couplings up to 100 cm^-1, one
    bath per site (lambda 35 cm^-1, 1 / rate 50 fs, 300 K, k exponentials)."""
    if disorder is None:
        e = rng.uniform(12000.0, 12600.0, sites)
        J = rng.uniform(-100.0, 100.0, (sites, sites))
        J = np.triu(J, 1) + (1j * np.triu(rng.uniform(-40.0, 40.0, (sites, sites)), 1) if complex_h else 0.0)
    else:
        e, J = disorder
        e = e + rng.normal(0.0, 50.0, sites)
    H = np.zeros((sites + ground, sites + ground), dtype=np.complex128)
    H[ground:, ground:] = np.diag(e - e.mean()) + J + np.conj(J).T
    tuples, plus, minus = _graph(sites * k, depth)
    nus, cs, delta, phi = _modes(35.0 * INVCM, 1.0 / (50.0 * FS), k, 300.0)
    n = sites + ground
    coupling = np.arange(-ground, sites, dtype=np.int32).reshape(n, 1)
    return SimpleNamespace(
        states=n, matsubaras=k, baths=sites, coupling=coupling, hamiltonian=_complex_pairs(H * INVCM), tuples=tuples,
        plus=plus, minus=minus, pf_same_sum=_complex_pairs(-(tuples @ np.tile(nus, sites))),
        pf_same=_complex_pairs(np.full(sites, delta)), pf_circ=_complex_pairs(np.full(sites, phi)),
        cbk=_complex_pairs(np.tile(cs, sites)))


def _pure_state(rng, n):
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    psi /= np.linalg.norm(psi)
    return np.outer(psi, psi.conj())


def _rng(case, seed):
    return np.random.default_rng([int(seed), len(case["kind"])])


def _precision(case):
    return heom_amd.HEOM_PRECISION_FP32 if case["precision"] == "fp32" else heom_amd.HEOM_PRECISION_FP64


# ---- inputs of each kind ------------------------------------------------------------------


def _propagate_inputs(case, seed):
    rng = _rng(case, seed)
    inst = _system(rng, case["sites"], case["modes_per_site"], case["depth"], case["complex_h"])
    return inst, _pure_state(rng, inst.states)


def _ensemble_inputs(case, seed):
    """The instances (populations first, then three absorption instances per realisation),
    their initial tops, start operators and trace operators."""
    rng = _rng(case, seed)
    n, members = case["sites"], case["members"]
    base = (rng.uniform(12000.0, 12600.0, n), np.triu(rng.uniform(-100.0, 100.0, (n, n)), 1))
    dirs = rng.normal(size=(n, 3))
    dirs /= np.linalg.norm(dirs, axis=1)[:, None]
    pops, las, depths = [], [], rng.integers(case["min_depth"], case["max_depth"] + 1, members)
    for d in depths:
        pop = _system(rng, n, 1, int(d), disorder=base)
        la = SimpleNamespace(**vars(pop))
        H = np.zeros((n + 1, n + 1, 2))
        H[1:, 1:] = pop.hamiltonian.reshape(n, n, 2)
        la.states, la.hamiltonian = n + 1, H.reshape(-1)
        la.coupling = np.arange(-1, n, dtype=np.int32).reshape(n + 1, 1)
        pops.append(pop)
        las.append(la)
    insts = pops + [la for la in las for _ in range(3)]
    N = n + 1
    tops = np.zeros((len(insts), N, N), dtype=np.complex128)
    start = np.zeros_like(tops)
    trace = np.zeros_like(tops)
    tops[:members, 1, 1] = 1.0  # |site_1><site_1|
    start[:members] = np.eye(N)
    tops[members:, 0, 0] = 1.0  # |g><g|, then the dipole operators of each component
    for t in range(3):
        start[members + t::3, 1:, 0] = dirs[:, t]
        trace[members + t::3, 0, 1:] = dirs[:, t]
    return insts, tops, start, trace


def _tss_inputs(case, seed):
    rng = _rng(case, seed)
    inst = _system(rng, case["sites"], case["modes_per_site"], case["depth"])
    n = inst.states
    H = inst.hamiltonian.reshape(n, n, 2)[..., 0]
    energies, vectors = np.linalg.eigh(H)
    boltzmann = np.exp(-(energies - energies.min()) / (K_B * 300.0))
    top = (vectors * (boltzmann / boltzmann.sum())) @ vectors.T
    setup = {"c": vectors.T.copy(), "eigenvalues": energies.astype(np.complex128), "epsilon": 1e14 + 0.0j}
    return inst, setup, top.astype(np.complex128)


def _adjoint_inputs(case, seed):
    rng = _rng(case, seed)
    inst = _system(rng, case["sites"], case["modes_per_site"], case["depth"])
    rows = case["steps"] // case["observe"] + 1
    op = np.zeros((inst.states, inst.states), dtype=np.complex128)
    op[1, 1] = 1.0
    weights = FS * 1e15 * rng.uniform(0.5, 1.5, rows).astype(np.complex128)
    return inst, _pure_state(rng, inst.states), op, weights


def _field_inputs(case, seed):
    rng = _rng(case, seed)
    inst = _system(rng, case["sites"], case["modes_per_site"], case["depth"], ground=True)
    N = inst.states
    tier = inst.tuples.sum(axis=1)
    shape = (tier.size, N, N)
    y = (rng.normal(size=shape) + 1j * rng.normal(size=shape)) * (0.3 ** tier)[:, None, None]
    y = 0.5 * (y + np.conj(np.swapaxes(y, 1, 2)))
    y[0] = _pure_state(rng, N)
    d_minus = np.zeros((N, N), dtype=np.complex128)
    d_minus[0, 1:] = rng.uniform(-1.0, 1.0, N - 1)
    times = FS * (np.arange(case["steps"])[:, None] + np.array([0.0, 0.5, 0.5, 1.0]))
    width = 0.2 * case["steps"] * FS
    E = 60.0 * INVCM * np.exp(-(times - 0.5 * case["steps"] * FS) ** 2 / (2.0 * width ** 2)) * np.exp(
        1j * (rng.uniform(0.0, 6.28) + 2.0e13 * times))
    H0 = inst.hamiltonian.reshape(N, N, 2) @ np.array([1.0, 1.0j])
    stage_h = H0 - E[..., None, None] * d_minus - np.conj(E)[..., None, None] * d_minus.T
    return inst, _complex_pairs(y), stage_h


# ---- what a user's program holds, and a pass ------------------------------------------------


def prepare(case, seed):
    state = SimpleNamespace(case=case)
    kind = case["kind"]
    if kind == "propagate":
        inst, top = _propagate_inputs(case, seed)
        state.handle = heom_amd.Handle.from_instance(inst, _precision(case))
        state.handle.use_graphs(case["graphs"])
        state.handle.set_top(top)
    elif kind == "ensemble":
        insts, state.tops, state.start, state.trace = _ensemble_inputs(case, seed)
        state.handle = heom_amd.Handle.from_instances(insts, _precision(case))
        state.handle.use_graphs(True)
    elif kind == "tss":
        inst, setup, top = _tss_inputs(case, seed)
        state.handle = heom_amd.Handle.thermal_state_search_from_instance(inst, setup)
        state.handle.set_top(top)
    elif kind == "adjoint":
        inst, state.top, state.op, state.weights = _adjoint_inputs(case, seed)
        state.handle = heom_amd.Handle.from_instance(inst)
    else:
        inst, state.checkpoint, state.stage_h = _field_inputs(case, seed)
        state.handle = heom_amd.Handle.from_instance(inst)
    return state


def run(state):
    case, h = state.case, state.handle
    kind = case["kind"]
    if kind == "propagate":
        pops, _ = h.propagate_observe(FS, case["steps"], case["observe"])
        return {"populations": pops, "top": h.get_top(), "norms": h.norms()}
    if kind == "ensemble":
        h.clear_state()
        h.set_top(state.tops)
        h.mmult_left(state.start)
        pops, traces = h.propagate_observe(2.0 * FS, case["steps"], case["observe"], state.trace)
        return {"populations": pops, "absorption": traces}
    if kind == "tss":
        tops = []
        for _ in range(case["iterations"] // case["observe"]):
            h.tss_step(case["observe"])
            tops.append(h.get_top())
        return {"tops": tops, "norms": h.norms()}
    if kind == "adjoint":
        h.clear_state()
        h.set_top(state.top)
        observed = h.adjoint_forward(FS, case["steps"], case["observe"], state.op)
        return {"observed": observed, "gradients": h.adjoint_backward(state.weights)}
    h.set_state(state.checkpoint)
    tops = h.propagate_timedep(FS, case["steps"], case["observe"], state.stage_h)
    return {"tops": tops, "state": h.get_state(), "norms": h.norms()}


# ---- bytes and operations of a pass ---------------------------------------------------------


def _evaluations(elements, states, k, complex_h, cbytes, count):
    """`count` evaluations of the operator on a state of `elements` matrix elements (N x N
    each ADO, one bath of k modes per site).  Every evaluation needs the whole result of
    the one before it, so a state beyond the last-level cache is read and written once
    by each; a smaller one is read and written once in all."""
    state = elements * cbytes
    flops = elements * (states * 2 * (8 if complex_h else 4) + 8 + 2 * k * 14 + 8) * count
    return 2 * state * (count if state > LLC_BYTES else 1), flops


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        mean = np.mean([_count(case["sites"], d) for d in range(case["min_depth"], case["max_depth"] + 1)])
        ados, n, k = case["members"] * mean, case["sites"], 1
        elements = ados * (n * n + 3 * (n + 1) ** 2)
        cb = 8 if case["precision"] == "fp32" else 16
        b, f = _evaluations(elements, n + 1, k, False, cb, 4 * case["steps"])
        return {"bytes": float(b), "flops": float(f)}
    n, k = case["sites"] + (kind == "field"), case["modes_per_site"]
    elements = _count(case["sites"] * k, case["depth"]) * n * n
    cb = 8 if case.get("precision") == "fp32" else 16
    if kind == "tss":
        # f_TSS has no commutator; the transform is four matrix products and a division
        b, f = _evaluations(elements, 0, k, False, cb, case["iterations"])
        return {"bytes": float(b), "flops": float(f + elements * case["iterations"] * (4 * n * 4 + 20))}
    if kind == "adjoint":
        b, f = _evaluations(elements, n, k, False, cb, 4 * case["steps"])
        # the forward stage vectors are written once and read once by the backward sweep
        traj = 2 * elements * cb * (4 * case["steps"] if 4 * case["steps"] * elements * cb > LLC_BYTES else 1)
        contract = elements * 4 * case["steps"] * (16 * n + 8 + 2 * k * 2 * 10)
        return {"bytes": float(b + traj), "flops": float(2 * f + contract)}
    if kind == "field":
        b, f = _evaluations(elements, n, k, True, cb, 4 * case["steps"])
        return {"bytes": float(b + 2 * elements * cb), "flops": float(f + 4 * elements)}
    b, f = _evaluations(elements, n, k, case["complex_h"], cb, 4 * case["steps"])
    return {"bytes": float(b), "flops": float(f)}


# ---- the same in 64 bits with plain torch ----------------------------------------------------


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Reference:
    """The HEOM right-hand side of one hierarchy shape for a stack of states
    [systems, ADOs, N, N] with one Hamiltonian each."""

    def __init__(self, inst, hamiltonians, parameters=None):
        dev, c = _device(), torch.complex128
        n, K, B = inst.states, inst.matsubaras, inst.baths

        def cplx(x):
            x = torch.as_tensor(np.asarray(x, dtype=np.float64).reshape(-1, 2), device=dev)
            return torch.complex(x[:, 0], x[:, 1])

        p = parameters or {"hamiltonian": torch.as_tensor(np.asarray(hamiltonians), device=dev, dtype=c),
                           "pf_same_sum": cplx(inst.pf_same_sum), "pf_same": cplx(inst.pf_same),
                           "pf_circ": cplx(inst.pf_circ), "cbk": cplx(inst.cbk)}
        self.p = p
        self.H = (p["hamiltonian"] / HBAR)[:, None]
        # how many baths equal to b the states i and j couple to
        coup = torch.zeros((B, n), device=dev, dtype=torch.float64)
        for s in range(n):
            for b in inst.coupling[s]:
                if b >= 0:
                    coup[int(b), s] += 1.0
        ci, cj = coup[:, :, None], coup[:, None, :]
        off = 1.0 - torch.eye(n, device=dev, dtype=torch.float64)
        gam = -((ci + cj) * off * p["pf_same"][:, None, None]).sum(0)
        self.diagonal = p["pf_same_sum"][:, None, None] + gam
        tuples = torch.as_tensor(np.asarray(inst.tuples), device=dev)
        plus = torch.as_tensor(np.asarray(inst.plus), device=dev).long()
        minus = torch.as_tensor(np.asarray(inst.minus), device=dev).long()
        self.terms = []
        for m in range(B * K):
            b, k = divmod(m, K)
            cm = p["cbk"][m]
            size = cm.abs()
            up = (ci[b] - cj[b]) * torch.sqrt(size / HBAR)
            down = 1j * (ci[b] - cj[b]) * cm / HBAR
            if k == 0:
                down = down + (ci[b] + cj[b]) * p["pf_circ"][b]
            down = down * torch.sqrt(HBAR / size)
            nm = tuples[:, m].double()
            has = torch.nonzero(plus[:, m] >= 0)[:, 0]
            low = torch.nonzero(minus[:, m] >= 0)[:, 0]
            self.terms.append((has, plus[has, m], 1j * torch.sqrt(nm[has] + 1.0)[:, None, None], up,
                               low, minus[low, m], torch.sqrt(nm[low])[:, None, None], down))

    def rhs(self, y, H=None):
        H = self.H if H is None else H
        f = 1j * (y @ H - H @ y) + self.diagonal * y
        for has, hi, sp, up, low, lo, sn, down in self.terms:
            f = f.index_add(1, has, (sp * up) * y[:, hi])
            f = f.index_add(1, low, (sn * down) * y[:, lo])
        return f

    def step(self, y, dt, stage_h=(None,) * 4):
        k1 = self.rhs(y, stage_h[0])
        k2 = self.rhs(y + 0.5 * dt * k1, stage_h[1])
        k3 = self.rhs(y + 0.5 * dt * k2, stage_h[2])
        k4 = self.rhs(y + dt * k3, stage_h[3])
        return y + dt / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)

    def start(self, tops):
        tops = torch.as_tensor(np.asarray(tops), device=_device(), dtype=torch.complex128)
        y = torch.zeros((tops.shape[0], self.diagonal.shape[0]) + tuple(tops.shape[1:]), device=tops.device,
                        dtype=tops.dtype)
        y[:, 0] = tops
        return y


def _hamiltonian(inst):
    h = np.asarray(inst.hamiltonian).reshape(inst.states, inst.states, 2)
    return h[..., 0] + 1j * h[..., 1]


def exact(case, seed):
    # on a CPU a right-hand side takes about 0.1 microseconds an element
    if _device() == "cpu" and work(case)["flops"] > 2e10:
        return None
    with torch.no_grad():
        return {"propagate": _exact_propagate, "ensemble": _exact_ensemble, "tss": _exact_tss,
                "adjoint": _exact_adjoint, "field": _exact_field}[case["kind"]](case, seed)


def _norms(y):
    return (y.real ** 2 + y.imag ** 2).sum(dim=(1, 2)).cpu().numpy()


def _exact_propagate(case, seed):
    inst, top = _propagate_inputs(case, seed)
    ref = _Reference(inst, _hamiltonian(inst)[None])
    y = ref.start(top[None])
    pops = []
    for s in range(case["steps"] + 1):
        if s:
            y = ref.step(y, FS)
        if s % case["observe"] == 0:
            pops.append(torch.diagonal(y[:, 0], dim1=1, dim2=2).real.cpu().numpy())
    return {"populations": np.stack(pops), "top": y[0, 0].cpu().numpy(), "norms": _norms(y[0])}


def _exact_ensemble(case, seed):
    insts, tops, start, trace = _ensemble_inputs(case, seed)
    N, rows = tops.shape[1], case["steps"] // case["observe"] + 1
    pops = np.zeros((rows, len(insts), N))
    traces = np.zeros((rows, len(insts)), dtype=np.complex128)
    key = lambda i: (insts[i].states, len(insts[i].tuples))  # noqa: E731
    for (n, _), group in itertools.groupby(sorted(range(len(insts)), key=key), key=key):
        ids = list(group)
        ref = _Reference(insts[ids[0]], np.stack([_hamiltonian(insts[i]) for i in ids]))
        y = ref.start((start[ids] @ tops[ids])[:, :n, :n])
        for s in range(case["steps"] + 1):
            if s:
                y = ref.step(y, 2.0 * FS)
            if s % case["observe"] == 0:
                top = y[:, 0].cpu().numpy()
                r = s // case["observe"]
                pops[r][ids, :n] = np.diagonal(top, axis1=1, axis2=2).real
                traces[r][ids] = np.einsum("kij,kji->k", trace[ids][:, :n, :n], top)
        del ref, y
    return {"populations": pops, "absorption": traces}


def _exact_tss(case, seed):
    inst, setup, top = _tss_inputs(case, seed)
    ref = _Reference(inst, np.zeros((1, inst.states, inst.states)))
    dev = _device()
    eps = setup["epsilon"]
    w = np.subtract.outer(setup["eigenvalues"], setup["eigenvalues"]) * 1j / HBAR
    S = ref.p["pf_same_sum"][:, None, None]
    denominator = torch.as_tensor(w, device=dev) + eps - S
    ref.diagonal = ref.diagonal - S + eps  # f_TSS: eps y in place of the commutator and S y
    C = torch.as_tensor(setup["c"].astype(np.complex128), device=dev)
    y, tops = ref.start(top[None]), []
    for s in range(1, case["iterations"] + 1):
        y = C.T @ ((C @ ref.rhs(y) @ C.T) / denominator) @ C
        if s % case["observe"] == 0:
            tops.append(y[0, 0].cpu().numpy())
    return {"tops": tops, "norms": _norms(y[0])}


def _exact_adjoint(case, seed):
    elements = _count(case["sites"] * case["modes_per_site"], case["depth"]) * case["sites"] ** 2
    if elements * case["steps"] * case["sites"] * case["modes_per_site"] > 2.5e8:
        return None  # the recorded graph of autograd grows with this
    inst, top, op, weights = _adjoint_inputs(case, seed)
    plain = _Reference(inst, _hamiltonian(inst)[None])
    with torch.enable_grad():
        p = {k: v.clone().requires_grad_(True) for k, v in plain.p.items()}
        ref = _Reference(inst, None, parameters=p)
        y0 = ref.start(top[None]).requires_grad_(True)
        O = torch.as_tensor(op, device=y0.device)
        w = torch.as_tensor(weights, device=y0.device)
        y, observed = y0, []
        for s in range(case["steps"] + 1):
            if s:
                y = ref.step(y, FS)
            if s % case["observe"] == 0:
                observed.append(torch.trace(O @ y[0, 0]))
        observed = torch.stack(observed)
        names = sorted(p)
        grads = torch.autograd.grad((w * observed).real.sum(), [p[k] for k in names] + [y0])
    g = {k: v.detach().cpu().numpy() for k, v in zip(names, grads)}
    g["state"] = _complex_pairs(grads[-1][0].detach().cpu().numpy())
    return {"observed": observed.detach().cpu().numpy()[:, None], "gradients": g}


def _exact_field(case, seed):
    inst, checkpoint, stage_h = _field_inputs(case, seed)
    n = inst.states
    ref = _Reference(inst, _hamiltonian(inst)[None])
    H = torch.as_tensor(stage_h / HBAR, device=_device())
    y = torch.as_tensor(checkpoint.reshape(-1, n, n, 2), device=_device())
    y = torch.complex(y[..., 0], y[..., 1])[None]
    tops = []
    for s in range(case["steps"] + 1):
        if s:
            y = ref.step(y, FS, H[s - 1])
        if s % case["observe"] == 0:
            tops.append(y[0, 0].cpu().numpy())
    return {"tops": np.stack(tops), "state": _complex_pairs(y[0].cpu().numpy()), "norms": _norms(y[0])}
