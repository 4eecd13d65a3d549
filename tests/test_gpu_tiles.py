"""The large-system kernel and the two thermal-state-search kernels where their tiling ends:
states at, below and above the multiples of 16 and 8 of the matrix tiles, hierarchies that do
not fill a 64-ADO tile, one ADO per wavefront and several, modes that couple to more elements
than a wavefront has lanes, more modes than lanes, element tables too large for LDS, real and
complex Hamiltonians and transforms, against the oracle.  Every result is one evaluation (the
RHS), one RK4 step or two search iterations: sums of at most a few hundred products, so 1e-12
in FP64, 1e-5 on FP32 storage (tier-0/1 ADOs: 1e-12) and 1e-10 through a search's transforms."""
import numpy as np
import pytest

import oracle as O
from helpers import as_complex, max_abs_rel, random_state
from test_gpu_parity import make_instance

pytestmark = pytest.mark.gpu

heom_amd = pytest.importorskip("heom_amd")

# N, matsubaras, depth, states per bath, complex H
CASES = [(9, 1, 2, 1, False), (17, 4, 1, 1, True), (16, 1, 2, 1, True), (17, 1, 3, 1, False), (17, 1, 4, 1, False),
         (24, 1, 1, 3, True), (25, 1, 2, 3, False), (25, 1, 3, 1, True), (32, 3, 1, 1, False), (32, 1, 2, 2, True)]


def case(N, K, D, states, complex_h=False):
    return make_instance(N, N, K, D, [[(b + 2 * s) % N for s in range(states)] for b in range(N)], seed=N + K,
                         complex_h=complex_h)


@pytest.mark.parametrize("N,K,D,states,complex_h", CASES)
def test_wide_matches_oracle(oracle_mod, N, K, D, states, complex_h):
    inst = case(N, K, D, states, complex_h)
    y = random_state(inst, 1)
    dt = 1e-15
    k1 = inst.rhs(y)
    k2 = inst.rhs(y + 0.5 * dt * k1)
    k3 = inst.rhs(y + 0.5 * dt * k2)
    step = y + dt / 6 * (k1 + 2 * k2 + 2 * k3 + inst.rhs(y + dt * k3))
    with heom_amd.Handle.from_instance(inst) as h:
        h.set_state(y)
        assert np.array_equal(h.get_state(), y)
        assert max_abs_rel(h.rhs(), k1) < 1e-12
        h.step_rk4(dt, 1)
        assert max_abs_rel(h.get_state(), step) < 1e-12
    t = np.nonzero(inst.graph.tuples.sum(axis=1) <= 1)[0]
    ys = as_complex(y.astype(np.float32).astype(np.float64), inst)
    ys[t] = as_complex(y, inst)[t]
    ref = as_complex(inst.rhs(np.ascontiguousarray(np.stack([ys.real, ys.imag], -1).reshape(-1))), inst)
    with heom_amd.Handle.from_instance(inst, precision=heom_amd.HEOM_PRECISION_FP32) as h:
        h.set_state(y)
        got = as_complex(h.rhs(), inst)
    assert max_abs_rel(got, ref) < 1e-5
    assert max_abs_rel(got[t], ref[t]) < 1e-12


@pytest.mark.parametrize("real_c", [True, False])
@pytest.mark.parametrize("N,K,D,states", [(2, 1, 9, 1), (3, 2, 3, 2), (5, 1, 3, 3), (7, 1, 4, 1), (8, 4, 1, 1), (8, 1, 3, 4)] +
                         [c[:4] for c in CASES])
def test_search_matches_oracle(oracle_mod, N, K, D, states, real_c):
    inst = case(N, K, D, states)
    s = O.thermal_state_setup(inst.hamiltonian_matrix(), 300.0)
    inst.set_hamiltonian(s["pseudo_hamiltonian"])
    if not real_c:
        rng = np.random.default_rng(N)
        q, _ = np.linalg.qr(rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N)))
        s = dict(s, c=q, eigenvalues=s["eigenvalues"] + 1j * rng.normal(size=N) * 1e-22)
    y = random_state(inst, 2)
    with heom_amd.Handle.thermal_state_search_from_instance(inst, s) as h:
        h.set_state(y)
        h.tss_step(2)
        got = h.get_state()
    inst.tss_step(y, s, 2)
    assert max_abs_rel(got, y) < 1e-10
