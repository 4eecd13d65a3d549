"""Large systems (N > 8) off the plain path, against the oracle: ADO norms and the norm
threshold's mask, masked and compacted hierarchies, masked searches, batches whose instances
differ in states, modes and couplings, mmult_left, the shapes in which every wavefront goes
through several ADOs (many ADOs; at 32 sites in FP64 with eight wavefronts per workgroup), and
baths that couple to all or to half of the sites beside one of its own per site."""
import numpy as np
import pytest

import oracle as O
from helpers import as_complex, make_instance, max_abs_rel, random_state
from test_gpu_batch_mixed import pad_state, random_states, split_state

pytestmark = pytest.mark.gpu

heom_amd = pytest.importorskip("heom_amd")
FP64, FP32 = heom_amd.HEOM_PRECISION_FP64, heom_amd.HEOM_PRECISION_FP32
DT = 1e-15


def local(N, D, K=1, seed=None, complex_h=False):
    return make_instance(N, N, K, D, [[i] for i in range(N)], seed=N if seed is None else seed, complex_h=complex_h)


def shared(N, D, reach, K=1, complex_h=False):
    """a bath per site and one more that couples to the first `reach` sites"""
    return make_instance(N, N + 1, K, D, [[i, N if i < reach else -1] for i in range(N)], seed=N + reach,
                         complex_h=complex_h)


def random_mask(inst, seed):
    m = np.where(np.random.default_rng(seed).random(inst.matrices) < 0.35, O.MASK_FALSE, O.MASK_TRUE).astype(np.uint8)
    m[0] = O.MASK_PROTECTED
    return m


def stored(inst, y, prec):
    """what a handle of this precision holds after set_state(y): tiers 0 and 1 stay in FP64"""
    if prec == FP64:
        return y
    z = as_complex(y.astype(np.float32).astype(np.float64), inst)
    t = inst.graph.tuples.sum(axis=1) <= 1
    z[t] = as_complex(y, inst)[t]
    return np.ascontiguousarray(np.stack([z.real, z.imag], -1).reshape(-1))


def rk4(inst, y):
    k1 = inst.rhs(y)
    k2 = inst.rhs(y + 0.5 * DT * k1)
    k3 = inst.rhs(y + 0.5 * DT * k2)
    return y + DT / 6 * (k1 + 2 * k2 + 2 * k3 + inst.rhs(y + DT * k3))


def check_rhs_and_step(inst, prec, seed=1):
    """one evaluation and one step: sums of a few hundred products (FP64 1e-12, FP32 1e-5)"""
    y = random_state(inst, seed)
    ys = stored(inst, y, prec)
    tol = 1e-12 if prec == FP64 else 1e-5
    with heom_amd.Handle.from_instance(inst, precision=prec) as h:
        h.set_state(y)
        assert np.array_equal(h.get_state(), ys)
        assert max_abs_rel(h.rhs(), inst.rhs(ys)) < tol
        h.step_rk4(DT, 1)
        assert max_abs_rel(h.get_state(), rk4(inst, ys)) < tol


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N,D", [(9, 3), (24, 2)])
def test_norms_and_threshold_mask(oracle_mod, N, D, prec):
    """the sum of up to 2 N^2 squares: 2e-13 relative, plus the storage's rounding in FP32"""
    inst = local(N, D)
    y = random_state(inst, 3)
    ref = inst.norms(y)
    order = np.sort(ref)
    threshold = 0.5 * (order[len(order) // 2] + order[len(order) // 2 + 1])
    with heom_amd.Handle.from_instance(inst, precision=prec) as h:
        h.set_state(y)
        got = h.norms()
        assert np.max(np.abs(got / ref - 1.0)) < (2e-13 if prec == FP64 else 2.5e-7)
        assert np.all(h.get_mask() == O.MASK_TRUE)
        got = h.norms(threshold)
        want = np.where(got <= threshold, O.MASK_FALSE, O.MASK_TRUE)
        assert np.array_equal(h.get_mask(), want)
        assert 0.25 < np.mean(want == O.MASK_FALSE) < 0.75
        rhs = h.rhs()
    inst.mask[:] = want
    ref = inst.rhs(stored(inst, y, prec))
    keep = want != O.MASK_FALSE
    assert max_abs_rel(as_complex(rhs, inst)[keep], as_complex(ref, inst)[keep]) < (1e-12 if prec == FP64 else 1e-5)


@pytest.mark.parametrize("N,D", [(9, 4), (24, 2), (32, 2)])
def test_masked_and_compacted(oracle_mod, N, D):
    inst = local(N, D)
    mask = random_mask(inst, N)
    keep = mask != O.MASK_FALSE
    y = random_state(inst, 5)
    inst.mask[:] = mask
    ref = y.copy()
    inst.propagate(ref, DT, 5, 5)
    state = {}
    for compact in (False, True):
        with heom_amd.Handle.from_instance(inst) as h:
            h.set_mask(mask)
            h.set_state(y)
            if compact:  # after the state: compaction moves it
                assert h.compact() == np.count_nonzero(keep)
                assert np.array_equal(as_complex(h.get_state(), inst)[keep], as_complex(y, inst)[keep])
            h.step_rk4(DT, 5)
            state[compact] = as_complex(h.get_state(), inst)
            if compact:
                got = h.norms()
                assert np.all(got[~keep] == 0) and np.all(state[True][~keep] == 0)
                want = np.sum(np.abs(state[True][keep]) ** 2, axis=(1, 2))
                assert np.max(np.abs(got[keep] / want - 1.0)) < 2e-13
    assert np.array_equal(state[True][keep], state[False][keep])
    assert max_abs_rel(state[True][keep], as_complex(ref, inst)[keep]) < 1e-10


@pytest.mark.parametrize("N,D", [(9, 4), (24, 2), (28, 2)])
def test_masked_search(oracle_mod, N, D):
    inst = local(N, D)
    s = O.thermal_state_setup(inst.hamiltonian_matrix(), 300.0)
    inst.set_hamiltonian(s["pseudo_hamiltonian"])
    mask = random_mask(inst, N + 1)
    y = random_state(inst, 4)
    with heom_amd.Handle.thermal_state_search_from_instance(inst, s) as h:
        h.set_mask(mask)
        h.set_state(y)
        h.tss_step(3)
        got = h.get_state()
    inst.mask[:] = mask
    inst.tss_step(y, s, 3)
    keep = mask != O.MASK_FALSE
    assert max_abs_rel(as_complex(got, inst)[keep], as_complex(y, inst)[keep]) < 1e-10


def mixed(N):
    """N sites; the same with a bath shared by all of them; fewer sites, two modes per bath;
    a ground state without a bath; N sites, another depth"""
    return [local(N, 2, seed=1), shared(N, 2, N), local(N - 3, 2, K=2, seed=2),
            make_instance(N, N - 1, 1, 3, [[-1]] + [[i] for i in range(N - 1)], seed=5), local(N, 3, seed=1)]


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N", [10, 18])
def test_mixed_batch(oracle_mod, N, prec):
    insts = mixed(N)
    ys = random_states(insts, 7)
    mx = np.random.default_rng(N).normal(size=(2, len(insts), N, N))
    mx = mx[0] + 1j * mx[1]
    with heom_amd.Handle.from_instances(insts, precision=prec) as h:
        h.set_state(pad_state(insts, ys, N))
        rhs = split_state(h.rhs(), insts, N)
        h.step_rk4(DT, 5)
        got = split_state(h.get_state(), insts, N)
        h.mmult_left(mx)
        product = split_state(h.get_state(), insts, N)
    tol = 1e-12 if prec == FP64 else 1e-5
    for k, inst in enumerate(insts):
        n = inst.states
        assert not np.any(got[k][:, n:, :]) and not np.any(got[k][:, :, n:])
        y = stored(inst, ys[k], prec)
        assert max_abs_rel(rhs[k][:, :n, :n], as_complex(inst.rhs(y), inst)) < tol, k
        inst.propagate(y, DT, 5, 5)
        assert max_abs_rel(got[k][:, :n, :n], as_complex(y, inst)) < tol, k
        # N products and sums a row, then the storage's rounding
        assert max_abs_rel(product[k], mx[k] @ got[k]) < (1e-13 if prec == FP64 else 1e-7), k


def test_mixed_search_batch(oracle_mod):
    insts = [local(10, 2, seed=1), shared(10, 2, 10), shared(10, 3, 5)]
    setups = []
    for inst in insts:
        s = O.thermal_state_setup(inst.hamiltonian_matrix(), 300.0)
        inst.set_hamiltonian(s["pseudo_hamiltonian"])
        setups.append(s)
    ys = random_states(insts, 9)
    with heom_amd.Handle.thermal_state_search_from_instances(insts, setups) as h:
        h.set_state(np.concatenate(ys))
        h.tss_step(2)
        got = split_state(h.get_state(), insts, 10)
    for k, (inst, s, y) in enumerate(zip(insts, setups, ys)):
        inst.tss_step(y, s, 2)
        assert max_abs_rel(got[k], as_complex(y, inst)) < 1e-10, k


# more ADOs than wavefronts run at once: N <= 16, 24 and 32; at 32 sites in FP64 by eights
@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N,D", [(9, 7), (18, 4), (32, 3)])
def test_several_ados_per_wavefront(oracle_mod, N, D, prec):
    check_rhs_and_step(local(N, D), prec)


# N, sites of the shared bath, depth, matsubaras, complex H: lists of up to N * N elements, so
# up to 16 rounds of 64 lanes for one mode and one round for the others; 73 modes
@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N,reach,D,K,complex_h", [(9, 9, 3, 1, False), (12, 6, 2, 2, True), (16, 16, 3, 1, False),
                                                   (24, 24, 2, 3, False), (24, 12, 3, 1, True), (32, 32, 2, 1, False)])
def test_shared_bath(oracle_mod, N, reach, D, K, complex_h, prec):
    check_rhs_and_step(shared(N, D, reach, K, complex_h), prec)


@pytest.mark.parametrize("N,reach,K", [(9, 9, 1), (12, 6, 2), (24, 24, 3), (32, 32, 1)])
def test_shared_bath_search(oracle_mod, N, reach, K):
    inst = shared(N, 2, reach, K)
    s = O.thermal_state_setup(inst.hamiltonian_matrix(), 300.0)
    inst.set_hamiltonian(s["pseudo_hamiltonian"])
    y = random_state(inst, 2)
    with heom_amd.Handle.thermal_state_search_from_instance(inst, s) as h:
        h.set_state(y)
        h.tss_step(2)
        got = h.get_state()
    inst.tss_step(y, s, 2)
    assert max_abs_rel(got, y) < 1e-10
