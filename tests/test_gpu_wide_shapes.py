"""Workgroup shapes of the large-system kernel: the one taken by default is among those that the
autotuner times and set_stage_config accepts, and all of them give the same bits, as do launches
with one ADO to a wavefront (which add the terms of ADOs with many edges by element) and with
several; the former against the oracle."""
import numpy as np
import pytest

from helpers import as_complex, make_instance, max_abs_rel, random_state

pytestmark = pytest.mark.gpu

heom_amd = pytest.importorskip("heom_amd")
FP64, FP32 = heom_amd.HEOM_PRECISION_FP64, heom_amd.HEOM_PRECISION_FP32


# 32 sites in FP64: by default eight wavefronts where each has several ADOs, else four
@pytest.mark.parametrize("N,D,prec", [(9, 3, FP64), (32, 2, FP64), (32, 3, FP64), (32, 3, FP32)])
def test_default_shape_is_a_candidate(N, D, prec):
    inst = make_instance(N, N, 1, D, [[i] for i in range(N)], seed=N)
    y = random_state(inst, 1)
    with heom_amd.Handle.from_instance(inst, precision=prec) as h:
        h.set_state(y)
        h.step_rk4(1e-15, 2)
        want = h.get_state()
        configs = h.autotune(steps=1)
        assert {c["ados_per_workgroup"] for c in configs} == {8, 4, 2, 1}
        for c in configs:
            h.set_stage_config(c)
            h.set_state(y)
            h.step_rk4(1e-15, 2)
            assert np.array_equal(h.get_state(), want), c


# N at the ends of two, three and four elements to a lane, two to eight terms an element, 64 and
# 68 modes; copies: so many instances of it that a wavefront gets several ADOs
BY_ELEMENT = [(9, 1, 3, 24), (11, 2, 2, 24), (12, 4, 2, 5), (13, 3, 2, 8), (14, 1, 2, 48), (16, 4, 2, 3), (16, 2, 1, 90)]


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N,K,D,copies", BY_ELEMENT)
def test_one_and_several_ados_per_wavefront_agree(N, K, D, copies, prec):
    inst = make_instance(N, N, K, D, [[i] for i in range(N)], seed=N + K, complex_h=N % 2 == 0)
    y = random_state(inst, 3)
    with heom_amd.Handle.from_instance(inst, precision=prec) as h:
        h.set_state(y)
        rhs = h.rhs()
        h.step_rk4(1e-15, 2)
        one = h.get_state()
    with heom_amd.Handle.from_instances([inst] * copies, precision=prec) as h:
        h.set_state(np.concatenate([y] * copies))
        assert np.array_equal(h.rhs().reshape(copies, -1), np.broadcast_to(rhs, (copies, rhs.size)))
        h.step_rk4(1e-15, 2)
        assert np.array_equal(h.get_state().reshape(copies, -1), np.broadcast_to(one, (copies, one.size)))


@pytest.mark.parametrize("N,B,K,D,every", [(9, 9, 1, 3, 1), (11, 11, 2, 2, 1), (12, 12, 4, 1, 1), (13, 13, 3, 2, 1),
                                           (14, 14, 1, 2, 1), (16, 16, 4, 1, 1), (16, 17, 4, 1, 1), (16, 8, 4, 2, 2)])
def test_terms_by_element_match_oracle(oracle_mod, N, B, K, D, every):
    inst = make_instance(N, B, K, D, [[i // every] for i in range(N)], seed=N + K)
    y = random_state(inst, 5)
    mask = np.where(np.random.default_rng(N).random(inst.matrices) < 0.2, 0, 1).astype(np.uint8)
    mask[0] = 2
    for m in (None, mask):
        keep = np.ones(inst.matrices, bool) if m is None else m != 0
        if m is not None:
            inst.mask[:] = m
        with heom_amd.Handle.from_instance(inst) as h:
            if m is not None:
                h.set_mask(m)
            h.set_state(y)
            got = h.rhs()
        assert max_abs_rel(as_complex(got, inst)[keep], as_complex(inst.rhs(y), inst)[keep]) < 1e-12
