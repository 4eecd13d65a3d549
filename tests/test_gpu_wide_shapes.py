"""Workgroup shapes of the large-system kernel: the one taken by default is among those that the
autotuner times and set_stage_config accepts, and all of them give the same bits."""
import numpy as np
import pytest

from helpers import make_instance, random_state

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
