"""heom_device_bytes counts what a handle holds beside its state: the constants of a search, added
state buffers, the scratch of an accumulating evaluation and the record of an adjoint sweep."""
import numpy as np
import pytest

import oracle as O
from helpers import make_instance

pytestmark = pytest.mark.gpu

heom_amd = pytest.importorskip("heom_amd")


@pytest.mark.parametrize("N,complex_c", [(5, False), (5, True), (12, False)])
def test_search_constants_are_counted(N, complex_c):
    inst = make_instance(N, N, 1, 2, [[i] for i in range(N)], seed=N)
    s = O.thermal_state_setup(inst.hamiltonian_matrix(), 300.0)
    if complex_c:
        s = dict(s, c=s["c"] * np.exp(0.3j))
    with heom_amd.Handle.from_instance(inst) as h:
        plain = h.device_bytes()
    with heom_amd.Handle.thermal_state_search_from_instance(inst, s) as h:
        # C (16 or, N <= 8 and real, twice 8 bytes an element), E_i - E_j, eps - S_u per slot
        constants = 16 * (2 * N * N + (inst.matrices + 1 + 63) // 64 * 64)
        assert h.device_bytes() >= plain + constants


def test_buffers_and_adjoint_record_are_counted():
    inst = make_instance(6, 6, 1, 2, [[i] for i in range(6)], seed=3)
    vector = 16 * 36 * 64  # 28 ADOs in one tile
    with heom_amd.Handle.from_instance(inst) as h:
        b0 = h.device_bytes()
        assert b0 >= 4 * vector
        h.add_buffers(2)
        b1 = h.device_bytes()
        assert b1 == b0 + 2 * vector
        h.clear_state()
        h.evaluate(0.0, 1e-15, src=0, out=1, out_base=0, out_coeff=0.5)
        assert h.device_bytes() == b1 + vector
        h.adjoint_forward(1e-15, 4, 1, np.eye(6), checkpoint_steps=2)
        assert h.device_bytes() >= b1 + vector + 2 * vector
