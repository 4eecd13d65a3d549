"""Compaction (heom_compact) of a batch whose instances have different baths: every instance
keeps its own bath prefactors in the compacted layout, against the oracle of that instance
with the same mask (five RK4 steps, 1e-10)."""
import numpy as np
import pytest

import oracle as O
from helpers import as_complex, make_instance, max_abs_rel
from test_gpu_batch_mixed import random_states, split_state

pytestmark = pytest.mark.gpu

heom_amd = pytest.importorskip("heom_amd")


@pytest.mark.parametrize("N,depths", [(4, (6, 5, 6)), (7, (4, 3, 4)), (8, (4, 3, 4)), (12, (3, 2, 3))])
def test_compacted_batch_keeps_bath_classes(oracle_mod, N, depths):
    # the seed sets the baths' lambda and 1/gamma; two instances share them
    insts = [make_instance(N, N, 1, D, [[i] for i in range(N)], seed=s) for D, s in zip(depths, (1, 2, 1))]
    masks = []
    for k, inst in enumerate(insts):
        m = np.where(np.random.default_rng(k).random(inst.matrices) < 0.6, O.MASK_FALSE, O.MASK_TRUE).astype(np.uint8)
        m[0] = O.MASK_PROTECTED
        masks.append(m)
    ys = random_states(insts, 4)
    with heom_amd.Handle.from_instances(insts) as h:
        h.set_mask(np.concatenate(masks))
        h.set_state(np.concatenate(ys))
        assert h.compact() == sum(np.count_nonzero(m) for m in masks)
        h.step_rk4(1e-15, 5)
        got = split_state(h.get_state(), insts, N)
    for k, (inst, mask, y) in enumerate(zip(insts, masks, ys)):
        inst.mask[:] = mask
        inst.propagate(y, 1e-15, 5, 5)
        keep = mask != O.MASK_FALSE
        assert max_abs_rel(got[k][keep], as_complex(y, inst)[keep]) < 1e-10, k
