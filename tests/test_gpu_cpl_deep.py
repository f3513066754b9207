"""Lists of at most 64 groups share a group's tops between eight wavefronts
(eri_cpld_*), longer ones between four (eri_cpls_*): every value is computed
by the same operations in the same order, so a list of 65 or more groups and
its quartets in lists of 64, 3 and 1 agree bit for bit.  Depths 1-3 mixed
within a list, one class of each shape that has the kernel and classes on
either side of the rule; first derivatives of one class through the g-shell
terms."""
import numpy as np
import pytest
import torch

import batch
import simint
from test_gpu_batch import _pool

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("am,deriv", [((2, 2, 2, 2), 0), ((3, 2, 3, 3), 0), ((3, 3, 3, 1), 0), ((2, 2, 3, 3), 0),
                                      ((3, 3, 3, 3), 0), ((3, 1, 2, 2), 0), ((2, 2, 2, 1), 0),
                                      ((3, 3, 2, 1), 1)])
def test_shortest_lists_equal_longer_ones(gpu, am, deriv):
    shells = _pool(seed=4, per_am=6, maxk=3)
    basis = simint.Basis(shells)
    rng = np.random.default_rng(sum(am))
    by = [[i for i, s in enumerate(shells) if s[0] == l] for l in range(4)]
    q = np.stack([rng.choice(by[l], 140) for l in am], axis=1)
    L = simint.lib()
    prev = L.simint_hip_class_list_kernel(*am)
    lanes = L.simint_hip_set_list_split(1)      # of the lane-per-quartet terms: by the list's length otherwise
    if not deriv:
        assert L.simint_hip_set_class_list_kernel(*am, simint.FAMILIES["cpl"]) >= 0

    def run(part):
        b = batch.QuartetBatch(basis, part, deriv=deriv)
        out = torch.full((b.out_doubles,), float("nan"), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        b.run(out.data_ptr())
        simint.synchronize()
        b.free()
        return out
    try:
        whole = run(q)
        parts = [run(q[a:b]) for a, b in ((0, 64), (64, 67), (67, 68), (68, 132), (132, 140))]
    finally:
        L.simint_hip_set_class_list_kernel(*am, prev)
        L.simint_hip_set_list_split(lanes)
    assert not bool(torch.isnan(whole).any())
    assert torch.equal(torch.cat(parts), whole)
    basis.free()
