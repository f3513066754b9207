"""Nuclear attraction of shells up to d with a recurrence per lane
(osoei_potential_direct): charge counts around and above a wavefront, depths
around a batch of primitive pairs, and higher shells in the same launch,
against the oracle and the long-double Hermite expansions.

Bar: helpers.parity_report (as tests/test_gpu_oei.py): the terms are the
oracle's, only their sum is taken in another order, so each block's error
against the long-double values stays within 4x the oracle's where that is
above 1e-14."""
import numpy as np
import pytest
import torch

import oracle
import simint
from helpers import REL_FLOOR, normalized_arrays, parity_report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncharge,depths,lmax", [(1, (1, 2), 2), (63, (6, 6), 2), (65, (5, 7), 3), (130, (1, 9), 2)])
def test_potential_lanes_over_primitives_and_charges(gpu, ncharge, depths, lmax):
    rng = np.random.default_rng(ncharge)
    shells = []
    for l in range(lmax + 1):
        for _ in range(2):
            n = int(rng.integers(depths[0], depths[1] + 1))
            shells.append((l, tuple(rng.uniform(-2.5, 2.5, 3)),
                           list(np.exp(rng.uniform(np.log(0.05), np.log(80.0), n))), list(rng.uniform(0.1, 1.0, n))))
    basis = simint.Basis(shells)
    sa = normalized_arrays(shells)
    pairs = [(i, j) for i in range(len(shells)) for j in range(len(shells))]
    Z, C = rng.integers(1, 20, ncharge).astype(np.float64), rng.uniform(-4, 4, (ncharge, 3))
    ref, off, n = oracle.osoei(sa, pairs, 2, Z, C)
    ex, _, _ = oracle.md_oei(sa, pairs, 2, Z, C, reference_boys=True)
    ds = simint.DeviceShells(basis)
    d_pairs = torch.tensor(np.array(pairs, dtype=np.int32).ravel(), device="cuda")
    d_off = torch.tensor(np.asarray(off, dtype=np.int64), device="cuda")
    ch = torch.tensor(np.column_stack([Z, C]).ravel(), dtype=torch.float64, device="cuda")
    out = torch.full((len(ref) + 1,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ds.compute("potential", len(pairs), d_pairs.data_ptr(), d_off.data_ptr(), out.data_ptr(), ncharge, ch.data_ptr())
    simint.synchronize()
    got = out.cpu().numpy()
    assert np.isnan(got[-1])
    ok, st = parity_report(got[:-1], ref, off, n, ex, floor=REL_FLOOR)
    assert ok, st
    ds.free()
    basis.free()
