"""Derivative lists whose terms add a quartet's primitive quartets in another
order than one lane does (several lanes a quartet, several wavefronts a group):
classes whose terms transfer up to two units of AM by HRR, contractions of up
to 1296 primitive quartets.  Accuracy: helpers.parity_report_deriv against the
analytic long-double derivatives.  Against the range call, which keeps the
order, the list may move by 1e-9 of its norm: 1296 terms of 2^-53 each, a
factor of 6^2 for two transfers over up to 5 bohr and 200 for the weight 2a
with exponents up to 100."""
import os
import re

import numpy as np
import pytest
import torch

import oracle
import simint
from conftest import PKG
from helpers import normalized_arrays, parity_report_deriv


def test_one_limit():
    """The two list families share the limit."""
    from emitter import hip_cpl
    text = open(os.path.join(PKG, "csrc", "runtime.hip")).read()
    assert int(re.search(r"constexpr int kReorderAM = (\d+);", text)[1]) == hip_cpl.SHARE_AM
    assert "lanes[k] = std::min(t.am[0], t.am[1]) + std::min(t.am[2], t.am[3]) <= kReorderAM;" in text
    assert "if (lanes[k]) a.split = list_split(" in text


@pytest.mark.gpu
@pytest.mark.parametrize("am", [(1, 1, 1, 0), (1, 1, 1, 1), (0, 2, 1, 1), (2, 1, 2, 0), (2, 1, 1, 0), (2, 2, 0, 1)])
def test_deep_derivative_lists(gpu, am):
    rng = np.random.default_rng(sum(x << 2 * k for k, x in enumerate(am)))
    nq = 6
    shells = [(l, tuple(rng.uniform(0, 3, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(100.0), 6))),
               list(rng.uniform(0.1, 1.0, 6))) for _ in range(nq) for l in am]
    ql = [tuple(range(4 * k, 4 * k + 4)) for k in range(nq)]
    basis = simint.Basis(shells)
    hp = simint.Pairs.from_pairs(basis, [q[:2] for q in ql])
    hq = simint.Pairs.from_pairs(basis, [q[2:] for q in ql])
    P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
    nc = 12 * int(np.prod([simint.ncart(l) for l in am]))
    idx = torch.arange(nq, dtype=torch.int32, device="cuda")
    at = nc * torch.arange(nq, dtype=torch.int64, device="cuda")
    work = torch.empty(simint.deriv1_worksize(P, Q, nq), dtype=torch.float64, device="cuda")
    out = [torch.full((nq * nc,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    simint.compute_deriv1_list(P, Q, nq, idx.data_ptr(), idx.data_ptr(), at.data_ptr(), work.data_ptr(),
                               out[0].data_ptr())
    # bra k against ket k alone
    lo = np.arange(nq, dtype=np.int32)
    simint.compute_deriv1_range(P, Q, 0, lo, lo + 1, work.data_ptr(), out[1].data_ptr())
    simint.synchronize()
    got, one = (o.cpu().numpy() for o in out)
    sa = normalized_arrays(shells)
    ref, offs, sizes = oracle.eri(sa, ql, deriv=1)
    ex, _, _ = oracle.md_eri_deriv1_analytic(sa, ql)
    for x in (got, one):
        ok, st = parity_report_deriv(x, ref, offs, sizes, ex)
        assert ok, st
    d = np.linalg.norm(got - one) / np.linalg.norm(one)
    print(am, "list against range: %.1e of the norm" % d)
    assert d <= 1e-9
    for h in (P, Q, hp, hq, basis):
        h.free()
