"""Small derivative ranges run their terms on side streams.

Calls of changing ranges share the caller's work buffer and the thread's
item and staging buffers, so a term that starts before its inputs are there,
or that is not waited for before the assembly or the next call, leaves wrong
derivatives: 24 calls queued without a wait are compared bit for bit with
the same calls waited for one by one.  Classes without staging kernels among
their terms, with some, and above the line of 2048 items (one stream)."""
import numpy as np
import pytest
import torch

import simint
from test_gpu_queue import _pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("am,nbra,nket", [((0, 0, 0, 0), 40, 130), ((1, 1, 2, 1), 6, 70), ((2, 1, 2, 0), 5, 66),
                                          ((3, 1, 1, 0), 3, 20), ((1, 0, 0, 0), 700, 200)])
def test_terms_side_by_side(gpu, am, nbra, nket):
    rng = np.random.default_rng(sum(am) + nbra)
    bb, hp, P = _pairs(rng, am[:2], nbra)
    bk, hq, Q = _pairs(rng, am[2:], nket)
    nc = 12 * int(np.prod([simint.ncart(l) for l in am]))
    plan = []
    for k in range(24):
        b0 = int(rng.integers(0, nbra)) if k % 4 else 0
        n = int(rng.integers(1, nbra - b0 + 1)) if k % 4 else nbra
        lo = None if k % 3 == 0 else rng.integers(0, nket // 2, n).astype(np.int32)
        hi = rng.integers(nket // 2, nket + 1, n).astype(np.int32)
        hi[0] = nket
        plan.append((b0, lo, hi, int((hi - (0 if lo is None else lo)).sum())))
    most = max(p[3] for p in plan)
    work = torch.empty(simint.deriv1_worksize(P, Q, most), dtype=torch.float64, device="cuda")
    size = sum(p[3] for p in plan) * nc
    ref = torch.full((size,), float("nan"), dtype=torch.float64, device="cuda")
    out = ref.clone()
    torch.cuda.synchronize()
    for dst, wait in ((ref, True), (out, False)):
        at = 0
        for b0, lo, hi, nq in plan:
            assert simint.compute_deriv1_range(P, Q, b0, lo, hi, work.data_ptr(), dst.data_ptr() + 8 * at) == nq
            at += nq * nc
            if wait:
                simint.synchronize()
    simint.synchronize()
    assert not bool(torch.isnan(ref).any())
    assert torch.equal(out, ref)
    for h in (P, Q, hp, hq, bb, bk):
        h.free()
