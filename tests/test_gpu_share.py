"""Small range launches whose items' primitive quartets several wavefronts
share (eri_lpqk_*, eri_lpqmk_*): bras of 1, 2, 9 and 36 primitives against
kets of 1, 5 and 30 (fewer bra primitives than wavefronts: the ket's are
shared too; fewer of both than wavefronts: some have none), FP64 against the
oracle and the long-double values, FP32-VRR against FP64.

Bar: helpers.parity_report for FP64 (the sum of up to 1080 like terms in
eight parts).  FP32-VRR: each contracted value is a sum of FP32-rounded
terms in FP64, relative error of a term a few 2^-24 per recurrence step; no
HRR in the classes compared, at most 4 steps of 5 operations: 100 x 6e-8 of
the largest integral of the quartet's primitives, taken as 1e-5."""
import numpy as np
import pytest
import torch

import oracle
import simint
from helpers import normalized_arrays, parity_report

pytestmark = pytest.mark.gpu


def _shell(rng, l, n):
    return (l, tuple(rng.uniform(0, 2.5, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(30.0), n))),
            list(rng.uniform(0.1, 1.0, n)))


@pytest.mark.parametrize("am", [(0, 0, 0, 0), (1, 0, 0, 0), (1, 0, 1, 0), (1, 1, 1, 0), (2, 1, 1, 0), (3, 0, 1, 0)])
@pytest.mark.parametrize("bra,ket", [((1, 1), (1, 1)), ((1, 2), (5, 6)), ((3, 3), (1, 5)), ((6, 6), (5, 6))])
def test_shared_items(gpu, am, bra, ket):
    rng = np.random.default_rng(sum(am) * 100 + sum(bra) * 10 + sum(ket))
    shells, pairs = [], [[], []]
    for side, depth, count in ((0, bra, 3), (1, ket, 70)):
        for _ in range(count):
            ij = []
            for l, n in zip(am[2 * side:2 * side + 2], depth):
                ij.append(len(shells))
                shells.append(_shell(rng, l, n))
            pairs[side].append(tuple(ij))
    basis = simint.Basis(shells)
    hp, hq = simint.Pairs.from_pairs(basis, pairs[0]), simint.Pairs.from_pairs(basis, pairs[1])
    P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
    nc = int(np.prod([simint.ncart(l) for l in am]))
    nk = np.array([70, 3, 64], dtype=np.int32)
    off = np.concatenate([[0], np.cumsum(nk * nc)[:-1]]).astype(np.int64)
    L = simint.lib()
    prev = L.simint_hip_class_kernel(*am)
    assert L.simint_hip_set_class_kernel(*am, 1) >= 0
    res = []
    try:
        for prec in (0, 1):
            out = torch.full((int(nk.sum()) * nc + 1,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            simint.compute_range(P, Q, 0, None, nk, off, out.data_ptr(), precision=prec)
            simint.synchronize()
            got = out.cpu().numpy()
            assert np.isnan(got[-1])
            res.append(got[:-1])
    finally:
        L.simint_hip_set_class_kernel(*am, prev)
    sel = [(b, k) for b in range(3) for k in (0, 1, 2, 63, 69) if k < nk[b]]
    ql = [pairs[0][b] + pairs[1][k] for b, k in sel]
    sa = normalized_arrays(shells)
    ref, offs, sizes = oracle.eri(sa, ql)
    ex, _, _ = oracle.md_eri(sa, ql, reference_boys=True)
    at = [int(off[b]) + k * nc for b, k in sel]
    got = np.concatenate([res[0][a:a + nc] for a in at])
    ok, st = parity_report(got, ref, offs, sizes, ex, floor=None)
    assert ok, st
    assert np.isfinite(res[1]).all()
    if not (min(am[0], am[1]) or min(am[2], am[3])):
        a, b = res[0].reshape(-1, nc), res[1].reshape(-1, nc)
        assert (np.abs(a - b).max(axis=1) <= 1e-5 * np.abs(a).max()).all()
    for h in (P, Q, hp, hq):
        h.free()
    basis.free()
