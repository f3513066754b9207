"""Primitive screening in the component-lane kernels: a primitive quartet that
is screened in all quartets of a group is left out, with its preparation where
a whole batch is.  Ranges and lists of every launch shape (one wavefront a
group, tops shared between two, four and eight, primitive quartets between
eight) against the oracle's screened integrals.

Bar: 1e-14 max(1, |integral|), or eight times the oracle's own rounding error
on that quartet (its unscreened integrals against the long-double ones) where
that is larger: screening leaves out terms of the same sums."""
import numpy as np
import pytest
import torch

import oracle
import simint
from helpers import normalized_arrays

pytestmark = pytest.mark.gpu

SCHWARZ = simint.SCREEN_SCHWARZ


def _shells(rng, l, n, depth):
    return [(l, tuple(rng.uniform(0, 4, 3)), list(np.exp(rng.uniform(np.log(0.05), np.log(40.0), depth))),
             list(rng.uniform(0.1, 1.0, depth))) for _ in range(n)]


@pytest.mark.parametrize("am,depth", [((1, 1, 1, 0), 4), ((2, 1, 2, 0), 4), ((2, 2, 1, 1), 3), ((2, 2, 2, 2), 3),
                                      ((3, 2, 1, 1), 3), ((3, 3, 3, 3), 2)])
def test_screened(gpu, am, depth):
    rng = np.random.default_rng(sum(x << 2 * k for k, x in enumerate(am)))
    shells = []
    for l in am:
        shells += _shells(rng, l, 3, depth)
    nbra, nket = 3, 6
    bras = [(k, 3 + k) for k in range(nbra)]
    kets = [(6 + k % 3, 9 + (k + k // 3) % 3) for k in range(nket)]
    ql = [b + k for b in bras for k in kets]
    sa = normalized_arrays(shells)
    plain, offs, sizes = oracle.eri(sa, ql)
    exact, _, _ = oracle.md_eri(sa, ql, reference_boys=True)
    basis = simint.Basis(shells)
    hp, hq = simint.Pairs.from_pairs(basis, bras, SCHWARZ), simint.Pairs.from_pairs(basis, kets, SCHWARZ)
    P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
    nc = int(np.prod([simint.ncart(l) for l in am]))
    L = simint.lib()
    prev = L.simint_hip_class_kernel(*am), L.simint_hip_class_list_kernel(*am)
    assert L.simint_hip_set_class_kernel(*am, 7) >= 0 and L.simint_hip_set_class_list_kernel(*am, 7) >= 0
    moved = 0.0
    try:
        for tol in (1e-6, 1e-3, 0.05, 1e3):
            ref, _, _ = oracle.eri(sa, ql, SCHWARZ, tol)
            moved = max(moved, np.abs(ref - plain).max())
            bar = np.maximum(1e-14 * np.maximum(1.0, np.abs(ref)),
                             8.0 * np.repeat([np.abs(plain[o:o + n] - exact[o:o + n]).max()
                                              for o, n in zip(offs, sizes)], sizes))
            out = torch.full((len(ql) * nc,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            simint.compute_range(P, Q, 0, None, np.full(nbra, nket, dtype=np.int32),
                                 nket * nc * np.arange(nbra, dtype=np.int64), out.data_ptr(), tol)
            simint.synchronize()
            assert (np.abs(out.cpu().numpy() - ref) <= bar).all(), ("range", tol)
            # 18 quartets (a list's shortest kernel), over and over for the others
            for n in (18, 18 * 40, 18 * 1500):
                if n * nc > 1 << 27:
                    continue
                q = np.arange(n) % len(ql)
                ib = torch.from_numpy((q // nket).astype(np.int32)).cuda()
                ik = torch.from_numpy((q % nket).astype(np.int32)).cuda()
                out = torch.full((n * nc,), float("nan"), dtype=torch.float64, device="cuda")
                at = torch.from_numpy(nc * np.arange(n, dtype=np.int64)).cuda()
                torch.cuda.synchronize()
                simint.compute_list(P, Q, n, ib.data_ptr(), ik.data_ptr(), at.data_ptr(), out.data_ptr(), tol)
                simint.synchronize()
                got = out.view(-1, len(ql) * nc)
                d = (got - torch.from_numpy(ref).cuda()).abs().amax(dim=0).cpu().numpy()
                assert (d <= bar).all(), ("list", n, tol)
    finally:
        L.simint_hip_set_class_kernel(*am, prev[0])
        L.simint_hip_set_class_list_kernel(*am, prev[1])
    assert moved > 0.0
    for h in (P, Q, hp, hq, basis):
        h.free()
