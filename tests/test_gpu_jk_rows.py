"""The per-bra J/K digestion against the one that adds every lane's updates
to global memory: few items (divided between a block's wavefronts) and more
than 1024, a block alone on its compute unit, no room in the local data share
for the lanes' sums of J_ab (nbf 1690 with a (dd| bra: 162 KB of rows, 9 KB or
more of sums, 160 KB in all), classes whose integrals are kept two a at a
time and classes that load row by row, ket ranges that start inside a tile.

Both sum the same products in other orders: normwise 1e-12, the bar of the
digestion against the oracle."""
import numpy as np
import pytest
import torch

import simint
from test_gpu_queue import _pairs

pytestmark = pytest.mark.gpu


def _digest(P, Q, lo, hi, off, out, nbf, funs, D, rows):
    J, K = (torch.zeros((nbf, nbf), dtype=torch.float64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    jk = simint.JK(nbf, 0, funs[0].data_ptr(), funs[1].data_ptr(), D.data_ptr(), J.data_ptr(), K.data_ptr())
    prev = simint.lib().simint_hip_set_jk_rows(rows)
    try:
        simint.compute_jk_range(P, Q, 0, lo, hi, off, out.data_ptr(), jk)
        simint.synchronize()
    finally:
        simint.lib().simint_hip_set_jk_rows(prev)
    return J, K


@pytest.mark.parametrize("am,nbra,nket,nbf", [
    ((0, 0, 0, 0), 7, 90, 60), ((1, 0, 0, 0), 45, 1600, 300), ((1, 1, 1, 1), 9, 70, 150), ((2, 0, 1, 1), 5, 130, 200),
    ((2, 1, 2, 2), 4, 65, 150), ((2, 2, 0, 0), 20, 70, 1690), ((2, 2, 1, 0), 30, 2300, 1200),
    ((2, 2, 2, 0), 3, 40, 150), ((3, 1, 1, 0), 4, 70, 120), ((3, 2, 3, 1), 2, 12, 120)])
def test_rows_against_atomics(gpu, am, nbra, nket, nbf):
    rng = np.random.default_rng(nbf + sum(am))
    bb, hp, P = _pairs(rng, am[:2], nbra, depth=1)
    bk, hq, Q = _pairs(rng, am[2:], nket, depth=1)
    nc = int(np.prod([simint.ncart(l) for l in am]))
    lo = rng.integers(0, nket // 3 + 1, nbra).astype(np.int32)
    hi = np.full(nbra, nket, dtype=np.int32)
    seg = (hi - lo).astype(np.int64) * nc
    off = np.concatenate([[0], np.cumsum(seg)[:-1]])
    out = torch.empty(int(seg.sum()), dtype=torch.float64, device="cuda")
    funs = [torch.from_numpy(rng.integers(0, nbf - 9, 2 * n).astype(np.int32)).cuda() for n in (nbra, nket)]
    D = torch.from_numpy(rng.uniform(-1, 1, (nbf, nbf))).cuda()
    D = (D + D.T).contiguous()
    J0, K0 = _digest(P, Q, lo, hi, off, out, nbf, funs, D, 0)
    J1, K1 = _digest(P, Q, lo, hi, off, out, nbf, funs, D, 1)
    for a, b in ((J1, J0), (K1, K0)):
        assert float(b.abs().max()) > 0
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
    for h in (P, Q, hp, hq, bb, bk):
        h.free()
