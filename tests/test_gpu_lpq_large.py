"""The lane-per-quartet range kernels as large launches run them.

A launch of few items runs other kernels than a large one (several wavefronts
an item, or the component-lane kernel of the class), also where family 1 is
selected; here every class that has a lane-per-quartet kernel runs it, on 2048
items: four bras over and over against three kets.

  * Every repetition has the same values, bit for bit.
  * They hold helpers.parity_report against the oracle and the long-double
    values (no floor: random quartets of all sizes).
  * The same quartets in launches of four items agree with them bit for bit:
    the kernels small launches run keep the order of every sum.  Classes
    without HRR whose wavefronts each sum a share of the primitive quartets
    (emitter share_kind "sum") add up to eight partial sums in place of one:
    there 16 roundings of 2^-53 of the sum of the terms' magnitudes, itself
    taken as at most 100 of the largest integral.
  * FP32-VRR (precision 1): finite, not the FP64 values, and within 1e-3 of the
    largest integral: 40 operations of 2^-24, times the HRR of up to four
    units over distances up to 4.4 bohr, 5.4^4 = 850 at most, is 2e-3 of the
    largest intermediate if everything conspires."""
import itertools

import numpy as np
import pytest
import torch

import oracle
import simint
from emitter import hip_lpq
from helpers import normalized_arrays, parity_report

pytestmark = pytest.mark.gpu

ITEMS = 2048


def _shell(rng, l, n):
    return (l, tuple(rng.uniform(0, 2.5, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(30.0), n))),
            list(rng.uniform(0.1, 1.0, n)))


@pytest.mark.parametrize("la,lb", list(itertools.product(range(4), repeat=2)))
def test_large_launches(gpu, la, lb):
    L = simint.lib()
    ran = 0
    for lc, ld in itertools.product(range(4), repeat=2):
        am = (la, lb, lc, ld)
        prev = L.simint_hip_class_kernel(*am)
        if L.simint_hip_set_class_kernel(*am, 1) < 0:
            continue
        rng = np.random.default_rng(1000 * la + 100 * lb + 10 * lc + ld)
        shells = []
        for _ in range(4):
            shells += [_shell(rng, la, 3), _shell(rng, lb, 2)]
        for _ in range(3):
            shells += [_shell(rng, lc, 2), _shell(rng, ld, 1)]
        bras = [(2 * k, 2 * k + 1) for k in range(4)]
        kets = [(8 + 2 * k, 9 + 2 * k) for k in range(3)]
        basis = simint.Basis(shells)
        hp, hq = simint.Pairs.from_pairs(basis, bras * (ITEMS // 4)), simint.Pairs.from_pairs(basis, kets)
        P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
        nc = int(np.prod([simint.ncart(l) for l in am]))

        def call(n, precision=0):
            out = torch.full((n * 3 * nc,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            simint.compute_range(P, Q, 0, None, np.full(n, 3, dtype=np.int32),
                                 3 * nc * np.arange(n, dtype=np.int64), out.data_ptr(), precision=precision)
            simint.synchronize()
            return out.view(-1, 12 * nc)
        try:
            big, small = call(ITEMS), call(4)
            low = call(ITEMS, 1) if max(am) <= 2 else None
        finally:
            L.simint_hip_set_class_kernel(*am, prev)
        assert bool((big == big[0]).all()), am
        got = big[0].cpu().numpy()
        ql = [b + k for b in bras for k in kets]
        sa = normalized_arrays(shells)
        ref, offs, sizes = oracle.eri(sa, ql)
        ex, _, _ = oracle.md_eri(sa, ql, reference_boys=True)
        ok, st = parity_report(got, ref, offs, sizes, ex, floor=None)
        assert ok, (am, st)
        if hip_lpq.share_kind(am) == "sum":
            d = (small[0] - big[0]).abs().max().item()
            assert d <= 16 * 2.0 ** -53 * 100 * np.abs(ref).max(), (am, d)
        else:
            assert torch.equal(small[0], big[0]), (am, (small[0] - big[0]).abs().max().item())
        if low is not None:
            assert bool((low == low[0]).all()), am
            d = np.abs(low[0].cpu().numpy() - ref).max()
            assert 0.0 < d <= 1e-3 * np.abs(ref).max(), (am, d)
            assert not torch.equal(low[0], big[0]), am
        ran += 1
        for h in (P, Q, hp, hq, basis):
            h.free()
    assert ran >= 6
