"""Which kernel a call runs by its size: on both sides of each line the call
with the built choice gives, bit for bit, what the family named there gives
when it is set.

  * (dp|dp) and (dd|pp) ranges: component-lane kernel below 1024 items or 16
    primitive quartets, the ket-top split kernel (family 5) from there on.
  * Lists: where the build chose component-lane kernels for streams of mixed
    depth, lists of even depth run the lane-per-quartet kernel from the class's
    "list_even" primitive quartets of tuning.json on; lists of uneven depth and
    shorter ones do not; nor does a class whose family was set.
  * The lists' values against the oracle (helpers.parity_report with the
    long-double values), on both sides.
  * simint_hip_reset_class_kernels brings the built choice back."""
import json
import os

import numpy as np
import pytest
import torch

import oracle
import simint
from conftest import PKG
from helpers import normalized_arrays, parity_report

pytestmark = pytest.mark.gpu

EVEN = json.load(open(os.path.join(PKG, "tuning.json")))["list_even"]


@pytest.fixture(autouse=True)
def built_choice(gpu):
    simint.lib().simint_hip_reset_class_kernels()
    yield
    simint.lib().simint_hip_reset_class_kernels()


def _am(name):
    return tuple("spdf".index(c) for c in name.split("_"))


def _pairs(rng, l1, l2, depths):
    """Pairs of shells of the given depths (a pair of depth d has d primitives
    on its first shell and one on the other)."""
    shells = []
    for d in depths:
        for l, n in ((l1, d), (l2, 1)):
            shells.append((l, tuple(rng.uniform(0, 2.5, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20.0), n))),
                           list(rng.uniform(0.1, 1.0, n))))
    return shells, [(2 * k, 2 * k + 1) for k in range(len(depths))]


def _device(shells, pairs, count):
    basis = simint.Basis(shells)
    hp = simint.Pairs.from_pairs(basis, [pairs[k % len(pairs)] for k in range(count)])
    P = simint.DevicePairs(hp)
    hp.free()
    basis.free()
    return P


@pytest.mark.parametrize("am", [(2, 1, 2, 1), (2, 2, 1, 1)])
def test_deep_ranges(gpu, am):
    L = simint.lib()
    rng = np.random.default_rng(sum(am))
    nc = int(np.prod([simint.ncart(l) for l in am]))
    for db, dk, items, family in ((4, 4, 1024, 5), (4, 4, 1023, 7), (5, 3, 1024, 7), (4, 5, 1100, 5)):
        P = _device(*_pairs(rng, am[0], am[1], [db] * 8), items)
        Q = _device(*_pairs(rng, am[2], am[3], [dk] * 2), 2)

        def call():
            out = torch.full((items * 2 * nc,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            simint.compute_range(P, Q, 0, None, np.full(items, 2, dtype=np.int32),
                                 2 * nc * np.arange(items, dtype=np.int64), out.data_ptr())
            simint.synchronize()
            return out
        built = call()
        assert L.simint_hip_set_class_kernel(*am, family) == 7
        want = call()
        assert bool(torch.isfinite(want).all()) and torch.equal(built, want), (db, dk, items)
        assert L.simint_hip_set_class_kernel(*am, 7) == family
        component = call()                    # set, so it stays
        if family == 7:
            assert torch.equal(component, want)
        else:
            d = (component - want).abs().max().item()
            assert d <= 1e-12 * want.abs().max().item(), d
        L.simint_hip_reset_class_kernels()
        assert L.simint_hip_class_kernel(*am) == 7 and torch.equal(call(), built)
        P.free()
        Q.free()


@pytest.mark.parametrize("name", sorted(EVEN))
def test_even_lists(gpu, name):
    L = simint.lib()
    am = _am(name)
    nc = int(np.prod([simint.ncart(l) for l in am]))
    rng = np.random.default_rng(sum(x << 2 * k for k, x in enumerate(am)))
    assert L.simint_hip_class_list_kernel(*am) == 7
    shallow, deep = EVEN[name]
    for even in (True, False):
        for line, db, dk in ((shallow, 3, 2), (deep, 4, 5)):
            # one deep bra among shallow ones: the same depth, not even
            sa, pa = _pairs(rng, am[0], am[1], [db] * 6 if even else [db] + [1] * 5)
            sb, pb = _pairs(rng, am[2], am[3], [dk] * 6 if even else [dk] + [1] * 5)
            P, Q = _device(sa, pa, 6), _device(sb, pb, 6)
            base = line or 12800
            for n in (-(-base // (db * dk)), -(-base // (db * dk)) - 1):
                if n * nc > 1 << 27:
                    continue
                q = np.arange(n) % 36
                ib = torch.from_numpy((q // 6).astype(np.int32)).cuda()
                ik = torch.from_numpy((q % 6).astype(np.int32)).cuda()
                at = torch.from_numpy(nc * np.arange(n, dtype=np.int64)).cuda()

                def call():
                    out = torch.full((n * nc,), float("nan"), dtype=torch.float64, device="cuda")
                    torch.cuda.synchronize()
                    simint.compute_list(P, Q, n, ib.data_ptr(), ik.data_ptr(), at.data_ptr(), out.data_ptr())
                    simint.synchronize()
                    return out
                built = call()
                family = 1 if even and line and n * db * dk >= line else 7
                assert L.simint_hip_set_class_list_kernel(*am, family) == 7
                assert torch.equal(built, call()), (even, line, n)
                L.simint_hip_reset_class_kernels()
                if n >= 36 and (db, dk) == (4, 5):
                    shells = sa + sb
                    ql = [pa[i] + tuple(len(sa) + x for x in pb[k]) for i in range(6) for k in range(6)]
                    arr = normalized_arrays(shells)
                    ref, offs, sizes = oracle.eri(arr, ql)
                    ex, _, _ = oracle.md_eri(arr, ql, reference_boys=True)
                    ok, st = parity_report(built[:36 * nc].cpu().numpy(), ref, offs, sizes, ex, floor=None)
                    assert ok, (name, st)
            P.free()
            Q.free()
