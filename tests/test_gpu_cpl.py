"""Component-lane kernels (emitter/hip_cpl.py) through their three entry
paths, each against the CPU oracle and the long-double values.

Bar: helpers.parity_report with the long-double values (per quartet at most
4x the oracle's own error where that is above 1e-14; the batch's worst and
median normwise errors at most 4x the oracle's).  The kernels transfer the
side of the smaller AM first, the oracle always the bra, so quartets of
bra-heavy classes round differently; the relative bar against the oracle
(1e-14 for quartets above 0.1) is kept."""
import itertools

import numpy as np
import pytest

import batch
import oracle
import simint
from helpers import normalized_arrays, parity_report
from test_gpu_batch import _pool, _stream
from test_gpu_eri import _f_shells

pytestmark = pytest.mark.gpu

CPL = simint.FAMILIES["cpl"]


def _select(setter, getter, classes, family):
    """Select a family where it is built; returns what was selected before."""
    prev = {}
    for am in classes:
        p = getter(*am)
        if setter(*am, family) >= 0:
            prev[am] = p
    return prev


@pytest.mark.parametrize("per_class,maxk,seed", [(1, 6, 1), (3, 2, 2)])
def test_lists_every_class(gpu, per_class, maxk, seed):
    """Short lists (the split kernels: one group of quartets a workgroup,
    its primitives shared), depths 1-6 mixed within a group, a repeated
    quartet and same-shell pairs."""
    import torch
    shells = _pool(seed=seed, per_am=6, maxk=maxk)
    basis = simint.Basis(shells)
    sa = normalized_arrays(shells)
    qs = _stream(shells, per_class=per_class, seed=seed)
    L = simint.lib()
    prev = _select(L.simint_hip_set_class_list_kernel, L.simint_hip_class_list_kernel,
                   itertools.product(range(4), repeat=4), CPL)
    assert len(prev) >= 190
    try:
        b = batch.QuartetBatch(basis, qs)
        out = torch.full((b.out_doubles,), float("nan"), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        b.run(out.data_ptr())
        simint.synchronize()
        got = out.cpu().numpy()
    finally:
        for am, f in prev.items():
            L.simint_hip_set_class_list_kernel(*am, f)
    ql = [tuple(x) for x in qs]
    ref, offs, sizes = oracle.eri(sa, ql)
    ex, _, _ = oracle.md_eri(sa, ql, reference_boys=True)
    ok, st = parity_report(got, ref, offs, sizes, ex)
    assert ok, st
    b.free()
    basis.free()


@pytest.mark.parametrize("am,n", [((2, 1, 2, 1), 12400), ((3, 1, 1, 1), 12300), ((1, 1, 2, 2), 12301)])
def test_long_lists_equal_short_ones(gpu, am, n):
    """A list above the split kernels' limit (a run of groups per wavefront,
    the last group partial) gives the values of the same quartets in short
    lists: the per-primitive arithmetic is the same, only the contraction
    order differs (at most 16 primitives of like size a quartet here, so a
    few ulp of the largest integral)."""
    import torch
    shells = [s for s in _pool(seed=9, per_am=8, maxk=2)]
    basis = simint.Basis(shells)
    rng = np.random.default_rng(3)
    by = {l: [i for i, s in enumerate(shells) if s[0] == l] for l in range(4)}
    few = np.array([[rng.choice(by[l]) for l in am] for _ in range(37)])
    long_ = few[np.arange(n) % len(few)]
    L = simint.lib()
    prev = _select(L.simint_hip_set_class_list_kernel, L.simint_hip_class_list_kernel, [am], CPL)
    assert prev
    res = []
    try:
        for q in (few, long_):
            b = batch.QuartetBatch(basis, q)
            out = torch.full((b.out_doubles,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            b.run(out.data_ptr())
            simint.synchronize()
            res.append(out.cpu().numpy().reshape(len(q), -1))
            b.free()
    finally:
        L.simint_hip_set_class_list_kernel(*am, prev[am])
    a, c = res[0][np.arange(n) % len(few)], res[1]
    assert np.isfinite(c).all()
    # the transfers amplify the ulp of the contracted inputs by at most the
    # pairs' extent in a 6-bohr cube to the power of the transferred AM
    amp = 11.0 ** (min(am[0], am[1]) + min(am[2], am[3]))
    assert np.abs(a - c).max() <= 64 * 2.2e-16 * amp * np.abs(a).max()
    basis.free()


def test_ranges_every_class(gpu):
    """Prefix launches of one item and of many, tiles of partial lanes
    (ket_lo inside a tile, ket_hi not a multiple of 64), every class up to f
    that has the family."""
    import torch
    shells = _f_shells(seed=21)
    basis = simint.Basis(shells)
    sa = normalized_arrays(shells)
    by = {l: [i for i, s in enumerate(shells) if s[0] == l] for l in range(4)}
    L = simint.lib()
    classes = list(itertools.product(range(4), repeat=4))
    prev = _select(L.simint_hip_set_class_kernel, L.simint_hip_class_kernel, classes, CPL)
    assert len(prev) >= 190
    try:
        for am in prev:
            pb = [(i, j) for i in by[am[0]] for j in by[am[1]]][:3]
            pk = [(i, j) for i in by[am[2]] for j in by[am[3]]] * 20      # 80 kets: a full and a partial tile
            hp, hq = simint.Pairs.from_pairs(basis, pb), simint.Pairs.from_pairs(basis, pk)
            P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
            nc = int(np.prod([simint.ncart(l) for l in am]))
            lo, hi = np.array([0, 61, 66], dtype=np.int32), np.array([1, 67, 66 + (sum(am) % 5)], dtype=np.int32)
            off = np.concatenate([[0], np.cumsum((hi - lo) * nc)[:-1]]).astype(np.int64)
            n = int((hi - lo).sum())
            out = torch.full((n * nc + 1,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            simint.compute_range(P, Q, 0, lo, hi, off, out.data_ptr())
            simint.synchronize()
            got = out.cpu().numpy()
            assert np.isnan(got[-1])
            ql = [pb[b] + pk[k] for b in range(3) for k in range(lo[b], hi[b])]
            ref, offs, sizes = oracle.eri(sa, ql)
            ex, _, _ = oracle.md_eri(sa, ql, reference_boys=True)
            ok, st = parity_report(got[:-1], ref, offs, sizes, ex)
            assert ok, (am, st)
            for h in (P, Q, hp, hq):
                h.free()
    finally:
        for am, f in prev.items():
            L.simint_hip_set_class_kernel(*am, f)
    basis.free()


def test_ranges_primitive_screen(gpu):
    """The primitive screen inside the kernel: skipped primitive quartets
    contribute nothing, as in the oracle's restatement."""
    shells = _f_shells(seed=33)
    basis = simint.Basis(shells)
    sa = normalized_arrays(shells)
    from test_gpu_eri import _check
    by = {l: [i for i, s in enumerate(shells) if s[0] == l] for l in range(4)}
    L = simint.lib()
    classes = [(2, 1, 2, 1), (2, 2, 1, 1), (1, 1, 2, 2), (3, 1, 2, 0)]
    prev = _select(L.simint_hip_set_class_kernel, L.simint_hip_class_kernel, classes, CPL)
    assert len(prev) == len(classes)
    try:
        for am in classes:
            _check(sa, basis, *[by[l] for l in am], simint.SCREEN_SCHWARZ, 1e-6)
    finally:
        for am, f in prev.items():
            L.simint_hip_set_class_kernel(*am, f)
    basis.free()
