"""Calls of one thread over a change of its stream (simint_hip_set_stream):
what an earlier call left queued on the stream before is not disturbed by the
calls on the next one."""
import ctypes

import numpy as np
import pytest
import torch

import simint

pytestmark = pytest.mark.gpu


def _shells(rng, ls, depth=2):
    return [(l, tuple(rng.uniform(-2, 2, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20.0), depth))),
             list(rng.uniform(0.1, 1.0, depth))) for l in ls]


def _busy(stream):
    """Queue some tens of milliseconds of work on a stream."""
    with torch.cuda.stream(stream):
        a = torch.ones(4096, 4096, dtype=torch.float64, device="cuda")
        b = torch.empty_like(a)
        for _ in range(40):
            torch.mm(a, a, out=b)
    return a, b


def test_one_electron_call_after_diag_on_another_stream(gpu):
    """diag queues the copy of its work items and returns; a one-electron
    drop-in call on the next stream fills the same staging buffer."""
    rng = np.random.default_rng(17)
    shells = _shells(rng, [1] * 24)
    basis = simint.Basis(shells)
    hp = simint.Pairs(basis, list(range(24)), list(range(24)))
    P = simint.DevicePairs(hp)
    want = torch.full((P.n * 81,), float("nan"), dtype=torch.float64, device="cuda")
    got = want.clone()
    torch.cuda.synchronize()
    simint.compute_diag(P, want.data_ptr())
    simint.synchronize()
    charges = (rng.uniform(1, 9, 2000), rng.uniform(-2, 2, (2000, 3)))
    rc, v0 = simint.compute_oei("potential", basis, 0, 1, charges)
    assert rc == 1
    side = torch.cuda.Stream()
    keep = _busy(side)
    L = simint.lib()
    try:
        assert L.simint_hip_set_stream(ctypes.c_void_p(side.cuda_stream)) == 0
        simint.compute_diag(P, got.data_ptr())
    finally:
        L.simint_hip_set_stream(None)
    rc, v1 = simint.compute_oei("potential", basis, 0, 1, charges)
    assert rc == 1 and np.array_equal(v0, v1)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and bool(torch.isfinite(want).all())
    del keep
    for h in (P, hp, basis):
        h.free()


def _range(rng, nbra, nket):
    """A (ps|ps) range call: pair handles, its arguments and its integrals."""
    shells = _shells(rng, [1, 0] * (nbra + nket))
    ij = [(2 * k, 2 * k + 1) for k in range(nbra + nket)]
    basis = simint.Basis(shells)
    hp, hq = simint.Pairs.from_pairs(basis, ij[:nbra]), simint.Pairs.from_pairs(basis, ij[nbra:])
    P, Q = simint.DevicePairs(hp), simint.DevicePairs(hq)
    args = (P, Q, 0, None, np.full(nbra, nket, dtype=np.int32), 9 * nket * np.arange(nbra, dtype=np.int64))
    want = torch.full((9 * nbra * nket,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    simint.compute_range(*args, want.data_ptr())
    simint.synchronize()
    return (P, Q, hp, hq, basis), args, want


def test_stream_destroyed_before_it_is_left(gpu):
    """The stream a range call ran on is gone when the thread leaves it; a new
    one may have its address."""
    hip = simint.lib()   # its own HIP runtime's symbols resolve through it
    handles, args, want = _range(np.random.default_rng(5), 40, 90)
    outs = []
    for k in range(4):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        assert hip.simint_hip_set_stream(s) == 0
        for _ in range(2):
            outs.append(torch.full_like(want, float("nan")))
            torch.cuda.synchronize()
            simint.compute_range(*args, outs[-1].data_ptr())
        simint.synchronize()
        assert hip.hipStreamDestroy(s) == 0
        if k % 2:
            assert hip.simint_hip_set_stream(None) == 0
            outs.append(torch.full_like(want, float("nan")))
            torch.cuda.synchronize()
            simint.compute_range(*args, outs[-1].data_ptr())
            simint.synchronize()
    assert hip.simint_hip_set_stream(None) == 0
    for o in outs:
        assert torch.equal(o, want)
    for h in handles:
        h.free()


def test_ranges_behind_work_of_the_stream_left(gpu):
    """Range calls on a stream that is busy, then others on the thread's own:
    the second ones' items take the place of the first ones' only once those
    have run."""
    rng = np.random.default_rng(6)
    h1, args1, want1 = _range(rng, 60, 200)
    h2, args2, want2 = _range(rng, 200, 60)
    got1, got2 = torch.full_like(want1, float("nan")), torch.full_like(want2, float("nan"))
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    keep = _busy(side)
    L = simint.lib()
    try:
        assert L.simint_hip_set_stream(ctypes.c_void_p(side.cuda_stream)) == 0
        simint.compute_range(*args1, got1.data_ptr())
        assert L.simint_hip_set_stream(None) == 0
        simint.compute_range(*args2, got2.data_ptr())
        assert L.simint_hip_set_stream(ctypes.c_void_p(side.cuda_stream)) == 0
        simint.compute_range(*args1, got1.data_ptr())
    finally:
        L.simint_hip_set_stream(None)
    torch.cuda.synchronize()
    assert torch.equal(got1, want1) and torch.equal(got2, want2)
    del keep
    for h in h1 + h2:
        h.free()
