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
