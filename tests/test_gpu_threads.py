"""Several host threads: derivative ranges whose terms run on the side streams
that the threads share, and calls that must be able to run side by side on the
card (each thread's own stream among the hardware queues, not all on one)."""
import ctypes
import threading
import time

import numpy as np
import pytest
import torch

import simint
from test_gpu_queue import _pairs

pytestmark = pytest.mark.gpu


def _run(fs):
    """The functions in a thread each, all started together; wall time."""
    gate = threading.Barrier(len(fs) + 1)
    bad = []

    def body(f):
        try:
            gate.wait()
            f()
            gate.wait()
        except Exception as e:   # noqa: BLE001 -- reported by the assertion below
            bad.append(e)
            gate.abort()
    ts = [threading.Thread(target=body, args=(f,)) for f in fs]
    for t in ts:
        t.start()
    t0 = 0.0
    try:
        gate.wait()
        t0 = time.perf_counter()
        gate.wait()
    except threading.BrokenBarrierError:
        pass
    wall = time.perf_counter() - t0
    for t in ts:
        t.join()
    assert not bad, bad
    return wall


def test_derivative_ranges_of_several_threads(gpu):
    sets = []
    for k, (am, nbra, nket) in enumerate([((1, 1, 2, 1), 6, 70), ((2, 1, 2, 0), 5, 66), ((3, 1, 1, 0), 3, 20),
                                          ((1, 0, 1, 0), 40, 90)]):
        rng = np.random.default_rng(40 + k)
        bb, hp, P = _pairs(rng, am[:2], nbra)
        bk, hq, Q = _pairs(rng, am[2:], nket)
        nc = 12 * int(np.prod([simint.ncart(l) for l in am]))
        hi = np.full(nbra, nket, dtype=np.int32)
        want = torch.full((nbra * nket * nc,), float("nan"), dtype=torch.float64, device="cuda")
        work = torch.empty(simint.deriv1_worksize(P, Q, nbra * nket), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        simint.compute_deriv1_range(P, Q, 0, None, hi, work.data_ptr(), want.data_ptr())
        simint.synchronize()
        assert bool(torch.isfinite(want).all())
        outs = [torch.full_like(want, float("nan")) for _ in range(8)]
        sets.append((P, Q, hi, work, want, outs, (hp, hq, bb, bk)))
    torch.cuda.synchronize()

    def caller(s):
        def f():
            for o in s[5]:
                simint.compute_deriv1_range(s[0], s[1], 0, None, s[2], s[3].data_ptr(), o.data_ptr())
            simint.synchronize()
        return f
    _run([caller(s) for s in sets])
    for P, Q, hi, work, want, outs, hs in sets:
        for o in outs:
            assert torch.equal(o, want)
        for h in (P, Q) + hs:
            h.free()


def test_calls_of_several_threads_side_by_side(gpu):
    """One call of 130 (pp) pairs with 64 of depth 11 is 130 wavefronts, an
    eighth of the card's SIMDs, for some 30 ms.  Four threads' calls one after
    another would take four times one; over the four hardware queues at most
    two of the streams share one, so twice."""
    rng = np.random.default_rng(9)
    bb, hp, P = _pairs(rng, (1, 1), 130, depth=11)
    bk, hq, Q = _pairs(rng, (1, 1), 64, depth=11)
    P.free()
    Q.free()

    def caller():
        out = np.zeros(81 * 130 * 64)
        for _ in range(3):
            assert simint.lib().simint_compute_eri(ctypes.byref(hp.mp), ctypes.byref(hq.mp), 0.0, None,
                                                   out.ctypes.data_as(simint.dptr)) == 130 * 64
    caller()
    one = min(_run([caller]) for _ in range(3))
    four = min(_run([caller] * 4) for _ in range(3))
    print("one thread %.1f ms, four %.1f ms" % (1e3 * one, 1e3 * four))
    assert one > 0.01 and four < 2.5 * one
    for h in (hp, hq, bb, bk):
        h.free()
