"""Large results of host-buffer calls cross PCIe through pinned slots that the
process has once, and a few threads copy them on into the caller's buffer.
Several callers at a time: one takes the slots, the others a plain copy, and
all get the device-resident integrals.  While the kernel of a call runs, its
copying threads sleep: the call costs about one processor, not one a thread."""
import ctypes
import threading
import time

import numpy as np
import pytest
import torch

import simint

pytestmark = pytest.mark.gpu


def _pairs(rng, n, depth):
    shells, ij = [], []
    for _ in range(n):
        for _ in range(2):
            shells.append((1, tuple(rng.uniform(0, 4, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20.0), depth))),
                           list(rng.uniform(0.1, 1.0, depth))))
        ij.append((len(shells) - 2, len(shells) - 1))
    basis = simint.Basis(shells)
    return basis, simint.Pairs.from_pairs(basis, ij)


def _call(hp, hq, out):
    return simint.lib().simint_compute_eri(ctypes.byref(hp.mp), ctypes.byref(hq.mp), 0.0, None,
                                           out.ctypes.data_as(simint.dptr))


def test_callers_at_a_time(gpu):
    """Four threads, six calls each, results of 2 to 27 MB (one piece, more
    than the slots, ragged)."""
    rng = np.random.default_rng(2)
    sets = []
    for n in (60, 113, 144, 203):
        basis, hp = _pairs(rng, n, 1)
        P = simint.DevicePairs(hp)
        dev = torch.full((81 * n * n,), float("nan"), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        simint.compute_range(P, P, 0, None, np.full(n, n, dtype=np.int32), 81 * n * np.arange(n, dtype=np.int64),
                             dev.data_ptr())
        simint.synchronize()
        sets.append((basis, hp, P, dev.cpu().numpy()))
    bad = []
    gate = threading.Barrier(4)

    def caller(k):
        gate.wait()
        for r in range(6):
            basis, hp, P, want = sets[(k + r) % 4]
            got = np.full(want.size + 1, np.nan)
            rc = _call(hp, hp, got)
            if rc != hp.mp.nshell12_clip ** 2 or not np.isnan(got[-1]) or not np.array_equal(got[:-1], want):
                bad.append((k, r, rc))
    threads = [threading.Thread(target=caller, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    for basis, hp, P, _ in sets:
        for h in (P, hp, basis):
            h.free()


def test_processor_time_of_a_long_call(gpu):
    """256 x 256 (pp) pairs of depth 12: some 100 ms of kernel, 42 MB of
    results.  The calling thread may spin while it waits (one processor);
    five more busy through the kernel would make it six."""
    basis, hp = _pairs(np.random.default_rng(3), 256, 12)
    got = np.zeros(81 * 256 * 256)
    assert _call(hp, hp, got) == 256 * 256
    c0, t0 = time.process_time(), time.perf_counter()
    assert _call(hp, hp, got) == 256 * 256
    cpu, wall = time.process_time() - c0, time.perf_counter() - t0
    print("processor time %.1f ms in %.1f ms" % (1e3 * cpu, 1e3 * wall))
    assert wall > 0.02 and cpu < 2.5 * wall
    hp.free()
    basis.free()
