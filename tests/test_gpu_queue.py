"""Range launches queued one behind another, and results on their way into a
caller's buffer.

Range launches describe their ranges in a ring of pinned memory (two halves
of 1 MiB) and share the thread's item and staging buffers: many launches of
changing ranges are queued without a wait, past both ends of the ring, over
a change of stream, and compared bit for bit with the same launches waited
for one by one.  A host-buffer call copies its results back in one kernel up
to 1 MiB and in 4 MiB pieces through four slots above: sizes at both edges,
one piece, a ragged last piece and more pieces than slots, against the
device-resident integrals of the same kernel."""
import ctypes

import numpy as np
import pytest
import torch

import simint

pytestmark = pytest.mark.gpu


def _pairs(rng, am, n, depth=2):
    shells, ij = [], []
    for _ in range(n):
        for l in am:
            shells.append((l, tuple(rng.uniform(0, 4, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20.0), depth))),
                           list(rng.uniform(0.1, 1.0, depth))))
        ij.append((len(shells) - 2, len(shells) - 1))
    basis = simint.Basis(shells)
    host = simint.Pairs.from_pairs(basis, ij)
    return basis, host, simint.DevicePairs(host)


@pytest.mark.parametrize("am", [(0, 0, 0, 0), (1, 1, 1, 0), (2, 2, 1, 1)])
def test_queued_ranges(gpu, am):
    rng = np.random.default_rng(7 + sum(am))
    nbra, nket, count = 150, 130, 24
    bb, hp, P = _pairs(rng, am[:2], nbra)
    bk, hq, Q = _pairs(rng, am[2:], nket)
    nc = int(np.prod([simint.ncart(l) for l in am]))
    plan, room = [], 0
    for k in range(count):
        b0 = int(rng.integers(0, nbra - 1))
        n = int(rng.integers(1, nbra - b0 + 1))
        lo = rng.integers(0, nket, n).astype(np.int32)
        hi = np.minimum(nket, lo + rng.integers(0, 90, n)).astype(np.int32)
        if k % 3 == 0:
            lo = None
        seg = (hi - (0 if lo is None else lo)).astype(np.int64) * nc
        off = room + np.concatenate([[0], np.cumsum(seg)[:-1]])
        room += int(seg.sum())
        plan.append((b0, lo, hi, off))
    ref = torch.full((room + 1,), float("nan"), dtype=torch.float64, device="cuda")
    out = ref.clone()
    torch.cuda.synchronize()
    for p in plan:
        simint.compute_range(P, Q, *p, ref.data_ptr())
        simint.synchronize()
    # about 2 KB a launch: enough rounds to pass both halves' ends twice
    rounds = 4 * (1 << 20) // sum(len(p[2]) * 20 for p in plan) + 2
    side = torch.cuda.Stream()
    L = simint.lib()
    try:
        for r in range(rounds):
            if r % 8 == 5:
                L.simint_hip_set_stream(ctypes.c_void_p(side.cuda_stream))
            if r % 8 == 7:
                L.simint_hip_set_stream(None)
            for p in plan if r < rounds - 1 else plan[::-1]:
                simint.compute_range(P, Q, *p, out.data_ptr())
    finally:
        L.simint_hip_set_stream(None)
    torch.cuda.synchronize()
    assert torch.equal(out[:-1], ref[:-1])
    assert bool(torch.isnan(out[-1])) and not bool(torch.isnan(out[:-1]).any())
    for h in (P, Q, hp, hq, bb, bk):
        h.free()


def test_range_refused_under_capture(gpu):
    rng = np.random.default_rng(3)
    b, hp, P = _pairs(rng, (1, 0), 5)
    out = torch.zeros(5 * 5 * 9, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    n = np.full(5, 5, dtype=np.int32)
    off = 45 * np.arange(5, dtype=np.int64)
    simint.compute_range(P, P, 0, None, n, off, out.data_ptr())
    L = simint.lib()
    assert L.simint_hip_capture_begin() == 0
    g = ctypes.c_void_p()
    try:
        with pytest.raises(RuntimeError):
            simint.compute_range(P, P, 0, None, n, off, out.data_ptr())
    finally:
        if L.simint_hip_capture_end(ctypes.byref(g)) == 0:
            L.simint_hip_graph_free(g)
    want = out.clone()
    out.zero_()
    torch.cuda.synchronize()
    simint.compute_range(P, P, 0, None, n, off, out.data_ptr())
    simint.synchronize()
    assert torch.equal(out, want)
    for h in (P, hp, b):
        h.free()


# values: 9, 131058, 131130 (1 MiB is 131072), 524286 and 524295 (4 MiB is
# 524288), six pieces, and sixteen and a bit
@pytest.mark.parametrize("nbra,nket", [(1, 1), (3, 4854), (2, 7285), (6, 9709), (5, 11651), (45, 7767), (77, 12107)])
def test_results_to_the_host(gpu, nbra, nket):
    rng = np.random.default_rng(nbra)
    bb, hp, P = _pairs(rng, (1, 0), nbra, depth=1)
    bk, hq, Q = _pairs(rng, (1, 0), nket, depth=1)
    nv = 9 * nbra * nket
    dev = torch.full((nv,), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    simint.compute_range(P, Q, 0, None, np.full(nbra, nket, dtype=np.int32),
                         9 * nket * np.arange(nbra, dtype=np.int64), dev.data_ptr())
    simint.synchronize()
    got = np.full(nv + 1, np.nan)
    rc = simint.lib().simint_compute_eri(ctypes.byref(hp.mp), ctypes.byref(hq.mp), 0.0, None,
                                         got.ctypes.data_as(simint.dptr))
    assert rc == nbra * nket
    assert np.isnan(got[-1])
    assert np.array_equal(got[:-1], dev.cpu().numpy())
    # and into memory the device reaches itself
    for kw in ({"pin_memory": True}, {"device": "cuda"}):
        into = torch.full((nv,), float("nan"), dtype=torch.float64, **kw)
        torch.cuda.synchronize()
        assert simint.lib().simint_compute_eri(ctypes.byref(hp.mp), ctypes.byref(hq.mp), 0.0, None,
                                               ctypes.cast(into.data_ptr(), simint.dptr)) == nbra * nket
        assert torch.equal(into.cpu(), dev.cpu())
    for h in (P, Q, hp, hq, bb, bk):
        h.free()
