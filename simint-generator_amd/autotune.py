"""Per-class kernel-family autotuner (runs on the GPU).

For every class, times each kernel family built for it -- lane-per-quartet
(registers), wave-per-quartet (LDS-staged, batched), the split
lane-per-quartet kernels with two group counts and, for bra-heavy d
classes, their ket-top-group variants, and the component-lane kernels -- on
the screened quartets of a synthetic system built with the 64-atom benchmark
recipe at a smaller size (classes that system does not have: on random shell
pairs of depth 1-3 in an 8-bohr cube), and writes the fastest family per class to tuning.json (read by the
build to set each class's default):

    python simint-generator_amd/autotune.py [--natom 16] [--reps 3] [--out PATH]
    python simint-generator_amd/autotune.py --lanes     # small launches ("lane_items")
    python simint-generator_amd/autotune.py --list [--split] [--even]   # quartet-list kernels

--list --split also times the lanes per quartet of the lane-per-quartet
list launches per class and records the counts that beat the automatic
choice ("list_split"; batch.QuartetBatch applies them).  --list --even times
lists of one depth and records from how many primitive quartets on the
lane-per-quartet kernel beats the component-lane one ("list_even").
"""
import argparse
import json
import os
import sys
import time

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--natom", type=int, default=16)
    ap.add_argument("--reps", type=int, default=3)
    ap.add_argument("--out", default=os.path.join(HERE, "tuning.json"))
    ap.add_argument("--list", action="store_true",
                    help="tune the quartet-list kernels on the batched all-classes stream instead "
                         "(merges 'list_family' into the output file)")
    ap.add_argument("--nquartet", type=int, default=200000)
    ap.add_argument("--split", action="store_true",
                    help="with --list: also time 1-16 lanes per quartet for the classes whose list kernel is "
                         "lane-per-quartet (merges 'list_split' into the output file)")
    ap.add_argument("--even", action="store_true",
                    help="with --list: also time lists of one depth in the classes whose list kernel is "
                         "component-lane (merges 'list_even' into the output file)")
    ap.add_argument("--lanes", action="store_true",
                    help="time the component-lane kernels against the lane-per-quartet ones on few items (merges "
                         "'lane_items' into the output file)")
    a = ap.parse_args()
    if a.lanes:
        return tune_lanes(a)
    if a.list:
        tune_lists(a)
        if a.split:
            tune_split(a)
        if a.even:
            tune_even(a)
        return None
    import torch
    import quartets
    import simint
    import workloads
    L = simint.lib()
    ss = quartets.ScreenedSet(workloads.grid_molecule(natom=a.natom, seed=0), tol=1e-12)
    out = torch.empty(ss.out_doubles, dtype=torch.float64, device="cuda")
    stream = torch.cuda.ExternalStream(L.simint_hip_stream())
    by = {}
    for ln in ss.launches:
        by.setdefault(ln.cls, []).append(ln)
    family = {}
    timings = {}
    for cls in sorted(by):
        name = quartets.simint_class_name(cls)
        prev = L.simint_hip_class_kernel(*cls)
        res = {}
        for fam, fname in ((1, "lpq"), (2, "wpq"), (3, "lpqs_a"), (4, "lpqs_b"), (5, "lpqsf_a"), (6, "lpqsf_b"),
                           (7, "cpl")):
            if L.simint_hip_set_class_kernel(*cls, fam) < 0:
                continue
            best = None
            for rep in range(a.reps + 1):
                e0 = torch.cuda.Event(enable_timing=True)
                e1 = torch.cuda.Event(enable_timing=True)
                e0.record(stream)
                for ln in by[cls]:
                    simint.compute_prefix(ln.bra.dev, ln.ket.dev, ln.b0, ln.nket, ln.off, out.data_ptr(), 0.0)
                e1.record(stream)
                simint.synchronize()
                ms = e0.elapsed_time(e1)
                if rep > 0:
                    best = ms if best is None else min(best, ms)
            res[fname] = best
        L.simint_hip_set_class_kernel(*cls, prev)
        if res:
            family[name] = min(res, key=res.get)
            timings[name] = res
            print("%-8s %s" % (name, "  ".join("%s %.3f ms" % kv for kv in sorted(res.items()))), flush=True)
    tune_other(a, family, timings)
    doc = json.load(open(a.out)) if os.path.exists(a.out) else {}
    doc.update({"workload": "64-atom recipe, %d atoms, Schwarz 1e-12, quartets of each class; "
                "the other classes: 96 x 512 random pairs of depth 1-3" % a.natom,
                "family": family, "timings_ms": timings,
                "generated": time.strftime("%Y-%m-%d %H:%M:%S")})
    with open(a.out, "w") as f:
        json.dump(doc, f, indent=1, sort_keys=True)
    print("wrote", a.out)


def tune_other(a, family, timings):
    """Prefix-kernel family of the classes up to f that the molecule recipe
    has none of: 96 bra against 512 ket pairs of shells of depth 1-3 with
    exponents log-uniform in [0.1, 50] in an 8-bohr cube."""
    import itertools
    import numpy as np
    import torch
    import quartets
    import simint
    L = simint.lib()
    rng = np.random.default_rng(0)
    shells = []
    for l in range(4):
        for _ in range(64):
            k = int(rng.integers(1, 4))
            shells.append((l, tuple(rng.uniform(0, 8, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(50), k))),
                           list(rng.uniform(0.1, 1.0, k))))
    basis = simint.Basis(shells)
    stream = torch.cuda.ExternalStream(L.simint_hip_stream())
    sets = {}
    for la, lb in itertools.product(range(4), repeat=2):
        for n in (96, 512):
            pr = [(64 * la + int(i), 64 * lb + int(j)) for i, j in rng.integers(0, 64, (n, 2))]
            pr.sort(key=lambda p: -len(shells[p[0]][2]) * len(shells[p[1]][2]))
            hp = simint.Pairs.from_pairs(basis, pr)
            sets[la, lb, n] = simint.DevicePairs(hp)
            hp.free()
    out = torch.empty(96 * 512 * 10000, dtype=torch.float64, device="cuda")
    for cls in itertools.product(range(4), repeat=4):
        name = quartets.simint_class_name(cls)
        if name in family:
            continue
        P, Q = sets[cls[0], cls[1], 96], sets[cls[2], cls[3], 512]
        nc = int(np.prod([simint.ncart(l) for l in cls]))
        nket = np.full(96, 512, dtype=np.int32)
        off = np.arange(96, dtype=np.int64) * 512 * nc
        prev = L.simint_hip_class_kernel(*cls)
        res = {}
        for fname, fam in simint.FAMILIES.items():
            if L.simint_hip_set_class_kernel(*cls, fam) < 0:
                continue
            for rep in range(a.reps + 1):
                e0 = torch.cuda.Event(enable_timing=True)
                e1 = torch.cuda.Event(enable_timing=True)
                e0.record(stream)
                simint.compute_prefix(P, Q, 0, nket, off, out.data_ptr())
                e1.record(stream)
                simint.synchronize()
                if rep > 0:
                    res[fname] = min(res.get(fname, 1e30), e0.elapsed_time(e1))
        L.simint_hip_set_class_kernel(*cls, prev)
        family[name] = min(res, key=res.get)
        timings[name] = res
        print("%-8s %s" % (name, "  ".join("%s %.3f ms" % kv for kv in sorted(res.items()))), flush=True)
    for d in sets.values():
        d.free()
    basis.free()


def tune_lists(a):
    """Quartet-list family per class, timed on a batched stream of the
    all-classes recipe (a 4096-shell pool, depths 1-6)."""
    import torch
    import batch
    import simint
    import workloads
    L = simint.lib()
    shells, q = workloads.all_class_stream(nquartet=a.nquartet, seed=1)
    basis = simint.Basis(shells)
    b = batch.QuartetBatch(basis, q)
    out = torch.empty(b.out_doubles, dtype=torch.float64, device="cuda")
    stream = torch.cuda.ExternalStream(L.simint_hip_stream())
    family, timings = {}, {}
    for g in b.groups:
        name = "_".join("spdfghik"[x] for x in g.cls)
        prev = L.simint_hip_class_list_kernel(*g.cls)
        res = {}
        for fam, fname in ((1, "lpq"), (2, "wpq"), (7, "cpl")):
            if L.simint_hip_set_class_list_kernel(*g.cls, fam) < 0:
                continue
            best = None
            for rep in range(a.reps + 1):
                e0 = torch.cuda.Event(enable_timing=True)
                e1 = torch.cuda.Event(enable_timing=True)
                e0.record(stream)
                simint.compute_list(g.P, g.Q, g.n, g.idx.data_ptr(), g.idx.data_ptr(), g.qout.data_ptr(),
                                    out.data_ptr())
                e1.record(stream)
                simint.synchronize()
                ms = e0.elapsed_time(e1)
                if rep > 0:
                    best = ms if best is None else min(best, ms)
            res[fname] = best
        L.simint_hip_set_class_list_kernel(*g.cls, prev)
        if res:
            family[name] = min(res, key=res.get)
            timings[name] = res
            print("%-8s %s" % (name, "  ".join("%s %.3f ms" % kv for kv in sorted(res.items()))), flush=True)
    doc = json.load(open(a.out)) if os.path.exists(a.out) else {}
    doc["list_family"] = family
    doc["list_timings_ms"] = timings
    doc["list_workload"] = "%d quartets of the all-classes stream recipe (seed 1)" % a.nquartet
    with open(a.out, "w") as f:
        json.dump(doc, f, indent=1, sort_keys=True)
    print("wrote", a.out)


def tune_split(a):
    """Lanes per quartet of the lane-per-quartet list launches, per class,
    on the same batched stream: every class whose list kernel (after the
    family tuning) is lane-per-quartet is timed with the automatic choice
    (0: about 65536 lanes per launch) and with 1, 2, 4, 8 and 16 lanes; a
    class keeps a fixed count only where it beats the automatic one by more
    than 2 %."""
    import torch
    import batch
    import simint
    import workloads
    L = simint.lib()
    if os.path.exists(a.out):
        simint.apply_tuning(a.out)
    shells, q = workloads.all_class_stream(nquartet=a.nquartet, seed=1)
    basis = simint.Basis(shells)
    b = batch.QuartetBatch(basis, q)
    out = torch.empty(b.out_doubles, dtype=torch.float64, device="cuda")
    stream = torch.cuda.ExternalStream(L.simint_hip_stream())
    split, timings = {}, {}
    for g in b.groups:
        if L.simint_hip_class_list_kernel(*g.cls) != 1:
            continue
        name = "_".join("spdfghik"[x] for x in g.cls)
        res = {}
        for lanes in (0, 1, 2, 4, 8, 16):
            prev = L.simint_hip_set_list_split(lanes)
            best = None
            for rep in range(a.reps + 1):
                e0 = torch.cuda.Event(enable_timing=True)
                e1 = torch.cuda.Event(enable_timing=True)
                e0.record(stream)
                simint.compute_list(g.P, g.Q, g.n, g.idx.data_ptr(), g.idx.data_ptr(), g.qout.data_ptr(),
                                    out.data_ptr())
                e1.record(stream)
                simint.synchronize()
                ms = e0.elapsed_time(e1)
                if rep > 0:
                    best = ms if best is None else min(best, ms)
            L.simint_hip_set_list_split(prev)
            res[lanes] = best
        timings[name] = res
        fastest = min(res, key=res.get)
        if fastest != 0 and res[fastest] < 0.98 * res[0]:
            split[name] = fastest
        print("%-8s %s" % (name, "  ".join("%d: %.3f ms" % kv for kv in sorted(res.items()))), flush=True)
    doc = json.load(open(a.out)) if os.path.exists(a.out) else {}
    doc["list_split"] = split
    doc["list_split_timings_ms"] = {k: {str(l): t for l, t in v.items()} for k, v in timings.items()}
    with open(a.out, "w") as f:
        json.dump(doc, f, indent=1, sort_keys=True)
    print("wrote", a.out, "(%d classes with a fixed lane count)" % len(split))


def tune_lanes(a):
    """Items (a bra against 64 kets) up to which a launch of a class that runs
    the lane-per-quartet kernel is not slower in the component-lane one, for
    1, 4, 9 and 16 and more (16, 36, 256) primitive quartets.  The other
    kernel, which small launches do not run, is timed on 256 items: up to one
    for every SIMD it takes the time of one (uncontracted quartets, which mostly
    store, a little more, so their line comes out high)."""
    import itertools
    import numpy as np
    import torch
    import quartets
    import simint
    from emitter import hip_lpq
    L = simint.lib()
    items = (4, 16, 32, 64, 96, 128)
    rng = np.random.default_rng(0)
    sets = {}
    for la, lb, depth in itertools.product(range(4), range(4), (1, 2, 3, 4)):
        shells = [(l, tuple(rng.uniform(0, 4, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20), depth))),
                   list(rng.uniform(0.1, 1.0, depth))) for _ in range(64) for l in (la, lb)]
        basis = simint.Basis(shells)
        hp = simint.Pairs.from_pairs(basis, [(2 * (k % 64), 2 * (k % 64) + 1) for k in range(256)])
        sets[la, lb, depth] = simint.DevicePairs(hp)
        hp.free()
        basis.free()
    out = torch.empty(256 * 64 * 1296, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def us(cls, dp, dq, n):
        nket = np.full(n, 64, dtype=np.int32)
        off = np.arange(n, dtype=np.int64) * 64 * int(np.prod([simint.ncart(l) for l in cls]))
        best = 1e30
        for rep in range(a.reps + 1):
            t0 = time.perf_counter()
            for _ in range(10):
                simint.compute_range(sets[cls[0], cls[1], dp], sets[cls[2], cls[3], dq], 0, None, nket, off,
                                     out.data_ptr())
            simint.synchronize()
            if rep > 0:
                best = min(best, time.perf_counter() - t0)
        return best
    found = {}
    for cls in itertools.product(range(4), repeat=4):
        if hip_lpq.share_kind(cls) != "lanes" or L.simint_hip_class_kernel(*cls) != 1:
            continue
        most = []
        for depths in (((1, 1),), ((2, 1),), ((3, 1),), ((2, 2), (3, 2), (4, 4))):
            good = items
            for dp, dq in depths:
                L.simint_hip_set_class_kernel(*cls, 1)
                ref = us(cls, dp, dq, 256)
                L.simint_hip_set_class_kernel(*cls, 7)
                t = [us(cls, dp, dq, n) for n in items]
                good = [n for k, n in enumerate(items) if n in good and max(t[:k + 1]) <= 1.03 * ref]
            most.append(max(good, default=0))
        found[quartets.simint_class_name(cls)] = most
        print("%-8s %s" % (quartets.simint_class_name(cls), most), flush=True)
    L.simint_hip_reset_class_kernels()
    for d in sets.values():
        d.free()
    doc = json.load(open(a.out)) if os.path.exists(a.out) else {}
    doc["lane_items"] = found
    with open(a.out, "w") as f:
        json.dump(doc, f, indent=1, sort_keys=True)
    print("wrote", a.out, "(%d classes)" % len(found))


def tune_even(a):
    """Lists of 50 to 51200 quartets of one depth: for every class whose list
    kernel (after the family tuning) is component-lane, the number of primitive
    quartets from which the lane-per-quartet kernel is taken, below 16 primitive
    quartets a quartet (timed at 1 and 4) and from there on (timed at 16 and
    256): the number that makes the timings' product least."""
    import itertools
    import math
    import numpy as np
    import torch
    import quartets
    import simint
    L = simint.lib()
    if os.path.exists(a.out):
        simint.apply_tuning(a.out)
    lens = (50, 200, 800, 3200, 12800, 51200)
    rng = np.random.default_rng(0)
    sets = {}
    for la, lb, k1, k2 in itertools.product(range(4), range(4), (1, 2, 4), (1, 2, 4)):
        if k2 > k1:
            continue
        shells = [(l, tuple(rng.uniform(0, 4, 3)), list(np.exp(rng.uniform(np.log(0.1), np.log(20), k))),
                   list(rng.uniform(0.1, 1.0, k))) for _ in range(64) for l, k in ((la, k1), (lb, k2))]
        basis = simint.Basis(shells)
        hp = simint.Pairs.from_pairs(basis, [(2 * k, 2 * k + 1) for k in range(64)])
        sets[la, lb, k1 * k2] = simint.DevicePairs(hp)
        hp.free()
        basis.free()
    index = [torch.from_numpy(rng.integers(0, 64, lens[-1]).astype(np.int32)).cuda() for _ in range(2)]
    out = torch.empty(lens[-1] * 3600, dtype=torch.float64, device="cuda")
    stream = torch.cuda.ExternalStream(L.simint_hip_stream())

    def ms(P, Q, n):
        best = None
        for rep in range(a.reps + 1):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            simint.compute_list(P, Q, n, index[0].data_ptr(), index[1].data_ptr(), 0, out.data_ptr())
            e1.record(stream)
            simint.synchronize()
            t = e0.elapsed_time(e1)
            if rep > 0:
                best = t if best is None else min(best, t)
        return best
    even = {}
    for cls in itertools.product(range(4), repeat=4):
        if L.simint_hip_class_list_kernel(*cls) != 7 or L.simint_hip_set_class_list_kernel(*cls, 1) < 0:
            continue
        t = {}
        for fam in (1, 7):
            L.simint_hip_set_class_list_kernel(*cls, fam)
            for kp, kq in ((1, 1), (2, 2), (4, 4), (16, 16)):
                for n in lens:
                    t[fam, kp * kq, n] = ms(sets[cls[0], cls[1], kp], sets[cls[2], cls[3], kq], n)
        line = []
        for depths in ((1, 4), (16, 256)):
            def cost(at):
                return sum(math.log(t[1 if at and n * k >= at else 7, k, n]) for k in depths for n in lens)
            line.append(min([0] + sorted({n * k for k in depths for n in lens}, reverse=True), key=cost))
        if any(line):
            even[quartets.simint_class_name(cls)] = line
            print("%-8s %s" % (quartets.simint_class_name(cls), line), flush=True)
    L.simint_hip_reset_class_kernels()
    for d in sets.values():
        d.free()
    doc = json.load(open(a.out)) if os.path.exists(a.out) else {}
    doc["list_even"] = even
    with open(a.out, "w") as f:
        json.dump(doc, f, indent=1, sort_keys=True)
    print("wrote", a.out, "(%d classes)" % len(even))


if __name__ == "__main__":
    main()
