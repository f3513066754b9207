"""The work this engine is timed on, and what its answers are checked against.

Six kinds of work, each through the calls a program makes:

  call     simint_compute_eri on host buffers: what a program written against
           simint's C API does, from one quartet a call to a block of pairs;
  list     a list of quartets of one class (simint_hip_compute_eri_list
           behind batch.QuartetBatch), integrals left on the GPU;
  stream   a list of quartets of every class up to f and every contraction
           depth, as one graph or spread over side streams; also its first
           derivatives;
  eri      every unique quartet of a molecule above a Schwarz threshold, in
           FP64 or with the FP32 recurrences for the small ones, or its
           first derivatives, all integrals kept;
  jk       the Coulomb and exchange matrices of a density over those
           quartets, the integrals going through a reused buffer;
  oei      overlap, kinetic energy and nuclear attraction of all shell pairs
           of a molecule.

Sizes are those of the repository's own benchmark (1000 (pp|pp) quartets, the
mixed-class stream, grid molecules of up to 64 atoms) and smaller ones of the
same recipes.  exact() evaluates the integrals by McMurchie-Davidson
expansions in torch, in 64 bits, from the shells alone.
"""
import json
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "simint-generator_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

STREAMS = 16   # side streams a batch is spread over (the benchmark's)


def listed():
    return [
        # one contracted (pp|pp) quartet a call: the smallest call of a
        # program that loops over quartets, all latency
        {"name": "call_one", "kind": "call", "am": "pppp", "npair": 1, "nket": 1, "depth": 3},
        # 528 x 528 (pp) pairs in one call: the benchmark's host-buffer
        # block, bound by the way back to the host
        {"name": "call_block", "kind": "call", "am": "pppp", "npair": 528, "nket": 528, "depth": 3},
        # 1000 (pp|pp) quartets of depth 3 on the GPU: an ordinary short list
        {"name": "list_pp", "kind": "list", "l": 1, "quartets": 1000, "depth": 3},
        # a small mixed-class stream (about 32 quartets a class), one graph
        # launch a pass: many short launches
        {"name": "stream_small", "kind": "stream", "quartets": 8192, "deriv": 0, "graph": True},
        # a large one queued on side streams: f classes and deep contractions
        {"name": "stream_large", "kind": "stream", "quartets": 300000, "deriv": 0, "graph": False},
        # first derivatives of a mixed-class stream (classes up to g inside)
        {"name": "stream_deriv", "kind": "stream", "quartets": 1500, "deriv": 1, "graph": False},
        # every integral of a small molecule, FP64: many launches of a few
        # thousand to a few hundred thousand quartets
        {"name": "eri_small", "kind": "eri", "atoms": 12, "mixed": False, "deriv": 0},
        # the same with the FP32 recurrences for quartets of small bounds
        {"name": "eri_mixed", "kind": "eri", "atoms": 15, "mixed": True, "deriv": 0},
        # first derivatives of a small molecule (one step of an optimiser)
        {"name": "eri_deriv", "kind": "eri", "atoms": 8, "mixed": False, "deriv": 1},
        # Coulomb and exchange of a small and of a large molecule (one
        # iteration of a self-consistent field)
        {"name": "jk_small", "kind": "jk", "atoms": 10, "mixed": False},
        {"name": "jk_large", "kind": "jk", "atoms": 64, "mixed": False},
        # one-electron matrices of a large molecule
        {"name": "oei_large", "kind": "oei", "atoms": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "list", "stream", "stream", "eri", "eri", "jk", "oei"])
    if kind == "call":
        am = "".join(rng.choice("spd") for _ in range(4))
        return {"kind": kind, "am": am, "npair": _log_int(rng, 1, 300), "nket": _log_int(rng, 1, 300),
                "depth": rng.randint(1, 5)}
    if kind == "list":
        return {"kind": kind, "l": rng.randint(0, 3), "quartets": _log_int(rng, 60, 20000), "depth": rng.randint(1, 4)}
    if kind == "stream":
        deriv = int(rng.random() < 0.4)
        lo, hi = (200, 1400) if deriv else (1000, 250000)
        return {"kind": kind, "quartets": _log_int(rng, lo, hi), "deriv": deriv, "graph": rng.random() < 0.5}
    if kind == "eri":
        deriv = int(rng.random() < 0.4)
        return {"kind": kind, "atoms": rng.randint(2, 8 if deriv else 16), "mixed": not deriv and rng.random() < 0.5,
                "deriv": deriv}
    if kind == "jk":
        return {"kind": kind, "atoms": _log_int(rng, 3, 50), "mixed": rng.random() < 0.5}
    return {"kind": kind, "atoms": _log_int(rng, 2, 64)}


# ------------------------------------------------------------- the workloads
def _shells(case, seed):
    """(shells, index data) of a case: shells as (l, centre, exponents,
    coefficients), made from the seed alone."""
    import workloads
    kind = case["kind"]
    if kind == "call":
        # the recipe of the (pp|pp) list: exponents log-uniform in [0.1, 20],
        # coefficients in [0.1, 1], centres in a 10-bohr cube
        rng = np.random.default_rng(seed)
        am = ["spdf".index(c) for c in case["am"]]
        sets = []
        shells = []
        for side, n in ((0, case["npair"]), (1, case["nket"])):
            pairs = []
            for _ in range(n):
                ij = []
                for l in am[2 * side:2 * side + 2]:
                    ij.append(len(shells))
                    shells.append((l, tuple(rng.uniform(0, 10, 3)),
                                   np.exp(rng.uniform(np.log(0.1), np.log(20.0), case["depth"])).tolist(),
                                   rng.uniform(0.1, 1.0, case["depth"]).tolist()))
                pairs.append(tuple(ij))
            sets.append(pairs)
        return shells, sets
    if kind == "list":
        rng = np.random.default_rng(seed)
        shells = [(case["l"], tuple(rng.uniform(0, 10, 3)),
                   np.exp(rng.uniform(np.log(0.1), np.log(20.0), case["depth"])).tolist(),
                   rng.uniform(0.1, 1.0, case["depth"]).tolist()) for _ in range(40)]
        return shells, rng.integers(0, 40, (case["quartets"], 4))
    if kind == "stream":
        # the pool of the benchmark's stream (1024 shells per AM, s to f);
        # the classes in a fixed random order, the shells by the seed, so
        # that every seed's integrals take the same room
        shells, _ = workloads.mixed_pool(seed)
        am = np.random.default_rng(1).integers(0, 4, (case["quartets"], 4))
        return shells, 1024 * am + np.random.default_rng(seed).integers(0, 1024, am.shape)
    return workloads.grid_molecule(natom=case["atoms"], seed=seed), None


def _ncart(l):
    return (l + 1) * (l + 2) // 2


def _oei_inputs(case, seed):
    """Shell pairs (i >= j), output offsets and the charges at the atoms."""
    shells, _ = _shells(case, seed)
    n = len(shells)
    i, j = np.tril_indices(n)
    nc = np.array([_ncart(s[0]) for s in shells], dtype=np.int64)
    size = nc[i] * nc[j]
    off = np.zeros(len(i), dtype=np.int64)
    off[1:] = np.cumsum(size)[:-1]
    centres = np.array([shells[6 * a][1] for a in range(case["atoms"])])
    charges = np.random.default_rng(seed).integers(1, 18, case["atoms"]).astype(np.float64)
    return shells, np.stack([i, j], axis=1).astype(np.int32), off, int(size.sum()), np.column_stack([charges, centres])


class State:
    """What a program holds between calls.  Its library handles go with it."""

    def __init__(self):
        self.handles = []

    def __del__(self):
        for h in reversed(self.handles):
            h.free()


def prepare(case, seed):
    import simint
    simint.lib().simint_init()
    s = State()
    s.kind = case["kind"]
    if s.kind == "call":
        shells, (bra, ket) = _shells(case, seed)
        basis = simint.Basis(shells)
        s.P = simint.Pairs.from_pairs(basis, bra)
        s.Q = simint.Pairs.from_pairs(basis, ket)
        s.handles = [basis, s.P, s.Q]
        n = len(bra) * len(ket)
        for c in case["am"]:
            n *= _ncart("spdf".index(c))
        s.out = np.empty(n)
        s.out[:] = 0.0          # touched once, as a buffer that a program keeps is
    elif s.kind in ("list", "stream"):
        import batch
        shells, q = _shells(case, seed)
        basis = simint.Basis(shells)
        s.batch = batch.QuartetBatch(basis, q, deriv=case.get("deriv", 0))
        s.out = torch.empty(s.batch.out_doubles, dtype=torch.float64, device="cuda")
        s.handles = [basis, s.batch]
        s.streams = STREAMS if s.kind == "stream" else None
        torch.cuda.synchronize()
        if case.get("graph"):
            s.graph = s.batch.capture(s.out.data_ptr(), streams=s.streams)
            s.handles.append(s.graph)
        else:
            s.graph = None
    elif s.kind in ("eri", "jk"):
        import quartets
        shells, _ = _shells(case, seed)
        mixed = 1e-4 if case["mixed"] else None
        s.set = quartets.ScreenedSet(shells, tol=1e-12, mixed=mixed, deriv=case.get("deriv", 0))
        s.handles = [s.set]
        if s.kind == "eri":
            size = [s.set.chunk_doubles(c) for c in range(s.set.nchunk)]
            s.start = np.concatenate([[0], np.cumsum(size)])
            # room for every quartet, as for a molecule whose geometry (and
            # so what the screen keeps) changes; the rest stays zero
            nc = np.array([_ncart(l[0]) for l in shells])
            i, j = np.tril_indices(len(shells))
            pair = nc[i] * nc[j]
            room = int(pair.sum()) ** 2 + int((pair ** 2).sum())
            s.out = torch.zeros(room // 2 * (12 if case["deriv"] else 1), dtype=torch.float64, device="cuda")
            n = s.set.deriv_worksize() if case["deriv"] else 0
            s.work = torch.empty(n, dtype=torch.float64, device="cuda") if n else None
        else:
            s.nbf = s.set.nbf()
            g = torch.Generator().manual_seed(seed)
            C = torch.rand((s.nbf, max(1, s.nbf // 4)), generator=g, dtype=torch.float64) - 0.5
            s.D = (C @ C.T / s.nbf).cuda()
            s.J = torch.zeros((s.nbf, s.nbf), dtype=torch.float64, device="cuda")
            s.K = torch.zeros_like(s.J)
            room = max(s.set.chunk_doubles(c) for c in range(s.set.nchunk))
            s.buffer = torch.empty(room, dtype=torch.float64, device="cuda")
    else:
        shells, pairs, off, n, charges = _oei_inputs(case, seed)
        basis = simint.Basis(shells)
        s.shells = simint.DeviceShells(basis)
        s.handles = [basis, s.shells]
        s.npair, s.ncharge = len(pairs), len(charges)
        s.pairs = torch.from_numpy(pairs.reshape(-1)).cuda()
        s.off = torch.from_numpy(off).cuda()
        s.charges = torch.from_numpy(charges.reshape(-1)).cuda()
        s.out = {k: torch.empty(n, dtype=torch.float64, device="cuda") for k in simint.OEI_KINDS}
    torch.cuda.synchronize()
    return s


def run(s):
    import ctypes
    import simint
    L = simint.lib()
    if s.kind == "call":
        rc = L.simint_compute_eri(ctypes.byref(s.P.mp), ctypes.byref(s.Q.mp), 0.0, None,
                                  s.out.ctypes.data_as(simint.dptr))
        if rc < 0:
            raise RuntimeError("simint_compute_eri: %d %s" % (rc, simint.last_error()))
        return s.out
    if s.kind in ("list", "stream"):
        if s.graph is not None:
            s.graph.launch()
        else:
            s.batch.run(s.out.data_ptr(), streams=s.streams)
        return s.out
    if s.kind == "eri":
        work = s.work.data_ptr() if s.work is not None else None
        for c in range(s.set.nchunk):
            s.set.run_pass(s.out.data_ptr() + 8 * int(s.start[c]), chunk=c, work_ptr=work)
        return s.out
    if s.kind == "jk":
        with torch.cuda.stream(torch.cuda.ExternalStream(L.simint_hip_stream())):
            s.J.zero_()
            s.K.zero_()
        s.set.run_jk(s.buffer.data_ptr(), s.D.data_ptr(), s.J.data_ptr(), s.K.data_ptr())
        simint.jk_symmetrize(s.nbf, s.J.data_ptr(), s.K.data_ptr())
        return {"J": s.J, "K": s.K}
    for kind, out in s.out.items():
        s.shells.compute(kind, s.npair, s.pairs.data_ptr(), s.off.data_ptr(), out.data_ptr(),
                         s.ncharge if kind == "potential" else 0, s.charges.data_ptr())
    return s.out


# ------------------------------------------------------------------ the work
def _class_table():
    with open(os.path.join(PKG, "csrc", "gen", "classes.json")) as f:
        return json.load(f)


def _per_quartet(table, am, K):
    c = table["_".join("spdf"[x] for x in am)]
    return K * (c["f_setup"] + c["f_vrr"] + c["f_boys"] + c["bcont"]) + c["f_hrr"], c["ncart"]


def work(case):
    """Bytes: every output value once and every shell's data once.  Flops:
    the reference recurrence's count per quartet (a fused multiply-add is
    two); for derivatives one count of the class per explicit centre, a
    lower bound of their (a+1) and (a-1) classes."""
    table = _class_table()
    kind = case["kind"]
    if kind == "call":
        n = case["npair"] * case["nket"]
        f, nc = _per_quartet(table, ["spdf".index(c) for c in case["am"]], case["depth"] ** 4)
        pairs = (case["npair"] + case["nket"]) * case["depth"] ** 2
        return {"bytes": 8.0 * (n * nc + 14 * pairs), "flops": float(n) * f}
    if kind in ("list", "stream"):
        shells, q = _shells(case, 0)
        am = np.array([s[0] for s in shells])[q]
        depth = np.array([len(s[2]) for s in shells], dtype=np.int64)[q].prod(axis=1)
        code, inv, count = np.unique(am @ np.array([64, 16, 4, 1]), return_inverse=True, return_counts=True)
        K = np.bincount(inv, weights=depth)
        flops = values = 0.0
        for c, n, k in zip(code, count, K):
            f1, nc = _per_quartet(table, [c // 64, c // 16 % 4, c // 4 % 4, c % 4], 1)
            f0, _ = _per_quartet(table, [c // 64, c // 16 % 4, c // 4 % 4, c % 4], 0)
            flops += float(k) * (f1 - f0) + float(n) * f0
            values += float(n) * nc
        d = 12 if case.get("deriv") else 1
        return {"bytes": 8.0 * (values * d + 2 * sum(len(s[2]) for s in shells) + 4 * len(q)),
                "flops": flops * (3 if d > 1 else 1)}
    if kind in ("eri", "jk"):
        import quartets
        shells, _ = _shells(case, 0)
        ss = quartets.ScreenedSet(shells, tol=1e-12, deriv=case.get("deriv", 0))
        flops, values, nbf, nq = ss.total_flops, ss.total_bytes, ss.nbf(), ss.total_quartets
        ss.free()
        if kind == "jk":
            # six updates of two flops per integral
            return {"bytes": 8.0 * 3 * nbf * nbf, "flops": flops + 12.0 * values / 8.0}
        return {"bytes": float(values), "flops": flops * (3 if case["deriv"] else 1)}
    shells, pairs, _, n, charges = _oei_inputs(case, 0)
    l = np.array([s[0] for s in shells])[pairs]
    k = np.array([len(s[2]) for s in shells], dtype=np.int64)[pairs].prod(axis=1)
    nc = ((l + 1) * (l + 2) // 2).prod(axis=1)
    # per primitive pair and charge: the Boys function (about 40) and, per
    # auxiliary order, two fused multiply-adds of every output component
    per = 40.0 + 4.0 * nc * (l.sum(axis=1) + 1)
    return {"bytes": 8.0 * (3 * n + 2 * sum(len(s[2]) for s in shells)), "flops": float((k * per).sum() * len(charges))}


# ------------------------------------------- the same values by another method
DEV = "cuda" if torch.cuda.is_available() else "cpu"
CHUNK_VALUES = 1 << 26   # doubles of the largest intermediate of one chunk


def _carts(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _hermites(L):
    return [(t, u, n - t - u) for n in range(L + 1) for t in range(n, -1, -1) for u in range(n - t, -1, -1)]


def _index(v):
    return torch.tensor(v, dtype=torch.long, device=DEV)


def _normalized(shells):
    """Coefficients of unit-normalised contracted x^l functions over
    normalised primitives, the primitives' own normalisation folded in."""
    out = []
    for l, _, al, co in shells:
        a, c = np.array(al), np.array(co)
        fact = float(np.prod(np.arange(2 * l - 1, 0, -2))) if l else 1.0
        c = c * a ** (0.5 * l + 0.75)
        p = a[:, None] + a[None, :]
        s = fact * (math.pi / p) ** 1.5 / (2.0 * p) ** l
        out.append(c / math.sqrt(float(c @ s @ c)))
    return out


def _boys(L, x):
    """F_0..F_L of every x, stacked in the last dimension."""
    small = x < 40.0
    xs = torch.where(small, x, torch.zeros_like(x))
    term = torch.full_like(x, 1.0 / (2 * L + 1))
    total = term.clone()
    for k in range(1, 190):
        term = term * (2.0 * xs) / (2 * L + 2 * k + 1)
        total = total + term
    low = [None] * (L + 1)
    ex = torch.exp(-xs)
    low[L] = ex * total
    for m in range(L - 1, -1, -1):
        low[m] = (2.0 * xs * low[m + 1] + ex) / (2 * m + 1)
    xl = torch.where(small, torch.full_like(x, 40.0), x)
    high = [0.5 * torch.sqrt(math.pi / xl) * torch.erf(torch.sqrt(xl))]
    ex = torch.exp(-xl)
    for m in range(L):
        high.append(((2 * m + 1) * high[m] - ex) / (2.0 * xl))
    return torch.stack([torch.where(small, a, b) for a, b in zip(low, high)], dim=-1)


def _expansion(la, lb, a, b, A, B):
    """Hermite expansion coefficients of the Cartesian products of a pair of
    primitives, the Gaussian product's exponential inside: E[n, ab, tuv]."""
    p = (a + b)[:, None]
    PA = -(b / (a + b))[:, None] * (A - B)
    PB = (a / (a + b))[:, None] * (A - B)
    h = 0.5 / p
    zero = torch.zeros_like(PA)
    E = {(0, 0, 0): torch.exp(-(a * b / (a + b))[:, None] * (A - B) ** 2)}

    def get(i, j, t):
        return E.get((i, j, t), zero)
    for i in range(la + 1):
        for j in range(lb + 1):
            if i == j == 0:
                continue
            X, (i0, j0) = (PA, (i - 1, j)) if i else (PB, (i, j - 1))
            for t in range(i + j + 1):
                E[i, j, t] = h * get(i0, j0, t - 1) + X * get(i0, j0, t) + (t + 1) * get(i0, j0, t + 1)
    L = la + lb
    T = torch.stack([get(i, j, t) for i in range(la + 1) for j in range(lb + 1) for t in range(L + 1)], dim=-1)
    prod = [(x, y) for x in _carts(la) for y in _carts(lb)]
    out = None
    for d in range(3):
        at = _index([[(x[d] * (lb + 1) + y[d]) * (L + 1) + t[d] for t in _hermites(L)] for x, y in prod])
        f = T[:, d, :][:, at]
        out = f if out is None else out * f
    return out


def _coulomb(L, alpha, R):
    """Hermite Coulomb integrals R_tuv, t+u+v <= L, without prefactor."""
    F = _boys(L, alpha * (R * R).sum(dim=1))
    cur = F[:, L:] * (-2.0 * alpha[:, None]) ** L
    for n in range(L - 1, -1, -1):
        herm = _hermites(L - n)
        where = {t: k for k, t in enumerate(_hermites(L - n - 1))}
        one, two, num, axis = [], [], [], []
        for t in herm[1:]:
            d = next(k for k in range(3) if t[k])
            e = tuple(v - (k == d) for k, v in enumerate(t))
            f = tuple(v - 2 * (k == d) for k, v in enumerate(t))
            one.append(where[e])
            two.append(where.get(f, 0))
            num.append(t[d] - 1 if f in where else 0)
            axis.append(d)
        rest = R[:, _index(axis)] * cur[:, _index(one)] \
            + torch.tensor(num, dtype=torch.float64, device=DEV) * cur[:, _index(two)]
        cur = torch.cat([F[:, n:n + 1] * (-2.0 * alpha[:, None]) ** n, rest], dim=1)
    return cur


class _Flat:
    """Shells as flat arrays on the device."""

    def __init__(self, shells):
        n = [len(s[2]) for s in shells]
        self.l = np.array([s[0] for s in shells])
        self.depth = np.array(n, dtype=np.int64)
        self.first = _index(np.concatenate([[0], np.cumsum(n)[:-1]]).tolist())
        self.exp = torch.tensor(np.concatenate([s[2] for s in shells]), dtype=torch.float64, device=DEV)
        self.coef = torch.tensor(np.concatenate(_normalized(shells)), dtype=torch.float64, device=DEV)
        self.xyz = torch.tensor(np.array([s[1] for s in shells]), dtype=torch.float64, device=DEV)

    def primitives(self, idx):
        """Every primitive tuple of the shell tuples idx: (tuple, primitive
        of each shell)."""
        k = torch.from_numpy(self.depth).to(DEV)[idx]
        n = k.prod(dim=1)
        t = torch.repeat_interleave(torch.arange(len(idx), device=DEV), n)
        r = torch.arange(int(n.sum()), device=DEV) - (torch.cumsum(n, 0) - n)[t]
        prim = []
        for c in range(idx.shape[1] - 1, -1, -1):
            kc = k[t, c]
            prim.insert(0, self.first[idx[t, c]] + r % kc)
            r = torch.div(r, kc, rounding_mode="floor")
        return t, prim


def _eri_class(flat, idx, am, weight=None):
    """(ab|cd) of the shell quadruples idx as functions of momenta am (which
    may differ from the shells' own), [n, ncart(abcd)]; weight: a centre
    whose primitives are weighted by twice their exponent."""
    la, lb, lc, ld = am
    Hb, Hk = _hermites(la + lb), _hermites(lc + ld)
    where = {t: k for k, t in enumerate(_hermites(sum(am)))}
    at = _index([[where[tuple(x + y for x, y in zip(t, u))] for u in Hk] for t in Hb])
    sign = torch.tensor([(-1.0) ** sum(u) for u in Hk], dtype=torch.float64, device=DEV)
    nab, ncd = _ncart(la) * _ncart(lb), _ncart(lc) * _ncart(ld)
    out = torch.zeros((len(idx), nab * ncd), dtype=torch.float64, device=DEV)
    t, prim = flat.primitives(idx)
    step = max(1, CHUNK_VALUES // max(len(Hb) * len(Hk), nab * len(Hb), ncd * len(Hk), nab * ncd, nab * len(Hk)))
    for s in range(0, len(t), step):
        q = t[s:s + step]
        pr = [x[s:s + step] for x in prim]
        a, b, c, d = (flat.exp[x] for x in pr)
        A, B, C, D = (flat.xyz[idx[q, k]] for k in range(4))
        p, r = a + b, c + d
        P = (a[:, None] * A + b[:, None] * B) / p[:, None]
        Q = (c[:, None] * C + d[:, None] * D) / r[:, None]
        f = 2.0 * math.pi ** 2.5 / (p * r * torch.sqrt(p + r))
        for x in pr:
            f = f * flat.coef[x]
        if weight is not None:
            f = f * 2.0 * flat.exp[pr[weight]]
        M = _coulomb(sum(am), p * r / (p + r), P - Q)[:, at] * sign
        Eb = _expansion(la, lb, a, b, A, B) * f[:, None, None]
        Ek = _expansion(lc, ld, c, d, C, D).transpose(1, 2).contiguous()
        out.index_add_(0, q, torch.matmul(torch.matmul(Eb, M), Ek).reshape(len(q), -1))
    return out


def _deriv_class(flat, idx, am):
    """First derivatives, [n, ncart(abcd), 12]: centres A, B, C from the
    (a+1) and (a-1) classes, D from translational invariance."""
    n = [_ncart(l) for l in am]
    out = torch.zeros([len(idx)] + n + [4, 3], dtype=torch.float64, device=DEV)
    for c in range(3):
        blocks = {}
        for s in (1, -1):
            m = list(am)
            m[c] += s
            if m[c] >= 0:
                blocks[s] = _eri_class(flat, idx, m, c if s > 0 else None).reshape(
                    [len(idx)] + [_ncart(l) for l in m])
        for k, e in enumerate(_carts(am[c])):
            for x in range(3):
                up = tuple(v + (y == x) for y, v in enumerate(e))
                v = blocks[1].select(c + 1, _carts(am[c] + 1).index(up)).clone()
                if e[x]:
                    down = tuple(v2 - (y == x) for y, v2 in enumerate(e))
                    v -= e[x] * blocks[-1].select(c + 1, _carts(am[c] - 1).index(down))
                out[..., c, x].select(c + 1, k).copy_(v)
    out[..., 3, :] = -out[..., :3, :].sum(dim=-2)
    return out.reshape(len(idx), -1)


def _exact_quartets(shells, q, deriv=0):
    """All integrals of the quartets q in their order, flat."""
    flat = _Flat(shells)
    am = flat.l[q]
    size = ((am + 1) * (am + 2) // 2).prod(axis=1) * (12 if deriv else 1)
    off = np.zeros(len(q), dtype=np.int64)
    off[1:] = np.cumsum(size)[:-1]
    out = torch.empty(int(size.sum()), dtype=torch.float64, device=DEV)
    code = am @ np.array([64, 16, 4, 1])
    for c in np.unique(code):
        sel = np.nonzero(code == c)[0]
        l = tuple(int(x) for x in am[sel[0]])
        idx = torch.from_numpy(q[sel]).to(DEV)
        v = _deriv_class(flat, idx, l) if deriv else _eri_class(flat, idx, l)
        at = torch.from_numpy(off[sel]).to(DEV)[:, None] + torch.arange(v.shape[1], device=DEV)
        out[at.reshape(-1)] = v.reshape(-1)
    return out


def _exact_jk(case, seed):
    """J and K of the full four-index tensor of a small molecule."""
    shells, _ = _shells(case, seed)
    flat = _Flat(shells)
    n = len(shells)
    first = np.concatenate([[0], np.cumsum([_ncart(s[0]) for s in shells])])
    nbf = int(first[-1])
    g = torch.Generator().manual_seed(seed)
    C = torch.rand((nbf, max(1, nbf // 4)), generator=g, dtype=torch.float64) - 0.5
    D = (C @ C.T / nbf).to(DEV)
    fun = torch.from_numpy(first[:-1]).to(DEV)
    bra = np.array([(i, j) for i in range(n) for j in range(i + 1)], dtype=np.int64)
    cls = flat.l[bra] @ np.array([4, 1])
    G = torch.zeros((nbf,) * 4, dtype=torch.float64, device=DEV)
    for cb in np.unique(cls):
        for ck in np.unique(cls):
            if ck > cb:
                continue
            x, y = bra[cls == cb], bra[cls == ck]
            q = np.concatenate([np.repeat(x, len(y), axis=0), np.tile(y, (len(x), 1))], axis=1)
            for s in range(0, len(q), 100000):
                idx = torch.from_numpy(q[s:s + 100000]).to(DEV)
                am = [int(v) for v in flat.l[q[s]]]
                v = _eri_class(flat, idx, am).reshape([len(idx)] + [_ncart(l) for l in am])
                at = [(fun[idx[:, k]].reshape(-1, 1, 1, 1, 1)
                       + torch.arange(_ncart(am[k]), device=DEV).reshape([-1 if m == k else 1 for m in range(4)]))
                      for k in range(4)]
                at = [z.expand(v.shape) for z in at]
                for b in ((0, 1), (1, 0)):
                    for k in ((2, 3), (3, 2)):
                        G[at[b[0]], at[b[1]], at[k[0]], at[k[1]]] = v
                        G[at[k[0]], at[k[1]], at[b[0]], at[b[1]]] = v
    J = (G.reshape(nbf * nbf, -1) @ D.reshape(-1)).reshape(nbf, nbf)
    K = torch.stack([(G[m].permute(1, 0, 2).reshape(nbf, -1) @ D.reshape(-1)) for m in range(nbf)])
    return {"J": J, "K": K}


def _exact_oei(case, seed):
    shells, pairs, off, n, charges = _oei_inputs(case, seed)
    flat = _Flat(shells)
    out = {k: torch.empty(n, dtype=torch.float64, device=DEV) for k in ("overlap", "ke", "potential")}
    Z = torch.from_numpy(charges[:, 0].copy()).to(DEV)
    X = torch.from_numpy(charges[:, 1:].copy()).to(DEV)
    code = flat.l[pairs] @ np.array([4, 1])
    for c in np.unique(code):
        sel = np.nonzero(code == c)[0]
        la, lb = (int(x) for x in flat.l[pairs[sel[0]]])
        idx = torch.from_numpy(pairs[sel].astype(np.int64)).to(DEV)
        t, (pa, pb) = flat.primitives(idx)
        a, b = flat.exp[pa], flat.exp[pb]
        A, B = flat.xyz[idx[t, 0]], flat.xyz[idx[t, 1]]
        p = a + b
        f = flat.coef[pa] * flat.coef[pb]

        def overlap(lb2, extra):
            E = _expansion(la, lb2, a, b, A, B)[:, :, 0]
            v = E * (f * extra * (math.pi / p) ** 1.5)[:, None]
            r = torch.zeros((len(idx), v.shape[1]), dtype=torch.float64, device=DEV)
            return r.index_add_(0, t, v).reshape(len(idx), _ncart(la), _ncart(lb2))
        one = torch.ones_like(b)
        S = overlap(lb, one)
        # -1/2 d2/dx2 of x^j e^(-b x^2): -2 b^2 x^(j+2) + b (2j+1) x^j - j(j-1)/2 x^(j-2)
        T = torch.zeros_like(S)
        up, same = overlap(lb + 2, -2.0 * b * b), overlap(lb, b)
        down = overlap(lb - 2, one) if lb >= 2 else None
        for k, e in enumerate(_carts(lb)):
            for d in range(3):
                T[:, :, k] += up[:, :, _carts(lb + 2).index(tuple(v + 2 * (y == d) for y, v in enumerate(e)))]
                T[:, :, k] += (2 * e[d] + 1) * same[:, :, k]
                if e[d] >= 2:
                    T[:, :, k] -= 0.5 * e[d] * (e[d] - 1) * \
                        down[:, :, _carts(lb - 2).index(tuple(v - 2 * (y == d) for y, v in enumerate(e)))]
        P = (a[:, None] * A + b[:, None] * B) / p[:, None]
        R = torch.zeros((len(p), len(_hermites(la + lb))), dtype=torch.float64, device=DEV)
        for z, x in zip(Z, X):
            R += z * _coulomb(la + lb, p, P - x)
        v = (_expansion(la, lb, a, b, A, B) * R[:, None, :]).sum(dim=2) * (-2.0 * math.pi / p * f)[:, None]
        V = torch.zeros((len(idx), v.shape[1]), dtype=torch.float64, device=DEV).index_add_(0, t, v)
        at = (torch.from_numpy(off[sel]).to(DEV)[:, None] + torch.arange(V.shape[1], device=DEV)).reshape(-1)
        for k, v in (("overlap", S), ("ke", T), ("potential", V)):
            out[k][at] = v.reshape(-1)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "call":
        shells, (bra, ket) = _shells(case, seed)
        if len(bra) * len(ket) * case["depth"] ** 4 > 2e6:
            return None         # the large blocks take too long
        q = np.array([x + y for x in bra for y in ket], dtype=np.int64)
        return _exact_quartets(shells, q).cpu().numpy()
    if kind in ("list", "stream"):
        if case["quartets"] > (1500 if kind == "list" else 9000):
            return None
        shells, q = _shells(case, seed)
        return _exact_quartets(shells, np.asarray(q, dtype=np.int64), case.get("deriv", 0))
    if kind == "jk":
        return _exact_jk(case, seed) if case["atoms"] <= 10 else None
    if kind == "oei":
        return _exact_oei(case, seed)
    return None                 # the layout of a screened set follows its plan
