"""HIP writer: component-lane (CPL) kernels for one (ab|cd) class.

For classes whose recurrence does not fit one lane's registers.  The VRR
reduces the side of the smaller total AM first (rrgraph: centres in the
order of their largest AM), so every value is built in two stages: up the
wide side E with the narrow side S at zero, then up the narrow side.  A lane
holds ONE component e of the wide side (all of AM 0 .. E_hi: 84 lanes for an
(ff| pair), and walks

1. its own chain (e0|00)^m from (00|00)^m: a component's reduction path runs
   along one direction at a time (lowest non-zero exponent first), so both
   sources of every step lie on the path; the direction's constants come
   from the local data share by a per-lane offset, and lanes of lower AM take
   identity steps first.  No lane needs another's values here;
2. the narrow side's components f in depth-first order, the same f in every
   lane at the same time (straight-line code, no descriptors): the vector
   (ef)^m, m = 0 .. S_hi - |f|, from the parent's and grandparent's vectors
   in the lane's registers, and from lane (e - 1_d)'s parent vector, which
   that lane left in the local data share;
3. the contraction of (e0|f0) for every top f in registers.

64 NS lane slots of a wavefront hold NQ quartets of NE components.  Per VRR
value that is at most one 8-byte read and one write of the local data share,
where the cooperative kernels (hip_wpq.py) read twelve values and a 32-byte
descriptor and wait at a barrier per level.  G wavefronts of a workgroup may
share the tops f between them, each walking the part of the tree its own
need and the chains once between them (one barrier a primitive quartet):
fewer accumulators a lane, and more hands on a deep quartet.  Or SW
wavefronts share the primitive quartets, which repeats nothing but adds the
contraction in another order.

HRR through the local data share, the reference's order: bra transfers with
one lane per (quartet, ket top), then ket transfers with one lane per
(quartet, bra component), then one contiguous copy to the output.  Every
step's arithmetic and order is the lane-per-quartet kernels' (setup:
generator/ostei/OSTEI_Writer.cpp:595-702; VRR: OSTEI_VRR_Writer.cpp:95-125;
HRR: OSTEI_HRR_Writer.cpp:22-99), so the values are theirs bit for bit
where the contraction runs in one lane there.

Bound: latency at one or two wavefronts a SIMD.  On the 256-atom system
(dd|dp) issues vector instructions in 42 % of the cycles (three to five FP64
operations per value), the local data share works in 41 %, HBM at 27 % of its
rate.  About two thirds of the kernels also keep some of their values in
scratch: the register bound (Plan.regs) counts the tree and the accumulators,
while in the HRR a lane holds a whole column.  Lists of the mixed-class stream
(all classes one after another, 100000 quartets): 560 ms with the cooperative
and lane-per-quartet kernels; the 186 classes that run these take 94 ms,
(ff|ff) 11.8 -> 3.4 ms, (ff|fd) 18.9 -> 2.7 ms, (dd|dd) 5.3 -> 0.9 ms.  Ranges
of a 24-atom molecule: (dd|dp) 2.02 -> 0.96 ms, (dp|dp) 1.70 -> 1.23, (dd|dd)
0.59 -> 0.32; random pairs: (ff|ff) 76.6 -> 29.4 ms, (fd|fd) 30.4 -> 5.6.
Screened primitive quartets are left out where a group's quartets all are.
"""
from functools import lru_cache

from .hip_lpq import class_name, _Writer
from .rrgraph import cart_index, carts, graph, mk_dir, ncart, step

ENT = 16           # primitive quartets per setup batch (one lane each), at most
QINFO = 8          # per quartet: AB and CD, output base
LDS_CU = 160 * 1024
AREA_GOOD = 22 * 1024    # HRR area up to which four to eight wavefronts share a CU
# List launches of at most SPLIT_GROUPS groups share a group between wavefronts
# where a quartet has SPLIT_DEEP primitive quartets or more, of SPLIT_SOME from
# SPLIT_DEPTH on (SPLIT_GROUPS where the unshared kernel has one wavefront a
# SIMD: 3200 (dd|dd) quartets of 16 take 146 us unshared and 137 shared, of
# (fd|pp) 54 and 81), of SPLIT_FEW (one a compute unit) whatever the depth: for
# one primitive quartet seven of eight wavefronts wait.  3200 (fp|ps) quartets
# of 1, 16 and 256 primitive quartets: 11, 38 and 474 us unshared, 57, 84 and
# 275 shared; 200: 10, 35 and 442, 7, 10 and 25.
SPLIT_GROUPS = 4096
SPLIT_SOME = 1024
SPLIT_FEW = 256
SPLIT_DEPTH = 16
SPLIT_DEEP = 64
SPLIT_W = 4              # between so many wavefronts (primitive quartets: up to twice as many)
# Lists of at most this many groups (four classes side by side then have one
# a compute unit) share a group's tops between twice as many wavefronts,
# where that shortens the longest wavefront's work to DEEP_GAIN of it.  The
# paths to the tops are walked by more of them: about 1.3 times the work in
# all, so longer lists, which fill the chip, do not.  256 classes of 32
# quartets: 16.0 ms with four wavefronts a group, 15.1 with eight.
DEEP_GROUPS = 64
DEEP_GAIN = 0.75
SUM_VALUES = 8           # accumulators added per round where primitive quartets are shared
# The most AM transferred in the HRR of a class that shares them: another order
# of the sum rounds otherwise, and the HRR amplifies it.  On the mixed-class
# stream (300000 quartets in a 30-bohr cube, 8 seeds) sharing moved a set by up
# to 2.5e-14 of its norm and single integrals by 1.8e-10 of its root mean
# square.  As terms of first derivatives, weighted by 2a, classes of 3 moved
# 1500 derivatives by up to 2e-8 of their norm, classes of 2 by 7e-12 (12
# seeds).  The lanes that share a derivative list's lane-per-quartet quartet
# keep the same limit (runtime.hip): with 2 they move it by 1.1e-14, with 3 by
# 1.2e-9.  Plain lane-per-quartet lists have none (classes of 3: 2.1e-12 of the
# norm, 2.8e-8 of the root mean square).  What sharing is worth, with limits of
# 3, 2 and 1: 8192 quartets 12.8, 16.0 and 20.4 ms, 300000 quartets 44.2, 47.8
# and 52.9, 1500 derivatives 48, 66 and 83; with the lanes at 2 as well 60.
SHARE_AM = 2

# primitive-quartet block of the local data share, in doubles
P_E, P_ID, P_EOVER, P_EO2, P_S, P_SOVER, P_SO2, P_O2PQ, P_F = 0, 6, 8, 9, 10, 16, 17, 18, 20


class Plan:
    """Sizes and tables of one class: G wavefronts share a group's tops, or
    SW wavefronts its primitive quartets.  With SPLIT_W or more of them (short
    lists, which leave the chip idle anyway) a wavefront takes the fewest
    lane slots."""

    def __init__(self, am, G, SW):
        g = self.g = graph(*am)
        self.am, self.G, self.SW, self.W = am, G, SW, G * SW
        assert G == 1 or SW == 1
        latency = self.latency = max(G, SW) >= SPLIT_W
        self.L = g.Ltot
        # the side reduced first is the narrow one (g.order lists centres in
        # the order of reduction)
        self.s_is_ket = g.f_hi <= g.e_hi
        bra = (g.e_lo, g.e_hi)
        ket = (g.f_lo, g.f_hi)
        (self.s_lo, self.s_hi), (self.e_lo, self.e_hi) = (ket, bra) if self.s_is_ket else (bra, ket)
        assert self.s_hi <= self.e_hi
        self.comps = [e for l in range(self.e_hi + 1) for e in carts(l)]
        self.NE = len(self.comps)
        self.index = {e: i for i, e in enumerate(self.comps)}
        self.first_top = self.index[carts(self.e_lo)[0]]
        self.net = self.NE - self.first_top
        self.stops = [f for l in range(self.s_lo, self.s_hi + 1) for f in carts(l)]
        la, lb, lc, ld = am
        self.nab, self.ncd = ncart(la) * ncart(lb), ncart(lc) * ncart(ld)
        self.nbt, self.nkt = len(g.bra_tops()), len(g.ket_tops())
        npc = P_F + self.L + 1
        while npc % 4 != 2:                                    # 16-byte rows, spread over the banks
            npc += 1
        self.npc = npc
        # published vectors: one buffer per depth with children
        self.pub_level = [0] * (self.s_hi + 1)
        n = 0
        for l in range(self.s_hi):
            self.pub_level[l] = n
            n += self.s_hi - l
        self.npub = n
        best = None
        for NS in (1, 2, 3):
            c = self._shape(NS)
            if c and latency and best:
                break
            if c and (best is None or c[0] > best[0] * 1.02):
                best = c
        if best is None:
            raise ValueError("class %s does not fit the component-lane kernel" % (am,))
        _, self.NS, self.NQ, self.HQ, self.hold, self.nch, self.area, self.ent, self.occ = best
        self._tree(self.NS)
        self.ps = self.NQ * self.NE + 1            # lanes beyond the components share the last slot
        self.blocks = self.ent * (self.npc + QINFO)
        self.lds_doubles = self.SW * self.blocks + self.area
        self.cc = -(-self.nab // self.nch)

    def chain_slots(self, part):
        """Lane slots whose chain wavefront `part` computes for all G."""
        return list(range(part, self.NS, self.G))

    def _tree(self, NS):
        """Children of every narrow component the tops' paths visit, and the
        tops shared between the G wavefronts: runs of the depth-first order
        of about equal work."""
        def path(f):
            out = [f]
            while sum(f):
                f = step(f, mk_dir(f), -1)
                out.append(f)
            return out
        need = set(x for f in self.stops for x in path(f)) | {(0, 0, 0)}
        self.children = {f: [] for f in need}
        for f in sorted(need, key=lambda f: (sum(f), cart_index(f))):
            if sum(f):
                self.children[step(f, mk_dir(f), -1)].append(f)
        order = []

        def visit(f):
            order.append(f)
            for c in self.children[f]:
                visit(c)
        visit((0, 0, 0))
        tops = set(self.stops)
        seq = [f for f in order if f in tops]

        def cost(part):
            return NS * sum(self.s_hi - sum(f) + 2 for f in set(x for f in part for x in path(f)))
        # a wavefront's work is its part of the tree and its share of the
        # chains; smallest largest work: grow each part up to a bound, raise
        # the bound
        own = [len(range(part, NS, self.G)) * sum(self.L - k for k in range(self.e_hi)) for part in range(self.G)]
        bound = (cost(seq) + sum(own)) // self.G
        while True:
            parts = [[] for _ in range(self.G)]
            at = 0
            for f in seq:
                while at < self.G and own[at] + cost(parts[at] + [f]) > bound:
                    at += 1
                if at == self.G:
                    break
                parts[at].append(f)
            if at < self.G:
                break
            bound += 1
        self.longest = bound
        self.parts = parts
        self.part_nodes = [set(x for f in p for x in path(f)) for p in self.parts]
        self.nacc = max(len(p) for p in self.parts)

    def root_doubles(self, ps):
        """Two buffers of the chains' results where wavefronts share them."""
        return 2 * (self.s_hi + 1) * ps if self.G > 1 else 0

    def regs(self, NS):
        """Rough VGPR count: path vectors, accumulators, constants."""
        path = (self.s_hi + 1) * (self.s_hi + 2) // 2
        chain = 2 * (self.L + 1)
        per = max(path + self.nacc, chain + 4) + 12
        return 2 * NS * per + 40

    def _hrr(self, NQ):
        """How the HRR of NQ quartets runs: HQ at a time, in place (each
        column of the tops becomes the column of its bra transfers) or with
        every lane holding its column's results while the rows pass through
        the area in nch parts; (rounds, doubles, HQ, hold, nch)."""
        best = None
        lanes = 64 * self.W
        ks = max(self.nkt, self.ncd) | 1
        for HQ in range(1, NQ + 1):
            if NQ % HQ:
                continue
            opts = [(False, 1, HQ * max(self.nbt, self.nab) * ks)]
            if HQ * self.nkt <= lanes:
                for nch in range(1, 7):
                    rows = -(-self.nab // nch)
                    opts.append((True, nch, HQ * max(self.nbt * (self.nkt | 1), rows * ks)))
            for hold, nch, area in opts:
                rows = -(-self.nab // nch)
                rounds = NQ // HQ * (-(-HQ * self.nkt // lanes) + nch * (-(-HQ * rows // lanes) + 0.5))
                key = (8 * area > AREA_GOOD * self.W, rounds if 8 * area <= AREA_GOOD * self.W else area, area)
                if best is None or key < best[0]:
                    best = (key, rounds, area, HQ, hold, nch)
        return best[1:]

    def _shape(self, NS):
        """Lane slots per wavefront: the share of the lanes at work times
        how well the wavefronts a SIMD holds hide each other's latencies."""
        NQ = min(64 * NS // self.NE, ENT)
        if NQ < 1:
            return None
        self._tree(NS)
        regs = self.regs(NS)
        if regs > 500:
            return None
        rounds, area, HQ, hold, nch = self._hrr(NQ)
        ps = NQ * self.NE + 1
        area = max(area, self.W * self.npub * ps + self.root_doubles(ps), SUM_VALUES * 64 * (self.SW - 1), 64)
        area += area % 2
        ent = ENT // NQ * NQ
        lds = 8 * (self.SW * ent * (self.npc + QINFO) + area)
        if lds > LDS_CU:
            return None
        occ = min(512 // regs, 4)
        held = min(occ, LDS_CU // lds * self.W / 4.0)
        eff = NQ * self.NE / (64.0 * NS)
        score = eff * (1.0 - 0.4 / max(1.0, held) ** 1.5) * (min(1.0, held) if held < 1 else 1.0)
        # register bound of the compiler: wavefronts per SIMD to leave room for
        bound = max(1, min(occ, 2 if self.latency else 4, -int(-held // 1)))
        return score, NS, NQ, HQ, hold, nch, area, ent, bound

    def lane_tables(self):
        """Per wide component: directions of its chain's E_hi steps (2 bits
        each, 3 = identity), exponent before each step (4 bits), exponents
        (4 bits per direction) and lane distance to e - 1_d (16 bits each,
        0 where the exponent is 0)."""
        rows = []
        for e in self.comps:
            path = []
            f = e
            while sum(f):
                d = mk_dir(f)
                path.append((d, f[d] - 1))
                f = step(f, d, -1)
            path.reverse()
            path = [(3, 0)] * (self.e_hi - len(path)) + path
            dirs = sum(d << (2 * k) for k, (d, _) in enumerate(path))
            ns = sum(n << (4 * k) for k, (_, n) in enumerate(path))
            ex = sum(e[d] << (4 * d) for d in range(3))
            dn = [self.index[e] - self.index[step(e, d, -1)] if e[d] else 0 for d in range(3)]
            rows.append((dirs, ns, ex, dn[0] | dn[1] << 8 | dn[2] << 16))
            assert max(dn) < 256
        return rows


@lru_cache(maxsize=None)
def plan(am, G=1, SW=1):
    return Plan(am, G, SW)


def split_plan(am):
    """Plan of the short-list kernel.  Sharing the primitive quartets
    repeats no work, but adds the contraction in another order; the HRR
    amplifies the difference by about the pairs' extent to the power of the
    AM it transfers, so classes that transfer more share the tops instead."""
    if min(am[0], am[1]) + min(am[2], am[3]) > SHARE_AM:
        return plan(am, SPLIT_W, 1)
    p = plan(am, 1, 2 * SPLIT_W)
    return p if 16 * p.lds_doubles <= LDS_CU else plan(am, 1, SPLIT_W)


def deep_plan(am):
    """Plan of the kernel for the shortest lists, or None.  Tops shared in
    another way leave every value's arithmetic as it is.  Eight wavefronts a
    workgroup leave 256 registers to each."""
    ps = split_plan(am)
    if ps.G == 1:
        return None
    try:
        p = plan(am, 2 * SPLIT_W, 1)
    except ValueError:
        return None
    if p.regs(p.NS) > 240 or p.NQ != ps.NQ or p.longest > DEEP_GAIN * ps.longest:
        return None
    return p


def base_G(am):
    """Wavefronts a workgroup of the range and long-list kernels: one where
    its HRR area leaves four of them a CU's local data share."""
    try:
        if 8 * plan(am, 1).area <= 2 * AREA_GOOD:
            return 1
    except ValueError:
        pass
    return 2


def candidate(am):
    """Classes this family is built for: a wide side of at least f in all,
    and a narrow side of at least p (the (gf|ss) derivative terms have no
    lane-per-quartet kernel; lower (ab|ss) classes run that); classes with
    an HRR and a wide side of d for their small launches."""
    g = graph(*am)
    wide, narrow = max(g.e_hi, g.f_hi), min(g.e_hi, g.f_hi)
    hrr = g.bra_hrr_needed() or g.ket_hrr_needed()
    if wide < (7 if narrow == 0 else 2 if hrr else 3):
        return False
    try:
        plan(am, base_G(am))
    except ValueError:
        return False
    return True


def emit_cpl(am):
    G = base_G(am)
    p, ps, pd = plan(am, G), split_plan(am), deep_plan(am)
    w = _Writer()
    w("// Generated by simint-generator_amd/emitter/hip_cpl.py -- class (%s)" % class_name(am).replace("_", ""))
    w('#include "../device_types.h"')
    w('#include "../boys_device.h"')
    w("")
    w("namespace {")
    w("constexpr int NE = %d, NPC = %d, QINFO = %d, DEEP_GROUPS = %d;" % (p.NE, p.npc, QINFO, DEEP_GROUPS))
    w("constexpr int SPLIT_GROUPS = %d, SPLIT_SOME = %d, SPLIT_FEW = %d, SPLIT_DEPTH = %d, SPLIT_DEEP = %d;"
      % (SPLIT_GROUPS, SPLIT_SOME if p.occ > 1 else SPLIT_GROUPS, SPLIT_FEW, SPLIT_DEPTH, SPLIT_DEEP))
    w("// per wide component: chain directions, chain exponents, exponents, lane distances to e - 1_d")
    w("__constant__ __attribute__((aligned(16))) unsigned int lane_tab[NE][4] = {")
    for r in p.lane_tables():
        w("    {%s}," % ", ".join("%du" % x for x in r))
    w("};")
    w("__device__ __forceinline__ void wave_fence()")
    w("{")
    w("    // one wavefront: its local data share operations complete in order,")
    w("    // only the compiler must keep them so")
    w('    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");')
    w("    __builtin_amdgcn_wave_barrier();")
    w("}")
    w("}  // namespace")
    w("")
    _emit_kernel(p, w, "range")
    _emit_kernel(p, w, "list")
    _emit_kernel(ps, w, "split")
    if pd:
        _emit_kernel(pd, w, "deep")
    _emit_launchers(p, ps, pd, w)
    return w.text()


def _emit_kernel(p, w, mode):
    """mode "range": a bra against the kets of a tile; "list": a run of
    groups of NQ quartets of a list; "split", "deep": the same with more
    wavefronts a group."""
    name = class_name(p.am)
    NS, NQ, G, SW = p.NS, p.NQ, p.G, p.SW
    listmode = mode != "range"
    kname = {"range": "eri_cpl_%s", "list": "eri_cpll_%s", "split": "eri_cpls_%s", "deep": "eri_cpld_%s"}[mode] % name
    w("__global__ void __launch_bounds__(%d, %d) %s(const %s A%s)"
      % (64 * p.W, p.occ, kname, "EriListArgs" if listmode else "EriArgs", ", int groups" if listmode else ""))
    w("{")
    w("    constexpr int NQ = %d, ENT = %d, PS = %d;" % (NQ, p.ent, p.ps))
    w("    // primitive-quartet blocks, quartet blocks, then published vectors")
    w("    // (recurrence) or rows of tops and results (HRR)")
    w("    __shared__ __attribute__((aligned(16))) double lds[%d];" % p.lds_doubles)
    w("    const int lane = threadIdx.x;")
    if p.W > 1:
        w("    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);")
        w("    const int tid = wave * 64 + lane;")
        w("    double *const area = lds + %d;" % (SW * p.blocks))
        w("    double *const pub = area + wave * %d;" % (p.npub * p.ps))
    else:
        w("    const int tid = lane;")
        w("    double *const area = lds + %d;" % p.blocks)
        w("    double *const pub = area;")
    if SW > 1:
        # each wavefront prepares its own primitive quartets; the HRR reads
        # the first one's quartet blocks (it always has a share)
        w("    double *const pc = lds + wave * %d;" % p.blocks)
        w("    double *const qmine = pc + ENT * NPC;")
        w("    double *const qi = lds + ENT * NPC;")
    else:
        w("    double *const pc = lds;")
        w("    double *const qi = lds + ENT * NPC;")
    if G > 1:
        w("    double *const roots = area + %d;   // two buffers of the chains' results" % (p.W * p.npub * p.ps))
        w("    int turn = 0;")
    w("    const double *__restrict__ grid = A.boys_grid;")
    w("    const bool screen = A.tol2 > 0.0;")
    if not listmode:
        w("    const WorkItem wi = A.items[blockIdx.x];")
        w("    const int ib0 = A.bra.poff[wi.bra];")
        w("    const int npb = A.bra.np[wi.bra];")
        w("    const int nq = A.ket.tnp[wi.tile];")
        w("    const long long kt = A.ket.toff[wi.tile];")
        w("    // this block's share of the item's kets, in groups of NQ")
        w("    const int ng = (wi.lane_hi - wi.lane_lo + NQ - 1) / NQ;")
        w("    const int gper = (ng + (int)gridDim.y - 1) / (int)gridDim.y;")
        w("    const int gbeg = (int)blockIdx.y * gper;")
        w("    const int gend = gbeg + gper < ng ? gbeg + gper : ng;")
        w("    const int q_first = wi.lane_lo, q_end = wi.lane_hi;")
        w("    const int K = npb * nq > 0 ? npb * nq : 1;   // no primitives: one that adds nothing")
    else:
        w("    const int q_first = 0, q_end = (int)A.nquartet;")
        w("    const int ngl = (q_end + NQ - 1) / NQ;")
        w("    const int gbeg = (int)blockIdx.x * groups;")
        w("    const int gend = gbeg + groups < ngl ? gbeg + groups : ngl;")
        w("    // primitive quartets of the deepest quartet of this block")
        w("    int K = 1;")
        w("    for (int q = gbeg * NQ + lane; q < gend * NQ && q < q_end; q += 64) {")
        w("        const int k = A.bra.np[A.qbra[q]] * A.ket.np[A.qket[q]];")
        w("        K = k > K ? k : K;")
        w("    }")
        w("#pragma unroll")
        w("    for (int o = 32; o > 0; o >>= 1) {")
        w("        const int k = __shfl_xor(K, o);")
        w("        K = k > K ? k : K;")
        w("    }")
        w("    K = __builtin_amdgcn_readfirstlane(K);")
    if SW > 1:
        w("    const int share = (K + %d) / %d;" % (SW - 1, SW))
        w("    const int p_end = (wave + 1) * share < K ? (wave + 1) * share : K;")
        w("    const int PBK = share < ENT / NQ ? share : ENT / NQ;")
        w("    const int GB = 1;")
    else:
        w("    const int p_end = K;")
        w("    const int PBK = K < ENT / NQ ? K : ENT / NQ;")
        w("    const int GB = PBK == K ? ENT / NQ / K : 1;   // groups per setup batch")
    for s in range(NS):
        w("    const int idx%d = %d + lane < NQ * NE ? %d + lane : NQ * NE;" % (s, 64 * s, 64 * s))
        w("    const bool use%d = idx%d < NQ * NE;" % (s, s))
        w("    const int w%d = use%d ? idx%d / NE : 0;" % (s, s, s))
        w("    const int e%d = use%d ? idx%d - w%d * NE : 0;" % (s, s, s, s))
        w("    const uint4 tab%d = *(const uint4 *)lane_tab[e%d];" % (s, s))
        for d in range(3):
            w("    const int nb%d_%d = idx%d - (int)((tab%d.w >> %d) & 255u);" % (s, d, s, s, 8 * d))
        for t in range(p.nacc):
            w("    double acc%d_%d = 0.0;" % (s, t))
    w("#pragma unroll 1")
    w("    for (int g0 = gbeg; g0 < gend; g0 += GB) {")
    w("#pragma unroll 1")
    w("        for (int p0 = %s; p0 < p_end; p0 += PBK) {" % ("wave * share" if SW > 1 else "0"))
    w("            const int npb_ = p_end - p0 < PBK ? p_end - p0 : PBK;")
    fence = "wave_fence();"
    sync = "__syncthreads();" if p.W > 1 else fence
    w("            " + (sync if SW == 1 else fence))
    _emit_setup(p, w, listmode)
    w("            " + (sync if SW == 1 else fence))
    if G > 1:
        w("            if (screen) alive = (unsigned)__builtin_amdgcn_readfirstlane((int)((const unsigned *)qi)[14]);")
    w("            unsigned every = 0;   // primitive quartet 0 of every quartet of a group")
    w("#pragma unroll")
    w("            for (int v = 0; v < NQ; ++v) every |= 1u << (v * PBK);")
    if SW > 1:
        w("            const int gi = 0;")
    else:
        w("#pragma unroll 1")
        w("            for (int gi = 0; gi < GB && g0 + gi < gend; ++gi) {")
    for part in range(G):
        if G > 1:
            w("                if (wave == %d) {" % part)
        w("#pragma unroll 1")
        w("                for (int pp = 0; pp < npb_; ++pp) {")
        w("                    if (((alive >> (gi * NQ * PBK + pp)) & every) == 0) continue;")
        _emit_vrr(p, w, part)
        w("                }")
        if G > 1:
            w("                }")
    if SW > 1:
        w("        }")
        w("        const int gi = 0;")
        w("        {")
        _emit_sum(p, w)
    else:
        w("                if (p0 + PBK < K) continue;")
    _emit_hrr(p, w, sync)
    w("            }")
    if SW == 1:
        w("        }")
    w("    }")
    w("}")
    w("")


def _emit_launchers(p, ps, pd, w):
    name = class_name(p.am)
    w('extern "C" hipError_t simint_launch_cpl_%s(const EriArgs *a, hipStream_t s)' % name)
    w("{")
    w("    if (a->nitems <= 0) return hipSuccess;")
    w("    // few items: several blocks share an item's kets")
    w("    const int most = (SIMINT_TILE + %d) / %d;" % (p.NQ - 1, p.NQ))
    w("    int ny = 1;")
    w("    while (ny < most && a->nitems * ny < 4096) ny *= 2;")
    w("    hipLaunchKernelGGL(eri_cpl_%s, dim3((unsigned)a->nitems, (unsigned)ny), dim3(64, %d), 0, s, *a);" % (name, p.G))
    w("    return hipGetLastError();")
    w("}")
    w("")
    w('extern "C" hipError_t simint_launch_cpll_%s(const EriListArgs *a, hipStream_t s)' % name)
    w("{")
    w("    if (a->nquartet <= 0) return hipSuccess;")
    w("    if (a->nquartet > 0x7fff0000LL) return hipErrorInvalidValue;")
    w("    long long ng = (a->nquartet + %d) / %d;" % (ps.NQ - 1, ps.NQ))
    if pd:
        w("    if (ng <= DEEP_GROUPS) {")
        w("        hipLaunchKernelGGL(eri_cpld_%s, dim3((unsigned)ng), dim3(64, %d), 0, s, *a, 1);" % (name, pd.W))
        w("        return hipGetLastError();")
        w("    }")
    w("    const long long depth = a->depth > 0 ? a->depth : SPLIT_DEEP;")
    w("    if (ng <= (depth >= SPLIT_DEEP ? SPLIT_GROUPS : depth >= SPLIT_DEPTH ? SPLIT_SOME : SPLIT_FEW)) {")
    w("        hipLaunchKernelGGL(eri_cpls_%s, dim3((unsigned)ng), dim3(64, %d), 0, s, *a, 1);" % (name, ps.W))
    w("        return hipGetLastError();")
    w("    }")
    w("    ng = (a->nquartet + %d) / %d;" % (p.NQ - 1, p.NQ))
    w("    const int groups = ng > 65536 ? 8 : ng > 16384 ? 2 : 1;")
    w("    hipLaunchKernelGGL(eri_cpll_%s, dim3((unsigned)((ng + groups - 1) / groups)), dim3(64, %d), 0, s, *a, groups);"
      % (name, p.G))
    w("    return hipGetLastError();")
    w("}")


def _emit_setup(p, w, listmode):
    """Lane t prepares primitive quartet t of the batch: group t / (NQ PBK),
    quartet slot, primitive p0 + t % PBK."""
    g = p.g
    bra_pa = "pa" if g.bra_j else "pb"
    ket_pa = "pa" if g.ket_l else "pb"
    ind = "                "
    w("            const bool mine = %s < GB * NQ * PBK;" % ("lane" if p.SW > 1 else "tid"))
    w("            bool live = false;")
    w("            const int r = lane / PBK, pl = p0 + lane - r * PBK;")
    w("            const int qx = q_first + g0 * NQ + r;")
    w("            const int q = qx < q_end ? qx : q_end - 1;")
    if not listmode:
        w("            int i = 0;")
        w("            long long kj = 0;")
        w("            if (mine) {")
        w(ind + "live = qx < q_end && pl < npb * nq;")
        w(ind + "if (live) {")
        w(ind + "    i = ib0 + pl / nq;")
        w(ind + "    kj = kt + q + (long long)SIMINT_TILE * (pl % nq);")
    else:
        w("            int i = 0, kj = 0, bp = 0, kp = 0;")
        w("            if (mine) {")
        w(ind + "bp = A.qbra[q], kp = A.qket[q];")
        w(ind + "const int nq = A.ket.np[kp];")
        w(ind + "live = qx < q_end && pl < A.bra.np[bp] * nq;")
        w(ind + "if (live) {")
        w(ind + "    i = A.bra.poff[bp] + pl / nq;")
        w(ind + "    kj = A.ket.poff[kp] + pl % nq;")
    w(ind + "    if (screen && (A.bra.screen[i] * A.ket_screen_max < A.tol2 ||")
    w(ind + "                   A.bra.screen[i] * A.ket.screen[kj] < A.tol2)) live = false;")
    w(ind + "}")
    w("            }")
    # 16 lanes at most: a primitive quartet that is screened in every quartet
    # of the group is left out, and the preparation of a batch of such
    w("            %s = screen ? (unsigned)__ballot(live) : ~0u;" % ("unsigned alive" if p.G > 1 else "const unsigned alive"))
    w("            if (alive != 0 && mine) {")
    w(ind + "double P_alpha = 1.0, P_inv = 1.0, P_prefac = 0.0, Q_alpha = 1.0, Q_inv = 1.0, Q_prefac = 0.0;")
    w(ind + "double PA0 = 0.0, PA1 = 0.0, PA2 = 0.0, QC0 = 0.0, QC1 = 0.0, QC2 = 0.0, PQx = 0.0, PQy = 0.0, PQz = 0.0;")
    w(ind + "if (live) {")
    w(ind + "    P_alpha = A.bra.alpha[i]; P_inv = A.bra.inv_alpha[i]; P_prefac = A.bra.prefac[i];")
    w(ind + "    Q_alpha = A.ket.alpha[kj]; Q_inv = A.ket.inv_alpha[kj]; Q_prefac = A.ket.prefac[kj];")
    w(ind + "    PA0 = A.bra.%sx[i]; PA1 = A.bra.%sy[i]; PA2 = A.bra.%sz[i];" % (bra_pa, bra_pa, bra_pa))
    w(ind + "    QC0 = A.ket.%sx[kj]; QC1 = A.ket.%sy[kj]; QC2 = A.ket.%sz[kj];" % (ket_pa, ket_pa, ket_pa))
    w(ind + "    PQx = A.bra.x[i] - A.ket.x[kj];")
    w(ind + "    PQy = A.bra.y[i] - A.ket.y[kj];")
    w(ind + "    PQz = A.bra.z[i] - A.ket.z[kj];")
    w(ind + "}")
    w(ind + "const double PQalpha_mul = P_alpha * Q_alpha;")
    w(ind + "const double PQalpha_sum = P_alpha + Q_alpha;")
    w(ind + "const double one_over_PQalpha_sum = 1.0 / PQalpha_sum;")
    w(ind + "double R2 = PQx * PQx;")
    w(ind + "R2 = fma(PQy, PQy, R2);")
    w(ind + "R2 = fma(PQz, PQz, R2);")
    w(ind + "const double alpha = PQalpha_mul * one_over_PQalpha_sum;")
    w(ind + "double F[%d];" % (p.L + 1))
    w(ind + "boys_eval<%d>(grid, R2 * alpha, F);" % p.L)
    w(ind + "const double prefac = (P_prefac * Q_prefac) * sqrt(one_over_PQalpha_sum);")
    w(ind + "const double a_over_p = (-alpha) * P_inv;")
    w(ind + "const double a_over_q = alpha * Q_inv;")
    w(ind + "double2 *const c = (double2 *)(pc + lane * NPC);")
    bra = [("PA%d" % d, "a_over_p * PQ%s" % "xyz"[d]) for d in range(3)] + [("a_over_p", "0.5 * P_inv")]
    ket = [("QC%d" % d, "a_over_q * PQ%s" % "xyz"[d]) for d in range(3)] + [("-a_over_q", "0.5 * Q_inv")]
    E, S = (bra, ket) if p.s_is_ket else (ket, bra)

    def put(at, a, b):
        w(ind + "c[%d] = make_double2(%s, %s);" % (at // 2, a, b))
    for d in range(3):
        put(P_E + 2 * d, *E[d])
        put(P_S + 2 * d, *S[d])
    put(P_ID, "1.0", "0.0")
    put(P_EOVER, *E[3])
    put(P_SOVER, *S[3])
    put(P_O2PQ, "0.5 * one_over_PQalpha_sum", "0.0")
    for m in range(0, p.L + 1, 2):
        put(P_F + m, "F[%d] * prefac" % m, "F[%d] * prefac" % (m + 1) if m < p.L else "0.0")
    w("            }")
    # the quartet's block for the HRR: with the last batch
    w("            if (mine && lane == r * PBK && p0 + PBK >= p_end) {")
    w(ind + "double *const h = %s + r * QINFO;" % ("qmine" if p.SW > 1 else "qi"))
    b, k = ("wi.bra", "(long long)wi.tile * SIMINT_TILE + q") if not listmode else ("bp", "kp")
    for c in range(3):
        w(ind + "h[%d] = A.bra.ab%s[%s];" % (c, "xyz"[c], b))
        w(ind + "h[%d] = A.ket.ab%s[%s];" % (3 + c, "xyz"[c], k))
    if listmode:
        w(ind + "((long long *)h)[6] = A.qout ? A.qout[q] : q * A.ostride;")
    else:
        w(ind + "((long long *)h)[6] = wi.obase + A.ket.col[(long long)wi.tile * SIMINT_TILE + q] * A.stride;")
    w("            }")
    if p.G > 1:
        w("            if (screen && tid == 0) ((unsigned *)qi)[14] = alive;   // read by the others behind the barrier")


def _emit_vrr(p, w, part):
    ind = "                    "
    L, NS = p.L, p.NS
    shared = p.NQ == 1        # one quartet: its constants serve every slot
    path0 = {}
    mine = p.chain_slots(part) if p.G > 1 else list(range(NS))
    if p.G > 1:
        w(ind + "double *const root = roots + turn * %d;" % ((p.s_hi + 1) * p.ps))
        w(ind + "turn ^= 1;")
    for s in range(NS):
        q = 0 if shared else s
        if s == q:
            w(ind + "const double *const c%d = pc + ((gi * NQ + w%d) * PBK + pp) * NPC;" % (s, s))
            w(ind + "const double2 eo%d = *(const double2 *)(c%d + %d), so%d = *(const double2 *)(c%d + %d);"
              % (s, s, P_EOVER, s, s, P_SOVER))
            w(ind + "const double o2pq%d = c%d[%d];" % (s, s, P_O2PQ))
            for m in range(L + 1) if mine and (shared or s in mine) else ():
                w(ind + "const double f%d_%d = c%d[%d];" % (s, m, s, P_F + m))
        # the lane's chain up the wide side
        if s not in mine:
            continue
        prev, cur = None, ["f%d_%d" % (q, m) for m in range(L + 1)]
        for k in range(1, p.e_hi + 1):
            w(ind + "const double2 ap%d_%d = *(const double2 *)(c%d + ((tab%d.x >> %d) & 3u) * 2);"
              % (s, k, q, s, 2 * (k - 1)))
            if k > 1:
                w(ind + "const double n%d_%d = (double)((tab%d.y >> %d) & 15u) * eo%d.y;" % (s, k, s, 4 * (k - 1), q))
            new = []
            for m in range(L - k + 1):
                v = "h%d_%d_%d" % (s, k, m)
                x = "fma(ap%d_%d.y, %s, ap%d_%d.x * %s)" % (s, k, cur[m + 1], s, k, cur[m])
                if k > 1:
                    x = "fma(n%d_%d, fma(eo%d.x, %s, %s), %s)" % (s, k, q, prev[m + 1], prev[m], x)
                w(ind + "const double %s = %s;" % (v, x))
                new.append(v)
            prev, cur = cur, new
        path0[s] = cur
        if p.G > 1:
            for m in range(p.s_hi + 1):
                w(ind + "root[%d + idx%d] = %s;" % (m * p.ps, s, cur[m]))
    if p.G > 1:
        # the other wavefronts write the other buffer only after the next one
        w(ind + "__syncthreads();")
    for s in range(NS):
        q = 0 if shared else s
        if p.G > 1 and p.parts[part]:
            path0[s] = []
            for m in range(p.s_hi + 1):
                w(ind + "const double r%d_%d = root[%d + idx%d];" % (s, m, m * p.ps, s))
                path0[s].append("r%d_%d" % (s, m))
        # (through an empty asm: hoisted out of the loop the exponents would
        # hold six registers a slot)
        w(ind + "unsigned z%d = tab%d.z;" % (s, s))
        w(ind + 'asm volatile("" : "+v"(z%d));' % s)
        for d in range(3):
            w(ind + "const double ox%d_%d = (double)((z%d >> %d) & 15u) * o2pq%d;" % (s, d, s, 4 * d, q))
    for s in range(NS):
        q = 0 if shared else s
        if s == q:
            for d in range(3):
                w(ind + "const double2 sp%d_%d = *(const double2 *)(c%d + %d);" % (s, d, s, P_S + 2 * d))
    # integer multiples of the narrow side's 1/2p
    most = max([0] + [f[mk_dir(f)] - 1 for f in p.part_nodes[part] if sum(f)])
    for s in range(NS):
        q = 0 if shared else s
        if s == q:
            for n in range(2, most + 1):
                w(ind + "const double sn%d_%d = %d.0 * so%d.y;" % (s, n, n, s))

    top = {f: t for t, f in enumerate(p.parts[part])}

    def accumulate(f, vec):
        if f in top:
            for s in range(NS):
                w(ind + "acc%d_%d += %s;" % (s, top[f], vec[s][0]))

    count = [0]

    def visit(f, vec, up):
        """f's vectors `vec` per slot; `up`: vectors of f's ancestors by component."""
        kids = [c for c in p.children[f] if c in p.part_nodes[part]]
        if not kids:
            return
        l = sum(f)
        if l or p.G == 1:
            for s in range(NS):
                for m in range(1, p.s_hi - l + 1):
                    w(ind + "pub[%d + idx%d] = %s;" % ((p.pub_level[l] + m - 1) * p.ps, s, vec[s][m]))
            w(ind + "wave_fence();")
        up = dict(up)
        up[f] = vec
        for c in kids:
            d = mk_dir(c)
            gp = up.get(step(f, d, -1)) if f[d] > 0 else None
            cv = {}
            for s in range(NS):
                q = 0 if shared else s
                cv[s] = []
                for m in range(p.s_hi - l):
                    v = "v%d" % count[0]
                    count[0] += 1
                    x = "fma(sp%d_%d.y, %s, sp%d_%d.x * %s)" % (q, d, vec[s][m + 1], q, d, vec[s][m])
                    if gp is not None:
                        n = c[d] - 1
                        cn = "so%d.y" % q if n == 1 else "sn%d_%d" % (q, n)
                        x = "fma(%s, fma(so%d.x, %s, %s), %s)" % (cn, q, gp[s][m + 1], gp[s][m], x)
                    at = "pub[%d" % ((p.pub_level[l] + m) * p.ps) if l or p.G == 1 else "root[%d" % ((m + 1) * p.ps)
                    x = "fma(ox%d_%d, %s + nb%d_%d], %s)" % (s, d, at, s, d, x)
                    w(ind + "const double %s = %s;" % (v, x))
                    cv[s].append(v)
            accumulate(c, cv)
            visit(c, cv, up)

    if not p.parts[part]:
        return
    origin = (0, 0, 0)
    accumulate(origin, path0)
    visit(origin, path0, {})
    # the next primitive quartet's publications must not overtake these reads
    w(ind + "wave_fence();")


def _emit_sum(p, w):
    """Add the wavefronts' accumulators to the first one's, SUM_VALUES at a
    time through the work area."""
    ind = "                "
    vals = ["acc%d_%d" % (s, t) for s in range(p.NS) for t in range(p.nacc)]
    for v0 in range(0, len(vals), SUM_VALUES):
        part = vals[v0:v0 + SUM_VALUES]
        w(ind + "__syncthreads();")
        w(ind + "if (wave != 0) {")
        w(ind + "    double *const x = area + (wave - 1) * %d + lane;" % (SUM_VALUES * 64))
        for k, v in enumerate(part):
            w(ind + "    x[%d] = %s;" % (64 * k, v))
        w(ind + "}")
        w(ind + "__syncthreads();")
        w(ind + "if (wave == 0) {")
        w("#pragma unroll 1")
        w(ind + "    for (int v = 0; v < %d; ++v) {" % (p.SW - 1))
        w(ind + "        const double *const x = area + v * %d + lane;" % (SUM_VALUES * 64))
        for k, v in enumerate(part):
            w(ind + "        %s += x[%d];" % (v, 64 * k))
        w(ind + "    }")
        w(ind + "}")


def _emit_hrr(p, w, sync):
    g = p.g
    ind = "                "
    bra_ops, bra_map, ket_ops, ket_map = g.hrr_program()
    la, lb, lc, ld = p.am
    bra_final = [(a, b) for a in carts(la) for b in carts(lb)]
    ket_final = [(c, d) for c in carts(lc) for d in carts(ld)]
    btop = {e: i for i, e in enumerate(g.bra_tops())}
    ktop = {f: i for i, f in enumerate(g.ket_tops())}
    NQ, HQ, lanes = p.NQ, p.HQ, 64 * p.W
    ks = max(p.nkt, p.ncd) | 1                       # row stride of results
    ts = (p.nkt | 1) if p.hold else ks               # row stride of tops
    trows = p.nbt if p.hold else max(p.nbt, p.nab)

    def transfers(ops, final, fmap, top, h):
        """Straight-line transfers of one column or row: the values of its
        final components."""
        names = {}

        def val(src):
            return "t%d" % top[src[1]] if src[0] == "top" else names[src[1], src[2]]
        for n, (dst, s0, s1, sign, d) in enumerate(ops):
            names[dst[1], dst[2]] = "x%d" % n
            w(ind + "        const double x%d = fma(%s%s[%d], %s, %s);" % (n, "" if sign > 0 else "-", h, d, val(s1), val(s0)))
        return [val(fmap[k]) for k in final]

    w("#pragma unroll 1")
    w(ind + "for (int h0 = 0; h0 < NQ; h0 += %d) {" % HQ)
    # tops to the area: row = bra top, column = ket top
    w(ind + "    " + sync)
    for part, tops in enumerate(p.parts):
        if not tops:
            continue
        if p.W > 1:
            w(ind + "    if (wave == %d) {" % part)
        for s in range(p.NS):
            w(ind + "    if (use%d && w%d >= h0 && w%d < h0 + %d && e%d >= %d) {" % (s, s, s, HQ, s, p.first_top))
            if p.s_is_ket:
                w(ind + "        double *const x = area + ((w%d - h0) * %d + e%d - %d) * %d;"
                  % (s, trows, s, p.first_top, ts))
            else:
                w(ind + "        double *const x = area + (w%d - h0) * %d + e%d - %d;"
                  % (s, trows * ts, s, p.first_top))
            for k, f in enumerate(tops):
                at = ktop[f] if p.s_is_ket else btop[f] * ts
                w(ind + "        x[%d] = acc%d_%d;" % (at, s, k))
            w(ind + "    }")
        if p.W > 1:
            w(ind + "    }")
    w(ind + "    " + sync)
    # bra transfers: one lane per (quartet, ket top)
    if p.hold:
        w(ind + "    const int bc = tid < %d ? tid : 0;" % (HQ * p.nkt))
        w(ind + "    const int bw = bc / %d, bk = bc - bw * %d;" % (p.nkt, p.nkt))
        w(ind + "    double " + ", ".join("y%d" % k for k in range(p.nab)) + ";")
        w(ind + "    {")
        w(ind + "        const double *const x = area + bw * %d + bk;" % (trows * ts))
        if bra_ops:
            w(ind + "        const double *const h = qi + (gi * NQ + h0 + bw) * QINFO;")
            w(ind + "        const double hv[3] = {h[0], h[1], h[2]};")
        for k in range(p.nbt):
            w(ind + "        const double t%d = x[%d];" % (k, k * ts))
        for k, v in enumerate(transfers(bra_ops, bra_final, bra_map, btop, "hv")):
            w(ind + "        y%d = %s;" % (k, v))
        w(ind + "    }")
    elif bra_ops:
        w("#pragma unroll 1")
        w(ind + "    for (int t = tid; t < %d; t += %d) {" % (HQ * p.nkt, lanes))
        w(ind + "        const int bw = t / %d, bk = t - bw * %d;" % (p.nkt, p.nkt))
        w(ind + "        double *const x = area + bw * %d + bk;" % (trows * ts))
        w(ind + "        const double *const h = qi + (gi * NQ + h0 + bw) * QINFO;")
        w(ind + "        const double hv[3] = {h[0], h[1], h[2]};")
        for k in range(p.nbt):
            w(ind + "        const double t%d = x[%d];" % (k, k * ts))
        for k, v in enumerate(transfers(bra_ops, bra_final, bra_map, btop, "hv")):
            w(ind + "        x[%d] = %s;" % (k * ts, v))
        w(ind + "    }")
    rows = [list(range(c, min(p.nab, c + p.cc))) for c in range(0, p.nab, p.cc)]
    for part in rows:
        nr = len(part)
        prow = p.cc if p.hold else trows                # rows per quartet in the area
        if p.hold:
            w(ind + "    " + sync)
            w(ind + "    if (tid < %d) {" % (HQ * p.nkt))
            w(ind + "        double *const x = area + bw * %d + bk;" % (prow * ks))
            for j, k in enumerate(part):
                w(ind + "        x[%d] = y%d;" % (j * ks, k))
            w(ind + "    }")
        w(ind + "    " + sync)
        if ket_ops:
            w("#pragma unroll 1")
            w(ind + "    for (int t = tid; t < %d; t += %d) {" % (HQ * nr, lanes))
            w(ind + "        const int kw = t / %d;" % nr)
            w(ind + "        double *const x = area + (kw * %d + t) * %d;" % (prow - nr, ks))
            w(ind + "        const double *const h = qi + (gi * NQ + h0 + kw) * QINFO;")
            w(ind + "        const double hv[3] = {h[3], h[4], h[5]};")
            for k in range(p.nkt):
                w(ind + "        const double t%d = x[%d];" % (k, k))
            for k, v in enumerate(transfers(ket_ops, ket_final, ket_map, ktop, "hv")):
                w(ind + "        x[%d] = %s;" % (k, v))
            w(ind + "    }")
            w(ind + "    " + sync)
        # the rows' values are contiguous in the output
        n = nr * p.ncd
        w(ind + "    for (int t = tid; t < %d; t += %d) {" % (HQ * n, lanes))
        w(ind + "        const int ow = t / %d, o = t - ow * %d;" % (n, n))
        w(ind + "        const int r = o / %d;" % p.ncd)
        w(ind + "        if (q_first + (g0 + gi) * NQ + h0 + ow < q_end)")
        w(ind + "            A.out[((const long long *)(qi + (gi * NQ + h0 + ow) * QINFO))[6] + %d + o] ="
          % (part[0] * p.ncd))
        w(ind + "                area[(ow * %d + r) * %d + o - r * %d];" % (prow, ks, p.ncd))
        w(ind + "    }")
    w(ind + "}")
    for s in range(p.NS):
        w(ind + " ".join("acc%d_%d = 0.0;" % (s, t) for t in range(p.nacc)))
    w(ind + sync)
