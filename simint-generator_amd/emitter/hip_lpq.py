"""HIP writer: lane-per-quartet (LPQ) kernels for one (ab|cd) class.

Mapping.  One wavefront (64 lanes) takes one work item: a bra shell pair,
uniform across the wave, against the 64 ket shell pairs of a ket tile, one
per lane.  Bra primitive data are wave-uniform scalar loads; ket primitive j
of every lane is one contiguous 512-byte run per field (tiled layout, see
csrc/device_types.h).  Each lane loops over bra x ket primitive pairs,
evaluates the Boys function, the Obara-Saika VRR as straight-line FP64 code
held in registers, and accumulates the contracted HRR inputs in registers;
then it runs the bra and ket HRR in registers and writes its ncart(abcd)
integrals in Psi4 order.

The arithmetic of every step is the reference's (setup:
generator/ostei/OSTEI_Writer.cpp:595-702; VRR: OSTEI_VRR_Writer.cpp:95-125;
HRR: OSTEI_HRR_Writer.cpp:22-99); only the (component, m) values that feed
the result are emitted.
"""
from .rrgraph import graph, carts, cart_index, ncart, I, J, K, L

AMCHAR = "spdfghik"


def class_name(am):
    return "_".join(AMCHAR[x] for x in am)


def _fmt_int(k):
    return "%d.0" % k


class _Writer:
    def __init__(self):
        self.lines = []

    def __call__(self, s=""):
        self.lines.append(s)

    def text(self):
        return "\n".join(self.lines) + "\n"


def emit_base(am, w, indent):
    """The primitive quartet's base values, into variables declared by the
    caller: Fp[m] = F_m(x) times the prefactor (m = 0..L), one_over_PQalpha_sum,
    alpha, PQx/PQy/PQz -- the same arithmetic emit_body uses."""
    Ltot = graph(*am).Ltot
    w(indent + "{")
    w(indent + "    const double PQalpha_mul = P_alpha * Q_alpha;")
    w(indent + "    const double PQalpha_sum = P_alpha + Q_alpha;")
    w(indent + "    one_over_PQalpha_sum = 1.0 / PQalpha_sum;")
    w(indent + "    PQx = P_x - Q_x;")
    w(indent + "    PQy = P_y - Q_y;")
    w(indent + "    PQz = P_z - Q_z;")
    w(indent + "    double R2 = PQx * PQx;")
    w(indent + "    R2 = fma(PQy, PQy, R2);")
    w(indent + "    R2 = fma(PQz, PQz, R2);")
    w(indent + "    alpha = PQalpha_mul * one_over_PQalpha_sum;")
    w(indent + "    const double F_x = R2 * alpha;")
    w(indent + "    double F[%d];" % (Ltot + 1))
    w(indent + "    boys_eval<%d>(grid, F_x, F);" % Ltot)
    w(indent + "    const double prefac = (P_prefac * Q_prefac) * sqrt(one_over_PQalpha_sum);")
    for m in range(Ltot + 1):
        w(indent + "    Fp[%d] = F[%d] * prefac;" % (m, m))
    w(indent + "}")


def emit_body(am, w, indent="        ", fp="double", keep=None, acc_tops=None, base="compute"):
    """Emit the per-primitive-quartet code (setup, Boys, VRR, accumulation).

    Assumes in scope: P_alpha, P_inv, P_prefac, P_x/y/z, P_PA or P_PB (x,y,z),
    Q_* likewise, grid, and accumulators acc<k> (double).  fp = "float":
    the Gaussian-product setup, the Boys function and the prefactor stay
    FP64; the VRR runs in FP32 on rounded copies of its inputs, and each
    result is accumulated into the FP64 accumulators.  base = "given": the
    values emit_base computes are already in scope (Fp[m], alpha,
    one_over_PQalpha_sum, PQx/PQy/PQz), so only the factors derived from
    them and the VRR are emitted."""
    given = base == "given"
    mixed = fp == "float"
    fm = "fmaf" if mixed else "fma"
    g = graph(*am)
    Ltot = g.Ltot
    # keep: the VRR nodes to emit (a closure of acc_tops); acc_tops: list of
    # (accumulator name, top key) -- by default every node and every top
    nodes = g.node_list if keep is None else [n for n in g.node_list if (n.q, n.m) in keep]
    if acc_tops is None:
        acc_tops = [("acc%d" % t, key) for t, key in enumerate(g.top_keys)]
    # The Boys values come from one evaluation at the class's total AM even
    # when a group of tops needs fewer orders, as in the reference (one
    # boys_F_split per primitive quartet): for x >= 36.5 the lower orders
    # then carry the same error pattern in every group, which the HRR
    # transfers between tops of different groups cancel -- with per-group
    # orders they did not, and (df|dd) lost 1e-7 normwise.
    used_steps = set(n.step for n in nodes if n.step is not None)
    # classes without HRR take 1/(p+q) and its square root from one refined
    # reciprocal square root (a few ulp): no HRR transfer amplifies it.  Only
    # in the lane-per-quartet kernels (their file carries the helpers); the
    # setup is FP64 in the mixed kernels too.
    fast = keep is None and not g.bra_hrr_needed() and not g.ket_hrr_needed() and not given
    if not given:
        _emit_setup(w, indent, Ltot, fast)
    _emit_vrr(g, nodes, acc_tops, w, indent, fp, mixed, fm, given, used_steps)


def _emit_setup(w, indent, Ltot, fast):
    w(indent + "const double PQalpha_mul = P_alpha * Q_alpha;")
    w(indent + "const double PQalpha_sum = P_alpha + Q_alpha;")
    if fast:
        w(indent + "const double rs_PQalpha_sum = rsqrt_nr(PQalpha_sum);")
        w(indent + "const double one_over_PQalpha_sum = rs_PQalpha_sum * rs_PQalpha_sum;")
    else:
        w(indent + "const double one_over_PQalpha_sum = 1.0 / PQalpha_sum;")
    w(indent + "const double PQx = P_x - Q_x;")
    w(indent + "const double PQy = P_y - Q_y;")
    w(indent + "const double PQz = P_z - Q_z;")
    w(indent + "double R2 = PQx * PQx;")
    w(indent + "R2 = fma(PQy, PQy, R2);")
    w(indent + "R2 = fma(PQz, PQz, R2);")
    w(indent + "const double alpha = PQalpha_mul * one_over_PQalpha_sum;")
    w(indent + "const double F_x = R2 * alpha;")
    w(indent + "double F[%d];" % (Ltot + 1))
    if fast:
        w(indent + "boys_eval_rs<%d>(grid, F_x, F);" % Ltot)
        w(indent + "const double prefac = (P_prefac * Q_prefac) * rs_PQalpha_sum;")
    else:
        w(indent + "boys_eval<%d>(grid, F_x, F);" % Ltot)
        w(indent + "const double prefac = (P_prefac * Q_prefac) * sqrt(one_over_PQalpha_sum);")


def _emit_vrr(g, nodes, acc_tops, w, indent, fp, mixed, fm, given, used_steps):
    has_bra = bool(used_steps & {I, J})
    has_ket = bool(used_steps & {K, L})
    # integer constants k/(2p), k/(2q), k/(2pq)
    need = {"2p": set(), "2q": set(), "2pq": set()}
    for n in nodes:
        if n.step is None:
            continue
        bra = n.step in (I, J)
        if n.src[2] is not None:
            need["2p" if bra else "2q"].add(n.fac[0])
        if n.src[4] is not None:
            need["2p" if bra else "2q"].add(n.fac[1])
        if n.src[6] is not None:
            need["2pq"].add(n.fac[2])
        if n.src[7] is not None:
            need["2pq"].add(n.fac[3])
    cv = (lambda e: "(float)(%s)" % e) if mixed else (lambda e: e)
    if need["2p"]:
        w(indent + "const %s one_over_2p = %s;" % (fp, cv("0.5 * P_inv")))
    if need["2q"]:
        w(indent + "const %s one_over_2q = %s;" % (fp, cv("0.5 * Q_inv")))
    if need["2pq"]:
        w(indent + "const %s one_over_2pq = %s;" % (fp, cv("0.5 * one_over_PQalpha_sum")))
    for kind in ("2p", "2q", "2pq"):
        for k in sorted(need[kind]):
            if k > 1:
                w(indent + "const %s c%d_%s = %s%s * one_over_%s;" % (fp, k, kind, _fmt_int(k), "f" if mixed else "",
                                                                     kind))
    if has_bra:
        w(indent + "const double a_over_p_d = (-alpha) * P_inv;")
        w(indent + "const %s a_over_p = %s;" % (fp, cv("a_over_p_d")))
        w(indent + "const %s aop_PQ[3] = {%s, %s, %s};" % (fp, cv("a_over_p_d * PQx"), cv("a_over_p_d * PQy"),
                                                           cv("a_over_p_d * PQz")))
    if has_ket:
        w(indent + "const double a_over_q_pos = alpha * Q_inv;")
        w(indent + "const %s aoq_PQ[3] = {%s, %s, %s};" % (fp, cv("a_over_q_pos * PQx"), cv("a_over_q_pos * PQy"),
                                                           cv("a_over_q_pos * PQz")))
        w(indent + "const %s a_over_q = %s;" % (fp, cv("-a_over_q_pos")))
    if mixed:
        # FP32 copies of the pair geometry the VRR steps use
        for side, dirs in (("P", (I, J)), ("Q", (K, L))):
            for arr in ("PA", "PB"):
                if any(n.step in dirs and ((arr == "PA") == (n.step in (I, K))) for n in nodes if n.step is not None):
                    w(indent + "const float f%s_%s[3] = {(float)%s_%s[0], (float)%s_%s[1], (float)%s_%s[2]};"
                      % (side, arr, side, arr, side, arr, side, arr))

    def cname(k, kind):
        return ("one_over_%s" % kind) if k == 1 else ("c%d_%s" % (k, kind))

    # each top is added to its accumulator right after it is computed, so
    # the value is dead unless a later node reads it (the node list is a
    # depth-first post-order over the tops)
    acc_of = {}
    for accname, key in acc_tops:
        acc_of.setdefault(key, []).append(accname)

    def accumulate(key, v):
        for accname in acc_of.get(key, ()):
            w(indent + "%s += %s;" % (accname, ("(double)%s" % v) if mixed else v))

    idx = {}
    for n in nodes:
        key = (n.q, n.m)
        v = "v%d" % len(idx)
        idx[key] = v
        if n.step is None:
            w(indent + "const %s %s = %s;" % (fp, v, cv(("Fp[%d]" if given else "F[%d] * prefac") % n.m)))
            accumulate(key, v)
            continue
        d = n.dir
        bra = n.step in (I, J)
        pfx = "f" if mixed else ""
        if n.step == I:
            pa = "%sP_PA[%d]" % (pfx, d)
        elif n.step == J:
            pa = "%sP_PB[%d]" % (pfx, d)
        elif n.step == K:
            pa = "%sQ_PA[%d]" % (pfx, d)
        else:
            pa = "%sQ_PB[%d]" % (pfx, d)
        aop = ("aop_PQ[%d]" if bra else "aoq_PQ[%d]") % d
        aover = "a_over_p" if bra else "a_over_q"
        k2 = "2p" if bra else "2q"
        s = [idx[x] if x is not None else None for x in n.src]
        expr = "%s * %s" % (pa, s[0])
        expr = "%s(%s, %s, %s)" % (fm, aop, s[1], expr)
        if s[2] is not None:
            expr = "%s(%s, %s(%s, %s, %s), %s)" % (fm, cname(n.fac[0], k2), fm, aover, s[3], s[2], expr)
        if s[4] is not None:
            expr = "%s(%s, %s(%s, %s, %s), %s)" % (fm, cname(n.fac[1], k2), fm, aover, s[5], s[4], expr)
        if s[6] is not None:
            expr = "%s(%s, %s, %s)" % (fm, cname(n.fac[2], "2pq"), s[6], expr)
        if s[7] is not None:
            expr = "%s(%s, %s, %s)" % (fm, cname(n.fac[3], "2pq"), s[7], expr)
        w(indent + "const %s %s = %s;" % (fp, v, expr))
        accumulate(key, v)


STAGE = 16   # output components per LDS slice (coalesced stores)


def _emit_flush(w, indent, k0, sl):
    """Write components [k0, k0 + sl) of the wave's quartets from the LDS
    slice: consecutive threads store consecutive doubles of one quartet's
    block, so every store instruction writes sl-double runs instead of 64
    scattered doubles."""
    w(indent + "__syncthreads();")
    w(indent + "for (int e = lane; e < %d; e += 64) {" % (64 * sl))
    w(indent + "    const int q = e / %d, j = e - q * %d;" % (sl, sl))
    w(indent + "    if (q >= wi.lane_lo && q < wi.lane_hi) A.out[ob[q] + %d + j] = xb[q * %d + j];" % (k0, STAGE + 1))
    w(indent + "}")
    w(indent + "__syncthreads();")


def emit_hrr(am, w, indent="    ", out="o", acc="acc", fp="double", staged=False):
    """Emit the bra then ket HRR on acc<k>, storing into out[k] (Psi4 order).
    fp = "float": the HRR runs in FP32 on rounded copies of the FP64
    contracted values and AB/CD; results are widened to FP64 on store.
    staged: results go through the LDS slices xb / ob (see _emit_flush)
    instead of straight to out[k]; every lane of the wave must run it."""
    mixed = fp == "float"
    fm = "fmaf" if mixed else "fma"
    g = graph(*am)
    la, lb, lc, ld = am
    bra_ops, bra_map, ket_ops, ket_map = g.hrr_program()
    ket_tops = g.ket_tops()
    bra_tops = g.bra_tops()
    nf = len(ket_tops)
    etop = {e: i for i, e in enumerate(bra_tops)}
    ftop = {f: i for i, f in enumerate(ket_tops)}

    if mixed:
        for t in range(len(g.tops)):
            w(indent + "const float f%s%d = (float)%s%d;" % (acc, t, acc, t))
        if g.bra_hrr_needed():
            w(indent + "const float fhAB[3] = {(float)hAB[0], (float)hAB[1], (float)hAB[2]};")
        if g.ket_hrr_needed():
            w(indent + "const float fhCD[3] = {(float)hCD[0], (float)hCD[1], (float)hCD[2]};")
    pre = "f" if mixed else ""

    def topvar(e, f):
        return "%s%s%d" % (pre, acc, etop[e] * nf + ftop[f])

    # bra HRR for every top ket component f -> names hb_<f>_<a>_<b>
    names = {}
    cnt = [0]

    def newname(prefix):
        cnt[0] += 1
        return "%s%d" % (prefix, cnt[0])

    def bra_val(src, f):
        if src[0] == "top":
            return topvar(src[1], f)
        return names[("b", f, src[1], src[2])]

    for f in ket_tops:
        for (dst, s0, s1, sign, d) in bra_ops:
            nm = newname("hb")
            names[("b", f, dst[1], dst[2])] = nm
            ab = ("%shAB[%d]" % (pre, d)) if sign > 0 else ("(-%shAB[%d])" % (pre, d))
            w(indent + "const %s %s = %s(%s, %s, %s);" % (fp, nm, fm, ab, bra_val(s1, f), bra_val(s0, f)))

    # ket HRR for every final bra component
    nb, nc, nd = ncart(lb), ncart(lc), ncart(ld)
    ntot = ncart(la) * nb * nc * nd
    for ia, a in enumerate(carts(la)):
        for ib, b in enumerate(carts(lb)):
            bm = bra_map[(a, b)]

            def abf(fc):
                return bra_val(bm, fc)

            def ket_val(src):
                if src[0] == "top":
                    return abf(src[1])
                return names[("k", a, b, src[1], src[2])]

            for (dst, s0, s1, sign, d) in ket_ops:
                nm = newname("hk")
                names[("k", a, b, dst[1], dst[2])] = nm
                cd = ("%shCD[%d]" % (pre, d)) if sign > 0 else ("(-%shCD[%d])" % (pre, d))
                w(indent + "const %s %s = %s(%s, %s, %s);" % (fp, nm, fm, cd, ket_val(s1), ket_val(s0)))
            for ic, c in enumerate(carts(lc)):
                for idd, dd in enumerate(carts(ld)):
                    k = ((ia * nb + ib) * nc + ic) * nd + idd
                    val = ket_val(ket_map[(c, dd)])
                    if mixed:
                        val = "(double)" + val
                    if staged:
                        w(indent + "xb[lane * %d + %d] = %s;" % (STAGE + 1, k % STAGE, val))
                        if (k + 1) % STAGE == 0 or k + 1 == ntot:
                            _emit_flush(w, indent, k - k % STAGE, k % STAGE + 1)
                    else:
                        w(indent + "%s[%d] = %s;" % (out, k, val))


def _emit_fast_setup(w, Ltot):
    """Helpers of the classes without HRR (emit_body's fast setup): x^-1/2
    from the hardware reciprocal square root refined by two Newton steps
    y <- y + y (1/2 - (x/2) y^2) (within a few ulp of the correctly rounded
    value; IEEE 1/x and sqrt are each about three times the instructions),
    and the Boys function with its long-range branch for L < 4 (all orders
    from longfac[m] x^-(m+1/2), boys.h:18-25) on that square root (L >= 4
    keeps boys_eval's branch)."""
    w("namespace {")
    w("__device__ __forceinline__ double rsqrt_nr(double x)")
    w("{")
    w("    double y = __builtin_amdgcn_rsq(x);")
    w("    const double h = 0.5 * x;")
    w("    double t = fma(-h * y, y, 0.5);")
    w("    y = fma(y, t, y);")
    w("    t = fma(-h * y, y, 0.5);")
    w("    return fma(y, t, y);")
    w("}")
    w("")
    w("template <int L>")
    w("__device__ __forceinline__ void boys_eval_rs(const double *__restrict__ grid, double x, double *F)")
    w("{")
    w("    if (L >= 4 || x < SIMINT_BOYS_MAXX) {")
    w("        boys_eval<L>(grid, x, F);")
    w("        return;")
    w("    }")
    w("    constexpr double longfac[] = SIMINT_BOYS_LONGFAC;")
    w("    double x2 = rsqrt_nr(x);")
    w("    const double x1 = x2 * x2;")
    w("#pragma unroll")
    w("    for (int n = 0; n <= L; n++) {")
    w("        F[n] = longfac[n] * x2;")
    w("        x2 *= x1;")
    w("    }")
    w("}")
    w("}  // namespace")
    w("")


def emit_lpq(am, mixed=False, lane_items=None):
    """Source of one class: the prefix kernel, the quartet-list kernel and,
    with mixed=True, the FP32-VRR prefix kernel (eri_lpqm_<class>)."""
    w = _Writer()
    w("// Generated by simint-generator_amd/emitter/hip_lpq.py -- class (%s)" % class_name(am).replace("_", ""))
    w('#include "../device_types.h"')
    w('#include "../boys_device.h"')
    w("")
    g = graph(*am)
    if not g.bra_hrr_needed() and not g.ket_hrr_needed():
        _emit_fast_setup(w, g.Ltot)
    _emit_lpq_prefix(am, w, "double")
    emit_lpq_list(am, w)
    if mixed:
        w("")
        _emit_lpq_prefix(am, w, "float")
    for fp in (("double", "float") if mixed else ("double",)):
        if share_kind(am) in ("sum", "turn"):
            _emit_lpq_prefix(am, w, fp, shared=share_kind(am))
        _emit_lpq_launcher(am, w, fp, lane_items)
    return w.text()


# Small launches: several wavefronts share an item's primitive quartets, eight
# at most and about as many as it has.  A 12-atom molecule's (ss|ss) launches are a
# few dozen items of up to 1296 primitive quartets: 82 us each with one
# wavefront an item, 24 us so.
# Classes without HRR add the wavefronts' sums at the end, while the launch has
# fewer than SHARE_ITEMS wavefronts (the chip holds 4096); of more than
# SHARE_TOPS sums up to SHARE_ITEMS / 2, one for every SIMD, which such a
# kernel's registers fill (1024 items of (fs|fs) take 369 us with one wavefront
# each, 405 with two and 500 with four, 256 of them 343, 204 and 133).  An HRR
# amplifies the rounding of another order of the sum, so the others keep it:
#  * (ab|ss) and (ss|cd): the wavefronts take the primitive quartets in turn,
#    leave the contracted terms in the local data share, and every contracted
#    value is added up by one of them in the order one wavefront alone adds it,
#    where all items' terms fit the compute units' local data shares at once:
#    256 items of 81 primitive quartets of (dd|ss) take 134 us with one
#    wavefront and 84 with four, 1024 of them 140 and 317; two wavefronts are
#    slower than one always;
#  * the rest run the component-lane kernel, which spreads a quartet over lanes
#    instead and gives the same values, up to a number of items by class and
#    depth (LANE_DEPTHS) that tuning.json's "lane_items" holds (autotune.py
#    --lanes: the most at which it is not slower): over the 60 classes it takes
#    0.58, 0.70 and 0.86 of the time with 32, 64 and 128 items of 16 primitive
#    quartets, 0.76, 0.85 and 0.98 with 4, but 1.12, 1.21 and 1.33 with 1; 128
#    items of 16 0.42 of it for (dd|ds) and 1.19 for (ps|pp).  Classes it does
#    not name: LANE_ITEMS_PER_DEPTH for each primitive quartet, up to LANE_ITEMS.
SHARE_ITEMS = 2048
SHARE_TOPS = 36
LANE_ITEMS = 128
LANE_ITEMS_PER_DEPTH = 8
LANE_DEPTHS = (4, 9, 16)    # "lane_items": below 4 primitive quartets, 9, 16, and from there on
SHARE_SUM = 8       # contracted values added per round at the end (classes without HRR)


def share_kind(am):
    """"sum", "turn" or "lanes" (see above); None: one wavefront an item
    whatever the launch."""
    from . import hip_cpl
    g = graph(*am)
    if not g.bra_hrr_needed() and not g.ket_hrr_needed():
        return "sum" if len(g.top_keys) <= 128 else None
    if min(g.e_hi, g.f_hi) == 0:
        return "turn" if len(g.top_keys) <= 32 else None
    return "lanes" if hip_cpl.candidate(am) else None


def share_waves(am):
    """Most wavefronts that share an item: "turn" keeps two buffers of their
    terms, at most 128 KB of the local data share; "sum" leaves 256
    registers a lane with eight, 512 with four."""
    ntop = len(graph(*am).top_keys)
    if share_kind(am) == "sum":
        return 8 if ntop <= 36 else 4
    return 8 if ntop <= 16 else 4 if ntop <= 32 else 2


def _emit_lpq_launcher(am, w, fp, lane_items=None):
    kname = ("lpqm_%s" if fp == "float" else "lpq_%s") % class_name(am)
    kind, most = share_kind(am), share_waves(am)
    if kind == "lanes" and fp == "double":
        w('extern "C" hipError_t simint_launch_cpl_%s(const EriArgs *a, hipStream_t s);' % class_name(am))
    w('extern "C" hipError_t simint_launch_%s(const EriArgs *a, hipStream_t s)' % kname)
    w("{")
    w("    if (a->nitems <= 0) return hipSuccess;")
    if kind:
        w("    const long long depth = a->depth > 0 ? a->depth : 4096;   // unknown: as deep ones")
    if kind == "lanes":
        if lane_items:
            test = "depth < %d ? %d : depth < %d ? %d : depth < %d ? %d : %d" % (
                LANE_DEPTHS[0], lane_items[0], LANE_DEPTHS[1], lane_items[1], LANE_DEPTHS[2], lane_items[2],
                lane_items[3])
        else:
            test = "%d * depth < %d ? %d * depth : %d" % (LANE_ITEMS_PER_DEPTH, LANE_ITEMS, LANE_ITEMS_PER_DEPTH,
                                                          LANE_ITEMS)
        w("    if (a->nitems <= (%s)) return simint_launch_cpl_%s(a, s);" % (test, class_name(am)))
    elif kind == "sum":
        w("    int waves = 1;")
        room = ("a->nitems * waves < %d" % SHARE_ITEMS if len(graph(*am).top_keys) <= SHARE_TOPS
                else "2 * a->nitems * waves <= %d" % (SHARE_ITEMS // 2))
        w("    while (waves < %d && waves < depth && %s) waves *= 2;" % (most, room))
        w("    if (waves > 1) {")
        w("        hipLaunchKernelGGL(eri_%s, dim3((unsigned)a->nitems), dim3(64, waves), 0, s, *a);"
          % kname.replace("_", "k_", 1))
        w("        return hipGetLastError();")
        w("    }")
    elif kind == "turn":
        terms = 2 * 512 * len(graph(*am).top_keys)   # of one wavefront, both buffers
        for waves in (8, 4):
            if waves <= most:
                w("    if (a->nitems <= %d && depth > %d%s) {"
                  % (256 * (160 * 1024 // (waves * terms)), waves // 2, "" if waves == most else " && depth <= %d" % waves))
                w("        hipLaunchKernelGGL(eri_%s, dim3((unsigned)a->nitems), dim3(64, %d), %du, s, *a);"
                  % (kname.replace("_", "k_", 1), waves, waves * terms))
                w("        return hipGetLastError();")
                w("    }")
    w("    hipLaunchKernelGGL(eri_%s, dim3((unsigned)a->nitems), dim3(64), 0, s, *a);" % kname)
    w("    return hipGetLastError();")
    w("}")
    w("")


def _emit_share_sum(ntop, most, w):
    """Add the wavefronts' sums to the first one's, which goes on alone."""
    w("    __shared__ double part[%d];" % ((most - 1) * SHARE_SUM * 64))
    for v0 in range(0, ntop, SHARE_SUM):
        vals = range(v0, min(ntop, v0 + SHARE_SUM))
        if v0:
            w("    __syncthreads();")
        w("    if (wave != 0) {")
        w("        double *const x = part + (wave - 1) * %d + lane;" % (SHARE_SUM * 64))
        for t in vals:
            w("        x[%d] = acc%d;" % (64 * (t - v0), t))
        w("    }")
        w("    __syncthreads();")
        w("    if (wave == 0) {")
        w("        for (int v = 0; v < waves - 1; ++v) {")
        w("            const double *const x = part + v * %d + lane;" % (SHARE_SUM * 64))
        for t in vals:
            w("            acc%d += x[%d];" % (t, 64 * (t - v0)))
        w("        }")
        w("    }")
    w("    if (wave != 0) return;")


def _emit_share_turn(ntop, most, w):
    """The round's terms of every wavefront to the local data share (two
    buffers by turns, one barrier a round), then the owned values' sums."""
    w("        double *const x = terms + turn * (waves * %d) + lane;" % (ntop * 64))
    w("        turn ^= 1;")
    for t in range(ntop):
        w("        x[(wave * %d + %d) * 64] = acc%d;" % (ntop, t, t))
    w("        __syncthreads();")
    w("#pragma unroll")
    w("        for (int k = 0; k < OWN; ++k) {")
    w("            const int t = wave + waves * k;")
    w("            if (t < %d) {" % ntop)
    w("                double y[%d];   // all loads before the sum" % most)
    w("#pragma unroll")
    w("                for (int v = 0; v < %d; ++v) y[v] = v < waves ? x[(v * %d + t) * 64] : 0.0;" % (most, ntop))
    w("#pragma unroll")
    w("                for (int v = 0; v < %d; ++v) own[k] += y[v];" % most)
    w("            }")
    w("        }")


def _emit_share_end(ntop, w):
    """Every sum to the first wavefront, which goes on alone."""
    w("    __syncthreads();")
    w("#pragma unroll")
    w("    for (int k = 0; k < OWN; ++k) {")
    w("        const int t = wave + waves * k;")
    w("        if (t < %d) terms[t * 64 + lane] = own[k];" % ntop)
    w("    }")
    w("    __syncthreads();")
    w("    if (wave != 0) return;")
    for t in range(ntop):
        w("    const double acc%d = terms[%d + lane];" % (t, 64 * t))


def _emit_lpq_prefix(am, w, fp, hrr_fp="double", shared=None):
    """shared: blockDim.y wavefronts share the item's primitive quartets
    ("sum", "turn": share_kind)."""
    g = graph(*am)
    name = class_name(am)
    ntop = len(g.top_keys)
    kname = ("eri_lpqm%s_%s" if fp == "float" else "eri_lpq%s_%s") % ("k" if shared else "", name)
    most = share_waves(am)
    w("__global__ void __launch_bounds__(%d) %s(const EriArgs A)" % (64 * most if shared else 64, kname))
    w("{")
    w("    const WorkItem wi = A.items[blockIdx.x];")
    w("    const int lane = threadIdx.x;")
    w("    const double *__restrict__ grid = A.boys_grid;")
    w("    const int ib0 = A.bra.poff[wi.bra];")
    w("    const int ib1 = ib0 + A.bra.np[wi.bra];")
    w("    const int nq = A.ket.tnp[wi.tile];")
    w("    const long long tl = (long long)wi.tile * SIMINT_TILE + lane;")
    w("    const long long kb = A.ket.toff[wi.tile] + lane;")
    w("    const bool screen = A.tol2 > 0.0;")
    if shared:
        w("    const int waves = (int)blockDim.y;")
        w("    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);")
    if shared == "sum":
        # strides over the bra primitives and, where those are fewer, the ket's
        w("    int istep = waves;")
        w("    while (istep > 1 && istep > ib1 - ib0) istep >>= 1;")
        w("    const int jstep = waves / istep;")
        w("    const int i0 = ib0 + wave / jstep, j0 = wave % jstep;")
    if shared == "turn":
        w("    extern __shared__ double terms[];")
        w("    constexpr int OWN = %d;   // values a wavefront adds up, with four of them or more" % ((ntop + 3) // 4))
        w("    double own[OWN];")
        w("#pragma unroll")
        w("    for (int k = 0; k < OWN; ++k) own[k] = 0.0;")
        w("    const int K = (ib1 - ib0) * nq;")
        w("    int turn = 0;")
    else:
        for t in range(ntop):
            w("    double acc%d = 0.0;" % t)
    bra_pa = "pa" if g.bra_j else "pb"
    ket_pa = "pa" if g.ket_l else "pb"
    if shared == "turn":
        w("    for (int p0 = 0; p0 < K; p0 += waves) {")
        for t in range(ntop):
            w("        double acc%d = 0.0;" % t)
        w("        const int p = p0 + wave;")
        w("        const int ii = p / nq;")
        w("        for (int once = p < K; once; once = 0) {")
        w("        const int i = ib0 + ii, j = p - ii * nq;")
    else:
        w("    for (int i = i0; i < ib1; i += istep) {" if shared else "    for (int i = ib0; i < ib1; ++i) {")
    w("        const double P_alpha = A.bra.alpha[i];")
    w("        const double P_inv = A.bra.inv_alpha[i];")
    w("        const double P_prefac = A.bra.prefac[i];")
    w("        const double P_x = A.bra.x[i], P_y = A.bra.y[i], P_z = A.bra.z[i];")
    w("        const double P_%s[3] = {A.bra.%sx[i], A.bra.%sy[i], A.bra.%sz[i]};"
      % ("PA" if g.bra_j else "PB", bra_pa, bra_pa, bra_pa))
    w("        const double P_screen = screen ? A.bra.screen[i] : 0.0;")
    w("        if (screen && P_screen * A.ket_screen_max < A.tol2) continue;")
    w({"turn": "        {", "sum": "        for (int j = j0; j < nq; j += jstep) {"}.get(
        shared, "        for (int j = 0; j < nq; ++j) {"))
    w("            const long long kj = kb + (long long)SIMINT_TILE * j;")
    w("            if (screen && A.ket.screen[kj] * P_screen < A.tol2) continue;")
    w("            const double Q_alpha = A.ket.alpha[kj];")
    w("            const double Q_inv = A.ket.inv_alpha[kj];")
    w("            const double Q_prefac = A.ket.prefac[kj];")
    w("            const double Q_x = A.ket.x[kj], Q_y = A.ket.y[kj], Q_z = A.ket.z[kj];")
    w("            const double Q_%s[3] = {A.ket.%sx[kj], A.ket.%sy[kj], A.ket.%sz[kj]};"
      % ("PA" if g.ket_l else "PB", ket_pa, ket_pa, ket_pa))
    emit_body(am, w, indent="            ", fp=fp)
    w("        }")
    w("    }")
    if shared == "sum":
        _emit_share_sum(ntop, most, w)
    if shared == "turn":
        _emit_share_turn(ntop, most, w)
        w("    }")
        _emit_share_end(ntop, w)
    # direct stores (through LDS slices measured 3% slower on these
    # compute-bound kernels)
    w("    if (lane < wi.lane_lo || lane >= wi.lane_hi) return;")
    w("    const long long colv = A.ket.col[tl];")
    w("    double *__restrict__ o = A.out + wi.obase + colv * A.stride;")
    if g.bra_hrr_needed():
        w("    const double hAB[3] = {A.bra.abx[wi.bra], A.bra.aby[wi.bra], A.bra.abz[wi.bra]};")
    if g.ket_hrr_needed():
        w("    const double hCD[3] = {A.ket.abx[tl], A.ket.aby[tl], A.ket.abz[tl]};")
    # the HRR stays FP64: its AB / CD transfers cancel strongly for the
    # far-apart pairs that have small Schwarz bounds, and FP32 there loses
    # far more than the ERI error budget
    emit_hrr(am, w, fp=hrr_fp)
    w("}")
    w("")


def emit_lpq_list(am, w):
    """Quartet-list variant: S = A.split lanes per quartet (a power of two
    up to 64); lanes 64k + l take quartet (64k + l) / S, with its own bra and
    ket pair (both read from the linear view, per-lane gathers).  Lane
    sub = l % S sums primitive quartets sub, sub + S, ... (bra-major order,
    as the reference's loops); the S partial sums are added across the
    lanes (xor butterfly), then lane sub = 0 runs the HRR and writes the
    contiguous output block.  With S = 1 the summation order is the
    lane-per-quartet kernels'."""
    g = graph(*am)
    name = class_name(am)
    ntop = len(g.top_keys)
    w("__global__ void __launch_bounds__(64) eri_lpql_%s(const EriListArgs A)" % name)
    w("{")
    w("    const int S = A.split;")
    w("    const long long gl = (long long)blockIdx.x * 64 + threadIdx.x;")
    w("    const long long q = gl / S;")
    w("    const int sub = (int)(gl - q * S);")
    w("    const bool valid = q < A.nquartet;")
    w("    // lanes past the list stay until the cross-lane sums")
    w("    const long long qc = valid ? q : A.nquartet - 1;")
    w("    const int bp = A.qbra[qc], kp = A.qket[qc];")
    w("    const double *__restrict__ grid = A.boys_grid;")
    w("    const int ib0 = A.bra.poff[bp];")
    w("    const int jb0 = A.ket.poff[kp];")
    w("    const int nqk = A.ket.np[kp];")
    w("    const int K = valid ? A.bra.np[bp] * nqk : 0;")
    w("    const bool screen = A.tol2 > 0.0;")
    for t in range(ntop):
        w("    double acc%d = 0.0;" % t)
    bra_pa = "pa" if g.bra_j else "pb"
    ket_pa = "pa" if g.ket_l else "pb"
    w("    int ii = 0, jj = sub;")
    w("    for (int p = sub; p < K; p += S) {")
    w("        while (jj >= nqk) { jj -= nqk; ++ii; }")
    w("        const int i = ib0 + ii, kj = jb0 + jj;")
    w("        jj += S;")
    w("        const double P_screen = screen ? A.bra.screen[i] : 0.0;")
    w("        if (screen && (P_screen * A.ket_screen_max < A.tol2 || A.ket.screen[kj] * P_screen < A.tol2)) continue;")
    w("        const double P_alpha = A.bra.alpha[i];")
    w("        const double P_inv = A.bra.inv_alpha[i];")
    w("        const double P_prefac = A.bra.prefac[i];")
    w("        const double P_x = A.bra.x[i], P_y = A.bra.y[i], P_z = A.bra.z[i];")
    w("        const double P_%s[3] = {A.bra.%sx[i], A.bra.%sy[i], A.bra.%sz[i]};"
      % ("PA" if g.bra_j else "PB", bra_pa, bra_pa, bra_pa))
    w("        {")
    w("            const double Q_alpha = A.ket.alpha[kj];")
    w("            const double Q_inv = A.ket.inv_alpha[kj];")
    w("            const double Q_prefac = A.ket.prefac[kj];")
    w("            const double Q_x = A.ket.x[kj], Q_y = A.ket.y[kj], Q_z = A.ket.z[kj];")
    w("            const double Q_%s[3] = {A.ket.%sx[kj], A.ket.%sy[kj], A.ket.%sz[kj]};"
      % ("PA" if g.ket_l else "PB", ket_pa, ket_pa, ket_pa))
    emit_body(am, w, indent="            ")
    w("        }")
    w("    }")
    w("    for (int o = 1; o < S; o <<= 1) {")
    for t in range(ntop):
        w("        acc%d += __shfl_xor(acc%d, o);" % (t, t))
    w("    }")
    w("    if (!valid || sub != 0) return;")
    w("    double *__restrict__ o = A.out + (A.qout ? A.qout[q] : q * A.ostride);")
    if g.bra_hrr_needed():
        w("    const double hAB[3] = {A.bra.abx[bp], A.bra.aby[bp], A.bra.abz[bp]};")
    if g.ket_hrr_needed():
        w("    const double hCD[3] = {A.ket.abx[kp], A.ket.aby[kp], A.ket.abz[kp]};")
    emit_hrr(am, w)
    w("}")
    w("")
    w('extern "C" hipError_t simint_launch_lpql_%s(const EriListArgs *a, hipStream_t s)' % name)
    w("{")
    w("    if (a->nquartet <= 0) return hipSuccess;")
    w("    if (a->split < 1 || a->split > 64 || (a->split & (a->split - 1))) return hipErrorInvalidValue;")
    w("    hipLaunchKernelGGL(eri_lpql_%s, dim3((unsigned)((a->nquartet * a->split + 63) / 64)), dim3(64), 0, s, *a);"
      % name)
    w("    return hipGetLastError();")
    w("}")
