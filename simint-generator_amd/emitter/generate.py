"""Emit every generated source of the engine into csrc/gen/.

  boys_grid.inc, boys_longfac.inc   Boys tables (emitter/boys_table.py)
  eri_lpq_<class>.hip               lane-per-quartet kernels (hip_lpq.py)
  eri_wpq_<class>.hip               wave-per-quartet kernels (hip_wpq.py)
  eri_cpl_<class>.hip               component-lane kernels (hip_cpl.py)
  eri_lpqs<G>_<class>.hip           split lane-per-quartet kernels, G bra-top
                                    groups (hip_lpqs.py)
  dispatch.cpp                      launcher tables + kernel-family choice
  classes.json                      per-class sizes and algorithmic FLOP counts
and include/simint/ostei/ostei_config.h (config_header.py).
Files are rewritten only when their text changes, so the build can reuse
objects.
"""
import itertools
import json
import os

from . import boys_table, config_header, hip_cpl, hip_lpq, hip_lpqs, hip_wpq
from .rrgraph import graph, ncart

# Lane-per-quartet kernels are built for every class.  The default family
# per class is lane-per-quartet when the compiler reports no scratch spills,
# else the split lane-per-quartet kernel where one is built, else
# wave-per-quartet (derivative terms with a g shell: component-lane);
# tuning.json (written by autotune.py from GPU timings of every family a
# class has) overrides the default.
# (the register kernels of the largest f classes are left out: their
# straight-line code runs to >10^5 statements and could only spill)
LPQ_MAX_TOPS = 1000
LPQ_MAX_NODES = 2200


def _write(path, text):
    if os.path.exists(path):
        with open(path) as f:
            if f.read() == text:
                return False
    tmp = path + ".tmp"
    with open(tmp, "w") as f:
        f.write(text)
    os.replace(tmp, path)
    return True


LPQS_MIN_TOPS = 64   # split kernels for classes with more contracted HRR inputs than this
LPQS_F_MAX_TOPS = 1500   # f classes: one split variant up to this size (the
LPQS_F_MAX_NODES = 5000  # (a+1) terms of the d-class derivatives are among them)


def lpqs_variants(am):
    """Group counts of the split kernels built for a class ([] = none).
    Classes whose bra carries at least the ket's AM split over bra tops (ket
    HRR first); the others over ket tops (bra HRR first): the ket-first order
    with the heavier transfer on the ket side measurably loses accuracy
    (median error 20x the reference algorithm's on (pp|ff))."""
    g = graph(*am)
    nt = len(g.top_keys)
    if nt <= LPQS_MIN_TOPS:
        return []
    if max(am) <= 2:
        return hip_lpqs.split_counts(am) if lpq_candidate(am) else []
    if max(am) == 3 and nt <= LPQS_F_MAX_TOPS and len(g.node_list) <= LPQS_F_MAX_NODES:
        return hip_lpqs.split_counts(am)[:1]
    return []


def lpqsf_variants(am):
    """Group counts of the ket-top split kernels built as a second choice for
    a d class whose default split kernels group bra tops: ket-top groups run
    the reference's HRR order (bra, then ket) and write their output straight
    through the local data share, so they stage less per quartet, at the cost
    of recomputing more of the VRR per group.  The autotuner picks."""
    if max(am) > 2 or hip_lpqs.split_kind(am) != "e" or not lpqs_variants(am):
        return []
    return hip_lpqs.split_counts(am, "f")


def deriv_term_classes(maxam):
    """Classes with one AM of maxam+1 that first derivatives of classes up to
    maxam need: the (a+1) terms of every centre but the first with the
    highest AM (ostei_deriv1_generator.cpp:96-124).  They run the
    component-lane kernels (the cooperative kernels are built for them too;
    a stream of 1500 first derivatives took 1220 ms with those, 137 ms with
    these)."""
    out = set()
    for am in itertools.product(range(maxam + 1), repeat=4):
        skip = am.index(max(am))
        for c in range(4):
            if c == skip:
                continue
            t = list(am)
            t[c] += 1
            if max(t) == maxam + 1:
                out.add(tuple(t))
    return sorted(out)


def classes(maxam):
    return list(itertools.product(range(maxam + 1), repeat=4))


def lpq_candidate(am):
    g = graph(*am)
    return len(g.tops) <= LPQ_MAX_TOPS and len(g.node_list) <= LPQ_MAX_NODES


def class_info(am):
    g = graph(*am)
    fc = g.flop_counts()
    la, lb, lc, ld = am
    return {
        "am": list(am),
        "L": g.Ltot,
        "ncart": ncart(la) * ncart(lb) * ncart(lc) * ncart(ld),
        "f_setup": fc["f_setup"],
        "f_vrr": fc["f_vrr"],
        "f_boys": fc["f_boys"],
        "bcont": fc["bcont"],
        "f_hrr": fc["f_hrr"],
        "prim": fc["prim"],
        "cont": fc["cont"],
        "vrr_nodes": len(g.node_list),
    }


MIXED_MAXAM = 2   # classes with an FP32-VRR/HRR variant (lane-per-quartet family)


def mixed_candidate(am):
    return max(am) <= MIXED_MAXAM


def dispatch_text(maxam, lpq, wpq, selection, lpqs=None, list_selection=None, lpqsf=None, cpl=(), deep=None,
                  even=None):
    # tables reach one AM above the maximum when derivative terms are built
    n = 1 + max(max(am) for am in wpq)
    lines = ["// Generated by simint-generator_amd/emitter/generate.py -- do not edit.",
             '#include <atomic>',
             '#include "../dispatch.h"',
             '#include "simint/simint_hip.h"',
             ""]
    for am in lpq:
        lines.append('extern "C" hipError_t simint_launch_lpq_%s(const EriArgs *, hipStream_t);' % hip_lpq.class_name(am))
    for am in wpq:
        lines.append('extern "C" hipError_t simint_launch_wpq_%s(const EriArgs *, hipStream_t);' % hip_lpq.class_name(am))
    for am in lpq:
        lines.append('extern "C" hipError_t simint_launch_lpql_%s(const EriListArgs *, hipStream_t);'
                     % hip_lpq.class_name(am))
    lpqm = [am for am in lpq if mixed_candidate(am)]
    for am in lpqm:
        lines.append('extern "C" hipError_t simint_launch_lpqm_%s(const EriArgs *, hipStream_t);'
                     % hip_lpq.class_name(am))
    lpqs = lpqs or {}
    for am, Gs in lpqs.items():
        for G in Gs:
            lines.append('extern "C" hipError_t simint_launch_%s(const EriArgs *, hipStream_t);'
                         % hip_lpqs.kernel_name(am, G))
    lpqsf = lpqsf or {}
    for am, Gs in lpqsf.items():
        for G in Gs:
            lines.append('extern "C" hipError_t simint_launch_%s(const EriArgs *, hipStream_t);'
                         % hip_lpqs.kernel_name(am, G, "f"))
    for am in wpq:
        lines.append('extern "C" hipError_t simint_launch_wpql_%s(const EriListArgs *, hipStream_t);'
                     % hip_lpq.class_name(am))
    for am in cpl:
        lines.append('extern "C" hipError_t simint_launch_cpl_%s(const EriArgs *, hipStream_t);' % hip_lpq.class_name(am))
        lines.append('extern "C" hipError_t simint_launch_cpll_%s(const EriListArgs *, hipStream_t);'
                     % hip_lpq.class_name(am))
    lines.append("")
    lines.append("namespace {")
    lines.append("constexpr int N = %d;" % n)

    def table(name, have, prefix, typ="simint_launch_fn", cell=None):
        lines.append("const %s %s[N][N][N][N] = {" % (typ, name))
        for a in range(n):
            lines.append(" {")
            for b in range(n):
                lines.append("  {")
                for c in range(n):
                    row = []
                    for d in range(n):
                        am = (a, b, c, d)
                        if cell is not None:
                            row.append(cell(am))
                            continue
                        row.append(("simint_launch_%s_%s" % (prefix, hip_lpq.class_name(am))) if am in have else "nullptr")
                    lines.append("   {" + ", ".join(row) + "},")
                lines.append("  },")
            lines.append(" },")
        lines.append("};")

    table("g_lpq", set(lpq), "lpq")
    table("g_wpq", set(wpq), "wpq")
    table("g_lpql", set(lpq), "lpql", "simint_list_launch_fn")
    table("g_lpqm", set(lpqm), "lpqm")

    def split_cell(k):
        def f(am):
            Gs = lpqs.get(am, [])
            return ("simint_launch_%s" % hip_lpqs.kernel_name(am, Gs[k])) if len(Gs) > k else "nullptr"
        return f
    table("g_lpqs_a", None, None, cell=split_cell(0))
    table("g_lpqs_b", None, None, cell=split_cell(1))
    table("g_stage", None, None, typ="int",
          cell=lambda am: str(hip_lpqs.staging_doubles(am) if lpqs.get(am) else 0))

    def splitf_cell(k):
        def f(am):
            Gs = lpqsf.get(am, [])
            return ("simint_launch_%s" % hip_lpqs.kernel_name(am, Gs[k], "f")) if len(Gs) > k else "nullptr"
        return f
    table("g_lpqs_c", None, None, cell=splitf_cell(0))
    table("g_lpqs_d", None, None, cell=splitf_cell(1))
    table("g_stage_f", None, None, typ="int",
          cell=lambda am: str(hip_lpqs.staging_doubles(am, "f") if lpqsf.get(am) else 0))
    table("g_wpql", set(wpq), "wpql", "simint_list_launch_fn")
    table("g_cpl", set(cpl), "cpl")
    table("g_cpll", set(cpl), "cpll", "simint_list_launch_fn")
    # the built-in choice carries BUILTIN: only it gives way to another family
    # by the size of a launch
    lines.append("constexpr int BUILTIN = 16, FAMILY = 15;")
    flat = []
    for am in itertools.product(range(n), repeat=4):
        flat.append("%d" % (selection[am] | 16) if am in selection else "0")
    lines.append("std::atomic<int> g_sel[N * N * N * N] = {" + ", ".join(flat) + "};")
    lines.append("const int g_sel_built[N * N * N * N] = {" + ", ".join(flat) + "};")
    flat = []
    for am in itertools.product(range(n), repeat=4):
        flat.append("%d" % ((list_selection or {}).get(am, 2) | 16))
    lines.append("std::atomic<int> g_sel_list[N * N * N * N] = {" + ", ".join(flat) + "};")
    lines.append("const int g_sel_list_built[N * N * N * N] = {" + ", ".join(flat) + "};")
    lines.append("const unsigned char g_deep[N * N * N * N] = {"
                 + ", ".join(str((deep or {}).get(am, 0)) for am in itertools.product(range(n), repeat=4)) + "};")
    lines.append("// primitive quartets from which a list of even depth runs the lane-per-quartet kernel: of")
    lines.append("// quartets of fewer than EVEN_DEPTH, and of deeper ones (0: never)")
    lines.append("constexpr int EVEN_DEPTH = %d;" % EVEN_DEPTH)
    lines.append("const int g_even[N * N * N * N][2] = {"
                 + ", ".join("{%d, %d}" % tuple((even or {}).get(am, (0, 0)))
                             for am in itertools.product(range(n), repeat=4)) + "};")
    lines.append("inline int idx(int a, int b, int c, int d) { return ((a * N + b) * N + c) * N + d; }")
    lines.append("inline bool in_range(int a, int b, int c, int d)")
    lines.append("{ return a >= 0 && b >= 0 && c >= 0 && d >= 0 && a < N && b < N && c < N && d < N; }")
    lines.append("}  // namespace")
    lines.append("")
    lines.append("simint_launch_fn simint_family_launch(int s, int la, int lb, int lc, int ld)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return nullptr;")
    lines.append("    if (s == 1) return g_lpq[la][lb][lc][ld];")
    lines.append("    if (s == 2) return g_wpq[la][lb][lc][ld];")
    lines.append("    if (s == 3) return g_lpqs_a[la][lb][lc][ld];")
    lines.append("    if (s == 4) return g_lpqs_b[la][lb][lc][ld];")
    lines.append("    if (s == 5) return g_lpqs_c[la][lb][lc][ld];")
    lines.append("    if (s == 6) return g_lpqs_d[la][lb][lc][ld];")
    lines.append("    if (s == 7) return g_cpl[la][lb][lc][ld];")
    lines.append("    return nullptr;")
    lines.append("}")
    lines.append("")
    lines.append("int simint_family_staging(int s, int la, int lb, int lc, int ld)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return 0;")
    lines.append("    if (s == 5 || s == 6) return g_stage_f[la][lb][lc][ld];")
    lines.append("    return (s == 3 || s == 4) ? g_stage[la][lb][lc][ld] : 0;")
    lines.append("}")
    lines.append("")
    lines.append("int simint_range_family(int la, int lb, int lc, int ld, long long items, long long depth)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return 0;")
    lines.append("    const int i = idx(la, lb, lc, ld);")
    lines.append("    const int s = g_sel[i].load(std::memory_order_relaxed);")
    lines.append("    if ((s & BUILTIN) && g_deep[i] && items >= %d && depth >= %d) return g_deep[i];" % (DEEP_ITEMS, DEEP_DEPTH))
    lines.append("    return s & FAMILY;")
    lines.append("}")
    lines.append("")
    lines.append("simint_launch_fn simint_dispatch(int la, int lb, int lc, int ld)")
    lines.append("{ return simint_family_launch(simint_range_family(la, lb, lc, ld, 0, 0), la, lb, lc, ld); }")
    lines.append("")
    lines.append("int simint_dispatch_staging(int la, int lb, int lc, int ld)")
    lines.append("{ return simint_family_staging(simint_range_family(la, lb, lc, ld, 0, 0), la, lb, lc, ld); }")
    lines.append("")
    lines.append("simint_launch_fn simint_dispatch_mixed(int la, int lb, int lc, int ld)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return nullptr;")
    lines.append("    const int s = g_sel[idx(la, lb, lc, ld)].load(std::memory_order_relaxed) & FAMILY;")
    lines.append("    return s == 1 ? g_lpqm[la][lb][lc][ld] : nullptr;")
    lines.append("}")
    lines.append("")
    lines.append("simint_list_launch_fn simint_dispatch_list(int la, int lb, int lc, int ld)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return nullptr;")
    lines.append("    const int s = g_sel_list[idx(la, lb, lc, ld)].load(std::memory_order_relaxed) & FAMILY;")
    lines.append("    if (s == 1 && g_lpql[la][lb][lc][ld]) return g_lpql[la][lb][lc][ld];")
    lines.append("    if (s == 7 && g_cpll[la][lb][lc][ld]) return g_cpll[la][lb][lc][ld];")
    lines.append("    return g_wpql[la][lb][lc][ld];")
    lines.append("}")
    lines.append("")
    lines.append("simint_list_launch_fn simint_dispatch_list_even(int la, int lb, int lc, int ld, long long n, long long depth)")
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return nullptr;")
    lines.append("    const int i = idx(la, lb, lc, ld);")
    lines.append("    const int from = g_even[i][depth >= EVEN_DEPTH];")
    lines.append("    if (g_sel_list[i].load(std::memory_order_relaxed) != (7 | BUILTIN) || from == 0 || n * depth < from) return nullptr;")
    lines.append("    return g_lpql[la][lb][lc][ld];")
    lines.append("}")
    lines.append("")
    lines.append('extern "C" int simint_hip_class_list_kernel(int la, int lb, int lc, int ld)')
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return 0;")
    lines.append("    return g_sel_list[idx(la, lb, lc, ld)].load() & FAMILY;")
    lines.append("}")
    lines.append("")
    lines.append('extern "C" int simint_hip_set_class_list_kernel(int la, int lb, int lc, int ld, int family)')
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return -1;")
    lines.append("    if (family == 1 && !g_lpql[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 2 && !g_wpql[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 7 && !g_cpll[la][lb][lc][ld]) return -1;")
    lines.append("    if (family != 1 && family != 2 && family != 7) return -1;")
    lines.append("    return g_sel_list[idx(la, lb, lc, ld)].exchange(family) & FAMILY;")
    lines.append("}")
    lines.append("")
    lines.append('extern "C" int simint_hip_class_kernel(int la, int lb, int lc, int ld)')
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return 0;")
    lines.append("    return g_sel[idx(la, lb, lc, ld)].load() & FAMILY;")
    lines.append("}")
    lines.append("")
    lines.append('extern "C" int simint_hip_set_class_kernel(int la, int lb, int lc, int ld, int family)')
    lines.append("{")
    lines.append("    if (!in_range(la, lb, lc, ld)) return -1;")
    lines.append("    if (family == 1 && !g_lpq[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 2 && !g_wpq[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 3 && !g_lpqs_a[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 4 && !g_lpqs_b[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 5 && !g_lpqs_c[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 6 && !g_lpqs_d[la][lb][lc][ld]) return -1;")
    lines.append("    if (family == 7 && !g_cpl[la][lb][lc][ld]) return -1;")
    lines.append("    if (family < 1 || family > 7) return -1;")
    lines.append("    return g_sel[idx(la, lb, lc, ld)].exchange(family) & FAMILY;")
    lines.append("}")
    lines.append("")
    lines.append('extern "C" void simint_hip_reset_class_kernels(void)')
    lines.append("{")
    lines.append("    for (int i = 0; i < N * N * N * N; i++) {")
    lines.append("        g_sel[i] = g_sel_built[i];")
    lines.append("        g_sel_list[i] = g_sel_list_built[i];")
    lines.append("    }")
    lines.append("}")
    return "\n".join(lines) + "\n"


FAMILIES = {"lpq": 1, "wpq": 2, "lpqs_a": 3, "lpqs_b": 4, "lpqsf_a": 5, "lpqsf_b": 6, "cpl": 7}


# The component-lane kernels spread one quartet over lanes; many deep quartets
# run faster where staging keeps every lane busy.  "deep_family" of tuning.json
# names the family of a class for launches of at least DEEP_ITEMS work items of
# DEEP_DEPTH primitive quartets: 4096 items of (dd|pp) take 1.57 ms in the
# component-lane kernel and 1.25 ms in the split one at 16 primitive quartets,
# 6.9 and 4.7 ms at 81; of (dp|dp) 1.37 and 1.23, 6.1 and 4.7 ms; at one
# primitive quartet 0.28 and 0.58 ms; 256 items of 81 0.55 and 1.15 ms.
DEEP_ITEMS = 1024
DEEP_DEPTH = 16
# Lists tuned to the component-lane kernels on a stream of mixed depths, whose
# lane-per-quartet wavefronts wait for their deepest lane: a list of even depth
# runs the lane-per-quartet kernel from "list_even" of tuning.json primitive
# quartets on (below EVEN_DEPTH a quartet, and from there; autotune.py --list
# --even).  3200 (fp|ps) quartets of 16 primitive quartets: 84 us in the
# component-lane kernels (38 unshared), 15 us in the other.
EVEN_DEPTH = 16


def load_tuning(pkg_root, key="family", names=FAMILIES):
    """Tuned value per class from tuning.json ("family": prefix kernels,
    "list_family": quartet-list kernels, "deep_family", "list_even",
    "lane_items"); names maps it to a number (None: as it is)."""
    path = os.path.join(pkg_root, "tuning.json")
    if not os.path.exists(path):
        return {}
    d = json.load(open(path))
    out = {}
    for name, fam in d.get(key, {}).items():
        out[tuple("spdfghik".index(c) for c in name.split("_"))] = names[fam] if names else fam
    return out


def generate(pkg_root, include_root, maxam, lpq_ok=None):
    """Write generated sources.  lpq_ok: set of classes whose LPQ build was
    spill-free (None = before the first compile: every candidate counts).
    Returns (lpq_classes, wpq_classes, selection, split groups, cpl_classes)."""
    gen = os.path.join(pkg_root, "csrc", "gen")
    os.makedirs(gen, exist_ok=True)
    boys_table.write(gen)
    cls = classes(maxam)
    lpq = [am for am in cls if lpq_candidate(am)]
    gterms = deriv_term_classes(maxam)
    wpq = list(cls) + gterms
    lane_items = load_tuning(pkg_root, "lane_items", None)
    for am in lpq:
        _write(os.path.join(gen, "eri_lpq_%s.hip" % hip_lpq.class_name(am)),
               hip_lpq.emit_lpq(am, mixed=mixed_candidate(am), lane_items=lane_items.get(am)))
    for am in wpq:
        _write(os.path.join(gen, "eri_wpq_%s.hip" % hip_lpq.class_name(am)), hip_wpq.emit_wpq(am))
    cpl = [am for am in wpq if hip_cpl.candidate(am)]
    for am in cpl:
        _write(os.path.join(gen, "eri_cpl_%s.hip" % hip_lpq.class_name(am)), hip_cpl.emit_cpl(am))
    lpqs = {}
    for am in cls:
        Gs = lpqs_variants(am)
        if Gs:
            lpqs[am] = Gs
            for G in Gs:
                _write(os.path.join(gen, "eri_%s.hip" % hip_lpqs.kernel_name(am, G)), hip_lpqs.emit_lpqs(am, G))
    lpqsf = {}
    for am in cls:
        Gs = lpqsf_variants(am)
        if Gs:
            lpqsf[am] = Gs
            for G in Gs:
                _write(os.path.join(gen, "eri_%s.hip" % hip_lpqs.kernel_name(am, G, "f")),
                       hip_lpqs.emit_lpqs(am, G, "f"))
    selection = {}
    tuned = load_tuning(pkg_root)

    def built(am, fam):
        if fam == 7:
            return am in cpl
        if fam < 3:
            return True
        if fam < 5:
            return len(lpqs.get(am, [])) > fam - 3
        return len(lpqsf.get(am, [])) > fam - 5
    for am in cls:
        if am in tuned and built(am, tuned[am]):
            selection[am] = tuned[am]
        elif am in lpq and (lpq_ok is None or am in lpq_ok):
            selection[am] = 1
        elif am in lpqs:
            selection[am] = 3
        else:
            selection[am] = 2
    for am in gterms:
        selection[am] = 7 if am in cpl else 2
    list_sel = {}
    tuned_list = load_tuning(pkg_root, "list_family")
    for am in cls:
        if am in tuned_list and tuned_list[am] in (1, 2, 7) and (tuned_list[am] == 2 or am in (lpq if tuned_list[am] == 1
                                                                                              else cpl)):
            list_sel[am] = tuned_list[am]
        elif am in lpq and (lpq_ok is None or am in lpq_ok):
            list_sel[am] = 1
        else:
            list_sel[am] = 2
    for am in gterms:
        list_sel[am] = selection[am]
    deep = {am: f for am, f in load_tuning(pkg_root, "deep_family").items() if built(am, f) and am in selection}
    even = {am: t for am, t in load_tuning(pkg_root, "list_even", None).items() if am in lpq and am in cpl}
    _write(os.path.join(gen, "dispatch.cpp"), dispatch_text(maxam, lpq, wpq, selection, lpqs, list_sel, lpqsf, cpl,
                                                        deep, even))
    fname = {v: k for k, v in FAMILIES.items()}
    info = {hip_lpq.class_name(am): dict(class_info(am), kernel=fname[selection[am]], split_groups=lpqs.get(am, []),
                                         split_kernels=[hip_lpqs.kernel_name(am, G) for G in lpqs.get(am, [])],
                                         split_kernels_f=[hip_lpqs.kernel_name(am, G, "f")
                                                          for G in lpqsf.get(am, [])])
            for am in cls}
    _write(os.path.join(gen, "classes.json"), json.dumps(info, indent=1, sort_keys=True))
    _write(os.path.join(include_root, "simint", "ostei", "ostei_config.h"),
           config_header.text(maxam, 1, maxam if gterms else maxam - 1))
    allsplit = dict(lpqs)
    allsplit.update({("f",) + am: Gs for am, Gs in lpqsf.items()})
    return lpq, wpq, selection, allsplit, cpl
