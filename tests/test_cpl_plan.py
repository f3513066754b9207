"""Component-lane kernels, checked on the CPU from their plan: the lane
tables walk every wide component's reduction path, no index leaves its area,
and the values of the two-stage recurrence equal the recurrence graph's."""
import itertools

import pytest

from emitter import generate, hip_cpl
from emitter.rrgraph import I, J, mk_dir, step

CLASSES = [am for am in generate.classes(3) + generate.deriv_term_classes(3) if hip_cpl.candidate(am)]


@pytest.mark.parametrize("G", [None, hip_cpl.SPLIT_W])
def test_plans_stay_inside_their_areas(G):
    """Both plans of every class: the base one and the short lists'."""
    assert len(CLASSES) >= 280
    for am in CLASSES:
        p = hip_cpl.split_plan(am) if G else hip_cpl.plan(am, hip_cpl.base_G(am))
        assert p.NQ >= 1 and p.NQ * p.NE <= 64 * p.NS and p.ent % p.NQ == 0 and p.NQ <= p.ent <= 64
        assert p.npc % 2 == 0 and p.area % 2 == 0 and 8 * p.lds_doubles <= hip_cpl.LDS_CU
        assert p.lds_doubles == p.SW * p.ent * (p.npc + hip_cpl.QINFO) + p.area
        # published vectors, the lanes beyond the components included
        assert p.ps > p.NQ * p.NE and p.W * p.npub * p.ps + p.root_doubles(p.ps) <= p.area
        # HRR: tops, then results, HQ quartets at a time
        ks = max(p.nkt, p.ncd) | 1
        assert p.NQ % p.HQ == 0 and p.cc * p.nch >= p.nab
        if p.hold:
            assert p.HQ * p.nkt <= 64 * p.W
            assert p.HQ * p.nbt * (p.nkt | 1) <= p.area and p.HQ * p.cc * ks <= p.area
        else:
            assert p.nch == 1 and p.HQ * max(p.nbt, p.nab) * ks <= p.area
        assert hip_cpl.P_F + p.L + 1 + (p.L % 2 == 0) <= p.npc
        # every top belongs to one wavefront, with its whole path
        assert sorted(f for part in p.parts for f in part) == sorted(p.stops) and len(p.parts) == p.G
        for part, nodes in zip(p.parts, p.part_nodes):
            assert len(part) <= p.nacc
            for f in part:
                while sum(f):
                    assert f in nodes
                    f = step(f, mk_dir(f), -1)
        for e, (dirs, ns, ex, dn) in zip(p.comps, p.lane_tables()):
            f = (0, 0, 0)
            for k in range(p.e_hi):
                d, n = (dirs >> 2 * k) & 3, (ns >> 4 * k) & 15
                if d == 3:
                    assert sum(f) == 0 and n == 0      # identity steps come first
                    continue
                assert n == f[d]
                f = step(f, d, 1)
            assert f == e
            for d in range(3):
                assert (ex >> 4 * d) & 15 == e[d]
                i = p.index[e] - ((dn >> 8 * d) & 255)
                assert i == (p.index[step(e, d, -1)] if e[d] else p.index[e])


@pytest.mark.parametrize("am", [(2, 1, 2, 1), (1, 0, 2, 2), (3, 2, 1, 1), (1, 2, 1, 3), (2, 2, 2, 2)])
def test_two_stage_recurrence_is_the_graphs(am):
    """Every top of the class from random inputs: the chain and tree with
    the kernel's tables against the recurrence graph, in exact rationals."""
    from fractions import Fraction as Q
    import random
    p = hip_cpl.plan(am)
    g = p.g
    rnd = random.Random(5)

    def r():
        return Q(rnd.randint(-9, 9) or 1, rnd.randint(1, 7))
    F = [r() for _ in range(p.L + 1)]
    sides = {}
    for side in ("bra", "ket"):
        sides[side] = {"A": [r() for _ in range(3)], "pq": [r() for _ in range(3)], "over": r(), "o2": r()}
    o2pq = r()
    val = {}
    for n in g.node_list:
        if n.step is None:
            val[n.q, n.m] = F[n.m]
            continue
        s = sides["bra" if n.step in (I, J) else "ket"]
        x = [val[k] if k is not None else 0 for k in n.src]
        v = s["A"][n.dir] * x[0] + s["pq"][n.dir] * x[1]
        v += n.fac[0] * s["o2"] * (x[2] + s["over"] * x[3]) + n.fac[1] * s["o2"] * (x[4] + s["over"] * x[5])
        val[n.q, n.m] = v + n.fac[2] * o2pq * x[6] + n.fac[3] * o2pq * x[7]
    E, S = (sides["bra"], sides["ket"]) if p.s_is_ket else (sides["ket"], sides["bra"])
    lanes = {}
    for e, (dirs, ns, ex, dn) in zip(p.comps, p.lane_tables()):
        prev, cur = None, list(F)
        for k in range(p.e_hi):
            d, n = (dirs >> 2 * k) & 3, (ns >> 4 * k) & 15
            a, b = (Q(1), Q(0)) if d == 3 else (E["A"][d], E["pq"][d])
            new = [a * cur[m] + b * cur[m + 1]
                   + (n * E["o2"] * (prev[m] + E["over"] * prev[m + 1]) if n else 0) for m in range(p.L - k)]
            prev, cur = cur, new
        assert len(cur) == p.s_hi + 1
        lanes[e] = {(0, 0, 0): cur}

    def visit(f):
        for c in p.children[f]:
            d = mk_dir(c)
            for e in p.comps:
                v, gp = lanes[e][f], lanes[e].get(step(f, d, -1) if f[d] else None)
                out = []
                for m in range(p.s_hi - sum(f)):
                    x = S["A"][d] * v[m] + S["pq"][d] * v[m + 1]
                    if gp is not None:
                        x += (c[d] - 1) * S["o2"] * (gp[m] + S["over"] * gp[m + 1])
                    if e[d]:
                        x += e[d] * o2pq * lanes[step(e, d, -1)][f][m + 1]
                    out.append(x)
                lanes[e][c] = out
            visit(c)
    visit((0, 0, 0))
    for (e, f), key in zip(g.tops, g.top_keys):
        wide, narrow = (e, f) if p.s_is_ket else (f, e)
        assert lanes[wide][narrow][0] == val[key], (am, e, f)


def test_every_deriv_term_class_is_built():
    assert all(hip_cpl.candidate(am) for am in generate.deriv_term_classes(3))
    assert all(hip_cpl.candidate(am) for am in itertools.product(range(4), repeat=4) if sum(am) >= 9)


def test_deep_plans_share_the_tops_in_another_way():
    """The shortest lists' plans: inside the local data share and 256
    registers, every top with its path in one wavefront, groups of the same
    quartets as the short lists' plan, less work for the longest wavefront."""
    deep = {am: p for am in CLASSES for p in [hip_cpl.deep_plan(am)] if p}
    assert 40 <= len(deep)
    for am, p in deep.items():
        ps = hip_cpl.split_plan(am)
        assert ps.G == hip_cpl.SPLIT_W and p.G == 2 * hip_cpl.SPLIT_W and p.SW == 1
        assert (p.NQ, p.NE) == (ps.NQ, ps.NE) and p.regs(p.NS) <= 240 and p.longest <= 0.75 * ps.longest
        assert 8 * p.lds_doubles <= hip_cpl.LDS_CU
        assert p.lds_doubles == p.ent * (p.npc + hip_cpl.QINFO) + p.area
        assert p.ps > p.NQ * p.NE and p.W * p.npub * p.ps + p.root_doubles(p.ps) <= p.area
        ks = max(p.nkt, p.ncd) | 1
        assert p.NQ % p.HQ == 0 and p.cc * p.nch >= p.nab
        if p.hold:
            assert p.HQ * p.nkt <= 64 * p.W
            assert p.HQ * p.nbt * (p.nkt | 1) <= p.area and p.HQ * p.cc * ks <= p.area
        else:
            assert p.nch == 1 and p.HQ * max(p.nbt, p.nab) * ks <= p.area
        assert sorted(f for part in p.parts for f in part) == sorted(p.stops) and len(p.parts) == p.G
        for part, nodes in zip(p.parts, p.part_nodes):
            assert len(part) <= p.nacc
            for f in part:
                while sum(f):
                    assert f in nodes
                    f = step(f, mk_dir(f), -1)


def test_screened_primitive_quartets_are_left_out():
    """The bits of the mask the primitive loop tests are those of the lanes
    that prepared that primitive quartet for the group's quartets, for every
    batch shape of every plan; and the emitted loops test them."""
    for am in CLASSES:
        for p in (hip_cpl.plan(am, hip_cpl.base_G(am)), hip_cpl.split_plan(am), hip_cpl.deep_plan(am)):
            if p is None:
                continue
            assert p.ent <= 16
            for PBK in range(1, p.ent // p.NQ + 1):
                every = sum(1 << (v * PBK) for v in range(p.NQ))
                GB = p.ent // p.NQ // PBK
                seen = set()
                for gi in range(GB):
                    for pp in range(PBK):
                        bits = {b for b in range(32) if every << (gi * p.NQ * PBK + pp) >> b & 1}
                        # block ((gi NQ + w) PBK + pp) is lane's, as the recurrence reads it
                        assert bits == {(gi * p.NQ + w) * PBK + pp for w in range(p.NQ)}
                        seen |= bits
                assert seen == set(range(GB * p.NQ * PBK))
    for am in [(1, 1, 1, 0), (2, 2, 2, 2), (3, 2, 3, 3)]:
        text = hip_cpl.emit_cpl(am)
        loops = text.split("for (int pp = 0; pp < npb_; ++pp) {\n")[1:]
        assert loops and all(
            x.lstrip().startswith("if (((alive >> (gi * NQ * PBK + pp)) & every) == 0) continue;") for x in loops)
