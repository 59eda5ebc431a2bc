"""Levels computed from an earlier level's set (KPlan::lev) on the CPU: for every
golden and central-node plan, the rows, bounds and exclusions that the engine
keeps on top of the base level's set -- restated here -- give the same candidate
sets as all of the level's constraints, over full bitmaps and, for plans that
read rows above their own position only, over bitmaps without mirrored bits.
The counts that follow from |C_2| alone (KPlan::closed) are checked the same
way.  The kernels are pinned by the GPU parity tests against the oracle."""
import random

import pytest

import beep_amd as B
from beep_amd import patterns as P


def plans():
    out = []
    for i, (_, e) in enumerate(P.central207()):
        for mode in (B.SGM, B.SGC):
            out.append((f"central{i}-{mode}", B.Plan.from_edges(*P.directed(e), mode)))
    for name in P.NAMES:
        for mode in (B.SGM, B.SGC):
            out.append((f"{name}-{mode}", B.Plan.from_edges(*P.directed(P.read_mtx_edges(name)), mode)))
    return [(n, p) for n, p in out if p.width >= 3]


def masks(p):
    qm = [set(q for q in p.qedge[l][1:]) for l in range(p.width)]
    sm = [set(s for s in p.sym[l] if s > 0) for l in range(p.width)]
    above = [set() for _ in range(p.width)]
    for l in range(1, p.width):
        for s in sm[l]:
            above[l] |= {s} | above[s]
    return qm, sm, above


def reduce_level(p, l, qm, sm, above, q, s, top):
    base, rq = 0, set(q)
    for b in range(2, min(l - 1, p.width - 2, top) + 1):
        if qm[b] <= q and sm[b] <= s and (not base or len(q - qm[b]) <= len(rq)):
            base, rq = b, q - qm[b]

    def implied(x):
        return any((t in s and x in above[t]) or (p.upper_rows and t in q and (t == x or x in above[t]))
                   for t in range(1, top))

    rs = {x for x in s if not (base and x in sm[base]) and not implied(x)}
    rx = {x for x in range(1, top) if not (x in s or x in q or (base and x < base) or implied(x))}
    return base, rq, rs, rx


def tail_summed(p, qm):
    return p.width >= 4 and (p.width - 2) not in qm[p.width - 1]


@pytest.mark.parametrize("seed", [1, 2])
def test_reduced_levels_give_the_full_levels_sets(seed):
    rng = random.Random(seed)
    for name, p in plans():
        qm, sm, above = masks(p)
        L, d = p.width, 11
        E = [[0] * d for _ in range(d)]
        for i in range(d):
            for j in range(i + 1, d):
                if rng.random() < 0.6:
                    E[i][j] = 1
                    E[j][i] = 0 if p.upper_rows else 1
        red = [None, None] + [reduce_level(p, l, qm, sm, above, qm[l], sm[l], l) for l in range(2, L)]
        # the last level: without x_{L-2}'s constraints, which are applied on top
        leaf_row, leaf_gt = L - 2 in qm[L - 1], L - 2 in sm[L - 1]
        if L >= 4:
            red[L - 1] = reduce_level(p, L - 1, qm, sm, above, qm[L - 1] - {L - 2}, sm[L - 1] - {L - 2}, L - 2)

        def full(l, x):
            return {i for i in range(d) if i not in x[1:l] and all(E[x[q]][i] for q in qm[l])
                    and all(i > x[s] for s in sm[l])}

        budget = [3000]

        def walk(l, x, sets):
            want = full(l, x)
            base, rq, rs, rx = red[l]
            got = {i for i in (sets[base] if base else range(d)) if all(E[x[q]][i] for q in rq)
                   and all(i > x[s] for s in rs) and all(i != x[t] for t in rx)}
            if l == L - 1 and L >= 4:
                y = x[L - 2]
                got = {i for i in got if (not leaf_row or E[y][i]) and (not leaf_gt or i > y)
                       and (leaf_row or leaf_gt or i != y)}
            assert got == want, (name, l, x)
            if l == L - 1:
                return
            for i in sorted(want):
                budget[0] -= 1
                if budget[0] < 0:
                    return
                walk(l + 1, x[:l] + [i], {**sets, l: got})

        for x1 in range(d):
            walk(2, [None, x1], {})


def test_counts_that_follow_from_c2():
    """kClosedPairs / kClosedOrdered / kClosedRow for 4-level plans with a summed last level."""
    rng = random.Random(3)
    seen = set()
    for name, p in plans():
        qm, sm, above = masks(p)
        L = p.width
        if L != 4 or not tail_summed(p, qm):
            continue
        gt = 2 in sm[3]
        base, rq, rs, rx = reduce_level(p, 3, qm, sm, above, qm[3], sm[3] - {2}, 2)
        if rq or rs:
            continue
        if base == 2 and not rx:
            kind = "pairs" if gt else "ordered"
        elif base == 0 and rx == {1} and not gt:
            kind = "row"
        else:
            continue
        seen.add(kind)
        for _ in range(20):
            d = rng.randint(3, 12)
            E = [[0] * d for _ in range(d)]
            for i in range(d):
                for j in range(i + 1, d):
                    if rng.random() < 0.5:
                        E[i][j] = 1
                        E[j][i] = 0 if p.upper_rows else 1
            for x1 in range(d):
                def cand(l, x):
                    return [i for i in range(d) if i not in x[1:l] and all(E[x[q]][i] for q in qm[l])
                            and all(i > x[s] for s in sm[l])]
                c2 = cand(2, [None, x1])
                want = sum(len(cand(3, [None, x1, x2])) for x2 in c2)
                c = len(c2)
                got = {"pairs": c * (c - 1) // 2, "ordered": c * (c - 1), "row": c * (d - 2)}[kind]
                assert got == want, (name, kind)
    assert {"pairs", "row"} <= seen
