"""The oracle's single stages pinned one by one.

Each stage of the restated schedule (seed matching, roles and the exact top
two, the mover threshold, isolated packing, two-hop pairing, LP proposals, the
afterburner, the repair gain bucket, repair destinations, donor eligibility
and receiver reservation) is run alone through the oracle's stage entry
points and checked against something it does not compute itself: hand-built
graphs with a known answer, brute-force dictionaries of affinities, exact cut
recounts, rational arithmetic, or the reference's own formula in the
reference's own words.  The hash constants and salts are checked against the
reference source text when the reference tree is present.
"""
import fractions
import math
import os
import re

import numpy as np
import pytest

from tests import graphs

REFERENCE = "/root/reference"
ORACLE_C = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle", "gp_oracle.c")


def mix32(x):
    """The reference's 32-bit finaliser (src/coarsen.cu:173-179)."""
    x &= 0xFFFFFFFF
    x ^= x >> 16
    x = (x * 0x7FEB352D) & 0xFFFFFFFF
    x ^= x >> 15
    x = (x * 0x846CA68B) & 0xFFFFFFFF
    return x ^ (x >> 16)


def role_salt(seed, level, round_):
    # src/coarsen.cu:743-745
    return (seed ^ ((level * 0x9E3779B9) & 0xFFFFFFFF) ^ ((round_ * 0x85EBCA6B) & 0xFFFFFFFF) ^ 0x27D4EB2D)


def tie_salt(seed, level, round_):
    # src/coarsen.cu:746-748
    return (seed ^ ((level * 0xC2B2AE35) & 0xFFFFFFFF) ^ ((round_ * 0x165667B1) & 0xFFFFFFFF) ^ 0xD3A2646C)


def rows(off, nbr, ew):
    """{v: [(u, w), ...]} from a CSR."""
    out = {}
    for v in range(len(off) - 1):
        out[v] = [(int(nbr[e]), 1 if ew is None else int(ew[e])) for e in range(off[v], off[v + 1])]
    return out


def cut_of(off, nbr, ew, lab):
    c = 0
    for v in range(len(off) - 1):
        for e in range(off[v], off[v + 1]):
            if lab[v] != lab[nbr[e]]:
                c += 1 if ew is None else int(ew[e])
    return c // 2


def path(weights, vw=None):
    n = len(weights) + 1
    return graphs.csr_from_edges(n, [(i, i + 1) for i in range(n - 1)], weights) + (
        np.ones(n, np.uint32) if vw is None else np.array(vw, np.uint32),)


# ------------------------------------------------- constants vs the reference
# (file, line, text that must appear on that line).  Each constant is also
# required in the oracle source.
REFERENCE_CONSTANTS = [
    ("src/coarsen.cu", 175, "0x7feb352dU"),
    ("src/coarsen.cu", 177, "0x846ca68bU"),
    ("src/refine.cu", 52, "0x7feb352dU"),
    ("src/refine.cu", 54, "0x846ca68bU"),
    ("src/coarsening/seed_matching.cuh", 8, "0x7feb352dU"),
    ("src/coarsen.cu", 520, "seed ^ (level * 0x9e3779b9U)"),
    ("src/coarsen.cu", 744, "0x9e3779b9U"),
    ("src/coarsen.cu", 745, "0x85ebca6bU) ^ 0x27d4eb2dU"),
    ("src/coarsen.cu", 747, "0xc2b2ae35U"),
    ("src/coarsen.cu", 748, "0x165667b1U) ^ 0xd3a2646cU"),
    ("src/refinement/incremental.cuh", 899, "maximum_edge<=1 ? 0.25 : 0.75"),
    ("src/refinement/incremental.cuh", 556, "max(2,min(49,25+static_cast<int>(ceil(log(-gain)/log(1.5)))))"),
    ("src/refinement/incremental.cuh", 549, "kBalanceBuckets=50"),
    ("src/refinement/incremental.cuh", 550, "kBalanceSections=16"),
    ("src/coarsening/seed_matching.cuh", 38, "degree > 1024"),
]


@pytest.mark.skipif(not os.path.isfile(os.path.join(REFERENCE, REFERENCE_CONSTANTS[0][0])),
                    reason="reference tree not present")
def test_constants_match_reference_source():
    oracle_text = open(ORACLE_C).read().lower().replace(" ", "")
    for rel, line, text in REFERENCE_CONSTANTS:
        with open(os.path.join(REFERENCE, rel)) as f:
            lines = f.read().split("\n")
        assert text in lines[line - 1], (rel, line, text, lines[line - 1])
        for const in re.findall(r"0x[0-9a-f]+", text):
            assert const.lower() in oracle_text, const
    # the Python finaliser used by these checks is the reference's, line by line
    body = open(os.path.join(REFERENCE, "src/coarsen.cu")).read().split("\n")[172:179]
    assert [l.strip() for l in body[1:6]] == ["x ^= x >> 16;", "x *= 0x7feb352dU;", "x ^= x >> 15;",
                                              "x *= 0x846ca68bU;", "return x ^ (x >> 16);"], body


# ------------------------------------------------------------ seed matching
def test_seed_match_takes_the_heaviest_edge(og):
    off, nbr, ew, vw = path([1, 5, 1])
    roots, count = og.seed_match(off, nbr, ew, vw, cap=10, salt=0)
    assert roots.tolist() == [0, 1, 1, 3] and count == 3


def test_seed_match_capacity_excludes_pairs(og):
    # 1 and 2 would pair over the weight-5 edge but 3 + 3 > cap 5, so each
    # falls back to its light edge and the pairs are (0,1) and (2,3).
    off, nbr, ew, vw = path([1, 5, 1], vw=[1, 3, 3, 1])
    roots, count = og.seed_match(off, nbr, ew, vw, cap=5, salt=0)
    assert roots.tolist() == [0, 0, 2, 2] and count == 2
    # A vertex heavier than the capacity pairs with nobody.
    roots, _ = og.seed_match(off, nbr, ew, np.array([1, 6, 1, 1], np.uint32), cap=5, salt=0)
    assert roots.tolist() == [0, 1, 2, 2]


def test_seed_match_needs_a_mutual_choice(og):
    # Star: the centre picks its heaviest leaf; every leaf picks the centre;
    # only the mutual pair merges.
    off, nbr, ew = graphs.csr_from_edges(5, [(0, 1), (0, 2), (0, 3), (0, 4)], [4, 3, 2, 1])
    roots, count = og.seed_match(off, nbr, ew, np.ones(5, np.uint32), cap=10, salt=7)
    assert roots.tolist() == [0, 0, 2, 3, 4] and count == 4


def test_seed_match_degree_limit(og):
    # A row longer than 1024 entries makes no choice (seed_matching.cuh:38).
    for leaves, merged in ((1024, True), (1025, False)):
        w = [1] * leaves
        w[0] = 9
        off, nbr, ew = graphs.csr_from_edges(leaves + 1, [(0, i) for i in range(1, leaves + 1)], w)
        roots, _ = og.seed_match(off, nbr, ew, np.ones(leaves + 1, np.uint32), cap=10, salt=0)
        assert (roots[1] == 0) == merged


def test_seed_match_ties_by_pair_hash(og):
    # Unit weights, vertex 0 with two leaves: the centre's choice between the
    # two equal edges is the larger mix32(lo ^ mix32(hi ^ salt)), then the
    # larger id; the leaves both choose 0.
    off, nbr, ew = graphs.csr_from_edges(3, [(0, 1), (0, 2)])
    outcomes = set()
    for salt in range(64):
        h1, h2 = mix32(0 ^ mix32(1 ^ salt)), mix32(0 ^ mix32(2 ^ salt))
        pick = 1 if (h1, 1) > (h2, 2) else 2
        roots, _ = og.seed_match(off, nbr, ew, np.ones(3, np.uint32), cap=10, salt=salt)
        want = [0, 0, 2] if pick == 1 else [0, 1, 0]
        assert roots.tolist() == want, salt
        outcomes.add(pick)
    assert outcomes == {1, 2}


def test_seed_match_is_order_free_and_mutual(og):
    # The result does not depend on the order of entries in a row, and every
    # cluster has at most two vertices joined by an edge.
    off, nbr, ew = graphs.random_graph(300, 900, seed=3, max_weight=3)
    vw = np.random.default_rng(1).integers(1, 4, 300).astype(np.uint32)
    roots, count = og.seed_match(off, nbr, ew, vw, cap=6, salt=99)
    rng = np.random.default_rng(2)
    nbr2, ew2 = nbr.copy(), ew.copy()
    for v in range(300):
        p = rng.permutation(off[v + 1] - off[v]) + off[v]
        nbr2[off[v]:off[v + 1]], ew2[off[v]:off[v + 1]] = nbr[p], ew[p]
    roots2, _ = og.seed_match(off, nbr2, ew2, vw, cap=6, salt=99)
    assert np.array_equal(roots, roots2)
    adj = rows(off, nbr, ew)
    assert count == len(set(roots.tolist()))
    for v in range(300):
        r = int(roots[v])
        if r != v:
            assert r < v and roots[r] == r and any(u == r for u, _ in adj[v])
            assert int(vw[v]) + int(vw[r]) <= 6


# -------------------------------------------------------- mover threshold
def test_mover_threshold_closed_form(og):
    # floor(2^32 * min(1/2, max(0, c - ceil(n/2)) / c)) (coarsen.cu:984-990)
    for n, c in ((1000, 1000), (1001, 1001), (1000, 700), (1000, 500), (1000, 400), (65536, 60000),
                 (4194304, 3000001), (12345, 9876)):
        frac = min(fractions.Fraction(1, 2), fractions.Fraction(max(0, c - (n + 1) // 2), c))
        assert og.mover_threshold(c, n) == math.floor(frac * 2 ** 32), (n, c)


# ------------------------------------------------ roles and exact top two
def _random_clustering(n, rng):
    clusters = np.arange(n, dtype=np.int32)
    for v in range(n):
        if rng.random() < 0.3:
            clusters[v] = clusters[int(rng.integers(0, v + 1))]
    return clusters


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_proposals_match_affinity_dictionary(og, seed):
    rng = np.random.default_rng(seed)
    n = 120
    off, nbr, ew = graphs.random_graph(n, 500, seed=seed + 10, max_weight=4)
    vw = rng.integers(1, 4, n).astype(np.uint32)
    clusters = _random_clustering(n, rng)
    cw = np.bincount(clusters, weights=vw, minlength=n).astype(np.uint64)
    cap, level, rnd, s = 9, 2, 1, 17
    threshold = og.mover_threshold(int((cw > 0).sum()), n)
    adj = rows(off, nbr, ew)
    for filter_roles, need_regret in ((1, 1), (1, 0), (0, 0)):
        got = og.proposals(off, nbr, ew, vw, clusters, cw, cap, s, level, rnd, filter_roles, threshold, need_regret)
        # roles: singleton roots whose hash falls below the threshold
        salt = role_salt(s, level, rnd)
        singleton = [clusters[v] == v and cw[v] == vw[v] for v in range(n)]
        roles = [singleton[v] and (not filter_roles or mix32(v ^ salt) < threshold) for v in range(n)]
        assert got["roles"].astype(bool).tolist() == roles
        tsalt = tie_salt(s, level, rnd)
        for v in range(n):
            src = int(clusters[v])
            if not roles[src]:
                assert got["proposals"][v] == 0x7FFFFFFF
                continue
            aff = {}
            for u, w in adj[v]:
                aff[int(clusters[u])] = aff.get(int(clusters[u]), 0) + w
            current = aff.pop(src, 0)
            cand = {}
            for c, a in aff.items():
                if filter_roles and (roles[c] or not (0 < cw[c] <= cap and cw[src] <= cap - cw[c])):
                    continue
                cand[c] = a
            best = max(cand.values(), default=0)
            if best <= current:
                assert got["proposals"][v] == 0x7FFFFFFF, v
                continue
            key = lambda c: (mix32(v ^ mix32(c) ^ tsalt), 0xFFFFFFFF - c)
            target = max((c for c in cand if cand[c] == best), key=key)
            assert got["proposals"][v] == target, (v, cand)
            assert got["gains"][v] == best - current
            assert got["ties"][v] == mix32(v ^ mix32(target) ^ tsalt)
            if filter_roles and need_regret:
                rest = sorted(cand.values())
                rest.remove(best)
                second = max(rest, default=0)
                assert got["regret"][v] == best - second, (v, cand)


def test_role_fraction_follows_threshold(og):
    # Movers are the singleton roots under the threshold: about frac * n of them.
    n = 20000
    off = np.zeros(n + 1, np.int32)
    clusters = np.arange(n, dtype=np.int32)
    cw = np.ones(n, np.uint64)
    vw = np.ones(n, np.uint32)
    for c in (20000, 15000, 11000):
        t = og.mover_threshold(c, n)
        got = og.proposals(off, np.zeros(0, np.int32), None, vw, clusters, cw, 4, 3, 0, 0, 1, t, 1)
        p = t / 2 ** 32
        movers = int(got["roles"].sum())
        assert abs(movers - p * n) < 5 * math.sqrt(n * p * (1 - p)) + 1, (c, movers, p * n)


# ---------------------------------------------------------- isolated packing
def test_pack_isolated_unit_bins(og):
    # Ten isolated vertices among others, cap 4: bins of the weight line hold
    # 4, 4 and 2 vertices, each joining its smallest member.
    n = 14
    edges = [(0, 1), (1, 2), (2, 3)]
    off, nbr, _ = graphs.csr_from_edges(n, edges)
    clusters = np.arange(n, dtype=np.int32)
    cw = np.ones(n, np.uint64)
    got, gw, ran = og.pack_isolated(off, np.ones(n, np.uint32), 4, clusters, cw)
    assert ran
    assert got[:4].tolist() == [0, 1, 2, 3]
    assert got[4:].tolist() == [4, 4, 4, 4, 8, 8, 8, 8, 12, 12]
    assert gw[[4, 8, 12]].tolist() == [4, 4, 2] and int(gw.sum()) == n


def test_pack_isolated_straddlers_stay_alone(og):
    off = np.zeros(7, np.int32)
    for w, want in (([3, 3, 3], [0, 1, 2]),                    # prefixes 3,6,9: 1 and 2 straddle edges
                    ([2, 2, 1, 3, 1, 1], [0, 0, 2, 2, 4, 4])):  # three bins of weight 4
        n = len(w)
        got, gw, _ = og.pack_isolated(off[:n + 1], np.array(w, np.uint32), 4, np.arange(n, dtype=np.int32),
                                      np.array(w, np.uint64))
        assert got.tolist() == want, w
        assert int(gw.max()) <= 4


def test_pack_isolated_interval_rule(og):
    rng = np.random.default_rng(8)
    for trial in range(20):
        n = 60
        w = rng.integers(1, 6, n)
        cap = int(rng.integers(5, 15))
        got, gw, _ = og.pack_isolated(np.zeros(n + 1, np.int32), w.astype(np.uint32), cap,
                                      np.arange(n, dtype=np.int32), w.astype(np.uint64))
        p, rep, want = 0, {}, list(range(n))
        bins = []
        for v in range(n):
            lo, hi = p, p + int(w[v])
            p = hi
            bins.append(lo // cap if lo // cap == (hi - 1) // cap else None)
        for v in range(n):
            if bins[v] is not None:
                rep.setdefault(bins[v], v)
                want[v] = rep[bins[v]]
        assert got.tolist() == want
        assert -(-p // cap) >= len(rep)  # at most ceil(W / C) bins
        assert int(gw.max()) <= cap


def test_pack_isolated_needs_two(og):
    _, _, ran = og.pack_isolated(np.zeros(2, np.int32), np.ones(1, np.uint32), 4, np.zeros(1, np.int32),
                                 np.ones(1, np.uint64))
    assert not ran


# -------------------------------------------------------------- two-hop
def _hub_leaves():
    # Cluster {0, 1} (not a singleton) and four leaves hanging off vertex 0
    # with edge weights 5, 4, 3, 2: each leaf's favourite is cluster 0 with
    # gain equal to its edge weight.
    off, nbr, ew = graphs.csr_from_edges(6, [(0, 1), (0, 2), (0, 3), (0, 4), (0, 5)], [1, 5, 4, 3, 2])
    clusters = np.array([0, 0, 2, 3, 4, 5], np.int32)
    cw = np.array([2, 0, 1, 1, 1, 1], np.uint64)
    return off, nbr, ew, np.ones(6, np.uint32), clusters, cw


def test_two_hop_pairs_by_gain(og):
    off, nbr, ew, vw, clusters, cw = _hub_leaves()
    got, gw = og.two_hop(off, nbr, ew, vw, clusters, cw, cap=2, seed=0, level=0, budget=10)
    # order by gain: 2, 3, 4, 5; the 2nd joins the 1st and the 4th the 3rd
    assert got.tolist() == [0, 0, 2, 2, 4, 4]
    assert gw.tolist() == [2, 0, 2, 0, 2, 0]


def test_two_hop_budget_and_capacity(og):
    off, nbr, ew, vw, clusters, cw = _hub_leaves()
    got, _ = og.two_hop(off, nbr, ew, vw, clusters, cw, cap=2, seed=0, level=0, budget=1)
    assert got.tolist() == [0, 0, 2, 2, 4, 5]
    got, _ = og.two_hop(off, nbr, ew, vw, clusters, cw, cap=1, seed=0, level=0, budget=10)
    assert got.tolist() == clusters.tolist()


# ------------------------------------------------------------ LP proposals
def _lp_brute(adj, n, k, lab, locks, vw, loads, cap, prices, filt):
    targets, gains = [-1] * n, [None] * n
    for v in range(n):
        if locks[v]:
            continue
        a = [0] * k
        for u, w in adj[v]:
            a[lab[u]] += w
        s = lab[v]
        cur, total = a[s], sum(a)
        if cur == total:
            continue
        best, target, score_best = 0, -1, None
        for p in range(k):
            if p == s or not a[p]:
                continue
            if prices is not None:
                slack = cap - int(loads[p])
                cost = float(prices[p]) * float(int(vw[v]) - slack) if int(vw[v]) > slack else 0.0
                score = float(a[p]) - cost
                if target < 0 or score > score_best:
                    best, target, score_best = a[p], p, score
            elif target < 0 or a[p] > best:
                best, target = a[p], p
        if target >= 0 and (best >= cur or cur - best < math.floor(fractions.Fraction(filt) * cur)):
            targets[v], gains[v] = target, best - cur
    return targets, gains


@pytest.mark.parametrize("weighted,priced", [(False, False), (True, False), (True, True), (False, True)])
def test_lp_proposals_brute_force(og, weighted, priced):
    rng = np.random.default_rng(21 + 2 * weighted + priced)
    n, k = 150, 5
    off, nbr, ew = graphs.random_graph(n, 600, seed=4, max_weight=6 if weighted else 1)
    ew = ew if weighted else None
    vw = rng.integers(1, 5, n).astype(np.uint32)
    lab = rng.integers(0, k, n).astype(np.int32)
    locks = (rng.random(n) < 0.2).astype(np.int32)
    loads = np.bincount(lab, weights=vw, minlength=k).astype(np.uint64)
    cap = int(loads.max()) + 3
    prices = rng.random(k) * 3 if priced else None
    filt = 0.75 if weighted else 0.25
    targets, gains, locks_after, count = og.lp_propose(off, nbr, ew, vw, k, lab, locks, loads, cap, prices, filt)
    want_t, want_g = _lp_brute(rows(off, nbr, ew), n, k, lab.tolist(), locks.tolist(), vw, loads, cap, prices, filt)
    assert targets.tolist() == want_t
    for v in range(n):
        if want_t[v] >= 0:
            assert gains[v] == want_g[v], v
    assert count == sum(t >= 0 for t in want_t) and not locks_after.any()


def test_lp_filter_examples(og):
    # Vertex 0 in part 0 with own-part weight 8: a move to a part of weight 7
    # is kept for filter 0.25 only when 8 - 7 < floor(0.25 * 8) = 2 (kept),
    # and one to a part of weight 6 is dropped (8 - 6 = 2, not < 2); with 0.75
    # (weighted graphs) the limit is floor(6) = 6.
    for other, filt, want in ((7, 0.25, 1), (6, 0.25, -1), (3, 0.75, 1), (2, 0.75, -1)):
        off, nbr, ew = graphs.csr_from_edges(3, [(0, 1), (0, 2)], [8, other])
        lab = np.array([0, 0, 1], np.int32)
        t, g, _, _ = og.lp_propose(off, nbr, ew, np.ones(3, np.uint32), 2, lab, np.zeros(3, np.int32),
                                   np.array([2, 1], np.uint64), 10, None, filt)
        assert t[0] == want, (other, filt)
        if want >= 0:
            assert g[0] == other - 8


def test_lp_ties_take_the_lowest_part(og):
    off, nbr, ew = graphs.csr_from_edges(4, [(0, 1), (0, 2), (0, 3)], [2, 2, 2])
    lab = np.array([0, 3, 1, 2], np.int32)
    t, g, _, _ = og.lp_propose(off, nbr, ew, np.ones(4, np.uint32), 4, lab, np.zeros(4, np.int32),
                               np.ones(4, np.uint64), 5, None, 0.75)
    assert t[0] == 1 and g[0] == 2


# ------------------------------------------------------------- afterburner
@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_afterburner_equals_sequential_recount(og, seed):
    # g~_v is the exact cut change of moving v after every candidate ranked
    # before it (larger gain, or equal gain and smaller id); keep iff >= 0.
    rng = np.random.default_rng(seed)
    n, k = 80, 4
    off, nbr, ew = graphs.random_graph(n, 300, seed=seed + 30, max_weight=5)
    lab = rng.integers(0, k, n).astype(np.int32)
    vw = np.ones(n, np.uint32)
    loads = np.bincount(lab, minlength=k).astype(np.uint64)
    targets, gains, _, _ = og.lp_propose(off, nbr, ew, vw, k, lab, np.zeros(n, np.int32), loads, n, None, 0.75)
    keep = og.afterburner(off, nbr, ew, vw, k, lab, loads, n, None, targets, gains)
    cand = [v for v in range(n) if targets[v] >= 0]
    assert len(cand) > 10
    for v in cand:
        before = lab.copy()
        for u in cand:
            if gains[u] > gains[v] or (gains[u] == gains[v] and u < v):
                before[u] = targets[u]
        after = before.copy()
        after[v] = targets[v]
        delta = cut_of(off, nbr, ew, before) - cut_of(off, nbr, ew, after)
        assert bool(keep[v]) == (delta >= 0), (v, delta)
    assert not keep[[v for v in range(n) if targets[v] < 0]].any()


def test_afterburner_price_adjustment(og):
    # Vertex 0 (part 0) gains 0 by moving to part 1; with prices the move is
    # kept iff cost(leave 0) - cost(enter 1) >= 0.
    off, nbr, ew = graphs.csr_from_edges(3, [(0, 1), (0, 2)], [3, 3])
    lab = np.array([0, 0, 1], np.int32)
    vw = np.array([4, 1, 1], np.uint32)
    targets = np.array([1, -1, -1], np.int32)
    gains = np.array([0, 0, 0], np.int64)
    for loads, prices, want in (([9, 8], [1.0, 1.0], True),    # slack 1 vs 2: cost 3 - 2 >= 0
                                ([8, 9], [1.0, 1.0], False),   # slack 2 vs 1: cost 2 - 3 < 0
                                ([8, 9], [2.0, 1.0], True)):   # 4 - 3 >= 0
        keep = og.afterburner(off, nbr, ew, vw, 2, lab, np.array(loads, np.uint64), 10,
                              np.array(prices), targets, gains)
        assert bool(keep[0]) == want, (loads, prices)


# -------------------------------------------------------- repair: buckets
def _near_power(x):
    j = math.log(x) / math.log(1.5)
    return abs(j - round(j)) < 1e-9


def test_gain_bucket_formula_sweep(og):
    # balance_gain_bucket (incremental.cuh:553-557) on a dense sweep away from
    # the exact powers of 1.5.
    assert og.gain_bucket(3.0) == 0 and og.gain_bucket(1e-300) == 0
    assert og.gain_bucket(0.0) == 1 and og.gain_bucket(-0.0) == 1
    for x in np.geomspace(1e-9, 1e9, 20001):
        x = float(x)
        if _near_power(x):
            continue
        want = max(2, min(49, 25 + math.ceil(math.log(x) / math.log(1.5))))
        assert og.gain_bucket(-x) == want, x


def test_gain_bucket_exact_powers(og):
    # 1.5^j (j >= 0) is exact in double: -1.5^j falls in bucket 25 + j, and
    # the next double above it in the next bucket (clamped to 49).
    for j in range(0, 24):
        x = 1.5 ** j
        assert fractions.Fraction(x) == fractions.Fraction(3, 2) ** j
        assert og.gain_bucket(-x) == min(49, 25 + j), j
        assert og.gain_bucket(-np.nextafter(x, np.inf)) == min(49, 26 + j), j
    assert og.gain_bucket(-1e30) == 49 and og.gain_bucket(-1e-30) == 2


# -------------------------------------------------- repair: destinations
def _dest_brute(adj, k, lab, vw, loads, cap, v):
    s = lab[v]
    w = int(vw[v])
    a = [0] * k
    for u, x in adj[v]:
        if u != v:
            a[lab[u]] += x
    fits = [p for p in range(k) if p != s and int(loads[p]) < cap and w <= cap - int(loads[p])]
    if a[s] != sum(a):
        best = None
        for p in fits:
            if a[p] and (best is None or (a[p], cap - int(loads[p])) > (a[best], cap - int(loads[best]))):
                best = p
        if best is not None:
            return best
    total = sum(cap - int(loads[p]) for p in fits)
    if not total:
        return -1
    ticket = mix32(v) % total
    for p in fits:
        if ticket < cap - int(loads[p]):
            return p
        ticket -= cap - int(loads[p])


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_repair_destination_brute_force(og, seed):
    rng = np.random.default_rng(seed)
    n, k = 100, 6
    off, nbr, ew = graphs.random_graph(n, 250, seed=seed + 50, max_weight=4)
    vw = rng.integers(1, 6, n).astype(np.uint32)
    lab = rng.integers(0, k, n).astype(np.int32)
    loads = np.bincount(lab, weights=vw, minlength=k).astype(np.uint64)
    cap = int(np.sort(loads)[k // 2]) + 2
    adj = rows(off, nbr, ew)
    for v in range(n):
        d, _, _ = og.repair_destination(off, nbr, ew, vw, k, lab, loads, cap, v)
        assert d == _dest_brute(adj, k, lab.tolist(), vw, loads, cap, v), v


# ----------------------------------------- repair: eligibility, reservation
def _repair_instance(seed, n=120, k=5):
    rng = np.random.default_rng(seed)
    off, nbr, ew = graphs.random_graph(n, 300, seed=seed + 70, max_weight=4)
    vw = rng.integers(1, 6, n).astype(np.uint32)
    lab = rng.integers(0, k, n).astype(np.int32)
    lab[rng.random(n) < 0.3] = 0  # part 0 overloaded
    loads = np.bincount(lab, weights=vw, minlength=k).astype(np.uint64)
    cap = int(np.sort(loads)[-2]) + 1
    return off, nbr, ew, vw, lab, loads, cap, k


@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_repair_eligibility_prefix(og, seed):
    # A donor is eligible iff the weight of its part's donors ordered before
    # it -- lower bucket, or same bucket and smaller id -- is below the excess.
    off, nbr, ew, vw, lab, loads, cap, k = _repair_instance(seed)
    got = og.repair_iteration(off, nbr, ew, vw, k, lab, loads, cap)
    adj = rows(off, nbr, ew)
    for s in range(k):
        donors = [v for v in range(len(lab)) if got["bucket"][v] >= 0 and lab[v] == s]
        if int(loads[s]) <= cap:
            assert not donors
            continue
        excess = int(loads[s]) - cap
        before = 0
        for v in sorted(donors, key=lambda v: (int(got["bucket"][v]), v)):
            assert bool(got["eligible"][v]) == (before < excess), (s, v, before, excess)
            before += int(vw[v])
        for v in donors:
            # bucket = part * 800 + gain bucket * 16 + mix32(v) % 16, gain per unit of relief
            d = int(got["first_choice"][v])
            assert d == _dest_brute(adj, k, lab.tolist(), vw, loads, cap, v)
            a = [0] * k
            for u, x in adj[v]:
                a[lab[u]] += x
            gpw = (a[d] - a[s]) / min(int(vw[v]), excess)
            assert got["bucket"][v] == s * 800 + og.gain_bucket(gpw) * 16 + mix32(v) % 16


def test_repair_eligibility_hand_example(og):
    # Part 0 holds four isolated vertices of weight 2 (load 8, cap 5, excess
    # 3); all gains are 0 (bucket 1), so donors order by hash section then
    # id: the first two (prefix 0 and 2 < 3) are eligible, the rest not.
    n = 6
    off = np.zeros(n + 1, np.int32)
    vw = np.array([2, 2, 2, 2, 1, 1], np.uint32)
    lab = np.array([0, 0, 0, 0, 1, 2], np.int32)
    loads = np.array([8, 1, 1], np.uint64)
    got = og.repair_iteration(off, np.zeros(0, np.int32), None, vw, 3, lab, loads, 5)
    order = sorted(range(4), key=lambda v: (mix32(v) % 16, v))
    assert [bool(got["eligible"][v]) for v in order] == [True, True, False, False]
    assert all(got["bucket"][v] == 16 + mix32(v) % 16 for v in range(4))


@pytest.mark.parametrize("seed", [0, 1, 2, 3, 4, 5])
def test_reservation_respects_receiver_slack(og, seed):
    off, nbr, ew, vw, lab, loads, cap, k = _repair_instance(seed)
    got = og.repair_iteration(off, nbr, ew, vw, k, lab, loads, cap)
    recv = got["receiver"]
    moved = recv >= 0
    assert moved.any()
    assert np.all(got["eligible"][moved])
    assert np.all(recv[moved] != lab[moved])
    incoming = np.bincount(recv[moved], weights=vw[moved], minlength=k)
    for p in range(k):
        slack = cap - int(loads[p]) if int(loads[p]) < cap else 0
        assert incoming[p] <= slack, (p, incoming[p], slack)
    # donors leave overloaded parts only
    for s in range(k):
        out = int(vw[moved & (lab == s)].sum())
        assert out == 0 or int(loads[s]) > cap


def test_reservation_tickets_in_vertex_order(og):
    # Isolated donors of weights 2, 2, 2, 1 in part 0 (load 7, cap 4, excess
    # 3) and two receivers of slack 3 (part 1) and 4 (part 2).  The
    # hash routing sends each donor somewhere first; per receiver the
    # requests are admitted in vertex order while they end within the slack,
    # and a rejected donor tries the other receiver in the next attempt.
    n = 5
    off = np.zeros(n + 1, np.int32)
    vw = np.array([2, 2, 2, 1, 1], np.uint32)
    lab = np.array([0, 0, 0, 0, 1], np.int32)
    loads = np.array([7, 1, 0], np.uint64)
    cap = 4
    got = og.repair_iteration(off, np.zeros(0, np.int32), None, vw, 3, lab, loads, cap)
    first = got["first_choice"]
    slack = {1: 3, 2: 4}
    used = {1: 0, 2: 0}
    want = [-1] * n
    pending = [v for v in range(4) if got["eligible"][v]]
    choice = {v: int(first[v]) for v in pending}
    tried = {v: set() for v in pending}
    for attempt in range(3):
        snapshot = dict(used)
        if attempt:
            choice = {}
            for v in pending:
                opts = [p for p in (1, 2) if p not in tried[v] and slack[p] - snapshot[p] >= int(vw[v])]
                choice[v] = max(opts, key=lambda p: (0, slack[p] - snapshot[p], -p)) if opts else -1
        if all(c < 0 for c in choice.values()):
            break
        batch = {1: 0, 2: 0}
        for v in sorted(choice):
            t = choice[v]
            if t < 0:
                continue
            tried[v].add(t)
            begin = used[t] + batch[t]
            batch[t] += int(vw[v])
            if begin + int(vw[v]) <= slack[t]:
                want[v] = t
        for p in (1, 2):
            used[p] += batch[p]
        pending = [v for v in pending if want[v] < 0]
    assert got["receiver"].tolist() == want
