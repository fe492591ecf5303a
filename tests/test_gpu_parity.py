"""GPU parity: every stage through the C ABI against the CPU oracle, bit-exact.

Inputs are seeded; sizes are chosen so the oracle finishes in seconds while still covering
the kernels' special paths (LDS vs global tables, small vs large hedges, cycles in pairing)."""
import ctypes as C

import numpy as np
import pytest

import gen
import gpu_stages as G
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # name, n, e, max_size, src_prob, max_src, dup, weights
    ("hgr_small", 300, 400, 6, 0.0, 1, 0.0, "unit"),
    ("hgr_wide", 2000, 1500, 40, 0.0, 1, 0.0, "int"),
    ("srcs", 1500, 1800, 12, 0.9, 3, 0.3, "int"),
    ("float_w", 800, 900, 9, 0.5, 2, 0.2, "float"),
    ("big_hedges", 3000, 120, 1200, 0.3, 2, 0.0, "unit"),
]


def make(case, rng):
    _, n, e, ms, sp, mxs, dup, w = case
    raw = O.HG(*gen.random_hypergraph(n, e, rng, max_size=ms, src_prob=sp, max_src=mxs, dup_prob=dup, weights=w))
    return O.dedup(raw)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_touching(dev, case, rng):
    hg = make(case, rng)
    L = G.Level(dev, hg)
    toff, tch, inb = L.build_touching()
    ro, rt, ri = O.touching(hg)
    assert np.array_equal(toff, ro) and np.array_equal(tch, rt) and np.array_equal(inb, ri)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_neighbors(dev, case, rng):
    hg = make(case, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    noff, nbr, _, _ = G.neighbors(dev, L)
    ro, rt, _ = O.touching(hg)
    eo, en = O.neighbors(hg, ro, rt)
    assert np.array_equal(noff, eo) and np.array_equal(nbr, en)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("cnc", [1, 4, 16])
def test_candidates(dev, case, cnc, rng):
    hg = make(case, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = rng.integers(1, 4, size=hg.n).astype(np.uint32)
    for omega, delta in ((6, 2**31 - 1), (4, 40)):
        pairs, scores, *_ = G.candidates(dev, L, sizes, cnc, omega, delta)
        ep, es = O.candidates(hg, ro, rt, ri, sizes, cnc, omega, delta)
        assert np.array_equal(pairs, ep), f"pairs differ (omega={omega}, delta={delta})"
        assert np.array_equal(scores, es)


def tier_graph(n, big_sizes, n_small, rng):
    """Mostly small hedges plus a few very large ones, so that their pins need candidate
    tables of every size class (LDS hash, LDS indexed by node id, HBM hash, HBM indexed)."""
    off, pins, srcc = [0], [], []
    for sz in big_sizes:
        nodes = rng.choice(n, size=sz, replace=False)
        pins.extend(int(x) for x in nodes)
        off.append(len(pins))
        srcc.append(1)
    for _ in range(n_small):
        sz = int(rng.integers(2, 6))
        nodes = rng.choice(n, size=sz, replace=False)
        pins.extend(int(x) for x in nodes)
        off.append(len(pins))
        srcc.append(int(rng.integers(0, 2)))
    e = len(srcc)
    w = (rng.random(e) * 3 + 0.5).astype(np.float32)
    return O.dedup(O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32), w))


@pytest.mark.parametrize("n,big,deltas", [
    (40000, (2500, 5000, 9000), (2**31 - 1, 30)),  # LDS hash (big), HBM hash (heavy)
    (20000, (9000,), (2**31 - 1, 30)),             # LDS indexed by id; HBM indexed by id with inbound counts
])
def test_candidates_table_tiers(dev, n, big, deltas, rng):
    hg = tier_graph(n, big, 3000, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = rng.integers(1, 3, size=hg.n).astype(np.uint32)
    for delta in deltas:
        pairs, scores, *_ = G.candidates(dev, L, sizes, 16, 6, delta)
        ep, es = O.candidates(hg, ro, rt, ri, sizes, 16, 6, delta)
        assert np.array_equal(pairs, ep), f"pairs differ (delta={delta})"
        assert np.array_equal(scores, es), f"scores differ (delta={delta})"


@pytest.mark.parametrize("pins", [1, 1023, 1024, 1025, 262143, 262144, 262145, 300001])
def test_construction_by_pins(dev, pins, rng):
    """Pin counts at the edges of the tiles of pins: hedges without pins in runs, at tile edges and at
    both ends, hedges of a few pins, and hedges of several tiles."""
    n, lens = max(2, pins // 8), [0, 0]
    left = pins
    while left:
        kind = rng.random()
        ln = 0 if kind < 0.2 else int(rng.integers(1, 9)) if kind < 0.999 else int(rng.integers(500, 20000))
        if left in (pins, pins - 1024, pins - 4096):
            lens += [0] * 5
        ln = min(ln, left, 1024 - (pins - left) if pins - left < 1024 else left)  # a hedge starts at pin 1024
        lens.append(ln)
        left -= ln
    lens = np.array(lens + [0, 0, 0])
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    p = rng.integers(0, n, size=pins).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 3, size=len(lens)), lens).astype(np.uint32)
    hg = O.HG(n, off, p, srcc, np.ones(len(lens), np.float32))
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    assert np.array_equal(dev.download(L.toff, n + 1, np.uint64), ro)
    assert np.array_equal(dev.download(L.tch, pins, np.uint32), rt)
    assert np.array_equal(dev.download(L.inb, n, np.uint32), ri)
    groups = rng.integers(0, n // 2, size=n).astype(np.uint32)
    groups[:2] = [0, n // 2 - 1]
    choff, cp, csrcc, *_ = G.coarsen_hedges(dev, L, dev.upload(groups))
    eo, ep, es = O.coarsen_hedges(hg, groups)
    assert np.array_equal(choff, eo) and np.array_equal(cp, ep) and np.array_equal(csrcc, es)


@pytest.mark.parametrize("short", [0, 300])
def test_candidates_long_hedges(dev, short, rng):
    """Hedges at the edges of the steps of the hedge-by-hedge traversal (64 pins a step, four steps
    a batch) with hubs in all of them, beside `short` hedges of a few pins that mix into the hubs'
    lists; contributions of zero, sources and destinations."""
    n, hubs = 9000, np.array([0, 17, 4321, 8998, 8999])
    lens = [128, 129, 191, 192, 193, 255, 256, 257, 258, 319, 320, 321, 511, 512, 513, 767, 769, 1024, 1025] * 4
    off, pins, srcc = [0], [], []
    for i, ln in enumerate(lens + [3, 5, 8] * (short // 3)):
        h = hubs[: 2 if ln < 9 else 5]
        row = np.concatenate([h, rng.choice(np.setdiff1d(np.arange(n), hubs), size=ln - len(h), replace=False)])
        pins.extend(int(x) for x in rng.permutation(row))
        off.append(len(pins))
        srcc.append(i % 3 if ln > 3 else 1)
    w = rng.random(len(srcc)).astype(np.float32)
    w[::4] = 0.0
    hg = O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32), w)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    for delta in (2**31 - 1, 40):
        pairs, scores, *_ = G.candidates(dev, L, sizes, 16, 6, delta)
        ep, es = O.candidates(hg, ro, rt, ri, sizes, 16, 6, delta)
        assert np.array_equal(pairs, ep) and np.array_equal(scores, es), delta


@pytest.mark.parametrize("delta", [2**31 - 1, 40])
def test_candidates_long_hedges_optimistic(dev, delta, rng):
    """Nodes whose tables are tried in LDS, with 1,024 touching hedges (64 a wave) of one length on
    either side of the line to the hedge-by-hedge traversal, and one hub with hedges of all of them."""
    n, lens = 50000, [128, 144, 159, 160, 161, 193]
    off, pins = [0], []
    for h, ln in enumerate(lens):
        pool = rng.choice(np.arange(10, n), size=4000, replace=False)  # distinct neighbours that fit
        for i in range(1024):
            row = np.concatenate([[h], [7] * (i % 16 == 0), rng.choice(pool, size=ln, replace=False)])[:ln]
            pins.extend(int(x) for x in rng.permutation(row))
            off.append(len(pins))
    e = len(off) - 1
    hg = O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.arange(e).astype(np.uint32) % 2,
              rng.random(e).astype(np.float32))
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    pairs, scores, *_ = G.candidates(dev, L, sizes, 16, 6, delta)
    ep, es = O.candidates(hg, ro, rt, ri, sizes, 16, 6, delta)
    assert np.array_equal(pairs, ep) and np.array_equal(scores, es)


@pytest.mark.parametrize("delta", [2**31 - 1, 1])
def test_candidates_of_two_billion_visits(dev, delta, rng):
    """A node of more than 2^31 visits on a level indexed by node id: its incidence list names one hedge
    of all nodes over and over (the stage takes the list as it is), with and without shared-inbound counts."""
    n, times = 16384, 131100
    assert times * (n - 1) >= 1 << 31
    hg = O.HG(n, np.array([0, n], np.uint64), rng.permutation(n).astype(np.uint32), np.ones(1, np.uint32),
              np.array([0.8], np.float32))
    L = G.Level(dev, hg)
    toff = np.full(n + 1, times, np.uint64)
    toff[0] = 0
    tch, inb = np.zeros(times, np.uint32), np.zeros(n, np.uint32)
    L.tch, L.toff, L.inb = (dev.upload(x) for x in (tch, toff, inb))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    print(f"case: {times * (n - 1)} visits, delta {delta}", flush=True)
    pairs, scores, *_ = G.candidates(dev, L, sizes, 4, 3, delta)
    ep, es = O.candidates(hg, toff, tch, inb, sizes, 4, 3, delta)
    assert ep[0] != 2**32 - 1
    assert np.array_equal(pairs, ep) and np.array_equal(scores, es)


def hub_graph(n, hubs, n_small, rng):
    """Hub nodes, each on `count` hedges of `size` pins drawn from a pool of `pool` nodes, so
    their visit bounds (and worst-case tables) are far above their distinct neighbours."""
    off, pins, srcc = [0], [], []
    for hub, count, size, pool in hubs:
        for _ in range(count):
            nodes = rng.choice(pool, size=size, replace=False)
            nodes = nodes[nodes != hub][: size - 1]
            pins.append(hub)
            pins.extend(int(x) for x in nodes)
            off.append(len(pins))
            srcc.append(1)
    for _ in range(n_small):
        sz = int(rng.integers(2, 6))
        pins.extend(int(x) for x in rng.choice(n, size=sz, replace=False))
        off.append(len(pins))
        srcc.append(int(rng.integers(0, 2)))
    w = (rng.random(len(srcc)) * 3 + 0.5).astype(np.float32)
    return O.dedup(O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32), w))


@pytest.mark.parametrize("n,hubs,expect", [
    # (hub, hedges, pins per hedge, pool): distinct neighbours ~20K, ~45K and ~75K
    (120000, [(7, 75, 400, 30000), (11, 141, 400, 120000), (13, 295, 400, 120000)],
     [(15000, 25000), (40400, 49000), (70000, 80000)]),
    # n = 50000: the hub's worst-case table is the whole level, indexed by node id
    (50000, [(5, 229, 400, 50000)], [(40400, 50000)]),
])
def test_candidates_heavy_tables(dev, n, hubs, expect, rng):
    """Nodes whose visit bound is far above their distinct neighbours, so they skip the
    guaranteed tiers: they are scored in the one-pass LDS table, the four-pass LDS table
    (one id class per pass), a 65536-slot HBM table at up to 3/4 load, or their worst-case
    HBM table (hashed, or indexed by node id), depending on the distinct count and on
    whether shared-inbound counts are kept (they shrink the LDS tables)."""
    hg = hub_graph(n, hubs, 4000, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    for (h, *_), (lo, hi) in zip(hubs, expect):
        idx = np.concatenate([np.arange(int(hg.off[e]), int(hg.off[e + 1])) for e in rt[ro[h]:ro[h + 1]]])
        nb = len(np.unique(hg.pins[idx]))
        assert lo < nb < hi, (h, nb)
    sizes = rng.integers(1, 3, size=hg.n).astype(np.uint32)
    for delta in (2**31 - 1, 30):
        pairs, scores, *_ = G.candidates(dev, L, sizes, 16, 6, delta)
        ep, es = O.candidates(hg, ro, rt, ri, sizes, 16, 6, delta)
        assert np.array_equal(pairs, ep), f"pairs differ (delta={delta})"
        assert np.array_equal(scores, es), f"scores differ (delta={delta})"


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 65535, 65536, 65537])
def test_candidates_by_size(dev, n, rng):
    """Levels whose nodes split into runs of 64 (and, above 65,536 nodes, of 128) when they are laid
    out by class: nodes without hedges, and hubs of every class with an LDS table by wave or workgroup."""
    if n < 64:
        hg = O.HG(n, np.array([0, 1], np.uint64), np.zeros(1, np.uint32), np.ones(1, np.uint32), np.ones(1, np.float32))
    else:
        hubs = [(h, c, 40, n) for h, c in ((0, 3), (1, 8), (n // 2, 20), (n - 1, 60), (n - 2, 110), (n - 3, 200))]
        hg = hub_graph(n, hubs, n // 4, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = rng.integers(1, 3, size=hg.n).astype(np.uint32)
    for delta in (2**31 - 1, 30):
        pairs, scores, *_ = G.candidates(dev, L, sizes, 4, 6, delta)
        ep, es = O.candidates(hg, ro, rt, ri, sizes, 4, 6, delta)
        assert np.array_equal(pairs, ep) and np.array_equal(scores, es), delta


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("cnc", [1, 3, 16])
def test_group_nodes(dev, case, cnc, rng):
    hg = make(case, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = np.ones(hg.n, np.uint32)
    omega, delta = 8, 2**31 - 1
    pairs, scores, d_sizes, d_pairs, d_scores = G.candidates(dev, L, sizes, cnc, omega, delta)
    k, groups, gs, ung, uoff, *_ = G.group_nodes(dev, hg.n, L.inb, d_pairs, d_scores, d_sizes, cnc, omega, delta)
    ek, eg, egs, eung, euoff, _ = O.group_nodes(hg.n, ri, pairs, scores, sizes, cnc, omega, delta)
    assert k == ek
    assert np.array_equal(groups, eg) and np.array_equal(gs, egs)
    assert np.array_equal(ung, eung) and np.array_equal(uoff, euoff)
    # invariants: groups of at most two nodes, each pair a candidate edge or an orphan pair
    counts = np.bincount(groups, minlength=k)
    assert counts.max() <= 2


def test_group_nodes_cycles(dev, rng):
    """Hand-made pointer rounds with 2-cycles and a 3-cycle in round 1."""
    n, cnc = 9, 2
    pairs = np.full(n * cnc, 0xFFFFFFFF, np.uint32)
    scores = np.zeros(n * cnc, np.uint32)

    def setp(v, i, t, s):
        pairs[v * cnc + i] = t
        scores[v * cnc + i] = s

    # round 0: chain 0->1->2, mutual 3<->4, 5 alone
    setp(0, 0, 1, 5); setp(1, 0, 2, 7); setp(2, 0, 1, 7); setp(3, 0, 4, 9); setp(4, 0, 3, 9)
    # round 1: 3-cycle 6->7->8->6 plus 5->6
    setp(6, 1, 7, 3); setp(7, 1, 8, 4); setp(8, 1, 6, 2); setp(5, 1, 6, 1)
    setp(6, 0, 0xFFFFFFFF, 0)
    inb = np.zeros(n, np.uint32)
    sizes = np.ones(n, np.uint32)
    d_inb, d_pairs, d_scores, d_sizes = (dev.upload(x) for x in (inb, pairs, scores, sizes))
    k, groups, *_ = G.group_nodes(dev, n, d_inb, d_pairs, d_scores, d_sizes, cnc, 10, 100)
    ek, eg, *_ = O.group_nodes(n, inb, pairs, scores, sizes, cnc, 10, 100)
    assert k == ek and np.array_equal(groups, eg)


@pytest.mark.parametrize("n", [1, 2, 64, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("cnc", [1, 4])
def test_group_nodes_by_size(dev, n, cnc, rng):
    """Levels at the edges of the one-workgroup pairing: random pointers (chains, cycles of all
    lengths, pointers to locked nodes and to the node itself), and orphans of many sizes."""
    pairs = rng.integers(0, n, size=(n, cnc)).astype(np.uint32)
    near = rng.random((n, cnc)) < 0.5  # half of them along one long cycle
    pairs[near] = ((np.arange(n)[:, None] + 1) % n * np.ones((1, cnc))).astype(np.uint32)[near]
    pairs[rng.random((n, cnc)) < 0.2] = 0xFFFFFFFF
    pairs[rng.random(n) < 0.3] = 0xFFFFFFFF  # orphans
    scores = rng.integers(0, 8, size=(n, cnc)).astype(np.uint32)
    sizes = rng.integers(1, 300, size=n).astype(np.uint32)
    inb = rng.integers(0, 50, size=n).astype(np.uint32)
    omega, delta = 310, 70
    d_inb, d_pairs, d_scores, d_sizes = (dev.upload(x) for x in (inb, pairs.ravel(), scores.ravel(), sizes))
    k, groups, gs, ung, uoff, *_ = G.group_nodes(dev, n, d_inb, d_pairs, d_scores, d_sizes, cnc, omega, delta)
    ek, eg, egs, eung, euoff, _ = O.group_nodes(n, inb, pairs.ravel(), scores.ravel(), sizes, cnc, omega, delta)
    assert k == ek and np.array_equal(groups, eg) and np.array_equal(gs, egs)
    assert np.array_equal(ung, eung) and np.array_equal(uoff, euoff)


@pytest.mark.parametrize("n", [100, 4096, 4097, 20000])
@pytest.mark.parametrize("omega", [1, 100, 70000])
def test_group_nodes_orphans_above_the_limit(dev, n, omega, rng):
    """Orphans are paired in the order of their sizes, also of sizes above the limit, whatever bits
    those have: sizes up to 2^31 - 1 (two of them do not wrap) beside sizes that fit in pairs."""
    pairs = np.full((n, 2), 0xFFFFFFFF, np.uint32)
    some = rng.random(n) < 0.2
    pairs[some, 0] = rng.integers(0, n, size=int(some.sum()))
    sizes = rng.integers(1, omega // 2 + 2, size=n).astype(np.uint32)
    above = rng.random(n) < 0.3
    sizes[above] = (2.0 ** rng.uniform(np.log2(omega + 1), 31, size=int(above.sum()))).astype(np.uint32)
    scores = rng.integers(0, 8, size=(n, 2)).astype(np.uint32)
    inb = rng.integers(0, 50, size=n).astype(np.uint32)
    d_inb, d_pairs, d_scores, d_sizes = (dev.upload(x) for x in (inb, pairs.ravel(), scores.ravel(), sizes))
    k, groups, gs, *_ = G.group_nodes(dev, n, d_inb, d_pairs, d_scores, d_sizes, 2, omega, 70)
    ek, eg, egs, *_ = O.group_nodes(n, inb, pairs.ravel(), scores.ravel(), sizes, 2, omega, 70)
    assert k == ek and np.array_equal(groups, eg) and np.array_equal(gs, egs)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_coarsening(dev, case, rng):
    """coarse hedges, coarse touching, coarse neighbours, uncoarsen"""
    hg = make(case, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    sizes = np.ones(hg.n, np.uint32)
    cnc = 4
    pairs, scores, d_sizes, d_pairs, d_scores = G.candidates(dev, L, sizes, cnc, 8, 2**31 - 1)
    k, groups, gs, ung, uoff, d_groups, *_ = G.group_nodes(dev, hg.n, L.inb, d_pairs, d_scores, d_sizes, cnc, 8,
                                                           2**31 - 1)
    choff, cp, csrcc, d_ch, d_co, d_cc = G.coarsen_hedges(dev, L, d_groups)
    eo, ep, es = O.coarsen_hedges(hg, groups)
    assert np.array_equal(choff, eo) and np.array_equal(cp, ep) and np.array_equal(csrcc, es)
    cto, ctt, cti = G.coarsen_touching(dev, d_ch, d_co, d_cc, k, hg.e)
    chg = O.HG(k, eo, ep, es, hg.w)
    xo, xt, xi = O.touching(chg)
    assert np.array_equal(cto, xo) and np.array_equal(ctt, xt) and np.array_equal(cti, xi)
    noff, nbr, d_nbr, d_noff = G.neighbors(dev, L)
    cno, cnb = G.coarsen_neighbors(dev, d_nbr, d_noff, d_groups, hg.n, k)
    eno, enb = O.coarsen_neighbors(hg.n, noff, nbr, groups, k)
    assert np.array_equal(cno, eno) and np.array_equal(cnb, enb)
    # the coarse neighbourhoods equal the neighbourhoods of the coarse hypergraph
    yo, yn = O.neighbors(chg, xo, xt)
    assert np.array_equal(cno, yo) and np.array_equal(cnb, yn)
    # uncoarsen
    cpart = rng.integers(0, 5, size=k).astype(np.uint32)
    d_cpart = dev.upload(cpart)
    d_part = dev.alloc(hg.n * 4)
    dev.check(dev.lib.hgp_uncoarsen(dev.ctx, G.V(d_groups), G.V(d_cpart), hg.n, G.V(d_part)), "uncoarsen")
    assert np.array_equal(dev.download(d_part, hg.n, np.uint32), cpart[groups])


REFINE_CASES = [
    ("kway_k2", 1, 2, "hgr_small"),
    ("kway_k8", 1, 8, "hgr_wide"),
    ("kway_k5_srcs", 1, 5, "srcs"),
    ("incc_k12", 0, 12, "srcs"),
    ("incc_k40_float", 0, 40, "float_w"),
    ("kway_big", 1, 4, "big_hedges"),
    # k-way up to 64 partitions scores from partition masks (both 32-bit words in use here),
    # above 64 from partition lists
    ("kway_k64_wide", 1, 64, "hgr_wide"),
    ("kway_k48_float", 1, 48, "float_w"),
    ("kway_k100_lists", 1, 100, "hgr_wide"),
]


def refine_setup(case_name, k, mode, rng):
    case = [c for c in CASES if c[0] == case_name][0]
    hg = make(case, rng)
    sizes = rng.integers(1, 3, size=hg.n).astype(np.uint32)
    part = rng.integers(0, k, size=hg.n).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    if mode == 1:
        omega = int(np.ceil(1.08 * sizes.sum() / k))
        delta = 2**31 - 1
    else:
        omega = int(psizes.max()) + 3
        inbs = O.inbound_sizes(hg, part, k)
        delta = int(inbs.max()) + 2
    return hg, sizes, part, psizes, omega, delta


@pytest.mark.parametrize("rc", REFINE_CASES, ids=[r[0] for r in REFINE_CASES])
@pytest.mark.parametrize("chainup", [False, True])
@pytest.mark.parametrize("fm_repeat", [0, 6, 13])
def test_refine_analyze(dev, rc, chainup, fm_repeat, rng):
    name, mode, k, case_name = rc
    hg, sizes, part, psizes, omega, delta = refine_setup(case_name, k, mode, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, fm_repeat, chainup, part, psizes)
    exp = O.refine_analyze(mode, omega, delta, 16, hg, ro, rt, ri, sizes, k, fm_repeat, chainup, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("mode,k,fm_repeat,chainup,n,e,max_size", [
    (1, 4096, 0, False, 4500, 10, 5000),   # gains table in LDS indexed by partition
    (0, 3000, 6, True, 4500, 10, 5000),
    (1, 22000, 0, True, 24000, 8, 9000),   # hashed LDS gains tables, some overflowing to HBM
    (0, 22000, 13, False, 24000, 8, 9000),
])
def test_refine_analyze_huge_lists(dev, mode, k, fm_repeat, chainup, n, e, max_size, rng):
    """Hedges of thousands of pins over thousands of partitions: partition lists longer than
    the LDS tables take the HBM-table path, and nodes adjacent to many partitions use the
    workgroup gain kernel (LDS tables indexed or hashed, HBM tables past 3/4 load)."""
    raw = O.HG(*gen.random_hypergraph(n, e, rng, max_size=max_size, src_prob=0.3, max_src=2, weights="unit"))
    hg = O.dedup(raw)
    sizes = rng.integers(1, 3, size=hg.n).astype(np.uint32)
    part = rng.integers(0, k, size=hg.n).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    lam = [len(np.unique(part[hg.pins[hg.off[e]:hg.off[e + 1]]])) for e in range(len(hg.off) - 1)]
    assert max(lam) > 2016, "the case must reach the HBM-table path"
    if mode == 1:
        omega, delta = int(np.ceil(1.08 * sizes.sum() / k)), 2**31 - 1
    else:
        omega, delta = int(psizes.max()) + 3, int(O.inbound_sizes(hg, part, k).max()) + 2
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, fm_repeat, chainup, part, psizes)
    exp = O.refine_analyze(mode, omega, delta, 16, hg, ro, rt, ri, sizes, k, fm_repeat, chainup, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("p", [1, 2, 63, 64, 65, 1023, 1025, 2048, 4097, 8191, 8192, 8193, 65535, 65536, 65537, 131072,
                               131073, 300001, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("n", [2, 100, 70000, 3000000])
def test_sorts_by_size(dev, p, n, rng):
    """The radix sorts at the edges of their kernels and tiles, by way of the incidence lists (32-bit
    keys with values, stable) and the coarse hedges (64-bit keys): one pass to seven, few and many
    distinct keys."""
    lens = np.minimum(rng.integers(1, 6, size=p), n).astype(np.int64)
    lens = lens[:int(np.searchsorted(np.cumsum(lens), p)) + 1]
    lens[-1] -= lens.sum() - p
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    e = len(lens)
    # distinct pins within a hedge: a random start and consecutive ids
    start = rng.integers(0, n, size=e)
    pos = np.arange(p) - np.repeat(off[:-1].astype(np.int64), lens)
    pins = ((np.repeat(start, lens) + pos) % n).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 2, size=e), lens).astype(np.uint32)
    hg = O.HG(n, off, pins, srcc, np.ones(e, np.float32))
    L = G.Level(dev, hg)
    toff, tch, inb = L.build_touching()
    hedge = np.repeat(np.arange(e, dtype=np.uint32), lens)
    key = pins.astype(np.int64) * 2 + (pos < np.repeat(srcc, lens))
    order = np.argsort(key, kind="stable")
    assert np.array_equal(tch, hedge[order])
    assert np.array_equal(toff, np.concatenate([[0], np.cumsum(np.bincount(pins, minlength=n))]).astype(np.uint64))
    assert np.array_equal(inb, np.bincount(pins[key % 2 == 0], minlength=n).astype(np.uint32))
    groups = (rng.permutation(n) // 2).astype(np.uint32)
    d_groups = dev.upload(groups)
    choff, cp, csrcc, *_ = G.coarsen_hedges(dev, L, d_groups)
    eo, ep, es = O.coarsen_hedges(hg, groups)
    assert np.array_equal(choff, eo) and np.array_equal(cp, ep) and np.array_equal(csrcc, es)
    for x in (d_groups, L.pins, L.off, L.srcc, L.w, L.tch, L.toff, L.inb):
        dev.free(x)


@pytest.mark.parametrize("mode,k,scale,chainup", [
    (1, 2, 1.0, False),            # whole-number gains: few varying bits, cycles of moves
    (0, 300, 1.0, True),
    (0, 4096, 0.37, False),        # the largest partition order ranked by counting
    (0, 4097, 0.37, False),        # ... and the smallest sorted one
    (0, 1 << 19, 16000.0, False),  # 64-bit keys (two sorts: test_refine_analyze_two_sorts)
    (0, 1 << 19, 16000.0, True),
])
def test_refine_analyze_move_keys(dev, mode, k, scale, chainup, rng):
    """The order of the moves over the bits of the gains that vary: unit and fractional weights,
    weights near the top of the fixed-point range on nodes of thousands of hedges."""
    heavy = scale > 1000
    n, e = 3000, 20000 if heavy else 3000
    n, off, pins, srcc, w = gen.random_hypergraph(n, e, rng, max_size=5, src_prob=0.3, max_src=1)
    rows = [list(pins[off[i]:off[i + 1]]) + ([0, 1] if heavy else []) for i in range(e)]  # two nodes of every hedge
    w = (np.ones(e) if scale == 1.0 else scale * (0.5 + 0.5 * rng.random(e))).astype(np.float32)
    hg = O.dedup(O.HG(n, np.cumsum([0] + [len(r) for r in rows]).astype(np.uint64),
                      np.array([x for r in rows for x in r], np.uint32), srcc, w))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    part = (rng.integers(0, min(k, 2000), size=n) + max(0, k - 2000)).astype(np.uint32)
    part[1] = part[0]
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega, delta = int(psizes.max()) + 2, 2**31 - 1
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, 0, chainup, part, psizes)
    exp = O.refine_analyze(mode, omega, delta, 16, hg, ro, rt, ri, sizes, k, 0, chainup, part, psizes)
    if heavy:
        bits = range_bits(exp["gains"][exp["moves"] != 2**32 - 1]) + (1 if chainup else (2 * k - 1).bit_length())
        assert 32 < bits <= 64, "the case must need a 64-bit key"
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("k,spread", [(1, 1), (70, 70), (70, 2), (40000, 40000)])
def test_partition_lists_by_hedge_length(dev, k, spread, rng):
    """Partition lists at the edges of their kernels (16 pins by thread, up to 64, 128 and 256 in a
    wave's registers, longer ones in LDS and HBM tables): the inbound sizes and lambda-1 that
    follow from them, with few and with many distinct partitions per hedge."""
    lens = [1, 2, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 2016, 2017, 2500] * 3
    n, off, pins, srcc = 4000, [0], [], []
    for i, ln in enumerate(lens):
        pins.extend(int(x) for x in rng.choice(n, size=ln, replace=False))
        off.append(len(pins))
        srcc.append(min(i % 3, ln))
    hg = O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32),
              rng.integers(1, 5, size=len(lens)).astype(np.float32))
    part = (rng.integers(0, spread, size=n) + k - spread).astype(np.uint32)
    L = G.Level(dev, hg)
    d_part = dev.upload(part)
    d_out = dev.alloc(4 * k)
    dev.check(dev.lib.hgp_inbound_sizes(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.srcc), G.V(d_part), hg.e, k,
                                        G.V(d_out)), "inbound sizes")
    assert np.array_equal(dev.download(d_out, k, np.uint32), O.inbound_sizes(hg, part, k))
    for p2 in (part, part + np.uint32(0xFFFE0000)):  # ids that fill 32 bits
        d_p2 = dev.upload(p2)
        km1 = C.c_int64()
        dev.check(dev.lib.hgp_connectivity(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.w), G.V(d_p2), hg.e, C.byref(km1)),
                  "connectivity")
        assert km1.value == O.connectivity_fixed(hg, part)


@pytest.mark.parametrize("short,long", [(1, 0), (200, 256), (200, 257), (65536, 0), (65537, 0), (65000, 1000), (0, 300)])
@pytest.mark.parametrize("k", [5, 9000])
def test_inbound_sizes_by_copies(dev, short, long, k, rng):
    """Inbound sizes added to one copy or to several: by the number of hedges, and by that of the longer
    ones, in registers, LDS and HBM tables, whose copies come after the short ones' counts."""
    n = 20000
    lens = np.concatenate([rng.integers(0, 17, size=short), np.resize([17, 64, 200, 256, 257, 600, 2500], long)])
    lens = rng.permutation(lens).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    pos = np.arange(int(off[-1])) - np.repeat(off[:-1].astype(np.int64), lens)
    pins = ((np.repeat(rng.integers(0, n, size=len(lens)), lens) + 7 * pos) % n).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 3, size=len(lens)), lens).astype(np.uint32)
    hg = O.HG(n, off, pins, srcc, np.ones(len(lens), np.float32))
    part = rng.integers(0, k, size=n).astype(np.uint32)
    L = G.Level(dev, hg)
    d_part, d_out = dev.upload(part), dev.alloc(4 * k)
    for _ in range(2):
        dev.check(dev.lib.hgp_inbound_sizes(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.srcc), G.V(d_part), hg.e, k,
                                            G.V(d_out)), "inbound sizes")
        assert np.array_equal(dev.download(d_out, k, np.uint32), O.inbound_sizes(hg, part, k))


@pytest.mark.parametrize("k", [5, 300, 66000])
@pytest.mark.parametrize("dup", [False, True])
def test_refine_analyze_inbound_by_hedge_size(dev, k, dup, rng):
    """The cascade kernels count which hedges leave and enter inbound sets: hedges of one pin, at
    the edges of every hedge class, with and without sources, and (not deduplicated) hedges that
    list a destination twice; k = 66000 takes the unpacked node records."""
    lens = [1, 2, 4, 5, 15, 16, 17, 63, 64, 65, 127, 128, 129, 1023, 1024, 1025, 2049] * 4 + [1, 2, 3] * 200
    n, off, pins, srcc = 3000, [0], [], []
    for i, ln in enumerate(lens):
        nodes = list(rng.choice(n, size=ln, replace=False))
        ns = min(int(rng.integers(0, 3)), ln - 1) if i % 3 else 0
        if dup and i % 2:
            nodes.append(nodes[int(rng.integers(ns, ln))])
        pins.extend(int(x) for x in nodes)
        off.append(len(pins))
        srcc.append(ns)
    hg = O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32),
              np.ones(len(lens), np.float32))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    part = rng.integers(0, min(k, 300), size=n).astype(np.uint32)
    part[:5] = k - 1 - np.arange(5)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega, delta = int(psizes.max()) + 3, int(O.inbound_sizes(hg, part, k).max()) - 1
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    got = G.refine_analyze(dev, L, sizes, k, 0, omega, delta, 16, 0, True, part, psizes)
    exp = O.refine_analyze(0, omega, delta, 16, hg, ro, rt, ri, sizes, k, 0, True, part, psizes)
    assert exp["iv"].any(), "the case must have inbound violations"
    # the cascade of a node listed twice is counted pin by pin on the device (the oracle applies
    # both pins at once), so seq and the best prefix are compared on deduplicated hedges only
    for key in ("moves", "gains", "ranks", "sv", "iv") + (() if dup else ("seq",)):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert dup or got["best"] == exp["best"]


@pytest.mark.parametrize("dup", [False, True])
@pytest.mark.parametrize("mode,k", [(0, 6), (1, 6), (0, 66000), (1, 66000)])
def test_refine_analyze_long_hedges(dev, mode, k, dup, rng):
    """Hedges cascaded by comparing all pins, at the edges of the LDS copy of the pins: sources from none
    to all, and (not deduplicated) nodes listed twice as destinations and as source and destination."""
    n, off, pins, srcc = 6000, [0], [], []
    for i, ln in enumerate([1025, 1026, 1500, 2047, 2048, 2049, 2050, 3001] * 3):
        nodes = list(rng.choice(n, size=ln, replace=False))
        ns = [0, 1, 3, ln // 2, ln - 1, ln][i % 6]
        if dup and 0 < ns < ln - 5:
            nodes[-1], nodes[-2] = nodes[0], nodes[-3]
        pins.extend(int(x) for x in nodes)
        off.append(len(pins))
        srcc.append(ns)
    e = len(srcc)
    hg = O.HG(n, np.array(off, np.uint64), np.array(pins, np.uint32), np.array(srcc, np.uint32),
              (rng.random(e) + 0.5).astype(np.float32))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    part = rng.integers(0, min(k, 300), size=n).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega = int(psizes.max()) + 3
    delta = 2**31 - 1 if mode else max(1, int(O.inbound_sizes(hg, part, k).max()) - 1)
    L = G.Level(dev, hg)
    L.build_touching()
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, 0, True, part, psizes)
    exp = O.refine_analyze(mode, omega, delta, 16, hg, *O.touching(hg), sizes, k, 0, True, part, psizes)
    # (a node listed twice: see test_refine_analyze_inbound_by_hedge_size)
    for key in ("moves", "gains", "ranks", "sv", "iv") + (() if dup else ("seq",)):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert dup or got["best"] == exp["best"]


@pytest.mark.parametrize("k", [40, 66000])
def test_refine_analyze_source_counts_above_the_length(dev, k, rng):
    """A source count above the hedge's length (the stages take device arrays as they are) makes all
    its pins sources, in the records of the small hedges too, where counts have five bits."""
    lens = np.resize([1, 2, 3, 4, 5, 8, 15, 16, 17, 40, 64, 65, 128, 129, 300, 1024, 1025], 1200)
    n, e = 3000, len(lens)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    pins = np.concatenate([rng.choice(n, size=ln, replace=False) for ln in lens]).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 3, size=e), lens).astype(np.uint32)
    high = rng.random(e) < 0.3
    srcc[high] = rng.choice(np.array([17, 31, 32, 33, 63, 1024, 1 << 16, 2**31, 2**32 - 1], np.uint32), size=int(high.sum()))
    assert (srcc > lens).any()
    hg = O.HG(n, off, pins, srcc, np.ones(e, np.float32))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    part = rng.integers(0, min(k, 300), size=n).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega, delta = int(psizes.max()) + 3, int(O.inbound_sizes(hg, part, k).max()) - 1
    L = G.Level(dev, hg)
    L.build_touching()
    for chainup in (False, True):
        got = G.refine_analyze(dev, L, sizes, k, 0, omega, delta, 16, 0, chainup, part, psizes)
        exp = O.refine_analyze(0, omega, delta, 16, hg, *O.touching(hg), sizes, k, 0, chainup, part, psizes)
        assert exp["iv"].any()
        for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
            assert np.array_equal(got[key], exp[key]), f"{key} differs (chainup={chainup})"
        assert got["best"] == exp["best"]


@pytest.mark.parametrize("n", [1, 2, 65, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 65536, 65537])
@pytest.mark.parametrize("mode,k", [(1, 40), (0, 40), (1, 3000), (0, 3000)])
def test_refine_analyze_by_level_size(dev, n, mode, k, rng):
    """Levels at the edges of the one-workgroup ranking (8,192 nodes) and events (4,096), of their
    items per thread, of the ranks whose counters fit LDS and of the tiles of the prefix sums;
    partitions by table and by scan."""
    lens = np.minimum(np.concatenate([rng.integers(1, 18, size=2 * n), rng.integers(17, 130, size=min(n, 200))]), n)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    start, step = rng.integers(0, n, size=len(lens)), 1 + 2 * rng.integers(0, 50, size=len(lens))
    pos = np.arange(int(off[-1])) - np.repeat(off[:-1].astype(np.int64), lens)
    pins = ((np.repeat(start, lens) + pos * np.repeat(step, lens)) % n).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 3, size=len(lens)), lens - 1).astype(np.uint32)
    hg = O.dedup(O.HG(n, off, pins, srcc, (rng.random(len(lens)) + 0.5).astype(np.float32)))
    sizes = rng.integers(1, 4, size=n).astype(np.uint32)
    part = rng.integers(0, k, size=n).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega, delta = int(psizes.max()) + 3, 2**31 - 1
    if mode == 0:
        delta = max(1, int(O.inbound_sizes(hg, part, k).max()) - 1)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    for chainup in (False, True):
        got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, 0, chainup, part, psizes)
        exp = O.refine_analyze(mode, omega, delta, 16, hg, ro, rt, ri, sizes, k, 0, chainup, part, psizes)
        for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
            assert np.array_equal(got[key], exp[key]), f"{key} differs (chainup={chainup})"
        assert got["best"] == exp["best"]


def inbound_violations(hg, part, moves, ranks, k, delta):
    """The running inbound violations from their definition: the destinations of every (hedge,
    partition) counted move by move in rank order, the inbound size of every partition from the
    counts that reach or leave zero, and its crossings of delta (a partition's first change starts
    from a valid state)."""
    lens = np.diff(hg.off.astype(np.int64))
    hedge = np.repeat(np.arange(hg.e), lens)
    dst = np.arange(len(hg.pins)) - hg.off[:-1].astype(np.int64)[hedge] >= hg.srcc.astype(np.int64)[hedge]
    hedge, node = hedge[dst], hg.pins[dst]
    own = hedge * k + part[node]  # (hedge, partition) of every destination
    m = moves[node] != 2**32 - 1
    rank = ranks[node].astype(np.int64)[m]
    key = np.concatenate([own[m], hedge[m] * k + moves[node].astype(np.int64)[m]])
    step, rank = np.concatenate([-np.ones(len(rank), np.int64), np.ones(len(rank), np.int64)]), np.tile(rank, 2)

    def running(key, step, start):  # sums up to each event of its key's run, added to the run's start
        total, first = np.cumsum(step), np.concatenate([[True], key[1:] != key[:-1]])
        return total - np.repeat((total - step)[first], np.diff(np.append(np.flatnonzero(first), len(key)))) + start

    o = np.lexsort((rank, key))
    key, step, rank = key[o], step[o], rank[o]
    ids, cnt = np.unique(own, return_counts=True)
    at = np.minimum(np.searchsorted(ids, key), len(ids) - 1)
    now = running(key, step, np.where(ids[at] == key, cnt[at], 0))
    change = (now > 0).astype(np.int64) - (now - step > 0)
    c = change != 0
    q, change, rank = key[c] % k, change[c], rank[c]
    o = np.lexsort((rank, q))
    q, change, rank = q[o], change[o], rank[o]
    size = running(q, change, np.bincount(ids % k, minlength=k)[q])
    was = (size - change > delta) & np.concatenate([[False], q[1:] == q[:-1]])
    return np.cumsum(np.bincount(rank, weights=(size > delta).astype(np.int64) - was, minlength=hg.n)).astype(np.int32)


@pytest.mark.parametrize("n,e,k,chainup", [
    (300_000, 300_000, 2000, False),         # above the ranks that have copies of the cascade's counters
    (300_000, 300_000, 2000, True),
    (600_000, (1 << 20) + 1, 1 << 24, True),  # partition, hedge and rank in more than 64 bits together
    (600_000, (1 << 20) + 1, 1 << 24, False),
])
def test_refine_analyze_inbound_many_ranks(dev, n, e, k, chainup, rng):
    """Inbound-constrained rounds of more than 262,144 moves: the cascade's counters in memory, the
    inbound events of many partitions, hedges of every cascade class.  (The oracle goes through all
    partitions for every node, so the largest case checks the violations alone, from their definition.)"""
    lens = rng.integers(1, 5, size=e)
    lens[rng.permutation(e)[:600]] = np.resize([16, 17, 64, 65, 128, 129, 700, 1024, 1025, 2049], 600)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    start, step = rng.integers(0, n, size=e), 1 + 2 * rng.integers(0, 50, size=e)
    pos = np.arange(int(off[-1])) - np.repeat(off[:-1].astype(np.int64), lens)
    pins = ((np.repeat(start, lens) + pos * np.repeat(step, lens)) % n).astype(np.uint32)
    srcc = np.minimum(rng.integers(0, 2, size=e), lens - 1).astype(np.uint32)
    hg = O.HG(n, off, pins, srcc, (rng.random(e) + 0.5).astype(np.float32))
    sizes = rng.integers(1, 4, size=n).astype(np.uint32)
    part = (np.arange(n) * 7 // 13 % min(k, 3000) * (k // min(k, 3000))).astype(np.uint32)
    psizes = np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)
    omega, delta = int(psizes.max()) + 3, max(1, int(O.inbound_sizes(hg, part, k).max()) - 1)
    L = G.Level(dev, hg)
    L.build_touching()
    got = G.refine_analyze(dev, L, sizes, k, 0, omega, delta, 16, 0, chainup, part, psizes)
    ranks = int((got["moves"] != 2**32 - 1).sum())
    assert ranks > 262144 and got["iv"].any()
    iv = inbound_violations(hg, part, got["moves"], got["ranks"], k, delta)
    assert np.array_equal(got["iv"][:ranks], iv[:ranks])
    if k >= 1 << 24:
        assert k.bit_length() + e.bit_length() + (ranks - 1).bit_length() > 64
        return
    exp = O.refine_analyze(0, omega, delta, 16, hg, *O.touching(hg), sizes, k, 0, chainup, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("movers", [1, 2, 3, 4, 5, 8, 9])
def test_refine_analyze_inbound_few_ranks(dev, movers, rng):
    """A device-wide inbound-constrained round of a handful of moves, all into one partition that is
    over its limit from the start: the first of its events counts as starting valid, no later one."""
    n, k = 5000, 12
    n, off, pins, srcc, w = gen.random_hypergraph(n, 8000, rng, max_size=12, src_prob=0.3, max_src=2)
    hg = O.dedup(O.HG(n, off, pins, srcc, w))
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    part = np.zeros(n, np.uint32)
    part[rng.permutation(n)[:movers]] = 1 + np.arange(movers) % (k - 1)
    psizes = np.full(k, 100, np.uint32)  # only partition 0 takes nodes
    psizes[0] = 1
    L = G.Level(dev, hg)
    L.build_touching()
    for delta in (10, int(O.inbound_sizes(hg, part, k).max())):
        for chainup in (False, True):
            exp = O.refine_analyze(0, 50, delta, 16, hg, *O.touching(hg), sizes, k, 0, chainup, part, psizes)
            assert int((exp["moves"] != 2**32 - 1).sum()) == movers
            got = G.refine_analyze(dev, L, sizes, k, 0, 50, delta, 16, 0, chainup, part, psizes)
            for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
                assert np.array_equal(got[key], exp[key]), f"{key} differs"
            assert got["best"] == exp["best"]


# (mode, n, k, chainup, hedges of each hub, where the keys are too wide).  By table a key is 13 bits of
# position, the partition and validity, and the range of the gains; by gain it holds no partition.
WIDE_CASES = [
    (1, 4000, 1000, False, 20000, "moves"),   # up to 4,096 nodes: found out after the round's last kernel
    (0, 4000, 1000, False, 20000, "moves"),
    (1, 8000, 1000, False, 20000, "moves"),   # above: found out before the cascade
    (0, 8000, 1000, False, 20000, "moves"),
    (1, 4000, 4, True, 270000, "moves"),
    (0, 8000, 4, True, 270000, "moves"),
    (1, 4000, 2, False, 110000, "chains"),    # every move fits, the sum of a chain's gains does not
    (1, 8000, 2, False, 110000, "chains"),
]


def wide_level(n, k, e, rng):
    """Hub 0, in partition 0, shares heavy hedges of two pins with nodes of partition 1, and hub 1 the
    other way round, so each gains them all; a few hedges of the smallest weight leave the gains
    without common trailing zeros."""
    part = rng.integers(0, min(k, 1000), size=n).astype(np.uint32)
    part[:2] = [0, 1]
    a, b = 2 + np.flatnonzero(part[2:] == 1), 2 + np.flatnonzero(part[2:] == 0)
    pairs = np.concatenate([np.stack([np.zeros(e, np.int64), rng.choice(a, e)], 1),
                            np.stack([np.ones(e, np.int64), rng.choice(b, e)], 1),
                            rng.permutation(np.arange(2, n))[:200].reshape(100, 2)])
    w = np.concatenate([16383 - rng.random(2 * e), np.full(100, 2.0 ** -18)]).astype(np.float32)
    hg = O.HG(n, 2 * np.arange(len(w) + 1).astype(np.uint64), pairs.ravel().astype(np.uint32), np.zeros(len(w), np.uint32), w)
    sizes = rng.integers(1, 3, size=n).astype(np.uint32)
    sizes[:2] = 1
    return hg, sizes, part, np.bincount(part, weights=sizes, minlength=k).astype(np.uint32)


def range_bits(gains):
    """Bits of the range of the gains above the trailing zeros that all share."""
    low = int(np.bitwise_or.reduce(gains))
    return ((int(gains.max()) - int(gains.min())) // (low & -low)).bit_length()


@pytest.mark.parametrize("mode,n,k,chainup,e,where", WIDE_CASES)
def test_refine_analyze_wide_keys_on_small_levels(dev, mode, n, k, chainup, e, where, rng):
    """Levels of up to 8,192 nodes whose keys do not fit the one-workgroup ranking are ranked
    device-wide instead, within the same round."""
    hg, sizes, part, psizes = wide_level(n, k, e, rng)
    omega = int(psizes.max()) + 2
    L = G.Level(dev, hg)
    L.build_touching()
    exp = O.refine_analyze(mode, omega, 2**31 - 1, 16, hg, *O.touching(hg), sizes, k, 0, chainup, part, psizes)
    gains = exp["gains"][exp["moves"] != 2**32 - 1]
    bits = range_bits(gains) + 13 + (1 if chainup else (2 * k - 1).bit_length())
    assert (bits > 64) == (where == "moves")
    if where == "chains":
        assert int(exp["ranks"][1]) == int(exp["ranks"][0]) + 1 or int(exp["ranks"][0]) == int(exp["ranks"][1]) + 1
        assert (int(exp["gains"][0]) + int(exp["gains"][1]) - int(gains.min())).bit_length() + 2 + 13 > 64
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, 2**31 - 1, 16, 0, chainup, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("mode", [0, 1])
def test_refine_analyze_two_sorts(dev, mode, rng):
    """Gain and partition bits together above 64: the device-wide ranking sorts by gain, then by partition."""
    n, k = 4000, 1 << 19
    hg, sizes, part, psizes = wide_level(n, k, 20000, rng)
    omega = int(psizes.max()) + 2
    L = G.Level(dev, hg)
    L.build_touching()
    exp = O.refine_analyze(mode, omega, 2**31 - 1, 16, hg, *O.touching(hg), sizes, k, 0, False, part, psizes)
    assert range_bits(exp["gains"][exp["moves"] != 2**32 - 1]) + (2 * k - 1).bit_length() > 64
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, 2**31 - 1, 16, 0, False, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]


@pytest.mark.parametrize("mode,n,k,chainup,e,where", [c for c in WIDE_CASES if not c[3]])
def test_refine_loop_wide_keys_on_small_levels(dev, mode, n, k, chainup, e, where, rng):
    """All rounds of such a level, whose layout is kept from round to round."""
    hg, sizes, part, psizes = wide_level(n, k, e, rng)
    omega = int(psizes.max()) + 2
    L = G.Level(dev, hg)
    L.build_touching()
    gp, gps, gpin = G.refine(dev, L, sizes, k, mode, omega, 2**31 - 1, 16, True, part, psizes)
    ep, eps_, epin = O.refine(mode, omega, 2**31 - 1, 16, hg, *O.touching(hg), sizes, k, True, part, psizes)
    assert np.array_equal(gp, ep) and np.array_equal(gps, eps_) and np.array_equal(gpin, epin)


@pytest.mark.parametrize("mode", [0, 1])
def test_refine_analyze_above_the_prefix_tiles(dev, mode, rng):
    """More ranks than the tiles of the prefix sums hold (4,096 of 4,096): single scans and a sweep for
    the best prefix.  A million hedges among a few thousand of the nodes and all of them."""
    n, e, k = 4096 * 4096 + 5000, 1_000_000, 2
    pins = rng.integers(0, n, size=3 * e).astype(np.uint32)
    pins[rng.random(3 * e) < 0.5] %= 4000
    hg = O.HG(n, 3 * np.arange(e + 1).astype(np.uint64), pins, (np.arange(e) % 2).astype(np.uint32),
              (rng.random(e) + 0.5).astype(np.float32))
    hg = O.dedup(hg)
    sizes = np.ones(n, np.uint32)
    part = rng.integers(0, k, size=n).astype(np.uint32)
    psizes = np.bincount(part, minlength=k).astype(np.uint32)
    omega = int(psizes.max()) + 2
    delta = int(O.inbound_sizes(hg, part, k).max()) - 1 if mode == 0 else 2**31 - 1
    print(f"case: {n} ranks, mode {mode}", flush=True)
    exp = O.refine_analyze(mode, omega, delta, 16, hg, *O.touching(hg), sizes, k, 0, True, part, psizes)
    assert int((exp["moves"] != 2**32 - 1).sum()) > 4096 * 4096
    L = G.Level(dev, hg)
    L.build_touching()
    got = G.refine_analyze(dev, L, sizes, k, mode, omega, delta, 16, 0, True, part, psizes)
    for key in ("moves", "gains", "ranks", "seq", "sv", "iv"):
        assert np.array_equal(got[key], exp[key]), f"{key} differs"
    assert got["best"] == exp["best"]
    for x in (L.pins, L.off, L.srcc, L.w, L.tch, L.toff, L.inb):
        dev.free(x)


@pytest.mark.parametrize("rc", REFINE_CASES, ids=[r[0] for r in REFINE_CASES])
def test_refine_loop(dev, rc, rng):
    name, mode, k, case_name = rc
    hg, sizes, part, psizes, omega, delta = refine_setup(case_name, k, mode, rng)
    L = G.Level(dev, hg)
    L.build_touching()
    ro, rt, ri = O.touching(hg)
    gp, gps, gpin = G.refine(dev, L, sizes, k, mode, omega, delta, 16, True, part, psizes)
    ep, eps_, epin = O.refine(mode, omega, delta, 16, hg, ro, rt, ri, sizes, k, True, part, psizes)
    assert np.array_equal(gp, ep) and np.array_equal(gps, eps_) and np.array_equal(gpin, epin)
    # the refined state is consistent and no worse than the start
    assert np.array_equal(np.bincount(gp, weights=sizes, minlength=k).astype(np.uint32), gps)
    assert O.connectivity_fixed(hg, gp) <= O.connectivity_fixed(hg, part)


def test_postprocess(dev, rng):
    n = 500
    ng = 120
    groups = rng.integers(0, ng, size=n).astype(np.uint32)
    groups = O.relabel(groups)[1]
    ng = int(groups.max()) + 1
    sizes = rng.integers(1, 4, size=n).astype(np.uint32)
    inb = rng.integers(0, 20, size=n).astype(np.uint32)
    gsizes = np.bincount(groups, weights=sizes, minlength=ng).astype(np.uint32)
    omega, delta = 60, 300
    d_sizes, d_inb, d_groups, d_gs = (dev.upload(x) for x in (sizes, inb, groups, gsizes))
    new = C.c_uint32()
    dev.check(dev.lib.hgp_greedy_merge_groups(dev.ctx, G.V(d_sizes), G.V(d_inb), n, ng, omega, delta, G.V(d_groups),
                                              G.V(d_gs), C.byref(new)), "greedy merge")
    en, eg, egs = O.greedy_merge_groups(n, ng, sizes, inb, omega, delta, groups, gsizes)
    assert new.value == en
    assert np.array_equal(dev.download(d_groups, n, np.uint32), eg)
    assert np.array_equal(dev.download(d_gs, en, np.uint32), egs)
    # small partitions merge + relabel
    k = 80
    part = rng.integers(0, k, size=n).astype(np.uint32)
    psz = np.bincount(part, minlength=k).astype(np.uint32)
    pinb = rng.integers(0, 50, size=k).astype(np.uint32)
    d_part, d_psz, d_pinb = (dev.upload(x) for x in (part, psz, pinb))
    dev.check(dev.lib.hgp_merge_small_partitions(dev.ctx, G.V(d_psz), G.V(d_pinb), n, k, 40, 200, G.V(d_part)), "msp")
    ep = O.merge_small_partitions(n, k, psz, pinb, 40, 200, part)
    gp = dev.download(d_part, n, np.uint32)
    assert np.array_equal(gp, ep)
    nk = C.c_uint32()
    dev.check(dev.lib.hgp_relabel_partitions(dev.ctx, n, G.V(d_part), C.byref(nk)), "relabel")
    ek, er = O.relabel(ep)
    assert nk.value == ek and np.array_equal(dev.download(d_part, n, np.uint32), er)


@pytest.mark.parametrize("case", CASES[:3], ids=[c[0] for c in CASES[:3]])
def test_inbound_and_connectivity(dev, case, rng):
    hg = make(case, rng)
    L = G.Level(dev, hg)
    k = 7
    part = rng.integers(0, k, size=hg.n).astype(np.uint32)
    d_part = dev.upload(part)
    d_out = dev.alloc(k * 4)
    dev.check(dev.lib.hgp_inbound_sizes(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.srcc), G.V(d_part), hg.e, k,
                                        G.V(d_out)), "inbound sizes")
    assert np.array_equal(dev.download(d_out, k, np.uint32), O.inbound_sizes(hg, part, k))
    km1 = C.c_int64()
    dev.check(dev.lib.hgp_connectivity(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.w), G.V(d_part), hg.e, C.byref(km1)),
              "connectivity")
    assert km1.value == O.connectivity_fixed(hg, part)


def ip_input_hypergraph(n, e, max_size, copies, rng):
    """Hedges with exact copies, copies with their pins permuted, repeated pins, single-pin
    hedges and weights that round to zero in fixed point."""
    hedges = []
    for _ in range(e):
        if hedges and rng.random() < copies:
            h = list(hedges[int(rng.integers(0, len(hedges)))])
            rng.shuffle(h)
        else:
            h = [int(x) for x in rng.choice(n, size=int(rng.integers(1, max_size + 1)), replace=False)]
            if rng.random() < 0.1:
                h.append(h[0])  # a repeated pin
        hedges.append(h)
    off = np.zeros(e + 1, np.uint64)
    off[1:] = np.cumsum([len(h) for h in hedges])
    pins = np.array([x for h in hedges for x in h], np.uint32)
    w = (rng.random(e) * 3).astype(np.float32)
    w[rng.random(e) < 0.05] = 1e-7
    return O.HG(n, off, pins, np.zeros(e, np.uint32), w)


def device_ip_input(dev, L, d_sizes, n, e, prune):
    m, p = C.c_uint32(), C.c_uint64()
    args = (dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.w), G.V(d_sizes), n, e, int(prune), C.byref(m), C.byref(p))
    dev.check(dev.lib.hgp_ip_input(*args, None, None, None), "ip input sizes")
    off = np.zeros(m.value + 1, np.uint64)
    pins = np.zeros(p.value, np.uint32)
    w = np.zeros(m.value, np.uint64)
    dev.check(dev.lib.hgp_ip_input(*args, off.ctypes.data_as(C.POINTER(C.c_uint64)),
                                   pins.ctypes.data_as(C.POINTER(C.c_uint32)),
                                   w.ctypes.data_as(C.POINTER(C.c_uint64))), "ip input")
    return off, pins, w


@pytest.mark.parametrize("prune", [0, 1, 4])
@pytest.mark.parametrize("n,e,max_size,copies", [(300, 2000, 5, 0.3), (5000, 40000, 12, 0.2), (64, 3000, 4, 0.6)])
def test_ip_input_device_equals_oracle(dev, n, e, max_size, copies, prune, rng):
    """The initial partitioner's input built on the device (hedge pruning, sort, merge of
    identical pin sets, summed weights) equals the oracle's restatement exactly."""
    hg = ip_input_hypergraph(n, e, max_size, copies, rng)
    L = G.Level(dev, hg)
    sizes = rng.integers(1, 5, size=n).astype(np.uint32)
    d_sizes = dev.upload(sizes)
    off, pins, w = device_ip_input(dev, L, d_sizes, n, e, prune)
    eo, ep, ew, _ = O.ip_input(hg, sizes, prune=prune)
    assert np.array_equal(off, eo) and np.array_equal(pins, ep) and np.array_equal(w, ew)
    assert 0 < len(w) < e


def test_initial_partition(dev, rng):
    hg = make(CASES[1], rng)
    L = G.Level(dev, hg)
    sizes = rng.integers(1, 5, size=hg.n).astype(np.uint32)
    k, eps = 8, 0.03
    omega = O.kway_omega(int(sizes.sum()), k, eps)
    d_sizes = dev.upload(sizes)
    pp, ps = G.V(), G.V()
    dev.check(dev.lib.hgp_initial_partition(dev.ctx, G.V(L.pins), G.V(L.off), G.V(L.w), hg.n, hg.e, L.p, G.V(d_sizes),
                                            k, eps, omega, 1, C.byref(pp), C.byref(ps)), "initial partition")
    gp = dev.download(pp.value, hg.n, np.uint32)
    ep, eps_ = O.initial_partition(hg, sizes, k, eps, omega)
    assert np.array_equal(gp, ep)
    assert np.array_equal(dev.download(ps.value, k, np.uint32), eps_)
    assert eps_.max() <= omega
