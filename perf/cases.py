"""Performance cases: what programs have this partitioner do, through its public entry points.

A case is one kind of call on one seeded workload:

* partition  whole partitionings, k-way or inbound-constrained, from device-resident CSR arrays
             (hgp_partition_device) or from a host model (hgp_partition, upload included);
* refine     one level's refinement, from a partition the caller brings (hgp_refine);
* contract   one coarsening level: incidence, candidates, pairing, coarse hedges and their
             incidence (hgp_build_touching .. hgp_coarsen_touching);
* evaluate   what is asked of a finished partition: lambda-1, inbound-set sizes and the
             quotient hypergraph (hgp_connectivity, hgp_inbound_sizes, hgp_quotient);
* serve      a burst of jobs through the serving loop (hgp_server_*).

Workloads come from the library's own generators: `random` (sizes 2 + Geom(1/2), uniform pins),
`netlist` (power-law nets with grid locality) and `snn` (8 layers of receptive fields).  Every
output is an integer, except the quotient's float weights.
"""
import ctypes as C
import math

import numpy as np
import torch

import axoncuda_amd as H

EPS = 0.03
LAYERS = 8
OMEGA, DELTA, MAX_PARTS = 1024, 4096, 1 << 20  # the inbound-constrained workload's -m
SCALE = 1 << 18  # fixed point of lambda-1
V = C.c_void_p
U32P = C.POINTER(C.c_uint32)


def _case(name, call, kind, size, **kw):
    c = {"name": name, "call": call, "kind": kind, "size": size, "k": 0, "ipm": False, "host": False, "fanout": 0,
         "jobs": 0}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest job: a random hypergraph of 80 thousand pins cut in two; launches and waits count
        _case("kway_random_20k_k2", "partition", "random", 20_000, k=2),
        # a block of a design straight from a loader, 64 parts
        _case("kway_netlist_100k_k64_host", "partition", "netlist", 100_000, k=64, host=True),
        # a serving-sized job of a million pins without locality
        _case("kway_random_250k_k8_host", "partition", "random", 250_007, k=8, host=True),
        # more parts than a 64-bit mask holds
        _case("kway_netlist_400k_k256", "partition", "netlist", 400_003, k=256),
        # the benchmark workload
        _case("kway_netlist_3200k_k64", "partition", "netlist", 3_200_000, k=64),
        # a small spiking network onto cores with an inbound limit
        _case("incc_snn_8x1156_f64_host", "partition", "snn", 1156, fanout=64, host=True),
        # an ordinary one, initial partitions merged
        _case("incc_snn_8x8191_f64_ipm", "partition", "snn", 8191, fanout=64, ipm=True),
        # improving a partition that the caller already has
        _case("refine_netlist_500k_k32", "refine", "netlist", 500_009, k=32),
        # one contraction of a design
        _case("contract_netlist_800k", "contract", "netlist", 800_000, k=64),
        # one contraction of a network of the full workload's fan-out (its widest neighbourhoods)
        _case("contract_snn_8x2048_f256", "contract", "snn", 2048, fanout=256),
        # scoring a partition and writing its quotient
        _case("evaluate_netlist_200k_k64", "evaluate", "netlist", 200_000, k=64),
        # a burst of mixed jobs through the serving loop
        _case("serve_12_jobs", "serve", "mixed", 400_000, jobs=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["kway", "kway", "kway", "incc", "incc", "refine", "contract", "contract", "evaluate", "serve"])
    if what == "kway":
        kind = rng.choice(["random", "netlist"])
        size = _log_int(rng, 15_000, 400_000 if kind == "random" else 2_000_000)
        c = _case("", "partition", kind, size, k=_log_int(rng, 2, 256), host=rng.random() < 0.5)
    elif what == "incc":
        c = _case("", "partition", "snn", _log_int(rng, 400, 8191), fanout=_log_int(rng, 16, 64),
                  ipm=rng.random() < 0.5, host=rng.random() < 0.5)
    elif what == "refine":
        c = _case("", "refine", rng.choice(["random", "netlist"]), _log_int(rng, 10_000, 1_000_000),
                  k=_log_int(rng, 2, 256))
    elif what == "contract":
        if rng.random() < 0.6:
            c = _case("", "contract", rng.choice(["random", "netlist"]), _log_int(rng, 5_000, 1_600_000), k=64)
        else:
            c = _case("", "contract", "snn", _log_int(rng, 400, 4000), fanout=_log_int(rng, 16, 256))
    elif what == "evaluate":
        c = _case("", "evaluate", rng.choice(["random", "netlist"]), _log_int(rng, 2_000, 2_000_000),
                  k=_log_int(rng, 2, 256))
    else:
        c = _case("", "serve", "mixed", _log_int(rng, 50_000, 400_000), jobs=rng.randint(4, 12))
    del c["name"]
    return c


# ---- handles a program opens once ---------------------------------------------------------

_handles = {}


def _stream():
    if "stream" not in _handles:
        _handles["stream"] = torch.cuda.Stream()
    return _handles["stream"]


def _device():
    """One context on a stream that the program's own tensor work shares."""
    if "device" not in _handles:
        dev = H.Device(0)
        dev.check(dev.lib.hgp_ctx_set_stream(dev.ctx, V(_stream().cuda_stream)), "stream")
        _handles["device"] = dev
    return _handles["device"]


def _server():
    if "server" not in _handles:
        _handles["server"] = H.Server(0, workers=4)
    return _handles["server"]


# ---- inputs -------------------------------------------------------------------------------

def _generate(kind, size, fanout, seed):
    if kind == "random":
        return H.Hypergraph.generate("random", n=size, e=size, max_size=64, seed=seed)
    if kind == "netlist":
        hg = H.Hypergraph.generate("netlist", n=size, e=round(size * 1.0625), alpha=2.5, max_size=1000, radius=8,
                                   frac_local=0.8, seed=seed)
        n, off, pins, srcc, w = hg.arrays()
        return H.Hypergraph.from_csr(n, off, pins, srcc, w, dedup=True)  # what a loader hands over
    grid = math.ceil(math.sqrt(size))
    sigma = max(4.0, math.sqrt(fanout))  # 16 for the full workload's fan-out of 256
    return H.Hypergraph.generate("snn", layers=LAYERS, per_layer=size, grid=grid, fanout=fanout, sigma=sigma,
                                 seed=seed)


def _pin_cap(case):
    """More pins than the generators give for a case (their mean and many standard deviations)."""
    _, e, pins = _shape(case)
    return int(pins + 100 * math.sqrt(e) + 1000)


def _params(n, k, ipm):
    prm = H.Params()
    H.load_library().hgp_default_params(C.byref(prm))
    prm.save_memory_up_to_level = 0
    if k:
        prm.mode, prm.kway, prm.epsilon = H.HGP_MODE_KWAY, k, EPS
        omega = int(np.ceil(np.float32(1 + np.float32(EPS)) * np.float32(n) / np.float32(k)))
        prm.max_nodes_per_part, prm.max_inbound_per_part, prm.max_parts = omega, 2**31 - 1, k
    else:
        prm.mode = H.HGP_MODE_INCC
        prm.max_nodes_per_part, prm.max_inbound_per_part, prm.max_parts = OMEGA, DELTA, MAX_PARTS
        prm.initial_partitions_merge = 1 if ipm else 0
    return prm


def _gpu(a):
    a = np.ascontiguousarray(a)
    if a.dtype.kind == "u":  # ids, counts and offsets: the same bits
        a = a.view(a.dtype.str.replace("u", "i"))
    return torch.from_numpy(a).cuda()


def _ptr(t):
    return V(t.data_ptr())


class _Csr:
    """The hypergraph as device tensors: pins (sources first), u64 offsets, source counts, weights."""

    def __init__(self, hg):
        self.n, off, pins, srcc, w = hg.arrays()
        self.e, self.p = len(srcc), len(pins)
        self.off, self.pins, self.srcc, self.w = _gpu(off), _gpu(pins), _gpu(srcc), _gpu(w)


def _partition_of(n, k, seed):
    """A partition as a caller brings it: runs of ids (rows of the grid), a few nodes out of place."""
    rng = np.random.default_rng(seed)
    part = (np.arange(n, dtype=np.int64) * k // n).astype(np.uint32)
    m = n // 20
    a, b = rng.permutation(n)[:m], rng.permutation(n)[:m]
    part[a] = part[b]
    part[rng.permutation(n)[:k]] = np.arange(k, dtype=np.uint32)  # every id is used
    return part


class _Owned:
    """Device arrays that a library call returned: seen as tensors, given back with hgp_free.
    keep() copies one whose length depends on the data into an array of the program's own (zeros
    after its end), as a program does that holds results in arrays of one size."""

    def __init__(self):
        self.ptrs = []

    def tensor(self, ptr, count, typestr):
        if not ptr.value:
            return torch.empty(0, dtype=torch.int32, device="cuda")
        self.ptrs.append(ptr.value)
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (ptr.value, False),
                                         "version": 2}
        return torch.as_tensor(self, device="cuda")

    def keep(self, t, where):
        where[: t.numel()].copy_(t, non_blocking=True)
        return where

    def free(self):
        dev = _device()
        for p in self.ptrs:
            dev.free(p)
        self.ptrs = []

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class _State:
    pass


def _jobs(case, seed):
    """Jobs of 10^4 .. `size` pins (spread over the logarithm, in a fixed mixed order), half random,
    half layered; k = 2, 8, 32 or inbound-constrained in turn."""
    count, jobs = case["jobs"], []
    for i in range(count):
        pins = math.exp(math.log(1e4) + (i * 0.618034 % 1.0) * (math.log(case["size"]) - math.log(1e4)))
        if i % 2 == 0:
            hg = _generate("random", max(64, int(pins / 4)), 0, seed * 64 + i)
        else:
            hg = _generate("snn", max(66, int(pins / ((LAYERS - 1) * 65))), 64, seed * 64 + i)
        jobs.append((hg, _params(hg.sizes()[0], (2, 8, 32, 0)[(i // 2 + i) % 4], False)))
    return jobs


def prepare(case, seed):
    s = _State()
    s.case = case
    call = case["call"]
    if call == "serve":
        s.server = _server()
        s.jobs = _jobs(case, seed)
        return s
    s.dev = dev = _device()
    hg = _generate(case["kind"], case["size"], case["fanout"], seed)
    n = hg.sizes()[0]
    s.prm = _params(n, case["k"], case["ipm"])
    s.out = _Owned()
    if call == "partition":
        s.part = np.zeros(n, np.int32)
        s.stats = H.RunStats()
        s.hg, s.csr = (hg, None) if case["host"] else (None, _Csr(hg))
        return s
    s.csr = g = _Csr(hg)
    s.sizes = torch.ones(n, dtype=torch.int32, device="cuda")
    cap = _pin_cap(case)
    if g.p > cap:
        raise RuntimeError("the generator's pins exceed their bound")
    words = lambda count: torch.zeros(count, dtype=torch.int32, device="cuda")  # noqa: E731
    longs = lambda count: torch.zeros(count, dtype=torch.int64, device="cuda")  # noqa: E731
    if call == "contract":
        s.own = {"tch": words(cap), "gsizes": words(n), "uoff": longs(n + 1), "hedges": words(cap), "ctch": words(cap),
                 "ctoff": longs(n + 1), "cinb": words(n)}
        cnc = s.prm.candidates_count
        s.pairs = torch.empty(n * cnc, dtype=torch.int32, device="cuda")
        s.scores = torch.empty(n * cnc, dtype=torch.int32, device="cuda")
        return s
    k = case["k"]
    part = _partition_of(n, k, seed)
    s.part0 = _gpu(part)
    if call == "evaluate":
        s.inbound = torch.empty(k, dtype=torch.int32, device="cuda")
        s.own = {"pins": words(cap), "off": longs(g.e + 1), "srcc": words(g.e),
                 "w": torch.zeros(g.e, dtype=torch.float32, device="cuda")}
        return s
    s.psizes0 = _gpu(np.bincount(part, minlength=k).astype(np.uint32))
    s.part, s.psizes = s.part0.clone(), s.psizes0.clone()
    torch.cuda.synchronize()
    s.touching = _Owned()
    s.tch, s.toff, s.inb = _touching(dev, s.touching, g.pins, g.off, g.srcc, n, g.e, dev.lib.hgp_build_touching)
    return s


# ---- one pass -----------------------------------------------------------------------------

def _touching(dev, owned, pins, off, srcc, n, e, build):
    ts, t, o, i = C.c_uint64(), V(), V(), V()
    dev.check(build(dev.ctx, _ptr(pins), _ptr(off), _ptr(srcc), n, e, C.byref(ts), C.byref(t), C.byref(o),
                    C.byref(i)), "touching")
    return owned.tensor(t, ts.value, "<i4"), owned.tensor(o, n + 1, "<i8"), owned.tensor(i, n, "<i4")


def _run_partition(s):
    dev, part = s.dev, s.part.ctypes.data_as(U32P)
    if s.hg is not None:
        st = dev.lib.hgp_partition(dev.ctx, C.byref(s.prm), s.hg.h, part, C.byref(s.stats))
    else:
        g = s.csr
        st = dev.lib.hgp_partition_device(dev.ctx, C.byref(s.prm), g.n, g.e, _ptr(g.pins), _ptr(g.off), _ptr(g.srcc),
                                          _ptr(g.w), part, C.byref(s.stats))
    dev.check(st, "partition")
    return {"part": s.part, "parts": s.stats.num_partitions, "levels": s.stats.levels}


def _run_refine(s):
    dev, g = s.dev, s.csr
    dev.check(dev.lib.hgp_memcpy_dtod(dev.ctx, _ptr(s.part), _ptr(s.part0), 4 * g.n), "copy")
    dev.check(dev.lib.hgp_memcpy_dtod(dev.ctx, _ptr(s.psizes), _ptr(s.psizes0), 4 * s.case["k"]), "copy")
    dev.check(dev.lib.hgp_refine(dev.ctx, C.byref(s.prm), _ptr(g.pins), _ptr(g.off), _ptr(g.srcc), _ptr(s.tch),
                                 _ptr(s.toff), _ptr(s.inb), _ptr(g.w), _ptr(s.sizes), 0, g.n, g.e, s.case["k"], 0,
                                 _ptr(s.part), _ptr(s.psizes), None), "refine")
    return {"part": s.part, "psizes": s.psizes}


def _run_contract(s):
    dev, g, p = s.dev, s.csr, s.prm
    s.out.free()
    own, cnc = s.out, p.candidates_count
    omega, delta = p.max_nodes_per_part, p.max_inbound_per_part
    tch, toff, inb = _touching(dev, own, g.pins, g.off, g.srcc, g.n, g.e, dev.lib.hgp_build_touching)
    dev.check(dev.lib.hgp_candidates(dev.ctx, _ptr(g.pins), _ptr(g.off), _ptr(g.srcc), _ptr(tch), _ptr(toff), _ptr(inb),
                                     _ptr(g.w), _ptr(s.sizes), g.n, g.e, cnc, omega, delta, _ptr(s.pairs),
                                     _ptr(s.scores)), "candidates")
    nn, gr, gs, ug, uo = C.c_uint32(), V(), V(), V(), V()
    dev.check(dev.lib.hgp_group_nodes(dev.ctx, _ptr(inb), _ptr(s.pairs), _ptr(s.scores), _ptr(s.sizes), g.n, cnc, omega,
                                      delta, C.byref(nn), C.byref(gr), C.byref(gs), C.byref(ug), C.byref(uo)), "groups")
    groups, gsizes = own.tensor(gr, g.n, "<i4"), own.tensor(gs, nn.value, "<i4")
    ungroups, uoff = own.tensor(ug, g.n, "<i4"), own.tensor(uo, nn.value + 1, "<i8")
    cs, ch, co, cc = C.c_uint64(), V(), V(), V()
    dev.check(dev.lib.hgp_coarsen_hedges(dev.ctx, _ptr(g.pins), _ptr(g.off), _ptr(g.srcc), _ptr(groups), g.e, g.p,
                                         C.byref(cs), C.byref(ch), C.byref(co), C.byref(cc)), "coarse hedges")
    hedges, hoff, srcc = own.tensor(ch, cs.value, "<i4"), own.tensor(co, g.e + 1, "<i8"), own.tensor(cc, g.e, "<i4")
    ctch, ctoff, cinb = _touching(dev, own, hedges, hoff, srcc, nn.value, g.e, dev.lib.hgp_coarsen_touching)
    kept = {"tch": tch, "gsizes": gsizes, "uoff": uoff, "hedges": hedges, "ctch": ctch, "ctoff": ctoff, "cinb": cinb}
    kept = {name: own.keep(t, s.own[name]) for name, t in kept.items()}
    return {"toff": toff, "inb": inb, "pairs": s.pairs, "scores": s.scores, "groups": groups, "ungroups": ungroups,
            "hoff": hoff, "srcc": srcc, **kept}


def _run_evaluate(s):
    dev, g, k = s.dev, s.csr, s.case["k"]
    s.out.free()
    own = s.out
    km1 = C.c_int64()
    dev.check(dev.lib.hgp_connectivity(dev.ctx, _ptr(g.pins), _ptr(g.off), _ptr(g.w), _ptr(s.part0), g.e,
                                       C.byref(km1)), "connectivity")
    dev.check(dev.lib.hgp_inbound_sizes(dev.ctx, _ptr(g.pins), _ptr(g.off), _ptr(g.srcc), _ptr(s.part0), g.e, k,
                                        _ptr(s.inbound)), "inbound sizes")
    kk, ee, pp, q, o, sc, w = C.c_uint32(), C.c_uint32(), C.c_uint64(), V(), V(), V(), V()
    dev.check(dev.lib.hgp_quotient(dev.ctx, _ptr(g.pins), _ptr(g.off), _ptr(g.srcc), _ptr(g.w), _ptr(s.part0), g.n, g.e,
                                   C.byref(kk), C.byref(ee), C.byref(pp), C.byref(q), C.byref(o), C.byref(sc),
                                   C.byref(w)), "quotient")
    got = {"pins": own.tensor(q, pp.value, "<i4"), "off": own.tensor(o, ee.value + 1, "<i8"),
           "srcc": own.tensor(sc, ee.value, "<i4"), "w": own.tensor(w, ee.value, "<f4")}
    return {"km1": km1.value, "inbound": s.inbound, **{name: own.keep(t, s.own[name]) for name, t in got.items()}}


def _run_serve(s):
    ids = [s.server.submit(hg, prm) for hg, prm in s.jobs]
    return [s.server.wait(i)[0].view(np.int32) for i in ids]


def run(state):
    with torch.cuda.stream(_stream()):
        return _run(state)


def _run(state):
    return {"partition": _run_partition, "refine": _run_refine, "contract": _run_contract, "evaluate": _run_evaluate,
            "serve": _run_serve}[state.case["call"]](state)


# ---- compulsory work and exact results -----------------------------------------------------

def _shape(case):
    """Nodes, hedges and the generators' mean number of pins."""
    size, kind = case["size"], case["kind"]
    if kind == "random":
        return size, size, 4.0 * size
    if kind == "netlist":
        e = round(size * 1.0625)
        return size, e, 4.54 * e
    e = (LAYERS - 1) * size
    return LAYERS * size, e, e * (case["fanout"] + 1.0)


def work(case):
    """Inputs read once (pins 4, offsets 8, source counts 4 and weights 4 bytes) and outputs written
    once.  Integer work only: no floating-point operation is compulsory."""
    if case["call"] == "serve":
        pins = case["jobs"] * (case["size"] - 1e4) / math.log(case["size"] / 1e4)
        return {"bytes": 8.0 * pins, "flops": 0}
    n, e, p = _shape(case)
    csr = 4 * p + 16 * e + 8
    if case["call"] == "partition":
        return {"bytes": csr + 4 * n, "flops": 0}
    if case["call"] == "refine":
        return {"bytes": csr + 4 * p + 20 * n + 4 * n, "flops": 0}
    if case["call"] == "contract":
        return {"bytes": csr + (4 * p + 12 * n) + 128 * n + 16 * n + 0.6 * (8 * p + 12 * n) + 12 * e, "flops": 0}
    return {"bytes": csr + 4 * n, "flops": 0}


def exact(case, seed):
    """lambda-1 from its definition.  The quotient's float weights are sums of unit weights, whole
    numbers, and have no separate value here."""
    if case["call"] != "evaluate":
        return None
    hg = _generate(case["kind"], case["size"], case["fanout"], seed)
    n, off, pins, srcc, w = hg.arrays()
    k = case["k"]
    part = _partition_of(n, k, seed).astype(np.int64)
    hedge = np.repeat(np.arange(len(srcc), dtype=np.int64), np.diff(off.astype(np.int64)))
    lam = np.bincount(np.unique(hedge * k + part[pins.astype(np.int64)]) // k, minlength=len(srcc))
    fixed = np.floor(w.astype(np.float64) * SCALE).astype(np.int64)
    km1 = int((fixed * np.maximum(lam - 1, 0)).sum())
    return {"km1": km1, "inbound": None, "pins": None, "off": None, "srcc": None, "w": None}
