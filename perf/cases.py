"""The work that users of this package have it do, as cases to be timed.

A case is one call through the public Python face: a finder that is kept and
run again, one call that builds, runs and frees everything, the entry point
that allocates nothing, a batch of graphs, and a server fed with requests.
All graphs come from the package's seeded generators in the sizes of its own
workloads (gmbe_amd/workloads.py) and tests, run as the command line runs them
(`-t 1 -o 1 -f`, bound_height 20, bound_size 1500).

Outputs are the count of maximal bicliques and the two digest words, as whole
64-bit numbers: they are the same for every correct traversal, so there is no
rounding to be compared against a value in higher precision.
"""
import math
import random

import numpy as np

from gmbe_amd import Batch, BiGraph, GenParams, IterFinderGpu6, Server, enumerate_graph
from gmbe_amd.finder import execute_static
from gmbe_amd.workloads import BOUND_HEIGHT, BOUND_SIZE, RUN_OPTION, gen_params

UNIFORM, POWERLAW, PLANTED = 1, 2, 3


def _graph(name, how, kind, nU, nV, m, cap=0, blocks=0, begin=0, stride=1):
    """A case on one generated graph. `how` is the entry point: "finder"
    (created once, executed on every pass), "oneshot" or "static". `begin` and
    `stride` choose the top-level vertices by processing rank (heaviest first)."""
    return dict(name=name, how=how, kind=kind, nU=nU, nV=nV, m=m, cap=cap, blocks=blocks,
                begin=begin, stride=stride)


def _powerlaw(name, scale, **more):
    """The gamma 2.1 power-law graph (100,000 x 200,000, 1.5M edges), scaled."""
    p = gen_params(2, scale)
    return _graph(name, "finder", POWERLAW, p.nU, p.nV, int(p.m), p.cap, **more)


def _planted(name, scale):
    """The gamma 2.0 graph with planted near-bicliques (50,000 x 1,000,000), scaled."""
    p = gen_params(3, scale)
    return _graph(name, "finder", PLANTED, p.nU, p.nV, int(p.m), p.cap, p.blocks)


def listed():
    return [
        # the smallest call: a few hundred edges, where launches and latency are all there is
        _graph("tiny_uniform", "finder", UNIFORM, 97, 61, 400),
        # the package's first workload: 2,000 x 1,500, 12,000 edges, a kept finder
        _graph("uniform_12k", "finder", UNIFORM, 2000, 1500, 12000),
        # the same size as a program with one graph calls it: create, run, free
        _graph("oneshot_12k", "oneshot", UNIFORM, 2000, 1500, 12000),
        # callers that cannot allocate device memory; odd sizes
        _graph("static_uniform", "static", UNIFORM, 1013, 797, 5501),
        # a sparse graph without hubs: many light top-level vertices
        _graph("uniform_240k", "finder", UNIFORM, 20011, 15013, 240000),
        # ordinary power-law graphs: a few hub subtrees hold most of the work
        _powerlaw("powerlaw_30k", 0.02),
        _graph("powerlaw_77k", "finder", POWERLAW, 5131, 10243, 77003, 1027),
        # dense overlapping near-bicliques: tens of millions of results
        _planted("planted_41k", 0.005),
        # the full-size power-law graph: its light top-level vertices, bound by
        # the two-hop neighbourhoods and not by the subtrees
        _powerlaw("powerlaw_1500k_light", 1.0, begin=20000),
        # and one in 400 of all its vertices, the largest hub among them
        _powerlaw("powerlaw_1500k_hubs", 1.0, stride=400),
        # many small graphs in one batch
        dict(name="batch_96", how="batch", n=96, lo=50, hi=2000, dlo=3.0, dhi=10.0),
        # a burst of requests to a server: half stand-alone graphs, half
        # two-hop neighbourhoods cut from the resident graph
        dict(name="serve_64", how="serve", n=64, lo=50, hi=2000, dlo=3.0, dhi=8.0, scale=0.1,
             max_edges=5000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "oneshot", "static", "powerlaw", "powerlaw",
                       "planted", "light", "hubs", "batch", "serve"])
    if kind in ("uniform", "oneshot", "static"):
        nU = _log_int(rng, 60, 2500 if kind == "static" else 20000)
        nV = max(50, int(nU * rng.uniform(0.5, 1.5)))
        m = int(max(nU, nV) * rng.uniform(4.0, 12.0))
        return {k: v for k, v in _graph("", "finder" if kind == "uniform" else kind, UNIFORM, nU, nV,
                                        m).items() if k != "name"}
    if kind == "powerlaw":
        scale = math.exp(rng.uniform(math.log(0.003), math.log(0.06)))
        nU, nV = int(100000 * scale), int(200000 * scale * rng.uniform(0.7, 1.3))
        c = _graph("", "finder", POWERLAW, nU, nV, int(1500000 * scale), max(300, int(20000 * scale)))
    elif kind == "planted":
        c = _planted("", rng.uniform(0.0015, 0.0045))
    elif kind == "light":
        c = _powerlaw("", 1.0, begin=rng.randrange(20000, 60000), stride=rng.randrange(1, 20))
    elif kind == "hubs":
        c = _powerlaw("", 1.0, begin=rng.randrange(600, 4000), stride=rng.randrange(100, 400))
    elif kind == "batch":
        c = dict(how="batch", n=_log_int(rng, 4, 96), lo=50, hi=2000, dlo=3.0, dhi=rng.uniform(5.0, 9.0))
    else:
        c = dict(how="serve", n=_log_int(rng, 4, 128), lo=50, hi=rng.randrange(500, 2000), dlo=3.0,
                 dhi=rng.uniform(5.0, 8.0), scale=0.1, max_edges=_log_int(rng, 500, 5000))
    c.pop("name", None)
    return c


def _generate(case, seed):
    p = GenParams()
    p.kind, p.nU, p.nV, p.m, p.seed = case["kind"], case["nU"], case["nV"], case["m"], seed
    p.gamma_u = p.gamma_v = 2.0 if case["kind"] == PLANTED else 2.1
    p.cap = case["cap"]
    if case["kind"] == PLANTED:
        q = gen_params(3)
        p.blocks, p.block_min, p.drop = case["blocks"], q.block_min, q.drop
        p.block_max = min(q.block_max, case["nU"], case["nV"])
    return BiGraph.generate(p)


def _small(case, rng):
    return BiGraph.generate_small(rng.getrandbits(63), case["lo"], case["hi"], case["dlo"],
                                  case["dhi"], 2.2)


def prepare(case, seed):
    rng = random.Random(seed)
    how = case["how"]
    if how == "batch":
        graphs = [_small(case, rng).derive(**RUN_OPTION) for _ in range(case["n"])]
        return dict(how=how, batch=Batch(graphs, BOUND_HEIGHT, BOUND_SIZE))
    if how == "serve":
        p = gen_params(2, case["scale"])
        p.seed = rng.getrandbits(63)
        resident = BiGraph.generate(p)
        requests = [(_small(case, rng), 0) if i % 2 else (None, rng.randrange(p.nU))
                    for i in range(case["n"])]
        server = Server(resident, slots=256, mem_budget=1 << 28, bound_height=BOUND_HEIGHT,
                        bound_size=BOUND_SIZE)
        return dict(how=how, server=server, requests=requests, max_edges=case["max_edges"])
    graph = _generate(case, seed).derive(**RUN_OPTION)
    if how != "finder":
        return dict(how=how, graph=graph)
    knobs = {}
    if case["begin"] or case["stride"] > 1:
        # part of a large graph: memory knobs that leave room for other finders on the card
        knobs = dict(root_begin=case["begin"], root_stride=case["stride"],
                     root_phase=case["begin"] % case["stride"], arena_kb=8192, ctx_kb=512)
    return dict(how=how, finder=IterFinderGpu6(graph, BOUND_HEIGHT, BOUND_SIZE, **knobs))


def _digest(results):
    """Rows of (maximal bicliques, hash sum, hash xor), the words as int64."""
    rows = [(r.maximal, r.hash_sum, r.hash_xor) for r in results]
    return np.array(rows, dtype=np.uint64).view(np.int64)


def run(state):
    how = state["how"]
    if how == "finder":
        return _digest([state["finder"].execute()])
    if how == "oneshot":
        return _digest([enumerate_graph(state["graph"], BOUND_HEIGHT, BOUND_SIZE)])
    if how == "static":
        return _digest([execute_static(state["graph"], BOUND_HEIGHT, BOUND_SIZE)])
    if how == "batch":
        per_graph, _ = state["batch"].execute()
        return _digest(per_graph)
    server, tickets, done = state["server"], [], {}
    for graph, u in state["requests"]:
        tickets.append(server.submit_graph(graph) if graph is not None
                       else server.submit_ego(u, state["max_edges"]))
    while len(done) < len(tickets):
        for d in server.poll(wait=True):
            done[d.ticket] = d
    done = [done[t] for t in tickets]
    return dict(status=np.array([d.status for d in done], dtype=np.int64), digest=_digest(done))


def _csr_bytes(nU, nV, m):
    """Both CSR directions, the offsets and the hash keys of each side."""
    return 8.0 * m + 16.0 * (nU + nV + 1)


def work(case):
    """Each graph read once and each result written once. The enumeration
    itself has no operation count that follows from the sizes."""
    if case["how"] in ("batch", "serve"):
        # the generator's means: sides log-uniform in [lo, hi], degrees uniform
        side = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        graph = _csr_bytes(side, side, side * (case["dlo"] + case["dhi"]) / 2) + 24.0
        if case["how"] == "batch":
            return dict(bytes=case["n"] * graph, flops=0)
        ego = 8.0 * case["max_edges"] + 24.0
        return dict(bytes=case["n"] * (graph + ego) / 2, flops=0)
    return dict(bytes=_csr_bytes(case["nU"], case["nV"], case["m"]) + 24.0, flops=0)
