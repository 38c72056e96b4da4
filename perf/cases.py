"""Workloads of the alias-method library, sized as its users size them, for timing it as a whole.

Every case goes through skywalker_amd.capi, the public view of the C interface, with the graph resident on the GPU and the
output buffers in hand, as a program that calls the library batch after batch keeps them.  Graphs are R-MAT (a, b, c, d =
.57, .19, .19, .05) of the sizes the configurations c1 to c5 of bench.py name, or rows of given lengths; weights are
uniform over [1, 100), uniform over (0, 1], or lognormal.

  build        tables of every vertex (the offline mode's first half)
  rebuild      the same from a weight array of the caller's, on rows of lengths spread evenly over the octaves: weights that
               a bias operator or a training step has just changed
  walk         DeepWalk or PPR on tables that exist, with or without the walk index
  node2vec     second-order walk: by rejection on the first-order tables, or with the table of every step
  online_walk  static-bias walk on a graph without tables: the rows the walkers reach are built on the way
  sample       k-hop neighbour sampling, on tables that exist or with the frontier's rows built on the way, children with
               replacement or distinct
"""
import ctypes
import math

import numpy as np
import torch

from skywalker_amd import capi

WEIGHTS = {"uniform": (capi.W_UNIFORM, 1.0, 100.0), "unit": (capi.W_UNIT, 0.0, 0.0),
           "lognormal1": (capi.W_LOGNORMAL, 0.0, 1.0), "lognormal2": (capi.W_LOGNORMAL, 0.0, 2.0)}
MAX_ENTRIES = 28 << 26


def listed():
    return [
        # smallest build: a graph of a unit test or of one community, where launches and waits are all there is
        dict(name="build_tiny", kind="build", scale=10, edge_factor=8, weights="uniform"),
        # an ordinary social graph (c2)
        dict(name="build_medium", kind="build", scale=20, edge_factor=16, weights="unit"),
        # the headline graph, 1.9 G entries (c5)
        dict(name="build_large", kind="build", scale=26, edge_factor=28, weights="lognormal2"),
        # rows of every length, none of them a round number, from weights the caller computed
        dict(name="rebuild_ragged", kind="rebuild", entries=40000003, max_degree=300007, weights="lognormal1"),
        # DeepWalk corpus of a small graph (c1)
        dict(name="deepwalk_small", kind="walk", scale=16, edge_factor=16, weights="uniform", walkers=4096, length=80,
             stop_prob=0.0, index=False),
        # a million walkers on the headline graph (c5): gathers from 30 GB
        dict(name="deepwalk_large", kind="walk", scale=26, edge_factor=28, weights="lognormal2", walkers=1000000, length=80,
             stop_prob=0.0, index=False),
        # PPR queries served again and again from one graph, for which the walk index pays
        dict(name="ppr_indexed", kind="walk", scale=24, edge_factor=16, weights="uniform", walkers=250007, length=100,
             stop_prob=0.15, index=True),
        # node2vec on a large graph (c4), tables in hand
        dict(name="node2vec_reject", kind="node2vec", scale=24, edge_factor=16, weights="uniform", walkers=40000, length=80,
             p=2.0, q=0.5, table=False),
        # the same law the way the reference samples it: the second-order table of every (walker, step)
        dict(name="node2vec_table", kind="node2vec", scale=18, edge_factor=16, weights="uniform", walkers=2000, length=40,
             p=2.0, q=0.5, table=True),
        # a few steps from a few thousand vertices of a large graph whose tables nobody will need
        dict(name="online_walk", kind="online_walk", scale=22, edge_factor=16, weights="lognormal1", walkers=10000, length=8,
             stop_prob=0.0),
        # mini-batches of a GNN's training loop: distinct neighbours, tables in hand
        dict(name="sage_minibatch", kind="sample", scale=20, edge_factor=16, weights="unit", seeds=1024, fanout="25,10",
             online=False, distinct=True),
        # one large batch, the tables of the frontier built on the way (c3)
        dict(name="sage_online", kind="sample", scale=22, edge_factor=32, weights="lognormal1", seeds=40000, fanout="25,10",
             online=True, distinct=False),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _graph(rng, lo, hi, most_entries):
    scale = rng.randint(lo, hi)
    ef = _log(rng, 3, 56)
    return dict(scale=scale, edge_factor=max(3, min(ef, most_entries >> scale)), weights=rng.choice(sorted(WEIGHTS)))


def draw(rng):
    kind = rng.choice(["build", "rebuild", "walk", "node2vec", "online_walk", "sample"])
    if kind == "build":
        return dict(kind=kind, **_graph(rng, 9, 26, MAX_ENTRIES))
    if kind == "rebuild":
        return dict(kind=kind, entries=_log(rng, 100000, 60000000), max_degree=_log(rng, 100, 1000000),
                    weights=rng.choice(sorted(WEIGHTS)))
    if kind == "walk":
        stop = rng.choice([0.0, 0.0, 0.15])
        return dict(kind=kind, **_graph(rng, 14, 26, MAX_ENTRIES), walkers=_log(rng, 100, 1000000),
                    length=rng.choice([100, 100, 50]) if stop else _log(rng, 5, 100), stop_prob=stop, index=rng.random() < 0.3)
    if kind == "node2vec":
        pq = dict(p=rng.choice([0.25, 0.5, 1.0, 2.0, 4.0]), q=rng.choice([0.5, 1.0, 2.0]))
        if rng.random() < 0.3:
            return dict(kind=kind, **_graph(rng, 10, 17, 16 << 17), walkers=_log(rng, 100, 2000), length=_log(rng, 5, 40),
                        table=True, **pq)
        return dict(kind=kind, **_graph(rng, 14, 24, 16 << 24), walkers=_log(rng, 100, 400000), length=_log(rng, 5, 80),
                    table=False, **pq)
    if kind == "online_walk":
        return dict(kind=kind, **_graph(rng, 14, 24, 16 << 24), walkers=_log(rng, 10, 40000), length=rng.randint(1, 16),
                    stop_prob=rng.choice([0.0, 0.0, 0.15]))
    fanout = rng.choice(["25,10", "10,10", "15,10,5", "20", "5,3", "32,7"])
    return dict(kind=kind, **_graph(rng, 12, 22, 32 << 22), seeds=_log(rng, 64, 40000 if fanout != "15,10,5" else 12000),
                fanout=fanout, online=rng.random() < 0.5, distinct=rng.random() < 0.5)


# ------------------------------------------------------------------------------------------------ states
class _View:
    """Device memory of the library as torch sees it (the CUDA array interface; HIP memory speaks it too)."""

    def __init__(self, ptr, count, typestr, stride, keep):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False), "strides": (stride,),
                                         "version": 2}
        self.keep = keep

    def tensor(self):
        return torch.as_tensor(self, device="cuda")


class _Buffer:
    """A torch tensor where capi takes one of its own arrays: anything with the address under `ptr`."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, ctypes.c_void_p(tensor.data_ptr())


def _filled(count, value):
    return _Buffer(torch.full((count,), value, dtype=torch.int32, device="cuda"))


def _fanout(case):
    return [1] + [int(k) for k in case["fanout"].split(",")]


def _degrees(case, seed):
    """Row lengths whose entries are spread evenly over the octaves from 1 to max_degree: the same ones for every seed, in an
    order of the seed's own."""
    rng = np.random.default_rng(case["entries"])
    parts, lo = [], 1
    octaves = case["max_degree"].bit_length()
    for _ in range(octaves):
        hi = min(2 * lo - 1, case["max_degree"])
        parts.append(rng.integers(lo, hi + 1, max(1, int(case["entries"] / octaves / ((lo + hi) / 2)))))
        lo *= 2
    degs = np.concatenate(parts)
    np.random.default_rng(seed).shuffle(degs)
    return degs


def prepare(case, seed):
    kind, s = case["kind"], {"case": case, "seed": seed}
    wk, wa, wb = WEIGHTS[case["weights"]]
    if kind == "rebuild":
        degs = _degrees(case, seed)
        g = capi.Graph.from_degrees(np.concatenate([[0], np.cumsum(degs)]).astype(np.uint32), seed, wk, wa, wb, seed)
        gen = torch.Generator(device="cuda").manual_seed(seed)
        w = torch.empty(g.E + 4, device="cuda")  # the library reads whole 16-byte vectors
        if wk == capi.W_LOGNORMAL:
            w.log_normal_(wa, wb, generator=gen)
        else:
            w.uniform_(wa, wb if wk == capi.W_UNIFORM else 1.0, generator=gen)
        s.update(g=g, weights=_Buffer(w))
        return s
    g = capi.Graph.rmat(case["scale"], case["edge_factor"], seed, wk, wa, wb, seed)
    s["g"] = g
    if kind == "build":
        return s
    n = case["seeds"] if kind == "sample" else case["walkers"]
    s["seeds"] = g.gen_seeds(seed, n)
    if kind == "sample":
        per_seed, lengths = capi.sample_layout(_fanout(case))
        s["out"] = (_filled(n * per_seed, -1), _filled(n * lengths, 0))
        g.set_option("sample_distinct", int(case["distinct"]))
    else:
        s["out"] = (_filled(n * (case["length"] + 1), -1), _filled(n, 0))
    if kind == "online_walk":
        g.set_option("online_full_build", 0)
    if kind == "walk" or (kind == "node2vec" and not case["table"]) or (kind == "sample" and not case["online"]):
        g.build_tables()
    if case.get("index"):
        g.build_walk_index()
    return s


def _tables(s):
    if "tables" not in s:  # the arrays stay where the first build put them
        g = s["g"]
        _, _, _, table, valid = g.device_ptrs()
        s["tables"] = {"prob": _View(table, g.E, "<f4", 8, g).tensor(), "alias": _View(table + 4, g.E, "<i4", 8, g).tensor(),
                       "valid": _View(valid, g.V, "|i1", 1, g).tensor()}
    return s["tables"]


def run(s):
    case, g = s["case"], s["g"]
    kind = case["kind"]
    if kind == "build":
        g.build_tables()
        return _tables(s)
    if kind == "rebuild":
        g.build_tables_from_weights(s["weights"])
        return _tables(s)
    if kind == "walk":
        _, _, sampled, _ = g.walk_offline(s["seeds"], case["length"], case["stop_prob"], s["seed"], out=s["out"])
    elif kind == "node2vec":
        bias = capi.BIAS_NODE2VEC if case["table"] else capi.BIAS_NODE2VEC_REJECT
        _, _, sampled, _ = g.walk_online(bias, case["p"], case["q"], s["seeds"], case["length"], 0.0, s["seed"], out=s["out"])
    elif kind == "online_walk":
        _, _, sampled, _ = g.walk_online(capi.BIAS_STATIC, 1.0, 1.0, s["seeds"], case["length"], case["stop_prob"], s["seed"],
                                         out=s["out"])
    else:
        fn = g.sample_online if case["online"] else g.sample_offline
        _, _, sampled, _ = fn(s["seeds"], _fanout(case), s["seed"], out=s["out"])
    return {"out": s["out"][0].tensor, "lengths": s["out"][1].tensor, "sampled": sampled}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _rmat_rows(case):
    """(rows, entries of each) by the number of one bits of the vertex id: what the generator gives on average."""
    s, e = case["scale"], case["edge_factor"] << case["scale"]
    return [(math.comb(s, k), e * 0.76 ** (s - k) * 0.24 ** k) for k in range(s + 1)]


def _live(case):
    """Share of the vertices that have an edge."""
    return sum(n * (1 - math.exp(-d)) for n, d in _rmat_rows(case)) / 2 ** case["scale"]


def _steps(case):
    """Steps of one walker on average: it ends where a vertex has no edge, which 0.14 / edge_factor of the edges lead to."""
    go, q = 1 - case.get("stop_prob", 0.0), 1 - min(0.5, 0.14 / case["edge_factor"])
    return _live(case) * sum(go ** k * q ** (k - 1) for k in range(1, case["length"] + 1))


def _entries_reached(case, draws):
    """Entries of the distinct rows that `draws` steps along random edges reach."""
    e = case["edge_factor"] << case["scale"]
    return sum(n * d * (1 - math.exp(-draws * d / e)) for n, d in _rmat_rows(case))


def work(case):
    kind = case["kind"]
    if kind in ("build", "rebuild"):
        if kind == "build":
            e, v = case["edge_factor"] << case["scale"], 1 << case["scale"]
        else:
            degs = _degrees(case, 0)
            e, v = int(degs.sum()), len(degs)
        # weight read, entry written, row offset read, flag written; a conversion, a sum, a product and a difference per entry
        return {"bytes": 12 * e + 5 * v, "flops": 4 * e}
    if kind == "sample":
        fan, parents, children, total = _fanout(case), case["seeds"], 0.0, 0.0
        filled = 0.35 * (case["edge_factor"] / 16) ** 0.25  # the first parents are ordinary vertices, later ones well connected
        reached = 0.0
        parents *= _live(case)
        for k in fan[1:]:
            reached += parents
            children = parents * k * min(1.0, filled)
            total += children * 16 + parents * 16  # entry, neighbour id, slot written; row bounds, parent, count
            parents, filled = children, 0.92
        if case["online"]:
            total += 12 * _entries_reached(case, reached)
        return {"bytes": total, "flops": 0}
    steps = case["walkers"] * _steps(case)
    # row bounds, entry, neighbour id, vertex written; start vertex, its slot and the length
    total = 24 * steps + 12 * case["walkers"]
    if kind == "online_walk":
        total += 12 * _entries_reached(case, steps)
    elif kind == "node2vec" and not case["table"]:
        total += 12 * steps  # at least one rejected or tested candidate's entry and membership
    elif kind == "node2vec":
        rows = _rmat_rows(case)
        total += 12 * steps * sum(n * d * d for n, d in rows) / sum(n * d for n, d in rows)
    return {"bytes": total, "flops": 0}


def tolerance(case):
    """Tables are a pure function of the weights by exact integer sums, draws one of the seed: every bit is determined."""
    return "exact"
