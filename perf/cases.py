"""Performance cases of dyng_amd: what a program that uses this framework has it do, each through the
public entry points, over the sizes of the benchmark's configurations (``bench.py``) and generic ones.

A case is a dict of plain values; ``listed()`` names twelve, ``draw(rng)`` gives more of the same
ranges. Inputs are drawn on the GPU from the seed alone: graphs with distinct non-loop edges
(Erdos-Renyi, RMAT, 4-neighbour grids with random shortcuts) and uniform integer weights, resident on
the device; batches of operations against them.

An update case's pass is one update: a state holds a few batches and, for each, the batch that undoes
it, and passes go through them in turn, so every pass finds the work of a running stream (a graph
whose rows carry the edits of earlier batches) and a state can be passed over any number of times.
The outputs are the trees as the result holds them on the device (distances and parents, whole) and the
update's counts.
"""

import ctypes
import math

import numpy as np
import torch

import dyng_amd as dyng
from dyng_amd import _lib, batched, hyper_sssp, mosp, sssp

DEVICE = "cuda:0"
RMAT_A, RMAT_B, RMAT_C = 0.57, 0.19, 0.19
GIVEN = 6  # batches of a state (each with its undoing)


def listed():
    return [
        # the smallest call: a handful of operations on a small graph, where latency and launches count
        {"name": "er1k_update10", "kind": "update", "graph": "er", "n": 1000, "m": 8000, "wmax": 100,
         "ops": 10, "mix": "ins_del", "host": False},
        # bench.py's er64k_mixed1k, its batches handed over as numpy arrays (the Python API's usual call)
        {"name": "er64k_update1k_host", "kind": "update", "graph": "er", "n": 65_536, "m": 1_048_576,
         "wmax": 100, "ops": 1000, "mix": "ins_del", "host": True},
        # a small batch on a large graph: the low end of bench.py's stream of uneven batches
        {"name": "rmat22_update1k", "kind": "update", "graph": "rmat", "n": 1 << 22, "m": 67_108_864,
         "wmax": 255, "ops": 1001, "mix": "ins_del", "host": False},
        # the headline workload (rmat22_mixed100k): 40 % insertions, 40 % deletions, 20 % reweights
        {"name": "rmat22_update100k", "kind": "update", "graph": "rmat", "n": 1 << 22, "m": 67_108_864,
         "wmax": 255, "ops": 100_000, "mix": "mixed", "host": False},
        # the high end of the stream of uneven batches (rmat23_learned)
        {"name": "rmat23_update1m", "kind": "update", "graph": "rmat", "n": 1 << 23, "m": 134_217_728,
         "wmax": 255, "ops": 1_000_000, "mix": "ins_del", "host": False},
        # a road-like graph (grid4096_tree10k): deep trees, 80 % of the deletions on tree edges
        {"name": "grid4096_update10k", "kind": "update", "graph": "grid", "n": 4096 * 4096, "m": 67_160_000,
         "wmax": 1000, "ops": 10_000, "mix": "tree", "host": False},
        # the first tree of a large skewed graph: compute from a source
        {"name": "rmat22_compute", "kind": "compute", "graph": "rmat", "n": 1 << 22, "m": 67_108_864, "wmax": 255},
        # the first tree of a deep graph, its side no power of two
        {"name": "grid1001_compute", "kind": "compute", "graph": "grid", "n": 1001 * 1001, "m": 4_008_000, "wmax": 1000},
        # several results on one graph: one batch, four sources (dyng_amd.update)
        {"name": "rmat20_four_trees", "kind": "several", "graph": "rmat", "n": 1 << 20, "m": 16_777_216,
         "wmax": 255, "ops": 10_007, "mix": "mixed", "results": 4},
        # MOSP with three objectives on its own graph format (appended rows, parallel edges allowed),
        # bench.py's preferences
        {"name": "rmat20_mosp3", "kind": "mosp", "graph": "rmat", "n": 1 << 20, "m": 16_777_216, "wmax": 255,
         "ops": 30_011, "mix": "ins_del", "objectives": 3, "costs": True},
        # many independent trees repaired in one launch (batched256_rmat): RMAT graphs of 2^10 to 2^16
        # vertices, 1 % of every instance's edges changed, the launch replayed from a hipGraph
        {"name": "batched64_rmat", "kind": "batched", "instances": 64, "low": 10.0, "high": 16.0, "wmax": 100},
        # shortest hyperpaths (hyper_uniform, half its size): hyperedge and incidence edits
        {"name": "hyper100k_update1k", "kind": "hyper", "vertices": 50_000, "hyperedges": 100_000, "wmax": 100,
         "ops": 1000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: every kind of the listed ones, sizes over the logarithm of their ranges."""
    kind = rng.choice(["update", "update", "update", "update", "compute", "several", "mosp", "batched", "hyper"])
    if kind == "batched":
        low = rng.uniform(8.0, 11.0)
        return {"kind": kind, "instances": rng.randint(8, 64), "low": round(low, 2),
                "high": round(rng.uniform(low + 1.0, 15.5), 2), "wmax": rng.choice([50, 100, 255])}
    if kind == "hyper":
        v = _log_int(rng, 2000, 50_000)
        return {"kind": kind, "vertices": v, "hyperedges": int(v * rng.uniform(1.0, 2.0)), "wmax": rng.choice([100, 255]),
                "ops": _log_int(rng, 8, max(9, min(1000, v // 20)))}
    graph = rng.choice(["er", "rmat", "rmat", "grid"])
    top = {"update": 22.0, "compute": 21.5, "several": 19.5, "mosp": 19.5}[kind]
    if graph == "grid":
        side = _log_int(rng, 50, min(2500, 2.0 ** (top / 2)))
        n, m, wmax = side * side, 4 * side * (side - 1), rng.choice([100, 1000])
        m += -(-m // 1000)
    else:
        n = _log_int(rng, 1000, 2.0 ** (min(top, 18.0) if graph == "er" else top))
        if graph == "rmat":
            n = 1 << max(10, n.bit_length() - 1)
        m, wmax = int(n * rng.uniform(6.0, 16.0)), rng.choice([100, 255])
    case = {"kind": kind, "graph": graph, "n": n, "m": m, "wmax": wmax}
    if kind == "compute":
        return case
    case["ops"] = _log_int(rng, 10, max(12, min(300_000, m // 40)))
    case["mix"] = rng.choice(["mixed", "ins_del"] if graph != "grid" else ["tree", "ins_del"])
    if kind == "update":
        case["host"] = rng.random() < 0.25
    elif kind == "several":
        case["results"] = rng.randint(2, 6)
    else:
        case["objectives"], case["mix"], case["costs"] = rng.randint(2, 4), "ins_del", rng.random() < 0.75
    return case


# ---- inputs, drawn on the GPU ----


def _generator(seed, part):
    g = torch.Generator(device=DEVICE)
    g.manual_seed((int(seed) * 1_000_003 + part) & 0x7FFFFFFFFFFFFFFF)
    return g


def _rand_int(gen, high, count):
    return torch.randint(0, int(high), (int(count),), generator=gen, device=DEVICE, dtype=torch.int64)


def _pairs(graph, n, count, gen):
    """`count` endpoint pairs as keys u * n + v: uniform, or RMAT's quadrants bit by bit."""
    if graph != "rmat":
        return _rand_int(gen, n, count) * n + _rand_int(gen, n, count)
    u = torch.zeros(count, dtype=torch.int64, device=DEVICE)
    v = torch.zeros(count, dtype=torch.int64, device=DEVICE)
    for _ in range(int(n).bit_length() - 1):
        r = torch.rand(count, generator=gen, device=DEVICE)
        u = 2 * u + (r >= RMAT_A + RMAT_B)
        v = 2 * v + (((r >= RMAT_A) & (r < RMAT_A + RMAT_B)) | (r >= RMAT_A + RMAT_B + RMAT_C))
    return u * n + v


def _distinct(graph, n, count, gen, avoid=None):
    """`count` distinct non-loop keys (sorted), none of them in `avoid` (sorted)."""
    keys, want = None, count
    while keys is None or len(keys) < count:
        new = _pairs(graph, n, want + want // 4 + 64, gen)
        new = new[new // n != new % n]
        if avoid is not None:
            at = torch.searchsorted(avoid, new).clamp_(max=len(avoid) - 1)
            new = new[avoid[at] != new]
        keys = torch.unique(new if keys is None else torch.cat([keys, new]))
        want = max(64, 2 * (count - len(keys)))
    if len(keys) > count:  # leave out random ones
        drop = torch.zeros(len(keys), dtype=torch.bool, device=DEVICE)
        drop[torch.randperm(len(keys), generator=gen, device=DEVICE)[: len(keys) - count]] = True
        keys = keys[~drop]
    return keys


def _grid_keys(n, m, gen):
    """The arcs between 4-neighbours of a square grid, and m - arcs random shortcuts (at least none)."""
    side = math.isqrt(n)
    v = torch.arange(n, dtype=torch.int64, device=DEVICE)
    c, r = v % side, v // side
    arcs = torch.cat([(v * n + v + d)[ok] for d, ok in ((1, c + 1 < side), (-1, c > 0), (side, r + 1 < side), (-side, r > 0))])
    arcs, _ = torch.sort(arcs)
    more = max(0, m - len(arcs))
    if not more:
        return arcs
    return torch.sort(torch.cat([arcs, _distinct("er", n, more, gen, avoid=arcs)]))[0]


def _keys(case, gen):
    if case["graph"] == "grid":
        return _grid_keys(case["n"], case["m"], gen)
    return _distinct(case["graph"], case["n"], case["m"], gen)


def _graph(n, keys, w, properties=None):
    """The device graph of an edge list that is on the device already: the library's C entry point takes
    device pointers (from_device = 1), which Graph.from_edges does not offer."""
    src, dst = (keys // n).to(torch.int32), (keys % n).to(torch.int32)
    w = w.to(torch.int32).contiguous()
    props = properties or dyng.GraphProperties()
    handle, native = ctypes.c_void_p(), props._native()
    torch.cuda.synchronize()
    _lib.check(_lib.lib().dyng_hip_graph_create_from_edges(
        0, ctypes.byref(native), n, len(keys), w.shape[1], src.data_ptr(), dst.data_ptr(), w.data_ptr(), 1, None,
        ctypes.byref(handle)))
    dyng.synchronize()
    return dyng.Graph._wrap(handle, dyng.Resources.hip(), props, w.shape[1])


def _array(x, host):
    a = np.ascontiguousarray(x.to(torch.int32).cpu().numpy())
    return a if host else dyng.DeviceArray(a)


def _edge_batch(n, ins, ins_w, dele, host):
    """Insertions `ins` (keys) with weights `ins_w` and deletions `dele` (keys) as an EdgeBatch."""
    return dyng.EdgeBatch(insert=(_array(ins // n, host), _array(ins % n, host), _array(ins_w, host)),
                          delete=(_array(dele // n, host), _array(dele % n, host)))


def _batches(case, n, keys, w, gen, host, parents=None):
    """GIVEN batches against the graph, each followed by the one that undoes it."""
    ops, mix, graph = case["ops"], case["mix"], case["graph"]
    wmax, K = case["wmax"], w.shape[1]
    tree = None
    if mix == "tree":
        v = torch.nonzero(parents >= 0).reshape(-1)
        tree = parents[v].to(torch.int64) * n + v
        tree = torch.searchsorted(keys, torch.sort(tree)[0])
    out = []
    for _ in range(GIVEN):
        if mix == "tree":  # half insertions, four tenths deletions of tree edges, one tenth of any edges
            n_ins, n_rew, n_tree = ops // 2, 0, min(len(tree), (2 * ops) // 5)
            n_del = max(0, ops - n_ins - n_tree)
        elif mix == "mixed":
            n_ins, n_rew, n_tree = (2 * ops) // 5, ops // 5, 0
            n_del = ops - n_ins - n_rew
        else:
            n_ins, n_rew, n_tree = ops // 2, 0, 0
            n_del = ops - n_ins
        new = _distinct(graph if graph != "grid" else "er", n, n_ins, gen, avoid=keys)
        new = new[torch.randperm(len(new), generator=gen, device=DEVICE)]
        new_w = 1 + _rand_int(gen, wmax, len(new) * K).reshape(-1, K)
        at = torch.randint(0, len(keys), (4 * (n_del + n_rew) + 64,), generator=gen, device=DEVICE)
        if n_tree:
            at = torch.cat([tree[torch.randperm(len(tree), generator=gen, device=DEVICE)[:n_tree]], at])
        # the first n_tree + n_del + n_rew distinct edges in the order they were drawn
        kept, first = torch.unique(at, return_inverse=True)
        when = torch.full((len(kept),), len(at), dtype=torch.int64, device=DEVICE)
        when.scatter_reduce_(0, first, torch.arange(len(at), device=DEVICE), "amin")
        at = at[torch.sort(when)[0][: n_tree + n_del + n_rew]]
        gone, again = at[: n_tree + n_del], at[n_tree + n_del:]
        again_w = 1 + _rand_int(gen, wmax, len(again) * K).reshape(-1, K)
        out.append(_edge_batch(n, torch.cat([new, keys[again]]), torch.cat([new_w, again_w]), keys[gone], host))
        out.append(_edge_batch(n, keys[at], w[at], new, host))
    return out


class _Memory:
    """Device memory of `owner` (a result) as torch's array interface names it. A tensor made from it holds
    it, and so the result: the memory lives as long as the tensor."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": kind, "version": 2}


def _view(state, name, owner, ptr, shape, kind):
    """A tensor over device memory of `owner`; made once while the memory stays where it is."""
    have = state["views"].get(name)
    if have is None or have[0] is not owner or have[1] != (ptr, shape):
        have = (owner, (ptr, shape), torch.as_tensor(_Memory(owner, ptr, shape, kind), device=DEVICE))
        state["views"][name] = have
    return have[2]


def _tree(state, name, result):
    d, p, n = result.device_arrays()
    return [_view(state, name + ".d", result, d, (n,), "<i8"), _view(state, name + ".p", result, p, (n,), "<i4")]


def _rows(rng, V, count, k):
    """`count` rows of `k` distinct vertices."""
    rows = rng.integers(0, V, (count, k))
    while True:
        again = (np.diff(np.sort(rows, axis=1), axis=1) == 0).any(axis=1)
        if not again.any():
            return rows
        rows[again] = rng.integers(0, V, (int(again.sum()), k))


def _prepare_hyper(case, seed):
    rng = np.random.default_rng(seed)
    V, H, ops, wmax = case["vertices"], case["hyperedges"], case["ops"], case["wmax"]
    half = H // 2  # hyperedges below it (of 4 members) are replaced, those above it (2 to 6) gain and lose members
    lists = list(_rows(rng, V, half, 4)) + [rng.integers(0, V, int(k)) for k in rng.integers(2, 7, H - half)]
    h = dyng.Hypergraph.from_lists(lists, rng.integers(1, wmax + 1, H), num_vertices=V)
    r = hyper_sssp.compute(h, int(np.argmax(np.bincount(np.concatenate(lists), minlength=V))))
    part, batches = max(1, ops // 4), []
    for _ in range(GIVEN):
        ids = half + rng.choice(H - half, 2 * part, replace=False)
        own = (ids[:part], np.asarray([lists[i][0] for i in ids[:part]]))
        other = (ids[part:], rng.integers(0, V, part))
        for lose, gain in ((own, other), (other, own)):
            batches.append(dyng.HyperedgeBatch(
                rng.choice(half, part, replace=False), list(_rows(rng, V, part, 4)), rng.integers(1, wmax + 1, part),
                delete_incidences=lose, insert_incidences=gain))
    return {"hypergraph": h, "tree": r, "batches": batches}


def _prepare_batched(case, seed):
    gen, graphs, sources, drawn = _generator(seed, 0), [], [], []
    count = case["instances"]
    for i in range(count):  # sizes spread over the logarithm of the range
        scale = int(case["low"] + (case["high"] - case["low"]) * i / max(1, count - 1))
        n, m = 1 << scale, 16 << scale
        keys = _distinct("rmat", n, m, gen)
        w = 1 + _rand_int(gen, case["wmax"], m).reshape(-1, 1)
        sources.append(torch.argmax(torch.bincount(keys // n, minlength=n)))
        drawn.append((n, keys, w))
        graphs.append((n, (keys // n).cpu().numpy(), (keys % n).cpu().numpy(), w.cpu().numpy()))
    inst = batched.Instances(graphs)
    tree = inst.compute([int(s) for s in sources])
    tree.set_tuning(sssp.Tuning(launch="graph"))
    total, batches = int(inst.offsets[-1]), []
    for _ in range(GIVEN):
        parts = [[] for _ in range(4)]
        for (n, keys, w), lo in zip(drawn, inst.offsets[:-1].tolist()):
            half = max(1, len(keys) // 200)
            new = _distinct("rmat", n, half, gen, avoid=keys)
            gone = torch.randperm(len(keys), generator=gen, device=DEVICE)[:half]
            up = lambda k: (k // n + lo) * total + k % n + lo  # noqa: E731
            for p, x in zip(parts, (up(new), 1 + _rand_int(gen, case["wmax"], half).reshape(-1, 1), up(keys[gone]), w[gone])):
                p.append(x)
        new, new_w, gone, gone_w = (torch.cat(p) for p in parts)
        batches += [_edge_batch(total, new, new_w, gone, False), _edge_batch(total, gone, gone_w, new, False)]
    return {"graph": inst.graph, "tree": tree, "batches": batches}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "hyper":
        state = _prepare_hyper(case, seed)
    elif kind == "batched":
        state = _prepare_batched(case, seed)
    else:
        gen, n, K = _generator(seed, 1), case["n"], case.get("objectives", 1)
        keys = _keys(case, gen)
        w = 1 + _rand_int(gen, case["wmax"], len(keys) * K).reshape(-1, K)
        g = _graph(n, keys, w, dyng.GraphProperties.mosp_compatible() if kind == "mosp" else None)
        degree = torch.bincount(keys // n, minlength=n)
        by_degree = torch.argsort(degree, descending=True, stable=True)
        source = int(by_degree[0]) if case["graph"] != "grid" else 0
        state = {"graph": g, "source": source}
        if kind == "update":
            state["tree"] = sssp.compute(g, source)
        elif kind == "several":
            state["trees"] = [sssp.compute(g, int(s)) for s in by_degree[: case["results"]]]
        elif kind == "mosp":
            state["paths"] = mosp.compute(g, source, preferences=[4 if k % 2 == 0 else 1 for k in range(K)],
                                          compute_path_costs=case["costs"])
        if kind != "compute":
            parents = None
            if case["mix"] == "tree":
                first = state.get("tree") or (state["trees"][0] if kind == "several" else state["paths"].tree(0))
                parents = torch.from_numpy(first.parents).to(DEVICE)
            state["batches"] = _batches(case, n, keys, w, gen, case.get("host", False), parents)
    state.update(kind=kind, views={}, turn=0)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return state


def run(state):
    """One pass: one update with the next batch, or one computation of a tree."""
    kind = state["kind"]
    if kind == "compute":
        state["tree"] = sssp.compute(state["graph"], state["source"])
        return _tree(state, "tree", state["tree"])
    batch = state["batches"][state["turn"]]
    state["turn"] = (state["turn"] + 1) % len(state["batches"])
    if kind == "hyper":
        st = hyper_sssp.update(state["hypergraph"], batch, state["tree"])
        return [state["tree"].hyperedge_distances, state["tree"].hyperedge_parents, st.line_graph_insertions,
                st.line_graph_deletions]
    g = state["graph"]
    if kind in ("update", "batched"):
        st = sssp.update(g, batch, state["tree"])
        return _tree(state, "tree", state["tree"]) + [st.affected, st.invalidated]
    if kind == "several":
        st = dyng.update(g, batch, *state["trees"])
        out = [s.affected for s in st]
        for i, t in enumerate(state["trees"]):
            out += _tree(state, "tree%d" % i, t)
        return out
    paths = state["paths"]
    st = mosp.update(g, batch, paths)
    d, p, n = paths.combined_device_arrays()
    out = [_view(state, "cd", paths, d, (n,), "<i8"), _view(state, "cp", paths, p, (n,), "<i4"), st.affected, st.combined_edges]
    if paths.options.compute_path_costs:
        c, n, k = paths.path_costs_device()
        out.append(_view(state, "costs", paths, c, (n, k), "<i8"))
    for k in range(paths.num_objectives):
        out += _tree(state, "tree%d" % k, paths.tree(k))
    return out


def work(case):
    """Bytes a pass cannot do without. An update reads its operations, and for each the row ends (8 B) and
    the entry (id and weights) in the out- and in-rows and the words of its two ends, and writes the entry;
    the trees' changed part depends on the data and is left out. A computation reads every row end and
    edge once and writes every distance and parent."""
    kind = case["kind"]
    if kind == "compute":
        return {"bytes": 8 * case["m"] + 20 * case["n"], "flops": 0}
    if kind == "hyper":
        # every edited hyperedge's members' other hyperedges become or cease to be neighbours
        pairs = case["ops"] * 4 * 4 * case["hyperedges"] // max(1, case["vertices"])
        return {"bytes": 40 * 2 * pairs + 12 * case["hyperedges"], "flops": 0}
    if kind == "batched":
        count = case["instances"]
        ops = sum(2 * max(1, (16 << int(case["low"] + (case["high"] - case["low"]) * i / max(1, count - 1))) // 200)
                  for i in range(count))
        return {"bytes": ops * (10 + 2 * 24 + 24), "flops": 0}
    K, ops = case.get("objectives", 1), case["ops"]
    trees = case.get("results", K)
    b = ops * (6 + 4 * K + 2 * (8 + 2 * (4 + 4 * K)) + 24 * trees)
    if kind == "mosp" and case["costs"]:
        b += case["n"] * (4 + 8 * K)  # the costs of every path
    return {"bytes": b, "flops": 0}


def tolerance(case):
    """Whole numbers, decided by the inputs: the canonical tree has the lowest-id parent on every tie."""
    return "exact"


def exact(case, seed):
    """No output is a floating-point number."""
    return None
