"""The measured workloads: what users of this package have it do, through its
public entry points, from host inputs to results in the caller's memory.

A case is a dict of plain values; ``kind`` names the path:

* ``leaf``: one synchronous leaf-cost call (task rows in, int64 cells out),
  the form a cost backend is called in by the leaf search;
* ``cursor``: one block of the deletion-set cursor, rows made on the device,
  improving-template masks out;
* ``batch``: a resident batch of (instance, k) segments, launched and read;
* ``batch_masks``: the same batch object given new rows for many instances,
  launched and read as improving masks;
* ``jv_call``: one synchronous JV proposal over a snapshot;
* ``jv_session``: a whole JV elimination of one graph, from the snapshot to
  the proof;
* ``jv_fleet``: the same for many independent graphs at once;
* ``ht_hamilton``: the Hamilton replies of many centers of one target;
* ``server``: a burst of mixed requests through the continuous-batching server.

Sizes are those of the package's workloads (``workloads.py``), of its tests
and benchmark, and of the leaf search's block size (4,096 rows).
"""
from __future__ import annotations

import itertools
import math

import numpy as np

from cudaedgeelimination_amd import backend, resident, workloads
from cudaedgeelimination_amd._lib import KOPT_TASK_DTYPE
from cudaedgeelimination_amd.graph import CEIL_2D, EUC_2D

TEMPLATES = {3: 4, 4: 25, 5: 208}
PAIRS = {3: 9, 4: 20, 5: 35}  # distinct port pairs the templates of one k use
INT64_MAX = np.iinfo(np.int64).max
BOX = 1_000_000            # the workloads' coordinate box
WIDE_BOX = 1 << 30         # coordinates beyond the 25-bit extent: 64-bit distances


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest leaf call: one 5-opt deletion set (208 cells), the end
        # of a search and the unit the reference's per-call latency is quoted on
        {"name": "leaf_k5_1row", "kind": "leaf", "k": 5, "rows": 1, "n": 4096, "type": EUC_2D, "box": BOX},
        # an ordinary, ragged call: a block that ran short, CEIL_2D
        {"name": "leaf_k4_1237rows", "kind": "leaf", "k": 4, "rows": 1237, "n": 5000, "type": CEIL_2D, "box": BOX},
        # the leaf search's full block
        {"name": "leaf_k5_4096rows", "kind": "leaf", "k": 5, "rows": 4096, "n": 15000, "type": EUC_2D, "box": BOX},
        # an instance with wide coordinates (geographic or scaled data)
        {"name": "leaf_wide_k5_1501rows", "kind": "leaf", "k": 5, "rows": 1501, "n": 15000, "type": EUC_2D,
         "box": WIDE_BOX},
        # the cursor's full block read as masks, the cheapest consumer form
        {"name": "cursor_k5_4096sets", "kind": "cursor", "k": 5, "rows": 4096, "first": 1000, "n": 15000,
         "tour": 400, "selectable": 120, "type": EUC_2D},
        # the 65,536-row leaf workload of the benchmark, resident rows, cells read back
        {"name": "batch_65536rows", "kind": "batch", "rows": 65536, "n": 15000},
        # many small instances in one launch: new rows uploaded, masks read back
        {"name": "batch_masks_64x4096", "kind": "batch_masks", "instances": 64, "rows": 4096, "n_hi": 4000},
        # one JV proposal over a 10-NN graph (the propose step as a backend call)
        {"name": "jv_call_n15000", "kind": "jv_call", "n": 15000, "neighbors": 10, "type": EUC_2D},
        # a whole JV run of the lattice workload: many ties, several epochs
        {"name": "jv_session_lattice60", "kind": "jv_session", "side": 60},
        # whole JV runs of many instances in lockstep
        {"name": "jv_fleet_64", "kind": "jv_fleet", "instances": 64, "n_hi": 4000},
        # every node of the served graph as a center of one target edge
        {"name": "ht_hamilton_n30000", "kind": "ht_hamilton", "n": 30000, "type": EUC_2D},
        # a burst of served requests, 20% of them JV rechecks
        {"name": "server_burst_60", "kind": "server", "requests": 60, "sizes": "1000,5000,15000,30000"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["leaf", "leaf", "leaf", "cursor", "batch", "batch_masks", "jv_call", "jv_session",
                       "jv_fleet", "ht_hamilton", "server"])
    dtype = rng.choice([EUC_2D, CEIL_2D])
    if kind == "leaf":
        k = rng.choice([3, 4, 5])
        return {"kind": kind, "k": k, "rows": _log_int(rng, 1, {3: 32768, 4: 16384, 5: 4096}[k]),
                "n": _log_int(rng, 200, 30000), "type": dtype, "box": rng.choice([BOX, BOX, WIDE_BOX])}
    if kind == "cursor":
        selectable = rng.randint(60, 240)
        return {"kind": kind, "k": rng.choice([4, 5]), "rows": _log_int(rng, 16, 4096),
                "first": rng.randint(0, 20000), "n": _log_int(rng, 1000, 30000), "tour": rng.randint(300, 900),
                "selectable": selectable, "type": dtype}
    if kind == "batch":
        return {"kind": kind, "rows": _log_int(rng, 512, 65536), "n": _log_int(rng, 1000, 15000)}
    if kind == "batch_masks":
        return {"kind": kind, "instances": rng.randint(2, 64), "rows": rng.randint(256, 4096),
                "n_hi": rng.randint(1000, 4000)}
    if kind == "jv_call":
        return {"kind": kind, "n": _log_int(rng, 300, 15000), "neighbors": rng.randint(6, 12), "type": dtype}
    if kind == "jv_session":
        return {"kind": kind, "side": rng.randint(17, 60)}
    if kind == "jv_fleet":
        return {"kind": kind, "instances": rng.randint(2, 64), "n_hi": rng.randint(1000, 4000)}
    if kind == "ht_hamilton":
        return {"kind": kind, "n": _log_int(rng, 300, 30000), "type": dtype}
    return {"kind": kind, "requests": rng.randint(8, 60),
            "sizes": ",".join(str(_log_int(rng, 1000, 30000)) for _ in range(rng.randint(1, 4)))}


# ------------------------------------------------------------------ inputs
# A case fixes every size (nodes, edge slots, rows, request sizes); the seed
# fixes the contents.
def _snapshot(seed: int, x, y, dtype: int, neighbors: int):
    """The k-NN union graph with a random few of its edges already gone, down
    to 0.53 n k of the 0.54 to 0.58 n k edges."""
    graph = workloads.knn_graph(x, y, dtype, neighbors)
    keep = _edges(len(x), neighbors)
    if graph.edge_count <= keep:
        return graph
    pick = np.sort(np.random.default_rng(seed ^ 0xED6E).permutation(graph.edge_count)[:keep])
    return type(graph).from_edges(graph.x, graph.y, dtype, graph.edge_u[pick], graph.edge_v[pick],
                                  graph.edge_weight[pick])


def _edges(n: int, neighbors: int) -> int:
    return n * neighbors * 53 // 100


def _graph(seed: int, n: int, dtype: int, neighbors: int, box: int = BOX):
    rng = np.random.default_rng(seed)
    return _snapshot(seed, rng.integers(0, box, n), rng.integers(0, box, n), dtype, neighbors)


def _lattice(seed: int, side: int):
    """A jittered lattice with 17% of its sites dropped (the multi-epoch
    workload's shape), 10-NN."""
    rng = np.random.default_rng(seed)
    site = np.sort(rng.permutation(side * side)[:_lattice_nodes(side)])
    jitter = rng.integers(-3, 4, (2, len(site)))
    return _snapshot(seed, 25 * (site % side) + jitter[0], 25 * (site // side) + jitter[1], EUC_2D, 10)


def _lattice_nodes(side: int) -> int:
    return side * side * 83 // 100


def _instance_nodes(case):
    """Node counts of the instances, spread evenly in log n over [200, n_hi]."""
    steps = max(case["instances"] - 1, 1)
    return [int(round(200 * (case["n_hi"] / 200) ** (i / steps))) for i in range(case["instances"])]


def _instances(case, seed: int):
    """Many small instances as in the many-instance workload: uniform or
    8-cluster coordinates in pairs, CEIL_2D at odd indices, 10-NN."""
    graphs = []
    for i, n in enumerate(_instance_nodes(case)):
        rng = np.random.default_rng([seed, i])
        if (i // 2) % 2 == 0:
            x, y = rng.integers(0, BOX, (2, n))
        else:
            centre = rng.integers(0, BOX, (2, 8))[:, rng.integers(0, 8, n)]
            x, y = np.clip(np.rint(centre + rng.normal(0, 20_000, (2, n))), 0, BOX).astype(np.int64)
        graphs.append(_snapshot(seed + i, x, y, CEIL_2D if i % 2 else EUC_2D, 10))
    return graphs


def _quota(rows: int):
    return 2048 * rows // 4096, 1229 * rows // 4096, rows - 2048 * rows // 4096 - 1229 * rows // 4096


def _requests(case, seed: int):
    """Graphs and a stream of served requests in the serving workload's
    distribution: leaf-cost queries lognormal in cells (median 2,896), k = 3 /
    4 / 5 at 50 / 30 / 20%, and 20% JV rechecks of lognormally many edge
    slots (median 256).  The case fixes the sizes, the seed the contents."""
    sizes = [int(s) for s in case["sizes"].split(",")]
    graphs = [_graph(seed + i, n, EUC_2D, 10) for i, n in enumerate(sizes)]
    fixed = np.random.default_rng([case["requests"], *sizes])
    rng = np.random.default_rng(seed)
    requests = []
    for _ in range(case["requests"]):
        g, k = int(fixed.integers(len(graphs))), int(fixed.choice([3, 4, 5], p=[0.5, 0.3, 0.2]))
        cells = float(np.clip(math.exp(fixed.normal(math.log(2896.0), 1.04)), 128, 65536))
        slots = int(np.clip(math.exp(fixed.normal(math.log(256.0), 1.0)), 16, 4096))
        if fixed.random() < 0.2:
            slots = min(slots, graphs[g].edge_count)
            requests.append((g, 0, rng.choice(graphs[g].edge_count, slots, replace=False).astype(np.int32)))
        else:
            rows = min(2048, math.ceil(cells / TEMPLATES[k]))
            requests.append((g, k, workloads.kopt_tasks(int(rng.integers(1 << 40)), graphs[g],
                                                        np.full(rows, k, np.uint8))))
    return graphs, requests


def _relabelled(seed: int, n: int, dtype: int):
    """One geometry per n under a seeded numbering of its nodes and a seeded
    shift, and one of its edges as the target: other ids and coordinates, the
    same number of replies."""
    base = _graph(n, n, dtype, 10)
    e = int(np.random.default_rng(n).integers(base.edge_count))
    rng = np.random.default_rng(seed)
    name = rng.permutation(n).astype(np.int32)
    x, y = np.empty(n, np.int64), np.empty(n, np.int64)
    x[name], y[name] = base.x + rng.integers(BOX), base.y + rng.integers(BOX)
    ends = np.sort(np.stack([name[base.edge_u], name[base.edge_v]]), axis=0)
    order = np.lexsort((ends[1], ends[0]))
    graph = type(base).from_edges(x, y, dtype, ends[0][order], ends[1][order], base.edge_weight[order])
    return graph, (int(ends[0, e]), int(ends[1, e]))


def _inputs(case, seed: int):
    """The host-side inputs of a case, from the seed alone."""
    kind = case["kind"]
    if kind == "leaf":
        graph = _graph(seed, case["n"], case["type"], 8, case["box"])
        tasks = workloads.kopt_tasks(seed ^ 0xA5A5, graph, np.full(case["rows"], case["k"], np.uint8))
        return graph, tasks
    if kind == "cursor":
        graph = _graph(seed, case["n"], case["type"], 8)
        return graph, workloads.tour_context(seed ^ 0x70, graph, case["tour"], case["selectable"])
    if kind == "batch":
        return workloads.config3(seed, case["n"], case["rows"])
    if kind == "batch_masks":
        return [(graph, {k: workloads.kopt_tasks(seed + 8 * i + k, graph, np.full(rows, k, np.uint8))
                         for k, rows in zip((3, 4, 5), _quota(case["rows"]))})
                for i, graph in enumerate(_instances(case, seed))]
    if kind == "jv_call":
        return _graph(seed, case["n"], case["type"], case["neighbors"])
    if kind == "jv_session":
        return _lattice(seed, case["side"])
    if kind == "jv_fleet":
        return _instances(case, seed)
    if kind == "ht_hamilton":
        graph, target = _relabelled(seed, case["n"], case["type"])
        centers = np.setdiff1d(np.arange(graph.dimension, dtype=np.int32), np.array(target, np.int32))
        return graph, target, centers
    return _requests(case, seed)


def prepare(case, seed):
    """The inputs and the handle (context, batch, server) a program keeps."""
    state = {"case": case, "ctx": backend.Context(0), "in": _inputs(case, seed)}
    ctx = state["ctx"]
    if case["kind"] in ("leaf", "cursor"):
        state["table"] = backend.build_kopt_reconnect_table(case["k"])
    elif case["kind"] == "batch":
        batch = state["batch"] = resident.KoptBatch(ctx)
        instance = batch.add_instance(state["in"].graph)
        rows = [state["in"].bucket(k) for k in (3, 4, 5)]
        batch.set_work([(instance, k, len(r)) for k, r in zip((3, 4, 5), rows)], np.concatenate(rows))
    elif case["kind"] == "batch_masks":
        batch = state["batch"] = resident.KoptBatch(ctx)
        batch.set_output("masks")
        segments, tasks = [], []
        for graph, work in state["in"]:
            instance = batch.add_instance(graph)
            for k, rows in work.items():
                segments.append((instance, k, len(rows)))
                tasks.append(rows)
        state["segments"], state["tasks"] = segments, np.concatenate(tasks)
    elif case["kind"] == "server":
        server = state["server"] = resident.KoptServer(ctx)
        graphs, requests = state["in"]
        leaf = [server.add_graph(g) for g in graphs]
        jv = [server.add_jv_graph(g) for g in graphs]
        state["requests"] = [(leaf[g] if k else jv[g], k, data) for g, k, data in requests]
    elif case["kind"] in ("jv_session", "jv_fleet"):
        slots = sum(g.edge_count for g in (state["in"] if case["kind"] == "jv_fleet" else [state["in"]]))
        state["proof"] = np.zeros(16 * slots, np.uint8)
    return state


# --------------------------------------------------------------- one pass
def _records(proofs, out):
    """The proofs' deterministic parts (everything before their timing lines),
    one after the other, zero to the end of `out`."""
    text = "".join(p[:p.index("metrics ")] for p in proofs).encode()
    out[:len(text)] = np.frombuffer(text, np.uint8)
    out[len(text):] = 0
    return out


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "leaf":
        graph, tasks = state["in"]
        return backend.evaluate_kopt_template_costs_cuda(graph, state["table"], tasks, ctx)[0]
    if kind == "cursor":
        graph, tour = state["in"]
        block = backend.evaluate_kopt_cursor_cuda(graph, state["table"], tour, case["k"], case["first"],
                                                  case["rows"], "masks", ctx)
        return [block.tasks.view(np.int64), block.positions.view(np.int32), block.masks.view(np.int32)]
    if kind == "batch":
        batch = state["batch"]
        batch.run()
        return [batch.segment_costs(i) for i in range(len(batch.segments))]
    if kind == "batch_masks":
        batch = state["batch"]
        batch.set_work(state["segments"], state["tasks"])
        batch.run()
        return batch.download_masks().view(np.int32)
    if kind == "jv_call":
        return backend.find_jv_witnesses(state["in"], ctx)[0]
    if kind == "jv_session":
        session = resident.JvSession(ctx, state["in"])
        r = session.run()
        active = session.active()
        session.close()
        return [active, _records([r.proof], state["proof"]), np.array([r.epochs, r.edges_scanned, r.proposed, r.committed]),
                np.array([r.initial_hash, r.final_hash], np.uint64).view(np.int64)]
    if kind == "jv_fleet":
        fleet = resident.JvFleet(ctx, state["in"])
        fleet.run()
        count = len(state["in"])
        active = np.concatenate([fleet.active(i) for i in range(count)])
        proofs = [fleet.proof(i) for i in range(count)]
        fleet.close()
        return [active, _records(proofs, state["proof"])]
    if kind == "ht_hamilton":
        graph, target, centers = state["in"]
        offsets, replies, _ = backend.evaluate_ht_hamilton_replies_cuda(graph, target, centers, ctx)
        return [offsets.view(np.int64), replies]
    server = state["server"]
    ids = server.submit_many(state["requests"])
    return [result for result, _ in server.wait_many(ids)]


# -------------------------------------------------------------------- work
def _kopt_work(rows, n, masks=False):
    """Rows, coordinates and templates read once, cells (or mask words)
    written once; per row each distinct pair's distance, per cell k sums."""
    cells = {k: r * TEMPLATES[k] for k, r in rows.items()}
    wide = max(k for k in rows if rows[k] or len(rows) == 1)
    out = sum(rows.values()) * ((TEMPLATES[wide] + 31) // 32) * 4 if masks else 8 * sum(cells.values())
    return {"bytes": 48 * sum(rows.values()) + out + 16 * n + 15 * sum(TEMPLATES[k] for k in rows),
            "flops": sum(10 * PAIRS[k] * r + k * cells[k] for k, r in rows.items())}


def _jv_work(n, m, a, epochs):
    """The snapshot read once per epoch, a witness per slot written; about 40
    distances and weights scored or tested per edge."""
    return {"bytes": epochs * (24 * m + 20 * n + 4 + 8 * a), "flops": epochs * m * 400}


def work(case):
    kind = case["kind"]
    if kind == "leaf":
        return _kopt_work({case["k"]: case["rows"]}, case["n"])
    if kind == "cursor":
        w = _kopt_work({case["k"]: case["rows"]}, case["n"], masks=True)
        w["bytes"] += 4 * case["k"] * case["rows"] + 12 * case["tour"] + 8 * case["selectable"]
        return w
    if kind == "batch":
        return _kopt_work(dict(zip((3, 4, 5), workloads.kopt_quota(case["rows"]))), case["n"])
    if kind == "batch_masks":
        rows = {k: q * case["instances"] for k, q in zip((3, 4, 5), _quota(case["rows"]))}
        return _kopt_work(rows, sum(_instance_nodes(case)), masks=True)
    if kind == "jv_call":
        m = _edges(case["n"], case["neighbors"])
        return _jv_work(case["n"], m, 2 * m, 1)
    if kind == "jv_session":
        n = _lattice_nodes(case["side"])
        return _jv_work(n, _edges(n, 10), 2 * _edges(n, 10), 2)
    if kind == "jv_fleet":
        n = sum(_instance_nodes(case))
        return _jv_work(n, _edges(n, 10), 2 * _edges(n, 10), 3)
    if kind == "ht_hamilton":
        n = case["n"]
        pairs = n * 55  # about C(11, 2) neighbour pairs per center
        return {"bytes": 24 * n + 46 * n + 12 * n + 12 * pairs, "flops": pairs * 12 + n * 11 * 50}
    cells = 5000 * case["requests"]  # lognormal, median 2,896 cells
    return {"bytes": 8 * cells + 48 * cells // 60, "flops": 6 * cells}


def tolerance(case):
    """Every output is a whole number that is defined exactly."""
    return "exact"


# ------------------------------------------------------------------- exact
def _distances(x, y, a, b, dtype):
    dx, dy = x[a] - x[b], y[a] - y[b]
    s = dx * dx + dy * dy  # below 2^62 in every box
    r = np.floor(np.sqrt(s.astype(np.float64))).astype(np.int64)
    r -= r * r > s
    r += (r + 1) * (r + 1) <= s
    return r + (((s - r * r) > r) if dtype == EUC_2D else (r * r != s))


def _cells(graph, k, ports):
    """[rows, T] reconnection costs from the rules: the added edges' distances
    summed; INT64_MAX when an added edge is a loop, equals a deleted edge or
    another added edge."""
    mates = backend.build_kopt_reconnect_table(k).templates["mate"][:, :2 * k].astype(np.int64)
    ports = ports[:, :2 * k].astype(np.int64)
    n = graph.dimension
    deleted = np.minimum(ports[:, 0::2], ports[:, 1::2]) * n + np.maximum(ports[:, 0::2], ports[:, 1::2])
    pair = {}
    for p, q in itertools.combinations(range(2 * k), 2):
        a, b = ports[:, p], ports[:, q]
        key = np.minimum(a, b) * n + np.maximum(a, b)
        pair[p, q] = (_distances(graph.x, graph.y, a, b, graph.distance_type), key,
                      (a == b) | (key[:, None] == deleted).any(axis=1))
    out = np.empty((len(ports), len(mates)), np.int64)
    for t, mate in enumerate(mates):
        edges = [pair[p, int(mate[p])] for p in range(2 * k) if p < mate[p]]
        bad = np.logical_or.reduce([e[2] for e in edges])
        for e, f in itertools.combinations(edges, 2):
            bad = bad | (e[1] == f[1])
        out[:, t] = np.where(bad, INT64_MAX, sum(e[0] for e in edges))
    return out


def _masks(cells, deleted_cost, words):
    bits = cells < deleted_cost[:, None]
    out = np.zeros((len(cells), words), np.uint32)
    for t in range(cells.shape[1]):
        out[:, t // 32] |= bits[:, t].astype(np.uint32) << np.uint32(t % 32)
    return out.view(np.int32)


def exact(case, seed):
    """The k-opt cells and masks from the rules in 64-bit integers.  The JV,
    HT and served outputs are decisions over such distances (witnesses,
    committed slots, reply lists), whose restatement here would take minutes."""
    kind = case["kind"]
    if kind == "leaf":
        graph, tasks = _inputs(case, seed)
        return _cells(graph, case["k"], tasks["port_nodes"]).reshape(-1)
    if kind == "cursor":
        graph, tour = _inputs(case, seed)
        k, length = case["k"], len(tour.tour)
        sets = itertools.combinations(range(1, len(tour.selectable)), k - 1)
        picked = np.array(list(itertools.islice(sets, case["first"], case["first"] + case["rows"])), np.int64)
        picked = np.concatenate([np.zeros((len(picked), 1), np.int64), picked], axis=1)
        positions = np.sort(tour.selectable.astype(np.int64)[picked], axis=1)
        tasks = np.zeros(len(positions), KOPT_TASK_DTYPE)
        tasks["port_nodes"][:, 0:2 * k:2] = tour.tour[positions]
        tasks["port_nodes"][:, 1:2 * k:2] = tour.tour[(positions + 1) % length]
        tasks["deleted_cost"] = tour.edge_costs[positions].sum(axis=1)
        cells = _cells(graph, k, tasks["port_nodes"])
        return [tasks.view(np.int64), positions.astype(np.int32),
                _masks(cells, tasks["deleted_cost"], (TEMPLATES[k] + 31) // 32)]
    if kind == "batch":
        work_ = _inputs(case, seed)
        return [_cells(work_.graph, k, work_.bucket(k)["port_nodes"]).reshape(-1) for k in (3, 4, 5)]
    if kind == "batch_masks":
        out = []
        for graph, work_ in _inputs(case, seed):
            for k, rows in work_.items():
                out.append(_masks(_cells(graph, k, rows["port_nodes"]), rows["deleted_cost"], 7))
        return np.concatenate(out)
    return None
