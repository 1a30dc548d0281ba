"""Performance cases of the batched shortest-path engine.

Each case is one call pattern of a program that routes on a resident graph,
through the public binding (``bf-new_amd/bfnew_amd.py``) and, for the
allocation-free entry, the C ABI behind it.  ``prepare`` makes what such a
program has in hand before the call (device, resident graph, workspace or
server, the new queries), ``run`` is one whole call from the queries to host
arrays with the results.

The graphs are the framework's synthetic tile grids (nodes with four edges
inside their tile and six to tiles 1, 2 and 6 away); a program keeps one
resident graph for many batches, so graphs are shared by the states of a case
and the seed makes the queries.
"""
import collections
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "bf-new_amd"))

import bfnew_amd as bfn  # noqa: E402

ENGINES = {"jacobi": bfn.JACOBI_PULL, "dense": bfn.DENSE_CHAOTIC_PUSH,
           "frontier": bfn.FRONTIER_PUSH, "mixed": bfn.FRONTIER_PUSH}
DEGREE = 10  # edges per node of the synthetic grids
KEPT_GRAPHS = 2


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _case(name, kind, tiles, queries, side, engine, control="persistent", **options):
    """Options, where a case does not say otherwise: point Jacobi sweeps and
    boundary pushes through LDS proposals (the engines' defaults), no graph
    replay, no push window, one terminal pair per query."""
    case = dict(kind=kind, tiles_x=tiles[0], tiles_y=tiles[1], nodes=tiles[2], graph_seed=2,
                queries=queries, side_min=side[0], side_max=side[1], unbounded=0.0, engine=engine,
                control=control, sweeps=1, boundary=0, replay_rounds=0, window=0.0, min_waves=0,
                per_claim=1, terminals=1)
    case.update(options)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest call: one net on a small device graph, engine defaults
        # (point Jacobi, one cooperative launch).  Launch and host latency.
        _case("one_net_16x16x64_default", "route", (16, 16, 64), 1, (4, 8), "jacobi"),
        # One net per call, the interactive / plain mode of the benchmark:
        # frontier push with closed tiles on the 64x64x256 graph.
        _case("one_net_64x64x256_frontier", "route", (64, 64, 256), 1, (4, 32), "frontier",
              sweeps=0, boundary=1),
        # A 32-lane batch as the reference's callers send it: point Jacobi
        # with host-polled chunks of eight rounds (the reference round counts).
        _case("lanes32_32x32x128_point_jacobi", "route", (32, 32, 128), 32, (4, 16), "jacobi",
              "chunked"),
        # The benchmark's second workload, a new batch of 64 nets per call,
        # with the autotuned entry of that size (frontier push, graph replay).
        _case("batch_64x64x256_q64_frontier", "route", (64, 64, 256), 64, (4, 32), "frontier",
              "chunked", sweeps=0, boundary=1, replay_rounds=17, min_waves=7, per_claim=2),
        # The same batch under block Jacobi in one persistent launch: the
        # deterministic engine with closed tiles.
        _case("batch_64x64x256_q64_block_jacobi", "route", (64, 64, 256), 64, (4, 32), "jacobi",
              sweeps=0),
        # Nets with several drivers and sinks on a ragged grid with an odd
        # tile size, dense push through LDS proposals.
        _case("fanout_45x37x301_q41_dense", "route", (45, 37, 301), 41, (3, 21), "dense", "chunked",
              sweeps=0, terminals=3),
        # Full label and predecessor images of a few nets (timing analysis,
        # run_with_distances callers).
        _case("images_64x64x256_q4", "images", (64, 64, 256), 4, (24, 24), "frontier", sweeps=0,
              boundary=1),
        # Small batch without any device allocation (under capture, in tight
        # serving loops).
        _case("static_32x32x128_q24", "static", (32, 32, 128), 24, (4, 16), "frontier", sweeps=0,
              boundary=1),
        # A burst of requests with the serving box mix into the continuous-
        # batching server, every response with its path.
        _case("serve_64x64x256_r384", "serve", (64, 64, 256), 384, (4, 64), "frontier", sweeps=0),
        # The headline workload: 256 nets on the 128x128x512 graph, the
        # resident batch run again (costs unchanged), paths to host.
        _case("batch_128x128x512_q256_again", "again", (128, 128, 512), 256, (4, 64), "frontier",
              "chunked", graph_seed=3, unbounded=0.01, sweeps=0, boundary=1, replay_rounds=40,
              window=5.0, min_waves=8, per_claim=2),
        # The same size as a new batch per call: description, upload,
        # preparation, relaxation and paths.
        _case("batch_128x128x512_q256_new", "route", (128, 128, 512), 256, (4, 64), "frontier",
              "chunked", graph_seed=3, unbounded=0.01, sweeps=0, boundary=1, replay_rounds=40,
              window=5.0, min_waves=8, per_claim=2),
        # Negotiated congestion at that size: route, re-cost every edge from
        # the occupancy of the paths, route again.
        _case("negotiate_128x128x512_q256", "negotiate", (128, 128, 512), 256, (4, 64), "frontier",
              "chunked", graph_seed=5, sweeps=0, boundary=1, replay_rounds=40, window=5.0,
              min_waves=8, per_claim=2),
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], its logarithm uniform."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["route"] * 5 + ["again"] * 2 + ["images", "static", "serve", "negotiate"])
    engine = rng.choice(["jacobi", "dense", "frontier", "frontier"])
    if kind == "serve":
        engine = rng.choice(["dense", "frontier"])
    while True:
        tiles = (_spread(rng, 8, 128), _spread(rng, 8, 128), _spread(rng, 33, 512))
        grid = min(tiles[0], tiles[1])
        lo = rng.randint(2, 8)
        hi = min(grid, max(lo, _spread(rng, 6, 64)))
        lo = min(lo, hi)
        queries = _spread(rng, 1, 256)
        if kind == "images":
            queries, lo = min(queries, 6), hi
        if kind == "negotiate":
            queries = max(queries, 16)
        if kind == "serve":
            queries, lo, hi = max(queries, 32), 4, 64
        slots = queries * (hi * hi if kind == "static" else _mean_tiles(tiles, lo, hi, kind, 0.0))
        nodes = tiles[0] * tiles[1] * tiles[2]
        limit = 2.4e7 if engine == "frontier" else 1.0e7
        if nodes > 3_000_000 or slots * tiles[2] > limit:
            continue
        if kind == "static" and slots * (8 * tiles[2] + 600) > 48 << 20:
            continue
        break
    case = _case(None, kind, tiles, queries, (lo, hi), engine,
                 rng.choice(["persistent", "chunked", "per_round"]),
                 graph_seed=rng.randint(1, 999), terminals=rng.choice([1, 1, 2, 5]))
    if kind in ("serve", "negotiate"):
        case.update(terminals=1)
    if kind == "route" and engine == "frontier" and rng.random() < 0.2:
        case.update(engine="mixed")  # an engine per query
    if engine != "jacobi" or rng.random() < 0.5 or kind != "route":
        case.update(sweeps=0)
    if engine != "jacobi" and (rng.random() < 0.7 or kind == "static"):
        case.update(boundary=1)
    if engine != "jacobi" and rng.random() < 0.4:
        case.update(window=float(rng.choice([3, 5, 9])))
    if kind in ("route", "again", "negotiate") and rng.random() < 0.4:
        case.update(control="chunked", replay_rounds=rng.choice([8, 16, 40]))
    if engine == "frontier":
        case.update(min_waves=rng.choice([0, 7, 8]), per_claim=rng.choice([1, 2]))
    return case


# ---------------------------------------------------------------------------
# State
# ---------------------------------------------------------------------------
_device = None
_graphs = collections.OrderedDict()


class _Graph:
    """A resident graph and the host graph it came from."""

    def __init__(self, case):
        global _device
        if _device is None:
            _device = bfn.Device(0)
        self.host = bfn.HostGraph.synthetic(case["tiles_x"], case["tiles_y"], case["nodes"],
                                            case["graph_seed"])
        self.device = bfn.DeviceGraph(_device, self.host.layout())
        self.costs = self.host.view()["node_costs"] if case["kind"] == "negotiate" else None

    def __del__(self):
        if getattr(self, "device", None) is not None:
            self.device.close()


def _graph(case):
    # A negotiating program owns its graph: its costs change.
    key = (case["tiles_x"], case["tiles_y"], case["nodes"], case["graph_seed"],
           case["kind"] == "negotiate")
    if key not in _graphs:
        while len(_graphs) >= KEPT_GRAPHS:
            _graphs.popitem(last=False)
        _graphs[key] = _Graph(case)
    _graphs.move_to_end(key)
    return _graphs[key]


class _State:
    def __init__(self, case):
        self.case = case
        self.graph = _graph(case)
        self.workspace = self.server = None

    def __del__(self):
        for owned in (self.workspace, self.server):
            if owned is not None:
                owned.close()


def _queries(case, graph, seed):
    """Sources, targets and selected tiles of each query: the generator's
    boxes with one driver and sink, and for fanout nets more nodes of the box."""
    qs = graph.host.synthetic_queries(case["queries"], seed=seed, side_min=case["side_min"],
                                      side_max=case["side_max"],
                                      unbounded_fraction=case["unbounded"],
                                      mix=1 if case["kind"] == "serve" else 0)
    rng = random.Random(seed)
    sources, targets, tiles = [], [], []
    for q in qs:
        t = graph.host.query_tiles(q)
        inside = t[t < case["tiles_x"] * case["tiles_y"]]  # the spill tile has no nodes

        def more(first):
            nodes = {int(first)}
            while len(nodes) < case["terminals"]:
                nodes.add(int(inside[rng.randrange(len(inside))]) * case["nodes"]
                          + rng.randrange(case["nodes"]))
            return sorted(nodes)

        sources.append(more(q.source))
        targets.append(more(q.target))
        tiles.append(t)
    return sources, targets, tiles


def _options(case):
    control = {"persistent": bfn.PERSISTENT, "chunked": bfn.CHUNKED,
               "per_round": bfn.PER_ROUND}[case["control"]]
    options = bfn.run_options(engine=ENGINES[case["engine"]], control_mode=control)
    tuning = bfn.tuning(tile_sweeps=case["sweeps"], boundary_mode=case["boundary"],
                        use_graph=1 if case["replay_rounds"] else 0,
                        graph_rounds=case["replay_rounds"], push_window=case["window"],
                        min_waves=case["min_waves"], items_per_claim=case["per_claim"])
    return options, tuning


def prepare(case, seed):
    s = _State(case)
    s.options, s.tuning = _options(case)
    s.sources, s.targets, s.tiles = _queries(case, s.graph, seed)
    s.batch = bfn.Batch(s.sources, s.targets, s.tiles)
    if case["engine"] == "mixed":
        s.batch.engines = [q % 3 for q in range(case["queries"])]
    if case["kind"] == "serve":
        s.server = bfn.Server(_device, s.graph.device, budget_bytes=2 << 30,
                              max_active_queries=1024, rounds_per_chunk=2,
                              engine=ENGINES[case["engine"]], tile_sweeps=case["sweeps"])
    elif case["kind"] != "static":
        s.workspace = bfn.Workspace(_device)
        if case["kind"] == "again":
            s.workspace.submit(s.graph.device, s.batch, s.options, s.tuning)
            s.workspace.path_arrays()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
PATH_ROOM = 160  # vertices per target that a program's path arrays hold


def _held(values, targets):
    """`values` in an array of the size that the program keeps for paths."""
    out = np.zeros(targets * PATH_ROOM, values.dtype)
    out[:len(values)] = values
    return out


def _routed(s, out):
    """What a router takes from a finished batch: convergence and every path."""
    status, per_query, _ = s.workspace.status()
    a = s.workspace.path_arrays()
    summaries, total = a["summaries"], int(a["offsets"][-1])
    out.update(converged=int(status.converged),
               distance=np.array(summaries["distance"]),
               source=np.array(summaries["selected_source"]),
               length=np.array(summaries["path_length"]),
               reconstruction=np.array(summaries["reconstruction"]), offsets=a["offsets"],
               vertices=_held(a["vertices"][:total], len(summaries)),
               labels=_held(a["labels"][:total], len(summaries)),
               edge_ids=_held(a["edge_ids"][:total], len(summaries)))
    if s.case["engine"] == "jacobi":  # its round counts are part of the result
        out["rounds"] = np.array([p.rounds_completed for p in per_query], np.int64)
    return out


def _run_route(s):
    s.workspace.submit(s.graph.device, s.batch, s.options, s.tuning)
    return _routed(s, {})


def _run_again(s):
    s.workspace.rerun()
    return _routed(s, {})


def _run_images(s):
    s.workspace.submit(s.graph.device, s.batch, s.options, s.tuning)
    n = range(len(s.sources))
    return {"distances": [s.workspace.distances(q) for q in n],
            "predecessors": [s.workspace.predecessors(q) for q in n],
            "region": [s.workspace.region_distances(q) for q in n]}


def _run_static(s):
    d = s.batch.desc()
    per_query = (bfn.QueryStatus * d.query_count)()
    distances = np.empty(int(s.batch.target_offsets[-1]), np.float32)
    lib = bfn.hip_lib()
    rc = lib.bfn_batch_run_static(s.graph.device.h, ctypes.byref(d), ctypes.byref(s.options),
                                  ctypes.byref(_static_tuning(s.tuning)), per_query,
                                  distances.ctypes.data_as(ctypes.c_void_p))
    if rc:
        raise RuntimeError(lib.bfn_last_error().decode())
    return {"distance": distances,
            "converged": np.array([p.converged for p in per_query], np.int64),
            "reached": np.array([p.reached_all_targets for p in per_query], np.int64)}


def _static_tuning(tuning):
    t = type(tuning).from_buffer_copy(tuning)
    t.use_graph = t.graph_rounds = 0  # graph replay needs an allocation
    return t


def _run_serve(s):
    for i, (source, target, tiles) in enumerate(zip(s.sources, s.targets, s.tiles)):
        s.server.submit(i, source[0], target[0], tiles)
    got = {}
    while len(got) < len(s.sources):
        for r in s.server.poll_paths(capacity=1024, timeout_ms=100, vertex_capacity=1 << 20):
            got[r["request_id"]] = r
    order = range(len(s.sources))
    return {"distance": np.array([got[i]["distance"] for i in order], np.float32),
            "length": np.array([got[i]["path_length"] for i in order], np.int64),
            "vertices": _held(np.concatenate([got[i]["vertices"] for i in order]), len(order)),
            "edge_ids": _held(np.concatenate([got[i]["edge_ids"] for i in order]), len(order))}


def _run_negotiate(s):
    graph = s.graph.device
    graph.update_node_costs(s.graph.costs)
    first, second = {}, {}
    s.workspace.submit(graph, s.batch, s.options, s.tuning)
    _routed(s, first)
    graph.update_node_costs_from_workspace(s.workspace)
    s.workspace.submit(graph, s.batch, s.options, s.tuning)
    _routed(s, second)
    return {"first": first, "second": second, "occupancy": s.workspace.occupancy()}


def run(state):
    return {"route": _run_route, "again": _run_again, "images": _run_images,
            "static": _run_static, "serve": _run_serve,
            "negotiate": _run_negotiate}[state.case["kind"]](state)


# ---------------------------------------------------------------------------
# Work, tolerance and the outputs in 64 bits
# ---------------------------------------------------------------------------
def _mean_tiles(tiles, lo, hi, kind, unbounded):
    """Mean selected tiles of a query whose box side is log-uniform in [lo, hi]."""
    grid = min(tiles[0], tiles[1])

    def square(a, b):
        a, b = min(a, grid), min(b, grid)
        return float(a * a) if a == b else (b * b - a * a) / (2 * math.log(b / a))

    everything = tiles[0] * tiles[1]
    if kind == "serve":
        return 0.7 * square(4, 8) + 0.25 * square(16, 32) + 0.05 * (
            square(64, 64) + everything) / 2
    return (1 - unbounded) * square(lo, hi) + unbounded * everything


def work(case):
    """Bytes: destination and weight of every edge of the selected tiles read
    once for the whole batch, each query's labels written once, the result
    images written once.  Operations: an add and a compare per edge and query."""
    tiles = (case["tiles_x"], case["tiles_y"], case["nodes"])
    per_query = _mean_tiles(tiles, case["side_min"], case["side_max"], case["kind"],
                            case["unbounded"])
    grid = tiles[0] * tiles[1]
    slots = case["queries"] * per_query
    touched = grid * (1 - math.exp(-slots / grid))
    nodes = case["nodes"]
    rounds = 2 if case["kind"] == "negotiate" else 1
    moved = rounds * (8 * DEGREE * nodes * touched + 4 * nodes * slots)
    if case["kind"] == "negotiate":
        # costs and occupancy read, every weight of both orientations written
        moved += 2 * (8 + 8 * DEGREE) * grid * nodes
    if case["kind"] == "images":
        moved += 8 * case["queries"] * grid * nodes + 4 * nodes * slots
    return {"bytes": moved, "flops": rounds * 2.0 * DEGREE * nodes * slots}


def tolerance(case):
    """Every schedule of the monotone fp32 relaxation reaches the same bits,
    and paths are chosen by the smallest edge id: outputs are the same bits."""
    return "exact"


def _labels64(layout, sources, tiles):
    """Shortest distances of one query in float64 (Bellman-Ford on tensors);
    +inf outside its tiles and where unreached."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    offsets = layout["tile_vertex_offsets"].astype(np.int64)
    rows = layout["csr_row_offsets"].astype(np.int64)
    spans = [(rows[offsets[t]], rows[offsets[t + 1]]) for t in tiles.tolist()]
    at = np.concatenate([np.arange(a, b) for a, b in spans])
    src = np.searchsorted(rows, at, side="right") - 1
    dst = layout["csr_destinations"][at].astype(np.int64)
    inside = np.zeros(layout["tile_count"], bool)
    inside[tiles] = True
    keep = inside[layout["owner_tiles"][dst]]
    src, dst = (torch.from_numpy(x[keep]).to(device) for x in (src, dst))
    w = torch.from_numpy(layout["csr_weights"][at[keep]].astype(np.float64)).to(device)
    d = torch.full((layout["vertex_count"],), math.inf, dtype=torch.float64, device=device)
    d[torch.tensor(sources, device=device)] = 0.0
    while True:
        n = d.scatter_reduce(0, dst, d[src] + w, "amin")
        if torch.equal(n, d):
            return d.cpu().numpy()
        d = n


def exact(case, seed):
    tiles = (case["tiles_x"], case["tiles_y"], case["nodes"])
    slots = case["queries"] * _mean_tiles(tiles, case["side_min"], case["side_max"], case["kind"],
                                          case["unbounded"])
    if slots * case["nodes"] > 8e6 or case["kind"] == "negotiate":
        return None  # too long on tensors; re-costed weights depend on the paths
    graph = _graph(case)
    sources, targets, selected = _queries(case, graph, seed)
    layout = graph.host.layout_arrays()
    labels = [_labels64(layout, s, t) for s, t in zip(sources, selected)]
    if case["kind"] == "images":
        offsets = layout["tile_vertex_offsets"].astype(np.int64)
        return {"distances": labels, "predecessors": None,
                "region": [np.concatenate([d[offsets[t]:offsets[t + 1]] for t in ts.tolist()])
                           for d, ts in zip(labels, selected)]}
    distance = np.concatenate([d[t] for d, t in zip(labels, targets)])
    return {"distance": distance}
