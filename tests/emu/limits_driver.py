"""Memory that the engine library named by argv[1] -- the CPU emulation of the
kernels -- takes, against what it says it takes: the check argv[2], one JSON
line on stdout with its failures."""
import ctypes
import json
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
TESTS = os.path.dirname(HERE)
ROOT = os.path.dirname(TESTS)
sys.path.insert(0, os.path.join(ROOT, "bf-new_amd"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
sys.path.insert(0, TESTS)

import numpy as np  # noqa: E402

import bfnew_amd as bfn  # noqa: E402
import oracle  # noqa: E402

bfn.HIP_LIB_PATH = sys.argv[1]

from helpers import bits, expected_paths, oracle_query, path_failures, with_node_costs  # noqa: E402

DEVICE, PINNED = 0, 1
FAILURES = []


def used(kind=DEVICE):
    f = bfn.hip_lib().emu_memory_used
    f.restype = ctypes.c_uint64
    return f(kind)


def check(ok, what):
    if not ok:
        FAILURES.append(what)


def refused(f):
    try:
        f()
    except bfn.BfnError as e:
        return e.code
    return 0


def graph(dev, x=8, y=8, nodes=32):
    hg = bfn.HostGraph.synthetic(x, y, nodes, 4, host_graph=True)
    return hg, bfn.DeviceGraph(dev, hg.layout())


def estimate(dev):
    """A batch's estimate covers the device memory of its submit, and is the
    smallest budget that admits it."""
    hg, dg = graph(dev)
    for count, engine, window in ((1, bfn.FRONTIER_PUSH, 0.0), (1, bfn.JACOBI_PULL, 0.0),
                                  (9, bfn.FRONTIER_PUSH, 3.0)):
        qs = hg.synthetic_queries(count, seed=5, side_min=2, side_max=4)
        batch = bfn.Batch([[q.source] for q in qs], [[q.target] for q in qs],
                          [hg.query_tiles(q) for q in qs])
        o = bfn.run_options(engine=engine, control_mode=bfn.CHUNKED)
        t = bfn.tuning(tile_sweeps=0, push_window=window)
        before = used()
        ws = bfn.Workspace(dev)
        need = ws.estimate(dg, batch, o)
        ws.submit(dg, batch, o, t)
        check(used() - before <= need, f"batch of {count}: {used() - before} bytes in use, estimate {need}")
        ws.close()
        check(used() == before, "memory left after the workspace")
        for budget, code in ((need, 0), (need - 1, 3)):
            ws = bfn.Workspace(dev, budget)
            got = refused(lambda: ws.submit(dg, batch, o, t))
            check(got == code, f"batch of {count}, budget {budget} of {need}: {got}")
            ws.close()


def server(dev):
    """A server's device memory stays within its budget."""
    _, dg = graph(dev)
    for budget, queries in ((256 << 10, 3), (1 << 20, 64), (8 << 20, 7)):
        before = used()
        s = bfn.Server(dev, dg, budget_bytes=budget, max_active_queries=queries)
        check(used() - before <= budget, f"server: {used() - before} bytes in use of {budget}")
        s.close()
        check(used() == before, "memory left after the server")


def largest(kind, n_bytes):
    bfn.hip_lib().emu_largest_allocation(kind, ctypes.c_uint64(n_bytes))


def workgroups():
    f = bfn.hip_lib().emu_workgroups
    f.restype = ctypes.c_uint64
    return f()


def expect_weights(dev, dg, view, costs):
    """Labels of one region under both weight orientations against the oracle."""
    tiles = np.arange(9, dtype=np.uint32)
    view["weights"] = costs[view["destinations"]]
    want, _ = oracle_query(view, [5], tiles)
    for engine in (bfn.JACOBI_PULL, bfn.FRONTIER_PUSH):
        ws = bfn.Workspace(dev)
        ws.submit(dg, bfn.Batch([[5]], [[100]], [tiles]),
                  bfn.run_options(engine=engine, control_mode=bfn.CHUNKED), bfn.tuning(tile_sweeps=0))
        check(np.array_equal(bits(ws.distances(0)), bits(want)), f"labels under engine {engine}")
        ws.close()


def costs(dev):
    """Node-cost updates: what they keep (the costs and the occupancy; on a
    large graph a second buffer where there is memory for it, and the update
    as before where there is none), and the workgroups of a small graph's."""
    half = np.float32(0.5)
    for dims, extra in (((16, 16, 33), 0), ((32, 32, 257), 1)):
        hg, dg = graph(dev, *dims)
        view = hg.view()
        V = view["vertex_count"]
        base = np.random.default_rng(V).uniform(0.5, 9.0, V).astype(np.float32)
        occupancy = (np.arange(V) % 3).astype(np.int32)
        before, at = used(), workgroups()
        dg.update_node_costs(base)
        groups = workgroups() - at
        blocks = -(-view["edge_count"] // 256)
        check(extra or groups <= 4 * blocks, f"{groups} workgroups for {view['edge_count']} edges")
        dg.update_node_costs(base * half)
        dg.update_node_costs(base, occupancy)
        kept = used() - before
        check(kept <= 4 * V * (2 + extra), f"{kept} bytes kept for {V} vertices")
        expect_weights(dev, dg, view, base * (np.float32(1.0) + half * occupancy.astype(np.float32)))
        bad = base.copy()
        bad[V - 1] = np.nan
        check(refused(lambda: dg.update_node_costs(bad)) == 1, "NaN costs accepted")
        dg.close()
    # no memory for more than the costs
    hg, dg = graph(dev, 32, 32, 257)
    dg.update_node_costs(base)
    largest(DEVICE, 0)
    check(refused(lambda: dg.update_node_costs(base + half)) == 0, "update without a second buffer")
    check(refused(lambda: dg.update_node_costs(bad)) == 1, "NaN costs accepted")
    largest(DEVICE, 1 << 40)
    expect_weights(dev, dg, view, base + half)
    dg.close()


def images(dev):
    """Label and predecessor images of a run of tiles, of tiles apart and of
    the whole graph, with pinned memory for them and without."""
    hg, dg = graph(dev, 9, 8, 33)
    view = hg.view()
    T = 72
    regions = [np.arange(T, dtype=np.uint32), np.arange(20, 31, dtype=np.uint32),
               np.array([0, 1, 2, 9, 10, 18, 70, 71], np.uint32), np.array([33], np.uint32)]
    sources = [[int(r[len(r) // 2]) * 33 + 4] for r in regions]
    ws = bfn.Workspace(dev)
    ws.submit(dg, bfn.Batch(sources, [[s[0] + 1] for s in sources], regions),
              bfn.run_options(engine=bfn.FRONTIER_PUSH, control_mode=bfn.CHUNKED), bfn.tuning(tile_sweeps=0))
    first = []
    for pinned in (1 << 40, 0):
        for q in (3, 2, 1, 0):  # growing, so that none fits what an earlier one took
            largest(PINNED, pinned)
            want, _ = oracle_query(view, sources[q], regions[q])
            where = oracle.region_vertices(view["tile_vertex_offsets"], regions[q])
            check(np.array_equal(bits(ws.distances(q)), bits(want)), f"labels of {q}, pinned {pinned}")
            check(np.array_equal(bits(ws.region_distances(q)), bits(want[where])), f"region of {q}")
            first.append(ws.predecessors(q))
        ws.close()
        largest(PINNED, 1 << 40)
        ws = bfn.Workspace(dev)
        ws.submit(dg, bfn.Batch(sources, [[s[0] + 1] for s in sources], regions),
                  bfn.run_options(engine=bfn.FRONTIER_PUSH, control_mode=bfn.CHUNKED), bfn.tuning(tile_sweeps=0))
    for a, b in zip(first[:4], first[4:]):
        check(np.array_equal(a, b), "predecessors with and without pinned memory")
    ws.close()
    dg.close()


def paths(dev):
    """Compact paths, some of them over zero-cost plateaus, as two calls (the
    first without arenas) and as one, with memory to write the paths early and
    without."""
    hg, dg = graph(dev, 9, 8, 32)
    rng = np.random.default_rng(2)
    costs = hg.view()["node_costs"].copy()
    costs[rng.random(len(costs)) < 0.05] = 0.0
    dg.update_node_costs(costs)
    view = with_node_costs(hg.view(), costs)
    tiles = np.arange(18, dtype=np.uint32)
    targets = sorted(int(v) for v in rng.choice(18 * 32, 60, False))
    want = expected_paths(view, [5], targets, tiles)
    walks = [w[1:] for w in want[1]]
    batch = bfn.Batch([[5]], [targets], [tiles])
    total = sum(len(v) for v, _ in walks)
    for device, pinned in ((1 << 40, 1 << 40), (12000, 1 << 40), (1 << 40, 4000)):
        for arenas_at_once in (False, True):
            what = (device, pinned, arenas_at_once)
            ws = bfn.Workspace(dev)
            ws.submit(dg, batch, bfn.run_options(engine=bfn.FRONTIER_PUSH, control_mode=bfn.CHUNKED),
                      bfn.tuning(tile_sweeps=0))
            largest(DEVICE, device)
            largest(PINNED, pinned)
            summaries = (bfn.TargetSummary * 60)()
            offsets, n = np.zeros(61, np.uint64), ctypes.c_uint64()
            out = [np.zeros(total, t) for t in (np.uint32, np.float32, np.uint32)]
            f, p = bfn.hip_lib().bfn_batch_paths, lambda a: a.ctypes.data_as(ctypes.c_void_p)
            if not arenas_at_once:
                rc = f(ws.h, summaries, p(offsets), None, None, None, 0, ctypes.byref(n))
                check(rc == 0 and n.value == total, f"summaries {what}: {rc}, {n.value} of {total} vertices")
            rc = f(ws.h, summaries, p(offsets), *(p(a) for a in out), total, ctypes.byref(n))
            check(rc == 0 and n.value == total, f"arenas {what}: {rc}")
            arrays = dict(summaries=np.ctypeslib.as_array(summaries), offsets=offsets, vertices=out[0],
                          labels=out[1], edge_ids=out[2])
            check(rc or path_failures(arrays, [want]) == [], f"paths {what}")
            largest(DEVICE, 1 << 40)
            largest(PINNED, 1 << 40)
            occupancy = np.zeros(view["vertex_count"], np.int32)
            for verts, _ in walks:
                occupancy[verts] += 1
            if rc == 0:
                check(np.array_equal(ws.occupancy(), occupancy), f"occupancy {what}")
            ws.close()
    dg.close()


def long_paths(dev):
    """Paths of more vertices than the room first made for them, on positive
    costs (tests/test_gpu_path_walks.py on a shorter strip)."""
    hg, dg = graph(dev, 300, 1, 4)
    view = with_node_costs(hg.view(), hg.view()["node_costs"])
    tiles = np.arange(300, dtype=np.uint32)
    targets = [1150, 1171, 1199]
    want = [expected_paths(view, [1], targets, tiles)]
    ws = bfn.Workspace(dev)
    ws.submit(dg, bfn.Batch([[1]], [targets], [tiles]),
              bfn.run_options(engine=bfn.FRONTIER_PUSH, control_mode=bfn.CHUNKED), bfn.tuning(tile_sweeps=0))
    for _ in range(2):
        arrays = ws.path_arrays()
        check(arrays["offsets"][-1] > 64 * 3, f"{arrays['offsets'][-1]} vertices")
        check(path_failures(arrays, want) == [], "paths")
        ws.rerun()
    ws.close()
    dg.close()


def main():
    dev = bfn.Device(0)
    globals()[sys.argv[2]](dev)
    dev.close()
    print(json.dumps(dict(check=sys.argv[2], failures=FAILURES)), flush=True)


if __name__ == "__main__":
    main()
