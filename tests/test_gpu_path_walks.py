"""Compact paths where the walk from a target cannot just follow the smallest
tight EdgeId: zero-weight plateaus (the walk can meet its own path), more
targets than frames to walk in (one-tile regions), several targets that share
their paths, and paths longer than the room first made for them; path by path
against the oracle's reconstruction."""
import numpy as np
import pytest

import bfnew_amd as bfn
import oracle
from helpers import bits, expected_paths, oracle_query, path_failures, tile_mask, with_node_costs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zero_share,nodes,targets", [(0.0, 16, 16), (0.0, 33, 5), (0.5, 16, 9),
                                                      (0.7, 33, 33), (0.2, 8, 3)])
def test_path_walks(device, zero_share, nodes, targets):
    hg = bfn.HostGraph.synthetic(40, 4, nodes, 5, host_graph=True)
    dg = bfn.DeviceGraph(device, hg.layout())
    view = hg.view()
    rng = np.random.default_rng(nodes + targets)
    costs = view["node_costs"].copy()
    costs[rng.random(len(costs)) < zero_share] = 0.0
    dg.update_node_costs(costs)
    view["weights"] = costs[view["destinations"]]
    heads = np.repeat(np.arange(len(costs)), np.diff(view["column_offsets"].astype(np.int64)))
    in_weights = costs[heads]
    # a one-tile region with as many targets as nodes, a strip, the whole grid
    regions = [np.array([41], np.uint32), np.arange(0, 12, dtype=np.uint32)]
    if zero_share == 0.0:  # on large plateaus the depth-first rule itself takes millions of steps
        regions.append(np.arange(160, dtype=np.uint32))
    sources, wanted = [], []
    for tiles in regions:
        inside = np.concatenate([np.arange(t * nodes, (t + 1) * nodes) for t in tiles])
        sources.append([int(inside[-1])])
        wanted.append(sorted(int(v) for v in rng.choice(inside, min(targets, len(inside)), False)))
    for engine in (bfn.JACOBI_PULL, bfn.FRONTIER_PUSH):
        ws = bfn.Workspace(device)
        batch = bfn.Batch(sources, wanted, regions)
        ws.submit(dg, batch, bfn.run_options(engine=engine, control_mode=bfn.CHUNKED),
                  bfn.tuning(tile_sweeps=0, boundary_mode=1))
        for _ in range(2):  # again on the workspace's kept frames, marks and room
            paths = ws.paths()
            at = 0
            for q, tiles in enumerate(regions):
                sel = tile_mask(view["tile_count"], tiles)
                labels, _ = oracle_query(view, sources[q], tiles)
                for target in batch.targets[q]:
                    p = paths[at]
                    at += 1
                    what, verts, edges = oracle.reconstruct(
                        view["vertex_count"], view["column_offsets"], view["sources"], in_weights,
                        view["in_edge_ids"], view["owner_tiles"], sel, labels, sources[q], target)
                    label = (zero_share, engine, q, target)
                    assert p["target"] == target, label
                    assert p["reconstruction"] == {"complete": 0, "unreachable": 1,
                                                   "no_tight_path": 3}[what], label
                    assert list(p["vertices"]) == list(verts), label
                    assert list(p["edge_ids"]) == list(edges), label
                    assert np.array_equal(bits(p["labels"]), bits(labels[verts])), label
            ws.rerun()
        ws.close()
    dg.close()


def test_paths_longer_than_the_first_room(device):
    """Paths of more than 64 vertices per target on positive costs: pass 2 has
    no room at first, and the paths are copied out of the frames that pass 1
    left; then room that an earlier batch grew."""
    hg = bfn.HostGraph.synthetic(400, 1, 4, 5, host_graph=True)
    dg = bfn.DeviceGraph(device, hg.layout())
    view = with_node_costs(hg.view(), hg.view()["node_costs"])
    assert view["node_costs"].min() > 0.0
    tiles = np.arange(400, dtype=np.uint32)
    sources, targets = [[1], [0, 6]], [[1502, 1540, 1571, 1599], [1450, 1588]]
    want = [expected_paths(view, s, t, tiles) for s, t in zip(sources, targets)]
    for engine in (bfn.JACOBI_PULL, bfn.FRONTIER_PUSH):
        ws = bfn.Workspace(device)
        ws.submit(dg, bfn.Batch(sources, targets, [tiles] * 2),
                  bfn.run_options(engine=engine, control_mode=bfn.CHUNKED),
                  bfn.tuning(tile_sweeps=0, boundary_mode=1))
        for _ in range(2):
            arrays = ws.path_arrays()
            assert arrays["offsets"][-1] > 64 * 6
            assert path_failures(arrays, want) == [], engine
            ws.rerun()
        ws.close()
    dg.close()


@pytest.mark.parametrize("zero_share", [0.03, 0.08])
def test_plateaus_of_many_queries(device, zero_share):
    """Batches where some queries have to be walked again by pass 2 and others
    do not: the first call leaves the former to the second."""
    hg = bfn.HostGraph.synthetic(24, 24, 32, 5, host_graph=True)
    dg = bfn.DeviceGraph(device, hg.layout())
    costs = hg.view()["node_costs"].copy()
    costs[np.random.default_rng(3).random(len(costs)) < zero_share] = 0.0
    dg.update_node_costs(costs)
    view = with_node_costs(hg.view(), costs)
    qs = hg.synthetic_queries(20, seed=4, side_min=2, side_max=6)
    tiles = [hg.query_tiles(q) for q in qs]
    want = [expected_paths(view, [q.source], [q.target], t) for q, t in zip(qs, tiles)]
    plateau = [any(labels[v] == labels[u] for v, u in zip(verts, verts[1:]))
               for labels, ((_, verts, _),) in want]
    assert any(plateau) and not all(plateau)
    ws = bfn.Workspace(device)
    ws.submit(dg, bfn.Batch([[q.source] for q in qs], [[q.target] for q in qs], tiles),
              bfn.run_options(engine=bfn.FRONTIER_PUSH, control_mode=bfn.CHUNKED),
              bfn.tuning(tile_sweeps=0, boundary_mode=1))
    for _ in range(2):
        assert path_failures(ws.path_arrays(), want) == []
        ws.rerun()
    ws.close()
    dg.close()
