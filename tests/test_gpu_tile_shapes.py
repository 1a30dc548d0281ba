"""Every engine and control mode on tile sizes at the edges of what a visit
stages at a time (64-word rows, two of a pulled slab and four of a proposal slab
together, the registers that hold a tile's internal records), against the oracle bit for bit.  The 9 x 8 grid
clamps its long edges, so tiles have between 5 and 13 neighbours, and the
boxes leave some of them out; the batches have fewer slots than work-list
classes and more, and claims of several items."""
import numpy as np
import pytest

import bfnew_amd as bfn
from helpers import bits, oracle_query

pytestmark = pytest.mark.gpu

CONFIGS = [
    dict(engine=bfn.JACOBI_PULL, control=bfn.PERSISTENT, sweeps=1, boundary=0),
    dict(engine=bfn.JACOBI_PULL, control=bfn.CHUNKED, sweeps=0, boundary=0),
    dict(engine=bfn.DENSE_CHAOTIC_PUSH, control=bfn.PER_ROUND, sweeps=0, boundary=0),
    dict(engine=bfn.FRONTIER_PUSH, control=bfn.PERSISTENT, sweeps=0, boundary=0),
    dict(engine=bfn.FRONTIER_PUSH, control=bfn.CHUNKED, sweeps=0, boundary=1, window=4.0,
         per_claim=5),
]


def check_grid(device, dims, block):
    hg = bfn.HostGraph.synthetic(*dims, 7, host_graph=True)
    view = hg.view()
    dg = bfn.DeviceGraph(device, hg.layout())
    rng = np.random.default_rng(dims[2])
    ends = rng.integers(0, view["vertex_count"], (7, 2))
    tiles = np.arange(dims[0] * dims[1], dtype=np.uint32)
    batch = bfn.Batch([[int(s)] for s, _ in ends], [[int(t)] for _, t in ends], [tiles] * 7)
    want = [oracle_query(view, [int(s)], tiles)[0] for s, _ in ends]
    for c in CONFIGS:
        print("grid", dims, block, c, flush=True)
        ws = bfn.Workspace(device)
        ws.submit(dg, batch, bfn.run_options(engine=c["engine"], control_mode=c["control"],
                                             rounds_per_chunk=3, block_size=block),
                  bfn.tuning(tile_sweeps=c["sweeps"], boundary_mode=c["boundary"],
                             push_window=c.get("window", 0.0),
                             items_per_claim=c.get("per_claim", 1)))
        assert ws.status()[0].converged == 1, c
        for i in range(len(ends)):
            assert np.array_equal(bits(ws.distances(i)), bits(want[i])), (c, i)
        ws.close()
    dg.close()


@pytest.mark.parametrize("dims,block", [((1, 1, 130), 64), ((2, 1, 257), 64), ((1, 1, 2049), 512),
                                        ((2, 1, 1023), 256), ((4, 1, 1025), 256),
                                        ((3, 3, 2000), 1024)])
def test_few_large_tiles_bit_exact(device, dims, block):
    """Grids of few tiles, whose slabs the whole workgroup takes one by one:
    sizes about its four words per thread."""
    check_grid(device, dims, block)


@pytest.mark.parametrize("nodes,block", [(1, 64), (2, 256), (63, 64), (64, 128), (65, 256),
                                         (129, 64), (257, 256), (301, 512), (513, 256),
                                         (640, 1024)])
def test_tile_shapes_bit_exact(device, nodes, block):
    hg = bfn.HostGraph.synthetic(9, 8, nodes, 7, host_graph=True)
    view = hg.view()
    dg = bfn.DeviceGraph(device, hg.layout())
    qs = hg.synthetic_queries(7, seed=nodes, side_min=2, side_max=8, unbounded_fraction=0.2)
    tiles = [hg.query_tiles(q) for q in qs]
    batch = bfn.Batch([[q.source] for q in qs], [[q.target] for q in qs], tiles)
    want = [oracle_query(view, [q.source], t)[0] for q, t in zip(qs, tiles)]
    for c in CONFIGS:
        print("tile shapes", nodes, block, c, flush=True)
        ws = bfn.Workspace(device)
        ws.submit(dg, batch, bfn.run_options(engine=c["engine"], control_mode=c["control"],
                                             rounds_per_chunk=3, block_size=block),
                  bfn.tuning(tile_sweeps=c["sweeps"], boundary_mode=c["boundary"],
                             push_window=c.get("window", 0.0),
                             items_per_claim=c.get("per_claim", 1)))
        assert ws.status()[0].converged == 1, c
        for i in range(len(qs)):
            assert np.array_equal(bits(ws.distances(i)), bits(want[i])), (c, i)
        ws.close()
    dg.close()


@pytest.mark.parametrize("sources", [1, 63, 64, 65, 300])
def test_many_sources_bit_exact(device, sources):
    """Sources of one query are taken by the lanes of a wave, several of them in
    one tile."""
    hg = bfn.HostGraph.synthetic(9, 8, 33, 7, host_graph=True)
    view = hg.view()
    dg = bfn.DeviceGraph(device, hg.layout())
    rng = np.random.default_rng(sources)
    tiles = np.arange(72, dtype=np.uint32)
    batch = bfn.Batch([sorted(int(v) for v in rng.choice(72 * 33, n, False)) for n in (sources, 2)],
                      [[7], [11]], [tiles] * 2)
    want = [oracle_query(view, s, tiles)[0] for s in batch.sources]
    for c in CONFIGS:
        ws = bfn.Workspace(device)
        ws.submit(dg, batch, bfn.run_options(engine=c["engine"], control_mode=c["control"]),
                  bfn.tuning(tile_sweeps=c["sweeps"], boundary_mode=c["boundary"],
                             push_window=c.get("window", 0.0)))
        assert ws.status()[0].converged == 1, c
        for i in range(2):
            assert np.array_equal(bits(ws.distances(i)), bits(want[i])), (c, i)
        ws.close()
    dg.close()
