"""Node costs on vertex counts that are no multiple of the kernels' blocks,
on both sides of the size up to which costs are checked on the host:
the weights of both orientations against the oracle, and refused costs
(negative, infinite, NaN) leaving the last accepted ones in place."""
import numpy as np
import pytest

import bfnew_amd as bfn
from helpers import bits, oracle_query

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(9, 8, 33), (32, 32, 257)])
def test_refused_costs_leave_the_last_ones(device, dims):
    hg = bfn.HostGraph.synthetic(*dims, 3, host_graph=True)
    view = hg.view()
    dg = bfn.DeviceGraph(device, hg.layout())
    costs = np.random.default_rng(1).uniform(0.5, 9.0, view["vertex_count"]).astype(np.float32)
    dg.update_node_costs(costs)
    for where, bad in ((0, -1.0), (255, np.inf), (view["vertex_count"] - 1, np.nan)):
        refused = costs + 1.0
        refused[where] = bad
        with pytest.raises(bfn.BfnError) as e:
            dg.update_node_costs(refused)
        assert e.value.code == 1
    tiles = np.arange(72, dtype=np.uint32)
    batch = bfn.Batch([[5]], [[2000]], [tiles])
    ws = bfn.Workspace(device)

    def expect(node_costs):
        view["weights"] = node_costs[view["destinations"]]
        want, _ = oracle_query(view, [5], tiles)
        for engine in (bfn.JACOBI_PULL, bfn.FRONTIER_PUSH):  # CSC and CSR weights
            ws.submit(dg, batch, bfn.run_options(engine=engine), bfn.tuning(tile_sweeps=0))
            assert np.array_equal(bits(ws.distances(0)), bits(want)), engine

    expect(costs)
    ws.path_arrays()
    occupancy = ws.occupancy()
    dg.update_node_costs_from_workspace(ws)  # on the accepted base costs
    expect(costs * (np.float32(1.0) + np.float32(0.5) * occupancy.astype(np.float32)))
    ws.close()
    dg.close()
