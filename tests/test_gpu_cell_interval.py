"""Where the cell list is built depends on the model's size and on the search
interval of its deck: by the controller's workgroup up to 700 (interval - 1)
nodes, by three launches above (in every step for interval 1).  Models on both
sides of the line against the oracle: candidate sets after rebuilds, and the
state bit for bit as the parity tests have it."""
import pytest

from peridem_amd import capi, configs
import oracle

from parity_util import compare_state, same_sets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("particles,nodes,interval", [(4, 60, 1), (4, 60, 2), (4, 60, 3), (9, 60, 3), (9, 100, 3)])
def test_cells_by_interval(particles, nodes, interval, graph):
    spec = configs.compressive_2d(n_particles=particles, nodes_per_particle=nodes, seed=2, interval=interval,
                                  R_lo=1e-3, R_hi=1.02e-3, pitch_factor=1.01, dt=2e-8, init_speed=5.0)
    print(f"[cells] {spec.n_nodes} nodes, interval {interval}, line {700 * (interval - 1)}, graph={graph}", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_FP64)
    r = oracle.OracleEngine(spec, 8)
    for e in (g, r):
        e.integrate_begin()
    if graph:
        g.integrate_cd_graph(31)
    else:
        g.integrate_cd(31)
    r.integrate_cd(31)
    a, b = g.neighbors(capi.NEIGH_CONTACT), r.neighbors(capi.NEIGH_CONTACT)
    assert b[0][-1] > 0 and same_sets(*a, *b)
    compare_state(g, r, tag=f"interval {interval}")
    g.close()
    r.close()
