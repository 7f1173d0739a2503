"""The contact search with particles that have left the grid of search cells
(its cell coordinates wrap around): inside it, across its border, many grid
widths away and beyond the range of cell coordinates.  The particles stay in
touching pairs, so there are candidates everywhere; the candidate sets equal
the oracle's (they are sets of nodes within a distance: no tolerance), in 2D
and 3D, from a fraction of a workgroup's nodes to more than 16384."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node, disk_mesh
from peridem_amd.model import ContactPairDeck, ModelBuilder, ZoneDeck
import oracle

from parity_util import same_sets

pytestmark = pytest.mark.gpu


def _pairs(dim, n, nodes):
    """n pairs of particles in a row, the two of a pair 0.7 mesh sizes apart."""
    h = 1e-3 * ((4.18879 / nodes) ** (1 / 3) if dim == 3 else (3.14159 / nodes / 0.866) ** 0.5)
    x, vol = (ball_mesh if dim == 3 else disk_mesh)(1e-3, h)
    cp = ContactPairDeck(contact_radius_factor=0.95, Kn=1e18, damping_on=False, friction_on=False)
    b = ModelBuilder(dim, 1e-9, [ZoneDeck(configs.rnp_material())], {(0, 0): cp}, search_factor=3.0)
    for k in range(n):
        for q in range(2):
            p = x + np.array([5e-3 * k, q * (np.ptp(x[:, 1]) + 0.7 * h), 0.0])
            b.add_particle(0, p, vol, center_node(p, p.mean(0), 1e-3), 1e-3)
    return b.build(name="pairs")


@pytest.mark.parametrize("where", ["inside", "border", "far", "beyond"])
@pytest.mark.parametrize("dim,n,nodes", [(2, 1, 100), (2, 8, 64), (3, 2, 520), (2, 40, 230)])
def test_candidates_outside_the_grid(dim, n, nodes, where):
    spec = _pairs(dim, n, nodes)
    print(f"[wrap] {dim}d pairs={n} nodes={spec.n_nodes} {where}", flush=True)
    rng = np.random.default_rng(n)
    ext = np.ptp(spec.x_ref, axis=0).max()
    amp = {"inside": 0.0, "border": 0.6, "far": 1e3, "beyond": 1e5 / ext}[where] * ext
    off = rng.uniform(-amp, amp, (n, 3))
    off[:, dim:] = 0.0
    x = spec.x_ref.copy()
    for k, p in enumerate(spec.particles):
        x[p["glob_start"]:p["glob_end"]] += off[k // 2]
    g, r = capi.GpuEngine(spec, capi.PREC_FP64, contact_capacity=512), oracle.OracleEngine(spec, 4)
    for e in (g, r):
        e.set_field(capi.FIELD_U, x - spec.x_ref)
        e.set_field(capi.FIELD_X, x)
        e.integrate_begin()
    a, b = g.neighbors(capi.NEIGH_CONTACT), r.neighbors(capi.NEIGH_CONTACT)
    assert np.diff(b[0]).sum() > 2 * n
    assert same_sets(*a, *b)
    g.close()
    r.close()
