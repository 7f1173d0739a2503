"""Damage and bond breaking of the mixed bond kernels at the ends of their range:
a stretch that is no number shows in the damage of the nodes that have it (and
of no others), and bonds whose ends have met break."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import center_node
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu

H = 2.0 ** -13  # positions and their differences are exact in FP32


def _model(n, dim, shuffle):
    ax = [np.arange(n if d < dim else 1) * H for d in range(3)]
    x = np.stack([a.ravel() for a in np.meshgrid(*ax, indexing="ij")], 1)
    if shuffle:
        x = x[np.random.default_rng(1).permutation(len(x))]
    b = ModelBuilder(dim, 1e-9, [ZoneDeck(configs.pdstate_material(K=5e7))], {}, multi_particle=False)
    b.add_particle(0, x, np.full(len(x), H ** dim), center_node(x, (0, 0, 0), 1e-3), n * H)
    return b.build(name="damage", h_override=[H])


SHAPES = [(12, 2, False), (9, 3, False), (60, 2, True), (16, 3, True)]  # closed tiles, HBM tiles


@pytest.mark.parametrize("n,dim,shuffle", SHAPES)
def test_nan_stretch_shows_in_the_damage(n, dim, shuffle):
    spec = _model(n, dim, shuffle)
    print(f"[damage] nan {n}^{dim} shuffle={shuffle}", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    assert (g.tile_counts()[1] > 0) == shuffle
    far = spec.n_nodes // 2
    u = np.zeros_like(spec.x_ref)
    u[far, 0] = 1e25  # its square is infinite in FP32
    g.set_field(capi.FIELD_U, u)
    g.integrate_begin()
    rp, cols = g.neighbors(capi.NEIGH_PD)
    want = np.zeros(spec.n_nodes, bool)
    want[far] = True
    want[cols[rp[far]:rp[far + 1]]] = True
    z = g.field(capi.FIELD_Z)
    np.testing.assert_array_equal(np.isnan(z), want)
    assert (z[~want] == 0.0).all()
    g.close()


@pytest.mark.parametrize("broken", [False, True])
@pytest.mark.parametrize("n,dim,shuffle", SHAPES)
def test_bonds_whose_ends_have_met(n, dim, shuffle, broken):
    spec = _model(n, dim, shuffle)
    print(f"[damage] met {n}^{dim} shuffle={shuffle} broken={broken}", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    r = oracle.OracleEngine(spec, 8)
    bonds = np.full(len(r.field(capi.FIELD_BONDS)), int(broken), np.uint8)
    for e in (g, r):
        e.set_field(capi.FIELD_BONDS, bonds)
        e.set_field(capi.FIELD_U, -spec.x_ref)  # all nodes at one point
        e.integrate_begin()
    assert (r.field(capi.FIELD_BONDS) == 1).all()
    np.testing.assert_array_equal(g.field(capi.FIELD_BONDS), r.field(capi.FIELD_BONDS))
    np.testing.assert_array_equal(g.field(capi.FIELD_THETA), r.field(capi.FIELD_THETA))  # zeros
    np.testing.assert_allclose(g.field(capi.FIELD_Z), r.field(capi.FIELD_Z), rtol=5e-6)
    np.testing.assert_array_equal(np.isnan(g.field(capi.FIELD_F)), np.isnan(r.field(capi.FIELD_F)))
    g.close()
    r.close()
