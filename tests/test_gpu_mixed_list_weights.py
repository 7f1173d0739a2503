"""Which bond weights a mixed-precision model stores: those of the LDS tiles'
distinct lists while the tiles read them, none where they evaluate them, and
HBM tiles' with the Gaussian influence function only.  Tiles with the same
entries share a list whatever their weights where these are evaluated."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu


def _model(kinds, inf=capi.INF_LINEAR):
    """One particle of 1021 nodes per kind: c a copy of the mesh, v with nodal
    volumes of its own, m with a mesh of its own, h numbered in any order
    (3000 nodes, HBM tiles)."""
    rng = np.random.default_rng(51)
    R = 1e-3
    h = R * (4.18879 / 1000) ** (1 / 3)
    b = ModelBuilder(3, 1e-9, [ZoneDeck(configs.pdstate_material(K=5e7, inf=inf))], {}, multi_particle=False)
    for k, kind in enumerate(kinds):
        x, vol = ball_mesh(R if kind != "h" else 1.45 * R, h)
        if kind == "v":
            vol = vol * rng.uniform(0.8, 1.2, len(x))
        elif kind == "m":
            x = x + 0.1 * h * rng.uniform(-1, 1, x.shape)
        elif kind == "h":
            x = x[rng.permutation(len(x))]
        x = np.rint(x * 2.0 ** 30) / 2.0 ** 30  # (copies are exact copies)
        b.add_particle(0, x + np.array([2.0 ** -7 * k, 0.0, 0.0]), vol, center_node(x, (0, 0, 0), R), R)
    return b.build(name="weights", h_override=[h] * len(kinds))


@pytest.mark.parametrize("kinds,inf,lists,evaluated,weights", [
    ("ccc", capi.INF_LINEAR, 1, False, "all"),
    ("cvv", capi.INF_LINEAR, 3, False, "all"),
    ("v" * 40, capi.INF_LINEAR, 1, True, "none"),          # 40 lists would be evaluated; then they are one
    ("m" * 40 + "vvc", capi.INF_CONST, 41, True, "none"),
    ("m" * 40 + "ch", capi.INF_LINEAR, 44, True, "none"),  # 3 HBM tiles
    ("vch", capi.INF_LINEAR, 5, False, "lds"),
    ("hvch", capi.INF_GAUSSIAN, 8, False, "all"),
    ("v" * 40, capi.INF_GAUSSIAN, 40, False, "all"),
])
def test_stored_weights(kinds, inf, lists, evaluated, weights):
    spec = _model(kinds, inf)
    print(f"[weights] {kinds[:4]}.. x{len(kinds)} inf={inf} nodes={spec.n_nodes}", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    n, entries, ev, w = g.list_info()
    print(f"[weights]   {n} lists of {entries} entries, {w} weights, evaluated={ev} tiles {g.tile_counts()}", flush=True)
    assert ev == evaluated and n == lists
    if weights == "lds":  # whole slices of 64 nodes and blocks of 8 bonds
        rp, _ = g.neighbors(capi.NEIGH_PD)
        bonds = rp[spec.particles[1]["glob_end"]]
        assert bonds <= w < 2 * bonds < entries
    else:
        assert w == (entries if weights == "all" else 0)
    r = oracle.OracleEngine(spec, 8)
    u = 3e-7 * np.sin(2 * np.pi * spec.x_ref[:, [1, 2, 0]] / 1e-3)
    for e in (g, r):
        e.set_field(capi.FIELD_U, u)
        e.set_field(capi.FIELD_X, spec.x_ref + u)
        e.integrate_begin()
    f, fr = g.field(capi.FIELD_F), r.field(capi.FIELD_F)
    den = np.abs(fr).max()
    assert np.abs(f - fr).max() < 1e-4 * den and np.sqrt(((f - fr) ** 2).sum(1).mean()) < 1e-5 * den
    g.close()
    r.close()
