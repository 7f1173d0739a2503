"""Vector fields read from the engine are what was written (bit for bit), in
2D (third component zero) and 3D, from a few nodes to more than the 131072 that
are read at a time."""
import numpy as np
import pytest

from peridem_amd import capi, configs

pytestmark = pytest.mark.gpu

MODELS = {
    "2d_small": lambda: configs.two_particle(h=4e-4),
    "2d_bed": lambda: configs.compressive_2d(n_particles=370, nodes_per_particle=400, R_lo=1e-3, R_hi=1.02e-3),
    "3d": lambda: configs.single_particle_3d(nodes=700),
}


@pytest.mark.parametrize("name", sorted(MODELS))
def test_fields_round_trip(name):
    spec = MODELS[name]()
    print(f"[fields] {name} nodes={spec.n_nodes}", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_FP64)
    np.testing.assert_array_equal(g.field(capi.FIELD_XREF), spec.x_ref)
    rng = np.random.default_rng(7)
    for f in (capi.FIELD_U, capi.FIELD_V, capi.FIELD_F, capi.FIELD_X):
        a = rng.normal(size=(spec.n_nodes, 3))
        a[:, spec.dim:] = 0.0
        g.set_field(f, a)
        np.testing.assert_array_equal(g.field(f), a)
    g.close()
