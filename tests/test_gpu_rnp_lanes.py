"""The RNP force pass at the sizes where its kernel changes (16 lanes per node,
4 lanes per node, pair tiles): the default kernel, the lane-group kernel in
workgroups of 64 and the pair-tile kernel give the same forces, damage, bonds
and state bit for bit, with bonds broken from the start and bonds breaking."""
import numpy as np
import pytest

from peridem_amd import capi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("particles,nodes,default", [(9, 37, 256), (40, 340, 256), (50, 400, 256), (240, 400, 512)])
def test_kernels_agree_at_every_size(particles, nodes, default):
    spec = configs.compressive_2d(n_particles=particles, nodes_per_particle=nodes, seed=3, R_lo=1.0e-3, R_hi=1.02e-3,
                                  pitch_factor=1.01)
    print(f"[rnp lanes] nodes={spec.n_nodes}", flush=True)
    rng = np.random.default_rng(particles)
    u = np.zeros_like(spec.x_ref)
    u[:, 0] = 2e-5 * np.sin(2 * np.pi * spec.x_ref[:, 1] / 1e-3)
    u[:, 1] = 3e-7 * np.cos(2 * np.pi * spec.x_ref[:, 0] / 1e-3)
    runs = []
    for tpb in (0, 64, 512):
        g = capi.GpuEngine(spec, capi.PREC_FP64)
        if tpb:
            g.set_launch_config(tpb)
        assert g.launch_config()[0] == (tpb or default)
        if not runs:
            start = g.field(capi.FIELD_BONDS)
            start[rng.random(len(start)) < 0.1] = 1
        g.set_field(capi.FIELD_U, u)
        g.set_field(capi.FIELD_X, spec.x_ref + u)
        g.set_field(capi.FIELD_BONDS, start)
        g.integrate_begin()
        g.integrate_cd_graph(5)
        runs.append([g.field(f) for f in (capi.FIELD_F, capi.FIELD_U, capi.FIELD_V, capi.FIELD_Z, capi.FIELD_BONDS)])
        g.close()
    assert np.isfinite(runs[0][0]).all()
    assert start.sum() < runs[0][4].sum() < len(start)
    for r in runs[1:]:
        for a, b in zip(runs[0], r):
            np.testing.assert_array_equal(a, b)
