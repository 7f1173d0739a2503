"""Mixed bond kernels that evaluate the bond weights (models of many different
meshes) at several mesh sizes against the FP64 oracle: the linear influence
function's slope p1 / (2 horizon h V) is a number of the model's units, and
the entries that pad a list to whole blocks must stay without effect whatever
it is.  Tolerances as in test_gpu_mixed.py: those of FP32 bond arithmetic,
1e-4 (max) and 1e-5 (RMS) of the largest force."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node, disk_mesh, transform
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu


def _model(dim, n, nodes, R, inf, j_scale):
    """n particles of radius 0.7 R to 1.3 R, all of different meshes.  j_scale
    multiplies the influence function, which forces and dilations do not
    depend on, so that the weighted volume of meshes below 0.07 mm stays in
    the accepted range."""
    rng = np.random.default_rng(21)
    mat = configs.pdstate_material(K=5e7, inf=inf)  # K far from 5 G / 3, where the dilation has no force
    h = R * ((4.18879 / nodes) ** (1 / 3) if dim == 3 else (3.14159 / nodes / 0.866) ** 0.5)
    ref, vol = (ball_mesh if dim == 3 else disk_mesh)(R, h)
    b = ModelBuilder(dim, 1e-8, [ZoneDeck(mat)], {}, multi_particle=False)
    for k in range(n):
        s = rng.uniform(0.7, 1.3)
        p = ref.copy()
        p[:, :dim] += 0.1 * h * rng.uniform(-1, 1, (len(p), dim))
        x = transform(p, (0, 0, 0), rng.uniform(0, 6.28), s)
        b.add_particle(0, x + np.array([5 * R * k, 0.0, 0.0]), vol * s ** dim, center_node(x, (0, 0, 0), R), R)
    spec = b.build(name="mixed_scales")
    spec.influence_fn_params = tuple(j_scale * p for p in spec.influence_fn_params)
    return spec


@pytest.mark.parametrize("broken", [False, True])
@pytest.mark.parametrize("dim,n,nodes,R,inf,j_scale", [
    (3, 42, 1000, 1.0e-3, capi.INF_LINEAR, 1.0),    # mesh size 0.11 to 0.21 mm
    (3, 42, 1000, 0.85e-3, capi.INF_LINEAR, 1.0),   # 0.09 to 0.18 mm
    (3, 42, 1000, 0.07e-3, capi.INF_LINEAR, 1e6),   # about 0.01 mm
    (3, 42, 1000, 7.0, capi.INF_LINEAR, 1.0),       # about 1 m
    (3, 42, 1000, 0.07e-3, capi.INF_CONST, 1e6),
    (2, 360, 380, 0.02e-3, capi.INF_LINEAR, 1e6),   # about 2 um
])
def test_evaluated_weights_at_scale(dim, n, nodes, R, inf, j_scale, broken):
    spec = _model(dim, n, nodes, R, inf, j_scale)
    print(f"[scales] {dim}D R={R} inf={inf} broken={broken} nodes={spec.n_nodes}", flush=True)
    u = np.zeros_like(spec.x_ref)
    for d in range(dim):
        u[:, d] = 3e-5 * R * np.sin(2 * np.pi * spec.x_ref[:, (d + 1) % dim] / R + d)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    assert g.list_info()[2], "the model reads its weights"
    r = oracle.OracleEngine(spec, 8)
    bonds = r.field(capi.FIELD_BONDS)
    if broken:
        # both ends of a few bonds in the first third of the particles
        rng = np.random.default_rng(22)
        rp, cols = r.neighbors(capi.NEIGH_PD)
        for i in range(0, spec.particles[n // 3]["glob_end"], 5):
            if rp[i + 1] > rp[i]:
                k = int(rng.integers(rp[i], rp[i + 1]))
                j = int(cols[k])
                bonds[k] = 1
                bonds[rp[j] + int(np.searchsorted(cols[rp[j]:rp[j + 1]], i))] = 1
    for e in (g, r):
        e.set_field(capi.FIELD_U, u)
        e.set_field(capi.FIELD_X, spec.x_ref + u)
        e.set_field(capi.FIELD_BONDS, bonds)
        e.integrate_begin()
    fr, tr, zr = r.field(capi.FIELD_F), r.field(capi.FIELD_THETA), r.field(capi.FIELD_Z)
    for fused in (True, False):
        if not fused:
            g.set_state_fusion(False)
            g.integrate_begin()
        fg, tg, zg = g.field(capi.FIELD_F), g.field(capi.FIELD_THETA), g.field(capi.FIELD_Z)
        assert np.isfinite(fg).all() and np.isfinite(tg).all()
        den = np.abs(fr).max()
        emax, erms = np.abs(fg - fr).max() / den, np.sqrt(((fg - fr) ** 2).sum(1).mean()) / den
        eth = np.abs(tg - tr).max() / np.abs(tr).max()
        ez = np.abs(zg - zr).max() / zr.max()
        print(f"[scales]   fused={fused}: max {emax:.2e} rms {erms:.2e} theta {eth:.2e} Z {ez:.2e}", flush=True)
        np.testing.assert_array_equal(g.field(capi.FIELD_BONDS), r.field(capi.FIELD_BONDS))
        assert emax < 1e-4 and erms < 1e-5 and eth < 1e-5 and ez < 5e-5
    g.close()
    r.close()
