"""HBM tiles of the mixed bond kernels (particles whose numbering spreads their
neighbors): 8 lanes a node or, in large models, one; an eighth of the tiles to
an XCD; nodes in mesh order or in any; weights evaluated, or read with the
Gaussian influence function.  Against the FP64 oracle (tolerances as in
test_gpu_mixed.py: 1e-4 max, 1e-5 RMS of the largest force), and a particle's
results bit for bit the same in a model of one particle and in one that takes
one lane."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu


def _model(copies, nodes, shuffle=True, inf=capi.INF_LINEAR):
    rng = np.random.default_rng(41)
    R = 1e-3
    h = R * (4.18879 / nodes) ** (1 / 3)
    x, vol = ball_mesh(R, h)
    if shuffle:
        x = x[rng.permutation(len(x))]
    b = ModelBuilder(3, 1e-9, [ZoneDeck(configs.pdstate_material(K=5e7, inf=inf))], {}, multi_particle=False)
    for k in range(copies):
        b.add_particle(0, x + np.array([5 * R * k, 0.0, 0.0]), vol, center_node(x, (0, 0, 0), R), R)
    return b.build(name="hbm", h_override=[h] * copies)


def _state(spec):
    """Displacements and broken bonds, the same for every copy."""
    n = spec.particles[0]["glob_end"]
    x = spec.x_ref[:n]
    u = np.tile(3e-7 * np.sin(2 * np.pi * x[:, [1, 2, 0]] / 1e-3), (len(spec.particles), 1))
    a = np.tile(np.random.default_rng(42).random(n), len(spec.particles))
    return u, a


def _run(e, spec):
    u, a = _state(spec)
    rp, cols = e.neighbors(capi.NEIGH_PD)
    rows = np.repeat(np.arange(spec.n_nodes), np.diff(rp))
    e.set_field(capi.FIELD_BONDS, ((a[rows] + a[cols]) * 7919.0 % 1.0 < 0.05).astype(np.uint8))
    e.set_field(capi.FIELD_U, u)
    e.set_field(capi.FIELD_X, spec.x_ref + u)
    e.integrate_begin()
    return tuple(e.field(k) for k in (capi.FIELD_F, capi.FIELD_THETA, capi.FIELD_Z, capi.FIELD_BONDS))


@pytest.mark.parametrize("copies,nodes,shuffle,inf", [
    (1, 2200, True, capi.INF_LINEAR), (4, 1500, True, capi.INF_LINEAR), (5, 2200, True, capi.INF_CONST),
    (2, 4000, False, capi.INF_LINEAR), (3, 2200, True, capi.INF_GAUSSIAN), (30, 2800, True, capi.INF_LINEAR),
    (20, 4000, False, capi.INF_LINEAR), (30, 2800, True, capi.INF_GAUSSIAN)])
def test_hbm_tiles(copies, nodes, shuffle, inf):
    spec = _model(copies, nodes, shuffle, inf)
    print(f"[hbm] {copies} x {nodes} shuffle={shuffle} inf={inf}: {spec.n_nodes} nodes", flush=True)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    assert g.tile_counts()[0] == 0
    r = oracle.OracleEngine(spec, 8)
    f, th, z, b = _run(g, spec)
    fr, tr, zr, br = _run(r, spec)
    den = np.abs(fr).max()
    emax, erms = np.abs(f - fr).max() / den, np.sqrt(((f - fr) ** 2).sum(1).mean()) / den
    eth, ez = np.abs(th - tr).max() / np.abs(tr).max(), np.abs(z - zr).max() / zr.max()
    print(f"[hbm]   tiles {g.tile_counts()}: max {emax:.2e} rms {erms:.2e} theta {eth:.2e} Z {ez:.2e}", flush=True)
    np.testing.assert_array_equal(b, br)
    assert emax < 1e-4 and erms < 1e-5 and eth < 1e-5 and ez < 5e-5
    g.close()
    r.close()


@pytest.mark.parametrize("shuffle,inf", [(True, capi.INF_LINEAR), (False, capi.INF_LINEAR), (True, capi.INF_GAUSSIAN)])
def test_lanes_agree(shuffle, inf):
    one, many = _model(1, 4000, shuffle, inf), _model(20, 4000, shuffle, inf)
    assert one.n_nodes <= 65536 < many.n_nodes
    out = []
    for spec in (one, many):
        g = capi.GpuEngine(spec, capi.PREC_MIXED)
        assert g.tile_counts()[0] == 0
        n = one.n_nodes
        out.append([a[:n] for a in _run(g, spec)[:3]])
        g.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
