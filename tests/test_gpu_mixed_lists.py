"""The shared neighbor lists of the mixed bond kernels against the FP64 oracle:
particles that share a list (copies of one mesh at other scales and angles),
particles that share none (every node moved), models of many different meshes
(the kernels then evaluate the bond weights), list lengths around the 8-bond
blocks, broken bonds in some blocks, bonds in the slack of the volume
correction's compare.  Tolerances as in test_gpu_mixed.py: those of FP32 bond
arithmetic, 1e-4 (max) and 1e-5 (RMS) of the largest force."""
import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node, disk_mesh, transform
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu


def _model(dim, meshes, inf, h=None):
    """One particle per mesh, far apart, no contact table needed."""
    mat = configs.pdstate_material(inf=inf)
    b = ModelBuilder(dim, 1e-8, [ZoneDeck(mat)], {}, multi_particle=False)
    for k, (x, vol) in enumerate(meshes):
        b.add_particle(0, x + np.array([5e-3 * k, 0.0, 0.0]), vol, center_node(x, (0, 0, 0), 1e-3), 1e-3)
    return b.build(name="mixed_lists", h_override=[h] + [None] * (len(meshes) - 1))


def _copies(dim, n, nodes, seed, jitter=0.0):
    rng = np.random.default_rng(seed)
    h = 1e-3 * ((4.18879 / nodes) ** (1 / 3) if dim == 3 else (3.14159 / nodes / 0.866) ** 0.5)
    ref, vol = (ball_mesh if dim == 3 else disk_mesh)(1e-3, h)
    out = []
    for _ in range(n):
        s = rng.uniform(0.7, 1.3)
        p = ref.copy()
        p[:, :dim] += jitter * h * rng.uniform(-1, 1, (len(p), dim))
        out.append((transform(p, (0, 0, 0), rng.uniform(0, 6.28), s), vol * s ** dim))
    return out


H_SLACK = 1e-4  # the mesh size handed to the model


def _slack_mesh():
    """A disk with some bonds longer than horizon - h/2 by half the slack of
    the relative compare (1e-5): their volume is not corrected."""
    x, vol = disk_mesh(1e-3, 1e-4)
    low = 2.5 * H_SLACK
    moved = 0
    for i in range(0, len(x), 37):
        d = np.linalg.norm(x - x[i], axis=1)
        j = int(np.argmin(np.abs(d - low)))
        x[j] = x[i] + (x[j] - x[i]) / d[j] * low * (1 + 5e-6)
        moved += 1
    assert moved > 3
    return [(x, vol)]


def _other_volumes(meshes, seed):
    """The same positions, so the same lists, with other nodal volumes."""
    rng = np.random.default_rng(seed)
    return [(x, vol * rng.uniform(0.8, 1.2, len(x))) for x, vol in meshes]


CASES = {
    "other_volumes_3d": lambda: _model(3, _copies(3, 2, 200, 12) + _other_volumes(_copies(3, 2, 200, 12), 13),
                                       capi.INF_LINEAR),
    "copies_3d": lambda: _model(3, _copies(3, 5, 300, 1), capi.INF_LINEAR),
    "copies_2d_const": lambda: _model(2, _copies(2, 7, 120, 2), capi.INF_CONST),
    "copies_2d_gauss": lambda: _model(2, _copies(2, 3, 367, 3), capi.INF_GAUSSIAN),
    "copies_and_others_3d": lambda: _model(3, _copies(3, 3, 120, 4) + _copies(3, 3, 120, 5, 0.1), capi.INF_LINEAR),
    "tiny_2d": lambda: _model(2, _copies(2, 2, 8, 6) + _copies(2, 2, 12, 7) + _copies(2, 2, 1300, 8), capi.INF_LINEAR),
    "many_meshes_3d": lambda: _model(3, _copies(3, 36, 1000, 9, 0.1), capi.INF_LINEAR),
    "slack_2d": lambda: _model(2, _slack_mesh(), capi.INF_LINEAR, H_SLACK),
    "many_meshes_slack_2d": lambda: _model(2, _slack_mesh() + _copies(2, 240, 380, 10, 0.1), capi.INF_CONST, H_SLACK),
}


@pytest.mark.parametrize("broken", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_lists_against_oracle(name, broken):
    spec = CASES[name]()
    print(f"[lists] {name} broken={broken} nodes={spec.n_nodes}", flush=True)
    rng = np.random.default_rng(11)
    u = np.zeros_like(spec.x_ref)
    for d in range(spec.dim):
        u[:, d] = 3e-7 * np.sin(2 * np.pi * spec.x_ref[:, (d + 1) % spec.dim] / 1e-3 + d)
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    r = oracle.OracleEngine(spec, 8)
    bonds = r.field(capi.FIELD_BONDS)
    if broken:
        # both ends of a few bonds, in most nodes of the first third of the particles
        rp, cols = r.neighbors(capi.NEIGH_PD)
        last = spec.particles[(len(spec.particles) - 1) // 3]["glob_end"]
        for i in range(0, last, 5):
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
    fg, fr = g.field(capi.FIELD_F), r.field(capi.FIELD_F)
    tg, tr = g.field(capi.FIELD_THETA), r.field(capi.FIELD_THETA)
    den = np.abs(fr).max()
    emax, erms = np.abs(fg - fr).max() / den, np.sqrt(((fg - fr) ** 2).sum(1).mean()) / den
    eth = np.abs(tg - tr).max() / np.abs(tr).max()
    ez = np.abs(g.field(capi.FIELD_Z) - r.field(capi.FIELD_Z)).max() / r.field(capi.FIELD_Z).max()
    print(f"[lists] {name} broken={broken}: max {emax:.2e} rms {erms:.2e} theta {eth:.2e} Z {ez:.2e}", flush=True)
    np.testing.assert_array_equal(g.field(capi.FIELD_BONDS), r.field(capi.FIELD_BONDS))
    assert den > 0.0 and emax < 1e-4 and erms < 1e-5 and eth < 1e-5 and ez < 5e-5
    # the two-pass kernels give the same bits as the fused one
    g.set_state_fusion(False)
    g.integrate_begin()
    np.testing.assert_array_equal(g.field(capi.FIELD_F), fg)
    np.testing.assert_array_equal(g.field(capi.FIELD_THETA), tg)
    g.close()
    r.close()
