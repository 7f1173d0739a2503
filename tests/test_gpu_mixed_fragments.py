"""Mixed bond kernels on particles whose parts have flown apart: the displacement
records of a particle are fixed-point numbers of 30 bits over the particle's
largest relative displacement, and nothing in the bond passes may be coarser.
The error against the FP64 oracle is held to that of the displacements rounded
to this step (the oracle's forces for the rounded displacements) plus that of
FP32 bond arithmetic, 1e-6 (RMS) and 1e-5 (max) of the largest force."""
import math

import numpy as np
import pytest

from peridem_amd import capi, configs
from peridem_amd.geometry import ball_mesh, center_node, disk_mesh
from peridem_amd.model import ModelBuilder, ZoneDeck
import oracle

pytestmark = pytest.mark.gpu


def _model(dim, nodes, shuffle):
    rng = np.random.default_rng(5)
    R = 1e-3
    h = R * ((4.18879 / nodes) ** (1 / 3) if dim == 3 else (3.14159 / nodes / 0.866) ** 0.5)
    x, vol = (ball_mesh if dim == 3 else disk_mesh)(R, h)
    if shuffle:
        p = rng.permutation(len(x))
        x, vol = x[p], vol[p]
    b = ModelBuilder(dim, 1e-9, [ZoneDeck(configs.pdstate_material(K=5e7, Gc=5e4))], {}, multi_particle=False)
    b.add_particle(0, x, vol, center_node(x, (0, 0, 0), R), R)
    return b.build(name="fragments")


@pytest.mark.parametrize("far", [0.01, 1.0])
@pytest.mark.parametrize("part", ["half", "first_node"])
@pytest.mark.parametrize("dim,nodes,shuffle,fused", [
    (2, 300, False, True), (3, 1000, False, True),   # a closed tile
    (2, 2500, False, True), (3, 1000, False, False),  # open LDS tiles
    (2, 2500, True, True), (3, 3000, True, True),    # HBM tiles
])
def test_fragments(dim, nodes, shuffle, fused, part, far):
    spec = _model(dim, nodes, shuffle)
    x = spec.x_ref
    print(f"[fragments] {dim}D {spec.n_nodes} shuffle={shuffle} fused={fused} {part} {far} m", flush=True)
    moved = x[:, 0] > 0.0 if part == "half" else np.arange(spec.n_nodes) == 0
    # large strains, where a bond's direction counts as much as its stretch
    u = np.zeros_like(x)
    for d in range(dim):
        u[:, d] = 0.2 * x[:, d] + 2e-5 * np.sin(2 * np.pi * x[:, (d + 1) % dim] / 1e-3 + d)
        u[moved, d] += far * (0.7, -0.9, 0.4)[d]
    g = capi.GpuEngine(spec, capi.PREC_MIXED)
    g.set_state_fusion(fused)
    lds, hbm = g.tile_counts()
    assert (hbm > 0) == shuffle and (lds > 0) != shuffle
    r = oracle.OracleEngine(spec, 8)
    rp, cols = r.neighbors(capi.NEIGH_PD)
    bonds = (moved[np.repeat(np.arange(spec.n_nodes), np.diff(rp))] != moved[cols]).astype(np.uint8)

    def forces(e, disp):
        e.set_field(capi.FIELD_U, disp)
        e.set_field(capi.FIELD_X, x + disp)
        e.set_field(capi.FIELD_BONDS, bonds)
        e.integrate_begin()
        return e.field(capi.FIELD_F), e.field(capi.FIELD_THETA)

    f, th = forces(r, u)
    np.testing.assert_array_equal(r.field(capi.FIELD_BONDS), bonds)  # no other bond breaks
    step = 2.0 ** (math.frexp(np.abs(u - u[0]).max())[1] - 29)
    fq, tq = forces(r, u[0] + np.rint((u - u[0]) / step) * step)
    fg, tg = forces(g, u)
    den, dth = np.abs(f).max(), np.abs(th).max()

    def rms(a):
        return np.sqrt((a ** 2).mean())

    print(f"[fragments]   max {np.abs(fg - f).max() / den:.2e} (rounded {np.abs(fq - f).max() / den:.2e}) rms "
          f"{rms(fg - f) / den:.2e} ({rms(fq - f) / den:.2e}) theta {rms(tg - th) / dth:.2e} ({rms(tq - th) / dth:.2e})",
          flush=True)
    # the rounding of another representative of the step's class: within a factor of 2
    assert rms(fg - f) <= 2.0 * rms(fq - f) + 1e-6 * den
    assert np.abs(fg - f).max() <= 2.0 * np.abs(fq - f).max() + 1e-5 * den
    assert rms(tg - th) <= 2.0 * rms(tq - th) + 1e-6 * dth
    g.close()
    r.close()
