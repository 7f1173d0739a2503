"""The FP64 state-based passes with a node's bonds dealt to four lanes against
the oracle: list lengths from 1 on (partial groups of four, the 32-bond words'
edges), broken bonds, bonds that break in the step, all influence functions.
Every operation runs in the oracle's order, so the results are equal (the
Gaussian influence function's exp may differ in the last ulp: 1e-13 of the
largest value)."""
import numpy as np
import pytest

from peridem_amd import capi
import oracle
from test_gpu_mixed_lists import _copies, _model

pytestmark = pytest.mark.gpu

CASES = {
    "tiny_2d": lambda: _model(2, _copies(2, 2, 8, 6) + _copies(2, 1, 12, 7) + _copies(2, 1, 90, 8), capi.INF_LINEAR),
    "disk_const": lambda: _model(2, _copies(2, 3, 367, 3), capi.INF_CONST),
    "disk_gauss": lambda: _model(2, _copies(2, 2, 150, 3), capi.INF_GAUSSIAN),
    "ball_linear": lambda: _model(3, _copies(3, 2, 300, 1), capi.INF_LINEAR),
    "ball_uneven": lambda: _model(3, _copies(3, 2, 37, 4, 0.1) + _copies(3, 1, 513, 5, 0.1), capi.INF_LINEAR),
}


@pytest.mark.parametrize("state", ["small", "breaking", "broken"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_state_passes_equal_oracle(name, state):
    spec = CASES[name]()
    print(f"[state64] {name} {state} nodes={spec.n_nodes}", flush=True)
    rng = np.random.default_rng(5)
    amp = 2e-5 if state == "breaking" else 3e-7
    u = np.zeros_like(spec.x_ref)
    for d in range(spec.dim):
        u[:, d] = amp * np.sin(2 * np.pi * spec.x_ref[:, (d + 1) % spec.dim] / 1e-3 + d)
    g, r = capi.GpuEngine(spec, capi.PREC_FP64), oracle.OracleEngine(spec, 4)
    bonds = r.field(capi.FIELD_BONDS)
    if state == "broken":
        bonds[rng.random(len(bonds)) < 0.2] = 1
    for e in (g, r):
        e.set_field(capi.FIELD_U, u)
        e.set_field(capi.FIELD_X, spec.x_ref + u)
        e.set_field(capi.FIELD_BONDS, bonds)
        e.integrate_begin()
    b = r.field(capi.FIELD_BONDS)
    np.testing.assert_array_equal(g.field(capi.FIELD_BONDS), b)
    if state == "breaking" and name != "tiny_2d":
        assert 0 < b.sum() < len(b)
    for f in (capi.FIELD_F, capi.FIELD_THETA, capi.FIELD_Z):
        a, c = g.field(f), r.field(f)
        if "gauss" in name:
            assert np.abs(a - c).max() <= (1e-6 if f == capi.FIELD_Z else 1e-13) * np.abs(c).max()
        else:
            np.testing.assert_array_equal(a, c)
    g.close()
    r.close()
