"""The SH traction rounds its product and its sum apart: T = Z (dV + a2v dA) + T0 with the
initial stress added to the rounded product, as in the rotated (P-SV) form of the solve.
With coefA2V = 1e-300 the acceleration's share is far below the last bit of the velocity
jump, so that the trial traction of a first step from a given velocity is known to the bit."""
import numpy as np
import pytest

from conftest import case_par
from sem2dpack_amd import builder, solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("structured", [True, False])
@pytest.mark.parametrize("case", ["sh_swf", "sh_kv", "sides_sh1"])  # the last one: one side
def test_trial_traction(case, structured, fp32):
    pb = builder.build(case_par(case), nsteps=4)
    f = pb.fault = dict(pb.fault, coefA2V=1e-300)
    s = solver.Solver(pb, bulk_fp32=fp32, structured=structured)
    rng = np.random.default_rng(3)
    v = np.zeros((1, pb.npoin))
    sides = [f["node1"]] if f["node2"] is None else [f["node1"], f["node2"]]
    for node in sides:
        v[0, node - 1] = rng.standard_normal(len(node))
    if fp32:
        v = v.astype(np.float32).astype(float)
    s.set_fields(v=v)
    s.step(1)
    v1 = v[0, f["node1"] - 1]
    jump = -2.0 * v1 if f["node2"] is None else v[0, f["node2"] - 1] - v1
    T0 = f["T0"][:, 0]
    want = (f["Z"][:, 0] * jump + T0) - T0
    got = s.fault_state()["Tstick"][0]
    assert np.all(np.abs(want) > 0)
    assert np.array_equal(got, want)
