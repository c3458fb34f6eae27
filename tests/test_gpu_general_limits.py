"""Problems of the general path that its node records cannot hold, or do not describe, in a
call of 64 steps, which takes the step by elements and nodes where it can: they take the
launches one by one, as in shorter calls, and give the same results bit for bit."""
import ctypes

import numpy as np
import pytest

from conftest import case_par
from sem2dpack_amd import builder, solver

pytestmark = pytest.mark.gpu

NT = 64


def same(pb, **kw):
    one = solver.Solver(pb, structured=False, **kw)
    many = solver.Solver(pb, structured=False, **kw)
    one.step(NT)
    many.step(NT // 2)
    many.step(NT // 2)
    for x, y, nm in zip(one.fields(), many.fields(), "dva"):
        assert np.any(x != 0), nm
        assert np.array_equal(x, y), nm
    one.step(3)  # the refusal is remembered or asked again: a call is taken either way
    many.step(3)
    assert np.array_equal(one.fields()[0], many.fields()[0])
    return one


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n", [127, 128])  # 254 and 256 entries: a count has 8 bits
def test_many_sources_at_a_node(n, fp32):
    pb = builder.build(case_par("mesh2d_psv"), nsteps=2 * NT)
    src = pb.sources[0]
    rng = np.random.default_rng(n)
    pb.sources = [dict(src, kind="force", iglob=pb.npoin // 2, dir=rng.standard_normal(2),
                       stf_table=rng.standard_normal(2 * NT)) for _ in range(n)]
    same(pb, bulk_fp32=fp32)


@pytest.mark.parametrize("fp32", [False, True])
def test_sources_added_between_calls(fp32):
    """records first, then more sources at a node than they hold"""
    pb = builder.build(case_par("mesh2d_psv"), nsteps=3 * NT)
    src, n = pb.sources[0], 128
    rng = np.random.default_rng(n)
    tab = np.ascontiguousarray(rng.standard_normal(3 * NT))
    more = rng.standard_normal((n, 2))

    def run(per_call):
        s = solver.Solver(pb, structured=False, bulk_fp32=fp32)
        for k in range(0, NT, per_call):
            s.step(per_call)
        for d in more:  # one call each, the table set for every one
            isrc = ctypes.c_int()
            s._check(s.api.set_force(s.h, pb.npoin // 2, solver._p(np.ascontiguousarray(d)), ctypes.byref(isrc)),
                     "set_force")
            s._check(s.api.set_stf(s.h, isrc.value, len(tab), solver._p(tab)), "set_stf")
        for k in range(0, 2 * NT, per_call):
            s.step(per_call)
        return s.fields()

    assert src["kind"] == "force"
    for x, y, nm in zip(run(NT), run(NT // 2), "dva"):
        assert np.array_equal(x, y), nm


@pytest.mark.parametrize("fp32", [False, True])
def test_stacey_ends_of_a_periodic_boundary_without_its_pairs(fp32):
    """sem2d_set_abso_periodic after a Stacey boundary, without sem2d_set_periodic"""
    pb = builder.build(case_par("psv_stacey"), nsteps=2 * NT)
    rng = np.random.default_rng(7)
    for ab in pb.abso:
        if ab.get("stacey") is not None:
            ab["periodic_ends"] = True
    # forces at the ends of the boundaries, where the terms differ
    src = pb.sources[0]
    pb.sources = [dict(src, kind="force", iglob=int(g), dir=rng.standard_normal(2),
                       stf_table=rng.standard_normal(2 * NT))
                  for ab in pb.abso for g in (ab["node"][0], ab["node"][-1])]
    same(pb, bulk_fp32=fp32)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("case", ["sh_swf", "psv_rsf"])
def test_a_fault_pair_of_one_node(case, fp32):
    """Both sides of the last pair are the same node: its tractions cancel there, so the
    fields are those without the pair (up to the roundings of adding and subtracting it:
    one of the bulk type's a step, of a force no larger than the others)."""
    pb = builder.build(case_par(case), nsteps=2 * NT)
    without = solver.Solver(pb, structured=False)
    f = pb.fault
    lone = int(np.setdiff1d(np.arange(1, pb.npoin + 1), np.r_[f["node1"], f["node2"]])[pb.npoin // 3])
    f = pb.fault = dict(f)
    for k in ("node1", "node2"):
        f[k] = np.r_[f[k], np.int32(lone)].astype(np.int32)
    n = len(f["node1"])
    for k, x in list(f.items()):
        if isinstance(x, np.ndarray) and x.ndim and len(x) == n - 1:
            f[k] = np.concatenate([x, x[n // 2:n // 2 + 1]])
    f["invM2"][-1] = f["invM1"][-1]
    one = same(pb, bulk_fp32=fp32)
    assert np.any(one.fault_state()["T"][:, -1] != 0)  # it does slip
    if not fp32:
        without.step(NT)
        without.step(3)
        for x, y, nm in zip(one.fields(), without.fields(), "dva"):
            assert np.linalg.norm(x - y) < 1e-9 * np.linalg.norm(y), nm
