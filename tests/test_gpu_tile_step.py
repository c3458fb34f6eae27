"""The tile kernel at the edges of its tiles (8 x 8 elements), and the state its steps hand
on inside one call: steps of one call pass the next step's predicted displacement and
velocity along and store d, v and a only at the call's end, steps called one by one store
them every time, with the same arithmetic on the same values."""
import numpy as np
import pytest

from sem2dpack_amd import builder, parfile, solver

pytestmark = pytest.mark.gpu

NT = 24
TOL = 1e-10  # the parity bar of FP64 runs against the oracle


def par(nx, nz, ndof, field, atnode, scheme="newmark", fault=False):
    sides = "".join(f"&BC_DEF tag={t}, kind='ABSORB' /\n" for t in (1, 2, 4))
    flt = ""
    if fault:
        flt = ("&BC_DEF tags=5,6, kind='DYNFLT' /\n&BC_DYNFLT friction='SWF', Tn=-120d6, Tt=82d6, oxi=1,9999,2 /\n"
               "&BC_DYNFLT_SWF Dc=0.4d0, MuS=0.677d0, MuD=0.525d0 /\n")
    lx, lz = 100.0 * nx, 100.0 * nz
    return (f"&GENERAL iexec=1, ngll=5, fmax=10d0, ndof={ndof}, title='tile edges', verbose='0000', ItInfo=1000 /\n"
            f"&MESH_DEF method='CARTESIAN' /\n"
            f"&MESH_CART xlim=0d0,{lx!r}, zlim=0d0,{lz!r}, nelem={nx},{nz}{', ezflt=-1' if fault else ''} /\n"
            "&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho=2670d0, cp=6000d0, cs=3464d0 /\n" + sides + flt +
            f"&TIME kind='{scheme}', NbSteps={NT}, Courant=0.3d0 /\n"
            f"&SRC_DEF stf='RICKER', coord={0.4 * lx!r},{0.6 * lz!r}, mechanism='FORCE' /\n"
            "&STF_RICKER f0=30d0, onset=0.04d0, ampli=1d9 /\n&SRC_FORCE angle=30d0 /\n"
            # the line crosses tile interiors, tile edges, the source and, in fault runs, the fault
            f"&REC_LINE number=23, first=0d0,0d0, last={lx!r},{lz!r}, field='{field}', isamp=2, "
            f"AtNode={'T' if atnode else 'F'} /\n")


def problem(nx, nz, ndof, varying=False, **kw):
    p = parfile.parse_par(par(nx, nz, ndof, **kw))
    if not varying:
        return builder.build(p)
    rng = np.random.default_rng(nx * 100 + nz)
    s = 1.0 + 0.1 * rng.random(nx * nz)
    mu = 2670.0 * 3464.0 ** 2 * s
    return builder.build(p, elem_props=(2670.0 * np.ones(nx * nz), mu, mu))


def both_ways(pb, fp32):
    one, many = solver.Solver(pb, bulk_fp32=fp32), solver.Solver(pb, bulk_fp32=fp32)
    one.step(NT)
    for _ in range(NT):
        many.step(1)
    return one, many


def same(a, b, what):
    assert np.array_equal(a, b), what


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("ndof", [1, 2])
@pytest.mark.parametrize("nx,nz", [(1, 1), (7, 9), (8, 8), (9, 17), (24, 16)])
def test_tile_edges(nx, nz, ndof, fp32, oracle_api):
    print(f"\n[tile edges {nx}x{nz} ndof={ndof} fp32={fp32}]", flush=True)
    pb = problem(nx, nz, ndof, field="V", atnode=True)
    one, many = both_ways(pb, fp32)
    for x, y, nm in zip(one.fields(), many.fields(), "dva"):
        same(x, y, nm)
    same(one.seismograms(), many.seismograms(), "seismograms")
    if fp32:
        return
    ref = solver.Solver(pb, api=oracle_api, compact=False)
    ref.step(NT)
    for x, y, nm in zip(list(one.fields()) + [one.seismograms()], list(ref.fields()) + [ref.seismograms()],
                        ("d", "v", "a", "seismograms")):
        assert np.linalg.norm(x - y) <= TOL * np.linalg.norm(y), nm


@pytest.mark.parametrize("field,atnode", [("D", True), ("A", True), ("V", False)])
@pytest.mark.parametrize("kw", [dict(fault=True), dict(scheme="leapfrog"), dict(varying=True)])
def test_recorded_fields(kw, field, atnode, oracle_api):
    """every recorded field, at nodes and interpolated, with a split fault on the way,
    the leapfrog scheme and per-element moduli"""
    print(f"\n[recorded {kw} {field} atnode={atnode}]", flush=True)
    pb = problem(17, 18, 2, field=field, atnode=atnode, **kw)
    one, many = both_ways(pb, False)
    same(one.seismograms(), many.seismograms(), "seismograms")
    for x, y, nm in zip(one.fields(), many.fields(), "dva"):
        same(x, y, nm)
    if kw.get("fault"):
        same(one.fault_records(), many.fault_records(), "fault records")
        same(one.potency(), many.potency(), "potency")
    ref = solver.Solver(pb, api=oracle_api, compact=False)
    ref.step(NT)
    x, y = one.seismograms(), ref.seismograms()
    assert np.linalg.norm(x - y) <= TOL * np.linalg.norm(y)
