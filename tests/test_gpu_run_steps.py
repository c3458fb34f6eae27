"""Runs of steps of small grids: many steps in one launch (16 or more in one call on a grid
whose tiles are resident together) against the same steps in short calls, which launch each
step by itself, with the same arithmetic on the same values in the same order: equal to the
bit.  A launch whose waits are cut short leaves the state alone, and its steps are taken one
by one."""
import numpy as np
import pytest

from sem2dpack_amd import builder, parfile, solver, workloads

pytestmark = pytest.mark.gpu

NT = 40


def par(nx, nz, ndof, scheme="newmark"):
    lx, lz = 100.0 * nx, 100.0 * nz
    return (f"&GENERAL iexec=1, ngll=5, fmax=10d0, ndof={ndof}, title='runs', verbose='0000', ItInfo=1000 /\n"
            "&MESH_DEF method='CARTESIAN' /\n"
            f"&MESH_CART xlim=0d0,{lx!r}, zlim=0d0,{lz!r}, nelem={nx},{nz} /\n"
            "&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho=2670d0, cp=6000d0, cs=3464d0 /\n"
            "&BC_DEF tag=1, kind='ABSORB' /\n&BC_DEF tag=2, kind='ABSORB' /\n"
            "&BC_DEF tag=4, kind='DIRNEU' /\n&BC_DIRNEU h='D', v='N' /\n"
            f"&TIME kind='{scheme}', NbSteps={NT}, Dt=8d-4 /\n"
            f"&SRC_DEF stf='RICKER', coord={0.4 * lx!r},{0.6 * lz!r}, mechanism='FORCE' /\n"
            "&STF_RICKER f0=60d0, onset=0.02d0, ampli=1d9 /\n&SRC_FORCE angle=30d0 /\n"
            # the line crosses tile interiors, tile edges and the source
            f"&REC_LINE number=23, first=0d0,0d0, last={lx!r},{lz!r}, field='V', isamp=3, AtNode=T /\n")


def problem(nx, nz, ndof, medium, **kw):
    p = parfile.parse_par(par(nx, nz, ndof, **kw))
    if medium == "uniform":  # one set of point coefficients
        return builder.build(p)
    if medium != "elements":  # moduli continuous across elements, or but for one element
        grid = workloads.layered_random_grid((0.0, 100.0 * nx + 400.0), (0.0, 100.0 * nz + 400.0), dx=400.0)
        pb = builder.build(p, material=workloads.hete1_material(*grid), per_element_coefs=False)
        if medium == "points":
            pb.lam_mu = np.array(pb.lam_mu)
            pb.lam_mu[0] *= 1.01
        return pb
    n, rng = nx * nz, np.random.default_rng(nx)
    mu = 2670.0 * 3464.0 ** 2 * (1 + 0.1 * rng.random(n))
    return builder.build(p, elem_props=(2670.0 * np.ones(n), mu, mu), per_element_coefs=False)


def run(pb, steps, **kw):
    s = solver.Solver(pb, **kw)
    for n in steps:
        s.step(n)
    return [*s.fields(), s.seismograms()]


def same(a, b):
    assert np.any(a[0] != 0)
    for x, y, what in zip(a, b, ("d", "v", "a", "seismograms")):
        assert np.array_equal(x, y), what


# 130 x 128 P-SV in FP64 is one column of tiles more than are resident together
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nx,nz,ndof,medium", [(1, 1, 2, "uniform"), (9, 17, 2, "elements"), (24, 16, 2, "nodes"),
                                               (128, 128, 2, "uniform"), (130, 128, 2, "nodes"),
                                               (7, 9, 1, "uniform"), (33, 25, 1, "elements"), (170, 178, 1, "nodes"),
                                               (24, 16, 2, "points"), (10, 9, 1, "points")])
def test_runs(nx, nz, ndof, medium, fp32):
    print(f"\n[runs {nx}x{nz} ndof={ndof} {medium} fp32={fp32}]", flush=True)
    pb = problem(nx, nz, ndof, medium)
    same(run(pb, [NT], bulk_fp32=fp32), run(pb, [8] * 5, bulk_fp32=fp32))


def test_runs_between_progress_rows():
    pb = problem(17, 18, 2, "uniform", scheme="leapfrog")
    same(run(pb, [3, NT - 3], itinfo=18), run(pb, [8] * 5, itinfo=18))


def test_a_run_that_gives_up(monkeypatch):
    """waits of no poll at all: sooner or later a tile finds a neighbour not there yet"""
    pb = problem(64, 64, 2, "uniform")
    want = run(pb, [8] * 5)
    monkeypatch.setenv("SEM2D_RUN_SPINS", "0")
    same(run(pb, [NT]), want)
