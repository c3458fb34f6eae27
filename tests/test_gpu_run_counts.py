"""Which calls are taken as a run of steps in one launch: those of 17 steps or more on a grid
of at most one tile per compute unit.  A run of a larger grid is not tried: its tiles would
wait for others that are not running until they give up."""
import pytest

from conftest import case_par
from sem2dpack_amd import builder, solver
from test_gpu_run_steps import NT, problem

pytestmark = pytest.mark.gpu


def counts(pb, steps=(NT,), **kw):
    s = solver.Solver(pb, **kw)
    for n in steps:
        s.step(n)
    return s.run_counts()


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nx,nz,ndof,medium", [(1, 1, 2, "uniform"), (24, 16, 2, "points"), (33, 25, 1, "elements"),
                                               (128, 128, 2, "nodes"), (121, 121, 1, "nodes")])
def test_runs_are_taken(nx, nz, ndof, medium, fp32):
    assert counts(problem(nx, nz, ndof, medium), bulk_fp32=fp32) == (1, 0)


# one tile more than the 256 compute units (a row of them), and the most that two
# workgroups on each could hold
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("nx,nz,ndof,medium", [(8, 8 * 257, 1, "uniform"), (129, 128, 2, "uniform"),
                                               (200, 150, 1, "nodes"), (170, 178, 1, "points"),
                                               (170, 178, 1, "elements")])
def test_no_runs_of_more_tiles_than_are_resident(nx, nz, ndof, medium, fp32):
    print(f"\n[no runs {nx}x{nz} ndof={ndof} {medium} fp32={fp32}]", flush=True)
    assert counts(problem(nx, nz, ndof, medium), bulk_fp32=fp32) == (0, 0)


def test_no_runs_in_short_calls_and_beside_a_fault():
    assert counts(problem(24, 16, 2, "uniform"), [16] * 3) == (0, 0)
    assert counts(problem(24, 16, 2, "uniform"), structured=False) == (0, 0)
    assert counts(builder.build(case_par("sh_swf"), nsteps=NT)) == (0, 0)


def test_progress_rows_cut_runs():
    assert counts(problem(24, 16, 2, "uniform"), itinfo=20) == (2, 0)


def test_a_run_that_gives_up_is_not_tried_again(monkeypatch):
    """waits of no poll at all: of several tiles the first one through finds the others missing"""
    monkeypatch.setenv("SEM2D_RUN_SPINS", "0")
    s = solver.Solver(problem(64, 64, 2, "uniform"))
    s.step(NT)
    assert s.run_counts() == (0, 1)
    monkeypatch.delenv("SEM2D_RUN_SPINS")
    s.step(NT)
    assert s.run_counts() == (0, 1)
