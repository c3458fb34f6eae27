"""sem2d_batch_config reports the tile kernel's launch as it is: workgroups of 384 threads
whatever was asked for, and no more workgroups than the tiles need."""
import pytest

from sem2dpack_amd import solver
from test_gpu_run_steps import problem

pytestmark = pytest.mark.gpu


def test_batch_reports_its_launch():
    pb = problem(24, 16, 2, "nodes")
    pb.dirichlet = []  # not batched
    b = solver.Batch([solver.Solver(pb) for _ in range(3)])
    tiles = 3 * 3 * 2
    for threads in (256, 512):
        b.set_config(threads, 0)
        assert b.config() == dict(threads=384, workgroups=(tiles + 7) // 8 * 8, ntiles=tiles)
    b.tune(1)
    assert b.config()["threads"] == 384
