"""Gradients on a grid split along a row of element edges (ezflt) with two stress-free
sides: the tiles of such a grid are two bands, each cut from its own first row, with one
node row more.  The halves do not interact, so each has a source; receivers on a diagonal
lie in tile interiors, on tile edges and between nodes of both.  J = <w, seismograms>; its
directional derivative is compared with the GPU forward's central difference, with the step
and the bar of the adjoint's other tests (truncation about 1e-8, round-off about 1e-9)."""
import numpy as np
import pytest

from sem2dpack_amd import adjoint

pytestmark = pytest.mark.gpu

NT = 90


def par(nx, nz, ez, field, atnode):
    lx, lz = 100.0 * nx, 100.0 * nz
    return ("&GENERAL iexec=1, ngll=5, fmax=10d0, ndof=2, title='split', verbose='0000', ItInfo=1000 /\n"
            "&MESH_DEF method='CARTESIAN' /\n"
            f"&MESH_CART xlim=0d0,{lx!r}, zlim=0d0,{lz!r}, nelem={nx},{nz}, ezflt={ez} /\n"
            "&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho=2670d0, cp=6000d0, cs=3464d0 /\n"
            + "".join(f"&BC_DEF tag={t}, kind='ABSORB' /\n" for t in (1, 2, 4)) +
            f"&TIME kind='newmark', NbSteps={NT}, Dt=8d-4 /\n"
            "&SRC_DEF stf='RICKER', mechanism='FORCE', file='sources.tab' /\n"
            "&STF_RICKER f0=30d0, onset=0.04d0, ampli=1d9 /\n&SRC_FORCE angle=30d0 /\n"
            f"&REC_LINE number=37, first=0d0,0d0, last={lx!r},{lz!r}, field='{field}', isamp=2, "
            f"AtNode={'T' if atnode else 'F'} /\n")


@pytest.mark.parametrize("field", ["D", "V", "A"])
@pytest.mark.parametrize("nx,nz,ez,atnode", [(20, 20, 10, True), (12, 12, 5, False), (9, 16, 8, True),
                                             (17, 20, 13, True)])
def test_gradient_of_a_split_grid(tmp_path, nx, nz, ez, atnode, field):
    print(f"\n[split adjoint {nx}x{nz} ezflt={ez} {field}]", flush=True)
    path = tmp_path / "Par.inp"
    path.write_text(par(nx, nz, ez, field, atnode))
    (tmp_path / "sources.tab").write_text("".join(f"{100.0 * nx * x!r} {100.0 * nz * z!r}\n"
                                                  for x, z in ((0.3, 0.25), (0.8, 0.8))))
    rng = np.random.default_rng(nx + 100 * nz)
    n = nx * nz
    mu = 2670.0 * 3464.0 ** 2 * (1 + 0.1 * rng.random(n))
    back = [2670.0 * (1 + 0.1 * rng.random(n)), 2670.0 * 6000.0 ** 2 - 2 * mu, mu]
    grads = []
    for seg in (0, 7):  # displacement history, checkpoints
        model = adjoint.SeismogramModel(str(path), seg=seg)
        seis = model.forward(*back)
        assert model._state.solver.adjoint_plan()[0] == (seg == 0)
        w = np.random.default_rng(1).standard_normal(seis.shape) / np.abs(seis).max()
        grads.append(model.backward(w))
        if seg:
            continue
        for k in range(3):
            dm = [(k == j) * 1e-4 * p * rng.standard_normal(n) for j, p in enumerate(back)]
            up = np.sum(w * model.forward(*[p + q for p, q in zip(back, dm)]))
            down = np.sum(w * model.forward(*[p - q for p, q in zip(back, dm)]))
            an = np.dot(grads[0][k], dm[k])
            assert abs(an - (up - down) / 2) < 1e-3 * abs(up - down) / 2, "rho lam mu".split()[k]
        model.close()
    adjoint.release()
    for a, b in zip(*grads):
        assert np.linalg.norm(a - b) < 1e-9 * np.linalg.norm(b)
