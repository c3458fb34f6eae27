"""Workloads of the time step, from a user's program: whole runs, time loops, ruptures,
a scenario ensemble and waveform gradients, with their inputs, their outputs, the work
they cannot do without and the values plain 64-bit torch gives for them.

Every input is made as a user makes it, from an input file's text through the builder.
All grids have square elements of 100 m unless they are layered.  Runs with an FP32 bulk
hand their outputs over as float32, which is what the solver holds them in and what the
seismogram and fault files store.
"""
import copy
import functools
import math

import numpy as np
import torch

from sem2dpack_amd import builder, parfile, solver, workloads

RHO, CP, CS = 2670.0, 6000.0, 3464.0


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a first run or a unit test of a set-up: the size of the Lamb's problem example
        # (NGLL 9, leapfrog, free surface), from a new solver to the fetched fields
        dict(name="run_psv_ngll9_40x20", kind="run", nx=40, nz=20, ndof=2, ngll=9, scheme="leapfrog", steps=400,
             fp32=False),
        # the reference's own CPU-runnable case, whole
        dict(name="run_psv_100x100", kind="run", nx=100, nz=100, ndof=2, ngll=5, scheme="newmark", steps=2000,
             fp32=False),
        # a run on a mesh that follows layer interfaces (general element geometry)
        dict(name="run_psv_layered_201x120", kind="run", nx=201, nz=120, ndof=2, ngll=5, scheme="layered", steps=2000,
             fp32=False),
        # a stretch of the time loop of a shot in a heterogeneous box: an antiplane one of
        # odd size, and the large in-plane one with each bulk precision
        dict(name="loop_sh_333x251_f32", kind="loop", nx=333, nz=251, ndof=1, steps=400, fp32=True),
        dict(name="loop_psv_1400x700", kind="loop", nx=1400, nz=700, ndof=2, steps=40, fp32=False),
        dict(name="loop_psv_1400x700_f32", kind="loop", nx=1400, nz=700, ndof=2, steps=40, fp32=True),
        # a stretch of a dynamic rupture: the antiplane slip-weakening configuration, with
        # each bulk precision, and an in-plane one with Kelvin-Voigt damping by the fault
        dict(name="rupture_sh_600x300", kind="rupture", nx=600, nz=300, ndof=1, kv=False, steps=300, fp32=False),
        dict(name="rupture_sh_600x300_f32", kind="rupture", nx=600, nz=300, ndof=1, kv=False, steps=300, fp32=True),
        dict(name="rupture_psv_kv_241x120", kind="rupture", nx=241, nz=120, ndof=2, kv=True, steps=200, fp32=False),
        # an ensemble of rate-and-state ruptures of uneven sizes advanced together
        dict(name="ensemble_rsf_24_f32", kind="ensemble", members=24, nx_min=100, nx_max=300, steps=128, fp32=True),
        # one gradient of an inversion: forward and adjoint, with the forward history in
        # memory, and with recomputed checkpoints
        dict(name="gradient_400x400", kind="gradient", nx=400, nz=400, steps=200, seg=0, fp32=False),
        dict(name="gradient_150x101_ckpt", kind="gradient", nx=150, nz=101, steps=300, seg=18, fp32=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "loop", "loop", "rupture", "rupture", "ensemble", "gradient"])
    c = dict(kind=kind)
    if kind == "run":
        scheme = rng.choice(["leapfrog", "newmark", "newmark", "layered"])
        # other orders than NGLL 5 are for small boxes
        ngll = rng.choice([4, 6, 7, 8, 9, 10]) if scheme == "leapfrog" and rng.random() < 0.5 else 5
        nx = _log(rng, 20, 60 if ngll != 5 else 240)
        c.update(nx=nx, nz=max(10, int(nx * rng.uniform(0.4, 1.0))), ndof=rng.choice([1, 2]), ngll=ngll,
                 scheme=scheme, steps=rng.randint(500, 2000), fp32=rng.random() < 0.3)
    elif kind == "loop":
        nx = _log(rng, 60, 1400)
        nz = max(30, int(nx * rng.uniform(0.4, 0.7)))
        c.update(nx=nx, nz=min(nz, 700), ndof=rng.choice([1, 2, 2]), steps=max(40, min(400, int(4e7 / (nx * nz)))),
                 fp32=rng.random() < 0.5)
    elif kind == "rupture":
        nx = _log(rng, 80, 600)
        ndof = rng.choice([1, 2])
        c.update(nx=nx, nz=max(32, 2 * int(nx * rng.uniform(0.2, 0.25))), ndof=ndof, kv=rng.random() < 0.4,
                 steps=rng.randint(100, 300), fp32=rng.random() < 0.5)
    elif kind == "ensemble":
        lo = rng.randint(60, 120)
        c.update(members=rng.randint(4, 24), nx_min=lo, nx_max=lo + rng.randint(20, 180), steps=rng.randint(64, 128),
                 fp32=rng.random() < 0.7)
    else:
        nx = _log(rng, 60, 400)
        steps = rng.randint(80, 200)
        c.update(nx=nx, nz=max(40, int(nx * rng.uniform(0.5, 1.0))), steps=steps,
                 seg=rng.choice([0, 0, int(math.ceil(math.sqrt(steps)))]), fp32=rng.random() < 0.4)
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
ABSORB = "".join(f"&BC_DEF tag={t}, kind='ABSORB' /\n" for t in (1, 2, 4))  # bottom, right, left


def _run_par(c, rng):
    """Point force below a free surface, absorbing sides and bottom; a line of receivers."""
    lx, lz = 100.0 * c["nx"], 100.0 * c["nz"]
    head = (f"&GENERAL iexec=1, ngll={c['ngll']}, fmax=20d0, ndof={c['ndof']}, title='point force', verbose='0000', "
            f"ItInfo=100000 /\n")
    if c["scheme"] == "layered":
        # three layers; the middle interface dips
        n1 = max(2, c["nz"] // 4)
        n2 = max(2, c["nz"] // 3)
        n3 = c["nz"] - n1 - n2
        z1, z2 = -100.0 * n1, -100.0 * (n1 + n2)
        dip = float(rng.uniform(0.1, 0.3)) * 100.0 * n1
        mesh = (f"&MESH_DEF method='LAYERED' /\n"
                f"&MESH_LAYERED xlim=0d0,{lx!r}, zmin={-lz!r}, nx={c['nx']}, nlayer=3 /\n"
                f"&MESH_LAYER nz={n1}, ztop=0d0 /\n&MESH_LAYER nz={n2}, ztopH='LINEAR' /\n"
                f"&DIST_LINEAR n=3 /\n 0d0 {z1!r}\n {0.6 * lx!r} {z1 + dip!r}\n {lx!r} {z1 - dip!r}\n"
                f"&MESH_LAYER nz={n3}, ztop={z2!r}, tag=3 /\n"
                "&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho=2100d0, cp=3000d0, cs=1600d0 /\n"
                "&MATERIAL tag=2, kind='ELAST' /\n&MAT_ELASTIC rho=2400d0, cp=4500d0, cs=2500d0 /\n"
                f"&MATERIAL tag=3, kind='ELAST' /\n&MAT_ELASTIC rho={RHO!r}, cp={CP!r}, cs={CS!r} /\n")
    else:
        mesh = (f"&MESH_DEF method='CARTESIAN' /\n"
                f"&MESH_CART xlim=0d0,{lx!r}, zlim={-lz!r},0d0, nelem={c['nx']},{c['nz']} /\n"
                f"&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho={RHO!r}, cp={CP!r}, cs={CS!r} /\n")
    f0 = float(rng.uniform(10.0, 20.0))
    time = "kind='leapfrog', " if c["scheme"] == "leapfrog" else "kind='newmark', "
    force = "&SRC_FORCE angle=0d0 /\n" if c["ndof"] == 2 else "&SRC_FORCE /\n"
    return (head + mesh + ABSORB + f"&TIME {time}NbSteps={c['steps']}, Courant=0.3d0 /\n"
            f"&SRC_DEF stf='RICKER', coord={float(rng.uniform(0.3, 0.7)) * lx!r},{-float(rng.uniform(0.2, 0.5)) * lz!r}, "
            f"mechanism='FORCE' /\n"
            f"&STF_RICKER f0={f0!r}, onset={1.1 / f0!r}, ampli={float(rng.uniform(0.5, 2.0))!r} /\n"
            + force +
            f"&REC_LINE number=9, first={0.1 * lx!r},0d0, last={0.9 * lx!r},0d0, field='V' /\n")


@functools.lru_cache(maxsize=1)
def _loop_medium(nx, nz, ndof):
    """The box of a survey: one medium (eight layers and a random perturbation), in which
    many shots are run.  The random field is drawn on a grid of 400 m."""
    lx, lz = 100.0 * nx, 100.0 * nz
    grid = workloads.layered_random_grid((0.0, lx + 400.0), (0.0, lz + 400.0), dx=400.0)
    par = workloads.par_throughput(nx, nz, lx, lz, nt=12000, nrec=64).replace("ndof=2", f"ndof={ndof}")
    if ndof == 1:
        par = par.replace("mechanism='EXPLOSION'", "mechanism='FORCE'").replace("&REC_LINE", "&SRC_FORCE /\n&REC_LINE")
    return builder.build(parfile.parse_par(par), material=workloads.hete1_material(*grid), per_element_coefs=False)


def _loop_problem(c, seed):
    """(problem, d, v): one shot in the medium, restarted from a wavefield in flight."""
    rng = np.random.Generator(np.random.PCG64(seed))
    base = _loop_medium(c["nx"], c["nz"], c["ndof"])
    pb = copy.copy(base)
    t = pb.dt * np.arange(1, pb.nt + 1)
    arg = (math.pi * rng.uniform(0.7, 1.5) * (t - 0.2)) ** 2
    pb.sources = [dict(base.sources[0], kind="force", iglob=int(rng.integers(1, pb.npoin + 1)),
                       dir=rng.standard_normal(c["ndof"]), stf_table=1e9 * (1 - 2 * arg) * np.exp(-arg))]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.as_tensor(pb.coord, device=dev)
    d = torch.zeros((c["ndof"], pb.npoin), dtype=torch.float64, device=dev)
    v = torch.zeros_like(d)
    for _ in range(4):  # plane waves of 0.5 to 3 km
        th, k = rng.uniform(0, 2 * math.pi), 2 * math.pi / rng.uniform(500.0, 3000.0)
        ph = x[:, 0] * (k * math.cos(th)) + x[:, 1] * (k * math.sin(th)) + rng.uniform(0, 2 * math.pi)
        pol = (math.cos(th), math.sin(th)) if c["ndof"] == 2 else (1.0,)
        om = k * 5000.0
        for q in range(c["ndof"]):
            d[q] += 1e-3 * pol[q] * torch.cos(ph)
            v[q] += 1e-3 * om * pol[q] * torch.sin(ph)
    return pb, d.cpu().numpy(), v.cpu().numpy()


def _rupture_par(c, rng):
    """Slip weakening on a split fault through the middle, nucleated by raised stress."""
    nx, nz = c["nx"], c["nz"]
    lx, lz = 100.0 * nx, 100.0 * nz
    r0 = float(rng.uniform(0.12, 0.16)) * lx
    tau = 1e6 * float(rng.uniform(81.6, 84.0))
    zone = ", fztag=2, fznz=2" if c["kv"] else ""
    kv = ("&MATERIAL tag=2, kind='ELAST','KV' /\n"
          f"&MAT_ELASTIC rho={RHO!r}, cp={CP!r}, cs={CS!r} /\n&MAT_KV eta=0.1d0 /\n") if c["kv"] else ""
    sides = "".join(f"&BC_DEF tag={t}, kind='ABSORB' /\n" for t in (1, 2, 3, 4))
    return (f"&GENERAL iexec=1, ngll=5, fmax=3d0, ndof={c['ndof']}, title='rupture', verbose='0000', ItInfo=100000 /\n"
            f"&MESH_DEF method='CARTESIAN' /\n"
            f"&MESH_CART xlim={-0.5 * lx!r},{0.5 * lx!r}, zlim={-0.5 * lz!r},{0.5 * lz!r}, nelem={nx},{nz}, "
            f"ezflt=-1{zone} /\n"
            f"&MATERIAL tag=1, kind='ELAST' /\n&MAT_ELASTIC rho={RHO!r}, cp={CP!r}, cs={CS!r} /\n" + kv + sides +
            f"&BC_DEF tags=5,6, kind='DYNFLT' /\n"
            f"&BC_DYNFLT friction='SWF', Tn=-120d6, TtH='PWCONR', otd=1d-1, oxi=1,{2 ** 31 - 1},4 /\n"
            f"&DIST_PWCONR num=2, ref=0d0,0d0 /\n{r0!r}\n{tau!r} 70d6\n"
            f"&BC_DYNFLT_SWF Dc=0.4d0, MuS=0.677d0, MuD=0.525d0 /\n"
            f"&TIME kind='newmark', NbSteps=12000, Courant=0.2d0 /\n")


def _ensemble_problems(c, seed):
    """The case's sizes; friction and stress of every member from the seed."""
    sizes = workloads.rupture_ensemble(c["members"], nx_min=c["nx_min"], nx_max=c["nx_max"])
    media = workloads.rupture_ensemble(c["members"], seed=seed)
    return [workloads.build_rupture(dict(z, a=m["a"], seed=m["seed"]), nt=8192) for z, m in zip(sizes, media)]


def _gradient_problem(c, seed):
    """(problem, observed traces): per-element model, 8 forces fired together, 48 receivers."""
    nx, nz = c["nx"], c["nz"]
    rng = np.random.Generator(np.random.PCG64(seed))
    par = workloads.par_adjoint(nx, nz, c["steps"], 48, f0=20.0, onset=0.055, dt="8.6d-4")
    par = par.replace(", file='sources.tab'", f", coord={50.0 * nx!r},{100.0 * nz - 1000.0!r}")
    rho, lam, mu = workloads.adjoint_models(nx, nz, seed=int(rng.integers(1 << 30)))[1]
    pb = builder.build(parfile.parse_par(par), per_element_coefs=False, elem_props=(rho, lam, mu))
    src = pb.sources[0]
    zs = np.nonzero(np.abs(pb.coord[:, 1] - (100.0 * nz - 500.0)) < 1.0)[0] + 1
    pb.sources = [dict(src, iglob=int(g), stf_table=float(rng.uniform(0.5, 1.5)) * src["stf_table"])
                  for g in rng.choice(zs, size=8, replace=False)]
    r = pb.receivers
    t = pb.dt * np.arange(r["nsamp"])[:, None, None]
    arrive = rng.uniform(0.05, 0.15, size=(1, 2, len(r["iglob"])))
    arg = (math.pi * 20.0 * (t - arrive)) ** 2
    return pb, 1e-13 * (1 - 2 * arg) * np.exp(-arg)


def _problem(c, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    par = _run_par(c, rng) if c["kind"] == "run" else _rupture_par(c, rng)
    return builder.build(parfile.parse_par(par))


# ---------------------------------------------------------------------------
# What a program holds before the call, and the call
# ---------------------------------------------------------------------------
def prepare(c, seed):
    kind, fp32 = c["kind"], c["fp32"]
    st = dict(c=c)
    if kind == "run":  # a new solver is part of the run
        st["pb"] = _problem(c, seed)
    elif kind == "loop":
        pb, d, v = _loop_problem(c, seed)
        st["s"] = solver.Solver(pb, bulk_fp32=fp32, keep_problem=False)
        st["s"].set_fields(d=d, v=v)
    elif kind == "rupture":
        st["s"] = solver.Solver(_problem(c, seed), bulk_fp32=fp32)
    elif kind == "ensemble":
        st["b"] = solver.Batch([solver.Solver(pb, bulk_fp32=fp32) for pb in _ensemble_problems(c, seed)])
        st["b"].tune(2)
    else:
        pb, st["obs"] = _gradient_problem(c, seed)
        st["s"] = solver.Solver(pb, bulk_fp32=fp32)
        st["s"].adjoint_init(c["steps"], c["seg"])
    return st


def _out(c, tree):
    return {k: np.asarray(x, dtype=np.float32) for k, x in tree.items()} if c["fp32"] else tree


def run(st):
    c = st["c"]
    if c["kind"] == "run":
        s = solver.Solver(st["pb"], bulk_fp32=c["fp32"])
        s.step(c["steps"])
        d, v, a = s.fields()
        out = dict(seis=s.seismograms(), d=d, v=v, a=a)
        s.close()
    elif c["kind"] == "loop":
        st["s"].step(c["steps"])
        out = dict(seis=st["s"].seismograms())
    elif c["kind"] == "rupture":
        st["s"].step(c["steps"])
        out = st["s"].fault_state()
    elif c["kind"] == "ensemble":
        b = st["b"]
        b.step(c["steps"])
        per = [b.fault_state(m) for m in range(c["members"])]
        out = {k: np.concatenate([p[k].ravel() for p in per]) for k in ("D", "V", "T", "MU", "Tstick")}
    else:
        s = st["s"]
        s.adjoint_forward()
        seis = s.seismograms()
        s.adjoint_backward(seis - st["obs"])
        lam, mu, mass, abso = s.adjoint_fetch()
        out = dict(seis=seis, lam=lam, mu=mu, mass=mass, abso=abso)
    return _out(c, out)


# ---------------------------------------------------------------------------
# The work of one pass
# ---------------------------------------------------------------------------
def work(c):
    """Per step: displacement and velocity read and written, the inverse mass, and the
    moduli where they vary, once per node (the acceleration follows from the forces);
    the products with H, the stresses and the update as operations.  A gradient reads
    the forward's displacement, acceleration and predicted velocity and the adjoint's
    displacement and velocity, and updates these and the mass sensitivity."""
    s = 4 if c["fp32"] else 8
    if c["kind"] == "ensemble":
        nxs = [(c["nx_min"] + c["nx_max"]) / 2] * c["members"]
        boxes = [(nx, nx / 2) for nx in nxs]
    else:
        boxes = [(c["nx"], c["nz"])]
    nd, ng = c.get("ndof", 2), c.get("ngll", 5)
    npoin = sum((nx * (ng - 1) + 1) * (nz * (ng - 1) + 1) for nx, nz in boxes)
    pts = sum(nx * nz for nx, nz in boxes) * ng * ng
    mod = (nd if c["kind"] in ("loop", "gradient") else 0)
    flops = pts * nd * (8 * ng + 12) + npoin * nd * 9
    words = 4 * nd + 1 + mod
    if c["kind"] == "gradient":
        flops, words = 3 * flops, words + 4 * nd + 1 + 2 * nd + 2 + mod
    return dict(bytes=float(c["steps"] * npoin * words * s), flops=float(c["steps"] * flops))


# ---------------------------------------------------------------------------
# The same in plain 64-bit torch
# ---------------------------------------------------------------------------
class _Exact:
    """The spectral-element time step on a problem's mesh, media, boundaries, sources and
    fault, written out with tensors: forces by differentiating through each element's own
    geometry, assembled by index_add."""

    def __init__(self, pb, dev):
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.pb, self.dev, self.t = pb, dev, t
        self.nd, self.npoin = pb.ndof, pb.npoin
        self.ib = torch.as_tensor(np.ascontiguousarray(pb.ibool).astype(np.int64) - 1, device=dev)  # [e][j][i]
        self.H = t(pb.hprime)  # [a][i] = h'_a(x_i)
        w = t(pb.wgll)
        x = t(pb.coord)[self.ib]  # [e][j][i][2]
        xi, eta = self._grad(x.permute(3, 0, 1, 2))
        J11, J21 = xi[0], xi[1]
        J12, J22 = eta[0], eta[1]
        det = J11 * J22 - J12 * J21
        self.xx, self.ex = J22 / det, -J21 / det  # dxi/dx, deta/dx
        self.xz, self.ez = -J12 / det, J11 / det  # dxi/dz, deta/dz
        self.wJ = w[None, :, None] * w[None, None, :] * det
        self.lam, self.mu = t(pb.lam), t(pb.mu)
        self.M = t(pb.mass_raw)
        self.leap = pb.scheme == "leapfrog"
        self.c3 = pb.dt if self.leap else 0.5 * pb.dt
        cm = 0.5 * pb.dt
        self.C = torch.zeros((self.nd, self.npoin), dtype=torch.float64, device=dev)
        self.skew = []  # boundaries at an angle: coefficients along and across the normal, normals
        Mt = self.M.clone()
        for ab in pb.abso:
            k = torch.as_tensor(ab["node"].astype(np.int64) - 1, device=dev)
            if ab.get("normals") is not None:
                self.skew.append((k, t(ab["C"].T), t(ab["normals"].T)))
                continue
            self.C[:, k] += t(ab["C"].T)
            Mt[:, k] += cm * t(ab["C"].T)
        self.rm = 1.0 / Mt
        self.kv = t(pb.kv_eta) if pb.kv_eta is not None else None
        self.src = [(int(q["iglob"]) - 1, t(q["dir"]) if self.nd == 2 else t([1.0]), np.asarray(q["stf_table"]))
                    for q in pb.sources]  # an antiplane force has no angle

    def _grad(self, U):
        return torch.einsum("ai,ceja->ceji", self.H, U), torch.einsum("aj,ceai->ceji", self.H, U)

    def force(self, d, v=None, lam=None, mu=None):
        lam, mu = (self.lam if lam is None else lam), (self.mu if mu is None else mu)
        U = d[:, self.ib]
        if self.kv is not None:
            U = U + self.kv * v[:, self.ib]
        gx, ge = self._grad(U)
        dx = gx * self.xx + ge * self.ex
        dz = gx * self.xz + ge * self.ez
        if self.nd == 2:
            sxx = (lam + 2 * mu) * dx[0] + lam * dz[1]
            szz = lam * dx[0] + (lam + 2 * mu) * dz[1]
            sxz = mu * (dz[0] + dx[1])
            S = torch.stack([sxx, sxz]), torch.stack([sxz, szz])
        else:
            S = mu * dx, mu * dz
        t1 = self.wJ * (S[0] * self.xx + S[1] * self.xz)
        t2 = self.wJ * (S[0] * self.ex + S[1] * self.ez)
        f = -(torch.einsum("ai,ceji->ceja", self.H, t1) + torch.einsum("bj,ceji->cebi", self.H, t2))
        return torch.zeros_like(d).index_add(1, self.ib.reshape(-1), f.reshape(self.nd, -1))

    def source(self, f, it):
        for g, dirv, tab in self.src:
            if it <= len(tab):
                f[:, g] += dirv * float(tab[it - 1])

    def step(self, d, v, a, it, fault=None):
        dt = self.pb.dt
        if self.leap:
            d = d + dt * v
        else:
            d = d + dt * v + 0.5 * dt * dt * a
            v = v + 0.5 * dt * a
        f = self.force(d, v)
        self.source(f, it)
        f = f - self.C * v
        for k, C, n in self.skew:
            vn = (v[:, k] * n).sum(0) * n
            f[:, k] -= C[0] * vn + C[1] * (v[:, k] - vn)
        if fault is not None:
            fault.apply(d, v, f)
        a = f * self.rm
        return d, v + self.c3 * a, a


class _SlipWeakening:
    """Linear slip weakening on node pairs (beta = 0), in the fault's frame."""

    def __init__(self, X):
        f, t, dev = X.pb.fault, X.t, X.dev
        self.nd = X.nd
        self.n1, self.n2 = (torch.as_tensor(f[k].astype(np.int64) - 1, device=dev) for k in ("node1", "node2"))
        self.n = t(f["n1"].T)
        self.B, self.i1, self.i2, self.Z = (t(f[k].T) for k in ("B", "invM1", "invM2", "Z"))
        self.T0 = t(f["T0"].T)
        self.coh, self.dc, self.mus, self.mud = (t(f[k]) for k in ("cohesion", "dc", "mus", "mud"))
        self.a2v, self.out = f["coefA2V"], None

    def _rot(self, x):
        return torch.stack([self.n[1] * x[0] - self.n[0] * x[1], self.n[0] * x[0] + self.n[1] * x[1]])

    def apply(self, d, v, f):
        dD, dV = d[:, self.n2] - d[:, self.n1], v[:, self.n2] - v[:, self.n1]
        dA = self.i2 * f[:, self.n2] - self.i1 * f[:, self.n1]
        T = self.Z * (dV + self.a2v * dA)
        if self.nd == 2:
            dD, dV, dA, T = (self._rot(x) for x in (dD, dV, dA, T))
        else:
            T = torch.cat([T, torch.zeros_like(T)])
        T = T + self.T0
        T[1] = torch.clamp(T[1], max=0.0)
        stick = T - self.T0
        th = dD[0].abs()
        mu = self.mus - (self.mus - self.mud) * torch.clamp(th / self.dc, max=1.0)
        T0 = torch.copysign(torch.minimum(T[0].abs(), self.coh - mu * T[1]), T[0])
        T = torch.stack([T0, T[1]]) - self.T0
        Tx = torch.stack([self.n[1] * T[0] + self.n[0] * T[1], -self.n[0] * T[0] + self.n[1] * T[1]]) \
            if self.nd == 2 else T[:1]
        f[:, self.n1] += self.B * Tx
        f[:, self.n2] -= self.B * Tx
        V = dV + self.a2v * (dA - T[:self.nd] / (self.Z * self.a2v))
        self.out = dict(D=dD, V=V, T=T, MU=mu, Tstick=stick)


def _exact_gradient(X, c, obs):
    """Reverse mode through the steps, in segments: per element lambda and mu, the mass and
    the absorbing coefficients (their share of the modified mass included) as leaves."""
    pb, n, dt = X.pb, c["steps"], X.pb.dt
    rec = torch.as_tensor(pb.receivers["iglob"].astype(np.int64) - 1, device=X.dev)
    leaf = [torch.zeros(pb.nelem, dtype=torch.float64, device=X.dev, requires_grad=True) for _ in range(2)]
    M = X.M[0].clone().requires_grad_()
    C = X.C.clone().requires_grad_()

    def advance(d, v, a, it):
        d = d + dt * v + 0.5 * dt * dt * a
        v = v + 0.5 * dt * a
        f = X.force(d, None, X.lam + leaf[0][:, None, None], X.mu + leaf[1][:, None, None])
        X.source(f, it)
        a = (f - C * v) / (M + 0.5 * dt * C)
        return d, v + 0.5 * dt * a, a

    seg = max(1, int(math.ceil(math.sqrt(n))))
    z = torch.zeros((2, pb.npoin), dtype=torch.float64, device=X.dev)
    st, keep, seis = (z, z, z), [], [torch.zeros(2, len(rec), dtype=torch.float64, device=X.dev)]
    with torch.no_grad():
        for it in range(1, n + 1):
            if (it - 1) % seg == 0:
                keep.append(st)
            st = advance(*st, it)
            seis.append(st[1][:, rec])
    seis = torch.stack(seis)
    res = seis - X.t(obs)
    leaves = leaf + [M, C]
    g = [torch.zeros_like(x) for x in leaves]
    adj = (z, z, z)
    for k in reversed(range(len(keep))):
        s0 = [x.detach().requires_grad_() for x in keep[k]]
        st, J = tuple(s0), 0.0
        for it in range(k * seg + 1, min(n, (k + 1) * seg) + 1):
            st = advance(*st, it)
            J = J + (st[1][:, rec] * res[it]).sum()
        J = J + sum((x * y).sum() for x, y in zip(st, adj))
        got = torch.autograd.grad(J, s0 + leaves, allow_unused=True)
        adj = tuple(x if x is not None else z for x in got[:3])
        g = [x + y for x, y in zip(g, got[3:])]
    on = X.C != 0
    return dict(seis=seis, lam=g[0], mu=g[1], mass=g[2], abso=torch.where(on.any(0)[None], g[3], torch.zeros_like(g[3])))


def exact(c, seed):
    """None for the ensemble: its rate-and-state solve stops at a tolerance of its own,
    so that its outputs have no value independent of the iteration."""
    if c["kind"] == "ensemble":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if c["kind"] == "gradient":
        pb, obs = _gradient_problem(c, seed)
        return {k: x.cpu().numpy() for k, x in _exact_gradient(_Exact(pb, dev), c, obs).items()}
    d = v = None
    if c["kind"] == "loop":
        pb, d, v = _loop_problem(c, seed)
    else:
        pb = _problem(c, seed)
    X = _Exact(pb, dev)
    d, v = (torch.zeros((X.nd, X.npoin), dtype=torch.float64, device=dev) if q is None else X.t(q) for q in (d, v))
    a = torch.zeros_like(d)
    fault = _SlipWeakening(X) if pb.fault is not None else None
    rec = None
    if pb.receivers is not None:
        rec = torch.as_tensor(pb.receivers["iglob"].astype(np.int64) - 1, device=dev)
        seis = [torch.zeros((X.nd, len(rec)), dtype=torch.float64, device=dev)]  # taken before the fields are set
    for it in range(1, c["steps"] + 1):
        d, v, a = X.step(d, v, a, it, fault)
        if rec is not None:
            seis.append(v[:, rec])
    if c["kind"] == "rupture":
        return {k: x.cpu().numpy() for k, x in fault.out.items()}
    out = dict(seis=torch.stack(seis))
    if c["kind"] == "run":
        out.update(d=d, v=v, a=a)
    return {k: x.cpu().numpy() for k, x in out.items()}
