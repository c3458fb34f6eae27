// Dynamic fault boundary: pointwise traction solve on split-node pairs.
// asinh, sinh and cosh follow the C library's decomposition (sem2d_libm.hpp).
//
// One lane per fault node pair.  All fault arithmetic is FP64 whatever the bulk type.  The
// pragmas below keep the front end from contracting products into sums; the backend, built
// with -ffp-contract=fast, still does where a product's only use is a sum, so where a bit
// matters the rounding is written out (fault_solve).
//   BC_DYNFLT_apply      SRC/bc_dynflt.f90:569-739
//   slip weakening       SRC/bc_dynflt_swf.f90:142-194
//   rate and state       SRC/bc_dynflt_rsf.f90:165-568 (two-pass rsf_solver,
//                        aging/slip/V-shape state updates, safeguarded
//                        Newton-bisection nr_solver returning the slip rate of
//                        its last function evaluation)
//   Coulomb normal law   SRC/bc_dynflt_normal.f90:118-136 (kind 1)
#pragma once
#include <hip/hip_runtime.h>

#include "sem2d_kernels.hpp"
#include "sem2d_libm.hpp"

namespace sem2d {

struct FaultDev {
  int np, ndof;
  const int *n1, *n2;                    // 0-based node pairs; n2[k] = -1 on a fault with one
                                         // side (on a domain boundary, SRC/bc_dynflt.f90:256-259)
  const double *nrm;                     // [2][np]
  const double *B, *invM1, *invM2, *Z;   // [ndof][np]
  const double *T0;                      // [2][np]
  const double *coh;                     // [np]
  double a2v, a2d, dt;
  int opening, law, kind, healing;
  const double *p0, *p1, *p2, *p3, *p4, *p5;  // friction parameters [np]
  const double *Tc, *coeft;              // RSF kind 1 helpers
  double *theta;                         // [np] state
  double *D, *V;                         // [ndof][np]
  double *T, *Tstick;                    // [2][np]
  double *MU, *sigma;                    // [np]
  int *nr_fail;                          // Newton iteration overflow flag
  // structured grids: Dirichlet components of the Dirichlet boundaries that act after
  // the fault, zeroed in the force of node 1 (bits 0-1) and node 2 (bits 2-3) before the
  // corrector (null: none)
  const unsigned char* dmask = nullptr;
  // structured grids: d and v after the step at both nodes of every pair, bulk type,
  // [d, v][node 1, node 2][ndof][np] (the field arrays hold the next step's predicted
  // values); the pairs' nodes in the deferred-node list (def2: -1 on one side)
  void* side = nullptr;
  const int *def1 = nullptr, *def2 = nullptr;
  // time-weakening friction (BC_DYNFLT_TWF): kind (0: none; law 3: time weakening alone),
  // parameters MuS, MuD, Mu0, X, Z, V, L, T, Dc and the fault node coordinates [2][np]
  int twf = 0;
  double tw[9] = {};
  const double* xz = nullptr;
  // normal stress response (BC_DYNFLT_NOR): 0 cohesion (sigma stays the initial normal
  // stress), 1 Coulomb, 2 Prakash-Clifton with time scale (nor_coef = exp(-dt/T)), 3 with
  // length scale (nor_coef = dt/L, nor_v = V)
  int nor_kind = 1;
  double nor_coef = 0.0, nor_v = 0.0;
};

// normal_update (SRC/bc_dynflt_normal.f90:122-140): the normal stress the friction law
// sees, from the previous one, the trial normal traction tn and the trial slip rate dv
__host__ __device__ inline double normal_sigma(int kind, double coef, double vc, double sig_old, double tn,
                                               double dv) {
  switch (kind) {
    case 0: return sig_old;
    case 2: return tn + coef * (sig_old - tn);
    case 3: return tn + exp(-(fabs(dv) + vc) * coef) * (sig_old - tn);
    default: return tn;
  }
}

// What the traction solve of a pair reads, loaded in one group: with the loads where the
// values are used, each behind the stores of the state before it (which may alias), a step
// waited for memory about ten times one after the other (600 x 300 SH elements, FP64: the
// launch after the tile kernel 13.9 us, with the pair's and the nodes' values in groups 9.4 us).
struct PairData {
  double B[2], iM1[2], iM2[2], Z[2], nx, nz, T0[2], sigma;
  double theta = 0, D = 0, V = 0, coh = 0, p0 = 0, p1 = 0, p2 = 0, p3 = 0, p4 = 0, p5 = 0, Tc = 0, coeft = 0;
};
template <int nd>
__device__ __forceinline__ PairData pair_load(const FaultDev& F, int k, bool two) {
  PairData P;
  const int np = F.np;
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    P.B[c] = F.B[c * np + k];
    P.iM1[c] = F.invM1[c * np + k];
    P.iM2[c] = two ? F.invM2[c * np + k] : 0.0;
    P.Z[c] = F.Z[c * np + k];
  }
  P.nx = F.nrm[k], P.nz = F.nrm[np + k];
  P.T0[0] = F.T0[k], P.T0[1] = F.T0[np + k];
  P.sigma = F.sigma[k];
  P.D = F.D[k];
  if (F.law != 2) P.coh = F.coh[k];
  if (F.law != 3) {
    P.theta = F.theta[k];
    P.p0 = F.p0[k], P.p1 = F.p1[k], P.p2 = F.p2[k], P.p3 = F.p3[k];
    if (F.law == 2 || F.kind > 2) P.p4 = F.p4[k];
  }
  if (F.law == 2) {
    P.V = F.V[k];
    if (F.kind == 4) P.p5 = F.p5[k];
    if (F.kind == 1) P.Tc = F.Tc[k], P.coeft = F.coeft[k];
  }
  return P;
}

// the pair's state after the step, and what its tractions add to the force of node 1 and take
// from that of node 2
struct PairOut {
  double D0, V0, T[2], Ts0, mu, bt[2];
};

#pragma clang fp contract(off)

__device__ inline double f_swf_mu(const FaultDev& F, const PairData& P, double th) {
  const double dc = P.p0, mus = P.p1, mud = P.p2;
  double mu;
  if (F.kind == 1) mu = mus - (mus - mud) * fmin(th / dc, 1.0);
  else if (F.kind == 2) mu = mud - (mud - mus) * exp(-th / dc);
  else mu = mud + (mus - mud) / pow(1.0 + th / dc, P.p4);
  return mu + P.p3 * th;
}

// twf_mu (SRC/bc_dynflt_twf.f90:129-183) of kind 1..3 with tw = MuS, MuD, Mu0, X, Z, V, L,
// T, Dc at point (x, z), time t, slip d; kind 3 leaves the points beyond V*T unset in the
// reference: they get huge(1d0) here (no weakening).  Host and device.
__host__ __device__ inline double twf_mu(int kind, const double* tw, double x, double z, double time, double d) {
  const double mus = tw[0], mud = tw[1], mu0 = tw[2], X = tw[3], Z = tw[4];
  const double V = tw[5], L = tw[6], T = tw[7], Dc = tw[8];
  const double big = 1.7976931348623157e308;
  const double dx = x - X, dz = z - Z;
  const double dist = sqrt(dx * dx + dz * dz);
  if (kind == 1 || kind == 2) {
    double t, r;
    if (kind == 1) {
      t = time + (mus - mu0) * L / ((mus - mud) * V);
      if (t > T) t = 0.0;
      r = V * t;
    } else {
      t = time + 0.5 * T * (1.0 - sqrt(1.0 - 4.0 * (mus - mu0) * L / ((mus - mud) * T * V)));
      t = fmin(t, T);
      r = V * t * (1.0 - t / T);
    }
    r = dist - r;
    if (r < -L) return mud;
    if (r <= L) return mus + (mus - mud) / L * r;
    return big;
  }
  if (dist <= V * T && d <= Dc) {
    if (dist < V * time - L) return mud;
    if (dist >= V * time - L && dist <= V * time) return mus + (mus - mud) / L * (dist - V * time);
  }
  return big;
}

__device__ inline double f_twf_mu(const FaultDev& F, int k, double time, double d) {
  return twf_mu(F.twf, F.tw, F.xz[k], F.xz[F.np + k], time, d);
}

__device__ inline double f_rsf_mu(const FaultDev& F, const PairData& P, double th, double v) {
  const double dc = P.p0, mus = P.p1, a = P.p2, b = P.p3, vs = P.p4;
  switch (F.kind) {
    case 1: return mus + a * fabs(v) / (fabs(v) + vs) - b * th / (th + dc);
    case 2:
    case 3: return a * libm::asinh(fabs(v) / (2.0 * vs) * exp((mus + b * log(vs * th / dc)) / a));
    default: return a * libm::asinh(fabs(v) / (2.0 * vs) * exp((mus + b * log(P.p5 * th / dc + 1)) / a));
  }
}

__device__ inline double f_rsf_theta(const FaultDev& F, const PairData& P, double theta, double v) {
  const double dc = P.p0, dt = F.dt;
  switch (F.kind) {
    case 1: {
      double tn = theta * P.coeft + P.Tc * fabs(v) * (1.0 - P.coeft);
      return tn < 1.0e-12 ? 0.0 : tn;
    }
    case 2:
    case 4: {
      const double x = fabs(v) / dc;
      const double ex = exp(-dt * x);
      if (dt * x > 1e-8) return theta * ex + (1.0 - ex) / x;
      return theta * ex + dt * (1.0 - 0.5 * dt * x);
    }
    default: {
      const double tn = dc / fabs(v);
      return tn * pow(theta / tn, exp(-dt / tn));
    }
  }
}

__device__ inline void f_fric(const FaultDev& F, const PairData& P, double theta, double tau, double tstick,
                              double sigma, double Z, double& fv, double& dfv, double& v) {
  const double dc = P.p0, mus = P.p1, a = P.p2, b = P.p3, vs = P.p4;
  double tmp = (F.kind == 4) ? mus + b * log(P.p5 * theta / dc + 1.0) : mus + b * log(vs * theta / dc);
  tmp = 2.0 * vs * exp(-tmp / a);
  v = libm::sinh(tau / (-sigma * a)) * tmp;
  fv = tstick - Z * v - tau;
  const double dv = libm::cosh(tau / (-sigma * a)) * tmp / (-sigma * a);
  dfv = -Z * dv - 1.0;
}

__device__ inline double f_nr_solver(const FaultDev& F, const PairData& P, double xL, double xR, double xacc,
                                     double theta, double tstick, double sigma, double Z, bool& ok) {
  double flow, fhigh, dfdx, v, xlow, xhigh, dx, dxold, fx;
  ok = true;
  f_fric(F, P, theta, xL, tstick, sigma, Z, flow, dfdx, v);
  f_fric(F, P, theta, xR, tstick, sigma, Z, fhigh, dfdx, v);
  double xl = xL, xr = xR;
  int guard = 0;
  while (flow * fhigh > 0 && guard++ < 2100) {
    xl = xl / 2.0;
    xr = xr * 2.0;
    f_fric(F, P, theta, xl, tstick, sigma, Z, flow, dfdx, v);
    f_fric(F, P, theta, xr, tstick, sigma, Z, fhigh, dfdx, v);
  }
  if (flow * fhigh > 0) { ok = false; return v; }
  if (flow == 0) return v;
  if (fhigh == 0) return v;
  if (flow < 0) { xlow = xl; xhigh = xr; } else { xhigh = xl; xlow = xr; }
  double xest = 0.5 * (xl + xr);
  dxold = fabs(xr - xl);
  dx = dxold;
  f_fric(F, P, theta, xest, tstick, sigma, Z, fx, dfdx, v);
  for (int is = 1; is <= 200; ++is) {
    if (((xest - xhigh) * dfdx - fx) * ((xest - xlow) * dfdx - fx) > 0 ||
        fabs(2 * fx) > fabs(dxold * dfdx)) {
      dxold = dx;
      dx = 0.5 * (xhigh - xlow);
      xest = xlow + dx;
      if (xlow == xest) return v;
    } else {
      dxold = dx;
      dx = fx / dfdx;
      const double tmp = xest;
      xest = xest - dx;
      if (tmp == xest) return v;
    }
    if (fabs(dx) < fabs(xacc)) {
      f_fric(F, P, theta, xest, tstick, sigma, Z, fx, dfdx, v);
      return v;
    }
    f_fric(F, P, theta, xest, tstick, sigma, Z, fx, dfdx, v);
    if (fx < 0) xlow = xest; else xhigh = xest;
  }
  ok = false;
  return v;
}

__device__ inline double f_rsf_v(const FaultDev& F, const PairData& P, double tstick, double sigma, double theta,
                                 double Z, bool& ok) {
  ok = true;
  if (F.kind == 1) {
    const double dc = P.p0, mus = P.p1, a = P.p2, b = P.p3, vs = P.p4;
    // rsf_mu_no_direct reads the stored state (the state before this step), not the
    // updated estimate: SRC/bc_dynflt_rsf.f90:189-196,338
    const double th0 = P.theta;
    const double mnd = mus - b * th0 / (th0 + dc);
    double v = (tstick + sigma * mnd) / Z;
    const double tmp = v - vs + sigma * a / Z;
    v = 0.5 * (tmp + sqrt(tmp * tmp + 4.0 * v * vs));
    v = fmax(0.0, v);
    return v < 1.0e-12 ? 0.0 : v;
  }
  const double tol = -0.001 * P.p2 * sigma;
  return f_nr_solver(F, P, fmin(0.0, tstick), fmax(0.0, tstick), tol, theta, tstick, sigma, Z, ok);
}

// One node component by component: the predicted displacement and velocity and the force.
template <typename R>
struct NodeState {
  R d[2] = {0, 0}, v[2] = {0, 0}, f[2] = {0, 0};
};

// Traction solve of pair k from the states of its nodes (n2 unused when two is false: a
// fault with one side); the fault state of the pair is updated and its tractions added to
// the nodes' forces.  time = it*dt of the step (SRC/main.f90:53), read by time-weakening
// friction only.
template <typename R, int nd>
__device__ inline PairOut fault_solve(const FaultDev& F, const PairData& P, int k, double time, bool two,
                                      NodeState<R>& n1, NodeState<R>& n2) {
  const int np = F.np;
  double dD[2] = {0, 0}, dV[2] = {0, 0}, dA[2] = {0, 0}, T[2] = {0, 0}, Ts[2];
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    if (two) {
      dD[c] = (double)n2.d[c] - (double)n1.d[c];
      dV[c] = (double)n2.v[c] - (double)n1.v[c];
      dA[c] = P.iM2[c] * (double)n2.f[c] - P.iM1[c] * (double)n1.f[c];
    } else {  // one side: get_jump, get_weighted_jump (SRC/bc_dynflt.f90:692-719)
      dD[c] = -2.0 * (double)n1.d[c];
      dV[c] = -2.0 * (double)n1.v[c];
      dA[c] = -2.0 * P.iM1[c] * (double)n1.f[c];
    }
    T[c] = P.Z[c] * (dV[c] + F.a2v * dA[c]);
    // rounded here: without the rotation (SH) the product would be fused with the addition of
    // the initial stress
    if (nd == 1) asm volatile("" : "+v"(T[c]));
  }
  const double nx = P.nx, nz = P.nz;
  if (nd == 2) {
    double r0, r1;
    r0 = nz * dD[0] - nx * dD[1]; r1 = nx * dD[0] + nz * dD[1]; dD[0] = r0; dD[1] = r1;
    r0 = nz * dV[0] - nx * dV[1]; r1 = nx * dV[0] + nz * dV[1]; dV[0] = r0; dV[1] = r1;
    r0 = nz * dA[0] - nx * dA[1]; r1 = nx * dA[0] + nz * dA[1]; dA[0] = r0; dA[1] = r1;
    r0 = nz * T[0] - nx * T[1];   r1 = nx * T[0] + nz * T[1];   T[0] = r0;  T[1] = r1;
  }
  if (nd == 1 || !two) T[1] = 0.0;  // SRC/bc_dynflt.f90:604
  T[0] = T[0] + P.T0[0];
  T[1] = T[1] + P.T0[1];
  if (F.opening) T[1] = fmin(T[1], 0.0);
  const double sigma = normal_sigma(F.nor_kind, F.nor_coef, F.nor_v, P.sigma, T[1], dV[0]);
  Ts[0] = T[0];
  Ts[1] = T[1];
  double th = P.theta, mu;  // friction state and coefficient
  if (F.law == 2) {
    const double vold = P.V, Z1 = P.Z[0];
    bool ok1, ok2;
    th = f_rsf_theta(F, P, P.theta, vold);
    double vst = f_rsf_v(F, P, T[0], sigma, th, Z1, ok1);
    th = f_rsf_theta(F, P, P.theta, 0.5 * (vold + vst));
    vst = f_rsf_v(F, P, T[0], sigma, th, Z1, ok2);
    if (!(ok1 && ok2)) atomicOr(F.nr_fail, 1);
    mu = f_rsf_mu(F, P, th, vst);
    // superimposed time weakening (SRC/bc_dynflt.f90:632)
    if (F.twf) mu = fmin(mu, f_twf_mu(F, k, time, P.D));
    const double strength = -mu * sigma;
    T[0] = copysign(fabs(strength), T[0]);
  } else if (F.law == 3) {  // time weakening alone (SRC/bc_dynflt.f90:656-657)
    mu = f_twf_mu(F, k, time, P.D);
    const double strength = P.coh - mu * sigma;
    T[0] = copysign(fmin(fabs(T[0]), strength), T[0]);
  } else {
    if (F.a2d == 0.0) {
      if (F.healing) {
        th = P.theta + fabs(dV[0]) * F.dt;
        if (fabs(dV[0]) < 1e-14) th = 0.0;
      } else {
        th = fabs(dD[0]);
      }
    } else {
      th = fabs(P.D);
    }
    mu = f_swf_mu(F, P, th);
    if (F.twf) mu = fmin(mu, f_twf_mu(F, k, time, P.D));  // :653
    const double strength = P.coh - mu * sigma;
    T[0] = copysign(fmin(fabs(T[0]), strength), T[0]);
  }
  T[0] = T[0] - P.T0[0];
  T[1] = T[1] - P.T0[1];
  Ts[0] = Ts[0] - P.T0[0];
  Ts[1] = Ts[1] - P.T0[1];
  double Tx[2] = {T[0], T[1]};
  if (nd == 2) {
    Tx[0] = nz * T[0] + nx * T[1];
    Tx[1] = -nx * T[0] + nz * T[1];
  }
  PairOut out;
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    // one rounding at node 1, two at node 2, however the compiler arranges the code around:
    // with FP32 fields a bit here grows to 1e-5 of a rupture's tractions in a hundred steps
    double bt = P.B[c] * Tx[c];
    asm volatile("" : "+v"(bt));
    n1.f[c] = (R)__builtin_fma(P.B[c], Tx[c], (double)n1.f[c]);
    if (two) n2.f[c] = (R)((double)n2.f[c] - bt);
    out.bt[c] = bt;
  }
  F.sigma[k] = sigma;
  if (F.law != 3) F.theta[k] = th;
  F.MU[k] = mu;
  F.T[k] = T[0];
  F.T[np + k] = T[1];
  F.Tstick[k] = Ts[0];
  F.Tstick[np + k] = Ts[1];
  out.T[0] = T[0], out.T[1] = T[1], out.Ts0 = Ts[0], out.mu = mu;
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    const double tf = T[c];
    const double da = dA[c] - tf / (P.Z[c] * F.a2v);
    const double D = dD[c] + F.a2d * da, V = dV[c] + F.a2v * da;
    F.D[c * np + k] = D;
    F.V[c * np + k] = V;
    if (c == 0) out.D0 = D, out.V0 = V;
  }
  return out;
}

// Fault of the general path: the pair's forces updated in place; every node is corrected
// afterwards.  Launched with 64 lanes per workgroup: the Newton iteration's registers are
// then not capped by the 1024-lane default (which spilled them to scratch).
template <typename R, int nd>
__global__ __launch_bounds__(64) void k_fault(FaultDev F, const R* d, const R* v, R* f, int npoin, double time) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= F.np) return;
  const int i1 = F.n1[k], i2 = F.n2[k];
  NodeState<R> n1, n2;
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    const size_t o = (size_t)c * npoin;
    n1.d[c] = d[o + i1];
    n1.v[c] = v[o + i1];
    n1.f[c] = f[o + i1];
    if (i2 >= 0) {
      n2.d[c] = d[o + i2];
      n2.v[c] = v[o + i2];
      n2.f[c] = f[o + i2];
    }
  }
  const PairOut po = fault_solve<R, nd>(F, pair_load<nd>(F, k, i2 >= 0), k, time, i2 >= 0, n1, n2);
#pragma unroll
  for (int c = 0; c < nd; ++c) {
    const size_t o = (size_t)c * npoin;
    f[o + i1] = n1.f[c];
    // a pair whose two sides are one node: both act on it
    if (i2 >= 0) f[o + i2] = i2 == i1 ? (R)((double)n1.f[c] - po.bt[c]) : n2.f[c];
  }
}

// fault record: out[6][nout] from the current state (SRC/bc_dynflt.f90:762-767)
__global__ void k_fault_record(FaultDev F, int oix1, int oixd, int nout, double* __restrict__ out) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= nout) return;
  const int k = oix1 - 1 + o * oixd;
  out[0 * nout + o] = F.D[k];
  out[1 * nout + o] = F.V[k];
  out[2 * nout + o] = F.T[k];
  out[3 * nout + o] = F.T[F.np + k];
  out[4 * nout + o] = F.MU[k];
  out[5 * nout + o] = F.Tstick[k];
}

// Per-side fault record (osides = T; export_side of get_side, SRC/bc_dynflt.f90:769-812):
// out[4*ndof][nout], rows d of side 1, d of side 2, v of side 1, v of side 2, each in
// the fault frame (t, n) for P-SV (rotate, SRC/bc_dynflt.f90:722-739); side 2 of a
// fault with one side is -(side 1).  FP64, no contraction, like the fault solve.
#pragma clang fp contract(off)
// side: from F.side instead of the fields.
template <typename R>
__global__ void k_fault_sides(FaultDev F, const R* __restrict__ d, const R* __restrict__ v, size_t stride,
                              int oix1, int oixd, int nout, double* __restrict__ out, int side_arrays) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= nout) return;
  const int k = oix1 - 1 + o * oixd;
  const int i1 = F.n1[k], i2 = F.n2[k];
  const int nd = F.ndof;
  int row = 0;
  for (int w = 0; w < 2; ++w)
    for (int side = 1; side <= 2; ++side) {
      const R* u = w == 0 ? d : v;
      double x[2] = {0.0, 0.0};
      for (int c = 0; c < nd; ++c) {
        if (side_arrays) {
          const R* sc = (const R*)F.side + ((size_t)(w * 2) * nd + c) * F.np + k;
          x[c] = side == 1 ? (double)sc[0] : (i2 >= 0 ? (double)sc[(size_t)nd * F.np] : -(double)sc[0]);
          continue;
        }
        const R* uc = u + (size_t)c * stride;
        x[c] = side == 1 ? (double)uc[i1] : (i2 >= 0 ? (double)uc[i2] : -(double)uc[i1]);
      }
      if (nd == 1) {
        out[(size_t)row * nout + o] = x[0];
      } else {
        const double n1x = F.nrm[k], n1z = F.nrm[F.np + k];
        out[(size_t)row * nout + o] = n1z * x[0] - n1x * x[1];
        out[(size_t)(row + 1) * nout + o] = n1x * x[0] + n1z * x[1];
      }
      row += nd;
    }
}
#pragma clang fp contract(on)

// Potency of the displacement and velocity jumps (BC_DYNFLT_potency,
// SRC/bc_dynflt.f90:832-855): P-SV p11, p22, p12 of d then of v, SH p13, p23 of d
// then of v, one row of 2*(ndof+1) values, over the fault pairs k0 .. k0+n-1.  One
// workgroup of 256 lanes: lane t sums pairs k0+t, k0+t+256, ..., then a fixed-shape
// tree, so the result is run-to-run identical.  The general path's rows and the row of
// step 0; the steps of a structured grid make theirs in potency_wave.
template <typename R>
__device__ __forceinline__ void potency_row(const FaultDev& F, int k0, int n, const R* __restrict__ d,
                                            const R* __restrict__ v, size_t stride, double* __restrict__ out,
                                            double (*red)[256]) {
  const int t = threadIdx.x, np = F.np;
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (int kl = t; kl < n; kl += 256) {
    const int k = k0 + kl;
    const int i1 = F.n1[k], i2 = F.n2[k];
    const double nx = F.nrm[k], nz = F.nrm[np + k], b = F.B[k];
    // get_jump (SRC/bc_dynflt.f90:692-704): x2 - x1, or -2 x1 on a one-sided fault
    auto jump = [&](int w, int c) {
      const R* x = (w == 0 ? d : v) + (size_t)c * stride;
      return i2 >= 0 ? (double)x[i2] - (double)x[i1] : -2.0 * (double)x[i1];
    };
    const double jd0 = jump(0, 0), jv0 = jump(1, 0);
    if (F.ndof == 2) {
      const double jd1 = jump(0, 1);
      const double jv1 = jump(1, 1);
      s[0] += nx * jd0 * b;
      s[1] += nz * jd1 * b;
      s[2] += (nx * jd1 + nz * jd0) * b;
      s[3] += nx * jv0 * b;
      s[4] += nz * jv1 * b;
      s[5] += (nx * jv1 + nz * jv0) * b;
    } else {
      s[0] += nx * jd0 * b;
      s[1] += nz * jd0 * b;
      s[2] += nx * jv0 * b;
      s[3] += nz * jv0 * b;
    }
  }
  for (int q = 0; q < 6; ++q) red[q][t] = s[q];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (t < w)
      for (int q = 0; q < 6; ++q) red[q][t] = red[q][t] + red[q][t + w];
    __syncthreads();
  }
  if (t == 0) {
    if (F.ndof == 2) {
      out[0] = red[0][0];
      out[1] = red[1][0];
      out[2] = 0.5 * red[2][0];
      out[3] = red[3][0];
      out[4] = red[4][0];
      out[5] = 0.5 * red[5][0];
    } else {
      out[0] = 0.5 * red[0][0];
      out[1] = 0.5 * red[1][0];
      out[2] = 0.5 * red[2][0];
      out[3] = 0.5 * red[3][0];
    }
  }
}

template <typename R>
__global__ __launch_bounds__(256) void k_fault_potency(FaultDev F, const R* __restrict__ d, const R* __restrict__ v,
                                                       size_t stride, double* __restrict__ out) {
  __shared__ double red[6][256];
  potency_row<R>(F, 0, F.np, d, v, stride, out, red);
}

// Per-step outputs of a fault on a structured grid, made where its pairs are finished.
// A wavefront takes wave[w] = (first pair, pairs, member, -): 64 pairs of one member at
// most, the member's wavefronts being member[m].x .. + member[m].y - 1 (a fault alone is
// member 0).
struct FaultOut {
  int nwave = 0;
  const int4* wave = nullptr;
  const int2* member = nullptr;
  // potency rows pot[member][pot_cap][2*(ndof+1)]: the row of this step is pot_row, or
  // pot_row + the device step counter; part [nwave][6] and cnt [members] are scratch (cnt
  // zero between launches)
  double *pot = nullptr, *part = nullptr;
  unsigned* cnt = nullptr;
  int pot_cap = 0, pot_row = 0;
  // fault records rec[sample][6][nout]: slot[k] is the output place of pair k or -1; the
  // sample is rec_slot (-1: none), or, with the device step counter, that of the steps
  // oit0, oit0 + oitd, ...
  const int* slot = nullptr;
  double* rec = nullptr;
  int nout = 0, rec_slot = -1, oit0 = 0, oitd = 1, nsamp = 0;
};

// Potency of one step from the jumps of a wavefront's pairs (dj, vj: the displacement and
// velocity jumps of this lane's pair, on: it has one): the wavefront's sums by a tree over
// its lanes, then, by the last wavefront of the member, the sums of its wavefronts in a
// fixed order.  The result does not depend on which wavefront is last and is the same for
// a fault alone and inside a batch.  (One workgroup over all pairs took 12 us of a 79 us
// step, 600 x 300 elements; this adds 1-2 us to the fault's.)
template <int nd>
__device__ inline void potency_wave(const PairData& P, const FaultOut& O, int w, int m, int2 mw, bool on,
                                    const double* dj, const double* vj, int row) {
  const int lane = threadIdx.x & 63;
  double s[6] = {0, 0, 0, 0, 0, 0};
  if (on) {
    const double nx = P.nx, nz = P.nz, b = P.B[0];
    if (nd == 2) {
      s[0] = nx * dj[0] * b;
      s[1] = nz * dj[1] * b;
      s[2] = (nx * dj[1] + nz * dj[0]) * b;
      s[3] = nx * vj[0] * b;
      s[4] = nz * vj[1] * b;
      s[5] = (nx * vj[1] + nz * vj[0]) * b;
    } else {
      s[0] = nx * dj[0] * b;
      s[1] = nz * dj[0] * b;
      s[2] = nx * vj[0] * b;
      s[3] = nz * vj[0] * b;
    }
  }
  auto tree = [&]() {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int q = 0; q < 6; ++q) s[q] = s[q] + __shfl_xor(s[q], o);
  };
  tree();
  unsigned before = 0;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 6; ++q)
      __hip_atomic_store(&O.part[(size_t)w * 6 + q], s[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the sums have to be in device memory before the count; they are stored past the L2
    // (agent scope), so waiting for the stores is enough, and the write-back of the whole L2
    // that a release at agent scope makes is not needed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    before = __hip_atomic_fetch_add(&O.cnt[m], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  before = __shfl(before, 0);
  if (before + 1 != (unsigned)mw.y) return;
  asm volatile("" ::: "memory");  // the sums are read (past the L2 too) after the count
#pragma unroll
  for (int q = 0; q < 6; ++q) s[q] = 0;
  for (int u = lane; u < mw.y; u += 64)
#pragma unroll
    for (int q = 0; q < 6; ++q)
      s[q] = s[q] + __hip_atomic_load(&O.part[(size_t)(mw.x + u) * 6 + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  tree();
  if (lane != 0) return;
  __hip_atomic_store(&O.cnt[m], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (row < 0 || row >= O.pot_cap) return;  // the host reserves the rows
  double* out = O.pot + ((size_t)m * O.pot_cap + row) * (2 * (nd + 1));
  if (nd == 2) {
    out[0] = s[0];
    out[1] = s[1];
    out[2] = 0.5 * s[2];
    out[3] = s[3];
    out[4] = s[4];
    out[5] = 0.5 * s[5];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = 0.5 * s[q];
  }
}

#pragma clang fp contract(on)

}  // namespace sem2d
