// Adjoint right-hand side and adjoint boundary conditions on the device.
//
// right_hand_side_adjoint_3d (src/equations/ns_rho_rhou_p.f90:257-536) is the
// continuous adjoint of the Euler part in the variables (rho, rho u, rho v,
// rho w, p / (gamma - 1)).  Along direction d it takes seven compact
// derivatives -- the five adjoint variables qs1..qs5, -u_d qs5 and the
// forward pressure p -- and combines them point-wise with the forward state
// q.  One sweep per direction applies all seven on register-resident blocks.
//
// With A = D qs1, B_m = D qs_{m+2} (m = 0,1,2), E = D qs5, F = D(-u_d qs5),
// P = D p, gdp = gamma p / (rho (gamma - 1)) and
//   S = sum_m u_m B_m + gdp E + qs5 P / rho
// the contributions of direction d (ns_rho_rhou_p.f90:317-372, 407-445,
// 475-514) are
//   r1        += u_d S
//   r_{d+2}   -= A + u_d B_d + S
//   r_{m+2}   -= u_d B_m            (m != d)
//   r5        -= (gamma - 1) (B_d + F) + gamma u_d E
// (the reference spells S out term by term; the sums agree to rounding).
// The sweeps run z, y, x; the x sweep adds the objective gradient g and
// finishes the RK4 stage of time_stepper_adjoint (rk_o4_e.f90:62-105,
// dt -> -dt).
#pragma once

#include <climits>

#include "boundary.hpp"
#include "sweeps.hpp"

namespace cruna {

// In FP64, a product that is about to be added to another product: which of the
// two a compiler fuses into the addition may differ between the kernels that
// this sweep is inlined into (the batched ones give the same bits).
template <typename T>
__device__ __forceinline__ void pin(T (&a)[PPT]) {
  if constexpr (sizeof(T) == 8) materialize(a);
}

// Hand the accumulated variable v on: intermediate sweeps store it; the last
// sweep adds g and applies the RK4 stage update.
template <bool LAST, int RK, typename T, typename IO>
__device__ __forceinline__ void finish(int v, T (&r)[PPT], const IO &io, long N, T *__restrict__ rhs,
                                       const double *__restrict__ gobj, const RkArgs<T> &rk) {
  if constexpr (!LAST) {
    io.st(rhs + v * N, r);
  } else {
    RkIn<RK, T> in;
    if constexpr (RK != RK_YLAST) rk_load<RK, T>(rk, v, io, N, in);
    if (gobj) {
      double gg[PPT];
      io.ld(gobj + v * N, gg);
      io.got(gg);
#pragma unroll
      for (int m = 0; m < PPT; ++m) r[m] = r[m] + T(gg[m]);
    }
    if constexpr (RK == RK_YLAST) {
      double q1[PPT];
      materialize(r);
      rk_ylast(rk, v, r, io, N, q1);
      io.st(rk.qn + v * N, q1);
    } else {
      rk_got<RK, T>(io, in);
      rk_store<RK, T>(rk, v, r, in, io, N, rhs);
    }
  }
}

// One adjoint sweep along DIR.
//   qs   : adjoint stage input (5 fields, type Q)
//   q0p  : device cell holding the forward state of the step (5 fields, FP64),
//          frozen over the stages; the cell lets one recorded launch sequence
//          serve every step of a backward loop (the slot is set on the device)
//   rhs  : 5 accumulator fields (written by the first sweep, z)
//   gobj : objective gradient g (5 fields) or null; added by the x sweep
// The x sweep (LAST) completes the stage: RK4 update RK (RkForm) with step
// rk.dt (negative for the backward integration).
template <typename T, typename Q, int DIR, int RK, typename Lines>
__device__ __forceinline__ void asweep_body(const ThreadPos &tp, const Q *qs,
                                            const double *const *__restrict__ q0p, T *__restrict__ rhs,
                                            const double *__restrict__ gobj, const Op<T> &op,
                                            const SweepGeom &g, double gamma, double inv_h, long N,
                                            const RkArgs<T> &rk, Lines &ln) {
  constexpr bool FIRST = DIR == 2, LAST = DIR == 0;
  const double *__restrict__ q = *q0p;
  const FieldIO<DIR, T> io(tp, g);
  const T ih = T(inv_h), gam = T(gamma), gm1 = T(gamma - 1.0), ggm = T(gamma / (gamma - 1.0));
  T ud[PPT], irho[PPT], S[PPT], R5[PPT], f[PPT], x[PPT], r[PPT];
  {
    T gdp[PPT], qs5[PPT];
    {
      T rho[PPT], md[PPT];
      io.ld(q, rho);
      io.ld(q + (1 + DIR) * N, md);
      io.ld(q + 4 * N, f);  // p
      io.ld(qs + 4 * N, qs5);
      issue_loads();
      io.got(rho);
      io.got(md);
      io.got(f);
      io.got(qs5);
#pragma unroll
      for (int m = 0; m < PPT; ++m) {
        irho[m] = T(1) / rho[m];
        ud[m] = md[m] * irho[m];
        gdp[m] = ggm * f[m] * irho[m];
      }
    }
    // P = D p
    ln.solve(op, f, x);
#pragma unroll
    for (int m = 0; m < PPT; ++m) S[m] = qs5[m] * irho[m] * (x[m] * ih);
    pin(S);
    // E = D qs5
    ln.solve(op, qs5, x);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T E = x[m] * ih;
      S[m] = S[m] + gdp[m] * E;
      R5[m] = gam * ud[m] * E;
      f[m] = -ud[m] * qs5[m];
    }
    pin(R5);
  }
  // F = D(-u_d qs5)
  ln.solve(op, f, x);
#pragma unroll
  for (int m = 0; m < PPT; ++m) R5[m] = R5[m] + gm1 * (x[m] * ih);
  // B_d = D qs_{d+2} completes r5 (the fences keep each group of loads next
  // to the solve it feeds, and the accumulators and forward momenta that a
  // solve's result meets are loaded after it, so that they take no registers
  // across it)
  T Ta[PPT];
  {
    asm volatile("" ::: "memory");
    io.ld(qs + (1 + DIR) * N, f);
    io.got(f);
    ln.solve(op, f, x);
    asm volatile("" ::: "memory");
    if (!FIRST) {
      io.ld(rhs + 4 * N, r);
      io.got(r);
    }
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T Bd = x[m] * ih;
      S[m] = S[m] + ud[m] * Bd;
      Ta[m] = ud[m] * Bd;
      R5[m] = R5[m] + gm1 * Bd;
      r[m] = FIRST ? -R5[m] : r[m] - R5[m];
    }
    pin(Ta);
    finish<LAST, RK>(4, r, io, N, rhs, gobj, rk);
  }
  // A = D qs1; A + u_d B_d waits in LDS (the thread's own slots) until the
  // end, which keeps the x sweep within 256 registers without spilling
  __shared__ T stash[PPT][NT];
  asm volatile("" ::: "memory");
  io.ld(qs, f);
  io.got(f);
  ln.solve(op, f, x);
#pragma unroll
  for (int m = 0; m < PPT; ++m) stash[m][threadIdx.x] = Ta[m] + x[m] * ih;
  // B_m = D qs_{m+2}, m != d
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (i == DIR) continue;
    T um[PPT];
    asm volatile("" ::: "memory");
    io.ld(qs + (1 + i) * N, f);
    io.got(f);
    ln.solve(op, f, x);
    asm volatile("" ::: "memory");
    io.ld(q + (1 + i) * N, um);
    if (!FIRST) io.ld(rhs + (1 + i) * N, r);
    io.got(um);
    if (!FIRST) io.got(r);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T Bm = x[m] * ih;
      S[m] = S[m] + (um[m] * irho[m]) * Bm;
      r[m] = FIRST ? -(ud[m] * Bm) : r[m] - ud[m] * Bm;
    }
    finish<LAST, RK>(1 + i, r, io, N, rhs, gobj, rk);
  }
  // r1 += u_d S, r_{d+2} -= A + u_d B_d + S
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const int var = v == 0 ? 0 : 1 + DIR;
    asm volatile("" ::: "memory");
    if (!FIRST) {
      io.ld(rhs + var * N, r);
      io.got(r);
    }
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T c = v == 0 ? ud[m] * S[m] : -(stash[m][threadIdx.x] + S[m]);
      r[m] = FIRST ? c : r[m] + c;
    }
    finish<LAST, RK>(var, r, io, N, rhs, gobj, rk);
  }
}

template <typename T, typename Q, int DIR, bool PER, int RK>
__global__ __launch_bounds__(NT) void k_asweep(const Q *qs, const double *const *__restrict__ q0p,
                                               T *__restrict__ rhs, const double *__restrict__ gobj,
                                               Op<T> op, SweepGeom g, double gamma, double inv_h, long N,
                                               RkArgs<T> rk) {
  const ThreadPos tp = thread_pos<DIR>(g);
  auto ln = make_lines<T, PER>(op, tp);
  asweep_body<T, Q, DIR, RK>(tp, qs, q0p, rhs, gobj, op, g, gamma, inv_h, N, rk, ln);
}

// characteristic_qs_k1d (src/boundaries/nonreflecting.f90:453-554) on the
// points of one box: removes the incoming adjoint characteristics of qs.
// shape (type 203, characteristic_qs_k4d, :596-601): the change toward zero
// is scaled by shape at the point.
template <typename Q>
__global__ __launch_bounds__(256) void k_bc_characteristic_qs(Q *__restrict__ qs,
                                                               const double *const *__restrict__ q0p,
                                                               BoxRow row, int n1, int n2, long N,
                                                               double gamma,
                                                               const double *__restrict__ kfield,
                                                               const double *__restrict__ shape) {
  // forward state at the point (201) or at its inner neighbour (200)
  const double *__restrict__ q = *q0p + row.aim_shift;
  const long nx = row.i1 - row.i0 + 1, ny = row.j1 - row.j0 + 1, nz = row.k1 - row.k0 + 1;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nx * ny * nz) return;
  const long i = row.i0 + t % nx, j = row.j0 + (t / nx) % ny, k = row.k0 + t / (nx * ny);
  const long o = i + (long)n1 * (j + (long)n2 * k);
  const double s1 = double(qs[o]), s2 = double(qs[N + o]), s3 = double(qs[2 * N + o]),
               s4 = double(qs[3 * N + o]), s5 = double(qs[4 * N + o]);
  // the row's normal, or the point's (202: characteristic_qs_k4d)
  const double kx = -(kfield ? kfield[o] : row.k[0]), ky = -(kfield ? kfield[N + o] : row.k[1]),
               kz = -(kfield ? kfield[2 * N + o] : row.k[2]);
  const double gm1 = gamma - 1.0;
  const double c = sqrt(gamma * (q[4 * N + o] / q[o]));
  const double g_c = gm1 / c;
  const double u = q[N + o] / q[o], v = q[2 * N + o] / q[o], w = q[3 * N + o] / q[o];
  // increments toward zero adjoint in the incoming waves
  const double sh = shape ? shape[o] : 1.0;
  const double d1 = -s1 * sh, d2 = -s2 * sh, d3 = -s3 * sh, d4 = -s4 * sh, d5 = -s5 * sh;
  const double ku = kx * u + ky * v + kz * w;
  const double kus = kx * d2 + ky * d3 + kz * d4;
  const double ruus = (d1 + u * d2 + v * d3 + w * d4) / c;
  const double rups = ruus + d5 / g_c;
  double drs = 0, dus = 0, dvs = 0, dws = 0, dps = 0;
  if (ku < 0.0) {  // entropy and vorticity waves enter
    drs = d1 + ku * kus;
    dus = d2 - kx * kus;
    dvs = d3 - ky * kus;
    dws = d4 - kz * kus;
    dps = -g_c * ruus;
  }
  if (ku + c < 0.0) {  // acoustic wave ku + c enters
    const double a = 0.5 * (kus + rups);
    drs = drs - ku * a;
    dus = dus + kx * a;
    dvs = dvs + ky * a;
    dws = dws + kz * a;
    dps = dps + g_c * a;
  }
  if (ku - c < 0.0) {  // acoustic wave ku - c enters
    const double a = 0.5 * (kus - rups);
    drs = drs - ku * a;
    dus = dus + kx * a;
    dvs = dvs + ky * a;
    dws = dws + kz * a;
    dps = dps - g_c * a;
  }
  qs[o] = Q(s1 + drs);
  qs[N + o] = Q(s2 + dus);
  qs[2 * N + o] = Q(s3 + dvs);
  qs[3 * N + o] = Q(s4 + dws);
  qs[4 * N + o] = Q(s5 + dps);
}

// sponge_rhss_correct (src/boundaries/sponge_layer_core.f90:107-151), the
// adjoint sponge of rows 400 when set_boundary_condition_rhss gets the
// forward state (the Euler adjoint, euler_rho_rhou_p.f90:384):
// rhss += sigma (qs1 - u.qs(2:4)/rho, qs(2:4)/rho, (gamma - 1) qs5), with qs
// the adjoint state the RHS was computed from and q the forward state.
template <typename T, typename Q>
__global__ __launch_bounds__(256) void k_sponge_rhss(T *__restrict__ rhs, const Q *__restrict__ qs,
                                                      const double *const *__restrict__ q0p,
                                                      const double *__restrict__ sigma, double gamma,
                                                      long N) {
  const long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= N) return;
  const double *__restrict__ q = *q0p;
  const double rho = q[o];
  const double u1 = q[N + o] / rho, u2 = q[2 * N + o] / rho, u3 = q[3 * N + o] / rho;
  const double s1 = double(qs[o]), s2 = double(qs[N + o]), s3 = double(qs[2 * N + o]),
               s4 = double(qs[3 * N + o]), s5 = double(qs[4 * N + o]);
  const double sg = sigma[o];
  const double r1 = 1.0 * s1 - u1 / rho * s2 - u2 / rho * s3 - u3 / rho * s4;
  rhs[o] = T(double(rhs[o]) + sg * r1);
  rhs[N + o] = T(double(rhs[N + o]) + sg * (1.0 / rho * s2));
  rhs[2 * N + o] = T(double(rhs[2 * N + o]) + sg * (1.0 / rho * s3));
  rhs[3 * N + o] = T(double(rhs[3 * N + o]) + sg * (1.0 / rho * s4));
  rhs[4 * N + o] = T(double(rhs[4 * N + o]) + sg * ((gamma - 1.0) * s5));
}

// sponge_qs (src/boundaries/sponge_layer_core.f90:155-167): qs <- qs - sigma qs.
template <typename Q>
__global__ __launch_bounds__(256) void k_bc_sponge_qs(Q *__restrict__ qs,
                                                       const double *__restrict__ sigma, long N) {
  const long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= N) return;
  const double s = sigma[o];
  if (s == 0.0) return;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const double x = double(qs[v * N + o]);
    qs[v * N + o] = Q(x - s * x);
  }
}

}  // namespace cruna
