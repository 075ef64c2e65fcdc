// Fused direct-RHS sweeps, filter sweep and single-derivative kernel.
//
// One RK stage of right_hand_side_direct_3d (src/equations/ns_rho_rhou_p.f90:31-253)
// is evaluated in six line sweeps; each sweep applies every compact
// derivative that runs along its direction, so the 42 Dx calls of the
// reference become 42 line solves on register-resident blocks:
//   S1 x : u_x v_x w_x, d/dx of (rho u), (rho u u_i), p, (p u), T and lambda T_x
//   S2 y : the same along y                                  (accumulates rhs)
//   S3 z : the same along z
//   S4 z : d/dz tau_{iz}
//   S5 y : d/dy tau_{iy}
//   S6 x : d/dx tau_{ix} and tau:grad(u), then the RK4 stage update
//          (src/time/rk_o4_e.f90:45-50)
// The pressure equation is accumulated as the bracket of ns_rho_rhou_p.f90:200-206
// and multiplied by (gamma - 1) once, as the reference does.
//
//
// Field layout in HBM: every field is f(n1,n2,n3) Fortran order; a state holds
// 5 fields at a stride of N = n1*n2*n3 elements.  The viscous stress and the
// dissipation use the velocity gradient only through its diagonal and the
// symmetric sums, so G holds 6 fields, and a seventh with the viscosity:
//   G0 = u_x, G1 = v_y, G2 = w_z, G3 = u_y + v_x, G4 = u_z + w_x, G5 = v_z + w_y,
//   G6 = mu(T) of the stage input
// (each sum is completed by the second sweep that contributes to it; the
// result equals the reference's u_y + v_x etc. bit for bit).  S1 x evaluates
// the viscosity law once per point and stage; S2, S3 and S4-S6 read it.
//
// FP64 Cartesian form (sweep1_y_stress, sweep12_z_stress): the later sweeps need the
// stresses, not the gradients, so a gradient field turns into a stress where
// it is complete: S2 y stores tau_12 (G3) and takes its y derivative at once, S3
// z stores tau_11, tau_22, tau_13, tau_23 (G0, G1, G4, G5), and each adds its part of
// tau:grad(u) to the pressure bracket.  S5 y then reads two fields and S6 x
// three, without the viscosity: 20 + 24 + 6 + 8 words per point and stage in
// S2, S3+S4, S5, S6 (before the RK update) instead of 20 + 23 + 12 + 12 (256^3, per
// stage: S5 0.327 -> 0.158 ms, S6 with the shorter update 0.836 -> 0.478, S3+S4
// 0.664 -> 0.688; the step 11.4 -> 10.3 ms).  Not in FP32, whose bits depend on the order of these sums, nor in the deformed-grid
// and penalised forms.
#pragma once

#include "line_solve.hpp"

namespace cruna {

struct Phys {
  double gamma;
  double gm1;        // gamma - 1
  double gt;         // gamma / (gamma - 1)
  double w_inv_r;    // W / R     (give_T)
  double mu0, T0;
  double visc_exp;
  int visc_law;      // 0 Sutherland, 1 power law
  double cp;         // gamma (R/W) / (gamma - 1)
  double Pr;
  double lam_coef;   // cp / Pr  (lambda = mu cp / Pr)
  double inv_T0;     // 1 / T0
  double inv_h[3];       // 1/dx_d
  double heat_inv_h[3];  // 1/dx_d, or 1 for the reference's unit-spacing heat flux
};

// Deformed grid with a diagonal metric whose entries M(d,d) are constant along
// the lines of direction d (every tensor-product stretch of a Cartesian grid:
// ns_rho_rhou_p_grid_transform.f90 with X_metric from grid_metric.f90).
// Stored per line of each direction and the Jacobian per point, in the
// compute precision.
template <typename T>
struct Metric {
  const T *m[3];  // M(d,d) of the line through (j,k) / (i,k) / (i,j): index ThreadPos::lidx
  const T *J;     // X_jacobian(n1,n2,n3)
};

// Volume penalisation (ns_rho_rhou_p_ev_phi.f90): the porosity phi and the
// stored 1/phi (volume_penalization's penalization(:,:,:,1:2)) per point.
template <typename T>
struct Penal {
  const T *phi;
  const T *inv_phi;
};

// Right-hand-side form of the sweeps: Cartesian (ns_rho_rhou_p), deformed
// grid with a tensor-product metric (ns_rho_rhou_p_grid_transform), or
// volume-penalised (ns_rho_rhou_p_ev_phi).
enum RhsForm { RHS_CART = 0, RHS_GT = 1, RHS_EV = 2 };

// give_mu, ns_rho_rhou_p_trafos.f90:119-142: mu0*(T/T0)**1.5*((T0+S1)/(T+S1)),
// or the power law mu0*(T/T0)**exp of the case-level override.
template <typename T>
__device__ __forceinline__ T viscosity(const Phys &ph, T Tk) {
  const T r = Tk * T(ph.inv_T0);
  // r > 0, so r**e = 2**(e log2 r) without pow's special-case branches
  if (ph.visc_law == 1) return T(ph.mu0) * exp2(T(ph.visc_exp) * log2(r));
  const T S1 = T(110.4);
  return T(ph.mu0) * (r * sqrt(r)) * ((T(ph.T0) + S1) / (Tk + S1));
}

// Issue point of a group of global loads: the compiler may not sink them below
// this line (it otherwise moves each point's loads down to its first use and
// serialises their latencies).
__device__ __forceinline__ void issue_loads() { asm volatile("" ::: "memory"); }

// Materialise a value here: the compiler otherwise sinks a computation to its
// (late) use and keeps all of its operands live across the line solves between.
template <typename T>
__device__ __forceinline__ void materialize(T (&a)[PPT]) {
#pragma unroll
  for (int m = 0; m < PPT; ++m) asm volatile("" : "+v"(a[m]));
}

// give_T (:57) and give_lambda (:169): T = (W/R) p / rho, lambda = mu cp / Pr,
// with 1/rho formed once per point by the caller
template <typename T>
__device__ __forceinline__ T temperature(const Phys &ph, T irho, T p) {
  return T(ph.w_inv_r) * p * irho;
}
template <typename T>
__device__ __forceinline__ T lambda_of(const Phys &ph, T mu) {
  return mu * T(ph.lam_coef);
}

// A thread's block is PPT consecutive points of its line.  Along x those are
// contiguous and 64-byte aligned (FP64), so they move as 16-byte vectors;
// along y/z they are PS elements apart.  Field accesses are raw buffer loads
// and stores: the field base in a buffer resource (SGPRs) and 32-bit byte
// offsets (the host checks that a field fits in 2 GiB).  Along x and y a
// block costs one offset VGPR: the distance m*PS between its points goes in
// the scalar offset.  Along z that distance is a multiple of the plane size
// (512 KiB at 256^2 FP64), and measured on the 256^3 step the z sweeps run
// 5-40 % faster with the point offsets in VGPRs and a zero scalar offset.
// Buffer accesses count against vmcnt only, so the line engine's LDS waits
// never wait for them.
typedef unsigned int bu2 __attribute__((ext_vector_type(2)));
typedef unsigned int bu4 __attribute__((ext_vector_type(4)));

// Buffer extent: 2 GiB from the field base (the host keeps one field below
// that).  An idle thread of a batched launch (IDLE_BASE) has the extent
// itself as its FP64 offset, so that its loads return zero and its stores are
// dropped by the buffer range check (which tests the per-thread offset); along
// z its point offsets stay below 4 GiB, as a field's plane distance times 7
// stays below 2 GiB.
constexpr unsigned FIELD_EXTENT = 0x80000000u;
static_assert(IDLE_BASE * 8 == FIELD_EXTENT, "idle FP64 offset is the buffer extent");

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *p) {
  // raw buffer (stride 0); word 3 is the gfx9 format word of a plain dword
  // buffer
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(FIELD_EXTENT), 0x00020000);
}

template <int DIR, typename T, typename Q>
__device__ __forceinline__ void ld(const Q *__restrict__ p, long base, long PS, T (&v)[PPT]) {
  const __amdgpu_buffer_rsrc_t r = rsrc(p);
  const unsigned vo = unsigned(base) * unsigned(sizeof(Q));
  if (DIR == 0) {
#pragma unroll
    for (int k = 0; k < PPT * int(sizeof(Q)) / 16; ++k) {
      const bu4 t = __builtin_amdgcn_raw_buffer_load_b128(r, vo, k * 16, 0);
      if constexpr (sizeof(Q) == 8) {
        v[2 * k] = T(__builtin_bit_cast(double, bu2{t[0], t[1]}));
        v[2 * k + 1] = T(__builtin_bit_cast(double, bu2{t[2], t[3]}));
      } else {
        // each element through a scalar: a bit cast of a vector element
        // lvalue reads the vector's first element
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const unsigned e = t[j];
          v[4 * k + j] = T(__builtin_bit_cast(float, e));
        }
      }
    }
  } else {
    const unsigned ps = unsigned(PS) * unsigned(sizeof(Q));
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const unsigned vm = DIR == 2 ? vo + m * ps : vo, sm = DIR == 2 ? 0u : m * ps;
      if constexpr (sizeof(Q) == 8)
        v[m] = T(__builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vm, sm, 0)));
      else
        v[m] = T(__builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vm, sm, 0)));
    }
  }
}

template <int DIR, typename T, typename Q>
__device__ __forceinline__ void st(Q *__restrict__ p, long base, long PS, const T (&v)[PPT]) {
  const __amdgpu_buffer_rsrc_t r = rsrc(p);
  const unsigned vo = unsigned(base) * unsigned(sizeof(Q));
  if (DIR == 0) {
#pragma unroll
    for (int k = 0; k < PPT * int(sizeof(Q)) / 16; ++k) {
      bu4 t;
      if constexpr (sizeof(Q) == 8) {
        const bu2 a = __builtin_bit_cast(bu2, double(v[2 * k])), b = __builtin_bit_cast(bu2, double(v[2 * k + 1]));
        t = bu4{a[0], a[1], b[0], b[1]};
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = __builtin_bit_cast(unsigned, float(v[4 * k + j]));
      }
      __builtin_amdgcn_raw_buffer_store_b128(t, r, vo, k * 16, 0);
    }
  } else {
    const unsigned ps = unsigned(PS) * unsigned(sizeof(Q));
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const unsigned vm = DIR == 2 ? vo + m * ps : vo, sm = DIR == 2 ? 0u : m * ps;
      if constexpr (sizeof(Q) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(bu2, double(v[m])), r, vm, sm, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, float(v[m])), r, vm, sm, 0);
    }
  }
}

// Field access of a sweep along DIR.  ld issues the loads of the thread's block,
// got (after all loads of a group are issued) makes the values the thread's
// own; st stores.  Along y and z got does nothing.  Along x a thread's block is
// 64 contiguous bytes (FP64), so thread-by-thread 16-byte accesses lie 64 bytes
// apart and each instruction touches every cache line of the wavefront's 4 KB,
// which makes the vector cache's request rate the limit.  In FP64 lane l moves
// chunk l of each contiguous 1 KB instead, and the blocks are exchanged through
// LDS within the wavefront (a lane's slot is 80 bytes, so that 8 lanes' 16-byte
// pieces fall on different banks).  Measured at 256^3: the x first-derivative
// sweep 456 -> 356 us (14 words per point: 4.1 -> 5.3 TB/s), at 128^3 59 -> 44 us,
// the x filter 38 -> 30 us.  FP32 (32-byte blocks) gained nothing and keeps the
// thread-by-thread form.
template <int DIR>
struct StridedIO {
  long B, PS;
  __device__ __forceinline__ StridedIO(const ThreadPos &tp, const SweepGeom &g, size_t = 0) : B(tp.base), PS(g.PS) {}
  template <typename Q, typename V>
  __device__ __forceinline__ void ld(const Q *__restrict__ p, V (&v)[PPT]) const {
    cruna::ld<DIR>(p, B, PS, v);
  }
  template <typename V>
  __device__ __forceinline__ void got(V (&)[PPT]) const {}
  template <typename Q, typename V>
  __device__ __forceinline__ void st(Q *__restrict__ p, const V (&v)[PPT]) const {
    cruna::st<DIR>(p, B, PS, v);
  }
};
template <int DIR, typename T>
struct FieldIO : StridedIO<DIR> {
  using StridedIO<DIR>::StridedIO;
};

constexpr int X_STAGE = 80;  // bytes of LDS per thread of an FP64 x sweep
inline size_t x_stage_bytes(int threads) { return (size_t)((threads + 63) / 64 * 64) * X_STAGE; }
// dynamic LDS of a sweep along dir in a work-group of `threads`
template <typename T>
size_t sweep_lds_bytes(int dir, int threads) {
  return line_lds_bytes<T>(threads) + (dir == 0 && sizeof(T) == 8 ? x_stage_bytes(threads) : 0);
}

template <>
struct FieldIO<0, double> {
  static constexpr int NCH = PPT / 2;  // 16-byte chunks of a block
  char *own, *raw;     // LDS: the lane's slot; the place of the chunks it moves
  unsigned off;        // byte offset of its first chunk in a field
  unsigned gstep, lstep;  // distance of its chunks in the field, in LDS
  // (behind the line engine's dynamic LDS, of engine_bytes)
  __device__ __forceinline__ FieldIO(const ThreadPos &tp, const SweepGeom &g)
      : FieldIO(tp, g, rec_lds_bytes(blockDim.x)) {}
  __device__ __forceinline__ FieldIO(const ThreadPos &tp, const SweepGeom &, size_t engine_bytes) {
    const unsigned lane = threadIdx.x & 63;
    char *stage = line_dyn + engine_bytes + (threadIdx.x >> 6) * (64 * X_STAGE);
    const bool idle = tp.base == IDLE_BASE;
    // lanes with a block: the first ones of the wavefront, their blocks one
    // after the other in memory
    const unsigned active = __popcll(__builtin_amdgcn_ballot_w64(!idle));
    const unsigned first = __builtin_amdgcn_readfirstlane(unsigned(tp.base)) * 8u;
    own = stage + lane * X_STAGE;
    if (active % NCH == 0 && active != 0) {
      // chunk k * active + lane of the wavefront, k = 0..3
      raw = idle ? own : stage + (lane / NCH) * X_STAGE + (lane % NCH) * 16;
      off = idle ? FIELD_EXTENT : first + lane * 16;
      gstep = active * 16;
      lstep = active / NCH * X_STAGE;
    } else {  // the lane's own block
      raw = own;
      off = idle ? FIELD_EXTENT : first + lane * 64;
      gstep = 16;
      lstep = 16;
    }
  }
  __device__ __forceinline__ static void order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
  __device__ __forceinline__ void ld(const double *__restrict__ p, double (&v)[PPT]) const {
    const __amdgpu_buffer_rsrc_t r = rsrc(p);
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      const bu4 t = __builtin_amdgcn_raw_buffer_load_b128(r, off, k * gstep, 0);
      v[2 * k] = __builtin_bit_cast(double, bu2{t[0], t[1]});
      v[2 * k + 1] = __builtin_bit_cast(double, bu2{t[2], t[3]});
    }
  }
  // (an idle lane's chunk k >= 1 would fall outside its slot: it writes nothing)
  __device__ __forceinline__ void got(double (&v)[PPT]) const {
#pragma unroll
    for (int k = 0; k < NCH; ++k)
      if (off != FIELD_EXTENT) *reinterpret_cast<double2 *>(raw + k * lstep) = double2{v[2 * k], v[2 * k + 1]};
    order();
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const double2 c = *reinterpret_cast<const double2 *>(own + j * 16);
      v[2 * j] = c.x;
      v[2 * j + 1] = c.y;
    }
    order();
  }
  __device__ __forceinline__ void st(double *__restrict__ p, const double (&v)[PPT]) const {
#pragma unroll
    for (int j = 0; j < NCH; ++j) *reinterpret_cast<double2 *>(own + j * 16) = double2{v[2 * j], v[2 * j + 1]};
    order();
    const __amdgpu_buffer_rsrc_t r = rsrc(p);
    static_assert(NCH == 4, "the registers held below");
    bu4 t[NCH];
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      // (an idle lane's store is dropped; it reads its own slot)
      t[k] = *reinterpret_cast<const bu4 *>(off != FIELD_EXTENT ? raw + k * lstep : own + k * 16);
      __builtin_amdgcn_raw_buffer_store_b128(t[k], r, off, k * gstep, 0);
    }
    // A store of 16 bytes still reads its data registers for two wait states
    // after it has been issued.  The compiler keeps other instructions off them
    // for that long, but not where the store's offset is a scalar register, as
    // here: an x sweep whose next multiplication took the last store's registers
    // wrote a product's half in place of the data in one line of 1500.  The
    // registers are held past the wait states.
    asm volatile("s_nop 1" ::"v"(t[0]), "v"(t[1]), "v"(t[2]), "v"(t[3]));
    order();
  }
};

// Work-group size limit of the Cartesian viscous sweeps: FP32 tiles take up
// to 32 y/z lines so that rows of floats are 128 bytes, as FP64 rows of 16.
template <typename T>
constexpr int sweep_nt() { return sizeof(T) == 4 ? NT_SWEEP32 : NT; }

// ----------------------------------------------------------------------------
// S1 / S2 / S3: first-derivative sweeps along DIR.
//   qs  : stage input state (5 fields, type Q)
//   rhs : 5 accumulator fields (S1 writes, S2/S3 read-modify-write)
//   G   : velocity-gradient fields (layout above)
// The solves are ordered so that each state field is live only while needed:
// the two transverse momentum components first (velocity gradient and
// momentum flux of each), then the DIR component, mass, pressure gradient,
// energy and heat flux with rho, rho u_DIR and p only.  Read-modify-write
// operands are fetched just before the line solve whose result they meet, so
// their latency hides behind the solve (the engine's barriers do not wait on
// global loads).
// GT: deformed grid (ns_rho_rhou_p_grid_transform.f90:31-330).  Every
// derivative along DIR is scaled by the line's metric entry M(DIR,DIR)
// (physical gradients, contravariant fluxes and the projected stresses all
// reduce to that for a diagonal metric); the heat flux takes the temperature
// gradient with h and lambda J inside, the outer derivative without h.
// EV: volume penalisation (ns_rho_rhou_p_ev_phi.f90:33-291): every flux
// carries phi inside its derivative and its divergence is multiplied by
// the stored 1/phi, distributed over the directions (the pressure
// gradient and u.grad(p) are not); both heat-flux derivatives take no h.
// What the fused z kernel's viscous part takes from its first-derivative
// part (k_sweep12_z, Cartesian form): the block's velocity gradients that the
// z sweep completes (s13 = u_z + w_x, s23 = v_z + w_y, w_z) and the
// viscosity in registers; the momentum RHS of the block in LDS (the thread's
// own slots) instead of a store and a reload through HBM.
template <typename T>
struct ZCarry {
  T s13[PPT], s23[PPT], wz[PPT], mu[PPT];
  T (*slots)[PPT][NT];  // LDS: [3][PPT][NT] momentum RHS (x, y, z)
  __device__ __forceinline__ T &mom(int i, int m) const { return slots[i][m][threadIdx.x]; }
};

template <typename T, typename Q, int DIR, int FORM, bool FUSE = false, typename Lines>
__device__ __forceinline__ void sweep1_body(const ThreadPos &tp, const Q *__restrict__ qs, T *__restrict__ rhs,
                                            T *__restrict__ G, const Op<T> &op, const SweepGeom &g,
                                            const Phys &ph, long N, const Metric<T> &mt, const Penal<T> &pe,
                                            Lines &ln, ZCarry<T> *zc = nullptr) {
  constexpr bool GT = FORM == RHS_GT, EV = FORM == RHS_EV;
  static_assert(!FUSE || (DIR == 2 && FORM == RHS_CART), "the fused z sweep is Cartesian");
  const FieldIO<DIR, T> io(tp, g);
  const T mline = GT ? mt.m[DIR][tp.lidx] : T(1);
  const T ih = GT ? T(ph.inv_h[DIR]) * mline : T(ph.inv_h[DIR]);
  // heat flux: inner (temperature) and outer derivative scales
  const T hin = GT ? ih : (EV ? T(1) : T(ph.heat_inv_h[DIR]));
  const T hout = GT ? mline : (EV ? T(1) : T(ph.heat_inv_h[DIR]));
  // penalisation: phi inside the fluxes, the stored 1/phi on their divergence
  T PH[PPT], IP[PPT];
  if (EV) {
    io.ld(pe.phi, PH);
    io.ld(pe.inv_phi, IP);
    io.got(PH);
    io.got(IP);
  }
  auto div = [&](int m, T v) -> T { return EV ? IP[m] * v : v; };
  // G slot of d(u_i)/dx_DIR and whether it completes a symmetric sum begun by
  // an earlier sweep: x writes u_x, v_x, w_x; y adds u_y to v_x and writes
  // v_y, w_y; z adds u_z to w_x, v_z to w_y and writes w_z
  auto gslot = [](int i) -> int {
    return DIR == 0 ? (i == 0 ? 0 : (i == 1 ? 3 : 4))
                    : (DIR == 1 ? (i == 0 ? 3 : (i == 1 ? 1 : 5)) : (i == 0 ? 4 : (i == 1 ? 5 : 2)));
  };
  auto gsum = [](int i) -> bool { return (DIR == 1 && i == 0) || (DIR == 2 && i < 2); };
  T irho[PPT], mom[PPT], p[PPT], f[PPT], x[PPT], y[PPT], r[PPT];
  io.ld(qs, f);
  io.ld(qs + (1 + DIR) * N, mom);
  if (DIR == 0) issue_loads();
  io.got(f);
  io.got(mom);
#pragma unroll
  for (int m = 0; m < PPT; ++m) irho[m] = T(1) / f[m];

  // transverse components i != DIR: d(u_i)/dx_DIR (ns_rho_rhou_p.f90:102-112)
  // and the momentum flux -d/dx_DIR (rho u_DIR u_i) (:138-172)
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = k == 0 ? (DIR == 0 ? 1 : 0) : (DIR == 2 ? 1 : 2);
    T ui[PPT], gs[PPT];
    asm volatile("" ::: "memory");
    io.ld(qs + (1 + i) * N, ui);
    if (gsum(i)) io.ld(G + gslot(i) * N, gs);
    issue_loads();
    io.got(ui);
    if (gsum(i)) io.got(gs);
#pragma unroll
    for (int m = 0; m < PPT; ++m) ui[m] = ui[m] * irho[m];
    ln.pair(
        op, ui, y,
        [&] {
#pragma unroll
          for (int m = 0; m < PPT; ++m) {
            y[m] = y[m] * ih;
            if (gsum(i)) y[m] = y[m] + gs[m];
          }
          io.st(G + gslot(i) * N, y);
          if constexpr (FUSE) {
#pragma unroll
            for (int m = 0; m < PPT; ++m) (k == 0 ? zc->s13 : zc->s23)[m] = y[m];
          }
        },
        [&] {
          if (DIR != 0) io.ld(rhs + (1 + i) * N, r);
          if (k == 1) io.ld(qs + 4 * N, p);  // in flight for the pressure terms
#pragma unroll
          for (int m = 0; m < PPT; ++m) f[m] = EV ? (PH[m] * mom[m]) * ui[m] : mom[m] * ui[m];
        },
        f, x,
        [&] {
          if (DIR != 0) io.got(r);
          if (k == 1) io.got(p);
#pragma unroll
          for (int m = 0; m < PPT; ++m) r[m] = DIR == 0 ? div(m, -(x[m] * ih)) : r[m] + div(m, -(x[m] * ih));
          if constexpr (FUSE) {
#pragma unroll
            for (int m = 0; m < PPT; ++m) zc->mom(i, m) = r[m];
          } else {
            io.st(rhs + (1 + i) * N, r);
          }
        });
  }

  // d(u_DIR)/dx_DIR, and mass: -d/dx_DIR (rho u_DIR) (:131-135)
  T ud[PPT];
#pragma unroll
  for (int m = 0; m < PPT; ++m) ud[m] = mom[m] * irho[m];
  ln.pair(
      op, ud, y,
      [&] {
#pragma unroll
        for (int m = 0; m < PPT; ++m) y[m] = y[m] * ih;
        io.st(G + DIR * N, y);
        if constexpr (FUSE) {
#pragma unroll
          for (int m = 0; m < PPT; ++m) zc->wz[m] = y[m];
        }
      },
      [&] {
        if (DIR != 0) io.ld(rhs, r);
#pragma unroll
        for (int m = 0; m < PPT; ++m) f[m] = EV ? PH[m] * mom[m] : mom[m];
      },
      f, x,
      [&] {
        if (DIR != 0) io.got(r);
#pragma unroll
        for (int m = 0; m < PPT; ++m) r[m] = DIR == 0 ? div(m, -(x[m] * ih)) : r[m] + div(m, -(x[m] * ih));
        io.st(rhs, r);
      });

  // pressure gradient p_DIR, and momentum DIR: -d/dx_DIR (rho u_DIR u_DIR) - p_DIR
  T pd[PPT];
  ln.pair(
      op, p, pd,
      [&] {
#pragma unroll
        for (int m = 0; m < PPT; ++m) pd[m] = pd[m] * ih;
      },
      [&] {
        if (DIR != 0) io.ld(rhs + (1 + DIR) * N, r);
#pragma unroll
        for (int m = 0; m < PPT; ++m) f[m] = EV ? (PH[m] * mom[m]) * ud[m] : mom[m] * ud[m];
      },
      f, x,
      [&] {
        if (DIR != 0) io.got(r);
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
          r[m] = DIR == 0 ? div(m, -(x[m] * ih)) : r[m] + div(m, -(x[m] * ih));
          r[m] = r[m] - pd[m];
        }
        if constexpr (FUSE) {
#pragma unroll
          for (int m = 0; m < PPT; ++m) zc->mom(DIR, m) = r[m];
        } else {
          io.st(rhs + (1 + DIR) * N, r);
        }
      });

  // pressure-equation bracket: gamma/(gamma-1) (-d(p u_DIR)) + u_DIR p_DIR
  // (:180-187), and the inner derivative of the heat flux d/dx_DIR (lambda
  // d/dx_DIR T) (:189-199); the x sweep evaluates the viscosity law and leaves
  // mu in G6 for the later sweeps of the stage
  T e[PPT], tk[PPT], mu[PPT], Jv[PPT];
#pragma unroll
  for (int m = 0; m < PPT; ++m) f[m] = EV ? (PH[m] * p[m]) * ud[m] : p[m] * ud[m];
  ln.pair(
      op, f, x,
      [&] {
#pragma unroll
        for (int m = 0; m < PPT; ++m) e[m] = div(m, T(ph.gt) * (-(x[m] * ih))) + ud[m] * pd[m];
      },
      [&] {
        if (DIR != 0) {
          io.ld(rhs + 4 * N, r);
          io.ld(G + 6 * N, mu);
        }
        if (GT) io.ld(mt.J, Jv);
        if (DIR != 0) {
          io.got(r);
          io.got(mu);
        }
        if (GT) io.got(Jv);
#pragma unroll
        for (int m = 0; m < PPT; ++m) tk[m] = temperature(ph, irho[m], p[m]);
        if (DIR == 0) {
#pragma unroll
          for (int m = 0; m < PPT; ++m) mu[m] = viscosity(ph, tk[m]);
          io.st(G + 6 * N, mu);
        }
        if constexpr (FUSE) {
#pragma unroll
          for (int m = 0; m < PPT; ++m) zc->mu[m] = mu[m];
        }
      },
      tk, y,
      [&] {
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
          const T lam = GT ? lambda_of(ph, mu[m]) * Jv[m]
                           : (EV ? PH[m] * lambda_of(ph, mu[m]) : lambda_of(ph, mu[m]));
          f[m] = lam * (y[m] * hin);
        }
      });
  ln.solve(op, f, x);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    e[m] = e[m] + div(m, x[m] * hout);
    if (DIR != 0) e[m] = r[m] + e[m];
  }
  io.st(rhs + 4 * N, e);
}

template <typename T, int FORM>
constexpr bool stress_form() { return sizeof(T) == 8 && FORM == RHS_CART; }

// These FP64 sweeps write every fused multiply-add out and contract nothing, so
// that the batched kernels, compiled apart, give the same bits.

// S1 x in FP64 (Cartesian form): two independent solves per exchange, the
// transverse momenta in flight while the solves before them run.
template <typename Lines>
__device__ __forceinline__ void sweep1_x_cart(const ThreadPos &tp, const double *__restrict__ qs,
                                              double *__restrict__ rhs, double *__restrict__ G, const RecOp &op,
                                              const SweepGeom &g, const Phys &ph, long N, Lines &ln) {
#pragma clang fp contract(off)
  const FieldIO<0, double> io(tp, g);
  const double ih = ph.inv_h[0], hh = ph.heat_inv_h[0];
  double irho[PPT], mom[PPT], u[PPT], p[PPT], lt[PPT], f[PPT], x[PPT], y[PPT];
  io.ld(qs, irho);
  io.ld(qs + N, mom);
  io.ld(qs + 4 * N, p);
  issue_loads();
  io.got(irho);
  io.got(mom);
  io.got(p);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    irho[m] = 1.0 / irho[m];
    f[m] = temperature(ph, irho[m], p[m]);
  }
#pragma unroll
  for (int m = 0; m < PPT; ++m) lt[m] = viscosity(ph, f[m]);
  io.st(G + 6 * N, lt);
  // p_x and the inner derivative of the heat flux
  double pd[PPT];
  ln.solve2(op, p, pd, f, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    u[m] = mom[m] * irho[m];
    lt[m] = lambda_of(ph, lt[m]) * (y[m] * hh);
    pd[m] = pd[m] * ih;
    f[m] = mom[m] * u[m];
    p[m] = p[m] * u[m];
  }
  // rho u, and the pressure bracket's flux with u p_x
  ln.solve2(op, f, x, p, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    x[m] = __builtin_fma(-x[m], ih, -pd[m]);
    p[m] = __builtin_fma(-ph.gt, y[m] * ih, u[m] * pd[m]);
  }
  io.st(rhs + N, x);
  asm volatile("" ::: "memory");
  // the heat flux completes the bracket; u_x
  double v[PPT];
  io.ld(qs + 2 * N, v);
  ln.solve2(op, lt, x, u, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    p[m] = __builtin_fma(x[m], hh, p[m]);
    y[m] = y[m] * ih;
  }
  io.st(rhs + 4 * N, p);
  io.st(G, y);
  // v_x, w_x and the fluxes rho u v, rho u w
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    io.got(v);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      u[m] = v[m] * irho[m];
      f[m] = mom[m] * u[m];
    }
    asm volatile("" ::: "memory");
    if (i == 0) io.ld(qs + 3 * N, v);
    ln.solve2(op, u, x, f, y);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      x[m] = x[m] * ih;
      y[m] = -(y[m] * ih);
    }
    io.st(G + (3 + i) * N, x);
    io.st(rhs + (2 + i) * N, y);
  }
  // mass
  ln.solve(op, mom, x);
#pragma unroll
  for (int m = 0; m < PPT; ++m) x[m] = -(x[m] * ih);
  io.st(rhs, x);
}

// S2 y in the stress form: the first-derivative sweep along y with tau_12.
template <typename Lines>
__device__ __forceinline__ void sweep1_y_stress(const ThreadPos &tp, const double *__restrict__ qs,
                                                double *__restrict__ rhs, double *__restrict__ G, const RecOp &op,
                                                const SweepGeom &g, const Phys &ph, long N, Lines &ln) {
#pragma clang fp contract(off)
  const long B = tp.base, PS = g.PS;
  const double ih = ph.inv_h[1], hh = ph.heat_inv_h[1];
  double irho[PPT], mom[PPT], p[PPT], mu[PPT], f[PPT], u[PPT], x[PPT], y[PPT], r[PPT], e[PPT], lt[PPT];
  ld<1>(qs, B, PS, irho);
  ld<1>(qs + 2 * N, B, PS, mom);
  ld<1>(qs + 4 * N, B, PS, p);
  ld<1>(qs + N, B, PS, u);
  ld<1>(G + 3 * N, B, PS, r);  // v_x
  ld<1>(G + 6 * N, B, PS, mu);
  issue_loads();
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    irho[m] = 1.0 / irho[m];
    u[m] = u[m] * irho[m];
    f[m] = temperature(ph, irho[m], p[m]);
  }
  // u_y, which completes tau_12, and the inner derivative of the heat flux
  ln.solve2(op, u, x, f, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    const double s12 = __builtin_fma(x[m], ih, r[m]);
    x[m] = mu[m] * s12;  // tau_12
    e[m] = x[m] * s12;   // its part of tau:grad(u)
    lt[m] = lambda_of(ph, mu[m]) * (y[m] * hh);
    f[m] = mom[m] * u[m];
  }
  materialize(e);
  materialize(lt);
  st<1>(G + 3 * N, B, PS, x);
  ld<1>(rhs + N, B, PS, r);
  // rho u: -d(rho v u)/dy + d(tau_12)/dy
  ln.solve2(op, x, u, f, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) r[m] = __builtin_fma(u[m] - y[m], ih, r[m]);
  st<1>(rhs + N, B, PS, r);
  asm volatile("" ::: "memory");
  // w_y and rho w
  ld<1>(qs + 3 * N, B, PS, u);
  ld<1>(rhs + 3 * N, B, PS, r);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    u[m] = u[m] * irho[m];
    f[m] = mom[m] * u[m];
  }
  ln.solve2(op, u, x, f, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    x[m] = x[m] * ih;
    r[m] = __builtin_fma(-y[m], ih, r[m]);
  }
  st<1>(G + 5 * N, B, PS, x);
  st<1>(rhs + 3 * N, B, PS, r);
  asm volatile("" ::: "memory");
  // v_y and mass
  ld<1>(rhs, B, PS, r);
#pragma unroll
  for (int m = 0; m < PPT; ++m) u[m] = mom[m] * irho[m];
  ln.solve2(op, u, x, mom, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    x[m] = x[m] * ih;
    r[m] = __builtin_fma(-y[m], ih, r[m]);
  }
  st<1>(G + N, B, PS, x);
  st<1>(rhs, B, PS, r);
  asm volatile("" ::: "memory");
  // p_y and rho v
  ld<1>(rhs + 2 * N, B, PS, r);
#pragma unroll
  for (int m = 0; m < PPT; ++m) f[m] = mom[m] * u[m];
  ln.solve2(op, p, x, f, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    r[m] = __builtin_fma(-(x[m] + y[m]), ih, r[m]);
    e[m] = __builtin_fma(u[m], x[m] * ih, e[m]);  // u.grad(p)
    f[m] = p[m] * u[m];
  }
  st<1>(rhs + 2 * N, B, PS, r);
  asm volatile("" ::: "memory");
  // pressure bracket
  ld<1>(rhs + 4 * N, B, PS, r);
  ln.solve2(op, f, x, lt, y);
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    e[m] = __builtin_fma(-ph.gt, x[m] * ih, e[m]);
    r[m] = r[m] + __builtin_fma(y[m], hh, e[m]);
  }
  st<1>(rhs + 4 * N, B, PS, r);
}

// S3 + S4 z in the stress form: the first-derivative sweep along z, the stresses
// and their z derivatives.  The z sweep is the last first-derivative sweep of a
// stage, so the gradients of the thread's block are complete in it.  The
// momentum RHS of x and y wait in LDS (the thread's own slots, stride 17: odd,
// no bank conflicts) for the last two solves.
constexpr int ZS_STRIDE = 2 * PPT + 1;
inline size_t z_stress_lds_bytes(int threads) {
  return rec_lds_bytes(threads) + (size_t)threads * ZS_STRIDE * sizeof(double);
}
template <typename Lines>
__device__ __forceinline__ void sweep12_z_stress(const ThreadPos &tp, const double *__restrict__ qs,
                                                 double *__restrict__ rhs, double *__restrict__ G, const RecOp &op,
                                                 const SweepGeom &g, const Phys &ph, long N, Lines &ln) {
#pragma clang fp contract(off)
  const long B = tp.base, PS = g.PS;
  const double ih = ph.inv_h[2], hh = ph.heat_inv_h[2];
  double *slot = reinterpret_cast<double *>(line_dyn) + rec_lds_bytes(blockDim.x) / sizeof(double) + threadIdx.x * ZS_STRIDE;
  double mom[PPT], w[PPT], p[PPT], t1[PPT], t2[PPT], t3[PPT], e[PPT], lt[PPT];
  {
    double irho[PPT], f[PPT], u[PPT], x[PPT], y[PPT], r[PPT], sx[PPT];
    ld<2>(qs, B, PS, irho);
    ld<2>(qs + 3 * N, B, PS, mom);
    // u_z (+ w_x), v_z (+ w_y) and the momentum fluxes rho w u, rho w v
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ld<2>(qs + (1 + i) * N, B, PS, u);
      ld<2>(G + (4 + i) * N, B, PS, sx);
      ld<2>(rhs + (1 + i) * N, B, PS, r);
      issue_loads();
#pragma unroll
      for (int m = 0; m < PPT; ++m) {
        if (i == 0) irho[m] = 1.0 / irho[m];
        u[m] = u[m] * irho[m];
        f[m] = mom[m] * u[m];
      }
      ln.solve2(op, u, x, f, y);
#pragma unroll
      for (int m = 0; m < PPT; ++m) {
        (i == 0 ? t1 : t2)[m] = __builtin_fma(x[m], ih, sx[m]);
        slot[i * PPT + m] = __builtin_fma(-y[m], ih, r[m]);
      }
      asm volatile("" ::: "memory");
    }
    // w_z and the inner derivative of the heat flux
    ld<2>(qs + 4 * N, B, PS, p);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      w[m] = mom[m] * irho[m];
      f[m] = temperature(ph, irho[m], p[m]);
    }
    ln.solve2(op, w, t3, f, lt);
  }
  asm volatile("" ::: "memory");
  {
    // the stresses (ns_rho_rhou_p.f90:115-128) and tau:grad(u) without tau_12
    double ux[PPT], vy[PPT], mu[PPT];
    ld<2>(G + 6 * N, B, PS, mu);
    ld<2>(G, B, PS, ux);
    ld<2>(G + N, B, PS, vy);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const double s13 = t1[m], s23 = t2[m], wz = t3[m] * ih;
      const double md = -2.0 / 3.0 * mu[m] * (ux[m] + vy[m] + wz);
      const double m2 = 2.0 * mu[m];
      const double t11 = __builtin_fma(m2, ux[m], md), t22 = __builtin_fma(m2, vy[m], md);
      t1[m] = mu[m] * s13;
      t2[m] = mu[m] * s23;
      t3[m] = __builtin_fma(m2, wz, md);
      e[m] = __builtin_fma(
          t11, ux[m], __builtin_fma(t22, vy[m], __builtin_fma(t3[m], wz, __builtin_fma(t1[m], s13, t2[m] * s23))));
      lt[m] = lambda_of(ph, mu[m]) * (lt[m] * hh);
      ux[m] = t11;
      vy[m] = t22;
    }
    materialize(e);
    materialize(lt);
    materialize(t3);
    st<2>(G, B, PS, ux);
    st<2>(G + N, B, PS, vy);
    st<2>(G + 4 * N, B, PS, t1);
    st<2>(G + 5 * N, B, PS, t2);
  }
  {
    // z derivatives of tau_13 and tau_23 complete the x and y momentum
    double x[PPT], y[PPT];
    ln.solve2(op, t1, x, t2, y);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      x[m] = __builtin_fma(x[m], ih, slot[m]);
      y[m] = __builtin_fma(y[m], ih, slot[PPT + m]);
    }
    st<2>(rhs + N, B, PS, x);
    st<2>(rhs + 2 * N, B, PS, y);
  }
  asm volatile("" ::: "memory");
  {
    // mass and the heat flux
    double x[PPT], r[PPT];
    ld<2>(rhs, B, PS, r);
    ln.solve2(op, mom, x, lt, t1);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      r[m] = __builtin_fma(-x[m], ih, r[m]);
      e[m] = __builtin_fma(t1[m], hh, e[m]);
    }
    st<2>(rhs, B, PS, r);
  }
  asm volatile("" ::: "memory");
  {
    // rho w: p_z, d(tau_33)/dz, the flux; and the pressure bracket
    double f[PPT], x[PPT], y[PPT], r[PPT], q[PPT];
    ld<2>(rhs + 3 * N, B, PS, r);
    ln.solve2(op, p, x, t3, y);
    ld<2>(rhs + 4 * N, B, PS, q);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      e[m] = __builtin_fma(w[m], x[m] * ih, e[m]);
      r[m] = __builtin_fma(y[m] - x[m], ih, r[m]);
      f[m] = mom[m] * w[m];
      p[m] = p[m] * w[m];
    }
    ln.solve2(op, f, x, p, y);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      r[m] = __builtin_fma(-x[m], ih, r[m]);
      q[m] = q[m] + __builtin_fma(-ph.gt, y[m] * ih, e[m]);
    }
    st<2>(rhs + 3 * N, B, PS, r);
    st<2>(rhs + 4 * N, B, PS, q);
  }
}

template <typename T, typename Q, int DIR, bool PER, int FORM>
__global__ __launch_bounds__(NT) void k_sweep1(const Q *__restrict__ qs, T *__restrict__ rhs,
                                                          T *__restrict__ G, Op<T> op, SweepGeom g,
                                                          Phys ph, long N, Metric<T> mt, Penal<T> pe) {
  const ThreadPos tp = thread_pos<DIR, DIR == 0>(g);
  auto ln = make_lines<T, PER>(op, tp);
  if constexpr (DIR == 0 && stress_form<T, FORM>())
    sweep1_x_cart(tp, qs, rhs, G, op, g, ph, N, ln);
  else if constexpr (DIR == 1 && stress_form<T, FORM>())
    sweep1_y_stress(tp, qs, rhs, G, op, g, ph, N, ln);
  else
    sweep1_body<T, Q, DIR, FORM>(tp, qs, rhs, G, op, g, ph, N, mt, pe, ln);
}

// RK4 stage update of a variable from its complete RHS k (rk_o4_e.f90:45-50,
// and :90-95 for the adjoint with dt -> -dt): stage inputs y2 = q0 + dt/2 k1,
// y3 = q0 + dt/2 k2, y4 = q0 + dt k3, and q1 = q0 + dt/6 (k1 + 2 k2 + 2 k3 + k4).
// Two forms:
//  * RK_Y, RK_YLAST (FP64 without boundary rows): no accumulator.  The stage
//    inputs are kept, each in its own buffer, and the last stage forms
//    q1 = q0 + ((y2 - q0) + 2 (y3 - q0) + (y4 - q0)) / 3 + dt/6 k4: 10 + 10 +
//    10 + 25 words per point and step instead of 15 + 20 + 20 + 10, and three
//    roundings at the size of q0 that enter q1 by 1/3, 2/3, 1/3 plus one, where
//    the accumulator takes four.
//  * RK_FIRST, RK_MID, RK_LAST: an accumulator of the arithmetic type T.
//    FP64 (contexts with boundary rows, which change the stage inputs or need
//    the complete RHS): the partial new state q0 + dt/6 k1 + dt/3 k2 + dt/3 k3.
//    FP32-mixed: the increment dt/6 k1 + dt/3 k2 + dt/3 k3 alone, in FP32, and
//    the last stage adds q0 in FP64; the increment is a step's change of the
//    state, so its FP32 rounding is far below that of the FP32 stage inputs.
// RK_RHS writes k into rhs instead (a single RHS evaluation).
// The form is a template parameter: its loads then stand in one block with the
// RHS's and are in flight together (as a runtime switch each was waited for
// before the next was issued).
enum RkForm { RK_FIRST = 0, RK_MID = 1, RK_LAST = 3, RK_RHS = 4, RK_Y = 5, RK_YLAST = 6 };

template <typename T>
struct RkArgs {
  double *qn;             // q0, and q1 after the last stage
  T *acc;                 // accumulator
  T *out;                 // next stage input
  const T *y2, *y3, *y4;  // RK_YLAST: the kept stage inputs
  double dt, c;           // step, and the stage's c dt
};

// What the update of one variable reads besides k.
template <int RK, typename T>
struct RkIn {
  double q0[PPT];
  T a[PPT], b[PPT], c[PPT];
};

// (issued; rk_got makes the values the thread's own)
template <int RK, typename T, typename IO>
__device__ __forceinline__ void rk_load(const RkArgs<T> &rk, int v, const IO &io, long N, RkIn<RK, T> &in) {
  if constexpr (RK == RK_RHS) return;
  if constexpr (!(RK == RK_LAST && sizeof(T) == 8)) io.ld(rk.qn + v * N, in.q0);
  if constexpr (RK == RK_MID || RK == RK_LAST) io.ld(rk.acc + v * N, in.a);
  if constexpr (RK == RK_YLAST) {
    io.ld(rk.y2 + v * N, in.a);
    io.ld(rk.y3 + v * N, in.b);
    io.ld(rk.y4 + v * N, in.c);
  }
}
template <int RK, typename T, typename IO>
__device__ __forceinline__ void rk_got(const IO &io, RkIn<RK, T> &in) {
  if constexpr (RK == RK_RHS) return;
  if constexpr (!(RK == RK_LAST && sizeof(T) == 8)) io.got(in.q0);
  if constexpr (RK == RK_MID || RK == RK_LAST || RK == RK_YLAST) io.got(in.a);
  if constexpr (RK == RK_YLAST) {
    io.got(in.b);
    io.got(in.c);
  }
}

// the new state q1 of the last stage
template <int RK, typename T>
__device__ __forceinline__ void rk_new_state(const RkArgs<T> &rk, const T (&k)[PPT], const RkIn<RK, T> &in,
                                             double (&q1)[PPT]) {
  const double dt = rk.dt;
#pragma unroll
  for (int m = 0; m < PPT; ++m) {
    if constexpr (RK == RK_YLAST) {
      const double d = (in.a[m] - in.q0[m]) + __builtin_fma(2.0, in.b[m] - in.q0[m], in.c[m] - in.q0[m]);
      q1[m] = in.q0[m] + __builtin_fma(d, 1.0 / 3.0, dt / 6.0 * k[m]);
    } else if constexpr (sizeof(T) == 8) {
      q1[m] = in.a[m] + dt / 6.0 * double(k[m]);
    } else {
      q1[m] = in.q0[m] + (double(in.a[m]) + dt / 6.0 * double(k[m]));
    }
  }
}

template <int RK, typename T, typename IO>
__device__ __forceinline__ void rk_store(const RkArgs<T> &rk, int v, const T (&k)[PPT], const RkIn<RK, T> &in,
                                         const IO &io, long N, T *rhs) {
  if constexpr (RK == RK_RHS) {
    io.st(rhs + v * N, k);
  } else if constexpr (RK == RK_LAST || RK == RK_YLAST) {
    double q1[PPT];
    rk_new_state<RK, T>(rk, k, in, q1);
    io.st(rk.qn + v * N, q1);
  } else {
    double a[PPT];
    if constexpr (RK != RK_Y) {
      // the accumulator's value after this stage
      const double base = sizeof(T) == 8 ? 1.0 : 0.0;  // FP32: the increment alone
      const double dt = rk.dt;
#pragma unroll
      for (int m = 0; m < PPT; ++m)
        a[m] = RK == RK_FIRST ? base * in.q0[m] + dt / 6.0 * double(k[m]) : in.a[m] + dt / 3.0 * double(k[m]);
      io.st(rk.acc + v * N, a);
    }
#pragma unroll
    for (int m = 0; m < PPT; ++m) a[m] = in.q0[m] + rk.c * double(k[m]);
    io.st(rk.out + v * N, a);
  }
}

// RK_YLAST's new state with one kept stage input live at a time, for the
// sweeps that have no registers for three
template <typename IO>
__device__ __forceinline__ void rk_ylast(const RkArgs<double> &rk, int v, const double (&k)[PPT], const IO &io, long N,
                                         double (&q1)[PPT]) {
  double q0[PPT], d[PPT];
  asm volatile("" ::: "memory");
  io.ld(rk.qn + v * N, q0);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    double y[PPT];
    io.ld((j == 0 ? rk.y2 : (j == 1 ? rk.y3 : rk.y4)) + v * N, y);
    if (j == 0) io.got(q0);
    io.got(y);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const double e = y[m] - q0[m];
      d[m] = j == 0 ? e : __builtin_fma(j == 1 ? 2.0 : 1.0, e, d[m]);
    }
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int m = 0; m < PPT; ++m) q1[m] = q0[m] + __builtin_fma(d[m], 1.0 / 3.0, rk.dt / 6.0 * k[m]);
}

// the form chosen at run time (uniform), for the sweeps whose instances are
// not worth one per form; Y: the forms without an accumulator
template <bool Y, typename T, typename IO>
__device__ __forceinline__ void rk_update(int form, const RkArgs<T> &rk, int v, const T (&k)[PPT], const IO &io,
                                          long N, T *rhs) {
#define CRUNA_RK(F)                                 \
  {                                                 \
    RkIn<F, T> in;                                  \
    rk_load<F, T>(rk, v, io, N, in);                \
    rk_got<F, T>(io, in);                           \
    rk_store<F, T>(rk, v, k, in, io, N, rhs);       \
  }
  if (form == RK_RHS) CRUNA_RK(RK_RHS)
  else if constexpr (Y) {
    if (form == RK_Y) {
      CRUNA_RK(RK_Y)
    } else {
      double q1[PPT];
      rk_ylast(rk, v, k, io, N, q1);
      io.st(rk.qn + v * N, q1);
    }
  } else {
    if (form == RK_FIRST) CRUNA_RK(RK_FIRST)
    else if (form == RK_MID) CRUNA_RK(RK_MID)
    else CRUNA_RK(RK_LAST)
  }
#undef CRUNA_RK
}
template <bool Y, typename T, typename IO>
__device__ __forceinline__ void rk_final(const RkArgs<T> &rk, int v, const T (&k)[PPT], const IO &io, long N,
                                         double (&q1)[PPT]) {
  if constexpr (Y) {
    rk_ylast(rk, v, k, io, N, q1);
  } else {
    RkIn<RK_LAST, T> in;
    rk_load<RK_LAST, T>(rk, v, io, N, in);
    rk_got<RK_LAST, T>(io, in);
    rk_new_state<RK_LAST, T>(rk, k, in, q1);
  }
}

// ----------------------------------------------------------------------------
// S4 (z) / S5 (y) / S6 (x): viscous fluxes d/dx_d tau_{i d}; the x sweep also
// adds tau:grad(u) (ns_rho_rhou_p.f90:202-205) and finishes the stage.
// RK: the x sweep's stage update (RkForm).
// FF (x sweep of the last stage only): also apply filter_i1 to
// the new state before storing it (the x filter of the step loop, fused
// because the x sweep holds complete x-lines); fop is that filter.  A
// separate instance, so that the other stages do not carry the filter
// solve's registers.
// The viscous sweeps read only G and rhs, so the next stage input (qs_out)
// may overwrite the current one in place.
// GT: deformed grid: d/dxi_d (M(d,d) tau_id) = M(d,d) d/dxi_d tau_id, and the
// last sweep multiplies every equation by X_jacobian and the dissipation once
// more (ns_rho_rhou_p_grid_transform.f90:190-276).
// EV: d/dx_d (phi tau_id), times the stored 1/phi (ns_rho_rhou_p_ev_phi.f90:161-201).
template <typename T, int DIR, int FORM, int RK, bool FF, typename Lines>
__device__ __forceinline__ void sweep2_body(const ThreadPos &tp, T *__restrict__ rhs, const T *__restrict__ G,
                                            const Op<T> &op, const Op<T> &fop, const SweepGeom &g,
                                            const Phys &ph, long N, const RkArgs<T> &rk, const Metric<T> &mt,
                                            const T *__restrict__ force, const Penal<T> &pe, Lines &ln) {
  static_assert(!FF || RK == RK_LAST || RK == RK_YLAST, "the x filter follows the last stage");
  constexpr bool GT = FORM == RHS_GT, EV = FORM == RHS_EV;
  constexpr bool LAST = DIR == 0;
  const FieldIO<DIR, T> io(tp, g);
  const T ih = GT ? T(ph.inv_h[DIR]) * mt.m[DIR][tp.lidx] : T(ph.inv_h[DIR]);
  constexpr bool ST = stress_form<T, FORM>();
  T t1[PPT], t2[PPT], t3[PPT], diss[PPT];
  if constexpr (ST) {
    // tau_11, tau_12, tau_13 (x) or tau_22, tau_23 (y)
    if (LAST) io.ld(G, t1);
    io.ld(G + (LAST ? 3 : 1) * N, t2);
    io.ld(G + (LAST ? 4 : 5) * N, t3);
    if (LAST) {
      issue_loads();
      io.got(t1);
      io.got(t2);
      io.got(t3);
    }
  } else {
    T mu[PPT], ux[PPT], vy[PPT], wz[PPT], sa[PPT], sb[PPT];
    io.ld(G + 6 * N, mu);
    io.ld(G + 0 * N, ux);
    io.ld(G + 1 * N, vy);
    io.ld(G + 2 * N, wz);
    // x: s12 = u_y + v_x, s13 = u_z + w_x;  y: s12, s23 = v_z + w_y;  z: s13, s23
    io.ld(G + (DIR == 2 ? 4 : 3) * N, sa);
    io.ld(G + (DIR == 0 ? 4 : 5) * N, sb);
    issue_loads();
    io.got(mu);
    io.got(ux);
    io.got(vy);
    io.got(wz);
    io.got(sa);
    io.got(sb);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T md = -2.0 / 3.0 * mu[m] * (ux[m] + vy[m] + wz[m]);
      const T t11 = md + 2 * mu[m] * ux[m], t22 = md + 2 * mu[m] * vy[m], t33 = md + 2 * mu[m] * wz[m];
      if (DIR == 0) {
        t1[m] = t11;            // tau_11
        t2[m] = mu[m] * sa[m];  // tau_21
        t3[m] = mu[m] * sb[m];  // tau_31
        // tau_ij du_i/dx_j = tau_11 u_x + tau_22 v_y + tau_33 w_z + mu (s12^2 + s13^2 + s23^2)
        diss[m] = t11 * ux[m] + t22 * vy[m] + t33 * wz[m] + t2[m] * sa[m] + t3[m] * sb[m];
      } else if (DIR == 1) {
        t1[m] = mu[m] * sa[m];  // tau_12
        t2[m] = t22;            // tau_22
        t3[m] = mu[m] * sb[m];  // tau_32
      } else {
        t1[m] = mu[m] * sa[m];  // tau_13
        t2[m] = mu[m] * sb[m];  // tau_23
        t3[m] = t33;            // tau_33
      }
    }
    // the stresses now, so that mu and the gradients are not kept across
    // the solves below
    materialize(t1);
    materialize(t2);
    materialize(t3);
    if (LAST) {
      io.ld(G + 5 * N, sa);
      io.got(sa);
#pragma unroll
      for (int m = 0; m < PPT; ++m) diss[m] = diss[m] + (mu[m] * sa[m]) * sa[m];
      materialize(diss);
    }
  }
  T Jv[PPT];
  if (LAST && GT) {
    io.ld(mt.J, Jv);
    io.got(Jv);
  }
  // the last sweep's complete RHS of variable v: what its RK4 update reads is
  // loaded together with the RHS; on the final stage optionally the x filter
  // of the new state
  auto finish = [&](int v, T(&k)[PPT], const RkIn<RK, T> &in) {
    // force (apply_force, ns_rho_rhou_p.f90:212): an additive term of the
    // complete RHS, here the learned closure; null when there is none
    if (force) {
      T fv[PPT];
      io.ld(force + v * N, fv);
      io.got(fv);
#pragma unroll
      for (int m = 0; m < PPT; ++m) k[m] = k[m] + fv[m];
    }
    if constexpr (FF) {
      double a[PPT];
      rk_new_state<RK, T>(rk, k, in, a);
      T f[PPT], x[PPT];
#pragma unroll
      for (int m = 0; m < PPT; ++m) f[m] = T(a[m]);
      ln.bind(fop);
      ln.template solve<true>(fop, f, x);
      ln.bind(op);
      io.st(rk.qn + v * N, x);
    } else {
      rk_store<RK, T>(rk, v, k, in, io, N, rhs);
    }
  };
  if constexpr (LAST) {
    // k_1 = rhs_1 (times J) and the pressure's (gamma - 1) (bracket +
    // tau:grad(u)) (ns_rho_rhou_p.f90:200-209) are complete already: their
    // updates go first, which frees the dissipation's registers for the solves
    // (the last stage of the form without an accumulator reads four more
    // fields per variable: it takes the two one after the other)
    // (FP32 keeps its registers for occupancy: 256^3 0.508 -> 0.478 ms)
    constexpr bool BOTH = RK != RK_YLAST && sizeof(T) == 8;
    T k[PPT], e[PPT];
    RkIn<RK, T> in, ie;
    io.ld(rhs, k);
    rk_load<RK, T>(rk, 0, io, N, in);
    if (BOTH) {
      io.ld(rhs + 4 * N, e);
      rk_load<RK, T>(rk, 4, io, N, ie);
    }
    issue_loads();
    if (RK != RK_RHS || GT || force) {
      io.got(k);
      rk_got<RK, T>(io, in);
      if (GT) {
#pragma unroll
        for (int m = 0; m < PPT; ++m) k[m] = Jv[m] * k[m];
      }
      finish(0, k, in);
    }
    if (!BOTH) {
      asm volatile("" ::: "memory");
      io.ld(rhs + 4 * N, e);
      rk_load<RK, T>(rk, 4, io, N, ie);
    }
    io.got(e);
    rk_got<RK, T>(io, ie);
#pragma unroll
    for (int m = 0; m < PPT; ++m)
      e[m] = GT ? (Jv[m] * T(ph.gm1)) * (e[m] + Jv[m] * diss[m]) : T(ph.gm1) * (ST ? e[m] : e[m] + diss[m]);
    finish(4, e, ie);
    asm volatile("" ::: "memory");
  }
  T IP[PPT];
  if (EV) {  // phi tau_id inside the derivative, 1/phi on it
    T PH[PPT];
    io.ld(pe.phi, PH);
    io.ld(pe.inv_phi, IP);
    io.got(PH);
    io.got(IP);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      t1[m] = PH[m] * t1[m];
      t2[m] = PH[m] * t2[m];
      t3[m] = PH[m] * t3[m];
    }
  }
  // z/y: read-modify-write of the momentum accumulators; x: the complete RHS
  // of that variable and its RK4 update
  auto complete = [&](int v, const T(&x)[PPT], T(&k)[PPT], RkIn<RK, T> &in) {
    io.got(k);
    if constexpr (LAST) rk_got<RK, T>(io, in);
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      k[m] = k[m] + (EV ? IP[m] * (x[m] * ih) : x[m] * ih);
      if (LAST && GT) k[m] = Jv[m] * k[m];
    }
    if constexpr (LAST)
      finish(v, k, in);
    else
      io.st(rhs + v * N, k);
  };
  if constexpr (ST && !LAST) {
    T x[PPT], y[PPT], k[PPT], l[PPT];
    RkIn<RK, T> none{};
    io.ld(rhs + 2 * N, k);
    io.ld(rhs + 3 * N, l);
    ln.solve2(op, t2, x, t3, y);
    complete(2, x, k, none);
    complete(3, y, l, none);
    return;
  }
  {
    // two stresses at once (FP64), the first accumulator in flight meanwhile
    T x[PPT], y[PPT], k[PPT];
    RkIn<RK, T> in;
    constexpr bool EARLY = RK != RK_YLAST && sizeof(T) == 8;
    if (EARLY) {
      io.ld(rhs + N, k);
      if constexpr (LAST) rk_load<RK, T>(rk, 1, io, N, in);
    }
    auto first = [&] {
      asm volatile("" ::: "memory");
      if (!EARLY) {
        io.ld(rhs + N, k);
        if constexpr (LAST) rk_load<RK, T>(rk, 1, io, N, in);
      }
      complete(1, x, k, in);
    };
    auto second = [&] {
      asm volatile("" ::: "memory");
      io.ld(rhs + 2 * N, k);
      if constexpr (LAST) rk_load<RK, T>(rk, 2, io, N, in);
      complete(2, y, k, in);
    };
    if constexpr (LAST) {
      ln.pair(op, t1, x, first, [] {}, t2, y, second);
    } else {
      // (y and z: with an FP32 result used before the next solve, the shear
      // layer's y sweep took 219 us instead of 186)
      ln.solve2(op, t1, x, t2, y);
      first();
      second();
    }
  }
  {
    T x[PPT], k[PPT];
    RkIn<RK, T> in;
    asm volatile("" ::: "memory");
    constexpr bool EARLY = RK != RK_YLAST && sizeof(T) == 8;
    if (EARLY) {
      io.ld(rhs + 3 * N, k);
      if constexpr (LAST) rk_load<RK, T>(rk, 3, io, N, in);
    }
    ln.solve(op, t3, x);
    if (!EARLY) {
      asm volatile("" ::: "memory");
      io.ld(rhs + 3 * N, k);
      if constexpr (LAST) rk_load<RK, T>(rk, 3, io, N, in);
    }
    complete(3, x, k, in);
  }
}

template <typename T, int DIR, bool PER, int FORM, int RK, bool FF>
__global__ __launch_bounds__(sweep_nt<T>()) void k_sweep2(T *__restrict__ rhs, const T *__restrict__ G,
                                                          Op<T> op, Op<T> fop, SweepGeom g, Phys ph,
                                                          long N, RkArgs<T> rk, Metric<T> mt,
                                                          const T *__restrict__ force, Penal<T> pe) {
  const ThreadPos tp = thread_pos<DIR, DIR == 1>(g);
  auto ln = make_lines<T, PER, sweep_nt<T>()>(op, tp);
  sweep2_body<T, DIR, FORM, RK, FF>(tp, rhs, G, op, fop, g, ph, N, rk, mt, force, pe, ln);
}

// S3 + S4: the z first-derivative sweep and the z viscous sweep as one
// kernel over the same z-line tiles.  The z sweep is the last
// first-derivative sweep of a stage, so once a thread has completed the
// velocity gradients of its block (w_z, u_z + w_x, v_z + w_y) the stresses
// of the block are known and the viscous z derivatives can follow at once.
// FP64 Cartesian form: sweep12_z_stress.  FP32 Cartesian form: the gradients and
// the viscosity stay in registers and the momentum RHS in LDS between the two
// parts (ZCarry), so the viscous part reads only u_x and v_y and writes the
// momentum RHS once.  The deformed-grid and penalised forms run the two sweep
// bodies one after the other.
template <typename T, typename Lines>
__device__ __forceinline__ void viscous_z_carry(const ThreadPos &tp, T *__restrict__ rhs, const T *__restrict__ G,
                                                const Op<T> &op, const SweepGeom &g, const Phys &ph, long N,
                                                Lines &ln, const ZCarry<T> &zc) {
  const long B = tp.base, PS = g.PS;
  const T ih = T(ph.inv_h[2]);
  T t1[PPT], t2[PPT], t3[PPT];
  {
    T ux[PPT], vy[PPT];
    ld<2>(G + 0 * N, B, PS, ux);
    ld<2>(G + 1 * N, B, PS, vy);
    issue_loads();
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
      const T mu = zc.mu[m], wz = zc.wz[m];
      const T md = -2.0 / 3.0 * mu * (ux[m] + vy[m] + wz);
      t1[m] = mu * zc.s13[m];  // tau_13
      t2[m] = mu * zc.s23[m];  // tau_23
      t3[m] = md + 2 * mu * wz;  // tau_33
    }
  }
  T x[PPT], y[PPT];
  auto put = [&](int i, T(&v)[PPT]) {
#pragma unroll
    for (int m = 0; m < PPT; ++m) v[m] = zc.mom(i, m) + v[m] * ih;
    st<2>(rhs + (1 + i) * N, B, PS, v);
  };
  ln.pair(op, t1, x, [&] { put(0, x); }, [] {}, t2, y, [&] { put(1, y); });
  ln.solve(op, t3, x);
  put(2, x);
}

template <typename T, typename Q, bool PER, int FORM>
__global__ __launch_bounds__(NT) void k_sweep12_z(const Q *__restrict__ qs, T *__restrict__ rhs,
                                                   T *__restrict__ G, Op<T> op, SweepGeom g, Phys ph,
                                                   long N, Metric<T> mt, Penal<T> pe) {
  const ThreadPos tp = thread_pos<2>(g);
  auto ln = make_lines<T, PER>(op, tp);
  if constexpr (stress_form<T, FORM>()) {
    sweep12_z_stress(tp, qs, rhs, G, op, g, ph, N, ln);
  } else if constexpr (FORM == RHS_CART) {
    __shared__ T mom[3][PPT][NT];
    ZCarry<T> zc;
    zc.slots = mom;
    sweep1_body<T, Q, 2, FORM, true>(tp, qs, rhs, G, op, g, ph, N, mt, pe, ln, &zc);
    viscous_z_carry<T>(tp, rhs, G, op, g, ph, N, ln, zc);
  } else {
    sweep1_body<T, Q, 2, FORM>(tp, qs, rhs, G, op, g, ph, N, mt, pe, ln);
    asm volatile("" ::: "memory");
    sweep2_body<T, 2, FORM, RK_RHS, false>(tp, rhs, G, op, op, g, ph, N, RkArgs<T>{}, mt, nullptr, pe, ln);
  }
}


// ----------------------------------------------------------------------------
// Single derivative (Dx1/2/3) of one field: out = (B^-1 A in) / h.
template <typename T, int DIR, bool PER>
__global__ __launch_bounds__(NT) void k_diff(const T *__restrict__ in, T *__restrict__ out,
                                             Op<T> op, SweepGeom g, double inv_h) {
  const ThreadPos tp = thread_pos<DIR>(g);
  auto ln = make_lines<T, PER>(op, tp);
  const FieldIO<DIR, T> io(tp, g);
  T f[PPT], x[PPT];
  io.ld(in, f);
  io.got(f);
  ln.solve(op, f, x);
#pragma unroll
  for (int m = 0; m < PPT; ++m) x[m] = x[m] * T(inv_h);
  io.st(out, x);
}

// Filter of nv fields in place (filter_4d): q = B_f^-1 A_f q per field.
template <typename T>
constexpr int filter_nt() { return sizeof(T) == 4 ? NT_FILTER32 : NT; }

// src: the fields to filter (FP64, or the compute precision); q64: where
// the filtered FP64 fields go (null: nowhere); copy: the filtered fields in
// the compute precision (null: nowhere).  src may be q64 or copy (in place:
// every thread loads its block before the line solve that the stores follow).
template <typename T, int DIR, typename S, typename LOp, typename Lines>
__device__ __forceinline__ void filter_body(const ThreadPos &tp, const S *src, double *q64, const LOp &op,
                                            const SweepGeom &g, long N, int nv, T *copy, Lines &ln) {
  const FieldIO<DIR, T> io(tp, g, Lines::dynamic_bytes(blockDim.x));
  double a[PPT];
  io.ld(src, a);
  for (int v = 0; v < nv; ++v) {
    T f[PPT], x[PPT];
    io.got(a);
#pragma unroll
    for (int m = 0; m < PPT; ++m) f[m] = T(a[m]);
    // the next field's loads fly while this one is filtered
    if (v + 1 < nv) io.ld(src + (v + 1) * N, a);
    ln.template solve<true>(op, f, x);
    if (q64) io.st(q64 + v * N, x);
    // the filtered state in the compute precision, when the next RK stage
    // or filter pass reads it (it equals the FP64 value converted back)
    if (copy) io.st(copy + v * N, x);
  }
}

template <typename T, int DIR, bool PER, typename S>
__global__ __launch_bounds__(filter_nt<T>()) void k_filter(const S *src, double *q64, Op<T> op, SweepGeom g,
                                                           long N, int nv, T *copy) {
  const ThreadPos tp = thread_pos<DIR>(g);
  auto ln = make_lines<T, PER, filter_nt<T>()>(op, tp);
  filter_body<T, DIR, S>(tp, src, q64, op, g, N, nv, copy, ln);
}

// The FP64 filter on the cyclic reduction, for the filter parameters that the
// recursions do not take (HostRecOp::usable).
template <int DIR, bool PER>
__global__ __launch_bounds__(NT) void k_filter_cr(const double *src, double *q64, LineOp<double> op, SweepGeom g,
                                                  long N, int nv) {
  __shared__ LineLds<double> lds;
  const ThreadPos tp = thread_pos<DIR>(g);
  CrLines<double, PER, NT> ln{lds, tp};
  filter_body<double, DIR, double>(tp, src, q64, op, g, N, nv, (double *)nullptr, ln);
}

}  // namespace cruna
