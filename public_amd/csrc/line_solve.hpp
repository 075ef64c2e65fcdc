// Device side of the block-partitioned line solve (tables: line_ops.hpp).
//
// A work-group owns TL complete grid lines along one direction; each thread
// owns one block of PPT = 8 consecutive points of one line (register
// resident).  Cross-thread traffic goes through LDS only for the explicit
// stencil halo (3 values per side) and the 2-unknown-per-block reduced
// system, so a derivative costs ~4 LDS accesses per point instead of the
// ~30 of a point-wise parallel cyclic reduction.  On periodic lines every
// table entry is the same for all threads and is read with scalar loads.
#pragma once

#include <hip/hip_runtime.h>

#include "line_ops.hpp"
#include "line_rec.hpp"

namespace cruna {

constexpr int NT = 512;  // max threads per work-group of the RHS sweeps
// the FP32 filter's and Cartesian sweeps' work-groups take up to 32 y/z lines
// (128-byte rows of floats)
constexpr int NT_FILTER32 = 1024;
constexpr int NT_SWEEP32 = 1024;

template <typename T>
struct LineOp {
  const T *I;  // [NI] interior blocks: stencil + local Thomas factors
  const T *M;  // [NTYPES][PPT][FE]  dense local operators: first, interior, last, before last
  const T *L;  // [NTYPES][PPT]
  const T *R;  // [NTYPES][PPT]
  const T *W;  // [K][nw][12]
  int n, NB, K, per;
  int spec2;   // open line: block NB-2 uses its own dense operator (type 3)
};

// Sweep geometry: which lines a work-group owns and where they live in HBM.
struct SweepGeom {
  int dir;        // 0: x (contiguous lines), 1: y, 2: z
  int n;          // line length
  int NB;         // blocks per line (n / PPT)
  int TL;         // lines per work-group
  int n1, n2, n3;
  long PS;        // distance between consecutive line points in memory
  int ntiles;     // work-groups in the grid
  int ntiles_in;  // (y/z) tiles along i
  long lines;     // batched launches: lines of the direction, taken TL at a time
  int back;       // first x sweep and second y sweep walk their tiles backwards
};

// Thread placement inside a tile.  The LDS slot of a (line, block) pair is the
// thread index; BS / LS are the slot strides between blocks / lines.
struct ThreadPos {
  int l, b;        // line in tile, block in line
  int BS, LS;
  long base;       // element offset of this thread's first point
  long lidx;       // index of the line in the plane across it: j + n2 k (x), i + n1 k (y), i + n1 j (z)
  bool wave_line;  // every line of the tile lies inside one wavefront
};

// Work-groups are dealt round-robin to the 8 XCDs; map consecutive tiles to the
// same XCD so that tiles sharing cache lines meet in the same L2.  rev: each
// XCD walks its tiles backwards.
__device__ inline int xcd_tile(int bid, int ntiles, bool rev = false) {
  if (ntiles % 8 != 0) return rev ? ntiles - 1 - bid : bid;
  const int per = ntiles / 8, t = bid / 8;
  return (bid % 8) * per + (rev ? per - 1 - t : t);
}

// Element offset of an idle thread's block: 2^28 FP64 elements is the 2 GiB
// buffer extent of the sweeps' field accesses (the host keeps every field
// below it), so an idle thread's loads return zero and its stores are dropped
// by the buffer range check.  FP64 fields only (the batched launches).
constexpr long IDLE_BASE = 1L << 28;

// Placement in tile `tile` of a sweep of geometry g (the launch has exactly
// TL x NB threads per work-group).
// BATCH (a batched launch over members of several sizes): tile t holds lines
// t*TL .. t*TL+TL-1 of the direction in line order (x: j + n2 k; y: i + n1 k;
// z: i + n1 j), so that a tile of any TL fills its work-group; the work-group
// may be larger than the tile, and the threads beyond it and the lines past
// the member's last line are idle: their block lies at IDLE_BASE and their
// exchange slots are those of block 0 of line 0, which they only read.
template <int DIR, bool BATCH = false>
__device__ inline ThreadPos thread_pos_tile(const SweepGeom &g, int tile) {
  ThreadPos t;
  const int tid = threadIdx.x;
  if (DIR == 0) {
    t.b = tid % g.NB;
    t.l = tid / g.NB;
    t.BS = 1;
    t.LS = g.NB;
    // x-lines take NB consecutive threads: with NB dividing the wavefront
    // size no line straddles two wavefronts
    t.wave_line = (64 % g.NB) == 0;
  } else {
    t.l = tid % g.TL;
    t.b = tid / g.TL;
    t.BS = g.TL;
    t.LS = 1;
    t.wave_line = false;
  }
  const long line = (long)tile * g.TL + t.l;
  if (BATCH && (tid >= g.TL * g.NB || line >= g.lines)) {
    t.l = 0;
    t.b = 0;
    t.base = IDLE_BASE;
    t.lidx = 0;
    return t;
  }
  if (DIR == 0) {
    t.base = line * g.n1 + (long)t.b * PPT;
    t.lidx = line;
  } else {
    long i, o;  // o: k for y-lines, j for z-lines
    if (BATCH) {
      // a member's lines are fewer than 2^31
      i = int(line) % g.n1;
      o = int(line) / g.n1;
    } else {
      i = (long)(tile % g.ntiles_in) * g.TL + t.l;
      o = tile / g.ntiles_in;
    }
    const long off = (DIR == 1) ? i + (long)g.n1 * g.n2 * o : i + (long)g.n1 * o;
    t.base = off + (long)t.b * PPT * g.PS;
    t.lidx = i + (long)g.n1 * o;
  }
  return t;
}

// (BACK: a sweep that follows one over the same planes and, where g.back is
// set, walks them backwards)
template <int DIR, bool BACK = false>
__device__ inline ThreadPos thread_pos(const SweepGeom &g) {
  return thread_pos_tile<DIR>(g, xcd_tile(blockIdx.x, g.ntiles, BACK && g.back));
}

// Work-group barrier that orders LDS traffic only.  __syncthreads() also waits
// for every outstanding global load, which would drain the prefetches the
// sweeps issue ahead of a line solve; this barrier leaves them in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Synchronisation point of the line engine: when each line lives inside one
// wavefront, the LDS exchange only has to be ordered within the wavefront
// (its LDS operations complete in issue order), so no work-group barrier is
// needed.
__device__ __forceinline__ void line_sync(bool wave_line) {
  if (wave_line) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  } else {
    lds_barrier();
  }
}

// LDS scratch of one work-group for the line engine, for up to NTM threads,
// indexed [value][thread slot]: consecutive lanes touch consecutive words
// (a thread-major [slot][value] layout put lanes 6 or 2 values apart, which
// the bank-conflict counters showed stalling every exchange).
template <typename T, int NTM = NT>
struct LineLds {
  T halo[2 * HALO][NTM];
  T z[2][2][NTM];
};

// x = B^-1 A f on the thread's block (unit spacing; the caller scales by 1/h).
// All threads of the work-group must call it together (barriers inside).
// Opaque copy of a uniform pointer: keeps the compiler from hoisting the table
// reads of one solve out of the surrounding sweep (which would pin ~130 table
// values in registers for the whole kernel); each solve re-reads them through
// the scalar cache instead.
// Tables are never written while a kernel runs, so uniform table reads may go
// through the scalar data cache: a pointer into the constant address space
// tells the compiler so.
template <typename T>
using cptr = const __attribute__((address_space(4))) T *;

template <typename T>
__device__ __forceinline__ cptr<T> launder_uniform(const T *p) {
  asm volatile("" : "+s"(p));
  return (cptr<T>)(p);
}

template <typename T, bool PER, int NTM>
__device__ __forceinline__ void line_solve(const LineOp<T> &op, LineLds<T, NTM> &s, const ThreadPos &tp,
                                           const T (&f)[PPT], T (&x)[PPT]) {
  const int tid = threadIdx.x;
  const int NB = op.NB;
  const int b = tp.b;
  // 1. halo exchange
#pragma unroll
  for (int m = 0; m < HALO; ++m) {
    s.halo[m][tid] = f[m];
    s.halo[HALO + m][tid] = f[PPT - HALO + m];
  }
  line_sync(tp.wave_line);
  const bool hasL = PER || b > 0;
  const bool hasR = PER || b < NB - 1;
  const int bl = b == 0 ? NB - 1 : b - 1;
  const int br = b == NB - 1 ? 0 : b + 1;
  const int sl = tp.l * tp.LS + bl * tp.BS;
  const int sr = tp.l * tp.LS + br * tp.BS;
  T fe[FE];
#pragma unroll
  for (int m = 0; m < HALO; ++m) {
    fe[m] = hasL ? s.halo[HALO + m][sl] : T(0);
    fe[HALO + PPT + m] = hasR ? s.halo[m][sr] : T(0);
  }
#pragma unroll
  for (int m = 0; m < PPT; ++m) fe[HALO + m] = f[m];
  // 2. local operator y = T_b^-1 A_b f: explicit stencil and an 8-point
  //    Thomas solve for interior blocks (every block of a periodic line); the
  //    two end blocks of an open line use their dense operator instead.
  T y[PPT];
  int ty = 1;
  {
    const cptr<T> I = launder_uniform(op.I);
    const T c0 = I[0], c1 = I[1], c2 = I[2], c3 = I[3], sg = I[4];
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      const T d1 = fe[HALO + i + 1] + sg * fe[HALO + i - 1];
      const T d2 = fe[HALO + i + 2] + sg * fe[HALO + i - 2];
      const T d3 = fe[HALO + i + 3] + sg * fe[HALO + i - 3];
      y[i] = c0 * fe[HALO + i] + c1 * d1 + c2 * d2 + c3 * d3;
    }
#pragma unroll
    for (int i = 1; i < PPT; ++i) y[i] = y[i] - I[4 + i] * y[i - 1];
    const T up = I[20];
    y[PPT - 1] = y[PPT - 1] * I[12 + PPT - 1];
#pragma unroll
    for (int i = PPT - 2; i >= 0; --i) y[i] = (y[i] - up * y[i + 1]) * I[12 + i];
  }
  if (!PER) {
    // the end blocks of an open line: one pass per block type present in the
    // wavefront, with that type's operator read through the scalar cache
    // (uniform), so that its 14 coefficients per row take no vector registers
    ty = b == 0 ? 0 : (b == NB - 1 ? 2 : ((b == NB - 2 && op.spec2) ? 3 : 1));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t == 1) continue;
      if (__builtin_amdgcn_ballot_w64(ty == t) == 0) continue;
      const cptr<T> Mb = launder_uniform(op.M + t * PPT * FE);
#pragma unroll 1
      for (int r = 0; r < PPT; ++r) {
        T acc = T(0);
#pragma unroll
        for (int j = 0; j < FE; ++j) acc += Mb[r * FE + j] * fe[j];
#pragma unroll
        for (int q = 0; q < PPT; ++q)
          if (q == r && ty == t) y[q] = acc;
      }
    }
  }
  // 3. reduced 2x2 block system by cyclic reduction over blocks
  T z0 = y[0], z1 = y[PPT - 1];
  int cur = 0;
  s.z[0][0][tid] = z0;
  s.z[0][1][tid] = z1;
  for (int k = 0; k < op.K; ++k) {
    line_sync(tp.wave_line);
    const int st = 1 << k;
    const bool hm = PER || b - st >= 0;
    const bool hp = PER || b + st < NB;
    int bm = b - st, bp = b + st;
    if (PER) {
      const int sr = st % NB;  // wave-uniform
      bm = b - sr;
      bm = bm < 0 ? bm + NB : bm;
      bp = b + sr;
      bp = bp >= NB ? bp - NB : bp;
    } else {
      bm = hm ? bm : b;
      bp = hp ? bp : b;
    }
    const int sm = tp.l * tp.LS + bm * tp.BS;
    const int sp = tp.l * tp.LS + bp * tp.BS;
    const T m0 = hm ? s.z[cur][0][sm] : T(0), m1 = hm ? s.z[cur][1][sm] : T(0);
    const T p0 = hp ? s.z[cur][0][sp] : T(0), p1 = hp ? s.z[cur][1][sp] : T(0);
    T w[12];
    if (PER) {
      const cptr<T> opW = launder_uniform(op.W);
#pragma unroll
      for (int i = 0; i < 12; ++i) w[i] = opW[k * 12 + i];
    } else {
#pragma unroll
      for (int i = 0; i < 12; ++i) w[i] = op.W[(k * NB + b) * 12 + i];
    }
    const T n0 = w[0] * z0 + w[1] * z1 + w[4] * m0 + w[5] * m1 + w[8] * p0 + w[9] * p1;
    const T n1 = w[2] * z0 + w[3] * z1 + w[6] * m0 + w[7] * m1 + w[10] * p0 + w[11] * p1;
    z0 = n0;
    z1 = n1;
    cur ^= 1;
    s.z[cur][0][tid] = z0;
    s.z[cur][1][tid] = z1;
  }
  line_sync(tp.wave_line);
  const T xl = hasL ? s.z[cur][1][sl] : T(0);
  const T xf = hasR ? s.z[cur][0][sr] : T(0);
  if (PER || ty == 1) {
    const cptr<T> opL = launder_uniform(op.L);
    const cptr<T> opR = launder_uniform(op.R);
#pragma unroll
    for (int r = 0; r < PPT; ++r) x[r] = y[r] + opL[PPT + r] * xl + opR[PPT + r] * xf;
  } else {
#pragma unroll
    for (int r = 0; r < PPT; ++r) x[r] = y[r];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (__builtin_amdgcn_ballot_w64(ty == t) == 0) continue;
      const cptr<T> L = launder_uniform(op.L + t * PPT);
      const cptr<T> R = launder_uniform(op.R + t * PPT);
#pragma unroll
      for (int r = 0; r < PPT; ++r) {
        const T v = y[r] + L[r] * xl + R[r] * xf;
        if (ty == t) x[r] = v;
      }
    }
  }
}

// ----------------------------------------------------------------------------
// FP64 engine (line_rec.hpp: the recursions, why and what they cost).

// LDS of the engine: REC_STRIDE doubles per thread (and a slot of zeros, what
// lies beyond an open line), value k of slot t at t REC_STRIDE + k: the halo
// values (2 H per field: two derivative fields with H = 2, or one filter field
// with H = 3), then u_L and x_F of up to two fields.  Every solve of a kernel,
// derivative or filter, keeps u_L and x_F in the same places: a value of one
// solve is rewritten by the next only after a barrier that follows its last
// read (halo: read before the second barrier, u_L before the third, x_F before
// the next solve's first).  The odd stride spreads consecutive lanes over all
// banks, and with the slots' addresses kept per thread every value is an
// immediate offset away.  Dynamic LDS, so that a work-group takes what its own
// size needs.
constexpr int REC_STRIDE = 13, REC_HALO = 8, REC_UL = 8, REC_XF = 10;
constexpr int REC_TEND = REC_ROWS * FE + 2 * PPT, REC_TSCAL = 2 * REC_TEND, REC_TAB = REC_TSCAL + 6;
// (a multiple of 16: what follows is accessed in 16-byte pieces)
__host__ __device__ inline size_t rec_lds_bytes(int threads) {
  return ((size_t)((threads + 1) * REC_STRIDE + REC_TAB) * sizeof(double) + 15) / 16 * 16;
}

template <typename T>
struct OpOf {
  typedef LineOp<T> type;
};
template <>
struct OpOf<double> {
  typedef RecOp type;
};
template <typename T>
using Op = typename OpOf<T>::type;

// The engine's arithmetic is written with explicit fused multiply-adds and
// contracts nothing else (also not with the operands' own products), so that
// a line gives the same bits in every kernel that it is inlined into.

// The lines of a work-group: solve(op, f, x) is x = B^-1 A f on the thread's
// block, solve2 two independent fields at once (all threads together, in the
// same order).  pair is two solves whose results are used at once, use1() and
// use2(), make2() preparing the second's input: CR, the cyclic reduction above,
// takes the fields one after the other, and no result or input of the second
// lives during the first; the recursions take both at once.  (With CR's
// results used after both solves, the FP32 first-derivative sweeps took 7 to
// 10 more registers, one wavefront per SIMD less, and the FP32-mixed step of an
// open 192^3 box 4 % longer.)
template <typename T, bool PER, int NTM>
struct CrLines {
  LineLds<T, NTM> &lds;
  const ThreadPos &tp;
  // dynamic LDS that the engine takes (its own is static)
  __host__ __device__ static size_t dynamic_bytes(int) { return 0; }
  template <bool FILT = false>
  __device__ __forceinline__ void solve(const LineOp<T> &op, const T (&f)[PPT], T (&x)[PPT]) {
    line_solve<T, PER>(op, lds, tp, f, x);
  }
  __device__ __forceinline__ void solve2(const LineOp<T> &op, const T (&f1)[PPT], T (&x1)[PPT], const T (&f2)[PPT],
                                         T (&x2)[PPT]) {
    line_solve<T, PER>(op, lds, tp, f1, x1);
    line_solve<T, PER>(op, lds, tp, f2, x2);
  }
  template <typename U1, typename M2, typename U2>
  __device__ __forceinline__ void pair(const LineOp<T> &op, const T (&f1)[PPT], T (&x1)[PPT], U1 use1, M2 make2,
                                       const T (&f2)[PPT], T (&x2)[PPT], U2 use2) {
    line_solve<T, PER>(op, lds, tp, f1, x1);
    use1();
    make2();
    line_solve<T, PER>(op, lds, tp, f2, x2);
    use2();
  }
  __device__ __forceinline__ void bind(const LineOp<T> &) {}
};

template <bool PER>
struct RecLines {
  __host__ __device__ static size_t dynamic_bytes(int threads) { return rec_lds_bytes(threads); }
  char *lds;                   // dynamic LDS
  int own;                     // byte offset of the thread's slot
  int lf[REC_WIN], rt[REC_WIN];  // slots of blocks b-1, b-2, ... and b+1, b+2, ...
  int b, NB, BS, line;         // block, blocks per line, slot stride of blocks, slot of block 0
  int nthreads;
  bool wave_line;
  double pwl, pwr;             // open: mu^(8 b - pf), mu^(n-1 - (8 b - pf) - 7)
  static constexpr int TAB_REGS = 1;
  double tv[TAB_REGS];         // open: entries of the closure table on their way to LDS
  bool pending = false;
  int keep[PPT];               // open: 0 for the thread's padding points, else all bits

  static constexpr int SLOT = REC_STRIDE * int(sizeof(double));
  __device__ __forceinline__ double get(int slot, int cell) const {
    return *reinterpret_cast<const double *>(lds + slot + cell * int(sizeof(double)));
  }
  __device__ __forceinline__ void put(int cell, double v) const {
    *reinterpret_cast<double *>(lds + own + cell * int(sizeof(double))) = v;
  }
  // slot of block t of the thread's line, 0 <= t < NB
  __device__ __forceinline__ int slot_of(int t) const { return (line + t * BS) * SLOT; }

  __device__ __forceinline__ RecLines(char *mem, const RecOp &op, const ThreadPos &tp) : lds(mem) {
    b = tp.b;
    NB = op.NB;
    BS = tp.BS;
    line = tp.l * tp.LS;
    nthreads = blockDim.x;
    wave_line = tp.wave_line;
    own = int(threadIdx.x) * SLOT;
    const int zero = nthreads * SLOT;
    int l = b, r = b;
#pragma unroll
    for (int m = 0; m < REC_WIN; ++m) {
      --l;
      ++r;
      if (PER) {
        l = l < 0 ? l + NB : l;
        r = r >= NB ? r - NB : r;
        lf[m] = slot_of(l);
        rt[m] = slot_of(r);
      } else {
        lf[m] = l >= 0 ? slot_of(l) : zero;
        rt[m] = r < NB ? slot_of(r) : zero;
      }
    }
    if (!PER) {
      for (int t = threadIdx.x; t < REC_STRIDE; t += nthreads)
        *reinterpret_cast<double *>(lds + zero + t * int(sizeof(double))) = 0.0;
      bind(op);
    }
  }
  // the closure table and powers of mu of an open line's op (the constructor
  // binds its own): loads issued here, stored to LDS by the next solve
  __device__ __forceinline__ void bind(const RecOp &op) {
    if (!PER) {
      pwl = op.tab[REC_PW + 2 * b];
      pwr = op.tab[REC_PW + 2 * b + 1];
      const int pad = (b == 0 ? op.zrow[0] : 0) | (b == NB - 1 ? op.zrow[1] : 0);
#pragma unroll
      for (int r = 0; r < PPT; ++r) keep[r] = ((pad >> r) & 1) - 1;
#pragma unroll
      for (int k = 0; k < TAB_REGS; ++k) {
        const int t = int(threadIdx.x) + k * nthreads;
        tv[k] = t < REC_TAB ? table_entry(op, t) : 0.0;
      }
      pending = true;
    }
  }
  // entry t of the closure table
  static __device__ __forceinline__ double table_entry(const RecOp &op, int t) {
    if (t >= REC_TSCAL) return op.tab[REC_SCAL + t - REC_TSCAL];
    const int e = t >= REC_TEND ? 1 : 0, o = t - e * REC_TEND;
    if (o >= REC_ROWS * FE) return op.tab[e * REC_END + PPT * FE + o - REC_ROWS * FE];
    const int r = (op.rows[e] >> (4 * (o / FE))) & 15;
    return r < PPT ? op.tab[e * REC_END + r * FE + o % FE] : 0.0;
  }
  __device__ __forceinline__ void store_table(const RecOp &op) {
    lds_barrier();  // the last op's table has been read
    double *tab = reinterpret_cast<double *>(lds + (nthreads + 1) * SLOT);
#pragma unroll
    for (int k = 0; k < TAB_REGS; ++k) {
      const int t = int(threadIdx.x) + k * nthreads;
      if (t < REC_TAB) tab[t] = tv[k];
    }
    for (int t = int(threadIdx.x) + TAB_REGS * nthreads; t < REC_TAB; t += nthreads) tab[t] = table_entry(op, t);
    lds_barrier();
    pending = false;
  }
  // the table of the thread's end of the line (any for the blocks between)
  __device__ __forceinline__ const double *end_table() const {
    return reinterpret_cast<const double *>(lds + (nthreads + 1) * SLOT) + (b == 0 ? 0 : REC_TEND);
  }
  // x where the thread's point is real, else y: two AND / BFI per value with
  // the masks kept per thread (compares and selects took four times the code)
  __device__ __forceinline__ double real_or(int r, double x, double y) const {
    const int2 a = __builtin_bit_cast(int2, x), c = __builtin_bit_cast(int2, y);
    return __builtin_bit_cast(double, int2{(a.x & keep[r]) | (c.x & ~keep[r]), (a.y & keep[r]) | (c.y & ~keep[r])});
  }
  __device__ __forceinline__ void zero_padding(double (&x)[PPT]) const {
#pragma unroll
    for (int r = 0; r < PPT; ++r) {
      const int2 a = __builtin_bit_cast(int2, x[r]);
      x[r] = __builtin_bit_cast(double, int2{a.x & keep[r], a.y & keep[r]});
    }
  }
  __device__ __forceinline__ void sync() const { line_sync(wave_line); }

  // sum_m rho^m value(block b -+ (1 + m)) of cell (the derivatives' mu never
  // needs more than REC_WIN terms)
  template <bool FILT>
  __device__ __forceinline__ double window(const RecOp &op, const int (&at)[REC_WIN], int dir, int cell) const {
#pragma clang fp contract(off)
    double v[REC_WIN];
#pragma unroll
    for (int m = 0; m < REC_WIN; ++m) v[m] = get(at[m], cell);
    if (!FILT || !op.slow) {
      double s = v[REC_WIN - 1];
#pragma unroll
      for (int m = REC_WIN - 2; m >= 0; --m) s = __builtin_fma(s, op.rho, v[m]);
      return s;
    }
    // slowly decaying filters: M terms, M at most the blocks of the line
    double s = 0.0;
    for (int m = op.M - 1; m >= 0; --m) {
      int t = b + dir * (1 + m);
      double u = 0.0;
      if (PER) {
        t = t < 0 ? t + NB : (t >= NB ? t - NB : t);
        u = get(slot_of(t), cell);
      } else if (t >= 0 && t < NB) {
        u = get(slot_of(t), cell);
      }
      s = __builtin_fma(s, op.rho, u);
    }
    return s * op.norm;
  }

  template <int NF, bool FILT>
  __device__ __forceinline__ void run(const RecOp &op, const double (&f)[NF][PPT], double (&x)[NF][PPT]) {
#pragma clang fp contract(off)
    constexpr int H = FILT ? 3 : 2, CELL = 2 * H;
    static_assert(NF * CELL <= REC_HALO && NF <= 2, "the fields' halo cells");
    if (!PER && pending) store_table(op);
    const bool end = !PER && (b == 0 || b == NB - 1);
    const bool padded = !PER && (op.zrow[0] | op.zrow[1]) != 0;
#pragma unroll
    for (int v = 0; v < NF; ++v)
#pragma unroll
      for (int m = 0; m < H; ++m) {
        put(v * CELL + m, f[v][m]);
        put(v * CELL + H + m, f[v][PPT - H + m]);
      }
    sync();
#pragma unroll
    for (int v = 0; v < NF; ++v) {
      double fe[PPT + 2 * H];
#pragma unroll
      for (int m = 0; m < H; ++m) {
        fe[m] = get(lf[0], v * CELL + H + m);
        fe[H + PPT + m] = get(rt[0], v * CELL + m);
      }
#pragma unroll
      for (int i = 0; i < PPT; ++i) fe[H + i] = f[v][i];
#pragma unroll
      for (int i = 0; i < PPT; ++i) {
        const double *e = fe + H + i;
        if (FILT)
          x[v][i] = __builtin_fma(op.s[0], e[0], __builtin_fma(op.s[1], e[1] + e[-1],
                                                              __builtin_fma(op.s[2], e[2] + e[-2], op.s[3] * (e[H] + e[-H]))));
        else
          x[v][i] = __builtin_fma(op.s[1], e[1] - e[-1], op.s[2] * (e[2] - e[-2]));
      }
      if (!PER) {
        // the closures' own rows and the padding of the two end blocks
        if (__builtin_amdgcn_ballot_w64(end) != 0) {
          const double *tab = end_table() + HALO - H;
          const int rows = b == 0 ? op.rows[0] : op.rows[1];
#pragma unroll 1
          for (int k = 0; k < op.nrow; ++k) {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < PPT + 2 * H; ++j) acc = __builtin_fma(tab[k * FE + j], fe[j], acc);
            const int r = end ? (rows >> (4 * k)) & 15 : 15;
#pragma unroll
            for (int q = 0; q < PPT; ++q) x[v][q] = q == r ? acc : x[v][q];
          }
          if (padded) zero_padding(x[v]);
        }
      }
#pragma unroll
      for (int i = 1; i < PPT; ++i) x[v][i] = __builtin_fma(op.mu, x[v][i - 1], x[v][i]);
      put(REC_UL + v, x[v][PPT - 1]);
    }
    sync();
#pragma unroll
    for (int v = 0; v < NF; ++v) {
      const double U = window<FILT>(op, lf, -1, REC_UL + v);
#pragma unroll
      for (int i = 0; i < PPT; ++i) x[v][i] = __builtin_fma(op.lp[i], U, x[v][i]);
      // nothing comes back from behind the last point
      if (padded && __builtin_amdgcn_ballot_w64(end) != 0) zero_padding(x[v]);
#pragma unroll
      for (int i = PPT - 2; i >= 0; --i) x[v][i] = __builtin_fma(op.mu, x[v][i + 1], x[v][i]);
      put(REC_XF + v, x[v][0]);
    }
    sync();
#pragma unroll
    for (int v = 0; v < NF; ++v) {
      const double X = window<FILT>(op, rt, +1, REC_XF + v);
#pragma unroll
      for (int i = 0; i < PPT; ++i) x[v][i] = __builtin_fma(op.lp[PPT - 1 - i], X, x[v][i]);
    }
    if (!PER) ends<NF, FILT>(op, f, x, end, padded);
  }

  // end corrections of an open line, then the padding rows
  template <int NF, bool FILT>
  __device__ __forceinline__ void ends(const RecOp &op, const double (&f)[NF][PPT], double (&x)[NF][PPT], bool end,
                                       bool padded) {
#pragma clang fp contract(off)
    const bool any = __builtin_amdgcn_ballot_w64(end) != 0;
    if (op.nend) {
      double kap[NF];
#pragma unroll
      for (int v = 0; v < NF; ++v) kap[v] = 0.0;
      if (any) {
        const double *c = end_table() + REC_ROWS * FE;
#pragma unroll
        for (int v = 0; v < NF; ++v) {
          double a = 0.0, k = 0.0;
#pragma unroll
          for (int r = 0; r < PPT; ++r) {
            a = __builtin_fma(c[r], x[v][r], a);
            k = __builtin_fma(c[PPT + r], x[v][r], k);
          }
          if (end) {
            put(REC_UL + v, a);  // u_L has been read (the exchange of x_F lies between)
            kap[v] = k;
          }
        }
      }
      sync();
      if (__builtin_amdgcn_ballot_w64(fabs(pwl) > 1e-19 || fabs(pwr) > 1e-19) != 0) {
        const double *t = reinterpret_cast<const double *>(lds + (nthreads + 1) * SLOT) + REC_TSCAL;
        const double gam = b == 0 ? t[4] : t[5];
        const int re = end ? (b == 0 ? op.rend[0] : op.rend[1]) : PPT;
#pragma unroll
        for (int v = 0; v < NF; ++v) {
          const double al = get(line * SLOT, REC_UL + v), ar = get(slot_of(NB - 1), REC_UL + v);
          const double sl = __builtin_fma(t[0], al, t[1] * ar), sr = __builtin_fma(t[2], ar, t[3] * al);
          const double l = sl * pwl, r = sr * pwr;
          x[v][0] += l;
          x[v][PPT - 1] += r;
#pragma unroll
          for (int i = 1; i < PPT; ++i) {
            x[v][i] = __builtin_fma(op.lp[i - 1], l, x[v][i]);
            x[v][PPT - 1 - i] = __builtin_fma(op.lp[i - 1], r, x[v][PPT - 1 - i]);
          }
          if (any) {
            const double k = __builtin_fma(gam, b == 0 ? sr : sl, kap[v]);
#pragma unroll
            for (int q = 0; q < PPT; ++q) x[v][q] = q == re ? x[v][q] + k : x[v][q];
          }
        }
      }
    }
    if (padded && any) {
#pragma unroll
      for (int v = 0; v < NF; ++v) {
        if (FILT) {
#pragma unroll
          for (int r = 0; r < PPT; ++r) x[v][r] = real_or(r, x[v][r], f[v][r]);
        } else {
          zero_padding(x[v]);
        }
      }
    }
  }

  template <bool FILT = false>
  __device__ __forceinline__ void solve(const RecOp &op, const double (&f)[PPT], double (&x)[PPT]) {
    double a[1][PPT], r[1][PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i) a[0][i] = f[i];
    run<1, FILT>(op, a, r);
#pragma unroll
    for (int i = 0; i < PPT; ++i) x[i] = r[0][i];
  }
  __device__ __forceinline__ void solve2(const RecOp &op, const double (&f1)[PPT], double (&x1)[PPT],
                                         const double (&f2)[PPT], double (&x2)[PPT]) {
    double a[2][PPT], r[2][PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      a[0][i] = f1[i];
      a[1][i] = f2[i];
    }
    run<2, false>(op, a, r);
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
      x1[i] = r[0][i];
      x2[i] = r[1][i];
    }
  }
  template <typename U1, typename M2, typename U2>
  __device__ __forceinline__ void pair(const RecOp &op, const double (&f1)[PPT], double (&x1)[PPT], U1 use1, M2 make2,
                                       const double (&f2)[PPT], double (&x2)[PPT], U2 use2) {
    make2();
    solve2(op, f1, x1, f2, x2);
    use1();
    use2();
  }
};

// The engine of a kernel in precision T (NTM: the largest work-group of the
// FP32 form's static LDS; FP64 launches pass rec_lds_bytes(threads))
extern __shared__ __align__(16) char line_dyn[];

template <typename T, bool PER, int NTM = NT>
__device__ __forceinline__ auto make_lines(const Op<T> &op, const ThreadPos &tp) {
  if constexpr (sizeof(T) == 8) {
    return RecLines<PER>(line_dyn, op, tp);
  } else {
    __shared__ LineLds<T, NTM> lds;
    return CrLines<T, PER, NTM>{lds, tp};
  }
}
// bytes of dynamic LDS that the engine takes in a work-group of `threads`
template <typename T>
size_t line_lds_bytes(int threads) {
  return sizeof(T) == 8 ? rec_lds_bytes(threads) : 0;
}

}  // namespace cruna
