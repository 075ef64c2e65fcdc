// Learned subfilter closure: a small 3-D CNN on a periodic S^3 grid, trained
// and evaluated with BF16 MFMA (FP32 accumulation).
//
// Network: 5 -> W -> W -> W -> 5 channels, 3x3x3 kernels with periodic
// padding, GELU (tanh form) after the three hidden layers.  Activations are
// stored channels-last, act[p][C] with p = i + S (j + S k) (+ S^3 b), and the
// channel counts are padded to multiples of 16 (zero weights and zero inputs
// in the padding), so every convolution is an implicit GEMM of 16x16 tiles:
//   forward       out[p][co] = b[co] + sum_t sum_ci in[p + o_t][ci] W[t][co][ci]
//   input grad    din[p][ci] = gelu'(z[p][ci]) sum_t sum_co dz[p - o_t][co] W[t][co][ci]
//   weight grad   dW[t][co][ci] = sum_p dz[p][co] in[p + o_t][ci]
// MFMA operand layouts (lane l of 64; both checked on the device):
// v_mfma_f32_16x16x16_bf16: A row l%16 holds K = 4(l/16)..+3, B column l%16
// holds K = 4(l/16)..+3; v_mfma_f32_16x16x32_bf16: the same with
// K = 8(l/16)..+7; both: D row 4(l/16)+r, column l%16, r = 0..3.
#pragma once

#include <hip/hip_runtime.h>

namespace cruna {

typedef unsigned short bf16;
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even (NaN stays NaN): the hardware's conversion
__device__ __forceinline__ bf16 to_bf16(float f) { return __builtin_bit_cast(bf16, (__bf16)f); }
__device__ __forceinline__ uint2 to_bf16(f32x4 v) {
  typedef __bf16 half4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint2, __builtin_convertvector(v, half4));
}
__device__ __forceinline__ float from_bf16(bf16 h) { return __uint_as_float((unsigned)h << 16); }

// GELU, tanh form: 0.5 z (1 + tanh(u)), u = c (z + a z^3), written with the
// logistic function s = 1 / (1 + exp(-2u)) (1 + tanh(u) = 2 s,
// 1 - tanh(u)^2 = 4 s (1 - s)) on the hardware exp2 and reciprocal:
//   gelu(z) = z s,   gelu'(z) = s + 2 z s (1 - s) c (1 + 3 a z^2)
__device__ __forceinline__ float gelu_sigma(float z) {
  const float c = 0.7978845608028654f, a = 0.044715f;
  const float u = c * (z + a * z * z * z);
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-2.8853900817779268f * u));  // 2 log2(e)
}
__device__ __forceinline__ float gelu(float z) { return z * gelu_sigma(z); }
__device__ __forceinline__ float gelu_grad(float z) {
  const float c = 0.7978845608028654f, a = 0.044715f;
  const float s = gelu_sigma(z);
  return s + 2.f * z * s * (1.f - s) * c * (1.f + 3.f * a * z * z);
}

// Geometry of a batch of boxes X x Y x Z, stored one after the other with
// p = i + X (j + Y k) + XYZ b: periodic boxes (a full field, wrapped at its
// faces) or crops whose outside reads as zero (a crop with a halo as wide as
// the network's reach gives exactly the periodic field's values at its
// centre).  Coordinates are found once per point with exact FP64 reciprocal
// division ((p + 1/2) / C is never within 1/(2C) of an integer).
struct ConvGeom {
  int X, Y, Z, periodic;
  double inv_x, inv_xy, inv_xyz;
};

struct Coord {
  int i, j, k;
  long base;  // index of the box's first point
};

__device__ __forceinline__ int exact_div(long p, double inv) { return (int)(((double)p + 0.5) * inv); }

__device__ __forceinline__ Coord coord_of(long p, const ConvGeom &g) {
  const long XY = (long)g.X * g.Y, XYZ = XY * g.Z;
  const int b = exact_div(p, g.inv_xyz);
  const long r = p - (long)b * XYZ;
  const int k = exact_div(r, g.inv_xy);
  const long r2 = r - (long)k * XY;
  const int j = exact_div(r2, g.inv_x);
  return Coord{(int)(r2 - (long)j * g.X), j, k, (long)b * XYZ};
}

enum ConvMode { CONV_GELU = 0, CONV_LINEAR = 1, CONV_BACKWARD = 2 };

// One convolution as an implicit GEMM on BF16 MFMA: out[p][co] over the 27
// taps and CK input channels of each point's neighbours.
// With 32 input channels a lane loads 16 bytes (channels 8(l/16)..+7) of a
// neighbour row per tap, the K = 32 operand of one v_mfma_f32_16x16x32_bf16;
// with 16 it loads 8 bytes for v_mfma_f32_16x16x16_bf16.
// CK: input (reduction) channels, CN: output channels.
//   CONV_GELU     : z = conv + bias; zsave <- bf16(z) (if set); out16 <- bf16(gelu(z))
//   CONV_LINEAR   : out32 <- conv + bias
//   CONV_BACKWARD : taps mirrored, W given as [t][CN][CK] of the transposed
//                   operator; out16 <- bf16(conv * gelu'(zin)) (zin: the
//                   pre-activations of this layer's input, CN channels)
// npts is a multiple of 64 and npts * 32 < 2^31 (checked by the host).
constexpr int CONV_TILES = 4;      // 16-point MFMA tiles per wavefront
constexpr int CONV_XCDS = 8;       // XCDs of the MI355X, each with its own L2
// The convolution with weights and input served from LDS: a work-group
// stages the layer's weights in LDS once and then walks tiles of 16 x 4 x 8 output points of one
// box (x, y, z; partial tiles at the box's far faces), loads each tile's
// input with a one-point halo, 18 x 6 x 10 points of CK channels, into LDS
// once (wrapped on periodic boxes, zero outside a crop), and takes all 27
// taps from there: each input row is read from L2 once per tile instead of
// once per tap; the next tile's rows are in flight (in registers) while a
// tile computes.  Wavefront w owns z-plane w of the tile and its 4 MFMA
// tiles are the plane's 4 x-rows of 16 points; it reuses every weight
// fragment for the 4 tiles, and each accumulator takes the taps in the
// order t = 9 dz + 3 dy + dx.  The work-groups are persistent: work-group g
// takes a contiguous range of tiles, the ranges of the work-groups on one
// XCD (g % 8) adjacent, so that neighbouring tiles share their halo rows in
// that XCD's L2.
constexpr int CT_X = 16, CT_Y = 4, CT_Z = 8;
constexpr int CT_THREADS = 64 * CT_Z;  // one wavefront per z-plane of the tile
constexpr int CH_X = CT_X + 2, CH_Y = CT_Y + 2, CH_Z = CT_Z + 2;
constexpr int CT_HALO = CH_X * CH_Y * CH_Z;  // input points per tile

template <int CK, int CN, int MODE>
__global__ __launch_bounds__(CT_THREADS) void k_conv_tile(const bf16 *__restrict__ in, const bf16 *__restrict__ W,
                                                   const float *__restrict__ bias, ConvGeom geo, long npts,
                                                   float *__restrict__ out32, bf16 *__restrict__ out16,
                                                   bf16 *__restrict__ zsave, const bf16 *__restrict__ zin) {
  // weight rows of CK channels: a fragment read (16 rows, 4 lane groups)
  // covers one contiguous run of LDS, free of bank conflicts
  __shared__ __align__(16) bf16 wl[27 * CN * CK];
  __shared__ __align__(16) bf16 xt[CT_HALO * CK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const bool per = geo.periodic != 0;
  const int X = geo.X, Y = geo.Y, Z = geo.Z;
  const long XY = (long)X * Y, XYZ = XY * Z;
  const int nbx = (X + CT_X - 1) / CT_X, nby = (Y + CT_Y - 1) / CT_Y, nbz = (Z + CT_Z - 1) / CT_Z;
  const int per_box = nbx * nby * nbz;
  const int ntiles = (int)(npts / XYZ) * per_box;
  // contiguous range of tiles of this work-group (see above)
  const int G = gridDim.x;
  const int slot = (blockIdx.x % CONV_XCDS) * ((G + CONV_XCDS - 1) / CONV_XCDS) + blockIdx.x / CONV_XCDS;
  const int chunk = (ntiles + G - 1) / G;
  const int t0 = slot * chunk, t1 = t0 + chunk < ntiles ? t0 + chunk : ntiles;
  constexpr int C8 = CK / 8;  // 16-byte pieces per input row
  constexpr int PIECES = CT_HALO * C8, PER_THREAD = (PIECES + CT_THREADS - 1) / CT_THREADS;
  // a tile's input rows: every load of the tile issued into registers
  // (the next tile's while the current one computes), then stored to LDS
  uint4 pre[PER_THREAD];
  auto fetch = [&](int tile) {
    const int b = tile / per_box, rem = tile % per_box;
    const int i0 = (rem % nbx) * CT_X, j0 = ((rem / nbx) % nby) * CT_Y, k0 = (rem / (nbx * nby)) * CT_Z;
    const long base = (long)b * XYZ;
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
      const int e = threadIdx.x + CT_THREADS * u;
      const int hp = e / C8, c8 = e % C8;
      int gi = i0 + hp % CH_X - 1, gj = j0 + (hp / CH_X) % CH_Y - 1, gk = k0 + hp / (CH_X * CH_Y) - 1;
      bool ok = e < PIECES;
      if (per) {
        gi = gi < 0 ? gi + X : (gi >= X ? gi - X : gi);
        gj = gj < 0 ? gj + Y : (gj >= Y ? gj - Y : gj);
        gk = gk < 0 ? gk + Z : (gk >= Z ? gk - Z : gk);
      } else {
        ok = ok && gi >= 0 && gi < X && gj >= 0 && gj < Y && gk >= 0 && gk < Z;
      }
      // points of a partial tile beyond the far face read a wrapped or zero
      // row: their outputs are not stored
      gi = gi < X ? gi : X - 1;
      gj = gj < Y ? gj : Y - 1;
      gk = gk < Z ? gk : Z - 1;
      const long gp = base + gi + X * ((long)gj + (long)Y * gk);
      pre[u] = ok ? *reinterpret_cast<const uint4 *>(in + gp * CK + c8 * 8) : uint4{0u, 0u, 0u, 0u};
    }
  };
  auto put = [&](bf16 *buf) {
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
      const int e = threadIdx.x + CT_THREADS * u;
      if (e < PIECES) *reinterpret_cast<uint4 *>(buf + (long)e * 8) = pre[u];
    }
  };
  {
    // the layer's weights, every load in flight together with the first tile's
    constexpr int WPIECES = 27 * CN * CK / 8, WPER = (WPIECES + CT_THREADS - 1) / CT_THREADS;
    uint4 v[WPER];
#pragma unroll
    for (int u = 0; u < WPER; ++u) {
      const int e = threadIdx.x + CT_THREADS * u;
      v[u] = e < WPIECES ? *reinterpret_cast<const uint4 *>(W + (long)e * 8) : uint4{0u, 0u, 0u, 0u};
    }
    if (t0 < t1) fetch(t0);
#pragma unroll
    for (int u = 0; u < WPER; ++u) {
      const int e = threadIdx.x + CT_THREADS * u;
      if (e < WPIECES) *reinterpret_cast<uint4 *>(wl + (long)e * 8) = v[u];
    }
  }
  f32x4 b4[CN / 16];
#pragma unroll
  for (int n = 0; n < CN / 16; ++n)
    b4[n] = MODE == CONV_BACKWARD ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4 *>(bias + n * 16 + 4 * kg);
  for (int tile = t0; tile < t1; ++tile) {
    __syncthreads();  // the previous tile's reads of xt are done
    put(xt);
    __syncthreads();
    if (tile + 1 < t1) fetch(tile + 1);
    const bf16 *x = xt;
    f32x4 acc[CONV_TILES][CN / 16];
#pragma unroll
    for (int j = 0; j < CONV_TILES; ++j)
#pragma unroll
      for (int n = 0; n < CN / 16; ++n) acc[j][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the 9 taps of each dz unrolled: the LDS reads of later taps issue
    // while the matrix cores work on earlier ones
#pragma unroll 1
    for (int dz = 0; dz < 3; ++dz)
#pragma unroll
      for (int dy = 0; dy < 3; ++dy)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const int t = 9 * dz + 3 * dy + dx;
          // neighbour (dx - 1, dy - 1, dz - 1), mirrored for the transposed operator
          const int ex = MODE == CONV_BACKWARD ? 2 - dx : dx, ey = MODE == CONV_BACKWARD ? 2 - dy : dy,
                    ez = MODE == CONV_BACKWARD ? 2 - dz : dz;
          const int row0 = ((wave + ez) * CH_Y + ey) * CH_X + r + ex;  // x-row j adds j * CH_X
          if constexpr (CK == 32) {
            uint4 a[CONV_TILES];
#pragma unroll
            for (int j = 0; j < CONV_TILES; ++j)
              a[j] = *reinterpret_cast<const uint4 *>(x + (row0 + j * CH_X) * CK + kg * 8);
#pragma unroll
            for (int n = 0; n < CN / 16; ++n) {
              const bf16x8 w = __builtin_bit_cast(
                  bf16x8, *reinterpret_cast<const uint4 *>(wl + (t * CN + n * 16 + r) * CK + kg * 8));
#pragma unroll
              for (int j = 0; j < CONV_TILES; ++j)
                acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8, a[j]), acc[j][n],
                                                                    0, 0, 0);
            }
          } else {
            static_assert(CK == 16, "16 or 32 input channels");
            bf16x4 a[CONV_TILES];
#pragma unroll
            for (int j = 0; j < CONV_TILES; ++j)
              a[j] = *reinterpret_cast<const bf16x4 *>(x + (row0 + j * CH_X) * CK + kg * 4);
#pragma unroll
            for (int n = 0; n < CN / 16; ++n) {
              const bf16x4 w = *reinterpret_cast<const bf16x4 *>(wl + (t * CN + n * 16 + r) * CK + kg * 4);
#pragma unroll
              for (int j = 0; j < CONV_TILES; ++j)
                acc[j][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, a[j], acc[j][n], 0, 0, 0);
            }
          }
        }
    const int b = tile / per_box, rem = tile % per_box;
    const int i0 = (rem % nbx) * CT_X, j0 = ((rem / nbx) % nby) * CT_Y, k0 = (rem / (nbx * nby)) * CT_Z;
    const long base = (long)b * XYZ;
    const int kk = k0 + wave;
    // a lane holds 4 consecutive channels of one point (channels are the matrix
    // rows): stores of 8 and 16 bytes.  With points as rows, single BF16 stores
    // and a rounding in integers the layers took 27 / 34 / 34 / 20 us at 64^3
    // (now 22 / 23 / 23 / 17); what bounds them is a tile's phases in turn.
    const int ii = i0 + r;
    const bool inside = ii < X && kk < Z;
#pragma unroll
    for (int j = 0; j < CONV_TILES; ++j) {
      const int jj = j0 + j;
      if (!inside || jj >= Y) continue;
      const long o0 = (base + ii + X * ((long)jj + (long)Y * kk)) * CN + 4 * kg;
#pragma unroll
      for (int n = 0; n < CN / 16; ++n) {
        const long o = o0 + n * 16;
        if (MODE == CONV_GELU) {
          const f32x4 z = acc[j][n] + b4[n];
          if (zsave) *reinterpret_cast<uint2 *>(zsave + o) = to_bf16(z);
          *reinterpret_cast<uint2 *>(out16 + o) = to_bf16(f32x4{gelu(z[0]), gelu(z[1]), gelu(z[2]), gelu(z[3])});
        } else if (MODE == CONV_LINEAR) {
          *reinterpret_cast<f32x4 *>(out32 + o) = acc[j][n] + b4[n];
        } else {
          const uint2 h = *reinterpret_cast<const uint2 *>(zin + o);
          f32x4 d;
#pragma unroll
          for (int rr = 0; rr < 4; ++rr)
            d[rr] = acc[j][n][rr] * gelu_grad(__uint_as_float(rr % 2 ? (rr / 2 ? h.y : h.x) & 0xffff0000u : (rr / 2 ? h.y : h.x) << 16));
          *reinterpret_cast<uint2 *>(out16 + o) = to_bf16(d);
        }
      }
    }
  }
}

// Weight gradient partials: work-group g sums dz[p][co] in[p + o_t][ci] over
// its tiles (16 x 4 x 8 points, as k_conv_tile's) into part[g][t][co][ci] for
// all 27 taps, as MFMA GEMMs with the points as reduction index.  A tile's dz and
// its input with a one-point halo are staged in LDS once, rows of channels as
// they lie in memory; the matrix operands, which run over points, come from
// the LDS transpose read (16 lanes read 4 rows of 16 channels and each gets the
// four values of its channel), so that a tap is nothing but another first row.
// Wavefront w takes the taps w, w + 8, ... and keeps their accumulators over all
// its tiles; wavefront 7 also sums dz (times ones) for the bias gradient.
// Bound by LDS reads (2 per channel block and 16 points) and by the staging of
// the next tile.  At 64^3 the 32 -> 32 layers take 40 us each, 16 -> 32 28 and
// 32 -> 16 30; a kernel that read and transposed every point once per tap took
// 217, 170 and 198.
constexpr int WG_MAX = 256;  // work-groups: one per CU (100 KB of LDS)

__device__ __forceinline__ bf16x4 read_points(const bf16 *p) {
  typedef __attribute__((address_space(3))) bf16x4 lds4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
}

template <int CI, int CO>
__global__ __launch_bounds__(CT_THREADS) void k_conv_wgrad(const bf16 *__restrict__ in, const bf16 *__restrict__ dz,
                                                          ConvGeom geo, long npts, float *__restrict__ part,
                                                          float *__restrict__ bpart) {
  constexpr int CT_PTS = CT_X * CT_Y * CT_Z, WAVES = CT_Z, TAPS = (27 + WAVES - 1) / WAVES;
  __shared__ __align__(16) bf16 dt[CT_PTS * CO];
  __shared__ __align__(16) bf16 xt[CT_HALO * CI];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const bool per = geo.periodic != 0;
  const int X = geo.X, Y = geo.Y, Z = geo.Z;
  const long XYZ = (long)X * Y * Z;
  const int nbx = (X + CT_X - 1) / CT_X, nby = (Y + CT_Y - 1) / CT_Y, nbz = (Z + CT_Z - 1) / CT_Z;
  const int per_box = nbx * nby * nbz;
  const int ntiles = (int)(npts / XYZ) * per_box;
  const int G = gridDim.x, chunk = (ntiles + G - 1) / G;
  const int t0 = blockIdx.x * chunk, t1 = t0 + chunk < ntiles ? t0 + chunk : ntiles;
  f32x4 acc[TAPS][CO / 16][CI / 16], bacc[CO / 16];
#pragma unroll
  for (int m = 0; m < CO / 16; ++m) {
    bacc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
      for (int n = 0; n < CI / 16; ++n) acc[k][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bf16x4 ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};  // 1 in BF16
  // row of this lane's 8 bytes of a 4 x 16 block: point 4 kg + r / 4, channels 4 (r % 4)..+3
  const int prow = 4 * kg + r / 4, pch = 4 * (r % 4);
  for (int tile = t0; tile < t1; ++tile) {
    const int b = tile / per_box, rem = tile % per_box;
    const int i0 = (rem % nbx) * CT_X, j0 = ((rem / nbx) % nby) * CT_Y, k0 = (rem / (nbx * nby)) * CT_Z;
    const long base = (long)b * XYZ;
    __syncthreads();  // the previous tile's reads are done
    for (int e = threadIdx.x; e < CT_PTS * (CO / 8); e += CT_THREADS) {
      const int q = e / (CO / 8), c8 = e % (CO / 8);
      const int gi = i0 + q % CT_X, gj = j0 + (q / CT_X) % CT_Y, gk = k0 + q / (CT_X * CT_Y);
      uint4 v = {0u, 0u, 0u, 0u};  // points beyond the box's far faces add nothing
      if (gi < X && gj < Y && gk < Z)
        v = *reinterpret_cast<const uint4 *>(dz + (base + gi + X * ((long)gj + (long)Y * gk)) * CO + c8 * 8);
      *reinterpret_cast<uint4 *>(dt + e * 8) = v;
    }
    for (int e = threadIdx.x; e < CT_HALO * (CI / 8); e += CT_THREADS) {
      const int q = e / (CI / 8), c8 = e % (CI / 8);
      int gi = i0 + q % CH_X - 1, gj = j0 + (q / CH_X) % CH_Y - 1, gk = k0 + q / (CH_X * CH_Y) - 1;
      bool ok = true;
      if (per) {
        gi = gi < 0 ? gi + X : (gi >= X ? gi - X : gi);
        gj = gj < 0 ? gj + Y : (gj >= Y ? gj - Y : gj);
        gk = gk < 0 ? gk + Z : (gk >= Z ? gk - Z : gk);
      } else {
        ok = gi >= 0 && gj >= 0 && gk >= 0;
      }
      ok = ok && gi < X && gj < Y && gk < Z;  // (wrapped once: further points meet dz = 0)
      uint4 v = {0u, 0u, 0u, 0u};
      if (ok) v = *reinterpret_cast<const uint4 *>(in + (base + gi + X * ((long)gj + (long)Y * gk)) * CI + c8 * 8);
      *reinterpret_cast<uint4 *>(xt + e * 8) = v;
    }
    __syncthreads();
    // the tile's x-rows of 16 points, one reduction step each
#pragma unroll 2
    for (int s = 0; s < CT_Y * CT_Z; ++s) {
      const int y = s % CT_Y, z = s / CT_Y;
      bf16x4 a[CO / 16];
#pragma unroll
      for (int m = 0; m < CO / 16; ++m) a[m] = read_points(dt + (s * CT_X + prow) * CO + m * 16 + pch);
      if (wave == WAVES - 1) {
#pragma unroll
        for (int m = 0; m < CO / 16; ++m)
          bacc[m] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], ones, bacc[m], 0, 0, 0);
      }
#pragma unroll
      for (int k = 0; k < TAPS; ++k) {
        const int t = wave + WAVES * k;
        if (t >= 27) continue;  // uniform in the wavefront
        const int dx = t % 3, dy = (t / 3) % 3, dzt = t / 9;
        const int row = ((z + dzt) * CH_Y + y + dy) * CH_X + dx + prow;
#pragma unroll
        for (int n = 0; n < CI / 16; ++n) {
          const bf16x4 x = read_points(xt + row * CI + n * 16 + pch);
#pragma unroll
          for (int m = 0; m < CO / 16; ++m)
            acc[k][m][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], x, acc[k][m][n], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < TAPS; ++k) {
    const int t = wave + WAVES * k;
    if (t >= 27) continue;
#pragma unroll
    for (int m = 0; m < CO / 16; ++m)
#pragma unroll
      for (int n = 0; n < CI / 16; ++n)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          part[(((long)blockIdx.x * 27 + t) * CO + m * 16 + 4 * kg + rr) * CI + n * 16 + r] = acc[k][m][n][rr];
  }
  if (wave == WAVES - 1 && r == 0) {
#pragma unroll
    for (int m = 0; m < CO / 16; ++m)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) bpart[(long)blockIdx.x * CO + m * 16 + 4 * kg + rr] = bacc[m][rr];
  }
}

// Sums of the work-groups' partials: dW[e] over nw weights and, in the last
// work-group, db[e] over nb <= 64 biases.  64 entries per work-group; its 16
// wavefronts take a sixteenth of the chunks each, several loads in flight (four
// wavefronts with one load at a time took 17 us for 256 chunks of 27648).
__global__ __launch_bounds__(1024) void k_sum_chunks(const float *__restrict__ part, const float *__restrict__ bpart,
                                                     int nchunks, int nw, int nb, float *__restrict__ dW,
                                                     float *__restrict__ db) {
  __shared__ float red[16][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool bias = blockIdx.x == gridDim.x - 1;
  const float *src = bias ? bpart : part;
  const int n = bias ? nb : nw, e = bias ? l : blockIdx.x * 64 + l;
  float s = 0.f;
  if (e < n) {
#pragma unroll 8
    for (int c = w; c < nchunks; c += 16) s += src[(long)c * n + e];
  }
  red[w][l] = s;
  __syncthreads();
  if (w == 0 && e < n) {
#pragma unroll
    for (int k = 1; k < 16; ++k) s += red[k][l];
    (bias ? db : dW)[e] = s;
  }
}

// Mean-square loss over the 5 real channels of out[p][16] against
// target[c][p], counting only the points at least `halo` away from their
// box's faces (all points for halo 0); dout[p][16] <- bf16(2 (out - target)
// / count) (zero elsewhere), partial loss sums per block into lpart.
__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ out, const float *__restrict__ target,
                                             long npts, ConvGeom geo, int halo, float scale,
                                             bf16 *__restrict__ dout, float *__restrict__ lpart) {
  __shared__ float red[256];
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  float s = 0.f;
  if (p < npts) {
    bool in = true;
    if (halo > 0) {
      const Coord cc = coord_of(p, geo);
      in = cc.i >= halo && cc.i < geo.X - halo && cc.j >= halo && cc.j < geo.Y - halo && cc.k >= halo &&
           cc.k < geo.Z - halo;
    }
    const f32x4 o = *reinterpret_cast<const f32x4 *>(out + p * 16);
    const float o4 = out[p * 16 + 4];
    float g[8] = {};
#pragma unroll
    for (int c = 0; c < 5; ++c)
      if (in) {
        const float d = (c < 4 ? o[c & 3] : o4) - target[c * npts + p];
        s += d * d;
        g[c] = scale * d;
      }
    const uint2 lo = to_bf16(f32x4{g[0], g[1], g[2], g[3]}), hi = to_bf16(f32x4{g[4], g[5], g[6], g[7]});
    uint4 *w = reinterpret_cast<uint4 *>(dout + p * 16);
    w[0] = uint4{lo.x, lo.y, hi.x, hi.y};
    w[1] = uint4{0u, 0u, 0u, 0u};
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

// One batch entry: a box of the training set and the offset of the window
// taken from it (the window's first point is the sample point (ox, oy, oz)).
struct CropSpec {
  const bf16 *feat;   // sample features [S^3][16]
  const float *tgt;   // sample targets [5][S^3]
  int ox, oy, oz, pad;
};

// Batch of windows X^3 (X = crop + 2 halo) cut from periodic S^3 samples:
// features of every window point, targets of every point (the loss masks
// the halo).  One thread per window point.
__global__ __launch_bounds__(256) void k_gather_crops(const CropSpec *__restrict__ spec, int S, ConvGeom geo,
                                                      long npts, bf16 *__restrict__ feat,
                                                      float *__restrict__ tgt) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  if (p >= npts) return;
  const Coord cc = coord_of(p, geo);
  const CropSpec sp = spec[cc.base / ((long)geo.X * geo.Y * geo.Z)];
  const int msk = S - 1;
  const int i = (sp.ox + cc.i) & msk, j = (sp.oy + cc.j) & msk, k = (sp.oz + cc.k) & msk;
  const long src = i + (long)S * (j + (long)S * k);
  const long S3 = (long)S * S * S;
  const uint4 *f = reinterpret_cast<const uint4 *>(sp.feat + src * 16);
  uint4 *d = reinterpret_cast<uint4 *>(feat + p * 16);
  d[0] = f[0];
  d[1] = f[1];
#pragma unroll
  for (int c = 0; c < 5; ++c) tgt[c * npts + p] = sp.tgt[c * S3 + src];
}

// Adam on the FP32 master parameters (bias-corrected step sizes from the host)
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, long n, float lr_t, float b1, float b2, float eps_t) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float gg = g[e];
  const float mm = b1 * m[e] + (1.f - b1) * gg;
  const float vv = b2 * v[e] + (1.f - b2) * gg * gg;
  m[e] = mm;
  v[e] = vv;
  w[e] = w[e] - lr_t * mm / (sqrtf(vv) + eps_t);
}

// BF16 copies of one layer's weights W[t][co][ci] (FP32, padded): the forward
// operand as is, and the transposed operand WT[t][ci][co] for the input grad.
__global__ void k_pack_weights(const float *__restrict__ w, int CO, int CI, bf16 *__restrict__ wf,
                               bf16 *__restrict__ wt) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 27L * CO * CI) return;
  const int t = (int)(e / ((long)CO * CI));
  const int co = (int)((e / CI) % CO), ci = (int)(e % CI);
  const bf16 h = to_bf16(w[e]);
  wf[e] = h;
  wt[((long)t * CI + ci) * CO + co] = h;
}

// Means of the 5 fields of a state, in a fixed summation order: partial
// sums of MEAN_BLOCKS grid-strided work-groups per field; the kernels that
// use the means add these up themselves (a launch less, 6 us; reading 10 KB of
// partial sums in every work-group costs 2).  The network sees every sample
// relative to its own means.
constexpr int MEAN_BLOCKS = 256;

// Sums over the work-group's 256 threads, as a tree (t takes t + 128, then t + 64, ...):
// valid in thread 0
template <int NF>
__device__ __forceinline__ void block_sums(double (&s)[NF], double (&red)[NF][128]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int w = 128; w >= 64; w >>= 1) {
    __syncthreads();
    if (t >= w && t < 2 * w) {
#pragma unroll
      for (int c = 0; c < NF; ++c) red[c][t - w] = s[c];
    }
    __syncthreads();
    if (t < w) {
#pragma unroll
      for (int c = 0; c < NF; ++c) s[c] += red[c][t];
    }
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1)
#pragma unroll
    for (int c = 0; c < NF; ++c) s[c] += __shfl_down(s[c], w);
}

// The means of the first NF fields from their partial sums, in every thread
template <int NF>
__device__ __forceinline__ void field_means(const double *__restrict__ part, long N, double (&mean)[NF]) {
  __shared__ double red[NF][128];
#pragma unroll
  for (int c = 0; c < NF; ++c) mean[c] = part[c * MEAN_BLOCKS + threadIdx.x];
  block_sums(mean, red);
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < NF; ++c) red[c][0] = mean[c] / (double)N;
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NF; ++c) mean[c] = red[c][0];
}

// work-group (b, c): partial sum b of field c
template <typename Q>
__global__ __launch_bounds__(256) void k_field_partials(const Q *__restrict__ q, long N,
                                                        double *__restrict__ part) {
  __shared__ double red[1][128];
  q += blockIdx.y * N;
  double s[1] = {0.0};
#pragma unroll 4
  for (long p = (long)blockIdx.x * 256 + threadIdx.x; p < N; p += MEAN_BLOCKS * 256) s[0] += (double)q[p];
  block_sums(s, red);
  if (threadIdx.x == 0) part[blockIdx.y * MEAN_BLOCKS + blockIdx.x] = s[0];
}

// Normalisation of a closure network (device copy, set by the host).
// Features: x_c = (q_c - mean_c) inv_std_c with the sample's field means;
// outputs: force_v = out_v out_std_v, times mean_p / p_ref for the pressure
// equation when p_ref > 0 (its residual scales with the mean pressure).
struct CnnNorm {
  float inv_std[5], out_std[5], out_inv_std[5];
  float gain[5];  // inference only: force_v = gain[v] x the network's term
  double p_ref;
};

__device__ __forceinline__ float pressure_scale(const CnnNorm &nm, const double *mean) {
  return nm.p_ref > 0.0 ? (float)(mean[4] / nm.p_ref) : 1.f;
}

// Network input from a state q (5 fields of N points, field-major, with their
// partial sums): channel c of point p = bf16(f32(q[c][p] - mean[c])
// inv_std[c]), channels 5..15 zero; mean[0..4] set.
template <typename Q>
__global__ __launch_bounds__(256) void k_pack_features(const Q *__restrict__ q, long N, const double *__restrict__ part,
                                                       const CnnNorm *__restrict__ nm, double *__restrict__ mean,
                                                       bf16 *__restrict__ feat) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  Q v[5] = {};
  if (p < N) {
#pragma unroll
    for (int c = 0; c < 5; ++c) v[c] = q[c * N + p];
  }
  double m[5];
  field_means(part, N, m);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 5; ++c) mean[c] = m[c];
  }
  if (p >= N) return;
  unsigned h[3];
#pragma unroll
  for (int c = 0; c < 6; c += 2) {
    const unsigned lo = to_bf16((float)((double)v[c] - m[c]) * nm->inv_std[c]);
    const unsigned hi = c + 1 < 5 ? to_bf16((float)((double)v[c + 1] - m[c + 1]) * nm->inv_std[c + 1]) : 0u;
    h[c / 2] = lo | (hi << 16);
  }
  uint4 *d = reinterpret_cast<uint4 *>(feat + p * 16);
  d[0] = uint4{h[0], h[1], h[2], 0u};
  d[1] = uint4{0u, 0u, 0u, 0u};
}

// Closure term in the solver's layout: force[v][p] = out[p][v] out_std[v] (x pressure scale) x gain[v],
// and the partial sums of its first 4 fields
template <typename T>
__global__ __launch_bounds__(256) void k_unpack_closure(const float *__restrict__ out, long N,
                                                        const CnnNorm *__restrict__ nm,
                                                        const double *__restrict__ mean, T *__restrict__ force,
                                                        double *__restrict__ part) {
  __shared__ double red[4][128];
  const float ps = pressure_scale(*nm, mean);
  float scale[5], gain[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    scale[v] = v == 4 ? nm->out_std[4] * ps : nm->out_std[v];
    gain[v] = nm->gain[v];
  }
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (long p = (long)blockIdx.x * 256 + threadIdx.x; p < N; p += MEAN_BLOCKS * 256) {
    const f32x4 o = *reinterpret_cast<const f32x4 *>(out + p * 16);
    const float o4 = out[p * 16 + 4];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const T f = T((v < 4 ? o[v & 3] : o4) * scale[v] * gain[v]);
      force[v * N + p] = f;
      if (v < 4) s[v & 3] += (double)f;
    }
  }
  block_sums(s, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) part[v * MEAN_BLOCKS + blockIdx.x] = s[v];
  }
}

// Zero domain mean for the closure terms of the conserved variables (rho,
// rho u, rho v, rho w): a subfilter term of a conservation law is the
// divergence of a subfilter flux and adds nothing to the domain total.
template <typename T>
__global__ __launch_bounds__(256) void k_remove_mean(T *__restrict__ force, long N, const double *__restrict__ part) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  T f[4] = {};
  if (p < N) {
#pragma unroll
    for (int v = 0; v < 4; ++v) f[v] = force[v * N + p];
  }
  double m[4];
  field_means(part, N, m);
  if (p >= N) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) force[v * N + p] = f[v] - T(m[v]);
}

// Normalised targets: tn[c][p] = target[c][p] out_inv_std[c] (/ pressure scale)
__global__ void k_scale_targets(const double *__restrict__ target, long N, const CnnNorm *__restrict__ nm,
                                const double *__restrict__ mean, float *__restrict__ tn) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const float ps = pressure_scale(*nm, mean);
  for (int c = 0; c < 5; ++c) {
    const float s = c == 4 ? nm->out_inv_std[4] / ps : nm->out_inv_std[c];
    tn[c * N + p] = (float)target[c * N + p] * s;
  }
}

// Box average of a state over f^3 blocks: out (m1, m2, m3, 5) with m = n / f.
template <typename T>
__global__ void k_box_average(const T *__restrict__ q, int n1, int n2, int n3, int f,
                              double *__restrict__ out) {
  const int m1 = n1 / f, m2 = n2 / f, m3 = n3 / f;
  const long M = (long)m1 * m2 * m3;
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 5 * M) return;
  const int v = (int)(e / M);
  const long r = e - (long)v * M;
  const int i = (int)(r % m1), j = (int)((r / m1) % m2), k = (int)(r / ((long)m1 * m2));
  const long N = (long)n1 * n2 * n3;
  double s = 0.0;
  for (int c = 0; c < f; ++c)
    for (int b = 0; b < f; ++b)
      for (int a = 0; a < f; ++a)
        s += (double)q[v * N + (i * f + a) + (long)n1 * ((j * f + b) + (long)n2 * (k * f + c))];
  out[e] = s / ((double)f * f * f);
}

}  // namespace cruna
