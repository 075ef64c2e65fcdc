// FP64 line solve by constant-coefficient recursions.
//
// The left matrix B of every compact scheme here is tridiag(a, d, a) away from
// the ends of an open line.  With alpha = a/d and lambda the root of
// lambda / (1 + lambda^2) = alpha inside the unit circle it factors exactly:
//   B = d / (1 + lambda^2) (I + lambda S-) (I + lambda S+)
// (S-, S+ the shifts along the line), so x = B^-1 A f is a forward and a
// backward recursion with the one coefficient mu = -lambda after the explicit
// stencil A, whose coefficients absorb the factor (1 + lambda^2) / d.  A thread owns 8 consecutive points of
// a line (as in line_solve.hpp):
//   1. halo exchange, stencil, and the forward recursion from a zero start;
//   2. the blocks' last values u_L give the value that really enters a block,
//      U_b = sum_m rho^m u_L(b-1-m), rho = mu^8; u_i += mu^(i+1) U;
//   3. the same backward: X_b = sum_m rho^m x_F(b+1+m), x_i += mu^(8-i) X.
// The sums stop where rho^m is below 2^-55 (5 terms for the o6 derivative, 6
// for the filter at alpha 0.35).  Three exchanges and about 72 FP64
// operations per 8 points, against five exchanges and about 130 of the
// cyclic reduction of line_solve.hpp, and the coefficients (the stencil's and
// mu^1..mu^8) fit in scalar registers for a whole kernel.  What a solve costs on
// small grids is its chain of LDS exchanges, table loads and dependent
// operations: measured per step against the cyclic reduction with its tables
// re-read in every solve, 32^3 286 -> 200 us, 64^3 390 -> 310 us, an open
// 60 x 65 x 70 box 1.28 -> 0.88 ms; the fused z kernel at 256^3 0.753 -> 0.664 ms
// (the other 256^3 sweeps are bound by HBM either way).
//
// Open lines: the factored matrix differs from B in rows 0, 1 and the last
// two.  The correction y = x - x~ of its solution x~ solves the homogeneous
// recurrence, y_i = sigma_L mu^i + sigma_R mu^(n-1-i) (plus kappa_L and
// kappa_R at the end points), and each end's two rows give (sigma, kappa) from
// the three end values of x~ and the other end's sigma.  The end threads
// publish their scalar A = C . x~ in one more exchange.
//
// FP32 keeps the cyclic reduction (line_solve.hpp), and with it the rounding of
// the FP32-mixed mode's line solves.
#pragma once

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <vector>

#include "line_ops.hpp"

namespace cruna {

constexpr int REC_WIN = 6;  // window terms kept as addresses (more: the slow loop)
// largest lambda of the recursion engine (alpha 0.4972): beyond it the end
// corrections' two modes mu^i and mu^(n-1-i) become alike, and the filter
// runs on the cyclic reduction of line_solve.hpp.  Up to there the recursions
// are the faster ones, also where their window takes the slow loop (alpha from
// 0.376 on: M = 7 terms at 0.38, 11 at 0.45, 44 at 0.497, at most one per block
// of the line), because the x filter then stays inside the last stage's x sweep.
// A step with filters on them, against one with the slow alphas on the cyclic
// reduction, at alpha 0.38 / 0.45 / 0.497: periodic 64^3 237 / 228 / 228 against
// 233 / 236 / 242 us, 256^3 9.67 / 9.63 / 9.67 against 9.98 / 9.99 / 10.03 ms;
// open 64^3 417 against 444 us throughout, 128^3 1.27 to 1.29 against 1.39 to
// 1.41 ms.
constexpr double REC_MAX_LAMBDA = 0.9;

// Table of an open line's ends (device memory; RecLines copies what it needs to LDS):
// per end (0 left, 1 right):
//   [0 .. 8 FE)  dense explicit rows of the end block (scaled)
//   [8 FE .. +8) C: A_end = C . x~ over the block's rows
//   [8 FE + 8 .. +8) K: kappa = K . x~ + gamma sigma(other end)
// then 6 scalars: sigma_L = t0 A_L + t1 A_R, sigma_R = t2 A_R + t3 A_L,
// gamma_L, gamma_R; then per block mu^(8 b - pf) and mu^(n-1 - (8 b - pf) - 7).
constexpr int REC_END = PPT * FE + 2 * PPT;
constexpr int REC_SCAL = 2 * REC_END;
constexpr int REC_PW = REC_SCAL + 6;
constexpr int REC_ROWS = 4;  // most rows of its own in an end block

struct RecOp {
  double s[4];     // stencil c0..c3 (scaled)
  double mu;       // -lambda
  double lp[PPT];  // mu^1..mu^8
  double rho;      // mu^8
  double norm;     // factor of a window that wraps the whole periodic line
  const double *tab;  // open lines: ends (above)
  int n, NB, per;
  int M;           // window terms of the slow form (at most the line's blocks)
  int slow;        // more than REC_WIN terms are needed
  int nend;        // 1: the ends need corrections
  int srow[2];     // bit r: row r of the first / last block has its own explicit row
  int zrow[2];     // bit r: row r of the first / last block is padding
  int rend[2];     // row of the first / last real point in its block
  int rows[2];     // srow as a list: row k in bits 4k..4k+3, 15 for none
  int nrow;        // the longer list's length (at most REC_ROWS)
};

struct HostRecOp {
  RecOp op{};
  std::vector<double> tab;
  bool usable = false;  // lambda within REC_MAX_LAMBDA
};

inline HostRecOp build_rec_op(OpKind kind, bool per, int n_real, double alpha) {
  using namespace detail;
  HostRecOp h;
  RecOp &op = h.op;
  std::vector<std::vector<std::pair<int, double>>> A;
  std::vector<double> lo, di, up;
  explicit_rows(kind, per, n_real, alpha, A);
  implicit_rows(kind, per, n_real, alpha, lo, di, up);
  const int n = padded_length(per, n_real), pf = front_padding(per, n_real), mid = n_real / 2;
  op.n = n;
  op.NB = n / PPT;
  op.per = per ? 1 : 0;
  const long double al = (long double)lo[mid] / di[mid];
  if (!(std::fabs((double)al) < 0.5)) return h;
  // (this form of the root keeps its digits for small alpha)
  const long double lam = 2.0L * al / (1.0L + std::sqrt(1.0L - 4.0L * al * al));
  if (std::fabs((double)lam) > REC_MAX_LAMBDA) return h;
  h.usable = true;
  const long double mu = -lam, sc = (1.0L + lam * lam) / di[mid];
  op.mu = (double)mu;
  std::vector<long double> pw(n_real + 2 * PPT + 1);
  pw[0] = 1.0L;
  for (size_t k = 1; k < pw.size(); ++k) pw[k] = pw[k - 1] * mu;
  for (int k = 0; k < PPT; ++k) op.lp[k] = (double)pw[k + 1];
  op.rho = (double)pw[PPT];
  op.norm = 1.0;
  op.M = 1;
  for (double r = op.rho; r > 0x1p-55; r *= op.rho) ++op.M;
  op.slow = op.M > REC_WIN ? 1 : 0;
  if (op.slow && kind != OP_FILTER) throw std::runtime_error("a derivative that decays too slowly");
  if (op.slow) {
    const int most = per ? op.NB : op.NB - 1;
    if (op.M > most) {
      op.M = std::max(most, 1);
      if (per) op.norm = 1.0 / (1.0 - std::pow(op.rho, op.NB));
    }
  }
  // interior stencil
  double c[7] = {0, 0, 0, 0, 0, 0, 0};
  const int ri = per ? 0 : (n_real >= 9 ? 4 : mid);
  for (auto &jc : A[ri]) {
    int off = jc.first - ri;
    if (per) off = ((off + n / 2) % n + n) % n - n / 2;
    c[off + 3] += jc.second;
  }
  for (int k = 0; k < 4; ++k) op.s[k] = (double)(sc * c[3 + k]);
  if (per) return h;

  // ---- open ends ----
  const int NB = op.NB, last = pf + n_real - 1;
  h.tab.assign(REC_PW + 2 * NB, 0.0);
  op.rend[0] = pf;
  op.rend[1] = last % PPT;
  auto interior = [&](int i) {
    if (A[i].size() != A[ri].size()) return false;
    for (size_t k = 0; k < A[i].size(); ++k)
      if (A[i][k].first - i != A[ri][k].first - ri || A[i][k].second != A[ri][k].second) return false;
    return true;
  };
  for (int i = 0; i < n_real; ++i) {
    if (interior(i)) continue;
    const int p = i + pf, e = i < mid ? 0 : 1, b = e == 0 ? 0 : NB - 1;
    if (p / PPT != b) throw std::runtime_error("closure rows beyond the two end blocks");
    op.srow[e] |= 1 << (p % PPT);
    for (auto &jc : A[i]) {
      const int j = jc.first + pf - b * PPT + HALO;
      const int reach = kind == OP_FILTER ? 3 : 2;  // halo points of the engine
      if (j < HALO - reach || j >= HALO + PPT + reach) throw std::runtime_error("closure row wider than the halo");
      h.tab[e * REC_END + (p % PPT) * FE + j] += (double)(sc * jc.second);
    }
  }
  for (int e = 0; e < 2; ++e) {
    int k = 0;
    op.rows[e] = (1 << 4 * REC_ROWS) - 1;
    for (int r = 0; r < PPT; ++r)
      if ((op.srow[e] >> r) & 1) {
        if (k == REC_ROWS) throw std::runtime_error("too many closure rows in a block");
        op.rows[e] ^= (15 ^ r) << 4 * k++;
      }
    op.nrow = std::max(op.nrow, k);
  }
  for (int r = 0; r < PPT; ++r) {
    if (r < pf) op.zrow[0] |= 1 << r;
    if (r > op.rend[1]) op.zrow[1] |= 1 << r;
  }
  auto mpow = [&](int k) -> long double { return k >= 0 ? pw[k] : 1.0L / pw[-k]; };
  // B normalised to (I + lambda L)(I + lambda U)'s scale, and its difference E
  auto Bn = [&](int i, int j) -> long double {
    return sc * (long double)(j == i ? di[i] : (j == i + 1 ? up[i] : (j == i - 1 ? lo[i] : 0.0)));
  };
  auto Bt = [&](int i, int j) -> long double {
    return j == i ? (i == 0 ? 1.0L : 1.0L + lam * lam) : ((j == i + 1 || j == i - 1) ? lam : 0.0L);
  };
  long double C[2][3] = {}, K[2][3] = {}, beta[2] = {}, gam[2] = {};
  const int N = n_real;
  bool differs = false;
  for (int e = 0; e < 2; ++e) {
    auto ix = [&](int k) { return e == 0 ? k : N - 1 - k; };
    long double E[2][3], b[2][3];
    for (int r = 0; r < 2; ++r)
      for (int k = 0; k < 3; ++k) {
        b[r][k] = Bn(ix(r), ix(k));
        E[r][k] = b[r][k] - Bt(ix(r), ix(k));
        if (std::fabs((double)E[r][k]) > 1e-17) differs = true;
      }
    if (lam == 0.0L) continue;
    const long double a11 = b[0][0] + b[0][1] * mu, a12 = b[0][0],
                      a21 = b[1][0] + b[1][1] * mu + b[1][2] * mu * mu, a22 = b[1][0];
    const long double det = a11 * a22 - a12 * a21;
    // (relative to the rows: a filter's second one is of the size of alpha)
    const long double size = std::max(std::fabs(a11), std::fabs(a12)) * std::max(std::fabs(a21), std::fabs(a22));
    if (!(std::fabs(det) > 1e-12L * size)) throw std::runtime_error("singular end closure");
    const long double i11 = a22 / det, i12 = -a12 / det, i21 = -a21 / det, i22 = a11 / det;
    for (int k = 0; k < 3; ++k) {
      C[e][k] = -(i11 * E[0][k] + i12 * E[1][k]);
      K[e][k] = -(i21 * E[0][k] + i22 * E[1][k]);
    }
    const long double f0 = b[0][0] * mpow(N - 1) + b[0][1] * mpow(N - 2);
    const long double f1 = b[1][0] * mpow(N - 1) + b[1][1] * mpow(N - 2) + b[1][2] * mpow(N - 3);
    beta[e] = -(i11 * f0 + i12 * f1);
    gam[e] = -(i21 * f0 + i22 * f1);
  }
  op.nend = lam != 0.0L && differs ? 1 : 0;
  if (op.nend) {
    for (int e = 0; e < 2; ++e)
      for (int k = 0; k < 3; ++k) {
        const int r = e == 0 ? pf + k : op.rend[1] - k;
        if (r < 0 || r >= PPT) throw std::runtime_error("end rows beyond their block");
        h.tab[e * REC_END + PPT * FE + r] = (double)C[e][k];
        h.tab[e * REC_END + PPT * FE + PPT + r] = (double)K[e][k];
      }
    const long double D = 1.0L - beta[0] * beta[1];
    double *t = h.tab.data() + REC_SCAL;
    t[0] = (double)(1.0L / D);
    t[1] = (double)(beta[0] / D);
    t[2] = (double)(1.0L / D);
    t[3] = (double)(beta[1] / D);
    t[4] = (double)gam[0];
    t[5] = (double)gam[1];
    for (int b = 0; b < NB; ++b) {
      h.tab[REC_PW + 2 * b] = (double)mpow(b * PPT - pf);
      h.tab[REC_PW + 2 * b + 1] = (double)mpow(N - 1 - (b * PPT - pf) - (PPT - 1));
    }
  }
  return h;
}

}  // namespace cruna
