// CPU emulation of the FP64 recursion engine (RecLines of
// public_amd/csrc/line_solve.hpp) driven by the host tables of
// public_amd/csrc/line_rec.hpp, compared with the oracle's LU-based cores on
// random lines: every scheme, periodic and open, padded open lines, lines
// shorter than the window and filters that decay slowly.
// Prints one line per case: kind scheme n alpha usable max_rel_err.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../oracle/cruna_oracle.h"
#include "../../public_amd/csrc/line_rec.hpp"

using namespace cruna;

static double window(const RecOp &op, const std::vector<double> &v, int b, int dir) {
  const bool slow = op.slow != 0;
  double s = 0.0;
  for (int m = (slow ? op.M : REC_WIN) - 1; m >= 0; --m) {
    int t = b + dir * (1 + m);
    double u = 0.0;
    if (op.per) u = v[((t % op.NB) + op.NB) % op.NB];
    else if (t >= 0 && t < op.NB) u = v[t];
    s = s * op.rho + u;
  }
  return slow ? s * op.norm : s;
}

static std::vector<double> emulate(const HostRecOp &h, bool filt, const std::vector<double> &f_real, int pf) {
  const RecOp &op = h.op;
  const int n = op.n, NB = op.NB, H = filt ? 3 : 2;
  std::vector<double> f(n, 0.0), x(n);
  for (size_t i = 0; i < f_real.size(); ++i) f[i + pf] = f_real[i];
  auto at = [&](int p) { return op.per ? f[((p % n) + n) % n] : (p >= 0 && p < n ? f[p] : 0.0); };
  const bool open = !op.per;
  auto masked = [&](int b, int r) {
    return open && ((b == 0 && ((op.zrow[0] >> r) & 1)) || (b == NB - 1 && ((op.zrow[1] >> r) & 1)));
  };
  std::vector<double> uL(NB), xF(NB);
  for (int p = 0; p < n; ++p) {
    double s = op.s[0] * at(p);
    for (int k = 1; k <= 3; ++k) s += op.s[k] * (filt ? at(p + k) + at(p - k) : at(p + k) - at(p - k));
    x[p] = s;
  }
  for (int e = 0; open && e < 2; ++e)
    for (int r = 0; r < PPT; ++r) {
      const int p = (e == 0 ? 0 : NB - 1) * PPT + r;
      if ((op.srow[e] >> r) & 1) {
        x[p] = 0.0;
        for (int j = HALO - H; j < HALO + PPT + H; ++j) x[p] += h.tab[e * REC_END + r * FE + j] * at(p - r - HALO + j);
      }
      if ((op.zrow[e] >> r) & 1) x[p] = 0.0;
    }
  for (int b = 0; b < NB; ++b) {
    for (int r = 1; r < PPT; ++r) x[b * PPT + r] += op.mu * x[b * PPT + r - 1];
    uL[b] = x[b * PPT + PPT - 1];
  }
  for (int b = 0; b < NB; ++b) {
    const double U = window(op, uL, b, -1);
    for (int r = 0; r < PPT; ++r) {
      x[b * PPT + r] += op.lp[r] * U;
      if (masked(b, r)) x[b * PPT + r] = 0.0;
    }
    for (int r = PPT - 2; r >= 0; --r) x[b * PPT + r] += op.mu * x[b * PPT + r + 1];
    xF[b] = x[b * PPT];
  }
  for (int b = 0; b < NB; ++b) {
    const double X = window(op, xF, b, +1);
    for (int r = 0; r < PPT; ++r) x[b * PPT + r] += op.lp[PPT - 1 - r] * X;
  }
  if (open && op.nend) {
    const double *t = h.tab.data() + REC_SCAL;
    double A[2] = {0, 0}, K[2] = {0, 0};
    for (int e = 0; e < 2; ++e)
      for (int r = 0; r < PPT; ++r) {
        const double v = x[(e == 0 ? 0 : NB - 1) * PPT + r], *c = h.tab.data() + e * REC_END + PPT * FE;
        A[e] += c[r] * v;
        K[e] += c[PPT + r] * v;
      }
    const double sl = t[0] * A[0] + t[1] * A[1], sr = t[2] * A[1] + t[3] * A[0];
    for (int b = 0; b < NB; ++b) {
      const double l = sl * t[6 + 2 * b], r = sr * t[6 + 2 * b + 1];
      for (int i = 0; i < PPT; ++i) {
        x[b * PPT + i] += (i ? op.lp[i - 1] : 1.0) * l;
        x[b * PPT + PPT - 1 - i] += (i ? op.lp[i - 1] : 1.0) * r;
      }
    }
    x[op.rend[0]] += K[0] + t[4] * sr;
    x[(NB - 1) * PPT + op.rend[1]] += K[1] + t[5] * sl;
  }
  for (int b = 0; b < NB; ++b)
    for (int r = 0; r < PPT; ++r)
      if (masked(b, r)) x[b * PPT + r] = filt ? f[b * PPT + r] : 0.0;
  return x;
}

int main() {
  std::mt19937_64 rng(7);
  std::normal_distribution<double> nd;
  const OpKind kinds[] = {OP_DIFF, OP_FILTER, OP_DIFF_O4E, OP_DIFF_O4P, OP_DIFF_O2E};
  const char *names[] = {"diff", "filter", "diffo4", "diffpade", "diffo2"};
  struct Case { int kind, per, n; double alpha; };
  std::vector<Case> cases;
  for (int kind = 0; kind < 5; ++kind) {
    for (int n : {16, 24, 40, 48, 64, 128, 256, 2048})
      if (kinds[kind] != OP_DIFF_O2E) cases.push_back({kind, 1, n, 0.35});
    for (int n : {9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 23, 24, 33, 40, 60, 65, 70, 128, 257, 2044})
      cases.push_back({kind, 0, n, 0.35});
  }
  // filters: from none to slow decay (both sides of the recursions' limit)
  for (double a : {-0.4, -0.1, 0.0, 0.1, 0.45, 0.49, 0.497, 0.4975, 0.4999, 0.5})
    for (int n : {16, 32, 64, 512}) {
      if (a != 0.5) cases.push_back({1, 1, n, a});
      cases.push_back({1, 0, n + 1, a});
    }
  for (const Case &c : cases) {
    const HostRecOp h = build_rec_op(kinds[c.kind], c.per, c.n, c.alpha);
    double worst = 0.0;
    for (int t = 0; t < 4 && h.usable; ++t) {
      std::vector<double> f(c.n);
      for (auto &v : f) v = nd(rng);
      std::vector<double> ref = f;
      const int sch = c.per ? ORC_PERIODIC : ORC_OPEN;
      if (c.kind == 0) orc_diff_core(sch, c.n, 1, ref.data(), 1.0);
      else if (c.kind == 1) orc_filter_core(sch, c.n, 1, ref.data(), c.alpha);
      else if (c.kind == 2) orc_diff_core_o4(sch, c.n, 1, ref.data(), 1.0);
      else if (c.kind == 3) orc_diff_core_pade(sch, c.n, 1, ref.data(), 1.0);
      else orc_diff_core_o2(c.n, 1, ref.data(), 1.0);
      const int pf = front_padding(c.per, c.n);
      const std::vector<double> x = emulate(h, c.kind == 1, f, pf);
      double num = 0, den = 0;
      for (int i = 0; i < c.n; ++i) {
        num = std::fmax(num, std::fabs(x[i + pf] - ref[i]));
        den = std::fmax(den, std::fabs(ref[i]));
      }
      for (int i = 0; i < h.op.n; ++i)
        if (i < pf || i >= pf + c.n) num = std::fmax(num, std::fabs(x[i]));
      worst = std::fmax(worst, num / den);
    }
    std::printf("%s %s %d %g %d %.3e\n", names[c.kind], c.per ? "periodic" : "open", c.n, c.alpha, h.usable ? 1 : 0,
                worst);
  }
  return 0;
}
