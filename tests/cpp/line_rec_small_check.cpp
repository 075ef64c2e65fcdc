// Filters of small alpha on the FP64 recursion engine: the same CPU emulation
// and reference cores as line_rec_check.cpp, on alphas down to the smallest
// FP64 number, periodic and open (padded) lines.
// Prints one line per case: scheme n alpha usable max_rel_err ("refused" where
// the tables cannot be built).
#define main line_rec_check_main
#include "line_rec_check.cpp"
#undef main

int main() {
  std::mt19937_64 rng(11);
  std::normal_distribution<double> nd;
  for (double size : {1e-3, 1e-4, 1e-6, 1e-7, 1e-8, 1e-9, 1e-10, 1e-11, 1e-12, 1e-14, 1e-16, 1e-17, 1e-30, 1e-300, 5e-324})
    for (double a : {size, -size})
      for (int n : {16, 64, 9, 13, 17, 65})
        for (int per = 0; per < 2; ++per) {
          if (per && n % PPT) continue;
          HostRecOp h;
          try {
            h = build_rec_op(OP_FILTER, per, n, a);
          } catch (const std::exception &) {
            std::printf("%s %d %g 0 refused\n", per ? "periodic" : "open", n, a);
            continue;
          }
          const int pf = front_padding(per, n);
          double worst = 0.0;
          for (int t = 0; t < 4; ++t) {
            std::vector<double> f(n);
            for (auto &v : f) v = nd(rng);
            std::vector<double> ref = f;
            orc_filter_core(per ? ORC_PERIODIC : ORC_OPEN, n, 1, ref.data(), a);
            const std::vector<double> x = emulate(h, true, f, pf);
            double num = 0, den = 0;
            for (int i = 0; i < n; ++i) {
              const double e = std::fabs(x[i + pf] - ref[i]);
              num = e <= num ? num : e;  // a NaN stays
              den = std::fmax(den, std::fabs(ref[i]));
            }
            const double r = num / den;
            worst = r <= worst ? worst : r;
          }
          std::printf("%s %d %g %d %.3e\n", per ? "periodic" : "open", n, a, h.usable ? 1 : 0, worst);
        }
  return 0;
}
