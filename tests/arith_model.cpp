// Prints the largest error, in units of 2^-24 relative, of the epilogue arithmetic in
// transformer_amd/csrc/arith.h against 64 bits: swiglu over gates of [-80, 80], and the quotient over
// mantissas and exponents of its operands; then the quotient at infinities, zeros and NaN.
#include <cmath>
#include <cstdio>
#include <random>

#include "../transformer_amd/csrc/arith.h"

int main() {
  const double unit = std::ldexp(1.0, -24);
  double es = 0, eq = 0;
  for (int i = -800000; i <= 800000; ++i) {
    const float g = float(i) * 1e-4f, u = 0.75f;
    if (g == 0.f) continue;
    const double ref = double(g) / (1.0 + std::exp(-double(g))) * double(u);
    es = std::fmax(es, std::fabs(double(msdc::swiglu(g, u)) - ref) / std::fabs(ref) / unit);
  }
  std::mt19937 rng(1);
  std::uniform_real_distribution<float> man(1.f, 2.f);
  std::uniform_int_distribution<int> ex(-20, 20);
  long differ = 0;
  for (int i = 0; i < 2000000; ++i) {
    const float a = std::ldexp(man(rng), ex(rng)), b = std::ldexp(man(rng), ex(rng));
    const float q = msdc::quotient(a, b, 1.f / b);
    differ += q != a / b;
    eq = std::fmax(eq, std::fabs(double(q) - double(a) / double(b)) / (double(a) / double(b)) / unit);
  }
  std::printf("swiglu %.3f quotient %.4f differ %ld\n", es, eq, differ);
  const float inf = INFINITY, nan = NAN;
  std::printf("edges %g %g %g %g\n", msdc::quotient(inf, 2.f, 0.5f), msdc::quotient(1.f, inf, 0.f),
              msdc::quotient(0.f, 2.f, 0.5f), msdc::quotient(nan, 2.f, 0.5f));
}
