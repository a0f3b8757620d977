// Host run of the complex 16-point DFT and the tangent-form twiddles of the
// log-mel kernel's FFT (scriptrs_amd/csrc/sfe_fft.hpp) against float64 DFTs.
// (The whole transform: tests/rdft_host_driver.cpp.)  No GPU is used.
//
// Prints one line per check and "bad N" at the end (N checks failed).
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <complex>
#include <random>
#include <vector>

#include "sfe_fft.hpp"

using sfe::cf;
typedef std::complex<double> C;

static int bad = 0;

static void check(const char* what, double err, double bound) {
  const bool ok = err <= bound;
  printf("%s: %.3e (bound %.1e) %s\n", what, err, bound, ok ? "ok" : "FAIL");
  if (!ok) ++bad;
}

static std::vector<C> dft(const std::vector<C>& x) {
  const size_t n = x.size();
  std::vector<C> y(n);
  for (size_t k = 0; k < n; ++k) {
    C s = 0;
    for (size_t m = 0; m < n; ++m) s += x[m] * std::polar(1.0, -2.0 * M_PI * (double)((k * m) % n) / (double)n);
    y[k] = s;
  }
  return y;
}

int main() {
  std::mt19937 rng(1234);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  const double u = ldexp(1.0, -24);

  // 16-point DFT, all scales 1: error relative to the input norm
  double e16 = 0;
  float ones[16];
  for (float& o : ones) o = 1.0f;
  for (int trial = 0; trial < 2000; ++trial) {
    cf a[16];
    std::vector<C> x(16);
    double nrm = 0;
    for (int m = 0; m < 16; ++m) {
      a[m] = {nd(rng), nd(rng)};
      x[m] = C(a[m].x, a[m].y);
      nrm += std::norm(x[m]);
    }
    sfe::dft16_scaled(a, ones);
    std::vector<C> y = dft(x);
    for (int k = 0; k < 16; ++k) e16 = fmax(e16, std::abs(C(a[k].x, a[k].y) - y[k]) / sqrt(nrm) / u);
  }
  // Twiddled inputs in tangent form, the cosines applied by dft16_scaled:
  // the DFT of a[m] e^{-i theta_m}, including theta = pi/2 and 3 pi/2 (as
  // a 2^-100 / 2^100 pair).
  double e16s = 0;
  std::uniform_real_distribution<double> ud(0.0, 2.0 * M_PI);
  for (int trial = 0; trial < 2000; ++trial) {
    cf a[16];
    float c[16];
    std::vector<C> x(16);
    double nrm = 0;
    for (int m = 0; m < 16; ++m) {
      const cf v = {nd(rng), nd(rng)};
      double th = m == 0 ? 0.0 : ud(rng);
      if (trial % 7 == 0 && m == 5) th = M_PI / 2;
      if (trial % 7 == 1 && m == 9) th = 3 * M_PI / 2;
      double cc = cos(th), tn;
      if (fabs(th - M_PI / 2) < 1e-12 || fabs(th - 3 * M_PI / 2) < 1e-12) {
        cc = ldexp(1.0, -100);
        tn = (th < M_PI ? 1.0 : -1.0) * ldexp(1.0, 100);
      } else {
        tn = sin(th) / cc;
      }
      a[m] = m == 0 ? v : sfe::tan_twiddle(v, (float)tn);
      c[m] = m == 0 ? 1.0f : (float)cc;
      x[m] = C(v.x, v.y) * std::polar(1.0, -th);
      nrm += std::norm(x[m]);
    }
    sfe::dft16_scaled(a, c);
    std::vector<C> y = dft(x);
    for (int k = 0; k < 16; ++k) e16s = fmax(e16s, std::abs(C(a[k].x, a[k].y) - y[k]) / sqrt(nrm) / u);
  }
  // A radix-4 x 4 DFT in f32: a few ulps of the input norm per output.
  check("dft16_scaled, max |err| / (|x| u)", e16, 16.0);
  check("tan_twiddle + dft16_scaled, max |err| / (|x| u)", e16s, 24.0);
  printf("bad %d\n", bad);
  return bad != 0;
}
