// Host run of the log-mel kernel's 32 x 16 real FFT (scriptrs_amd/csrc/
// sfe_fft.hpp rdft32_windowed, tan_twiddle, dft16_scaled) with the device
// tables, against float64 DFTs; of its mel schedule against the filterbank;
// and of the raw log-mel layout.  Argument: a sample rate.  No GPU is used.
//
// Prints one line per check and "bad N" at the end (N checks failed).
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <complex>
#include <random>
#include <set>
#include <vector>

#include "sfe_fft.hpp"
#include "sfe_internal.hpp"

using sfe::cf;
typedef std::complex<double> C;

static int bad = 0;

static void check(const char* what, double err, double bound) {
  const bool ok = err <= bound;
  printf("%s: %.3e (bound %.1e) %s\n", what, err, bound, ok ? "ok" : "FAIL");
  if (!ok) ++bad;
}

static C root(int m, int n) { return std::polar(1.0, -2.0 * M_PI * (double)(((m % n) + n) % n) / (double)n); }

int main(int argc, char** argv) {
  const int rate = argc > 1 ? atoi(argv[1]) : 16000;
  std::mt19937 rng(99);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  const double u = ldexp(1.0, -24);

  double e32 = 0;
  for (int trial = 0; trial < 1000; ++trial) {
    float y[25], w[25];
    double nrm = 0;
    for (int i = 0; i < 25; ++i) {
      y[i] = nd(rng);
      w[i] = fabsf(nd(rng));
      nrm += (double)y[i] * w[i] * y[i] * w[i];
    }
    cf Y[16];
    sfe::rdft32_windowed(y, w, Y);
    for (int k = 0; k <= 16; ++k) {
      C s = 0;
      for (int i = 0; i < 25; ++i) s += (double)y[i] * (double)w[i] * root(k * (i - 12), 32);
      const C got = k == 0 ? C(Y[0].x, 0) : (k == 16 ? C(Y[0].y, 0) : C(Y[k].x, Y[k].y));
      e32 = fmax(e32, std::abs(got - s) / sqrt(nrm) / u);
    }
  }
  // 6 levels of additions and constant factors: a few ulps of the input norm
  check("rdft32_windowed, max |err| / (|x w| u)", e32, 16.0);

  sfe::DevTables tb;
  if (!sfe::build_dev_tables(rate, &tb)) {
    printf("tables failed\nbad 1\n");
    return 1;
  }
  // Whole frames as the kernel computes them: |X_k|^2, k = 1 .. 256.
  double emag = 0, especial = 0, equiet = 0;
  for (int trial = 0; trial < 200; ++trial) {
    std::vector<float> y(400);
    const float amp = trial % 4 == 0 ? 1e-3f : 1.0f;
    for (float& v : y) v = amp * nd(rng);
    if (trial % 5 == 1)  // a loud low tone over near silence: low-energy bins next to a strong one
      for (int n = 0; n < 400; ++n) y[n] = 0.5f * sinf(0.05f * n) + 1e-5f * nd(rng);
    cf X[16][16];
    for (int c = 0; c < 16; ++c) {
      float v[25], w[25];
      for (int i = 0; i < 25; ++i) {
        v[i] = y[16 * i + c];
        w[i] = tb.window[16 * i + c];
      }
      cf a[16];
      sfe::rdft32_windowed(v, w, a);
      for (int k = 0; k < 16; ++k) X[k][c] = k == 0 ? a[0] : sfe::tan_twiddle(a[k], tb.tan512[c * 16 + k]);
    }
    std::vector<double> P(257, 0.0);
    for (int k1 = 1; k1 < 16; ++k1) {
      cf a[16];
      float ct[16];
      for (int c = 0; c < 16; ++c) {
        a[c] = X[k1][c];
        ct[c] = tb.cos512[k1 * 16 + c];
      }
      sfe::dft16_scaled(a, ct);
      for (int k2 = 0; k2 < 16; ++k2) {
        const int k = k1 + 32 * k2;
        P[k <= 256 ? k : 512 - k] = (double)fmaf(a[k2].y, a[k2].y, a[k2].x * a[k2].x);
      }
    }
    // the special columns: two half sums of each block, then added
    for (int q = 0; q < 8; ++q) {
      float row[2][4];
      for (int h = 0; h < 2; ++h)
        for (int i = 0; i < 4; ++i) {
          float acc = 0.0f;
          for (int s = 0; s < 8; ++s) {
            const float v = q < 4 ? X[0][8 * h + s].x : X[0][8 * h + s].y;
            acc = fmaf(reinterpret_cast<const float*>(&tb.special[s / 4][4 * (8 * h + q) + i])[s % 4], v, acc);
          }
          row[h][i] = acc;
        }
      for (int h = 0; h < 2; ++h) {
        const float re = row[0][2 * h] + row[1][2 * h], im = row[0][2 * h + 1] + row[1][2 * h + 1];
        P[sfe::special_bin(q, h)] = (double)fmaf(im, im, re * re);
      }
    }
    double nrm = 0;
    for (int n = 0; n < 400; ++n) nrm += pow((double)y[n] * tb.window[n], 2);
    // |X_k| to within a small multiple of u log2(N) |x| (the error any f32
    // FFT carries, independent of the bin)
    const double scale = u * 9.0 * sqrt(nrm) * sqrt(512.0);
    for (int k = 1; k <= 256; ++k) {
      C s = 0;
      for (int n = 0; n < 400; ++n) s += (double)y[n] * (double)tb.window[n] * root(k * n, 512);
      const double e = fabs(sqrt(P[k]) - std::abs(s)) / scale;
      emag = fmax(emag, e);
      if (k % 16 == 0) especial = fmax(especial, e);
      if (trial % 5 == 1 && std::abs(s) < 1e-3) equiet = fmax(equiet, e);
    }
  }
  check("frame |X_k|, max err / (u log2(512) |x| sqrt(512))", emag, 1.0);
  check("bins that are multiples of 16, same scale", especial, 1.0);
  check("low-energy bins of a loud tone, same scale", equiet, 1.0);

  // The mel schedule holds every nonzero weight of every filter exactly, and
  // reads bins 1 .. 256 only.
  std::vector<float> fb((size_t)sfe::kMel * sfe::kBins);
  sfe::mel_filterbank(sfe::kNfft, sfe::kMel, rate, fb.data());
  double wrong = 0;
  int first = 0;
  for (int i = 0; i < sfe::kMelSlots; ++i) {
    const int S = sfe::kMelSteps[tb.schedule][i];
    for (int L = 0; L < 64; ++L) {
      std::vector<float> row(sfe::kBins, 0.0f);
      const int k0 = tb.mel_k0[i][L];
      if (k0 < 1 || k0 + S > sfe::kBins) ++wrong;
      else
        for (int s = 0; s < S; ++s)
          row[k0 + s] = reinterpret_cast<const float*>(&tb.mel_w[(first + s) / 4][L])[(first + s) % 4];
      for (int k = 0; k < sfe::kBins; ++k) wrong += row[k] != fb[(size_t)(64 * i + L) * sfe::kBins + k];
    }
    first += S;
  }
  check("mel weights that differ from the filterbank", wrong, 0.0);

  // The raw layout: 32 frames x 128 features fill two tiles, each slot once.
  std::set<int64_t> slots;
  for (int f = 0; f < 32; ++f)
    for (int m = 0; m < sfe::kMel; ++m)
      slots.insert(sfe::raw_frame(f) + sfe::kRawSlab * (m / 16) + 4 * (m % 16));
  check("raw slots missing", 2.0 * sfe::kRawTile - (double)slots.size(), 0.0);
  check("raw slot range", (double)(*slots.rbegin() + 1), 2.0 * sfe::kRawTile);
  printf("bad %d\n", bad);
  return bad != 0;
}
