// Host-side construction of the constant tables the kernels read.
//
// hann_window and mel_filterbank follow src/frontend.rs:161-223 with the
// reference's operation order and precision (f32 for the window, f64 for
// the mel points and triangle weights with an f32 cast, then an f32
// multiply by the f32-cast Slaney norm).  This file is built with
// -ffp-contract=off so each operation rounds as in the reference.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "sfe_internal.hpp"

namespace sfe {

void hann_window(int win, float* out) {
  const float pi = 3.14159265358979323846f;  // std::f32::consts::PI
  for (int n = 0; n < win; ++n) {
    float num = (2.0f * pi) * (float)n;
    float den = (float)win - 1.0f;
    out[n] = 0.5f - 0.5f * cosf(num / den);
  }
}

namespace {
const double kFsp = 200.0 / 3.0;            // F_SP, src/frontend.rs:167
const double kMinLogHz = 1000.0;            // MIN_LOG_HZ
const double kLogStep = 0.06875177742094912;  // LOG_STEP = ln(6.4)/27

double hz_to_mel(double hz) {
  const double min_log_mel = kMinLogHz / kFsp;
  return hz < kMinLogHz ? hz / kFsp : min_log_mel + log(hz / kMinLogHz) / kLogStep;
}

double mel_to_hz(double mel) {
  const double min_log_mel = kMinLogHz / kFsp;
  return mel < min_log_mel ? mel * kFsp : kMinLogHz * exp((mel - min_log_mel) * kLogStep);
}
}  // namespace

void mel_filterbank(int n_fft, int n_mels, int sample_rate, float* out) {
  const int bins = n_fft / 2 + 1;
  const double mel_min = hz_to_mel(0.0);
  const double mel_max = hz_to_mel((double)sample_rate / 2.0);
  std::vector<double> pts(n_mels + 2), freqs(bins), diffs(n_mels + 1);
  for (int i = 0; i <= n_mels + 1; ++i)
    pts[i] = mel_to_hz(mel_min + (mel_max - mel_min) * (double)i / (double)(n_mels + 1));
  for (int k = 0; k < bins; ++k) freqs[k] = (double)k * (double)sample_rate / (double)n_fft;
  for (int i = 0; i <= n_mels; ++i) diffs[i] = pts[i + 1] - pts[i];
  for (int m = 0; m < n_mels; ++m)
    for (int k = 0; k < bins; ++k) {
      double lower = (freqs[k] - pts[m]) / diffs[m];
      double upper = (pts[m + 2] - freqs[k]) / diffs[m + 1];
      double v = lower < upper ? lower : upper;
      out[(size_t)m * bins + k] = (float)(v > 0.0 ? v : 0.0);
    }
  for (int m = 0; m < n_mels; ++m) {
    float enorm = (float)(2.0 / (pts[m + 2] - pts[m]));
    for (int k = 0; k < bins; ++k) out[(size_t)m * bins + k] *= enorm;
  }
}

namespace {
// Chooses k0[j] >= 1 in (hi[j] - S, lo[j]] with distinct k0[j] mod 16, as far as a
// matching (augmenting paths) finds one; the others keep lo[j].
void spread_banks(const int (&lo)[16], const int (&hi)[16], int S, int (&k0)[16]) {
  int owner[16];  // bank group -> lane
  for (int& o : owner) o = -1;
  struct Search {
    const int (&lo)[16];
    const int (&hi)[16];
    int S;
    int (&k0)[16];
    int (&owner)[16];
    bool seen[16];
    bool place(int j) {
      for (int k = lo[j]; k >= 1 && k > hi[j] - S; --k) {
        const int u = k % 16;
        if (seen[u]) continue;
        seen[u] = true;
        if (owner[u] < 0 || place(owner[u])) {
          owner[u] = j;
          k0[j] = k;
          return true;
        }
      }
      return false;
    }
  };
  for (int j = 0; j < 16; ++j) {
    Search s{lo, hi, S, k0, owner, {}};
    s.place(j);
  }
}
}  // namespace

bool build_dev_tables(int sample_rate, DevTables* t) {
  memset(t, 0, sizeof(*t));
  hann_window(kWin, t->window);
  for (int k = 0; k < 16; ++k)
    for (int c = 0; c < 16; ++c) {
      const double th = 2.0 * M_PI * (double)(k * c) / 512.0;
      t->tan512[k * 16 + c] = (float)(sin(th) / cos(th));
      t->cos512[k * 16 + c] = (float)cos(th);
    }
  for (int L = 0; L < 64; ++L) {
    // rows i = 0..3 of a block: real and imaginary parts of its two bins
    const int j = L / 4, i = L % 4, bin = special_bin(j % 8, i / 2);
    for (int s = 0; s < 8; ++s) {
      const int m = (bin * (8 * (j / 8) + s)) % 512;  // a multiple of 16
      const double th = 2.0 * M_PI * (double)m / 512.0;
      const bool zero = i % 2 == 0 ? m % 256 == 128 : m % 256 == 0;
      reinterpret_cast<float*>(&t->special[s / 4][L])[s % 4] = zero ? 0.0f : (float)(i % 2 == 0 ? cos(th) : -sin(th));
    }
  }
  std::vector<float> fb((size_t)kMel * kBins);
  mel_filterbank(kNfft, kMel, sample_rate, fb.data());
  // The sample rates taken and their schedule follow from the band edges of
  // blocks of 4 filters: from a first bin that is a multiple of 4, the blocks
  // of filters 0..63 span at most 8 bins and those of 64..127 at most 32
  // (schedule 0), or 12 and 48 (schedule 1, which may also run 3 bins past
  // the spectrum).  Rates outside are refused; the slots of kMelSteps hold
  // every filter of those inside.
  auto fits = [&](int low, int high, int bins) -> bool {
    for (int f0 = 0; f0 < kMel; f0 += 4) {
      const int S = f0 < 64 ? low : high;
      int lo = -1, hi = -1;
      for (int m = f0; m < f0 + 4; ++m)
        for (int k = 0; k < kBins; ++k)
          if (fb[(size_t)m * kBins + k] != 0.0f) {
            if (lo < 0 || k < lo) lo = k;
            if (k > hi) hi = k;
          }
      if (lo < 0) lo = hi = 0;
      int k0 = lo / 4 * 4;
      if (k0 + S > bins) k0 = (bins - S) / 4 * 4;
      if (lo < k0 || hi >= k0 + S) return false;
    }
    return true;
  };
  if (fits(8, 32, kBins)) t->schedule = 0;
  else if (fits(12, 48, kBins + 3)) t->schedule = 1;
  else return false;
  int first = 0;  // steps before the slot's
  for (int i = 0; i < kMelSlots; ++i) {
    const int S = kMelSteps[t->schedule][i];
    for (int g = 0; g < 64; g += 16) {
      int lo[16], hi[16], k0[16];
      for (int j = 0; j < 16; ++j) {
        const float* f = &fb[(size_t)(64 * i + g + j) * kBins];
        lo[j] = 0, hi[j] = kBins - 1;
        while (lo[j] < kBins && f[lo[j]] == 0.0f) ++lo[j];
        while (hi[j] > lo[j] && f[hi[j]] == 0.0f) --hi[j];
        if (lo[j] == kBins) lo[j] = hi[j] = 1;  // an all-zero filter
        lo[j] = std::min(lo[j], kBins - S);
        if (hi[j] >= lo[j] + S) return false;
        k0[j] = lo[j];
      }
      // Bin 0 has no weight at any rate (0 Hz is the first filter's edge) and
      // is never read: the kernel leaves it undefined.
      // 16 lanes' 16-byte reads of power bins fall on 16 groups of banks:
      // slot 1's filters are wider apart than the first bins of slot 0's,
      // which mostly share bins, so where the slot is wider than the filter
      // its first bin is moved down to spread them.
      if (i == 1) spread_banks(lo, hi, S, k0);
      for (int j = 0; j < 16; ++j) {
        const float* f = &fb[(size_t)(64 * i + g + j) * kBins];
        t->mel_k0[i][g + j] = k0[j];
        for (int s = 0; s < S; ++s)
          reinterpret_cast<float*>(&t->mel_w[(first + s) / 4][g + j])[(first + s) % 4] = f[k0[j] + s];
      }
    }
    first += S;
  }
  return true;
}

}  // namespace sfe
