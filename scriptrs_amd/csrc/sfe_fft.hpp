// Register-level pieces of the log-mel kernel's 512-point real FFT, written
// for both the device and the host so that the host tests
// (tests/rdft_host_driver.cpp, tests/fft_host_driver.cpp) run the same
// arithmetic against float64 DFTs.
//
// The transform is 32 x 16: each of 16 lanes runs a real 32-point DFT over its
// registers (rdft32_windowed), the inter-stage twiddles are applied in tangent
// form (tan_twiddle), the block is transposed (through LDS in the kernel) and a
// complex 16-point DFT, the twiddles' cosines fused into its inner layer,
// finishes it (dft16_scaled).  Its instruction count is what the kernel's time
// goes to, so the constant multiplications are folded into fused multiply-adds:
//  * the window product of the first DFT's inputs goes into its first
//    additions (fma(v, w, .));
//  * an internal twiddle e^{-i theta} is written as cos(theta) (1 - i
//    tan(theta)) (theta = pi/8, 3pi/8 through 1/tan) or sqrt(1/2) (1 - i):
//    the bracket costs two fmas or two additions, and the common factor
//    (cos(pi/8) or sqrt(1/2)) multiplies the outer layer's additions as fmas.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace sfe {

struct __align__(8) cf {
  float x, y;
};

__host__ __device__ __forceinline__ cf cadd(cf a, cf b) { return {a.x + b.x, a.y + b.y}; }
__host__ __device__ __forceinline__ cf csub(cf a, cf b) { return {a.x - b.x, a.y - b.y}; }
// c + s v and c - s v for a real s
__host__ __device__ __forceinline__ cf cfma(float s, cf v, cf c) { return {fmaf(s, v.x, c.x), fmaf(s, v.y, c.y)}; }

namespace fftc {
constexpr float kR = 0.70710678118654752f;   // sqrt(1/2) = cos(pi/4)
constexpr float kC1 = 0.92387953251128674f;  // cos(pi/8)
constexpr float kT1 = 0.41421356237309505f;  // tan(pi/8)
}  // namespace fftc

// 4-point forward DFT in place on (a0, a1, a2, a3).
__host__ __device__ __forceinline__ void dft4(cf& a0, cf& a1, cf& a2, cf& a3) {
  const cf t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = csub(a1, a3);
  a0 = cadd(t0, t2);
  a2 = csub(t0, t2);
  a1 = {t1.x + t3.y, t1.y - t3.x};  // t1 - i t3
  a3 = {t1.x - t3.y, t1.y + t3.x};  // t1 + i t3
}

// The outputs of a radix-4 butterfly from t0 = v0 + v2, t1 = v0 - v2 and
// t2 = k s, t3 = k d (k real, applied here as fmas):
//   y0 = t0 + t2, y2 = t0 - t2, y1 = t1 - i t3, y3 = t1 + i t3.
__host__ __device__ __forceinline__ void bfly_out(cf t0, cf t1, float k, cf s, cf d, cf& y0, cf& y1, cf& y2,
                                                  cf& y3) {
  y0 = cfma(k, s, t0);
  y2 = cfma(-k, s, t0);
  y1 = {fmaf(k, d.y, t1.x), fmaf(-k, d.x, t1.y)};
  y3 = {fmaf(-k, d.y, t1.x), fmaf(k, d.x, t1.y)};
}

// u e^{-i pi/8} = cos(pi/8) g1(u), g1(u) = (x + y t, y - x t), t = tan(pi/8)
__host__ __device__ __forceinline__ cf g1(cf u) { return {fmaf(u.y, fftc::kT1, u.x), fmaf(-u.x, fftc::kT1, u.y)}; }
// u e^{-3 i pi/8} = cos(pi/8) g3(u), g3(u) = (x t + y, y t - x)
__host__ __device__ __forceinline__ cf g3(cf u) { return {fmaf(u.x, fftc::kT1, u.y), fmaf(u.y, fftc::kT1, -u.x)}; }

// Outer layer of a 16-point DFT: a[p + 4c] holds the inner layer's U[p][c]
// (inner DFT over q of the inputs m = p + 4q, output index c).  Applies the
// twiddles e^{-2 pi i p c / 16} and the 4-point DFTs over p, and leaves
// X[k] at a[k] (natural order).
__host__ __device__ __forceinline__ void dft16_outer(cf (&a)[16]) {
  using namespace fftc;
  cf y[16];
  // c = 0: no twiddles
  {
    cf v0 = a[0], v1 = a[1], v2 = a[2], v3 = a[3];
    dft4(v0, v1, v2, v3);
    y[0] = v0, y[4] = v1, y[8] = v2, y[12] = v3;
  }
  // c = 1: v1 = U e^{-i pi/8}, v2 = U e^{-i pi/4}, v3 = U e^{-3 i pi/8}
  {
    const cf u2 = {a[6].x + a[6].y, a[6].y - a[6].x};  // v2 = kR u2
    const cf t0 = cfma(kR, u2, a[4]), t1 = cfma(-kR, u2, a[4]);
    const cf h1 = g1(a[5]), h3 = g3(a[7]);               // v1 = kC1 h1, v3 = kC1 h3
    bfly_out(t0, t1, kC1, cadd(h1, h3), csub(h1, h3), y[1], y[5], y[9], y[13]);
  }
  // c = 2: v1 = U e^{-i pi/4}, v2 = U e^{-i pi/2} = -i U, v3 = U e^{-3 i pi/4}
  {
    const cf t0 = {a[8].x + a[10].y, a[8].y - a[10].x};
    const cf t1 = {a[8].x - a[10].y, a[8].y + a[10].x};
    const cf u1 = {a[9].x + a[9].y, a[9].y - a[9].x};       // v1 = kR u1
    const float w = a[11].x + a[11].y;
    const cf u3 = {a[11].y - a[11].x, -w};                 // v3 = kR u3
    bfly_out(t0, t1, kR, cadd(u1, u3), csub(u1, u3), y[2], y[6], y[10], y[14]);
  }
  // c = 3: v1 = U e^{-3 i pi/8}, v2 = U e^{-3 i pi/4}, v3 = U e^{-9 i pi/8} = -U e^{-i pi/8}
  {
    const cf u2 = {a[14].y - a[14].x, -(a[14].x + a[14].y)};  // v2 = kR u2
    const cf t0 = cfma(kR, u2, a[12]), t1 = cfma(-kR, u2, a[12]);
    const cf h1 = g3(a[13]), h3 = g1(a[15]);                 // v1 = kC1 h1, v3 = -kC1 h3
    bfly_out(t0, t1, kC1, csub(h1, h3), cadd(h1, h3), y[3], y[7], y[11], y[15]);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) a[i] = y[i];
}

// Inter-stage twiddle in tangent form: a e^{-i theta} = cos(theta) g with
// g = (x + y tan(theta), y - x tan(theta)), two fmas; the cosine is applied
// by the next stage (dft16_scaled).
__host__ __device__ __forceinline__ cf tan_twiddle(cf a, float t) {
  return {fmaf(a.y, t, a.x), fmaf(-a.x, t, a.y)};
}

// 16-point forward DFT of the inputs c[m] a[m] (real scale factors, c[0] =
// 1 and not read), into a[k], natural order.  The scales are fused into the
// inner layer: per inner DFT (inputs p, p + 4, p + 8, p + 12) the first
// input of each pair is scaled by a multiplication and the second by the
// fmas of the pair's sum and difference.
__host__ __device__ __forceinline__ void dft16_scaled(cf (&a)[16], const float (&c)[16]) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const cf x0 = p == 0 ? a[0] : cf{c[p] * a[p].x, c[p] * a[p].y};
    const cf x1 = {c[p + 4] * a[p + 4].x, c[p + 4] * a[p + 4].y};
    const float c2 = c[p + 8], c3 = c[p + 12];
    const cf t0 = cfma(c2, a[p + 8], x0), t1 = cfma(-c2, a[p + 8], x0);
    const cf t2 = cfma(c3, a[p + 12], x1), t3 = cfma(-c3, a[p + 12], x1);
    a[p] = cadd(t0, t2);
    a[p + 8] = csub(t0, t2);
    a[p + 4] = {t1.x + t3.y, t1.y - t3.x};   // t1 - i t3
    a[p + 12] = {t1.x - t3.y, t1.y + t3.x};  // t1 + i t3
  }
  dft16_outer(a);
}

// 8-point DCT-II of g[0..5], 0, 0: sum over i of g[i] cos(pi k (2 i + 1) /
// 16), as x[k] times the scale kDct8[k], which the caller applies in its
// fmas.
namespace fftc {
constexpr float kK1 = 0.98078528040323045f;  // cos(pi/16)
constexpr float kA3 = 0.84775906502257351f;  // cos(3 pi/16) / cos(pi/16)
constexpr float kA5 = 0.56645449735052156f;  // cos(5 pi/16) / cos(pi/16)
constexpr float kA7 = 0.19891236737965801f;  // cos(7 pi/16) / cos(pi/16)
}  // namespace fftc
__host__ __device__ __forceinline__ void dct8_6(const float (&g)[6], float (&x)[8]) {
  using namespace fftc;
  const float s2 = g[2] + g[5], d2 = g[2] - g[5];
  const float s3 = g[3] + g[4], d3 = g[3] - g[4];
  const float a = g[0] + s3, c = g[0] - s3;
  const float b = g[1] + s2, d = g[1] - s2;
  x[0] = a + b;
  x[4] = a - b;
  x[2] = fmaf(kT1, d, c);
  x[6] = fmaf(kT1, c, -d);
  x[1] = fmaf(kA7, d3, fmaf(kA5, d2, fmaf(kA3, g[1], g[0])));
  x[3] = fmaf(-kA3, g[0], fmaf(kA7, g[1], fmaf(kA5, d3, d2)));
  x[5] = fmaf(-kA3, d3, fmaf(-kA7, d2, fmaf(-kA5, g[0], g[1])));
  x[7] = fmaf(-kA7, g[0], fmaf(kA5, g[1], fmaf(-kA3, d2, d3)));
}

// 32-point DFT of the real, windowed inputs v[i] = w[i] y[i] at positions b
// = i - 12 (i < 25; the other 7 positions are zero), into Y[k] = sum over b
// of v e^{-2 pi i k b / 32}: Y[k] at y[k] for 0 < k < 16, and the real Y[0]
// and Y[16] as y[0] = (Y[0], Y[16]).
//
// With the origin at the middle input, the real part takes the sums of the
// pairs +-b and the imaginary part their differences (the window product
// rides in both), and each half splits again by the parity of b: cosines or
// sines of even b are a 16-point transform of the same kind, those of odd b
// an 8-point DCT-II (dct8_6; sin(pi k m / 16) = +-cos(pi (8 - k) m / 16) for
// odd m).  153 operations.
__host__ __device__ __forceinline__ void rdft32_windowed(const float (&y)[25], const float (&w)[25], cf (&Y)[16]) {
  using namespace fftc;
  float e[13], o[13];
#pragma unroll
  for (int b = 1; b <= 12; ++b) {
    const float m = w[12 - b] * y[12 - b];
    e[b] = fmaf(w[12 + b], y[12 + b], m);
    // odd b: the sign (-1)^((b - 1) / 2) of the sine's DCT-II form
    o[b] = b % 4 == 3 ? fmaf(-w[12 + b], y[12 + b], m) : fmaf(w[12 + b], y[12 + b], -m);
  }
  e[0] = w[12] * y[12];
  // cosines, even b: ev[k] = sum over j of e[2 j] cos(pi k j / 8), k <= 8
  float ev[9], od[8];
  {
    const float u = e[0] + e[8], d = e[0] - e[8], p = e[4] + e[12], q = e[4] - e[12];
    const float g = e[6] + e[10], t = e[6] - e[10];
    const float z0 = u + p, z1 = fmaf(kR, q, e[0]), z3 = fmaf(-kR, q, e[0]);
    const float o0 = e[2] + g, o2 = e[2] - g, o1 = fmaf(kT1, t, e[2]), o3 = fmaf(kT1, e[2], -t);
    ev[0] = z0 + o0;
    ev[8] = z0 - o0;
    ev[1] = fmaf(kC1, o1, z1);
    ev[7] = fmaf(-kC1, o1, z1);
    ev[2] = fmaf(kR, o2, d);
    ev[6] = fmaf(-kR, o2, d);
    ev[3] = fmaf(kC1, o3, z3);
    ev[5] = fmaf(-kC1, o3, z3);
    ev[4] = u - p;
    const float h[6] = {e[1], e[3], e[5], e[7], e[9], e[11]};
    dct8_6(h, od);
  }
  // sines, even b: se[k] = sum over j of o[2 j] sin(pi k j / 8), 1 <= k <= 7
  float se[8], so[8];
  {
    const float v = o[4] + o[12], s2 = o[4] - o[12], s1 = fmaf(kR, v, o[8]), s3 = fmaf(kR, v, -o[8]);
    const float m1 = o[6] + o[10], m2 = o[6] - o[10];
    const float h1 = fmaf(kT1, o[2], m1), h3 = fmaf(-kT1, m1, o[2]), h2 = o[2] + m2;
    se[1] = fmaf(kC1, h1, s1);
    se[7] = fmaf(kC1, h1, -s1);
    se[2] = fmaf(kR, h2, s2);
    se[6] = fmaf(kR, h2, -s2);
    se[3] = fmaf(kC1, h3, s3);
    se[5] = fmaf(kC1, h3, -s3);
    se[4] = o[2] - m2;
    const float h[6] = {o[1], o[3], o[5], o[7], o[9], o[11]};
    dct8_6(h, so);  // so[8 - k]: the sum over odd b at k
  }
  constexpr float sc[8] = {1.0f, kK1, kC1, -kK1, kR, -kK1, kC1, -kK1};
  Y[0] = {ev[0] + od[0], ev[0] - od[0]};
  Y[8] = {ev[8], -so[0]};
#pragma unroll
  for (int k = 1; k < 8; ++k) {
    Y[k].x = fmaf(sc[k], od[k], ev[k]);
    Y[16 - k].x = fmaf(-sc[k], od[k], ev[k]);
    Y[k].y = fmaf(-sc[8 - k], so[8 - k], -se[k]);
    Y[16 - k].y = fmaf(-sc[8 - k], so[8 - k], se[k]);
  }
}

}  // namespace sfe
