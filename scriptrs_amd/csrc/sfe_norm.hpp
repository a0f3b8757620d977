// The normalisation (normalize_columns, src/frontend.rs:225-241): device code
// and launches, compiled into two code objects.  sfe_kernels.hip holds the
// kernels of items whose quads are quads of their regions (SHIFT = false, every
// call of the long-form planner), sfe_norm_shift.hip those of calls with items
// that start inside a quad of their shared region, four instances of each body.
// A process loads a code object with its first kernel: with both in one, the
// first call of a process took 3.9 ms instead of 2.7.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sfe_internal.hpp"
#include "sfe_rounds.hpp"
#include "sfe_seqsum.hpp"

namespace sfe {

// Measurement builds (compiled with -DSFE_TIMESTAMPS, never the product
// library): the kernels write s_memrealtime stamps (a 100 MHz clock shared
// by all CUs) into a device buffer the host registers with
// sfe_debug_stamps.  Log-mel: per wave (blockIdx * waves + wave) 8 words at
// kStampLogmel: start, loop entry (end of the prologue), end, units
// processed, (unused), item descriptors loaded (after their first use).
// (A stamp after the workgroup barrier of the mel table made the compiler
// spill registers in the main loop, so there is none.)  Normalisation: per
// workgroup 4 words at kStampNorm: start, first statistics reduced (its loads
// have landed), statistics published, end.  Every launch overwrites its
// region.
#ifdef SFE_TIMESTAMPS
constexpr int64_t kStampLogmel = 0;
constexpr int64_t kStampNorm = 8 * 65536;
__device__ unsigned long long* g_stamps;
__device__ long long g_stamp_words;
__device__ __forceinline__ void stamp(int64_t word, unsigned long long v) {
  if (g_stamps && word < g_stamp_words) g_stamps[word] = v;
}
__device__ __forceinline__ unsigned long long stamp_now() { return __builtin_amdgcn_s_memrealtime(); }
#define SFE_STAMP(word, value) stamp((word), (value))
#else
#define SFE_STAMP(word, value) ((void)0)
#endif

namespace {

constexpr float kLn2 = 0.69314718055994531f;

// Raw value loaded by the normalisation kernel: RN(log2 * ln 2).
__device__ __forceinline__ float4 ln2_scale(float4 v) {
#pragma clang fp contract(off)  // rounded on its own, never fused into a later add
  return make_float4(v.x * kLn2, v.y * kLn2, v.z * kLn2, v.w * kLn2);
}

__device__ __forceinline__ float ln2_scale(float v) {
#pragma clang fp contract(off)
  return v * kLn2;
}

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);                                            // round to nearest even
  return (uint16_t)(u >> 16);
}

// Statistics of a row whose values are all bitwise equal to x0: digital
// silence, and at sample rates past 24 kHz every row of a filter so narrow that
// it holds no bin.  This is where the reference's sequential f32 sums decide
// the result: their rounding leaves x - mean != 0 (about +-0.93 for digital
// silence), so the sums are those of its loops (src/frontend.rs:230-236).
//
// What bounds it: a serial chain on one lane, while the rest of the workgroup
// waits, in every workgroup of a long item (norm_finish).  Walking the row is
// 2 T dependent additions, a sequential_sum about 4 per doubling of T.  Calls
// with the rows walked / as sequential sums: 24 silent clips of 90 s 1200 /
// 164 us (406 when one workgroup normalised a whole long item), 8 of 15 s 63 /
// 28, 64 clips of 480,000 samples at 48 kHz 406 / 140.
__device__ __forceinline__ void constant_row_stats(float x0, int T, float* mean_out, float* sd_out) {
#pragma clang fp contract(off)  // every f32 operation rounded, as the reference's
  float a = x0, mean = 0.0f, var = 0.0f;
#pragma unroll 1  // one copy of the sum's code: the store phase follows it
  for (int pass = 0; pass < 2; ++pass) {
    const float sum = sequential_sum(a, T);
    if (pass == 0) {
      mean = __fdiv_rn(sum, (float)T);
      const float d = x0 - mean;
      a = d * d;
    } else {
      var = __fdiv_rn(sum, (float)T - 1.0f);
    }
  }
  *mean_out = mean;
  *sd_out = __fsqrt_rn(var) + 1e-5f;
}

// normalize_columns (src/frontend.rs:225-241).  Input: raw log-mel in
// 16-frame tiles of 8 slabs (as the log-mel kernel writes it).
// Output: feature-major ([128][T] per item, the reference's memory order).
//
// One workgroup of W waves per (item, slab of 16 features).  Loads: in round
// j, lane i of wave v holds the 4 frames of quad 4 (W j + v) + i / 16 of
// feature i % 16, one float4, and a wave's load is 1 KB of one raw tile.
// Items of up to 16 W N frames are read from HBM once and held in registers
// (N float4s per lane); longer ones go in segments (norm_segment).  Stores: chunks
// of 4 rounds are transposed through LDS and each lane writes 4 consecutive
// frames of one feature row, so a store instruction covers 16 / W rows of
// contiguous bytes (rows are only 4-byte aligned when T is odd; gfx950 takes
// unaligned 16-byte stores).
//
// Statistics: per quad (4 frames of one feature, the same quads whatever the
// workgroup's shape) the f32 sum of (x - x0) (x0 the feature's first value)
// is accumulated in f64, then reduced across lanes by shuffles and across
// waves through LDS, always in the same order, so results are deterministic;
// the sum of squared deviations from the f32 mean likewise.  Then out = (x -
// mean) / (sqrt(var) + 1e-5) in f32, var over T - 1 (T == 1 gives NaN, as the
// reference).  A feature whose values are all equal (squared deviations that
// sum to exactly 0: the f32 mean is then that value) replays the reference's
// sequential f32 sums (constant_row_stats).
constexpr int kSlabF = 16;  // features per slab
constexpr int kSlabs = kMel / kSlabF;
// Fourth word of a raw buffer resource (no format conversion, no swizzle).
constexpr int kBufWord3 = 0x00020000;

// Shape of a normalisation workgroup of W waves.
template <int W>
struct NormShape {
  static constexpr int kThreads = 64 * W;
  static constexpr int kSpan = kTile * W;                 // frames per round
  static constexpr int kChunk = 4 * kSpan;                // frames per LDS transpose
  static constexpr int kTStride = kChunk + 4;             // LDS row stride (floats), rows 16-byte aligned
  static constexpr int kRowsPerWave = kSlabF / W;
  static constexpr int kLanesPerRow = 64 / kRowsPerWave;  // each writes 4 frames per store
  static_assert(4 * kLanesPerRow == kSpan, "a store instruction covers one round of a row");
};

// A normalisation workgroup's LDS.  Two transpose buffers in the 4-wave form
// (chunk ch stages into tb[ch % 2]: the next chunk's staging does not wait for
// this chunk's stores, one barrier per chunk); one in the 8-wave form, whose
// buffer is twice as large.
constexpr int kSumParts = 8;
template <int W>
struct NormLds {
  static constexpr int kTBufs = W == 4 ? 2 : 1;
  double red[kSumParts * kSlabF];
  float st[3 * kSlabF];
  __attribute__((aligned(16))) float tb[kTBufs][kSlabF * NormShape<W>::kTStride];
};

// Workgroup sum over the lanes that hold the same feature (lane % 16 equal)
// and the waves; every lane gets its own feature's total.  v[k] holds the
// lane's sum over rounds j = k mod 8 / W: tile 4 j + w of a 4-wave workgroup is
// tile 8 (j / 2) + w + 4 (j % 2) of an 8-wave one, so both add the same 8 sums
// in the same order and the results do not depend on the form.
template <int W>
__device__ __forceinline__ double slab_sum(double (&v)[kSumParts / W], double* red, int lane, int w) {
#pragma unroll
  for (int k = 0; k < kSumParts / W; ++k) {
    v[k] += __shfl_xor(v[k], 16, 64);
    v[k] += __shfl_xor(v[k], 32, 64);
    if (lane < kSlabF) red[(w + W * k) * kSlabF + lane] = v[k];
  }
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int u = 0; u < kSumParts; ++u) t += red[u * kSlabF + lane % kSlabF];
  __syncthreads();  // red is reused by the next reduction
  return t;
}

// (x - mean) / sd, correctly rounded, from r = RN(1 / sd): q = RN(d r) is
// within one ulp of d / sd, and one residual step q + r fma(-sd, q, d)
// rounds to RN(d / sd) (Markstein's theorem; d and sd are far from overflow
// and underflow here).  Three VALU operations instead of a full division.
__device__ __forceinline__ float norm_div(float x, float mean, float sd, float r) {
  const float d = __fsub_rn(x, mean);
  const float q = __fmul_rn(d, r);
  return __fmaf_rn(__fmaf_rn(-sd, q, d), r, q);
}

// f32 mean from the sum S of (x - x0) over T values.
__device__ __forceinline__ float row_mean(float x0, double S, int T) { return (float)((double)x0 + S / (double)T); }

// Per-feature (mean, sd, 1/sd) of the slab, published in LDS for the store
// phase by wave 0's lanes 0..15, one feature each.  S: sum of (x - x0), Q:
// sum of squared deviations from the f32 mean.
__device__ __forceinline__ void publish_stats(double S, double Q, bool constant, float x0, int T, int lane, int w,
                                              float* st) {
  if (w == 0 && lane < kSlabF) {
    float mean, sd;
    if (__builtin_expect(constant, 0)) {
      constant_row_stats(x0, T, &mean, &sd);
    } else {
      mean = row_mean(x0, S, T);
      sd = __fadd_rn(__fsqrt_rn((float)(Q / (double)(T - 1))), 1e-5f);
    }
    st[3 * lane] = mean;
    st[3 * lane + 1] = sd;
    st[3 * lane + 2] = __fdiv_rn(1.0f, sd);
  }
  __syncthreads();
}

__device__ __forceinline__ void put4(float* o, float4 y) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  *reinterpret_cast<f4u*>(o) = f4u{y.x, y.y, y.z, y.w};
}
__device__ __forceinline__ void put4(uint16_t* o, float4 y) {
  typedef uint16_t u4u __attribute__((ext_vector_type(4), aligned(2)));
  *reinterpret_cast<u4u*>(o) = u4u{f32_to_bf16(y.x), f32_to_bf16(y.y), f32_to_bf16(y.z), f32_to_bf16(y.w)};
}
__device__ __forceinline__ void put1(float* o, float y) { *o = y; }
__device__ __forceinline__ void put1(uint16_t* o, float y) { *o = f32_to_bf16(y); }

// Store phase of one chunk: its frames are in tb[16][kTStride]
// (feature-major); wave v writes rows R v .. R v + R - 1 (R = 16 / W).
template <int W, typename O>
__device__ __forceinline__ void store_chunk(const float* tb, const float* st, int t0, int T, int rs, int lane, int w,
                                            O* __restrict__ ob) {
  using S = NormShape<W>;
  const int r = S::kRowsPerWave * w + lane / S::kLanesPerRow;
  const float mean = st[3 * r], sd = st[3 * r + 1], rc = st[3 * r + 2];
  O* orow = ob + (size_t)r * rs;
#pragma unroll
  for (int s = 0; s < S::kChunk / S::kSpan; ++s) {
    const int k = 4 * (lane % S::kLanesPerRow) + S::kSpan * s;
    const float4 x = *reinterpret_cast<const float4*>(tb + r * S::kTStride + k);
    const float4 y = make_float4(norm_div(x.x, mean, sd, rc), norm_div(x.y, mean, sd, rc),
                                 norm_div(x.z, mean, sd, rc), norm_div(x.w, mean, sd, rc));
    const int t = t0 + k;
    if (t + 3 < T) {
      put4(orow + t, y);
    } else {
      if (t < T) put1(orow + t, y.x);
      if (t + 1 < T) put1(orow + t + 1, y.y);
      if (t + 2 < T) put1(orow + t + 2, y.z);
    }
  }
}

// Zeroes frames [T, rs) of the slab's 16 rows (the encoder-input padding,
// src/model.rs:266-271).
template <int W, typename O>
__device__ __forceinline__ void zero_tail(O* __restrict__ ob, int T, int rs, int lane, int w) {
  const int tail = rs - T;
  for (int e = w * 64 + lane; e < kSlabF * tail; e += W * 64) put1(ob + (size_t)(e / tail) * rs + T + e % tail, 0.0f);
}

template <int W>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t round_buffer(const Rounds<W>& rd) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(rd.base), 0, kNormBufRange, kBufWord3);
}

// The lane's N quads (Rounds): raw buffer loads from the uniform base, all
// issued before any is used (a load under a per-lane branch would wait for
// itself).  One 16-byte load a quad where the item's quads are quads of its
// regions (SHIFT = 0); the 4 - SHIFT frames from one quad of the shared region
// and the SHIFT from the next in two loads where it starts inside one.
template <int SHIFT, int W, int N>
__device__ __forceinline__ void load_rounds(const Rounds<W>& rd, float4 (&v)[N]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef float f32x3 __attribute__((ext_vector_type(3)));
  const __amdgpu_buffer_rsrc_t rsrc = round_buffer(rd);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if constexpr (SHIFT == 0) {
      v[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, rd.buf_off(j), 0, 0));
    } else {
      const int o0 = rd.template elem_off<SHIFT>(j, 0), o1 = rd.template elem_off<SHIFT>(j, kQuad - SHIFT);
      if constexpr (SHIFT == 1) {
        const f32x3 a = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(rsrc, o0, 0, 0));
        const float b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, o1, 0, 0));
        v[j] = make_float4(a.x, a.y, a.z, b);
      } else if constexpr (SHIFT == 2) {
        const f32x2 a = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, o0, 0, 0));
        const f32x2 b = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, o1, 0, 0));
        v[j] = make_float4(a.x, a.y, b.x, b.y);
      } else {
        const float a = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, o0, 0, 0));
        const f32x3 b = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(rsrc, o1, 0, 0));
        v[j] = make_float4(a, b.x, b.y, b.z);
      }
      __builtin_amdgcn_sched_barrier(0);  // one round's addresses at a time: they take registers beside v
    }
  }
  // (Left to itself the scheduler moves the first uses, and their waits, up
  // among the loads.)
  __builtin_amdgcn_sched_barrier(0);
}

// Adds the f32 sum over a quad of (x - p) to s; elements past the item (index >= n)
// left out.  (all is uniform and rarely false: an empty asm keeps the masked
// form behind a branch, another the sum where it is written; moved past the
// branches of later rounds, it would keep all their differences allocated.)
__device__ __forceinline__ void add_dev(double& s, const float4& v, float p, bool all, int n) {
  float d0 = v.x - p, d1 = v.y - p, d2 = v.z - p, d3 = v.w - p;
  if (!all) {
    asm volatile("" : "+v"(n));
    d0 = n > 0 ? d0 : 0.0f;
    d1 = n > 1 ? d1 : 0.0f;
    d2 = n > 2 ? d2 : 0.0f;
    d3 = n > 3 ? d3 : 0.0f;
  }
  s += (double)((d0 + d1) + (d2 + d3));
  asm volatile("" : "+v"(s));
}
// The same of (x - p)^2.
__device__ __forceinline__ void add_sq(double& s, const float4& v, float p, bool all, int n) {
  float d0 = v.x - p, d1 = v.y - p, d2 = v.z - p, d3 = v.w - p;
  if (!all) {
    asm volatile("" : "+v"(n));
    d0 = n > 0 ? d0 : 0.0f;
    d1 = n > 1 ? d1 : 0.0f;
    d2 = n > 2 ? d2 : 0.0f;
    d3 = n > 3 ? d3 : 0.0f;
  }
  s += (double)(fmaf(d1, d1, d0 * d0) + fmaf(d3, d3, d2 * d2));
  asm volatile("" : "+v"(s));
}

// W waves, N float4 registers per lane: an item of up to 16 W N frames, held
// in registers and read once.  Every N sums the same quads, so the class does
// not change the result.  `work` is the (item, slab) index; items longer than
// kNormRegFrames are left to norm_segment and norm_finish.
template <int SHIFT, int W, int N, typename O>
__device__ __forceinline__ void norm_body(const float* __restrict__ raw, const Item* __restrict__ items, int work,
                                          int pad_to, O* __restrict__ out, NormLds<W>& lds) {
  static_assert(N % 4 == 0, "whole chunks");
  using S = NormShape<W>;
  constexpr int kSpan = S::kSpan;
  constexpr int kChunk = S::kChunk;
  constexpr int kTBufs = NormLds<W>::kTBufs;
  double* red = lds.red;
  float* st = lds.st;
  const int item = work / kSlabs;
#ifdef SFE_TIMESTAMPS
  const int64_t sn = kStampNorm + 4 * (int64_t)work;
  if (threadIdx.x == 0) SFE_STAMP(sn, stamp_now());
#endif
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int slab = work % kSlabs;
  const Item it = items[item];
  const int T = it.T;
  if (T > kNormRegFrames) return;
  const Rounds<W> rd(raw, it, slab, lane, w, 0);
  const int rs = pad_to > 0 ? pad_to : T;  // output row length
  O* ob = out + it.dst_off + (size_t)(kSlabF * slab) * rs;
  if (pad_to > 0) zero_tail<W>(ob, T, rs, lane, w);
  // Frame 0 is always at out_off: below f_lo for an item that shares frames,
  // and an item with its own region has grid_off = out_off.
  const float x0 = ln2_scale(raw[it.out_off + kRawSlab * slab + 4 * (lane & 15)]);
  // The chunk's columns of this lane's quads.
  auto stage = [&](float* t, int jr, const float4& v) {
    *reinterpret_cast<float4*>(t + (lane & 15) * S::kTStride + kSpan * jr + kQuad * rd.q) = v;
  };
  const int chunks = (T + kChunk - 1) / kChunk;

  constexpr int K = kSumParts / W;
  double sp[K] = {}, qp[K] = {};
  float4 v[N];
  // (Loads in place, without load_rounds or a barrier behind them: the schedules
  // that the compiler makes of those forms took 75.0 to 76.1 us of normalisation
  // on the 1 h recording, this one 74.1, between events.)
  if constexpr (SHIFT == 0) {
    const __amdgpu_buffer_rsrc_t rsrc = round_buffer(rd);
#pragma unroll
    for (int j = 0; j < N; ++j)
      v[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, rd.buf_off(j), 0, 0));
  } else {
    load_rounds<SHIFT>(rd, v);
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    v[j] = ln2_scale(v[j]);
    add_dev(sp[j % K], v[j], x0, Rounds<W>::full(j, T), rd.left - kSpan * j);
  }
  const double s = slab_sum<W>(sp, red, lane, w);
#ifdef SFE_TIMESTAMPS
  if (threadIdx.x == 0) SFE_STAMP(sn + 1, stamp_now());
#endif
  const float m = row_mean(x0, s, T);
#pragma unroll
  for (int j = 0; j < N; ++j) add_sq(qp[j % K], v[j], m, Rounds<W>::full(j, T), rd.left - kSpan * j);
  const double sq = slab_sum<W>(qp, red, lane, w);
  publish_stats(s, sq, sq == 0.0, x0, T, lane, w, st);
#ifdef SFE_TIMESTAMPS
  if (threadIdx.x == 0) SFE_STAMP(sn + 2, stamp_now());
#endif
#pragma unroll
  for (int ch = 0; ch < N / 4; ++ch) {
    if (ch < chunks) {
      float* t = lds.tb[ch % kTBufs];
#pragma unroll
      for (int jr = 0; jr < 4; ++jr) stage(t, jr, v[4 * ch + jr]);
      __syncthreads();
      store_chunk<W>(t, st, kChunk * ch, T, rs, lane, w, ob);
      if (kTBufs == 1) __syncthreads();
    }
  }
#ifdef SFE_TIMESTAMPS
  if (threadIdx.x == 0) SFE_STAMP(sn + 3, stamp_now());
#endif
}

// Workgroups of kNormMainWaves waves; workgroup b normalises slab b % 8 of
// item b / 8.
constexpr int kNormMainWaves = 4;
constexpr int kNormWideWaves = 8;

// Runs body<shift> for the item's own shift: one instance a value, each with
// its loads and nothing to choose per load.  (Chosen inside one instance, the
// loads of all four forms meet in the same registers, which took 107 a lane
// instead of 74 in the 12-round class.)  716 windows of 15 s every 5.01 s: 152
// us, against 144 on a grid of 4 hops (5.00 s); four 4-byte loads a quad, for
// any shift, took 222.  The call, whose log-mel is then one shared region
// instead of one per residue, 501 -> 265 us; 1 h in windows of 15 s every 13.01
// s 195 -> 180.
template <bool SHIFT, class F>
__device__ __forceinline__ void with_shift(const Item& it, F&& body) {
  const int s = SHIFT ? it.gshift % kQuad : 0;
  if (s == 0) body(std::integral_constant<int, 0>());
  else if (s == 1) body(std::integral_constant<int, 1>());
  else if (s == 2) body(std::integral_constant<int, 2>());
  else body(std::integral_constant<int, 3>());
}

template <bool SHIFT, int N, typename O>
__global__ __launch_bounds__(64 * kNormMainWaves) void sfe_norm_kernel(const float* __restrict__ raw,
                                                                       const Item* __restrict__ items, int pad_to,
                                                                       O* __restrict__ out) {
  __shared__ NormLds<kNormMainWaves> lds;
  const int b = blockIdx.x;
  with_shift<SHIFT>(items[b / kSlabs],
                    [&](auto s) { norm_body<s(), kNormMainWaves, N>(raw, items, b, pad_to, out, lds); });
}

// Long items, in segments of seg_frames(T) frames, chunks of 512 in registers.
//
// norm_segment leaves per (segment, slab) the sums S of (x - x0) and V of (x
// - x0)^2, x0 the item's first value of the feature.  V comes from squared
// deviations from the chunk's own f32 mean, moved to x0 in f64, so it carries
// no f32 cancellation; it is exactly 0 where all values equal x0.
// norm_finish adds the item's segments in order, has the sum of squared
// deviations from the f32 mean m as V - 2 (m - x0) S + T (m - x0)^2 (f64: the
// terms exceed it at most about T-fold), and writes its segment.
//
// What bounds it: memory.  One workgroup per (item, slab) streaming the item
// three times left 24 clips of 20-90 s on 192 workgroups (79 us); segments
// read it twice, the second time mostly from the Infinity Cache, and fill the
// machine: 15 us for the sums (67 MB, 4.5 TB/s) and 26 us for the rest (67 MB
// in, 67 MB out, 5.2 TB/s).  Shorter items stay whole: held in registers they
// are read once, and 256 clips of 1-20 s take 49 us.
constexpr int kSegRounds = kSegFrames / (kTile * kNormMainWaves);

template <int SHIFT>
__device__ __forceinline__ void norm_segment(const float* __restrict__ raw, const Item* __restrict__ items,
                                             const int32_t* __restrict__ seg_item, int work,
                                             double2* __restrict__ parts, NormLds<kNormMainWaves>& lds) {
  constexpr int W = kNormMainWaves;
  constexpr int kSpan = NormShape<W>::kSpan;
  double* red = lds.red;
  const int seg = work / kSlabs, slab = work % kSlabs;
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const Item it = items[seg_item[seg]];
  const int sf = seg_frames(it.T), t0 = sf * (seg - it.seg0);
  const int t1 = t0 + sf < it.T ? t0 + sf : it.T;
  const float x0 = ln2_scale(raw[it.out_off + kRawSlab * slab + 4 * (lane & 15)]);
  double S = 0.0, V = 0.0;
  for (int t = t0; t < t1; t += kSegFrames) {
    const int n = t1 - t < kSegFrames ? t1 - t : kSegFrames;
    const Rounds<W> rd(raw, it, slab, lane, w, t / kQuad);
    float4 v[kSegRounds];
    load_rounds<SHIFT>(rd, v);
    constexpr int K = kSumParts / W;
    double sp[K] = {}, qp[K] = {};
#pragma unroll
    for (int j = 0; j < kSegRounds; ++j) {
      v[j] = ln2_scale(v[j]);
      add_dev(sp[j % K], v[j], x0, Rounds<W>::full(j, n), rd.left - kSpan * j);
    }
    const double s = slab_sum<W>(sp, red, lane, w);
    const float m = row_mean(x0, s, n);
#pragma unroll
    for (int j = 0; j < kSegRounds; ++j) add_sq(qp[j % K], v[j], m, Rounds<W>::full(j, n), rd.left - kSpan * j);
    const double sq = slab_sum<W>(qp, red, lane, w);
    const double d = (double)m - (double)x0, r = s - n * d;  // r: sum of (x - m)
    S += s;
    V += sq + 2.0 * d * r + n * (d * d);
  }
  if (w == 0 && lane < kSlabF) parts[(size_t)work * kSlabF + lane] = make_double2(S, V);
}

template <int SHIFT, typename O>
__device__ __forceinline__ void norm_finish(const float* __restrict__ raw, const Item* __restrict__ items,
                                            const int32_t* __restrict__ seg_item, int work,
                                            const double2* __restrict__ parts, int pad_to, O* __restrict__ out,
                                            NormLds<kNormMainWaves>& lds) {
  constexpr int W = kNormMainWaves;
  using NS = NormShape<W>;
  double* red = lds.red;
  float* st = lds.st;
  const int seg = work / kSlabs, slab = work % kSlabs;
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const Item it = items[seg_item[seg]];
  const int T = it.T;
  const int sf = seg_frames(T), n_segs = (T - 1) / sf + 1, t0 = sf * (seg - it.seg0);
  const int t1 = t0 + sf < T ? t0 + sf : T;
  const int rs = pad_to > 0 ? pad_to : T;
  O* ob = out + it.dst_off + (size_t)(kSlabF * slab) * rs;
  if (pad_to > 0 && t1 == T) zero_tail<W>(ob, T, rs, lane, w);
  const float x0 = ln2_scale(raw[it.out_off + kRawSlab * slab + 4 * (lane & 15)]);
  float4 v[kSegRounds];
  auto load = [&](int t) { load_rounds<SHIFT>(Rounds<W>(raw, it, slab, lane, w, t / kQuad), v); };
  load(t0);
  // Segment k of the item: wave k % 4, lanes 16 (k / 4 % 4) ..
  double Sp[kSumParts / W] = {}, Vp[kSumParts / W] = {};
  for (int k = w + W * (lane >> 4); k < n_segs; k += 4 * W) {
    const double2 p = parts[((size_t)(it.seg0 + k) * kSlabs + slab) * kSlabF + (lane & 15)];
    Sp[0] += p.x;
    Vp[0] += p.y;
  }
  const double S = slab_sum<W>(Sp, red, lane, w);
  const double V = slab_sum<W>(Vp, red, lane, w);
  const double d = (double)row_mean(x0, S, T) - (double)x0;
  publish_stats(S, fmax(V - 2.0 * d * S + T * (d * d), 0.0), V == 0.0, x0, T, lane, w, st);
  for (int t = t0; t < t1; t += kSegFrames) {
    if (t > t0) load(t);
#pragma unroll
    for (int ch = 0; ch < kSegRounds / 4; ++ch) {
#pragma unroll
      for (int jr = 0; jr < 4; ++jr)
        *reinterpret_cast<float4*>(lds.tb[ch % 2] + (lane & 15) * NS::kTStride + NS::kSpan * jr + 16 * w +
                                   kQuad * (lane >> 4)) = ln2_scale(v[4 * ch + jr]);
      __syncthreads();
      store_chunk<W>(lds.tb[ch % 2], st, t + NS::kChunk * ch, t1, rs, lane, w, ob);
    }
  }
}

// Workgroups [0, 8 n_segs): the long items' segments; the rest normalise the
// other items.  A launch runs those from `first` on.
template <bool SHIFT, int N, typename O>
__global__ __launch_bounds__(64 * kNormMainWaves) void sfe_norm_long_kernel(
    const float* __restrict__ raw, const Item* __restrict__ items, int first, int n_segs,
    const int32_t* __restrict__ seg_item, double2* __restrict__ parts, int pad_to, O* __restrict__ out) {
  __shared__ NormLds<kNormMainWaves> lds;
  const int b = first + blockIdx.x, rest = b - kSlabs * n_segs;
  if (rest < 0)
    with_shift<SHIFT>(items[seg_item[b / kSlabs]],
                      [&](auto s) { norm_segment<s()>(raw, items, seg_item, b, parts, lds); });
  else
    with_shift<SHIFT>(items[rest / kSlabs],
                      [&](auto s) { norm_body<s(), kNormMainWaves, N>(raw, items, rest, pad_to, out, lds); });
}

template <bool SHIFT, typename O>
__global__ __launch_bounds__(64 * kNormMainWaves) void sfe_norm_finish_kernel(
    const float* __restrict__ raw, const Item* __restrict__ items, int first, const int32_t* __restrict__ seg_item,
    const double2* __restrict__ parts, int pad_to, O* __restrict__ out) {
  __shared__ NormLds<kNormMainWaves> lds;
  const int b = first + blockIdx.x;
  with_shift<SHIFT>(items[seg_item[b / kSlabs]],
                    [&](auto s) { norm_finish<s()>(raw, items, seg_item, b, parts, pad_to, out, lds); });
}

template <bool SHIFT, int N, typename O>
__global__ __launch_bounds__(64 * kNormWideWaves) void sfe_norm_wide_kernel(const float* __restrict__ raw,
                                                                            const Item* __restrict__ items,
                                                                            int pad_to, O* __restrict__ out) {
  __shared__ NormLds<kNormWideWaves> lds;
  const int b = blockIdx.x;
  with_shift<SHIFT>(items[b / kSlabs],
                    [&](auto s) { norm_body<s(), kNormWideWaves, N>(raw, items, b, pad_to, out, lds); });
}

template <bool SHIFT, typename O>
hipError_t launch_norm_t(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, int cus,
                         int pad_to, O* out, int n_segs, const int32_t* seg_item, double2* parts,
                         hipStream_t stream) {
  using S = NormShape<kNormMainWaves>;
  using SW = NormShape<kNormWideWaves>;
  static_assert(kNormShortFrames == S::kSpan * 8, "the 4-wave form's smallest class");
  const int64_t blocks = (int64_t)n_items * kSlabs, seg_blocks = (int64_t)n_segs * kSlabs;
  if (blocks + seg_blocks > INT32_MAX) return hipErrorInvalidValue;  // (the kernels' 32-bit workgroup numbers)
  if (n_segs > 0) {
    // Long items among them: their segments' sums beside the other items,
    // then the segments themselves.
    const hipError_t e = for_launches(seg_blocks + blocks, S::kThreads, [&](int64_t first, unsigned n) {
      sfe_norm_long_kernel<SHIFT, kNormRegFrames / S::kSpan, O><<<dim3(n), dim3(S::kThreads), 0, stream>>>(
          raw, items, (int)first, n_segs, seg_item, parts, pad_to, out);
      return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    return for_launches(seg_blocks, S::kThreads, [&](int64_t first, unsigned n) {
      sfe_norm_finish_kernel<SHIFT, O><<<dim3(n), dim3(S::kThreads), 0, stream>>>(raw, items, (int)first, seg_item,
                                                                                 parts, pad_to, out);
      return hipGetLastError();
    });
  }
  // (SHIFT has 4-wave kernels for short items only: 1,172 windows of 2 s every
  // 0.51 s 49 us, 66 with 8 waves.  Longer tasks that share frames are mostly of
  // one length, where the 8-wave form is the faster one, and it loses 4% at most.)
  if ((SHIFT && max_T > kNormShortFrames) || norm_wide(n_items, max_T, sum_T, cus)) {
    return for_launches(blocks, SW::kThreads, [&](int64_t first, unsigned n) {
      const Item* it = items + first / kSlabs;
      const dim3 grid(n), block(SW::kThreads);
      if (max_T <= SW::kSpan * 8) sfe_norm_wide_kernel<SHIFT, 8, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
      else if (max_T <= SW::kSpan * 12)
        sfe_norm_wide_kernel<SHIFT, 12, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
      else sfe_norm_wide_kernel<SHIFT, 16, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
      return hipGetLastError();
    });
  }
  // Registers per lane sized to the longest item (N float4s hold kSpan N
  // frames).
  return for_launches(blocks, S::kThreads, [&](int64_t first, unsigned n) {
    const Item* it = items + first / kSlabs;
    const dim3 grid(n), block(S::kThreads);
    if (SHIFT || max_T <= S::kSpan * 8) {
      sfe_norm_kernel<SHIFT, 8, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
    } else if constexpr (!SHIFT) {
      if (max_T <= S::kSpan * 16) sfe_norm_kernel<false, 16, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
      else if (max_T <= S::kSpan * 24) sfe_norm_kernel<false, 24, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
      else sfe_norm_kernel<false, 32, O><<<grid, block, 0, stream>>>(raw, it, pad_to, out);
    }
    return hipGetLastError();
  });
}

template <bool SHIFT>
hipError_t launch_norm_form(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, int cus,
                            int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                            hipStream_t stream) {
  auto go = [&](auto* o) {
    return launch_norm_t<SHIFT>(raw, items, n_items, max_T, sum_T, cus, pad_to, o, n_segs, seg_item,
                                static_cast<double2*>(parts), stream);
  };
  return out_bf16 ? go(static_cast<uint16_t*>(out)) : go(static_cast<float*>(out));
}

}  // namespace

}  // namespace sfe
