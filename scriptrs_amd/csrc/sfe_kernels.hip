// CDNA4 (gfx950) kernels of the log-mel front end.
//
// sfe_logmel_kernel fuses, per quad of 4 frames of one item, everything
// ParakeetFeatureExtractor::extract does before normalisation
// (src/frontend.rs:104-147, :150-159):
//   preemphasis restarted at the item start -> 256-zero padding ->
//   400-tap left-aligned Hann window -> 512-point real FFT -> |X|^2 ->
//   128x257 Slaney mel contraction -> ln(x + 2^-24)
// and writes the raw log-mel to scratch in tiles of 16 frames (8 slabs of 16
// features, 4 consecutive frames of a feature together), in base 2 (the
// normalisation kernel multiplies by ln 2 as it loads).
// The normalisation (sfe_norm.hpp) then applies normalize_columns
// (src/frontend.rs:225-241) per (item, feature) and writes the reference's feature-major layout
// ([128][T] per item).
//
// FFT mapping: the 512-point real FFT is 32 x 16 with tap n = 16 (b + 12) +
// c: 16 lanes own one frame; lane c runs a real 32-point DFT over b in its
// registers (25 of the 32 inputs are inside the 400-tap window), applies the
// inter-stage twiddles, a 16 x 16 transpose goes through LDS, and lane k1
// finishes bins k1 + 32 k2 (of 512) with a complex 16-point DFT over c.  A
// real transform has no even/odd split: every bin's power comes straight
// from it, and only the columns k1 = 0 and 16 (bins that are multiples of
// 16), which are real, are finished apart, on the matrix cores.  A 64-wide
// wavefront transforms 4 frames at once.
//
// What bounds it: vector issue.  An f32 MFMA takes the vector ALU with it on
// this GPU (measured with one wave of each per SIMD: 16x16x4 32 cycles, 4x4x1
// about 9, none of it overlapped; bf16 MFMAs do overlap), so 4x4x1 products
// pay only where they are fewer than 4/9 of the vector operations, which take
// 4 cycles each: the 8 of the special columns here (against 32 fmas), while
// the mel sums (68 fmas a quad) left them (40 MFMAs, 86 issue slots) and a
// first stage on them (32 16x16x4) was 20% slower than this kernel.  522
// vector instructions a quad against 582 of the 16 x 16 complex FFT with its
// split; 1 h recording 112 -> 102 us in f32, 115 -> 93 us an hour in 16-bit
// PCM (f32 also waits on memory: 420 MB in 102 us), 256 ragged clips 85 -> 76
// us.  LDS is next: about 470 of 560 cycles a quad (16-byte reads take half
// the cycles of the same bytes in smaller ones).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sfe_fft.hpp"
#include "sfe_internal.hpp"
#include "sfe_norm.hpp"
#include "sfe_pcm.hpp"

namespace sfe {

namespace {

// Log-mel workgroups hold independent waves: 4 (three workgroups per CU)
// for launches that do not fill the machine, 12 (one per CU, all of its
// waves sharing one work counter) for those that do.
constexpr int kWavesSmall = kLogmelWavesSmall;
constexpr int kWavesBig = kLogmelWavesBig;
constexpr int kXRow = 36;                            // floats per transpose row (16 complex): 16 rows' 16-byte reads
                                                     // fall on distinct banks
constexpr int kSlot = 16 * kXRow + 12;               // floats per frame slot: the 4 frames' rows 0 on distinct banks
constexpr float kGuard = 5.9604644775390625e-08f;    // 2^-24, src/frontend.rs:111

// Orders LDS traffic among the lanes of one wavefront: earlier LDS writes of
// all lanes are visible to later reads, and the compiler keeps LDS accesses
// on their side of it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Work of one wave: units taken one at a time from its workgroup's range; a
// unit (a quad) is 4 consecutive frames of one item.  Waves are independent
// but for that counter: each owns an LDS region in which its quad's samples,
// FFT transpose and power spectra live in turn, and contracts its own 4
// frames with all 128 filters.  The only workgroup barrier is the one after
// the mel weights are staged in LDS at kernel start.
constexpr int kSpan = 3 * kHop + kWin;  // samples under 4 consecutive frames (880)
// Span sample j sits at span_at(j): 16 floats of padding per hop put the 4
// frames' reads of a tap on distinct banks (a hop alone is a multiple of 32).
__host__ __device__ constexpr int span_at(int j) { return j + 16 * (j / kHop); }
constexpr int kWaveBuf = 4 * kSlot;     // floats: 4 transpose slots; also holds the span and the power spectra
static_assert(span_at(kSpan) <= kWaveBuf, "span must fit the wave buffer");
static_assert(4 * kBins <= kWaveBuf, "power spectra ([bin][frame]) fit the wave buffer");
static_assert(kXRow % 4 == 0 && kSlot % 4 == 0, "transpose rows are 16-byte aligned");
constexpr int kSpanVec = (kSpan + 255) / 256;  // 16-byte loads per lane (4)
static_assert(kSpan % 4 == 0, "span is whole float4s");

// The 880 samples under one wave's quad: span sample j is item sample
// s0 + j, valid for j in [jlo, jhi).
template <typename S>
struct Span {
  const S* xb;
  int64_t s0;
  int jlo, jhi;
  bool interior;  // the whole span lies inside the item, after its first sample
};

template <typename S>
__device__ __forceinline__ Span<S> make_span(const Item& it, const S* samples, int u) {
  const int fw = (u - it.unit_off + it.q0) * kQuad;
  Span<S> sp;
  sp.s0 = (int64_t)fw * kHop - kPad;
  sp.jlo = sp.s0 < 0 ? (int)(-sp.s0) : 0;
  sp.jhi = (int)(it.len - sp.s0 < (int64_t)kSpan ? (it.len - sp.s0 > 0 ? it.len - sp.s0 : 0) : (int64_t)kSpan);
  sp.xb = samples + it.start + sp.s0;
  sp.interior = sp.jlo == 0 && sp.jhi == kSpan && sp.s0 > 0;
  return sp;
}

// Issues the loads of an interior span (lane L: samples 4L + 256 h + 0..3)
// and, per lane, the sample before its first vector (4L - 1), which is that
// vector's preemphasis neighbour.  The per-lane address keeps it a vector
// load: a scalar load would share lgkmcnt with LDS, and every later LDS wait
// would also wait for it.  Other spans are read when processed.  Samples
// stay raw (undecoded) in registers until used.
template <typename S>
__device__ __forceinline__ void prefetch_span(const Span<S>& sp, int lane, typename Pcm<S>::V4 (&v)[kSpanVec], S& xm1) {
  if (!sp.interior) return;
#pragma unroll
  for (int h = 0; h < kSpanVec; ++h) {
    const int j = 4 * lane + 256 * h;
    v[h] = Pcm<S>::load4(sp.xb + (j < kSpan ? j : 0));
  }
  // (At an index the compiler cannot relate to the vectors': it would load
  // the neighbour and three samples as one vector and wait for it here to
  // put the samples in place.)
  int before = 4 * lane - 1;
  asm("" : "+v"(before));
  xm1 = sp.xb[before];
}

// Guarded log (src/frontend.rs:111-113) in base 2: log2(v + 2^-24), where
// the guard 2^-24 is already in v (the mel accumulators start at it).  The
// log-mel value is this times ln 2, rounded to f32, which the normalisation
// kernel applies as it loads the raw values (ln2_scale), so the VALU-bound
// log-mel kernel does one operation less per value.  A mel value that adds
// nothing to the guard gives log2(2^-24) = -24 exactly, and -24 * f32(ln 2)
// rounds to f32(ln 2^-24), the reference's value for digital silence.
// Raw log-mel is written in tiles of 16 frames: 8 slabs of 16 features, each
// [4 quads][16 features][4 frames] (1 KB).  Lane L holds the quad's 4 frames
// of filters L and 64 + L: two aligned 16-byte stores per lane, each store
// instruction writing 4 slabs x 256 contiguous bytes.  The normalisation
// kernel, which works per (item, slab), reads 1 KB contiguous per load
// instruction and finds each lane's 4 values in output order.

__device__ __forceinline__ float4 log4(const float4& v) {
  return make_float4(__log2f(v.x), __log2f(v.y), __log2f(v.z), __log2f(v.w));
}
__device__ __forceinline__ float4 fma4(float a, const float4& b, const float4& c) {
  return make_float4(fmaf(a, b.x, c.x), fmaf(a, b.y, c.y), fmaf(a, b.z, c.z), fmaf(a, b.w, c.w));
}

// An MFMA's operands stay allocated until its result d is in use (the empty
// asm reads all three).  Otherwise the register allocator may give an MFMA a
// destination overlapping one of its own operands (their last use).  Whether
// v_mfma_f32_4x4x1_16b_f32 reads every block's operands before its
// destination is written is not documented, so this kernel never relies on
// it: the build rejects any MFMA whose destination overlaps its A or B
// operand in the generated assembly.
__device__ __forceinline__ void mfma_hold(f32x4& d, float a, float b) { asm volatile("" : "+v"(d) : "v"(a), "v"(b)); }

template <typename S, int NW, int SCH>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(kLogmelWavesPerSimd, kLogmelWavesPerSimd)))
void sfe_logmel_kernel(const S* __restrict__ samples, const Item* __restrict__ items, int n_items, int unit0,
                       int n_units, const DevTables* __restrict__ tb, float coef, Decode dc, float* __restrict__ out,
                       const int32_t* __restrict__ wave_item) {
  constexpr int kWaves = NW;
  constexpr int kThreads = 64 * NW;
  constexpr int kMelVec = mel_vec(SCH);
  __shared__ __align__(16) float wbuf[kWaves][kWaveBuf];
  __shared__ __align__(16) float4 mel_w[kMelVec][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;  // frame of this lane within the wave's 4
#ifdef SFE_TIMESTAMPS
  // (the word index is recomputed where used: kept live it cost a register)
#define SFE_LOGMEL_WORD (kStampLogmel + 8 * ((int64_t)blockIdx.x * NW + w))
  if (lane == 0) SFE_STAMP(SFE_LOGMEL_WORD, stamp_now());
  int n_done = 0;
#endif
  const int l = lane & 15;

  // Work: workgroup b owns units [wb, we) of this launch's [unit0, unit0 +
  // n_units) (items[].unit_off counts in the same numbering; logmel_share,
  // which weights 4-wave grids' slots), and its waves take them one at a
  // time through an LDS counter, so a wave that gets less issue on its SIMD
  // takes fewer units.
  __shared__ int wg_next;
  int wb, we;
  logmel_share(gridDim.x, blockIdx.x, NW, unit0, n_units, &wb, &we);
  if (tid == 0) wg_next = wb + kWaves;  // each wave's first unit is wb + w

  // Mel weights, shared by the workgroup's waves.
#pragma unroll
  for (int i0 = 0; i0 < kMelVec * 64; i0 += kThreads)  // (a wave-uniform loop)
    if (i0 + tid < kMelVec * 64) mel_w[(i0 + tid) / 64][(i0 + tid) % 64] = tb->mel_w[(i0 + tid) / 64][(i0 + tid) % 64];
  // (With schedule 1's longer mel sums the special columns' operands do not
  // fit the registers: they are read from LDS each time.)
  constexpr bool kSpecialLds = SCH == 1;
  __shared__ __align__(16) float4 special[kSpecialLds ? 2 : 1][64];
  if constexpr (kSpecialLds) {
    if (tid < 128) special[tid / 64][tid % 64] = tb->special[tid / 64][tid % 64];
  }
  __syncthreads();

  // Per-lane constants: window taps of this lane's FFT inputs, inter-stage
  // twiddles (tangents for it as a first-stage lane, cosines as a
  // second-stage lane), the special columns' operands.
  float wv[25];
#pragma unroll
  for (int i = 0; i < 25; ++i) wv[i] = tb->window[16 * i + l];
  float tt[16], ct[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    tt[k] = tb->tan512[l * 16 + k];
    ct[k] = tb->cos512[l * 16 + k];
  }
  float4 sw0 = {}, sw1 = {};
  if constexpr (!kSpecialLds) sw0 = tb->special[0][lane], sw1 = tb->special[1][lane];

  float* sb = wbuf[w];
  // Span samples 4 lane + 256 h, h < 4, as this lane writes them.
  float* span_w[kSpanVec];
#pragma unroll
  for (int h = 0; h < kSpanVec; ++h) span_w[h] = sb + span_at(4 * lane + 256 * h);
  // First-stage inputs: samples 160 g + 16 i + l of the span (i < 25).
  const float* fin = sb + span_at(g * kHop) + l;
  // Transpose slots [frame][k1][c]: written as (g, k1, l), read as (g, l, c).
  float* xw = sb + kSlot * g + 2 * l;
  const float* xr = sb + kSlot * g + kXRow * l;
  // Special columns: lane 4 j + n reads inputs 8 (j / 8) .. of frame n's row
  // 0, which holds (Y[0], Y[16]): Y[0] for j % 8 < 4.
  const float* xs = sb + kSlot * (lane & 3) + 16 * (lane >> 5) + ((lane >> 4) & 1);
  // Power spectra [bin][frame] (bin 0 holds no power and is not read): bins l
  // + 32 k2 and 32 m - l of frame g; this
  // lane's special bin of frame lane % 4 (after the halves are exchanged, h =
  // lane / 32).
  float* p_lo = sb + 4 * l + g;
  float* p_hi = sb + 4 * (32 - l) + g;
  float* p_sp = sb + 4 * special_bin((lane >> 2) & 7, lane >> 5) + (lane & 3);
  // Mel: filters lane and 64 + lane of all 4 frames, from each one's first bin.
  const float4* pm0 = reinterpret_cast<const float4*>(sb) + tb->mel_k0[0][lane];
  const float4* pm1 = reinterpret_cast<const float4*>(sb) + tb->mel_k0[1][lane];
  // Store offset of this lane's first filter within a raw tile (the second's
  // is 4 slabs on).
  const int so = kRawSlab * (lane >> 4) + 4 * (lane & 15);

  const int u_first = wb + w;
  if (u_first >= we) {
#ifdef SFE_TIMESTAMPS
    if (lane == 0) {
      const unsigned long long t = stamp_now();
      SFE_STAMP(SFE_LOGMEL_WORD + 1, t);
      SFE_STAMP(SFE_LOGMEL_WORD + 2, t);
      SFE_STAMP(SFE_LOGMEL_WORD + 3, 0ull);
    }
#endif
    return;
  }
  // The unit after the one being prefetched is taken one iteration ahead
  // (lane 0's LDS add), so its result is in by the time it is needed.
  int grab = 0;
  if (lane == 0) grab = atomicAdd(&wg_next, 1);
  // Item descriptors stay in scalar registers: it_c is the item of the unit
  // being prefetched, it_n the item after it, loaded one item ahead so an
  // item boundary never waits on memory.  Every item spans at least one unit.
  int li = 0;
  if (wave_item) {
    li = wave_item[(int64_t)blockIdx.x * NW + w];  // from the host (logmel_wave_items)
  } else {
    int hi = n_items - 1;
    while (li < hi) {
      int mid = (li + hi + 1) >> 1;
      if (items[mid].unit_off <= u_first) li = mid;
      else hi = mid - 1;
    }
  }
  Item it_c = items[li];
  Item it_n = items[li + 1 < n_items ? li + 1 : li];
  // The samples of unit u + 1 are loaded into registers while unit u is
  // transformed, so the global-load latency hides behind the FFT.
  Span<S> sp_n = make_span(it_c, samples, u_first);
#ifdef SFE_TIMESTAMPS
  // (after the first use of the item descriptor, which waits for it)
  if (lane == 0) SFE_STAMP(SFE_LOGMEL_WORD + 5, stamp_now());
#endif
  typename Pcm<S>::V4 nv[kSpanVec] = {};
  S nxm1 = 0;
  prefetch_span(sp_n, lane, nv, nxm1);

  for (int u = u_first, un; u < we; u = un) {
#ifdef SFE_TIMESTAMPS
    // (stamped here rather than before the loop: there it cost a register)
    if (n_done == 0 && lane == 0) SFE_STAMP(SFE_LOGMEL_WORD + 1, stamp_now());
    n_done = __builtin_amdgcn_readfirstlane(n_done) + 1;
#endif
    const Item it = it_c;
    const Span<S> sp = sp_n;
    // (for a span that is not interior nv holds stale values, decoded and
    // never used)
    float4 cv[kSpanVec];
#pragma unroll
    for (int h = 0; h < kSpanVec; ++h) cv[h] = Pcm<S>::dec4(nv[h], dc);
    const float cxm1 = Pcm<S>::dec(nxm1, dc);

    // From here to the FFT's input reads the wave runs at priority 1: the
    // span's LDS writes and the next quad's loads are a round trip the wave
    // waits on before any arithmetic, and issuing it ahead of the SIMD's
    // other waves (in their FFT arithmetic) shortens that wait.
    __builtin_amdgcn_s_setprio(1);
    // ---- 1. preemphasised, zero-padded samples of this wave's 4 frames
    // y[0] = x[0], y[s] = x[s] - coef * x[s-1] (separately rounded, as
    // src/frontend.rs:157 computes it), zero outside [0, L).  The previous
    // quad's mel reads of this buffer were issued earlier, and LDS
    // operations of a wave complete in order.
    if (sp.interior) {
#pragma clang fp contract(off)
#pragma unroll
      for (int h = 0; h < kSpanVec; ++h) {
        const int j = 4 * lane + 256 * h;
        // x[j - 1]: for h = 0 the lane's own prefetched neighbour; else lane
        // L - 1's last sample, lane 0 taking the previous vector's lane 63.
        float p0 = cxm1;
        if (h > 0) {
          const float edge = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cv[h - 1].w), 63));
          p0 = __int_as_float(
              __builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(cv[h].w), 0x138, 0xf, 0xf, false));
        }
        float4 y;
        y.x = cv[h].x - coef * p0;
        y.y = cv[h].y - coef * cv[h].x;
        y.z = cv[h].z - coef * cv[h].y;
        y.w = cv[h].w - coef * cv[h].z;
        if (j < kSpan) *reinterpret_cast<float4*>(span_w[h]) = y;
      }
    } else {
      // span crossing the item's start or end: per-sample bounds
#pragma unroll
      for (int h = 0; h < kSpanVec; ++h) {
        const int j = 4 * lane + 256 * h;
        if (j < kSpan) {
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
            const int je = j + e;
            float v = 0.0f;
            if (je >= sp.jlo && je < sp.jhi) {
              const float cur = Pcm<S>::dec(sp.xb[je], dc);
              // item sample 0 (je == jlo with the span starting before the item)
              v = (je == sp.jlo && sp.s0 <= 0) ? cur : cur - coef * Pcm<S>::dec(sp.xb[je - 1], dc);
            }
            y[e] = v;
          }
          *reinterpret_cast<float4*>(span_w[h]) = make_float4(y[0], y[1], y[2], y[3]);
        }
      }
    }
    // Then the next unit's samples are requested.
    un = __builtin_amdgcn_readfirstlane(grab);
    if (un < we) {
      if (lane == 0) grab = atomicAdd(&wg_next, 1);
      // (units only increase: the items are walked forward)
      while (li + 1 < n_items && un >= it_n.unit_off) {
        ++li;
        it_c = it_n;
        it_n = items[li + 1 < n_items ? li + 1 : li];
      }
      sp_n = make_span(it_c, samples, un);
      prefetch_span(sp_n, lane, nv, nxm1);
    }
    wave_lds_sync();

    // ---- 2. 512-point real FFT of frame g, first stage: lane l owns taps
    // 16 i + l
    float y[25];
#pragma unroll
    for (int i = 0; i < 25; ++i) y[i] = fin[span_at(16 * i)];
    wave_lds_sync();  // the transpose below reuses the span's LDS
    __builtin_amdgcn_s_setprio(0);
    cf a[16];
    rdft32_windowed(y, wv, a);  // a[k1] = Y[k1] of column l; a[0] = (Y[0], Y[16])
#pragma unroll
    for (int k1 = 1; k1 < 16; ++k1) a[k1] = tan_twiddle(a[k1], tt[k1]);
#pragma unroll
    for (int k1 = 0; k1 < 16; ++k1) *reinterpret_cast<cf*>(xw + kXRow * k1) = a[k1];
    wave_lds_sync();
    // From the transposed reads to the mel sums the wave runs at raised
    // priority: it is then on a chain of LDS round trips (transpose, power
    // spectra), and letting it issue ahead of the SIMD's other waves, which
    // are in their first stage, shortens that chain.
    __builtin_amdgcn_s_setprio(2);
    // Second stage: lane l owns row k1 = l (lane 0's row is the special
    // columns', whose transform is replaced below).
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const float4 v = *reinterpret_cast<const float4*>(xr + 4 * m);
      a[2 * m] = {v.x, v.y};
      a[2 * m + 1] = {v.z, v.w};
    }
    float ys[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) ys[s] = xs[2 * s];
    wave_lds_sync();  // the power spectra overwrite the transpose slots
    if constexpr (kSpecialLds) sw0 = special[0][lane], sw1 = special[1][lane];
    f32x4 spec = {0.0f, 0.0f, 0.0f, 0.0f};
    const float sw[8] = {sw0.x, sw0.y, sw0.z, sw0.w, sw1.x, sw1.y, sw1.z, sw1.w};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      spec = __builtin_amdgcn_mfma_f32_4x4x1f32(sw[s], ys[s], spec, 0, 0, 0);
      mfma_hold(spec, sw[s], ys[s]);
    }
    dft16_scaled(a, ct);  // a[k2] = X[l + 32 k2] (the twiddles' cosines applied here)
#pragma unroll
    for (int k2 = 0; k2 < 8; ++k2) {
      p_lo[4 * 32 * k2] = fmaf(a[k2].y, a[k2].y, a[k2].x * a[k2].x);
      p_hi[4 * 32 * (7 - k2)] = fmaf(a[8 + k2].y, a[8 + k2].y, a[8 + k2].x * a[8 + k2].x);
    }
    {
      // The two halves of the special sums are 32 lanes apart: exchanging
      // halves of rows 0, 2 (real) and 1, 3 (imaginary) leaves one bin a lane.
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(spec[0]), __float_as_uint(spec[2]), false, false);
      const auto i = __builtin_amdgcn_permlane32_swap(__float_as_uint(spec[1]), __float_as_uint(spec[3]), false, false);
      const float re = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      const float im = __uint_as_float(i[0]) + __uint_as_float(i[1]);
      *p_sp = fmaf(im, im, re * re);  // after lane 0's own writes: LDS operations of a wave complete in order
    }
    wave_lds_sync();

    // ---- 3. mel: lane L sums filters L and 64 + L of the 4 frames.  The
    // guard 2^-24 of the log (src/frontend.rs:111) is added first instead of
    // last.  Digital silence still sums to exactly 2^-24.
    float4 m0 = make_float4(kGuard, kGuard, kGuard, kGuard), m1 = m0;
    {
      constexpr int kS0 = kMelSteps[SCH][0], kS1 = kMelSteps[SCH][1];
      float wt[4 * kMelVec];
#pragma unroll
      for (int v = 0; v < kMelVec; ++v) {
        const float4 q = mel_w[v][lane];
        wt[4 * v] = q.x;
        wt[4 * v + 1] = q.y;
        wt[4 * v + 2] = q.z;
        wt[4 * v + 3] = q.w;
      }
#pragma unroll
      for (int s = 0; s < kS0; ++s) m0 = fma4(wt[s], pm0[s], m0);
#pragma unroll
      for (int s = 0; s < kS1; ++s) m1 = fma4(wt[kS0 + s], pm1[s], m1);
    }
    __builtin_amdgcn_s_setprio(0);
    // Every frame of the quad is stored: frames past the item's end land in
    // its last tile's padding, which nothing reads.
    {
      float* o = out + it.out_off + raw_quad(u - it.unit_off + it.q0) + so;
      *reinterpret_cast<float4*>(o) = log4(m0);
      *reinterpret_cast<float4*>(o + 4 * kRawSlab) = log4(m1);
    }
  }
#ifdef SFE_TIMESTAMPS
  if (lane == 0) {
    SFE_STAMP(SFE_LOGMEL_WORD + 2, stamp_now());
    SFE_STAMP(SFE_LOGMEL_WORD + 3, (unsigned long long)__builtin_amdgcn_readfirstlane(n_done));
  }
#endif
}

// Copies a call's tables from pinned host memory.  A copy on the DMA engine
// takes the stream from one queue to another and back, which left 12-15 us
// between the kernels of calls whose tables differ; this kernel takes 2.5 us
// for 4 KB and 5 us for 45 KB (256 items), bound by the round trips over the
// host link, and leaves no gap.
constexpr int kUploadThreads = 256;
__global__ __launch_bounds__(kUploadThreads) void sfe_upload_kernel(const uint4* __restrict__ src,
                                                                  uint4* __restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * kUploadThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kUploadThreads)
    dst[i] = src[i];
}

}  // namespace

bool stamps_built() {
#ifdef SFE_TIMESTAMPS
  return true;
#else
  return false;
#endif
}

hipError_t set_stamp_buffer(void* buf, int64_t words) {
#ifdef SFE_TIMESTAMPS
  unsigned long long* p = static_cast<unsigned long long*>(buf);
  long long n = words;
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(g_stamps), &p, sizeof(p));
  if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(g_stamp_words), &n, sizeof(n));
  return e;
#else
  (void)buf;
  (void)words;
  return hipErrorNotSupported;
#endif
}

int64_t tiles_for(int64_t T) { return (T + kTile - 1) / kTile; }
int64_t units_for(int64_t T) { return (T + kQuad - 1) / kQuad; }

hipError_t launch_upload(const void* src, void* dst, size_t bytes, hipStream_t stream) {
  const size_t n = (bytes + 15) / 16;
  if (n == 0) return hipSuccess;
  const unsigned blocks = (unsigned)std::min<size_t>((n + kUploadThreads - 1) / kUploadThreads, 1024);
  sfe_upload_kernel<<<dim3(blocks), dim3(kUploadThreads), 0, stream>>>(static_cast<const uint4*>(src),
                                                                     static_cast<uint4*>(dst), n);
  return hipGetLastError();
}

template <int NW, int SCH>
hipError_t launch_logmel_t(const void* samples, int pcm, const Decode& dc, const Item* items, int n_items, int unit0,
                           int n_units, const DevTables* tables, float preemph, float* raw_out, int grid,
                           const int32_t* wave_item, hipStream_t stream) {
  const dim3 g(grid), b(64 * NW);
  if (pcm == kPcmI16)
    sfe_logmel_kernel<int16_t, NW, SCH><<<g, b, 0, stream>>>(static_cast<const int16_t*>(samples), items, n_items,
                                                             unit0, n_units, tables, preemph, dc, raw_out, wave_item);
  else if (pcm == kPcmI32)
    sfe_logmel_kernel<int32_t, NW, SCH><<<g, b, 0, stream>>>(static_cast<const int32_t*>(samples), items, n_items,
                                                             unit0, n_units, tables, preemph, dc, raw_out, wave_item);
  else
    sfe_logmel_kernel<float, NW, SCH><<<g, b, 0, stream>>>(static_cast<const float*>(samples), items, n_items, unit0,
                                                           n_units, tables, preemph, dc, raw_out, wave_item);
  return hipGetLastError();
}

template <int NW>
hipError_t launch_logmel_s(int schedule, const void* samples, int pcm, const Decode& dc, const Item* items,
                           int n_items, int unit0, int n_units, const DevTables* tables, float preemph, float* raw_out,
                           int grid, const int32_t* wave_item, hipStream_t stream) {
  if (schedule == 1)
    return launch_logmel_t<NW, 1>(samples, pcm, dc, items, n_items, unit0, n_units, tables, preemph, raw_out, grid,
                                  wave_item, stream);
  return launch_logmel_t<NW, 0>(samples, pcm, dc, items, n_items, unit0, n_units, tables, preemph, raw_out, grid,
                                wave_item, stream);
}

void logmel_wave_items(const Item* items, int n_items, int unit0, int n_units, LogmelGrid g, int32_t* out) {
  for (int b = 0; b < g.blocks; ++b) {
    int wb, we;
    logmel_share(g.blocks, b, g.waves, unit0, n_units, &wb, &we);
    for (int w = 0; w < g.waves; ++w) {
      const int u = wb + w;
      int li = 0;
      if (u < we) {
        int hi = n_items - 1;
        while (li < hi) {  // the last item whose unit_off <= u
          const int mid = (li + hi + 1) >> 1;
          if (items[mid].unit_off <= u) li = mid;
          else hi = mid - 1;
        }
      }
      out[(size_t)b * g.waves + w] = li;
    }
  }
}

hipError_t launch_logmel(const void* samples, int pcm, float pcm_scale, const Item* items, int n_items, int unit0,
                         int n_units, const DevTables* tables, int schedule, float preemph, float* raw_out, int cus,
                         const int32_t* wave_item, hipStream_t stream) {
  if (n_units <= 0) return hipSuccess;
  Decode dc{pcm_scale, 1.0f / pcm_scale, 1.0 / (double)pcm_scale};  // the host's divisions are correctly rounded
  const LogmelGrid g = logmel_grid(n_units, cus);
  if (g.waves == kWavesBig)
    return launch_logmel_s<kWavesBig>(schedule, samples, pcm, dc, items, n_items, unit0, n_units, tables, preemph,
                                      raw_out, g.blocks, wave_item, stream);
  return launch_logmel_s<kWavesSmall>(schedule, samples, pcm, dc, items, n_items, unit0, n_units, tables, preemph,
                                      raw_out, g.blocks, wave_item, stream);
}

hipError_t launch_norm(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, bool shifted,
                       int cus, int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                       hipStream_t stream) {
  if (n_items <= 0) return hipSuccess;
  if (shifted)
    return launch_norm_shifted(raw, items, n_items, max_T, sum_T, cus, pad_to, out, out_bf16, n_segs, seg_item, parts,
                               stream);
  return launch_norm_form<false>(raw, items, n_items, max_T, sum_T, cus, pad_to, out, out_bf16, n_segs, seg_item, parts,
                                 stream);
}

}  // namespace sfe
