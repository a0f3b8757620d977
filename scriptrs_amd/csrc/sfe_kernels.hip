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
// sfe_norm_kernel then applies normalize_columns (src/frontend.rs:225-241)
// per (item, feature) and writes the reference's feature-major layout
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
#include <type_traits>

#include "sfe_fft.hpp"
#include "sfe_internal.hpp"
#include "sfe_pcm.hpp"
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

// Log-mel workgroups hold independent waves: 4 (three workgroups per CU)
// for launches that do not fill the machine, 12 (one per CU, all of its
// waves sharing one work counter) for those that do.
constexpr int kWavesSmall = kLogmelWavesSmall;
constexpr int kWavesBig = kLogmelWavesBig;
constexpr int kXRow = 36;                            // floats per transpose row (16 complex): 16 rows' 16-byte reads
                                                     // fall on distinct banks
constexpr int kSlot = 16 * kXRow + 12;               // floats per frame slot: the 4 frames' rows 0 on distinct banks
constexpr float kGuard = 5.9604644775390625e-08f;    // 2^-24, src/frontend.rs:111
constexpr float kLn2 = 0.69314718055994531f;

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
// Raw value loaded by the normalisation kernel: RN(log2 * ln 2).
__device__ __forceinline__ float4 ln2_scale(float4 v) {
#pragma clang fp contract(off)  // rounded on its own, never fused into a later add
  return make_float4(v.x * kLn2, v.y * kLn2, v.z * kLn2, v.w * kLn2);
}

__device__ __forceinline__ float ln2_scale(float v) {
#pragma clang fp contract(off)
  return v * kLn2;
}

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

// The lane's N quads (Rounds): raw buffer loads from the uniform base, all
// issued before any is used (a load under a per-lane branch would wait for
// itself).  One 16-byte load a quad where the item's quads are quads of its
// regions (SHIFT = 0); the 4 - SHIFT frames from one quad of the shared region
// and the SHIFT from the next in two loads where it starts inside one.
template <int SHIFT, int W, int N>
__device__ __forceinline__ void load_rounds(const Rounds<W>& rd, float4 (&v)[N]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef float f32x3 __attribute__((ext_vector_type(3)));
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(rd.base), 0, kNormBufRange, kBufWord3);
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
  load_rounds<SHIFT>(rd, v);
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

hipError_t launch_norm(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, bool shifted,
                       int cus, int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                       hipStream_t stream) {
  if (n_items <= 0) return hipSuccess;
  double2* p = static_cast<double2*>(parts);
  auto go = [&](auto* o) {
    return shifted ? launch_norm_t<true>(raw, items, n_items, max_T, sum_T, cus, pad_to, o, n_segs, seg_item, p, stream)
                   : launch_norm_t<false>(raw, items, n_items, max_T, sum_T, cus, pad_to, o, n_segs, seg_item, p,
                                          stream);
  };
  return out_bf16 ? go(static_cast<uint16_t*>(out)) : go(static_cast<float*>(out));
}

}  // namespace sfe
