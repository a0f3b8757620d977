// Internal declarations shared by the kernels and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>
#include <stdint.h>

#include <vector>

namespace sfe {

// Shape the kernels are specialised to: TranscriptionConfig::default()
// (src/config.rs:30-44).
constexpr int kNfft = 512;
constexpr int kWin = 400;
constexpr int kHop = 160;
constexpr int kMel = 128;
constexpr int kBins = kNfft / 2 + 1;  // 257
constexpr int kPad = kNfft / 2;       // 256 zeros each side (src/frontend.rs:124-125)

// Mel contraction schedule.  One wave contracts the power spectra of its own
// 4 frames: lane L sums filters L and 64 + L (slots 0 and 1) of all 4, slot i
// over kMelSteps[schedule][i] consecutive bins from the filter's own first
// bin (from the device table), so the dense 128x257 product is never formed.
// Schedule 0 fits the Slaney filterbank at 16, 22.05 and 24 kHz (504 nonzero
// weights); schedule 1 the other sample rates taken (build_dev_tables).
constexpr int kSchedules = 2;
constexpr int kMelSlots = 2;
constexpr int kMelSteps[kSchedules][kMelSlots] = {{3, 14}, {4, 20}};
constexpr int mel_vec(int schedule) { return (kMelSteps[schedule][0] + kMelSteps[schedule][1] + 3) / 4; }
constexpr int kMelVecMax = mel_vec(1);  // float4 weights per lane, either schedule
static_assert(mel_vec(0) <= kMelVecMax, "the weight table holds either schedule");

// Raw log-mel (log2; times ln 2 is the log-mel) lives in scratch in tiles
// of 16 frames (kRawTile floats): 8 slabs of 16 features, slab s holding
// features 16 s .. 16 s + 15 as [4 quads][16 features][4 frames], so that the
// 4 frames of one feature that a log-mel lane computes are 16 bytes.  Frame f
// of a region whose tile 0 holds frames 0..15 has its slab 0, feature 0 at
// region + raw_frame(f); feature m of slab s 256 s + 4 m floats on.
constexpr int kTile = 16;              // frames per raw tile
constexpr int kRawTile = kTile * 128;  // raw scratch floats per tile of 16 frames
constexpr int kRawSlab = 256;          // floats per slab of a tile
constexpr int kQuad = 4;               // frames per unit of work (one wave pass) of the log-mel kernel
__host__ __device__ constexpr int64_t raw_quad(int64_t q) { return kRawTile * (q >> 2) + 64 * (q & 3); }
__host__ __device__ constexpr int64_t raw_frame(int64_t f) { return raw_quad(f >> 2) + (f & 3); }

// One entry of either kernel's table.
//
// Log-mel entries: frames 4 q0 .. 4 (q0 + n_units) - 1 of samples[start,
// start + len) (preemphasis restarting at `start`, zero padding outside),
// frame f written to raw[out_off + raw_frame(f)]; its units (4-frame quads)
// are numbered from unit_off.  Entries are whole items, or parts of them
// (first or last quads), or spans that several overlapping items share.
//
// Normalisation entries, one per featurized item (a clip or a long-form
// chunk task) of T frames, written to out[dst_off + m*S + t] (S = T, or the
// padded row length of the encoder-input layout).  Frame f of its raw
// log-mel is read from raw[grid_off + raw_frame(f + gshift)] for f in
// [f_lo, f_hi], raw[tail_off + raw_frame(f)] past f_hi and raw[out_off +
// raw_frame(f)] below f_lo.  An item with its own region has f_lo = 0,
// f_hi = T - 1, grid_off = out_off and gshift = 0.  Else f_lo and f_hi + 1 are
// multiples of 4: the regions meet at whole quads of the item.
struct Item {
  int64_t start;
  int64_t len;
  int64_t out_off;
  int64_t dst_off;
  int64_t grid_off;
  int64_t tail_off;
  int32_t T;         // len / hop + 1
  int32_t unit_off;  // log-mel: first unit, relative to the launch
  int32_t n_units;   // log-mel: units of the entry
  int32_t q0;        // log-mel: first quad of the entry within its frames
  int32_t f_lo, f_hi, gshift;
  int32_t seg0;      // normalisation: first segment of a long item (norm_segments)
};
static_assert(sizeof(Item) == 80, "item table layout");

// An item with its own raw region at out_off (both kernels' view).
inline Item own_item(int64_t start, int64_t len, int64_t out_off, int64_t dst_off, int32_t unit_off) {
  Item it{};
  it.start = start;
  it.len = len;
  it.out_off = out_off;
  it.dst_off = dst_off;
  it.grid_off = out_off;
  it.tail_off = out_off;
  it.T = (int32_t)(len / kHop + 1);
  it.unit_off = unit_off;
  it.n_units = (int32_t)((it.T + kQuad - 1) / kQuad);
  it.q0 = 0;
  it.f_lo = 0;
  it.f_hi = it.T - 1;
  it.gshift = 0;
  return it;
}

// Shared frames (sfe_share.cpp).  Frames of overlapping items whose samples
// lie at least one sample inside each item and whose starts agree modulo the
// hop are computed once: items' own regions keep only their first quad and
// their last quads, and a shared log-mel entry per run of such items covers
// the union of their interior frames.  Given items with their own regions
// (own_item; out_off ignored), plan_table fills one table, table[0, *n_lm)
// with the log-mel entries and table[*n_lm, *n_lm + n) with the
// normalisation entries in item order, and returns the raw tiles they use.
// With share = false, or where sharing saves no quads, every item keeps its
// own region.  table holds (kPlanEntriesPerItem + 1) n entries; nothing is
// allocated when ws was reserved for at least n items.
constexpr int kPlanEntriesPerItem = 3;  // log-mel entries per item at most
struct PlanWorkspace {
  struct Span {
    int idx;              // item index
    int64_t res, lo, hi;  // start mod hop; interior frames in recording frame indices
  };
  struct Run {
    int64_t res, lo, hi;   // union of interior frames (recording frame indices)
    int64_t vstart, vend;  // samples of the shared entry
    int64_t cv;            // vstart / hop
    int64_t grid;          // out_off of the shared entry once placed, else -1
    int k0, k1;            // members: sp[k0, k1)
  };
  struct Piece {
    int64_t pos;  // recording position of the first frame
    int32_t seq;  // creation order
    Item e;
  };
  std::vector<Span> sp;
  std::vector<int> run_of;
  std::vector<Run> runs;
  std::vector<Piece> pieces;
  void reserve(size_t n);
};
int64_t plan_table(const Item* items, int n, bool share, PlanWorkspace* ws, Item* table, size_t* n_lm);
// Normalisation entries reordered longest first (in 256-frame classes, call
// order within one); allocates nothing.
void order_norm(Item* norm, int n);
// Long items (more than kNormRegFrames frames, what a normalisation workgroup
// holds in registers) are normalised in segments of seg_frames(T) frames, at
// most 64 an item (sfe_kernels.hip norm_segment).  norm_segments numbers the
// segments of table entries norm[0, n) (Item::seg0), writes each segment's
// entry index to seg_item unless it is null, and returns their count.  A
// segment leaves kSegPartBytes of partial sums.
constexpr int kNormRegFrames = 2048;
constexpr int kSegFrames = 512;
constexpr int kSegPartBytes = kMel * 2 * (int)sizeof(double);
__host__ __device__ constexpr int seg_frames(int T) { return kSegFrames * ((T - 1) / (64 * kSegFrames) + 1); }
inline int64_t norm_segments(Item* norm, int n, int32_t* seg_item) {
  int64_t segs = 0;
  for (int i = 0; i < n; ++i) {
    if (norm[i].T <= kNormRegFrames) continue;
    norm[i].seg0 = (int32_t)segs;
    const int k = (norm[i].T - 1) / seg_frames(norm[i].T) + 1;
    for (int s = 0; s < k && seg_item; ++s) seg_item[segs + s] = i;
    segs += k;
  }
  return segs;
}
// Frames of one run's shared entry at most (512 MB of raw log-mel), and
// members of one run at most (each with at most 3 tiles of its own, 384 MB
// in all): an item's first and last tiles follow its run's shared region,
// and every frame of the item lies within kNormBufRange bytes of the
// region's start (the normalisation kernel's 32-bit buffer offsets).
constexpr int64_t kMaxShareFrames = (int64_t)1 << 20;
constexpr int kMaxShareMembers = 1 << 14;
constexpr int kNormBufRange = 0x7ffffff0;
static_assert(kMaxShareFrames * kRawTile / kTile * 4 + (int64_t)kMaxShareMembers * 3 * kRawTile * 4 +
                      (int64_t)2 * kRawTile * 4 <
                  kNormBufRange,
              "a run's regions fit the normalisation kernel's offsets");

// Constant tables, uploaded once per context.
struct DevTables {
  float window[kNfft];       // hann_window(400), zero past 400
  // Inter-stage twiddles e^{-2 pi i k c / 512} (k, c < 16) of the log-mel
  // kernel's 32 x 16 FFT in tangent form (sfe_fft.hpp tan_twiddle), both
  // symmetric: tan512[c * 16 + k] is read by lane c of the first stage,
  // cos512[k * 16 + c] by lane k of the second (dft16_scaled).  Never pi / 2
  // (k c = 128 needs a factor of 16).
  float tan512[256];
  float cos512[256];
  // Operands of the special columns' MFMAs (the bins that are multiples of
  // 16): steps 0..3 and 4..7 of lane 4 j + i; see special_bin.
  float4 special[2][64];
  // Mel weights: step s of lane L's concatenated slots at mel_w[s / 4][L],
  // component s % 4; each filter's first bin.
  float4 mel_w[kMelVecMax][64];
  int32_t mel_k0[kMelSlots][64];
  int32_t schedule;         // index into kMelSteps
};

// Special columns of the log-mel kernel's FFT: block j (of 16) sums half j / 8
// of the inputs of pair q = j % 8; the pair's two bins (h = 0, 1) are
// multiples of 32 from Y[0] (q < 4) or odd multiples of 16 from Y[16].
__host__ __device__ constexpr int special_bin(int q, int h) {
  return q < 4 ? 32 * (2 * q + 1 + h) : 16 + 32 * (2 * (q - 4) + h);
}

// Host table builders (sfe_tables.cpp).
void hann_window(int win, float* out);
void mel_filterbank(int n_fft, int n_mels, int sample_rate, float* out);
// Returns false if the filterbank fits no mel schedule.
bool build_dev_tables(int sample_rate, DevTables* t);

// Kernel launchers (sfe_kernels.hip).  All asynchronous on `stream`.
int64_t tiles_for(int64_t T);
int64_t units_for(int64_t T);  // quads of an item: ceil(T / 4)
// cus: the device's compute units (the log-mel grid is persistent: at most
// the workgroups resident at once).  Input sample formats: f32, or integer PCM (16-bit or 32-bit containers)
// decoded as value / pcm_scale in the kernel.
constexpr int kPcmF32 = 0;
constexpr int kPcmI16 = 1;
constexpr int kPcmI32 = 2;
// A launch holds fewer than 2^32 threads: `blocks` workgroups of `threads` go
// in launches of at most that, in multiples of 8 workgroups.  go(first, n)
// launches workgroups [first, first + n).
template <class F>
hipError_t for_launches(int64_t blocks, int threads, F&& go) {
  const int64_t most = UINT32_MAX / threads / 8 * 8;
  for (int64_t first = 0; first < blocks; first += most) {
    const hipError_t e = go(first, (unsigned)(blocks - first < most ? blocks - first : most));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Copies bytes (rounded up to 16; both sides 16-byte aligned and with room for
// that) from pinned host memory to the device with a kernel on `stream`.
hipError_t launch_upload(const void* src, void* dst, size_t bytes, hipStream_t stream);
// Units [unit0, unit0 + n_units) in the numbering of items[].unit_off.
// Timestamp buffer of measurement builds (-DSFE_TIMESTAMPS, sfe_kernels.hip);
// stamps_built() is false and set_stamp_buffer fails in the product build.
bool stamps_built();
hipError_t set_stamp_buffer(void* buf, int64_t words);
constexpr int kLogmelWavesPerSimd = 3;
// Log-mel launch shape: launches with at least 4 units per wave on every
// CU's 12 waves take one 12-wave workgroup per CU; smaller ones 4-wave
// workgroups, up to 3 per CU, each wave taking at least one unit.
constexpr int kLogmelWavesSmall = 4;
constexpr int kLogmelWavesBig = 12;
struct LogmelGrid {
  int waves;   // per workgroup
  int blocks;  // workgroups
};
inline LogmelGrid logmel_grid(int n_units, int cus) {
  if ((int64_t)n_units >= (int64_t)4 * kLogmelWavesBig * cus) {
    const int want = (n_units + kLogmelWavesBig - 1) / kLogmelWavesBig;
    return {kLogmelWavesBig, want < cus ? want : cus};
  }
  const int want = (n_units + kLogmelWavesSmall - 1) / kLogmelWavesSmall;
  const int cap = kLogmelWavesPerSimd * cus;
  return {kLogmelWavesSmall, want < cap ? want : cap};
}
// Units [*wb, *we) of workgroup b of G workgroups of NW waves, over units
// [unit0, unit0 + n_units).  4-wave grids run 3 workgroups per CU, dispatched
// a CU slot at a time, and a SIMD issues its oldest wave first, so the later
// slots run slower: their shares are weighted 11 : 10 : 9 by slot (blocks in
// thirds of the grid) when every wave has at least 8 units.  The log-mel
// kernel and the host's first-item table (logmel_wave_items) both use this.
__host__ __device__ inline void logmel_share(int64_t G, int64_t b, int NW, int unit0, int n_units, int* wb, int* we) {
  const int64_t B1 = G / 3, B2 = 2 * G / 3;
  const bool weighted = NW == kLogmelWavesSmall && G >= 3 && (int64_t)n_units >= (int64_t)8 * NW * G;
  auto cum = [=](int64_t c) -> int64_t {  // share of the blocks before block c
    if (!weighted) return c;
    const int64_t c1 = c < B1 ? c : B1, c2 = c < B1 ? 0 : (c < B2 ? c - B1 : B2 - B1), c3 = c > B2 ? c - B2 : 0;
    return 11 * c1 + 10 * c2 + 9 * c3;
  };
  const int64_t tot = cum(G);
  *wb = unit0 + (int)((int64_t)n_units * cum(b) / tot);
  *we = unit0 + (int)((int64_t)n_units * cum(b + 1) / tot);
}
// Item of each wave's first unit, for a launch of grid g over units
// [unit0, unit0 + n_units) of items[0, n_items) (sorted by unit_off):
// out[b * g.waves + w] = the last item whose unit_off <= wb + w (0 for a wave
// with no unit).  The kernel then skips its item search, a chain of
// dependent loads at the start of every wave.  At most kMaxLogmelWaves
// entries; larger grids go without (the kernel searches).
constexpr int kMaxLogmelWaves = 4096;
void logmel_wave_items(const Item* items, int n_items, int unit0, int n_units, LogmelGrid g, int32_t* out);
// wave_item: the table above on the device for this launch, or null.
// schedule: the tables' mel schedule (DevTables::schedule).
hipError_t launch_logmel(const void* samples, int pcm, float pcm_scale, const Item* items, int n_items, int unit0,
                         int n_units, const DevTables* tables, int schedule, float preemph, float* raw_out, int cus,
                         const int32_t* wave_item, hipStream_t stream);
// Workgroup form of a normalisation launch without long items: 8 waves (128
// frames per round, 33 KB of LDS for the 512-frame transpose chunks, half the
// registers per lane, 3 per CU) or 4 (64 frames per round, 4 per CU).  With 8,
// each item is loaded, reduced and stored by twice the waves, but fewer items
// are resident at once, and items of few rounds leave waves without a quad.
// Normalisation times, 4-wave / 8-wave (of items up to 512 frames between
// events, which add about 2 us):
// * past 512 frames: one 10 s clip 6.8 / 5.3 us, 40 ragged clips 12.2 / 10.2,
//   10 min long form (47 chunks) 18.0 / 15.2, 64 x 15 s 20.3 / 18.5, 1 h (280
//   chunks) 77 / 72, 8 h to bf16 436 / 428; but 128 clips of 1-15 s 18.9 / 20.5,
//   256 of 1-20 s 50.2 / 52, 128 of 7.5-15 s 25.0 / 26.1: once the items no
//   longer fit at 3 per CU, the 8-wave form needs them of nearly one length
//   (measured down to 7/8 of the longest on average: 128 of 11-15 s 30.6 /
//   30.1);
// * up to 256 frames: 1 clip of 2 s 6.8 / 7.3, 48 of 2 s 8.2 / 9.1, 97 of 1 s
//   9.0 / 11.3, 300 of 0.5 s 16.3 / 20.9, 1,200 of 2 s 55 / 64;
// * between, 8 waves only while every workgroup has a CU to itself (32 x 4 s
//   8.5 / 8.2, 48 x 4 s 9.5 / 9.9, 96 x 5 s 12.6 / 13.0, 128 x 5 s 14.1 / 14.4) or
//   where 4-wave ones of nearly 512 frames no longer fit at 4 per CU (160 x 5 s
//   18.6 / 17.9, 1,200 x 5 s 108 / 103; 600 x 4 s 44.3 / 45.9).
constexpr int kNormShortFrames = 512;
constexpr int kNormWidePerCu = 3;
inline bool norm_wide(int n_items, int max_T, int64_t sum_T, int cus) {
  const int64_t groups = (int64_t)n_items * (kMel / 16);  // one per slab of 16 features
  const bool even = 8 * sum_T >= (int64_t)7 * max_T * n_items;
  if (groups <= cus) return max_T > kNormShortFrames / 2;
  if (max_T <= kNormShortFrames) return even && 8 * max_T > 7 * kNormShortFrames && groups > (int64_t)4 * cus;
  return groups <= (int64_t)kNormWidePerCu * cus || even;
}

// Normalises raw (f32 log2 values in 16-frame tiles, see Item) per (item, feature)
// and writes feature-major [128][T] per item to out (f32, must not alias
// raw) or bf16 (uint16_t*) when out_bf16 is set.  max_T: the longest item's
// frame count (sizes the kernel's register budget); sum_T: all items' frames;
// shifted: whether any item has gshift % kQuad != 0; cus: the device's
// compute units.  pad_to > 0: rows of pad_to frames, zero past T (the encoder
// input layout).  n_segs, seg_item, parts: the long items' segments
// (norm_segments over items), the device copy of their entry indexes and
// n_segs * kSegPartBytes of scratch.
hipError_t launch_norm(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, bool shifted,
                       int cus, int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                       hipStream_t stream);
// launch_norm's `shifted` calls (sfe_norm_shift.hip).
hipError_t launch_norm_shifted(const float* raw, const Item* items, int n_items, int max_T, int64_t sum_T, int cus,
                               int pad_to, void* out, bool out_bf16, int n_segs, const int32_t* seg_item, void* parts,
                               hipStream_t stream);

// Static scratch of the allocation-free entry point (sfe_noalloc.hip): an
// item table of up to kNoAllocMaxItems items, then kNoAllocRawBytes of raw
// log-mel (kNoAllocRawBytes / (kRawTile * 4) 16-frame tiles), then the partial
// sums of long items.
constexpr int kNoAllocMaxItems = 4096;
// (a plan has at most kPlanEntriesPerItem log-mel entries and one
// normalisation entry per item)
constexpr size_t kNoAllocRawBytes = (size_t)64 << 20;
// Segments of long items within that much raw log-mel: each item's last one
// may be short, and a long item has more than 4.
constexpr int kNoAllocMaxSegs = (int)(kNoAllocRawBytes / (kRawTile * 4) * kTile / kSegFrames * 5 / 4) + 1;
constexpr size_t kNoAllocItemBytes = ((size_t)(kPlanEntriesPerItem + 1) * kNoAllocMaxItems * sizeof(Item) +
                                      (kMaxLogmelWaves + kNoAllocMaxSegs) * sizeof(int32_t) + 255) / 256 * 256;
constexpr size_t kNoAllocPartBytes = (size_t)kNoAllocMaxSegs * kSegPartBytes;
// Device address of this device's static scratch (looked up once per device).
hipError_t noalloc_scratch(int device, void** out);
// Host lock of a device's static scratch (held for a whole call), and the
// device-side order of calls on it: noalloc_order makes `stream` wait for
// the previous call's end when that call ran on another stream, noalloc_mark
// records this call's end on `stream`.  Both need the lock held.
hipError_t noalloc_lock(int device, std::unique_lock<std::mutex>* lock);
hipError_t noalloc_order(int device, hipStream_t stream);
hipError_t noalloc_mark(int device, hipStream_t stream);

// Silero VAD model inputs (sfe_vad.hip): [64 context | 512 window] f32 per
// 512-sample window (src/long_form/vad.rs:62-99, src/constants.rs).
constexpr int kVadWin = 512;
constexpr int kVadCtx = 64;
constexpr int kVadRow = kVadWin + kVadCtx;
int64_t vad_num_windows(int64_t len);  // ceil(len / 512); 0 for len <= 0
// Writes vad_num_windows(len) rows of kVadRow floats to out (16-byte aligned).
hipError_t launch_vad_frames(const void* samples, int pcm, float pcm_scale, int64_t len, float* out,
                             hipStream_t stream);

}  // namespace sfe
