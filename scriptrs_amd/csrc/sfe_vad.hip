// Silero VAD model-input framing on the GPU.
//
// The reference's VAD loop (src/long_form/vad.rs:62-99) walks the recording
// in 512-sample windows (VAD_WINDOW_SAMPLES, src/constants.rs) and feeds the
// model [64 context | 512 window] = 576 samples per window.  The context is
// zero for the first window and the last 64 samples of the previous window
// otherwise; a short last window is padded with its own last sample.  Every
// window but the last is full, so the previous window's tail is plain
// recording, and the whole sequence of model inputs is one gather:
//
//   out[w][p] = x(512 w - 64 + p),  p in [0, 576),
//   x(i) = 0 for i < 0, recording[min(i, len - 1)] otherwise.
//
// The kernel writes that [n_windows][576] f32 array (the model's input
// tensors back to back), decoding integer PCM on the fly.  It moves
// 4 B/sample in (f32; 2 for 16-bit PCM) and 4.5 B/sample out, and is bound
// by HBM bandwidth: no arithmetic beyond the decode.  The 64-sample context
// re-read hits L2 (the neighbouring window is mostly the same workgroup's).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sfe_internal.hpp"
#include "sfe_pcm.hpp"

namespace sfe {
namespace {

constexpr int kVadRowVec = kVadRow / 4;   // 144 float4 per model input
// One float4 of output per thread: 576 threads, 9 whole waves, write 4 rows.
// What bounds it: memory, and how evenly the workgroups keep it busy.  With 9
// float4s per thread (16 rows of 256 threads) the 1 h recording took 90 us (490
// MB, 5.4 TB/s; 71 us for 16-bit PCM), with 3 (192 threads) 84, with one 80
// and 61; 288 threads (4.5 waves) 78 and 67.
constexpr int kVadRowsPerBlock = 4;
constexpr int kVadThreads = kVadRowsPerBlock * kVadRowVec;  // 576
static_assert(kVadThreads % 64 == 0, "whole waves");
static_assert(kVadCtx % 4 == 0 && kVadWin % 4 == 0, "rows start on float4 boundaries of the recording");

// Recordings whose samples and rows together exceed the 256 MB Infinity Cache
// are read past the caches where a sample is 4 bytes: 1 h 75 us against 80
// with plain loads, 2 h 155 against 162.  Smaller ones, whose samples may
// still be cached, are not (20 min 26 us against 23, 1 min 3.4 against 2.7),
// and 16-bit PCM is not at any size measured (1 h 64 us against 61).
constexpr int64_t kVadStreamBytes = (int64_t)256 << 20;

template <typename S>
__device__ __forceinline__ float vad_sample(const S* x, int64_t len, int64_t i, const Decode& d) {
  if (i < 0) return 0.0f;
  return Pcm<S>::dec(x[i < len ? i : len - 1], d);
}

// One workgroup writes kVadRowsPerBlock model inputs, thread t float4 t of
// them (from row0), so a wave's loads and stores are contiguous except across a
// row boundary.  STREAM: nontemporal loads.
template <typename S, bool STREAM>
__global__ __launch_bounds__(kVadThreads) void sfe_vad_frames_kernel(const S* __restrict__ x, int64_t len,
                                                                     int64_t row0, int64_t n_windows, Decode dc,
                                                                     float* __restrict__ out) {
  const int r = (int)threadIdx.x / kVadRowVec;
  const int p = 4 * ((int)threadIdx.x - r * kVadRowVec);
  const int64_t w = row0 + (int64_t)blockIdx.x * kVadRowsPerBlock + r;
  if (w >= n_windows) return;
  const int64_t i = w * kVadWin - kVadCtx + p;
  float4 v;
  if (i >= 0 && i + 4 <= len) {
    typedef typename Pcm<S>::V4 V4;
    const V4* q = reinterpret_cast<const V4*>(x + i);
    v = Pcm<S>::dec4(STREAM ? __builtin_nontemporal_load(q) : *q, dc);
  } else {
    v = make_float4(vad_sample(x, len, i, dc), vad_sample(x, len, i + 1, dc), vad_sample(x, len, i + 2, dc),
                    vad_sample(x, len, i + 3, dc));
  }
  // Nontemporal stores: the output is not read again by this kernel (1 h
  // recording 78 us against 82 with plain stores).
  typedef float F4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(F4{v.x, v.y, v.z, v.w}, reinterpret_cast<F4*>(out + w * kVadRow + p));
}

template <typename S>
hipError_t launch_vad(const void* samples, int64_t len, int64_t n, const Decode& dc, float* out, hipStream_t stream) {
  const S* x = static_cast<const S*>(samples);
  const bool streamed = sizeof(S) == 4 && 4 * (len + kVadRow * n) > kVadStreamBytes;
  return for_launches((n + kVadRowsPerBlock - 1) / kVadRowsPerBlock, kVadThreads, [&](int64_t first, unsigned blocks) {
    const int64_t row0 = first * kVadRowsPerBlock;
    if (streamed)
      sfe_vad_frames_kernel<S, true><<<dim3(blocks), dim3(kVadThreads), 0, stream>>>(x, len, row0, n, dc, out);
    else
      sfe_vad_frames_kernel<S, false><<<dim3(blocks), dim3(kVadThreads), 0, stream>>>(x, len, row0, n, dc, out);
    return hipGetLastError();
  });
}

}  // namespace

int64_t vad_num_windows(int64_t len) { return len <= 0 ? 0 : (len + kVadWin - 1) / kVadWin; }

hipError_t launch_vad_frames(const void* samples, int pcm, float pcm_scale, int64_t len, float* out,
                             hipStream_t stream) {
  const int64_t n = vad_num_windows(len);
  if (n == 0) return hipSuccess;
  const Decode dc{pcm_scale, 1.0f / pcm_scale, 1.0 / (double)pcm_scale};
  if (pcm == kPcmI16) return launch_vad<int16_t>(samples, len, n, dc, out, stream);
  if (pcm == kPcmI32) return launch_vad<int32_t>(samples, len, n, dc, out, stream);
  return launch_vad<float>(samples, len, n, dc, out, stream);
}

}  // namespace sfe
