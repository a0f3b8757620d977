// The C ABI's host code (sfe_capi.cpp, sfe_share.cpp, sfe_tables.cpp) over a
// host stand-in of the HIP runtime and of the kernel launchers, for what a call
// leaves behind while its work is still queued: the pinned staging of the
// tables, the device copy of them, and the order of calls across streams.
//
// A stream is a list of operations that run as late as they may: only when the
// host waits for them, or for something that must come after them.  So a
// staging piece, a table or a scratch buffer that is written again too early
// gives wrong outputs here every time, where on a GPU it would be a race.  The
// stand-in of the normalisation writes, for each entry of the table that is on
// the "device" when it runs, a number made of the entry's start and length to
// the entry's place in the output.
//
// argv[1]: the scenario.  Prints "bad N" at the end.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <functional>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "scriptrs_fe.h"
#include "sfe_internal.hpp"

using sfe::Item;

// ---- runtime ---------------------------------------------------------------
struct Op {
  std::function<void()> run;
  bool kernel;
};
struct ihipStream_t {
  std::vector<Op> ops;
  size_t done = 0;
};
struct ihipEvent_t {
  ihipStream_t* s = nullptr;
  size_t at = 0;
};
static std::vector<std::unique_ptr<ihipStream_t>> g_streams;
static ihipStream_t g_null;
static long g_kernels_run = 0;  // by host waits
static long g_waits = 0;        // host waits that found something to run
static bool g_capturing = false;
static int g_fail_norm = 0;     // the next launches of the normalisation that fail
static long g_fail_new = -1;    // the allocation that fails (counted down to 0)
void* operator new(size_t n) {
  if (g_fail_new >= 0 && g_fail_new-- == 0) throw std::bad_alloc();
  return malloc(n);
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static ihipStream_t* st(hipStream_t s) { return s ? s : &g_null; }
static void run_to(ihipStream_t* s, size_t n) {
  while (s->done < n) {
    Op op = s->ops[s->done++];
    g_kernels_run += op.kernel;
    op.run();
  }
}
static void enqueue(hipStream_t s, std::function<void()> f, bool kernel) { st(s)->ops.push_back({std::move(f), kernel}); }
static void host_wait(ihipStream_t* s, size_t n) {
  g_waits += s->done < n;
  run_to(s, n);
}
static void drain() {
  host_wait(&g_null, g_null.ops.size());
  for (auto& s : g_streams) host_wait(s.get(), s->ops.size());
}

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return drain(), hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return *p = calloc(1, n + 16), hipSuccess; }
hipError_t hipFree(void* p) { return drain(), free(p), hipSuccess; }
// (freed pinned memory is kept, overwritten: an upload still queued from it shows)
static std::vector<std::pair<void*, size_t>> g_pinned;
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n);
  g_pinned.push_back({*p, n});
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  for (auto& m : g_pinned)
    if (m.first == p) memset(p, 0xEE, m.second);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  enqueue(q, [=] { memcpy(d, s, n); }, false);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  g_streams.emplace_back(new ihipStream_t);
  return *s = g_streams.back().get(), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return host_wait(st(s), st(s)->ops.size()), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) {
  *c = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  ihipStream_t* from = e->s;
  const size_t at = e->at;
  if (from) enqueue(s, [=] { run_to(from, at); }, false);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new ihipEvent_t, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->s = st(s);
  e->at = st(s)->ops.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->s) host_wait(e->s, e->at);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 0, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
}

// ---- kernels ---------------------------------------------------------------
static long g_bad = 0;
static float mark(int64_t start, int64_t len) { return (float)((start * 31 + len) % 1000003); }

namespace sfe {
int64_t tiles_for(int64_t T) { return (T + kTile - 1) / kTile; }
int64_t units_for(int64_t T) { return (T + kQuad - 1) / kQuad; }
bool stamps_built() { return false; }
hipError_t set_stamp_buffer(void*, int64_t) { return hipErrorNotSupported; }
hipError_t launch_upload(const void* src, void* dst, size_t bytes, hipStream_t s) {
  enqueue(s, [=] { memcpy(dst, src, (bytes + 15) / 16 * 16); }, false);
  return hipSuccess;
}
void logmel_wave_items(const Item*, int, int, int, LogmelGrid g, int32_t* out) {
  for (int i = 0; i < g.blocks * g.waves; ++i) out[i] = 1000 + i;
}
hipError_t launch_logmel(const void*, int, float, const Item* items, int n, int unit0, int n_units, const DevTables*,
                         int, float, float*, int cus, const int32_t* wave_item, hipStream_t s) {
  enqueue(s, [=] {
    int units = unit0;
    for (int i = 0; i < n; ++i) g_bad += items[i].unit_off != units, units += items[i].n_units;
    g_bad += units != unit0 + n_units;
    const LogmelGrid g = logmel_grid(n_units, cus);
    for (int i = 0; wave_item && i < g.blocks * g.waves; ++i) g_bad += wave_item[i] != 1000 + i;
  }, true);
  return hipSuccess;
}
hipError_t launch_norm(const float*, const Item* items, int n, int, int64_t, bool, int, int, void* out, bool, int n_segs,
                       const int32_t* seg_item, void*, hipStream_t s) {
  if (g_fail_norm > 0) return --g_fail_norm, hipErrorInvalidConfiguration;
  float* o = static_cast<float*>(out);
  enqueue(s, [=] {
    for (int i = 0; i < n; ++i) o[items[i].dst_off] = mark(items[i].start, items[i].len);
    for (int k = 0; k < n_segs; ++k) {
      const int i = seg_item[k];
      g_bad += i < 0 || i >= n || items[i].T <= kNormRegFrames || items[i].seg0 > k;
    }
  }, true);
  return hipSuccess;
}
hipError_t launch_vad_frames(const void*, int, float, int64_t, float*, hipStream_t) { return hipSuccess; }
int64_t vad_num_windows(int64_t len) { return (len + 511) / 512; }
// the static scratch: its calls are ordered as in sfe_noalloc.hip
static std::vector<unsigned char> g_noalloc(kNoAllocItemBytes + 64);
static std::mutex g_mu;
static hipEvent_t g_ev = new ihipEvent_t;
hipError_t noalloc_scratch(int, void** out) { return *out = g_noalloc.data(), hipSuccess; }
hipError_t noalloc_lock(int, std::unique_lock<std::mutex>* l) { return *l = std::unique_lock<std::mutex>(g_mu), hipSuccess; }
hipError_t noalloc_order(int, hipStream_t s) { return hipStreamWaitEvent(s, g_ev, 0); }
hipError_t noalloc_mark(int, hipStream_t s) { return hipEventRecord(g_ev, s); }
}  // namespace sfe

// ---- scenarios -------------------------------------------------------------
struct Call {
  std::vector<sfe_chunk> tasks;
  std::vector<int64_t> fo;
  std::vector<float> out;
};
static std::vector<std::unique_ptr<Call>> g_calls;
static sfe_ctx* g_ctx;
static float g_samples[1];

// n tasks of about `len` samples, different in every call.
static Call* make(int n, int64_t len, int seed) {
  g_calls.emplace_back(new Call);
  Call* c = g_calls.back().get();
  int64_t at = seed * 7 + 1, frames = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t l = len + (seed * 13 + i * 5) % 157;
    c->tasks.push_back({at, at + l, at, 0});
    frames += l / 160 + 1;
    at += l + 3;
  }
  c->fo.resize(n + 1);
  c->out.assign((size_t)frames * 128, -1.0f);
  return c;
}
static int run(Call* c, hipStream_t s, bool noalloc = false) {
  auto f = noalloc ? sfe_extract_chunks_noalloc : sfe_extract_chunks;
  return f(g_ctx, g_samples, c->tasks.back().audio_end, c->tasks.data(), (int)c->tasks.size(), SFE_F32, c->out.data(),
           c->fo.data(), s);
}
static int run_streamed(Call* c, std::vector<float>* host) {
  host->assign((size_t)c->tasks.back().audio_end, 0.0f);
  return sfe_extract_chunks_streamed(g_ctx, host->data(), c->tasks.back().audio_end, c->tasks.data(),
                                     (int)c->tasks.size(), SFE_F32, c->out.data(), c->fo.data(), 960000);
}
static void check(Call* c, const char* what, int64_t rebase = 0) {
  long wrong = 0;
  for (size_t i = 0; i < c->tasks.size(); ++i)
    wrong += c->out[128 * c->fo[i]] != mark(c->tasks[i].audio_start - rebase, c->tasks[i].audio_end - c->tasks[i].audio_start);
  if (wrong) printf("%s: %ld of %zu tasks wrong\n", what, wrong, c->tasks.size());
  g_bad += wrong;
}
static void check_all(const char* what) {
  drain();
  for (auto& c : g_calls) check(c.get(), what);
  g_calls.clear();
}
static void expect(bool ok, const char* what) {
  if (!ok) printf("%s\n", what);
  g_bad += !ok;
}

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  sfe_config cfg;
  sfe_config_default(&cfg);
  if (sfe_create(&cfg, 0, &g_ctx)) return 2;
  hipStream_t a = nullptr, b = nullptr;
  hipStreamCreateWithFlags(&a, 0);
  hipStreamCreateWithFlags(&b, 0);
  // the context grows its device buffers for the largest call first, so that
  // growing does not drain the streams later
  auto warm = [&](int n, int64_t len) { run(make(n, len, 999), a), check_all("warm"); };

  if (name == "turns") {
    // calls of one stream, no host wait between them: many turns of the ring,
    // small, large and past the ring's first size, long tasks among them
    warm(9000, 1600);
    for (int k = 0; k < 120; ++k) {
      const int n = k % 5 == 0 ? 4000 + 37 * k : 1 + 11 * k;
      expect(run(make(n, k % 7 == 3 && n < 500 ? 400000 : 1600, k), a) == SFE_OK, "call failed");
    }
    check_all("turns");
  } else if (name == "streams") {
    // the same over two streams in turn
    warm(6000, 1600);
    for (int k = 0; k < 80; ++k) expect(run(make(k % 4 == 1 ? 5000 - k : 3 + k, 1600, k), k % 2 ? b : a) == SFE_OK, "call failed");
    check_all("streams");
  } else if (name == "grow") {
    // a table that grows the ring alone (the device buffers have room), with
    // uploads queued on both streams; then tables that grow everything
    warm(1000, 160000);
    for (int n : {8000, 8100}) run(make(n, 1600, n), a);
    for (int k = 0; k < 9; ++k) run(make(50 + k, 1600, k), k % 2 ? b : a);
    expect(run(make(9000, 1600, 5), a) == SFE_OK, "call failed");
    check_all("grow the ring");
    for (int k = 0; k < 14; ++k) expect(run(make(100 << k % 13, 800, k), k % 2 ? b : a) == SFE_OK, "call failed");
    check_all("grow");
  } else if (name == "mixed") {
    // resident, allocation-free and streamed calls on one context
    warm(3000, 1600);
    for (int k = 0; k < 40; ++k) {
      Call* c = make(k % 3 == 0 ? 4096 : 50 + k, 1600, k);
      if (k % 10 == 9) {
        std::vector<float> host;
        expect(run_streamed(c, &host) == SFE_OK, "streamed call failed");
        check(c, "streamed", c->tasks[0].audio_start);  // one batch, re-based to its first sample
        g_calls.pop_back();
      } else {
        expect(run(c, k % 4 == 2 ? b : a, k % 2 == 0) == SFE_OK, "call failed");
      }
    }
    check_all("mixed");
  } else if (name == "ahead") {
    // the host runs at least one call ahead of the device, whatever the tables'
    // size: no call waits for the kernels of the call before it
    for (bool noalloc : {true, false})
      for (int n : {300, 2500, 4096}) {
        warm(n, 1600);
        run(make(n, 1600, 1), a, noalloc);
        check_all("ahead");
        g_kernels_run = 0;
        for (int k = 0; k < 12; ++k) {
          expect(run(make(n, 1600, k + 2), a, noalloc) == SFE_OK, "call failed");
          // after call k (counting from 0) at most the k - 1 first have run
          if (g_kernels_run > 2 * (k > 1 ? k - 1 : 0)) {
            printf("%s calls of %d tasks: %ld kernels run after call %d\n", noalloc ? "noalloc" : "resident", n,
                   g_kernels_run, k);
            ++g_bad;
            break;
          }
        }
        check_all("ahead");
      }
  } else if (name == "failed") {
    // a call whose normalisation does not launch leaves its upload and its
    // log-mel queued on its stream; the calls after it come on another one
    auto fails = [&](Call* c, hipStream_t s, bool noalloc = false) {
      g_fail_norm = 1;
      expect(run(c, s, noalloc) == SFE_HIP_ERROR, "the launch did not fail");
      g_fail_norm = 0;
      std::fill(c->out.begin(), c->out.end(), -1.0f);
    };
    // the first call of the context fails; then one that failed after others.
    // The same table again: its upload must have run.
    for (int k = 0; k < 3; ++k) {
      Call* c = make(20 + k, 1600, k);
      fails(c, a);
      expect(run(c, b) == SFE_OK, "call failed");
      hipStreamSynchronize(b);
      check(c, "same table after a failed call");
      check_all("same table after a failed call");
    }
    // other tables: the failed call's upload must not come after theirs
    for (int k = 0; k < 3; ++k) {
      fails(make(20, 1600, 40 + k), a);
      g_calls.pop_back();
      Call* c = make(30, 1600, k);
      expect(run(c, b) == SFE_OK, "call failed");
      hipStreamSynchronize(b);
      drain();
      std::fill(c->out.begin(), c->out.end(), -1.0f);
      expect(run(c, b) == SFE_OK, "call failed");
      check_all("other table after a failed call");
    }
    // a clip from host memory, a streamed recording
    std::vector<float> x(1600), y(128 * 11);
    g_fail_norm = 1;
    expect(sfe_extract(g_ctx, x.data(), 1600, y.data(), (int64_t)y.size()) == SFE_HIP_ERROR, "the launch did not fail");
    g_waits = 0;
    expect(sfe_extract(g_ctx, x.data(), 1600, y.data(), (int64_t)y.size()) == SFE_OK, "call failed");
    expect(g_waits == 2, "a clip after a failed one waits for it before it writes the staging");
    g_fail_norm = 1;
    std::vector<float> host;
    expect(run_streamed(make(40, 1600, 3), &host) == SFE_HIP_ERROR, "the launch did not fail");
    g_calls.pop_back();
    Call* c = make(30, 1600, 5);
    expect(run(c, b) == SFE_OK, "call failed");
    hipStreamSynchronize(b);
    drain();
    std::fill(c->out.begin(), c->out.end(), -1.0f);
    expect(run(c, b) == SFE_OK, "call failed");
    check_all("after a failed streamed call");
    // the static scratch, from another context: its upload, then the failed
    // call's as late as it may come, then its kernels
    sfe_ctx* other = g_ctx;
    fails(make(25, 1600, 7), a, true);
    g_calls.pop_back();
    if (sfe_create(&cfg, 0, &g_ctx)) return 2;
    expect(run(make(25, 1600, 8), b, true) == SFE_OK, "call failed");
    run_to(::st(b), ::st(b)->ops.size() - 2);
    check_all("static scratch after a failed call");
    sfe_destroy(other);
    // and a context without failures waits for nothing
    g_waits = 0;
    for (int k = 0; k < 4; ++k) run(make(5, 1600, 20 + k), b);
    expect(g_waits == 0, "calls without a failure wait");
    check_all("after");
  } else if (name == "memory") {
    // each of a call's host allocations fails in turn: the calls after it, with
    // the plan from before it and with its own, are right
    warm(300, 1600);
    int failures = 0;
    for (int k = 0; k < 100; ++k) {
      Call* before = make(60, 1600, 3 * k);
      expect(run(before, a) == SFE_OK, "call failed");
      Call* c = make(400 + 10 * k, 1603, 3 * k + 1);  // (more tasks than any before: every list grows)
      g_fail_new = k;
      const int rc = run(c, a);
      g_fail_new = -1;
      drain();
      std::fill(before->out.begin(), before->out.end(), -1.0f);
      expect(run(before, a) == SFE_OK && run(c, a) == SFE_OK, "call failed");
      check_all("after a failed allocation");
      if (rc == SFE_OK) break;
      ++failures;
    }
    expect(failures > 5 && failures < 100, "allocations failed");
  } else {
    return 3;
  }
  drain();
  sfe_destroy(g_ctx);
  printf("bad %ld\n", g_bad);
  return g_bad != 0;
}
