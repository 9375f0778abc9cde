// The engine's and the front end's host code on a runtime of ordinary memory:
// what the calls do to locks, events and staging when something fails or
// engines part, which a GPU run does not show.  Kernel launches do nothing,
// except that the per-frame launcher copies the plane.  Built and run by
// test_host_calls.py, one case per process: exit status 0 passes.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>
#include <string>
#include <vector>

#include "../include/nf3d.h"
#include "../neo_fft3d_amd/csrc/nf3d_internal.h"
#include "../neo_fft3d_amd/csrc/nf3d_mlp_batch.h"

#define CHECK(c)                                                        \
  do {                                                                  \
    if (!(c)) {                                                         \
      printf("line %d: %s\n", __LINE__, #c);                            \
      fflush(stdout);                                                   \
      _Exit(1);                                                         \
    }                                                                   \
  } while (0)

// ------------------------------------------------------------ the runtime
namespace {
int pinned_left = -1;                   // pinned allocations granted before they are refused (-1: all)
int pinned_throw = -1;                  // ... before one throws
int compute_units = 256;
int events_made = 0;
std::set<hipEvent_t> events;            // living events
std::map<hipEvent_t, hipStream_t> recorded;  // stream of an event's latest record
struct Wait {
  hipStream_t on;
  hipStream_t record;
};
std::vector<Wait> waits;
std::vector<hipStream_t> synced;        // streams of the events waited for on the host
std::vector<int> run_jobs;              // jobs of each Wiener-3D launch
char handles[4096];
int next_handle = 1;
template <class T>
T handle() {
  return reinterpret_cast<T>(&handles[next_handle++]);
}
hipStream_t stream(int k) { return reinterpret_cast<hipStream_t>(&handles[4000 + k]); }
hipError_t fresh_event(hipEvent_t* e) {
  *e = handle<hipEvent_t>();
  events.insert(*e);
  events_made++;
  return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  if (a != hipDeviceAttributeMultiprocessorCount) return hipErrorInvalidValue;
  *v = compute_units;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMalloc(void** p, size_t n) {
  *p = calloc(n, 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (pinned_throw >= 0 && pinned_throw-- == 0) throw std::bad_alloc();
  if (pinned_left == 0) return hipErrorOutOfMemory;
  if (pinned_left > 0) pinned_left--;
  return hipMalloc(p, n);
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemset(void* p, int v, size_t n) {
  memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
  for (size_t y = 0; y < h; y++) memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }  // pageable
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  CHECK(events.count(e));
  waits.push_back(Wait{s, recorded[e]});
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = handle<hipGraph_t>();
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = handle<hipGraphExec_t>();
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return fresh_event(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return fresh_event(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  CHECK(events.erase(e) == 1);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  CHECK(events.count(e));
  recorded[e] = s;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  CHECK(events.count(e));
  synced.push_back(recorded[e]);
  return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
// (no network here)
int nf3d_mlp_features(nf3d_mlp*, const void*, int, void*, void*) { return -1; }
int nf3d_mlp_predict(nf3d_mlp*, const void*, int, float*, int, float, void*, void*, char*, size_t) { return -1; }
long long nf3d_mlp_work_bytes(const nf3d_mlp*, int) { return 0; }
void nf3d_mlp_dims(const nf3d_mlp*, int*) {}
}
int nf3d_mlp_features_batch(nf3d_mlp*, void const* const*, int const*, int, void*, void*) { return -1; }

namespace nf3d {
hipError_t launch_tile(int, int, int, int, int, int, const TileLaunch& l, hipStream_t) {
  const PlaneJob& J = l.job[0];
  if (J.dst)
    for (int y = 0; y < J.Hc; y++) memcpy(J.dst + y * J.dst_pitch, J.src + y * J.src_pitch, (size_t)J.Wc * J.pix);
  return hipSuccess;
}
hipError_t launch_run(int mode, int, int, int, int, int, const RunBatch& b, hipStream_t) {
  if (mode == MODE_W3D) run_jobs.push_back(b.njobs);
  return hipSuccess;
}
hipError_t launch_seam_run(int, int, int, const RunBatch&, hipStream_t) { return hipSuccess; }
hipError_t launch_pattern(const PatternJob&, hipStream_t) { return hipSuccess; }
hipError_t launch_pattern_regions(const PatternJob&, int, int, float*, float*, float, hipStream_t) { return hipSuccess; }
hipError_t launch_dft_mfma(const void*, void*, int, int, int, float, hipStream_t) { return hipSuccess; }
const void* mfma_dft_table(int, hipError_t*) { return nullptr; }
bool mfma_dft_supported(int, int) { return true; }
bool block_shape_supported(int, int) { return true; }
int tile_blocks_per_wg(int bw, int bh) { return 128 / std::max(bw / 2 + 1, bh / 2); }
int run_blocks_per_wg(int bw, int bh, int) { return tile_blocks_per_wg(bw, bh); }
}  // namespace nf3d

// -------------------------------------------------------------- the cases
namespace {
constexpr int W = 192, H = 128, FRAMES = 24;

struct Planes {
  std::vector<std::vector<uint8_t>> p;
  std::vector<const void*> src;
  std::vector<void*> dst;
  Planes(int w, int h) {
    for (int k = 0; k < 2 * FRAMES; k++) {
      p.emplace_back((size_t)w * h);
      for (size_t i = 0; i < p.back().size(); i++) p.back()[i] = (uint8_t)(k * 37 + i * 11);
    }
    for (int k = 0; k < FRAMES; k++) {
      src.push_back(p[k].data());
      dst.push_back(p[FRAMES + k].data());
    }
  }
};

nf3d_engine* engine(int bt, int block = 16) {
  nf3d_params prm;
  nf3d_params_defaults(&prm, 2.0f);
  prm.bt = bt;
  prm.bw = prm.bh = block;
  prm.ow = prm.oh = block / 4;
  nf3d_format fmt{};
  fmt.bits_per_sample = 8;
  fmt.num_planes = 1;
  nf3d_engine* e = nullptr;
  char err[256] = {0};
  CHECK(nf3d_engine_create(&prm, &fmt, W, H, FRAMES, 0, &e, err, sizeof err) == 0);
  return e;
}

// A call of frames [first, first + count) of every engine on stream s.
void batch(const std::vector<nf3d_engine*>& es, Planes& P, int first, int count, hipStream_t s) {
  std::vector<nf3d_run_item> it;
  for (nf3d_engine* e : es) it.push_back(nf3d_run_item{e, first, count, P.src.data(), W, P.dst.data(), W});
  char err[256] = {0};
  CHECK(nf3d_run_device_batch(it.data(), (int)it.size(), s, err, sizeof err) == 0);
}

bool waited_for(hipStream_t on, hipStream_t record) {
  for (const Wait& w : waits)
    if (w.on == on && w.record == record) return true;
  return false;
}

// A call that lacks a frame of its window leaves no frame recorded in the
// ring that nothing transformed.
void missing_frame() {
  Planes P(W, H);
  for (int device = 0; device < 2; device++) {
    nf3d_engine* e = engine(3);
    char err[256] = {0};
    const nf3d_frame_ref two[2] = {{5, P.src[5], W}, {6, P.src[6], W}};
    const nf3d_frame_ref all[3] = {{4, P.src[4], W}, two[0], two[1]};
    auto get = [&](const nf3d_frame_ref* r, int n) {
      return device ? nf3d_engine_get_frame_device(e, 5, r, n, P.dst[5], W, stream(1), err, sizeof err)
                    : nf3d_engine_get_frame(e, 5, r, n, P.dst[5], W, err, sizeof err);
    };
    CHECK(get(two, 2) == -1);
    for (int k = 4; k <= 6; k++) CHECK(!nf3d_engine_cache_refresh(e, k));
    CHECK(get(all, 3) == 0);
    for (int k = 4; k <= 6; k++) CHECK(nf3d_engine_cache_refresh(e, k));
    nf3d_engine_destroy(e);
  }
}

// A frame of a 4:2:0 filter (bt = 1).
struct Frame {
  nf3d_filter* f = nullptr;
  std::vector<uint8_t> in, out;
  nf3d_frame_planes fr{};
  void* dst[4] = {};
  int stride[4] = {W, W / 2, W / 2, 0};
  Frame() : in(W * H * 3 / 2), out(in.size()) {
    nf3d_format fmt{};
    fmt.color_family = 1;
    fmt.bits_per_sample = 8;
    fmt.ssw = fmt.ssh = 1;
    fmt.num_planes = 3;
    char err[256] = {0};
    CHECK(nf3d_filter_create("bt=1;bw=16;bh=16;ow=4;oh=4", &fmt, W, H, FRAMES, &f, err, sizeof err) == 0);
    for (size_t i = 0; i < in.size(); i++) in[i] = (uint8_t)(i * 7 + (i >> 8));
    size_t o = 0;
    for (int p = 0; p < 3; p++) {
      fr.data[p] = &in[o];
      fr.stride[p] = stride[p];
      dst[p] = &out[o];
      o += (size_t)stride[p] * (p ? H / 2 : H);
    }
  }
  int get(std::string* msg = nullptr) {
    char err[256] = {0};
    std::fill(out.begin(), out.end(), 0);
    const int rc = nf3d_filter_get_frame(f, 0, &fr, 1, dst, stride, err, sizeof err);
    if (msg) *msg = err;
    return rc;
  }
};

// An exception in the pinned allocation `at` of a frame, so while one of its
// planes is queued: an error, and every plane's engine is free again (a lock
// left behind would stop the next call for good).
void frame_throws() {
  for (int at = 0; at < 6; at++) {
    Frame F;
    std::string msg;
    pinned_throw = at;
    CHECK(F.get(&msg) == -1);
    CHECK(!msg.empty());
    pinned_throw = -1;
    CHECK(F.get() == 0);
    CHECK(F.out == F.in);
    nf3d_filter_destroy(F.f);
  }
}

// Page-locked memory refused: the frame comes all the same, then and after.
void pinned_refused() {
  for (int at = 0; at <= 6; at++) {
    Frame F;
    pinned_left = at;
    CHECK(F.get() == 0);
    CHECK(F.out == F.in);
    CHECK(F.get() == 0);
    CHECK(F.out == F.in);
    pinned_left = -1;
    CHECK(F.get() == 0);
    CHECK(F.out == F.in);
    nf3d_filter_destroy(F.f);
  }
}

// Engines that met in one batch and part: each waits for the batch, not for
// what the others did later; no events are made once the calls repeat; an
// engine's mark outlives it.
void engines_part() {
  Planes P(W, H);
  nf3d_engine *a = engine(1), *b = engine(1), *c = engine(1);
  batch({a, b, c}, P, 0, 2, stream(1));
  batch({a}, P, 2, 2, stream(2));
  CHECK(waited_for(stream(2), stream(1)));
  batch({b}, P, 2, 2, stream(3));
  CHECK(waited_for(stream(3), stream(1)) && !waited_for(stream(3), stream(2)));
  synced.clear();
  nf3d_engine_sync(c);
  CHECK(synced == std::vector<hipStream_t>{stream(1)});
  // together again on a fourth stream: the batch waits for both
  batch({a, b}, P, 4, 2, stream(4));
  CHECK(waited_for(stream(4), stream(2)) && waited_for(stream(4), stream(3)));
  for (int k = 0; k < 4; k++) batch({a, b, c}, P, 6, 2, stream(5));
  const int made = events_made;
  for (int k = 0; k < 40; k++) batch({a, b, c}, P, 6, 2, stream(5));
  for (int k = 0; k < 40; k++) {
    batch({a, b, c}, P, 6, 2, stream(5));
    batch({a}, P, 8, 2, stream(6));
  }
  CHECK(events_made <= made + 1);
  nf3d_engine_destroy(a);
  waits.clear();
  batch({b, c}, P, 8, 2, stream(7));
  CHECK(waited_for(stream(7), stream(5)));
  nf3d_engine_destroy(b);
  nf3d_engine_sync(c);
  nf3d_engine_destroy(c);
  CHECK(events.empty());
}

// Where Wiener-3D runs go in pairs: twice the tiles on the device's three
// workgroups per CU, and runs of four frames, or, past two per CU, of six in
// blocks of 48 rows with bt = 5.
void pairs() {
  Planes P(W, H);
  for (int block : {16, 32, 48}) {
    for (int bt : {2, 3, 5}) {
      int geo[7];
      nf3d_engine* e = engine(bt, block);
      nf3d_engine_geometry(e, geo);
      nf3d_engine_destroy(e);
      const int per = nf3d::tile_blocks_per_wg(block, block), wgs = 2 * geo[1] * ((geo[0] + per - 1) / per);
      for (int cus : {(wgs - 1) / 3, (wgs + 2) / 3, (wgs - 1) / 2, (wgs + 1) / 2}) {
        compute_units = cus;
        const int least = wgs > 3 * cus ? FRAMES : bt == 5 && block == 48 && wgs > 2 * cus ? 6 : 4;
        e = engine(bt, block);
        for (int whole : {7, 8, 10, 11, 12, 15}) {
          run_jobs.clear();
          batch({e}, P, bt / 2, whole, stream(1));
          CHECK(run_jobs == std::vector<int>{whole >= 2 * least ? 2 : 1});
        }
        nf3d_engine_destroy(e);
      }
    }
  }
}

// Captured batches: pairs only where all engines share their launches.
void captured_pairs() {
  Planes P(W, H);
  for (int second : {16, 24}) {
    nf3d_engine *a = engine(3), *b = engine(3, second);
    std::vector<nf3d_run_item> it;
    for (nf3d_engine* e : {a, b}) it.push_back(nf3d_run_item{e, 0, 20, P.src.data(), W, P.dst.data(), W});
    nf3d_graph* g = nullptr;
    char err[256] = {0};
    run_jobs.clear();
    CHECK(nf3d_run_device_batch_graph(it.data(), 2, stream(1), &g, err, sizeof err) == 0);
    // (18 whole windows a plane: pairs of 9 frames, or launches of 9)
    CHECK(run_jobs == (second == 16 ? std::vector<int>{4} : std::vector<int>(4, 1)));
    CHECK(nf3d_graph_launch(g, stream(1)) == 0);
    nf3d_graph_destroy(g);
    run_jobs.clear();
    batch({a, b}, P, 0, 20, stream(1));
    CHECK(run_jobs == (second == 16 ? std::vector<int>{4} : std::vector<int>(2, 2)));
    nf3d_engine_destroy(a);
    nf3d_engine_destroy(b);
  }
}
}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "missing_frame") missing_frame();
  else if (name == "frame_throws") frame_throws();
  else if (name == "pinned_refused") pinned_refused();
  else if (name == "engines_part") engines_part();
  else if (name == "pairs") pairs();
  else if (name == "captured_pairs") captured_pairs();
  else return 2;
  return 0;
}
