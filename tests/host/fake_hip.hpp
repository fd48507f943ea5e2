// fake_hip.hpp -- a stand-in for the HIP runtime and the library's kernels, so that the
// host code (flip_api.cpp, hash_api.cpp, unet_api.cpp) runs on a machine without a GPU.
//
// Device memory is host memory in a table of live allocations. Work on a stream is queued
// and runs only when something waits for that stream; a copy on the null stream does not
// wait for others, as for the runtime's non-blocking streams. Kernels are reduced to what
// the tests look at: pressure element 0 counts the sweeps that made the buffer, a residual
// is a power of that count, bins hold how many records were counted.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "aqflip.h"
#include "aqflip_hash.h"
#include "aqflip_internal.h"
#include "aqflip_unet.h"
#include "mgpcg.h"
#include "unet_internal.h"

namespace fake {

using Work = std::function<void()>;
struct Stream {
  std::deque<Work> queue;
  std::vector<Work>* capture = nullptr;
  bool invalid = false;  // a launch failed during the capture
};
struct Graph {
  std::vector<Work> work;
};
struct Event {
  long long at = 0;
};
struct Block {
  size_t size;
  int dev;
};

inline std::map<char*, Block> live;
inline std::vector<Stream*> streams;
inline size_t capacity = (size_t)-1;  // of a device
inline int device = 0;
inline std::string fail_launch;       // a launch of this name fails,
inline int fail_skip = 0;             // after so many of them
inline hipError_t last_error = hipSuccess;
inline bool check_bins = true;        // a scatter's offsets have to end at its record count
inline long long launches = 0, graph_launches = 0, captures = 0;
inline std::map<std::string, long long> count;  // launches by name, replayed ones too
inline double rate = 0.99, drop_at = 1e30;      // the residual's factor per sweep; 1e-3 of it from drop_at on

inline int mg_iters = 0;

inline size_t used(int dev) {
  size_t n = 0;
  for (const auto& b : live) n += b.second.dev == dev ? b.second.size : 0;
  return n;
}
// [p, p + n) lies in one live allocation.
inline void check(const void* p, size_t n) {
  auto b = live.upper_bound((char*)p);
  if (b != live.begin() && (--b, (char*)p + n <= b->first + b->second.size)) return;
  std::fprintf(stderr, "kernel argument outside every live allocation\n");
  std::exit(3);
}
inline void run(Stream* s) {
  while (!s->queue.empty()) {
    Work w = std::move(s->queue.front());
    s->queue.pop_front();
    w();
  }
}
inline size_t pending() {
  size_t n = 0;
  for (Stream* s : streams) n += s->queue.size();
  return n;
}
inline void put(hipStream_t s, Work w) {
  Stream* f = (Stream*)s;
  if (!f)
    w();
  else if (f->capture)
    f->capture->push_back(std::move(w));
  else
    f->queue.push_back(std::move(w));
}
inline void launch(const char* name, hipStream_t s, Work w = [] {}) {
  if (fail_launch == name && fail_skip-- == 0) {
    fail_skip = 0;
    fail_launch.clear();
    last_error = hipErrorLaunchFailure;
    if (s && ((Stream*)s)->capture) ((Stream*)s)->invalid = true;
    return;
  }
  ++launches;
  put(s, [name = std::string(name), w] {
    ++count[name];
    w();
  });
}

}  // namespace fake

// ---- the runtime
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (fake::used(fake::device) + n > fake::capacity) return fake::last_error = hipErrorOutOfMemory;
  *p = std::malloc(n);
  std::memset(*p, 0xcd, n);
  fake::live[(char*)*p] = {n, fake::device};
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  for (fake::Stream* s : fake::streams) fake::run(s);
  fake::check(p, 1);
  fake::live.erase((char*)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { return *d = p, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = fake::device, hipSuccess; }
hipError_t hipSetDevice(int d) { return fake::device = d, hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = fake::last_error;
  fake::last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  fake::streams.push_back(new fake::Stream);
  *s = (hipStream_t)fake::streams.back();
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (s) fake::run((fake::Stream*)s);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {  // polling lets the stream go on by one piece of work
  fake::Stream* f = (fake::Stream*)s;
  if (f->queue.empty()) return hipSuccess;
  fake::Work w = std::move(f->queue.front());
  f->queue.pop_front();
  w();
  return hipErrorNotReady;
}
hipError_t hipStreamDestroy(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  ((fake::Stream*)s)->capture = new std::vector<fake::Work>;
  ++fake::captures;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
  fake::Stream* f = (fake::Stream*)s;
  *g = f->invalid ? nullptr : (hipGraph_t) new fake::Graph{*f->capture};
  f->capture = nullptr;
  const hipError_t e = f->invalid ? hipErrorStreamCaptureInvalidated : hipSuccess;
  f->invalid = false;
  return e;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t) new fake::Graph(*(fake::Graph*)g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  ++fake::graph_launches;
  for (const fake::Work& w : ((fake::Graph*)e)->work) fake::put(s, w);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete (fake::Graph*)g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return delete (fake::Graph*)e, hipSuccess; }
// An event's time is the number of launches before it.
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t) new fake::Event, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (fake::Event*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return ((fake::Event*)e)->at = fake::launches, hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(((fake::Event*)b)->at - ((fake::Event*)a)->at);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
  if (kind == hipMemcpyHostToDevice) {  // pageable: staged before the call returns
    std::vector<char> staged((const char*)s, (const char*)s + n);
    fake::put(st, [d, staged] { std::memcpy(d, staged.data(), staged.size()); });
  } else {
    fake::put(st, [d, s, n] { std::memcpy(d, s, n); });
    if (kind == hipMemcpyDeviceToHost) return hipStreamSynchronize(st);
  }
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  fake::put(s, [p, v, n] { std::memset(p, v, n); });
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = (void*)s, hipSuccess; }
}

// ---- the library's kernels
namespace aqf {
using fake::launch;
void launch_fill_u32(void* p, uint32_t v, long long n, hipStream_t s) {
  launch("fill", s, [=] { std::fill_n((uint32_t*)p, n, v); });
}
void launch_residual(const Geom&, Grid gr, int pb, double*, double* out, hipStream_t s, SweepReport* report,
                     int* reports) {
  launch("residual", s, [=] {
    const double r = std::pow(fake::rate, gr.p[pb][0]) * (gr.p[pb][0] >= fake::drop_at ? 1e-3 : 1.0);
    out[0] = r * r, out[1] = 1.0;
    if (!report) return;
    const int c = ++*reports;
    report[c & 1] = SweepReport{out[0], out[1], c};
  });
}
void launch_copy_cells(const Geom& G, const float* src, float* dst, hipStream_t s) {
  launch("copy_cells", s, [src, dst, n = (size_t)G.ncell] { std::memcpy(dst, src, n * 4); });
}
void launch_jacobi(const Geom&, Grid gr, int pin, int, int, hipStream_t s) {
  launch("jacobi", s, [=] { gr.p[pin ^ 1][0] = gr.p[pin][0] + 1; });
}
int tile_sweeps() { return 4; }
bool tile_full(const Geom&) { return true; }
void launch_jacobi_tile(const Geom&, Grid gr, int pin, int, int, hipStream_t s) {
  launch("tile", s, [=] { gr.p[pin ^ 1][0] = gr.p[pin][0] + 4; });
}
void launch_tile_pair(const Geom&, Grid, int, int, int, float, double, int, int, hipStream_t s) { launch("tile_pair", s); }
void launch_jacobi_diffusion(const Geom&, Grid, int, int, int, int, float, double, int, int, int, int, hipStream_t s) {
  launch("pair", s);
}
bool small_grid(const Geom& G, int) { return G.ncells_hash <= 20000; }
void launch_sweeps_small(const Geom&, Grid gr, int, int pb, int, int nj, int, float, double, int, int, int, hipStream_t s) {
  launch("small", s, [=] { gr.p[pb][0] += (float)nj; });
}
void launch_diffusion(const Geom&, Grid, int, int, float, double, int, int, int, hipStream_t s) { launch("diffusion", s); }
void launch_fill_pressure_zero(const Geom& G, Grid gr, int pb, hipStream_t s) {
  launch("pressure_zero", s, [=, n = G.ncell] { std::fill_n(gr.p[pb], n, 0.f); });
}
int sweep_chunks(const Geom& G) { return (G.ncells_hash + 511) / 512; }
int sweep_table_entries(const Geom&) { return 64; }
void set_listed_grids(const Geom&, Grid&, int) {}
int seed_block_size() { return 256; }
void launch_hash_records(const Geom&, const float* rec, long long n, int stride, Bins B, hipStream_t s) {
  launch("hash_records", s, [=] {
    fake::check(rec, (size_t)n * stride * 4), fake::check(B.hash, (size_t)n * 4), fake::check(B.rank, (size_t)n * 4);
    B.count[0] += (int)n;
  });
}
void launch_scan(const Geom& G, Bins B, hipStream_t s, int*, int*) {
  launch("scan", s, [B, n = G.ncells_hash] {
    B.offsets[n] = 0;
    for (int c = 0; c < n; ++c) B.offsets[n] += B.count[c], B.count[c] = 0;
  });
}
void launch_scatter_segsort(const Geom& G, long long n, Bins B, hipStream_t s) {
  launch("scatter", s, [B, n, nc = G.ncells_hash] {
    fake::check(B.perm, (size_t)n * 4);
    if (fake::check_bins && B.offsets[nc] != n) std::fprintf(stderr, "offsets hold %d records of %lld\n", B.offsets[nc], n), std::exit(4);
  });
}
size_t radix_counts(long long n) { return (size_t)((n + 1023) / 1024 * 512); }
int radix_passes(const Geom&) { return 2; }
uint32_t* launch_radix_sort(const Geom&, const float*, long long n, int, const RadixBufs& R, hipStream_t s) {
  launch("radix", s, [R, n] {
    for (const void* p : {(const void*)R.keys[0], (const void*)R.keys[1], (const void*)R.vals[0], (const void*)R.vals[1]})
      fake::check(p, (size_t)n * 4);
    fake::check(R.counts, radix_counts(n) * 4), fake::check(R.offsets, radix_counts(n) * 4 + 4), fake::check(R.partials, 4);
  });
  return R.keys[0];
}
void launch_hash_outputs(long long, int, const HashSorted&, const float*, int*, int*, float*, hipStream_t s) {
  launch("outputs", s);
}
void launch_export_field(const Geom&, const ExportField& f, long long first, long long n, void* out, hipStream_t s) {
  launch("export_field", s, [=] {
    const size_t w = f.kind == ExportField::kVector || f.kind == ExportField::kBits ? 4 : 1;
    fake::check(out, n * w * 4);
    for (long long i = 0; i < n; ++i) std::fill_n((int*)out + i * w, w, (int)(first + i));
  });
}
#define AQ_FAKE(name, ...) \
  void launch_##name(__VA_ARGS__, hipStream_t s) { launch(#name, s); }
void launch_seed_count(const SeedVolume&, const SeedParams&, long long nc, int* counts, hipStream_t s) {
  launch("seed_count", s, [=] { std::fill_n(counts, (nc + 255) / 256, 0); });
}
AQ_FAKE(seed_write, const SeedVolume&, const SeedParams&, long long, const int*, long long, Particles)
AQ_FAKE(hash_count, const Geom&, Particles, long long, Bins)
AQ_FAKE(scatter_sort_gather, const Geom&, Particles, Particles, long long, int, Bins)
AQ_FAKE(export_particles, Particles, long long, int, float*, float*, float4*)
AQ_FAKE(p2g, const Geom&, Particles, long long, int, Bins, Grid, int, int, int, StepParams)
AQ_FAKE(gravity_boundary, const Geom&, Grid, int, StepParams, int, int)
AQ_FAKE(divergence, const Geom&, Grid, int, Bins)
AQ_FAKE(refresh_rhs, const Geom&, Grid)
AQ_FAKE(active_list, const Geom&, Grid)
AQ_FAKE(air_pressure_zero, const Geom&, Grid, int)
AQ_FAKE(project, const Geom&, Grid, int, int, int)
AQ_FAKE(build_nvo, const Geom&, Grid, int)
AQ_FAKE(g2p, const Geom&, Particles, long long, int, Grid, int, int, StepParams)
AQ_FAKE(advect, const Geom&, Particles, long long, Grid, int, StepParams)
AQ_FAKE(g2p_advect_hash, const Geom&, Particles, long long, int, Grid, int, int, StepParams, Bins)
AQ_FAKE(stats, const Geom&, Particles, long long, int, Grid, double*, int, double*)
#undef AQ_FAKE
void launch_extrapolate(const Geom&, Grid, int, int, bool, hipStream_t s, bool) { launch("extrapolate", s); }
MgLevel mg_level(int X, int Y, int Z) {
  MgLevel L{};
  L.X = X, L.Y = Y, L.Z = Z, L.n = X * Y * Z;
  return L;
}
int mg_tail_level(const MgLevels& H) { return H.count - 1; }
size_t mg_part_size(const MgLevels&) { return 64; }
// Solved after fake::mg_iters iterations.
void mg_start(const Geom&, const MgLevels&, const MgVectors& V, const uint8_t*, const float*, const float*, double,
              int max_iters, int check_every, hipStream_t s) {
  launch("mg_start", s, [=] {
    *V.S = MgScalars{};
    V.S->max_iters = max_iters, V.S->check_every = check_every;
    *V.report = MgReport{1.0, fake::mg_iters == 0, 1};
  });
}
void mg_iterate(const MgLevels&, const MgVectors& V, int, hipStream_t s) {
  launch("mg_iterate", s, [V] {
    MgScalars& S = *V.S;
    if (++S.it % S.check_every && S.it != S.max_iters) return;
    const bool stop = S.it >= fake::mg_iters;
    *V.report = MgReport{stop ? 0.0 : 1.0, stop, S.it + 1};
  });
}
void mg_finish(const Geom&, const MgLevels&, const MgVectors&, float*, hipStream_t s) { launch("mg_finish", s); }
}  // namespace aqf

// ---- the network's kernels
namespace aqu {
using aqf::Geom;
#define AQ_FAKE(name, ...) \
  void name(__VA_ARGS__, hipStream_t s) { fake::launch(#name, s); }
AQ_FAKE(conv3_dgrad, int, int, const Vol&, const __bf16*, const __bf16*, float*)
AQ_FAKE(conv3_dgrad_relu, int, const Vol&, const __bf16*, const __bf16*, const __bf16*, int, int, __bf16*)
AQ_FAKE(conv3_dgrad_concat, int, int, const Vol&, const __bf16*, const __bf16*, float*, const __bf16*, __bf16*)
AQ_FAKE(conv3_wgrad, int, int, const Vol&, const __bf16*, const __bf16*, int, int, float*, float*, int, float*, float*)
AQ_FAKE(skip_bwd, const Vol&, int, const __bf16*, int, const float*, const float*, __bf16*)
AQ_FAKE(avgpool, const Vol&, int, const __bf16*, int, int, __bf16*)
AQ_FAKE(upsample, const Vol&, int, const __bf16*, __bf16*, int, int)
AQ_FAKE(head_bwd, long long, const __bf16*, const float*, const float*, __bf16*, float*, int, float*)
AQ_FAKE(masked_mse, long long, const float*, const float*, const float*, double*, int, double*, float*)
AQ_FAKE(adam, long long, float*, const float*, float*, float*, float, float, float, float)
AQ_FAKE(pack_weights, int, int, const float*, __bf16*, __bf16*)
AQ_FAKE(mfma_probe, const float*, const float*, float*)
AQ_FAKE(nn_sigma, const Geom&, const uint8_t*, const float*, double*, int, double*)
AQ_FAKE(nn_input, const Geom&, const uint8_t*, const float*, const double*, __bf16*, float*)
AQ_FAKE(nn_target, const Geom&, const uint8_t*, const float*, const double*, float, float*)
AQ_FAKE(nn_guess_gather, const Geom&, const uint8_t*, const float*, float*, float*)
AQ_FAKE(nn_restrict, int, int, int, const float*, const float*, float*, float*)
AQ_FAKE(nn_input_dense, long long, const float*, const float*, double*, int, double*, __bf16*)
AQ_FAKE(nn_output_dense, long long, const float*, const float*, const double*, float, float*)
AQ_FAKE(nn_prolong, int, int, int, const float*, float*)
AQ_FAKE(nn_scatter_scaled, const Geom&, const uint8_t*, const float*, const float*, float*, double*, int, double*)
AQ_FAKE(nn_residual, const Geom&, const uint8_t*, const float*, const float*, float*)
AQ_FAKE(nn_axpy, const Geom&, const uint8_t*, const float*, float*)
#undef AQ_FAKE
void host_input(long long V, const float* x2, __bf16* x0, hipStream_t s) {
  fake::launch("host_input", s, [=] { fake::check(x2, V * 8), fake::check(x0, V * 16); });
}
void conv3_forward(int cin, int cout, const Vol& v, const __bf16* X, int xs, int, const __bf16*, const float*, __bf16* Y,
                   int ys, int, hipStream_t s) {
  const size_t V = (size_t)v.B * v.D * v.H * v.W;
  fake::launch("conv3_forward", s, [=] { fake::check(X, V * xs * 2), fake::check(Y, V * ys * 2); });
}
void head_fwd(long long V, int C, const __bf16* X, const float*, const float*, float* y, hipStream_t s) {
  fake::launch("head_fwd", s, [=] { fake::check(X, (size_t)V * C * 2), fake::check(y, (size_t)V * 4); });
}
}  // namespace aqu
