// flip_api.cpp -- C ABI of libaqflip (include/aqflip.h).
//
// Host orchestration of Fluid_3D_FLIP::Fluid (Fluid/Fluid_3D_FLIP.cu:316-505) for
// one GPU: every stage is enqueued on the handle's own HIP stream with no host
// synchronisation inside a step (the reference synchronises about 30 times per
// step); entry points synchronise once before returning. Errors come back as
// aq_status with a thread-local message instead of exit().
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/aqflip.h"
#include "../../include/aqflip_unet.h"
#include "aqflip_internal.h"
#include "flip_view.h"
#include "mgpcg.h"

namespace aqf {
int64_t seed_scene(const aq_flip_config& cfg, std::vector<float>* pos, std::vector<float>* frac);
}

using namespace aqf;

namespace {

thread_local std::string g_err;

aq_status fail(aq_status s, const std::string& msg) {
  g_err = msg;
  return s;
}

#define HIP_TRY(expr)                                                                         \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess) {                                                                   \
      (void)hipGetLastError(); /* reported here, not by the next call */                      \
      return fail(e_ == hipErrorOutOfMemory ? AQ_ENOMEM : AQ_EHIP,                            \
                  std::string(#expr) + ": " + hipGetErrorString(e_));                         \
    }                                                                                         \
  } while (0)

#define AQ_TRY(expr)              \
  do {                            \
    aq_status s_ = (expr);        \
    if (s_ != AQ_OK) return s_;   \
  } while (0)

// Device memory of handles, kept for the next handle. Mapping and unmapping a handle's
// memory cost more than a short scene's steps (64^3: 1 + 7 ms against 0.37 ms a step;
// 256^3: 7 + 11 ms, and 150 ms once a process had cycled through the card's memory), so a
// destroyed handle's blocks are kept and handed to the next request that they fit. Blocks
// enter after their handle's streams have been synchronised and are cleared by whoever
// takes them, so neither threads nor streams matter beyond the lock. Bounded: at most
// kKeepBytes per device, and a block that kKeepPuts later ones passed over is freed. All are
// when an allocation of this library fails (device_malloc) and when the caller asks for it
// (aq_flip_release_memory); nothing else in the process or outside it can. Blocks below
// kKeepMin are not kept: the runtime serves those from its own chunks.
class BlockCache {
 public:
  // size, device: the block's, for put().
  hipError_t get(size_t bytes, void** p, size_t* size, int* device) {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    *device = dev;
    *size = bytes;
    if (bytes < kKeepMin) return device_malloc(p, bytes);
    *size = (bytes + kGranule - 1) / kGranule * kGranule;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      auto best = blocks_.end();
      for (auto b = blocks_.begin(); b != blocks_.end(); ++b)
        if (b->dev == dev && b->size >= bytes && b->size <= *size + *size / 4 &&
            (best == blocks_.end() || b->size < best->size))
          best = b;
      if (best != blocks_.end()) {
        *p = best->p;
        *size = best->size;
        blocks_.erase(best);
        return hipSuccess;
      }
    }
    return device_malloc(p, *size);
  }
  // p: no work on it is pending.
  void put(void* p, size_t size, int dev) {
    if (size < kKeepMin) {
      (void)hipFree(p);
      return;
    }
    std::lock_guard<std::mutex> lock(mutex_);
    try {
      blocks_.push_back(Block{p, size, dev, ++puts_});
    } catch (const std::bad_alloc&) {
      (void)hipFree(p);
      return;
    }
    size_t held = 0;  // newest first, what fits the bound stays
    for (size_t i = blocks_.size(); i-- > 0;) {
      const Block& b = blocks_[i];
      if (b.dev != dev) continue;
      held += b.size;
      if (held <= kKeepBytes && puts_ - b.at < kKeepPuts) continue;
      held -= b.size;
      (void)hipFree(b.p);
      blocks_.erase(blocks_.begin() + (long)i);
    }
  }
  // Frees every block; whether there was one.
  bool release() {
    std::lock_guard<std::mutex> lock(mutex_);
    const bool any = !blocks_.empty();
    for (const Block& b : blocks_) (void)hipFree(b.p);
    blocks_.clear();
    return any;
  }

 private:
  static constexpr size_t kGranule = 1 << 21, kKeepMin = 1 << 20, kKeepBytes = 12ull << 30;
  static constexpr uint64_t kKeepPuts = 64;
  struct Block {
    void* p;
    size_t size;
    int dev;
    uint64_t at;
  };
  std::mutex mutex_;
  std::vector<Block> blocks_;
  uint64_t puts_ = 0;
};
// Never destroyed: at process exit the runtime may be gone before it, and the memory goes
// with the process.
BlockCache& block_cache() {
  static BlockCache* c = new BlockCache;
  return *c;
}

int boundary_coverage(int A, int B, bool ref) {
  const int pairs = (A + 1) * (B + 1);
  if (!ref) return pairs;
  const int total = A * B;
  const int nt = std::min(1024, total);
  // divUp (Common/Commons.h:7-13)
  const int blocks = nt == 0 ? 1 : (total % nt != 0 ? total / nt + 1 : total / nt);
  return (int)std::min<long long>((long long)blocks * nt, pairs);
}

}  // namespace

struct aq_flip {
  aq_flip_config cfg{};
  Geom G{};
  int K = 1;
  long long Np = 0;
  hipStream_t stream = nullptr;
  // Diffusion of the phase fractions depends on neither pressure nor velocities, so
  // inside a step its sweeps run on a second stream, concurrently with the pressure
  // solve, projection and extrapolation (fork after the divergence pass, join before
  // the step ends).
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  bool overlap = true;
  // With the fixed-sweep solver, diffusion sweeps share launches with pressure sweeps
  // (fused_pressure_diffusion) instead of running on the second stream.
  bool fuse = true;
  // Paired diffusion sweeps after one that changed no bit skip their identical work.
  bool skip_fixed = true;
  int listed_grid = 0;  // 0: the default listed sweep grids; n: at most n workgroups
  struct Alloc {
    void* p;
    size_t size;
    int dev;
  };
  std::vector<Alloc> allocs;

  Particles P[2]{};
  int cur = 0;
  Grid gr{};
  int nv = 0, hv = 0, pb = 0, nf = 0;  // current buffer of each ping-pong pair
  // air_clean[i]: pressure buffer i holds 0 on every AIR cell of the current content.
  bool air_clean[2] = {false, false};
  bool p2g_content = false;  // every interior cell is AIR or FLUID (see content_changed)
  long long fluid = 0;       // FLUID cells to expect (see expect_fluid)
  Bins B{};
  StepParams sp{};
  int nparts_red = 0;
  double* red_partial = nullptr;
  double* red_out = nullptr;
  float physicalTime = 0.f;

  // Pressure solve mode (fixed sweeps as the reference, or to a tolerance).
  aq_flip_solver solver{AQ_SOLVE_FIXED, 1e-4, 100000, 50, 20, 0};
  aq_unet* net = nullptr;
  aq_flip_solver_stats sstats{};
  // Scratch of field exports beyond a particle array, at most kExportBytes.
  void* export_buf = nullptr;
  size_t export_cap = 0;
  static constexpr size_t kExportBytes = 32 << 20;
  float* p_keep = nullptr;  // the iterate before a U-Net correction (allocated on first use)

  bool timing = false;
  double stage_ms[AQ_STAGE_COUNT]{};
  int64_t stage_calls[AQ_STAGE_COUNT]{};
  // Stage timing: event pairs recorded on this handle's stream while a step is
  // enqueued, read back only at the synchronisation point that ends the call.
  struct Mark {
    int stage;
    hipEvent_t a, b;
    int64_t passes;
  };
  // Captured steps: one executable graph per ping-pong state at step entry (odd
  // pass counts alternate buffers between steps), with the state it leaves.
  struct StepGraph {
    int key[7];
    int next[7];
    hipGraph_t graph;
    hipGraphExec_t exec;
  };
  std::vector<StepGraph> graphs;
  bool use_graphs = true;
  bool nvo_valid = false;  // gr.nvo matches newVelocity and velocity (see graph_step)
  // Tolerance solves: k Jacobi sweeps plus the FP64 residual kernels between two
  // host checks, captured once per (pressure buffer, AIR-clean state, kind of content, k).
  struct SweepGraph {
    int key[6];   // pb, air_clean[0], air_clean[1], p2g_content, k, whether the iterate is kept first
    int next[3];  // pb, air_clean[0], air_clean[1] afterwards
    hipGraph_t graph;
    hipGraphExec_t exec;
  };
  std::vector<SweepGraph> sweep_graphs;
  // 16 chunk lengths and buffer states, each on either kind of content and with the iterate
  // kept or not.
  static constexpr size_t kMaxSweepGraphs = 16 * 4;
  SweepReport* report = nullptr;  // pinned, two; the device's view of it
  SweepReport* report_dev = nullptr;
  int* reports = nullptr;         // device count of the reports written
  int reports_due = 0;            // and of those enqueued
  bool reports_lost = false;      // an error came between: the two may differ
  float* p_ahead = nullptr;       // the iterate before the chunk that runs ahead
  // Multigrid-preconditioned CG (allocated on first use). The iteration's launches are
  // captured once per parity from the handle's second solve on.
  struct MgState {
    MgLevels H{};
    MgVectors V{};
    MgReport* report = nullptr;  // pinned
    long long solves = 0;
    bool running = false;  // a solve has begun and has not come to its end
    hipGraph_t graph[2] = {};
    hipGraphExec_t exec[2] = {};
    ~MgState() {
      for (int k = 0; k < 2; ++k) {
        if (exec[k]) hipGraphExecDestroy(exec[k]);
        if (graph[k]) hipGraphDestroy(graph[k]);
      }
      if (report) hipHostFree(report);
    }
  };
  MgState* mg = nullptr;
  std::vector<hipEvent_t> event_pool;
  std::vector<Mark> pending;
  size_t pool_used = 0;
  hipEvent_t open_event = nullptr;

  ~aq_flip() {
    if (stream) hipStreamSynchronize(stream);
    delete mg;
    if (report) hipHostFree(report);
    for (StepGraph& g : graphs) {
      hipGraphExecDestroy(g.exec);
      hipGraphDestroy(g.graph);
    }
    for (SweepGraph& g : sweep_graphs) {
      hipGraphExecDestroy(g.exec);
      hipGraphDestroy(g.graph);
    }
    if (side) hipStreamSynchronize(side);
    for (const Alloc& a : allocs) block_cache().put(a.p, a.size, a.dev);
    for (hipEvent_t e : event_pool) hipEventDestroy(e);
    if (ev_fork) hipEventDestroy(ev_fork);
    if (ev_join) hipEventDestroy(ev_join);
    if (side) hipStreamDestroy(side);
    if (stream) hipStreamDestroy(stream);
  }

  // Zeroed.
  aq_status alloc(void** p, size_t bytes) {
    size_t size = 0;
    int dev = 0;
    HIP_TRY(block_cache().get(bytes, p, &size, &dev));
    allocs.push_back({*p, size, dev});
    HIP_TRY(hipMemsetAsync(*p, 0, bytes, stream));
    return AQ_OK;
  }
  template <typename T>
  aq_status allocT(T** p, size_t n) {
    return alloc((void**)p, std::max<size_t>(n, 1) * sizeof(T));
  }

  hipEvent_t next_event() {
    if (pool_used == event_pool.size()) {
      hipEvent_t e = nullptr;
      if (hipEventCreate(&e) != hipSuccess) return nullptr;
      event_pool.push_back(e);
    }
    return event_pool[pool_used++];
  }
  void begin(int st) {
    (void)st;
    if (!timing) return;
    open_event = next_event();
    if (open_event) hipEventRecord(open_event, stream);
  }
  void end(int st, int64_t passes = 1) {
    if (!timing || !open_event) return;
    hipEvent_t e = next_event();
    if (!e) return;
    hipEventRecord(e, stream);
    pending.push_back({st, open_event, e, passes});
    open_event = nullptr;
  }
  // Called after the stream has been synchronised.
  aq_status collect() {
    for (const Mark& m : pending) {
      float ms = 0.f;
      HIP_TRY(hipEventElapsedTime(&ms, m.a, m.b));
      stage_ms[m.stage] += ms;
      stage_calls[m.stage] += m.passes;
    }
    pending.clear();
    pool_used = 0;
    return AQ_OK;
  }
};

namespace {

aq_status validate(const aq_flip_config* c) {
  if (!c) return fail(AQ_EINVAL, "null config");
  for (int a = 0; a < 3; ++a)
    if (c->size[a] < 1 || c->size[a] > 1024)
      return fail(AQ_EINVAL, "grid size must be in [1, 1024] on every axis");
  if ((long long)c->size[0] * c->size[1] * c->size[2] > (1ll << 30))
    return fail(AQ_EINVAL, "grid too large");
  if (c->phase_count > 4) return fail(AQ_EINVAL, "Only supports up to 4 phases");
  if (c->phase_count < 1) return fail(AQ_EINVAL, "phase_count must be >= 1");
  if (c->n_volumes < 0 || c->n_volumes > AQ_MAX_VOLUMES)
    return fail(AQ_EINVAL, "n_volumes out of range");
  if (!(c->grid_physical_size > 0) || !std::isfinite(c->grid_physical_size))
    return fail(AQ_EINVAL, "grid_physical_size must be positive");
  if (!std::isfinite(c->dt) || !std::isfinite(c->flip_coeff))
    return fail(AQ_EINVAL, "dt and flip_coeff must be finite");
  if (c->pressure_iters < 0 || c->diffusion_iters < 0)
    return fail(AQ_EINVAL, "iteration counts must be >= 0");
  if (c->pressure_init != AQ_PRESSURE_ZERO && c->pressure_init != AQ_PRESSURE_PREVIOUS)
    return fail(AQ_EINVAL, "pressure_init must be AQ_PRESSURE_ZERO or AQ_PRESSURE_PREVIOUS");
  return AQ_OK;
}

// Number of volume-fraction channels in use: phases 0..K-1 can be non-zero; the
// remaining channels are provably zero throughout the step.
int channels_for(const aq_flip_config& c, const float* frac4, long long n) {
  int K = std::max(1, std::min(4, c.phase_count));
  for (int i = 0; i < c.n_volumes; ++i)
    if (c.volumes[i].phase >= 0 && c.volumes[i].phase < 4) K = std::max(K, c.volumes[i].phase + 1);
  if (frac4)
    for (long long i = 0; i < n; ++i)
      for (int a = 3; a >= K; --a)
        if (frac4[4 * i + a] != 0.f) {
          K = a + 1;
          break;
        }
  return K;
}

// Positions must hash into the grid (calcHashImpl would index out of range otherwise).
// cells: how many cells they lie in, where a choice of kernels depends on it (below 2^20 cells),
// else 0.
aq_status check_positions(const aq_flip* h, const float* pos, long long n, long long* cells) {
  const int S[3] = {h->G.X, h->G.Y, h->G.Z};
  std::vector<bool> seen(h->G.ncells_hash < kTileLongCells ? (size_t)h->G.ncells_hash : 0);
  *cells = 0;
  for (long long i = 0; i < n; ++i) {
    int c[3];
    for (int a = 0; a < 3; ++a) {
      const float v = pos[3 * i + a];
      if (!(v >= 0.f) || (c[a] = (int)(v / h->G.h)) >= S[a])
        return fail(AQ_EINVAL, "particle " + std::to_string(i) + " lies outside the grid");
    }
    if (seen.empty()) continue;
    const size_t at = ((size_t)c[0] * S[1] + c[1]) * S[2] + c[2];
    *cells += !seen[at];
    seen[at] = true;
  }
  return AQ_OK;
}

// Hands out the arrays of one block, 256 bytes apart at least; without a base it only
// measures.
struct Carver {
  char* base = nullptr;
  size_t at = 0;
  template <typename T>
  void take(T** p, size_t n) {
    *p = base ? (T*)(base + at) : nullptr;
    at += (std::max<size_t>(n, 1) * sizeof(T) + 255) / 256 * 256;
  }
};
void carve_arrays(aq_flip* h, Carver& c) {
  const Geom& G = h->G;
  const size_t Np = (size_t)h->Np, nc = (size_t)G.ncell, nch = (size_t)G.ncells_hash;
  for (int b = 0; b < 2; ++b) {
    c.take(&h->P[b].a, Np);
    c.take(&h->P[b].b, Np);
    c.take(&h->P[b].c, Np);
  }
  Grid& gr = h->gr;
  c.take(&gr.content, nc);
  for (int a = 0; a < 3; ++a) {
    c.take(&gr.vel[a], nc);
    c.take(&gr.nvel[0][a], nc);
    c.take(&gr.nvel[1][a], nc);
    c.take(&gr.nvo[a], nc);
  }
  for (int b = 0; b < 2; ++b) {
    c.take(&gr.hasvel[b], nc);
    c.take(&gr.p[b], nc);
  }
  c.take(&gr.div, nc);
  c.take(&gr.rhs, nc);
  c.take(&gr.density, nc);
  // One flag per 256-cell block plus one slot that stays 0, so the sweep kernels'
  // pairs of blocks never read past the array.
  c.take(&gr.active, (nch + 255) / 256 + 1);
  c.take(&gr.alist, (size_t)sweep_chunks(G) + 1);
  c.take(&gr.btab, (size_t)sweep_table_entries(G));
  c.take(&gr.tactive, (size_t)sweep_tiles(G));
  c.take(&gr.tlist, (size_t)sweep_tiles(G) + 1);
  c.take(&gr.ttab, (size_t)tile_grid(G));
  c.take(&gr.dchange, 4);
  c.take(&gr.stepstamp, 1);
  c.take(&gr.rowstamp, (size_t)(G.X + 1) * (G.Y + 1));
  for (int a = 0; a < 4; ++a) {
    c.take(&gr.vf[a], nc);
    c.take(&gr.nvf[0][a], nc);
    c.take(&gr.nvf[1][a], nc);
  }
  c.take(&h->B.count, nch);
  c.take(&h->B.offsets, nch + 1);
  c.take(&h->B.partials, (nch + 4095) / 4096 + 1);
  c.take(&h->B.hash, Np);
  c.take(&h->B.rank, Np);
  c.take(&h->B.perm, Np);
  c.take(&h->B.multi, nch);  // zeroed here; k_segsort clears what it reads
  h->nparts_red = 512;  // volume statistics: 512 partial rows of 16 columns
  // (the residual uses two columns per sweep chunk)
  c.take(&h->red_partial, std::max<size_t>((size_t)h->nparts_red * 16, 2 * (size_t)sweep_chunks(G)));
  c.take(&h->red_out, 16);
}

aq_status setup(aq_flip* h, const aq_flip_config* cfg, long long Np) {
  h->cfg = *cfg;
  Geom& G = h->G;
  G.X = cfg->size[0];
  G.Y = cfg->size[1];
  G.Z = cfg->size[2];
  G.EY = G.Y + 1;
  G.EZ = ((G.Z + 1) + 7) / 8 * 8;
  G.sx = (long long)G.EY * G.EZ;
  G.ncell = (long long)(G.X + 1) * G.sx;
  G.ncells_hash = G.X * G.Y * G.Z;
  G.nfaces = (G.X + 1) * (G.Y + 1) * (G.Z + 1);
  G.h = cfg->grid_physical_size / (float)G.Y;  // Fluid_3D_FLIP.cu:444
  G.inv_h = 1.0 / (double)G.h;
  G.divZ = make_fastdiv((uint32_t)G.Z);
  G.divYZ = make_fastdiv((uint32_t)(G.Y * G.Z));
  G.divZ1 = make_fastdiv((uint32_t)(G.Z + 1));
  G.divYZ1 = make_fastdiv((uint32_t)((G.Y + 1) * (G.Z + 1)));
  h->Np = Np;

  StepParams& sp = h->sp;
  sp.dt = cfg->dt;
  sp.flip = cfg->flip_coeff;
  for (int a = 0; a < 3; ++a) sp.g[a] = cfg->gravity[a];
  for (int a = 0; a < 4; ++a) sp.rho[a] = cfg->phase_densities[a];
  sp.lambda = (cfg->diffusion_coeff * cfg->dt) / (G.h * G.h);  // Fluid_3D_common.cu:86
  sp.inv_cc = 1.0 / (double)(1.f + 2.f * sp.lambda);             // Fluid_3D_kernels.cu:538
  const bool ref = cfg->ref_boundary_coverage != 0;
  sp.coverX = boundary_coverage(G.Y, G.Z, ref);
  sp.coverY = boundary_coverage(G.X, G.Z, ref);
  sp.coverZ = boundary_coverage(G.X, G.Y, ref);

  HIP_TRY(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  HIP_TRY(hipStreamCreateWithFlags(&h->side, hipStreamNonBlocking));
  HIP_TRY(hipEventCreateWithFlags(&h->ev_fork, hipEventDisableTiming));
  HIP_TRY(hipEventCreateWithFlags(&h->ev_join, hipEventDisableTiming));
  // One block for every array: measured first, then carved.
  Carver c;
  carve_arrays(h, c);
  AQ_TRY(h->alloc((void**)&c.base, c.at));
  c.at = 0;
  carve_arrays(h, c);
  set_listed_grids(G, h->gr, h->listed_grid);
  return AQ_OK;
}

void refresh_rhs(aq_flip* h) { launch_refresh_rhs(h->G, h->gr, h->stream); }

aq_status upload_particles(aq_flip* h, const float* pos, const float* vel, const float* frac4) {
  const long long n = h->Np;
  std::vector<float4> a((size_t)n), b((size_t)n), c((size_t)n);
  for (long long i = 0; i < n; ++i) {
    const float* p = pos + 3 * i;
    float v[3] = {0.f, 0.f, 0.f}, f[4] = {0.f, 0.f, 0.f, 0.f};
    if (vel)
      for (int k = 0; k < 3; ++k) v[k] = vel[3 * i + k];
    if (frac4)
      for (int k = 0; k < 4; ++k) f[k] = frac4[4 * i + k];
    a[i] = make_float4(p[0], p[1], p[2], v[0]);
    b[i] = make_float4(v[1], v[2], f[0], f[1]);
    c[i] = make_float4(f[2], f[3], 0.f, 0.f);
  }
  const Particles& P = h->P[h->cur];
  HIP_TRY(hipMemcpyAsync(P.a, a.data(), n * sizeof(float4), hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(P.b, b.data(), n * sizeof(float4), hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(P.c, c.data(), n * sizeof(float4), hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return AQ_OK;
}

// ---- stages --------------------------------------------------------------

// New FLUID/AIR marking: AIR cells of either pressure buffer may hold old values.
// p2g: the marking is P2G's, AIR or FLUID on every interior cell (an upload may hold others).
void content_changed(aq_flip* h, bool p2g) {
  h->air_clean[0] = h->air_clean[1] = false;
  h->p2g_content = p2g;
}

// hash is already binned (count filled): scan, scatter, segment sort, gather, P2G.
// Inside a step the P2G kernel is timed in its own bucket (split = true).
void transfer_after_count(aq_flip* h, bool split = false) {
  launch_scan(h->G, h->B, h->stream);
  launch_scatter_sort_gather(h->G, h->P[h->cur], h->P[h->cur ^ 1], h->Np, h->K, h->B, h->stream);
  h->cur ^= 1;
  if (split) {
    h->end(AQ_STAGE_TRANSFER_TO_GRID);
    h->begin(AQ_STAGE_P2G);
  }
  launch_p2g(h->G, h->P[h->cur], h->Np, h->K, h->B, h->gr, h->nv, h->hv, h->nf, h->sp, h->stream);
  if (split) h->end(AQ_STAGE_P2G);
  content_changed(h, true);
}

void clear_bins(aq_flip* h) { launch_fill_u32(h->B.count, 0u, h->G.ncells_hash, h->stream); }

void stage_transfer(aq_flip* h) {
  clear_bins(h);
  launch_hash_count(h->G, h->P[h->cur], h->Np, h->B, h->stream);
  transfer_after_count(h);
}

// n Jacobi sweeps. Every sweep leaves 0 on all AIR cells of its output buffer, so
// a sweep whose output buffer already holds those zeros may skip AIR cells and
// blocks without FLUID (the result is identical); otherwise it writes every cell.
// from_zero: the sweeps start from the zero guess; the first one does not read the
// input buffer (its neighbours are 0) and writes every cell, so neither buffer needs
// clearing first.
//
// Small grids run all n sweeps in one launch, in place. One workgroup per chain does the
// work, so the rule weighs the FLUID cells to expect (times K with the diffusion chain beside
// it) against tile launches of four sweeps. Microseconds per step, one launch / tiles, sweep counts in brackets: 16^3 with 1,160
// FLUID cells 109/164 (100), 81/86 (16), with 3,900 146/170 (100); 24^3 with 3,900 165/175
// (100), 102/94 (16); 27^3 with 5,600 205/177 (100). Both chains, 100 sweeps each, K = 2: 16^3
// with 1,160 107/175, with 3,900 and phases mixing 286/296, 18^3 with 5,500 608/464; K = 4,
// mixing: 12^3 with 1,640 403/430, 16^3 with 3,900 587/440.
constexpr int kSmallSweeps = 16;
// With four phases the line lies lower for the sake of a longer diffusion chain, whose rest is
// quicker in launches of its own (30 + 100 sweeps, 1,210 FLUID cells mixing: 394/364).
constexpr long long kSmallPressure = 4096, kSmallPaired = 8192, kSmallPaired4 = 4500;
bool small_cells(const aq_flip* h, int K) {
  return small_grid(h->G, K) && (K > 1 ? h->fluid * K <= (K < 4 ? kSmallPaired : kSmallPaired4) : h->fluid <= kSmallPressure);
}
bool small_sweeps(const aq_flip* h, int n, int K) {
  return n >= kSmallSweeps && h->p2g_content && small_cells(h, K);
}
void jacobi_sweeps(aq_flip* h, int n, bool from_zero = false) {
  if (small_sweeps(h, n, 1)) {
    launch_sweeps_small(h->G, h->gr, 1, h->pb, from_zero ? 1 : 0, n, h->nf, 0.f, 1.0, 0, 0, 0, h->stream);
    h->air_clean[h->pb] = true;
    return;
  }
  const bool tiles = h->p2g_content && tile_fits(h->G);
  for (int i = 0; i < n;) {
    const int out = h->pb ^ 1;
    const bool z = from_zero && i == 0, full = z || !h->air_clean[out];
    if (tiles && n - i >= tile_sweeps() && (!full || tile_full(h->G))) {
      launch_jacobi_tile(h->G, h->gr, h->pb, full ? 1 : 0, z ? 1 : 0, h->stream);
      i += tile_sweeps();
    } else {
      launch_jacobi(h->G, h->gr, h->pb, full ? 1 : 0, z ? 1 : 0, h->stream);
      ++i;
    }
    h->air_clean[out] = true;
    h->pb = out;
  }
}

// Zero pressure start: both buffers cleared.
void zero_pressure(aq_flip* h) {
  launch_fill_pressure_zero(h->G, h->gr, h->pb, h->stream);
  launch_fill_pressure_zero(h->G, h->gr, h->pb ^ 1, h->stream);
  h->air_clean[0] = h->air_clean[1] = true;
}
// The fixed-sweep solve: pressure_iters sweeps from the configured start.
void fixed_sweeps(aq_flip* h) {
  const bool zero = h->cfg.pressure_init == AQ_PRESSURE_ZERO;
  if (zero && h->cfg.pressure_iters == 0) zero_pressure(h);
  jacobi_sweeps(h, h->cfg.pressure_iters, zero);
}

void stage_pressure(aq_flip* h) { fixed_sweeps(h); }

// Inside a step (in_step) the second and third passes visit only the face rows this
// step's P2G stamped (k_extrapolate); the stage on its own runs every pass in full.
// Inside a step the last pass also writes the interleaved (newVelocity, velocity) copy the
// next step's G2P samples (gr.nvo), on the rows it visits.
void stage_extrapolate(aq_flip* h, bool in_step = false) {
  for (int i = 0; i < 3; ++i) {  // maxDistance = 3 (Fluid_3D_common.cu:74)
    launch_extrapolate(h->G, h->gr, h->nv, h->hv, in_step && i > 0, h->stream, in_step && i == 2);
    h->nv ^= 1;
    h->hv ^= 1;
  }
}

// Diffusion sweeps first..diffusion_iters-1 of the step (first > 0: after `launch` paired
// launches). After paired sweeps every kRecordEvery-th, the first among them, records whether
// it changed a bit, under the next launch's number.
constexpr int kRecordEvery = 4;
void diffusion_sweeps(aq_flip* h, hipStream_t s, int first = 0, int launch = 0) {
  const bool chained = first > 0 && h->skip_fixed;
  for (int i = first; i < h->cfg.diffusion_iters; ++i) {  // the first sweep also copies AIR cells across
    const bool record = chained && (i - first) % kRecordEvery == 0;
    launch_diffusion(h->G, h->gr, h->K, h->nf, h->sp.lambda, h->sp.inv_cc, i == 0 ? 1 : 0, chained ? launch - 1 : -1,
                     record ? launch : -1, s);
    launch += record;
    h->nf ^= 1;
  }
}

// Fixed-sweep pressure solve and the diffusion sweeps together: the first
// min(pressure_iters, diffusion_iters) sweeps of each share launches, one or several of
// each at a time, the rest of the longer chain has its own. Same iterates as the two loops.
void fused_pressure_diffusion(aq_flip* h) {
  const bool zero = h->cfg.pressure_init == AQ_PRESSURE_ZERO;  // first sweep from the zero guess
  const int n = std::min(h->cfg.pressure_iters, h->cfg.diffusion_iters);
  h->begin(AQ_STAGE_PRESSURE_DIFFUSION);
  const bool small = small_sweeps(h, n, h->K);
  const bool whole = small && !h->timing;  // both chains to their ends, side by side
  if (small) {  // (timed, the longer chain's rest has launches and a bucket of its own)
    launch_sweeps_small(h->G, h->gr, h->K, h->pb, zero ? 1 : 0, whole ? h->cfg.pressure_iters : n, h->nf, h->sp.lambda,
                        h->sp.inv_cc, whole ? h->cfg.diffusion_iters : n, n, h->skip_fixed ? 1 : 0, h->stream);
    h->air_clean[h->pb] = true;
  }
  int launch = 0;  // the step's paired launches, numbered for the diffusion's skipping
  for (int i = 0; i < n && !small; ++launch) {
    const int out = h->pb ^ 1;
    const bool z = zero && i == 0, full = z || !h->air_clean[out];
    if (i > 0 && !full && n - i >= tile_sweeps() && tile_pairs(h->G, h->K, h->fluid)) {
      launch_tile_pair(h->G, h->gr, h->K, h->pb, h->nf, h->sp.lambda, h->sp.inv_cc, launch, h->skip_fixed ? 1 : 0,
                       h->stream);
      i += tile_sweeps();
    } else {
      launch_jacobi_diffusion(h->G, h->gr, h->K, h->pb, full ? 1 : 0, h->nf, h->sp.lambda, h->sp.inv_cc,
                              i == 0 ? 1 : 0, z ? 1 : 0, launch, h->skip_fixed ? 1 : 0, h->stream);
      ++i;
    }
    h->air_clean[out] = true;
    h->pb = out;
    h->nf ^= 1;
  }
  h->end(AQ_STAGE_PRESSURE_DIFFUSION, n);
  h->begin(AQ_STAGE_PRESSURE);
  if (!whole) jacobi_sweeps(h, h->cfg.pressure_iters - n);
  h->end(AQ_STAGE_PRESSURE, h->cfg.pressure_iters - n);
  h->begin(AQ_STAGE_DIFFUSION);
  if (!small)
    diffusion_sweeps(h, h->stream, n, launch);
  else if (!whole && h->cfg.diffusion_iters > n)
    launch_sweeps_small(h->G, h->gr, h->K, h->pb, 0, 0, h->nf, h->sp.lambda, h->sp.inv_cc, h->cfg.diffusion_iters - n, 0,
                        1, h->stream);
  h->end(AQ_STAGE_DIFFUSION, h->cfg.diffusion_iters - n);
}

// inStep: the grid fractions were produced by this step's P2G, so with a single
// channel they are exactly 1 (FLUID) or 0 (AIR) and every sweep is the identity;
// Jacobi with >= 1 sweep has already zeroed AIR pressure.
// Returns the number of diffusion sweeps run.
int stage_diffusion(aq_flip* h, bool inStep) {
  if (h->cfg.diffusion_iters <= 0) return 0;
  if (!inStep || h->cfg.pressure_iters == 0) launch_air_pressure_zero(h->G, h->gr, h->pb, h->stream);
  if (inStep && h->K == 1) return 0;
  diffusion_sweeps(h, h->stream);
  return h->cfg.diffusion_iters;
}

aq_status run_stage(aq_flip* h, int st) {
  if (st == AQ_STAGE_PRESSURE_DIFFUSION || st == AQ_STAGE_P2G)
    return fail(AQ_EINVAL, "timing bucket: runs only inside a step");
  h->nvo_valid = false;
  if (st < 0 || st >= AQ_STAGE_COUNT) return fail(AQ_EINVAL, "unknown stage");
  int64_t passes = 1;
  h->begin(st);
  switch (st) {
    case AQ_STAGE_G2P: launch_g2p(h->G, h->P[h->cur], h->Np, h->K, h->gr, h->nv, h->nf, h->sp, h->stream); break;
    case AQ_STAGE_ADVECT: launch_advect(h->G, h->P[h->cur], h->Np, h->gr, h->nv, h->sp, h->stream); break;
    case AQ_STAGE_TRANSFER_TO_GRID:
      stage_transfer(h);
      refresh_rhs(h);  // content changed: re-mark AIR for Jacobi
      break;
    case AQ_STAGE_GRAVITY: launch_gravity_boundary(h->G, h->gr, h->nv, h->sp, 1, 0, h->stream); break;
    case AQ_STAGE_BOUNDARY: launch_gravity_boundary(h->G, h->gr, h->nv, h->sp, 0, 1, h->stream); break;
    case AQ_STAGE_DIVERGENCE: launch_divergence(h->G, h->gr, h->nv, h->B, h->stream); break;
    case AQ_STAGE_PRESSURE:
      stage_pressure(h);
      passes = h->cfg.pressure_iters;
      break;
    case AQ_STAGE_PROJECT: launch_project(h->G, h->gr, h->nv, h->hv, h->pb, h->stream); break;
    case AQ_STAGE_EXTRAPOLATE:
      stage_extrapolate(h);
      passes = 3;
      break;
    case AQ_STAGE_DIFFUSION: passes = stage_diffusion(h, false); break;
    default: break;
  }
  HIP_TRY(hipGetLastError());
  h->end(st, passes);
  return AQ_OK;
}

// ---- multigrid-preconditioned CG ---------------------------------------------
aq_status mg_setup(aq_flip* h) {
  if (h->mg) return AQ_OK;
  std::unique_ptr<aq_flip::MgState> M(new aq_flip::MgState);
  const Geom& G = h->G;
  MgLevels& H = M->H;
  int X = G.X, Y = G.Y, Z = G.Z;
  auto guarded = [&](auto** p, const MgLevel& L) -> aq_status {
    AQ_TRY(h->allocT(p, (size_t)L.n + 2 * (size_t)mg_guard(L)));
    *p += mg_guard(L);
    return AQ_OK;
  };
  for (;;) {  // halve every axis down to a few cells
    MgLevel& L = H.L[H.count++];
    L = mg_level(X, Y, Z);
    AQ_TRY(guarded(&L.code, L));
    for (float** p : {&L.f, &L.u, &L.t}) AQ_TRY(guarded(p, L));
    if (std::max(X, std::max(Y, Z)) <= 4) break;
    X = (X + 1) / 2, Y = (Y + 1) / 2, Z = (Z + 1) / 2;
  }
  H.tail = mg_tail_level(H);
  MgVectors& V = M->V;
  for (double** p : {&V.x, &V.r, &V.q, &V.d[0], &V.d[1]}) AQ_TRY(guarded(p, H.L[0]));
  AQ_TRY(h->allocT(&V.part, mg_part_size(H)));
  AQ_TRY(h->allocT(&V.S, 1));
  HIP_TRY(hipHostMalloc((void**)&M->report, sizeof(MgReport), hipHostMallocMapped));
  HIP_TRY(hipHostGetDevicePointer((void**)&V.report, M->report, 0));
  h->mg = M.release();
  return AQ_OK;
}

// Waits until *seq has reached want. Every report is written by a kernel already
// queued on the stream; if the stream runs empty without it, a launch failed.
aq_status wait_report(aq_flip* h, const int* seq, int want) {
  auto there = [&] { return __atomic_load_n(seq, __ATOMIC_ACQUIRE) >= want; };
  for (unsigned spin = 1; !there(); ++spin) {
    if (spin % 4096) continue;
    const hipError_t e = hipStreamQuery(h->stream);
    if (e == hipErrorNotReady) continue;
    if (e != hipSuccess) return fail(AQ_EHIP, std::string("solver: ") + hipGetErrorString(e));
    if (!there()) return fail(AQ_EHIP, "solver: the residual was not reported");
  }
  return AQ_OK;
}
aq_status mg_wait(aq_flip* h, int seq) { return wait_report(h, &h->mg->report->seq, seq); }

aq_status mg_enqueue(aq_flip* h, int odd) {
  aq_flip::MgState& M = *h->mg;
  if (h->timing || !h->use_graphs || M.solves == 0) {
    mg_iterate(M.H, M.V, odd, h->stream);
    return AQ_OK;
  }
  if (!M.exec[odd]) {
    HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    mg_iterate(M.H, M.V, odd, h->stream);
    const hipError_t e = hipStreamEndCapture(h->stream, &M.graph[odd]);
    if (e != hipSuccess) {
      (void)hipGetLastError();  // reported here, not by the next call
      return fail(AQ_EHIP, std::string("MG-PCG capture: ") + hipGetErrorString(e));
    }
    HIP_TRY(hipGraphInstantiate(&M.exec[odd], M.graph[odd], nullptr, nullptr, 0));
  }
  HIP_TRY(hipGraphLaunch(M.exec[odd], h->stream));
  return AQ_OK;
}

// Solve A p = b to an FP64 relative residual <= tol with MG-preconditioned CG in FP64,
// starting from the current pressure (or zero), and store the result as FP32. The
// residual of an iteration is reported before its V-cycle, so the next iteration is
// queued while the V-cycle runs.
aq_status mgpcg_solve(aq_flip* h, double tol, int max_iters, int check_every, bool from_current,
                      int* iters, double* rel) {
  AQ_TRY(mg_setup(h));
  aq_flip::MgState& M = *h->mg;
  // A completed solve has no report left to write; one that failed may have some queued.
  if (M.running) HIP_TRY(hipStreamSynchronize(h->stream));
  M.running = true;
  M.report->seq = 0;
  float* p = h->gr.p[h->pb];
  mg_start(h->G, M.H, M.V, h->gr.content, h->gr.rhs, from_current ? p : nullptr, tol, max_iters, check_every,
           h->stream);
  AQ_TRY(mg_wait(h, 1));
  int it = 0;
  while (!M.report->stop && it < max_iters) {
    const int next = (int)std::min<long long>(max_iters, ((long long)it / check_every + 1) * check_every);
    for (; it < next; ++it) AQ_TRY(mg_enqueue(h, it & 1));
    AQ_TRY(mg_wait(h, it + 1));
  }
  mg_finish(h->G, M.H, M.V, p, h->stream);
  HIP_TRY(hipGetLastError());
  ++M.solves;
  M.running = false;
  h->air_clean[h->pb] = true;  // AIR cells written 0
  *iters = it;
  *rel = M.report->res;
  return AQ_OK;
}

// Reads back the residual sums the residual kernels left in red_out.
aq_status residual_read(aq_flip* h, double* rel) {
  double o[2];
  HIP_TRY(hipMemcpyAsync(o, h->red_out, sizeof(o), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  *rel = o[1] > 0 ? std::sqrt(o[0]) / std::sqrt(o[1]) : std::sqrt(o[0]);
  return AQ_OK;
}

aq_status residual_now(aq_flip* h, double* rel) {
  launch_residual(h->G, h->gr, h->pb, h->red_partial, h->red_out, h->stream);
  HIP_TRY(hipGetLastError());
  return residual_read(h, rel);
}

// k Jacobi sweeps, then the FP64 residual of the result; with `keep` the iterate before
// them is copied to p_ahead first. Replayed from a captured
// graph (host-launched sweeps cannot keep up with the GPU: about 5.6 against 3.6 us
// per sweep at 128^3); eager while stage timing is on or graphs are switched off.
aq_status enqueue_sweeps(aq_flip* h, int k, bool keep) {
  if (!h->report) {
    AQ_TRY(h->allocT(&h->reports, 1));
    HIP_TRY(hipHostMalloc((void**)&h->report, 2 * sizeof(SweepReport), hipHostMallocMapped));
    h->report[0].seq = h->report[1].seq = 0;
    HIP_TRY(hipHostGetDevicePointer((void**)&h->report_dev, h->report, 0));
  }
  if (keep && !h->p_ahead) AQ_TRY(h->allocT(&h->p_ahead, (size_t)h->G.ncell));
  if (h->reports_lost) {
    HIP_TRY(hipMemcpyAsync(&h->reports_due, h->reports, sizeof(int), hipMemcpyDeviceToHost, h->stream));
    HIP_TRY(hipStreamSynchronize(h->stream));
  }
  h->reports_lost = true;  // until this report is queued
  auto queued = [h] {
    ++h->reports_due;
    h->reports_lost = false;
    return AQ_OK;
  };
  auto enqueue = [&] {
    if (keep) launch_copy_cells(h->G, h->gr.p[h->pb], h->p_ahead, h->stream);
    jacobi_sweeps(h, k);
    launch_residual(h->G, h->gr, h->pb, h->red_partial, h->red_out, h->stream, h->report_dev, h->reports);
  };
  const int key[6] = {h->pb, h->air_clean[0], h->air_clean[1], h->p2g_content, k, keep};
  const bool graphs = !h->timing && h->use_graphs;
  if (graphs) {
    for (auto& g : h->sweep_graphs) {
      if (std::memcmp(g.key, key, sizeof(key)) == 0) {
        HIP_TRY(hipGraphLaunch(g.exec, h->stream));
        h->pb = g.next[0], h->air_clean[0] = g.next[1] != 0, h->air_clean[1] = g.next[2] != 0;
        return queued();
      }
    }
  }
  if (!graphs || h->sweep_graphs.size() >= aq_flip::kMaxSweepGraphs) {  // (unusual chunk lengths)
    enqueue();
    HIP_TRY(hipGetLastError());
    return queued();
  }
  aq_flip::SweepGraph g{};
  std::memcpy(g.key, key, sizeof(key));
  HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  enqueue();
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(h->stream, &graph);
  if (e != hipSuccess) {
    if (graph) hipGraphDestroy(graph);
    (void)hipGetLastError();  // reported here, not by the next call
    h->pb = key[0], h->air_clean[0] = key[1] != 0, h->air_clean[1] = key[2] != 0;  // no sweep has run
    return fail(AQ_EHIP, std::string("sweep capture: ") + hipGetErrorString(e));
  }
  g.graph = graph;
  HIP_TRY(hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0));
  g.next[0] = h->pb, g.next[1] = h->air_clean[0], g.next[2] = h->air_clean[1];
  h->sweep_graphs.push_back(g);
  HIP_TRY(hipGraphLaunch(g.exec, h->stream));
  return queued();
}

// Sweeps in chunks of `every` up to `budget`, each chunk's residual read while the next
// one already runs: a chunk is queued before its predecessor's residual is known when the
// fall of the last two lets expect that this will not end the solve, and undone by finish()
// where it did. 64^3, a check every 50 sweeps: 24.0 -> 20.4 ms for 10,700 sweeps. A solve that
// ends sooner than expected has queued up to kMaxAhead sweeps for nothing, which the entry
// points wait for; longer chunks gain less than they risk and are not queued ahead.
struct ChunkedSweeps {
  aq_flip* h;
  int every, budget;
  double tol, res;             // res: the last known residual
  double before = 0;           // and the one before it (0: none)
  int done = 0, flying = 0;    // sweeps reported; of the chunk queued ahead
  int pb = 0;                  // state before that chunk
  bool clean[2] = {false, false};
  // Up to here: the copy then takes 7 us (8 bytes a cell), and a wait is little next to a chunk.
  static constexpr long long kMaxCells = 1 << 22;
  static constexpr int kMaxAhead = 128;

  aq_status next() {
    const int k = flying ? flying : std::min(every, budget - done);
    if (!flying) AQ_TRY(enqueue_sweeps(h, k, false));
    const int due = h->reports_due;
    flying = std::min(every, budget - done - k);
    if (flying > 0 && flying <= kMaxAhead && before > 0 && res * (res / before) > tol && res < before && !h->timing && h->use_graphs &&
        h->G.ncell <= kMaxCells) {
      pb = h->pb;
      std::copy(h->air_clean, h->air_clean + 2, clean);
      AQ_TRY(enqueue_sweeps(h, flying, true));
    } else {
      flying = 0;
    }
    if (const aq_status st = wait_report(h, &h->report[due & 1].seq, due); st != AQ_OK) {
      h->reports_lost = true;
      return st;
    }
    const SweepReport& r = h->report[due & 1];
    before = res;
    res = r.bb > 0 ? std::sqrt(r.rr) / std::sqrt(r.bb) : std::sqrt(r.rr);
    done += k;
    return AQ_OK;
  }
  aq_status finish() {
    if (!flying) return AQ_OK;
    launch_copy_cells(h->G, h->p_ahead, h->gr.p[pb], h->stream);
    HIP_TRY(hipGetLastError());
    h->pb = pb;
    std::copy(clean, clean + 2, h->air_clean);
    flying = 0;
    return AQ_OK;
  }
};

// Jacobi sweeps from the current pressure until the FP64 relative residual is
// <= tol (checked every check_every sweeps) or `budget` sweeps are spent. With
// detect_stall, `stall_checks` consecutive checks without a 1% improvement over
// the best residual (or a non-finite residual) end the solve as stalled.
aq_status sweep_to_tol(aq_flip* h, int budget, bool detect_stall, int* sweeps, double* res,
                       bool* stalled) {
  const aq_flip_solver& S = h->solver;
  *sweeps = 0;
  *stalled = false;
  AQ_TRY(residual_now(h, res));
  ChunkedSweeps C{h, S.check_every, budget, S.tol, *res};
  double best = *res;
  int flat = 0;
  while (!(C.res <= S.tol) && C.done < budget) {
    if (!std::isfinite(C.res)) {
      *stalled = true;
      break;
    }
    AQ_TRY(C.next());
    if (detect_stall) {
      if (std::isfinite(C.res) && C.res < 0.99 * best) {
        best = C.res;
        flat = 0;
      } else if (++flat >= S.stall_checks || !std::isfinite(C.res)) {
        *stalled = true;
        break;
      }
    }
  }
  AQ_TRY(C.finish());
  *sweeps = C.done;
  *res = C.res;
  return AQ_OK;
}

// Refinement of a U-Net guess already in the pressure buffer: Jacobi to the solver's
// tol within `budget` sweeps, the network correcting the iterate from its residual
// every nn_refresh sweeps (0: never). While the residual at the end of each chunk of
// sweeps keeps falling by at least 1 % from the previous chunk's, every correction is
// kept: the network removes smooth error that Jacobi is slow on while adding
// high-frequency residual that the following sweeps remove, so the residual right after
// a correction, or even one chunk later on a large grid, says little. Once a chunk
// ends within 1 % of the previous one (Jacobi near its FP32 round-off floor, where the
// network's output is mostly noise), the next correction is judged by the residual
// after the sweeps that follow it: if that is not below the residual before the
// correction, the iterate from before it is restored bit for bit and Jacobi continues
// without further corrections.
aq_status nn_refine(aq_flip* h, aq_unet* net, int budget, int nn_refresh, int* total, double* res,
                    bool* stalled, bool* fallback, int64_t* corrections, int64_t* rejected) {
  const size_t bytes = (size_t)h->G.ncell * sizeof(float);
  int left = budget, sweeps = 0;
  bool correcting = nn_refresh > 0;
  bool judging = false;  // the last chunk followed a correction that is being judged
  double before = 0;     // residual of the iterate saved in p_keep
  double last = 0;       // residual at the end of the previous chunk
  bool have_last = false;
  int pb_keep = 0;
  bool clean_keep = false;
  *total = 0;
  for (;;) {
    const int chunk = correcting ? std::min(nn_refresh, left) : left;
    AQ_TRY(sweep_to_tol(h, chunk, true, &sweeps, res, stalled));
    *total += sweeps;
    left -= sweeps;
    const bool flat = have_last && !(*res < 0.99 * last);
    last = *res;
    have_last = true;
    if (judging) {
      judging = false;
      if (!(*res <= h->solver.tol) && !(*res < before)) {
        // restore the iterate from before the correction
        HIP_TRY(hipMemcpyAsync(h->gr.p[pb_keep], h->p_keep, bytes, hipMemcpyDeviceToDevice, h->stream));
        h->pb = pb_keep;
        h->air_clean[pb_keep] = clean_keep;
        *res = before;
        *stalled = false;
        *rejected += 1;
        correcting = false;
        if (left > 0) continue;
      }
    }
    if (!std::isfinite(*res)) *fallback = true;
    if (*fallback || *res <= h->solver.tol || left <= 0 || *stalled || !correcting) break;
    if (flat) {  // keep a copy of the iterate: this correction will be judged
      if (!h->p_keep) AQ_TRY(h->allocT(&h->p_keep, (size_t)h->G.ncell));
      pb_keep = h->pb;
      clean_keep = h->air_clean[h->pb];
      HIP_TRY(hipMemcpyAsync(h->p_keep, h->gr.p[h->pb], bytes, hipMemcpyDeviceToDevice, h->stream));
    }
    before = *res;
    AQ_TRY(aq_flip_nn_correct(h, net));
    *corrections += 1;
    judging = flat;
  }
  return AQ_OK;
}

// The pressure solve of one step, per the selected mode.
aq_status pressure_stage(aq_flip* h) {
  aq_flip_solver_stats& st = h->sstats;
  if (h->solver.mode == AQ_SOLVE_FIXED) {
    h->begin(AQ_STAGE_PRESSURE);  // the Jacobi sweeps
    fixed_sweeps(h);
    h->end(AQ_STAGE_PRESSURE, h->cfg.pressure_iters);
    return AQ_OK;
  }
  h->begin(AQ_STAGE_PRESSURE);
  int sweeps = 0, total = 0;
  double res = 0, guess = 1.0;
  bool stalled = false, fallback = false;
  bool mg_converged = false;  // MGPCG: the CG residual reached tol
  if (h->solver.mode == AQ_SOLVE_TOL_NN) {
    if (!h->net) return fail(AQ_EINVAL, "AQ_SOLVE_TOL_NN needs a U-Net");
    AQ_TRY(aq_flip_nn_guess(h, h->net));
    h->air_clean[h->pb] = true;  // the guess is 0 on AIR cells
    AQ_TRY(residual_now(h, &guess));
    // Jacobi converges to the same fixed point from any finite start, so only a
    // non-finite guess or refinement is rejected for the zero-guess solve. A finite
    // guess that stalls has reached FP32 Jacobi's round-off floor, where a solve from
    // zero would stall as well.
    if (!std::isfinite(guess)) fallback = true;
    // Refine with Jacobi; every nn_refresh sweeps (if set) the network corrects the
    // iterate from its residual, then Jacobi continues.
    if (!fallback)
      AQ_TRY(nn_refine(h, h->net, h->solver.max_iters, h->solver.nn_refresh, &total, &res, &stalled,
                       &fallback, &st.nn_corrections, &st.nn_rejected));
  }
  if (h->solver.mode == AQ_SOLVE_MGPCG) {
    const bool from_current = h->cfg.pressure_init == AQ_PRESSURE_PREVIOUS;
    int it = 0;
    double cg = 0;
    AQ_TRY(mgpcg_solve(h, h->solver.tol, h->solver.max_iters, h->solver.check_every, from_current, &it, &cg));
    AQ_TRY(residual_now(h, &res));  // of the stored FP32 field (reported)
    mg_converged = cg <= h->solver.tol;
    total = it;
    guess = 1.0;
  }
  if (h->solver.mode == AQ_SOLVE_TOL_ZERO || fallback) {
    zero_pressure(h);
    AQ_TRY(sweep_to_tol(h, std::max(0, h->solver.max_iters), true, &sweeps, &res, &stalled));
    total += sweeps;
    if (h->solver.mode == AQ_SOLVE_TOL_ZERO) guess = 1.0;
  }
  h->end(AQ_STAGE_PRESSURE, total);
  st.solves += 1;
  st.sweeps += total;
  st.fallbacks += fallback ? 1 : 0;
  const bool reached = h->solver.mode == AQ_SOLVE_MGPCG ? mg_converged : res <= h->solver.tol;
  st.capped += reached ? 0 : 1;
  st.last_sweeps = total;
  st.last_residual = res;
  st.last_guess_residual = guess;
  st.last_fallback = fallback ? 1 : 0;
  return AQ_OK;
}

// Fluid::simulationStep (Fluid/Fluid_3D_FLIP.cu:316-352). G2P, advection, hashing
// and bin counting are one particle pass; gravity and boundary one face pass.
// The bin counts are zero on entry: allocated so, and every scan sets them back to zero.
aq_status enqueue_step(aq_flip* h) {
  h->begin(AQ_STAGE_G2P);
  launch_g2p_advect_hash(h->G, h->P[h->cur], h->Np, h->K, h->gr, h->nv, h->nf, h->sp, h->B, h->stream);
  h->end(AQ_STAGE_G2P);
  h->begin(AQ_STAGE_TRANSFER_TO_GRID);
  transfer_after_count(h, true);  // ends the bucket before P2G, which is timed as AQ_STAGE_P2G
  h->begin(AQ_STAGE_GRAVITY);
  launch_gravity_boundary(h->G, h->gr, h->nv, h->sp, 1, 1, h->stream);
  h->end(AQ_STAGE_GRAVITY);
  h->begin(AQ_STAGE_DIVERGENCE);
  launch_divergence(h->G, h->gr, h->nv, h->B, h->stream);
  h->end(AQ_STAGE_DIVERGENCE);
  // Diffusion reads the fractions, content and active-block flags, all final after
  // the divergence pass, and writes only the fractions, which nothing before the
  // next step's G2P reads. (Stage timing keeps the reference's sequential order.)
  const bool fused = h->fuse && h->solver.mode == AQ_SOLVE_FIXED &&
                     h->cfg.diffusion_iters > 0 && h->K > 1 && h->cfg.pressure_iters > 0;
  const bool side = !fused && h->overlap && !h->timing && h->cfg.diffusion_iters > 0 && h->K > 1;
  if (side) {
    HIP_TRY(hipEventRecord(h->ev_fork, h->stream));
    HIP_TRY(hipStreamWaitEvent(h->side, h->ev_fork, 0));
    diffusion_sweeps(h, h->side);
    HIP_TRY(hipEventRecord(h->ev_join, h->side));
  }
  if (fused) {
    fused_pressure_diffusion(h);
  } else if (const aq_status ps = pressure_stage(h); ps != AQ_OK) {
    if (side) hipStreamWaitEvent(h->stream, h->ev_join, 0);  // never leave the fork open
    return ps;
  }
  h->begin(AQ_STAGE_PROJECT);
  launch_project(h->G, h->gr, h->nv, h->hv, h->pb, h->stream);
  h->end(AQ_STAGE_PROJECT);
  h->begin(AQ_STAGE_EXTRAPOLATE);
  stage_extrapolate(h, true);
  h->end(AQ_STAGE_EXTRAPOLATE, 3);
  if (side) {
    if (h->cfg.pressure_iters == 0) launch_air_pressure_zero(h->G, h->gr, h->pb, h->stream);
    HIP_TRY(hipStreamWaitEvent(h->stream, h->ev_join, 0));
  } else if (!fused) {
    h->begin(AQ_STAGE_DIFFUSION);
    h->end(AQ_STAGE_DIFFUSION, stage_diffusion(h, true));
  }
  HIP_TRY(hipGetLastError());
  h->physicalTime += h->cfg.dt;
  return AQ_OK;
}

void drop_graphs(aq_flip* h) {
  hipStreamSynchronize(h->stream);
  for (auto& g : h->graphs) {
    hipGraphExecDestroy(g.exec);
    hipGraphDestroy(g.graph);
  }
  h->graphs.clear();
}

// FLUID cells to expect: those that hold particles now, or what the particles fill at the
// seeding density of 8 per cell if that is more. Captured launches that the choice of kernels
// would no longer make are dropped. (27^3 cells with one particle in each, 100 sweeps a step:
// 340 us with a sweep per launch, 550 in one launch as 8 per cell let expect, now 166.)
void expect_fluid(aq_flip* h, long long cells) {
  const auto routes = [h] {
    return (small_cells(h, 1) ? 1 : 0) | (small_cells(h, h->K) ? 2 : 0) | (tile_pairs(h->G, h->K, h->fluid) ? 4 : 0);
  };
  const int before = routes();
  h->fluid = std::min((long long)h->G.ncells_hash, std::max(cells, (h->Np + 7) / 8));
  if (routes() == before) return;
  drop_graphs(h);
  for (auto& g : h->sweep_graphs) {
    hipGraphExecDestroy(g.exec);
    hipGraphDestroy(g.graph);
  }
  h->sweep_graphs.clear();
}

void state_of(const aq_flip* h, int k[7]) {
  k[0] = h->cur, k[1] = h->nv, k[2] = h->hv, k[3] = h->pb, k[4] = h->nf;
  k[5] = h->air_clean[0], k[6] = h->air_clean[1];
}
void set_state(aq_flip* h, const int k[7]) {
  h->cur = k[0], h->nv = k[1], h->hv = k[2], h->pb = k[3], h->nf = k[4];
  h->air_clean[0] = k[5] != 0, h->air_clean[1] = k[6] != 0;
}

// One step through a captured graph (eager launches when timing is on, so the
// stage events sit on the stream between kernels).
// A step's G2P reads new and old velocity from gr.nvo, which the previous step's last
// extrapolation pass wrote on every row a particle's first sample can touch (the rows
// within 4 of a cell row holding FLUID; a particle's corners lie within one row of its
// FLUID cell). Anything else that changes the velocities, or a fresh handle, leaves it
// stale, and the copy is then rebuilt in full first.
aq_status graph_step(aq_flip* h) {
  if (!h->nvo_valid) {
    launch_build_nvo(h->G, h->gr, h->nv, h->stream);
    h->nvo_valid = true;
  }
  if (h->timing || !h->use_graphs || h->solver.mode != AQ_SOLVE_FIXED) return enqueue_step(h);
  int key[7];
  state_of(h, key);
  for (auto& g : h->graphs) {
    if (std::memcmp(g.key, key, sizeof(key)) == 0) {
      HIP_TRY(hipGraphLaunch(g.exec, h->stream));
      set_state(h, g.next);
      h->p2g_content = true;
      h->physicalTime += h->cfg.dt;
      return AQ_OK;
    }
  }
  aq_flip::StepGraph g{};
  std::memcpy(g.key, key, sizeof(key));
  HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  aq_status st = enqueue_step(h);
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(h->stream, &graph);
  if (st != AQ_OK) {
    if (graph) hipGraphDestroy(graph);
    return st;
  }
  if (e != hipSuccess) return fail(AQ_EHIP, std::string("step capture: ") + hipGetErrorString(e));
  g.graph = graph;
  HIP_TRY(hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0));
  state_of(h, g.next);
  h->graphs.push_back(g);
  HIP_TRY(hipGraphLaunch(g.exec, h->stream));
  return AQ_OK;
}

// ---- particle seeding on the GPU ------------------------------------------
// The volumes of a scene as the GPU seeder walks them, with per-block output
// offsets from a counting pass (seed_kernels.hip); identical to seed_scene's output.
struct SeedPlan {
  SeedParams sp{};
  std::vector<SeedVolume> vols;
  std::vector<long long> nc;                // candidates per volume (cells x 8)
  std::vector<std::vector<int>> offsets;    // per volume: exclusive prefix of block counts
  std::vector<long long> first;             // per volume: index of its first particle
  long long total = 0;
};

bool in_unit_cube(const float c[3]) {
  for (int a = 0; a < 3; ++a)
    if (c[a] < 0 || c[a] > 1) return false;
  return true;
}

aq_status plan_seeding(const aq_flip_config& cfg, SeedPlan* plan) {
  const int S[3] = {cfg.size[0], cfg.size[1], cfg.size[2]};
  const float h = cfg.grid_physical_size / (float)cfg.size[1];
  plan->sp.seed = cfg.seed;
  plan->sp.h = h;
  plan->sp.jitter = cfg.particle_jitter;
  for (int a = 0; a < 3; ++a) plan->sp.S[a] = S[a];
  uint64_t draws = 0;
  for (int i = 0; i < cfg.n_volumes; ++i) {
    const aq_flip_volume& v = cfg.volumes[i];
    SeedVolume sv{};
    sv.phase = v.phase;
    if (v.shape == AQ_SHAPE_BOX) {
      if (!in_unit_cube(v.box_min) || !in_unit_cube(v.box_max)) continue;
      // createSquareFluid's loops: z, then x, then y, each from (int)(min*S) while (float)i < max*S
      const int order[3] = {2, 0, 1};
      for (int j = 0; j < 3; ++j) {
        const int a = order[j];
        const int lo = (int)(v.box_min[a] * (float)S[a]);
        int cnt = 0;
        for (int c = lo; (float)c < v.box_max[a] * (float)S[a]; ++c) ++cnt;
        sv.n[j] = cnt;
        sv.o[j] = lo;
        sv.axis[j] = a;
      }
    } else if (v.shape == AQ_SHAPE_SPHERE) {
      if (!in_unit_cube(v.center)) continue;
      // createSphereFluid visits every cell: y, then x, then z
      const int order[3] = {1, 0, 2};
      for (int j = 0; j < 3; ++j) {
        sv.n[j] = S[order[j]];
        sv.o[j] = 0;
        sv.axis[j] = order[j];
      }
      sv.sphere = 1;
      for (int a = 0; a < 3; ++a) sv.cc[a] = (v.center[a] * (float)S[a]) * h;
      sv.limit = (v.radius * h) * (float)S[1];
    } else {
      continue;
    }
    sv.base = draws;
    const long long cells = (long long)std::max(sv.n[0], 0) * std::max(sv.n[1], 0) * std::max(sv.n[2], 0);
    draws += (uint64_t)cells * 24u;
    if (cells == 0) continue;
    plan->vols.push_back(sv);
    plan->nc.push_back(cells * 8);
  }
  if (plan->vols.empty()) return AQ_OK;  // nothing to seed (no device work)
  // counting pass
  hipStream_t s = nullptr;
  HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  const int B = seed_block_size();
  long long maxb = 1;
  for (long long nc : plan->nc) maxb = std::max(maxb, (nc + B - 1) / B);
  int* d_counts = nullptr;
  hipError_t e = device_malloc((void**)&d_counts, (size_t)maxb * sizeof(int));
  for (size_t i = 0; i < plan->vols.size() && e == hipSuccess; ++i) {
    const long long nb = (plan->nc[i] + B - 1) / B;
    launch_seed_count(plan->vols[i], plan->sp, plan->nc[i], d_counts, s);
    std::vector<int> counts((size_t)nb);
    e = hipMemcpyAsync(counts.data(), d_counts, (size_t)nb * sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    std::vector<int> off((size_t)nb);
    long long run = 0;
    for (long long b = 0; b < nb; ++b) {
      off[(size_t)b] = (int)run;
      run += counts[(size_t)b];
    }
    plan->first.push_back(plan->total);
    plan->total += run;
    plan->offsets.push_back(std::move(off));
  }
  if (d_counts) hipFree(d_counts);
  hipStreamDestroy(s);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(AQ_EHIP, std::string("seeding: ") + hipGetErrorString(e));
  }
  if (plan->total > (1ll << 31) - 1) return fail(AQ_EINVAL, "too many particles");
  return AQ_OK;
}

// Write the planned particles into the handle's current particle buffer.
aq_status write_seeded(aq_flip* h, const SeedPlan& plan) {
  long long maxb = 1;
  for (const auto& o : plan.offsets) maxb = std::max<long long>(maxb, (long long)o.size());
  int* d_off = nullptr;
  HIP_TRY(device_malloc((void**)&d_off, (size_t)maxb * sizeof(int)));
  hipError_t e = hipSuccess;
  for (size_t i = 0; i < plan.vols.size() && e == hipSuccess; ++i) {
    e = hipMemcpyAsync(d_off, plan.offsets[i].data(), plan.offsets[i].size() * sizeof(int),
                       hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) {
      launch_seed_write(plan.vols[i], plan.sp, plan.nc[i], d_off, plan.first[i], h->P[h->cur], h->stream);
      e = hipStreamSynchronize(h->stream);  // d_off is reused by the next volume
    }
  }
  hipFree(d_off);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(AQ_EHIP, std::string("seeding: ") + hipGetErrorString(e));
  }
  return AQ_OK;
}

// Switches for measurements: AQFLIP_NO_GRAPH=1 (eager launches), AQFLIP_NO_OVERLAP=1
// (diffusion after the pressure solve on one stream), AQFLIP_NO_FUSE=1 (no fused
// pressure + diffusion sweeps), AQFLIP_NO_FIXED_POINT_SKIP=1 (paired diffusion sweeps
// always computed). Results are identical in every combination.
void read_env(aq_flip* h) {
  if (const char* env = std::getenv("AQFLIP_NO_GRAPH")) h->use_graphs = env[0] == '0';
  if (const char* env = std::getenv("AQFLIP_NO_OVERLAP")) h->overlap = env[0] != '1';
  if (const char* env = std::getenv("AQFLIP_NO_FUSE")) h->fuse = env[0] != '1';
  if (const char* env = std::getenv("AQFLIP_NO_FIXED_POINT_SKIP")) h->skip_fixed = env[0] != '1';
  if (const char* env = std::getenv("AQFLIP_LISTED_GRID")) h->listed_grid = std::max(0, std::atoi(env));
}

aq_status create_common(const aq_flip_config* cfg, const float* pos, const float* vel,
                        const float* frac4, long long n, aq_flip** out, const SeedPlan* plan = nullptr) {
  aq_flip* h = new aq_flip;
  read_env(h);
  aq_status st = setup(h, cfg, n);
  if (plan) {  // seeded on the device: positions are clamped into the domain by construction
    h->K = channels_for(*cfg, nullptr, 0);
    if (st == AQ_OK) expect_fluid(h, 0);
    if (st == AQ_OK) st = write_seeded(h, *plan);
  } else {
    long long cells = 0;
    if (st == AQ_OK) st = check_positions(h, pos, n, &cells);
    if (st == AQ_OK) {
      h->K = channels_for(*cfg, frac4, n);
      expect_fluid(h, cells);
      st = upload_particles(h, pos, vel, frac4);
    }
  }
  if (st == AQ_OK) {
    // Fluid::init: fixBoundary, then transferToGrid (Fluid_3D_FLIP.cu:485,500).
    launch_gravity_boundary(h->G, h->gr, h->nv, h->sp, 0, 1, h->stream);
    stage_transfer(h);
    refresh_rhs(h);
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess) st = fail(AQ_EHIP, std::string("init: ") + hipGetErrorString(e));
  }
  if (st != AQ_OK) {
    delete h;
    return st;
  }
  *out = h;
  return AQ_OK;
}

size_t field_elems(const aq_flip* h, int field, int* width, bool* isInt) {
  const Geom& G = h->G;
  const size_t e1 = (size_t)(G.X + 1) * (G.Y + 1) * (G.Z + 1), e0 = (size_t)G.X * G.Y * G.Z;
  *isInt = false;
  switch (field) {
    case AQ_FIELD_CONTENT: *width = 1; *isInt = true; return e1;
    case AQ_FIELD_VELOCITY:
    case AQ_FIELD_NEW_VELOCITY: *width = 4; return e1;
    case AQ_FIELD_PRESSURE:
    case AQ_FIELD_DIVERGENCE:
    case AQ_FIELD_DENSITY: *width = 1; return e0;
    case AQ_FIELD_PARTICLE_COUNT: *width = 1; *isInt = true; return e0;
    case AQ_FIELD_HAS_VELOCITY: *width = 4; *isInt = true; return e0;
    case AQ_FIELD_VOLUME_FRACTIONS:
    case AQ_FIELD_NEW_VOLUME_FRACTIONS: *width = 4; return e0;
  }
  *width = 0;
  return 0;
}

template <typename T>
aq_status d2h(aq_flip* h, std::vector<T>& dst, const void* src, size_t n) {
  dst.resize(n);
  HIP_TRY(hipMemcpyAsync(dst.data(), src, n * sizeof(T), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return AQ_OK;
}
template <typename T>
aq_status h2d(aq_flip* h, void* dst, const std::vector<T>& src) {
  HIP_TRY(hipMemcpyAsync(dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return AQ_OK;
}

// Small exports: copied as stored and rearranged here, without a launch before the copy. Us,
// here / on the GPU: a pressure of 16^3 11 / 25, 33^3 20 / 29, 50^3 45 / 46, content of 33^3
// 25 / 30, 40^3 38 / 35; 1,162 particles 24 / 54, 3,922 32 / 62 (one phase 77 / 122), 18,137
// 193 / 86. Fields of several arrays, a copy each, are quicker on the GPU at every size.
constexpr size_t kHostElements = 40000;
constexpr long long kHostParticles = 4096;
aq_status field_on_host(aq_flip* h, const ExportField& f, size_t n, uint32_t* out) {
  const Geom& G = h->G;
  const bool bytes = f.kind == ExportField::kByte || f.kind == ExportField::kBits;
  std::vector<uint8_t> raw;
  AQ_TRY(d2h(h, raw, f.src[0], f.kind == ExportField::kCount ? (n + 1) * 4 : (size_t)G.ncell * (bytes ? 1 : 4)));
  const uint32_t* words = (const uint32_t*)raw.data();
  if (f.kind == ExportField::kCount) {  // cellEnd - cellStart (Fluid/Fluid_3D_FLIP.cu:180)
    for (size_t o = 0; o < n; ++o) out[o] = words[o + 1] - words[o] - (words[o + 1] > words[o]);
    return AQ_OK;
  }
  const int X = G.X + f.face, Y = G.Y + f.face, Z = G.Z + f.face;
  for (int x = 0; x < X; ++x)
    for (int y = 0; y < Y; ++y) {
      const uint8_t* r = raw.data() + G.g(x, y, 0);
      const uint32_t* w = words + (bytes ? 0 : G.g(x, y, 0));
      uint32_t* o = out + ((size_t)x * Y + y) * Z * (f.kind == ExportField::kVector || f.kind == ExportField::kBits ? 4 : 1);
      switch (f.kind) {
        case ExportField::kScalar: std::memcpy(o, w, (size_t)Z * 4); break;
        case ExportField::kByte:
          for (int z = 0; z < Z; ++z) o[z] = r[z];
          break;
        case ExportField::kBits:
          for (int z = 0; z < Z; ++z, o += 4) o[0] = r[z] & 1, o[1] = r[z] >> 1 & 1, o[2] = r[z] >> 2 & 1, o[3] = 0;
          break;
        default:  // kVector, one array
          for (int z = 0; z < Z; ++z, o += 4) o[0] = w[z], o[1] = o[2] = o[3] = 0;
      }
    }
  return AQ_OK;
}
aq_status particles_on_host(aq_flip* h, float* pos, float* vel, float* frac4) {
  const size_t n = (size_t)h->Np;
  const Particles& P = h->P[h->cur];
  std::vector<float4> a, b, c;
  AQ_TRY(d2h(h, a, P.a, n));
  AQ_TRY(d2h(h, b, P.b, n));
  if (frac4 && h->K > 2) AQ_TRY(d2h(h, c, P.c, n));
  for (size_t i = 0; i < n; ++i) {
    if (pos) pos[3 * i] = a[i].x, pos[3 * i + 1] = a[i].y, pos[3 * i + 2] = a[i].z;
    if (vel) vel[3 * i] = a[i].w, vel[3 * i + 1] = b[i].x, vel[3 * i + 2] = b[i].y;
    if (!frac4) continue;
    frac4[4 * i] = b[i].z;
    frac4[4 * i + 1] = h->K > 1 ? b[i].w : 0.f;
    frac4[4 * i + 2] = h->K > 2 ? c[i].x : 0.f;
    frac4[4 * i + 3] = h->K > 3 ? c[i].y : 0.f;
  }
  return AQ_OK;
}

}  // namespace

namespace aqf {
hipError_t device_malloc(void** p, size_t bytes) {
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory || !block_cache().release()) return e;
  (void)hipGetLastError();
  return hipMalloc(p, bytes);
}
FlipView flip_view(aq_flip* h) { return FlipView{h->G, &h->gr, &h->pb, h->stream}; }
void set_last_error(const std::string& msg) { g_err = msg; }
}  // namespace aqf

extern "C" {

aq_status aq_flip_set_solver(aq_flip* h, const aq_flip_solver* s, aq_unet* net) {
  if (!h || !s) return fail(AQ_EINVAL, "null argument");
  if (s->mode < AQ_SOLVE_FIXED || s->mode > AQ_SOLVE_MGPCG) return fail(AQ_EINVAL, "unknown solver mode");
  if (s->mode != AQ_SOLVE_FIXED && (!(s->tol > 0) || s->max_iters < 0 || s->check_every < 1 ||
                                    s->stall_checks < 1 || s->nn_refresh < 0))
    return fail(AQ_EINVAL, "tolerance solves need tol > 0, max_iters >= 0, check_every >= 1, "
                           "stall_checks >= 1, nn_refresh >= 0");
  if (s->mode == AQ_SOLVE_TOL_NN && !net) return fail(AQ_EINVAL, "AQ_SOLVE_TOL_NN needs a U-Net");
  if (s->mode == AQ_SOLVE_TOL_NN && (h->G.X % 4 || h->G.Y % 4 || h->G.Z % 4))
    return fail(AQ_EINVAL, "the U-Net needs grid extents that are multiples of 4");
  h->solver = *s;
  h->net = net;
  return AQ_OK;
}

aq_status aq_flip_solve_pressure_nn(aq_flip* h, aq_unet* net, double tol, int32_t max_iters,
                                    int32_t check_every, int32_t nn_refresh, int32_t* iters_out,
                                    double* rel_out, int32_t* corrections_out, int32_t* rejected_out) {
  if (!h || !net || max_iters < 0 || check_every < 1 || nn_refresh < 0) return fail(AQ_EINVAL, "bad argument");
  const aq_flip_solver keep = h->solver;
  h->solver.tol = tol;
  h->solver.check_every = check_every;
  int total = 0;
  double res = 0;
  bool stalled = false, fallback = false;
  int64_t corr = 0, rej = 0;
  aq_status st = aq_flip_nn_guess(h, net);
  if (st == AQ_OK) {
    h->air_clean[h->pb] = true;  // the guess is 0 on AIR cells
    st = nn_refine(h, net, max_iters, nn_refresh, &total, &res, &stalled, &fallback, &corr, &rej);
  }
  h->solver = keep;
  if (st != AQ_OK) return st;
  HIP_TRY(hipStreamSynchronize(h->stream));  // a chunk queued ahead may still be running
  if (iters_out) *iters_out = total;
  if (rel_out) *rel_out = res;
  if (corrections_out) *corrections_out = (int32_t)corr;
  if (rejected_out) *rejected_out = (int32_t)rej;
  if (!(res <= tol)) return fail(AQ_ESTALL, fallback ? "U-Net refinement is not finite" : "pressure solve did not reach tol");
  return AQ_OK;
}

aq_status aq_flip_solver_stats_get(aq_flip* h, aq_flip_solver_stats* out, int32_t reset) {
  if (!h || !out) return fail(AQ_EINVAL, "null argument");
  *out = h->sstats;
  if (reset) h->sstats = aq_flip_solver_stats{};
  return AQ_OK;
}

aq_status aq_flip_config_default(aq_flip_config* c) {
  if (!c) return fail(AQ_EINVAL, "null config");
  std::memset(c, 0, sizeof(*c));
  // ConfigFLIP (Fluid/FluidConfig.cuh:41-50)
  c->size[0] = c->size[1] = c->size[2] = 50;
  c->pressure_iters = 100;
  c->diffusion_iters = 100;
  c->dt = 0.033f;
  c->flip_coeff = 0.95f;
  c->particle_jitter = 0.05f;
  c->grid_physical_size = 10.f;  // Fluid_3D_FLIP.cuh:62
  // FluidConfig (Fluid/FluidConfig.cuh:68-97)
  c->gravity[0] = 0.f;
  c->gravity[1] = -9.8f;
  c->gravity[2] = 0.f;
  c->phase_count = 2;
  for (int a = 0; a < 4; ++a) c->phase_densities[a] = 1.f;
  c->diffusion_coeff = 0.001f;
  c->pressure_init = AQ_PRESSURE_PREVIOUS;
  c->ref_boundary_coverage = 1;
  c->seed = 0;
  // Default scene: a pool and a ball (InitializationVolume, FluidConfig.cuh:20-39).
  c->n_volumes = 2;
  aq_flip_volume& box = c->volumes[0];
  box.shape = AQ_SHAPE_BOX;
  box.box_min[0] = box.box_min[1] = box.box_min[2] = 0.f;
  box.box_max[0] = 1.f;
  box.box_max[1] = 0.1875f;
  box.box_max[2] = 1.f;
  box.center[0] = 0.5f;
  box.center[1] = 0.75f;
  box.center[2] = 0.5f;
  box.radius = 0.125f;
  box.phase = 0;
  c->volumes[1] = box;
  c->volumes[1].shape = AQ_SHAPE_SPHERE;
  return AQ_OK;
}

aq_status aq_flip_seed_particles(const aq_flip_config* cfg, float* pos, float* frac4,
                                 int64_t capacity, int64_t* n_out) {
  AQ_TRY(validate(cfg));
  if (!n_out) return fail(AQ_EINVAL, "null n_out");
  if (!pos) {
    *n_out = seed_scene(*cfg, nullptr, nullptr);
    return AQ_OK;
  }
  std::vector<float> p, f;
  const int64_t n = seed_scene(*cfg, &p, &f);
  *n_out = n;
  if (capacity < n) return fail(AQ_EINVAL, "capacity smaller than the particle count");
  std::memcpy(pos, p.data(), p.size() * sizeof(float));
  if (frac4) std::memcpy(frac4, f.data(), f.size() * sizeof(float));
  return AQ_OK;
}

aq_status aq_flip_create(const aq_flip_config* cfg, aq_flip** out) {
  AQ_TRY(validate(cfg));
  if (!out) return fail(AQ_EINVAL, "null out");
  SeedPlan plan;
  AQ_TRY(plan_seeding(*cfg, &plan));
  if (plan.total <= 0) return fail(AQ_EINVAL, "the configured volumes produce no particles");
  return create_common(cfg, nullptr, nullptr, nullptr, plan.total, out, &plan);
}

aq_status aq_flip_create_with_particles(const aq_flip_config* cfg, const float* pos,
                                        const float* vel, const float* frac4, int64_t n,
                                        aq_flip** out) {
  AQ_TRY(validate(cfg));
  if (!out || !pos) return fail(AQ_EINVAL, "null argument");
  if (n <= 0 || n > (1ll << 31) - 1) return fail(AQ_EINVAL, "particle count out of range");
  return create_common(cfg, pos, vel, frac4, n, out);
}

void aq_flip_destroy(aq_flip* h) { delete h; }

void aq_flip_release_memory(void) { block_cache().release(); }

aq_status aq_flip_step(aq_flip* h) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  AQ_TRY(graph_step(h));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return h->collect();
}

aq_status aq_flip_steps(aq_flip* h, int32_t count) {
  if (!h || count < 0) return fail(AQ_EINVAL, "bad argument");
  for (int i = 0; i < count; ++i) AQ_TRY(graph_step(h));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return h->collect();
}

aq_status aq_flip_run_stage(aq_flip* h, int32_t stage) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  if (stage < 0 || stage >= AQ_STAGE_COUNT) return fail(AQ_EINVAL, "unknown stage");
  AQ_TRY(run_stage(h, stage));
  HIP_TRY(hipStreamSynchronize(h->stream));
  return h->collect();
}

int64_t aq_flip_particle_count(const aq_flip* h) { return h ? h->Np : 0; }

// Arrays a and b of the particle buffer that a step overwrites next serve as scratch between
// steps, 16 bytes per particle each. (c does not: with up to two phases no step writes it, and
// the fractions in it have to stay 0.) Fractions follow in a launch of their own, in order
// behind the copies that read the scratch.
aq_status aq_flip_get_particles(aq_flip* h, float* pos, float* vel, float* frac4) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  const size_t n = (size_t)h->Np;
  const Particles &P = h->P[h->cur], &S = h->P[h->cur ^ 1];
  if (h->Np <= kHostParticles) return particles_on_host(h, pos, vel, frac4);
  if (pos || vel) {
    launch_export_particles(P, h->Np, h->K, pos ? (float*)S.a : nullptr, vel ? (float*)S.b : nullptr, nullptr,
                            h->stream);
    HIP_TRY(hipGetLastError());
    if (pos) HIP_TRY(hipMemcpyAsync(pos, S.a, n * 3 * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    if (vel) HIP_TRY(hipMemcpyAsync(vel, S.b, n * 3 * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  }
  if (frac4) {
    launch_export_particles(P, h->Np, h->K, nullptr, nullptr, S.a, h->stream);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(frac4, S.a, n * 4 * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return AQ_OK;
}

aq_status aq_flip_set_particles(aq_flip* h, const float* pos, const float* vel, const float* frac4,
                                int64_t n) {
  if (!h || !pos) return fail(AQ_EINVAL, "null argument");
  if (n != h->Np) return fail(AQ_EINVAL, "particle count differs from the handle's");
  long long cells = 0;
  AQ_TRY(check_positions(h, pos, n, &cells));
  const int K = std::max(h->K, channels_for(h->cfg, frac4, n));
  if (K != h->K) drop_graphs(h);
  h->K = K;
  expect_fluid(h, cells);
  return upload_particles(h, pos, vel, frac4);
}

size_t aq_flip_field_bytes(const aq_flip* h, int32_t field) {
  if (!h) return 0;
  int w;
  bool isInt;
  const size_t n = field_elems(h, field, &w, &isInt);
  return n * (size_t)w * 4;
}

aq_status aq_flip_get_field(aq_flip* h, int32_t field, void* dst, size_t bytes) {
  if (!h || !dst) return fail(AQ_EINVAL, "null argument");
  int w;
  bool isInt;
  const size_t n = field_elems(h, field, &w, &isInt);
  if (n == 0) return fail(AQ_EINVAL, "unknown field");
  if (bytes != n * w * 4) return fail(AQ_EINVAL, "byte count does not match the field");
  const Grid& gr = h->gr;
  ExportField f{ExportField::kScalar, false, {}};
  switch (field) {
    case AQ_FIELD_CONTENT: f = {ExportField::kByte, true, {gr.content}}; break;
    case AQ_FIELD_VELOCITY: f = {ExportField::kVector, true, {gr.vel[0], gr.vel[1], gr.vel[2]}}; break;
    case AQ_FIELD_NEW_VELOCITY:
      f = {ExportField::kVector, true, {gr.nvel[h->nv][0], gr.nvel[h->nv][1], gr.nvel[h->nv][2]}};
      break;
    case AQ_FIELD_PRESSURE: f.src[0] = gr.p[h->pb]; break;
    case AQ_FIELD_DIVERGENCE: f.src[0] = gr.div; break;
    case AQ_FIELD_DENSITY: f.src[0] = gr.density; break;
    case AQ_FIELD_PARTICLE_COUNT: f = {ExportField::kCount, false, {h->B.offsets}}; break;
    case AQ_FIELD_HAS_VELOCITY: f = {ExportField::kBits, false, {gr.hasvel[h->hv]}}; break;
    default:  // the volume fractions
      f.kind = ExportField::kVector;
      for (int a = 0; a < h->K; ++a) f.src[a] = field == AQ_FIELD_VOLUME_FRACTIONS ? gr.vf[a] : gr.nvf[h->nf][a];
  }
  if (!f.src[1] && n <= kHostElements) return field_on_host(h, f, n, (uint32_t*)dst);
  // Scratch: an array of the idle particle buffer (see aq_flip_get_particles), or one of its
  // own, kept, where that is small; a field larger than it is exported in pieces.
  const size_t elem = w * 4, particles = (size_t)h->Np * sizeof(float4);
  char* scratch = (char*)h->P[h->cur ^ 1].a;
  size_t cap = particles;
  if (const size_t want = std::min(bytes, aq_flip::kExportBytes); particles < want) {
    void* p = nullptr;
    if (h->export_cap < want && h->alloc(&p, want) == AQ_OK) h->export_buf = p, h->export_cap = want;
    if (h->export_cap > cap) scratch = (char*)h->export_buf, cap = h->export_cap;  // (else out of memory: make do)
  }
  for (size_t done = 0; done < n;) {
    const size_t m = std::min(n - done, cap / elem);
    launch_export_field(h->G, f, (long long)done, (long long)m, scratch, h->stream);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync((char*)dst + done * elem, scratch, m * elem, hipMemcpyDeviceToHost, h->stream));
    done += m;
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  return AQ_OK;
}

aq_status aq_flip_set_field(aq_flip* h, int32_t field, const void* src, size_t bytes) {
  if (!h || !src) return fail(AQ_EINVAL, "null argument");
  h->nvo_valid = false;
  int w;
  bool isInt;
  const size_t n = field_elems(h, field, &w, &isInt);
  if (n == 0) return fail(AQ_EINVAL, "unknown field");
  if (field == AQ_FIELD_PARTICLE_COUNT)
    return fail(AQ_EINVAL, "particleCount is derived from the cell bins and cannot be set");
  if (bytes != n * w * 4) return fail(AQ_EINVAL, "byte count does not match the field");
  const Geom& G = h->G;
  const size_t nc = (size_t)G.ncell;
  const float* F = (const float*)src;
  const int32_t* I = (const int32_t*)src;
  const bool face = (field == AQ_FIELD_CONTENT || field == AQ_FIELD_VELOCITY ||
                     field == AQ_FIELD_NEW_VELOCITY);
  const int EX = face ? G.X + 1 : G.X, EYe = face ? G.Y + 1 : G.Y, EZe = face ? G.Z + 1 : G.Z;
  auto each = [&](auto&& fn) {
    size_t o = 0;
    for (int x = 0; x < EX; ++x)
      for (int y = 0; y < EYe; ++y)
        for (int z = 0; z < EZe; ++z, ++o) fn(o, (size_t)G.g(x, y, z));
  };
  switch (field) {
    case AQ_FIELD_CONTENT: {
      std::vector<uint8_t> c;
      AQ_TRY(d2h(h, c, h->gr.content, nc));
      each([&](size_t o, size_t g) { c[g] = (uint8_t)I[o]; });
      AQ_TRY(h2d(h, h->gr.content, c));
      content_changed(h, false);
      refresh_rhs(h);
      HIP_TRY(hipStreamSynchronize(h->stream));
      break;
    }
    case AQ_FIELD_VELOCITY:
    case AQ_FIELD_NEW_VELOCITY: {
      for (int a = 0; a < 3; ++a) {
        float* d = field == AQ_FIELD_VELOCITY ? h->gr.vel[a] : h->gr.nvel[h->nv][a];
        std::vector<float> v;
        AQ_TRY(d2h(h, v, d, nc));
        each([&](size_t o, size_t g) { v[g] = F[4 * o + a]; });
        AQ_TRY(h2d(h, d, v));
      }
      break;
    }
    case AQ_FIELD_PRESSURE:
    case AQ_FIELD_DIVERGENCE:
    case AQ_FIELD_DENSITY: {
      float* d = field == AQ_FIELD_PRESSURE ? h->gr.p[h->pb]
                 : field == AQ_FIELD_DIVERGENCE ? h->gr.div
                                                : h->gr.density;
      std::vector<float> v;
      AQ_TRY(d2h(h, v, d, nc));
      each([&](size_t o, size_t g) { v[g] = F[o]; });
      AQ_TRY(h2d(h, d, v));
      if (field == AQ_FIELD_PRESSURE) h->air_clean[h->pb] = false;
      if (field != AQ_FIELD_PRESSURE) {
        // keep the Jacobi right-hand side consistent with divergence*density
        refresh_rhs(h);
        HIP_TRY(hipStreamSynchronize(h->stream));
      }
      break;
    }
    case AQ_FIELD_HAS_VELOCITY: {
      std::vector<uint8_t> v;
      AQ_TRY(d2h(h, v, h->gr.hasvel[h->hv], nc));
      each([&](size_t o, size_t g) {
        v[g] = (uint8_t)((I[4 * o] ? 1 : 0) | (I[4 * o + 1] ? 2 : 0) | (I[4 * o + 2] ? 4 : 0));
      });
      AQ_TRY(h2d(h, h->gr.hasvel[h->hv], v));
      break;
    }
    case AQ_FIELD_VOLUME_FRACTIONS:
    case AQ_FIELD_NEW_VOLUME_FRACTIONS: {
      int need = 1;
      for (size_t o = 0; o < n; ++o)
        for (int a = 3; a >= need; --a)
          if (F[4 * o + a] != 0.f) {
            need = a + 1;
            break;
          }
      if (need > h->K) {
        drop_graphs(h);
        h->K = need;
      }
      for (int a = 0; a < h->K; ++a) {
        float* d = field == AQ_FIELD_VOLUME_FRACTIONS ? h->gr.vf[a] : h->gr.nvf[h->nf][a];
        std::vector<float> v;
        AQ_TRY(d2h(h, v, d, nc));
        each([&](size_t o, size_t g) { v[g] = F[4 * o + a]; });
        AQ_TRY(h2d(h, d, v));
      }
      break;
    }
  }
  return AQ_OK;
}

aq_status aq_flip_get_cells(aq_flip* h, int32_t* cell_start, int32_t* cell_end, int32_t* hash,
                            int32_t* perm) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  const Geom& G = h->G;
  std::vector<int> off;
  AQ_TRY(d2h(h, off, h->B.offsets, (size_t)G.ncells_hash + 1));
  const size_t e1 = (size_t)(G.X + 1) * (G.Y + 1) * (G.Z + 1);
  if (cell_start || cell_end) {
    // Reference convention: cellStart/cellEnd sized (X+1)(Y+1)(Z+1), inclusive end,
    // -1 where empty (Fluid_3D_common.cuh:47-48, Fluid_kernels.cuh:3-22).
    for (size_t c = 0; c < e1; ++c) {
      int s = -1, e = -1;
      if (c < (size_t)G.ncells_hash && off[c + 1] > off[c]) {
        s = off[c];
        e = off[c + 1] - 1;
      }
      if (cell_start) cell_start[c] = s;
      if (cell_end) cell_end[c] = e;
    }
  }
  if (hash)
    for (int c = 0; c < G.ncells_hash; ++c)
      for (int k = off[c]; k < off[c + 1]; ++k) hash[k] = c;
  if (perm) {
    std::vector<int> p;
    AQ_TRY(d2h(h, p, h->B.perm, (size_t)h->Np));
    std::memcpy(perm, p.data(), p.size() * sizeof(int));
  }
  return AQ_OK;
}

aq_status aq_flip_residual_fp64(aq_flip* h, double* rel) {
  if (!h || !rel) return fail(AQ_EINVAL, "null argument");
  launch_residual(h->G, h->gr, h->pb, h->red_partial, h->red_out, h->stream);
  HIP_TRY(hipGetLastError());
  double o[2];
  HIP_TRY(hipMemcpyAsync(o, h->red_out, sizeof(o), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  *rel = o[1] > 0 ? std::sqrt(o[0]) / std::sqrt(o[1]) : std::sqrt(o[0]);
  return AQ_OK;
}

aq_status aq_flip_volume_stats(aq_flip* h, aq_flip_stats* out) {
  if (!h || !out) return fail(AQ_EINVAL, "null argument");
  launch_stats(h->G, h->P[h->cur], h->Np, h->K, h->gr, h->red_partial, h->nparts_red, h->red_out, h->stream);
  HIP_TRY(hipGetLastError());
  double o[16];
  HIP_TRY(hipMemcpyAsync(o, h->red_out, sizeof(o), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  out->particles = h->Np;
  out->fluid_cells = (int64_t)o[4];
  for (int a = 0; a < 4; ++a) out->phase_sum[a] = a < h->K ? o[a] : 0.0;
  out->mean_ppc = out->fluid_cells > 0 ? (double)h->Np / (double)out->fluid_cells : 0.0;
  for (int a = 0; a < 3; ++a) {
    out->pos_min[a] = -o[5 + a];
    out->pos_max[a] = o[8 + a];
  }
  return AQ_OK;
}

aq_status aq_flip_solve_pressure(aq_flip* h, double tol, int32_t max_iters, int32_t check_every,
                                 int32_t* iters_out, double* rel_out) {
  if (!h || max_iters < 0 || check_every < 1) return fail(AQ_EINVAL, "bad argument");
  int it = 0;
  double rel = 0;
  AQ_TRY(aq_flip_residual_fp64(h, &rel));
  ChunkedSweeps C{h, check_every, max_iters, tol, rel};
  while (!(C.res <= tol) && C.done < max_iters) AQ_TRY(C.next());
  AQ_TRY(C.finish());
  HIP_TRY(hipStreamSynchronize(h->stream));  // a chunk queued ahead may still be running
  it = C.done;
  rel = C.res;
  if (iters_out) *iters_out = it;
  if (rel_out) *rel_out = rel;
  if (!(rel <= tol)) return fail(AQ_ESTALL, "pressure solve reached its iteration cap");
  return AQ_OK;
}

// ---- snapshots ---------------------------------------------------------------
extern "C++" {
namespace {

constexpr char kSnapMagic[8] = {'A', 'Q', 'F', 'L', 'I', 'P', 'S', 'N'};

// Every device array that carries state between calls, tagged in a fixed order.
// Ping-pong pairs contribute their current buffer only.
struct SnapArray {
  uint32_t tag;
  void* ptr;
  size_t bytes;
};
std::vector<SnapArray> snapshot_arrays(aq_flip* h) {
  const Geom& G = h->G;
  const size_t nc = (size_t)G.ncell, np = (size_t)h->Np, nh = (size_t)G.ncells_hash;
  Grid& gr = h->gr;
  std::vector<SnapArray> a;
  const Particles& P = h->P[h->cur];
  a.push_back({1, P.a, np * sizeof(float4)});
  a.push_back({2, P.b, np * sizeof(float4)});
  if (h->K > 2) a.push_back({3, P.c, np * sizeof(float4)});
  a.push_back({10, gr.content, nc});
  for (int c = 0; c < 3; ++c) a.push_back({11u + c, gr.vel[c], nc * 4});
  for (int c = 0; c < 3; ++c) a.push_back({14u + c, gr.nvel[h->nv][c], nc * 4});
  a.push_back({17, gr.hasvel[h->hv], nc});
  a.push_back({18, gr.p[h->pb], nc * 4});
  a.push_back({19, gr.div, nc * 4});
  a.push_back({20, gr.rhs, nc * 4});
  a.push_back({21, gr.density, nc * 4});
  for (int c = 0; c < h->K; ++c) a.push_back({30u + c, gr.vf[c], nc * 4});
  for (int c = 0; c < h->K; ++c) a.push_back({40u + c, gr.nvf[h->nf][c], nc * 4});
  a.push_back({50, gr.active, ((nh + 255) / 256 + 1) * sizeof(uint32_t)});
  a.push_back({60, h->B.offsets, (nh + 1) * sizeof(int)});
  a.push_back({61, h->B.hash, np * sizeof(int)});
  a.push_back({62, h->B.perm, np * sizeof(int)});
  return a;
}

// Configuration fields in a fixed order (independent of the struct's padding).
template <typename IO>
void config_fields(IO&& io, aq_flip_config& c) {
  for (int a = 0; a < 3; ++a) io(c.size[a]);
  io(c.dt), io(c.flip_coeff), io(c.particle_jitter), io(c.grid_physical_size);
  io(c.pressure_iters), io(c.diffusion_iters), io(c.phase_count);
  for (int a = 0; a < 3; ++a) io(c.gravity[a]);
  for (int a = 0; a < 4; ++a) io(c.phase_densities[a]);
  io(c.diffusion_coeff), io(c.pressure_init), io(c.ref_boundary_coverage), io(c.seed), io(c.n_volumes);
  for (int i = 0; i < AQ_MAX_VOLUMES; ++i) {
    aq_flip_volume& v = c.volumes[i];
    io(v.shape);
    for (int a = 0; a < 3; ++a) io(v.box_min[a]);
    for (int a = 0; a < 3; ++a) io(v.box_max[a]);
    for (int a = 0; a < 3; ++a) io(v.center[a]);
    io(v.radius), io(v.phase);
  }
}

}  // namespace
}  // extern "C++"

aq_status aq_flip_save(aq_flip* h, const char* path) {
  if (!h || !path) return fail(AQ_EINVAL, "null argument");
  HIP_TRY(hipStreamSynchronize(h->stream));
  FILE* f = std::fopen(path, "wb");
  if (!f) return fail(AQ_EINVAL, std::string("cannot open ") + path + " for writing");
  bool ok = true;
  auto put = [&](const void* p, size_t n) { ok = ok && std::fwrite(p, 1, n, f) == n; };
  auto io = [&](auto& v) { put(&v, sizeof(v)); };
  put(kSnapMagic, 8);
  uint32_t version = AQ_SNAPSHOT_VERSION;
  io(version);
  aq_flip_config cfg = h->cfg;
  config_fields(io, cfg);
  int64_t np = h->Np;
  int32_t K = h->K, nsec = 0;
  float t = h->physicalTime;
  io(np), io(K), io(t);
  const std::vector<SnapArray> arrays = snapshot_arrays(h);
  nsec = (int32_t)arrays.size();
  io(nsec);
  std::vector<char> buf;
  for (const SnapArray& a : arrays) {
    uint32_t tag = a.tag;
    uint64_t bytes = a.bytes;
    io(tag), io(bytes);
    buf.resize(a.bytes);
    if (hipMemcpy(buf.data(), a.ptr, a.bytes, hipMemcpyDeviceToHost) != hipSuccess) ok = false;
    put(buf.data(), a.bytes);
  }
  ok = (std::fclose(f) == 0) && ok;
  if (!ok) return fail(AQ_EHIP, std::string("writing the snapshot ") + path + " failed");
  return AQ_OK;
}

aq_status aq_flip_load(const char* path, aq_flip** out) {
  if (!path || !out) return fail(AQ_EINVAL, "null argument");
  *out = nullptr;
  FILE* f = std::fopen(path, "rb");
  if (!f) return fail(AQ_EINVAL, std::string("cannot open ") + path);
  bool ok = true;
  auto get = [&](void* p, size_t n) { ok = ok && std::fread(p, 1, n, f) == n; };
  auto io = [&](auto& v) { get(&v, sizeof(v)); };
  auto bail = [&](aq_status st, const std::string& msg) {
    std::fclose(f);
    return fail(st, msg);
  };
  char magic[8];
  get(magic, 8);
  uint32_t version = 0;
  io(version);
  if (!ok || std::memcmp(magic, kSnapMagic, 8) != 0) return bail(AQ_EINVAL, "not a libaqflip snapshot");
  if (version != AQ_SNAPSHOT_VERSION)
    return bail(AQ_EINVAL, "snapshot format version " + std::to_string(version) + " is not supported");
  aq_flip_config cfg{};
  config_fields(io, cfg);
  int64_t np = 0;
  int32_t K = 0, nsec = 0;
  float t = 0.f;
  io(np), io(K), io(t), io(nsec);
  if (!ok) return bail(AQ_EINVAL, "truncated snapshot header");
  if (validate(&cfg) != AQ_OK) return bail(AQ_EINVAL, std::string("snapshot configuration: ") + aq_last_error());
  if (np <= 0 || np > (1ll << 31) - 1 || K < 1 || K > 4) return bail(AQ_EINVAL, "corrupt snapshot state");
  aq_flip* h = new aq_flip;
  read_env(h);
  aq_status st = setup(h, &cfg, np);
  // The sections arrive by copies that do not wait for the handle's stream: the clear of its
  // memory has to be over before the first.
  if (st == AQ_OK && hipStreamSynchronize(h->stream) != hipSuccess)
    st = fail(AQ_EHIP, "snapshot: clearing the handle's memory failed");
  if (st != AQ_OK) {
    delete h;
    return bail(st, aq_last_error());
  }
  h->K = K;
  h->physicalTime = t;
  const std::vector<SnapArray> arrays = snapshot_arrays(h);
  if ((size_t)nsec != arrays.size()) {
    delete h;
    return bail(AQ_EINVAL, "snapshot sections do not match its configuration");
  }
  std::vector<char> buf;
  for (const SnapArray& a : arrays) {
    uint32_t tag = 0;
    uint64_t bytes = 0;
    io(tag), io(bytes);
    if (!ok || tag != a.tag || bytes != a.bytes) {
      delete h;
      return bail(AQ_EINVAL, "corrupt snapshot section " + std::to_string(a.tag));
    }
    buf.resize(a.bytes);
    get(buf.data(), a.bytes);
    if (!ok || hipMemcpy(a.ptr, buf.data(), a.bytes, hipMemcpyHostToDevice) != hipSuccess) {
      delete h;
      return bail(AQ_EINVAL, "truncated snapshot section " + std::to_string(a.tag));
    }
    if (a.ptr == h->B.offsets) {  // as the particles were binned last
      const int* off = (const int*)buf.data();
      long long cells = 0;
      for (int c = 0; c < h->G.ncells_hash; ++c) cells += off[c + 1] > off[c];
      expect_fluid(h, cells);
    }
  }
  std::fclose(f);
  // Pressure buffers: only the current one was saved, so neither is known to hold 0
  // on every AIR cell; the next sweeps write them fully (same values either way).
  h->air_clean[0] = h->air_clean[1] = false;
  launch_active_list(h->G, h->gr, h->stream);  // derived from the restored flags
  if (hipStreamSynchronize(h->stream) != hipSuccess) {
    delete h;
    return bail(AQ_EHIP, "snapshot: rebuilding the active list failed");
  }
  *out = h;
  return AQ_OK;
}

aq_status aq_flip_solve_pressure_mgpcg(aq_flip* h, double tol, int32_t max_iters, int32_t check_every,
                                       int32_t from_current, int32_t* iters_out, double* rel_out) {
  if (!h || max_iters < 0 || check_every < 1 || !(tol > 0)) return fail(AQ_EINVAL, "bad argument");
  int it = 0;
  double cg = 0, rel = 0;
  AQ_TRY(mgpcg_solve(h, tol, max_iters, check_every, from_current != 0, &it, &cg));
  AQ_TRY(residual_now(h, &rel));
  if (iters_out) *iters_out = it;
  if (rel_out) *rel_out = rel;
  if (!(cg <= tol)) return fail(AQ_ESTALL, "MG-PCG reached its iteration cap");
  return AQ_OK;
}

aq_status aq_flip_set_timing(aq_flip* h, int32_t enable) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  h->timing = enable != 0;
  return AQ_OK;
}
aq_status aq_flip_get_timing(aq_flip* h, double* stage_ms, int64_t* stage_calls) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  for (int i = 0; i < AQ_STAGE_COUNT; ++i) {
    if (stage_ms) stage_ms[i] = h->stage_ms[i];
    if (stage_calls) stage_calls[i] = h->stage_calls[i];
  }
  return AQ_OK;
}
aq_status aq_flip_paired_diffusion_computed(aq_flip* h, int64_t* count) {
  if (!h || !count) return fail(AQ_EINVAL, "null argument");
  uint32_t v = 0;
  HIP_TRY(hipStreamSynchronize(h->stream));
  HIP_TRY(hipMemcpy(&v, h->gr.dchange + 3, sizeof(v), hipMemcpyDeviceToHost));
  *count = (int64_t)v;
  return AQ_OK;
}

aq_status aq_flip_reset_timing(aq_flip* h) {
  if (!h) return fail(AQ_EINVAL, "null handle");
  for (int i = 0; i < AQ_STAGE_COUNT; ++i) {
    h->stage_ms[i] = 0;
    h->stage_calls[i] = 0;
  }
  return AQ_OK;
}

double aq_flip_physical_time(const aq_flip* h) { return h ? (double)h->physicalTime : 0.0; }

aq_status aq_flip_get_center(const aq_flip* h, float* center) {
  if (!h || !center) return fail(AQ_EINVAL, "null argument");
  // Fluid::getCenter returns gridPhysicalSize/2 on every axis (Fluid_3D_FLIP.cu:728-730).
  for (int a = 0; a < 3; ++a) center[a] = h->cfg.grid_physical_size / 2;
  return AQ_OK;
}
float aq_flip_container_size(const aq_flip* h) { return h ? h->cfg.grid_physical_size : 0.f; }

const char* aq_last_error(void) { return g_err.c_str(); }

const char* aq_flip_version(void) { return "aqflip 0.1.0 (gfx950)"; }

}  // extern "C"
