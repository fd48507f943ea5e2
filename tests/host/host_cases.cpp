// host_cases.cpp -- the library's host code over fake_hip.hpp, one case per run:
//   host_cases NAME DIR      exit status 0: passed
#include "fake_hip.hpp"

#include <fstream>
#include <iterator>

#define REQUIRE(cond)                                                         \
  do {                                                                        \
    if (!(cond)) {                                                            \
      std::fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #cond, aq_last_error()); \
      std::exit(1);                                                           \
    }                                                                         \
  } while (0)

namespace {

std::string dir;

aq_flip_config config(int n, int phases = 1) {
  aq_flip_config c;
  REQUIRE(aq_flip_config_default(&c) == AQ_OK);
  c.size[0] = c.size[1] = c.size[2] = n;
  c.phase_count = phases;
  return c;
}
// A handle with `np` particles spread over the grid.
aq_flip* create(const aq_flip_config& c, int np = 64) {
  std::vector<float> pos(3 * np), frac(4 * np, 0.f);
  const float h = c.grid_physical_size / (float)c.size[1];
  for (int i = 0; i < np; ++i) {
    for (int a = 0; a < 3; ++a) pos[3 * i + a] = h * (0.5f + (float)((i + a) % c.size[a]));
    frac[4 * i] = 1.f;
  }
  aq_flip* f = nullptr;
  REQUIRE(aq_flip_create_with_particles(&c, pos.data(), nullptr, frac.data(), np, &f) == AQ_OK);
  return f;
}
std::string saved(aq_flip* f, const std::string& name) {
  const std::string path = dir + "/" + name;
  REQUIRE(aq_flip_save(f, path.c_str()) == AQ_OK);
  std::ifstream in(path, std::ios::binary);
  return std::string(std::istreambuf_iterator<char>(in), {});
}

// The clear of a new handle's memory must not run over the sections of its snapshot.
void load_after_clear() {
  aq_flip* f = create(config(32));
  const std::vector<float> p(32 * 32 * 32, 1.5f);
  REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, p.data(), p.size() * 4) == AQ_OK);
  const std::string first = saved(f, "first");
  aq_flip_destroy(f);
  aq_flip* g = nullptr;
  REQUIRE(aq_flip_load((dir + "/first").c_str(), &g) == AQ_OK);
  REQUIRE(saved(g, "second") == first);
  aq_flip_destroy(g);
}

// A counting sort that fails after its counts leaves them dirty, whatever succeeds next.
void hash_after_a_failed_sort() {
  aq_hash* h = nullptr;
  REQUIRE(aq_hash_create(4, 4, 4, 1.f, 4096, &h) == AQ_OK);
  const std::vector<float> rec(3 * 4096, 0.5f);
  REQUIRE(aq_hash_sort_host(h, rec.data(), 100, 3, nullptr, nullptr, nullptr, nullptr, 0, nullptr) == AQ_OK);
  fake::check_bins = false;
  fake::fail_launch = "scan";
  REQUIRE(aq_hash_sort_host(h, rec.data(), 100, 3, nullptr, nullptr, nullptr, nullptr, 0, nullptr) != AQ_OK);
  REQUIRE(aq_hash_sort_host(h, rec.data(), 4096, 3, nullptr, nullptr, nullptr, nullptr, 0, nullptr) == AQ_OK);
  REQUIRE(fake::count["radix"] == 1);  // the crowded sort, which does not touch the counts
  fake::check_bins = true;
  for (int i = 0; i < 2; ++i)
    REQUIRE(aq_hash_sort_host(h, rec.data(), 100, 3, nullptr, nullptr, nullptr, nullptr, 0, nullptr) == AQ_OK);
  aq_hash_destroy(h);
}

// Records are sorted by radix only where the cells are crowded or the records many and wide:
// elsewhere the counting sort is the faster one for records that come nearly sorted.
void sort_by_density() {
  struct Case {
    int side, n, stride;
    bool radix;
  };
  const std::vector<float> rec(12 * 786432, 0.5f);
  for (const Case& c : {Case{4, 64 * 32, 3, false}, {4, 64 * 32 + 1, 3, true}, {10, 4000, 3, false}, {10, 20000, 12, false},
                        {12, 60000, 3, true}, {3, 800, 3, false}, {3, 2000, 3, false}, {3, 2048, 3, true},
                        {40, 786432, 8, false}, {40, 786432, 12, true}, {40, 786431, 12, false}, {59, 786432, 12, false}}) {
    aq_hash* h = nullptr;
    REQUIRE(aq_hash_create(c.side, c.side, c.side, 1.f, c.n, &h) == AQ_OK);
    const long long before = fake::count["radix"];
    REQUIRE(aq_hash_sort_host(h, rec.data(), c.n, c.stride, nullptr, nullptr, nullptr, nullptr, 0, nullptr) == AQ_OK);
    REQUIRE(fake::count["radix"] - before == c.radix);
    aq_hash_destroy(h);
  }
}

// A sort that runs out of memory while its buffers grow leaves none of the old ones in use.
void hash_after_failed_growth() {
  const auto sort = [](aq_hash* h, const float* rec, long long n) {
    return aq_hash_sort_host(h, rec, n, 3, nullptr, nullptr, nullptr, nullptr, 0, nullptr);
  };
  const std::vector<float> rec(3 * 8192, 0.5f);
  for (int cells : {4, 2}) {  // 4^3: 1,000 records are no crowded sort there; 2^3: 2,100 are one
    const long long n = cells == 4 ? 1000 : 2100;
    for (int room = 1; room <= 40; ++room) {  // each allocation of the growth in turn
      aq_hash* h = nullptr;
      fake::capacity = (size_t)-1;
      REQUIRE(aq_hash_create(cells, cells, cells, 1.f, n, &h) == AQ_OK);
      REQUIRE(sort(h, rec.data(), n) == AQ_OK);
      fake::capacity = fake::used(0) + (size_t)room * 8192;
      (void)sort(h, rec.data(), 8192);
      (void)sort(h, rec.data(), n);  // may fail for the larger buffers that are there by now
      fake::capacity = (size_t)-1;
      REQUIRE(sort(h, rec.data(), n) == AQ_OK);
      aq_hash_destroy(h);
      REQUIRE(fake::used(0) == 0);
    }
  }
}

// A solve that ends while its next chunk is queued ahead returns with nothing left on the
// stream, and with the iterate, sweep count and residual of the chunk that reached tol.
void solve_returns_idle() {
  aq_flip* f = create(config(16));
  const std::vector<float> zero(16 * 16 * 16, 0.f);
  fake::drop_at = 195;  // sooner than the last two residuals let expect
  for (int every : {10, 20}) {
    REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, zero.data(), zero.size() * 4) == AQ_OK);
    int32_t it = 0;
    double rel = 0, now = 0;
    const long long undone = fake::count["copy_cells"];
    REQUIRE(aq_flip_solve_pressure(f, 0.01, 5000, every, &it, &rel) == AQ_OK);
    REQUIRE(fake::pending() == 0);
    REQUIRE(fake::count["copy_cells"] > undone);  // a chunk was queued ahead
    REQUIRE(it == 200 && std::abs(rel - 1e-3 * std::pow(0.99, 200)) < 1e-12);
    REQUIRE(aq_flip_residual_fp64(f, &now) == AQ_OK && now == rel);
  }
  aq_flip_destroy(f);
}

// One failed launch in a tolerance solve fails that solve only.
void solves_after_a_failed_launch() {
  for (const char* eager : {"1", "0"}) {
    setenv("AQFLIP_NO_GRAPH", eager, 1);
    aq_flip* f = create(config(16));
    const std::vector<float> zero(16 * 16 * 16, 0.f);
    for (const char* name : {"", "residual", "small", "copy_cells", ""}) {
      REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, zero.data(), zero.size() * 4) == AQ_OK);
      REQUIRE(aq_flip_solve_pressure(f, 0.9, 20, 20, nullptr, nullptr) == AQ_OK);
      fake::fail_launch = name;
      const aq_status st = aq_flip_solve_pressure(f, 0.2, 1000, 20, nullptr, nullptr);
      REQUIRE(st != AQ_OK || !fake::fail_launch.empty() || !*name);
      fake::fail_launch.clear();
      REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, zero.data(), zero.size() * 4) == AQ_OK);
      int32_t it = 0;
      REQUIRE(aq_flip_solve_pressure(f, 0.5, 1000, 20, &it, nullptr) == AQ_OK);
      REQUIRE(it == 80);
    }
    aq_flip_destroy(f);
  }
}

// Sweeps whose capture fails have not run: the pressure is still the iterate before them.
void iterate_after_a_failed_capture() {
  aq_flip* f = create(config(33));
  const std::vector<float> zero(33 * 33 * 33, 0.f);
  REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, zero.data(), zero.size() * 4) == AQ_OK);
  REQUIRE(aq_flip_solve_pressure(f, 1e-9, 20, 20, nullptr, nullptr) == AQ_ESTALL);
  fake::fail_launch = "tile";
  REQUIRE(aq_flip_solve_pressure(f, 1e-9, 12, 12, nullptr, nullptr) == AQ_EHIP);
  double rel = 0;
  REQUIRE(aq_flip_residual_fp64(f, &rel) == AQ_OK && std::abs(rel - std::pow(0.99, 20)) < 1e-12);
  aq_flip_destroy(f);
}

// A step marks every interior cell AIR or FLUID, replayed or not: solves after it take
// several sweeps to a launch again.
void replayed_step_marks_content() {
  aq_flip* f = create(config(33));
  std::vector<int32_t> content(34 * 34 * 34, 0);
  const long long captured = fake::captures;
  for (int i = 0; i < 8; ++i) {
    REQUIRE(aq_flip_set_field(f, AQ_FIELD_CONTENT, content.data(), content.size() * 4) == AQ_OK);
    REQUIRE(aq_flip_step(f) == AQ_OK);
  }
  REQUIRE(fake::captures - captured < 8);  // some of the steps were replayed
  const long long single = fake::count["jacobi"];
  REQUIRE(aq_flip_solve_pressure(f, 1e-9, 40, 40, nullptr, nullptr) == AQ_ESTALL);
  REQUIRE(fake::count["jacobi"] == single && fake::count["tile"] >= 10);
  aq_flip_destroy(f);
}

// Timed steps of small grids: a stage that counts sweeps has the launches that ran them.
void timed_small_steps() {
  for (const auto& iters : {std::pair<int, int>{100, 30}, {30, 100}, {40, 40}, {20, 25}, {25, 20}}) {
    aq_flip_config c = config(16, 2);
    c.pressure_iters = iters.first, c.diffusion_iters = iters.second;
    aq_flip* f = create(c);
    REQUIRE(aq_flip_set_timing(f, 1) == AQ_OK && aq_flip_steps(f, 2) == AQ_OK);
    double ms[AQ_STAGE_COUNT];
    int64_t passes[AQ_STAGE_COUNT];
    REQUIRE(aq_flip_get_timing(f, ms, passes) == AQ_OK);
    const int n = std::min(iters.first, iters.second);
    REQUIRE(fake::count["small"] > 0 && passes[AQ_STAGE_PRESSURE_DIFFUSION] == 2 * n);
    REQUIRE(passes[AQ_STAGE_PRESSURE] == 2 * (iters.first - n) && passes[AQ_STAGE_DIFFUSION] == 2 * (iters.second - n));
    for (int st : {AQ_STAGE_PRESSURE_DIFFUSION, AQ_STAGE_PRESSURE, AQ_STAGE_DIFFUSION})
      REQUIRE((passes[st] > 0) == (ms[st] > 0));  // (the stand-in's milliseconds are launches)
    aq_flip_destroy(f);
  }
}

// Eight chunk lengths of a handle's tolerance solves replay their graphs, on either kind of
// content, with or without a chunk queued ahead.
void eight_chunk_lengths_replay() {
  aq_flip* f = create(config(33));
  const std::vector<float> zero(33 * 33 * 33, 0.f);
  std::vector<int32_t> content(34 * 34 * 34, 0);
  const auto solve_all = [&] {
    for (int k = 1; k <= 8; ++k) {  // k * 8 sweeps: the pressure ends in the buffer it began in
      fake::rate = 0.99;
      REQUIRE(aq_flip_set_field(f, AQ_FIELD_PRESSURE, zero.data(), zero.size() * 4) == AQ_OK);
      REQUIRE(aq_flip_solve_pressure(f, 1e-9, k * 8 * 4, k * 8, nullptr, nullptr) == AQ_ESTALL);
    }
  };
  for (bool uploaded : {false, true}) {
    if (uploaded) REQUIRE(aq_flip_set_field(f, AQ_FIELD_CONTENT, content.data(), content.size() * 4) == AQ_OK);
    solve_all();
    solve_all();  // (the second round starts from other buffer states)
    const long long captured = fake::captures, launched = fake::launches;
    solve_all();
    // every chunk is a replay: only the residual at each solve's start is launched
    REQUIRE(fake::captures == captured && fake::launches - launched <= 2 * 8);
  }
  aq_flip_destroy(f);
}

// The memory kept from destroyed handles serves the library's other allocations when there
// is no more, and goes back to the device when asked.
void kept_memory_is_given_back() {
  const auto keep = [] {
    fake::capacity = (size_t)-1;
    aq_flip_destroy(create(config(112)));
    REQUIRE(fake::used(0) > 1 << 20);
    fake::capacity = fake::used(0);
  };
  keep();
  aq_hash* h = nullptr;
  REQUIRE(aq_hash_create(8, 8, 8, 1.f, 1000, &h) == AQ_OK);
  aq_hash_destroy(h);
  keep();
  aq_unet_config uc;
  aq_unet* net = nullptr;
  REQUIRE(aq_unet_config_default(&uc) == AQ_OK && aq_unet_create(&uc, &net) == AQ_OK);
  aq_unet_destroy(net);
  keep();
  aq_flip* f = nullptr;  // (the stand-in's seeder counts no particles)
  const aq_flip_config c = config(64);
  REQUIRE(aq_flip_create(&c, &f) == AQ_EINVAL);
  keep();
  aq_flip_release_memory();
  REQUIRE(fake::used(0) == 0);
}

// A block that was allocated with another device current is kept for that device.
void kept_blocks_stay_on_their_device() {
  const aq_flip_config c = config(64);
  const auto solve = [&](int device) {
    aq_flip* f = create(c);
    fake::device = device, fake::mg_iters = 2;
    const size_t before = fake::used(device);
    REQUIRE(aq_flip_solve_pressure_mgpcg(f, 1e-6, 10, 1, 0, nullptr, nullptr) == AQ_OK);
    const size_t added = fake::used(device) - before;
    fake::device = 0;
    aq_flip_destroy(f);
    return added;
  };
  const size_t size = solve(1);
  REQUIRE(size > 0 && solve(0) == size);
  aq_flip_release_memory();
}

// A network that runs out of memory while its activations grow leaves none of the old ones
// in use.
void network_after_failed_growth() {
  aq_unet_config uc;
  aq_unet* net = nullptr;
  REQUIRE(aq_unet_config_default(&uc) == AQ_OK && aq_unet_create(&uc, &net) == AQ_OK);
  std::vector<float> x(2 * 16 * 16 * 16, 0.f), y(16 * 16 * 16);
  const auto forward = [&](int n) { return aq_unet_forward_host(net, x.data(), 1, n, n, n, y.data()); };
  aq_flip* f = create(config(16));
  const auto reserve = [&](int samples) { return aq_unet_dataset_reserve(net, samples, 16, 16, 16); };
  REQUIRE(forward(8) == AQ_OK && reserve(2) == AQ_OK && aq_unet_dataset_add_flip(net, f) == AQ_OK);
  fake::capacity = fake::used(0) + 200000;
  REQUIRE(forward(16) != AQ_OK);
  (void)forward(8);
  REQUIRE(reserve(64) != AQ_OK && aq_unet_dataset_size(net) == 0);
  fake::capacity = (size_t)-1;
  REQUIRE(forward(8) == AQ_OK && forward(16) == AQ_OK);
  REQUIRE(aq_unet_dataset_add_flip(net, f) != AQ_OK);  // nothing is reserved
  REQUIRE(reserve(2) == AQ_OK && aq_unet_dataset_add_flip(net, f) == AQ_OK && aq_unet_dataset_size(net) == 1);
  aq_flip_destroy(f);
  aq_unet_destroy(net);
}

// An export takes a bounded scratch buffer at most, and works without any memory left.
void exports_need_little_memory() {
  for (bool room : {true, false}) {
    aq_flip* f = create(config(130), room ? 64 : 5000);
    fake::capacity = fake::used(0) + (room ? 33 << 20 : 0);
    for (int field : {AQ_FIELD_PRESSURE, AQ_FIELD_VELOCITY, AQ_FIELD_HAS_VELOCITY}) {
      std::vector<int> out(aq_flip_field_bytes(f, field) / 4, -1);
      REQUIRE(aq_flip_get_field(f, field, out.data(), out.size() * 4) == AQ_OK);
      const size_t w = field == AQ_FIELD_PRESSURE ? 1 : 4;
      for (size_t i = 0; i < out.size(); ++i) REQUIRE(out[i] == (int)(i / w));  // as the stand-in fills them
    }
    fake::capacity = (size_t)-1;
    aq_flip_destroy(f);
    aq_flip_release_memory();
  }
}

// Whether a small grid's sweeps run in one launch goes by the cells that hold particles, however
// few there are in each, through uploads and snapshots.
void sparse_particles_on_small_grids() {
  const int n = 24;
  aq_flip_config c = config(n);
  c.diffusion_iters = 0;
  const float h = c.grid_physical_size / n;
  std::vector<float> everywhere, corner;
  for (int i = 0; i < n * n * n; ++i)
    for (int a : {i / (n * n), i / n % n, i % n}) {
      everywhere.push_back(h * ((float)a + 0.5f));
      corner.push_back(h * ((float)(a % 8) + 0.5f));
    }
  const auto one_launch = [](aq_flip* f) {
    const long long small = fake::count["small"];
    REQUIRE(aq_flip_steps(f, 3) == AQ_OK && fake::pending() == 0);
    return fake::count["small"] > small;
  };
  aq_flip* f = nullptr;
  REQUIRE(aq_flip_create_with_particles(&c, everywhere.data(), nullptr, nullptr, n * n * n, &f) == AQ_OK);
  REQUIRE(!one_launch(f));  // 13,824 cells
  REQUIRE(aq_flip_set_particles(f, corner.data(), nullptr, nullptr, n * n * n) == AQ_OK);
  REQUIRE(one_launch(f));  // 512 cells; 1,728 at eight per cell
  REQUIRE(aq_flip_set_particles(f, everywhere.data(), nullptr, nullptr, n * n * n) == AQ_OK);
  REQUIRE(!one_launch(f));
  aq_flip_destroy(f);
  // a snapshot counts the cells of its bins (the stand-in bins nothing: none hold particles)
  REQUIRE(aq_flip_create_with_particles(&c, everywhere.data(), nullptr, nullptr, n * n * n, &f) == AQ_OK);
  (void)saved(f, "sparse");
  aq_flip_destroy(f);
  REQUIRE(aq_flip_load((dir + "/sparse").c_str(), &f) == AQ_OK);
  REQUIRE(one_launch(f));
  aq_flip_destroy(f);
}

// Paired sweeps run on tiles where those that hold FLUID are few, by the number of phases.
void paired_tiles_by_fluid() {
  struct Case {
    int x, y, z, phases;
    double fluid;
    bool tiles;
  };
  for (const Case& c : {Case{33, 33, 33, 4, 0.95, true}, {48, 48, 48, 4, 0.95, true}, {50, 50, 50, 4, 0.95, false},
                        {48, 48, 48, 3, 0.95, true}, {50, 50, 50, 3, 0.95, false}, {50, 50, 50, 3, 0.3, true},
                        {80, 80, 80, 3, 0.3, false}, {64, 64, 64, 2, 0.95, true}, {72, 72, 72, 2, 0.95, false},
                        {72, 72, 72, 2, 0.3, true}, {90, 90, 90, 2, 0.53, false}, {256, 4, 256, 2, 1.0, false},
                        {101, 101, 101, 2, 0.1, true}, {102, 102, 102, 2, 0.1, false}}) {
    aqf::Geom G{};
    G.X = c.x, G.Y = c.y, G.Z = c.z, G.ncells_hash = c.x * c.y * c.z;
    REQUIRE(aqf::tile_pairs(G, c.phases, (long long)(c.fluid * G.ncells_hash)) == c.tiles);
  }
}

// With four phases fewer FLUID cells take the one launch.
void four_phases_on_small_grids() {
  for (int phases : {2, 3, 4}) {
    aq_flip_config c = config(16, phases);
    aq_flip* f = create(c, 8 * 1300);
    const long long small = fake::count["small"];
    REQUIRE(aq_flip_step(f) == AQ_OK);
    REQUIRE((fake::count["small"] > small) == (phases < 4));
    aq_flip_destroy(f);
  }
}

// Every tile has a workgroup of its own as long as there are enough, in whole groups.
void one_workgroup_per_tile() {
  for (int n : {1, 8, 9, 16, 17, 20, 28, 33, 40, 50, 56, 64, 72, 101}) {
    aqf::Geom G{};
    G.X = G.Y = G.Z = n, G.ncells_hash = n * n * n;
    const int tiles = aqf::sweep_tiles(G), grid = aqf::tile_grid(G);
    REQUIRE(grid <= 512 && (grid == 512 || grid >= tiles) && grid < tiles + 8 && (grid < 8 || grid % 8 == 0));
  }
}

// Sweeps run on tiles where the grid fills them or needs few of them.
void tiles_fit_the_grid() {
  struct Case {
    int x, y, z;
    bool fits;
  };
  for (const Case& c : {Case{33, 33, 33, true}, {64, 64, 64, true}, {100, 100, 100, true}, {130, 130, 65, true},
                        {256, 256, 256, true}, {256, 256, 1, true}, {1, 256, 256, true}, {1024, 8, 8, true},
                        {512, 512, 3, true}, {512, 512, 1, false}, {512, 512, 2, false}, {512, 512, 4, false},
                        {512, 512, 12, false}, {512, 512, 16, true}, {1024, 1024, 1, false}, {1024, 1, 1024, false},
                        {1024, 1024, 8, false}, {1024, 1024, 16, true}, {1024, 1024, 1024, true}}) {
    aqf::Geom G{};
    G.X = c.x, G.Y = c.y, G.Z = c.z, G.ncells_hash = c.x * c.y * c.z;
    REQUIRE(aqf::tile_fits(G) == c.fits);
  }
  aq_flip_config c = config(512);
  c.size[2] = 2;
  aq_flip* f = create(c);
  REQUIRE(aq_flip_run_stage(f, AQ_STAGE_PRESSURE) == AQ_OK);
  REQUIRE(fake::count["tile"] == 0 && fake::count["jacobi"] == c.pressure_iters);
  aq_flip_destroy(f);
}

// What a failed MG-PCG solve has left on the stream does not answer for the next one.
void mgpcg_after_a_failed_solve() {
  aq_flip* f = create(config(16));
  const auto solve = [&](int* it) { return aq_flip_solve_pressure_mgpcg(f, 1e-6, 100, 2, 0, it, nullptr); };
  int32_t it = 0;
  fake::mg_iters = 8;
  REQUIRE(solve(&it) == AQ_OK && it == 8);
  fake::fail_launch = "mg_iterate";  // the capture of the odd iterations, behind a queued even one
  fake::fail_skip = 1;
  REQUIRE(solve(&it) != AQ_OK && fake::pending() > 0);
  for (int i = 0; i < 2; ++i) REQUIRE(solve(&it) == AQ_OK && it == 8);
  aq_flip_destroy(f);
}

const std::map<std::string, void (*)()> cases = {
    {"four_phases_on_small_grids", four_phases_on_small_grids},
    {"paired_tiles_by_fluid", paired_tiles_by_fluid},
    {"sparse_particles_on_small_grids", sparse_particles_on_small_grids},
    {"one_workgroup_per_tile", one_workgroup_per_tile},
    {"tiles_fit_the_grid", tiles_fit_the_grid},
    {"exports_need_little_memory", exports_need_little_memory},
    {"sort_by_density", sort_by_density},
    {"network_after_failed_growth", network_after_failed_growth},
    {"kept_blocks_stay_on_their_device", kept_blocks_stay_on_their_device},
    {"kept_memory_is_given_back", kept_memory_is_given_back},
    {"eight_chunk_lengths_replay", eight_chunk_lengths_replay},
    {"timed_small_steps", timed_small_steps},
    {"replayed_step_marks_content", replayed_step_marks_content},
    {"iterate_after_a_failed_capture", iterate_after_a_failed_capture},
    {"mgpcg_after_a_failed_solve", mgpcg_after_a_failed_solve},
    {"solves_after_a_failed_launch", solves_after_a_failed_launch},
    {"solve_returns_idle", solve_returns_idle},
    {"hash_after_failed_growth", hash_after_failed_growth},
    {"hash_after_a_failed_sort", hash_after_a_failed_sort},
    {"load_after_clear", load_after_clear},
};

}  // namespace

int main(int argc, char** argv) {
  if (argc == 1) {
    for (const auto& c : cases) std::puts(c.first.c_str());
    return 0;
  }
  dir = argc > 2 ? argv[2] : ".";
  cases.at(argv[1])();
  return 0;
}
