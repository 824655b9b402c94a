// Host checks of what the library does around its kernels, on the HIP runtime
// of fake_hip.h.  Each check has a name, given as the argument.
#include <chrono>
#include <vector>

#include "fake_hip.h"
#include "ripples_amd.h"

namespace {

void require(bool ok, const char *what) {
  if (ok) return;
  printf("%s: %s\n", what, rip_last_error());
  exit(1);
}

bool is(const std::string &kernel, const char *name) { return kernel.find(name) != std::string::npos; }

// In-neighbours v + 1 .. v + 4 of every v.
rip_graph *ring(int model, uint32_t n) {
  std::vector<uint64_t> index(n + 1);
  std::vector<uint32_t> edges;
  for (uint32_t v = 0; v < n; ++v) {
    for (uint32_t d = 1; d <= 4; ++d) edges.push_back((v + d) % n);
    index[v + 1] = edges.size();
  }
  const std::vector<float> w(edges.size(), 0.2f);
  rip_graph *g;
  require(rip_graph_create(0, model, n, edges.size(), index.data(), edges.data(), w.data(), &g) == 0,
          "graph");
  return g;
}

// The count of samples that outgrew the lanes or waves (word 3 of the control
// words), set where the kernels clear it.
void set_long(const std::string &kernel, void **args, uint64_t count) {
  for (const char *k : {"reset_lane_kernel", "reset_stage_kernel", "reset_wave_kernel"})
    if (is(kernel, k)) (**static_cast<uint64_t ***>(static_cast<void *>(args)))[3] = count;
}

// A grid call that fails after its search began leaves colour masks and bitmaps
// behind: the next call must clear them before its own search.
void grid_scratch_after_failure() {
  const uint32_t n = 4000;
  rip_tune t{};
  t.colors = 64;
  bool cut = false;   // some call failed in that state
  for (long at = 0;; ++at) {
    rip_graph *g = ring(RIP_IC, n);
    rip_pool *p;
    require(rip_pool_create(g, 1, &p) == 0, "pool");
    bool searched = false, cleared = true;
    g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t, void **args) {
      set_long(kernel, args, 64);
      if (!is(kernel, "grid_seed_kernel")) return;
      searched = true;
      if (!cleared) {
        printf("failure %ld: the next call searched in what was left\n", at);
        exit(1);
      }
    };
    g_fail_at = at;
    g_failed = false;
    require(rip_pool_sample(p, 100, &t) == (g_failed ? RIP_ENOMEM : 0), "first call");
    g_fail_at = -1;
    if (g_failed && searched) {
      cut = true;
      cleared = false;
      g_on_fill = [&](size_t bytes) { cleared = cleared || bytes >= 16ull * n; };
      require(rip_pool_sample(p, 100, &t) == 0, "second call");
      g_on_fill = [](size_t) {};
    }
    g_on_launch = end_rounds;
    rip_pool_destroy(p);
    rip_graph_destroy(g);
    if (!g_failed) break;
  }
  require(cut, "no call failed after its search began");
}

// A kernel's limit of dynamic LDS belongs to the process: a call on a small
// graph must not lower what a call on a large one, in another thread, is about
// to launch with.
void lds_limit_is_kept() {
  std::map<std::string, int> limit;
  std::map<std::string, int> launched;
  bool lowered = false;
  g_on_attribute = [&](const std::string &kernel, int attribute, int value) {
    if (attribute != 8) return;   // hipFuncAttributeMaxDynamicSharedMemorySize
    lowered = lowered || value < limit[kernel];
    limit[kernel] = value;
  };
  g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t lds, void **args) {
    set_long(kernel, args, 1);
    if (lds == 0) return;
    ++launched[kernel];
    if (lds > static_cast<size_t>(limit[kernel])) require(false, kernel.c_str());
  };
  for (const uint32_t n : {400000u, 2000u}) {
    for (const int model : {RIP_IC, RIP_LT}) {
      rip_graph *g = ring(model, n);
      const uint32_t seed = 3;
      uint64_t act;
      uint32_t lev;
      require(rip_spread(g, &seed, 1, 1, 0, 1, &act, &lev) == 0, "spread");
      if (model == RIP_IC) {
        rip_pool *p;
        require(rip_pool_create(g, 1, &p) == 0, "pool");
        require(rip_pool_sample(p, 100, nullptr) == 0, "sample");
        rip_pool_destroy(p);
      }
      rip_graph_destroy(g);
    }
  }
  size_t both = 0;
  for (const auto &k : launched) both += k.second == 2 ? 1 : 0;
  require(both == 3, "the team and both spread kernels did not run on both graphs");
  require(!lowered, "a limit was lowered");
}

// With little device memory left, samplers take less scratch, not an error.
void scratch_fits_little_memory() {
  g_cus = 256;
  g_on_launch = [](const std::string &kernel, Dim3, Dim3, size_t, void **args) {
    set_long(kernel, args, 300);
  };
  const struct {
    const char *what;
    uint32_t n;
    uint64_t sets;
    size_t left;   // bytes
  } cases[] = {
      {"wave stage and grid", (1u << 20) + 1, 1000, 160u << 20},
      {"wave stage and teams", 1u << 20, 1000, 130u << 20},
      {"lanes, wave stage and teams", 1u << 20, 5000, 260u << 20},
  };
  for (const auto &c : cases) {
    rip_graph *g = ring(RIP_IC, c.n);
    rip_pool *p;
    require(rip_pool_create(g, 1, &p) == 0, "pool");
    g_memory = used() + c.left;
    require(rip_pool_sample(p, c.sets, nullptr) == 0, c.what);
    require(rip_pool_sample(p, c.sets, nullptr) == 0, c.what);
    g_memory = 64ull << 30;
    require(rip_pool_sample(p, c.sets, nullptr) == 0, c.what);
    rip_pool_destroy(p);
    rip_graph_destroy(g);
  }
}

// Counts need no scratch beside the counts themselves: they do not fail where
// there is no room for the buckets.
void counts_fit_little_memory() {
  const uint32_t n = 1000, size = 10;
  const uint64_t sets = 60000;
  rip_graph *g = ring(RIP_IC, n);
  rip_pool *p;
  require(rip_pool_create(g, 1, &p) == 0, "pool");
  std::vector<uint64_t> off(1, 0);
  std::vector<uint32_t> ver, counts(n);
  for (uint64_t s = 0; s < sets; ++s) {
    for (uint32_t i = 0; i < size; ++i) ver.push_back(s % (n - size) + i);
    off.push_back(ver.size());
  }
  require(rip_pool_append_host(p, sets, off.data(), ver.data()) == 0, "append");
  bool buckets = false, members = false;
  g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t, void **) {
    buckets = buckets || is(kernel, "bucket_count_kernel");
    members = members || is(kernel, "member_count_kernel");
  };
  g_memory = used() + (1u << 20);
  require(rip_pool_count(p, sets, counts.data()) == 0, "counts");
  require(members && !buckets, "not counted member by member");
  g_memory = 64ull << 30;
  require(rip_pool_count(p, sets, counts.data()) == 0, "counts");
  require(buckets, "not counted by bucket");
  rip_pool_destroy(p);
  rip_graph_destroy(g);
}

// A pool of `sets` sets of `size` vertices each, from a moving start.
rip_pool *runs(rip_graph *g, uint32_t n, uint64_t sets, uint32_t size) {
  rip_pool *p;
  require(rip_pool_create(g, 1, &p) == 0, "pool");
  std::vector<uint64_t> off(1, 0);
  std::vector<uint32_t> ver;
  for (uint64_t s = 0; s < sets; ++s) {
    for (uint32_t i = 0; i < size; ++i) ver.push_back(s * 7 % (n - size) + i);
    off.push_back(ver.size());
  }
  require(rip_pool_append_host(p, sets, off.data(), ver.data()) == 0, "append");
  return p;
}

int select(rip_pool *p, uint64_t sets, uint32_t k) {
  std::vector<uint32_t> seeds(k);
  uint32_t got;
  uint64_t covered;
  return rip_pool_select(p, sets, k, seeds.data(), &got, &covered);
}

// A few long sets are walked by as many workgroups as their members fill, as
// many short ones are.
void long_sets_fill_the_chip() {
  rip_graph *g = ring(RIP_IC, 100000);
  const struct {
    uint64_t sets;
    uint32_t size;
    uint32_t least, most;   // workgroups
  } cases[] = {{800, 1000, 100, 1024}, {100, 5000, 13, 1024}, {20, 10, 1, 3}, {60000, 10, 100, 1024}};
  for (const auto &c : cases) {
    rip_pool *p = runs(g, 100000, c.sets, c.size);
    int walks = 0;
    g_on_launch = [&](const std::string &kernel, Dim3 grid, Dim3 block, size_t lds, void **args) {
      end_rounds(kernel, grid, block, lds, args);
      for (const char *k : {"bucket_size", "bucket_deal", "member_count", "top_index"})
        if (is(kernel, k)) {
          ++walks;
          if (grid.x < c.least || grid.x > c.most) {
            printf("%s: %u workgroups for %llu sets of %u\n", kernel.c_str(), grid.x,
                   static_cast<unsigned long long>(c.sets), c.size);
            exit(1);
          }
        }
    };
    require(select(p, c.sets, 3) == 0, "select");
    require(walks >= 2, "no counts or index");
    g_on_launch = end_rounds;
    rip_pool_destroy(p);
  }
  rip_graph_destroy(g);
}

// Rounds whose list holds many members together run on the whole chip, also
// where the pool has few sets; pools of short sets stay with one workgroup.
void long_lists_go_wide() {
  rip_graph *g = ring(RIP_IC, 100000);
  const struct {
    uint64_t sets;
    uint32_t size;
    bool wide;
  } cases[] = {{1000, 300, true}, {1000, 20, false}, {4000, 20, false}, {5000, 20, true}};
  for (const auto &c : cases) {
    rip_pool *p = runs(g, 100000, c.sets, c.size);
    int wide = 0;
    g_on_launch = [&](const std::string &kernel, Dim3 grid, Dim3 block, size_t lds, void **args) {
      end_rounds(kernel, grid, block, lds, args);
      if (is(kernel, "top_rounds") && grid.x > 1) ++wide;
    };
    require(select(p, c.sets, 3) == 0, "select");
    require((wide != 0) == c.wide, c.wide ? "one workgroup for long lists" : "wide rounds for short lists");
    g_on_launch = end_rounds;
    rip_pool_destroy(p);
  }
  rip_graph_destroy(g);
}

// A selection whose passes yield a round or two and leave most sets there turns
// to the full index after two of them; one whose passes yield more goes on.
void poor_passes_end() {
  const uint32_t n = 100000;
  rip_graph *g = ring(RIP_IC, n);
  const struct {
    uint32_t rounds, covered;
    int least, most;   // passes
  } cases[] = {{1, 5, 2, 2}, {15, 150, 2, 2}, {20, 100, 8, 12}, {1, 600, 3, 12}};
  for (const auto &c : cases) {
    rip_pool *p = runs(g, n, 1000, 20);
    int passes = 0;
    bool full = false;
    g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t, void **args) {
      if (is(kernel, "top_rounds")) set_rounds(args, c.rounds, c.covered, 2);
      if (is(kernel, "top_index")) ++passes;
      full = full || is(kernel, "fill_inverted");
    };
    require(select(p, 1000, 500) == 0, "select");
    if (passes < c.least || passes > c.most || !full) {
      printf("%d passes of %u rounds, full index: %d\n", passes, c.rounds, full);
      exit(1);
    }
    g_on_launch = end_rounds;
    rip_pool_destroy(p);
  }
  rip_graph_destroy(g);
}

// However many seeds are asked for, no graph holds more than some 25,000 nodes.
void graphs_stay_bounded() {
  rip_graph *g = ring(RIP_IC, 20000);
  rip_pool *plain = runs(g, 20000, 1000, 20), *dense = runs(g, 20000, 500, 10000);
  int argmax = 0;
  g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t, void **args) {
    if (is(kernel, "top_rounds")) set_rounds(args, 0, 0, 2);   // no round among candidates
    if (is(kernel, "argmax_kernel")) ++argmax;
  };
  for (const auto &c : {std::make_pair(plain, 1000), std::make_pair(dense, 500)})
    for (const uint32_t k : {10u, 4096u, 60000u}) {
      argmax = 0;
      require(select(c.first, c.second, k) == 0, "select");
      require(argmax == static_cast<int>(k), "not a round per seed");
    }
  if (g_largest_graph < 4096 || g_largest_graph > 25000) {
    printf("%d launches in a graph\n", g_largest_graph);
    exit(1);
  }
  g_on_launch = end_rounds;
  rip_pool_destroy(plain);
  rip_pool_destroy(dense);
  rip_graph_destroy(g);
}

// Spread workgroups have as many threads as leave 16 waves to a CU, by how many
// of them it holds: one each where two bitmaps do not fit its 160 KiB of LDS.
void spread_fills_its_cus() {
  const struct {
    int model;
    uint32_t n;
    uint64_t replicas;
    uint32_t threads;
  } cases[] = {
      {RIP_IC, 700001, 8, 1024}, {RIP_IC, 700001, 4, 1024}, {RIP_IC, 1000003, 64, 1024},
      {RIP_IC, 600000, 8, 512},  {RIP_IC, 300000, 64, 256}, {RIP_IC, 2000, 8, 512},
      {RIP_LT, 400000, 8, 1024}, {RIP_LT, 280000, 8, 512},
  };
  for (const auto &c : cases) {
    rip_graph *g = ring(c.model, c.n);
    const uint32_t seed = 3;
    std::vector<uint64_t> act(c.replicas);
    std::vector<uint32_t> lev(c.replicas);
    uint32_t threads = 0;
    g_on_launch = [&](const std::string &kernel, Dim3, Dim3 block, size_t, void **) {
      if (is(kernel, "spread_")) threads = block.x;
    };
    require(rip_spread(g, &seed, 1, 1, 0, c.replicas, act.data(), lev.data()) == 0, "spread");
    if (threads != c.threads) {
      printf("%u threads for %llu replicas on %u vertices, not %u\n", threads,
             static_cast<unsigned long long>(c.replicas), c.n, c.threads);
      exit(1);
    }
    rip_graph_destroy(g);
  }
}

// A graph whose large sets the team sampler takes and one where the grid does
// share no autotuned setting, alike as they are.
void tuned_settings_part_at_the_team_line() {
  rip_tune t{};
  double ms;
  uint32_t tried = 0;
  rip_graph *above = ring(RIP_IC, (1u << 20) + 5), *alike = ring(RIP_IC, (1u << 20) + 9);
  rip_graph *below = ring(RIP_IC, (1u << 20) - 5);
  require(rip_autotune(above, 2000, 1, &t, &ms, &tried) == 0 && tried > 0, "tune");
  require(rip_autotune(alike, 2000, 0, &t, &ms, &tried) == 0 && tried == 0, "a graph alike was timed again");
  require(rip_autotune(below, 2000, 0, &t, &ms, &tried) == 0 && tried > 0,
          "a setting timed with the grid was taken over");
  rip_graph_destroy(above);
  rip_graph_destroy(alike);
  rip_graph_destroy(below);
}

// The autotuner's settings with the wave stage differ in what they run: each in
// turn made the fastest, the last has another output chunk, not another lane
// capacity, which those lanes do not heed.
void staged_settings_differ() {
  rip_graph *g = ring(RIP_IC, 5000);
  rip_tune t{};
  double ms;
  uint32_t tried = 0;
  int staged = 0;
  g_on_launch = [&](const std::string &kernel, Dim3, Dim3, size_t, void **) {
    int wait = is(kernel, "ic_lane_kernel") ? 40 : 0;
    if (is(kernel, "ic_short_kernel")) wait = 30 - 5 * ++staged;   // two a setting
    for (const auto end = std::chrono::steady_clock::now() + std::chrono::milliseconds(wait);
         std::chrono::steady_clock::now() < end;) {}
  };
  require(rip_autotune(g, 20000, 1, &t, &ms, &tried) == 0, "tune");
  g_on_launch = end_rounds;
  if (staged < 6 || !t.wave_stage || t.queue_cap != 64 || t.out_chunk != 1024) {
    printf("after %d calls: queue_cap %u, wave_stage %u, out_chunk %u\n", staged, t.queue_cap, t.wave_stage,
           t.out_chunk);
    exit(1);
  }
  rip_graph_destroy(g);
}

// What destroyed pools left to their graph goes back to the device when asked
// for; live pools keep theirs.
void idle_memory_is_given_back() {
  rip_graph *g = ring(RIP_IC, 5000);
  const size_t graph = used();
  rip_pool *live_pool = runs(g, 5000, 1000, 10);
  const size_t with_live = used();
  rip_pool *p = runs(g, 5000, 60000, 10);
  require(select(p, 60000, 5) == 0, "select");
  rip_pool_destroy(p);
  require(used() > with_live, "nothing was kept");
  require(rip_graph_trim(g) == 0, "trim");
  if (used() > with_live + 8192) {   // a stream kit's control words
    printf("%zu bytes after, %zu before\n", used(), with_live);
    exit(1);
  }
  require(select(live_pool, 1000, 5) == 0, "select");
  rip_pool_destroy(live_pool);
  require(rip_graph_trim(g) == 0, "trim");
  require(used() <= graph + 16384, "idle blocks are left");
  rip_graph_destroy(g);
  require(rip_graph_trim(nullptr) == RIP_EINVAL, "no graph");
}

}  // namespace

int main(int argc, char **argv) {
  const std::map<std::string, void (*)()> checks = {
      {"grid_scratch_after_failure", grid_scratch_after_failure},
      {"lds_limit_is_kept", lds_limit_is_kept},
      {"scratch_fits_little_memory", scratch_fits_little_memory},
      {"counts_fit_little_memory", counts_fit_little_memory},
      {"long_sets_fill_the_chip", long_sets_fill_the_chip},
      {"long_lists_go_wide", long_lists_go_wide},
      {"poor_passes_end", poor_passes_end},
      {"graphs_stay_bounded", graphs_stay_bounded},
      {"spread_fills_its_cus", spread_fills_its_cus},
      {"tuned_settings_part_at_the_team_line", tuned_settings_part_at_the_team_line},
      {"staged_settings_differ", staged_settings_differ},
      {"idle_memory_is_given_back", idle_memory_is_given_back},
  };
  const auto it = argc == 2 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  it->second();
  return 0;
}
