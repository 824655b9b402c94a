// Host check of what a failed device allocation leaves behind: the library on
// a HIP runtime (fake_hip.h) whose allocations fail from the n-th of a call on.
//
// For every n: a small call, a larger one that fails, the small one again; and
// a small one that fails, then again.  A buffer whose capacity still claims
// room after the failure would not be allocated by the last call, so there must
// be as many allocations alive as after the small calls alone (idle blocks
// aside, which a failure frees).
#include <functional>
#include <vector>

#include "fake_hip.h"
#include "ripples_amd.h"

namespace {

void require(bool ok, const char *what) {
  if (ok) return;
  printf("%s: %s\n", what, rip_last_error());
  exit(1);
}

// A graph, a pool of it, and a call of a small and of a large size.
struct Case {
  const char *name;
  int model;
  uint32_t n;
  std::function<void(rip_pool *)> fill;                    // the pool before the calls
  std::function<int(rip_graph *, rip_pool *, bool)> call;  // large or not
};

// Allocations alive after small, [large, failing from its n-th allocation on,]
// small; n < 0: without the large call; fresh: a small call in the place of
// the first two.
size_t alive(const Case &c, long n, bool fresh, bool *failed) {
  // in-neighbours v + 1 .. v + 4 of every v
  std::vector<uint64_t> index(c.n + 1);
  std::vector<uint32_t> edges;
  std::vector<float> w;
  for (uint32_t v = 0; v < c.n; ++v) {
    for (uint32_t d = 1; d <= 4; ++d) {
      edges.push_back((v + d) % c.n);
      w.push_back(0.2f);
    }
    index[v + 1] = edges.size();
  }
  rip_graph *g;
  rip_pool *p;
  require(rip_graph_create(0, c.model, c.n, edges.size(), index.data(), edges.data(), w.data(), &g) == 0, c.name);
  require(rip_pool_create(g, 1, &p) == 0, c.name);
  if (c.fill) c.fill(p);
  if (!fresh) require(c.call(g, p, false) == 0, c.name);
  if (n >= 0) {
    g_fail_at = n;
    g_failed = false;
    const int rc = c.call(g, p, !fresh);
    g_fail_at = -1;
    require(rc == (g_failed ? RIP_ENOMEM : 0), c.name);
    *failed = g_failed;
  }
  require(c.call(g, p, false) == 0, c.name);
  rip_graph *none;
  g_fail_at = 0;   // the idle blocks go
  require(rip_graph_create(0, c.model, c.n, edges.size(), index.data(), edges.data(), w.data(), &none) ==
              RIP_ENOMEM, c.name);
  g_fail_at = -1;
  const size_t count = live().size();
  rip_pool_destroy(p);
  rip_graph_destroy(g);
  if (!live().empty()) {
    printf("%s: %zu allocations left\n", c.name, live().size());
    exit(1);
  }
  return count;
}

// `sets` sets of `size` vertices each, from a moving start.
void append(rip_pool *p, uint32_t n, uint64_t sets, uint32_t size) {
  std::vector<uint64_t> off(1, 0);
  std::vector<uint32_t> ver;
  for (uint64_t s = 0; s < sets; ++s) {
    const uint32_t a = static_cast<uint32_t>(s * 7 % (n - size));
    for (uint32_t i = 0; i < size; ++i) ver.push_back(a + i);
    off.push_back(ver.size());
  }
  require(rip_pool_append_host(p, sets, off.data(), ver.data()) == 0, "append");
}

int select(rip_pool *p, uint64_t sets, uint32_t k) {
  std::vector<uint32_t> seeds(k);
  uint32_t got;
  uint64_t covered;
  return rip_pool_select(p, sets, k, seeds.data(), &got, &covered);
}

int sample(rip_pool *p, bool large, uint32_t sampler, uint32_t colors = 0) {
  rip_tune t{};
  t.sampler = sampler;
  t.colors = colors;
  return rip_pool_sample(p, large ? 60000 : 100, &t);
}

// The same when samples outgrow what the first kernels hold: the kernels that
// clear the count of them (word 3 of the control words) leave that many.
int sample_long(rip_pool *p, bool large, uint32_t sampler, uint32_t colors = 0) {
  g_on_launch = [large](const std::string &kernel, Dim3, Dim3, size_t, void **args) {
    for (const char *k : {"reset_lane_kernel", "reset_stage_kernel", "reset_wave_kernel", "reset_long_kernel"})
      if (kernel.find(k) != std::string::npos)
        (**static_cast<uint64_t ***>(static_cast<void *>(args)))[3] = large ? 40000 : 64;
  };
  const int rc = sample(p, large, sampler, colors);
  g_on_launch = end_rounds;
  return rc;
}

int spread(rip_graph *g, bool large) {
  const uint32_t seeds[] = {1, 2};
  uint64_t act[64];
  uint32_t lev[64];
  return rip_spread(g, seeds, 2, 1, 0, large ? 64 : 1, act, lev);
}

}  // namespace

int main() {
  const std::vector<Case> cases = {
      {"plain selection", RIP_IC, 2000, [](rip_pool *p) { append(p, 2000, 30000, 6); },
       [](rip_graph *, rip_pool *p, bool l) { return select(p, l ? 30000 : 10, l ? 90 : 3); }},
      {"dense selection", RIP_IC, 20000,
       [](rip_pool *p) { append(p, 20000, 500, 10000); },
       [](rip_graph *, rip_pool *p, bool l) { return select(p, l ? 500 : 450, l ? 9 : 3); }},
      {"coverage", RIP_IC, 2000, [](rip_pool *p) { append(p, 2000, 100, 6); },
       [](rip_graph *, rip_pool *p, bool l) {
         const std::vector<uint32_t> seeds(l ? 1000 : 2, 5);
         uint64_t covered;
         return rip_pool_coverage(p, 100, seeds.data(), static_cast<uint32_t>(seeds.size()), &covered);
       }},
      {"spread, IC", RIP_IC, 2000, nullptr, [](rip_graph *g, rip_pool *, bool l) { return spread(g, l); }},
      {"spread, LT", RIP_LT, 2000, nullptr, [](rip_graph *g, rip_pool *, bool l) { return spread(g, l); }},
      {"LT", RIP_LT, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample(p, l, 0); }},
      {"IC", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample(p, l, RIP_SAMPLER_AUTO); }},
      {"IC, waves", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample(p, l, RIP_SAMPLER_WAVE); }},
      {"IC, lanes", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample(p, l, RIP_SAMPLER_LANE); }},
      {"IC, colours", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample(p, l, RIP_SAMPLER_COLOUR); }},
      {"IC, grid", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample_long(p, l, RIP_SAMPLER_AUTO, 64); }},
      {"IC, teams", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample_long(p, l, RIP_SAMPLER_AUTO); }},
      {"IC, large by waves", RIP_IC, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample_long(p, l, RIP_SAMPLER_WAVE); }},
      {"LT, long walks", RIP_LT, 2000, nullptr, [](rip_graph *, rip_pool *p, bool l) { return sample_long(p, l, 0); }},
  };
  int bad = 0;   // calls left without a buffer
  for (const Case &c : cases) {
    bool failed = false;
    const size_t want = alive(c, -1, false, &failed);
    for (const bool fresh : {false, true}) {
      long n = 0;
      for (failed = true; failed; ++n) {
        const size_t got = alive(c, n, fresh, &failed);
        if (failed && got < want) {
          printf("%s: %zu allocations after a failure of number %ld%s, %zu without\n", c.name, got, n,
                 fresh ? " of the first call" : "", want);
          ++bad;
        }
      }
      printf("%s: %ld failures\n", c.name, n - 1);
      if (n < 2) ++bad;   // the call must allocate
    }
  }
  if (g_null) printf("%d copies or fills of a null buffer\n", g_null);
  return bad != 0 || g_null != 0;
}
