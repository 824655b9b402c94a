// Host check of what a failed device allocation leaves behind: the library on
// a HIP runtime made here, whose device memory is host memory, whose kernels do
// nothing, and whose allocations fail from the n-th of a call on.
//
// For every n: a small call, a larger one that fails, the small one again.  A
// buffer whose capacity still claims room after the failure would not be
// allocated by the last call, so there must be as many allocations alive as
// after the small calls alone (idle blocks aside, which a failure frees).
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "ripples_amd.h"

namespace {

struct Dim3 {
  uint32_t x, y, z;
};

std::set<void *> &live() {
  static std::set<void *> s;
  return s;
}

std::map<const void *, std::string> &kernels() {   // host function -> kernel name
  static std::map<const void *, std::string> m;
  return m;
}

long g_fail_at = -1;   // allocations left before they fail; < 0: never
bool g_failed = false;
int g_null = 0;        // copies and fills of a null buffer

struct {
  Dim3 grid, block;
  size_t lds;
  void *stream;
} g_call;

}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  kernels()[host] = name;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void *stream) {
  g_call = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *lds, void **stream) {
  *grid = g_call.grid;
  *block = g_call.block;
  *lds = g_call.lds;
  *stream = g_call.stream;
  return 0;
}
int hipLaunchKernel(const void *f, Dim3, Dim3, void **args, size_t, void *) {
  // the selection's rounds: its state (the first pointer) says that every set
  // is covered (word 10)
  if (kernels()[f].find("top_rounds_kernel") != std::string::npos)
    (**static_cast<uint32_t ***>(static_cast<void *>(args)))[10] = 1;
  return 0;
}
int hipMalloc(void **p, size_t bytes) {
  if (g_fail_at == 0) {
    g_failed = true;
    *p = nullptr;
    return 2;
  }
  if (g_fail_at > 0) --g_fail_at;
  *p = calloc(bytes, 1);
  live().insert(*p);
  return 0;
}
int hipFree(void *p) {
  live().erase(p);
  free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t bytes, unsigned) { return (*p = calloc(bytes, 1)) ? 0 : 2; }
int hipHostFree(void *p) {
  free(p);
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  if (d && s)
    memcpy(d, s, n);
  else if (n)
    ++g_null;
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) { return hipMemcpy(d, s, n, kind); }
int hipMemset(void *p, int v, size_t n) {
  if (p)
    memset(p, v, n);
  else if (n)
    ++g_null;
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t n, void *) { return hipMemset(p, v, n); }
int hipMemGetInfo(size_t *f, size_t *t) {
  *f = *t = 64ull << 30;
  return 0;
}
int hipDeviceTotalMem(size_t *t, int) {
  *t = 64ull << 30;
  return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
  *v = 4;
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *v, const void *, int, size_t) {
  *v = 2;
  return 0;
}
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 0;
  return 0;
}
static int handle(void **h) {
  *h = malloc(1);
  return 0;
}
int hipEventCreate(void **e) { return handle(e); }
int hipStreamCreateWithFlags(void **s, unsigned) { return handle(s); }
int hipStreamEndCapture(void *, void **g) { return handle(g); }
int hipGraphInstantiate(void **x, void *, void *, char *, size_t) { return handle(x); }
int hipEventDestroy(void *) { return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipStreamBeginCapture(void *, int) { return 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
int hipGraphLaunch(void *, void *) { return 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDevice(int *d) { return *d = 0; }
int hipGetDeviceCount(int *n) {
  *n = 1;
  return 0;
}
int hipGetLastError() { return 0; }
const char *hipGetErrorString(int) { return "out of memory"; }
}

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
// small; n < 0: without the large call.
size_t alive(const Case &c, long n, bool *failed) {
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
  require(c.call(g, p, false) == 0, c.name);
  if (n >= 0) {
    g_fail_at = n;
    g_failed = false;
    const int rc = c.call(g, p, true);
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

int sample(rip_pool *p, bool large, uint32_t sampler) {
  rip_tune t{};
  t.sampler = sampler;
  return rip_pool_sample(p, large ? 60000 : 100, &t);
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
  };
  int bad = 0;   // calls left without a buffer
  for (const Case &c : cases) {
    bool failed = false;
    const size_t want = alive(c, -1, &failed);
    long n = 0;
    for (failed = true; failed; ++n) {
      const size_t got = alive(c, n, &failed);
      if (failed && got < want) {
        printf("%s: %zu allocations after a failure of number %ld, %zu without\n", c.name, got, n, want);
        ++bad;
      }
    }
    printf("%s: %ld failures\n", c.name, n - 1);
    if (n < 2) ++bad;   // the large call must allocate
  }
  if (g_null) printf("%d copies or fills of a null buffer\n", g_null);
  return bad != 0 || g_null != 0;
}
