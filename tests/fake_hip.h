// A HIP runtime for host checks of the library: device memory is host memory,
// kernels do nothing, and what the library asks of the runtime can be limited
// and watched.  Include it in one file, linked with -rdynamic, so that the
// library's calls find these definitions before the real ones.
#pragma once

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>

namespace {

struct Dim3 {
  uint32_t x, y, z;
};

std::map<void *, size_t> &live() {   // device allocations and their sizes
  static std::map<void *, size_t> m;
  return m;
}

std::map<const void *, std::string> &kernels() {   // host function -> kernel name
  static std::map<const void *, std::string> m;
  return m;
}

long g_fail_at = -1;   // allocations left before they fail; < 0: never
bool g_failed = false;
int g_null = 0;        // copies and fills of a null buffer
size_t g_memory = 64ull << 30;   // device memory there is
int g_cus = 4;                   // compute units
int g_last = 0;                  // the error that hipGetLastError returns next

size_t used() {
  size_t bytes = 0;
  for (const auto &b : live()) bytes += b.second;
  return bytes;
}

struct {
  Dim3 grid, block;
  size_t lds;
  void *stream;
} g_call;

// Ends a pass of the selection's rounds: their state (the first pointer of
// top_rounds_kernel) gets the rounds done (word 8), the sets they cover (9) and
// why they ended (10; 1: every set is covered, 2: the candidates ran out).
void set_rounds(void **args, uint32_t rounds, uint32_t covered, uint32_t why) {
  uint32_t *state = **static_cast<uint32_t ***>(static_cast<void *>(args));
  state[8] = rounds;
  state[9] = covered;
  state[10] = why;
}

// A kernel launch and its arguments; the default covers every set at once.
void end_rounds(const std::string &kernel, Dim3, Dim3, size_t, void **args) {
  if (kernel.find("top_rounds_kernel") != std::string::npos) set_rounds(args, 0, 0, 1);
}
std::function<void(const std::string &, Dim3, Dim3, size_t, void **)> g_on_launch = end_rounds;
int g_captured = -1;             // launches of the capture under way; < 0: none
int g_largest_graph = 0;         // launches of the largest capture
std::function<void(const std::string &, int, int)> g_on_attribute = [](const std::string &, int, int) {};
std::function<void(size_t)> g_on_fill = [](size_t) {};   // bytes of a fill of device memory

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
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t lds, void *) {
  if (g_captured >= 0) ++g_captured;
  g_on_launch(kernels()[f], grid, block, lds, args);
  return 0;
}
int hipMalloc(void **p, size_t bytes) {
  if (g_fail_at == 0 || used() + bytes > g_memory) {
    g_failed = true;
    *p = nullptr;
    return g_last = 2;
  }
  if (g_fail_at > 0) --g_fail_at;
  *p = calloc(bytes, 1);
  live()[*p] = bytes;
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
  g_on_fill(n);
  if (p)
    memset(p, v, n);
  else if (n)
    ++g_null;
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t n, void *) { return hipMemset(p, v, n); }
int hipMemGetInfo(size_t *f, size_t *t) {
  *f = g_memory - used();
  *t = 64ull << 30;
  return 0;
}
int hipDeviceTotalMem(size_t *t, int) {
  *t = 64ull << 30;
  return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
  *v = g_cus;
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
int hipStreamEndCapture(void *, void **g) {
  if (g_captured > g_largest_graph) g_largest_graph = g_captured;
  g_captured = -1;
  return handle(g);
}
int hipGraphInstantiate(void **x, void *, void *, char *, size_t) { return handle(x); }
int hipEventDestroy(void *) { return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipStreamBeginCapture(void *, int) { return g_captured = 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
int hipGraphLaunch(void *, void *) { return 0; }
int hipFuncSetAttribute(const void *f, int attribute, int value) {
  g_on_attribute(kernels()[f], attribute, value);
  return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDevice(int *d) { return *d = 0; }
int hipGetDeviceCount(int *n) {
  *n = 1;
  return 0;
}
int hipGetLastError() {   // an error stays until it is asked for
  const int e = g_last;
  g_last = 0;
  return e;
}
const char *hipGetErrorString(int) { return "out of memory"; }
}
