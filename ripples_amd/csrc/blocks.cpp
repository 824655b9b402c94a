// Idle device blocks and stream kits of a graph's pools (internal.h).
//
// A driver allocates its pools anew on every call, and a pool's buffers grow
// as its sets do: 46 pairs of hipMalloc and hipFree in an IMM run under LT on
// 2^20 vertices, 51 on R-MAT scale 22 under weighted cascade, tens to hundreds
// of microseconds for each large block, and every hipFree waits for the whole
// device, other pools' streams included.  So blocks that a pool gives up wait
// here for the next pool of the same graph: 12.4 ms to 5.1 and 44 to 33 ms for
// those two runs, 66 to 33 ms for twelve queries served together.
#include <algorithm>
#include <set>

#include "internal.h"

namespace rip {
namespace {

// Idle memory a graph may hold: a 64th of the device's (4.5 of 288 GB), in at
// most this many blocks; pools of a few gigabytes find their buffers again.
constexpr uint64_t kIdleShare = 64;
constexpr size_t kIdleBlocks = 256;
constexpr size_t kIdleKits = 8;

struct Registry {
  std::mutex mu;
  std::set<BlockCache *> all;
};

// Never destroyed: objects may outlive static destruction.
Registry &registry() {
  static Registry *r = new Registry;
  return *r;
}

}  // namespace

BlockCache::BlockCache(int device) : device_(device) {
  limit_ = device_total_bytes(device) / kIdleShare;
  std::lock_guard<std::mutex> hold(registry().mu);
  registry().all.insert(this);
}

BlockCache::~BlockCache() {
  {
    std::lock_guard<std::mutex> hold(registry().mu);
    registry().all.erase(this);
  }
  close();
}

void *BlockCache::take(size_t bytes) {
  {
    std::lock_guard<std::mutex> hold(mu_);
    // the smallest idle block that fits, at most a quarter larger
    auto best = idle_.end();
    for (auto it = idle_.begin(); it != idle_.end(); ++it)
      if (it->bytes >= bytes && it->bytes <= bytes + bytes / 4 + 4096 &&
          (best == idle_.end() || it->bytes < best->bytes))
        best = it;
    if (best != idle_.end()) {
      void *p = best->p;
      lent_[p] = best->bytes;
      idle_bytes_ -= best->bytes;
      idle_.erase(best);
      return p;
    }
  }
  void *p = device_malloc(bytes);
  std::lock_guard<std::mutex> hold(mu_);
  lent_[p] = bytes;
  return p;
}

void BlockCache::give(void *p, bool keep) {
  std::vector<void *> drop;
  {
    std::lock_guard<std::mutex> hold(mu_);
    const auto it = lent_.find(p);
    const size_t bytes = it == lent_.end() ? 0 : it->second;
    if (it != lent_.end()) lent_.erase(it);
    if (!keep || closed_ || bytes == 0 || bytes > limit_) {
      drop.push_back(p);
    } else {
      idle_.push_back({p, bytes});
      idle_bytes_ += bytes;
      // the longest idle leave first
      while (idle_bytes_ > limit_ || idle_.size() > kIdleBlocks) {
        drop.push_back(idle_.front().p);
        idle_bytes_ -= idle_.front().bytes;
        idle_.pop_front();
      }
    }
  }
  for (void *d : drop) (void)hipFree(d);
}

bool BlockCache::take_kit(StreamKit *kit) {
  std::lock_guard<std::mutex> hold(mu_);
  if (kits_.empty()) return false;
  *kit = kits_.back();
  kits_.pop_back();
  return true;
}

bool BlockCache::give_kit(const StreamKit &kit) {
  std::lock_guard<std::mutex> hold(mu_);
  if (closed_ || kits_.size() >= kIdleKits) return false;
  kits_.push_back(kit);
  return true;
}

void BlockCache::release() {
  std::list<Block> drop;
  {
    std::lock_guard<std::mutex> hold(mu_);
    drop.swap(idle_);
    idle_bytes_ = 0;
  }
  for (const Block &b : drop) (void)hipFree(b.p);
}

void BlockCache::close() {
  std::vector<StreamKit> kits;
  {
    std::lock_guard<std::mutex> hold(mu_);
    closed_ = true;
    kits.swap(kits_);
  }
  release();
  for (StreamKit &k : kits) kit_destroy(k);
}

size_t BlockCache::idle_bytes() {
  std::lock_guard<std::mutex> hold(mu_);
  return idle_bytes_;
}

// Runs f on every cache of a device.
template <typename F>
static void each_cache(int device, F &&f) {
  std::lock_guard<std::mutex> hold(registry().mu);
  for (BlockCache *c : registry().all)
    if (c->device() == device) f(c);
}

void *device_malloc(size_t bytes) {
  void *p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e != hipSuccess) {
    // the idle blocks of this device's graphs go first
    int dev = 0;
    (void)hipGetLastError();
    (void)hipGetDevice(&dev);
    each_cache(dev, [](BlockCache *c) { c->release(); });
    e = hipMalloc(&p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();   // or the next call's launch check finds it
    throw Error(-2, std::string("hipMalloc of ") + std::to_string(bytes) +
                        " bytes failed: " + hipGetErrorString(e));
  }
  return p;
}

uint64_t device_total_bytes(int device) {
  size_t total_b = 0;
  RIP_HIP(hipDeviceTotalMem(&total_b, device));
  return total_b;
}

uint64_t device_free_bytes() {
  size_t free_b = 0, total_b = 0;
  RIP_HIP(hipMemGetInfo(&free_b, &total_b));
  int dev = 0;
  RIP_HIP(hipGetDevice(&dev));
  uint64_t idle = 0;
  each_cache(dev, [&](BlockCache *c) { idle += c->idle_bytes(); });
  return std::min<uint64_t>(total_b, free_b + idle);
}

void kit_create(StreamKit *k) {
  RIP_HIP(hipStreamCreateWithFlags(&k->stream, hipStreamNonBlocking));
  for (hipEvent_t &e : k->ev) RIP_HIP(hipEventCreate(&e));
  k->d_ctl = dev_alloc<unsigned long long>(kCtlWords);
  // pinned, so reading the control words back after a launch is one DMA
  // rather than a copy staged through a driver buffer
  RIP_HIP(hipHostMalloc(reinterpret_cast<void **>(&k->h_ctl),
                        sizeof(unsigned long long) * kCtlWords, hipHostMallocDefault));
}

void kit_destroy(StreamKit &k) {
  dev_free(k.d_ctl);
  if (k.h_ctl) (void)hipHostFree(k.h_ctl);
  for (hipEvent_t e : k.ev)
    if (e) (void)hipEventDestroy(e);
  if (k.stream) (void)hipStreamDestroy(k.stream);
  k = StreamKit{};
}

}  // namespace rip
