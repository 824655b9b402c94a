// Forward Monte Carlo spread of a seed set under IC or LT: the check of a
// seed set's influence (include/ripples/diffusion_simulation.h:73-178, driven
// by tools/simulator.cc:100-171), one replica per persistent workgroup at a
// time.
//
// Replica r draws from the sample stream r of the given seed (the same
// per-sample construction the samplers use): element 1 + f is the IC coin of
// forward edge f, live iff (x >> 40) < floor(w * 2^24); element 1 + v is the
// LT threshold of v, U = ((x >> 40) + 1) * 2^-24.  The forward CSR lists, for
// each u, the targets of the transposed entries with source u in transposed
// position order; it is built once per graph on first use.
//
// One replica per workgroup at a time, as many threads as leave no CU idle;
// the bitmap of active vertices (LT: and of candidates) is in LDS where it
// fits.
// IC: level-synchronous breadth-first search; a wave takes 64 frontier
// vertices, long rows by the whole wave, the edges of the short ones dealt
// out over its lanes.  Levels count the layers processed, the seed layer
// included.
// LT: per level, every vertex activated in the previous level adds the weight
// of each out-edge to its target's sum, in double precision and any order; a
// target that is inactive becomes a candidate (deduplicated by a bitmap).  A
// candidate activates when its active in-neighbours' weights, added in CSR
// order in float, reach its threshold: the double sum decides where it is
// further from the threshold than the float sum's rounding can be, and only
// else the row is read and added up in order.  Activations take effect at the
// end of the level.  Levels count the iterations, the last one (activating
// nothing) included.
//
// Both are bound by the latency of a level's dependent loads (vertex, record,
// edge, target), so what counts is lanes at work per CU: 256 replicas of 50
// seeds under IC with U[0,0.1] weights at 262,144 vertices take 3.6 ms (23.8
// with workgroups of 256 threads, a wave per vertex and the bitmap in device
// memory), and of 20 seeds under LT at 100,003 vertices 5.4 ms (180 when every
// level also added each candidate's row anew, one weight at a time).
#include <algorithm>
#include <vector>

#include "device_util.h"
#include "ic_common.h"
#include "internal.h"

namespace rip {
namespace {

struct alignas(16) FwdRec {
  uint64_t ja, jb;  // P^(1 + fbegin(u)): coin of u's first out-edge
  uint64_t ta, tb;  // P^(1 + u): LT threshold of u
  uint32_t begin, end;
  uint32_t pad[2];
};

__global__ void build_fwd_kernel(const unsigned long long *fidx, uint32_t n, Affine step,
                                 FwdRec *rec) {
  const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  FwdRec r;
  const Affine j = aff_pow(step, 1 + fidx[u]);
  const Affine t = aff_pow(step, 1 + static_cast<uint64_t>(u));
  r.ja = j.a;
  r.jb = j.b;
  r.ta = t.a;
  r.tb = t.b;
  r.begin = static_cast<uint32_t>(fidx[u]);
  r.end = static_cast<uint32_t>(fidx[u + 1]);
  r.pad[0] = r.pad[1] = 0;
  rec[u] = r;
}

struct SpreadParams {
  const FwdRec *fwd;
  const uint32_t *fdst;
  const uint32_t *fval;  // IC threshold or LT weight bits of each forward edge
  const VertexRec *vrec; // transposed rows (LT in-edges)
  const uint32_t *ids;
  const uint32_t *val;   // LT weight bits of each transposed edge
  uint32_t n;
  const uint32_t *seeds;
  uint32_t nseeds;
  uint64_t seed;
  uint64_t first;
  uint64_t count;
  unsigned long long *act_out;
  uint32_t *lev_out;
  unsigned long long *ctl;  // [0]: replica counter
  uint32_t *scratch;        // per workgroup: LT sums, queue, LT candidates, bitmaps, 2 words
  uint64_t per_wg;          // its words
  uint64_t words;           // 32-bit words per bitmap
  Affine step;
};

// Bitmaps in device memory are written with atomics, which complete in the
// L2: they are read past the vector L1.
template <bool kLds>
__device__ inline bool test_bit(const uint32_t *bm, uint32_t v) {
  const uint32_t w = kLds ? bm[v >> 5]
                          : __hip_atomic_load(&bm[v >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return (w >> (v & 31)) & 1u;
}

// Zeroes the word of v; barrier() makes it so for the workgroup's atomics.
template <bool kLds>
__device__ inline void clear_bits(uint32_t *bm, uint32_t v) {
  if (kLds)
    bm[v >> 5] = 0u;
  else
    __hip_atomic_store(&bm[v >> 5], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A workgroup barrier after the waves' own accesses to memory are done.
__device__ inline void barrier() {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
}

// Sets bit v; true when this call set it.
__device__ inline bool set_bit(uint32_t *bm, uint32_t v) {
  const uint32_t b = 1u << (v & 31);
  return !(atomicOr(&bm[v >> 5], b) & b);
}

// Appends v of the lanes with pred to list at *len (LDS): one atomic a wave.
__device__ inline void append(bool pred, uint32_t v, uint32_t *list, uint32_t *len) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(len, static_cast<uint32_t>(__popcll(m)));
  at = uniform_u32(at);
  if (pred) list[at + __popcll(m & lanes_below())] = v;
}

// The edges of up to 64 rows, lane l holding row (begin, deg): f(valid, j, e,
// k) with every lane, edge e = begin of row j + k.  Rows longer than 64 by the
// whole wave, 64 edges in order at a time; the others' edges dealt out.
template <typename F>
__device__ inline void for_row_edges(uint32_t begin, uint32_t deg, F &&f) {
  const uint32_t lane = lane_id();
  for (uint64_t m = __ballot(deg > 64); m; m &= m - 1) {
    const int j = __ffsll(static_cast<unsigned long long>(m)) - 1;
    const uint32_t b = __builtin_amdgcn_readlane(begin, j), d = __builtin_amdgcn_readlane(deg, j);
    for (uint32_t k0 = 0; k0 < d; k0 += 64) f(k0 + lane < d, static_cast<uint32_t>(j), b + k0 + lane, k0 + lane);
  }
  const uint32_t len = deg > 64 ? 0u : deg;
  const uint32_t incl = wave_inclusive_scan(len);
  const uint32_t total = uniform_u32(__shfl(incl, 63, 64));
  for (uint32_t i0 = 0; i0 < total; i0 += 64) {
    const uint32_t i = i0 + lane;
    uint32_t j = 0;   // the first row whose inclusive prefix passes i
#pragma unroll
    for (uint32_t s = 32; s > 0; s >>= 1)
      if (__shfl(incl, static_cast<int>(j + s - 1), 64) <= i) j += s;
    const int src = static_cast<int>(std::min(j, 63u));
    const uint32_t k = i - (__shfl(incl, src, 64) - __shfl(len, src, 64));
    f(i < total, static_cast<uint32_t>(src), __shfl(begin, src, 64) + k, k);
  }
}

// The workgroup's next replica (every thread gets it).
__device__ inline unsigned long long next_replica(unsigned long long *ctl, unsigned long long *s_r) {
  barrier();
  if (threadIdx.x == 0) *s_r = atomicAdd(&ctl[0], 1ull);
  __syncthreads();
  return *s_r;
}

// Takes the vertices [lo, hi) of a level, 64 to a wave or fewer when they are
// few: f(have, position) with every lane.
template <uint32_t NW, typename F>
__device__ inline void for_level(uint32_t lo, uint32_t hi, uint32_t *s_next, F &&f) {
  const uint32_t chunk = std::min(64u, std::max(4u, (hi - lo + NW - 1) / NW));
  for (;;) {
    uint32_t b = 0;
    if (lane_id() == 0) b = lo + atomicAdd(s_next, chunk);
    b = uniform_u32(b);
    if (b >= hi) break;
    f(lane_id() < std::min(chunk, hi - b), b + lane_id());
  }
}

template <int BT, bool kLds>
__global__ void __launch_bounds__(BT) spread_ic_kernel(SpreadParams P) {
  extern __shared__ uint32_t s_bits[];
  __shared__ Affine s_pow[64];   // P^j
  __shared__ uint32_t s_len, s_next;
  __shared__ unsigned long long s_r;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  uint32_t *queue = P.scratch + static_cast<uint64_t>(blockIdx.x) * P.per_wg;
  uint32_t *act = kLds ? s_bits : queue + P.n;
  if (tid < 64) s_pow[tid] = aff_pow(P.step, tid);
  if (kLds)
    for (uint32_t w = tid; w < P.words; w += BT) act[w] = 0;
  const Affine j64 = uniform_affine(aff_pow(P.step, 64));
  for (;;) {
    const unsigned long long r = next_replica(P.ctl, &s_r);
    if (r >= P.count) break;
    if (tid == 0) s_len = s_next = 0;
    __syncthreads();
    const uint64_t z = sample_z(P.seed, P.first + r);
    for (uint32_t i = tid; i < P.nseeds; i += BT) {
      const uint32_t v = P.seeds[i];
      if (set_bit(act, v)) queue[atomicAdd(&s_len, 1u)] = v;
    }
    __syncthreads();
    uint32_t lo = 0, hi = s_len, lev = 0;
    __syncthreads();
    while (lo < hi) {
      ++lev;
      for_level<BT / 64>(lo, hi, &s_next, [&](bool have, uint32_t at) {
        uint32_t begin = 0, deg = 0;
        uint64_t x0 = 0;   // coin of the row's first edge
        if (have) {
          const FwdRec fr = P.fwd[queue[at]];
          begin = fr.begin;
          deg = fr.end - fr.begin;
          x0 = fr.ja * z + fr.jb;
        }
        uint64_t xl = 0;   // long rows: the lane's coin, 64 edges further each time
        for_row_edges(begin, deg, [&](bool valid, uint32_t j, uint32_t f, uint32_t k) {
          // (every lane shuffles: the row's own lane may have no edge here)
          const uint64_t xr = __shfl(x0, static_cast<int>(j), 64);
          xl = k < 64 ? aff_apply(s_pow[k & 63u], xr) : aff_apply(j64, xl);
          const bool live = valid && static_cast<uint32_t>(xl >> 40) < P.fval[f];
          uint32_t v = 0;
          bool fresh = false;
          if (live) {
            v = P.fdst[f];
            fresh = !test_bit<kLds>(act, v) && set_bit(act, v);
          }
          append(fresh, v, queue, &s_len);
        });
      });
      __syncthreads();
      lo = hi;
      hi = s_len;
      if (tid == 0) s_next = 0;
      __syncthreads();
    }
    if (tid == 0) {
      P.act_out[r] = hi;
      P.lev_out[r] = lev;
    }
    for (uint32_t i = tid; i < hi; i += BT) clear_bits<kLds>(act, queue[i]);
  }
}

// Whether the weights of v's active in-neighbours, added in CSR order in
// float, reach its threshold; a wave for one candidate.
template <bool kLds>
__device__ inline bool lt_reaches(const SpreadParams &P, const uint32_t *act, uint32_t v, float th) {
  const uint32_t lane = lane_id();
  const VertexRec vr = P.vrec[v];
  float total = 0.0f;
  for (uint32_t e0 = vr.begin; e0 < vr.end; e0 += 64) {
    const uint32_t e = e0 + lane;
    const bool on = e < vr.end && test_bit<kLds>(act, P.ids[e]);
    const float wv = on ? __uint_as_float(P.val[e]) : 0.0f;
    for (uint64_t bal = __ballot(on); bal; bal &= bal - 1)
      total += __shfl(wv, __ffsll(static_cast<unsigned long long>(bal)) - 1, 64);
  }
  return total >= th;
}

// The sums are zero between replicas, or known not to be: one that met fewer than
// this share of n edges clears those of its targets as it ends, after any other
// all are cleared before the next.  1,024 replicas of 5 seeds that reach a
// handful of 2^22 vertices: 5.9 ms when each cleared them all, 0.12 this way; 512
// of 20 seeds on 2^18 vertices with weights of 0.3 to 0.9 a row 0.37 to 2.07 and
// 0.17 to 1.68.  Lines of n and n / 16 measured the same.
constexpr uint32_t kClearShare = 4;

template <int BT, bool kLds>
__global__ void __launch_bounds__(BT) spread_lt_kernel(SpreadParams P) {
  extern __shared__ uint32_t s_bits[];
  __shared__ uint32_t s_len, s_next, s_nc, s_edges;
  __shared__ unsigned long long s_r;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  // whether sums are left from the workgroup's last replica, of an earlier launch
  // perhaps
  uint32_t *left = P.scratch + static_cast<uint64_t>(blockIdx.x + 1) * P.per_wg - 2;
  bool dirty = *left != 0;
  double *sum = reinterpret_cast<double *>(P.scratch + static_cast<uint64_t>(blockIdx.x) * P.per_wg);
  uint32_t *queue = reinterpret_cast<uint32_t *>(sum + P.n);
  uint32_t *clist = queue + P.n;
  uint32_t *act = kLds ? s_bits : clist + P.n;
  uint32_t *cand = act + P.words;
  if (kLds)
    for (uint32_t w = tid; w < 2 * P.words; w += BT) act[w] = 0;
  for (;;) {
    const unsigned long long r = next_replica(P.ctl, &s_r);
    if (r >= P.count) break;
    if (tid == 0) s_len = s_next = s_nc = s_edges = 0;
    if (dirty)
      for (uint32_t v = tid; v < P.n; v += BT) sum[v] = 0.0;
    __syncthreads();
    const uint64_t z = sample_z(P.seed, P.first + r);
    for (uint32_t i = tid; i < P.nseeds; i += BT) {
      const uint32_t v = P.seeds[i];
      if (set_bit(act, v)) queue[atomicAdd(&s_len, 1u)] = v;
    }
    barrier();   // the zeroes are in place before the atomics
    uint32_t lo = 0, hi = s_len, lev = 0, edges = 0;
    __syncthreads();
    do {
      ++lev;
      // the last level's activations add to their targets' sums
      for_level<BT / 64>(lo, hi, &s_next, [&](bool have, uint32_t at) {
        uint32_t begin = 0, deg = 0;
        if (have) {
          const FwdRec fr = P.fwd[queue[at]];
          begin = fr.begin;
          deg = fr.end - fr.begin;
          edges += deg;
        }
        for_row_edges(begin, deg, [&](bool valid, uint32_t, uint32_t f, uint32_t) {
          uint32_t v = 0;
          bool fresh = false;
          if (valid) {
            v = P.fdst[f];
            if (!test_bit<kLds>(act, v)) {
              unsafeAtomicAdd(&sum[v], static_cast<double>(__uint_as_float(P.fval[f])));
              fresh = !test_bit<kLds>(cand, v) && set_bit(cand, v);
            }
          }
          append(fresh, v, clist, &s_nc);
        });
      });
      barrier();   // the sums are complete before they are read
      const uint32_t nc = s_nc;
      if (tid == 0) s_next = 0;
      // a lane per candidate; whole waves, for the doubtful ones
      for (uint32_t c0 = tid - lane; c0 < nc; c0 += BT) {
        const bool have = c0 + lane < nc;
        const uint32_t v = have ? clist[c0 + lane] : 0u;
        bool on = false, doubt = false;
        float th = 0.0f;
        if (have) {
          const FwdRec fr = P.fwd[v];
          th = u01(fr.ta * z + fr.tb);
          const double S = __hip_atomic_load(&sum[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          // k nonnegative floats added one by one: within (k - 1) 2^-24 of
          // the sum, relative, to first order; k is at most the in-degree
          const uint32_t d = P.vrec[v].end - P.vrec[v].begin;
          const double err = S * (static_cast<double>(d) + 2.0) * 0x1p-23;
          doubt = (P.vrec[v].flags & kRowScalar) != 0 || d >= (1u << 20) ||
                  !(S - err >= th || S + err < th);
          on = !doubt && S >= th;
        }
        for (uint64_t m = __ballot(doubt); m; m &= m - 1) {
          const int j = __ffsll(static_cast<unsigned long long>(m)) - 1;
          const bool reached = lt_reaches<kLds>(P, act, __builtin_amdgcn_readlane(v, j), __shfl(th, j, 64));
          if (static_cast<int>(lane) == j) on = reached;
        }
        append(on, v, queue, &s_len);
      }
      __syncthreads();
      const uint32_t len = s_len;
      for (uint32_t i = hi + tid; i < len; i += BT) set_bit(act, queue[i]);
      for (uint32_t i = tid; i < nc; i += BT) clear_bits<kLds>(cand, clist[i]);
      barrier();
      if (tid == 0) s_nc = 0;
      lo = hi;
      hi = len;
      __syncthreads();
    } while (lo < hi);
    if (tid == 0) {
      P.act_out[r] = hi;
      P.lev_out[r] = lev;
    }
    for (uint32_t i = tid; i < hi; i += BT) clear_bits<kLds>(act, queue[i]);
    // (next_replica() waits for these stores before the next atomics)
    edges = wave_sum(edges);
    if (lane == 0) atomicAdd(&s_edges, edges);
    __syncthreads();
    dirty = s_edges >= P.n / kClearShare;
    if (!dirty) {
      for_level<BT / 64>(0, hi, &s_next, [&](bool have, uint32_t at) {
        uint32_t begin = 0, deg = 0;
        if (have) {
          const FwdRec fr = P.fwd[queue[at]];
          begin = fr.begin;
          deg = fr.end - fr.begin;
        }
        for_row_edges(begin, deg, [&](bool valid, uint32_t, uint32_t f, uint32_t) {
          if (valid) sum[P.fdst[f]] = 0.0;
        });
      });
    }
  }
  if (tid == 0) *left = dirty ? 1u : 0u;
}

using SpreadKernel = void (*)(SpreadParams);

template <int BT>
SpreadKernel spread_kernel_of(int model, bool lds) {
  if (model == RIP_IC) return lds ? &spread_ic_kernel<BT, true> : &spread_ic_kernel<BT, false>;
  return lds ? &spread_lt_kernel<BT, true> : &spread_lt_kernel<BT, false>;
}

// Bytes of bitmaps a workgroup may keep in LDS, and of a CU's LDS; a workgroup
// takes some 1.2 KiB besides its bitmaps.
constexpr uint64_t kSpreadLds = 128u << 10;
constexpr uint64_t kCuLds = 160u << 10, kSpreadTables = 2u << 10;

}  // namespace

// Forward CSR of the graph (once): rows by source in transposed-position
// order, with the per-vertex stream jumps.
static void ensure_forward(rip_graph *g) {
  if (g->fwd.d_rec) return;
  const uint32_t n = g->n;
  const uint64_t m = g->m;
  std::vector<VertexRec> vr(n);
  std::vector<uint32_t> ids(m + kEdgePad), val(m + kEdgePad);
  RIP_HIP(hipMemcpy(vr.data(), g->d_vrec, sizeof(VertexRec) * n, hipMemcpyDeviceToHost));
  RIP_HIP(hipMemcpy(ids.data(), g->d_ids, sizeof(uint32_t) * (m + kEdgePad), hipMemcpyDeviceToHost));
  RIP_HIP(hipMemcpy(val.data(), g->d_val, sizeof(uint32_t) * (m + kEdgePad), hipMemcpyDeviceToHost));
  std::vector<unsigned long long> fidx(static_cast<size_t>(n) + 1, 0);
  for (uint64_t i = 0; i < m; ++i) ++fidx[ids[i] + 1];
  for (uint32_t u = 0; u < n; ++u) fidx[u + 1] += fidx[u];
  std::vector<unsigned long long> cur(fidx.begin(), fidx.end() - 1);
  std::vector<uint32_t> fdst(m + 1), fval(m + 1);
  for (uint32_t v = 0; v < n; ++v)
    for (uint32_t i = vr[v].begin; i < vr[v].end; ++i) {
      const unsigned long long f = cur[ids[i]]++;
      fdst[f] = v;
      fval[f] = val[i];  // IC: the edge's integer threshold
    }
  unsigned long long *d_fidx = nullptr;
  try {
    g->fwd.d_rec = dev_alloc<uint8_t>(sizeof(FwdRec) * n);
    g->fwd.d_dst = dev_alloc<uint32_t>(m + 1);
    g->fwd.d_val = dev_alloc<uint32_t>(m + 1);
    d_fidx = dev_alloc<unsigned long long>(static_cast<size_t>(n) + 1);
    RIP_HIP(hipMemcpy(d_fidx, fidx.data(), sizeof(unsigned long long) * (n + 1), hipMemcpyHostToDevice));
    RIP_HIP(hipMemcpy(g->fwd.d_dst, fdst.data(), sizeof(uint32_t) * (m + 1), hipMemcpyHostToDevice));
    RIP_HIP(hipMemcpy(g->fwd.d_val, fval.data(), sizeof(uint32_t) * (m + 1), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(build_fwd_kernel, dim3((n + 255) / 256), dim3(256), 0, 0, d_fidx, n, g->step,
                       reinterpret_cast<FwdRec *>(g->fwd.d_rec));
    RIP_HIP(hipGetLastError());
    RIP_HIP(hipDeviceSynchronize());
  } catch (...) {
    dev_free(d_fidx);
    dev_free(g->fwd.d_rec);
    dev_free(g->fwd.d_dst);
    dev_free(g->fwd.d_val);
    throw;
  }
  dev_free(d_fidx);
}

void spread_run(rip_graph *g, const uint32_t *seeds, uint32_t nseeds, uint64_t seed,
                uint64_t first, uint64_t count, uint64_t *activated, uint32_t *levels) {
  RIP_REQUIRE(nseeds == 0 || seeds, -1, "spread: seeds is NULL");
  RIP_REQUIRE(count == 0 || (activated && levels), -1, "spread: output arrays are NULL");
  for (uint32_t i = 0; i < nseeds; ++i)
    RIP_REQUIRE(seeds[i] < g->n, -1, "spread: seed vertex out of range");
  if (count == 0) return;
  std::lock_guard<std::mutex> lock(g->sampler_mu);
  RIP_HIP(hipSetDevice(g->device));
  ensure_forward(g);
  const uint64_t n = g->n, words = (n + 31) / 32;
  const bool ic = g->model == RIP_IC;
  const uint64_t bitmaps = 4 * words * (ic ? 1 : 2);   // bytes
  const bool lds = bitmaps <= kSpreadLds;
  // 32-bit words per workgroup: queue, bitmaps outside LDS; LT: sums, candidates
  // and, last, whether sums are left
  const uint64_t per_wg = ((ic ? n : 4 * n) + (lds ? 0 : bitmaps / 4) + 1) / 2 * 2 + 2;
  const uint64_t free_b = device_free_bytes();
  const uint64_t held = g->fwd.wgs * g->fwd.per_wg * 4;
  const uint64_t budget = std::min<uint64_t>((free_b + held) / 8, 16ull << 30);
  uint64_t wgs = std::max<uint64_t>(1, std::min<uint64_t>({count, 1024, budget / (per_wg * 4)}));
  if (g->fwd.per_wg != per_wg || g->fwd.wgs < wgs) {
    dev_free(g->fwd.d_scratch);
    g->fwd.wgs = 0;   // until the new scratch is there
    g->fwd.d_scratch = dev_alloc<uint32_t>(wgs * per_wg);
    RIP_HIP(hipMemset(g->fwd.d_scratch, 0, sizeof(uint32_t) * wgs * per_wg));
    g->fwd.wgs = wgs;
    g->fwd.per_wg = per_wg;
  }
  wgs = std::min<uint64_t>(wgs, g->fwd.wgs);
  unsigned long long *d_ctl = nullptr, *d_act = nullptr;
  uint32_t *d_lev = nullptr, *d_seeds = nullptr;
  try {
    d_ctl = dev_alloc<unsigned long long>(1);
    d_act = dev_alloc<unsigned long long>(count);
    d_lev = dev_alloc<uint32_t>(count);
    d_seeds = dev_alloc<uint32_t>(nseeds);
    RIP_HIP(hipMemset(d_ctl, 0, sizeof(unsigned long long)));
    if (nseeds)
      RIP_HIP(hipMemcpy(d_seeds, seeds, sizeof(uint32_t) * nseeds, hipMemcpyHostToDevice));
    SpreadParams P;
    P.fwd = reinterpret_cast<const FwdRec *>(g->fwd.d_rec);
    P.fdst = g->fwd.d_dst;
    P.fval = g->fwd.d_val;
    P.vrec = g->d_vrec;
    P.ids = g->d_ids;
    P.val = g->d_val;
    P.n = g->n;
    P.seeds = d_seeds;
    P.nseeds = nseeds;
    P.seed = seed;
    P.first = first;
    P.count = count;
    P.act_out = d_act;
    P.lev_out = d_lev;
    P.ctl = d_ctl;
    P.scratch = g->fwd.d_scratch;
    P.per_wg = per_wg;
    P.words = words;
    P.step = g->step;
    // 16 waves to a CU: as many threads per workgroup as its share of them,
    // by how many workgroups there are and how many bitmaps fit (512 replicas
    // under IC, U[0,0.1], on 1,000,003 vertices, one bitmap to a CU: 52.5 ms
    // with 512 threads, 30.4 with 1024)
    const uint32_t lds_bytes = lds ? static_cast<uint32_t>(bitmaps) : 0u;
    const uint64_t per_cu = std::min<uint64_t>((wgs + cu_count() - 1) / cu_count(),
                                               lds_bytes ? kCuLds / (lds_bytes + kSpreadTables) : 4);
    const uint32_t bt = per_cu <= 1 ? 1024u : per_cu <= 3 ? 512u : 256u;
    const SpreadKernel kernel = bt == 1024   ? spread_kernel_of<1024>(g->model, lds)
                                : bt == 512 ? spread_kernel_of<512>(g->model, lds)
                                            : spread_kernel_of<256>(g->model, lds);
    // the limit belongs to the process: one value for every graph, as calls on
    // others may be about to launch
    RIP_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(kSpreadLds)));
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(wgs)), dim3(bt), lds_bytes, 0, P);
    RIP_HIP(hipGetLastError());
    RIP_HIP(hipDeviceSynchronize());
    std::vector<unsigned long long> a(count);
    RIP_HIP(hipMemcpy(a.data(), d_act, sizeof(unsigned long long) * count, hipMemcpyDeviceToHost));
    RIP_HIP(hipMemcpy(levels, d_lev, sizeof(uint32_t) * count, hipMemcpyDeviceToHost));
    for (uint64_t i = 0; i < count; ++i) activated[i] = a[i];
  } catch (...) {
    dev_free(d_ctl);
    dev_free(d_act);
    dev_free(d_lev);
    dev_free(d_seeds);
    throw;
  }
  dev_free(d_ctl);
  dev_free(d_act);
  dev_free(d_lev);
  dev_free(d_seeds);
}

}  // namespace rip
