// Seed selection of plain pools among the vertices with the most sets.
//
// Greedy max coverage (FindMostInfluentialSet,
// include/ripples/find_most_influential.h:85-174, lowest-id ties) only ever
// needs the counts of vertices that can still be the maximum.  Counts never
// grow, so with the kTopMax vertices of largest count as candidates and a
// bound no other vertex's key passes, the rounds run on the candidates alone
// until the best of them falls below the bound:
//   1. counts[v] of every vertex (count_plain: by vertex bucket in LDS);
//   2. the candidates: a histogram of the counts in bins of 1/64 of their
//      size gives the bins that hold at most kTopMax vertices together; when
//      room is left and the next bin is a single value, its lowest ids too;
//   3. per set a record of the candidates it holds (16-bit ranks), and per
//      candidate the sets that hold it;
//   4. rounds: the sets of the round's seed not covered yet are marked and
//      the counts of the candidates they hold drop.  A round whose seed lists
//      many sets runs on the whole GPU, a launch each; the last workgroup of
//      the launch goes on with the rounds of short lists by itself, the counts
//      in LDS, up to the next long one.
// When the best candidate falls below the bound, counts and candidates are
// taken anew over the uncovered sets and the rounds go on.  Every set is
// killed at most once, and a kill touches its candidate members only: of
// 60M set members on R-MAT scale 22 weighted cascade about a tenth.
#include <algorithm>
#include <vector>

#include "device_util.h"
#include "internal.h"
#include "select_common.h"

namespace rip {
namespace {

constexpr uint32_t kBT = 256;
// Candidates at a time.  More of them mean fewer passes over the pool (a
// restart each time the best falls below the bound) but longer lists of sets
// already covered: IMM on R-MAT scale 22 weighted cascade (k = 200) took 56,
// 47, 45.5 and 44.5 ms with 8192, 4096, 2048 and 1024, with 512 as with 1024.
constexpr uint32_t kTopMax = 1024;

// ------------------------------------------------------------------ counts
// Counts through vertex buckets of 2^14: the members are dealt to their
// buckets as 16-bit offsets, each bucket is counted in LDS, and the counts
// reach memory with one atomic per vertex and slice instead of one per
// member (hub counters take hundreds of thousands of members).
constexpr uint32_t kBucketBits = 14;
constexpr uint32_t kBucketWidth = 1u << kBucketBits;
constexpr uint32_t kMaxBuckets = 2048;
constexpr uint32_t kSlice = 1u << 16;       // members a workgroup counts
constexpr uint64_t kBucketMin = 1ull << 19; // members from which the buckets pay
constexpr uint32_t kCountBT = 512;

// Sets a wave walks at a time: 64, fewer (a power of two) while the chip is not
// full and a wave keeps four members a lane.  With 64 everywhere a pool of a few
// long sets was walked by a few workgroups: the counts of 820 sets of 1100 took
// 1.90 ms (0.18 now), those of 10,000 of 205 (U[0,0.1], 4096 vertices) 0.56
// (0.11) and a selection on them 2.5 ms.
constexpr uint64_t kFullBlocks = 512;
inline uint32_t wave_sets(uint64_t num_sets, uint64_t total) {
  uint32_t step = 64;
  while (step > 1 && num_sets < kFullBlocks * (kCountBT / 64) * step &&
         total * step > 512 * num_sets)
    step /= 2;
  return step;
}

// The sets of a block of `blocks`: an even share, rounded up to whole waves.
__device__ inline uint64_t share_of(uint64_t num_sets, uint32_t blocks, uint32_t step) {
  return ((num_sets + blocks - 1) / blocks + step - 1) / step * step;
}

// f(member, set) over the block's share of sets [0, num_sets), `step` to a wave
// at a time, covered ones (covered != nullptr) left out.
template <int BT, typename F>
__device__ inline void for_block_members(const unsigned long long *set_off,
                                         const uint32_t *set_len, const uint32_t *data,
                                         uint64_t num_sets, uint32_t step,
                                         const uint8_t *covered, uint32_t (*s_pre)[65],
                                         unsigned long long (*s_off)[64], F &&f) {
  const uint32_t lane = lane_id(), wid = threadIdx.x >> 6;
  const uint64_t per = share_of(num_sets, gridDim.x, step);
  const uint64_t sb = blockIdx.x * per;
  const uint64_t se = sb + per < num_sets ? sb + per : num_sets;
  for (uint64_t w = sb + wid * step; w < se; w += BT / 64 * step) {
    const uint64_t s = w + lane;
    const bool live = lane < step && s < se && !(covered && covered[s]);
    for_each_run_element(live ? set_off[s] : 0ull, live ? set_len[s] : 0u, data, s_pre[wid],
                         s_off[wid], [&](uint32_t v, uint32_t j) { f(v, w + j); });
  }
}

// Members of each bucket (bcnt), and where the block's own start within each
// (where[block][bucket]).
__global__ void __launch_bounds__(kCountBT)
bucket_size_kernel(const unsigned long long *set_off, const uint32_t *set_len,
                   const uint32_t *data, uint64_t num_sets, uint32_t step, const uint8_t *covered,
                   uint32_t buckets, uint32_t *bcnt, uint32_t *where) {
  __shared__ uint32_t hist[kMaxBuckets];
  __shared__ uint32_t s_pre[kCountBT / 64][65];
  __shared__ unsigned long long s_off[kCountBT / 64][64];
  for (uint32_t b = threadIdx.x; b < buckets; b += kCountBT) hist[b] = 0;
  __syncthreads();
  for_block_members<kCountBT>(set_off, set_len, data, num_sets, step, covered, s_pre, s_off,
                              [&](uint32_t v, uint64_t) { atomicAdd(&hist[v >> kBucketBits], 1u); });
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < buckets; b += kCountBT)
    where[static_cast<uint64_t>(blockIdx.x) * buckets + b] = hist[b] ? atomicAdd(&bcnt[b], hist[b]) : 0u;
}

// One block: bstart[b] = members of the buckets before b, sstart[b] = their
// slices, for b in [0, buckets].
__global__ void __launch_bounds__(1024) bucket_scan_kernel(const uint32_t *bcnt, uint32_t buckets,
                                                           uint32_t *bstart, uint32_t *sstart) {
  __shared__ uint32_t s_tmp[1024 / 64];
  uint32_t run = 0, srun = 0;
  for (uint32_t b0 = 0; b0 < buckets; b0 += 1024) {
    const uint32_t b = b0 + threadIdx.x;
    const uint32_t c = b < buckets ? bcnt[b] : 0u;
    uint32_t tot, stot;
    const uint32_t pre = block_exclusive_scan<1024>(c, s_tmp, &tot);
    const uint32_t spre = block_exclusive_scan<1024>((c + kSlice - 1) / kSlice, s_tmp, &stot);
    if (b < buckets) {
      bstart[b] = run + pre;
      sstart[b] = srun + spre;
    }
    run += tot;
    srun += stot;
  }
  if (threadIdx.x == 0) {
    bstart[buckets] = run;
    sstart[buckets] = srun;
  }
}

// Each member's offset in its bucket to part[], the block's own after where.
__global__ void __launch_bounds__(kCountBT)
bucket_deal_kernel(const unsigned long long *set_off, const uint32_t *set_len,
                   const uint32_t *data, uint64_t num_sets, uint32_t step, const uint8_t *covered,
                   uint32_t buckets, const uint32_t *bstart, const uint32_t *where,
                   uint16_t *part) {
  __shared__ uint32_t cur[kMaxBuckets];
  __shared__ uint32_t s_pre[kCountBT / 64][65];
  __shared__ unsigned long long s_off[kCountBT / 64][64];
  for (uint32_t b = threadIdx.x; b < buckets; b += kCountBT)
    cur[b] = bstart[b] + where[static_cast<uint64_t>(blockIdx.x) * buckets + b];
  __syncthreads();
  for_block_members<kCountBT>(set_off, set_len, data, num_sets, step, covered, s_pre, s_off,
                              [&](uint32_t v, uint64_t) {
                                part[atomicAdd(&cur[v >> kBucketBits], 1u)] =
                                    static_cast<uint16_t>(v & (kBucketWidth - 1));
                              });
}

// Block i counts slice i: its vertices' counts by LDS atomics, then one
// global atomic per vertex met.
__global__ void __launch_bounds__(kCountBT)
bucket_count_kernel(const uint16_t *part, const uint32_t *bstart, const uint32_t *sstart,
                    uint32_t buckets, uint32_t n, uint32_t *counts) {
  __shared__ uint32_t hist[kBucketWidth];
  if (blockIdx.x >= sstart[buckets]) return;   // block-uniform
  uint32_t lo = 0, hi = buckets;
  while (lo < hi) {                            // the last bucket starting at or before this slice
    const uint32_t mid = (lo + hi) >> 1;
    if (sstart[mid + 1] <= blockIdx.x) lo = mid + 1;
    else hi = mid;
  }
  const uint32_t v0 = lo << kBucketBits;
  const uint32_t width = n - v0 < kBucketWidth ? n - v0 : kBucketWidth;
  const uint32_t b = bstart[lo] + (blockIdx.x - sstart[lo]) * kSlice;
  const uint32_t e = min(b + kSlice, bstart[lo + 1]);
  for (uint32_t i = threadIdx.x; i < width; i += kCountBT) hist[i] = 0;
  __syncthreads();
  for (uint32_t i = b + threadIdx.x; i < e; i += kCountBT * 4) {
    uint32_t v[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) v[u] = i + u * kCountBT < e ? part[i + u * kCountBT] : width;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u)
      if (v[u] < width) atomicAdd(&hist[v[u]], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < width; i += kCountBT)
    if (hist[i]) atomicAdd(&counts[v0 + i], hist[i]);
}

// Small pools: one atomic per member.
__global__ void __launch_bounds__(kCountBT)
member_count_kernel(const unsigned long long *set_off, const uint32_t *set_len,
                    const uint32_t *data, uint64_t num_sets, uint32_t step,
                    const uint8_t *covered, uint32_t *counts) {
  __shared__ uint32_t s_pre[kCountBT / 64][65];
  __shared__ unsigned long long s_off[kCountBT / 64][64];
  for_block_members<kCountBT>(set_off, set_len, data, num_sets, step, covered, s_pre, s_off,
                              [&](uint32_t v, uint64_t) { atomicAdd(&counts[v], 1u); });
}

__global__ void zero_u32_kernel(uint32_t *p, uint64_t n) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    p[i] = 0;
}

// -------------------------------------------------------------- candidates
// Words of the device state (TopState::w) the kernels below share.
enum : int {
  kTopBin = 0,     // counts in bins above this one are candidates
  kTopTie,         // count value whose lowest ids join them (0: none)
  kTopRoom,        // how many of those there is room for
  kTopTieEnd,      // ids below this join
  kTopBound,       // no other vertex has a count above this
  kTopN,           // candidates
  kTopMembers,     // ranks in the members array
  kTopDone,        // blocks of the current kernel that finished
  kTopRound,       // rounds done
  kTopCovered,     // sets covered by them
  kTopStop,        // why the rounds ended: kStopNone, kStopAll, kStopBound
  kTopRank,        // the candidate of the next round, its list long
  kTopGain,        // and its count
  kTopWords
};
enum : uint32_t { kStopNone = 0, kStopAll = 1, kStopBound = 2 };

constexpr uint32_t kBins = 28 * 64;   // 64 per power of two from 64 up: one per value below 128
constexpr uint32_t kTile = 1024;      // vertices per tile: ties join by whole tiles

// Monotone in the count: counts below 64 have a bin each, larger ones share
// one with the counts of the same leading seven bits.
__device__ inline uint32_t count_bin(uint32_t c) {
  if (c < 64) return c;
  const uint32_t e = 31 - __clz(static_cast<int>(c));   // 6..31
  return (e - 5) * 64 + ((c >> (e - 6)) & 63u);
}

// The largest count of bin b.
__device__ inline uint32_t bin_top(uint32_t b) {
  if (b < 64) return b;
  const uint32_t e = b / 64 + 5;
  return static_cast<uint32_t>(((static_cast<uint64_t>(64 + (b & 63u)) + 1) << (e - 6)) - 1);
}

struct TopState {
  uint32_t w[kTopWords];
  uint32_t hist[kBins];
};

// Whether this is the last block of the launch to get here (every thread
// gets the answer).  What the other blocks wrote before is then there: each
// waits for its waves' accesses and writes back its XCD's L2 before it counts
// itself done, and the last one drops what its own L1 and L2 hold after the
// count, so that plain loads (the rounds' records) find it as atomic ones do.
// One fence per block, not per wave: an agent-scope release writes back the
// XCD's L2, and 8,000 of them took 0.13 ms.
__device__ inline bool last_block(uint32_t *done, uint32_t *s_flag) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    const uint32_t d = atomicAdd(done, 1u);
    *s_flag = d + 1 == gridDim.x;
    if (*s_flag) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      atomicExch(done, 0u);
    }
  }
  __syncthreads();
  return *s_flag != 0;
}

__device__ inline uint32_t load_u32(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr uint32_t kPickBT = 1024;    // a thread per vertex of a tile
constexpr uint32_t kHistPer = 4;      // vertices per thread and step of the histogram

// Histogram of the counts of [0, n) over the bins; the last block picks the
// bins above which at most kTopMax vertices lie.
__global__ void __launch_bounds__(kPickBT) top_hist_kernel(const uint32_t *counts, uint32_t n,
                                                           TopState *st) {
  __shared__ uint32_t hist[kBins];
  __shared__ uint32_t s_tmp[kPickBT / 64];
  __shared__ uint32_t s_flag, s_cut, s_sum;
  for (uint32_t i = threadIdx.x; i < kBins; i += kPickBT) hist[i] = 0;
  __syncthreads();
  for (uint64_t v0 = static_cast<uint64_t>(blockIdx.x) * kHistPer * kPickBT; v0 < n;
       v0 += static_cast<uint64_t>(gridDim.x) * kHistPer * kPickBT) {
    uint32_t c[kHistPer];
#pragma unroll
    for (uint32_t i = 0; i < kHistPer; ++i) {
      const uint64_t v = v0 + i * kPickBT + threadIdx.x;
      c[i] = v < n ? counts[v] : 0u;
    }
#pragma unroll
    for (uint32_t i = 0; i < kHistPer; ++i)
      if (c[i]) atomicAdd(&hist[count_bin(c[i])], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kBins; i += kPickBT)
    if (hist[i]) atomicAdd(&st->hist[i], hist[i]);
  if (!last_block(&st->w[kTopDone], &s_flag)) return;
  // vertices in bin b and above, two bins a thread from the top down; the
  // bins above the cut are those whose sum fits
  if (threadIdx.x == 0) {
    s_cut = 0;
    s_sum = 0;
  }
  const uint32_t hi = kBins - 1 - 2 * threadIdx.x, lo = hi - 1;   // kBins is even
  const bool have = 2 * threadIdx.x < kBins;
  const uint32_t ch = have ? load_u32(&st->hist[hi]) : 0u;
  const uint32_t cl = have ? load_u32(&st->hist[lo]) : 0u;
  uint32_t tot;
  const uint32_t pre = block_exclusive_scan<kPickBT>(ch + cl, s_tmp, &tot);
  if (have) {
    // the highest bin >= 1 that does not fit (bin 0 holds no counted vertex)
    if (hi >= 1 && pre + ch > kTopMax) atomicMax(&s_cut, hi);
    else if (lo >= 1 && pre + ch + cl > kTopMax) atomicMax(&s_cut, lo);
  }
  __syncthreads();
  const uint32_t cut = s_cut;    // 0: every vertex in a set is a candidate
  if (have && hi == cut) s_sum = pre;
  if (have && lo == cut) s_sum = pre + ch;
  __syncthreads();
  if (threadIdx.x != 0) return;
  st->w[kTopBin] = cut;
  st->w[kTopTie] = cut < 128 ? cut : 0u;   // one value per bin up to 127
  st->w[kTopRoom] = kTopMax - s_sum;
  st->w[kTopTieEnd] = 0;
  st->w[kTopBound] = bin_top(cut);
}

// Candidates of each tile of kTile vertices, without the ties and the ties
// alone; the last block finds how many whole tiles of ties there is room for
// and where each tile's candidates start.
__global__ void __launch_bounds__(kPickBT) top_tiles_kernel(const uint32_t *counts, uint32_t n,
                                                            TopState *st, uint32_t *tiles,
                                                            uint32_t ntiles) {
  __shared__ uint32_t s_tmp[kPickBT / 64];
  __shared__ uint32_t s_flag, s_end;
  const uint32_t cut = st->w[kTopBin], tie = st->w[kTopTie];
  uint32_t *sure = tiles, *ties = tiles + ntiles;
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const uint64_t v = static_cast<uint64_t>(t) * kTile + threadIdx.x;
    const uint32_t x = v < n ? counts[v] : 0u;
    // candidates in the low half, ties in the high half (at most kTile each)
    const uint32_t c = x == 0 ? 0u : count_bin(x) > cut ? 1u : x == tie ? 1u << 16 : 0u;
    uint32_t tot;
    (void)block_exclusive_scan<kPickBT>(c, s_tmp, &tot);
    if (threadIdx.x == 0) {
      atomicExch(&sure[t], tot & 0xFFFFu);
      atomicExch(&ties[t], tot >> 16);
    }
  }
  if (!last_block(&st->w[kTopDone], &s_flag)) return;
  if (threadIdx.x == 0) s_end = ntiles;
  __syncthreads();
  const uint32_t room = st->w[kTopRoom];
  uint32_t run = 0;
  for (uint32_t t0 = 0; tie != 0 && t0 < ntiles; t0 += kPickBT) {
    const uint32_t t = t0 + threadIdx.x;
    const uint32_t c = t < ntiles ? load_u32(&ties[t]) : 0u;
    uint32_t tot;
    const uint32_t pre = block_exclusive_scan<kPickBT>(c, s_tmp, &tot);
    if (t < ntiles && run + pre + c > room) atomicMin(&s_end, t);
    run += tot;
    __syncthreads();
    if (s_end < ntiles) break;   // the same for every thread
  }
  const uint32_t end = tie ? s_end : 0u;
  run = 0;
  for (uint32_t t0 = 0; t0 < ntiles; t0 += kPickBT) {
    const uint32_t t = t0 + threadIdx.x;
    const uint32_t c = t < ntiles ? load_u32(&sure[t]) + (t < end ? load_u32(&ties[t]) : 0u) : 0u;
    uint32_t tot;
    const uint32_t pre = block_exclusive_scan<kPickBT>(c, s_tmp, &tot);
    if (t < ntiles) sure[t] = run + pre;
    run += tot;
  }
  if (threadIdx.x == 0) {
    st->w[kTopTieEnd] = static_cast<uint32_t>(
        std::min<uint64_t>(static_cast<uint64_t>(end) * kTile, n));
    st->w[kTopN] = run;
  }
}

// Lists the candidates in id order (so a lower rank is a lower id) with their
// counts, their ranks by vertex, and a bitmap of who is one; the last block
// makes each candidate's place in the index.
__global__ void __launch_bounds__(kPickBT)
top_pick_kernel(const uint32_t *counts, uint32_t n, TopState *st, const uint32_t *tiles,
                uint32_t ntiles, uint32_t *cand, uint32_t *cnt, uint16_t *rank,
                unsigned long long *is_cand, uint32_t *cstart, uint32_t *ccur) {
  __shared__ uint32_t s_tmp[kPickBT / 64];
  __shared__ uint32_t s_flag;
  const uint32_t cut = st->w[kTopBin], tie = st->w[kTopTie], tie_end = st->w[kTopTieEnd];
  for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const uint64_t v = static_cast<uint64_t>(t) * kTile + threadIdx.x;
    const uint32_t c = v < n ? counts[v] : 0u;
    const bool in = c != 0 && (count_bin(c) > cut || (c == tie && v < tie_end));
    uint32_t tot;
    const uint32_t r = tiles[t] + block_exclusive_scan<kPickBT>(in ? 1u : 0u, s_tmp, &tot);
    if (in) {
      cand[r] = static_cast<uint32_t>(v);
      atomicExch(&cnt[r], c);
    }
    const uint64_t m = __ballot(in);
    if (v < n) {
      rank[v] = static_cast<uint16_t>(r);   // read for candidates only
      if (lane_id() == 0) is_cand[v >> 6] = m;
    }
  }
  if (!last_block(&st->w[kTopDone], &s_flag)) return;
  const uint32_t nc = st->w[kTopN];
  uint32_t run = 0;
  for (uint32_t c0 = 0; c0 < nc; c0 += kPickBT) {
    const uint32_t c = c0 + threadIdx.x;
    const uint32_t x = c < nc ? load_u32(&cnt[c]) : 0u;
    uint32_t tot;
    const uint32_t pre = block_exclusive_scan<kPickBT>(x, s_tmp, &tot);
    if (c < nc) {
      cstart[c] = run + pre;
      ccur[c] = run + pre;
    }
    run += tot;
  }
  if (threadIdx.x == 0) cstart[nc] = run;
}

// ------------------------------------------------------------------- index
// Per set a record of the ranks of its candidates: up to kInline in the
// record itself, more in the members array.  Per candidate its sets (inv from
// cstart).  A block finds the candidates among the members of its sets (a
// bitmap of n bits says who is one, so most members cost one access that the
// L2 holds), keeps them in LDS, reserves its room in every candidate's list
// and in the members with one atomic each, and then writes.  60M members on
// 4.2M vertices: looking the ranks up in their table instead, once to count
// and once to write, took 1.6 ms.
constexpr uint32_t kIndexSets = 1024;   // sets of a block at a time
constexpr uint32_t kStash = 8192;       // candidates kept in LDS of them
constexpr uint32_t kInline = 6;
constexpr uint32_t kRecCovered = 0x80000000u;

struct alignas(16) SetRec {
  uint32_t w[3];   // six ranks, or w[0] = where they are in the members
  uint32_t len;    // candidates of the set; kRecCovered once it is covered
};

__global__ void __launch_bounds__(kCountBT)
top_index_kernel(const unsigned long long *set_off, const uint32_t *set_len,
                 const uint32_t *data, uint64_t num_sets, uint32_t step, const uint8_t *covered,
                 const uint16_t *rank, const unsigned long long *is_cand, TopState *st,
                 uint32_t *ccur, uint32_t *inv, SetRec *rec, uint16_t *members) {
  __shared__ uint32_t hist[kTopMax];
  __shared__ uint32_t s_cnt[kIndexSets];
  __shared__ uint32_t s_hit[kStash];      // rank << 16 | set in the chunk
  __shared__ uint32_t s_tmp[kCountBT / 64];
  __shared__ uint32_t s_base, s_hits;
  __shared__ uint32_t s_pre[kCountBT / 64][65];
  __shared__ unsigned long long s_off[kCountBT / 64][64];
  const uint32_t nc = st->w[kTopN];
  const uint32_t lane = lane_id(), wid = threadIdx.x >> 6;
  const uint64_t per = share_of(num_sets, gridDim.x, step);
  const uint64_t sb = blockIdx.x * per;
  const uint64_t se = sb + per < num_sets ? sb + per : num_sets;
  for (uint64_t b = sb; b < se; b += kIndexSets) {
    const uint64_t e = b + kIndexSets < se ? b + kIndexSets : se;
    for (uint32_t i = threadIdx.x; i < nc; i += kCountBT) hist[i] = 0;
    for (uint32_t i = threadIdx.x; i < kIndexSets; i += kCountBT) s_cnt[i] = 0;
    if (threadIdx.x == 0) s_hits = 0;
    __syncthreads();
    // f(rank, set in the chunk) for the candidates in the chunk's sets
    auto for_hits = [&](auto &&f) {
      for (uint64_t w = b + wid * step; w < e; w += kCountBT / 64 * step) {
        const uint64_t s = w + lane;
        const bool live = lane < step && s < e && !(covered && covered[s]);
        for_each_run_element(live ? set_off[s] : 0ull, live ? set_len[s] : 0u, data, s_pre[wid],
                             s_off[wid], [&](uint32_t v, uint32_t j) {
                               if ((is_cand[v >> 6] >> (v & 63u)) & 1ull)
                                 f(rank[v], static_cast<uint32_t>(w - b) + j);
                             });
      }
    };
    for_hits([&](uint32_t r, uint32_t j) {
      atomicAdd(&hist[r], 1u);
      atomicAdd(&s_cnt[j], 1u);
      const uint32_t at = atomicAdd(&s_hits, 1u);
      if (at < kStash) s_hit[at] = (r << 16) | j;
    });
    __syncthreads();
    // room in the candidates' lists and, for long sets, among the members
    for (uint32_t i = threadIdx.x; i < nc; i += kCountBT)
      if (hist[i]) hist[i] = atomicAdd(&ccur[i], hist[i]);
    constexpr uint32_t kPer = kIndexSets / kCountBT;
    uint32_t mine[kPer], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      mine[q] = s_cnt[threadIdx.x * kPer + q];
      sum += mine[q] > kInline ? mine[q] : 0u;
    }
    uint32_t tot;
    uint32_t at = block_exclusive_scan<kCountBT>(sum, s_tmp, &tot);
    if (threadIdx.x == 0) s_base = tot ? atomicAdd(&st->w[kTopMembers], tot) : 0u;
    __syncthreads();
    at += s_base;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
      const uint64_t s = b + threadIdx.x * kPer + q;
      const bool large = mine[q] > kInline;
      if (s < e) {
        if (large) rec[s].w[0] = at;
        rec[s].len = mine[q];
      }
      // where the set's next rank goes: kRecCovered marks the members array
      s_cnt[threadIdx.x * kPer + q] = large ? kRecCovered | at : 0u;
      if (large) at += mine[q];
    }
    __syncthreads();
    auto place = [&](uint32_t r, uint32_t j) {
      inv[atomicAdd(&hist[r], 1u)] = static_cast<uint32_t>(b + j);
      const uint32_t a = atomicAdd(&s_cnt[j], 1u);
      if (a & kRecCovered)
        members[a & ~kRecCovered] = static_cast<uint16_t>(r);
      else
        reinterpret_cast<uint16_t *>(&rec[b + j])[a] = static_cast<uint16_t>(r);
    };
    if (s_hits <= kStash) {
      for (uint32_t i = threadIdx.x; i < s_hits; i += kCountBT) place(s_hit[i] >> 16, s_hit[i] & 0xFFFFu);
    } else {
      for_hits(place);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ rounds
struct TopRounds {
  TopState *st;
  const uint32_t *cand;
  uint32_t *cnt;
  const uint32_t *cstart;
  const uint32_t *inv;
  SetRec *rec;
  const uint16_t *members;
  uint8_t *covered;
  uint64_t num_sets;
  uint32_t *picked;           // per round its candidate: the rank, once its launch ends the vertex
};

// What a candidate must pass to be picked: counts above the bound are safe,
// and equal ones among the ids the tie tiles took (no other vertex of that
// count has a lower id).
struct TopBound {
  uint32_t bound, tie, tie_end;
  __device__ explicit TopBound(const TopState *st)
      : bound(st->w[kTopBound]), tie(st->w[kTopTie]), tie_end(st->w[kTopTieEnd]) {}
  __device__ bool safe(const TopRounds &R, uint32_t gain, uint32_t r) const {
    return gain > bound || (tie != 0 && gain == tie && R.cand[r] < tie_end);
  }
};

// Marks up to K of the sets listed at inv[p], inv[p + stride], ... (below e)
// covered, and f(rank) for each candidate of those that were not: the K lists
// entries, then the K records, are read together.
template <int K, typename F>
__device__ inline void kill_sets(const TopRounds &R, uint32_t p, uint32_t stride, uint32_t e,
                                 F &&f) {
  uint32_t s[K];
  uint4 rec[K];
#pragma unroll
  for (int u = 0; u < K; ++u) s[u] = p + u * stride < e ? R.inv[p + u * stride] : 0xFFFFFFFFu;
#pragma unroll
  for (int u = 0; u < K; ++u)
    rec[u] = s[u] != 0xFFFFFFFFu ? *reinterpret_cast<const uint4 *>(&R.rec[s[u]])
                                 : make_uint4(0, 0, 0, kRecCovered);
#pragma unroll
  for (int u = 0; u < K; ++u) {
    if (rec[u].w & kRecCovered) continue;
    R.rec[s[u]].len = rec[u].w | kRecCovered;
    R.covered[s[u]] = 1;
    const uint32_t l = rec[u].w;
    if (l <= kInline) {
      if (l > 0) f(rec[u].x & 0xFFFFu);
      if (l > 1) f(rec[u].x >> 16);
      if (l > 2) f(rec[u].y & 0xFFFFu);
      if (l > 3) f(rec[u].y >> 16);
      if (l > 4) f(rec[u].z & 0xFFFFu);
      if (l > 5) f(rec[u].z >> 16);
    } else {
      for (uint32_t q = 0; q < l; q += 8) {
        uint32_t m[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) m[i] = q + i < l ? R.members[rec[u].x + q + i] : 0u;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
          if (q + i < l) f(m[i]);
      }
    }
  }
}

// Rounds of seeds that list this many sets or more run on the whole GPU: one
// workgroup takes 4,096 sets of a list at a time, and a launch of its own
// costs about as much as one such turn (lines of 2,048 and 4,096 measured
// alike, 8,192 and 16,384 slower: 12 served queries 66, 66, 78 and 83 ms).
constexpr uint32_t kWideList = 4096;
// That line is for sets of a few candidates each (two on R-MAT scale 22 under
// weighted cascade).  Where they hold more it lies at this many together: one
// workgroup takes some 120 us for 4,095 sets of 150 candidates, whose LDS
// decrements meet on a few counters (10,000 sets of 205 under U[0,0.1] on 4096
// vertices, k = 10: 1.82 ms by sets alone, 0.91 with this line).
constexpr uint32_t kWideMembers = 8 * kWideList;
constexpr uint32_t kWideBlocks = 64;
constexpr uint32_t kRoundLaunches = 16;
constexpr uint32_t kRoundBT = 1024;
static_assert(kTopMax <= kRoundBT, "one candidate a thread");

// Rounds from the state's on: the long one pending on the whole GPU, then the
// following ones by one workgroup up to the next long one (with `all`, long
// ones too) or the end.  None is pending before the first launch, which is of
// one block: the others of a larger grid could find the state already moved.
__global__ void __launch_bounds__(kRoundBT) top_rounds_kernel(TopRounds R, uint32_t k,
                                                              uint32_t all) {
  __shared__ uint32_t cnt[kTopMax];
  __shared__ uint32_t start[kTopMax + 1];
  __shared__ uint2 s_w[kRoundBT / 64];   // per wave its best: count, rank
  __shared__ uint32_t s_flag;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  uint32_t *w = R.st->w;
  uint32_t i = w[kTopRound], cov = w[kTopCovered];
  const uint32_t stopped = w[kTopStop], gain0 = w[kTopGain], r0 = w[kTopRank];
  const uint32_t nc = w[kTopN];
  if (stopped != kStopNone || i == k) return;         // the same for every block
  if (gain0 != 0) {
    for (uint32_t c = tid; c < nc; c += kRoundBT) cnt[c] = 0;
    __syncthreads();
    const uint32_t b = R.cstart[r0], e = R.cstart[r0 + 1], stride = gridDim.x * kRoundBT;
    for (uint32_t p = b + blockIdx.x * kRoundBT + tid; p < e; p += 4 * stride)
      kill_sets<4>(R, p, stride, e, [&](uint32_t m) { atomicAdd(&cnt[m], 1u); });
    __syncthreads();
    for (uint32_t c = tid; c < nc; c += kRoundBT)
      if (cnt[c]) atomicSub(&R.cnt[c], cnt[c]);
    if (!last_block(&w[kTopDone], &s_flag)) return;
    if (tid == 0) R.picked[i] = r0;
    ++i;
    cov += gain0;
  }
  const uint32_t first = gain0 != 0 ? i - 1 : i;
  const TopBound bound(R.st);
  const bool bounded = w[kTopBin] != 0;   // vertices in sets exist outside the candidates
  for (uint32_t c = tid; c < nc; c += kRoundBT) {
    cnt[c] = load_u32(&R.cnt[c]);
    start[c] = R.cstart[c];
  }
  const uint32_t held = R.cstart[nc];     // the sets' candidates together
  if (tid == 0) start[nc] = held;
  const uint64_t each = held / R.num_sets;
  const uint32_t wide = each <= kWideMembers / kWideList
                            ? kWideList
                            : max(64u, static_cast<uint32_t>(kWideMembers / each));
  uint32_t stop = kStopNone, rank = 0, gain = 0;
  for (;;) {
    __syncthreads();
    // the best candidate, ties to the lower rank; one candidate a thread.  The
    // counts alone go through the wave, by DPP: with (count, rank) pairs and
    // shuffles IMM under LT on 2^20 vertices took 5.08 ms instead of 4.82,
    // twelve served queries 29.5 instead of 28.7
    const uint32_t mine = tid < nc ? cnt[tid] : 0u;
    const uint32_t m = wave_max_u32(mine);
    const uint32_t l = __ffsll(static_cast<unsigned long long>(__ballot(mine == m))) - 1;
    if (lane == 0) s_w[tid >> 6] = make_uint2(m, tid + l);
    __syncthreads();
    const uint2 top = s_w[lane % (kRoundBT / 64)];
    gain = wave_max_u32(top.x);
    rank = __builtin_amdgcn_readlane(
        top.y, __ffsll(static_cast<unsigned long long>(__ballot(top.x == gain))) - 1);
    if (i == k) {
      gain = 0;
      break;
    }
    if (gain == 0 || !bound.safe(R, gain, rank)) {
      stop = bounded ? kStopBound : kStopAll;
      break;
    }
    const uint32_t b = start[rank], e = start[rank + 1];
    if (e - b >= wide && !all) break;             // for the next launch
    for (uint32_t p = b + tid; p < e; p += 4 * kRoundBT)
      kill_sets<4>(R, p, kRoundBT, e, [&](uint32_t m) { atomicSub(&cnt[m], 1u); });
    if (tid == 0) R.picked[i] = rank;
    cov += gain;
    ++i;
  }
  for (uint32_t c = tid; c < nc; c += kRoundBT) R.cnt[c] = cnt[c];
  for (uint32_t q = first + tid; q < i; q += kRoundBT) R.picked[q] = R.cand[R.picked[q]];
  if (tid == 0) {
    w[kTopRound] = i;
    w[kTopCovered] = cov;
    w[kTopStop] = stop;
    w[kTopRank] = rank;
    w[kTopGain] = stop == kStopNone ? gain : 0u;
  }
}

}  // namespace

// When the candidates run out (the best falls below the bound) another pass over
// the pool finds new ones; after this many passes in a row of fewer rounds than
// this the full index takes over.  A pass costs 0.1 to 1 ms, a round of the full
// index some 8 us more than one among candidates.  R-MAT pools of 0.6 to 19M
// members under cascade and LT yield 17 to 200 rounds in the first pass and 140
// to 1000 in each later one, two or three passes for k = 1000 and up to eleven
// for k = 5000; one of large sets (U[0,0.1], 10,000 sets of 205 on 4096 vertices)
// 1 in the first and 900 in the next.  Forty cliques of 1100 vertices, each
// vertex of a clique in all its sets (0.9M members, k = 10), yield one a pass.
constexpr uint32_t kPoorRounds = 16, kPoorPasses = 2;

// counts[v] (cleared first) = sets of [0, num_sets) holding v, covered ones
// (covered != nullptr) left out; total: at least the members there are.
void count_plain(rip_pool *p, uint64_t num_sets, uint64_t total, const uint8_t *covered) {
  SelectScratch &s = p->sel;
  hipStream_t st = p->stream;
  const uint32_t n = p->g->n;
  hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_for(n, kBT * 4, 2048)), dim3(kBT), 0, st,
                     s.d_counts, static_cast<uint64_t>(n));
  if (num_sets == 0 || total == 0) return;
  const uint32_t buckets = (n + kBucketWidth - 1) >> kBucketBits;
  const uint32_t step = wave_sets(num_sets, total), block_sets = step * (kCountBT / 64);
  const uint32_t blocks = grid_for(num_sets, block_sets, 1024);
  bool deal = total >= kBucketMin && total < (1ull << 32) - kSlice && buckets <= kMaxBuckets;
  if (deal) {
    const uint64_t words = 3ull * (buckets + 1) + static_cast<uint64_t>(blocks) * buckets +
                           (total + 1) / 2;
    if (s.cap_part < words) {
      pool_free(p, s.d_part);
      s.cap_part = 0;
      try {
        s.d_part = pool_alloc<uint32_t>(p, words);
        s.cap_part = words;
      } catch (const Error &e) {
        if (e.code != RIP_ENOMEM) throw;
        deal = false;   // no room for the buckets: an atomic per member needs none
      }
    }
  }
  if (!deal) {
    hipLaunchKernelGGL(member_count_kernel, dim3(grid_for(num_sets, block_sets, 4096)),
                       dim3(kCountBT), 0, st, p->d_off, p->d_len, p->d_data, num_sets, step,
                       covered, s.d_counts);
    RIP_HIP(hipGetLastError());
    return;
  }
  uint32_t *bcnt = s.d_part, *bstart = bcnt + buckets + 1, *sstart = bstart + buckets + 1;
  uint32_t *where = sstart + buckets + 1;
  uint16_t *part = reinterpret_cast<uint16_t *>(where + static_cast<uint64_t>(blocks) * buckets);
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(kBT), 0, st, bcnt,
                     static_cast<uint64_t>(buckets));
  hipLaunchKernelGGL(bucket_size_kernel, dim3(blocks), dim3(kCountBT), 0, st, p->d_off, p->d_len,
                     p->d_data, num_sets, step, covered, buckets, bcnt, where);
  hipLaunchKernelGGL(bucket_scan_kernel, dim3(1), dim3(1024), 0, st, bcnt, buckets, bstart, sstart);
  hipLaunchKernelGGL(bucket_deal_kernel, dim3(blocks), dim3(kCountBT), 0, st, p->d_off, p->d_len,
                     p->d_data, num_sets, step, covered, buckets, bstart, where, part);
  hipLaunchKernelGGL(bucket_count_kernel,
                     dim3(static_cast<uint32_t>(total / kSlice) + buckets), dim3(kCountBT), 0, st,
                     part, bstart, sstart, buckets, n, s.d_counts);
  RIP_HIP(hipGetLastError());
}

// Greedy selection over sets [0, num_sets) of a plain pool (total members)
// into seeds[0, k); the counts of all vertices are in d_counts and the
// covered flags clear.  Returns the seeds found; *covered gets the sets they
// cover and *finished whether the selection is complete.  When it is not (the
// candidates' counts kept falling below the bound), the seeds returned are
// its first ones and the covered flags theirs.
uint32_t select_top(rip_pool *p, uint64_t num_sets, uint64_t total, uint32_t k, uint32_t *seeds,
                    uint64_t *covered, bool *finished) {
  SelectScratch &s = p->sel;
  hipStream_t st = p->stream;
  const uint32_t n = p->g->n;
  const uint32_t ntiles = (n + kTile - 1) / kTile;
  const uint64_t nwords = (static_cast<uint64_t>(n) + 63) / 64;
  if (!s.d_top) s.d_top = pool_alloc<uint8_t>(p, sizeof(TopState));
  if (s.top_n != n) {
    pool_free(p, s.d_rank);
    pool_free(p, s.d_cand);
    s.top_n = 0;
    // ranks, then the bitmap of the candidates
    s.d_rank = pool_alloc<uint16_t>(p, 4 * nwords + 4 * ((n + 3ull) / 4));
    // candidates, their counts, starts and cursors; the tiles' two counts
    s.d_cand = pool_alloc<uint32_t>(p, 4ull * (kTopMax + 1) + 2ull * ntiles);
    s.top_n = n;
  }
  if (s.cap_top_sets < num_sets) {
    pool_free(p, s.d_rec);
    const uint64_t cap = std::max<uint64_t>(num_sets, s.cap_top_sets + s.cap_top_sets / 2);
    s.cap_top_sets = 0;
    s.d_rec = pool_alloc<uint8_t>(p, sizeof(SetRec) * cap);
    s.cap_top_sets = cap;
  }
  if (s.cap_members < total) {
    pool_free(p, s.d_members);
    const uint64_t cap = std::max<uint64_t>(total, s.cap_members + s.cap_members / 2);
    s.cap_members = 0;
    s.d_members = pool_alloc<uint16_t>(p, cap);
    s.cap_members = cap;
  }
  TopState *ts = reinterpret_cast<TopState *>(s.d_top);
  uint32_t *cand = s.d_cand, *cnt = cand + kTopMax + 1, *cstart = cnt + kTopMax + 1;
  uint32_t *ccur = cstart + kTopMax + 1, *tiles = ccur + kTopMax + 1;
  unsigned long long *is_cand = reinterpret_cast<unsigned long long *>(s.d_rank + 4 * ((n + 3ull) / 4));
  const TopRounds R{ts, cand, cnt, cstart, s.d_inv, reinterpret_cast<SetRec *>(s.d_rec),
                    s.d_members, s.d_covered, std::max<uint64_t>(num_sets, 1),
                    reinterpret_cast<uint32_t *>(s.d_keys)};
  const uint32_t step = wave_sets(num_sets, total);
  uint32_t got = 0, restarts = 0, poor = 0;
  uint64_t cov = 0;
  std::vector<uint32_t> picked(k);
  *finished = false;
  for (;;) {
    const uint32_t left = k - got;
    const uint8_t *cflags = got ? s.d_covered : nullptr;
    if (got) count_plain(p, num_sets, total, cflags);
    hipLaunchKernelGGL(zero_u32_kernel, dim3(2), dim3(kBT), 0, st, reinterpret_cast<uint32_t *>(ts),
                       sizeof(TopState) / 4ull);
    const uint32_t vgrid = grid_for(n, kTile, 512);
    hipLaunchKernelGGL(top_hist_kernel, dim3(vgrid), dim3(kPickBT), 0, st, s.d_counts, n, ts);
    hipLaunchKernelGGL(top_tiles_kernel, dim3(vgrid), dim3(kPickBT), 0, st, s.d_counts, n, ts,
                       tiles, ntiles);
    hipLaunchKernelGGL(top_pick_kernel, dim3(vgrid), dim3(kPickBT), 0, st, s.d_counts, n, ts, tiles,
                       ntiles, cand, cnt, s.d_rank, is_cand, cstart, ccur);
    hipLaunchKernelGGL(top_index_kernel, dim3(grid_for(num_sets, step * (kCountBT / 64), 1024)),
                       dim3(kCountBT), 0, st, p->d_off, p->d_len, p->d_data, num_sets, step, cflags,
                       s.d_rank, is_cand, ts, ccur, s.d_inv, R.rec, s.d_members);
    // launches until the rounds are done: one when no list can be long, else
    // a few between looks at the state (one with no long round pending ends
    // the selection or costs its launch only)
    uint32_t w[kTopWords];
    const bool all = num_sets < kWideList && total < 4 * kWideMembers;
    hipLaunchKernelGGL(top_rounds_kernel, dim3(1), dim3(kRoundBT), 0, st, R, left, all ? 1u : 0u);
    do {
      for (uint32_t i = 0; i < (all ? 0u : kRoundLaunches); ++i)
        hipLaunchKernelGGL(top_rounds_kernel, dim3(kWideBlocks), dim3(kRoundBT), 0, st, R, left, 0u);
      RIP_HIP(hipGetLastError());
      RIP_HIP(hipMemcpyAsync(w, ts->w, sizeof(w), hipMemcpyDeviceToHost, st));
      RIP_HIP(hipMemcpyAsync(picked.data(), R.picked, sizeof(uint32_t) * left,
                             hipMemcpyDeviceToHost, st));
      RIP_HIP(hipStreamSynchronize(st));
    } while (w[kTopStop] == kStopNone && w[kTopRound] < left);
    std::copy(picked.begin(), picked.begin() + w[kTopRound], seeds + got);
    got += w[kTopRound];
    cov += w[kTopCovered];
    if (got == k || w[kTopStop] == kStopAll) {
      *finished = true;
      break;
    }
    // passes over the pool that yield few rounds and leave most sets there: the
    // candidates share their sets, and the full index is the better form
    const uint64_t before = num_sets - (cov - w[kTopCovered]);
    poor = w[kTopRound] < kPoorRounds && 2ull * w[kTopCovered] < before ? poor + 1 : 0;
    if (poor == kPoorPasses || ++restarts > 8 + k / 256 || w[kTopRound] == 0) break;
  }
  *covered = cov;
  return got;
}

}  // namespace rip
