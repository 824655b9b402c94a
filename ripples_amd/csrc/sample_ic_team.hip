// Team sampler: the IC samples that outgrow a lane or a wave, one reverse BFS
// per workgroup, on graphs whose visited bits fit in LDS.
//
// Semantics are those of AddRRRSet (add_rrrset.h:105-157) under the stream
// contract (common.h, ic_gap.h): the set is the reverse closure of the root
// over live edges, the same as the other samplers' and the oracle's.
//
// A discovery is one LDS atomic on the workgroup's bitmap, where the colour
// groups of the grid sampler make two device-scope atomics (their pairs of
// colour masks hold the visited and the pending colours of every vertex); in
// return rows are read once per sample, not once per group and level, which
// graphs this small serve from the L2 and the memory-side cache.  With U[0,0.1]
// weights the sampling of an IMM run took 24 ms of grid levels and 3.3 ms of
// their output at 65,536 vertices, and 34 and 3.3 ms at 262,144; the team
// kernels take 7 and 11 ms and their output 0.5.  What bounds them is the
// latency of the dependent loads of a row (record, then candidates), with the
// 16 waves per CU their registers allow.  The waves of
// the workgroup take the vertices of a level 64 at a time from a queue in
// device memory, their rows split into gap blocks (ic_expand.h).
//
// The finished bitmap is written out as a row of n bits.  Then, per group of
// 64 samples: a group whose sets hold more than 2 * hot_n hot members keeps
// them as bits of a column of the pool's column store (the rows transposed 64
// x 32 bits at a time), and the other members of every set are written as its
// sorted list, the bits in order.
#include <algorithm>

#include "device_util.h"
#include "ic_common.h"
#include "ic_expand.h"
#include "ic_gap.h"
#include "internal.h"

namespace rip {
namespace {

struct TeamParams {
  const VertexRec *vrec;
  const uint32_t *ids;
  const uint32_t *val;
  uint32_t n, nw;              // vertices, words of a bitmap
  Affine step;
  uint64_t seed;
  uint64_t first;
  const uint32_t *sample_ids;  // local sample indices of the batch, or nullptr
  uint64_t local0;             // the batch's first local index
  uint32_t count;              // samples of the batch
  uint32_t *queue;             // workgroups x n
  uint32_t *rows;              // samples x nw
  uint32_t *size, *hot;        // samples: members, hot members
  const uint32_t *hot_mask;
  unsigned long long *ctl;
};

__device__ inline uint64_t team_sample(const TeamParams &P, uint32_t i) {
  return P.first + (P.sample_ids ? P.sample_ids[i] : P.local0 + i);
}

template <int BT>
__global__ void __launch_bounds__(BT, 4) ic_team_kernel(TeamParams P) {
  constexpr uint32_t NW = BT / 64;
  extern __shared__ uint32_t s_bits[];   // nw words
  __shared__ Affine s_p2[64];
  __shared__ IcGapTab s_tab;
  __shared__ uint32_t s_idx, s_next, s_tail, s_hot;
  const uint32_t tid = threadIdx.x, lane = lane_id();
  uint32_t *queue = P.queue + static_cast<uint64_t>(blockIdx.x) * P.n;
  if (tid == 0) fill_step_powers(P.step, s_p2);
  ic_load_tables(&s_tab);
  for (uint32_t w = tid; w < P.nw; w += BT) s_bits[w] = 0;
  unsigned long long st_cand = 0, st_draws = 0, st_exp = 0, st_bytes = 0, st_live = 0;
  // marks a batch's live edges' sources; the first visits join the queue
  auto take = [&](const bool (&live)[kUnitBatch], const uint32_t (&src)[kUnitBatch], uint32_t) {
    bool fresh[kUnitBatch];
    uint64_t m[kUnitBatch];
    uint32_t total = 0;
#pragma unroll
    for (uint32_t i = 0; i < kUnitBatch; ++i) {
      const uint32_t bit = 1u << (src[i] & 31u);
      fresh[i] = live[i] && !(atomicOr(&s_bits[src[i] >> 5], bit) & bit);
      m[i] = __ballot(fresh[i]);
      total += static_cast<uint32_t>(__popcll(m[i]));
    }
    if (total == 0) return true;
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&s_tail, total);
    at = uniform_u32(at);
#pragma unroll
    for (uint32_t i = 0; i < kUnitBatch; ++i) {
      if (fresh[i]) queue[at + __popcll(m[i] & lanes_below())] = src[i];
      at += static_cast<uint32_t>(__popcll(m[i]));
    }
    return true;
  };
  for (;;) {
    __syncthreads();
    if (tid == 0) s_idx = static_cast<uint32_t>(atomicAdd(&P.ctl[kCtlBigCounter], 1ull));
    __syncthreads();
    const uint32_t idx = s_idx;
    if (idx >= P.count) break;
    const uint64_t z = sample_z(P.seed, team_sample(P, idx));
    const uint32_t root = uniform_index(z, P.n);
    if (tid == 0) {
      s_bits[root >> 5] = 1u << (root & 31u);
      queue[0] = root;
      s_tail = 1;
      s_next = 0;
      s_hot = 0;
    }
    __syncthreads();
    uint32_t lo = 0, hi = 1;
    while (lo < hi) {
      // the level's vertices, at most 64 to a wave and spread over the waves
      // when they are few
      const uint32_t chunk = std::min(64u, std::max(8u, (hi - lo + NW - 1) / NW));
      for (;;) {
        uint32_t b = 0;
        if (lane == 0) b = atomicAdd(&s_next, chunk);
        b = uniform_u32(b);
        if (b >= hi) break;
        const uint32_t take_n = std::min(chunk, hi - b);
        const bool have = lane < take_n;
        VertexRec rec{};
        if (have) rec = P.vrec[queue[b + lane]];
        st_exp += have ? 1u : 0u;
        expand_rows_units<true>(P.ids, P.val, have, rec, z, 0u, s_p2, &s_tab, st_cand, st_draws, st_bytes,
                          st_live, take);
      }
      __syncthreads();
      lo = hi;
      hi = s_tail;
      if (tid == 0) s_next = lo;
      __syncthreads();
    }
    // the finished bitmap as a row, cleared for the next sample
    uint32_t *row = P.rows + static_cast<uint64_t>(idx) * P.nw;
    uint32_t hot = 0;
    for (uint32_t w = tid; w < P.nw; w += BT) {
      const uint32_t x = s_bits[w];
      row[w] = x;
      s_bits[w] = 0;
      hot += static_cast<uint32_t>(__popc(x & P.hot_mask[w]));
    }
    for (int d = 32; d > 0; d >>= 1) hot += __shfl_xor(hot, d, 64);
    if (lane == 0 && hot) atomicAdd(&s_hot, hot);
    __syncthreads();
    if (tid == 0) {
      P.size[idx] = hi;
      P.hot[idx] = s_hot;
    }
  }
  st_bytes += static_cast<unsigned long long>(kIcRecBytes) * st_exp;
  report_stats(P.ctl, st_bytes, st_cand, st_draws, st_exp, st_live);
}

__global__ void team_reset_kernel(unsigned long long *ctl) { ctl[kCtlBigCounter] = 0; }

// ------------------------------------------------------------------ output
struct TeamOut {
  uint32_t n, nw, count;
  const uint32_t *rows, *size, *hot;
  unsigned long long *base;   // samples: pool offset of each list
  uint32_t *gcol;             // groups: the group's column, or kNoGroup
  uint32_t *gfail;            // groups: pool space ran out (nothing is written)
  const uint32_t *hot_mask, *hot_index;
  uint32_t hot_n;
  unsigned long long *const *colptr;
  uint32_t *gsample, *gref;
  uint32_t group_base;
  unsigned long long *set_off;
  uint32_t *set_len, *data;
  uint64_t cap_data;
  unsigned long long *ctl;
};

// Per group of 64 samples (thread j = sample j): the column decision, one
// reservation of pool space, the sets' offsets and lengths.
__global__ void __launch_bounds__(64) team_group_kernel(TeamParams P, TeamOut O) {
  const uint32_t j = threadIdx.x, i = blockIdx.x * 64 + j;
  const bool has = i < O.count;
  const uint32_t size = has ? O.size[i] : 0u, hot = has ? O.hot[i] : 0u;
  unsigned long long all_hot = hot;
  for (int d = 32; d > 0; d >>= 1) all_hot += __shfl_xor(all_hot, d, 64);
  // a column costs 8 bytes per hot vertex, lists 4 per member
  uint32_t col = kNoGroup;
  if (all_hot > 2ull * O.hot_n) {
    if (j == 0)
      col = O.group_base + static_cast<uint32_t>(atomicAdd(&O.ctl[kCtlGroupCounter2], 1ull));
    col = uniform_u32(col);
  }
  const uint32_t len = size - (col != kNoGroup ? hot : 0u);
  unsigned long long incl = len;
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long y = __shfl_up(incl, d, 64);
    if (j >= static_cast<uint32_t>(d)) incl += y;
  }
  const unsigned long long total = __shfl(incl, 63, 64);
  unsigned long long base = 0;
  if (j == 0) base = atomicAdd(&O.ctl[kCtlDataBump], total);
  base = uniform_u64(base);
  const bool fail = base + total > O.cap_data;
  if (j == 0) {
    if (fail) atomicOr(&O.ctl[kCtlOverflow], 1ull);
    if (col != kNoGroup) atomicAdd(&O.ctl[kCtlElems], all_hot);
    O.gcol[blockIdx.x] = col;
    O.gfail[blockIdx.x] = fail ? 1u : 0u;
  }
  const unsigned long long mine = base + incl - len;
  uint32_t sid = kNoGroup;
  if (has) {
    sid = static_cast<uint32_t>(team_sample(P, i));
    O.base[i] = mine;
    if (fail) {
      O.set_len[sid] = kLenFail;
    } else {
      O.set_off[sid] = mine;
      O.set_len[sid] = len;
    }
    if (col != kNoGroup) O.gref[sid] = (col << 6) | j;
  }
  if (col != kNoGroup) O.gsample[64ull * col + j] = sid;
  report_stats(O.ctl, has && !fail ? 4ull * len : 0ull, 0, 0, 0, 0);
}

// Each sample's members outside its group's column as its sorted list: the
// bits of its row in order, a word to a thread.
__global__ void __launch_bounds__(256) team_list_kernel(TeamOut O) {
  __shared__ uint32_t s_tmp[256 / 64];
  for (uint32_t i = blockIdx.x; i < O.count; i += gridDim.x) {
    if (O.gfail[i >> 6]) continue;   // the call is redone with more pool space
    const bool col = O.gcol[i >> 6] != kNoGroup;
    const uint32_t *row = O.rows + static_cast<uint64_t>(i) * O.nw;
    unsigned long long at = O.base[i];
    for (uint32_t w0 = 0; w0 < O.nw; w0 += 256) {
      const uint32_t w = w0 + threadIdx.x;
      uint32_t x = w < O.nw ? row[w] : 0u;
      if (col && x) x &= ~O.hot_mask[w];
      uint32_t tot;
      unsigned long long p = at + block_exclusive_scan<256>(static_cast<uint32_t>(__popc(x)), s_tmp, &tot);
      for (; x; x &= x - 1) O.data[p++] = w * 32 + static_cast<uint32_t>(__ffs(static_cast<int>(x)) - 1);
      at += tot;
    }
  }
}

// The columns: 64 words of the 64 rows of a group to a wave, transposed
// through LDS; word by word, ballot b of the rows' bits is the colour mask of
// vertex b of the word.
__global__ void __launch_bounds__(64) team_column_kernel(TeamOut O, uint32_t tiles) {
  __shared__ uint32_t s_w[64][65];
  const uint32_t g = blockIdx.x / tiles, w0 = blockIdx.x % tiles * 64, lane = threadIdx.x;
  const uint32_t col = O.gcol[g];
  if (col == kNoGroup || O.gfail[g]) return;
  unsigned long long *c = O.colptr[col];
  const uint32_t w = w0 + lane;
  for (uint32_t j = 0; j < 64; ++j) {
    const uint32_t i = g * 64 + j;
    s_w[j][lane] = i < O.count && w < O.nw ? O.rows[static_cast<uint64_t>(i) * O.nw + w] : 0u;
  }
  __syncthreads();
  for (uint32_t q = 0; q < 64 && w0 + q < O.nw; ++q) {
    const uint32_t hm = O.hot_mask[w0 + q];
    if (hm == 0) continue;   // the same for every lane
    const uint32_t x = s_w[lane][q];
    unsigned long long keep = 0;
#pragma unroll
    for (uint32_t b = 0; b < 32; ++b) {
      const unsigned long long m = __ballot((x >> b) & 1u);
      if (lane == b) keep = m;
    }
    if (lane < 32 && ((hm >> lane) & 1u)) c[O.hot_index[(w0 + q) * 32 + lane]] = keep;
  }
}

// Workgroups of a size that fit on a CU with `lds` bytes of bitmap.
int team_blocks_per_cu(const void *kernel, int bt, uint32_t lds) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, bt, lds) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return per_cu;
}

const void *team_kernel_ptr(uint32_t bt) {
  switch (bt) {
    case 256: return reinterpret_cast<const void *>(&ic_team_kernel<256>);
    case 512: return reinterpret_cast<const void *>(&ic_team_kernel<512>);
    default: return reinterpret_cast<const void *>(&ic_team_kernel<1024>);
  }
}

}  // namespace

void team_scratch_free(TeamScratch &s) {
  dev_free(s.d_queue);
  dev_free(s.d_rows);
  dev_free(s.d_tables);
  s = TeamScratch{};
}

// Samples first + ids[i] (first + i without ids), i in [0, count).  Returns
// the kernel launches made; nothing is synchronised.
uint32_t ic_team_launch(rip_pool *p, uint64_t first, uint64_t count, const uint32_t *ids) {
  if (count == 0) return 0;
  rip_graph *g = p->g;
  hipStream_t st = p->stream;
  TeamScratch &s = g->team;
  const uint32_t n = g->n, nw = (n + 31) / 32, lds = 4 * nw;
  pool_reserve_groups(p, p->groups + static_cast<uint32_t>((count + 63) / 64));
  // workgroups of 256 threads while four of them (the register limit of 16
  // waves per CU) find room for their bitmaps, larger ones for larger
  // bitmaps, and the largest when the samples are too few to fill the CUs
  // (262,144 vertices, calls of a few hundred large samples: IMM 16.0 ms with
  // this line, 18.5 with it at a quarter of the samples, the same at four
  // times them)
  const int cus = cu_count();
  uint32_t bt = lds <= (32u << 10) ? 256u : lds <= (64u << 10) ? 512u : 1024u;
  while (bt < 1024 && count * bt < static_cast<uint64_t>(cus) * 1024) bt *= 2;
  const void *kernel = team_kernel_ptr(bt);
  // the limit belongs to the process: one value for every graph, as calls on
  // others may be about to launch
  RIP_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(kTeamMaxNodes / 8)));
  const uint64_t resident = static_cast<uint64_t>(cus) *
                            team_blocks_per_cu(kernel, static_cast<int>(bt), lds);
  // a batch's rows take at most 1 GiB, and at least a group of samples; rows
  // and queues stay within an eighth of the memory they may use (free plus what
  // they already hold) when that is less
  const uint64_t row_bytes = 4ull * nw;
  uint64_t batch = std::min<uint64_t>(
      (count + 63) / 64 * 64, std::max<uint64_t>(64, (1ull << 30) / row_bytes / 64 * 64));
  uint64_t wgs = std::min<uint64_t>(resident, batch);
  if (s.queue_words < wgs * n || s.row_words < batch * nw) {
    const uint64_t budget = (device_free_bytes() + 4 * (s.queue_words + s.row_words)) / 8;
    batch = std::min(batch, std::max<uint64_t>({64, s.row_words / nw / 64 * 64,
                                                budget / 2 / row_bytes / 64 * 64}));
    wgs = std::min({wgs, batch, std::max<uint64_t>({1, s.queue_words / n, budget / 2 / (4ull * n)})});
  }
  if (s.queue_words < wgs * n) {
    dev_free(s.d_queue);
    s.queue_words = 0;
    s.d_queue = dev_alloc<uint32_t>(wgs * n);
    s.queue_words = wgs * n;
  }
  if (s.row_words < batch * nw) {
    dev_free(s.d_rows);
    s.row_words = 0;
    s.d_rows = dev_alloc<uint32_t>(batch * nw);
    s.row_words = batch * nw;
  }
  if (s.samples < batch) {
    dev_free(s.d_tables);
    s.samples = 0;
    // per sample its list's offset (64 bits), size and hot members; per group
    // its column and whether it failed
    s.d_tables = dev_alloc<uint32_t>(4 * batch + 2 * (batch / 64));
    s.samples = batch;
  }
  TeamParams P;
  P.vrec = g->d_vrec;
  P.ids = g->d_ids;
  P.val = g->d_val;
  P.n = n;
  P.nw = nw;
  P.step = g->step;
  P.seed = p->seed;
  P.first = first;
  P.queue = s.d_queue;
  P.rows = s.d_rows;
  P.size = s.d_tables + 2 * batch;
  P.hot = P.size + batch;
  P.hot_mask = g->d_hot_mask;
  P.ctl = p->d_ctl;
  TeamOut O;
  O.n = n;
  O.nw = nw;
  O.rows = P.rows;
  O.size = P.size;
  O.hot = P.hot;
  O.base = reinterpret_cast<unsigned long long *>(s.d_tables);
  O.gcol = P.hot + batch;
  O.gfail = O.gcol + batch / 64;
  O.hot_mask = g->d_hot_mask;
  O.hot_index = g->d_hot_index;
  O.hot_n = g->hot_n;
  O.colptr = p->d_colptr;
  O.gsample = p->d_gsample;
  O.gref = p->d_gref;
  O.group_base = p->groups;
  O.set_off = p->d_off;
  O.set_len = p->d_len;
  O.data = p->d_data;
  O.cap_data = p->cap_data;
  O.ctl = p->d_ctl;
  const uint32_t tiles = (nw + 63) / 64;
  uint32_t launches = 0;
  RIP_HIP(hipEventRecord(p->ev3, st));
  for (uint64_t b0 = 0; b0 < count; b0 += batch) {
    P.sample_ids = ids ? ids + b0 : nullptr;
    P.local0 = b0;
    P.count = static_cast<uint32_t>(std::min<uint64_t>(batch, count - b0));
    O.count = P.count;
    const uint32_t groups = (P.count + 63) / 64;
    const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>(wgs, P.count));
    hipLaunchKernelGGL(team_reset_kernel, dim3(1), dim3(1), 0, st, p->d_ctl);
    switch (bt) {
      case 256: hipLaunchKernelGGL((ic_team_kernel<256>), dim3(grid), dim3(256), lds, st, P); break;
      case 512: hipLaunchKernelGGL((ic_team_kernel<512>), dim3(grid), dim3(512), lds, st, P); break;
      default: hipLaunchKernelGGL((ic_team_kernel<1024>), dim3(grid), dim3(1024), lds, st, P); break;
    }
    RIP_HIP(hipGetLastError());
    RIP_HIP(hipEventRecord(p->ev4, st));
    hipLaunchKernelGGL(team_group_kernel, dim3(groups), dim3(64), 0, st, P, O);
    hipLaunchKernelGGL(team_list_kernel, dim3(std::min(P.count, 8192u)), dim3(256), 0, st, O);
    hipLaunchKernelGGL(team_column_kernel, dim3(groups * tiles), dim3(64), 0, st, O, tiles);
    RIP_HIP(hipGetLastError());
    launches += 5;
    ++p->grid_levels;
  }
  p->team_ran = true;
  return launches;
}

}  // namespace rip
