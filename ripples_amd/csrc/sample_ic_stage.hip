// Wave stage: the IC samples between a lane's list and the large sets, several
// per wave at a time.
//
// Semantics are those of AddRRRSet (include/ripples/add_rrrset.h:105-157)
// under the per-sample stream contract of common.h and ic_gap.h; the set is
// the reverse closure of the root over live edges, so any expansion order
// gives the sets of the other samplers and the oracle bit for bit.
//
// A frontier of these samples is thin (ten vertices on average on R-MAT scale
// 22 under weighted cascade, and 42 rounds deep), so a wave holds kPack
// samples in slots and fills its 64 lanes with queued vertices of all of
// them.  Per slot:
//   tab   (LDS)   visited vertices + 1, open addressing, 0 = empty, for the
//                 first of them, up to three quarters of the table
//   htab  (HBM)   the later ones, 2 cap slots, cleared when a sample used it
//   list  (HBM)   BFS queue and set, in discovery order, cap vertices; its
//                 last 64 also in LDS
//   tail  (LDS)   its length, bumped by the lanes that append
// and, in lane k's registers, slot k's head.  A round takes up to 64 queued
// vertices, draws their rows' gap blocks (ic_expand.h), queues the live edges
// in LDS and marks their in-neighbours kMark to a lane at a time, so that it
// waits for three trips to memory (records, ids, HBM tables) whatever it
// finds.  Sets of up to 64 vertices are sorted in registers on the way out,
// longer ones written as they are and sorted by stage_sort_kernel; samples
// that outgrow cap are listed for the large-set samplers.
//
// What bounds it: a round is some 300 vector instructions in dependent chains
// of 64-bit arithmetic besides those three trips, about 12 us on a full chip
// and 4 on an empty one, for one vertex as for 64; and the longest samples go
// through hundreds of rounds, about 1 ms however few samples there are.  IMM on
// R-MAT scale 22 under weighted cascade, one sample per wave and visited checks
// edge by edge: 33.0 ms; slots 32.0; marks together 29.6; the lanes in front
// cut to 16 vertices 28.3; sets sorted in registers and list ends in LDS 27.6;
// counters and claims of the waves off one line 24.3.
#include <algorithm>

#include "device_util.h"
#include "ic_common.h"
#include "ic_expand.h"
#include "ic_gap.h"
#include "internal.h"

namespace rip {
namespace {

constexpr int kStageBT = 256;
constexpr uint32_t kPack = 4;             // samples a wave holds
constexpr uint32_t kSortWave = 512;       // longest set sorted by one wave
constexpr uint32_t kMark = 3;             // queued edges a lane marks at once
constexpr uint32_t kQueue = 64 * (kMark + kUnitBatch);  // a wave's queue of live edges
constexpr uint32_t kStageCap = 4096;      // longest set of the stage
// A wave holds fewer samples when there are few: two to claim per slot, so that
// the long ones spread (one measured the same, four 5% slower on IMM on R-MAT
// scale 22 under weighted cascade, where eight slots measured as four).
constexpr uint64_t kSlotShare = 2;
// The stage's cap where the team sampler takes the rest: a sample that
// reaches a giant component is soon seen to, and the stage's work on it is
// lost.  IMM with U[0,0.1] weights at 65,536 vertices took 23.9, 17.2, 15.9
// and 15.7 ms with 4096, 2048, 1024 and 512; OPIM-C with weighted cascade at
// 200,003 vertices 6.0 ms down to 1024 and 7.9 with 512.
constexpr uint32_t kStageCapTeam = 1024;
// LDS tables per wave: with sets of at most 1024 vertices most never leave one
// of 2048 words; longer ones do, and four workgroups a CU are worth more.
constexpr uint32_t kTab = 1024, kTabTeam = 2048;

struct StageParams {
  const VertexRec *vrec;
  const uint32_t *ids;
  const uint32_t *val;
  uint32_t n;
  Affine step;
  uint64_t seed;
  uint64_t first;
  uint64_t count;
  uint32_t *htab;              // waves x kPack x 2 cap
  uint32_t *list;              // waves x kPack x cap
  uint32_t cap;                // a power of two
  uint32_t slots;              // samples a wave holds in this call: 1, 2, .., kPack
  uint32_t *big_ids;           // samples left for the large-set samplers (kCtlLongCount)
  uint32_t *sort_ids;          // sets written unsorted (kCtlSortCount)
  unsigned long long *set_off;
  uint32_t *set_len;
  uint32_t *data;
  uint64_t cap_data;
  unsigned long long *ctl;
  uint32_t chunk;              // pool elements a wave reserves at a time
  const uint32_t *sample_ids;  // optional: local index -> sample index (minus first)
};

// Inserts v into a wave's LDS table of a power of two slots (vertex + 1, 0 =
// empty; always some empty); true if it was not there yet.
__device__ inline bool mark(uint32_t *t, uint32_t mask, uint32_t v) {
  const uint32_t want = v + 1u;
  uint32_t h = hash_vertex(v) & mask;
  for (;;) {
    const uint32_t cur = atomicCAS(&t[h], 0u, want);
    if (cur == 0) return true;
    if (cur == want) return false;
    h = (h + 1) & mask;
  }
}

// Whether v is in a wave's LDS table.
__device__ inline bool marked(const uint32_t *t, uint32_t mask, uint32_t v) {
  const uint32_t want = v + 1u;
  uint32_t h = hash_vertex(v) & mask;
  for (;;) {
    const uint32_t cur = __hip_atomic_load(&t[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    if (cur == want) return true;
    if (cur == 0) return false;
    h = (h + 1) & mask;
  }
}

// Sorts the values of a wave's lanes, w of them (a power of two; the lanes
// from w on hold values of their own).
__device__ inline uint32_t lane_sort(uint32_t x, uint32_t w) {
  const uint32_t lane = lane_id();
  for (uint32_t k = 2; k <= w; k <<= 1)
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      const uint32_t y = __shfl_xor(x, static_cast<int>(j), 64);
      const bool up = (lane & k) == 0, low = (lane & j) == 0;
      x = up == low ? min(x, y) : max(x, y);
    }
  return x;
}

// TAB: words of the LDS tables of a wave's slots together.
template <int BT, uint32_t TAB>
__global__ void __launch_bounds__(BT, 4) ic_stage_kernel(StageParams P) {
  constexpr uint32_t NW = BT / 64;
  __shared__ alignas(16) uint32_t s_tab[NW][TAB];
  __shared__ uint32_t s_ring[NW][kPack][64];   // the last vertices of the slots' lists
  __shared__ uint32_t s_qe[NW][kQueue];
  __shared__ uint8_t s_qs[NW][kQueue];
  __shared__ uint32_t s_tail[NW][kPack], s_big[NW][kPack], s_local[NW][kPack];
  __shared__ uint64_t s_z[NW][kPack];
  __shared__ Affine s_p2[64];                 // P^(2^j): jumps between gap blocks
  __shared__ IcGapTab s_gap;
  __shared__ unsigned long long s_out;        // the workgroup's first output
  const uint32_t lane = lane_id();
  const uint32_t wid = threadIdx.x >> 6;
  const uint64_t wave = static_cast<uint64_t>(blockIdx.x) * NW + wid;
  if (threadIdx.x == 0) {
    s_out = atomicAdd(&P.ctl[kCtlDataBump], static_cast<unsigned long long>(NW) * P.chunk);
    fill_step_powers(P.step, s_p2);
  }
  ic_load_tables(&s_gap);
  if (lane < kPack) s_tail[wid][lane] = s_big[wid][lane] = 0;
  __syncthreads();
  const uint32_t cap = P.cap, hmask = 2 * cap - 1;
  // a slot's LDS table, and the vertices it takes
  const uint32_t tab = TAB / P.slots, near = tab / 4 * 3;
  uint32_t *tabs = s_tab[wid];
  uint32_t *htab = P.htab + wave * kPack * 2 * cap;
  uint32_t *list = P.list + wave * kPack * cap;
  // the wave's reserved output [out_cur, out_end) (wave-uniform), the first of
  // it reserved for all waves together; the rest of a chunk that cannot take the
  // next set stays a gap in the pool's data
  unsigned long long out_cur = s_out + static_cast<unsigned long long>(wid) * P.chunk;
  unsigned long long out_end = out_cur + P.chunk;
  unsigned long long st_cand = 0, st_draws = 0, st_exp = 0, st_bytes = 0, st_live = 0;
  uint32_t head = 0;       // lane k: slot k's
  bool held = false;       // lane k: slot k has a sample
  bool left = true;        // samples may be left to claim (wave-uniform)
  // the wave's first samples are its own, later ones claimed past everyone's
  const uint64_t own = static_cast<uint64_t>(gridDim.x) * NW * P.slots;
  bool first = true;

  uint32_t qn = 0;         // edges queued (wave-uniform)

  // appends u to the slot's list
  auto append = [&](uint32_t slot, uint32_t u) {
    const uint32_t at = atomicAdd(&s_tail[wid][slot], 1u);
    s_ring[wid][slot][at & 63u] = u;
    if (at < cap)
      list[slot * cap + at] = u;
    else
      s_big[wid][slot] = 1;
  };
  // Marks the in-neighbours of the last 64 kMark queued edges, or all when
  // they are fewer: their ids together, then the LDS tables, then the HBM
  // tables together.
  auto discover = [&]() {
    const uint32_t now = min(qn, 64u * kMark), q0 = qn - now;
    uint32_t u[kMark], slot[kMark], seen[kMark];
    bool far[kMark];
#pragma unroll
    for (uint32_t i = 0; i < kMark; ++i) {
      const uint32_t at = q0 + i * 64 + lane;
      far[i] = at < qn;
      slot[i] = far[i] ? s_qs[wid][at] : 0u;
      u[i] = far[i] ? P.ids[s_qe[wid][at]] : 0u;
    }
#pragma unroll
    for (uint32_t i = 0; i < kMark; ++i) {
      if (far[i]) {
        // at most 64 vertices join a slot's LDS table before its tail, which
        // only grows, is read again
        const uint32_t tail = __hip_atomic_load(&s_tail[wid][slot[i]], __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WAVEFRONT);
        uint32_t *t = tabs + slot[i] * tab;
        if (tail >= cap) {
          s_big[wid][slot[i]] = 1;
          far[i] = false;
        } else if (tail + 64u <= near) {
          if (mark(t, tab - 1, u[i])) append(slot[i], u[i]);
          far[i] = false;
        } else if (marked(t, tab - 1, u[i])) {
          far[i] = false;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (uint32_t i = 0; i < kMark; ++i)
      if (far[i])
        seen[i] = atomicCAS(&htab[slot[i] * 2 * cap + (hash_vertex(u[i]) & hmask)], 0u, u[i] + 1u);
#pragma unroll
    for (uint32_t i = 0; i < kMark; ++i) {
      if (far[i]) {
        uint32_t h = hash_vertex(u[i]) & hmask;
        while (seen[i] != 0 && seen[i] != u[i] + 1u) {
          h = (h + 1) & hmask;
          seen[i] = atomicCAS(&htab[slot[i] * 2 * cap + h], 0u, u[i] + 1u);
        }
        if (seen[i] == 0) append(slot[i], u[i]);
      }
    }
    qn = q0;
  };
  // queues the live ones of a batch of edges
  auto take = [&](const bool (&live)[kUnitBatch], const uint32_t (&e)[kUnitBatch], uint32_t slot) {
#pragma unroll
    for (uint32_t i = 0; i < kUnitBatch; ++i) {
      const uint64_t m = __ballot(live[i]);
      if (live[i]) {
        const uint32_t at = qn + static_cast<uint32_t>(__popcll(m & lanes_below()));
        s_qe[wid][at] = e[i];
        s_qs[wid][at] = static_cast<uint8_t>(slot);
      }
      qn += static_cast<uint32_t>(__popcll(m));
    }
    if (qn >= 64 * kMark) discover();
    return true;
  };

  for (;;) {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    uint32_t tail = lane < kPack ? s_tail[wid][lane] : 0u;
    const bool big = lane < kPack && s_big[wid][lane] != 0;
    const uint64_t bigs = __ballot(held && big);
    // ------------------------------------------------ finished samples
    for (uint64_t m = __ballot(held && (big || head == tail)); m; m &= m - 1) {
      const uint32_t k = __ffsll(static_cast<unsigned long long>(m)) - 1;
      const uint32_t len = __builtin_amdgcn_readlane(tail, k);
      const uint32_t local = uniform_u32(s_local[wid][k]);
      const uint64_t s = P.first + local;
      if (len + 64u > near) {
        // the LDS table was left: clear the other one
        uint4 *h = reinterpret_cast<uint4 *>(htab + k * 2 * cap);
        for (uint32_t i = lane; i < cap / 2; i += 64) h[i] = make_uint4(0, 0, 0, 0);
      }
      if (lane == k) held = false;
      if ((bigs >> k) & 1ull) {
        if (lane == 0) {
          const unsigned long long b = atomicAdd(&P.ctl[kCtlLongCount], 1ull);
          P.big_ids[b] = local;
        }
        continue;
      }
      if (out_end - out_cur < len) {
        const unsigned long long want = len > P.chunk ? len : P.chunk;
        unsigned long long nb = 0;
        if (lane == 0) nb = atomicAdd(&P.ctl[kCtlDataBump], want);
        nb = uniform_u64(nb);
        out_cur = nb;
        out_end = nb + want;
      }
      const unsigned long long base = out_cur;
      out_cur += len;
      if (base + len > P.cap_data) {
        if (lane == 0) {
          atomicOr(&P.ctl[kCtlOverflow], 1ull);
          P.set_len[s] = kLenFail;
        }
        continue;
      }
      const uint32_t *l = list + k * cap;
      if (len <= 64) {
        uint32_t w = 1;
        while (w < len) w <<= 1;
        const uint32_t x = lane_sort(lane < len ? l[lane] : kEmptyVertex, w);
        if (lane < len) P.data[base + lane] = x;
      } else {
        for (uint32_t i = lane; i < len; i += 64) P.data[base + i] = l[i];
      }
      if (lane == 0) {
        // the short ones from the front of sort_ids, the long ones from its end
        if (len > kSortWave) {
          const unsigned long long q = atomicAdd(&P.ctl[kCtlBigCounter], 1ull);
          P.sort_ids[P.count - 1 - q] = local;
        } else if (len > 64) {
          const unsigned long long q = atomicAdd(&P.ctl[kCtlSortCount], 1ull);
          P.sort_ids[q] = local;
        }
        P.set_off[s] = base;
        P.set_len[s] = len;
        st_bytes += 4ull * len;
      }
    }
    // ----------------------------------------------------- new samples
    if (left) {
      const bool idle = lane < P.slots && !held;
      const uint64_t m = __ballot(idle);
      if (m) {
        unsigned long long i0 = wave * P.slots;
        if (!first) {
          if (lane == 0)
            i0 = atomicAdd(&P.ctl[kCtlGroupCounter], static_cast<unsigned long long>(__popcll(m)));
          i0 = own + uniform_u64(i0);
        }
        const unsigned long long i = i0 + __popcll(m & lanes_below());
        left = first ? own < P.count : i0 + __popcll(m) < P.count;
        first = false;
        const bool got = idle && i < P.count;
        uint32_t root = 0;
        if (got) {
          const uint32_t local = P.sample_ids ? P.sample_ids[i] : static_cast<uint32_t>(i);
          const uint64_t z = sample_z(P.seed, P.first + local);
          root = uniform_index(z, P.n);
          s_local[wid][lane] = local;
          s_z[wid][lane] = z;
          s_tail[wid][lane] = 1;
          s_big[wid][lane] = 0;
          list[lane * cap] = root;
          s_ring[wid][lane][0] = root;
          head = 0;
          tail = 1;
          held = true;
        }
        for (uint64_t c = __ballot(got); c; c &= c - 1) {
          uint4 *t = reinterpret_cast<uint4 *>(
              tabs + (__ffsll(static_cast<unsigned long long>(c)) - 1) * tab);
          for (uint32_t q = lane; q < tab / 4; q += 64) t[q] = make_uint4(0, 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        if (got) tabs[lane * tab + (hash_vertex(root) & (tab - 1))] = root + 1u;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      }
    }
    if (__ballot(held) == 0) break;
    // ------------------------------------- a round: up to 64 queued vertices
    const uint32_t queued = held ? tail - head : 0u;
    uint32_t used = 0, slot = 0, pos = 0, end = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPack; ++k) {
      const uint32_t a = min(static_cast<uint32_t>(__builtin_amdgcn_readlane(queued, k)), 64u - used);
      const uint32_t h = __builtin_amdgcn_readlane(head, k), l = __builtin_amdgcn_readlane(tail, k);
      if (lane >= used && lane < used + a) {
        slot = k;
        pos = h + lane - used;
        end = l;
      }
      if (lane == k) head += a;
      used += a;
    }
    const bool have = lane < used;
    VertexRec rec{};
    uint64_t z = 0;
    if (have) {
      rec = P.vrec[end - pos <= 64 ? s_ring[wid][slot][pos & 63u] : list[slot * cap + pos]];
      z = s_z[wid][slot];
      ++st_exp;
    }
    expand_rows_units<false>(P.ids, P.val, have, rec, z, slot, s_p2, &s_gap, st_cand, st_draws,
                             st_bytes, st_live, take);
    while (qn) discover();
  }
  report_stats(P.ctl, st_bytes + kIcRecBytes * st_exp, st_cand, st_draws, st_exp, st_live);
}

// Sorts 64 R values of a wave, R to a lane; value r of lane l ends up with the
// (l R + r)-th.
template <uint32_t R>
__device__ inline void wave_sort(uint32_t (&x)[R]) {
  const uint32_t lane = lane_id();
#pragma unroll
  for (uint32_t k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      if (j >= R) {
        const bool keep_min = ((lane & (k / R)) == 0) == ((lane & (j / R)) == 0);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
          const uint32_t y = __shfl_xor(x[r], static_cast<int>(j / R), 64);
          x[r] = keep_min ? min(x[r], y) : max(x[r], y);
        }
      } else {
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
          if (r & j) continue;
          const bool up = k < R ? (r & k) == 0 : (lane & (k / R)) == 0;
          const uint32_t lo = min(x[r], x[r | j]), hi = max(x[r], x[r | j]);
          x[r] = up ? lo : hi;
          x[r | j] = up ? hi : lo;
        }
      }
    }
  }
}

template <uint32_t R>
__device__ inline void sort_set(uint32_t *d, uint32_t len) {
  uint32_t x[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t i = r * 64 + lane_id();
    x[r] = i < len ? d[i] : kEmptyVertex;
  }
  wave_sort<R>(x);
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t i = lane_id() * R + r;
    if (i < len) d[i] = x[r];
  }
}

// Sorts the sets the stage wrote unsorted: those past kSortWave vertices a
// workgroup each (bitonic in LDS), the others a wave each in registers, where
// a step of the network costs two to four instructions a value instead of some
// seven.
template <int BT, uint32_t CAP>
__global__ void __launch_bounds__(BT) stage_sort_kernel(const uint32_t *sort_ids, uint64_t count,
                                                        const unsigned long long *ctl,
                                                        uint64_t first,
                                                        const unsigned long long *set_off,
                                                        const uint32_t *set_len, uint32_t *data) {
  __shared__ uint32_t a[CAP];
  const uint64_t nlong = ctl[kCtlBigCounter], nshort = ctl[kCtlSortCount];
  for (uint64_t i = blockIdx.x; i < nlong; i += gridDim.x) {
    const uint64_t s = first + sort_ids[count - 1 - i];
    const unsigned long long off = set_off[s];
    const uint32_t len = set_len[s];
    uint32_t w = 2 * kSortWave;
    while (w < len) w <<= 1;
    for (uint32_t j = threadIdx.x; j < w; j += BT) a[j] = j < len ? data[off + j] : kEmptyVertex;
    __syncthreads();
    for (uint32_t k = 2; k <= w; k <<= 1) {
      for (uint32_t j = k >> 1; j > 0; j >>= 1) {
        for (uint32_t t = threadIdx.x; t < w / 2; t += BT) {
          const uint32_t p = ((t & ~(j - 1)) << 1) | (t & (j - 1)), q = p | j;
          const uint32_t x = a[p], y = a[q];
          if ((x > y) == ((p & k) == 0)) {
            a[p] = y;
            a[q] = x;
          }
        }
        __syncthreads();
      }
    }
    for (uint32_t j = threadIdx.x; j < len; j += BT) data[off + j] = a[j];
    __syncthreads();
  }
  const uint64_t waves = static_cast<uint64_t>(gridDim.x) * (BT / 64);
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * (BT / 64) + (threadIdx.x >> 6); i < nshort;
       i += waves) {
    const uint64_t s = first + uniform_u32(sort_ids[i]);
    uint32_t *d = data + uniform_u64(set_off[s]);
    const uint32_t len = uniform_u32(set_len[s]);
    if (len <= 128)
      sort_set<2>(d, len);
    else if (len <= 256)
      sort_set<4>(d, len);
    else
      sort_set<8>(d, len);
  }
}

__global__ void reset_stage_kernel(unsigned long long *ctl) {
  ctl[kCtlGroupCounter] = 0;
  ctl[kCtlLongCount] = 0;
  ctl[kCtlSortCount] = 0;
  ctl[kCtlBigCounter] = 0;
}

}  // namespace

// Samples first + ids[i] (first + i without ids), i in [0, count), through the
// stage.  Returns the number left for the large-set samplers (their local
// indices are in g->wave.d_big).
uint64_t ic_stage_launch(rip_pool *p, uint64_t first, uint64_t count, const uint32_t *ids,
                         uint32_t out_chunk, bool record_events) {
  constexpr int BT = kStageBT;
  rip_graph *g = p->g;
  WaveScratch &w = g->wave;
  const uint32_t cap = g->n <= kTeamMaxNodes ? kStageCapTeam : kStageCap;
  // the output slack is sized for the waves and chunks of ic_wave_blocks
  const uint32_t plain = ic_wave_blocks(count);
  const void *kernel = cap == kStageCap
                           ? reinterpret_cast<const void *>(&ic_stage_kernel<BT, kTab>)
                           : reinterpret_cast<const void *>(&ic_stage_kernel<BT, kTabTeam>);
  const uint32_t resident =
      std::min<uint32_t>(plain, static_cast<uint32_t>(blocks_per_cu(kernel, BT) * cu_count()));
  uint64_t waves = static_cast<uint64_t>(resident) * (BT / 64);
  const uint64_t wave_bytes = 12ull * kPack * cap;   // tables 8 cap, lists 4 cap a slot
  if (w.stage_waves < waves) {
    // fewer waves where the scratch would pass an eighth of the memory it may
    // use (free plus what it already holds)
    const uint64_t budget = (device_free_bytes() + w.stage_waves * wave_bytes) / 8;
    const uint64_t fit = std::max<uint64_t>(1, budget / (wave_bytes * (BT / 64))) * (BT / 64);
    waves = std::min(waves, std::max(fit, w.stage_waves));
  }
  const uint32_t blocks = static_cast<uint32_t>(waves / (BT / 64));
  if (w.stage_waves < waves) {
    dev_free(w.d_shtab);
    dev_free(w.d_slist);
    w.stage_waves = 0;
    w.d_shtab = dev_alloc<uint32_t>(waves * kPack * 2 * cap);
    w.d_slist = dev_alloc<uint32_t>(waves * kPack * cap);
    // zero once; the kernel leaves it so
    RIP_HIP(hipMemsetAsync(w.d_shtab, 0, sizeof(uint32_t) * waves * kPack * 2 * cap, p->stream));
    w.stage_waves = waves;
  }
  if (w.cap_big < count) {
    dev_free(w.d_big);
    w.cap_big = 0;
    w.d_big = dev_alloc<uint32_t>(count);
    w.cap_big = count;
  }
  if (w.cap_ssort < count) {
    dev_free(w.d_ssort);
    w.cap_ssort = 0;
    w.d_ssort = dev_alloc<uint32_t>(count);
    w.cap_ssort = count;
  }
  StageParams P;
  P.vrec = g->d_vrec;
  P.ids = g->d_ids;
  P.val = g->d_val;
  P.n = g->n;
  P.step = g->step;
  P.seed = p->seed;
  P.first = first;
  P.count = count;
  P.htab = w.d_shtab;
  P.list = w.d_slist;
  P.cap = cap;
  P.slots = 1;
  while (P.slots < kPack && 2 * P.slots * kSlotShare * waves <= count) P.slots *= 2;
  P.big_ids = w.d_big;
  P.sort_ids = w.d_ssort;
  P.set_off = p->d_off;
  P.set_len = p->d_len;
  P.data = p->d_data;
  P.cap_data = p->cap_data;
  P.ctl = p->d_ctl;
  P.chunk = ic_chunk(p, count, out_chunk, static_cast<uint64_t>(plain) * (BT / 64));
  P.sample_ids = ids;
  hipLaunchKernelGGL(reset_stage_kernel, dim3(1), dim3(1), 0, p->stream, p->d_ctl);
  if (record_events) RIP_HIP(hipEventRecord(p->ev0, p->stream));
  RIP_HIP(hipEventRecord(p->ev3, p->stream));
  const uint32_t sorters = static_cast<uint32_t>(
      std::max<uint64_t>(1, std::min<uint64_t>(count, 2048)));
  if (cap == kStageCap) {
    hipLaunchKernelGGL((ic_stage_kernel<BT, kTab>), dim3(blocks), dim3(BT), 0, p->stream, P);
    hipLaunchKernelGGL((stage_sort_kernel<256, kStageCap>), dim3(sorters), dim3(256), 0, p->stream,
                       P.sort_ids, count, P.ctl, first, P.set_off, P.set_len, P.data);
  } else {
    hipLaunchKernelGGL((ic_stage_kernel<BT, kTabTeam>), dim3(blocks), dim3(BT), 0, p->stream, P);
    hipLaunchKernelGGL((stage_sort_kernel<256, kStageCapTeam>), dim3(sorters), dim3(256), 0,
                       p->stream, P.sort_ids, count, P.ctl, first, P.set_off, P.set_len, P.data);
  }
  RIP_HIP(hipGetLastError());
  if (record_events) RIP_HIP(hipEventRecord(p->ev1, p->stream));
  RIP_HIP(hipEventRecord(p->ev4, p->stream));
  pool_read_ctl(p, record_events);
  float ms = 0.0f;
  RIP_HIP(hipEventElapsedTime(&ms, p->ev3, p->ev4));
  p->wave_ms = ms;
  p->wave_ran = true;
  for (int i = 0; i < RIP_STAT_COUNT; ++i) p->wave_stats[i] = p->h_ctl[kCtlStatBytes + i];
  return p->h_ctl[kCtlLongCount];
}

void stage_scratch_free(WaveScratch &w) {
  dev_free(w.d_shtab);
  dev_free(w.d_slist);
  dev_free(w.d_ssort);
  w.stage_waves = w.cap_ssort = 0;
}

}  // namespace rip
