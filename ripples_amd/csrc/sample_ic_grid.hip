// Grid sampler: the IC samples that outgrow a lane's list, 64 per colour
// group and many groups per batch, expanded by the whole GPU one BFS level at
// a time.
//
// Semantics are those of AddRRRSet (add_rrrset.h:105-157) under the stream
// contract (common.h, ic_gap.h): the set is the reverse closure of the root
// over live edges, so any expansion order gives the sets of the other
// samplers and the oracle bit for bit.  The colour-per-sample idea is that of
// BatchedBFSNeighborColor (batched_add_rrrset.h:184-257); the reference's GPU
// form runs one BFS level per kernel as well (gpu/bfs.h:1338-1680).
//
// Samples that reach a giant component (R-MAT with U[0,0.1] or U[0,0.02]
// weights) visit hundreds of thousands of vertices each.  Per group g (64
// samples, colour c = bit c) the scratch holds
//   vp[g][v] = (vis, pend) : colour masks of the visited and of the not yet
//                            expanded colours of vertex v, side by side in
//                            one 16-byte pair (dense, n pairs per group), so
//                            a discovery's two atomics touch one cache line
//   bm0[g], bm1[g]        : bitmap of the group's union and its summary
// so the groups of a batch cost 16 bytes per vertex each, which bounds the
// batch by memory rather than by the number of workgroups: every level is
// one persistent kernel over the frontier items (g, v) of all groups of the
// batch.  A wave takes 64 items, a lane each: its pending colours with one
// exchange, its record, and the number of its units, a unit being one colour
// and one gap block.  The wave's units are dealt out over its lanes 64 at a
// time, the colours of a block side by side (they read the same few lines of
// thresholds); a lane draws its block's candidates, reads their thresholds
// together, and the live edges join a queue of the wave in LDS.  When the
// queue holds 64 kDiscover of them they are discovered at once, kDiscover to a
// lane and stage by stage: the in-neighbours, the vis words (most edges in a
// giant component reach vertices the colour has visited), the atomicOr on
// vis, on the union bitmap and on pend; (g, u) joins the next frontier when
// its pend word was zero, through another queue in LDS.  Items of kHeavyUnits
// units or more (hub rows pending for many colours) are cut into segments
// that a second kernel of the level spreads over all waves.  A frontier longer
// than its buffer sets an overflow flag; the vertices it could not list keep
// their pend bits, and a scan of pend finds them once the listed frontier is
// done.
//
// What bounds it: requests to memory, 16 waves a CU holding dozens each and
// meeting no workgroup barrier.  20,000 sets of an R-MAT graph of 2^24
// vertices with U[0,0.02] weights (1.8e9 live edges, 3.7e9 candidates): 94 ms
// in these kernels, where random 8-byte loads (55e9/s) and atomics (20e9/s) of
// the live and the fresh edges alone take about that long.  Chunks of rows
// per workgroup, expanded in barriered phases, took 320 ms.  Batches of 2, 3,
// 4, 6 and 8 discoveries a lane (pool call and selection): 222, 170, 145, 126
// and 125 ms while every batch reserved its own frontier entries, 117 ms for 3
// and 4 with the queue of entries, whose LDS costs larger batches the fourth
// workgroup of a CU (126 ms).
//
// After the last level, one workgroup per group reads its union in vertex
// order from the bitmaps (clearing them and vis), keeps the group's hot
// members in a column of the pool's column store when they are many, and
// writes each colour's sorted list through one reservation of pool space.
#include <algorithm>
#include <vector>

#include "device_util.h"
#include "ic_common.h"
#include "ic_expand.h"
#include "ic_gap.h"
#include "internal.h"

namespace rip {
namespace {

constexpr int kExpBT = 256;            // level and tail kernels
constexpr uint32_t kDiscover = 3;      // queued edges a lane discovers at once
constexpr uint32_t kQueue = 64 * (kDiscover + kUnitBatch);  // a wave's queue of live edges
constexpr uint32_t kHeavyUnits = 2048; // units from which an item is cut up (8192: the same time)
constexpr uint32_t kSegUnits = 1024;   // units of a segment
constexpr uint32_t kOut = 128;         // a wave's queue of frontier entries
constexpr uint32_t kMinTake = 8;       // fewest items a wave takes at a time
constexpr int kGridWaves = 4;          // waves a SIMD holds (a quarter of LDS per workgroup)
// level counters kept on the device (a ring), and levels enqueued per host
// synchronisation: a BFS of hundreds of narrow levels costs a launch per
// level, not a round trip
constexpr uint32_t kRing = 64;
constexpr uint32_t kLevelsPerSync = 16;
// a frontier of at most this many items is expanded by one workgroup that
// runs level after level with a barrier between them (no launch per level):
// the long thin tails of deep samples (32 to 128 measured the same).
constexpr uint64_t kTailItems = 128;

// room for the heavy items of a level and their segments (8 and 8 MiB), no
// more than a level may list; what finds none is expanded by its own wave
constexpr uint32_t kHeavyCap = 1u << 19, kSegCap = 1u << 20;

// control words of the grid scratch
enum : int { kGOver = 0, kGLevels = 1, kGCount = 2, kGTail = 3, kGWords = 4 };

struct GridParams {
  const VertexRec *vrec;
  const uint32_t *ids;
  const uint32_t *val;
  uint32_t n;
  Affine step;
  unsigned long long *vp;          // groups x n pairs (visited, pending colours)
  uint32_t *bm0, *bm1;             // groups x nw0, groups x nw1
  uint32_t nw0, nw1;
  const unsigned long long *z;     // groups x 64: element 0 of each colour's sample
  const unsigned long long *cur;   // frontier items g << 32 | v
  uint64_t ncur;
  unsigned long long *next;        // next frontier
  unsigned long long *next_cnt;    // its length (counts every append, also past cap)
  uint64_t cap;                    // capacity of next
  unsigned long long *gctl;        // control words: overflow flag, level count
  unsigned long long *ring;        // per level L, words k kRing + L % kRing: frontier length,
                                   // items taken, heavy items, their segments, segments taken
  unsigned long long *heavy;       // heavy items of a level: (g << 32 | v, colours) pairs
  unsigned long long *segs;        // their segments: heavy index << 32 | segment
  uint32_t heavy_cap, seg_cap;
  unsigned long long *buf[2];      // level L reads buf[L % 2], writes buf[(L + 1) % 2]
  unsigned long long *ctl;         // the pool's control words (work counters)
};

// The j-th set bit of m (j < popcount(m)).
__device__ inline uint32_t nth_bit(uint64_t m, uint32_t j) {
  uint32_t pos = 0;
  uint32_t c = __popc(static_cast<uint32_t>(m));
  uint32_t w = static_cast<uint32_t>(m);
  if (j >= c) {
    j -= c;
    w = static_cast<uint32_t>(m >> 32);
    pos = 32;
  }
  c = __popc(w & 0xFFFFu);
  if (j >= c) { j -= c; w >>= 16; pos += 16; }
  c = __popc(w & 0xFFu);
  if (j >= c) { j -= c; w >>= 8; pos += 8; }
  c = __popc(w & 0xFu);
  if (j >= c) { j -= c; w >>= 4; pos += 4; }
  c = __popc(w & 0x3u);
  if (j >= c) { j -= c; w >>= 2; pos += 2; }
  if (j >= (w & 1u)) pos += 1;
  return pos;
}

// Marks the colours `bits` of group g discovered at u (for lanes with live
// set); (g, u) joins the next frontier when its pend word was zero.  Every
// lane of the wave must call it.
__device__ inline void grid_discover(const GridParams &P, bool live, uint32_t g, uint32_t u,
                                     unsigned long long bits) {
  bool push = false;
  if (live) {
    const uint64_t idx = static_cast<uint64_t>(g) * P.n + u;
    // vis is written by atomics, which complete in L2; the read goes there too
    unsigned long long old = __hip_atomic_load(&P.vp[2 * idx], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
    if (bits & ~old) {
      old = atomicOr(&P.vp[2 * idx], bits);
      const unsigned long long fresh = bits & ~old;
      if (fresh) {
        if (old == 0) {
          uint32_t *b0 = P.bm0 + static_cast<uint64_t>(g) * P.nw0;
          const uint32_t o0 = atomicOr(&b0[u >> 5], 1u << (u & 31u));
          if (o0 == 0)
            atomicOr(&P.bm1[static_cast<uint64_t>(g) * P.nw1 + (u >> 10)], 1u << ((u >> 5) & 31u));
        }
        push = atomicOr(&P.vp[2 * idx + 1], fresh) == 0;
      }
    }
  }
  const uint64_t m = __ballot(push);
  if (m == 0) return;
  const uint32_t leader = __ffsll(static_cast<unsigned long long>(m)) - 1;
  unsigned long long base = 0;
  if (lane_id() == leader) base = atomicAdd(P.next_cnt, static_cast<unsigned long long>(__popcll(m)));
  base = __shfl(base, static_cast<int>(leader), 64);
  if (push) {
    const unsigned long long at = base + __popcll(m & lanes_below());
    if (at < P.cap) P.next[at] = (static_cast<unsigned long long>(g) << 32) | u;
  }
}

__device__ inline unsigned long long wave_or_u64(unsigned long long v) {
  for (int d = 32; d > 0; d >>= 1) v |= __shfl_xor(v, d, 64);
  return v;
}

// Batch start: the root of every colour of every group (one 64-lane block
// per group; lanes past the group's colours have no sample).
__global__ void __launch_bounds__(64) grid_seed_kernel(GridParams P, const uint32_t *nb) {
  const uint32_t g = blockIdx.x, c = threadIdx.x;
  const bool has = c < nb[g];
  const unsigned long long z = P.z[64ull * g + c];
  const uint32_t root = has ? uniform_index(z, P.n) : 0u;
  grid_discover(P, has, g, root, 1ull << c);
}

enum : int { kRFront = 0, kRTaken = 1, kRHeavy = 2, kRSegs = 3, kRSegTaken = 4, kRWords = 5 };

__device__ inline unsigned long long *ring_word(const GridParams &P, int k, uint32_t L) {
  return &P.ring[static_cast<uint32_t>(k) * kRing + L % kRing];
}

// A row to expand: the vertex's record, the group and its pending colours.
struct Row {
  uint64_t q, ja, jb;
  unsigned long long M;
  double inv;
  uint32_t begin, deg, ufull, ulast, g;
  uint32_t tf;      // thr | beta << 25 | (threshold shared by the row) << 30
};
static_assert(sizeof(Row) == 64 && kIcOne < 1u << 25 && kIcBetaMax < 32, "packed row");

// A workgroup's tables, and per wave the rows being expanded and the queue of
// live edges to discover (the edge, and group << 6 | colour) and that of the
// next level's entries.
template <int BT>
struct ExpandLds {
  Affine p2[64];
  IcGapTab tab;
  Row row[BT / 64][64];
  uint32_t qe[BT / 64][kQueue], qg[BT / 64][kQueue];
  unsigned long long qo[BT / 64][kOut];
};

// A wave's side of the expansion; every lane of the wave calls each method.
template <int BT>
struct Expander {
  const GridParams &P;
  ExpandLds<BT> &S;
  const uint32_t wid, lane;
  uint32_t qn = 0, on = 0;   // edges and frontier entries queued (wave-uniform)
  // a lane's work: blocks drawn and gaps after a block's first, candidates
  // and those whose threshold was read, live edges, rows
  uint32_t gaps = 0, cand = 0, vals = 0, live = 0, exp = 0;

  __device__ Expander(const GridParams &p, ExpandLds<BT> &s)
      : P(p), S(s), wid(threadIdx.x >> 6), lane(lane_id()) {}

  // Appends the wave's frontier entries to the next level's list.
  __device__ void flush() {
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(P.next_cnt, static_cast<unsigned long long>(on));
    base = uniform_u64(base);
    for (uint32_t i = lane; i < on; i += 64)
      if (base + i < P.cap) P.next[base + i] = S.qo[wid][i];
    on = 0;
  }

  // Discovers the last 64 kDiscover queued edges, or all when they are fewer,
  // stage by stage over a lane's kDiscover entries, so that each stage's
  // requests are in flight together.  Entries may name the same (g, u): the
  // atomics on vis settle which of them finds a colour fresh.
  __device__ void discover() {
    const uint32_t take = min(qn, 64u * kDiscover), q0 = qn - take;
    uint32_t gc[kDiscover], u[kDiscover];
    bool fresh[kDiscover], first[kDiscover], push[kDiscover];
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      const uint32_t at = q0 + i * 64 + lane;
      fresh[i] = at < qn;
      gc[i] = fresh[i] ? S.qg[wid][at] : 0u;
      u[i] = fresh[i] ? P.ids[S.qe[wid][at]] : 0u;
    }
    auto vis = [&](uint32_t i) {
      return &P.vp[2 * (static_cast<uint64_t>(gc[i] >> 6) * P.n + u[i])];
    };
    unsigned long long old[kDiscover];
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      // vis is written by atomics, which complete in L2; the read goes there too
      old[i] = fresh[i] ? __hip_atomic_load(vis(i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
    }
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      fresh[i] = fresh[i] && ((old[i] >> (gc[i] & 63u)) & 1ull) == 0;
      if (fresh[i]) old[i] = atomicOr(vis(i), 1ull << (gc[i] & 63u));
    }
    // the bitmap's and the pend word's atomics go out together; the summary
    // bit needs the bitmap's old word
    uint32_t o0[kDiscover];
    unsigned long long pend[kDiscover];
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      fresh[i] = fresh[i] && ((old[i] >> (gc[i] & 63u)) & 1ull) == 0;
      first[i] = fresh[i] && old[i] == 0;
      o0[i] = 0;
      pend[i] = 0;
      if (first[i])
        o0[i] = atomicOr(&P.bm0[static_cast<uint64_t>(gc[i] >> 6) * P.nw0 + (u[i] >> 5)],
                         1u << (u[i] & 31u));
      if (fresh[i]) pend[i] = atomicOr(vis(i) + 1, 1ull << (gc[i] & 63u));
    }
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      push[i] = fresh[i] && pend[i] == 0;
      if (first[i] && o0[i] == 0)
        atomicOr(&P.bm1[static_cast<uint64_t>(gc[i] >> 6) * P.nw1 + (u[i] >> 10)],
                 1u << ((u[i] >> 5) & 31u));
    }
#pragma unroll
    for (uint32_t i = 0; i < kDiscover; ++i) {
      const uint64_t m = __ballot(push[i]);
      const uint32_t k = static_cast<uint32_t>(__popcll(m));
      if (on + k > kOut) flush();
      if (push[i])
        S.qo[wid][on + __popcll(m & lanes_below())] =
            (static_cast<unsigned long long>(gc[i] >> 6) << 32) | u[i];
      on += k;
    }
    qn = q0;
  }

  // Expands `units` units of each lane's row, from its unit rbase on; unit r
  // of a row is block r / |M| for the r % |M|-th of its colours M.
  __device__ void run(uint32_t units, uint64_t rbase) {
    const uint32_t incl = wave_inclusive_scan(units);
    const uint32_t total = uniform_u32(__shfl(incl, 63, 64));
    const Affine A = uniform_affine(S.p2[0]), A2 = uniform_affine(S.p2[1]);
    for (uint32_t u0 = 0; u0 < total; u0 += 64) {
      const uint32_t u = u0 + lane;
      uint32_t j = 0;   // the first lane whose inclusive prefix passes u
#pragma unroll
      for (uint32_t s = 32; s > 0; s >>= 1)
        if (__shfl(incl, static_cast<int>(j + s - 1), 64) <= u) j += s;
      const uint32_t before = __shfl(incl, static_cast<int>(j ? j - 1 : 0), 64);
      uint32_t gc = 0, e0 = 0, len = 0, T = 0;
      uint64_t x = 0, q = 0;
      double inv = 0.0;
      bool uniform = true, more = false;
      if (u < total) {
        const Row &R = S.row[wid][j];
        const uint64_t r = rbase + (u - (j ? before : 0u));
        const unsigned long long M = R.M;
        const uint32_t ncol = static_cast<uint32_t>(__popcll(M));
        const uint32_t k = r >> 32 ? static_cast<uint32_t>(r / ncol)
                                   : static_cast<uint32_t>(r) / ncol;
        const uint32_t c = nth_bit(M, static_cast<uint32_t>(r - static_cast<uint64_t>(k) * ncol));
        const uint32_t tf = R.tf, beta = (tf >> 25) & 31u;
        gc = (R.g << 6) | c;
        // block k's first element: 2 B k elements after the row's first
        x = R.ja * P.z[gc] + R.jb;
        e0 = R.begin + (k << beta);
        len = min(R.deg - (k << beta), 1u << beta);
        T = tf & 0x1FFFFFFu;
        q = R.q;
        inv = R.inv;
        uniform = (tf >> 30) != 0;
        for (uint32_t kk = k, bit = beta + 1; kk; kk >>= 1, ++bit)
          if (kk & 1) x = aff_apply(S.p2[bit], x);
        ++gaps;
        // a block without candidates costs one compare
        more = (x >> 32) + 1 > (len == 1u << beta ? R.ufull : R.ulast);
      }
      uint32_t pos = 0;
      while (__ballot(more)) {
        uint32_t ce[kUnitBatch], th[kUnitBatch], t[kUnitBatch];
        const uint32_t nc = ic_draw_block<kUnitBatch>(x, pos, more, len, T, q, inv, uniform, A, A2,
                                                      &S.tab, ce, th);
        gaps += nc - (nc != 0 && pos == len ? 1u : 0u);
#pragma unroll
        for (uint32_t i = 0; i < kUnitBatch; ++i)
          t[i] = i < nc && !uniform ? P.val[e0 + ce[i]] : 0xFFFFFFFFu;
        cand += nc;
        if (!uniform) vals += nc;
#pragma unroll
        for (uint32_t i = 0; i < kUnitBatch; ++i) {
          const bool on = i < nc && t[i] > th[i];
          const uint64_t m = __ballot(on);
          if (on) {
            const uint32_t at = qn + static_cast<uint32_t>(__popcll(m & lanes_below()));
            S.qe[wid][at] = e0 + ce[i];
            S.qg[wid][at] = gc;
            ++live;
          }
          qn += static_cast<uint32_t>(__popcll(m));
        }
        if (qn >= 64 * kDiscover) discover();
      }
    }
  }

  // Lane's row: vertex v of group g, pending for the colours M (0: none).
  // Returns its units.
  __device__ uint64_t load(uint32_t g, uint32_t v, unsigned long long M) {
    if (!M) return 0;
    const VertexRec rv = P.vrec[v];
    if (!rv.thr) return 0;
    const uint32_t beta = (rv.flags >> kBetaShift) & 31u;
    S.row[wid][lane] = Row{rv.q, rv.ja, rv.jb, M, rv.inv, rv.begin, rv.end - rv.begin, rv.ufull,
                           rv.ulast, g,
                           rv.thr | beta << 25 | (rv.flags & kRowUniform ? 1u << 30 : 0u)};
    return static_cast<uint64_t>(__popcll(M)) * (((rv.end - rv.begin - 1) >> beta) + 1);
  }

  // Leaves an item of `all` units to the level's heavy kernel; false when
  // there is no room for it.
  __device__ bool defer(uint32_t L, unsigned long long item, unsigned long long M, uint64_t all) {
    const uint64_t nseg = (all + kSegUnits - 1) / kSegUnits;
    const unsigned long long h = atomicAdd(ring_word(P, kRHeavy, L), 1ull);
    if (h >= P.heavy_cap) return false;
    P.heavy[2 * h] = item;
    P.heavy[2 * h + 1] = M;
    const unsigned long long s0 = atomicAdd(ring_word(P, kRSegs, L), nseg);
    const bool fits = s0 + nseg <= P.seg_cap;
    const uint64_t end = fits ? s0 + nseg : P.seg_cap;
    for (uint64_t i = s0; i < end; ++i) P.segs[i] = fits ? (h << 32) | (i - s0) : ~0ull;
    return fits;
  }

  // Up to 64 frontier items, one per lane, of level L; with `here` also the
  // heavy ones are expanded by this wave.
  __device__ void items(bool have, unsigned long long item, uint32_t L, bool here) {
    const uint32_t g = static_cast<uint32_t>(item >> 32), v = static_cast<uint32_t>(item);
    // the colours still to expand at v; a repeated item finds none
    unsigned long long M = 0;
    if (have) M = atomicExch(&P.vp[2 * (static_cast<uint64_t>(g) * P.n + v) + 1], 0ull);
    if (M) ++exp;
    const uint64_t all = load(g, v, M);
    uint64_t left = 0;     // units of a heavy item to expand here
    uint32_t units = static_cast<uint32_t>(all);
    if (all >= kHeavyUnits) {
      units = 0;
      if (here || !defer(L, item, M, all)) left = all;
    }
    // the light items together, then the heavy ones one by one
    uint64_t from = 0;
    for (;;) {
      run(units, from);
      const uint64_t m = __ballot(left != 0);
      if (!m) break;
      const uint32_t j = __ffsll(static_cast<unsigned long long>(m)) - 1;
      const uint64_t lj = uniform_u64(__shfl(left, static_cast<int>(j), 64));
      const uint64_t aj = uniform_u64(__shfl(all, static_cast<int>(j), 64));
      const uint32_t now = static_cast<uint32_t>(min(lj, static_cast<uint64_t>(1) << 30));
      from = aj - lj;
      units = lane == j ? now : 0u;
      if (lane == j) left -= now;
    }
  }

  __device__ void finish() {
    while (qn) discover();
    if (on) flush();
  }

  __device__ void report() {
    report_stats(P.ctl, static_cast<unsigned long long>(kIcRecBytes) * exp + 4ull * vals + 4ull * live,
                 cand, static_cast<unsigned long long>(gaps) + vals, exp, live);
  }
};

template <int BT>
__device__ inline void expand_tables(const GridParams &P, ExpandLds<BT> &S) {
  if (threadIdx.x == 0) fill_step_powers(P.step, S.p2);
  ic_load_tables(&S.tab);
  __syncthreads();
}

// BFS level L: the frontier is buf[L % 2][0, n) with n the level's frontier
// length (its first cap entries when it overflowed, which raises the overflow
// flag); waves take up to 64 items at a time, fewer when the frontier would
// leave waves without any.  Levels are enqueued ahead of the host: a level
// whose frontier is empty costs its launches only.
template <int BT>
__global__ void __launch_bounds__(BT, kGridWaves) grid_level_kernel(GridParams P, uint32_t L) {
  constexpr uint32_t NW = BT / 64;
  __shared__ ExpandLds<BT> S;
  const uint64_t raw = __hip_atomic_load(ring_word(P, kRFront, L), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  const uint64_t ncur = raw < P.cap ? raw : P.cap;
  if (blockIdx.x == 0 && threadIdx.x == 0 && ncur) {
    P.gctl[kGLevels] += 1;
    if (raw > P.cap) P.gctl[kGOver] = 1;
  }
  const uint64_t waves = static_cast<uint64_t>(gridDim.x) * NW;
  const uint64_t each = (ncur + waves - 1) / waves;
  const uint32_t take = each >= 64 ? 64u : max(kMinTake, static_cast<uint32_t>(each));
  if (static_cast<uint64_t>(blockIdx.x) * NW * take >= ncur) return;   // no items for it
  P.next = L & 1u ? P.buf[0] : P.buf[1];
  P.next_cnt = ring_word(P, kRFront, L + 1);
  const unsigned long long *cur = L & 1u ? P.buf[1] : P.buf[0];
  expand_tables<BT>(P, S);
  Expander<BT> E(P, S);
  // a wave's first items are its own, later ones claimed past everyone's
  const uint64_t own = waves * take;
  for (uint64_t i0 = (static_cast<uint64_t>(blockIdx.x) * NW + E.wid) * take; i0 < ncur;) {
    const bool have = E.lane < take && i0 + E.lane < ncur;
    E.items(have, have ? cur[i0 + E.lane] : 0ull, L, false);
    if (own >= ncur) break;
    unsigned long long c = 0;
    if (E.lane == 0) c = atomicAdd(ring_word(P, kRTaken, L), static_cast<unsigned long long>(take));
    i0 = own + uniform_u64(c);
  }
  E.finish();
  E.report();
}

// The segments of level L's heavy items, one to a wave at a time.
template <int BT>
__global__ void __launch_bounds__(BT, kGridWaves) grid_heavy_kernel(GridParams P, uint32_t L) {
  __shared__ ExpandLds<BT> S;
  const uint64_t raw = __hip_atomic_load(ring_word(P, kRSegs, L), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  const uint64_t nseg = raw < P.seg_cap ? raw : P.seg_cap;
  if (static_cast<uint64_t>(blockIdx.x) * (BT / 64) >= nseg) return;
  P.next = L & 1u ? P.buf[0] : P.buf[1];
  P.next_cnt = ring_word(P, kRFront, L + 1);
  expand_tables<BT>(P, S);
  Expander<BT> E(P, S);
  for (;;) {
    unsigned long long i = 0;
    if (E.lane == 0) i = atomicAdd(ring_word(P, kRSegTaken, L), 1ull);
    i = uniform_u64(i);
    if (i >= nseg) break;
    const unsigned long long s = uniform_u64(P.segs[i]);
    if (s == ~0ull) continue;
    const unsigned long long item = P.heavy[2 * (s >> 32)], M = P.heavy[2 * (s >> 32) + 1];
    const uint64_t all = E.load(static_cast<uint32_t>(item >> 32), static_cast<uint32_t>(item),
                                E.lane == 0 ? M : 0ull);
    const uint64_t a = (s & 0xFFFFFFFFull) * kSegUnits;
    E.run(all > a ? static_cast<uint32_t>(min(all - a, static_cast<uint64_t>(kSegUnits))) : 0u, a);
  }
  E.finish();
  E.report();
}

// Levels L0, L0 + 1, ... by one workgroup while the frontier holds between 1
// and tail_cap items: each level zeroes the next level's length, expands its
// items, an even share to each wave, and meets the next level at a barrier.
// Stops at the first level whose frontier is empty or longer than tail_cap and
// leaves its number in gctl[kGTail]; that level's length stays in the ring for
// the level kernels.
template <int BT>
__global__ void __launch_bounds__(BT, kGridWaves) grid_tail_kernel(GridParams P, uint32_t L0,
                                                          uint64_t tail_cap) {
  constexpr uint32_t NW = BT / 64;
  __shared__ ExpandLds<BT> S;
  __shared__ unsigned long long s_n;
  const uint32_t tid = threadIdx.x;
  expand_tables<BT>(P, S);
  Expander<BT> E(P, S);
  uint32_t L = L0;
  for (;; ++L) {
    // the previous level's appends are done: the waves' own stores first
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
      const unsigned long long raw = __hip_atomic_load(ring_word(P, kRFront, L), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
      s_n = raw;
      if (raw != 0 && raw <= tail_cap) {
        __hip_atomic_store(ring_word(P, kRFront, L + 1), 0ull, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        P.gctl[kGLevels] += 1;
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const uint64_t ncur = s_n;
    if (ncur == 0 || ncur > tail_cap) break;
    P.next = L & 1u ? P.buf[0] : P.buf[1];
    P.next_cnt = ring_word(P, kRFront, L + 1);
    const unsigned long long *cur = L & 1u ? P.buf[1] : P.buf[0];
    const uint64_t share = min(64ull, (ncur + NW - 1) / NW);
    for (uint64_t i0 = E.wid * share; i0 < ncur; i0 += NW * share) {
      const bool have = E.lane < share && i0 + E.lane < ncur;
      E.items(have, have ? cur[i0 + E.lane] : 0ull, L, true);
    }
    E.finish();
  }
  if (tid == 0) P.gctl[kGTail] = L;
  E.report();
}

// Zeroes the frontier lengths of levels a .. a + k - 1 and the other counters
// of levels a - 1 .. a + k - 2 (ring indices mod kRing), or, with `all`, the
// whole ring and the control words.
__global__ void grid_ring_kernel(unsigned long long *ring, unsigned long long *gctl, uint32_t a,
                                 uint32_t k, uint32_t all) {
  const uint32_t i = threadIdx.x;
  if (all) {
    for (uint32_t j = i; j < kRWords * kRing; j += blockDim.x) ring[j] = 0;
    if (i < kGWords) gctl[i] = 0;
    return;
  }
  if (i < k) {
    ring[(a + i) % kRing] = 0;
    for (uint32_t w = 1; w < kRWords; ++w) ring[w * kRing + (a + i - 1) % kRing] = 0;
  }
}

// Frontier from the pend words (after an overflow): every (g, v) of groups
// [0, groups) with colours still to expand.
__global__ void grid_rebuild_kernel(GridParams P, uint32_t groups) {
  const uint64_t total = static_cast<uint64_t>(groups) * P.n;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * blockDim.x; i0 < total; i0 += stride) {
    const uint64_t i = i0 + threadIdx.x;
    const bool push = i < total && __hip_atomic_load(&P.vp[2 * i + 1], __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT) != 0;
    const uint64_t m = __ballot(push);
    if (m == 0) continue;
    const uint32_t leader = __ffsll(static_cast<unsigned long long>(m)) - 1;
    unsigned long long base = 0;
    if (lane_id() == leader)
      base = atomicAdd(P.next_cnt, static_cast<unsigned long long>(__popcll(m)));
    base = __shfl(base, static_cast<int>(leader), 64);
    if (push) {
      const unsigned long long at = base + __popcll(m & lanes_below());
      const uint64_t g = i / P.n, v = i - g * P.n;
      if (at < P.cap) P.next[at] = (g << 32) | v;
    }
  }
}


// Union size of every group: the set bits of its bitmap.
__global__ void __launch_bounds__(1024) grid_union_kernel(const uint32_t *bm0, uint32_t nw0,
                                                          unsigned long long *out) {
  __shared__ uint32_t s_w[16];
  const uint32_t *b = bm0 + static_cast<uint64_t>(blockIdx.x) * nw0;
  uint32_t acc = 0;
#pragma unroll 8
  for (uint32_t i = threadIdx.x; i < nw0; i += 1024) acc += __popc(b[i]);
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (uint32_t w = 0; w < 16; ++w) t += s_w[w];
    out[blockIdx.x] = t;
  }
}

// ------------------------------------------------------------------ output
// After a batch's last level the groups' sets are written in four steps,
// each spread over many workgroups per group:
//   1. union lists: the group's bitmap is cut into kRanges ranges of summary
//      words; one kernel counts each range's members, the next writes them in
//      vertex order into the group's staging (list + colour masks), clearing
//      bitmaps and vis on the way;
//   2. per chunk of kChunk staging entries (one wave each): members of each
//      colour, all and hot ones;
//   3. per group: the column decision, each colour's offsets over the chunks,
//      one reservation of pool space, the sets' offsets and lengths;
//   4. per chunk: hot members into the group's column (when it has one), the
//      rest scattered to their colours' sorted lists.
constexpr uint32_t kRanges = 256;   // a wave each in step 1
constexpr uint32_t kChunk = 2048;   // staging entries per wave of steps 2 and 4

struct OutParams {
  uint32_t n, nw0, nw1;
  unsigned long long *vp;
  uint32_t *bm0, *bm1;
  uint32_t g0;                          // first group of this sub-batch
  uint32_t groups;                      // groups of the sub-batch
  const unsigned long long *soff;       // per group of the sub-batch: staging offset
  uint32_t *slist;                      // staging: union lists
  unsigned long long *smask;            // staging: union masks
  unsigned long long *rc;               // groups x kRanges: range member counts
  const unsigned long long *cbase;      // groups + 1: first chunk of each group
  const unsigned long long *usz;        // groups: union sizes
  uint32_t *cc;                         // chunks x 64: members per colour (then offsets)
  uint32_t *cch;                        // chunks x 64: hot members per colour
  unsigned long long *dbase;            // groups x 64: pool offset of each colour's list
  uint32_t *gcol;                       // groups: column of the group, or kNoGroup
  uint32_t *gfail;                      // groups: pool space ran out (nothing is written)
  const uint32_t *sid;                  // groups x 64 sample ids (kNoGroup: none)
  const uint32_t *nb;                   // colours per group
  unsigned long long *set_off;
  uint32_t *set_len;
  uint32_t *data;
  uint64_t cap_data;
  unsigned long long *ctl;
  // column store (colptr == nullptr: every set a list)
  unsigned long long *const *colptr;
  uint32_t *gsample;
  uint32_t *gref;
  const uint32_t *hot_index;
  uint32_t hot_n;
  uint32_t group_base;
};

// Summary words [lo, hi) of range r of a group with nw1 of them.
__device__ inline void range_of(uint32_t nw1, uint32_t r, uint32_t *lo, uint32_t *hi) {
  *lo = static_cast<uint32_t>(static_cast<uint64_t>(nw1) * r / kRanges);
  *hi = static_cast<uint32_t>(static_cast<uint64_t>(nw1) * (r + 1) / kRanges);
}

// f(w, word) for summary words [lo, hi), two at a time: each lane gets one of
// their 64 bitmap words (0 where the summary has no bit), word w + lane.
template <typename F>
__device__ inline void range_words(const uint32_t *bm0, const uint32_t *bm1, uint32_t lo,
                                   uint32_t hi, F &&f) {
  const uint32_t lane = lane_id();
  for (uint32_t w1i = lo; w1i < hi; w1i += 2) {
    const uint32_t mine = w1i + (lane >> 5);
    const uint32_t s1 = mine < hi ? bm1[mine] : 0u;
    const uint32_t w = w1i * 32;
    f(w, (s1 >> (lane & 31u)) & 1u ? bm0[w + lane] : 0u);
  }
}

// Step 1a: members of each (group, range).
__global__ void __launch_bounds__(64) out_range_count_kernel(OutParams P) {
  const uint32_t i = blockIdx.x / kRanges, r = blockIdx.x % kRanges;
  const uint32_t g = P.g0 + i;
  uint32_t lo, hi;
  range_of(P.nw1, r, &lo, &hi);
  uint32_t cnt = 0;
  range_words(P.bm0 + static_cast<uint64_t>(g) * P.nw0, P.bm1 + static_cast<uint64_t>(g) * P.nw1,
              lo, hi, [&](uint32_t, uint32_t word) { cnt += __popc(word); });
  cnt = wave_sum(cnt);
  if (lane_id() == 0) P.rc[blockIdx.x] = cnt;
}

// Step 1b: the members of each (group, range) into the staging in vertex
// order, a lane per member; bitmaps and vis cleared on the way.  256 groups on
// an R-MAT graph of 2^24 vertices (U[0,0.02] weights): 1.4 ms, 5.6 with a lane
// per summary word that wrote its members one by one through atomics.
__global__ void __launch_bounds__(64) out_range_write_kernel(OutParams P) {
  const uint32_t i = blockIdx.x / kRanges, r = blockIdx.x % kRanges;
  const uint32_t g = P.g0 + i, lane = lane_id();
  uint32_t *bm0 = P.bm0 + static_cast<uint64_t>(g) * P.nw0;
  uint32_t *bm1 = P.bm1 + static_cast<uint64_t>(g) * P.nw1;
  unsigned long long *vp = P.vp + 2 * static_cast<uint64_t>(g) * P.n;
  unsigned long long at = 0;
  for (uint32_t q = lane; q < r; q += 64) at += P.rc[i * kRanges + q];
  for (int d = 32; d > 0; d >>= 1) at += __shfl_xor(at, d, 64);
  uint32_t *list = P.slist + P.soff[i];
  unsigned long long *masks = P.smask + P.soff[i];
  uint32_t lo, hi;
  range_of(P.nw1, r, &lo, &hi);
  range_words(bm0, bm1, lo, hi, [&](uint32_t w, uint32_t word) {
    const uint32_t cnt = __popc(word), incl = wave_inclusive_scan(cnt);
    const uint32_t total = uniform_u32(__shfl(incl, 63, 64));
    if (total == 0) return;
    if (word) bm0[w + lane] = 0;
    if (lane == 0) bm1[w / 32] = 0;
    if (lane == 32 && w / 32 + 1 < hi) bm1[w / 32 + 1] = 0;
    for (uint32_t t0 = 0; t0 < total; t0 += 64) {
      const uint32_t t = t0 + lane;
      uint32_t j = 0;   // the first lane whose inclusive prefix passes t
#pragma unroll
      for (uint32_t d = 32; d > 0; d >>= 1)
        if (__shfl(incl, static_cast<int>(j + d - 1), 64) <= t) j += d;
      const int src = static_cast<int>(min(j, 63u));
      const uint32_t k = t - (__shfl(incl, src, 64) - __shfl(cnt, src, 64));
      const uint32_t bits = __shfl(word, src, 64);
      if (t < total) {
        const uint32_t v = (w + src) * 32 + nth_bit(bits, k);
        list[at + t] = v;
        masks[at + t] = vp[2ull * v];
        vp[2ull * v] = 0;
      }
    }
    at += total;
  });
}

// The group of chunk c (cbase is ascending, groups + 1 entries).
__device__ inline uint32_t group_of_chunk(const unsigned long long *cbase, uint32_t groups,
                                          uint64_t c) {
  uint32_t lo = 0, hi = groups;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (cbase[mid + 1] <= c) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// The wave's 64 x 64 bit matrix (lane l holds row l) transposed.
__device__ inline unsigned long long transpose64(unsigned long long x) {
  const uint32_t lane = lane_id();
  unsigned long long m = 0x00000000FFFFFFFFull;   // the columns without bit s
#pragma unroll
  for (uint32_t s = 32; s > 0; s >>= 1, m ^= m << s) {
    const unsigned long long y = __shfl_xor(x, static_cast<int>(s), 64);
    x = lane & s ? (x & ~m) | ((y >> s) & m) : (x & m) | ((y & m) << s);
  }
  return x;
}

// Step 2: per chunk (one wave), members of each colour, all and hot: 64 members'
// masks are transposed, so that a lane counts its colour at once.  That is about
// 100 instructions, against 8 for each colour they hold by ballots (20,000 sets
// on an R-MAT graph of 2^24 vertices and a selection: 105.4 ms by ballots, 104.2
// so; twenty sets on one of 2^21 2.20 either way).
__global__ void __launch_bounds__(64) out_chunk_count_kernel(OutParams P) {
  const uint64_t c = blockIdx.x;
  const uint32_t i = group_of_chunk(P.cbase, P.groups, c);
  const uint32_t lane = lane_id();
  const uint64_t e0 = (c - P.cbase[i]) * kChunk;
  const uint64_t e1 = min(e0 + kChunk, P.usz[i]);
  const uint32_t *list = P.slist + P.soff[i];
  const unsigned long long *masks = P.smask + P.soff[i];
  uint32_t all = 0, hot = 0;   // lane j: colour j's counts
  for (uint64_t t = e0; t < e1; t += 64) {
    const uint64_t e = t + lane;
    const bool h = P.colptr && e < e1 && P.hot_index[list[e]] != kNotHot;
    const unsigned long long col = transpose64(e < e1 ? masks[e] : 0ull);
    all += static_cast<uint32_t>(__popcll(col));
    hot += static_cast<uint32_t>(__popcll(col & __ballot(h)));
  }
  P.cc[c * 64 + lane] = all;
  P.cch[c * 64 + lane] = hot;
}

// Step 3: per group, lane j of each wave = colour j: the column decision,
// colour j's list offsets over the group's chunks, one pool reservation.  The
// chunks are shared out over 16 waves: one wave takes 1.9 ms for a group's two
// megabytes of counts (the same graph), 16 under 0.3.
constexpr uint32_t kGroupWaves = 16;

__global__ void __launch_bounds__(64 * kGroupWaves) out_group_kernel(OutParams P) {
  __shared__ unsigned long long s_hot, s_base;
  __shared__ uint32_t s_col, s_fail;
  __shared__ unsigned long long s_tot[64];
  __shared__ uint32_t s_all[kGroupWaves][64], s_chot[kGroupWaves][64];
  const uint32_t i = blockIdx.x, g = P.g0 + i, j = lane_id(), wid = threadIdx.x >> 6;
  const uint32_t nb = P.nb[g];
  const uint64_t chunks = P.cbase[i + 1] - P.cbase[i];
  const uint64_t c0 = P.cbase[i] + chunks * wid / kGroupWaves;
  const uint64_t c1 = P.cbase[i] + chunks * (wid + 1) / kGroupWaves;
  uint32_t all = 0, mine_hot = 0;
#pragma unroll 4
  for (uint64_t c = c0; c < c1; ++c) {
    all += P.cc[c * 64 + j];
    mine_hot += P.cch[c * 64 + j];
  }
  s_all[wid][j] = all;
  s_chot[wid][j] = mine_hot;
  __syncthreads();
  if (wid == 0) {
    unsigned long long hot = 0;
    for (uint32_t w = 0; w < kGroupWaves; ++w) hot += s_chot[w][j];
    for (int d = 32; d > 0; d >>= 1) hot += __shfl_xor(hot, d, 64);
    if (j == 0) {
      s_hot = hot;
      s_col = kNoGroup;
      // a column costs 8 bytes per hot vertex, lists 4 per member
      if (P.colptr && hot > 2ull * P.hot_n)
        s_col = P.group_base + static_cast<uint32_t>(atomicAdd(&P.ctl[kCtlGroupCounter2], 1ull));
    }
  }
  __syncthreads();
  const bool col = s_col != kNoGroup;
  // colour j's offsets in its list, chunk by chunk, eight read together
  uint32_t run = 0;
  for (uint32_t w = 0; w < wid; ++w) run += s_all[w][j] - (col ? s_chot[w][j] : 0u);
  for (uint64_t c = c0; c < c1; c += 8) {
    uint32_t k[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q)
      k[q] = c + q < c1 ? P.cc[(c + q) * 64 + j] - (col ? P.cch[(c + q) * 64 + j] : 0u) : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
      if (c + q < c1) P.cc[(c + q) * 64 + j] = run;
      run += k[q];
    }
  }
  if (wid == kGroupWaves - 1) s_tot[j] = run;
  __syncthreads();
  if (wid != 0) return;
  if (j == 0) {
    unsigned long long acc = 0;
    for (uint32_t q = 0; q < nb; ++q) acc += s_tot[q];
    const unsigned long long base = atomicAdd(&P.ctl[kCtlDataBump], acc);
    s_base = base;
    s_fail = 0;
    if (base + acc > P.cap_data) {
      s_fail = 1;
      atomicOr(&P.ctl[kCtlOverflow], 1ull);
    }
    if (col) atomicAdd(&P.ctl[kCtlElems], s_hot);
    P.gcol[i] = s_col;
    P.gfail[i] = s_fail;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");   // one wave from here on
  unsigned long long mine = s_base;
  for (uint32_t q = 0; q < j; ++q) mine += s_tot[q];
  P.dbase[i * 64ull + j] = mine;
  if (j < nb) {
    const uint32_t sid = P.sid[64ull * g + j];
    if (s_fail) {
      P.set_len[sid] = kLenFail;
    } else {
      P.set_off[sid] = mine;
      P.set_len[sid] = static_cast<uint32_t>(s_tot[j]);
    }
    if (col) P.gref[sid] = (s_col << 6) | j;
  }
  if (col) P.gsample[64ull * s_col + j] = j < nb ? P.sid[64ull * g + j] : kNoGroup;
  unsigned long long bytes = s_fail ? 0ull : 4ull * s_tot[j];
  report_stats(P.ctl, bytes, 0, 0, 0, 0);
}

// Step 3b: the columns of the sub-batch's column groups start at zero.
__global__ void out_column_clear_kernel(OutParams P) {
  const uint64_t total = static_cast<uint64_t>(P.groups) * P.hot_n;
  for (uint64_t t = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
       t += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint32_t i = static_cast<uint32_t>(t / P.hot_n);
    const uint32_t cg = P.gcol[i];
    if (cg != kNoGroup && !P.gfail[i]) P.colptr[cg][t - static_cast<uint64_t>(i) * P.hot_n] = 0ull;
  }
}

// Step 4: per chunk (one wave), hot members into the column (column
// groups), the rest to their colours' lists in vertex order.
__global__ void __launch_bounds__(64) out_scatter_kernel(OutParams P) {
  const uint64_t c = blockIdx.x;
  const uint32_t i = group_of_chunk(P.cbase, P.groups, c);
  if (P.gfail[i]) return;   // the call is redone with more pool space
  const uint32_t lane = lane_id();
  const uint32_t cg = P.gcol[i];
  const unsigned long long base = P.dbase[i * 64ull + lane];   // lane j: colour j
  const uint64_t e0 = (c - P.cbase[i]) * kChunk;
  const uint64_t e1 = min(e0 + kChunk, P.usz[i]);
  const uint32_t *list = P.slist + P.soff[i];
  const unsigned long long *masks = P.smask + P.soff[i];
  unsigned long long *colv = cg != kNoGroup ? P.colptr[cg] : nullptr;
  unsigned long long pos = base + P.cc[c * 64 + lane];   // lane j: next slot of colour j
  for (uint64_t t = e0; t < e1; t += 64) {
    const uint64_t e = t + lane;
    unsigned long long m = 0;
    uint32_t v = 0;
    if (e < e1) {
      m = masks[e];
      v = list[e];
      if (colv) {
        const uint32_t h = P.hot_index[v];
        if (h != kNotHot) {
          colv[h] = m;
          m = 0;
        }
      }
    }
    for (unsigned long long u = uniform_u64(wave_or_u64(m)); u; u &= u - 1) {
      const uint32_t col = static_cast<uint32_t>(__ffsll(u) - 1);
      const uint64_t b = __ballot((m >> col) & 1ull);
      const unsigned long long at = __shfl(pos, static_cast<int>(col), 64);
      if ((m >> col) & 1ull) P.data[at + __popcll(b & lanes_below())] = v;
      if (lane == col) pos += __popcll(b);
    }
  }
}

// Element 0 and sample id of every colour of the batch's groups: group g
// holds samples b0 + g C + c, c < C (C = colors); colours c >= C have none.
__global__ void grid_samples_kernel(uint64_t seed, uint64_t first, const uint32_t *ids,
                                    uint64_t b0, uint64_t count, uint32_t groups, uint32_t C,
                                    unsigned long long *z, uint32_t *sid, uint32_t *nb) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 64u * groups) return;
  const uint32_t g = i >> 6, c = i & 63u;
  const uint64_t t0 = b0 + static_cast<uint64_t>(g) * C;   // the group's first sample
  const uint64_t t = t0 + c;
  const bool has = c < C && t < count;
  const uint64_t s = has ? first + (ids ? ids[t] : t) : 0;
  z[i] = has ? sample_z(seed, s) : 0ull;
  sid[i] = has ? static_cast<uint32_t>(s) : kNoGroup;
  if (c == 0) {
    const uint64_t left = count > t0 ? count - t0 : 0;
    nb[g] = static_cast<uint32_t>(left < C ? left : C);
  }
}

// Bytes of one group's scratch: vis and pend, the union bitmap and summary.
uint64_t group_bytes(uint32_t n) {
  return 16ull * n + 4ull * ((n + 31) / 32) + 4ull * ((n + 1023) / 1024);
}

}  // namespace

// Groups per batch and frontier capacity for `count` samples.
static void grid_plan(const rip_graph *g, uint64_t count, uint32_t colors, uint32_t *groups,
                      uint64_t *fcap) {
  const uint64_t free_b = device_free_bytes();
  const GridScratch &s = g->grid;
  const uint64_t held = s.n == g->n ? s.groups * group_bytes(g->n) + 16ull * s.fcap : 0;
  // the scratch stays within an eighth of the memory it may use, 32 GiB at most
  const uint64_t budget = std::min<uint64_t>((free_b + held) / 8, 32ull << 30);
  const uint64_t per = group_bytes(g->n) + 16ull * std::min<uint64_t>(g->n, 1u << 22);
  uint64_t G = std::max<uint64_t>(1, budget / per);
  G = std::min<uint64_t>({G, 256, (count + colors - 1) / colors});
  *groups = static_cast<uint32_t>(G);
  // room for every group's frontier up to 2^22 vertices, and for one whole
  // union (the output staging reuses the frontier buffers)
  *fcap = std::max<uint64_t>(g->n, G * std::min<uint64_t>(g->n, 1u << 22));
}

static void grid_ensure(rip_graph *g, uint32_t groups, uint64_t fcap, hipStream_t st) {
  GridScratch &s = g->grid;
  const uint32_t n = g->n;
  if (s.searching || s.n != n || s.groups < groups) {
    dev_free(s.d_vis);
    dev_free(s.d_bm0);
    dev_free(s.d_bm1);
    dev_free(s.d_z);
    dev_free(s.d_sid);
    dev_free(s.d_nb);
    s.groups = 0;
    const uint64_t nw0 = (n + 31) / 32, nw1 = (n + 1023) / 1024;
    s.d_vis = dev_alloc<unsigned long long>(2ull * groups * n);
    s.d_bm0 = dev_alloc<uint32_t>(groups * nw0);
    s.d_bm1 = dev_alloc<uint32_t>(groups * nw1);
    s.d_z = dev_alloc<unsigned long long>(64ull * groups);
    s.d_sid = dev_alloc<uint32_t>(64ull * groups);
    s.d_nb = dev_alloc<uint32_t>(groups);
    // zero once; every batch leaves them zero again
    RIP_HIP(hipMemsetAsync(s.d_vis, 0, 16ull * groups * n, st));
    RIP_HIP(hipMemsetAsync(s.d_bm0, 0, 4ull * groups * nw0, st));
    RIP_HIP(hipMemsetAsync(s.d_bm1, 0, 4ull * groups * nw1, st));
    s.groups = groups;
    s.n = n;
    s.searching = false;
  }
  if (s.fcap < fcap) {
    dev_free(s.d_fa);
    dev_free(s.d_fb);
    s.fcap = 0;
    s.d_fa = dev_alloc<unsigned long long>(fcap);
    s.d_fb = dev_alloc<unsigned long long>(fcap);
    s.fcap = fcap;
  }
  // (each by itself: an allocation that fails leaves the rest for the next call)
  if (!s.d_ring) s.d_ring = dev_alloc<unsigned long long>(kRWords * kRing);
  if (!s.d_heavy) s.d_heavy = dev_alloc<unsigned long long>(2ull * kHeavyCap);
  if (!s.d_segs) s.d_segs = dev_alloc<unsigned long long>(kSegCap);
  if (!s.d_gctl) s.d_gctl = dev_alloc<unsigned long long>(kGWords);
  if (!s.d_union) s.d_union = dev_alloc<unsigned long long>(256);
  if (!s.h_ctl)
    RIP_HIP(hipHostMalloc(reinterpret_cast<void **>(&s.h_ctl), sizeof(unsigned long long) * 256,
                          hipHostMallocDefault));
}

// Room for `words` 64-bit words of output tables.
static void grid_out_arena(GridScratch &s, uint64_t words) {
  if (s.out_words >= words) return;
  dev_free(s.d_out);
  s.out_words = 0;
  s.d_out = dev_alloc<unsigned long long>(words);
  s.out_words = words;
}

// Reads `count` words of device memory into the scratch's pinned buffer.
static const unsigned long long *grid_read(GridScratch &s, const unsigned long long *src,
                                           uint32_t count, hipStream_t st) {
  RIP_HIP(hipMemcpyAsync(s.h_ctl, src, sizeof(unsigned long long) * count,
                         hipMemcpyDeviceToHost, st));
  RIP_HIP(hipStreamSynchronize(st));
  return s.h_ctl;
}

void grid_scratch_free(GridScratch &s) {
  dev_free(s.d_vis);
  dev_free(s.d_bm0);
  dev_free(s.d_bm1);
  dev_free(s.d_z);
  dev_free(s.d_sid);
  dev_free(s.d_nb);
  dev_free(s.d_fa);
  dev_free(s.d_fb);
  dev_free(s.d_gctl);
  dev_free(s.d_union);
  dev_free(s.d_ring);
  dev_free(s.d_heavy);
  dev_free(s.d_segs);
  dev_free(s.d_out);
  s.out_words = 0;
  if (s.h_ctl) (void)hipHostFree(s.h_ctl);
  s.h_ctl = nullptr;
  s.groups = 0;
  s.fcap = 0;
  s.n = 0;
  s.searching = false;
}

// Samples first + ids[i] (first + i without ids), i in [0, count), with the
// grid sampler; with columns, groups with many hot members go to the pool's
// column store.  Returns the kernel launches made.
uint32_t ic_grid_launch(rip_pool *p, uint64_t first, uint64_t count, const uint32_t *ids,
                        bool columns, uint32_t frontier_cap, uint32_t colors) {
  if (count == 0) return 0;
  RIP_REQUIRE(colors >= 1 && colors <= 64, RIP_EINVAL, "tune: colors must be in [1, 64]");
  const uint32_t C = colors;
  rip_graph *gr = p->g;
  hipStream_t st = p->stream;
  uint32_t G = 0;
  uint64_t fcap = 0;
  grid_plan(gr, count, C, &G, &fcap);
  grid_ensure(gr, G, fcap, st);
  GridScratch &s = gr->grid;
  const uint64_t total_groups = (count + C - 1) / C;
  if (columns) pool_reserve_groups(p, p->groups + static_cast<uint32_t>(total_groups));
  const uint32_t n = gr->n;
  GridParams P;
  P.vrec = gr->d_vrec;
  P.ids = gr->d_ids;
  P.val = gr->d_val;
  P.n = n;
  P.step = gr->step;
  P.vp = s.d_vis;
  P.bm0 = s.d_bm0;
  P.bm1 = s.d_bm1;
  P.nw0 = (n + 31) / 32;
  P.nw1 = (n + 1023) / 1024;
  P.z = s.d_z;
  // entries a level may list: the buffer, or fewer when asked (the buffers
  // keep room for one whole union, the output staging)
  const uint64_t lcap = frontier_cap ? std::min<uint64_t>(frontier_cap, s.fcap) : s.fcap;
  P.cap = lcap;
  const uint64_t tail_cap = std::min<uint64_t>(kTailItems, lcap);
  P.gctl = s.d_gctl;
  P.ctl = p->d_ctl;
  P.ring = s.d_ring;
  P.heavy = s.d_heavy;
  P.segs = s.d_segs;
  P.heavy_cap = static_cast<uint32_t>(std::min<uint64_t>(kHeavyCap, lcap));
  P.seg_cap = static_cast<uint32_t>(std::min<uint64_t>(kSegCap, lcap));
  P.buf[0] = s.d_fa;
  P.buf[1] = s.d_fb;
  const int per_cu = blocks_per_cu(reinterpret_cast<const void *>(&grid_level_kernel<kExpBT>),
                                   kExpBT);
  const uint32_t exp_grid = static_cast<uint32_t>(per_cu * cu_count());
  uint32_t launches = 0;
  s.searching = true;   // an error from here on leaves masks and bitmaps set
  for (uint64_t b0 = 0; b0 < count; b0 += static_cast<uint64_t>(C) * G) {
    const uint32_t Gb = static_cast<uint32_t>(std::min<uint64_t>(G, (count - b0 + C - 1) / C));
    hipLaunchKernelGGL(grid_samples_kernel, dim3((64 * Gb + 255) / 256), dim3(256), 0, st,
                       p->seed, first, ids, b0, count, Gb, C, s.d_z, s.d_sid, s.d_nb);
    hipLaunchKernelGGL(grid_ring_kernel, dim3(1), dim3(256), 0, st, s.d_ring, s.d_gctl, 0u,
                       0u, 1u);
    // level 0: the roots, in buf[0]
    P.next = s.d_fa;
    P.next_cnt = &s.d_ring[0];
    hipLaunchKernelGGL(grid_seed_kernel, dim3(Gb), dim3(64), 0, st, P,
                       static_cast<const uint32_t *>(s.d_nb));
    launches += 3;
    uint32_t L = 0;            // the level whose frontier is ring[L % kRing]
    bool dirty = false;        // some vertices with pend bits are in no list
    const uint32_t levels0 = p->grid_levels;
    auto frontier_len = [&](uint32_t level) {
      RIP_HIP(hipMemcpyAsync(s.h_ctl + kGWords, s.d_ring + level % kRing,
                             sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
      RIP_HIP(hipStreamSynchronize(st));
      return static_cast<uint64_t>(s.h_ctl[kGWords]);
    };
    uint64_t pending = frontier_len(L);
    for (;;) {
      if (pending == 0) {
        if (!dirty) break;
        // the vertices the overflowing lists could not hold, as level L
        P.next = P.buf[L & 1u];
        P.next_cnt = &s.d_ring[L % kRing];
        hipLaunchKernelGGL(grid_rebuild_kernel, dim3(2048), dim3(256), 0, st, P, Gb);
        launches += 1;
        pending = frontier_len(L);
        dirty = pending > lcap;
        if (pending == 0) break;
        continue;
      }
      RIP_HIP(hipEventRecord(p->ev3, st));
      if (pending <= tail_cap) {
        // a thin frontier: one workgroup runs the levels until it widens
        hipLaunchKernelGGL((grid_tail_kernel<kExpBT>), dim3(1), dim3(kExpBT), 0, st, P, L,
                           tail_cap);
        launches += 1;
      } else {
        // kLevelsPerSync levels, then one look at the frontier length
        hipLaunchKernelGGL(grid_ring_kernel, dim3(1), dim3(kLevelsPerSync), 0, st, s.d_ring,
                           s.d_gctl, L + 1, kLevelsPerSync, 0u);
        for (uint32_t i = 0; i < kLevelsPerSync; ++i) {
          hipLaunchKernelGGL((grid_level_kernel<kExpBT>), dim3(exp_grid), dim3(kExpBT), 0, st, P,
                             L + i);
          hipLaunchKernelGGL((grid_heavy_kernel<kExpBT>), dim3(exp_grid), dim3(kExpBT), 0, st, P,
                             L + i);
        }
        launches += 1 + 2 * kLevelsPerSync;
      }
      RIP_HIP(hipGetLastError());
      RIP_HIP(hipEventRecord(p->ev4, st));
      const unsigned long long *h = grid_read(s, s.d_gctl, kGWords, st);
      if (pending <= tail_cap) {
        L = static_cast<uint32_t>(h[kGTail]);
      } else {
        L += kLevelsPerSync;
        if (h[kGOver] != 0) dirty = true;
      }
      p->grid_levels = levels0 + static_cast<uint32_t>(h[kGLevels]);
      float ms = 0.0f;
      RIP_HIP(hipEventElapsedTime(&ms, p->ev3, p->ev4));
      p->grid_ms += ms;
      pending = frontier_len(L);
      if (pending > lcap) dirty = true;
    }
    // output: groups whose unions fit the staging together share a launch
    hipLaunchKernelGGL(grid_union_kernel, dim3(Gb), dim3(1024), 0, st, s.d_bm0, P.nw0, s.d_union);
    std::vector<unsigned long long> usz(Gb);
    const unsigned long long *h = grid_read(s, s.d_union, Gb, st);
    std::copy(h, h + Gb, usz.begin());
    OutParams O;
    O.n = n;
    O.nw0 = P.nw0;
    O.nw1 = P.nw1;
    O.vp = s.d_vis;
    O.bm0 = s.d_bm0;
    O.bm1 = s.d_bm1;
    O.slist = reinterpret_cast<uint32_t *>(s.d_fa);
    O.smask = s.d_fb;
    O.sid = s.d_sid;
    O.nb = s.d_nb;
    O.set_off = p->d_off;
    O.set_len = p->d_len;
    O.data = p->d_data;
    O.cap_data = p->cap_data;
    O.ctl = p->d_ctl;
    O.colptr = columns ? p->d_colptr : nullptr;
    O.gsample = columns ? p->d_gsample : nullptr;
    O.gref = columns ? p->d_gref : nullptr;
    O.hot_index = columns ? gr->d_hot_index : nullptr;
    O.hot_n = columns ? gr->hot_n : 0;
    O.group_base = p->groups;
    for (uint32_t a = 0; a < Gb;) {
      // groups a, a + 1, ... while their unions fit the staging together (one
      // always does); their staging offsets and chunks
      std::vector<unsigned long long> off, cb(1, 0);
      unsigned long long acc = 0;
      uint32_t e = a;
      while (e < Gb && (e == a || acc + usz[e] <= s.fcap)) {
        off.push_back(acc);
        acc += usz[e];
        cb.push_back(cb.back() + (usz[e] + kChunk - 1) / kChunk);
        ++e;
      }
      const uint32_t m = e - a;
      const uint64_t chunks = cb.back();
      // device tables of the sub-batch, carved from the output arena
      const uint64_t words = 4ull * m + kRanges * static_cast<uint64_t>(m) + 64ull * m +
                             64ull * chunks + 2;   // u64 words
      grid_out_arena(s, words);
      unsigned long long *w = s.d_out;
      unsigned long long *d_soff = w;          w += m;
      unsigned long long *d_cbase = w;         w += m + 1;
      unsigned long long *d_usz = w;           w += m;
      unsigned long long *d_rc = w;            w += static_cast<uint64_t>(kRanges) * m;
      unsigned long long *d_dbase = w;         w += 64ull * m;
      uint32_t *d_cc = reinterpret_cast<uint32_t *>(w);
      uint32_t *d_cch = d_cc + 64ull * chunks; w += 64ull * chunks;
      uint32_t *d_gcol = reinterpret_cast<uint32_t *>(w);
      uint32_t *d_gfail = d_gcol + m;          w += m;
      std::vector<unsigned long long> up(3ull * m + 1);
      std::copy(off.begin(), off.end(), up.begin());
      std::copy(cb.begin(), cb.end(), up.begin() + m);
      std::copy(usz.begin() + a, usz.begin() + e, up.begin() + 2 * m + 1);
      RIP_HIP(hipMemcpyAsync(s.d_out, up.data(), sizeof(unsigned long long) * up.size(),
                             hipMemcpyHostToDevice, st));
      O.g0 = a;
      O.groups = m;
      O.soff = d_soff;
      O.cbase = d_cbase;
      O.usz = d_usz;
      O.rc = d_rc;
      O.dbase = d_dbase;
      O.cc = d_cc;
      O.cch = d_cch;
      O.gcol = d_gcol;
      O.gfail = d_gfail;
      hipLaunchKernelGGL(out_range_count_kernel, dim3(m * kRanges), dim3(64), 0, st, O);
      hipLaunchKernelGGL(out_range_write_kernel, dim3(m * kRanges), dim3(64), 0, st, O);
      hipLaunchKernelGGL(out_chunk_count_kernel, dim3(static_cast<uint32_t>(chunks)), dim3(64), 0,
                         st, O);
      hipLaunchKernelGGL(out_group_kernel, dim3(m), dim3(64 * kGroupWaves), 0, st, O);
      if (columns)
        hipLaunchKernelGGL(out_column_clear_kernel, dim3(4096), dim3(256), 0, st, O);
      hipLaunchKernelGGL(out_scatter_kernel, dim3(static_cast<uint32_t>(chunks)), dim3(64), 0, st,
                         O);
      RIP_HIP(hipGetLastError());
      RIP_HIP(hipStreamSynchronize(st));   // `up` and the staging are reused
      launches += 6;
      a = e;
    }
    launches += 1;
  }
  s.searching = false;
  return launches;
}

}  // namespace rip
