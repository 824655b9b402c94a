// Row expansion shared by the IC samplers that take 64 vertices of one sample
// at a time (wave stage, team sampler).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "device_util.h"
#include "ic_common.h"
#include "ic_gap.h"

namespace rip {

// Candidates a lane collects before their edges are read together (a block
// draws two or three; four spill the team kernel's registers and measured 3%
// slower there, two 4%).
constexpr uint32_t kUnitBatch = 3;

// Expands up to 64 queued vertices of the sample whose element 0 is z at
// once, lane l holding the record rv of one (when `have`).  The rows' gap
// blocks are the units of work: 64 units at a time, one per lane, found by a
// wave scan of the block counts when some row has several (a hub's blocks
// spread over the lanes instead of queueing in one).  A lane draws up to
// kUnitBatch candidates of its block (arithmetic only), then the wave reads
// their thresholds and in-neighbours together, so a unit waits for one trip
// to memory, not one per candidate; take(live, src) gets every batch.  Against one draw per lane and
// step, a whole row per lane: the stage's kernels of an IMM run on R-MAT scale
// 22 weighted cascade took 13.5 ms instead of 15.6 (rows of one block there;
// hub rows of U[0,0.1] graphs have hundreds).  Every lane of the wave must
// call it.  Returns false as soon as take() does.
template <typename Take>
__device__ inline bool expand_rows_units(const uint32_t *ids, const uint32_t *val, bool have,
                                         const VertexRec &rv, uint64_t z,
                                         const Affine *p2, const IcGapTab *tab,
                                         unsigned long long &st_cand,
                                         unsigned long long &st_draws,
                                         unsigned long long &st_bytes,
                                         unsigned long long &st_live, Take &&take) {
  const uint32_t lane = lane_id();
  const bool row = have && rv.thr != 0;            // else no edge of the row can be live
  const uint32_t rdeg = rv.end - rv.begin;
  const uint32_t nblk = row ? ((rdeg - 1) >> ((rv.flags >> kBetaShift) & 31u)) + 1 : 0u;
  const uint64_t x0 = rv.ja * z + rv.jb;           // the row's first element
  const bool single = __ballot(nblk > 1) == 0;     // a lane's unit is its own row
  const uint32_t incl = single ? 0u : wave_inclusive_scan(nblk);
  const uint32_t total = single ? 64u : uniform_u32(__shfl(incl, 63, 64));
  const Affine P = uniform_affine(p2[0]), P2 = uniform_affine(p2[1]);
  for (uint32_t u0 = 0; u0 < total; u0 += 64) {
    uint32_t e0 = rv.begin, len = 0, T = rv.thr;
    uint64_t q = rv.q, x = x0;
    double inv = rv.inv;
    bool uniform = (rv.flags & kRowUniform) != 0;
    bool skip = true;
    if (single) {
      if (row) {
        len = rdeg;                                // one block, at most its full length
        const uint32_t beta = (rv.flags >> kBetaShift) & 31u;
        skip = (x >> 32) + 1 <= (len == (1u << beta) ? rv.ufull : rv.ulast);
      }
    } else {
      // unit u is block k of the row of lane j, the first whose inclusive
      // prefix passes u
      const uint32_t u = u0 + lane;
      uint32_t j = 0;
#pragma unroll
      for (uint32_t s = 32; s > 0; s >>= 1) {
        const uint32_t v = __shfl(incl, static_cast<int>(j + s - 1), 64);
        if (v <= u) j += s;
      }
      const int src = static_cast<int>(min(j, 63u));
      const uint32_t k = u - (__shfl(incl, src, 64) - __shfl(nblk, src, 64));
      const uint32_t begin = __shfl(rv.begin, src, 64), deg = __shfl(rdeg, src, 64);
      const uint32_t flags = __shfl(rv.flags, src, 64);
      const uint32_t ufull = __shfl(rv.ufull, src, 64), ulast = __shfl(rv.ulast, src, 64);
      T = __shfl(rv.thr, src, 64);
      q = __shfl(rv.q, src, 64);
      inv = __shfl(rv.inv, src, 64);
      x = __shfl(x0, src, 64);
      uniform = (flags & kRowUniform) != 0;
      if (u < total) {
        const uint32_t beta = (flags >> kBetaShift) & 31u;
        e0 = begin + (k << beta);
        len = min(deg - (k << beta), 1u << beta);
        // block k's first element: 2 B k elements after the row's first
        for (uint32_t kk = k, bit = beta + 1; kk; kk >>= 1, ++bit)
          if (kk & 1) x = aff_apply(p2[bit], x);
        skip = (x >> 32) + 1 <= (len == (1u << beta) ? ufull : ulast);
      }
    }
    // a block without candidates costs one compare
    if (len) ++st_draws;
    bool more = len != 0 && !skip;
    uint32_t pos = 0;
    while (__ballot(more)) {
      uint32_t ce[kUnitBatch], th[kUnitBatch];
      uint32_t nc = 0;
#pragma unroll
      for (uint32_t i = 0; i < kUnitBatch; ++i) {
        ce[i] = 0;
        th[i] = 0;
        if (more) {
          const uint32_t gap = ic_gap_draw(x, q, inv, tab);
          if (gap >= len - pos) {
            more = false;
          } else {
            pos += gap;
            ce[i] = e0 + pos;
            // kept iff the edge's threshold t passes this (ic_accept:
            // hi32(a) T < t 2^32 for the acceptance element a)
            if (!uniform)
              th[i] = static_cast<uint32_t>(((aff_apply(P, x) >> 32) * T) >> 32);
            nc = i + 1;
            if (++pos < len) {
              x = aff_apply(P2, x);                // next gap element
              ++st_draws;
            } else {
              more = false;
            }
          }
        }
      }
      uint32_t t[kUnitBatch], src[kUnitBatch];
#pragma unroll
      for (uint32_t i = 0; i < kUnitBatch; ++i) {
        t[i] = 0xFFFFFFFFu;                        // rows sharing one threshold keep every candidate
        src[i] = 0;
        if (i < nc) {
          src[i] = ids[ce[i]];
          if (!uniform) t[i] = val[ce[i]];
        }
      }
      st_cand += nc;
      if (!uniform) {
        st_draws += nc;
        st_bytes += 4 * nc;
      }
      bool live[kUnitBatch];
#pragma unroll
      for (uint32_t i = 0; i < kUnitBatch; ++i) {
        live[i] = i < nc && t[i] > th[i];
        if (live[i]) {
          ++st_live;
          st_bytes += 4;
        }
      }
      if (!take(live, src)) return false;
    }
  }
  return true;
}

}  // namespace rip
