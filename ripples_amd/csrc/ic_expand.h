// Row expansion shared by the IC samplers that take 64 queued vertices at a
// time (wave stage, team sampler).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "device_util.h"
#include "ic_common.h"
#include "ic_gap.h"

namespace rip {

// Candidates a lane draws before their edges are read together (a block has
// two or three; in the team kernel four measured 3% slower and two 4%).
constexpr uint32_t kUnitBatch = 3;

// Draws of up to K candidates of a gap block, for lanes with `more` set: the
// next element x, pos of the block's len edges passed.  e[i] gets the i-th
// candidate's position in the block and h[i] what its threshold must pass (0
// for `uniform` rows, which keep every candidate); returns how many there
// are, with x, pos and more moved on.  K elements and their gaps are computed
// whether or not the block ends before them, apart from each other: one draw
// is a chain of some forty dependent instructions, which is what a wave waits
// for when it draws them one by one.
template <int K>
__device__ inline uint32_t ic_draw_block(uint64_t &x, uint32_t &pos, bool &more, uint32_t len,
                                         uint32_t T, uint64_t q, double inv, bool uniform,
                                         const Affine &A, const Affine &A2, const IcGapTab *tab,
                                         uint32_t (&e)[K], uint32_t (&h)[K]) {
  uint64_t xs[K];
  double fg[K];
  uint32_t gap[K];
  xs[0] = x;
#pragma unroll
  for (int i = 1; i < K; ++i) xs[i] = aff_apply(A2, xs[i - 1]);
#pragma unroll
  for (int i = 0; i < K; ++i) fg[i] = ic_gap_real(xs[i], inv, tab);
  bool sure = true;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    sure = sure && ic_gap_sure(fg[i], inv);
    gap[i] = static_cast<uint32_t>(__builtin_floor(fg[i]));
  }
  if (more && !sure) {
#pragma unroll 1
    for (int i = 0; i < K; ++i)
      if (!ic_gap_sure(fg[i], inv)) gap[i] = ic_gap_near(xs[i], q, fg[i]);
  }
  uint32_t n = 0;
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const bool is = more && gap[i] < len - pos;
    e[i] = is ? pos + gap[i] : 0u;
    h[i] = is && !uniform ? static_cast<uint32_t>(((aff_apply(A, xs[i]) >> 32) * T) >> 32) : 0u;
    if (is) pos = e[i] + 1;
    n += is ? 1u : 0u;
    more = is && pos < len;
  }
  x = aff_apply(A2, xs[K - 1]);
  return n;
}

// Expands up to 64 queued vertices at once, lane l holding the record rv of
// one (when `have`), the element 0 z of its sample and the caller's tag of it.
// The rows' gap blocks are the units of work: 64 units at a time, one per lane,
// found by a wave scan of the block counts when some row has several (a hub's
// blocks spread over the lanes instead of queueing in one).  A lane draws up to
// kUnitBatch candidates of its block (arithmetic only), then the wave reads
// their thresholds and in-neighbours together, so a unit waits for one trip to
// memory, not one per candidate; take(live, src, tag) gets every batch (without
// kIds the edges in place of their in-neighbours, which are not read).  Every
// lane of the wave must call it.  Returns false as soon as take() does.
template <bool kIds, typename Take>
__device__ inline bool expand_rows_units(const uint32_t *ids, const uint32_t *val, bool have,
                                         const VertexRec &rv, uint64_t z, uint32_t tag,
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
    uint32_t utag = tag;
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
      utag = __shfl(tag, src, 64);
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
      const uint32_t nc = ic_draw_block<kUnitBatch>(x, pos, more, len, T, q, inv, uniform, P, P2, tab,
                                                    ce, th);
      st_draws += nc - (nc != 0 && pos == len ? 1u : 0u);
      uint32_t t[kUnitBatch], src[kUnitBatch];
#pragma unroll
      for (uint32_t i = 0; i < kUnitBatch; ++i) {
        t[i] = 0xFFFFFFFFu;                        // rows sharing one threshold keep every candidate
        src[i] = 0;
        if (i < nc) {
          src[i] = kIds ? ids[e0 + ce[i]] : e0 + ce[i];
          if (!uniform) t[i] = val[e0 + ce[i]];
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
      if (!take(live, src, utag)) return false;
    }
  }
  return true;
}

}  // namespace rip
