// pair_sched.h -- the balanced pair schedule of the tile kernels (SPH pair
// passes, Newton-h): device code included by k_sph.hip and k_hsolve.hip.
#pragma once

#include "fsph_internal.h"

namespace fsph {
namespace sched {

// ---------------------------------------------------------------------------
// Balanced pair schedule of one chunk.
//
// Row k of the chunk's mask (CH candidates; candidate j is bit j%32 of word
// j/32) marks the neighbours of group particle k among the chunk's
// candidates.  The chunk's P pairs, in (k, j) order, are cut into NT runs
// of q = ceil(P/NT) pairs and thread l walks run l, so every thread walks
// the same number of pairs however unevenly they fall on the particles.
// A run covers whole rows plus at most two partial rows: the row it starts
// in (which may have begun in an earlier run) and the row it ends in (which
// may go on in a later run).  Thread l writes the partial result of row k to
// slot l + k: along the (row, run) pieces in order one of the two, or both,
// grow by one, so no two pieces share a slot and row k's pieces are the
// consecutive slots k + la .. k + lb for the first and last runs la <= lb
// that hold its pairs.  After the walk thread k adds them up in run order.
// The result depends only on the tile, not on timing.
// ---------------------------------------------------------------------------
template <int NT> struct Sched {
  int off[NT + 1];  // pairs before row k; off[k] = P for k >= gc
  int wsum[NT / 64];
};

template <class T, int NV, int NT> struct Parts {
  T v[NV][2 * NT];
};

// Inclusive scan over the wavefront with DPP moves (no LDS round trips).
__device__ inline int wave_scan_incl(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // bcast 15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // bcast 31
  return v;
}

// Row offsets of the chunk (requires the staged masks; gc <= NT); returns P.
// Thread t passes whether row t takes part (a row that does not has no
// pairs in the schedule).
template <int NT>
__device__ inline int schedule(Sched<NT> &S, const uint32_t *smask, int nw,
                               int gc, bool row_on = true) {
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  int n = 0;
  if (t < gc && row_on)
    for (int w = 0; w < nw; ++w) n += __popc(smask[w * gc + t]);
  const int inc = wave_scan_incl(n);
  int total = 0, before = 0;
  if (NT == 64) {
    total = __builtin_amdgcn_readlane(inc, 63);
  } else {
    if (lane == 63) S.wsum[wv] = inc;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NT / 64; ++v) {
      if (v < wv) before += S.wsum[v];
      total += S.wsum[v];
    }
  }
  S.off[t] = inc - n + before;
  if (t == 0) S.off[NT] = total;
  __syncthreads();
  return total;
}

// x without its r lowest set bits (r < popc(x)).
__device__ inline uint32_t drop_low(uint32_t x, int r) {
  uint32_t y = x;
  int pos = 0;
#pragma unroll
  for (int w = 16; w > 0; w >>= 1) {
    const int n = __popc(y & ((1u << w) - 1u));
    if (n <= r) {
      r -= n;
      y >>= w;
      pos += w;
    }
  }
  return x & (~0u << pos);
}

// Bits of one row over the chunk, 64 candidates per word, the current word
// first; `base` is the candidate of its bit 0.
template <int CH> struct RowBits {
  static constexpr int W = CH / 64;
  uint64_t b[W];
  int base;
  __device__ inline void load(const uint32_t *smask, int gc, int k) {
#pragma unroll
    for (int i = 0; i < W; ++i)
      b[i] = (uint64_t)smask[(2 * i + 1) * gc + k] << 32 |
             smask[2 * i * gc + k];
    base = 0;
  }
  __device__ inline void next_word() {
#pragma unroll
    for (int i = 0; i + 1 < W; ++i) b[i] = b[i + 1];
    b[W - 1] = 0;
    base += 64;
  }
  // drops the r lowest bits (r < number of bits)
  __device__ inline void drop(int r) {
    for (int n; W > 1 && (n = __popcll(b[0])) <= r;) {
      r -= n;
      next_word();
    }
    uint32_t lo = (uint32_t)b[0], hi = (uint32_t)(b[0] >> 32);
    const int n = __popc(lo);
    if (r < n) {
      lo = drop_low(lo, r);
    } else {
      lo = 0;
      hi = drop_low(hi, r - n);
    }
    b[0] = (uint64_t)hi << 32 | lo;
  }
  // the lowest candidate, removed (some bit must be left)
  __device__ inline int pop() {
    if (W > 1)
      while (b[0] == 0) next_word();
    const int j = base + __builtin_ctzll(b[0]);
    b[0] &= b[0] - 1;
    return j;
  }
};

// Walks this thread's run: load(k) when the run enters row k, pair(j, valid)
// for its pairs, flush(k) when the run leaves row k.
//
// kPairs pairs of a row are taken per iteration, without a branch between
// them (the ones past the row's or the run's end come with valid false and
// must add nothing): some thread of the wavefront changes rows in nearly
// every iteration, so that code is paid once for kPairs pairs, and their
// LDS reads and chains overlap.  The row's bits stay in registers.  The
// acceleration pass (FP32, chunk 128) went from 341 to 273 us on Sedov 64^3
// and 726 to 596 us on the 1M star; three pairs measured 318 and 703 us, four
// 332 and 737 (more of them past a row's end, more registers).
constexpr int kPairs = 2;
template <int CH, int NT, class Load, class Pair, class Flush>
__device__ inline void walk_run(const Sched<NT> &S, const uint32_t *smask,
                                int gc, int total, Load &&load, Pair &&pair,
                                Flush &&flush) {
  const int q = (total + NT - 1) / NT;
  const int p0 = (int)threadIdx.x * q, p1 = min(p0 + q, total);
  if (p0 >= p1) return;
  int k = 0;
#pragma unroll
  for (int s = NT / 2; s > 0; s >>= 1)
    if (S.off[k + s] <= p0) k += s;
  int rend = S.off[k + 1];
  RowBits<CH> row;
  row.load(smask, gc, k);
  row.drop(p0 - S.off[k]);
  load(k);
  for (int p = p0; p < p1;) {
    if (p == rend) {
      flush(k);
      ++k;
      while (S.off[k + 1] <= p) ++k;
      rend = S.off[k + 1];
      row.load(smask, gc, k);
      load(k);
    }
    const int lim = min(rend, p1) - p;
    int j[kPairs];
    j[0] = row.pop();
#pragma unroll
    for (int u = 1; u < kPairs; ++u) {
      j[u] = j[0];
      if (u < lim) j[u] = row.pop();
    }
#pragma unroll
    for (int u = 0; u < kPairs; ++u) pair(j[u], u == 0 || u < lim);
    p += min(lim, kPairs);
  }
  flush(k);
}

template <class T, int NV, int NT>
__device__ inline void put(Parts<T, NV, NT> &R, int i, int k, T v) {
  R.v[i][(int)threadIdx.x + k] = v;
}

// Row k's results of this chunk into v (after the walk; the row must hold
// pairs): its pieces in run order, added up or, for the components whose bit
// is set in MAXED, the largest.  The runs that hold the row's first and last
// pair are quotients by the run length: exact through FP32, as the numbers
// stay below 2^15 and (pair + 0.5) / q is at least 0.5 / q from an integer.
template <unsigned MAXED, class T, int NV, int NT>
__device__ inline void row_results(const Sched<NT> &S,
                                   const Parts<T, NV, NT> &R, int k, int total,
                                   T (&v)[NV]) {
  const float rq = 1.0f / (float)((total + NT - 1) / NT);
  const int la = (int)(((float)S.off[k] + 0.5f) * rq);
  const int lb = (int)(((float)S.off[k + 1] - 0.5f) * rq);
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = R.v[i][k + la];
  for (int l = la + 1; l <= lb; ++l)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const T u = R.v[i][k + l];
      v[i] = MAXED >> i & 1u ? (v[i] < u ? u : v[i]) : v[i] + u;
    }
}

}  // namespace sched
}  // namespace fsph
