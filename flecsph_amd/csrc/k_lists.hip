// k_lists.hip -- the neighbour lists as arrays of sorted particle indices
// (fsph_neighbor_lists): the tiles' candidates and mask bits are expanded on
// the device, every row in ascending index, and copied out once.
//
// Bound by the copy to the host (8 bytes per neighbour).  Expanding on the
// host instead (one copy per tile, then a sort of every row) took 39 ms for
// the 38,880-particle Sod tube (60 neighbours); now the tree, the lists and
// their copy take 1.6 ms, 0.09 of it this kernel.
#include "fsph_internal.h"

namespace fsph {

namespace {

constexpr int kLT = 256;         // threads: four wavefronts, a row each
constexpr int kSortMax = 4096;   // candidates sorted in LDS

struct ListArgs {
  const int32_t *tstart, *tcount, *tslot, *tccount, *cand;
  const int64_t *tmoff;
  const uint32_t *mask;
  int64_t ccap, nt;
  const int64_t *off;  // row offsets, n + 1
  int64_t r0, r1;      // rows written by this launch
  int64_t *out;        // entry off[r0] is out[0]
  int *bad;            // set when a row does not hold its count
};

// Appends to row `row` (already holding cnt entries) the particles of the
// lanes that hold one, in lane order; never past the row's end.
__device__ inline int append(const ListArgs &a, int64_t row, int cnt,
                             bool in, int32_t id) {
  const uint64_t m = __ballot(in);
  const int lane = threadIdx.x & 63;
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
  const int64_t at = a.off[row] + cnt + __popcll(m & below);
  if (in && at < a.off[row + 1]) a.out[at - a.off[a.r0]] = id;
  return cnt + __popcll(m);
}

// One workgroup per tile.  The tile's candidates are brought into ascending
// order once (64 rows share them): up to kSortMax of them with a bitonic
// sort of (index, position) in LDS.  Then a wavefront takes a row, 64
// candidates in that order at a time: each lane looks its candidate's bit up
// in the row's mask words and a ballot packs the neighbours.  A tile with
// more candidates (a few very wide spheres) goes through windows of kSortMax
// particle indices: a table gives each index its position in the tile.
__global__ __launch_bounds__(kLT) void k_lists(ListArgs a) {
  __shared__ uint64_t srt[kSortMax];
  __shared__ uint32_t wbuf[kLT / 64][kSortMax / 32];
  __shared__ int lo_s, hi_s;
  const int64_t t = xcd_item(blockIdx.x, gridDim.x);
  const int64_t ts = a.tstart[t];
  const int tc = a.tcount[t], cc = a.tccount[t];
  const int k0 = (int)(a.r0 > ts ? (a.r0 - ts < tc ? a.r0 - ts : tc) : 0);
  const int k1 = (int)(a.r1 > ts ? (a.r1 - ts < tc ? a.r1 - ts : tc) : 0);
  if (k0 >= k1) return;
  const int32_t *cand = a.cand + (int64_t)a.tslot[t] * a.ccap;
  const uint32_t *mask = a.mask + a.tmoff[t];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (cc <= kSortMax) {
    int m = 64;
    while (m < cc) m <<= 1;
    for (int i = threadIdx.x; i < m; i += kLT)
      srt[i] = i < cc ? ((uint64_t)(uint32_t)cand[i] << 32) | (uint32_t)i
                      : ~0ull;
    __syncthreads();
    for (int k = 2; k <= m; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int q = threadIdx.x; q < m / 2; q += kLT) {
          const int i = 2 * q - (q & (j - 1)), l = i + j;
          const uint64_t x = srt[i], y = srt[l];
          if ((x > y) == ((i & k) == 0)) {
            srt[i] = y;
            srt[l] = x;
          }
        }
        __syncthreads();
      }
    const int nw = (cc + 31) >> 5;
    // (uniform trip count: the barriers order each wavefront's row buffer)
    for (int kk = k0; kk < k1; kk += kLT / 64) {
      const int k = kk + w;
      if (k < k1)
        for (int q = lane; q < nw; q += 64)
          wbuf[w][q] = mask[(int64_t)q * tc + k];
      __syncthreads();
      if (k < k1) {
        const int64_t row = ts + k;
        int cnt = 0;
        for (int s = 0; s < cc; s += 64) {
          bool in = false;
          int32_t id = 0;
          if (s + lane < cc) {
            const uint64_t e = srt[s + lane];
            const uint32_t j = (uint32_t)e;
            id = (int32_t)(e >> 32);
            in = wbuf[w][j >> 5] >> (j & 31u) & 1u;
          }
          cnt = append(a, row, cnt, in, id);
        }
        if (lane == 0 && cnt != a.off[row + 1] - a.off[row])
          atomicOr(a.bad, 1);
      }
      __syncthreads();
    }
    return;
  }
  if (threadIdx.x == 0) {
    lo_s = INT32_MAX;
    hi_s = -1;
  }
  __syncthreads();
  int lo = INT32_MAX, hi = -1;
  for (int i = threadIdx.x; i < cc; i += kLT) {
    lo = min(lo, cand[i]);
    hi = max(hi, cand[i]);
  }
  atomicMin(&lo_s, lo);
  atomicMax(&hi_s, hi);
  __syncthreads();
  // rows' counts so far live in srt's upper half, the window's table below
  int32_t *pos = reinterpret_cast<int32_t *>(srt);
  int32_t *done = pos + kSortMax;
  for (int k = threadIdx.x; k < tc; k += kLT) done[k] = 0;
  const int64_t first = lo_s, last = hi_s;
  for (int64_t b = first; b <= last; b += kSortMax) {
    for (int i = threadIdx.x; i < kSortMax; i += kLT) pos[i] = -1;
    __syncthreads();
    for (int i = threadIdx.x; i < cc; i += kLT) {
      const int64_t r = (int64_t)cand[i] - b;
      if (r >= 0 && r < kSortMax) pos[r] = i;
    }
    __syncthreads();
    for (int k = k0 + w; k < k1; k += kLT / 64) {
      const int64_t row = ts + k;
      int cnt = done[k];
      for (int s = 0; s < kSortMax; s += 64) {
        const int32_t j = pos[s + lane];
        const bool in =
            j >= 0 && (mask[(int64_t)(j >> 5) * tc + k] >> (j & 31) & 1u);
        cnt = append(a, row, cnt, in, (int32_t)(b + s + lane));
      }
      if (lane == 0) done[k] = cnt;
    }
    __syncthreads();
  }
  for (int k = k0 + (int)threadIdx.x; k < k1; k += kLT)
    if (done[k] != a.off[ts + k + 1] - a.off[ts + k]) atomicOr(a.bad, 1);
}

}  // namespace

// Entries expanded per launch: the device buffer is bounded by this (128
// MiB) whatever the lists' size, unless one row alone is longer.
constexpr int64_t kListPart = (int64_t)1 << 24;

int stage_lists(Ctx *c, int64_t *off, int64_t *ids, int64_t cap) {
  const int64_t n = c->n;
  FSPH_TRY(ensure(c, c->list_off, (size_t)(n + 2) * 8));
  int64_t *doff = c->list_off.as<int64_t>();
  int *bad = reinterpret_cast<int *>(doff + n + 1);
  FSPH_TRY(scan_i32_to_i64(c, c->f[PF_NNGB].as<int32_t>(), doff, n));
  FSPH_HIP(c, hipMemsetAsync(bad, 0, sizeof(int), c->stream));
  FSPH_HIP(c, hipMemcpyAsync(off, doff, (size_t)(n + 1) * 8,
                             hipMemcpyDeviceToHost, c->stream));
  int64_t total = 0;
  FSPH_TRY(read_scan_total(c, doff + n, &total));
  if (!ids) return FSPH_OK;
  if (cap < total) return fail(c, FSPH_E_CAP, "ids buffer too small");
  for (int64_t r0 = 0; r0 < n;) {
    // as many whole rows as fit a part, at least one
    int64_t r1 = std::upper_bound(off + r0 + 1, off + n + 1,
                                  off[r0] + kListPart) - off - 1;
    if (r1 <= r0) r1 = r0 + 1;
    const int64_t m = off[r1] - off[r0];
    if (m > 0) {
      FSPH_TRY(ensure(c, c->list_ids, (size_t)m * 8));
      const ListArgs a{c->tstart.as<int32_t>(), c->tcount.as<int32_t>(),
                       c->tslot.as<int32_t>(),  c->tccount.as<int32_t>(),
                       c->cand.as<int32_t>(),   c->tmoff.as<int64_t>(),
                       c->mask.as<uint32_t>(),  c->ccap,
                       c->nt,                   doff,
                       r0,                      r1,
                       c->list_ids.as<int64_t>(), bad};
      k_lists<<<(unsigned)c->nt, kLT, 0, c->stream>>>(a);
      FSPH_HIP(c, hipGetLastError());
      FSPH_HIP(c, hipMemcpyAsync(ids + off[r0], c->list_ids.p, (size_t)m * 8,
                                 hipMemcpyDeviceToHost, c->stream));
    }
    r0 = r1;
  }
  int wrong = 0;
  FSPH_HIP(c, hipMemcpyAsync(&wrong, bad, sizeof(int), hipMemcpyDeviceToHost,
                             c->stream));
  FSPH_HIP(c, hipStreamSynchronize(c->stream));
  if (wrong) return fail(c, FSPH_E_ARG, "inconsistent neighbour count");
  return FSPH_OK;
}

}  // namespace fsph
