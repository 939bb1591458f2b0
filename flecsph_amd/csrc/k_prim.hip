// k_prim.hip -- device primitives: block/wave scans and an exclusive scan
// over int64: one workgroup for up to 16,384 items, otherwise one pass over
// tiles of 4,096 items that take their prefix from the tiles before them
// (decoupled look-back).
#include "fsph_internal.h"

namespace fsph {

namespace {

constexpr int kScanThreads = 256;

// Inclusive scan over the wavefront with DPP moves (both halves of the word;
// the sum carries between them).
template <int CTRL, int ROWS>
__device__ inline int64_t dpp_add(int64_t v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS,
                                             0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(
      0, (int)(uint32_t)((uint64_t)v >> 32), CTRL, ROWS, 0xf, false);
  return v + (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ inline int64_t wave_inclusive_scan(int64_t v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // lane 15 of rows 0, 2 to rows 1, 3
  return dpp_add<0x143, 0xc>(v);  // lane 31 to rows 2, 3
}
__device__ inline int64_t last_lane(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi =
      __builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), 63);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Exclusive scan of the ROWS x 64 consecutive items from `base` that a
// wavefront owns, lane l holding item 64 r + l of row r (so that loads and
// stores are coalesced; with each thread holding consecutive items, 128
// bytes apart from its neighbour's, the one-workgroup scan took 17 us for
// 10,000 items, half of it waiting for the strided loads).  v: the items,
// then their prefixes.  Returns the sum.
template <int ROWS, class In>
__device__ inline int64_t scan_rows(const In *in, int64_t base, int rows,
                                    int64_t n, int64_t (&v)[ROWS]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int64_t i = base + r * 64 + lane;
    v[r] = r < rows && i < n ? (int64_t)in[i] : 0;
  }
  int64_t run = 0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    if (r < rows) {
      const int64_t inc = wave_inclusive_scan(v[r]);
      v[r] = run + inc - v[r];
      run += last_lane(inc);
    }
  return run;
}
template <int ROWS>
__device__ inline void put_rows(int64_t *out, int64_t base, int rows,
                                int64_t n, int64_t ex,
                                const int64_t (&v)[ROWS]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int64_t i = base + r * 64 + lane;
    if (r < rows && i < n) out[i] = ex + v[r];
  }
}

// Single-pass scan.  Each workgroup draws its tile from a counter (so every
// tile before it has started), scans its items, publishes its total, and
// wave 0 walks back over the published states of the preceding tiles, 64 at
// a time, until it meets one that holds its inclusive prefix.  A state is
// one 64-bit word (2 status bits over a 62-bit signed value) written and
// read atomically at device scope.  Two halves of states alternate between
// scans: the running scan clears the other half and its counter for the
// next one, so no clearing launch is needed.
constexpr int kOneItems = 16;
constexpr int64_t kOneTile = (int64_t)kScanThreads * kOneItems;
constexpr uint64_t kStAgg = 1ull << 62, kStInc = 2ull << 62;
constexpr uint64_t kStVal = (1ull << 62) - 1;
constexpr int kSpinLimit = 1 << 20;  // a safety bound: predecessors run

__device__ inline uint64_t st_load(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_store(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int64_t st_value(uint64_t w) {
  return (int64_t)(w << 2) >> 2;
}
__device__ inline int64_t wave_sum(int64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

struct ScanState {
  uint64_t *st;     // this scan's tile states
  uint64_t *clear;  // the other half (cleared here)
  int64_t cap;      // states per half
  unsigned *ctr, *ctr_clear;
  int *flags;
};

template <class In>
__global__ __launch_bounds__(kScanThreads) void k_scan_one(
    const In *in, int64_t n, int64_t *out, ScanState S) {
  __shared__ int tile_s;
  __shared__ int64_t prefix_s;
  if (threadIdx.x == 0) tile_s = (int)atomicAdd(S.ctr, 1u);
  __syncthreads();
  const int tile = tile_s, nt = (int)gridDim.x, lane = threadIdx.x & 63;
  if (tile >= nt) {  // a counter left dirty by a scan that never ran
    if (threadIdx.x == 0) atomicOr(S.flags, kFlagScanStall);
    return;
  }
  for (int64_t j = (int64_t)tile * kScanThreads + threadIdx.x; j < S.cap;
       j += (int64_t)nt * kScanThreads)
    S.clear[j] = 0;
  if (tile == 0 && threadIdx.x == 0) *S.ctr_clear = 0;
  __shared__ int64_t wsum[kScanThreads / 64];
  const int w = threadIdx.x >> 6;
  const int64_t base = (int64_t)tile * kOneTile + w * (kOneItems * 64);
  int64_t v[kOneItems];
  const int64_t s = scan_rows<kOneItems>(in, base, kOneItems, n, v);
  if (lane == 0) wsum[w] = s;
  __syncthreads();
  int64_t ex = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kScanThreads / 64; ++i) {
    if (i < w) ex += wsum[i];
    tot += wsum[i];
  }
  if (threadIdx.x < 64) {
    int64_t excl = 0;
    if (tile == 0) {
      if (lane == 0) st_store(&S.st[0], kStInc | ((uint64_t)tot & kStVal));
    } else {
      if (lane == 0) st_store(&S.st[tile], kStAgg | ((uint64_t)tot & kStVal));
      int64_t j0 = tile - 1;
      int spins = 0;
      bool stalled = false;
      while (true) {
        const int64_t j = j0 - lane;
        uint64_t w = j >= 0 ? st_load(&S.st[j]) : kStInc;
        while (__ballot((w >> 62) == 0)) {
          if (++spins > kSpinLimit) {
            stalled = true;
            break;
          }
          if ((w >> 62) == 0) w = st_load(&S.st[j]);
        }
        if (stalled) break;
        const uint64_t inc = __ballot((w >> 62) == 2);
        const int64_t val = st_value(w);
        if (inc) {
          const int first = __builtin_ctzll(inc);
          excl += wave_sum(lane <= first ? val : 0);
          break;
        }
        excl += wave_sum(val);
        j0 -= 64;
      }
      if (stalled && lane == 0) atomicOr(S.flags, kFlagScanStall);
      if (lane == 0)
        st_store(&S.st[tile], kStInc | ((uint64_t)(excl + tot) & kStVal));
    }
    if (lane == 0) prefix_s = excl;
  }
  __syncthreads();
  put_rows(out, base, kOneItems, n, prefix_s + ex, v);
  if (tile == nt - 1 && threadIdx.x == 0) out[n] = prefix_s + tot;
}


// One-workgroup scan: wavefront w takes the w-th run of `rows` x 64 items
// (every item is read before a prefix is written, so in may equal out).
constexpr int kSmallThreads = 1024;
constexpr int kSmallItems = 16;
constexpr int64_t kSmallMax = (int64_t)kSmallThreads * kSmallItems;

template <class In>
__global__ __launch_bounds__(kSmallThreads) void k_scan_small(
    const In *in, int64_t n, int64_t *out) {
  __shared__ int64_t wsum[kSmallThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rows = (int)((n + kSmallThreads - 1) / kSmallThreads);
  const int64_t base = (int64_t)w * rows * 64;
  int64_t v[kSmallItems];
  const int64_t s = scan_rows<kSmallItems>(in, base, rows, n, v);
  if (lane == 0) wsum[w] = s;
  __syncthreads();
  int64_t ex = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kSmallThreads / 64; ++i) {
    if (i < w) ex += wsum[i];
    tot += wsum[i];
  }
  put_rows(out, base, rows, n, ex, v);
  if (threadIdx.x == 0) out[n] = tot;
}

template <class In>
int scan_impl(Ctx *c, const In *in, int64_t *out, int64_t n) {
  if (n <= 0) {
    FSPH_HIP(c, hipMemsetAsync(out, 0, sizeof(int64_t), c->stream));
    return 0;
  }
  if (n <= kSmallMax) {
    k_scan_small<In><<<1, kSmallThreads, 0, c->stream>>>(in, n, out);
    return hip_check(c, hipGetLastError(), "scan");
  }
  const int64_t nt = (n + kOneTile - 1) / kOneTile;
  if (nt > c->scan_cap) {
    const int64_t cap = nt + nt / 2 + 64;
    const size_t bytes = (size_t)(2 * cap + 2) * sizeof(uint64_t);
    FSPH_TRY(ensure(c, c->scan_state, bytes));
    FSPH_HIP(c, hipMemsetAsync(c->scan_state.p, 0, bytes, c->stream));
    c->scan_cap = cap;
    c->scan_parity = 0;
  }
  const int p = c->scan_parity;
  c->scan_parity ^= 1;
  uint64_t *st = c->scan_state.as<uint64_t>();
  unsigned *ctr = reinterpret_cast<unsigned *>(st + 2 * c->scan_cap);
  const ScanState S{st + p * c->scan_cap, st + (1 - p) * c->scan_cap,
                    c->scan_cap, ctr + 2 * p, ctr + 2 * (1 - p),
                    c->flags.as<int>() + kScanWord};
  k_scan_one<In><<<(unsigned)nt, kScanThreads, 0, c->stream>>>(in, n, out, S);
  return hip_check(c, hipGetLastError(), "scan");
}

}  // namespace

int scan_i64(Ctx *c, const int64_t *in, int64_t *out, int64_t n) {
  return scan_impl<int64_t>(c, in, out, n);
}

int scan_i32_to_i64(Ctx *c, const int32_t *in, int64_t *out, int64_t n) {
  return scan_impl<int32_t>(c, in, out, n);
}

}  // namespace fsph
