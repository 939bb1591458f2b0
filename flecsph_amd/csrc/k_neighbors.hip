// k_neighbors.hip -- neighbour tiles of every SPH group.
//
// tree_topology::traversal_sph (tree_topology.h:213-442) visits, for each
// group G, every node whose ancestors all pass two tests against G: the
// node box intersects G's box (intersects_box_box), and the node box is
// within h_k of some particle k of G (intersects_sphere_box).  Leaves under
// accepted nodes are then kept if they pass a centre-of-mass filter and
// d(k,b) <= max(h_k, h_b).  Here one wavefront per group walks the octree
// with an LDS stack, 64 nodes per step, and appends reached leaves to the
// group's candidate tile; a second kernel finds, for every (tile row,
// candidate) pair, whether the reference's predicate holds and stores it as a
// bitmask row per particle: mask[moff[t] + w*rows + k] bit j <=> candidate
// 32w+j neighbours row k.  The SPH passes stage candidates in LDS and walk
// these bits.
// Both decide nearly every test in FP32, on coordinates relative to the unit,
// where the rounding cannot change the outcome, and the others in FP64 in the
// reference's operation order without FMA contraction, so nodes and bits are
// the reference's.  The gather form (tiles of the smoothing-length solver)
// needs only the masks to be exact: its traversal keeps a superset, by balls
// about the nodes' centres of mass and spheres about eight particles.
#include <cfloat>

#include <type_traits>

#include "fsph_internal.h"
#include "pair_sched.h"

namespace fsph {

namespace {

constexpr int kW = 64;          // one wavefront per group
// LDS traversal stack (node indices) in three sizes: the smaller, the more
// groups are resident per CU (the 1M polytrope's groups need at most about
// 420 entries: 512 entries give about 5.9 wavefronts per SIMD, 1024 about
// 4.5).  A traversal that overflows is run again with the next size, which
// the context keeps from then on (one state for the SPH tiles and one for
// the gather tiles).
constexpr int kStackSmall = 512, kStackMid = 1024, kStackLarge = 4096;
constexpr int kMaxGroup = 128;  // tree_topology::sub_entities_
constexpr int kRowBlock = 8;    // mask rows tested as one unrolled block

__device__ inline bool box_box(const double *a, const double *b) {
  // intersects_box_box(min1,max1,min2,max2), tree_geometry.h:306-314
  return !((a[3] < b[0] || a[4] < b[1] || a[5] < b[2]) ||
           (b[3] < a[0] || b[4] < a[1] || b[5] < a[2]));
}

__device__ inline bool sphere_box(const double *bx, double c0, double c1,
                                  double c2, double r) {
  // intersects_sphere_box, tree_geometry.h:329-341
#pragma clang fp contract(off)
  double x0 = c0 < bx[3] ? c0 : bx[3];
  double x1 = c1 < bx[4] ? c1 : bx[4];
  double x2 = c2 < bx[5] ? c2 : bx[5];
  x0 = x0 < bx[0] ? bx[0] : x0;
  x1 = x1 < bx[1] ? bx[1] : x1;
  x2 = x2 < bx[2] ? bx[2] : x2;
  const double dist =
      (x0 - c0) * (x0 - c0) + (x1 - c1) * (x1 - c1) + (x2 - c2) * (x2 - c2);
  return dist <= r * r;
}

__device__ inline bool within_distance2(double a0, double a1, double a2,
                                        double b0, double b1, double b2,
                                        double r) {
  // within_distance2, tree_geometry.h:272-276
#pragma clang fp contract(off)
  const double d =
      (a0 - b0) * (a0 - b0) + (a1 - b1) * (a1 - b1) + (a2 - b2) * (a2 - b2);
  return d <= r * r;
}

__device__ inline float lane_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

struct TravArgs {
  const double *x, *y, *z, *h;
  const double *box;     // 6 per node
  const double *com, *nrad;  // 3 and 1 per node (gather form)
  const int32_t *child;  // 8 per node
  const int32_t *gstart, *gcount, *gnode;
  int32_t *cand;
  int32_t *ccount;
  int64_t ccap;
  int *flags;
  // gather form (smoothing-length solver): sphere radius rscale * h_k and
  // no group-box test; the SPH form takes h_k and the box test.
  double rscale;
  const float *hprop;    // gather radius base instead of h (or null)
  const int32_t *glist;  // tile slot -> group (or null: slot = group)
  // batched mode: the walk starts at the root of the group's instance
  const int32_t *inst, *root;
  // out, per row: position relative to the unit's first particle and
  // squared radius in FP32, what the masks screen with
  float4 *rowrel;
  int64_t *words;  // out: the unit's mask words (rows x 32-candidate words)
};

// MAXG: the largest group (64 when group_max <= 64, else kMaxGroup), which
// sizes the group's LDS arrays.
//
// A node passes the sphere test if some particle's sphere meets its box.
// The test is FP64 in the reference's operation order; nearly every node is
// decided by FP32 forms of it, in coordinates relative to the group's first
// particle and in units of R, the largest coordinate or sphere bound of the
// group there: every value that can decide a test is at most 2, its rounding
// at most 2^-23, and the rounding of d^2 - r^2 below 18 * 2^-24, so a
// difference beyond kScreen = 2^-19 has the exact test's sign.
//   1. lanes = nodes: for every eight particles, the sphere about all their
//      spheres (a node that meets none of these is rejected) and the sphere
//      of the particle nearest its centre (a node that meets one of these is
//      accepted).
//   2. lanes = particles: the nodes still open, one after the other (the
//      node's box from its lane, the spheres in registers).
//   3. where no sphere accepts a node and one is too close to tell, the exact
//      test, lanes = particles, from memory.
// The gather form, whose masks decide, needs a superset of the leaves within
// the particles' own radii: there a node is kept if the ball about its centre
// of mass that holds its particles meets the sphere about some eight (the
// ball has no margin of h / 2 around the particles, as the box has, and costs
// fewer operations), and the leaves under kept nodes, 64 at a time in the
// order they were reached, stay candidates if they lie in such a sphere.
// Particles far apart for their radii (a diffuse tile beside a dense clump,
// which the sphere about eight of them may hold although no own sphere comes
// near it) are tested by their own spheres instead: where such an eight's
// sphere has more than kSparse times the largest own radius (1.5 to 2.5 times
// for particles with 40 to 100 neighbours each), and where a walk by eights
// overflows the largest stack or kFineCap candidates or more, which starts it
// over (below that the capacity grows: 300 neighbours each need 8,192, and
// starting over on every call took 10% longer).
// Where the screen is off (a position that is not a number or infinite in the
// unit's first particle, or a scale beyond FP32's reach), its nodes take the
// exact box test and the leaves under them all stay, so that a particle whose
// position is not a number still meets nothing.
//
// Measured: SPH form 551 -> 290 us for 1.5M particles of a collapse, 505 ->
// 286 for a 1M polytrope, 200 -> 99 for 64^3 (testing each node's own
// particles in FP64, one after the other, waited for the slowest lane: the
// one node of 64 that meets many groups of eight and no sphere); gather form
// 2,560 -> 800 us (1,260 with three scattered coordinate loads per leaf child
// in place of the queue).  Filtering the SPH form's leaves the same way takes
// 40% of the masks' work off and costs as much here: 64^3 was slower.
constexpr int kEight = 8;
constexpr float kSparse = 8.f;
constexpr int64_t kFineCap = 16384;
constexpr float kScreen = 1.0f / (1 << 19);

// d^2 - r^2 of the box l .. h and the sphere p (r^2 in p.w)
__device__ inline float sphere_gap(const float (&l)[3], const float (&h)[3],
                                   const float4 &p) {
  const float dx = fmaxf(fmaxf(l[0] - p.x, p.x - h[0]), 0.f),
              dy = fmaxf(fmaxf(l[1] - p.y, p.y - h[1]), 0.f),
              dz = fmaxf(fmaxf(l[2] - p.z, p.z - h[2]), 0.f);
  return __builtin_fmaf(
      dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, -p.w)));
}
template <int kStack, int MAXG, bool GF>
__global__ __launch_bounds__(kW) void k_traverse(TravArgs a) {
#pragma clang fp contract(off)
  // x, y, z, r^2 of the screen (gather form, after the eights are made: r),
  // then of each eight the sphere about them (r); the sphere of the one inside
  constexpr int kOuter = MAXG, kSph = MAXG + MAXG / kEight;
  __shared__ float4 sph[kSph], inner[MAXG / kEight];
  float4 *const outer = sph + kOuter;
  __shared__ int32_t leaves[GF ? 9 * kW : 1];  // reached, not yet filtered
  __shared__ int32_t stk[kStack];
  constexpr int NK = MAXG / kW;
  const int lane = threadIdx.x;
  const int64_t gi = xcd_item(blockIdx.x, gridDim.x);
  const int64_t g = a.glist ? a.glist[gi] : gi;
  const int64_t gs = a.gstart[g];
  const int gc = a.gcount[g];
  const int gn = GF ? -1 : a.gnode[g];
  auto radius = [&](int64_t p) {
    return !GF ? a.h[p] : a.rscale * (a.hprop ? (double)a.hprop[p] : a.h[p]);
  };
  const double c0 = a.x[gs], c1 = a.y[gs], c2 = a.z[gs];
  double X[NK][3], rad[NK], R = 0;
  float4 own[NK];  // this lane's spheres
#pragma unroll
  for (int q = 0; q < NK; ++q) {
    const int k = lane + q * kW;
    if (k >= gc) continue;
    X[q][0] = a.x[gs + k];
    X[q][1] = a.y[gs + k];
    X[q][2] = a.z[gs + k];
    rad[q] = radius(gs + k);
    const double e0 = X[q][0] - c0, e1 = X[q][1] - c1, e2 = X[q][2] - c2;
    a.rowrel[gs + k] = make_float4((float)e0, (float)e1, (float)e2,
                                   (float)(rad[q] * rad[q]));
    R = fmax(R, fmax(fmax(fabs(e0), fabs(e1)), fabs(e2)) + fabs(rad[q]));
  }
  for (int o = 32; o > 0; o >>= 1) R = fmax(R, __shfl_xor(R, o, 64));
  // (outside this range, infinities included, every test is the exact one)
  const bool scr = R > 1e-150 && R < 1e150 && c0 - c0 + c1 - c1 + c2 - c2 == 0;
  const double inv = scr ? 1.0 / R : 0.0;
#pragma unroll
  for (int q = 0; q < NK; ++q) {
    const int k = lane + q * kW;
    // past the group, or with a NaN: a sphere that nothing meets
    const double nan = k < gc ? X[q][0] + X[q][1] + X[q][2] + rad[q] : NAN;
    own[q] = nan == nan ? make_float4((float)((X[q][0] - c0) * inv),
                                      (float)((X[q][1] - c1) * inv),
                                      (float)((X[q][2] - c2) * inv),
                                      (float)((rad[q] * inv) * (rad[q] * inv)))
                        : make_float4(0.f, 0.f, 0.f, -4.f);
    sph[k] = own[q];
  }
  double gb[6];
  if (gn >= 0) {
    for (int d = 0; d < 6; ++d) gb[d] = a.box[6 * (int64_t)gn + d];
  } else {
    // Without a group node (gather mode, single-particle groups): the box
    // hull of the group's spheres, widened by 1e-9 of |centre| + radius,
    // well beyond the rounding of the sphere test.  A node that meets a
    // sphere meets the hull, so testing it first only saves sphere tests.
    for (int d = 0; d < 3; ++d) {
      gb[d] = DBL_MAX;
      gb[d + 3] = -DBL_MAX;
    }
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      if (lane + q * kW >= gc) continue;
      for (int d = 0; d < 3; ++d) {
        const double r = rad[q] + 1e-9 * (fabs(X[q][d]) + rad[q]);
        gb[d] = fmin(gb[d], X[q][d] - r);
        gb[d + 3] = fmax(gb[d + 3], X[q][d] + r);
      }
    }
    for (int o = 32; o > 0; o >>= 1)
      for (int d = 0; d < 3; ++d) {
        gb[d] = fmin(gb[d], __shfl_xor(gb[d], o, 64));
        gb[d + 3] = fmax(gb[d + 3], __shfl_xor(gb[d + 3], o, 64));
      }
  }
  __syncthreads();
  const int n8 = (gc + kEight - 1) / kEight;
  if (lane >= n8 && lane < MAXG / kEight) {  // (the loops below go in pairs)
    outer[lane] = make_float4(INFINITY, 0.f, 0.f, 0.f);
    inner[lane] = make_float4(0.f, 0.f, 0.f, -4.f);
  }
  bool sparse = false;
  if (lane < n8) {
    float lo[3] = {INFINITY, INFINITY, INFINITY},
          hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    float4 p[kEight];
#pragma unroll
    for (int u = 0; u < kEight; ++u) {
      p[u] = sph[lane * kEight + u];
      if (p[u].w < 0.f) continue;
      const float c[3] = {p[u].x, p[u].y, p[u].z};
      for (int d = 0; d < 3; ++d) {
        lo[d] = fminf(lo[d], c[d]);
        hi[d] = fmaxf(hi[d], c[d]);
      }
    }
    const float m[3] = {0.5f * (lo[0] + hi[0]), 0.5f * (lo[1] + hi[1]),
                        0.5f * (lo[2] + hi[2])};
    float far = -1.f, best = INFINITY, rmax = 0.f;
    float4 in = make_float4(0.f, 0.f, 0.f, -4.f);
#pragma unroll
    for (int u = 0; u < kEight; ++u) {
      if (p[u].w < 0.f) continue;
      const float e0 = p[u].x - m[0], e1 = p[u].y - m[1], e2 = p[u].z - m[2];
      const float dd = sqrtf(e0 * e0 + e1 * e1 + e2 * e2);
      far = fmaxf(far, dd + sqrtf(p[u].w));
      rmax = fmaxf(rmax, p[u].w);
      if (dd < best) {
        best = dd;
        in = p[u];
      }
    }
    // (|centre| <= 1 and far <= 5: 4 kScreen is many of their roundings, and
    // of those of the tests below; eight NaNs meet nothing)
    outer[lane] = far < 0.f ? make_float4(INFINITY, 0.f, 0.f, 0.f)
                            : make_float4(m[0], m[1], m[2],
                                          far + 4.f * kScreen);
    inner[lane] = in;
    sparse = far > kSparse * sqrtf(rmax);
  }
  // gather form: the spheres tested, the eights' or the particles' own
  int q_lo = kOuter, q_hi = kOuter + n8;
  if (GF && __ballot(sparse)) {
    q_lo = 0;
    q_hi = gc;
  }
  if (lane == 0) stk[0] = a.root ? a.root[a.inst[gs]] : 0;  // root
  __syncthreads();
  if (GF) {
#pragma unroll
    for (int q = 0; q < NK; ++q)
      sph[lane + q * kW] =
          own[q].w < 0.f ? make_float4(INFINITY, 0.f, 0.f, 0.f)
                         : make_float4(own[q].x, own[q].y, own[q].z,
                                       sqrtf(own[q].w) + 4.f * kScreen);
    __syncthreads();
  }
  // Whether the ball of radius r about e (normalised) meets some of these
  // spheres.  The margins of the spheres' radii are many roundings of
  // coordinates and radii up to 5, the factor many of larger ones; a NaN
  // meets every sphere.
  auto meets = [&](float e0, float e1, float e2, float r) {
    bool miss = true;
    for (int q0 = q_lo; q0 < q_hi; q0 += 2)
#pragma unroll
      for (int q = q0; q < q0 + 2; ++q) {
        const float4 o = sph[q];
        const float f0 = e0 - o.x, f1 = e1 - o.y, f2 = e2 - o.z, s = r + o.w;
        miss &= __builtin_fmaf(f0, f0, __builtin_fmaf(f1, f1, f2 * f2)) >
                s * s * (1.f + 4.f * kScreen);
      }
    return !miss;
  };
  int sp = 1, nl = 0;
  int64_t ncand = 0;
  const int64_t cbase = gi * a.ccap;
  bool overflow = false;
  // (gather form) after an overflow of a walk by eights: from the root again
  auto again = [&] {
    q_lo = 0;
    q_hi = gc;
    overflow = false;
    sp = 1;
    nl = 0;
    ncand = 0;
    __syncthreads();
    if (lane == 0) stk[0] = a.root ? a.root[a.inst[gs]] : 0;
    __syncthreads();
  };
  while (sp > 0) {
    const int nb = sp < kW ? sp : kW;
    sp -= nb;
    const int node = lane < nb ? stk[sp + lane] : -1;
    __syncthreads();
    bool acc = false;
    // the children are loaded with the box or ball (one memory latency per
    // step; a rejected node's are not used)
    int32_t ch[8];
    if (GF) {
      if (node >= 0) {
        const double *nc = a.com + 3 * (int64_t)node;
        const int32_t *nch = a.child + 8 * (int64_t)node;
        const float e0 = (float)((nc[0] - c0) * inv),
                    e1 = (float)((nc[1] - c1) * inv),
                    e2 = (float)((nc[2] - c2) * inv);
        const float r = (float)(a.nrad[node] * inv);
        for (int j = 0; j < 8; ++j) ch[j] = nch[j];
        if (scr) {
          acc = meets(e0, e1, e2, r);
        } else {
          for (int64_t p = gs; p < gs + gc && !acc; ++p)
            acc = sphere_box(a.box + 6 * (int64_t)node, a.x[p], a.y[p],
                             a.z[p], radius(p));
        }
      }
    } else {
      double bx[6] = {0, 0, 0, 0, 0, 0};
      bool open = false;
      if (node >= 0) {
        const double *nbx = a.box + 6 * (int64_t)node;
        const int32_t *nch = a.child + 8 * (int64_t)node;
        for (int d = 0; d < 6; ++d) bx[d] = nbx[d];
        for (int j = 0; j < 8; ++j) ch[j] = nch[j];
        open = box_box(bx, gb);
      }
      const float l[3] = {(float)((bx[0] - c0) * inv),
                          (float)((bx[1] - c1) * inv),
                          (float)((bx[2] - c2) * inv)},
                  h[3] = {(float)((bx[3] - c0) * inv),
                          (float)((bx[4] - c1) * inv),
                          (float)((bx[5] - c2) * inv)};
      if (scr) {
        float to = INFINITY, ti = INFINITY;
        for (int q0 = 0; q0 < n8; q0 += 2)
#pragma unroll
          for (int q = q0; q < q0 + 2; ++q) {
            float4 o = outer[q];
            o.w *= o.w;
            to = fminf(to, sphere_gap(l, h, o));
            ti = fminf(ti, sphere_gap(l, h, inner[q]));
          }
        acc = open && ti < -kScreen;
        open = open && !acc && to <= 0.f;
      }
      uint64_t todo = __ballot(open);
      while (todo) {
        const int u = __builtin_ctzll(todo);
        todo &= todo - 1;
        bool in = false, unsure = !scr;
        if (scr) {
          float lu[3], hu[3], t = INFINITY;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            lu[d] = lane_f(l[d], u);
            hu[d] = lane_f(h[d], u);
          }
#pragma unroll
          for (int q = 0; q < NK; ++q)
            t = fminf(t, sphere_gap(lu, hu, own[q]));
          in = t < -kScreen;
          unsure = t <= kScreen;
        }
        uint64_t hit = __ballot(in);
        if (!hit && __ballot(unsure)) {
          const double *nbx =
              a.box + 6 * (int64_t)__builtin_amdgcn_readlane(node, u);
          bool ex = false;
#pragma unroll
          for (int q = 0; q < NK; ++q) {
            const int64_t p = gs + lane + q * kW;
            if (unsure && lane + q * kW < gc)
              ex |= sphere_box(nbx, a.x[p], a.y[p], a.z[p], radius(p));
          }
          hit = __ballot(ex);
        }
        if (lane == u) acc = hit != 0;
      }
    }
    int nnode = 0, nleaf = 0;
    if (acc) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        nnode += ch[j] >= 0;
        nleaf += ch[j] <= -2;
      }
    }
    // both counts are at most 512 over the wavefront: one packed scan
    const int cnt = nnode | nleaf << 16;
    const int inc = sched::wave_scan_incl(cnt);
    const int all = __builtin_amdgcn_readlane(inc, 63);
    const int tn = all & 0xffff, tl = all >> 16;
    if (sp + tn > kStack) {
      if (GF && kStack == kStackLarge && scr && q_lo) {
        again();
        continue;
      }
      overflow = true;
      if (lane == 0) atomicOr(a.flags, kFlagStack);
      break;
    }
    if (!GF && ncand + tl > a.ccap) {
      overflow = true;
      if (lane == 0) atomicOr(a.flags, kFlagCand);
      break;
    }
    if (acc) {
      int qn = sp + ((inc - cnt) & 0xffff);
      int ql = nl + ((inc - cnt) >> 16);
      int32_t *lp = GF ? leaves : a.cand + cbase + ncand;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (ch[j] >= 0)
          stk[qn++] = ch[j];
        else if (ch[j] <= -2)
          lp[ql++] = (int32_t)leaf_of(ch[j]);
      }
    }
    sp += tn;
    if (GF)
      nl += tl;
    else
      ncand += tl;
    __syncthreads();
    if (!GF) continue;
    int done = 0;
    while (nl - done >= kW || (sp == 0 && nl > done)) {
      const bool on = lane < nl - done;
      const int64_t p = on ? leaves[done + lane] : gs;
      const float e0 = (float)((a.x[p] - c0) * inv),
                  e1 = (float)((a.y[p] - c1) * inv),
                  e2 = (float)((a.z[p] - c2) * inv);
      const bool keep = on && (!scr || meets(e0, e1, e2, 0.f));
      const uint64_t km = __ballot(keep);
      const int nk = __popcll(km);
      if (ncand + nk > a.ccap) {
        overflow = true;
        break;
      }
      if (keep)
        a.cand[cbase + ncand + __popcll(km & ((1ull << lane) - 1))] =
            (int32_t)p;
      ncand += nk;
      done += kW;
    }
    if (overflow) {
      if (scr && q_lo && a.ccap >= kFineCap) {
        again();
        continue;
      }
      if (lane == 0) atomicOr(a.flags, kFlagCand);
      break;
    }
    if (done && nl > done) {  // fewer than kW are left: to the front
      const int32_t v = leaves[min(done + lane, 9 * kW - 1)];
      __syncthreads();
      leaves[lane] = v;
    }
    nl = max(nl - done, 0);
    __syncthreads();
  }
  if (lane == 0) {  // (an overflowed walk leaves zero candidates)
    const int32_t cc = overflow ? 0 : (int32_t)ncand;
    a.ccount[gi] = cc;
    a.words[gi] = (int64_t)gc * ((cc + 31) / 32);
  }
}

// Mailbox of the tile stage: [0] error flags, [1] mask words.
__global__ void k_tile_mail(const int *__restrict__ flags,
                            const int64_t *__restrict__ words,
                            int64_t *__restrict__ mail) {
  if (threadIdx.x == 0) {
    mail_put(mail + 0, flags[0] | flags[kScanWord]);
    mail_put(mail + 1, *words);
  }
}

struct MaskArgs {
  const double *x, *y, *z, *h;
  const double *com, *rad, *lap;
  const int32_t *gstart, *gcount, *gnode;
  int32_t *cand, *ccount;  // traversal output per slot
  const int64_t *moff;
  int64_t ccap;
  uint32_t *mask;
  int32_t *nngb;  // may be null
  // gather mode: bit set iff r_kb < rscale * h_k (strict, own radius only)
  double rscale;
  const float *hprop;    // gather radius base instead of h (or null)
  const int32_t *glist;  // tile slot -> group (or null)
  // SPH tiles: each tile's group, rows and candidate slot, and the outputs
  // per tile (gather units are their own tiles, compacted in place into
  // ccount/cand/mask at moff)
  const int32_t *tgrp, *tstart, *tcount, *tslot;
  int32_t *tcc;
  int64_t *tmo;
  const float4 *rowrel;  // written by the traversal
};

// Bit compress (the "compress" of Hacker's Delight, 2nd ed., section 7-4):
// moves the bits of x selected by m to the low end in order.  The five
// shift masks depend on m only, so they are computed once per mask word and
// applied to every row's word.
struct Compress {
  uint32_t mv[5];
};
__device__ inline Compress compress_masks(uint32_t m) {
  Compress c;
  uint32_t mk = ~m << 1;
  for (int i = 0; i < 5; ++i) {
    uint32_t mp = mk ^ (mk << 1);
    mp ^= mp << 2;
    mp ^= mp << 4;
    mp ^= mp << 8;
    mp ^= mp << 16;
    const uint32_t mv = mp & m;
    c.mv[i] = mv;
    m = (m ^ mv) | (mv >> (1 << i));
    mk &= ~mp;
  }
  return c;
}
__device__ inline uint32_t compress(uint32_t x, uint32_t m, const Compress &c) {
  x &= m;
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const uint32_t t = x & c.mv[i];
    x = (x ^ t) | (t >> (1 << i));
  }
  return x;
}

// Row data is read through the scalar cache (the row index is uniform over
// the wavefront): constant-address-space views.
typedef const __attribute__((address_space(4))) double *ConstD;
typedef const __attribute__((address_space(4))) float *ConstF;
__device__ inline ConstD const_view(const double *p) {
  return (ConstD)(uintptr_t)p;
}
__device__ inline ConstF const_view(const float4 *p) {
  return (ConstF)(uintptr_t)p;
}

// v_writelane_b32: `old` with lane `lane` (uniform) replaced by v (uniform).
// The compiler has no __builtin_ form of it; the intrinsic is named (a name it
// does not know fails to link) and not written as inline assembly because an
// instruction that reads a scalar register needs two wait states after the
// comparison that writes it, which the compiler keeps for the instructions it
// knows and not for the text of an assembly block.
__device__ int write_lane(int v, int lane, int old)
    __asm("llvm.amdgcn.writelane.i32");

// Neighbour bits of one tile.  GATHER selects the gather-mode predicate at
// compile time.  One wavefront per tile holds 64 candidates per round, one
// per lane, and takes the rows one after the other: a row's comparison over
// the wavefront is the row's 64 mask bits in a scalar register pair (no bits
// are put together lane by lane), which a v_writelane per word hands to the
// lane that owns the row.
//
// The rows are tested in FP32 first, on positions relative to the unit's
// first particle (scalar loads of the traversal's rowrel): an FP32 add,
// multiply or FMA issues in 2.5 cycles here, an FP64 one in 5.  With
// u = d^2 - max(h_k^2, h_b^2) in FP32 and R the largest coordinate, row or
// candidate, the rounding of the coordinates (2^-24 R each), of d^2 and of
// the bound moves u by less than 84 R^2 2^-24 + max(h^2) 2^-22; outside
// tau = 2^-17 max(R^2, h^2) the sign of u decides, and a round of rows with
// a u inside it (or not a number; about one in a hundred rounds) is tested
// over in FP64 with the reference's operations.  A tau too small to be
// normal counts as infinite: everything is then tested in FP64.  So it is
// from 2^107 on, where tau becomes not a number: d^2 (at most 12 R^2) or h^2
// may overflow there, and an infinite u says nothing of the exact one's sign.
// d <= max(h_k, h_b)^2 is tested there as d <= h_k^2 or d <= h_b^2: squaring
// and rounding are monotone, so the outcome is the same.
//
// Rows go in unrolled blocks of kRowBlock, whose lane numbers and loads are
// then constants: with one scalar unit for four SIMDs, the scalar
// instructions of a loop over rows (mask bookkeeping, lane number, loop)
// bounded it.  The last block may run over the tile's end: its extra rows
// are other tiles' (or the buffer's padding) and their lanes are cleared.
// Sedov 64^3 (474,552 rows and copies) 418 -> 214 us, 1M star 1,000 -> 512,
// 1.5M collapse 1,594 -> 987 and 1,036 -> 713 (gather), against lanes that
// held (row, word) pairs, read the candidates from LDS and put the words
// together bit by bit in FP64; it issues a VALU instruction per 4.3 cycles
// and SIMD there, 13 per row and round.  A hull box over every eight rows
// that skips the rounds which miss it saved nothing: 64 candidates in a row
// cover about the extent of a tile.
//
// The candidates that are no neighbour of any of the tile's rows are
// dropped (about a third on Sedov 64^3): the round's row masks are ORed
// over the lanes, the used candidates are written in order to the tile's
// candidate slot, and every row's bits are compressed to the same used
// positions, so the pair passes stage and walk only used candidates in an
// unchanged order.  A group cut into two tiles has a wavefront for each
// (one for both took as long as the largest group: 1.9 wavefronts per SIMD
// were resident on average on Sedov 64^3), whose candidates go to slots of
// their own; otherwise they are compacted in place, ahead of the reads.  The
// neighbour predicate is the group's (its candidates and its centre-of-mass
// filter) whatever the cut.
template <bool GATHER, int NR>
__global__ __launch_bounds__(kW) void k_masks(MaskArgs a) {
#pragma clang fp contract(off)
  __shared__ double ph2[NR * kW];
  const int lane = threadIdx.x;
  const int64_t t = xcd_item(blockIdx.x, gridDim.x);
  const int64_t g = GATHER ? (a.glist ? a.glist[t] : t) : a.tgrp[t];
  const int64_t g0 = a.gstart[g];  // the unit's first particle
  const int64_t gs = GATHER ? g0 : a.tstart[t];
  const int gc = GATHER ? a.gcount[g] : a.tcount[t];
  const int gn = GATHER ? -1 : a.gnode[g];
  const int64_t cslot = GATHER ? t : g;
  const int cc = a.ccount[cslot];
  const int64_t cbase = cslot * a.ccap;
  const int64_t cout = GATHER ? cbase : (int64_t)a.tslot[t] * a.ccap;
  // the group's mask words hold its tiles one after the other
  const int64_t mout = a.moff[cslot] + (gs - g0) * ((cc + 31) >> 5);
  const double ox = a.x[g0], oy = a.y[g0], oz = a.z[g0];
  const float inf = __builtin_inff();
  float scale2 = 0.f;  // max of the rows' R^2 and squared radii
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int k = lane + r * kW;
    if (k < gc) {
      const double h = !GATHER ? a.h[gs + k]
                               : a.rscale * (a.hprop ? (double)a.hprop[gs + k]
                                                     : a.h[gs + k]);
      ph2[k] = h * h;
      const float4 q = a.rowrel[gs + k];
      const float m = fmaxf(fmaxf(fabsf(q.x), fabsf(q.y)), fabsf(q.z));
      scale2 = fmaxf(scale2, fmaxf(m * m, q.w));
    }
  }
  for (int o = 32; o > 0; o >>= 1)
    scale2 = fmaxf(scale2, __shfl_xor(scale2, o, 64));
  __syncthreads();
  const ConstD X = const_view(a.x + gs), Y = const_view(a.y + gs),
               Z = const_view(a.z + gs);
  const ConstF RR = const_view(a.rowrel + gs);
  double gcom[3] = {0, 0, 0}, gext_lap = 0, grad = 0;
  if (gn >= 0) {
    gcom[0] = a.com[3 * (int64_t)gn];
    gcom[1] = a.com[3 * (int64_t)gn + 1];
    gcom[2] = a.com[3 * (int64_t)gn + 2];
    gext_lap = a.lap[gn];
    grad = a.rad[gn];
  }
  // compaction state: used candidates so far, words written and bits
  // pending (per row k = lane + 64 r)
  int64_t used_so_far = 0;
  uint64_t pend[NR] = {};
  int nb = 0, wi = 0, cnt[NR] = {};
  // The next round's candidates are loaded while the current round's rows
  // are tested, their indices one round earlier still.
  double rx = 0, ry = 0, rz = 0, rh = 0;
  auto index_of = [&](int r0) {
    const int j = r0 + lane;
    return j < cc ? a.cand[cbase + j] : -1;
  };
  auto fetch = [&](int32_t b) {
    if (b < 0) return;
    rx = a.x[b];
    ry = a.y[b];
    rz = a.z[b];
    rh = a.h[b];
  };
  int32_t ccur = index_of(0);
  fetch(ccur);
  int32_t cnext = index_of(kW);
  for (int r0 = 0; r0 < cc; r0 += kW) {
    // a lane without a candidate, or whose candidate fails the
    // centre-of-mass filter, is infinitely far away
    const double cx = rx, cy = ry, cz = rz, ch2 = rh * rh;
    bool on = ccur >= 0;
    if (gn >= 0) {
      // COM filter, tree_topology.h:365-371
      const double ext = ((rh < gext_lap) ? gext_lap : rh) + grad;
      on = on && within_distance2(cx, cy, cz, gcom[0], gcom[1], gcom[2], ext);
    }
    const float fx = on ? (float)(cx - ox) : inf, fy = (float)(cy - oy),
                fz = (float)(cz - oz), fh2 = GATHER ? 0.f : (float)ch2;
    float tau = inf;
    {
      const float m = fmaxf(fmaxf(fabsf((float)(cx - ox)), fabsf(fy)),
                            fabsf(fz));
      const float t2 = 0x1p-17f * fmaxf(scale2, fmaxf(m * m, fh2));
      // (0 for a finite product, else not a number)
      if (t2 > 0x1p-100f) tau = __builtin_fmaf(t2 * 0x1p21f, 0.f, t2);
    }
    const uint64_t far = __ballot(!on);
    fetch(cnext);
    const int32_t cafter = index_of(r0 + 2 * kW);
    // bits of row k over the round's candidates, in lane k % 64
    uint32_t lo[NR] = {}, hi[NR] = {};
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int nrow = gc - r * kW;
#pragma unroll
      for (int k0 = 0; k0 < kW; k0 += kRowBlock) {
        if (k0 >= nrow) break;
        float q[4 * kRowBlock];
#pragma unroll
        for (int u = 0; u < 4 * kRowBlock; ++u)
          q[u] = RR[4 * (r * kW + k0) + u];
        uint64_t amb = 0;
#pragma unroll
        for (int v = 0; v < kRowBlock; ++v) {
          const float d0 = q[4 * v] - fx, d1 = q[4 * v + 1] - fy,
                      d2 = q[4 * v + 2] - fz;
          const float d = __builtin_fmaf(
              d2, d2, __builtin_fmaf(d1, d1, d0 * d0));
          // (the median with infinity: a maximum without the second
          // instruction that quiets the loaded operand)
          const float u =
              d - (GATHER ? q[4 * v + 3]
                          : __builtin_amdgcn_fmed3f(q[4 * v + 3], fh2, inf));
          const uint64_t m = __ballot(u <= -tau);
          amb |= __ballot(!(fabsf(u) >= tau));
          lo[r] = (uint32_t)write_lane((int)(uint32_t)m, k0 + v, (int)lo[r]);
          hi[r] = (uint32_t)write_lane((int)(uint32_t)(m >> 32), k0 + v,
                                       (int)hi[r]);
        }
        if (amb & ~far) {
          const int k1 = min(k0 + kRowBlock, nrow);
          for (int k = k0; k < k1; ++k) {
            const int kr = r * kW + k;
            const double qh2 = ph2[kr];
            const double e0 = X[kr] - cx, e1 = Y[kr] - cy, e2 = Z[kr] - cz;
            const double e = e0 * e0 + e1 * e1 + e2 * e2;
            // tree_topology.h:372-379: d^2 <= max(h_k, h_b)^2
            const uint64_t m =
                (GATHER ? __ballot(e < qh2)
                        : __ballot(e <= qh2) | __ballot(e <= ch2)) & ~far;
            lo[r] = (uint32_t)write_lane((int)(uint32_t)m, k, (int)lo[r]);
            hi[r] = (uint32_t)write_lane((int)(uint32_t)(m >> 32), k,
                                         (int)hi[r]);
          }
        }
      }
      if (lane >= nrow) lo[r] = hi[r] = 0;
      cnt[r] += __popc(lo[r]) + __popc(hi[r]);
    }
    uint32_t v0 = lo[0], v1 = hi[0];
    if (NR == 2) {
      v0 |= lo[NR - 1];
      v1 |= hi[NR - 1];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      v0 |= __shfl_xor(v0, o, 64);
      v1 |= __shfl_xor(v1, o, 64);
    }
    const uint32_t u0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)v0);
    const uint32_t u1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)v1);
    const uint64_t used = (uint64_t)u1 << 32 | u0;
    if (used) {
      const int n0 = __popc(u0), n1 = __popc(u1);
      const Compress c0 = compress_masks(u0), c1 = compress_masks(u1);
      if (used >> lane & 1ull)
        a.cand[cout + used_so_far +
               __popcll(used & ((1ull << lane) - 1ull))] = ccur;
      // each row's bits at the used positions, appended after the bits of
      // the earlier rounds (the same positions for every row of the tile)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const int k = lane + r * kW;
        if (k >= gc) continue;
        uint64_t acc = pend[r];
        int nbl = nb, wil = wi;
        auto put = [&](uint32_t bits, int n) {
          acc |= (uint64_t)bits << nbl;
          nbl += n;
          if (nbl >= 32) {
            a.mask[mout + (int64_t)wil * gc + k] = (uint32_t)acc;
            acc >>= 32;
            nbl -= 32;
            ++wil;
          }
        };
        put(compress(lo[r], u0, c0), n0);
        put(compress(hi[r], u1, c1), n1);
        pend[r] = acc;
      }
      nb += n0 + n1;
      wi += nb >> 5;
      nb &= 31;
      used_so_far += n0 + n1;
    }
    ccur = cnext;
    cnext = cafter;
  }
  if (nb > 0)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int k = lane + r * kW;
      if (k < gc) a.mask[mout + (int64_t)wi * gc + k] = (uint32_t)pend[r];
    }
  if (lane == 0) {
    if (GATHER) {
      a.ccount[t] = (int32_t)used_so_far;
    } else {
      a.tcc[t] = (int32_t)used_so_far;
      a.tmo[t] = mout;
    }
  }
  if (a.nngb)
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (lane + r * kW < gc) a.nngb[gs + r * kW + lane] = cnt[r];
}

struct TileBufs {
  DBuf &cand, &ccount, &moff, &mask;
  int64_t &ccap, &words;
};

// SPH mode: the traversal and the masks run per group (the group decides
// the candidates, tree_topology.h:213-442) and the masks kernel writes the
// group's tiles.  Gather mode: the predicate involves only the particle's
// own radius, so the units are the tiles themselves (nt of them, or the ngl
// listed in glist).
int build_tiles(Ctx *c, TileBufs tb, bool gather, double scale,
                int32_t *nngb, const float *hprop, const int32_t *glist,
                int64_t ngl) {
  const int64_t nu = glist ? ngl : (gather ? c->nt : c->ng);
  if (nu <= 0) return 0;
  const int32_t *ustart = gather ? c->tstart.as<int32_t>()
                                 : c->gstart.as<int32_t>();
  const int32_t *ucount = gather ? c->tcount.as<int32_t>()
                                 : c->gcount.as<int32_t>();
  // candidate slots: one per unit, plus two per split group
  const int64_t nslots = nu + (gather ? 0 : 2 * c->nsplit);
  // rows of the largest unit (sizes the kernels' LDS arrays)
  const bool u64 = (gather ? c->tiles_w : c->groups_max) <= kW;
  FSPH_TRY(ensure(c, tb.ccount, (size_t)nu * 4));
  FSPH_TRY(ensure(c, tb.moff, (size_t)(nu + 1) * 8));
  FSPH_TRY(ensure(c, c->rowrel, (size_t)(c->pcap + kW) * sizeof(float4)));
  for (int attempt = 0;; ++attempt) {
    FSPH_TRY(ensure(c, tb.cand, (size_t)nslots * tb.ccap * 4));
    // (update_iteration has cleared the flags for the SPH tiles' first try)
    if (gather || attempt)
      FSPH_HIP(c, hipMemsetAsync(c->flags.p, 0, sizeof(int), c->stream));
    TravArgs t{c->f[PF_X].as<double>(), c->f[PF_Y].as<double>(),
               c->f[PF_Z].as<double>(), c->f[PF_H].as<double>(),
               c->nbox.as<double>(),    c->ncom.as<double>(),
               c->nrad.as<double>(),    c->nchild.as<int32_t>(),
               ustart,                  ucount,
               gather ? nullptr : c->gnode.as<int32_t>(),
               tb.cand.as<int32_t>(),
               tb.ccount.as<int32_t>(), tb.ccap,
               c->flags.as<int>(),      scale,
               hprop,                   glist,
               c->batch.n_inst ? c->f[PF_INST].as<int32_t>() : nullptr,
               c->batch.n_inst ? c->batch.root.as<int32_t>() : nullptr,
               c->rowrel.as<float4>(),  tb.moff.as<int64_t>()};
    {
      PhaseTimer tm(c, gather ? FSPH_T_H : FSPH_T_TRAVERSE);
      const int tier = c->stack_tier[gather ? 1 : 0];
      auto go = [&](auto gf) {
        constexpr bool GF = decltype(gf)::value;
        auto run = [&](auto stack) {
          constexpr int S = decltype(stack)::value;
          if (u64)
            k_traverse<S, kW, GF><<<(unsigned)nu, kW, 0, c->stream>>>(t);
          else
            k_traverse<S, kMaxGroup, GF>
                <<<(unsigned)nu, kW, 0, c->stream>>>(t);
        };
        if (tier >= 2)
          run(std::integral_constant<int, kStackLarge>{});
        else if (tier == 1)
          run(std::integral_constant<int, kStackMid>{});
        else
          run(std::integral_constant<int, kStackSmall>{});
      };
      if (gather)
        go(std::true_type{});
      else
        go(std::false_type{});
    }
    FSPH_HIP(c, hipGetLastError());
    // mask offsets, then the flags and the word count in one read-back
    FSPH_TRY(scan_i64(c, tb.moff.as<int64_t>(), tb.moff.as<int64_t>(), nu));
    k_tile_mail<<<1, 64, 0, c->stream>>>(c->flags.as<int>(),
                                         tb.moff.as<int64_t>() + nu,
                                         c->mail_d);
    FSPH_TRY(read_mail(c));
    const int fl = (int)c->mail_h[0];
    if (fl & kFlagScanStall)
      return fail(c, FSPH_E_HIP, "scan: a tile's look-back did not complete");
    if (fl & kFlagStack) {
      int &tier = c->stack_tier[gather ? 1 : 0];
      if (tier >= 2)
        return fail(c, FSPH_E_CAP, "neighbour traversal stack overflow");
      ++tier;
      continue;
    }
    if (fl & kFlagCand) {
      if (attempt >= 6)
        return fail(c, FSPH_E_CAP, "candidate tile overflow (cap %lld)",
                    (long long)tb.ccap);
      tb.ccap *= 2;
      continue;
    }
    break;
  }
  const int64_t words = c->mail_h[1];
  tb.words = words;
  FSPH_TRY(ensure(c, tb.mask, (size_t)(words > 0 ? words : 1) * 4));
  const bool tiled = !gather;
  if (tiled) {
    FSPH_TRY(ensure(c, c->tccount, (size_t)c->nt * 4));
    FSPH_TRY(ensure(c, c->tmoff, (size_t)c->nt * 8));
  }
  MaskArgs m{c->f[PF_X].as<double>(), c->f[PF_Y].as<double>(),
             c->f[PF_Z].as<double>(), c->f[PF_H].as<double>(),
             c->ncom.as<double>(),    c->nrad.as<double>(),
             c->nlap.as<double>(),    ustart,
             ucount,                  gather ? nullptr : c->gnode.as<int32_t>(),
             tb.cand.as<int32_t>(),   tb.ccount.as<int32_t>(),
             tb.moff.as<int64_t>(),   tb.ccap,
             tb.mask.as<uint32_t>(),  nngb,
             scale,                   hprop,
             glist,
             tiled ? c->tgrp.as<int32_t>() : nullptr,
             c->tstart.as<int32_t>(), c->tcount.as<int32_t>(),
             tiled ? c->tslot.as<int32_t>() : nullptr,
             tiled ? c->tccount.as<int32_t>() : nullptr,
             tiled ? c->tmoff.as<int64_t>() : nullptr,
             c->rowrel.as<float4>()};
  {
    PhaseTimer tm(c, gather ? FSPH_T_H : FSPH_T_MASKS);
    // rows of the widest tile: one or two per lane
    const unsigned nw = (unsigned)(gather ? nu : c->nt);
    if (gather && u64)
      k_masks<true, 1><<<nw, kW, 0, c->stream>>>(m);
    else if (gather)
      k_masks<true, 2><<<nw, kW, 0, c->stream>>>(m);
    else if (c->tiles_w <= kW)
      k_masks<false, 1><<<nw, kW, 0, c->stream>>>(m);
    else
      k_masks<false, 2><<<nw, kW, 0, c->stream>>>(m);
  }
  return hip_check(c, hipGetLastError(), "k_masks");
}

}  // namespace

int stage_neighbors(Ctx *c) {
  TileBufs tb{c->cand, c->ccount, c->moff, c->mask, c->ccap, c->mask_words};
  return build_tiles(c, tb, false, 1.0, c->f[PF_NNGB].as<int32_t>(), nullptr,
                     nullptr, -1);
}

int stage_gather_tiles(Ctx *c, double scale, const float *hprop,
                       const int32_t *glist, int64_t ngl) {
  TileBufs tb{c->gcand, c->gccount, c->gmoff, c->gmask, c->gccap,
              c->gmask_words};
  return build_tiles(c, tb, true, scale, nullptr, hprop, glist, ngl);
}

}  // namespace fsph
