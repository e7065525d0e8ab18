// Contact-resolved velocity pass on the device
// (self_collision_cloth.cpp:355-456, bvh_aabb.cpp).
//
//  refit      the leaves, then one launch per tree depth, bottom-up.
//  traverse   one wave walks the BVH in pre-order for a group of leaves
//             (stackless, the subtree end of every node is its skip link) and
//             lists every later leaf whose box overlaps: exactly the leaf
//             pairs the reference's recursion visits, oriented the same way
//             (the leaf under the LCA's child 0 first).
//  narrow     the 6 face-vertex and 9 edge-edge tests of each pair, numbered
//             in the reference's order: the tests that a pair needs are listed,
//             then run one per thread, and a block's records are appended at
//             one place.
//  select     records are radix-sorted by canonical key; for a key found as
//             both face-vertex and edge-edge the visit that comes first in the
//             reference's depth-first order wins (std::set keeps the first
//             insertion, bvh_aabb.h:96-102).
//  impulses   Gauss-Seidel in key order, scheduled in rounds: a contact runs
//             once every earlier contact sharing a vertex has run, so each
//             velocity sees exactly the updates it sees sequentially.  What
//             does not depend on velocities (a proximity contact's distance
//             and weights) is formed for all contacts at once before.
//  zones      rigid impact zones by union-find in one workgroup, zone sums in
//             ascending vertex order.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>

#include "cs_contact.hpp"
#include "cs_math.hpp"
#include "cs_solve.hpp"

namespace cs {

namespace {
constexpr int kTB = 256;
inline unsigned grid_for(long n, int tb = kTB) { return (unsigned)((n + tb - 1) / tb); }
enum Counter : int {
  kRaw = 0,       // narrow-phase records emitted
  kGroups = 1,    // distinct contacts
  kDoneCnt = 2,   // contacts whose impulse has run
  kCand = 3,      // overlapping leaf pairs found by the traversal
  kReady = 4,     // contacts with no earlier contact on their vertices
  kQueryCounters = 8,  // a query clears counters [0, kQueryCounters)
  kZoneVerts = 8, // vertices in impact zones after the last zone pass
  kNumCounters = 16
};
}  // namespace

__device__ __forceinline__ Box load_box(const double* bb, int n) {
  Box b;
  b.lx = bb[6 * n + 0];
  b.hx = bb[6 * n + 1];
  b.ly = bb[6 * n + 2];
  b.hy = bb[6 * n + 3];
  b.lz = bb[6 * n + 4];
  b.hz = bb[6 * n + 5];
  return b;
}
__device__ __forceinline__ void store_box(double* bb, int n, const Box& b) {
  bb[6 * n + 0] = b.lx;
  bb[6 * n + 1] = b.hx;
  bb[6 * n + 2] = b.ly;
  bb[6 * n + 3] = b.hy;
  bb[6 * n + 4] = b.lz;
  bb[6 * n + 5] = b.hz;
}

// ---------------------------------------------------------------------------
// refit (bvh_aabb.cpp:23-106)

// Leaf boxes from their triangles; the internal nodes follow level by level
// (k_refit_merge), deepest first.  A box merge is a componentwise min / max,
// exact in any order, so the boxes are the reference's.
__global__ void k_refit_leaves(DevCloth c, const double* X, const double* U, double delta,
                               double dt, int ccd) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= c.nt) return;
  const int i0 = c.tri[3 * t], i1 = c.tri[3 * t + 1], i2 = c.tri[3 * t + 2];
  Box b;
  if (ccd) {
    const double eps = 1.0e-10;
    b = box_point(at(X, i0), eps);
    box_grow(b, at(X, i1), eps);
    box_grow(b, at(X, i2), eps);
    box_grow(b, advanced(X, U, dt, i0), eps);
    box_grow(b, advanced(X, U, dt, i1), eps);
    box_grow(b, advanced(X, U, dt, i2), eps);
  } else {
    const double eps = delta * 0.5;
    b = box_point(at(X, i0), eps);
    box_grow(b, at(X, i1), eps);
    box_grow(b, at(X, i2), eps);
  }
  const int L = c.leaf_of[t];
  store_box(c.bb, L, b);
  store_box(c.rbb, c.pre[L], b);
}

// the internal nodes among refit_order[b .. e) (one depth): box = merge of
// the children's boxes, written by earlier launches
__global__ void k_refit_merge(DevCloth c, int b, int e) {
  const int k = b + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (k >= e) return;
  const int n = c.refit_order[k];
  if (c.node[3 * n + 2] == -1) return;  // a leaf: boxed from its triangle
  const Box m = box_merge(load_box(c.bb, c.node[3 * n + 1]), load_box(c.bb, c.node[3 * n + 2]));
  store_box(c.bb, n, m);
  store_box(c.rbb, c.pre[n], m);
}

// ---------------------------------------------------------------------------
// narrow phase

// canonical key of a contact element (bvh_aabb.h:68-95): a face-vertex key
// lists the face ascending then the vertex; an edge-edge key starts with the
// edge holding the smallest index, each edge ascending
__device__ __forceinline__ void canonical(bool fv, int j0, int j1, int j2, int j3, int k[4]) {
  if (fv) {
    int a = j0, b = j1, d = j2, t;
    if (a > b) { t = a; a = b; b = t; }
    if (b > d) { t = b; b = d; d = t; }
    if (a > b) { t = a; a = b; b = t; }
    k[0] = a;
    k[1] = b;
    k[2] = d;
    k[3] = j3;
  } else {
    const int a0 = min(j0, j1), a1 = max(j0, j1), b0 = min(j2, j3), b1 = max(j2, j3);
    if (a0 < b0) {
      k[0] = a0; k[1] = a1; k[2] = b0; k[3] = b1;
    } else {
      k[0] = b0; k[1] = b1; k[2] = a0; k[3] = a1;
    }
  }
}

struct Emit {
  int* counters;
  int cap;
  int* rkey;
  int* rinfo;
  int* rpair;
  __device__ void operator()(int slot, bool fv, int test, int first, int second, int j0, int j1,
                             int j2, int j3) const {
    int k[4];
    canonical(fv, j0, j1, j2, j3, k);
    rkey[4 * slot + 0] = k[0];
    rkey[4 * slot + 1] = k[1];
    rkey[4 * slot + 2] = k[2];
    rkey[4 * slot + 3] = k[3];
    rinfo[slot] = (fv ? 1 : 0) | (test << 1);
    rpair[2 * slot] = first;
    rpair[2 * slot + 1] = second;
  }
};

// Leaf-leaf tests of overlapping leaf pairs: face-vertex 0..5 then edge-edge
// 6..14 (bvh_aabb.cpp:475-536 proximity, 833-900 continuous).
//
// A block takes kTB pairs.  First every thread forms, for its pair, which of
// the fifteen tests pass their own first conditions (a shared vertex, boxes
// apart: cheap and the same on every lane) and lists those in LDS, face tests
// from the front and edge tests from the back; then the block's threads take
// the listed tests one each (one thread per pair running its tests in turn
// executed the long part of each test for almost every wave) and list the
// hits, whose records go out behind one atomic of the block on the global
// counter: an atomic per record cost about 22 ns each, which was nearly all of
// the kernel (397 000 records of a 253 x 397 drop: 8.8 ms, now 1.6; 57 000
// of a folded 176^2 sheet: 1.05 ms, now 0.22).
constexpr int kNarrowTests = 15;

// vertices of one test of the leaf pair (L, M): a face of one leaf and a
// vertex of the other, or an edge of each
struct NarrowTest {
  int i[4];
  int face;  // leaf node of the face
  int face_tri;
};
__device__ __forceinline__ NarrowTest narrow_test(const DevCloth& c, int test, int L, int M) {
  const int it = c.node[3 * L + 1], jt = c.node[3 * M + 1];
  NarrowTest t;
  if (test < 6) {
    const int ft = test < 3 ? it : jt, vt = test < 3 ? jt : it;
    t.face = test < 3 ? L : M;
    t.face_tri = ft;
    t.i[0] = c.tri[3 * ft];
    t.i[1] = c.tri[3 * ft + 1];
    t.i[2] = c.tri[3 * ft + 2];
    t.i[3] = c.tri[3 * vt + (test < 3 ? test : test - 3)];
  } else {
    const int a = (test - 6) / 3, b = (test - 6) - 3 * a;
    t.face = t.face_tri = 0;
    t.i[0] = c.tri[3 * it + a];
    t.i[1] = c.tri[3 * it + (a == 2 ? 0 : a + 1)];
    t.i[2] = c.tri[3 * jt + b];
    t.i[3] = c.tri[3 * jt + (b == 2 ? 0 : b + 1)];
  }
  return t;
}

// the tests of a pair that get past their first conditions (each exactly the
// ones that fv_near, ee_near, fv_sweep and ee_sweep begin with)
template <bool kCcd>
__device__ __forceinline__ unsigned narrow_mask(const DevCloth& c, const double* X,
                                                const double* U, double dt, double delta, int L,
                                                int M) {
  const int it = c.node[3 * L + 1], jt = c.node[3 * M + 1];
  const int iv[3] = {c.tri[3 * it], c.tri[3 * it + 1], c.tri[3 * it + 2]};
  const int jv[3] = {c.tri[3 * jt], c.tri[3 * jt + 1], c.tri[3 * jt + 2]};
  Vec3 P[3], Q[3], Pe[3], Qe[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    P[a] = at(X, iv[a]);
    Q[a] = at(X, jv[a]);
    if (kCcd) {
      Pe[a] = advanced(X, U, dt, iv[a]);
      Qe[a] = advanced(X, U, dt, jv[a]);
    }
  }
  // the proximity face tests read the box of the node whose id equals the
  // triangle id (bvh_aabb.cpp:490-507)
  const Box bi = load_box(c.bb, kCcd ? L : it), bj = load_box(c.bb, kCcd ? M : jt);
  const double eps = 1.0e-10;
  unsigned mask = 0;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const bool di = jv[a] != iv[0] && jv[a] != iv[1] && jv[a] != iv[2];
    const bool dj = iv[a] != jv[0] && iv[a] != jv[1] && iv[a] != jv[2];
    if (kCcd) {
      Box q = box_point(Q[a], eps), p = box_point(P[a], eps);
      box_grow(q, Qe[a], eps);
      box_grow(p, Pe[a], eps);
      mask |= di && overlap(bi, q) ? 1u << a : 0u;
      mask |= dj && overlap(bj, p) ? 8u << a : 0u;
    } else {
      mask |= di && inside(bi, Q[a]) ? 1u << a : 0u;
      mask |= dj && inside(bj, P[a]) ? 8u << a : 0u;
    }
  }
  if (kCcd) {
    Box ep[3], eq[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int a1 = a == 2 ? 0 : a + 1;
      ep[a] = box_point(P[a], eps);
      box_grow(ep[a], P[a1], eps);
      box_grow(ep[a], Pe[a], eps);
      box_grow(ep[a], Pe[a1], eps);
      eq[a] = box_point(Q[a], eps);
      box_grow(eq[a], Q[a1], eps);
      box_grow(eq[a], Qe[a], eps);
      box_grow(eq[a], Qe[a1], eps);
    }
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const int i0 = iv[a], i1 = iv[a == 2 ? 0 : a + 1], j0 = jv[b], j1 = jv[b == 2 ? 0 : b + 1];
        const bool far = i0 == j0 || i0 == j1 || i1 == j0 || i1 == j1 || !overlap(ep[a], eq[b]);
        mask |= far ? 0u : 64u << (3 * a + b);
      }
  } else {
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const int a1 = a == 2 ? 0 : a + 1, b1 = b == 2 ? 0 : b + 1;
        const int i0 = iv[a], i1 = iv[a1], j0 = jv[b], j1 = jv[b1];
        const bool far = i0 == j0 || i0 == j1 || i1 == j0 || i1 == j1 ||
                         ee_apart(P[a], P[a1], Q[b], Q[b1], delta);
        mask |= far ? 0u : 64u << (3 * a + b);
      }
  }
  return mask;
}

// n overlapping leaf pairs (n <= the buffer's capacity)
template <bool kCcd>
__global__ __launch_bounds__(kTB) void k_narrow(DevCloth c, const double* X, const double* U,
                                                double dt, double delta, int n, const int* cand,
                                                Emit emit) {
  constexpr int kEnd = kTB * kNarrowTests;
  // entries: pair of the block << 4 | test
  __shared__ unsigned short list[kEnd];
  __shared__ unsigned short hits[kEnd];
  __shared__ int nfv, nee, nhit, base;
  const int tid = threadIdx.x, p0 = blockIdx.x * kTB;
  if (tid == 0) nfv = nee = nhit = 0;
  __syncthreads();
  unsigned mask = 0;
  if (p0 + tid < n)
    mask = narrow_mask<kCcd>(c, X, U, dt, delta, cand[2 * (p0 + tid)], cand[2 * (p0 + tid) + 1]);
  if (mask & 63u) {
    int at = atomicAdd(&nfv, __popc(mask & 63u));
    for (unsigned m = mask & 63u; m; m &= m - 1)
      list[at++] = (unsigned short)(tid << 4 | (__ffs((int)m) - 1));
  }
  if (mask >> 6) {
    int at = kEnd - 1 - atomicAdd(&nee, __popc(mask >> 6));
    for (unsigned m = mask >> 6; m; m &= m - 1)
      list[at--] = (unsigned short)(tid << 4 | (__ffs((int)m) + 5));
  }
  __syncthreads();
  const int tests_fv = nfv, tests_ee = nee;
  for (int q = tid; q < tests_fv; q += kTB) {
    const int e = list[q], test = e & 15;
    const NarrowTest t = narrow_test(c, test, cand[2 * (p0 + (e >> 4))], cand[2 * (p0 + (e >> 4)) + 1]);
    const Box b = load_box(c.bb, kCcd ? t.face : t.face_tri);
    const Vec3 a0 = at(X, t.i[0]), a1 = at(X, t.i[1]), a2 = at(X, t.i[2]), a3 = at(X, t.i[3]);
    bool hit;
    if (kCcd)
      hit = fv_sweep(t.i[0], t.i[1], t.i[2], t.i[3], a0, a1, a2, a3, advanced(X, U, dt, t.i[0]),
                     advanced(X, U, dt, t.i[1]), advanced(X, U, dt, t.i[2]),
                     advanced(X, U, dt, t.i[3]), b);
    else
      hit = fv_near(t.i[0], t.i[1], t.i[2], t.i[3], a0, a1, a2, a3, b, delta);
    if (hit) hits[atomicAdd(&nhit, 1)] = (unsigned short)e;
  }
  for (int q = tid; q < tests_ee; q += kTB) {
    const int e = list[kEnd - 1 - q], test = e & 15;
    const NarrowTest t = narrow_test(c, test, cand[2 * (p0 + (e >> 4))], cand[2 * (p0 + (e >> 4)) + 1]);
    const Vec3 p = at(X, t.i[0]), p1 = at(X, t.i[1]), r = at(X, t.i[2]), r1 = at(X, t.i[3]);
    bool hit;
    if (kCcd)
      hit = ee_sweep(t.i[0], t.i[1], t.i[2], t.i[3], p, p1, r, r1, advanced(X, U, dt, t.i[0]),
                     advanced(X, U, dt, t.i[1]), advanced(X, U, dt, t.i[2]),
                     advanced(X, U, dt, t.i[3]));
    else
      hit = ee_near(t.i[0], t.i[1], t.i[2], t.i[3], p, p1, r, r1, delta);
    if (hit) hits[atomicAdd(&nhit, 1)] = (unsigned short)e;
  }
  __syncthreads();
  const int total = nhit;
  if (total == 0) return;
  if (tid == 0) base = atomicAdd(&emit.counters[kRaw], total);
  __syncthreads();
  for (int q = tid; q < total && base + q < emit.cap; q += kTB) {
    const int e = hits[q], test = e & 15;
    const int L = cand[2 * (p0 + (e >> 4))], M = cand[2 * (p0 + (e >> 4)) + 1];
    const NarrowTest t = narrow_test(c, test, L, M);
    emit(base + q, test < 6, test, L, M, t.i[0], t.i[1], t.i[2], t.i[3]);
  }
}

// Overlapping leaf pairs (L, M), M after L in pre-order, as the reference's
// pair recursion finds them (bvh_aabb.cpp:461-474, 544-556): the records are
// sorted by key afterwards and k_select orders visits by the tree alone, so
// the order in which pairs are found does not matter.
//
// One wave per 64 consecutive leaves in pre-order.  Each lane's own walk is a
// pre-order scan from the root that skips a subtree (jumps to its end) when
// it holds no leaf after the lane's leaf or its box does not overlap the
// leaf's box, and records every leaf it reaches after its own.  The wave walks
// the union of its lanes' walks: at rank r a lane takes part iff r is at or
// past the end of the last subtree it skipped, so every lane tests exactly
// the nodes its own walk tests; the wave goes on to r + 1 if any lane
// descends, else to the end of r's subtree, the first rank at which any lane
// takes part again.  The node data are read by wave-uniform rank (scalar
// loads of rend / rbb / by_pre), the leaf's box stays in registers, and the
// pairs go through an LDS buffer, one counter atomic per kTravBuf pairs.
constexpr int kTravBuf = 512;

// overlap() evaluated without short-circuit branches (each comparison as
// written there, so NaN coordinates behave the same), which keeps all six
// bounds of a box in one round of loads
__device__ __forceinline__ bool overlap_all(const Box& a, const Box& b) {
  return !(a.hx < b.lx) & !(a.lx > b.hx) & !(a.hy < b.ly) & !(a.ly > b.hy) & !(a.hz < b.lz) &
         !(a.lz > b.hz);
}

__device__ __forceinline__ void trav_flush(const int2* buf, int fill, int* __restrict__ counters,
                                           int cap, int2* __restrict__ cand) {
  __syncthreads();  // the buffer's entries, written by every lane
  int base = 0;
  if (threadIdx.x == 0) base = atomicAdd(&counters[kCand], fill);
  base = __shfl(base, 0);
  for (int i = (int)threadIdx.x; i < fill; i += 64)
    if (base + i < cap) cand[base + i] = buf[i];
  __syncthreads();  // read out before the buffer is reused
}

__global__ __launch_bounds__(64) void k_traverse(int nnode, int nt, int per,
                                                 const int* __restrict__ leaf_rank,
                                                 const int* __restrict__ rend,
                                                 const double* __restrict__ rbb,
                                                 const int* __restrict__ by_pre,
                                                 int* __restrict__ counters, int cap,
                                                 int2* __restrict__ cand) {
  __shared__ int2 buf[kTravBuf];
  // per (1..64) leaves per wave: fewer leaves make shorter union walks and
  // more waves, which pays where the tree is small and few waves would run
  const int k = (int)(blockIdx.x * per + threadIdx.x);
  int rl = 0, L = -1, skip = INT_MAX;  // lanes past the last leaf never take part
  Box bl{};
  if ((int)threadIdx.x < per && k < nt) {
    rl = leaf_rank[k];
    L = by_pre[rl];
    bl = load_box(rbb, rl);
    skip = 0;
  }
  int fill = 0;
  int r = 0;
  while (r < nnode) {
    // all three loads issue together (no branch between them and their use)
    const int end = rend[r];
    const Box b = load_box(rbb, r);
    const int m = by_pre[r];
    const bool alive = r >= skip;
    const bool down = alive & (end > rl + 1) & overlap_all(bl, b);
    const bool hit = down & (end == r + 1) & (r > rl);
    skip = (alive & !down) ? end : skip;
    const unsigned long long hm = __ballot(hit);
    if (hm) {
      const int cnt = __popcll(hm);
      if (fill + cnt > kTravBuf) {
        trav_flush(buf, fill, counters, cap, cand);
        fill = 0;
      }
      if (hit) {
        const int below = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(hm >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((unsigned)hm, 0u));
        buf[fill + below] = make_int2(L, m);
      }
      fill += cnt;
    }
    r = __ballot(down) ? r + 1 : end;
  }
  if (fill) trav_flush(buf, fill, counters, cap, cand);
}

// ---------------------------------------------------------------------------
// selection: sort by key, then per key the first visit in depth-first order

__global__ void k_make_keys(const int* rkey, int n, int nbits, int pass, uint64_t* key, int* idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t k0 = (uint64_t)rkey[4 * i], k1 = (uint64_t)rkey[4 * i + 1];
  const uint64_t k2 = (uint64_t)rkey[4 * i + 2], k3 = (uint64_t)rkey[4 * i + 3];
  uint64_t k;
  if (pass == 0)  // whole key fits in 64 bits
    k = (((k0 << nbits | k1) << nbits | k2) << nbits) | k3;
  else if (pass == 1)  // least significant part of a two-pass sort
    k = k3;
  else
    k = ((k0 << nbits | k1) << nbits) | k2;
  key[i] = k;
  if (pass != 2) idx[i] = i;
}

__global__ void k_rekey(const int* rkey, const int* order, int n, int nbits, uint64_t* key) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int r = order[i];
  const uint64_t k0 = (uint64_t)rkey[4 * r], k1 = (uint64_t)rkey[4 * r + 1];
  const uint64_t k2 = (uint64_t)rkey[4 * r + 2];
  key[i] = ((k0 << nbits | k1) << nbits) | k2;
}

__device__ __forceinline__ bool same_key(const int* rkey, int a, int b) {
  return rkey[4 * a] == rkey[4 * b] && rkey[4 * a + 1] == rkey[4 * b + 1] &&
         rkey[4 * a + 2] == rkey[4 * b + 2] && rkey[4 * a + 3] == rkey[4 * b + 3];
}

__global__ void k_heads(const int* rkey, const int* order, int n, int* head) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  head[i] = (i == 0 || !same_key(rkey, order[i], order[i - 1])) ? 1 : 0;
}

__device__ __forceinline__ bool in_subtree(const DevCloth& c, int n, int leaf) {
  const int r = c.pre[leaf];
  return c.pre[n] <= r && r < c.pre_end[n];
}

// Does visit (L0, M0, test t0) come before (L1, M1, t1) in the reference's
// traversal?  self(N) visits the pairs whose LCA is N before those of its
// subtrees (LCAs in pre-order); within one LCA the pair recursion descends
// both sides at once and orders children pairs (00, 10, 01, 11)
// (bvh_aabb.cpp:461-474, 550-556).
__device__ bool visited_before(const DevCloth& c, int L0, int M0, int t0, int L1, int M1, int t1) {
  if (L0 == L1 && M0 == M1) return t0 < t1;
  int A0 = L0;
  while (!in_subtree(c, A0, M0)) A0 = c.node[3 * A0];
  int A1 = L1;
  while (!in_subtree(c, A1, M1)) A1 = c.node[3 * A1];
  if (A0 != A1) return c.pre[A0] < c.pre[A1];
  int X = c.node[3 * A0 + 1], Y = c.node[3 * A0 + 2];
  for (int guard = 0; guard < 4 * c.nnode; guard++) {
    const bool lx = c.node[3 * X + 2] == -1, ly = c.node[3 * Y + 2] == -1;
    const int xb0 = lx ? 0 : (in_subtree(c, c.node[3 * X + 1], L0) ? 0 : 1);
    const int xb1 = lx ? 0 : (in_subtree(c, c.node[3 * X + 1], L1) ? 0 : 1);
    const int yb0 = ly ? 0 : (in_subtree(c, c.node[3 * Y + 1], M0) ? 0 : 1);
    const int yb1 = ly ? 0 : (in_subtree(c, c.node[3 * Y + 1], M1) ? 0 : 1);
    const int d0 = xb0 + 2 * yb0, d1 = xb1 + 2 * yb1;
    if (d0 != d1) return d0 < d1;
    if (lx && ly) return false;  // identical pairs (handled above)
    if (!lx) X = c.node[3 * X + 1 + xb0];
    if (!ly) Y = c.node[3 * Y + 1 + yb0];
  }
  return false;
}

__global__ void k_select(DevCloth c, const int* rkey, const int* rinfo, const int* rpair,
                         const int* order, const int* head, const int* gpos, int n, int* ce,
                         int* counters) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (i == n - 1) counters[kGroups] = gpos[i] + head[i];
  if (!head[i]) return;
  int e = i + 1;
  while (e < n && !head[e]) e++;
  int w = order[i];
  bool mixed = false;
  for (int k = i + 1; k < e; k++) mixed |= ((rinfo[order[k]] ^ rinfo[w]) & 1) != 0;
  if (mixed) {
    for (int k = i + 1; k < e; k++) {
      const int r = order[k];
      if (visited_before(c, rpair[2 * r], rpair[2 * r + 1], rinfo[r] >> 1, rpair[2 * w],
                         rpair[2 * w + 1], rinfo[w] >> 1))
        w = r;
    }
  }
  const int g = gpos[i];
  ce[5 * g] = rinfo[w] & 1;
  for (int q = 0; q < 4; q++) ce[5 * g + 1 + q] = rkey[4 * w + q];
}

// ---------------------------------------------------------------------------
// impulses (self_collision_cloth.cpp:20-212)

__device__ __forceinline__ void vel_add(double* U, int i, double a, double b, double d) {
  U[3 * i] += a;
  U[3 * i + 1] += b;
  U[3 * i + 2] += d;
}

// the impulse of a continuous contact
__device__ void impulse_ccd(const int* e, const double* X, double* U, double delta, double dt,
                            double m) {
  const int i0 = e[1], i1 = e[2], i2 = e[3], i3 = e[4];
  const Vec3 p0 = at(X, i0), p1 = at(X, i1), p2 = at(X, i2), p3 = at(X, i3);
  const Vec3 v0 = at(U, i0), v1 = at(U, i1), v2 = at(U, i2), v3 = at(U, i3);
  // end positions are p + v, not p + dt v (self_collision_cloth.cpp:141)
  const double t = coplanar_time(p0, p1, p2, p3, p0 + v0, p1 + v1, p2 + v2, p3 + v3);
  if (t < 0 || t > 1) return;
  if (e[0]) {  // face (i0,i1,i2) - vertex i3
    double w0, w1;
    {
      const double dist =
          face_vertex(p0 + t * v0, p1 + t * v1, p2 + t * v2, p3 + t * v3, w0, w1);
      if (w0 < 0 || w0 > 1) return;
      if (w1 < 0 || w1 > 1) return;
      if (dist > delta) return;
    }
    const double w2 = 1.0 - w0 - w1;
    const Vec3 pc = w0 * p0 + w1 * p1 + w2 * p2;
    const Vec3 nrm = unit(p3 - pc);
    const double rel = dot(v3 - w0 * v0 - w1 * v1 - w2 * v2, nrm);
    if (rel > 0.1 * delta / dt) return;
    const double imp = m * (0.1 * delta / dt - rel);
    double j = 2 * imp / (1.0 + w0 * w0 + w1 * w1 + w2 * w2);
    j /= m;
    j *= 0.1;
    vel_add(U, i0, -nrm.x * j * w0, -nrm.y * j * w0, -nrm.z * j * w0);
    vel_add(U, i1, -nrm.x * j * w1, -nrm.y * j * w1, -nrm.z * j * w1);
    vel_add(U, i2, -nrm.x * j * w2, -nrm.y * j * w2, -nrm.z * j * w2);
    vel_add(U, i3, +nrm.x * j, +nrm.y * j, +nrm.z * j);
  } else {  // edge (i0,i1) - edge (i2,i3)
    double wa, wb;
    {
      const double dist = edge_edge(p0 + t * v0, p1 + t * v1, p2 + t * v2, p3 + t * v3, wa, wb);
      if (wa < 0 || wa > 1) return;
      if (wb < 0 || wb > 1) return;
      if (dist > delta) return;
    }
    const Vec3 ca = (1 - wa) * p0 + wa * p1;
    const Vec3 cb = (1 - wb) * p2 + wb * p3;
    const Vec3 nrm = unit(cb - ca);
    const double rel = dot((1 - wb) * v2 + wb * v3 - (1 - wa) * v0 - wa * v1, nrm);
    if (rel > 0.1 * delta / dt) return;
    const double imp = m * (0.1 * delta / dt - rel);
    double j = 2 * imp / (wa * wa + (1 - wa) * (1 - wa) + wb * wb + (1 - wb) * (1 - wb));
    j /= m;
    j *= 0.1;
    vel_add(U, i0, -nrm.x * j * (1 - wa), -nrm.y * j * (1 - wa), -nrm.z * j * (1 - wa));
    vel_add(U, i1, -nrm.x * j * wa, -nrm.y * j * wa, -nrm.z * j * wa);
    vel_add(U, i2, +nrm.x * j * (1 - wb), +nrm.y * j * (1 - wb), +nrm.z * j * (1 - wb));
    vel_add(U, i3, +nrm.x * j * wb, +nrm.y * j * wb, +nrm.z * j * wb);
  }
}

// What a proximity impulse takes from the positions alone: formed for every
// contact at once before the sequential schedule, whose chain then holds only
// the velocities (in the continuous passes the time of impact depends on them:
// impulse_ccd).  One 128-byte line per contact.
struct alignas(128) ImpulseGeom {
  double c[4];     // weights of the four velocities (face-vertex: c[3] is 1)
  double n[3];     // contact normal
  double limit;    // 0.1 depth / dt
  double elastic;  // dt k depth
  double den;      // sum of the squared weights
  int v[4];        // vertices
  int kind;        // 0: no impulse, 1: face-vertex, 2: edge-edge
};

__global__ void k_impulse_geom(const int* ce, int g, const double* X, double delta, double k,
                               double dt, ImpulseGeom* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g) return;
  const int* e = ce + 5 * i;
  ImpulseGeom o;
  for (int a = 0; a < 4; a++) o.v[a] = e[1 + a];
  const Vec3 p0 = at(X, o.v[0]), p1 = at(X, o.v[1]), p2 = at(X, o.v[2]), p3 = at(X, o.v[3]);
  o.kind = 0;
  Vec3 nrm;
  double depth;
  if (e[0]) {
    double w0, w1;
    const double dist = face_vertex(p0, p1, p2, p3, w0, w1);
    if (!(w0 < 0 || w0 > 1) && !(w1 < 0 || w1 > 1) && !(dist > delta)) o.kind = 1;
    const double w2 = 1.0 - w0 - w1;
    const Vec3 pc = w0 * p0 + w1 * p1 + w2 * p2;
    nrm = unit(p3 - pc);
    depth = delta - dot(p3 - pc, nrm);
    o.c[0] = w0;
    o.c[1] = w1;
    o.c[2] = w2;
    o.c[3] = 1.0;
    o.den = 1 + w0 * w0 + w1 * w1 + w2 * w2;
  } else {
    double wa, wb;
    const double dist = edge_edge(p0, p1, p2, p3, wa, wb);
    if (!(wa < 0 || wa > 1) && !(wb < 0 || wb > 1) && !(dist > delta)) o.kind = 2;
    const Vec3 ca = (1 - wa) * p0 + wa * p1;
    const Vec3 cb = (1 - wb) * p2 + wb * p3;
    nrm = unit(cb - ca);
    depth = delta - norm(cb - ca);
    o.c[0] = 1 - wa;
    o.c[1] = wa;
    o.c[2] = 1 - wb;
    o.c[3] = wb;
    o.den = wa * wa + (1 - wa) * (1 - wa) + wb * wb + (1 - wb) * (1 - wb);
  }
  o.n[0] = nrm.x;
  o.n[1] = nrm.y;
  o.n[2] = nrm.z;
  o.limit = 0.1 * depth / dt;
  o.elastic = dt * k * depth;
  out[i] = o;
}

// the velocity part of a proximity impulse, the reference's operations in its
// order
__device__ __forceinline__ void impulse_velocity(const ImpulseGeom& o, Vec3 v0, Vec3 v1, Vec3 v2,
                                                 Vec3 v3, double* U, double m) {
  if (o.kind == 0) return;
  const Vec3 nrm = mk(o.n[0], o.n[1], o.n[2]);
  const double rel = o.kind == 1
                         ? dot(v3 - o.c[0] * v0 - o.c[1] * v1 - o.c[2] * v2, nrm)
                         : dot(o.c[2] * v2 + o.c[3] * v3 - o.c[0] * v0 - o.c[1] * v1, nrm);
  if (rel > o.limit) return;
  const double ie = m * (o.limit - rel);
  const double imin = (o.elastic < ie) ? o.elastic : ie;
  double j = 2 * imin / o.den;
  j /= m;
  j *= 0.25;
  // face-vertex: +n on the vertex, -n on the face; edge-edge: -n on the first
  // edge, +n on the second (a product with the weight 1 changes nothing)
  const double s2 = o.kind == 1 ? -1.0 : 1.0;
  auto put = [&](int v, const Vec3& u, double sx, double c) {
    U[3 * v] = u.x + sx * nrm.x * j * c;
    U[3 * v + 1] = u.y + sx * nrm.y * j * c;
    U[3 * v + 2] = u.z + sx * nrm.z * j * c;
  };
  put(o.v[0], v0, -1.0, o.c[0]);
  put(o.v[1], v1, -1.0, o.c[1]);
  put(o.v[2], v2, s2, o.c[2]);
  put(o.v[3], v3, 1.0, o.c[3]);
}

__global__ void k_inc_count(const int* ce, int g, int* vcount) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g) return;
  for (int a = 0; a < 4; a++) atomicAdd(&vcount[ce[5 * i + 1 + a]], 1);
}

__global__ void k_inc_fill(const int* ce, int g, const int* vstart, int* vfill, int* inc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g) return;
  for (int a = 0; a < 4; a++) {
    const int v = ce[5 * i + 1 + a];
    inc[vstart[v] + atomicAdd(&vfill[v], 1)] = 4 * i + a;
  }
}

// order each vertex's incidences by contact and link every incidence to the
// previous and the next contact on that vertex
__global__ void k_inc_link(int np, const int* vstart, int* inc, int* pred, int* succ) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= np) return;
  const int b = vstart[v], e = vstart[v + 1];
  for (int i = b + 1; i < e; i++) {
    const int x = inc[i];
    int j = i - 1;
    while (j >= b && inc[j] > x) {
      inc[j + 1] = inc[j];
      j--;
    }
    inc[j + 1] = x;
  }
  for (int i = b; i < e; i++) {
    pred[inc[i]] = (i == b) ? -1 : (inc[i - 1] >> 2);
    succ[inc[i]] = (i + 1 == e) ? -1 : (inc[i + 1] >> 2);
  }
}

// contacts with no earlier contact on their vertices start the schedule
__global__ void k_impulse_ready(int g, const int* pred, int* npred, int* ready, int* counters) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g) return;
  int c = 0;
  for (int a = 0; a < 4; a++) c += pred[4 * i + a] >= 0 ? 1 : 0;
  npred[i] = c;
  if (c == 0) ready[atomicAdd(&counters[kReady], 1)] = i;
}

// a workgroup barrier that orders LDS only: loads and stores stay in flight
__device__ __forceinline__ void lds_only_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Runs the ready contacts and every contact that becomes ready, round by
// round, in one workgroup: a contact is ready once every earlier contact on
// its vertices has run.  The contacts of a round share no vertex and each
// reads its vertices' velocities after every earlier contact on them has
// written them, so the velocities are those of the key-order Gauss-Seidel
// sweep.  Every contact enters a list once, so the loop ends after at most
// g contacts; the count of those run goes to counters[kDoneCnt].
//
// What bounds it: the chain of memory latencies of a round, times the rounds
// (3122 for the 120 343 contacts of a folded 256^2 sheet).  So in proximity
// passes half of the workgroup runs contacts and the other half fetches: a
// running contact first releases its successors (they only run in the next
// round, after the barrier that ends this one) and loads its velocities;
// behind an LDS-only barrier the runners form and store the impulses while the
// fetchers load the released contacts' geometry and successors, which come
// from far memory, into LDS for the next round, every load of a thread in
// flight at once.  The four counter atomics of a contact are all in flight
// together, at workgroup scope (no other workgroup touches the counters).
// What a round has beyond the runners' contacts every thread helps to run
// first.  In a continuous pass, where nothing can be fetched ahead (the
// geometry depends on the velocities), every thread runs contacts.
// Against 1024 threads that each load their own data, and against 256 runners
// with one load of a fetcher in flight: folded 256^2 sheet 14.8 / 7.1 / 6.6 ms
// (2.1 us per round), 253 x 397 drop 38 / 20.1 / 18.2 ms, four stacked 128^2
// sheets 10.1 / 6.4 / 5.1 ms, and four stacked 512^2 sheets, whose 23 035
// rounds have about 290 contacts, 215 / 259 / 193 ms; 384 runners: 7.4, 20.1,
// 5.5 and 204 ms.
// Released contacts are listed in LDS up to lds_cap, the rest of a longer round
// in the global lists; the first kDrainRecs of a round have their data in LDS
// (two rounds of them and the lists fill 140 of 160 KB), others load it
// themselves.  lds_cap (at most kDrainLds) is smaller only for
// tests (the CLOTHSIM_DRAIN_LDS environment variable).
constexpr int kDrainLds = 4096;
constexpr int kDrainRun = 512;   // runners, and as many fetchers
constexpr int kDrainRecs = 384;  // contacts of a round whose data is in LDS
constexpr int kDrainPieces = (int)sizeof(ImpulseGeom) / 16 + 1;  // 16 bytes each: geometry, successors
constexpr int kDrainCcd = 1024;  // threads of a continuous pass
static_assert(sizeof(ImpulseGeom) % 16 == 0, "a contact's geometry moves in 16-byte pieces");

// kGeom: a proximity pass (else a continuous one, which reads ce, X, delta, dt)
template <bool kGeom>
__global__ __launch_bounds__(kGeom ? 2 * kDrainRun : kDrainCcd) void k_impulse_drain(
    const int* ce, const int* succ, int* npred, int* ready0, int* ready1, const double* X, double* U,
    double delta, double dt, double m, int* counters, int lds_cap, const ImpulseGeom* geom) {
  constexpr int kThreads = kGeom ? 2 * kDrainRun : kDrainCcd;
  constexpr int kRun = kGeom ? kDrainRun : 0;  // contacts of a round that the runners take
  __shared__ int count[2];  // contacts released for the next round, in turn
  __shared__ int lists[2][kDrainLds];
  __shared__ int4 rec[2][kGeom ? kDrainRecs : 1][kDrainPieces];
  const int tid = threadIdx.x;
  int n = counters[kReady];
  int *gcur = ready0, *gnxt = ready1;  // the first round's list and the spills
  int cur = 0;                         // the LDS list and data of this round
  bool first = true;                   // the first round reads k_impulse_ready's list
  int done = 0;
  // data is fetched for contacts listed in LDS (a spilled entry is not visible
  // behind the LDS-only barrier)
  const int recs = min(kDrainRecs, lds_cap);
  if (tid < 2) count[tid] = 0;
  __syncthreads();
  auto listed = [&](int t) { return (first || t >= lds_cap) ? gcur[t] : lists[cur][t]; };
  auto release = [&](int c) {
    const int pos = atomicAdd(&count[cur ^ 1], 1);
    if (pos < lds_cap)
      lists[cur ^ 1][pos] = c;
    else
      gnxt[pos] = c;
  };
  // releases the successors of contact i; loads its velocities in between
  auto begin = [&](int i, const int4& sc, const ImpulseGeom& o, Vec3 (&v)[4]) {
    const int s4[4] = {sc.x, sc.y, sc.z, sc.w};
    int left[4];
#pragma unroll
    for (int a = 0; a < 4; a++)
      // unconditional, so that the four are in flight together: without a
      // successor the contact's own counter, which nothing reads any more
      left[a] = __hip_atomic_fetch_sub(&npred[s4[a] >= 0 ? s4[a] : i], 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
    if (kGeom)
#pragma unroll
      for (int a = 0; a < 4; a++) v[a] = at(U, o.v[a]);
#pragma unroll
    for (int a = 0; a < 4; a++)
      if (s4[a] >= 0 && left[a] == 1) release(s4[a]);
  };
  auto finish = [&](int i, const ImpulseGeom& o, const Vec3 (&v)[4]) {
    if (kGeom)
      impulse_velocity(o, v[0], v[1], v[2], v[3], U, m);
    else
      impulse_ccd(ce + 5 * i, X, U, delta, dt, m);
  };
  while (n > 0) {
    ImpulseGeom o{};
    Vec3 v[4];
    int i = -1;
    // what the runners do not take, on every thread
    for (int t = kRun + tid; t < n; t += kThreads) {
      const int c = listed(t);
      if (kGeom) o = geom[c];
      begin(c, reinterpret_cast<const int4*>(succ)[c], o, v);
      finish(c, o, v);
    }
    if (kGeom && tid < min(n, kRun)) {
      i = listed(tid);
      int4 sc;
      if (!first && tid < recs) {
        int4 w[kDrainPieces];
#pragma unroll
        for (int p = 0; p < kDrainPieces; p++) w[p] = rec[cur][tid][p];
        __builtin_memcpy(&o, w, sizeof(o));
        sc = w[kDrainPieces - 1];
      } else {
        o = geom[i];
        sc = reinterpret_cast<const int4*>(succ)[i];
      }
      begin(i, sc, o, v);
    }
    lds_only_barrier();  // the next round's list is complete; loads stay in flight
    const int next = count[cur ^ 1];
    if (i >= 0) finish(i, o, v);
    if (tid == 0) count[cur] = 0;  // read by every thread before the barrier above
    const int pieces = min(next, recs) * kDrainPieces;
    if (kGeom && tid - kRun >= 0 && tid - kRun < pieces) {
      // every load issued before the first is stored (past the end: the last piece)
      int4 w[kDrainPieces];
#pragma unroll
      for (int u = 0; u < kDrainPieces; u++) {
        const int q = min(tid - kRun + u * kDrainRun, pieces - 1);
        const int e = q / kDrainPieces, p = q - e * kDrainPieces;
        const int c = lists[cur ^ 1][e];
        w[u] = p < kDrainPieces - 1 ? reinterpret_cast<const int4*>(geom + c)[p]
                                    : reinterpret_cast<const int4*>(succ)[c];
      }
#pragma unroll
      for (int u = 0; u < kDrainPieces; u++) {
        const int q = tid - kRun + u * kDrainRun;
        if (q < pieces) (&rec[cur ^ 1][0][0])[q] = w[u];
      }
    }
    done += n;
    __syncthreads();  // the round's velocities and the next round's data are complete
    n = next;
    int* tmp = gcur;
    gcur = gnxt;
    gnxt = tmp;
    cur ^= 1;
    first = false;
  }
  if (tid == 0) counters[kDoneCnt] = done;
}

// ---------------------------------------------------------------------------
// rigid impact zones (self_collision_cloth.cpp:220-348), one workgroup

__device__ int zfind(int* par, int v) {
  while (par[v] != v) {
    par[v] = par[par[v]];
    v = par[v];
  }
  return v;
}
__device__ int zfind_ro(const int* par, int v) {
  while (par[v] != v) v = par[v];
  return v;
}

// block-wide exclusive scan of one int per thread; the block total goes to *total
__device__ int block_excl_scan(int x, int* total) {
  __shared__ int ws[16];
  __shared__ int tot;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int v = x;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(v, o, 64);
    if (lane >= o) v += y;
  }
  if (lane == 63) ws[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
      const int t = ws[w];
      ws[w] = acc;
      acc += t;
    }
    tot = acc;
  }
  __syncthreads();
  const int ex = v - x + ws[wid];
  const int t = tot;
  __syncthreads();
  *total = t;
  return ex;
}

__global__ __launch_bounds__(1024) void k_riz_pass(DevCloth c, const int* ce, int g, int* zpar,
                                                   int* zroot, int* zmemb, int* zroots,
                                                   const double* X, const double* U0, double* U,
                                                   int* counters) {
  // 1. zones touched by each contact through a vertex or its 1-ring; merge
  //    (only the partition matters: zone order never changes a result).
  //    Each touched zone is joined to the first one found as it is found, so
  //    any number of zones merges; membership (zpar >= 0) is what the
  //    reference tests, and a merge does not change it.
  if (threadIdx.x == 0) {
    for (int e = 0; e < g; e++) {
      const int* n4 = ce + 5 * e + 1;
      int root = -1;
      for (int a = 0; a < 4; a++) {
        const int v = n4[a];
        if (zpar[v] >= 0) {
          const int r = zfind(zpar, v);
          if (root < 0) root = r; else if (r != root) zpar[r] = root;
        }
        for (int q = c.ring_ptr[v]; q < c.ring_ptr[v + 1]; q++) {
          const int w = c.ring[q];
          if (zpar[w] < 0) continue;
          const int r = zfind(zpar, w);
          if (root < 0) root = r; else if (r != root) zpar[r] = root;
        }
      }
      if (root < 0) {
        root = n4[0];
        zpar[root] = root;
      }
      for (int a = 0; a < 4; a++)
        if (zpar[n4[a]] < 0) zpar[n4[a]] = root;
    }
  }
  __syncthreads();
  // 2. zone members in ascending vertex order, and the zone roots
  __shared__ int s_off, s_roff;
  if (threadIdx.x == 0) {
    s_off = 0;
    s_roff = 0;
  }
  __syncthreads();
  for (int base = 0; base < c.np; base += blockDim.x) {
    const int v = base + threadIdx.x;
    int in = 0, isroot = 0;
    if (v < c.np && zpar[v] >= 0) {
      const int r = zfind_ro(zpar, v);
      in = 1;
      isroot = (r == v);
      zroot[v] = r;
    }
    int tot, rtot;
    const int pos = block_excl_scan(in, &tot);
    const int rpos = block_excl_scan(isroot, &rtot);
    if (in) zmemb[s_off + pos] = v;
    if (isroot) zroots[s_roff + rpos] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      s_off += tot;
      s_roff += rtot;
    }
    __syncthreads();
  }
  const int nm = s_off, nz = s_roff;
  if (threadIdx.x == 0) counters[kZoneVerts] = nm;
  // 3. rigid velocity per zone from the pre-zone velocities U0
  for (int z = threadIdx.x; z < nz; z += blockDim.x) {
    const int R = zroots[z];
    Vec3 gc = mk(0, 0, 0), av = mk(0, 0, 0);
    int cnt = 0;
    for (int q = 0; q < nm; q++) {
      const int v = zmemb[q];
      if (zroot[v] != R) continue;
      gc = gc + at(X, v);
      av = av + at(U0, v);
      cnt++;
    }
    const double dn = (double)cnt;
    if (!(fabs(dn) < 1.e-16)) {  // operator/= guard (vector3d.h:63-67)
      gc = mk(gc.x / dn, gc.y / dn, gc.z / dn);
      av = mk(av.x / dn, av.y / dn, av.z / dn);
    }
    Vec3 L = mk(0, 0, 0);
    double I[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int q = 0; q < nm; q++) {
      const int v = zmemb[q];
      if (zroot[v] != R) continue;
      const Vec3 p = at(X, v), u = at(U0, v);
      L = L + cross(p - gc, u - av);
      const Vec3 r = p - gc;
      const double uu = dot(u, u);  // |v|^2 where a rigid inertia uses |r|^2 (:327-329)
      I[0] += uu - r.x * r.x;
      I[1] += -r.x * r.y;
      I[2] += -r.x * r.z;
      I[3] += -r.y * r.x;
      I[4] += uu - r.y * r.y;
      I[5] += -r.y * r.z;
      I[6] += -r.z * r.x;
      I[7] += -r.z * r.y;
      I[8] += uu - r.z * r.z;
    }
    const double det = +I[0] * I[4] * I[8] + I[3] * I[7] * I[2] + I[6] * I[1] * I[5] -
                       I[0] * I[7] * I[5] - I[6] * I[4] * I[2] - I[3] * I[1] * I[8];
    const double id = 1.0 / det;
    double J[9];
    J[0] = id * (I[4] * I[8] - I[5] * I[7]);
    J[1] = id * (I[2] * I[7] - I[1] * I[8]);
    J[2] = id * (I[1] * I[5] - I[2] * I[4]);
    J[3] = id * (I[5] * I[6] - I[3] * I[8]);
    J[4] = id * (I[0] * I[8] - I[2] * I[6]);
    J[5] = id * (I[2] * I[3] - I[0] * I[5]);
    J[6] = id * (I[3] * I[7] - I[4] * I[6]);
    J[7] = id * (I[1] * I[6] - I[0] * I[7]);
    J[8] = id * (I[0] * I[4] - I[1] * I[3]);
    const Vec3 om = mk(J[0] * L.x + J[1] * L.y + J[2] * L.z, J[3] * L.x + J[4] * L.y + J[5] * L.z,
                       J[6] * L.x + J[7] * L.y + J[8] * L.z);
    for (int q = 0; q < nm; q++) {
      const int v = zmemb[q];
      if (zroot[v] != R) continue;
      const Vec3 rr = cross(at(X, v) - gc, om);
      U[3 * v] = av.x + -rr.x;
      U[3 * v + 1] = av.y + -rr.y;
      U[3 * v + 2] = av.z + -rr.z;
    }
  }
}

// ---------------------------------------------------------------------------
// after the contact pass (self_contact_sparse/main.cpp:246-261,
// solve_internal_sparse.h:329-369)

__global__ void k_advance(DevCloth c, double dt) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 3 * c.np) return;
  c.x[e] = c.x1[e] + c.v[e] * dt;
}

__global__ void k_velocity_update(DevCloth c, Params P) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= c.np) return;
  double g[3] = {0.0, 0.0, 0.0};
  for (int s = c.grad_src_ptr[i]; s < c.grad_src_ptr[i + 1]; s++) {
    const int src = c.grad_src[s];
    const double* e = (src >= 0) ? c.etri + (size_t)(src / 3) * 90 + 81 + (src % 3) * 3
                                 : c.eq + (size_t)(-src - 1) * 3;
    g[0] += e[0];
    g[1] += e[1];
    g[2] += e[2];
  }
  for (int k = 0; k < 3; k++) g[k] -= P.mass * P.grav[k];
  double* v = c.v + 3 * i;
  if (c.bc[i] != 0) v[0] = v[1] = v[2] = 0;
  for (int k = 0; k < 3; k++) v[k] += -(0.5 * P.dt / P.mass) * g[k];
}

// ---------------------------------------------------------------------------
// host side

namespace {

// device buffers of the contact state: allocated and released in the order
// of the cloth's stream s, without synchronising the device
template <typename T>
int dalloc(T** p, size_t n, hipStream_t s) {
  return dev_alloc((void**)p, sizeof(T) * (n ? n : 1), s);
}
template <typename T>
void dfree(T*& p, hipStream_t s) {
  dev_free(p, s);
  p = nullptr;
}

int grow_records(ContactState& cs, int need, hipStream_t s) {
  if (need <= cs.cap) return kOk;
  CS_HIP(hipStreamSynchronize(s));
  int cap = std::max(need + need / 2, 1 << 16);
  dfree(cs.rkey, s);
  dfree(cs.rinfo, s);
  dfree(cs.rpair, s);
  dfree(cs.skey[0], s);
  dfree(cs.skey[1], s);
  dfree(cs.sidx[0], s);
  dfree(cs.sidx[1], s);
  dfree(cs.head, s);
  dfree(cs.gpos, s);
  dfree(cs.ce, s);
  dfree(cs.pred, s);
  dfree(cs.succ, s);
  dfree(cs.npred, s);
  dfree(cs.ready[0], s);
  dfree(cs.ready[1], s);
  dfree(cs.inc, s);
  dev_free(cs.tmp, s);
  cs.tmp = nullptr;
  cs.cap = 0;
  if (int st = dalloc(&cs.rkey, 4L * cap, s)) return st;
  if (int st = dalloc(&cs.rinfo, cap, s)) return st;
  if (int st = dalloc(&cs.rpair, 2L * cap, s)) return st;
  if (int st = dalloc(&cs.skey[0], cap, s)) return st;
  if (int st = dalloc(&cs.skey[1], cap, s)) return st;
  if (int st = dalloc(&cs.sidx[0], cap, s)) return st;
  if (int st = dalloc(&cs.sidx[1], cap, s)) return st;
  if (int st = dalloc(&cs.head, cap, s)) return st;
  if (int st = dalloc(&cs.gpos, cap, s)) return st;
  if (int st = dalloc(&cs.ce, 5L * cap, s)) return st;
  if (int st = dalloc(&cs.pred, 4L * cap, s)) return st;
  if (int st = dalloc(&cs.succ, 4L * cap, s)) return st;
  if (int st = dalloc(&cs.npred, cap, s)) return st;
  if (int st = dalloc(&cs.ready[0], cap, s)) return st;
  if (int st = dalloc(&cs.ready[1], cap, s)) return st;
  if (int st = dalloc(&cs.inc, 4L * cap, s)) return st;
  // temporary storage for the largest sort / scan
  size_t a = 0, b = 0, c2 = 0;
  CS_HIP(rocprim::radix_sort_pairs(nullptr, a, cs.skey[0], cs.skey[1], cs.sidx[0], cs.sidx[1],
                                   (unsigned)cap, 0, 64, s));
  CS_HIP(rocprim::exclusive_scan(nullptr, b, cs.head, cs.gpos, 0, (size_t)cap,
                                 rocprim::plus<int>(), s));
  CS_HIP(rocprim::exclusive_scan(nullptr, c2, cs.vcount, cs.vstart, 0, (size_t)cs.np + 1,
                                 rocprim::plus<int>(), s));
  cs.tmp_bytes = std::max(a, std::max(b, c2)) + 256;
  if (int st = dev_alloc(&cs.tmp, cs.tmp_bytes, s)) return st;
  cs.cap = cap;
  return kOk;
}

int grow_cand(ContactState& cs, int need, hipStream_t s) {
  if (need <= cs.cand_cap) return kOk;
  CS_HIP(hipStreamSynchronize(s));
  const int cap = std::max(need + need / 2, 1 << 16);
  dfree(cs.cand, s);
  cs.cand_cap = 0;
  if (int st = dalloc(&cs.cand, 2L * cap, s)) return st;
  cs.cand_cap = cap;
  return kOk;
}

int read_counters(ContactState& cs, hipStream_t s) {
  CS_HIP(hipMemcpyAsync(cs.hcounters, cs.counters, sizeof(int) * kNumCounters,
                        hipMemcpyDeviceToHost, s));
  CS_HIP(hipStreamSynchronize(s));
  return kOk;
}

int refit(ContactState& cs, const DevCloth& d, hipStream_t s, const double* X, const double* U,
          double delta, double dt, int ccd) {
  hipLaunchKernelGGL(k_refit_leaves, dim3(grid_for(d.nt)), dim3(kTB), 0, s, d, X, U, delta, dt,
                     ccd);
  for (size_t l = 0; l + 1 < cs.refit_lvl.size(); l++) {
    const int b = cs.refit_lvl[l], e = cs.refit_lvl[l + 1];
    if (e > b) hipLaunchKernelGGL(k_refit_merge, dim3(grid_for(e - b)), dim3(kTB), 0, s, d, b, e);
  }
  CS_HIP(hipGetLastError());
  return kOk;
}

// refit + traverse + select: the contact set into cs.ce, its size into *g
int query(ContactState& cs, const DevCloth& d, hipStream_t s, const double* X, const double* U,
          double delta, double dt, int ccd, int* g) {
  if (int st = refit(cs, d, s, X, U, delta, dt, ccd)) return st;
  int ncand = 0;
  for (int attempt = 0; attempt < 2; attempt++) {
    CS_HIP(hipMemsetAsync(cs.counters, 0, sizeof(int) * kQueryCounters, s));
    // leaves per wave: 64, halved (down to 16) while the launch would have
    // fewer than 2048 waves, so that a small tree's walks spread over more waves
    int per = 64;
    while (per > 16 && (d.nt + per - 1) / per < 2048) per /= 2;
    hipLaunchKernelGGL(k_traverse, dim3((d.nt + per - 1) / per), dim3(64), 0, s, d.nnode, d.nt, per,
                       d.leaf_rank, d.rend, d.rbb, d.by_pre, cs.counters, cs.cand_cap,
                       reinterpret_cast<int2*>(cs.cand));
    CS_HIP(hipGetLastError());
    if (int st = read_counters(cs, s)) return st;
    ncand = cs.hcounters[kCand];
    if (ncand <= cs.cand_cap) break;
    if (int st = grow_cand(cs, ncand, s)) return st;
  }
  int raw = 0;
  for (int attempt = 0; attempt < 2 && ncand > 0; attempt++) {
    CS_HIP(hipMemsetAsync(cs.counters + kRaw, 0, sizeof(int), s));
    Emit em{cs.counters, cs.cap, cs.rkey, cs.rinfo, cs.rpair};
    if (ccd)
      hipLaunchKernelGGL(k_narrow<true>, dim3(grid_for(ncand)), dim3(kTB), 0, s, d, X, U, dt, delta,
                         ncand, cs.cand, em);
    else
      hipLaunchKernelGGL(k_narrow<false>, dim3(grid_for(ncand)), dim3(kTB), 0, s, d, X, U, dt,
                         delta, ncand, cs.cand, em);
    CS_HIP(hipGetLastError());
    if (int st = read_counters(cs, s)) return st;
    raw = cs.hcounters[kRaw];
    if (raw <= cs.cap) break;
    if (int st = grow_records(cs, raw, s)) return st;
  }
  if (raw == 0) {
    *g = 0;
    return kOk;
  }
  // radix sort of the records by canonical key
  const int nb = cs.nbits;
  const int* order = nullptr;
  size_t tb = cs.tmp_bytes;
  if (4 * nb <= 64) {
    hipLaunchKernelGGL(k_make_keys, dim3(grid_for(raw)), dim3(kTB), 0, s, cs.rkey, raw, nb, 0,
                       cs.skey[0], cs.sidx[0]);
    CS_HIP(rocprim::radix_sort_pairs(cs.tmp, tb, cs.skey[0], cs.skey[1], cs.sidx[0], cs.sidx[1],
                                     (unsigned)raw, 0, 4 * nb, s));
    order = cs.sidx[1];
  } else {
    hipLaunchKernelGGL(k_make_keys, dim3(grid_for(raw)), dim3(kTB), 0, s, cs.rkey, raw, nb, 1,
                       cs.skey[0], cs.sidx[0]);
    CS_HIP(rocprim::radix_sort_pairs(cs.tmp, tb, cs.skey[0], cs.skey[1], cs.sidx[0], cs.sidx[1],
                                     (unsigned)raw, 0, nb, s));
    hipLaunchKernelGGL(k_rekey, dim3(grid_for(raw)), dim3(kTB), 0, s, cs.rkey, cs.sidx[1], raw, nb,
                       cs.skey[0]);
    tb = cs.tmp_bytes;
    CS_HIP(rocprim::radix_sort_pairs(cs.tmp, tb, cs.skey[0], cs.skey[1], cs.sidx[1], cs.sidx[0],
                                     (unsigned)raw, 0, 3 * nb, s));
    order = cs.sidx[0];
  }
  hipLaunchKernelGGL(k_heads, dim3(grid_for(raw)), dim3(kTB), 0, s, cs.rkey, order, raw, cs.head);
  tb = cs.tmp_bytes;
  CS_HIP(rocprim::exclusive_scan(cs.tmp, tb, cs.head, cs.gpos, 0, (size_t)raw,
                                 rocprim::plus<int>(), s));
  hipLaunchKernelGGL(k_select, dim3(grid_for(raw)), dim3(kTB), 0, s, d, cs.rkey, cs.rinfo,
                     cs.rpair, order, cs.head, cs.gpos, raw, cs.ce, cs.counters);
  CS_HIP(hipGetLastError());
  if (int st = read_counters(cs, s)) return st;
  *g = cs.hcounters[kGroups];
  return kOk;
}

// Gauss-Seidel impulses over cs.ce[0..g) in key order
int impulses(ContactState& cs, const DevCloth& d, const Params& P, hipStream_t s, const double* X,
             double* U, int g, int ccd) {
  if (g == 0) return kOk;
  CS_HIP(hipMemsetAsync(cs.vcount, 0, sizeof(int) * (d.np + 1), s));
  CS_HIP(hipMemsetAsync(cs.vfill, 0, sizeof(int) * (d.np + 1), s));
  hipLaunchKernelGGL(k_inc_count, dim3(grid_for(g)), dim3(kTB), 0, s, cs.ce, g, cs.vcount);
  size_t tb = cs.tmp_bytes;
  CS_HIP(rocprim::exclusive_scan(cs.tmp, tb, cs.vcount, cs.vstart, 0, (size_t)d.np + 1,
                                 rocprim::plus<int>(), s));
  hipLaunchKernelGGL(k_inc_fill, dim3(grid_for(g)), dim3(kTB), 0, s, cs.ce, g, cs.vstart, cs.vfill,
                     cs.inc);
  hipLaunchKernelGGL(k_inc_link, dim3(grid_for(d.np)), dim3(kTB), 0, s, d.np, cs.vstart, cs.inc,
                     cs.pred, cs.succ);
  CS_HIP(hipMemsetAsync(cs.counters + kDoneCnt, 0, sizeof(int), s));
  CS_HIP(hipMemsetAsync(cs.counters + kReady, 0, sizeof(int), s));
  hipLaunchKernelGGL(k_impulse_ready, dim3(grid_for(g)), dim3(kTB), 0, s, g, cs.pred, cs.npred,
                     cs.ready[0], cs.counters);
  if (!ccd) {
    if (g > cs.geom_cap) {
      dev_free(cs.geom, s);
      cs.geom = nullptr;
      cs.geom_cap = 0;
      const int cap = g + g / 2;
      if (int st = dev_alloc(&cs.geom, sizeof(ImpulseGeom) * cap, s)) return st;
      cs.geom_cap = cap;
    }
    hipLaunchKernelGGL(k_impulse_geom, dim3(grid_for(g)), dim3(kTB), 0, s, cs.ce, g, X, P.clearance,
                       P.k_contact, P.dt, (ImpulseGeom*)cs.geom);
  }
  int lds_cap = kDrainLds;
  if (const char* e = getenv("CLOTHSIM_DRAIN_LDS")) lds_cap = std::min(std::max(atoi(e), 1), kDrainLds);
  if (ccd)
    hipLaunchKernelGGL(k_impulse_drain<false>, dim3(1), dim3(kDrainCcd), 0, s, cs.ce, cs.succ,
                       cs.npred, cs.ready[0], cs.ready[1], X, U, P.clearance, P.dt, P.mass,
                       cs.counters, lds_cap, (const ImpulseGeom*)nullptr);
  else
    hipLaunchKernelGGL(k_impulse_drain<true>, dim3(1), dim3(2 * kDrainRun), 0, s, cs.ce, cs.succ,
                       cs.npred, cs.ready[0], cs.ready[1], X, U, P.clearance, P.dt, P.mass,
                       cs.counters, lds_cap, (const ImpulseGeom*)cs.geom);
  CS_HIP(hipGetLastError());
  if (int st = read_counters(cs, s)) return st;
  if (cs.hcounters[kDoneCnt] != g) {
    set_error("impulse schedule did not drain");
    return kHipError;
  }
  return kOk;
}

}  // namespace

int contact_init(ContactState& cs, const MeshSetup& S, const DevCloth& d, hipStream_t s) {
  cs.np = S.np;
  cs.nt = S.nt;
  cs.nnode = S.nnode;
  int nb = 1;
  while ((1 << nb) < S.np) nb++;
  cs.nbits = nb;
  if (3 * nb > 64) {
    set_error("mesh too large for the contact keys");
    return kBadArg;
  }
  if (int st = dalloc(&cs.vcount, S.np + 1, s)) return st;
  if (int st = dalloc(&cs.vstart, S.np + 1, s)) return st;
  if (int st = dalloc(&cs.vfill, S.np + 1, s)) return st;
  if (int st = dalloc(&cs.counters, kNumCounters, s)) return st;
  cs.refit_lvl = S.refit_lvl_ptr;
  if (int st = dalloc(&cs.zpar, S.np, s)) return st;
  if (int st = dalloc(&cs.zroot, S.np, s)) return st;
  if (int st = dalloc(&cs.zmemb, S.np, s)) return st;
  if (int st = dalloc(&cs.zroots, S.np, s)) return st;
  if (int st = dalloc(&cs.u0, 3L * S.np, s)) return st;
  if (int st = dalloc(&cs.qx, 3L * S.np, s)) return st;
  if (int st = dalloc(&cs.qv, 3L * S.np, s)) return st;
  if (int st = pinned_alloc((void**)&cs.hcounters, sizeof(int) * kNumCounters)) return st;
  CS_HIP(hipMemsetAsync(cs.counters, 0, sizeof(int) * kNumCounters, s));
  if (int st = grow_cand(cs, std::max(8 * S.nt, 1 << 16), s)) return st;
  return grow_records(cs, std::max(8 * S.nt, 1 << 16), s);
}

void contact_release(ContactState& cs, hipStream_t s) {
  dfree(cs.cand, s);
  cs.cand_cap = 0;
  dfree(cs.rkey, s);
  dfree(cs.rinfo, s);
  dfree(cs.rpair, s);
  dfree(cs.skey[0], s);
  dfree(cs.skey[1], s);
  dfree(cs.sidx[0], s);
  dfree(cs.sidx[1], s);
  dfree(cs.head, s);
  dfree(cs.gpos, s);
  dfree(cs.ce, s);
  dfree(cs.pred, s);
  dfree(cs.succ, s);
  dfree(cs.npred, s);
  dfree(cs.ready[0], s);
  dfree(cs.ready[1], s);
  dfree(cs.inc, s);
  dfree(cs.vcount, s);
  dfree(cs.vstart, s);
  dfree(cs.vfill, s);
  dfree(cs.counters, s);
  dfree(cs.zpar, s);
  dfree(cs.zroot, s);
  dfree(cs.zmemb, s);
  dfree(cs.zroots, s);
  dfree(cs.u0, s);
  dfree(cs.qx, s);
  dfree(cs.qv, s);
  dev_free(cs.tmp, s);
  cs.tmp = nullptr;
  dev_free(cs.geom, s);
  cs.geom = nullptr;
  cs.geom_cap = 0;
  pinned_free(cs.hcounters);
  cs.hcounters = nullptr;
}

int contact_resolve(ContactState& cs, const MeshSetup& S, const DevCloth& d, const Params& P,
                    hipStream_t s, int* applied, cs_step_stats* stats, Prof* prof) {
  (void)S;
  ProfScope ps(prof, kProfContact);
  const double* X = d.x1;
  double* U = d.v;
  int g = 0;
  if (stats) {
    stats->n_prox = 0;
    stats->n_ccd_pass = 0;
    for (int k = 0; k < 5; k++) stats->n_ccd[k] = 0;
    stats->n_riz_pass = 0;
    stats->n_riz_vertices = 0;
  }
  // one proximity pass
  if (int st = query(cs, d, s, X, U, P.clearance, P.dt, 0, &g)) return st;
  *applied = g > 0;
  if (stats) stats->n_prox = g;
  if (int st = impulses(cs, d, P, s, X, U, g, 0)) return st;
  // up to five continuous passes
  for (int it = 0; it < 5; it++) {
    if (int st = query(cs, d, s, X, U, P.clearance, P.dt, 1, &g)) return st;
    if (g == 0) return kOk;
    *applied = 1;
    if (stats) {
      stats->n_ccd[it] = g;
      stats->n_ccd_pass = it + 1;
    }
    if (int st = impulses(cs, d, P, s, X, U, g, 1)) return st;
  }
  // rigid impact zones, up to 100 passes
  CS_HIP(hipMemcpyAsync(cs.u0, U, sizeof(double) * 3 * d.np, hipMemcpyDeviceToDevice, s));
  CS_HIP(hipMemsetAsync(cs.zpar, 0xff, sizeof(int) * d.np, s));
  CS_HIP(hipMemsetAsync(cs.counters + kZoneVerts, 0, sizeof(int), s));
  for (int it = 0; it < 100; it++) {
    if (int st = query(cs, d, s, X, U, P.clearance, P.dt, 1, &g)) return st;
    if (g == 0) break;
    hipLaunchKernelGGL(k_riz_pass, dim3(1), dim3(1024), 0, s, d, cs.ce, g, cs.zpar, cs.zroot,
                       cs.zmemb, cs.zroots, X, (const double*)cs.u0, U, cs.counters);
    CS_HIP(hipGetLastError());
    if (stats) stats->n_riz_pass = it + 1;
  }
  if (stats && stats->n_riz_pass > 0) {
    if (int st = read_counters(cs, s)) return st;
    stats->n_riz_vertices = cs.hcounters[kZoneVerts];
  }
  return kOk;
}

int update_velocity(const DevCloth& d, const Params& P, hipStream_t s) {
  if (int st = launch_gradients(d, P, s)) return st;
  hipLaunchKernelGGL(k_velocity_update, dim3(grid_for(d.np)), dim3(kTB), 0, s, d, P);
  CS_HIP(hipGetLastError());
  return kOk;
}

int post_contact_update(const DevCloth& d, const Params& P, hipStream_t s) {
  hipLaunchKernelGGL(k_advance, dim3(grid_for(3L * d.np)), dim3(kTB), 0, s, d, P.dt);
  CS_HIP(hipGetLastError());
  return update_velocity(d, P, s);
}

int contact_refit_host(ContactState& cs, const MeshSetup& S, const DevCloth& d, hipStream_t s,
                       const double* xyz, const double* uvw, double delta, double dt, double* bb) {
  const size_t n = sizeof(double) * 3 * d.np;
  CS_HIP(hipMemcpyAsync(cs.qx, xyz, n, hipMemcpyHostToDevice, s));
  if (uvw) CS_HIP(hipMemcpyAsync(cs.qv, uvw, n, hipMemcpyHostToDevice, s));
  if (int st = refit(cs, d, s, cs.qx, cs.qv, delta, dt, uvw ? 1 : 0)) return st;
  if (bb) CS_HIP(hipMemcpyAsync(bb, d.bb, sizeof(double) * 6 * S.nnode, hipMemcpyDeviceToHost, s));
  CS_HIP(hipStreamSynchronize(s));
  return kOk;
}

int contact_query_host(ContactState& cs, const MeshSetup& S, const DevCloth& d, hipStream_t s,
                       const double* xyz, const double* uvw, double delta, double dt, int* out,
                       int cap, int* n) {
  (void)S;
  const size_t bytes = sizeof(double) * 3 * d.np;
  CS_HIP(hipMemcpyAsync(cs.qx, xyz, bytes, hipMemcpyHostToDevice, s));
  if (uvw) CS_HIP(hipMemcpyAsync(cs.qv, uvw, bytes, hipMemcpyHostToDevice, s));
  int g = 0;
  if (int st = query(cs, d, s, cs.qx, cs.qv, delta, dt, uvw ? 1 : 0, &g)) return st;
  if (n) *n = g;
  const int m = std::min(g, cap);
  if (out && m > 0)
    CS_HIP(hipMemcpyAsync(out, cs.ce, sizeof(int) * 5 * m, hipMemcpyDeviceToHost, s));
  CS_HIP(hipStreamSynchronize(s));
  return kOk;
}

}  // namespace cs
