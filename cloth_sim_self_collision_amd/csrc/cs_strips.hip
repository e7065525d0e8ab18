// The triangular sweeps by strips: one wave sweeps a contiguous strip of rows
// (cs_strips.hpp), strips run on different CUs, and a strip takes the rows it
// needs of the strips before it as they are finished.
//
// Work of a wave, per sub-level: eight lanes per row, two halves of four.  Lane
// r (0..2) of a half forms component r of the products of its half's blocks
// (lane 3 idles); the first half then subtracts its own products and, read
// across the halves, the second half's.  The operations of a row are the
// reference's (ilu_sparse.cpp:185-215, 295-324), in its order: t_r = rhs_r
// minus the blocks' products in column order, forward then z_r = d_r0 t0 +
// d_r1 t1 + d_r2 t2.  Two halves because a sub-level lasts as long as one
// wave's instructions: with four lanes per row (16 rows per sub-level, half
// the strips) a sub-level took 314 ns and the 256^2 sheet's sweep 511 us.
// A wave needs no barrier: its own rows go through an LDS ring that only it
// uses (one wave's LDS operations execute in order).
//
// Handoff between strips.  A sweep's results are stored with device scope to
// the array that also is its result (forward: the backward sweep's
// right-hand side st_sb, backward: z), which holds "not written yet" before:
// a signalling NaN, which no arithmetic produces.  A reader takes the value
// once it is there; 8-byte accesses are single, so value and readiness cannot
// disagree and neither fences nor flags are needed.  Readers load four
// sub-levels ahead, so a strip that trails the one before it by the latency
// of a store and a load never waits; the first sub-levels of a strip do.
// z is marked by the kernels that write r before the sweep (k_pcg_init,
// k_update_rx, the gather of a single solve); st_sb by the backward sweep
// itself once it has consumed an entry (every forward reader of row i is a
// row j > i that a block couples to i, and i's backward step comes after j's,
// the pattern being symmetric).
//
// Order.  The waves claim strips from one counter: the forward strips in
// order, then the backward ones.  A claimed strip only ever waits for strips
// claimed before it, by waves that are running, so every wait ends whatever
// number of workgroups is resident (a bound on the wait reports an error
// instead of hanging should that ever fail).  The last claim resets the
// counter.
//
// What a wave reads is laid out in the order it reads it: per sub-level one
// record of 1 KiB pieces (16 bytes per lane): metadata (LDS offsets of the
// column rows, where the result goes), the coefficients, for the forward
// sweep D^-1 and the right-hand side.  All addresses of a sub-level are one
// scalar base plus the lane.
//
// What bounds it: the sub-levels on the longest path, about 0.2 us each (70
// instructions of one wave; 0.16 us without the loads), and 1.25 us for every
// strip boundary that path crosses (a device-scope store seen by a
// device-scope load).  Measured per launch, sheets of 32^2 / 128^2 / 256^2
// vertices: 52 / 198 / 391 us, against 74 / 455 / 1263 us for one workgroup
// with a barrier per sub-level (k_ilu_apply_quad), which keeps to one CU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "cs_device.hpp"
#include "cs_solve.hpp"
#include "cs_strips.hpp"

namespace cs {

namespace {

constexpr int kPiece = 1024;       // bytes per piece: 16 per lane
constexpr int kSets = kStripGroup; // register sets: sub-levels whose loads are in flight
constexpr int kSpinMax = 1 << 22;  // polls of one wait before it is given up

typedef int int4v __attribute__((ext_vector_type(4)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));

// blocks per half, and what a lane's 3 per block take in FP64 pairs / FP32 quads
__host__ __device__ constexpr int strip_half(int K) { return (K + 1) / 2; }
__host__ __device__ constexpr int strip_pairs(int K) { return (3 * strip_half(K) + 1) / 2; }
__host__ __device__ constexpr int strip_quads(int K) { return (3 * strip_half(K) + 3) / 4; }
// metadata word that holds the offset to store to, after the LDS offsets
__host__ __device__ constexpr int strip_out(int K) { return (strip_half(K) + 1) / 2; }
// pieces of a record: metadata, coefficients (FP32 quads use the first of the
// pairs' pieces), forward also D^-1 in two
__host__ __device__ constexpr int strip_pieces(bool fwd, int K) {
  return 1 + strip_pairs(K) + (fwd ? 2 : 0);
}
static_assert(strip_pieces(true, kMaxBlocksPerRow) <= 16 && strip_half(kMaxBlocksPerRow) <= 4,
              "a record's pieces are in reach of two offset registers, its metadata in one");

// device-scope accesses of results by 32-bit byte offset; an offset past the
// array (kStripNone) stores nothing and reads 0
constexpr int kDevScope = 16;  // sc1
__device__ __forceinline__ double res_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  const uint2v w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, kDevScope);
  return __hiloint2double((int)w.y, (int)w.x);
}
__device__ __forceinline__ void res_store(__amdgpu_buffer_rsrc_t r, unsigned off, double v) {
  uint2v w;
  w.x = (unsigned)__double2loint(v);
  w.y = (unsigned)__double2hiint(v);
  __builtin_amdgcn_raw_buffer_store_b64(w, r, (int)off, 0, kDevScope);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t res_of(double* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00027000);
}

template <int j>
__device__ __forceinline__ double quad_lane(double v) {
  constexpr int ctrl = j | (j << 2) | (j << 4) | (j << 6);
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// the value of the same component's lane in the other half (first half only:
// lane i reads lane i + 4 of its row of sixteen)
__device__ __forceinline__ double other_half(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x104, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x104, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// what a sub-level needs, loaded ahead
template <int K>
struct Set {
  unsigned meta[strip_out(K) + 1];  // the blocks' LDS offsets in pairs, where to store
  double a[3 * strip_half(K)];
  double d[3];
  double rhs;
  double imp;  // the imported rows' values
};

// one sweep's operands
struct Sweep {
  const char* rec;             // records
  const int4v* src;            // import offsets, four sub-levels per entry
  __amdgpu_buffer_rsrc_t res;  // the array written and imported from
  __amdgpu_buffer_rsrc_t sbr;  // forward results (the backward right-hand side)
  int polls;                   // of one wait before it is given up
};

template <class T>
__device__ __forceinline__ T piece_load(const char* rec, unsigned v0, unsigned v1, int p) {
  // eight pieces in reach of one offset register's immediates
  const unsigned v = p < 8 ? v0 : v1;
  const int imm = (p & 7) * kPiece - 4096;
  const auto g = (const __attribute__((address_space(1))) char*)rec;
  return *(const __attribute__((address_space(1))) T*)(g + v + imm);
}

template <bool kFwd, int K, bool F32>
__device__ __forceinline__ void set_load(Set<K>& q, const Sweep& w, int sub, unsigned src,
                                         unsigned v0, unsigned v1) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef float f4 __attribute__((ext_vector_type(4)));
  // only what is used is loaded (a last piece with one value as one value):
  // the compiler reuses an unused register of a load in flight, and waits for it
  constexpr int NB = strip_pairs(K), NV = 3 * strip_half(K);
  const char* rec = w.rec + (size_t)sub * (strip_pieces(kFwd, K) * kPiece);
  typedef unsigned words __attribute__((ext_vector_type(strip_out(K) + 1)));
  const words m = piece_load<words>(rec, v0, v1, 0);
#pragma unroll
  for (int j = 0; j <= strip_out(K); j++) q.meta[j] = m[j];
  if constexpr (F32) {
#pragma unroll
    for (int p = 0; 4 * p < NV; p++) {
      if (4 * p + 1 == NV) {
        q.a[4 * p] = (double)piece_load<float>(rec, v0, v1, 1 + p);
        continue;
      }
      const f4 x = piece_load<f4>(rec, v0, v1, 1 + p);
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (4 * p + j < NV) q.a[4 * p + j] = (double)x[j];
    }
  } else {
#pragma unroll
    for (int p = 0; 2 * p < NV; p++) {
      if (2 * p + 1 == NV) {
        q.a[2 * p] = piece_load<double>(rec, v0, v1, 1 + p);
        continue;
      }
      const d2 x = piece_load<d2>(rec, v0, v1, 1 + p);
      q.a[2 * p] = x.x;
      q.a[2 * p + 1] = x.y;
    }
  }
  if (kFwd) {
    const d2 x = piece_load<d2>(rec, v0, v1, 1 + NB);
    const d2 y = piece_load<d2>(rec, v0, v1, 2 + NB);
    q.d[0] = x.x;
    q.d[1] = x.y;
    q.d[2] = y.x;
    q.rhs = y.y;
  } else {
    q.rhs = res_load(w.sbr, (unsigned)sub * 512u + threadIdx.x * 8);
  }
  q.imp = res_load(w.res, src);
}

// some lane's import (backward: or right-hand side) is not there yet
template <bool kFwd>
__device__ __forceinline__ bool waiting(double imp, double rhs) {
  unsigned long long w = __builtin_amdgcn_ballot_w64(not_yet(imp));
  if (!kFwd) w |= __builtin_amdgcn_ballot_w64(not_yet(rhs));
  return w != 0ull;
}

// Polls until the imports (and, backward, the right-hand sides) of sub-level
// `sub`, in set n, are there.  Each poll also reloads what is missing of the
// two sub-levels after it, whose loads were issued too early as well: polling
// them one after another made a strip trail the one before it by 2.7 us, four
// round trips, instead of about one.
// Past the bound on the wait the wave goes on with what it has (`gave_up`,
// wave-uniform: it waits no more), the launches after this one do not wait at
// all, and the solve reports the error.
template <bool kFwd, int K>
__device__ __forceinline__ void set_wait(Set<K> (&q)[kSets], int n, const Sweep& w, int sub,
                                         const unsigned (&src)[3], int& gave_up) {
  if (gave_up) return;
  int polls = 0;
  do {
    asm volatile("" ::: "memory");  // every poll loads again
#pragma unroll
    for (int m = 0; m < 3; m++) {
      Set<K>& p = q[(n + m) % kSets];
      if (not_yet(p.imp)) p.imp = res_load(w.res, src[m]);
      if (!kFwd && not_yet(p.rhs))
        p.rhs = res_load(w.sbr, (unsigned)(sub + m) * 512u + threadIdx.x * 8);
    }
  } while (waiting<kFwd>(q[n].imp, q[n].rhs) && ++polls < w.polls);
  gave_up = __builtin_amdgcn_readfirstlane(polls >= w.polls);
}

// the column rows' entries of a lane's blocks
template <int K>
struct Cols {
  double2 y01[strip_half(K)];
  double y2[strip_half(K)];
};

// Sub-level `sub`'s imports into the ring, then its ring reads issued.  lds:
// this lane's place in sub-level 0's ring entries.
template <bool kFwd, int K>
__device__ __forceinline__ void set_read(Set<K> (&sets)[kSets], int n, Cols<K>& y, const Sweep& w,
                                         int sub, const unsigned (&src)[3], const char* ring0,
                                         char* lds, unsigned ringmask, int& gave_up) {
  Set<K>& q = sets[n];
  if (__builtin_expect(waiting<kFwd>(q.imp, q.rhs), 0))
    set_wait<kFwd, K>(sets, n, w, sub, src, gave_up);
  char* ring = lds + ((unsigned)(sub * kStripSub) & ringmask);
  *reinterpret_cast<double*>(ring + kStripRows * kStripEntry) = q.imp;
#pragma unroll
  for (int k = 0; k < strip_half(K); k++) {
    const char* e = ring0 + ((q.meta[k / 2] >> (16 * (k % 2))) & 0xffffu);
    y.y01[k] = *reinterpret_cast<const double2*>(e);
    y.y2[k] = *reinterpret_cast<const double*>(e + 16);
  }
}

// the sub-level's rows from what was read, into the ring (the second half's
// lanes have entries that nothing reads); returns the lane's result
template <bool kFwd, int K>
__device__ __forceinline__ double set_compute(const Set<K>& q, const Cols<K>& y, int sub,
                                              char* lds, unsigned ringmask) {
  constexpr int KH = strip_half(K);
  double pr[KH];
#pragma unroll
  for (int k = 0; k < KH; k++)
    pr[k] = q.a[3 * k] * y.y01[k].x + q.a[3 * k + 1] * y.y01[k].y + q.a[3 * k + 2] * y.y2[k];
  double t = q.rhs;
#pragma unroll
  for (int k = 0; k < KH; k++) t = t - pr[k];
#pragma unroll
  for (int k = 0; k < KH; k++) t = t - other_half(pr[k]);
  double z = t;
  if (kFwd) {
    const double t0 = quad_lane<0>(t), t1 = quad_lane<1>(t), t2 = quad_lane<2>(t);
    z = q.d[0] * t0 + q.d[1] * t1 + q.d[2] * t2;
  }
  *reinterpret_cast<double*>(lds + ((unsigned)(sub * kStripSub) & ringmask)) = z;
  return z;
}

template <bool kFwd, int K>
__device__ __forceinline__ void set_store(const Set<K>& q, const Sweep& w, int sub, double z) {
  const int out = (int)q.meta[strip_out(K)];  // negative: not a lane with a result
  res_store(w.res, (unsigned)out, z);
  // consumed: the next launch finds this right-hand side unwritten again
  if (!kFwd)
    res_store(w.sbr, (unsigned)(out >> 31) | ((unsigned)sub * 512u + threadIdx.x * 8), unwritten());
}

// Sub-levels [first, end) of one strip (a multiple of kStripGroup).  The loads
// of the next kSets sub-levels are in flight while one is computed (past the
// strip's end they read the next strip's records or the tail, unused).  After
// a sub-level's results are in the ring the next one's ring reads go out
// first, then the global stores and the loads that refill its registers: their
// issue (a dozen instructions) covers the LDS latency.
template <bool kFwd, int K, bool F32>
__device__ __forceinline__ void strip_sweep(const Sweep& w, int first, int end, char* ring0,
                                            unsigned ringmask, int& gave_up) {
  // this lane's place in a sub-level's ring entries
  const unsigned lane = threadIdx.x;
  char* lds = ring0 + kStripZero + (lane >> 3) * kStripEntry + (lane & 3) * 8 +
              (lane >> 2 & 1) * (2 * kStripRows * kStripEntry);
  const unsigned v0 = threadIdx.x * 16 + 4096, v1 = v0 + 8192;
  // (global pointers: the compiler cannot prove a batch table's pointers global,
  // and flat loads would also wait on the LDS counter)
  auto srcp = (const __attribute__((address_space(1))) int4v*)w.src +
              (size_t)(first / kStripGroup) * 64 + threadIdx.x;
  int4v s0 = srcp[0], s1 = srcp[64];
  Set<K> q[kSets];
  Cols<K> y;
#pragma unroll
  for (int j = 0; j < kSets; j++) {
    // in the order the loop refills them: a wait in the loop is for the loads
    // issued since, counted over both ways into it
    set_load<kFwd, K, F32>(q[j], w, first + j, (unsigned)s0[j], v0, v1);
    __builtin_amdgcn_sched_barrier(0);
  }
  // import offsets of the sub-level n positions into a group of s0 and the two after it
  auto src3 = [&](int n, unsigned (&src)[3]) {
#pragma unroll
    for (int m = 0; m < 3; m++)
      src[m] = (unsigned)(n + m < kSets ? s0[(n + m) % kSets] : s1[(n + m) % kSets]);
  };
  {
    unsigned src[3];
    src3(0, src);
    set_read<kFwd, K>(q, 0, y, w, first, src, ring0, lds, ringmask, gave_up);
  }
  for (int sub = first; sub < end; sub += kSets) {
    const int4v s2 = srcp[128];
    srcp += 64;
#pragma unroll
    for (int j = 0; j < kSets; j++) {
      const double z = set_compute<kFwd, K>(q[j], y, sub + j, lds, ringmask);
      // past the end this reads a sub-level of another strip, or the tail:
      // nothing to wait for then
      if (j + 1 < kSets || sub + kSets < end) {
        unsigned src[3];
        src3(j + 1, src);
        set_read<kFwd, K>(q, (j + 1) % kSets, y, w, sub + j + 1, src, ring0, lds, ringmask,
                          gave_up);
      }
      __builtin_amdgcn_sched_barrier(0);
      set_store<kFwd, K>(q[j], w, sub + j, z);
      set_load<kFwd, K, F32>(q[j], w, sub + kSets + j, (unsigned)s1[j], v0, v1);
      __builtin_amdgcn_sched_barrier(0);
    }
    s0 = s1;
    s1 = s2;
  }
}

}  // namespace

template <int K, bool F32, class Sel>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_strip_sweep(Sel sel, int polls) {
  const DevCloth c = sel.cloth();
  if (c.flags[kSkip]) return;
  extern __shared__ char lds[];
  if (threadIdx.x < kStripZero / 8) reinterpret_cast<double*>(lds)[threadIdx.x] = 0.0;
  const unsigned ringmask = (unsigned)(c.st_ring * kStripSub) - 1u;
  const int total = c.st_nf + c.st_nb;
  Sweep f, b;
  f.rec = c.st_frec;
  f.src = reinterpret_cast<const int4v*>(c.st_fsrc);
  f.sbr = b.sbr = res_of(c.st_sb, (unsigned)c.st_nsb * 512u);
  f.res = f.sbr;
  b.rec = c.st_brec;
  b.src = reinterpret_cast<const int4v*>(c.st_bsrc);
  b.res = res_of(c.z, (unsigned)c.np * 24u);
  f.polls = b.polls = polls;
  int gave_up = c.flags[kSweepErr];  // by an earlier launch
  while (true) {
    int t = 0;
    if (threadIdx.x == 0)
      t = __hip_atomic_fetch_add(c.st_ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t = __builtin_amdgcn_readfirstlane(t);
    if (t >= total) {
      // every workgroup makes one claim past the end; the last one resets
      if (t == total + (int)gridDim.x - 1 && threadIdx.x == 0) store_device(c.st_ticket, 0);
      return;
    }
    if (t < c.st_nf)
      strip_sweep<true, K, F32>(f, c.st_fptr[t], c.st_fptr[t + 1], lds, ringmask, gave_up);
    else
      strip_sweep<false, K, F32>(b, c.st_bptr[t - c.st_nf], c.st_bptr[t - c.st_nf + 1], lds,
                                 ringmask, gave_up);
    if (gave_up && threadIdx.x == 0) store_device(c.flags + kSweepErr, 1);
  }
}

// The factor into the records.  One lane per (sub-level, lane): its values
// v = 3 k + j (entry (r, j) of block k) in pairs, FP64 or rounded to FP32 in
// quads; rows past the strip and lane 3 get zeros.
template <class Sel>
__global__ void k_strip_pack(Sel sel) {
  const DevCloth c = sel.cloth();
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = id & 63;
  int sub = id >> 6;
  const bool fwd = sub < c.st_nsf;
  if (!fwd) sub -= c.st_nsf;
  if (!fwd && sub >= c.st_nsb) return;
  const int K = c.kpack, NB = strip_pairs(K), KH = strip_half(K), r = lane & 3;
  const int half = lane >> 2 & 1;
  const int i = r == 3 ? -1 : (fwd ? c.st_frow : c.st_brow)[sub * kStripRows + (lane >> 3)];
  char* rec = (fwd ? c.st_frec : c.st_brec) + (size_t)sub * (strip_pieces(fwd, K) * kPiece) +
              lane * 16;
  const int first = i < 0 ? 0 : (fwd ? c.rowptr[i] : c.diaind[i]) + half * KH;
  const int cnt = i < 0 ? 0 : min((fwd ? c.diaind[i] : c.rowptr[i + 1]) - first, KH);
  const double* src = c.fcrs + (size_t)first * 9;
  auto value = [&](int v) {
    const int k = v / 3, j = v - 3 * k;
    return k < cnt ? src[k * 9 + r * 3 + j] : 0.0;
  };
  if (c.precision) {
    for (int p = 0; p < strip_quads(K); p++)
      *reinterpret_cast<float4*>(rec + (1 + p) * kPiece) =
          make_float4((float)value(4 * p), (float)value(4 * p + 1), (float)value(4 * p + 2),
                      (float)value(4 * p + 3));
  } else {
    for (int p = 0; p < NB; p++)
      *reinterpret_cast<double2*>(rec + (1 + p) * kPiece) =
          make_double2(value(2 * p), value(2 * p + 1));
  }
  if (fwd) {
    const bool has = i >= 0 && half == 0;
    const double* d = c.fdia + (has ? (size_t)i * 9 + r * 3 : 0);
    *reinterpret_cast<double2*>(rec + (1 + NB) * kPiece) =
        has ? make_double2(d[0], d[1]) : make_double2(0.0, 0.0);
    *reinterpret_cast<double2*>(rec + (2 + NB) * kPiece) = make_double2(has ? d[2] : 0.0, 0.0);
  }
}

// The records' metadata and the import offsets from the plan's arrays (row and
// LDS offsets per slot, imported rows).  One thread per (sub-level, lane);
// lane l: row l / 8 of the sub-level, blocks 0 .. kh - 1 (l & 4 == 0) or
// kh .. k - 1, component l & 3 (3: none); import l / 4.
__global__ void k_strip_meta(DevCloth c, int fwd, const unsigned short* col, const int* import,
                             const int* bslot) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = id & 63, sub = id >> 6;
  if (sub >= (fwd ? c.st_nsf : c.st_nsb) + kStripTail) return;
  const int k = c.kpack, kh = strip_half(k), r = lane & 3, half = lane >> 2 & 1;
  const int slot = sub * kStripRows + (lane >> 3);
  const int i = (fwd ? c.st_frow : c.st_brow)[slot];
  const int j = import[sub * kStripImports + (lane >> 2)];
  // where component r of row n is in the sweep's result
  auto result = [&](int n) {
    return fwd ? (unsigned)((bslot[n] * 8 + r) * 8) : (unsigned)((3 * n + r) * 8);
  };
  int* src = const_cast<int*>(fwd ? c.st_fsrc : c.st_bsrc);
  src[((sub / kStripGroup) * 64 + lane) * kStripGroup + sub % kStripGroup] =
      (int)(r < 3 && j >= 0 ? result(j) : kStripNone);
  unsigned short w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int m = 0; m < kh && half * kh + m < k; m++) w[m] = col[(size_t)slot * k + half * kh + m];
  const unsigned out = r < 3 && half == 0 && i >= 0 ? result(i) : kStripNone;
  const int at = (kh + 1) / 2 * 2;
  w[at] = (unsigned short)(out & 0xffffu);
  w[at + 1] = (unsigned short)(out >> 16);
  char* rec = (fwd ? c.st_frec : c.st_brec) + (size_t)sub * (strip_pieces(fwd, k) * kPiece);
  __builtin_memcpy(rec + lane * 16, w, 16);
}

// st_sb as the first launch expects it: unwritten where a row's result goes,
// zero elsewhere; the tickets at zero; the rows of the slots
__global__ void k_strip_reset(DevCloth c) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e == 0) {
    c.st_ticket[0] = c.st_ticket[1] = 0;
    c.flags[kSweepErr] = 0;
  }
  if (e < (c.st_nsf + kStripTail) * kStripRows) {
    const int i = c.st_frow[e];
    int* m = const_cast<int*>(c.st_rows) + 8 * e;
    m[0] = i;
    m[1] = i < 0 ? 0 : c.rowptr[i];
    m[2] = i < 0 ? 0 : c.diaind[i] - c.rowptr[i];
    m[3] = i < 0 ? 0 : c.rowptr[i + 1] - c.rowptr[i];
    m[4] = i < 0 ? 0 : c.fu_ptr[i];
    m[5] = i < 0 ? 0 : c.fu_ptr[i + 1] - c.fu_ptr[i];
    m[6] = m[7] = 0;
  }
  if (e >= (c.st_nsb + kStripTail) * 64) return;
  const int lane = e & 63;
  c.st_sb[e] =
      (lane & 7) < 3 && c.st_brow[(e >> 6) * kStripRows + (lane >> 3)] >= 0 ? unwritten() : 0.0;
}

// ---------------------------------------------------------------------------
// Block ILU(0) by strips (ilu_sparse.cpp:387-401, 507-569), the strips of the
// forward sweep: two waves per strip, sixteen lanes per row, the eight rows of
// a sub-level at once.  A row's operations are ilu_row's (cs_solve.hip) in its
// order, as in k_ilu_factor_staged: the updates that share a lower block L_ik
// target distinct blocks and run at once, one per lane, with k ascending.
//
// The upper blocks of other rows are taken as they are finished, by the same
// strip or by others: fcrs holds "not written yet" before (k_strip_unwritten),
// each is stored with device scope, and the lane that needs one polls it.  (An
// upper block is always a product with D^-1, so it is never the marker.)
// Strips are claimed in order and wait only for strips claimed before; the two
// waves of a strip, which wait for each other, are one workgroup.  What does
// not depend on other rows (the row's place, its update list, its matrix
// blocks) is loaded one or two sub-levels ahead.
//
// What bounds it: per sub-level a store and a load of device scope, the up to
// eight dependent update rounds and the 3 x 3 inverse, about 5.5 us, times
// the levels (one workgroup walking the levels: 19 us each at 256^2).
constexpr int kFsLanes = 16;   // lanes per row
constexpr int kFsLayers = 2;   // updates a lane keeps in registers
constexpr int kFsBlocks = 2 * kMaxBlocksPerRow + 1;  // blocks of a row at most, the diagonal included
constexpr int kFsVals = (9 * kFsBlocks + kFsLanes - 1) / kFsLanes;
constexpr int kFsSlot = 9 * kFsBlocks + 2;  // doubles per row in LDS
constexpr int kFsThreads = kStripRows * kFsLanes;

// every off-diagonal block of the factor unwritten, no singular pivot seen
template <class Sel>
__global__ void k_strip_unwritten(Sel sel) {
  const DevCloth c = sel.cloth();
  const long n = 9L * c.nnz;
  const long stride = (long)gridDim.x * blockDim.x;
  const long e0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e0 == 0) c.flags[kNsing] = 0;
  for (long e = e0; e < n; e += stride) gstore(c.fcrs + e, unwritten());
  for (long e = e0; e < c.np; e += stride) gstore(c.ising + e, 0);
}

struct FsRow {  // a slot's row: where it is, its blocks and updates
  int i, rb, low, deg, u0, nu;
};
struct FsUpdates {
  int code[kFsLayers];  // lower block | target << 8, -1: none
  unsigned at[kFsLayers];  // byte offset of the upper block used
};

__device__ __forceinline__ FsRow fs_row(const DevCloth& c, int slot) {
  const auto p = (const __attribute__((address_space(1))) int4v*)c.st_rows + 2 * slot;
  const int4v a = p[0], b = p[1];
  return FsRow{a.x, a.y, a.z, a.w, b.x, b.y};
}
__device__ __forceinline__ void fs_updates(const DevCloth& c, const FsRow& r, int t,
                                           FsUpdates& u) {
#pragma unroll
  for (int m = 0; m < kFsLayers; m++) {
    const int e = t + m * kFsLanes;
    const bool has = e < r.nu;
    const int p = has ? r.u0 + e : 0;
    const int code = gptr(c.fu_code)[p], kj = gptr(c.fu_kj)[p];
    u.code[m] = has ? code : -1;
    u.at[m] = has ? 72u * (unsigned)kj : kStripNone;
  }
}
// the row's matrix blocks, then its diagonal block: value q on lane q % 16
__device__ __forceinline__ void fs_matrix(const DevCloth& c, const FsRow& r, int t,
                                          double (&v)[kFsVals]) {
  const int n = 9 * r.deg;
#pragma unroll
  for (int m = 0; m < kFsVals; m++) {
    const int q = t + m * kFsLanes;
    double x = 0.0;
    if (r.i >= 0 && q < n + 9)
      x = q < n ? gptr(c.crs)[(size_t)r.rb * 9 + q] : gptr(c.dia)[(size_t)r.i * 9 + (q - n)];
    v[m] = x;
  }
}
__device__ __forceinline__ void fs_block(__amdgpu_buffer_rsrc_t f, unsigned at, double (&u)[9]) {
#pragma unroll
  for (int q = 0; q < 9; q++) u[q] = res_load(f, at == kStripNone ? at : at + 8 * q);
}
__device__ __forceinline__ bool fs_missing(const double (&u)[9]) {
  bool w = false;
#pragma unroll
  for (int q = 0; q < 9; q++) w = w || not_yet(u[q]);
  return w;
}
// A_ij -= L_ik U_kj on the row in LDS (diagonal block after the others)
__device__ __forceinline__ void fs_apply(double* sl, int deg, int code, const double (&u)[9]) {
  const double* l = sl + (code & 0xff) * 9;
  const int tg = (code >> 8) & 0xff;
  double* a = sl + (tg == kFuDiag ? deg : tg) * 9;
#pragma unroll
  for (int r = 0; r < 3; r++) {
    const double l0 = l[r * 3 + 0], l1 = l[r * 3 + 1], l2 = l[r * 3 + 2];
    a[r * 3 + 0] -= l0 * u[0] + l1 * u[3] + l2 * u[6];
    a[r * 3 + 1] -= l0 * u[1] + l1 * u[4] + l2 * u[7];
    a[r * 3 + 2] -= l0 * u[2] + l1 * u[5] + l2 * u[8];
  }
}

template <class Sel>
__global__ __launch_bounds__(kFsThreads) void k_strip_factor(Sel sel, int polls_max) {
  const DevCloth c = sel.cloth();
  __shared__ double stage[kStripRows * kFsSlot];
  __shared__ int s_strip;
  const int grp = threadIdx.x / kFsLanes, t = threadIdx.x % kFsLanes;
  double* sl = stage + grp * kFsSlot;
  const __amdgpu_buffer_rsrc_t f = res_of(c.fcrs, (unsigned)c.nnz * 72u);
  if (threadIdx.x == 0)
    s_strip = __hip_atomic_fetch_add(c.st_ticket + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int strip = __builtin_amdgcn_readfirstlane(s_strip);
  // every workgroup makes one claim; the last one resets
  if (strip == (int)gridDim.x - 1 && threadIdx.x == 0) store_device(c.st_ticket + 1, 0);
  if (strip >= c.st_nf) return;
  const int first = c.st_fptr[strip], end = c.st_fptr[strip + 1];
  int gave_up = c.flags[kSweepErr];  // a strip before this one
  FsRow r = fs_row(c, first * kStripRows + grp), rn = fs_row(c, (first + 1) * kStripRows + grp);
  FsUpdates up;
  double av[kFsVals];
  fs_updates(c, r, t, up);
  fs_matrix(c, r, t, av);
  for (int sub = first; sub < end; sub++) {
    double u[kFsLayers][9];
#pragma unroll
    for (int m = 0; m < kFsLayers; m++) fs_block(f, up.at[m], u[m]);
    // ahead (past the strip's end: another strip's rows or the tail, unused)
    const FsRow rnn = fs_row(c, (sub + 2) * kStripRows + grp);
    FsUpdates upn;
    double avn[kFsVals];
    fs_updates(c, rn, t, upn);
    fs_matrix(c, rn, t, avn);
    const int nv = r.i >= 0 ? 9 * (r.deg + 1) : 0;
#pragma unroll
    for (int m = 0; m < kFsVals; m++)
      if (t + m * kFsLanes < nv) sl[t + m * kFsLanes] = av[m];
    int polls = 0;
    while (!gave_up && __builtin_amdgcn_ballot_w64(fs_missing(u[0]) || fs_missing(u[1])) != 0ull) {
      asm volatile("" ::: "memory");  // every poll loads again
#pragma unroll
      for (int m = 0; m < kFsLayers; m++)
        if (fs_missing(u[m])) fs_block(f, up.at[m], u[m]);
      gave_up = __builtin_amdgcn_readfirstlane(++polls >= polls_max);
    }
    wave_lds_sync();
    bool late = false;  // this lane gave up on an update beyond the registers
    for (int k = 0; k < r.low; k++) {
#pragma unroll
      for (int m = 0; m < kFsLayers; m++)
        if (up.code[m] >= 0 && (up.code[m] & 0xff) == k) fs_apply(sl, r.deg, up.code[m], u[m]);
      // updates beyond the registers (a closed strip of four columns has 35 per row)
      for (int e = t + kFsLayers * kFsLanes; e < r.nu; e += kFsLanes) {
        const int cd = gptr(c.fu_code)[r.u0 + e];
        if ((cd & 0xff) != k) continue;
        double x[9];
        int n = 0;
        do {
          asm volatile("" ::: "memory");
          fs_block(f, 72u * (unsigned)gptr(c.fu_kj)[r.u0 + e], x);
        } while (!gave_up && !late && fs_missing(x) && ++n < polls_max);
        late = late || n >= polls_max;
        fs_apply(sl, r.deg, cd, x);
      }
      wave_lds_sync();
    }
    if (__builtin_amdgcn_ballot_w64(late) != 0ull) gave_up = 1;
    double* d = sl + r.deg * 9;
    if (t == 0 && r.i >= 0) {
      const double det = +d[0] * d[4] * d[8] + d[3] * d[7] * d[2] + d[6] * d[1] * d[5] -
                         d[0] * d[7] * d[5] - d[6] * d[4] * d[2] - d[3] * d[1] * d[8];
      if (fabs(det) > 1.0e-30) {
        const double id = 1.0 / det;
        double w[9];
        for (int q = 0; q < 9; q++) w[q] = d[q];
        d[0] = id * (w[4] * w[8] - w[5] * w[7]);
        d[1] = id * (w[2] * w[7] - w[1] * w[8]);
        d[2] = id * (w[1] * w[5] - w[2] * w[4]);
        d[3] = id * (w[5] * w[6] - w[3] * w[8]);
        d[4] = id * (w[0] * w[8] - w[2] * w[6]);
        d[5] = id * (w[2] * w[3] - w[0] * w[5]);
        d[6] = id * (w[3] * w[7] - w[4] * w[6]);
        d[7] = id * (w[1] * w[6] - w[0] * w[7]);
        d[8] = id * (w[0] * w[4] - w[1] * w[3]);
      } else {
        gstore(c.ising + r.i, 1);
        atomicAdd(&c.flags[kNsing], 1);
      }
    }
    wave_lds_sync();
    // upper blocks first (others wait for them): D^-1 U, one block row each
    const int up_rows = r.i >= 0 ? 3 * (r.deg - r.low) : 0;
    for (int q = t; q < up_rows; q += kFsLanes) {
      const int b = q / 3, row = q - 3 * b;
      const double* w = sl + (r.low + b) * 9;
      const double d0 = d[row * 3], d1 = d[row * 3 + 1], d2 = d[row * 3 + 2];
      const unsigned at = 72u * (unsigned)(r.rb + r.low + b) + 24u * row;
      res_store(f, at, d0 * w[0] + d1 * w[3] + d2 * w[6]);
      res_store(f, at + 8, d0 * w[1] + d1 * w[4] + d2 * w[7]);
      res_store(f, at + 16, d0 * w[2] + d1 * w[5] + d2 * w[8]);
    }
    const int low = r.i >= 0 ? 9 * r.low : 0;
    for (int q = t; q < low; q += kFsLanes) res_store(f, 72u * (unsigned)r.rb + 8u * q, sl[q]);
    if (r.i >= 0 && t < 9) gstore(c.fdia + (size_t)r.i * 9 + t, d[t]);
    wave_lds_sync();  // the slot is reused by the next row
    r = rn;
    rn = rnn;
    up = upn;
#pragma unroll
    for (int m = 0; m < kFsVals; m++) av[m] = avn[m];
  }
  if (gave_up && (threadIdx.x & 63) == 0) store_device(c.flags + kSweepErr, 1);
}

// a single solve's right-hand side x (row order) into the records, z unwritten
__global__ void k_strip_rhs(DevCloth c, const double* x) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 3 * c.np) return;
  strip_put_rhs(c, e, x[e]);
}

// ---------------------------------------------------------------------------

bool strips_ok(const DevCloth& c) { return c.st_nf > 0 && c.sweep_variant != 1; }

// polls of one wait: kSpinMax, or fewer (0: every wait is given up) for tests
// of what follows a wait that was given up (CLOTHSIM_STRIP_POLLS)
static int wait_polls() {
  const char* e = getenv("CLOTHSIM_STRIP_POLLS");
  return e ? std::min(std::max(atoi(e), 0), kSpinMax) : kSpinMax;
}

int strip_record_bytes(bool fwd, int K) { return strip_pieces(fwd, K) * kPiece; }
int strip_rhs_offset(int K) { return (strip_pairs(K) + 2) * kPiece + 8; }

template <bool F32, class Sel>
static void launch_k(int k, dim3 grid, size_t lds, const Sel& sel, hipStream_t s) {
  const dim3 tb(64);
  const int polls = wait_polls();
  switch (k) {
    case 1: hipLaunchKernelGGL((k_strip_sweep<1, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 2: hipLaunchKernelGGL((k_strip_sweep<2, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 3: hipLaunchKernelGGL((k_strip_sweep<3, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 4: hipLaunchKernelGGL((k_strip_sweep<4, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 5: hipLaunchKernelGGL((k_strip_sweep<5, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 6: hipLaunchKernelGGL((k_strip_sweep<6, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    case 7: hipLaunchKernelGGL((k_strip_sweep<7, F32, Sel>), grid, tb, lds, s, sel, polls); break;
    default: hipLaunchKernelGGL((k_strip_sweep<8, F32, Sel>), grid, tb, lds, s, sel, polls); break;
  }
}

void launch_strip_sweep(const DevCloth& c, hipStream_t s) {
  const dim3 grid(std::max(c.st_nf, c.st_nb));
  const size_t lds = kStripZero + (size_t)c.st_ring * kStripSub;
  if (c.precision)
    launch_k<true>(c.kpack, grid, lds, One{c, {}}, s);
  else
    launch_k<false>(c.kpack, grid, lds, One{c, {}}, s);
}

void launch_strip_sweep_batch(const BatchView& b, hipStream_t s) {
  const dim3 grid(b.max_strips, b.n);
  const size_t lds = kStripZero + (size_t)b.max_ring * kStripSub;
  const Many m{b.tab, b.ptab};
  if (b.f32)
    launch_k<true>(b.kpack, grid, lds, m, s);
  else
    launch_k<false>(b.kpack, grid, lds, m, s);
}

bool strip_factor_ok(const DevCloth& c) { return c.st_nf > 0 && c.fu_blocks > 0; }

void launch_strip_factor(const DevCloth& c, hipStream_t s) {
  const unsigned fill = (unsigned)std::min<long>(2048, (9L * c.nnz + 255) / 256 + 1);
  hipLaunchKernelGGL(k_strip_unwritten<One>, dim3(fill), dim3(256), 0, s, One{c, {}});
  hipLaunchKernelGGL(k_strip_factor<One>, dim3(c.st_nf), dim3(kFsThreads), 0, s, One{c, {}},
                     wait_polls());
}

void launch_strip_factor_batch(const BatchView& b, hipStream_t s) {
  const Many m{b.tab, b.ptab};
  const unsigned fill = (unsigned)std::min<long>(256, (9L * b.max_nnz + 255) / 256 + 1);
  hipLaunchKernelGGL(k_strip_unwritten<Many>, dim3(fill, b.n), dim3(256), 0, s, m);
  hipLaunchKernelGGL(k_strip_factor<Many>, dim3(b.max_strips, b.n), dim3(kFsThreads), 0, s, m,
                     wait_polls());
}

int launch_strip_pack(const DevCloth& c, hipStream_t s) {
  const unsigned lanes = (unsigned)(c.st_nsf + c.st_nsb) * 64u;
  hipLaunchKernelGGL(k_strip_pack<One>, dim3((lanes + 255) / 256), dim3(256), 0, s, One{c, {}});
  CS_HIP(hipGetLastError());
  return kOk;
}

void launch_strip_pack_batch(const BatchView& b, hipStream_t s) {
  hipLaunchKernelGGL(k_strip_pack<Many>, dim3((unsigned)b.max_subs / 4, b.n), dim3(256), 0, s,
                     Many{b.tab, b.ptab});
}

int launch_strip_meta(const DevCloth& c, bool fwd, const unsigned short* col, const int* import,
                      const int* bslot, hipStream_t s) {
  const unsigned lanes = (unsigned)((fwd ? c.st_nsf : c.st_nsb) + kStripTail) * 64u;
  hipLaunchKernelGGL(k_strip_meta, dim3((lanes + 255) / 256), dim3(256), 0, s, c, fwd ? 1 : 0, col,
                     import, bslot);
  CS_HIP(hipGetLastError());
  return kOk;
}

int launch_strip_reset(const DevCloth& c, hipStream_t s) {
  const unsigned n = (unsigned)(std::max(c.st_nsf, c.st_nsb) + kStripTail) * 64u;
  hipLaunchKernelGGL(k_strip_reset, dim3((n + 255) / 256), dim3(256), 0, s, c);
  CS_HIP(hipGetLastError());
  return kOk;
}

void launch_strip_rhs(const DevCloth& c, const double* x, hipStream_t s) {
  hipLaunchKernelGGL(k_strip_rhs, dim3((3u * c.np + 255) / 256), dim3(256), 0, s, c, x);
}

}  // namespace cs
