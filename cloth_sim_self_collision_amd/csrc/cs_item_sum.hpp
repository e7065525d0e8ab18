// The left-to-right sum of cs_ordered_sum.hpp for sums whose running value
// changes binade often (the PCG's (r, z) products cancel by ten orders of
// magnitude): each tile is cut into items instead of having one summary.
//
// An item is one addend x added by itself (or +0), followed by a run of
// addends that are integers in the ulps of one binade.  Every tile predicts
// the running sum at each of its addends from approximate prefixes; an addend
// that takes the predicted sum into another binade, is a rounding tie or does
// not fit the binade's integers begins a new item as its x, and so does a
// change of the predicted binade.  Of a run the item holds the total N (as a
// double in units of the sum) and the least and greatest inclusive prefix.
//
// The chain then does two dependent additions per item, s += x and s += N,
// instead of walking the addends of every tile in which the binade changes.
// s += N equals the run's sequential additions when s lies in the run's binade
// and every prefix keeps it inside (see cs_ordered_sum.hpp; N is then exact
// and so is the addition).  Those conditions are tested for 64 items at a time
// from the s recorded at each; where one fails (a wrong prediction) the sum
// goes back to that item, whose x is a plain addition and always right, and
// the rest of its tile is walked from its addends.  Wrong predictions cost
// time, never accuracy.
//
// What bounds it: the chain on one wave, about 8 ns per item and 1.5 us per
// window of staged items (one summary per tile: 0.6 us per walker step and 6.5
// ns per addend near every binade change).  Measured, a PCG's reductions over
// their number, by events around the launches of one iteration: 256^2 sheet
// 160 -> 38 us, 128^2 75 -> 22 us, 61 x 96 drop 54 -> 12 us, 32^2 31 -> 10 us
// ((r, z) and (r, r) share a launch now).  In these solves one tile in
// 200 to 50000 is walked because a prediction missed.  cs_ordered_sum_noalloc
// keeps one summary per tile (k_sum_exact): its scratch is a small static array.
#pragma once

#include "cs_ordered_sum.hpp"

namespace cs {

constexpr int kItemCap = 256;  // items of a tile at most (more: the tile is walked)
constexpr int kItemWin = 512;  // items the chain stages at a time
constexpr int kItemPass = 4;   // items a lane stages at a time
constexpr int kItemNone = -2;  // code of an item without a run

// device scratch of one sum, kItemCap items per tile
struct SumItem {
  double x;        // added first
  double n;        // the run's total
  long long lo, hi;  // least and greatest prefix of the run, in ulps
  int code;        // sign and exponent the run needs, kItemNone: no run
  int elem;        // the run's first addend in the tile
};
static_assert(sizeof(SumItem) == 40, "items are stored and loaded in 8-byte words");

struct ItemShared {
  double wd[kSumWaves], wp[kSumWaves];
  long long wl[kSumWaves];
  int wi[kSumWaves], wc[kSumWaves];
  int last;
  alignas(16) double2 xn[kItemWin + 8];
  double mid[kItemWin + 8];  // the sum after each item's x
  long long lo[kItemWin], hi[kItemWin];
  long long start[kItemCap + 1];  // integer prefix at each item's run
  int code[kItemWin], elem[kItemWin];
  int at[64];  // first staged item of each tile of the window
  alignas(16) double buf[kSumBuf];
};

// Addend i of a job: t[i], or with kSelf and a dot product x[i] * y[i] formed
// where it is needed.  Sums of at most kSelfTiles tiles take kSelf: every tile
// adds up the tiles before it itself, which saves the launch of k_sum_tiles
// but costs the last tile about 2 us per tile before it.  Mean reduction of a
// PCG, with and without: 14.3 / 17.1 us at 2 tiles, 16.3 / 17.8 at 3, 20.0 /
// 18.5 at 5, 23.5 / 19.7 at 8, 40 / 25.6 at 18: the line lies between 3 and 5.
constexpr int kSelfTiles = 4;
template <bool kSelf>
__device__ __forceinline__ double sum_term(const SumJob& job, int i) {
  if (kSelf && job.x) return gload(job.x + i) * gload(job.y + i);
  return gload(job.t + i);
}

__device__ __forceinline__ int normal_code(double s) { return sum_normal(s) ? sign_exp(s) : -1; }
// exponent of a normal double from its sign_exp
__device__ __forceinline__ int code_exp(int code) { return (code & 0x7ff) - 1023; }

__device__ __forceinline__ double wave_incl_scan_f64(double x) {
  x = x + dpp_f64<0x111, 0xf>(x);
  x = x + dpp_f64<0x112, 0xf>(x);
  x = x + dpp_f64<0x114, 0xf>(x);
  x = x + dpp_f64<0x118, 0xf>(x);
  x = x + dpp_f64<0x142, 0xa>(x);
  x = x + dpp_f64<0x143, 0xc>(x);
  return x;
}
__device__ __forceinline__ int wave_scan_dpp32(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

// Items of tile b into sh (and their count, -1: more than kItemCap); the
// block calls it, kSumBlock threads of kSumPer consecutive addends each.
template <bool kSelf>
__device__ __forceinline__ int tile_items(const SumJob& job, int b, ItemShared& sh) {
  const int n = job.n;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const double two53 = 9007199254740992.0;
  const long long huge = 1LL << 60;
  const int e0 = b * kSumTile + tid * kSumPer;
  double x[kSumPer], loc[kSumPer];
  double run = 0.0;
#pragma unroll
  for (int j = 0; j < kSumPer; j++) {
    x[j] = e0 + j < n ? sum_term<kSelf>(job, e0 + j) : 0.0;
    run += x[j];
    loc[j] = run;
  }
  double p = 0.0;  // approximate sum of the tiles before
  if (kSelf)
    for (int j = tid; j < b * kSumTile; j += kSumBlock) p += sum_term<kSelf>(job, j);
  else
    for (int j = tid; j < b; j += kSumBlock) p += gload(job.w.tsum + j);
  p = wave_incl_scan_f64(p);
  const double incl = wave_incl_scan_f64(run);
  if (lane == 63) {
    sh.wp[wid] = p;
    sh.wd[wid] = incl;
  }
  __syncthreads();
  double base = 0.0;
#pragma unroll
  for (int w = 0; w < kSumWaves; w++) base += sh.wp[w];
#pragma unroll
  for (int w = 0; w < kSumWaves; w++)
    if (w < wid) base += sh.wd[w];
  base += incl - run;
  // predicted codes before and after each addend
  int cb[kSumPer], ca[kSumPer];
  long long q[kSumPer];
  bool single[kSumPer];
  int prev = normal_code(base);
#pragma unroll
  for (int j = 0; j < kSumPer; j++) {
    const bool real = e0 + j < n;
    cb[j] = prev;
    ca[j] = real ? normal_code(base + loc[j]) : prev;
    const double r = ldexp(x[j], 52 - code_exp(cb[j]));
    const double ri = rint(r);
    const bool conv = cb[j] >= 0 && ca[j] == cb[j] && fabs(r) < two53 && fabs(r - ri) != 0.5;
    single[j] = real && !conv;
    q[j] = conv ? (long long)ri : 0;
    prev = ca[j];
  }
  // the code after the addend before this thread's first
  int before = __shfl_up(ca[kSumPer - 1], 1, 64);
  if (lane == 63) sh.wc[wid] = ca[kSumPer - 1];
  __syncthreads();
  if (lane == 0) before = wid == 0 ? -3 : sh.wc[wid - 1];
  int flags = 0, nf = 0;
  long long sum = 0;
#pragma unroll
  for (int j = 0; j < kSumPer; j++) {
    const bool real = e0 + j < n;
    const int pc = j == 0 ? before : ca[j - 1];
    const bool f = single[j] || (real && pc != cb[j]);
    flags |= f ? 1 << j : 0;
    nf += f ? 1 : 0;
    sum = sum + q[j];
  }
  const int nfi = wave_scan_dpp32(nf);
  const long long si = wave_scan_dpp64(sum);
  if (lane == 63) {
    sh.wi[wid] = nfi;
    sh.wl[wid] = si;
  }
  __syncthreads();
  int id = nfi - nf - 1, count = 0;
  long long pre = si - sum, total = 0;
#pragma unroll
  for (int w = 0; w < kSumWaves; w++) {
    if (w < wid) {
      id += sh.wi[w];
      pre += sh.wl[w];
    }
    count += sh.wi[w];
    total += sh.wl[w];
  }
  if (count > kItemCap) return -1;  // the same on every thread
  const int id0 = id;
  const long long pre0 = pre;
#pragma unroll
  for (int j = 0; j < kSumPer; j++) {
    if (flags >> j & 1) {
      id++;
      sh.start[id] = pre;
      sh.xn[id].x = single[j] ? x[j] : 0.0;
      sh.code[id] = single[j] ? ca[j] : cb[j];
      sh.elem[id] = tid * kSumPer + j + (single[j] ? 1 : 0);
      sh.lo[id] = LLONG_MAX;
      sh.hi[id] = LLONG_MIN;
    }
    pre += q[j];
  }
  if (tid == 0) sh.start[count] = total;
  __syncthreads();
  // prefixes of the runs: a wave whose addends all belong to one run reduces
  // them first
  id = id0;
  pre = pre0;
  const int first = __builtin_amdgcn_readfirstlane(id0);
  const bool plain = (flags == 0 && id0 == first && e0 + kSumPer <= n);
  if (__builtin_amdgcn_ballot_w64(!plain) == 0ull && first >= 0) {
    long long mn = LLONG_MAX, mx = LLONG_MIN;
    const long long s0 = sh.start[first];
#pragma unroll
    for (int j = 0; j < kSumPer; j++) {
      pre += q[j];
      mn = min(mn, pre - s0);
      mx = max(mx, pre - s0);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mn = min(mn, (long long)__shfl_xor(mn, o, 64));
      mx = max(mx, (long long)__shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
      atomicMin(&sh.lo[first], mn);
      atomicMax(&sh.hi[first], mx);
    }
  } else {
#pragma unroll
    for (int j = 0; j < kSumPer; j++) {
      if (flags >> j & 1) id++;
      pre += q[j];
      if (e0 + j < n && !single[j]) {
        atomicMin(&sh.lo[id], pre - sh.start[id]);
        atomicMax(&sh.hi[id], pre - sh.start[id]);
      }
    }
  }
  __syncthreads();
  if (tid < count) {
    const long long lo = sh.lo[tid], hi = sh.hi[tid];
    const long long N = sh.start[tid + 1] - sh.start[tid];
    if (lo > hi) {
      sh.code[tid] = kItemNone;
      sh.xn[tid].y = 0.0;
    } else {
      sh.xn[tid].y = ldexp((double)N, code_exp(sh.code[tid]) - 52);
      sh.lo[tid] = max(lo, -huge);  // so that adding an integer view cannot wrap
      sh.hi[tid] = min(hi, huge);
    }
  }
  return count;
}

// the run's conditions on the sum s at its start
__device__ __forceinline__ bool run_applies(double s, int code, long long lo, long long hi) {
  const long long lo52 = (1LL << 52) + 1, hi53 = (1LL << 53) - 1;
  if (!sum_normal(s) || sign_exp(s) != code) return false;
  const long long S = (long long)ldexp(s, 52 - code_exp(code));
  return s > 0.0 ? (S + lo >= lo52 && S + hi <= hi53) : (S + lo >= -hi53 && S + hi <= -lo52);
}

// tile b from its addends, from addend `pos` of the tile on
template <bool kSelf>
__device__ __forceinline__ double walk_tile(double s, int b, int pos, const SumJob& job,
                                            double* buf, unsigned long long* stats) {
  const int begin = b * kSumTile, len = min(job.n, begin + kSumTile) - begin;
  if (len <= pos) return s;
#pragma unroll
  for (int r = 0; r < kSumTile / 64; r++) {
    const int i = r * 64 + ((int)threadIdx.x & 63);
    buf[i] = sum_term<kSelf>(job, begin + min(i, len - 1));
  }
  wave_lds_sync();
  s = wave_walk(buf, len, s, stats, pos);
  wave_lds_sync();
  return s;
}

// adds count items (padded with zeros to a multiple of 8) onto s
__device__ __forceinline__ double add_items(double s, int count, ItemShared& sh) {
  double2 w[8];
#pragma unroll
  for (int j = 0; j < 8; j++) w[j] = sh.xn[j];
  for (int q = 0; q < count; q += 8) {
    double2 v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = sh.xn[min(q + 8 + j, kItemWin + 7)];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      s = s + w[j].x;
      sh.mid[q + j] = s;  // every lane the same value
      s = s + w[j].y;
    }
#pragma unroll
    for (int j = 0; j < 8; j++) w[j] = v[j];
  }
  return s;
}

// The sum of the tiles from their items, on one wave (every lane holds s).
// Windows of 64 tiles, one per lane; `walked` counts the tiles walked.
template <bool kSelf>
__device__ __forceinline__ double chain_items(const SumJob& job, ItemShared& sh, int& walked) {
  const SumItem* items = job.w.items;
  const int* counts = job.w.code;
  unsigned long long* stats = job.w.stats;
  const int lane = threadIdx.x & 63, nt = sum_tiles(job.n);
  double s = 0.0;
  int bb = 0;
  while (bb < nt && !isnan(s)) {
    const int k = bb + lane;
    const bool in = k < nt;
    const SumItem* it = items + (size_t)min(k, nt - 1) * kItemCap;
    const int cnt = in ? load_device(counts + k) : 0;
    int f = 0;  // leading tiles applied at once: one run each, all in one binade
    if (__builtin_amdgcn_ballot_w64(in && cnt == 1) & 1ull) {
      const bool one = in && cnt == 1;
      const double x = one ? load_device(&it->x) : 1.0;
      const double nd = one ? load_device(&it->n) : 0.0;
      const long long lo = one ? load_device(&it->lo) : 0, hi = one ? load_device(&it->hi) : 0;
      const int code = one ? load_device(&it->code) : -1;
      if (sum_normal(s)) {
        const int c = sign_exp(s), e = code_exp(c);
        const bool same = one && x == 0.0 && code == c;
        const long long N = same ? (long long)ldexp(nd, 52 - e) : 0;
        const long long S = (long long)ldexp(s, 52 - e);
        const long long incl = wave_scan_dpp64(N), at = S + incl - N;
        const long long lo52 = (1LL << 52) + 1, hi53 = (1LL << 53) - 1;
        const bool ok = same && (s > 0.0 ? (at + lo >= lo52 && at + hi <= hi53)
                                         : (at + lo >= -hi53 && at + hi <= -lo52));
        const unsigned long long bad = __builtin_amdgcn_ballot_w64(!ok);
        f = bad ? __ffsll((long long)bad) - 1 : 64;
        if (f > 0) s = ldexp((double)(S + readlane64(incl, f - 1)), e - 52);
      }
    }
    if (f >= 8 || bb + f >= nt) {  // worth a window of its own
      bb += f;
      continue;
    }
    // the items of the next tiles, as many as fit, up to a tile without items
    const int use = lane >= f && in ? cnt : 0;
    const int incl = wave_scan_dpp32(max(use, 0));
    const unsigned long long stop =
        __builtin_amdgcn_ballot_w64(!in || (lane >= f && (cnt < 0 || incl > kItemWin)));
    const int g = stop ? __ffsll((long long)stop) - 1 : 64;  // tiles bb + f .. bb + g - 1
    if (g == f) {  // (a tile has at most kItemCap < kItemWin items: this one has none)
      s = walk_tile<kSelf>(s, bb + f, 0, job, sh.buf, stats);
      walked++;
      bb += f + 1;
      continue;
    }
    const int total = __builtin_amdgcn_readlane(incl, g - 1);
    const int mine = lane >= f && lane < g ? cnt : 0, at = incl - max(use, 0);
    // staged side by side: lane l takes the items l, l + 64, ..., whose tiles
    // it finds in the list of the tiles' first items; every load of a pass is
    // issued before its first store
    sh.at[lane] = lane < g ? at : INT_MAX;
    wave_lds_sync();
    for (int q0 = lane; q0 < total; q0 += 64 * kItemPass) {
      int src[kItemPass];
#pragma unroll
      for (int u = 0; u < kItemPass; u++) {
        const int q = min(q0 + 64 * u, total - 1);
        int l = 0;  // the last tile whose first item is at most q
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) l += sh.at[l + o] <= q ? o : 0;
        src[u] = (bb + l) * kItemCap + (q - sh.at[l]);
      }
      double x[kItemPass], nd[kItemPass];
      long long lo[kItemPass], hi[kItemPass], ce[kItemPass];
#pragma unroll
      for (int u = 0; u < kItemPass; u++) {
        const SumItem* i = items + src[u];
        x[u] = load_device(&i->x);
        nd[u] = load_device(&i->n);
        lo[u] = load_device(&i->lo);
        hi[u] = load_device(&i->hi);
        ce[u] = load_device(reinterpret_cast<const long long*>(&i->code));
      }
#pragma unroll
      for (int u = 0; u < kItemPass; u++) {
        const int d = min(q0 + 64 * u, total - 1);  // past the end: the last item again
        sh.xn[d] = make_double2(x[u], nd[u]);
        sh.lo[d] = lo[u];
        sh.hi[d] = hi[u];
        sh.code[d] = (int)ce[u];
        sh.elem[d] = (int)(ce[u] >> 32);
      }
    }
    if (lane < 8) sh.xn[total + lane] = make_double2(0.0, 0.0);
    wave_lds_sync();
    s = add_items(s, total, sh);
    wave_lds_sync();
    int fail = -1;
    for (int q0 = 0; q0 < total && fail < 0; q0 += 64) {
      const int q = q0 + lane;
      bool ok = true;
      if (q < total) {
        const int code = sh.code[q];
        ok = code == kItemNone || run_applies(sh.mid[q], code, sh.lo[q], sh.hi[q]);
      }
      const unsigned long long bad = __builtin_amdgcn_ballot_w64(!ok);
      if (bad) fail = q0 + __ffsll((long long)bad) - 1;
    }
    if (fail < 0) {
      bb += g;
      continue;
    }
    // back to the failing item: its x was added, its run is walked
    s = sh.mid[fail];
    const unsigned long long own =
        __builtin_amdgcn_ballot_w64(mine > 0 && at <= fail && fail < at + mine);
    const int l = __ffsll((long long)own) - 1;
    const int elem = __builtin_amdgcn_readfirstlane(sh.elem[fail]);
    s = walk_tile<kSelf>(s, bb + l, elem, job, sh.buf, stats);
    walked++;
    bb += l + 1;
  }
  return s;
}

// Tile items, then the chain in the last block of the job to finish;
// src.finish(s) runs on one thread with the exact sum.  Same grid as
// k_sum_tiles, which runs before it unless kSelf.
template <class Src, bool kSelf>
__global__ __launch_bounds__(kSumBlock) void k_sum_items(Src src) {
  const SumJob job = src.job();
  if (job.skip && *job.skip) return;
  const SumScratch& w = job.w;
  const int b = blockIdx.x, nt = sum_tiles(job.n), tid = threadIdx.x;
  if (b >= nt) return;
  __shared__ ItemShared sh;
  {
    const int count = tile_items<kSelf>(job, b, sh);
    if (tid < count) {
      SumItem* i = w.items + (size_t)b * kItemCap + tid;
      store_device(&i->x, sh.xn[tid].x);
      store_device(&i->n, sh.xn[tid].y);
      store_device(&i->lo, sh.lo[tid]);
      store_device(&i->hi, sh.hi[tid]);
      store_device(reinterpret_cast<long long*>(&i->code),
                   (long long)(unsigned)sh.code[tid] | (long long)sh.elem[tid] << 32);
    }
    if (tid == 0) store_device(w.code + b, count);
    // stored and read with device-scope accesses and complete before the
    // ticket is taken: no device-scope fence (k_sum_exact)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) sh.last = atomicAdd(w.ticket, 1u) == (unsigned)(nt - 1);
  }
  __syncthreads();
  if (!sh.last || tid >= 64) return;
  const unsigned long long chain_t0 = w.stats ? wall_clock64() : 0;
  if (tid == 0) store_device(w.ticket, 0u);
  int walked = 0;
  const double s = chain_items<kSelf>(job, sh, walked);
  if (tid == 0) {
    src.finish(s);
    if (w.stats) {
      atomicAdd(w.stats + kStatSums, 1ull);
      atomicAdd(w.stats + kStatTiles, (unsigned long long)nt);
      atomicAdd(w.stats + kStatFast, (unsigned long long)(nt - walked));
      atomicAdd(w.stats + kStatChainTicks, wall_clock64() - chain_t0);
    }
  }
}

// jobs = grid rows, sums = sums per job (blockIdx.z); max_n = the largest job's
// length; the jobs' scratch has items
template <class Src>
inline void launch_item_sum(const Src& src, int max_n, int jobs, hipStream_t stream,
                            int sums = 1) {
  const dim3 grid(sum_tiles(max_n), jobs, sums);
  if (sum_tiles(max_n) <= kSelfTiles) {
    hipLaunchKernelGGL((k_sum_items<Src, true>), grid, dim3(kSumBlock), 0, stream, src);
    return;
  }
  hipLaunchKernelGGL(k_sum_tiles<Src>, grid, dim3(kSumBlock), 0, stream, src);
  hipLaunchKernelGGL((k_sum_items<Src, false>), grid, dim3(kSumBlock), 0, stream, src);
}

}  // namespace cs
