// Host launchers of the implicit internal solve (cs_solve.hip).
#pragma once

#include "cs_device.hpp"

namespace cs {

// the packed (quad) sweep applies: packed factor, LDS ring proven safe,
// sub-level pointers fit
// the quad sweep addresses its operands with 32-bit byte offsets (at most
// 3 * np 16-byte pairs per array)
inline bool quad_ok(const DevCloth& c) {
  return c.kpack > 0 && c.ring_ok &&
         48LL * c.np < (1LL << 32);
}

// the quad sweep's workgroup waves and vector loads per wave per forward /
// backward sub-level; false when the row-by-row sweep runs instead
bool sweep_shape(const DevCloth& c, int* waves, int* loads_fwd, int* loads_bwd);
// blocks of a staged ILU row (the widest row plus the diagonal) that the
// staged factorisation can hold, 0 if a row is too wide for it
int ilu_stage_blocks(int widest_row);
int launch_bend_setup(const DevCloth& c, const Params& P, hipStream_t s);
// element kernels + gather assembly of A and b (after boundary conditions)
int launch_assemble(const DevCloth& c, const Params& P, hipStream_t s, Prof* prof = nullptr);
// block ILU(0) of the assembled system; *packed: the packed copies are stale,
// and with `solve` the one that this cloth's solve needs is made
int launch_ilu(const DevCloth& c, int* packed, bool solve, hipStream_t s, Prof* prof = nullptr);
// rearrange the factor for the packed sweeps (after any change of fdia/fcrs)
int launch_pack_factor(const DevCloth& c, hipStream_t s);
// sweeps by strips (cs_strips.hip): one wave per strip of rows.  strips_ok:
// the cloth's sweeps take them (the mesh fits and the row-by-row sweep is not
// selected)
bool strips_ok(const DevCloth& c);
int strip_record_bytes(bool fwd, int K);
int strip_rhs_offset(int K);
// the records' metadata and the import offsets from device copies of the plan
// (cs_strips.hpp: col and import of that sweep, slot of the backward one)
int launch_strip_meta(const DevCloth& c, bool fwd, const unsigned short* col, const int* import,
                      const int* bslot, hipStream_t s);
int launch_strip_pack(const DevCloth& c, hipStream_t s);   // the factor into the records
int launch_strip_reset(const DevCloth& c, hipStream_t s);  // before the first sweep, or after kSweepErr
void launch_strip_rhs(const DevCloth& c, const double* x, hipStream_t s);
void launch_strip_sweep(const DevCloth& c, hipStream_t s);
// block ILU(0) of the assembled system by strips (the pivot flags included)
void launch_strip_factor(const DevCloth& c, hipStream_t s);
bool strip_factor_ok(const DevCloth& c);
// which packed copies of the factor are current (they are made when a solve
// first needs them)
enum Packed : int { kPackedQuad = 1, kPackedStrips = 2 };
int ensure_packed(const DevCloth& c, bool strips, int* packed, hipStream_t s);
int launch_matvec(const DevCloth& c, double alpha, const double* x, double beta, double* y,
                  hipStream_t s);
// dst = (LU)^-1 src; with the strip sweeps dst must be c.z
int launch_ilu_apply(const DevCloth& c, const double* src, double* dst, int* packed,
                     hipStream_t s);
// the one-workgroup PCG solve (k_pcg_wg) applies to this cloth
bool pcg_wg_ok(const DevCloth& c);
// Solve_PCG from dx = 0 with r = b; poll convergence every `poll` iterations
// (the one-workgroup solve needs no poll)
int run_pcg(const DevCloth& c, double tol, int maxit, int* host_flags, int* packed, hipStream_t s,
            int poll, Prof* prof = nullptr);
// x[v] = rest[v] + off for the swept vertices
int launch_apply_sweep(const DevCloth& c, const int* verts, int n, const double off[3],
                       hipStream_t s);
// membrane and bending gradients only (UpdateIntermidiateVelocity)
int launch_gradients(const DevCloth& c, const Params& P, hipStream_t s);
int launch_finish_internal(const DevCloth& c, const Params& P, hipStream_t s);

// a batch of cloths as the batched kernels see it: device tables of the
// cloths' DevCloth and Params, and the largest sizes (grid extents)
struct BatchView {
  const DevCloth* tab;
  const Params* ptab;
  int n;
  int max_np, max_nt, max_nq, max_nnz, max_wmax;
  int max_qwidth, max_ncomp;  // widest sweep sub-level, most components of a cloth
  int max_fu_blocks;  // staged factorisation: blocks per row slot (0: some cloth cannot)
  bool piped;  // every cloth can use the packed (quad) sweep ...
  int kpack;   // ... with this many packed blocks per row
  bool wg;     // every cloth takes the one-workgroup PCG solve (one workgroup per cloth)
  bool f32;    // every cloth's packed sweep coefficients are FP32 (mixed precision)
  bool strips;  // every cloth's sweeps go by strips
  bool strip_factor;  // every cloth is factorised by strips
  int max_strips, max_ring, max_subs;  // most strips of a sweep, LDS ring sub-levels, sub-levels of both sweeps
  const int2* rowmap;  // the SpMV's blocks: (cloth, first row), kSpmvRows rows each
  int nrowblk;         // entries of rowmap
  const int2* vecmap;  // the vector update's blocks: (cloth, first of 3 np entries)
  int nvecblk;         // entries of vecmap
};
// rows per block of the batched SpMV and entries per block of the batched
// vector update (their block maps are built with these steps)
constexpr int kSpmvRows = 16;
constexpr int kVecBlock = 256;
// StepTime_InternalDynamicsILU for every cloth of the batch (start positions
// saved, assembly, ILU(0), PCG, x += dx, v = dx/dt); dgather/hgather hold n
// ints (device / pinned host) for the convergence poll
int batch_internal_step(const BatchView& b, double tol, int maxit, int poll, int* dgather,
                        int* hgather, hipStream_t s, Prof* prof = nullptr);
void launch_strip_sweep_batch(const BatchView& b, hipStream_t s);
void launch_strip_pack_batch(const BatchView& b, hipStream_t s);
void launch_strip_factor_batch(const BatchView& b, hipStream_t s);

}  // namespace cs
