// ostc_kernels.hpp -- host-side launcher declarations for the HIP kernels.
#pragma once
#include <algorithm>
#include "ostc_ops.hpp"
#include "ostc_parallel.hpp"

namespace ostc {

// per-block (reference-shaped) path, ostc_kernels_plain.hip
void plain_rhs(const DevBlock& B, const Params& P, hipStream_t st, long long* n);
void plain_update(const DevBlock& B, double dt, int rk, hipStream_t st, long long* n);
void plain_local_dt(const DevBlock& B, const Params& P, hipStream_t st, long long* n);
void min_reduce(const double* in, long long len, double* scratch, int n_first, hipStream_t st, long long* n);
void padded_pass(const DevBlock& B, int slot, int what, hipStream_t st, long long* n);
void count_pass(unsigned long long* pass, int lo, int hi, hipStream_t st, long long* n);
void sponge_mean(const DevBlock& B, const unsigned long long* iter, hipStream_t st, long long* n);
// n_wg workgroups of a launch; face_state: far-field or inflow ops among them
void ops_launch(const DevBlock* blocks, const DevOp* ops, const OpWg* wgs, int n_wg, bool face_state, int slot, int src,
                bool props, hipStream_t st, long long* n);
// parallel faces (ring slot 0): pack into / unpack from buf + f.offset
void par_pack(const DevBlock& B, const ParFace& f, double* buf, hipStream_t st);
void par_unpack(const DevBlock& B, const ParFace& f, const double* recv, const double* sent, hipStream_t st);
void store_last(const DevBlock& B, hipStream_t st);
void residual_partial(const DevBlock& B, double* out4, int nblk, hipStream_t st);

// dual time stepping + DPLUR on the per-block path, ostc_kernels_dual.hip
struct DualBlock {
  double* qn1;      // q^(n-1), 5 padded planes
  double* qn_star;  // J/(2 dt) (4 q^n - q^(n-1)), 5 interior planes
  double* sr;       // inviscid spectral radii along xi, eta, zeta, 3 interior planes
  double* dq0;      // dt dq / diag, 5 interior planes
  double* dqk;      // the DPLUR iterate, 5 interior planes
  double* last;     // rho, |V|, p, T of the last inner iteration, then their squared change
};
void dual_qn_star(const DevBlock& B, const DualBlock& D, double dt, hipStream_t st, long long* n);
void dual_pre(const DevBlock& B, const Params& P, const DualBlock& D, double dt, double diag_factor, hipStream_t st,
              long long* n);
void dual_dplur(const DevBlock& B, const DualBlock& D, double diag_factor, hipStream_t st, long long* n);
void dual_update(const DevBlock& B, hipStream_t st, long long* n);
void dual_last_store(const DevBlock& B, const DualBlock& D, hipStream_t st);
void dual_last_square(const DevBlock& B, const DualBlock& D, double* out4, int nblk, hipStream_t st);

// batched path, ostc_kernels_sweep.hip and ostc_kernels_fused.hip
struct FusedArgs {
  const DevBlock* blocks;
  const int* tile_block;     // block of each tile
  int n_tiles;
  int in, out;               // ring slots read / written
  double ra, rb, rc;         // SSP-RK3 coefficients of this stage
  const double* dt;          // device dt (bit pattern of a positive double)
  Params P;
  int xcd_remap;             // 1: contiguous tile chunks per XCD
  int target_block;          // >= 0: only this block's tiles (dq mode)
  int to_dq;                 // sweeps: the residual goes to the block's dq instead of res (sweep_launch)
};

struct TileShape { int tx, ty, tz, waves_per_eu; };  // waves_per_eu: occupancy hint given to the compiler
int fused_shape_count(int scheme);
TileShape fused_shape(int scheme, int index);
// Launches the tile kernels of table entry `index`; mode 0 = RK update,
// mode 1 = write dq only, mode 2 = RK update with the inviscid part in a kernel
// of its own.  Returns the dynamic LDS bytes used, or -1 (not a characteristic
// scheme, or a tile too large).
int fused_launch(int index, int mode, const FusedArgs& a, int n_wg, hipStream_t st);
int fused_lds_bytes(int scheme, int index);
// Work list of the inviscid sweeps (ostc_kernels_sweep.hip).  x: one workgroup
// per item, padded points `first` on of the block's interior rows; y, z: one
// wave per item, 64 columns from `first`, cells c0 .. c0 + n - 1 of each.
struct SweepItem { int block, first, c0, n; };
struct SweepPlan { const SweepItem* items[4]; int n[4]; };
bool sweep_scheme(int scheme);    // component-wise WENO: 50, 51, 71
int sweep_valid(int scheme);      // padded points a wave of the x sweep advances by
int visc_cells_per_wg();          // ... and a workgroup of the viscous kernel
void sweep_launch(FusedArgs a, const SweepPlan& s, bool update, hipStream_t st, long long* n);
// about n_wg workgroups over all blocks; max_cells: interior nodes of the largest
void dt_rows(const FusedArgs& a, int n_blocks, long long max_cells, int n_wg, double* dt_bits, hipStream_t st,
             long long* n);

// reverse mode, ostc_kernels_adjoint.hip
struct VjpArgs {
  int mx, my, mz, g, sx, sy;
  long long sz, n0;
  const double* cv;      // state the RHS was evaluated at (5 planes, padded)
  const double* bv;      // its primitives (6 planes, padded)
  const double* mul;     // its viscosity (padded)
  const double* jac;
  const double* met;
  const double* w;       // dq cotangent (5 planes, interior)
  double* lam;           // cv cotangent (5 planes, padded), accumulated
  double* fs;            // viscous face cotangents: 3 directions x 16 planes
  long long fs_stride;   // plane stride of fs, >= vjp_face_stride()
  double* gs;            // partial gathers of the viscous cotangents: 8 planes over [-1, m]^3
  long long gs_stride;   // plane stride of gs, >= vjp_gather_stride()
  Params P;
};
long long vjp_face_stride(int mx, int my, int mz);
long long vjp_gather_stride(int mx, int my, int mz);
void rhs_vjp(const VjpArgs& a, hipStream_t st, long long* n);
void adj_stage_pre(const DevBlock& B, double* lam, double* lam_qn, double* w, double ra, double rb, double cdt,
                   hipStream_t st);
void adj_stage_qn(const DevBlock& B, double* lam, double* lam_qn, hipStream_t st);
void adj_bc_ops(const DevBlock& B, const DevOp* ops, const OpWg* wgs, int n_wg, double* lam, hipStream_t st);

constexpr int kMaxModes = 64;
struct FourierModes {        // see ostc_fourier in abi.h
  int n;
  int comp[kMaxModes], kx[kMaxModes], kz[kMaxModes], trig[kMaxModes];
  double amp[kMaxModes];
  double y0, dx, dy, dz, lx, lz, delta, yc, du;
};
struct ThetaParams {         // see ostc_theta in abi.h
  double u1, u2, rho0, du, dy;
  int ni, nk;
};
void fourier_add(const DevBlock& B, const FourierModes& F, double* bv, hipStream_t st);
int fourier_grad_parts();
void fourier_grad(const DevBlock& B, const FourierModes& F, const double* lam, const double* cv, double* part,
                  double* grad, hipStream_t st);
void theta_eval(const DevBlock& B, const ThetaParams& T, const double* cv, double* rows, double* coef, double* theta,
                hipStream_t st);
void theta_seed(const DevBlock& B, const ThetaParams& T, const double* coef, double* lam, hipStream_t st);
// The momentum thickness with its row sums, coefficients and result in a
// file-scope device array (4 kThetaMaxRows + 1 doubles per GPU) instead of
// library-allocated memory; `scratch_ptr` comes from theta_scratch_ptr.
constexpr int kThetaMaxRows = 16384;
int theta_scratch_ptr(int device, double** scratch_ptr);

}  // namespace ostc
