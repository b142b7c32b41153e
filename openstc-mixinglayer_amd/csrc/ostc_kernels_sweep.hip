// ostc_kernels_sweep.hip -- the component-wise inviscid residual of every
// block of a batched stage (WENO5-JS 50, WENO-Z5 51, WENO-Z7 71) as three
// sweeps without workgroup barriers: dq = s - dFx, then dq -= dFy, then
// dq -= dFz, in the reference's order (src/RK.cuh:113-139), s the sponge term;
// then the viscous fluxes and the RK update.  A step leaves the block's dq
// array alone: between the kernels dq lies in planes of its own (a.to_dq: in
// the array).  In the primitives of the slot that the stage writes, which are
// free until then, its rows would be padded, and cut lines: 24 blocks 2 % slower.
//
// One tile kernel per stage did all of this with dq in registers (24 blocks,
// 12.5 M nodes: 4.5 ms a stage).  It moved the fewest bytes, but it waited half
// of its time: six staging phases with workgroup barriers, the split fluxes of
// a point evaluated 6.4 times, a third of its instructions spent on indexes.
// Here a wave depends on no other wave.  The price is dq, stored and read
// between the kernels (0.3 KB a node and stage).  Measured on the same case:
// x sweep 0.43 ms (4.1 TB/s), y 0.59 (5.0), z 0.55 (5.2), viscous + update 1.40
// (6.9 GB, 4.9 TB/s); when they took the tile kernel's place the step went from
// 14.4 to 10.1 ms (10.2 in the present rounding), 16^3 nodes from 114 to 111 us,
// 101x75x49 nodes with WENO-Z7 from 603 to 495 us.
#include "ostc_stage.hpp"

namespace ostc {

namespace {

// The five split fluxes along metric row k at one point and its
// Jacobian-weighted metric row (src/WENO.cu:697-720).
struct SplitPoint { double fp[5], fm[5], mj[3]; };

struct PointIn { double q[5], p, t, k[3], jac; };

template <int D>
__device__ __forceinline__ PointIn load_point(const StageBlock& B, int o) {
  PointIn I;
  const int s = B.sz;
  const unsigned b = 8u * (unsigned)o;
#pragma unroll
  for (int l = 0; l < 5; ++l) I.q[l] = ld(B.cvi + l * s, b);
  I.p = ld(B.bvi + 4 * s, b);
  I.t = ld(B.bvi + 5 * s, b);
#pragma unroll
  for (int c = 0; c < 3; ++c) I.k[c] = ld(B.met + (3 * D + c) * s, b);
  I.jac = ld(B.jac, b);
  return I;
}

// In the reference's order and rounding (lf_split5), with the short quotient
// and roots.  Products of J / 2 with U, lambda and p rounded first, a rounded
// reciprocal of rho and fused sums save a third of the instructions (16^3
// nodes 68.1 -> 66.5 us, 24 blocks 10.20 -> 10.11 ms), but the transverse
// velocities of a step are then 6 to 12 % further from 64-bit whole-array
// arithmetic.
__device__ __forceinline__ SplitPoint split_point(const PointIn& I) {
  SplitPoint S;
  const double U = div64(I.q[1] * I.k[0] + I.q[2] * I.k[1] + I.q[3] * I.k[2], I.q[0]);
  const double c_grad = sqrt64(kGamma * kRAir * I.t) * sqrt64(I.k[0] * I.k[0] + I.k[1] * I.k[1] + I.k[2] * I.k[2]);
  const double lambda = fabs(U) + c_grad, hj = 0.5 * I.jac;
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    const double f = l == 0 ? U * I.q[0] : (l == 4 ? U * (I.q[4] + I.p) : U * I.q[l] + I.p * I.k[l - 1]);
    S.fp[l] = hj * (f + lambda * I.q[l]);
    S.fm[l] = hj * (f - lambda * I.q[l]);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) S.mj[c] = I.k[c] * I.jac;
  return S;
}

// The WENO epsilon of rho, the momenta and the energy (src/WENO.cu:1469-1482).
__device__ __forceinline__ void face_eps(const Params& P, const double* a, const double* b, double e[3]) {
  weno_eps(P, a[0], a[1], a[2], b[0], b[1], b[2], e);
}

}  // namespace

// x sweep.  A wave takes 64 consecutive padded points of a block's interior
// rows (whole cache lines, rows of any length), each lane one split-flux
// point; the split fluxes go through the wave's own LDS words, each lane then
// forms the face to its right and gets the one to its left from the next lane.
// 64 - 2R lanes update their cell: the halo is 10 % for WENO-Z5 instead of the
// 37 % of a 16-cell tile, and no wave waits for another.
template <int SCHEME>
__global__ __launch_bounds__(256) void k_sweep_x(FusedArgs A, const SweepItem* items) {
  constexpr int R = Stencil<SCHEME>::R, W = Stencil<SCHEME>::W, VALID = 64 - 2 * R;
  __shared__ double lds[4][13][64];
  const SweepItem it = items[blockIdx.x];
  if (A.target_block >= 0 && it.block != A.target_block) return;
  const StageBlock B = stage_block(A.blocks[it.block], A.in, A.out);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = B.sx * B.my * B.mz;
  const int qf = it.first + wave * VALID + lane, qc = min(qf, n - 1);
  const int row = qc / B.sx, ii = qc - row * B.sx, k = row / B.my, j = row - k * B.my, i = ii - B.g;
  const int o = poff(B, i, j, k);
  double(*L)[64] = lds[wave];
  {
    const SplitPoint S = split_point(load_point<0>(B, o));
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      L[l][lane] = S.fp[l];
      L[5 + l][lane] = S.fm[l];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) L[10 + c][lane] = S.mj[c];
  }
  // a wave's LDS accesses complete in order; the compiler must keep that order
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int c = min(max(lane, R - 1), 63 - R);  // lanes without a face repeat a neighbour's
  double e[3];
  {
    const double a[3] = {L[10][c], L[11][c], L[12][c]}, b[3] = {L[10][c + 1], L[11][c + 1], L[12][c + 1]};
    face_eps(A.P, a, b, e);
  }
  double diff[5];
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    double vp[W], vm[W];
#pragma unroll
    for (int r = 0; r < W; ++r) {
      vp[r] = L[l][c - W / 2 + r];
      vm[r] = L[5 + l][c - W / 2 + 1 + r];
    }
    const double f = weno_face<SCHEME>(vp, vm, e[l == 0 ? 0 : (l == 4 ? 2 : 1)]);
    diff[l] = f - __shfl_up(f, 1, 64);
  }
  if (lane < R || lane > 63 - R || qf >= n || i < 0 || i >= B.mx) return;
  const gptr<double> res = A.to_dq ? B.dq : B.res;
  const int q0 = (k * B.my + j) * B.mx + i, n0 = (int)B.n0, s = B.sz;
  if (B.sp_sigma) {
    // sponge_layer_source (src/SpongeLayer.cu:68-160), the first term of the
    // stage's dq as in compute_source: dq -= sigma (cv - mean)
    const double sigma = B.sp_jac ? B.sp_sigma[q0] * B.jac[o] : B.sp_sigma[q0];
#pragma unroll
    for (int l = 0; l < 5; ++l)
      res[q0 + l * n0] = (0.0 - sigma * (B.cvi[o + l * s] - B.sp_mean[q0 + l * n0])) - diff[l];
  } else {
#pragma unroll
    for (int l = 0; l < 5; ++l) st(res + l * n0, 8u * (unsigned)q0, 0.0 - diff[l]);
  }
}

// y (D = 1) and z (D = 2) sweeps.  A wave takes 64 columns, consecutive in i
// (then in the third index), and marches along D over the item's cells: each
// step reads one point per lane, splits its fluxes once, and forms one face
// from the last 2R points, which stay in registers.  No LDS, no barrier, and
// a point is split once (plus 2R at the ends of an item) where the tiles of
// k_fused split it 2.5 times along each of y and z.
template <int D, int SCHEME>
__global__ __launch_bounds__(64, 2) void k_sweep_march(FusedArgs A, const SweepItem* items) {
  constexpr int R = Stencil<SCHEME>::R, W = Stencil<SCHEME>::W;
  const SweepItem it = items[blockIdx.x];
  if (A.target_block >= 0 && it.block != A.target_block) return;
  const StageBlock B = stage_block(A.blocks[it.block], A.in, A.out);
  const gptr<double> res = A.to_dq ? B.dq : B.res;
  const int third = D == 1 ? B.mz : B.my, n0 = (int)B.n0;
  const int col = it.first + (int)threadIdx.x, cc = min(col, B.mx * third - 1);
  const bool store = col == cc;
  const int i = cc % B.mx, a = cc / B.mx;
  const int step = D == 1 ? B.sx : B.sx * B.sy, dstep = D == 1 ? B.mx : B.mx * B.my;
  int o = D == 1 ? poff(B, i, it.c0 - R, a) : poff(B, i, a, it.c0 - R);  // next point to load
  int q = D == 1 ? (a * B.my + it.c0) * B.mx + i : (it.c0 * B.my + a) * B.mx + i;  // next cell to update
  double fp[5][W + 1], fm[5][W];  // points t-W..t of F+, t-W+1..t of F-
  double mj[R + 1][3];            // Jacobian-weighted metric rows of t-R..t
  double left[5];
  // Z5, JS: the next point is loaded a step ahead and the march is unrolled
  // over one turn of the window, so the window never moves (228 VGPRs); Z7's
  // window leaves no registers for either (252 VGPRs without, 56 spilled with).
  constexpr bool PREFETCH = W == 5;
  constexpr int TURN = PREFETCH ? W + 1 : 1;
  PointIn next;
  if constexpr (PREFETCH) next = load_point<D>(B, o);
  auto push = [&](const SplitPoint& S) {
#pragma unroll
    for (int l = 0; l < 5; ++l) {
#pragma unroll
      for (int r = 0; r < W; ++r) fp[l][r] = fp[l][r + 1];
      fp[l][W] = S.fp[l];
#pragma unroll
      for (int r = 0; r + 1 < W; ++r) fm[l][r] = fm[l][r + 1];
      fm[l][W - 1] = S.fm[l];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int r = 0; r < R; ++r) mj[r][c] = mj[r + 1][c];
      mj[R][c] = S.mj[c];
    }
  };
  auto advance = [&](bool more) {
    if constexpr (PREFETCH) {
      const PointIn cur = next;
      if (more) {
        o += step;
        next = load_point<D>(B, o);
      }
      push(split_point(cur));
    } else {
      push(split_point(load_point<D>(B, o)));
      o += step;
    }
    // keep the scheduler from mixing the steps of the unrolled march: their
    // loads and faces would all be live at once (340 bytes of scratch a lane)
    __builtin_amdgcn_sched_barrier(0);
  };
  auto face = [&](double* f) {
    double e[3];
    face_eps(A.P, mj[0], mj[1], e);
#pragma unroll
    for (int l = 0; l < 5; ++l) f[l] = weno_face<SCHEME>(fp[l], fm[l], e[l == 0 ? 0 : (l == 4 ? 2 : 1)]);
  };
#pragma unroll
  for (int r = 0; r < 2 * R; ++r) advance(true);
  face(left);
#pragma unroll TURN
  for (int c = 0; c < it.n; ++c) {
    double dq[5];
#pragma unroll
    for (int l = 0; l < 5; ++l) dq[l] = ld(res + l * n0, 8u * (unsigned)q);
    advance(c + 1 < it.n);
    double f[5];
    face(f);
#pragma unroll
    for (int l = 0; l < 5; ++l) {
      if (store) st(res + l * n0, 8u * (unsigned)q, dq[l] - (f[l] - left[l]));
      left[l] = f[l];
    }
    q += dstep;
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ------------------------------------------- viscous fluxes and RK update

// The value of the next / the previous lane (the end lanes keep their own):
// a whole-wave shift by one lane in the VALU, no LDS.
__device__ __forceinline__ double lane_after(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  v.x = __builtin_amdgcn_update_dpp(v.x, v.x, 0x130, 0xf, 0xf, false);
  v.y = __builtin_amdgcn_update_dpp(v.y, v.y, 0x130, 0xf, 0xf, false);
  return __builtin_bit_cast(double, v);
}
__device__ __forceinline__ double lane_before(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  v.x = __builtin_amdgcn_update_dpp(v.x, v.x, 0x138, 0xf, 0xf, false);
  v.y = __builtin_amdgcn_update_dpp(v.y, v.y, 0x138, 0xf, 0xf, false);
  return __builtin_bit_cast(double, v);
}

namespace {

struct V4 { double v[4]; };                       // u, v, w, T
struct Geo { double met[9], jac, mu; };

__device__ __forceinline__ V4 load_v4(const StageBlock& B, int o) {
  const int s = B.sz;
  const unsigned b = 8u * (unsigned)o;
  return V4{{ld(B.bvi + s, b), ld(B.bvi + 2 * s, b), ld(B.bvi + 3 * s, b), ld(B.bvi + 5 * s, b)}};
}
__device__ __forceinline__ Geo load_geo(const StageBlock& B, int o) {
  Geo G;
  const unsigned b = 8u * (unsigned)o;
#pragma unroll
  for (int c = 0; c < 9; ++c) G.met[c] = ld(B.met + c * B.sz, b);
  G.jac = ld(B.jac, b);
  G.mu = ld(B.muli, b);
  return G;
}
__device__ __forceinline__ V4 minus(const V4& a, const V4& b) {
  V4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r.v[q] = a.v[q] - b.v[q];
  return r;
}
__device__ __forceinline__ V4 along_x(const V4& f) {  // f(i+1) - f(i-1)
  V4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r.v[q] = lane_after(f.v[q]) - lane_before(f.v[q]);
  return r;
}
__device__ __forceinline__ V4 after(const V4& f) {
  V4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r.v[q] = lane_after(f.v[q]);
  return r;
}
__device__ __forceinline__ Geo after(const Geo& g) {
  Geo r;
#pragma unroll
  for (int c = 0; c < 9; ++c) r.met[c] = lane_after(g.met[c]);
  r.jac = lane_after(g.jac);
  r.mu = lane_after(g.mu);
  return r;
}

// Viscous flux of the face of direction D between cells a (lower) and b
// (src/ViscousScheme.cuh:23-909): their values, their central differences
// p(i+1) - p(i-1) along the two other directions E1 < E2, and their geometry.
// Products and sums may be contracted: the viscous fluxes are a small part of
// the residual and are not differences of large terms.
template <int D>
__device__ __forceinline__ V4 visc_face(const V4& fa, const V4& fb, const V4& a1, const V4& b1, const V4& a2,
                                        const V4& b2, const Geo& ga, const Geo& gb, double prandtl) {
#pragma clang fp contract(fast)
  constexpr int E1 = D == 0 ? 1 : 0, E2 = D == 2 ? 1 : 2;
  double m[9], k[3];
#pragma unroll
  for (int c = 0; c < 9; ++c) m[c] = ga.met[c] + gb.met[c];
#pragma unroll
  for (int c = 0; c < 3; ++c) k[c] = 0.5 * (ga.met[3 * D + c] * ga.jac + gb.met[3 * D + c] * gb.jac);
  double g[4][3];  // physical gradients of u, v, w, T; m holds twice the face metric
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const double d = 0.5 * (fb.v[q] - fa.v[q]), e1 = 0.125 * (a1.v[q] + b1.v[q]), e2 = 0.125 * (a2.v[q] + b2.v[q]);
#pragma unroll
    for (int c = 0; c < 3; ++c) g[q][c] = d * m[3 * D + c] + e1 * m[3 * E1 + c] + e2 * m[3 * E2 + c];
  }
  const double mu = 0.5 * (ga.mu + gb.mu), mu2 = mu + mu;
  const double third = (g[0][0] + g[1][1] + g[2][2]) * (1.0 / 3.0);
  const double xx = mu2 * (g[0][0] - third), yy = mu2 * (g[1][1] - third), zz = mu2 * (g[2][2] - third);
  const double xy = mu * (g[0][1] + g[1][0]), xz = mu * (g[0][2] + g[2][0]), yz = mu * (g[1][2] + g[2][1]);
  V4 f;
  f.v[0] = k[0] * xx + k[1] * xy + k[2] * xz;
  f.v[1] = k[0] * xy + k[1] * yy + k[2] * yz;
  f.v[2] = k[0] * xz + k[1] * yz + k[2] * zz;
  constexpr double cp{kGamma * kRu / kMwAir / (kGamma - 1)};
  const double heat = mu * (cp / prandtl) * (k[0] * g[3][0] + k[1] * g[3][1] + k[2] * g[3][2]);
  f.v[3] = 0.5 * ((fa.v[0] + fb.v[0]) * f.v[0] + (fa.v[1] + fb.v[1]) * f.v[1] + (fa.v[2] + fb.v[2]) * f.v[2]) + heat;
  return f;
}

// update_cv_and_bv_rk<Air> (src/RK.cuh:230-284) and the interior part of
// update_physical_properties<Air> (src/FieldOperation.cuh:107-140) at padded
// offset p, in the order and rounding of the per-block update (fused sums and
// rounded reciprocals: density 20 % further from 64-bit whole-array arithmetic,
// and no faster).
__device__ __forceinline__ void stage_update(const FusedArgs& A, const StageBlock& B, int p, double dt, double jac,
                                             const double dq[5]) {
  const int s = B.sz;
  const unsigned b = 8u * (unsigned)p;
  const double dt_div_jac = div64(dt, jac);
  double c[5];
#pragma unroll
  for (int l = 0; l < 5; ++l) {
    c[l] = A.ra * ld(B.qn + l * s, b) + A.rb * ld(B.cvi + l * s, b) + A.rc * dt_div_jac * dq[l];
    st(B.cvo + l * s, b, c[l]);
  }
  const double density_inv = div64(1.0, c[0]);
  const double u = c[1] * density_inv, v = c[2] * density_inv, w = c[3] * density_inv;
  const double V2 = u * u + v * v + w * w;
  const double pr = (kGamma - 1) * (c[4] - 0.5 * c[0] * V2);
  const double T = div64(pr * kMwAir * density_inv, kRu, 1.0 / kRu);
  st(B.bvo, b, c[0]);
  st(B.bvo + s, b, u);
  st(B.bvo + 2 * s, b, v);
  st(B.bvo + 3 * s, b, w);
  st(B.bvo + 4 * s, b, pr);
  st(B.bvo + 5 * s, b, T);
  st(B.mulo, b, sutherland(T));
  constexpr double c_temp{kGamma * kRu / kMwAir};
  st(B.mach, b, div64(sqrt(V2), sqrt(c_temp * T)));
}

}  // namespace

// Viscous fluxes of all three directions added to the stored inviscid dq
// (VISC), then the RK update of ring slot `out`; UPDATE false: dq is written
// to the block's array instead.  As in the x sweep a wave takes 64 consecutive
// padded points of the interior rows, one cell a lane: the x face is shared with
// the neighbouring lane (62 of 64 update), the two y and the two z faces are
// formed here.  u, v, w, T of the nine rows of the cells' yz cross section are
// loaded at once into the wave's own LDS words (held in registers they spill:
// 82 of 256), from which each face reads what it needs, x neighbours
// included.  Five faces a cell instead of three, but no workgroup barrier, and
// every load is a whole row segment; the rows beside and above are read from
// L2, since consecutive workgroups go to one XCD.
constexpr int kVWaves = 2;  // waves of a workgroup: 18 KB of LDS each, eight waves a CU
template <int VISC, bool UPDATE>
__global__ __launch_bounds__(64 * kVWaves, 2) void k_visc_update_rows(FusedArgs A, const SweepItem* items) {
  __shared__ double lds[VISC ? kVWaves : 1][9][4][VISC ? 64 : 1];
  const int G = gridDim.x, x = blockIdx.x % 8, per = G / 8, rest = G % 8;
  const SweepItem it = items[x * per + min(x, rest) + blockIdx.x / 8];
  if (A.target_block >= 0 && it.block != A.target_block) return;
  const StageBlock B = stage_block(A.blocks[it.block], A.in, A.out);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n = B.sx * B.my * B.mz, n0 = (int)B.n0;
  const int qf = it.first + wave * 62 + lane, qc = min(qf, n - 1);
  const int row = qc / B.sx, i = qc - row * B.sx - B.g, k = row / B.my, j = row - k * B.my;
  const bool store = lane > 0 && lane < 63 && qf < n && i >= 0 && i < B.mx;
  const int sy = B.sx, sz = B.sx * B.sy, o = poff(B, i, j, k);
  const gptr<double> res = UPDATE ? B.res : B.dq;
  const int q = (k * B.my + j) * B.mx + i;
  double dq[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (store) {
#pragma unroll
    for (int l = 0; l < 5; ++l) dq[l] = ld(res + l * n0, 8u * (unsigned)q);
  }
  double jac = 1.0;
  if constexpr (VISC) {
    const Geo g0 = load_geo(B, o);
    Geo gn = load_geo(B, o + sy);
    auto* L = lds[wave];  // [3 (k - 1, k, k + 1) + (j - 1, j, j + 1)][u, v, w, T][lane]
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const V4 f = load_v4(B, o + (c - 1) * sz + (r - 1) * sy);
#pragma unroll
        for (int v = 0; v < 4; ++v) L[3 * c + r][v][lane] = f.v[v];
      }
    // a wave's LDS accesses complete in order; the compiler must keep that order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    jac = g0.jac;
    const double pr = A.P.prandtl;
    __builtin_amdgcn_sched_barrier(0);
    const int lm = max(lane - 1, 0), lp = min(lane + 1, 63);
    auto val = [&](int r, int at) { return V4{{L[r][0][at], L[r][1][at], L[r][2][at], L[r][3][at]}}; };
    auto dx = [&](int r) { return minus(val(r, lp), val(r, lm)); };
    auto dy = [&](int c, int at) { return minus(val(3 * c + 2, at), val(3 * c, at)); };
    auto dz = [&](int r, int at) { return minus(val(6 + r, at), val(r, at)); };
    {
      const V4 g = visc_face<0>(val(4, lane), val(4, lp), dy(1, lane), dy(1, lp), dz(1, lane), dz(1, lp), g0, after(g0),
                                pr);
#pragma unroll
      for (int l = 0; l < 4; ++l) dq[l + 1] += g.v[l] - lane_before(g.v[l]);
    }
    // Between the faces: one face's operands and the next one's geometry live
    // at a time.  The empty asm makes a face's result exist at its place (left
    // alone, the evaluation sinks to its use behind the next face and keeps its
    // operands live: 142 registers spilled).
    auto done = [](V4& f) {
      asm volatile("" : "+v"(f.v[0]), "+v"(f.v[1]), "+v"(f.v[2]), "+v"(f.v[3])::"memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    V4 sum = {{dq[1], dq[2], dq[3], dq[4]}};
    done(sum);
    Geo gl = load_geo(B, o - sy);
    V4 up = visc_face<1>(val(4, lane), val(5, lane), dx(4), dx(5), dz(1, lane), dz(2, lane), g0, gn, pr);
    done(up);
    gn = load_geo(B, o + sz);
    V4 dn = visc_face<1>(val(3, lane), val(4, lane), dx(3), dx(4), dz(0, lane), dz(1, lane), gl, g0, pr);
#pragma unroll
    for (int l = 0; l < 4; ++l) sum.v[l] += up.v[l] - dn.v[l];
    done(sum);
    gl = load_geo(B, o - sz);
    up = visc_face<2>(val(4, lane), val(7, lane), dx(4), dx(7), dy(1, lane), dy(2, lane), g0, gn, pr);
    done(up);
    dn = visc_face<2>(val(1, lane), val(4, lane), dx(1), dx(4), dy(0, lane), dy(1, lane), gl, g0, pr);
#pragma unroll
    for (int l = 0; l < 4; ++l) dq[l + 1] = sum.v[l] + (up.v[l] - dn.v[l]);
  } else if (store) {
    jac = ld(B.jac, 8u * (unsigned)o);
  }
  if (!store) return;
  if constexpr (UPDATE) {
    stage_update(A, B, o, *A.dt, jac, dq);
  } else {
#pragma unroll
    for (int l = 0; l < 5; ++l) st(res + l * n0, 8u * (unsigned)q, dq[l]);
  }
}

int visc_cells_per_wg() { return kVWaves * 62; }

template <int SCHEME>
static void sweeps(const FusedArgs& a, const SweepPlan& s, hipStream_t st) {
  hipLaunchKernelGGL(k_sweep_x<SCHEME>, dim3(s.n[0]), dim3(256), 0, st, a, s.items[0]);
  hipLaunchKernelGGL((k_sweep_march<1, SCHEME>), dim3(s.n[1]), dim3(64), 0, st, a, s.items[1]);
  hipLaunchKernelGGL((k_sweep_march<2, SCHEME>), dim3(s.n[2]), dim3(64), 0, st, a, s.items[2]);
}

bool sweep_scheme(int scheme) { return scheme == 50 || scheme == 51 || scheme == 71; }

int sweep_valid(int scheme) { return 64 - 2 * (scheme == 71 ? Stencil<71>::R : Stencil<51>::R); }

void sweep_launch(FusedArgs a, const SweepPlan& s, bool update, hipStream_t st, long long* n) {
  a.to_dq = !update;
  if (a.P.scheme == 50) sweeps<50>(a, s, st);
  else if (a.P.scheme == 71) sweeps<71>(a, s, st);
  else sweeps<51>(a, s, st);
  *n += 3;
  if (!update && !a.P.visc) return;
  const dim3 grid(s.n[3]), wg(64 * kVWaves);
  if (!a.P.visc) hipLaunchKernelGGL((k_visc_update_rows<0, true>), grid, wg, 0, st, a, s.items[3]);
  else if (update) hipLaunchKernelGGL((k_visc_update_rows<1, true>), grid, wg, 0, st, a, s.items[3]);
  else hipLaunchKernelGGL((k_visc_update_rows<1, false>), grid, wg, 0, st, a, s.items[3]);
  ++*n;
}

}  // namespace ostc
