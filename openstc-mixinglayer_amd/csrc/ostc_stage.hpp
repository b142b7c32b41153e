// ostc_stage.hpp -- what one stage of the batched path reads and writes of a
// block, for the sweep and tile kernels.
#pragma once
#include "ostc_kernels.hpp"

namespace ostc {

// What one stage reads and writes of a block, with the arrays as pointers
// into global memory.  The block table is itself read from memory, so the
// pointers it holds are generic to the compiler, which would then access
// every array with flat instructions: those wait on the LDS counter as well
// and need 64-bit addresses per lane.
struct StageBlock {
  int mx, my, mz, g, sx, sy, sz;  // sz fits 32 bits: the host refuses 9 sz >= 2^31
  int ntx, nty, tile_base, sp_jac;
  long long n0;
  gptr<const double> cvi, bvi, muli, qn, jac, met, sp_sigma, sp_mean;
  gptr<double> cvo, bvo, mulo, mach, dq, res;
};

__device__ __forceinline__ StageBlock stage_block(const DevBlock& B, int in, int out) {
  StageBlock S;
  S.mx = B.mx; S.my = B.my; S.mz = B.mz; S.g = B.g; S.sx = B.sx; S.sy = B.sy; S.sz = (int)B.sz;
  S.ntx = B.ntx; S.nty = B.nty; S.tile_base = B.tile_base; S.sp_jac = B.sp_jac;
  S.n0 = B.n0;
  S.cvi = (gptr<const double>)B.cv[in];
  S.bvi = (gptr<const double>)B.bv[in];
  S.muli = (gptr<const double>)B.mul[in];
  S.qn = (gptr<const double>)B.cv[0];
  S.jac = (gptr<const double>)B.jac;
  S.met = (gptr<const double>)B.met;
  S.sp_sigma = (gptr<const double>)B.sp_sigma;
  S.sp_mean = (gptr<const double>)B.sp_mean;
  S.cvo = (gptr<double>)B.cv[out];
  S.bvo = (gptr<double>)B.bv[out];
  S.mulo = (gptr<double>)B.mul[out];
  S.mach = (gptr<double>)B.mach;
  S.dq = (gptr<double>)B.dq;
  S.res = (gptr<double>)B.res;
  return S;
}

// 32-bit offset of node (i, j, k) in a padded plane; the host refuses blocks
// whose 9 metric planes would not fit 2^31 doubles.
__device__ __forceinline__ int poff(const StageBlock& b, int i, int j, int k) {
  return ((k + b.g) * b.sy + (j + b.g)) * b.sx + (i + b.g);
}

// A plane's double at a byte offset of 32 bits.  The plane's address is the
// same for the whole wave, so it stays in scalar registers and the access has
// one vector register of address; an index of type int has to be widened and
// scaled per plane, two vector registers for each of a kernel's tens of loads.
__device__ __forceinline__ double ld(gptr<const double> plane, unsigned byte) {
  return *(gptr<const double>)((gptr<const char>)plane + byte);
}
__device__ __forceinline__ double ld(gptr<double> plane, unsigned byte) {
  return *(gptr<double>)((gptr<char>)plane + byte);
}
__device__ __forceinline__ void st(gptr<double> plane, unsigned byte, double v) {
  *(gptr<double>)((gptr<char>)plane + byte) = v;
}

}  // namespace ostc
