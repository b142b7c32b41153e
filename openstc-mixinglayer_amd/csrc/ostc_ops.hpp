// ostc_ops.hpp -- ghost-layer work items (boundary conditions, inner-face
// exchange, properties, cv-from-bv) as one list of boxes, many independent ops
// per launch.
#pragma once
#include "ostc_device.hpp"
#include "ostc_inflow.hpp"

namespace ostc {

enum OpType : int {
  OP_BC_OUTFLOW = 0,   // apply_outflow,  src/BoundCond.cuh:205-233
  OP_BC_PERIODIC = 1,  // apply_periodic, src/BoundCond.cuh:1443-1486
  OP_COMM = 2,         // inner_communication, src/DataCommunication.cuh:60-105
  OP_PROPS = 3,        // update_physical_properties<Air>, src/FieldOperation.cuh:107-140
  OP_CV_FROM_BV = 4,   // compute_cv_from_bv, src/FieldOperation.cuh:40-76
  OP_COPY_BV = 5,      // bv of slot `src` -> slot `slot` (ghost rims read by boundary ops)
  OP_BC_FARFIELD = 6,  // apply_farfield<Air>, src/BoundCond.cuh:755-1022
  OP_BC_INFLOW = 7,    // apply_inflow<Air>, src/BoundCond.cuh:235-612
};

// Doubles of one far-field state on the device, the layout of ostc_farfield:
// density, u, v, w, pressure, temperature, acoustic_speed, entropy,
// specific_heat_ratio, mw, sv[16].
constexpr int kFarfieldDoubles = 26;

struct DevOp {
  int type;
  int block, target;
  int axis, side;
  int lo[3];           // box origin (block indices, ghosts negative)
  int n[3];            // box extents
  int shared;          // OP_COMM: index along axis of the shared node layer
  int tcode[3];        // OP_COMM: target index along d = toff[d] + sgn * (index along p), tcode[d] = sgn * (p + 1)
  int toff[3];
  int flags;           // OP_COMM bit 0: also recompute the target's cv on the shared layer
  long long count;     // n[0]*n[1]*n[2]
  int layers;          // ghost layers as items of their own (OP_BC_OUTFLOW, OP_BC_PERIODIC), else 1
  const double* ff;    // OP_BC_FARFIELD: the state of the face's label (kFarfieldDoubles);
                       // OP_BC_INFLOW: the inflow state (kInflowDoubles)
  const double* aux;   // OP_BC_INFLOW: y of every op point (the face layer), in op point order
  const unsigned long long* pass;  // OP_BC_INFLOW: boundary-condition passes per block so far
};

// Largest ngg (WENO-Z7).
constexpr int kMaxGhost = 4;

// A workgroup of a launch: its op and its first item (point and layer).
struct OpWg { int op, first; };
constexpr int kOpWg = 256;

// The arrays of ring slot `slot` of a block.  The block table is itself read
// from memory, so the pointers it holds are generic to the compiler; as
// pointers into global memory the accesses are not flat instructions.
struct NodeArrays {
  gptr<double> bv, cv, mul, mach;
  long long s;
};
__device__ __forceinline__ NodeArrays node_arrays(const DevBlock& B, int slot) {
  return {(gptr<double>)B.bv[slot], (gptr<double>)B.cv[slot], (gptr<double>)B.mul[slot], (gptr<double>)B.mach, B.sz};
}
struct NodeState { double q[6]; };
__device__ __forceinline__ NodeState get_node(const NodeArrays& N, long long p) {
  NodeState n;
#pragma unroll
  for (int l = 0; l < 6; ++l) n.q[l] = N.bv[p + l * N.s];
  return n;
}

// compute_cv_from_bv_1_point<Air> (src/FieldOperation.cuh:40-76)
__device__ __forceinline__ void put_cv(const NodeArrays& N, long long p, const NodeState& n) {
  const double rho = n.q[0];
  N.cv[p] = rho;
  N.cv[p + N.s] = rho * n.q[1];
  N.cv[p + 2 * N.s] = rho * n.q[2];
  N.cv[p + 3 * N.s] = rho * n.q[3];
  N.cv[p + 4 * N.s] = total_energy(rho, n.q[1], n.q[2], n.q[3], n.q[4]);
}

// update_physical_properties<Air> at one point (src/FieldOperation.cuh:107-140):
// Sutherland viscosity and the Mach number.
__device__ __forceinline__ void put_props(const NodeArrays& N, long long p, const NodeState& n) {
  const double t = n.q[5];
  const double V = sqrt(n.q[1] * n.q[1] + n.q[2] * n.q[2] + n.q[3] * n.q[3]);
  constexpr double c_temp{kGamma * kRu / kMwAir};
  N.mul[p] = sutherland(t);
  N.mach[p] = V / sqrt(c_temp * t);
}

// Writes the primitives of a node and, from the same registers, its cv and,
// with `props`, its properties.  An op loads everything it reads before its
// first store, so a point costs one memory round trip rather than one per
// store the next load might alias.
__device__ __forceinline__ void put_node(const NodeArrays& N, long long p, const NodeState& n, bool with_cv,
                                         bool props) {
#pragma unroll
  for (int l = 0; l < 6; ++l) N.bv[p + l * N.s] = n.q[l];
  if (with_cv) put_cv(N, p, n);
  if (props) put_props(N, p, n);
}

// One item of an op.  Every op reads and writes the ring slot `slot` of
// cv/bv/mul.  With `props`, each op also recomputes the properties of every
// node whose primitives it writes, and the rim copy carries the viscosity of
// slot `src` along: then no separate properties pass over the ghost layers is
// needed (a node no op writes keeps the primitives and properties every slot
// was initialised with).  FACE_STATE: the launch may hold far-field and inflow
// ops, whose powers and random numbers the others should not pay registers for.
template <bool FACE_STATE>
__device__ __forceinline__ void op_item(const DevBlock* blocks, const DevOp& op, int item, int slot, int src,
                                        bool props) {
  const int pts = op.n[0] * op.n[1] * op.n[2], ax = op.axis, side = op.side;
  if (item >= pts * op.layers) return;
  // the layers of an x face are neighbours in memory, those of a y or z face
  // are planes
  const int t = ax == 0 ? item / op.layers : item % pts, g = 1 + (ax == 0 ? item % op.layers : item / pts);
  const int u = t / op.n[0], v = u / op.n[1];
  const int i = op.lo[0] + t - u * op.n[0], j = op.lo[1] + u - v * op.n[1], k = op.lo[2] + v;
  const DevBlock& B = blocks[op.block];
  const NodeArrays N = node_arrays(B, slot);
  const int di = ax == 0 ? side : 0, dj = ax == 1 ? side : 0, dk = ax == 2 ? side : 0;
  switch (op.type) {
    case OP_BC_OUTFLOW: {
      put_node(N, pidx(B, i + g * di, j + g * dj, k + g * dk), get_node(N, pidx(B, i, j, k)), true, props);
      break;
    }
    case OP_BC_PERIODIC: {
      const int m = ax == 0 ? B.mx : (ax == 1 ? B.my : B.mz), from = side < 0 ? m - 1 : 0;
      const int si = ax == 0 ? from : i, sj = ax == 1 ? from : j, sk = ax == 2 ? from : k;
      put_node(N, pidx(B, i + g * di, j + g * dj, k + g * dk),
               get_node(N, pidx(B, si + g * di, sj + g * dj, sk + g * dk)), true, props);
      break;
    }
    case OP_COMM: {
      const DevBlock& Tg = blocks[op.target];
      const NodeArrays M = node_arrays(Tg, slot);
      auto src_index = [&](int code) {
        const int q = (code < 0 ? -code : code) - 1;
        const int x = q == 0 ? i : (q == 1 ? j : k);
        return code < 0 ? -x : x;
      };
      const long long p = pidx(B, i, j, k), pt = pidx(Tg, op.toff[0] + src_index(op.tcode[0]),
                                                      op.toff[1] + src_index(op.tcode[1]),
                                                      op.toff[2] + src_index(op.tcode[2]));
      NodeState n = get_node(M, pt);
      if ((ax == 0 ? i : (ax == 1 ? j : k)) == op.shared) {
        const NodeState own = get_node(N, p);
#pragma unroll
        for (int l = 0; l < 6; ++l) n.q[l] = 0.5 * (n.q[l] + own.q[l]);
        put_node(M, pt, n, (op.flags & 1) != 0, props);
      }
      put_node(N, p, n, true, props);
      break;
    }
    case OP_PROPS: {
      const long long p = pidx(B, i, j, k);
      put_props(N, p, get_node(N, p));
      break;
    }
    case OP_COPY_BV: {
      const long long p = pidx(B, i, j, k);
      const NodeArrays S = node_arrays(B, src);
      const NodeState n = get_node(S, p);
      const double mu = props ? S.mul[p] : 0.0;
      put_node(N, p, n, false, false);
      if (props) N.mul[p] = mu;
      break;
    }
    case OP_BC_INFLOW: {
      if constexpr (FACE_STATE) {
        NodeState n;
        inflow_state(op.ff, op.aux[t], op.pass[op.block], inflow_point(ax, i, j, k, B.mx, B.my, B.g), n.q);
        for (int l = 0; l <= B.g; ++l) put_node(N, pidx(B, i + l * di, j + l * dj, k + l * dk), n, true, props);
      }
      break;
    }
    case OP_BC_FARFIELD: {
      // Each face point (and ngg beyond on the tangential directions) decides
      // from its own normal Mach number: supersonic inflow takes the far field
      // on the face point and its ghosts, supersonic outflow copies the face
      // point to the ghosts, subsonic faces take the state from the outgoing
      // Riemann invariant of the face point and the incoming one of the far
      // field, with the far field's entropy and tangential velocity on
      // inflow and the face point's on outflow.
      if constexpr (FACE_STATE) {
        const double* F = op.ff;
        const long long p = pidx(B, i, j, k), s = B.sz;
        double nx = B.met[p + (3 * ax) * s], ny = B.met[p + (3 * ax + 1) * s], nz = B.met[p + (3 * ax + 2) * s];
        const double grad_n_inv = side / sqrt(nx * nx + ny * ny + nz * nz);
        nx *= grad_n_inv;
        ny *= grad_n_inv;
        nz *= grad_n_inv;
        const NodeState b = get_node(N, p);
        const double u_b = b.q[1], v_b = b.q[2], w_b = b.q[3];
        const double u_face = nx * u_b + ny * v_b + nz * w_b;
        const double p_b = b.q[4], rho_b = b.q[0];
        const double a_b = sqrt(kGamma * p_b / rho_b);
        const double mach_b = u_face / a_b;
        NodeState st = b;
        bool face_too = true;
        if (mach_b <= -1) {
          for (int l = 0; l < 6; ++l) st.q[l] = F[l];
        } else if (mach_b >= 1) {
          face_too = false;
        } else {
          const double riemann_pos = u_face + 2 * a_b / (kGamma - 1);
          const double u_inf = F[1] * nx + F[2] * ny + F[3] * nz;
          const double riemann_neg = u_inf - 2 * F[6] / (F[8] - 1);
          const double Un = 0.5 * (riemann_pos + riemann_neg);
          const double c_b = 0.25 * (kGamma - 1) * (riemann_pos - riemann_neg);
          double s_b;
          if (mach_b <= 0) {
            s_b = F[7];
            st.q[1] = F[1] + (Un - u_inf) * nx;
            st.q[2] = F[2] + (Un - u_inf) * ny;
            st.q[3] = F[3] + (Un - u_inf) * nz;
          } else {
            s_b = p_b / pow(rho_b, kGamma);
            st.q[1] = u_b + (Un - u_face) * nx;
            st.q[2] = v_b + (Un - u_face) * ny;
            st.q[3] = w_b + (Un - u_face) * nz;
          }
          st.q[0] = pow(c_b * c_b / (kGamma * s_b), 1 / (kGamma - 1));
          st.q[4] = st.q[0] * c_b * c_b / kGamma;
          st.q[5] = st.q[4] * kMwAir / (st.q[0] * kRu);
        }
        if (face_too) put_node(N, p, st, true, props);
        for (int l = 1; l <= B.g; ++l) put_node(N, pidx(B, i + l * di, j + l * dj, k + l * dk), st, true, props);
      }
      break;
    }
    default:
      break;
  }
}

}  // namespace ostc
