// Half-edge arguments shared by UpdateBCs and the Jacobian's boundary part.
#pragma once
#include "common.h"

namespace pcfd {

// threads per workgroup of the half-edge kernels: one wavefront, so that a
// few thousand half-edges spread over the chip
constexpr int kBndBlock = 64;

struct BndArgs {
  int nbnd, nnode, ntot, ntag, nbnode;
  const int *bnd_nodes, *he_ptr, *he_node, *he_src;
  const int4* he_desc;  // by list position: half-edge id, face tag, BC type, wall-normal neighbour (noSlip; else -1)
  const double *he_a, *qref, *twall;
  double gamma;
  double* q;
  double* seen;  // 5 x nbnode, by list position: a resetting node's state once the half-edge has been walked
};

// the node state half-edge p (list position) sees
__device__ __forceinline__ void bnd_seen(const BndArgs& A, int p, double* QL) {
  const int i = A.he_node[p];
#pragma unroll
  for (int k = 0; k < 5; ++k) QL[k] = i < 0 ? A.seen[k * A.nbnode + p] : A.q[k * A.ntot + i];
}

// the state of an adiabatic noSlip half-edge's wall-normal neighbour nn
__device__ __forceinline__ void wall_normal_state(const BndArgs& A, int p, int nn, double* Q) {
  const int s = A.he_src[p];
#pragma unroll
  for (int k = 0; k < 5; ++k) Q[k] = s >= 0 ? A.seen[k * A.nbnode + s] : A.q[k * A.ntot + nn];
}

BndArgs bnd_args(Ctx& c);
// the walk of the nodes that have resetting half-edges: their phantoms and
// `seen`; q's interior part is not written
void launch_bnd_resets(Ctx& c, hipStream_t s);

}  // namespace pcfd
