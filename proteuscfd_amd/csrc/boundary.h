// Half-edge arguments shared by UpdateBCs and the Jacobian's boundary part.
#pragma once
#include "common.h"

namespace pcfd {

// threads per workgroup of the half-edge kernels: one wavefront, so that a
// few thousand half-edges spread over the chip
constexpr int kBndBlock = 64;

struct BndArgs {
  int nbnd, nnode, ntot, ntag, nbnode, nrst;
  const int *bnd_nodes, *rst, *he_ptr, *he_node;
  const int4* he_desc;  // by list position: half-edge id, face tag, BC type, wall-normal neighbour (noSlip; else -1)
  const double *he_a, *qref, *twall;
  double gamma;
  double* q;
  double* seen;  // 5 x nbnode, by list position: the node state a half-edge of a resetting node sees
};

// the node state half-edge p (list position) sees
__device__ __forceinline__ void bnd_seen(const BndArgs& A, int p, double* QL) {
  const int i = A.he_node[p];
#pragma unroll
  for (int k = 0; k < 5; ++k) QL[k] = i < 0 ? A.seen[k * A.nbnode + p] : A.q[k * A.ntot + i];
}

BndArgs bnd_args(Ctx& c);
// the resets of the nodes that have any: into q, or (Qb set) into Qb with q's interior part untouched
void launch_bnd_resets(Ctx& c, hipStream_t s, double* Qb);

}  // namespace pcfd
