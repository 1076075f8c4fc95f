// Exact rates of the surrogate's fallback cells.  The kernel is compiled in the
// unit whose path asks for the rates, so that they have that path's powers and
// its rounding (the finite-rate solver's unit contracts no products): an FR
// solve in which every node falls back has the bits of one with exact rates.
#pragma once
#include "chem_model.h"

namespace pcfd {

constexpr int kSurNs = 5;  // the surrogate is built for five species

// entry t of the compacted list lives in the pass p with off[p] <= t < off[p+1]
// (binary search)
template <typename P>
__global__ void __launch_bounds__(kChemBlock) k_wdot_list(const ChemDev* __restrict__ md, int npass,
                                                         const int* __restrict__ lst, const int* __restrict__ off,
                                                         const double* __restrict__ rhoi,
                                                         const double* __restrict__ T, double* __restrict__ wdot) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= off[npass]) return;
  int lo = 0, hi = npass;  // off[lo] <= t < off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= t) lo = mid;
    else hi = mid;
  }
  const int c = lst[(long long)lo * 64 + (t - off[lo])];
  const ChemDev& m = *md;
  double r[kSurNs], w[kSurNs];
#pragma unroll
  for (int k = 0; k < kSurNs; ++k) r[k] = rhoi[(long long)c * kSurNs + k];
  wdot_of<kSurNs, P>(m, r, T[c], w);
#pragma unroll
  for (int k = 0; k < kSurNs; ++k) wdot[(long long)c * kSurNs + k] = w[k];
}

using WdotList = void (*)(const ChemDev*, int, const int*, const int*, const double*, const double*, double*);

// Surrogate pass + fixed-order scan of the per-pass fallback counts + exact
// rates of the fallback list by `exact` (kernels_mlp.hip), on the mlp's stream,
// which is synchronised on return; lst/cnt/off hold at least npass*64, npass and
// npass+1 ints.
int surrogate_launch(pcfd_chem* chem, pcfd_mlp& m, const pcfd_surrogate_desc* d, int n, const double* rhoi,
                     const double* T, double* wdot, int* lst, int* cnt, int* off, WdotList exact, int* nfallback,
                     double* ms);

}  // namespace pcfd
