// First-order finite-difference block Jacobian and the inverses of its diagonal.
//
// Reference: ComputeSpatialJacobian (ucs/jacobian.tcc:129-210) scatters per
// edge A[R][L] += -dF/dQL and A[L][R] += dF/dQR (Kernel_NumJac :253-304),
// adds boundary blocks to the diagonal with the boundary state re-evaluated
// under perturbation (Bkernel_NumJac :458-535), then sums each column's
// off-diagonal blocks onto the diagonal (Kernel_Diag_NumJac :436-456), and
// ContributeTemporalTerms adds vol/dt (:213-250).
//
// Here five lanes own one block row of the SELL matrix, a column each (12
// rows a wavefront, in SELL row order): they write the row's off-diagonal
// blocks and accumulate its diagonal (boundary part first, then edges in
// ascending neighbour order, then the temporal term), so every entry has a
// single writer.  Storage type T is double
// (plain) or float (chosen form); the differences are always taken in FP64.
#include <stdexcept>

#include "boundary.h"
#include "common.h"
#include "physics.h"

namespace pcfd {

struct JacArgs {
  int nnode, ntot, nrow_pad, sym2d;
  double gamma;
  const int *gwidth, *gbase, *gcol, *gslot;
  const double* gnrm;
  long long gstride;
  const double *vol, *dt;
  const double* q;
  const int *srow, *sbase;
  const double* xyz;       // SoA, for the viscous directional weights
  ViscParams vp;
  int flux_alg;            // 1: algebraic flux (generic form only)
  int centred;             // 1: centred differences, jacobianFieldType 1 (generic form only)
  int bcentred;            // 1: centred boundary differences, jacobianBoundaryType 1
  int* nonfinite;          // cleared by the rows, set by k_prepare_sgs
};

// One-sided differences with h = 1e-8 (ucs/jacobian.tcc:268): the quotient
// is taken as a product with 1/h = 1e8, which is exact in binary64, so it
// differs from the division by h at most in the last bit.
constexpr double kInvH = 1.0e8;
// centred differences (Kernel_NumJac_Centered, ucs/jacobian.tcc:307-367):
// the quotient by 2h as a product with 1/(2h) = 5e7, exact in binary64
constexpr double kInv2H = 5.0e7;

// Five lanes per block row: lane c of a row's group owns perturbation
// column c -- it writes column c of every block of the row and accumulates
// column c of the diagonal.  Each block entry is produced by exactly the
// same finite difference as a one-thread-per-row evaluation, with a fifth
// of the live state per lane.  A wavefront holds 12 rows (lanes 60-63 idle).
__device__ __forceinline__ void perturb(const double* Q, int c, double h, double* QP) {
#pragma unroll
  for (int k = 0; k < 5; ++k) QP[k] = Q[k] + (k == c ? h : 0.0);
}

// Boundary half-edges (Bkernel_NumJac).  k_bnd_resets has walked the nodes'
// resets; then every half-edge has a thread for its boundary state and
// unperturbed flux (k_jac_bnd_base), every (half-edge, column) one for the
// perturbed evaluation (k_jac_bnd_cols), and k_jac_bnd_sum adds a node's
// half-edges in their order into its part Db of the diagonal block
// (Db[t*25 + r*5 + c], t = boundary-node index).  One thread a (node, column)
// that walked the half-edges took 95 us on the 386 boundary nodes of the 8^3
// bump, 126 us on the 36k-node plate, 259 us on the 416k-node one; the four
// passes take 36, 60 and 160 us.
//
// With A.bcentred (Bkernel_NumJac_Centered, ucs/jacobian.tcc:538-640, at the
// default jacobianBoundaryEval 0) column c is (F(q+h e_c, BC(q+h e_c)) -
// F(q-h e_c, QR)) / 2h: the +h side re-evaluates the boundary state, the -h
// side keeps the unperturbed one QR.  bnd_down() forms that -h flux.
template <bool ALG>
__device__ __forceinline__ void bnd_down(const double* QL, const double* QR, int c, const double* a, double gamma,
                                         int sym2d, double* fD) {
  double QPD[5];
  perturb(QL, c, -1.0e-8, QPD);
  num_flux<ALG>(QPD, QR, a, gamma, sym2d, fD);
}
// rec[p]: the boundary state QR and the flux the columns difference against
// (one-sided form), or for a centred Dirichlet half-edge the +h side's flux
template <bool ALG>
__global__ void __launch_bounds__(kBndBlock) k_jac_bnd_base(BndArgs B, int sym2d, int cen, double* __restrict__ rec) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= B.nbnode) return;
  const int4 d = B.he_desc[p];
  const int h = d.x, tag = d.y, type = d.z, ph = B.nnode + h;
  const double a[4] = {B.he_a[h], B.he_a[B.nbnode + h], B.he_a[2 * B.nbnode + h], B.he_a[3 * B.nbnode + h]};
  double QL[5], QR[5], Qr[5];
  bnd_seen(B, p, QL);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    QR[k] = B.q[k * B.ntot + ph];
    Qr[k] = B.qref[k * B.ntag + tag];
  }
  // noSlip and Dirichlet phantoms are set by k_bnd_resets
  if (type != BC_NOSLIP && !is_dirichlet(type) && bc_state(type, QL, QR, Qr, B.qref[5 * B.ntag + tag], a, B.gamma)) {
#pragma unroll
    for (int k = 0; k < 5; ++k) B.q[k * B.ntot + ph] = QR[k];
  }
  double fS[5] = {0, 0, 0, 0, 0};
  if (!cen || is_dirichlet(type)) num_flux<ALG>(QL, QR, a, B.gamma, sym2d, fS);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    rec[(long long)p * 10 + k] = QR[k];
    rec[(long long)p * 10 + 5 + k] = fS[k];
  }
}

template <bool ALG>
__global__ void __launch_bounds__(kBndBlock) k_jac_bnd_cols(BndArgs B, int sym2d, int cen,
                                                           const double* __restrict__ rec,
                                                           double* __restrict__ col) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 5LL * B.nbnode) return;
  const int p = (int)(t / 5), c = (int)(t % 5);
  const int4 d = B.he_desc[p];
  const int h = d.x, tag = d.y, type = d.z;
  const double a[4] = {B.he_a[h], B.he_a[B.nbnode + h], B.he_a[2 * B.nbnode + h], B.he_a[3 * B.nbnode + h]};
  const double w = cen ? kInv2H : kInvH;
  double QL[5], QR[5], fS[5], fL[5], Dc[5] = {0, 0, 0, 0, 0};
  bnd_seen(B, p, QL);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    QR[k] = rec[(long long)p * 10 + k];
    fS[k] = rec[(long long)p * 10 + 5 + k];
  }
  bool live = true;
  if (is_dirichlet(type)) {
    // QL = QR = Qref and every perturbed evaluation resets both to Qref, so
    // the one-sided contribution is exactly zero; the centred one keeps its
    // -h side: (F(Qref, Qref) - F(Qref - h e_c, Qref)) / 2h
    live = cen != 0;
#pragma unroll
    for (int k = 0; k < 5; ++k) fL[k] = fS[k];
  } else {
    double QPL[5], QPR[5] = {QR[0], QR[1], QR[2], QR[3], QR[4]};
    perturb(QL, c, 1.0e-8, QPL);
    if (type == BC_NOSLIP) {
      // CalculateBoundaryVariables hard-sets the wall node for the base and
      // for every perturbed state (ucs/jacobian.tcc:484-512)
      const double tw = B.twall[tag];
      const int nn = d.w;
      live = !(tw < 0.0 && nn < 0);
      double nQ[5] = {0, 0, 0, 0, 0};
      if (tw < 0.0 && live) wall_normal_state(B, p, nn, nQ);
      noslip_state(QPL, QPR, tw, nQ, B.gamma);
    } else {
      double Qr[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) Qr[k] = B.qref[k * B.ntag + tag];
      bc_state(type, QPL, QPR, Qr, B.qref[5 * B.ntag + tag], a, B.gamma);
    }
    num_flux<ALG>(QPL, QPR, a, B.gamma, sym2d, fL);
  }
  if (live) {
    if (cen) bnd_down<ALG>(QL, QR, c, a, B.gamma, sym2d, fS);
#pragma unroll
    for (int rr = 0; rr < 5; ++rr) Dc[rr] = (fL[rr] - fS[rr]) * w;
  }
#pragma unroll
  for (int rr = 0; rr < 5; ++rr) col[t * 5 + rr] = Dc[rr];
}

// ... and the nodes' states after the re-evaluation to Qb
__global__ void __launch_bounds__(kBlock) k_jac_bnd_sum(BndArgs B, const double* __restrict__ col,
                                                       double* __restrict__ Db, double* __restrict__ Qb) {
  const long long t25 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t25 >= 25LL * B.nbnd) return;
  const int t = (int)(t25 / 25), k = (int)(t25 % 25);  // k = column * 5 + row, as col stores them
  const int i = B.bnd_nodes[t];
  const int p1 = B.he_ptr[i + 1];
  if (k < 5) Qb[5LL * t + k] = B.he_node[p1 - 1] < 0 ? B.seen[k * B.nbnode + p1 - 1] : B.q[k * B.ntot + i];
  double s = 0.0;
  for (int p = B.he_ptr[i]; p < p1; ++p) s += col[25LL * p + k];
  Db[25LL * t + (k % 5) * 5 + k / 5] = s;
}

// the edge flux of the generic form, evaluated from node i's side (x is
// node i's state); a is the canonical n0 -> n1 normal, `left` whether i is n0
__device__ __forceinline__ void jac_flux(const JacArgs& A, const double* x, const double* y, const double* ai,
                                         const double* a, bool left, double* F) {
  if (A.flux_alg) alg_flux(x, y, ai, A.gamma, F);
  else if (roe_flux_fast(x, y, ai, A.gamma, A.sym2d, F) && !left) roe_flux_canonical(y, x, a, A.gamma, A.sym2d, F);
}

// GENERIC = false: Roe flux, one-sided differences (the reference defaults),
// with the own node's Roe-side quantities formed once per row.
// GENERIC = true: the flux (Roe or algebraic) and the difference form
// (one-sided or centred) chosen at run time, each evaluation from scratch.
template <typename T, bool VISC, bool GENERIC>
__global__ void __launch_bounds__(kBlock) k_jacobian(JacArgs A, const int* __restrict__ bidx,
                                                    const double* __restrict__ Db, const double* __restrict__ Qb,
                                                    T* __restrict__ Moff, T* __restrict__ Dg) {
  const int lane64 = threadIdx.x & 63;
  if (lane64 >= 60) return;
  const int r = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * 12 + lane64 / 5;
  const int c = lane64 % 5;
  if (r >= A.nrow_pad) return;
  if (r == 0 && c == 0) *A.nonfinite = 0;
  const int i = A.srow[r];
  if (i < 0) return;
  const int chunk = r >> 6, lane = r & 63;
  const double h = 1.0e-8;
  const double gamma = A.gamma;
  double Dc[5] = {0, 0, 0, 0, 0};  // column c of the diagonal block
  const int bt = bidx[i];
  if (bt >= 0) {
    // boundary contributions come first, as Bdriver runs before Kernel_Diag_NumJac
#pragma unroll
    for (int rr = 0; rr < 5; ++rr) Dc[rr] = Db[(long long)bt * 25 + rr * 5 + c];
  }
  double qi[5], xi[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 5; ++k) qi[k] = A.q[k * A.ntot + i];
  if (VISC) {
    xi[0] = A.xyz[i];
    xi[1] = A.xyz[A.nnode + i];
    xi[2] = A.xyz[2 * A.nnode + i];
  }
  // --- interior edges (Kernel_NumJac): row blocks + diagonal column sums ---
  // Each edge flux is evaluated from this node's side: G(x, y) = F(x, y, n_i)
  // with n_i the face normal pointing out of node i.  The Roe flux with the
  // Harten-Hyman fix is antisymmetric, F(L, R, a) = -F(R, L, -a), so the
  // reference's F(L, R, a) is +G when i is the left node and -G when it is
  // the right node, and the two signs cancel in what the row needs:
  //   diagonal column c:   -A[j][i] column c = (G(q_i + h e_c, q_j) - G(q_i, q_j)) / h
  //   off-diagonal column c:  A[i][j] column c = (G(q_i, q_j + h e_c) - G(q_i, q_j)) / h
  // (the same one-sided differences as the reference's (L,R) evaluation up
  // to the rounding of the flux).  The own node's states, unperturbed and
  // perturbed in component c, are formed once per row.
  // (with centred differences: dcol = (G(q_i + h e_c, q_j) - G(q_i - h e_c, q_j)) / 2h,
  //  offc = (G(q_i, q_j + h e_c) - G(q_i, q_j - h e_c)) / 2h)
  double qiP[5], qiM[5];
  perturb(qi, c, h, qiP);
  perturb(qi, c, -h, qiM);
  RoeSide S0, SP;
  if constexpr (!GENERIC) {
    roe_side_state(qi, gamma, S0);
    roe_side_state(qiP, gamma, SP);
  }
  const long long gb = (long long)A.gbase[i >> 6] * kW + (i & 63);
  const int w = A.gwidth[i >> 6];
  T* ob = Moff + (long long)A.sbase[chunk] * 25 * kW + lane + (long long)c * kW;
  const int g0 = lane64 - c;  // first lane of this row's group of five
  double fSg[5] = {0, 0, 0, 0, 0};
  for (int s = 0; s < w; ++s) {
    const long long gi = gb + (long long)s * kW;
    const int j = A.gcol[gi];
    if (j < 0) break;
    const bool left = i < j;
    const double a[4] = {A.gnrm[gi], A.gnrm[A.gstride + gi], A.gnrm[2 * A.gstride + gi], A.gnrm[3 * A.gstride + gi]};
    const double sg = left ? 1.0 : -1.0;
    const double ai[4] = {sg * a[0], sg * a[1], sg * a[2], a[3]};  // out of node i
    double qj[5], qjP[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) qj[k] = A.q[k * A.ntot + j];
    perturb(qj, c, h, qjP);
    T* blk = ob + (long long)A.gslot[gi] * 25 * kW;
    // offc: column c of this row's block A[i][j]; dcol: this edge's part of
    // column c of the diagonal block
    double offc[5], dcol[5];
    if constexpr (!GENERIC) {
      // The unperturbed flux G(q_i, q_j) is the same for the row's five
      // lanes: at every fifth slot, lane c evaluates it for slot s + c, and
      // each lane then takes slot s's value from lane s % 5 of its group.
      // (Inviscid rows only: with the viscous columns the extra registers
      // cost more than the four flux evaluations they save.)
      if (!VISC && s % 5 == 0) {
        const int sc = s + c;
        const long long gic = gb + (long long)sc * kW;
        const int jc = sc < w ? A.gcol[gic] : -1;
#pragma unroll
        for (int k = 0; k < 5; ++k) fSg[k] = 0.0;
        if (jc >= 0) {
          const double sgc = i < jc ? 1.0 : -1.0;
          const double aic[4] = {sgc * A.gnrm[gic], sgc * A.gnrm[A.gstride + gic], sgc * A.gnrm[2 * A.gstride + gic],
                                 A.gnrm[3 * A.gstride + gic]};
          double qc[5];
#pragma unroll
          for (int k = 0; k < 5; ++k) qc[k] = A.q[k * A.ntot + jc];
          RoeSide Sc = S0, Sjc;
          roe_side_th(Sc, aic);
          roe_side(qc, aic, gamma, Sjc);
          if (roe_flux_s(qi, Sc, qc, Sjc, aic, gamma, A.sym2d, fSg) && i > jc) {
            const double ac[4] = {-aic[0], -aic[1], -aic[2], aic[3]};
            roe_flux_canonical(qc, qi, ac, gamma, A.sym2d, fSg);
          }
        }
      }
      roe_side_th(S0, ai);
      roe_side_th(SP, ai);
      RoeSide Sj, SjP;
      roe_side(qj, ai, gamma, Sj);
      double fS[5], fP[5];
      if constexpr (VISC) {
        if (roe_flux_s(qi, S0, qj, Sj, ai, gamma, A.sym2d, fS) && !left)
          roe_flux_canonical(qj, qi, a, gamma, A.sym2d, fS);
      } else {
#pragma unroll
        for (int k = 0; k < 5; ++k) fS[k] = __shfl(fSg[k], g0 + s % 5);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (roe_flux_s(qiP, SP, qj, Sj, ai, gamma, A.sym2d, fP) && !left)
        roe_flux_canonical(qj, qiP, a, gamma, A.sym2d, fP);
#pragma unroll
      for (int rr = 0; rr < 5; ++rr) dcol[rr] = (fP[rr] - fS[rr]) * kInvH;
      __builtin_amdgcn_sched_barrier(0);
      roe_side(qjP, ai, gamma, SjP);
      if (roe_flux_s(qi, S0, qjP, SjP, ai, gamma, A.sym2d, fP) && !left)
        roe_flux_canonical(qjP, qi, a, gamma, A.sym2d, fP);
#pragma unroll
      for (int rr = 0; rr < 5; ++rr) offc[rr] = (fP[rr] - fS[rr]) * kInvH;
      __builtin_amdgcn_sched_barrier(0);
    } else {
      double fA[5], fB[5];
      if (A.centred) {
        double qjM[5];
        perturb(qj, c, -h, qjM);
        jac_flux(A, qiP, qj, ai, a, left, fA);
        jac_flux(A, qiM, qj, ai, a, left, fB);
#pragma unroll
        for (int rr = 0; rr < 5; ++rr) dcol[rr] = (fA[rr] - fB[rr]) * kInv2H;
        jac_flux(A, qi, qjP, ai, a, left, fA);
        jac_flux(A, qi, qjM, ai, a, left, fB);
#pragma unroll
        for (int rr = 0; rr < 5; ++rr) offc[rr] = (fA[rr] - fB[rr]) * kInv2H;
      } else {
        jac_flux(A, qi, qj, ai, a, left, fB);
        jac_flux(A, qiP, qj, ai, a, left, fA);
#pragma unroll
        for (int rr = 0; rr < 5; ++rr) dcol[rr] = (fA[rr] - fB[rr]) * kInvH;
        jac_flux(A, qi, qjP, ai, a, left, fA);
#pragma unroll
        for (int rr = 0; rr < 5; ++rr) offc[rr] = (fA[rr] - fB[rr]) * kInvH;
      }
    }
    if (VISC) {
      // Kernel_Viscous_Jac (ucs/jacobian.tcc:734-767): A[R][L] += aL,
      // A[L][R] += aR, added before the column sums; it runs after the
      // boundary Jacobian has hard-set wall / Dirichlet nodes, so boundary
      // nodes enter with their re-evaluated states
      const double xj[3] = {A.xyz[j], A.xyz[A.nnode + j], A.xyz[2 * A.nnode + j]};
      double vi[5], vj[5];
      const int bj = bidx[j];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        vi[k] = bt >= 0 ? Qb[(long long)bt * 5 + k] : qi[k];
        vj[k] = bj >= 0 ? Qb[(long long)bj * 5 + k] : qj[k];
      }
      double vL[5], vR[5];
      visc_jac_cols(c, left ? vi : vj, left ? vj : vi, left ? xi : xj, left ? xj : xi, a, A.vp, vL, vR);
#pragma unroll
      for (int rr = 0; rr < 5; ++rr) {
        offc[rr] += left ? vR[rr] : vL[rr];
        dcol[rr] -= left ? vL[rr] : vR[rr];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int rr = 0; rr < 5; ++rr) {
      blk[rr * 5 * kW] = (T)offc[rr];
      Dc[rr] += dcol[rr];
    }
  }
  // --- temporal term, steady pseudo-time: A_ii += 1*vol/dtau ---
  const double vt = 1.0 * A.vol[i] / A.dt[i];
#pragma unroll
  for (int rr = 0; rr < 5; ++rr)
    if (rr == c) Dc[rr] += vt;
  T* dg = Dg + (long long)chunk * 25 * kW + lane + (long long)c * kW;
#pragma unroll
  for (int rr = 0; rr < 5; ++rr) dg[rr * 5 * kW] = (T)Dc[rr];
}

// Dirichlet / sonic-inflow and noSlip overwrites of boundary node states,
// deferred until all rows have read the pre-update states (the reference
// applies them inside Bkernel_NumJac after Kernel_NumJac has run): the
// states the boundary part ended with are copied into q.
__global__ void __launch_bounds__(kBlock) k_commit_hardset(int nbnd, int ntot, const int* __restrict__ bnd_nodes,
                                                          const double* __restrict__ Qb, double* __restrict__ q) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nbnd) return;
  const int i = bnd_nodes[t];
#pragma unroll
  for (int k = 0; k < 5; ++k) q[k * ntot + i] = Qb[(long long)t * 5 + k];
}

// Bkernel_BC_Jac_Modify -> ModifyViscousWallJacobian (ucs/bc.tcc:747-900,
// ucs/compressible.tcc:1577-1606) after the temporal terms: per noSlip
// half-edge, BlankSubRow (ucs/crsmatrix.tcc:525-541) zeroes sub-row r of
// every block of the row and puts 1 on the diagonal; isothermal walls then
// tie the energy change to the density change, adiabatic walls tie density
// and energy to the wall-normal neighbour.  Of a node's half-edges the last
// noSlip one decides sub-rows 1-4 and the last adiabatic one sub-row 0, so one
// thread per (boundary node, slot) writes the end state (slot `w` of the grid:
// the diagonal).  One thread a node that replayed every half-edge: 71 us on
// the 36k-node plate; now 8 us.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_noslip_rows(BndArgs B, const int* __restrict__ spos,
                                                       const int* __restrict__ swidth, const int* __restrict__ sbase,
                                                       const int* __restrict__ scol, T* __restrict__ Moff,
                                                       T* __restrict__ Dg) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= B.nbnd) return;
  const int i = B.bnd_nodes[t];
  if (B.he_node[B.he_ptr[i]] >= 0) return;  // no half-edge resets it
  int last = -1, adia = -1;  // list positions
  for (int p = B.he_ptr[i]; p < B.he_ptr[i + 1]; ++p) {
    if (B.he_desc[p].z != BC_NOSLIP) continue;
    last = p;
    if (B.twall[B.he_desc[p].y] < 0.0) adia = p;
  }
  if (last < 0) return;
  const int r = spos[i];
  const int chunk = r >> 6, lane = r & 63, s = blockIdx.y;
  const bool last_adia = last == adia;
  if (s == (int)gridDim.y - 1) {  // the diagonal block
    T* dg = Dg + (long long)chunk * 25 * kW + lane;
    const double tw = B.twall[B.he_desc[last].y], g = B.gamma, v2 = 0.0;
#pragma unroll
    for (int rr = 0; rr < 5; ++rr) {
      if (rr == 0 && adia < 0) continue;
#pragma unroll
      for (int k = 0; k < 5; ++k) dg[(rr * 5 + k) * kW] = (T)(k == rr ? 1 : 0);
    }
    if (!last_adia) dg[20 * kW] = (T)(-(tw / (g * (g - 1.0)) + 0.5 * v2));
    return;
  }
  if (s >= swidth[chunk]) return;
  const long long sb = (long long)sbase[chunk] + s;
  const int col = scol[sb * kW + lane];
  if (col < 0) return;  // padding
  T* blk = Moff + sb * 25 * kW + lane;
#pragma unroll
  for (int rr = 0; rr < 5; ++rr) {
    if (rr == 0 && adia < 0) continue;
#pragma unroll
    for (int k = 0; k < 5; ++k) blk[(rr * 5 + k) * kW] = (T)0;
  }
  // the last adiabatic half-edge's wall-normal neighbour
  const int nn = adia >= 0 ? B.he_desc[adia].w : -1;
  if (nn < 0 || col != spos[nn]) return;
  blk[0 * kW] = (T)-1.0;
  if (last_adia) blk[24 * kW] = (T)-1.0;
}

static JacArgs jac_args(Ctx& c) {
  const pcfd_params& p = c.prm;
  return JacArgs{c.nnode, c.ntot, c.nrow_pad, p.symmetry2d, p.gamma, c.d.gwidth, c.d.gbase, c.d.gcol, c.d.gslot,
                 c.d.gnrm, c.nslot_g * kW, c.d.vol, c.d.dt, c.d.q, c.d.srow, c.d.sbase, c.d.xyz,
                 ViscParams{p.gamma, p.re_tilde, p.prandtl, p.prandtl_t, p.sutherland_s, p.symmetry2d},
                 p.flux_type == PCFD_FLUX_ALGEBRAIC ? 1 : 0, p.jac_field_type == 1 ? 1 : 0,
                 p.jac_boundary_type == 1 ? 1 : 0, c.d.icount + 1};
}

static void jac_boundary(Ctx& c, const JacArgs& A, hipStream_t s) {
  if (c.nbnd == 0) return;
  launch_bnd_resets(c, s);
  const BndArgs B = bnd_args(c);
  // per half-edge, until the rows fill the array: boundary state and unperturbed
  // flux (10), the columns of the diagonal's boundary part (25)
  double* const jhe = c.prm.precision == PCFD_CHOSEN_FP32 ? reinterpret_cast<double*>(c.d.Mf) : c.d.Md;
  double* const jcol = jhe + 10 * (size_t)c.nbnode;
  hipLaunchKernelGGL(A.flux_alg ? k_jac_bnd_base<true> : k_jac_bnd_base<false>, dim3(nblk(c.nbnode, kBndBlock)),
                     dim3(kBndBlock), 0, s, B, A.sym2d, A.bcentred, jhe);
  PCFD_HIP(hipGetLastError());
  hipLaunchKernelGGL(A.flux_alg ? k_jac_bnd_cols<true> : k_jac_bnd_cols<false>, dim3(nblk(5LL * c.nbnode, kBndBlock)),
                     dim3(kBndBlock), 0, s, B, A.sym2d, A.bcentred, jhe, jcol);
  PCFD_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_jac_bnd_sum, dim3(nblk(25LL * c.nbnd)), dim3(kBlock), 0, s, B, jcol, c.d.jdb, c.d.jqb);
  PCFD_HIP(hipGetLastError());
}

static void jac_commit(Ctx& c, hipStream_t s) {
  if (c.nbnd == 0) return;
  hipLaunchKernelGGL(k_commit_hardset, dim3(nblk(c.nbnd)), dim3(kBlock), 0, s, c.nbnd, c.ntot, c.d.bnd_nodes,
                     c.d.jqb, c.d.q);
  PCFD_HIP(hipGetLastError());
}

static void jac_rows(Ctx& c, const JacArgs& A, hipStream_t s) {
  const pcfd_params& p = c.prm;
  const long long waves = (c.nrow_pad + 11) / 12;  // 12 rows x 5 lanes per wavefront
  const int grid = nblk(waves * kW);
  const bool f32 = p.precision == PCFD_CHOSEN_FP32;
  const bool gen = A.flux_alg || A.centred;
  if (f32) {
    auto kern = p.viscous ? (gen ? k_jacobian<float, true, true> : k_jacobian<float, true, false>)
                          : (gen ? k_jacobian<float, false, true> : k_jacobian<float, false, false>);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, s, A, c.d.bidx, c.d.jdb, c.d.jqb, c.d.Mf, c.d.Df);
  } else {
    auto kern = p.viscous ? (gen ? k_jacobian<double, true, true> : k_jacobian<double, true, false>)
                          : (gen ? k_jacobian<double, false, true> : k_jacobian<double, false, false>);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, s, A, c.d.bidx, c.d.jdb, c.d.jqb, c.d.Md, c.d.Dd);
  }
  PCFD_HIP(hipGetLastError());
}

static void jac_noslip(Ctx& c, hipStream_t s) {
  if (!c.has_noslip) return;
  const dim3 grid(nblk(c.nbnd), c.max_swidth + 1);
  if (c.prm.precision == PCFD_CHOSEN_FP32)
    hipLaunchKernelGGL(k_noslip_rows<float>, grid, dim3(kBlock), 0, s, bnd_args(c), c.d.spos, c.d.swidth, c.d.sbase,
                       c.d.scol, c.d.Mf, c.d.Df);
  else
    hipLaunchKernelGGL(k_noslip_rows<double>, grid, dim3(kBlock), 0, s, bnd_args(c), c.d.spos, c.d.swidth,
                       c.d.sbase, c.d.scol, c.d.Md, c.d.Dd);
  PCFD_HIP(hipGetLastError());
}

// In reference order on the library stream: boundary part (phantom states,
// boundary diagonal contributions), rows, then the hard-set commit.
void launch_jacobian(Ctx& c) {
  const JacArgs A = jac_args(c);
  sub_begin(c);
  jac_boundary(c, A, c.stream);
  jac_rows(c, A, c.stream);
  jac_commit(c, c.stream);
  jac_noslip(c, c.stream);
  sub_end(c, 11);
}

// The rows on the second stream, overlapping the time step, BCs, gradient,
// limiter and residual that follow on the library stream (they touch
// neither the matrix nor, with the states the rows read kept apart, the rows'
// inputs).  The rows read the states from before the hard-set commit -- a
// snapshot when the case has hard-set nodes, q itself otherwise (then
// nothing on the library stream writes interior states before the join) --
// and the dt array the caller then retires (the new time step goes to the
// other buffer).  jacobian_join() orders the library stream after the rows.
void launch_jacobian_overlapped(Ctx& c) {
  JacArgs A = jac_args(c);
  jac_boundary(c, A, c.stream);
  if (!c.rst_level.empty()) {
    PCFD_HIP(hipMemcpyAsync(c.d.qjac, c.d.q, sizeof(double) * 5 * (size_t)c.ntot, hipMemcpyDeviceToDevice,
                            c.stream));
    A.q = c.d.qjac;
    jac_commit(c, c.stream);
  }
  PCFD_HIP(hipEventRecord(c.ev_fork, c.stream));
  PCFD_HIP(hipStreamWaitEvent(c.stream2, c.ev_fork, 0));
  if (c.timing) PCFD_HIP(hipEventRecord(c.ev4, c.stream2));
  jac_rows(c, A, c.stream2);
  jac_noslip(c, c.stream2);
  if (c.timing) PCFD_HIP(hipEventRecord(c.ev5, c.stream2));
  PCFD_HIP(hipEventRecord(c.ev_join, c.stream2));
  c.jac_pending = true;
}

void jacobian_join(Ctx& c) {
  if (!c.jac_pending) return;
  PCFD_HIP(hipStreamWaitEvent(c.stream, c.ev_join, 0));
  c.jac_pending = false;
  if (c.timing) {
    PCFD_HIP(hipEventSynchronize(c.ev5));
    float ms = 0.f;
    PCFD_HIP(hipEventElapsedTime(&ms, c.ev4, c.ev5));
    c.phase_ms[5] += ms;
    c.phase_ms[11] += ms;
  }
}

// PrepareSGS (ucs/crsmatrix.tcc:839-876): the reference factors each diagonal
// block (LU with partial pivoting, ucs/matrix.h:110-190) and every row update
// solves with the factor.  Here the block is replaced by its inverse, from
// the same elimination (rows swapped physically: compile-time register
// indices, no scratch) applied to the unit columns, so a row update is one
// 5x5 product.  The elimination runs in FP64 for both storage types.
//
// A block that holds a NaN or an infinity is reported: an off-diagonal block
// holds one only where a diagonal block does (its column's, which sums it, or
// where that node's rows are hard-set its own row's, which has the same flux),
// and the first sweep then takes nothing for granted (k_sgs_color).
template <typename T>
__global__ void __launch_bounds__(kBlock) k_prepare_sgs(int nrow_pad, const int* __restrict__ srow,
                                                       T* __restrict__ Dg, int* __restrict__ nonfinite) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrow_pad || srow[r] < 0) return;
  T* a = Dg + (long long)(r >> 6) * 25 * kW + (r & 63);
  double A[25];
#pragma unroll
  for (int k = 0; k < 25; ++k) A[k] = (double)a[k * kW];
  double z = 0.0;
#pragma unroll
  for (int k = 0; k < 25; ++k) z += 0.0 * A[k];
  if (z != 0.0) atomicOr(nonfinite, 1);  // NaN
  int p[5] = {0, 1, 2, 3, 4};
  int row = 0;  // persists across columns, like the reference's
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    double large = 0;
#pragma unroll
    for (int j = c; j < 5; ++j) {
      double v = A[j * 5 + c];
      if (fabs(v) > fabs(large)) {
        large = v;
        row = j;
      }
    }
#pragma unroll
    for (int j = c + 1; j < 5; ++j) {
      if (j == row) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          double t = A[c * 5 + k];
          A[c * 5 + k] = A[j * 5 + k];
          A[j * 5 + k] = t;
        }
        int t = p[c];
        p[c] = p[j];
        p[j] = t;
      }
    }
    large = 1.0 / large;
#pragma unroll
    for (int j = c + 1; j < 5; ++j) A[j * 5 + c] *= large;
#pragma unroll
    for (int j = c + 1; j < 5; ++j)
#pragma unroll
      for (int k = c + 1; k < 5; ++k) A[j * 5 + k] -= A[j * 5 + c] * A[c * 5 + k];
  }
  double id[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) id[k] = 1.0 / A[k * 5 + k];
  // column `col` of the inverse: the unit vector, permuted, through both factors
#pragma unroll
  for (int col = 0; col < 5; ++col) {
    double y[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      double s = (p[k] == col) ? 1.0 : 0.0;
#pragma unroll
      for (int c = 0; c < k; ++c) s -= A[k * 5 + c] * y[c];
      y[k] = s;
    }
#pragma unroll
    for (int k = 4; k >= 0; --k) {
      double s = y[k];
#pragma unroll
      for (int c = 4; c > k; --c) s -= A[k * 5 + c] * y[c];
      y[k] = s * id[k];
      a[(k * 5 + col) * kW] = (T)y[k];
    }
  }
}

void launch_prepare_sgs(Ctx& c) {
  if (c.prm.precision == PCFD_CHOSEN_FP32)
    hipLaunchKernelGGL(k_prepare_sgs<float>, dim3(nblk(c.nrow_pad)), dim3(kBlock), 0, c.stream, c.nrow_pad, c.d.srow,
                       c.d.Df, c.d.icount + 1);
  else
    hipLaunchKernelGGL(k_prepare_sgs<double>, dim3(nblk(c.nrow_pad)), dim3(kBlock), 0, c.stream, c.nrow_pad,
                       c.d.srow, c.d.Dd, c.d.icount + 1);
  PCFD_HIP(hipGetLastError());
}

}  // namespace pcfd
