// Multicolour symmetric block Gauss-Seidel (CRS::SGS, ucs/crs.tcc:61-173).
//
// The reference sweeps rows 0..n-1 then n-1..0 with the newest x.  Rows of
// one colour share no off-diagonal block, so sweeping colour by colour is
// exactly Gauss-Seidel in the colour-sorted row order (and its reverse on the
// way back); within a colour all rows update in parallel.  Blocks are read
// from the SELL layout (the 64 rows of a chunk read one 512-byte (FP64) /
// 256-byte (FP32) line per block entry).  While sweeping, x is 5-wide AoS in
// SELL row order: a pass writes its rows contiguously, and since a colour's
// values lie together, the lines a gather pulls in hold only values of the
// colours the pass reads.
#include <stdexcept>

#include "common.h"
#include "physics.h"

namespace pcfd {

// b (node-order SoA, FP64) -> SELL row order [chunk][eq][lane] in type T
template <typename T>
__global__ void __launch_bounds__(kBlock) k_pack_b(int nrow_pad, int nnode, const int* __restrict__ srow,
                                                  const double* __restrict__ b, T* __restrict__ bs) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrow_pad) return;
  const int i = srow[r];
  T* o = bs + (long long)(r >> 6) * 5 * kW + (r & 63);
#pragma unroll
  for (int k = 0; k < 5; ++k) o[k * kW] = (i >= 0) ? (T)b[k * nnode + i] : (T)0;
}

// Block-matrix entries are read once per symmetric sweep.  A matrix larger
// than the 256 MiB Infinity Cache is loaded non-temporally (it then leaves
// the gathered x lines in L2); a smaller one stays in that cache from sweep
// to sweep and is loaded plainly.  Eight sweeps, non-temporal / plain: bump
// 41^3 FP64 (216 MB) 0.72 / 0.56 ms; bump 64^3 FP32 (401 MB) 0.91 / 0.94;
// bump 100^3 FP32 (1.5 GB) 2.53 / 2.76, FP64 (3 GB) 5.27 / 5.56.
constexpr double kCacheBytes = 256.0 * 1024.0 * 1024.0;

template <bool NT, typename T>
__device__ __forceinline__ T mload(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// One colour pass over half of each row.  In a forward pass the neighbours
// of higher colours still hold the values the last backward pass left, and
// the row's sum over them is what that pass formed; likewise a backward pass
// finds the lower-colour sum of the forward pass unchanged.  So a pass reads
// only the blocks whose neighbours have moved since (the lower-colour run
// forwards, the higher-colour run backwards) and takes the other half's sum
// from `ps`, where it leaves its own: every off-diagonal block is read once
// per symmetric sweep instead of twice.  In the first forward sweep the
// higher-colour neighbours are zero and their blocks are left out, unless the
// matrix holds NaNs or infinities (`nonfinite` given and set): those times zero
// are NaN, and the rows that have them are the rows an update leaves out.
//
// LPR lanes share a row and take alternate slots; their partial sums are
// combined with a fixed exchange (all lanes end with the same value) before
// the first of them applies the inverse of the diagonal block.
//
// What bounds it: a large colour streams its blocks (bump 100^3, eight
// sweeps: 13.6 GB in 2.49 ms FP32, 27.1 GB in 5.05 ms FP64, 5.4 TB/s; a
// plain device copy reaches 4.8).  A small one waits: for the chain of
// dependent loads (row, chunk, column, x, each ~0.5 us), which more lanes per
// row shorten, and for its own instructions, which every CU fetches anew at
// each launch (a straight-line LU solve here cost 14 us a pass on 268
// workgroups whose first instructions missed together, and 0.6 us when
// repeated within a launch).  Hence the inverse: 25 multiply-adds.
// Eight sweeps before (both halves read each way, LU solve) -> now: bump 8^3
// FP64 0.50 -> 0.28 ms, bump 41^3 1.30 -> 0.56 FP64, 0.81 -> 0.38 FP32, bump
// 64^3 2.89 -> 1.74, 1.51 -> 0.91, bump 100^3 8.74 -> 5.05, 4.10 -> 2.49.
template <typename T, int LPR, bool NT>
__global__ void __launch_bounds__(kBlock) k_sgs_color(int row0, int nrows, int backward, int use_ps, int save_ps,
                                                     const int* __restrict__ srow, const int* __restrict__ swidth,
                                                     const int* __restrict__ swidth_lo,
                                                     const int* __restrict__ sbase, const int* __restrict__ scol,
                                                     const T* __restrict__ Moff, const T* __restrict__ Dg,
                                                     const T* __restrict__ bs, T* __restrict__ ps,
                                                     T* __restrict__ x, T* __restrict__ xnode,
                                                     const int* __restrict__ nonfinite) {
  constexpr int RPW = 64 / LPR;  // rows per wavefront
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int l64 = threadIdx.x & 63;
  const int sub = l64 / RPW;
  const int local = (t >> 6) * RPW + l64 % RPW;
  const bool inr = local < nrows;
  const int r = row0 + (inr ? local : 0);
  const int i = inr ? srow[r] : -1;
  const int chunk = r >> 6, lane = r & 63;
  T acc[5] = {0, 0, 0, 0, 0};
  if (i >= 0) {
    const int wl = swidth_lo[chunk];
    const int s0 = backward ? wl : 0, w = backward ? swidth[chunk] : wl;
    const long long cb = (long long)sbase[chunk] * kW + lane;
    const T* mb = Moff + (long long)sbase[chunk] * 25 * kW + lane;
    // the next slot's row index is loaded one iteration ahead, so this
    // slot's x and block loads issue without waiting for it
    int jn = (s0 + sub < w) ? scol[cb + (long long)(s0 + sub) * kW] : -1;
    for (int s = s0 + sub; s < w; s += LPR) {
      const int j = jn;
      if (j < 0) break;
      jn = (s + LPR < w) ? scol[cb + (long long)(s + LPR) * kW] : -1;
      const T* xj = x + (long long)j * 5;
      const T x0 = xj[0], x1 = xj[1], x2 = xj[2], x3 = xj[3], x4 = xj[4];
      const T* blk = mb + (long long)s * 25 * kW;
#pragma unroll
      for (int rr = 0; rr < 5; ++rr) {
        T v = mload<NT>(blk + (rr * 5 + 0) * kW) * x0;
        v += mload<NT>(blk + (rr * 5 + 1) * kW) * x1;
        v += mload<NT>(blk + (rr * 5 + 2) * kW) * x2;
        v += mload<NT>(blk + (rr * 5 + 3) * kW) * x3;
        v += mload<NT>(blk + (rr * 5 + 4) * kW) * x4;
        acc[rr] += v;
      }
    }
    if (nonfinite && __builtin_expect(*nonfinite != 0, 0)) {
      const int wu = swidth[chunk];
      for (int s = wl + sub; s < wu && scol[cb + (long long)s * kW] >= 0; s += LPR) {
        const T* blk = mb + (long long)s * 25 * kW;
#pragma unroll 1
        for (int k = 0; k < 5; ++k)
#pragma unroll
          for (int rr = 0; rr < 5; ++rr) acc[rr] += blk[(rr * 5 + k) * kW] * (T)0;
      }
    }
  }
#pragma unroll
  for (int m = 32; m >= RPW; m >>= 1) {
#pragma unroll
    for (int k = 0; k < 5; ++k) acc[k] += __shfl_xor(acc[k], m);
  }
  if (i < 0 || sub != 0) return;
  T rhs[5];
  const long long v0 = (long long)chunk * 5 * kW + lane;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    T s = acc[k];
    if (use_ps) s += ps[v0 + k * kW];
    if (save_ps) ps[v0 + k * kW] = acc[k];
    rhs[k] = bs[v0 + k * kW] - s;
  }
  const T* dg = Dg + (long long)chunk * 25 * kW + lane;
  T v[5];
#pragma unroll
  for (int rr = 0; rr < 5; ++rr) {
    v[rr] = mload<NT>(dg + rr * 5 * kW) * rhs[0];
#pragma unroll
    for (int k = 1; k < 5; ++k) v[rr] += mload<NT>(dg + (rr * 5 + k) * kW) * rhs[k];
  }
  T* xo = x + (long long)r * 5;
#pragma unroll
  for (int k = 0; k < 5; ++k) xo[k] = v[k];
  if (xnode) {
    T* xn = xnode + (long long)i * 5;
#pragma unroll
    for (int k = 0; k < 5; ++k) xn[k] = v[k];
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_zero(long long n, T* __restrict__ x) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = (T)0;
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_sumsq_x(int nrow, const T* __restrict__ x, double* __restrict__ red) {
  __shared__ double sh[kBlock];
  double s = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nrow; i += gridDim.x * blockDim.x) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      double v = (double)x[(long long)i * 5 + k];
      s += v * v;
    }
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) red[blockIdx.x] = sh[0];
}

template <typename T>
static double xnorm(Ctx& c, const T* x) {
  const int nb = 512;
  hipLaunchKernelGGL(k_sumsq_x<T>, dim3(nb), dim3(kBlock), 0, c.stream, c.nrow_pad, x, c.d.red);
  PCFD_HIP(hipGetLastError());
  double h[nb];
  PCFD_HIP(hipMemcpyAsync(h, c.d.red, sizeof(h), hipMemcpyDeviceToHost, c.stream));
  PCFD_HIP(hipStreamSynchronize(c.stream));
  double s = 0.0;
  for (int k = 0; k < nb; ++k) s += h[k];
  return std::sqrt(s) / (double)(5LL * c.nnode);
}

// Lanes per row of a colour of `nrows` rows: enough wavefronts to cover the
// chip's latency, no more (each lane's share of a 128-byte line of block
// entries shrinks with LPR).  Eight sweeps at 8 / 4 / 2 / 1 lanes, ms: 183 rows
// a colour 0.28 / 0.32 / 0.39 / 0.45 (FP64); 2.3k rows 0.31 / 0.35 / 0.46 /
// 0.69 (FP64); 9k rows 0.39 / 0.37 / 0.45 / 0.53 (FP32); 18.5k rows 0.66 / 0.60 /
// 0.56 / 0.78 (FP64); 69k rows 2.36 / 1.80 / 1.74 / 1.95 (FP64); 258k rows 8.5 /
// 5.65 / 5.27 / 5.05 (FP64).
static int lanes_per_row(int nrows) { return nrows <= 4096 ? 8 : nrows <= 12288 ? 4 : nrows <= 131072 ? 2 : 1; }

template <typename T, bool NT>
static void sgs_pass(Ctx& c, int row0, int nrows, bool backward, bool use_ps, bool save_ps, const T* Moff,
                     const T* Dg, const T* bs, T* ps, T* x, T* xnode, const int* nonfinite) {
  const int lpr = lanes_per_row(nrows);
  auto kern = lpr == 1 ? k_sgs_color<T, 1, NT>
              : lpr == 2 ? k_sgs_color<T, 2, NT> : lpr == 4 ? k_sgs_color<T, 4, NT> : k_sgs_color<T, 8, NT>;
  hipLaunchKernelGGL(kern, dim3(nblk((long long)nrows * lpr)), dim3(kBlock), 0, c.stream, row0, nrows, (int)backward,
                     (int)use_ps, (int)save_ps, c.d.srow, c.d.swidth, c.d.swidth_lo, c.d.sbase, c.d.scol, Moff, Dg,
                     bs, ps, x, xnode, nonfinite);
  PCFD_HIP(hipGetLastError());
}

template <typename T>
static void sgs_impl(Ctx& c, int nsgs, const T* Moff, const T* Dg, T* bs, T* ps, T* x, T* xnode, double* delta) {
  if (nsgs == 0) {
    const long long n5 = 5LL * c.nnode;
    hipLaunchKernelGGL(k_zero<T>, dim3(nblk(n5)), dim3(kBlock), 0, c.stream, n5, xnode);
    PCFD_HIP(hipGetLastError());
    if (delta) *delta = 0.0;
    return;
  }
  hipLaunchKernelGGL(k_pack_b<T>, dim3(nblk(c.nrow_pad)), dim3(kBlock), 0, c.stream, c.nrow_pad, c.nnode, c.d.srow,
                     c.d.b, bs);
  PCFD_HIP(hipGetLastError());
  double xold = 0.0, xn = 0.0;
  // A colour pass directly after a pass over the same colour (the turn of
  // each symmetric sweep, and the start of the next forward sweep) reads the
  // same neighbour x and writes the same values bit for bit: the rows of a
  // colour never read each other.  Those passes are skipped.  x = 0 at the
  // start, so the first forward sweep has no higher-colour sums: it reads
  // only values it has written, and x needs no clearing.  The first and the
  // last colour have neighbours on one side only and keep no partial sums.
  const int C = c.ncolor;
  const bool streamed = (double)c.nslot_s * kW * 25 * sizeof(T) > kCacheBytes;
  int last = -1;
  for (int it = 0; it < nsgs; ++it) {
    sub_begin(c);
    for (int dir = 0; dir < 2; ++dir) {
      for (int cc = 0; cc < C; ++cc) {
        const int col = dir == 0 ? cc : C - 1 - cc;
        if (col == last) continue;
        last = col;
        const bool inner = col > 0 && col < C - 1;
        const bool first_pass = it == 0 && dir == 0;
        // the pass after which the colour's x does not change any more
        const bool last_pass = C == 1 || (it == nsgs - 1 && (dir == 1 || col == C - 1));
        const int row0 = c.color_chunk[col] * kW;
        const int nrows = (c.color_chunk[col + 1] - c.color_chunk[col]) * kW;
        (streamed ? sgs_pass<T, true> : sgs_pass<T, false>)(c, row0, nrows, dir == 1, inner && !first_pass,
                                                            inner && !last_pass, Moff, Dg, bs, ps, x,
                                                            last_pass ? xnode : nullptr,
                                                            first_pass ? c.d.icount + 1 : nullptr);
      }
    }
    sub_end(c, 9);
    if (delta && it >= nsgs - 2) {
      xold = xn;
      xn = xnorm(c, x);
    }
  }
  if (delta) *delta = std::fabs(xold - xn);
}

void launch_sgs(Ctx& c, int nsgs, double* delta) {
  if (c.prm.precision == PCFD_CHOSEN_FP32)
    sgs_impl<float>(c, nsgs, c.d.Mf, c.d.Df, c.d.bsf, c.d.psf, c.d.xsf, c.d.xf, delta);
  else
    sgs_impl<double>(c, nsgs, c.d.Md, c.d.Dd, c.d.bsd, c.d.psd, c.d.xsd, c.d.xd, delta);
}

}  // namespace pcfd
