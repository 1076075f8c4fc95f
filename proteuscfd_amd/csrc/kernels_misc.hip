// Solution update: NaN/Inf rows of the correction zeroed, then ApplyDQ
// (ucs/solutionSpace.tcc:772-804, ucs/compressible.tcc:928-993), and the
// explicit update (ExplicitSolve, ucs/solve.tcc:70-101).
#include <algorithm>
#include <stdexcept>
#include <vector>

#include "common.h"
#include "fill.h"
#include "physics.h"
#include "scan.h"

namespace pcfd {

template <typename T>
__global__ void __launch_bounds__(kBlock) k_apply_dq(int nnode, int ntot, double gamma, T* __restrict__ x,
                                                    double* __restrict__ q, int* __restrict__ count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnode) return;
  double dq[5], Q[5];
  bool zero = false;
  T* xi = x + (long long)i * 5;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    dq[k] = (double)xi[k];
    if (__builtin_isnan(dq[k]) || __builtin_isinf(dq[k])) zero = true;
    Q[k] = q[k * ntot + i];
  }
  if (zero) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      dq[k] = 0.0;
      xi[k] = (T)0;
    }
    atomicAdd(count, 1);
  }
  apply_dq(dq, Q, gamma);
#pragma unroll
  for (int k = 0; k < 5; ++k) q[k * ntot + i] = Q[k];
}

// ExplicitSolve x = b*dt/vol with ApplyDQ, then NewtonIterate's update, which
// applies the same x a second time (the reference calls ApplyDQ in both).
__global__ void __launch_bounds__(kBlock) k_explicit(int nnode, int ntot, double gamma, const double* __restrict__ b,
                                                    const double* __restrict__ dt, const double* __restrict__ vol,
                                                    double* __restrict__ q, int* __restrict__ count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnode) return;
  double dq[5], Q[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    dq[k] = b[k * nnode + i] * dt[i] / vol[i];
    Q[k] = q[k * ntot + i];
  }
  apply_dq(dq, Q, gamma);
  bool zero = false;
#pragma unroll
  for (int k = 0; k < 5; ++k)
    if (__builtin_isnan(dq[k]) || __builtin_isinf(dq[k])) zero = true;
  if (zero) {
#pragma unroll
    for (int k = 0; k < 5; ++k) dq[k] = 0.0;
    atomicAdd(count, 1);
  }
  apply_dq(dq, Q, gamma);
#pragma unroll
  for (int k = 0; k < 5; ++k) q[k * ntot + i] = Q[k];
}

__global__ void k_zero_int(int* p) { *p = 0; }

__global__ void __launch_bounds__(kBlock) k_zero_words(size_t n, unsigned* __restrict__ p) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

void launch_zero(hipStream_t stream, void* p, size_t n) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_zero_words, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream, n,
                     (unsigned*)p);
  PCFD_HIP(hipGetLastError());
}

// One stage of the four-stage Runge-Kutta extension: Q = Q0 + a dt/vol b
// through ApplyDQ; a row whose correction is NaN/Inf keeps Q0 (counted).
__global__ void __launch_bounds__(kBlock) k_rk_stage(int nnode, int ntot, double gamma, double a,
                                                    const double* __restrict__ b, const double* __restrict__ dt,
                                                    const double* __restrict__ vol, const double* __restrict__ q0,
                                                    double* __restrict__ q, int* __restrict__ count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnode) return;
  double dq[5], Q[5];
  bool zero = false;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    dq[k] = a * (b[k * nnode + i] * dt[i] / vol[i]);
    if (__builtin_isnan(dq[k]) || __builtin_isinf(dq[k])) zero = true;
    Q[k] = q0[k * ntot + i];
  }
  if (zero) {
#pragma unroll
    for (int k = 0; k < 5; ++k) dq[k] = 0.0;
    atomicAdd(count, 1);
  }
  apply_dq(dq, Q, gamma);
#pragma unroll
  for (int k = 0; k < 5; ++k) q[k * ntot + i] = Q[k];
}

void launch_zero_count(Ctx& c) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, c.stream, c.d.icount);
  PCFD_HIP(hipGetLastError());
}

void launch_rk_stage(Ctx& c, double a, const double* q0) {
  hipLaunchKernelGGL(k_rk_stage, dim3(nblk(c.nnode)), dim3(kBlock), 0, c.stream, c.nnode, c.ntot, c.prm.gamma, a,
                     c.d.b, c.d.dt, c.d.vol, q0, c.d.q, c.d.icount);
  PCFD_HIP(hipGetLastError());
}

// Exclusive prefix sum of per-pass counts (one workgroup of 1024, fixed
// order): off[p] = sum of cnt[0..p-1], off[npass] = total.  Used to compact
// lists in order without atomics (the surrogate's fallback cells, the
// pressure clip's candidate edges).
// Counts are read in coalesced tiles of 1024, up to kScanTiles tiles at a
// time so their loads are in flight together; each tile is scanned with
// wavefront shuffles plus one pass over the 16 wavefront totals.
constexpr int kScanBlock = 1024;
constexpr int kScanTiles = 16;

__global__ void __launch_bounds__(kScanBlock) k_scan_counts(int npass, const int* __restrict__ cnt,
                                                                int* __restrict__ off) {
  __shared__ int wsum[kScanBlock / 64];
  __shared__ int carry_sh;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  if (t == 0) carry_sh = 0;
  __syncthreads();
  for (int base = 0; base < npass; base += kScanBlock * kScanTiles) {
    int v[kScanTiles];
#pragma unroll
    for (int k = 0; k < kScanTiles; ++k) {
      const int p = base + k * kScanBlock + t;
      v[k] = p < npass ? cnt[p] : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanTiles; ++k) {
      // inclusive scan within the wavefront
      int x = v[k];
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
      }
      if (lane == 63) wsum[wv] = x;
      __syncthreads();
      int before = carry_sh;
      for (int u = 0; u < wv; ++u) before += wsum[u];
      const int p = base + k * kScanBlock + t;
      if (p < npass) off[p] = before + x - v[k];
      __syncthreads();
      if (t == kScanBlock - 1) carry_sh = before + x;
      __syncthreads();
    }
  }
  if (t == 0) off[npass] = carry_sh;
}

void launch_scan_counts(hipStream_t stream, int n, const int* cnt, int* off) {
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(kScanBlock), 0, stream, n, cnt, off);
  PCFD_HIP(hipGetLastError());
}


void launch_apply_dq(Ctx& c, int explicit_mode, int* nzeroed) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, c.stream, c.d.icount);
  PCFD_HIP(hipGetLastError());
  if (explicit_mode) {
    hipLaunchKernelGGL(k_explicit, dim3(nblk(c.nnode)), dim3(kBlock), 0, c.stream, c.nnode, c.ntot, c.prm.gamma,
                       c.d.b, c.d.dt, c.d.vol, c.d.q, c.d.icount);
  } else if (c.prm.precision == PCFD_CHOSEN_FP32) {
    hipLaunchKernelGGL(k_apply_dq<float>, dim3(nblk(c.nnode)), dim3(kBlock), 0, c.stream, c.nnode, c.ntot,
                       c.prm.gamma, c.d.xf, c.d.q, c.d.icount);
  } else {
    hipLaunchKernelGGL(k_apply_dq<double>, dim3(nblk(c.nnode)), dim3(kBlock), 0, c.stream, c.nnode, c.ntot,
                       c.prm.gamma, c.d.xd, c.d.q, c.d.icount);
  }
  PCFD_HIP(hipGetLastError());
  if (nzeroed) {
    PCFD_HIP(hipMemcpyAsync(nzeroed, c.d.icount, sizeof(int), hipMemcpyDeviceToHost, c.stream));
    PCFD_HIP(hipStreamSynchronize(c.stream));
  }
}

// ---- callers' arrays ---------------------------------------------------------
// A caller's arrays hold a node's components together, the device one array a
// component.  The reordering is the device's: it is one pass at memory speed
// there, and the caller's array is filled by a single copy.  (On the host, with
// its own buffer between the copy and the reordering, the gradient of 39k nodes,
// 8.5 MB, took 1450 us to reach the caller; 650 so.)

// aos[i * stride + k] = soa[k * ld + i], k < ncomp
__global__ void __launch_bounds__(kBlock) k_to_aos(long long n, int ncomp, int ld, const double* __restrict__ soa,
                                                  double* __restrict__ aos) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * ncomp) return;
  aos[t] = soa[t % ncomp * ld + t / ncomp];
}

__global__ void __launch_bounds__(kBlock) k_from_aos(int n, int ncomp, int ld, int stride,
                                                    const double* __restrict__ aos, double* __restrict__ soa) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int k = 0; k < ncomp; ++k) soa[(long long)k * ld + i] = aos[(long long)i * stride + k];
}

// rows of the full state: the conservative values and what follows from them,
// in the host's arithmetic (no contracted products)
__global__ void __launch_bounds__(kBlock) k_full_state(int ntot, double gamma, const double* __restrict__ q,
                                                      double* __restrict__ aos) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ntot) return;
  double Q[10];
#pragma unroll
  for (int k = 0; k < 5; ++k) Q[k] = q[(long long)k * ntot + i];
  const double gm1 = gamma - 1.0;
  const double u = Q[1] / Q[0], v = Q[2] / Q[0], w = Q[3] / Q[0];
  const double P = gm1 * (Q[4] - 0.5 * Q[0] * (u * u + v * v + w * w));
  const double v2h = 0.5 * (u * u + v * v + w * w);
  Q[5] = gamma * (gm1 * (Q[4] - Q[0] * v2h)) / Q[0];
  Q[6] = P;
  Q[7] = u;
  Q[8] = v;
  Q[9] = w;
#pragma unroll
  for (int k = 0; k < 10; ++k) aos[(long long)i * 10 + k] = Q[k];
}

__global__ void __launch_bounds__(kBlock) k_ones(size_t n, double* __restrict__ v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = 1.0;
}

static double* aos_space(Ctx& c, size_t n) {
  if (c.d.aos_n < n) {
    // the stream may still be reading the old one
    PCFD_HIP(hipStreamSynchronize(c.stream));
    if (c.d.aos) PCFD_HIP(hipFree(c.d.aos));
    c.d.aos = nullptr;
    c.d.aos_n = 0;
    PCFD_HIP(hipMalloc((void**)&c.d.aos, sizeof(double) * n));
    c.d.aos_n = n;
  }
  return c.d.aos;
}

// Where a kernel leaves or finds a caller's array of n values: up to pin_n in
// pinned host memory, which the host copies to or from itself, more in device
// memory.  A copy engine's start costs more than the kernel's own trip over the
// bus: 37k values went up in 137 and came down in 154 us through device memory,
// in 26 and 30 through pinned; at 220k both took 80-100 and 130-140.
static double* space_of(Ctx& c, size_t n) { return n <= c.pin_n ? c.pin_dev + kPinHead : aos_space(c, n); }

// the n rows of ncomp values a kernel has left there into the caller's rows of
// `stride` values, the stream's work done on return
static void rows_to_host(Ctx& c, size_t n, int ncomp, double* host, int stride) {
  const size_t m = n * ncomp;
  const double* src = c.pin + kPinHead;
  std::vector<double> s;
  if (m <= c.pin_n) {
    PCFD_HIP(hipStreamSynchronize(c.stream));
    if (stride == ncomp) std::copy(src, src + m, host);
  } else {
    double* to = host;
    if (stride != ncomp) {
      s.resize(m);
      src = to = s.data();
    }
    PCFD_HIP(hipMemcpyAsync(to, c.d.aos, sizeof(double) * m, hipMemcpyDeviceToHost, c.stream));
    PCFD_HIP(hipStreamSynchronize(c.stream));
  }
  if (stride != ncomp)
    for (size_t i = 0; i < n; ++i)
      for (int k = 0; k < ncomp; ++k) host[i * stride + k] = src[i * ncomp + k];
}

void soa_to_host(Ctx& c, const double* soa, int ld, int n, int ncomp, double* host) {
  const size_t m = (size_t)n * ncomp;
  if (ncomp == 1 && m > c.pin_n) {
    PCFD_HIP(hipMemcpyAsync(host, soa, sizeof(double) * m, hipMemcpyDeviceToHost, c.stream));
    PCFD_HIP(hipStreamSynchronize(c.stream));
    return;
  }
  hipLaunchKernelGGL(k_to_aos, dim3((unsigned)((m + kBlock - 1) / kBlock)), dim3(kBlock), 0, c.stream, (long long)n,
                     ncomp, ld, soa, space_of(c, m));
  PCFD_HIP(hipGetLastError());
  rows_to_host(c, n, ncomp, host, ncomp);
}

// rows of up to kWide values go up as they are; of wider ones only what is read
constexpr int kWide = 10;

void soa_from_host(Ctx& c, double* soa, int ld, int n, int ncomp, const double* host, int stride) {
  std::vector<double> s;
  if (stride > kWide) {
    s.resize((size_t)n * ncomp);
    for (size_t i = 0; i < (size_t)n; ++i)
      for (int k = 0; k < ncomp; ++k) s[i * ncomp + k] = host[i * stride + k];
    host = s.data();
    stride = ncomp;
  }
  // the last row's columns past the components are not read: a caller's array
  // may end with them
  const size_t m = (size_t)(n - 1) * stride + ncomp;
  double* aos = space_of(c, m);
  if (m <= c.pin_n) {
    // nothing on the stream still reads the pinned rows: every use waits for its own
    std::copy(host, host + m, c.pin + kPinHead);
  } else {
    PCFD_HIP(hipMemcpyAsync(aos, host, sizeof(double) * m, hipMemcpyHostToDevice, c.stream));
  }
  hipLaunchKernelGGL(k_from_aos, dim3(nblk(n)), dim3(kBlock), 0, c.stream, n, ncomp, ld, stride, aos, soa);
  PCFD_HIP(hipGetLastError());
  PCFD_HIP(hipStreamSynchronize(c.stream));
}

void state_to_host(Ctx& c, double gamma, double* host, int nvars) {
  const int ncol = nvars >= 10 ? 10 : 5;
  double* aos = space_of(c, (size_t)c.ntot * ncol);
  if (ncol == 10)
    hipLaunchKernelGGL(k_full_state, dim3(nblk(c.ntot)), dim3(kBlock), 0, c.stream, c.ntot, gamma, c.d.q, aos);
  else
    hipLaunchKernelGGL(k_to_aos, dim3((unsigned)((5LL * c.ntot + kBlock - 1) / kBlock)), dim3(kBlock), 0, c.stream,
                       (long long)c.ntot, 5, c.ntot, c.d.q, aos);
  PCFD_HIP(hipGetLastError());
  rows_to_host(c, (size_t)c.ntot, ncol, host, nvars);
}

void launch_ones(Ctx& c, size_t n, double* v) {
  hipLaunchKernelGGL(k_ones, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, c.stream, n, v);
  PCFD_HIP(hipGetLastError());
}

}  // namespace pcfd
