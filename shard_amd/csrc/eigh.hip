// Top eigenpairs of a symmetric float64 matrix on gfx950: the PCA basis of a
// layer's key covariance (the quantities _compress_k takes from svd_lowrank,
// cache.py:376-378).
//
//   1. Householder tridiagonalization, one launch per column (k_tridiag).
//   2. k_tri_eig, a wave per wanted eigenvalue: multisection with Sturm counts
//      (64 points a pass), then the eigenvector of the tridiagonal matrix by a
//      twisted factorization.
//   3. k_back, a wave per eigenvector: the reflectors applied in reverse.
//
// The vectors of eigenvalues closer than about 1e-7 of the largest one lose
// orthogonality in step 2 (no reorthogonalization): the caller checks V^T V and
// the residual and takes a library routine where they miss its bound.
#include "common.h"

namespace shard {

constexpr int kEigMax = 1024;         // largest order
constexpr int kEigE = kEigMax / 64;   // elements per lane of a row

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 0xF, 0xF, false);
  const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sum over the wave, in every lane (a fixed order).
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_f64<kDppXor1>(v);
  v += dpp_f64<kDppXor2>(v);
  v += dpp_f64<kDppHalfMirror>(v);
  v += dpp_f64<kDppMirror>(v);
  uint64_t u = __builtin_bit_cast(uint64_t, v);
  auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)u, false, false);
  auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  v = __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
      __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
  u = __builtin_bit_cast(uint64_t, v);
  lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)u, false, false);
  hi = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}

// Launch k of the tridiagonalization (k = 0 .. n - 2).  On entry the rows of A
// hold the matrix after the updates of columns 0 .. k - 2; row k - 1 of V is
// the reflector of column k - 1 (leading element 1 at k, zeros before), pin =
// A v of it.  Every workgroup forms the whole of w = tau p - tau^2 (p . v) v / 2
// and, from row k, the updated column k and its reflector (a few thousand
// operations, cheaper than a second launch), then each wave updates one row
// i > k with v w^T + w v^T and takes its product with the new reflector:
// one launch, one pass over the trailing matrix, per column.  The last
// workgroup, active to the end, writes d, e, tau and V's row k.  5.2 us a launch
// at n = 1024 (6.6 ms the whole solve; 5.9 traced with other work on the GPU), the
// launch itself and two block reductions; the matrix (8 MB, read and written once
// a launch) stays in the last-level cache.
__global__ __launch_bounds__(256)
void k_tridiag(double* __restrict__ A, int n, int k, const double* __restrict__ pin,
               double* __restrict__ pout, double* __restrict__ V, double* __restrict__ d,
               double* __restrict__ e, double* __restrict__ tau) {
  __shared__ double vo[kEigMax], wo[kEigMax], vn[kEigMax];
  __shared__ double part[4], part2[4], head[2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x * 4 + 3 <= k) return;  // no row left (whole workgroup)
  const int i = (int)blockIdx.x * 4 + w;     // this wave's row
  const bool mine = i > k && i < n;
  const int m0 = (k + 1) >> 6;               // 64-column groups before it are done
  double row[kEigE];
#pragma unroll
  for (int m = 0; m < kEigE; ++m) {
    const int j = lane + 64 * m;
    row[m] = (m >= m0 && mine && j < n) ? A[(int64_t)i * n + j] : 0.0;
  }
  // ---- w of the previous reflector
  constexpr int TE = kEigMax / 256;
  double pv[TE], vv[TE], ak[TE], dot = 0.0;
#pragma unroll
  for (int m = 0; m < TE; ++m) {
    const int j = tid + 256 * m;
    const bool in = j >= k && j < n;
    vv[m] = in && k > 0 ? V[(int64_t)(k - 1) * n + j] : 0.0;
    pv[m] = in && k > 0 ? pin[j] : 0.0;
    ak[m] = in ? A[(int64_t)k * n + j] : 0.0;
    dot += vv[m] * pv[m];
  }
  const double t = k > 0 ? tau[k - 1] : 0.0;
  dot = wave_sum(dot);
  if (lane == 0) part[w] = dot;
  __syncthreads();
  const double half = 0.5 * t * t * (part[0] + part[1] + part[2] + part[3]);
#pragma unroll
  for (int m = 0; m < TE; ++m) {
    pv[m] = t * pv[m] - half * vv[m];
    const int j = tid + 256 * m;
    vo[j] = vv[m];
    wo[j] = pv[m];
  }
  __syncthreads();
  // ---- column k after that update, and its reflector
  const double vk = vo[k], wk = wo[k];
  double sq = 0.0;
#pragma unroll
  for (int m = 0; m < TE; ++m) {
    const int j = tid + 256 * m;
    ak[m] -= vv[m] * wk + pv[m] * vk;
    if (j > k + 1) sq += ak[m] * ak[m];  // elements past n are zero
    if (j == k) head[0] = ak[m];
    if (j == k + 1) head[1] = ak[m];
  }
  sq = wave_sum(sq);
  if (lane == 0) part2[w] = sq;
  __syncthreads();
  sq = part2[0] + part2[1] + part2[2] + part2[3];
  const double alpha = head[1];
  double beta = alpha, tn = 0.0, scale = 0.0;
  if (sq > 0.0) {
    beta = -copysign(sqrt(alpha * alpha + sq), alpha);
    tn = (beta - alpha) / beta;
    scale = 1.0 / (alpha - beta);
  }
  const bool last = blockIdx.x == gridDim.x - 1;
#pragma unroll
  for (int m = 0; m < TE; ++m) {
    const int j = tid + 256 * m;
    const double x = j <= k ? 0.0 : j == k + 1 ? 1.0 : ak[m] * scale;
    vn[j] = x;
    if (last && j < n) V[(int64_t)k * n + j] = x;
  }
  if (last && tid == 0) {
    d[k] = head[0];
    e[k] = beta;
    tau[k] = tn;
  }
  __syncthreads();
  // ---- the wave's row: rank-2 update, product with the new reflector
  if (!mine) return;
  const double vi = vo[i], wi = wo[i];
  double p = 0.0;
#pragma unroll
  for (int m = 0; m < kEigE; ++m) {
    if (m < m0) continue;
    const int j = lane + 64 * m;
    if (j < n) {
      const double x = row[m] - vi * wo[j] - wi * vo[j];
      A[(int64_t)i * n + j] = x;
      p += x * vn[j];
      if (k == n - 2 && j == n - 1) d[n - 1] = x;
    }
  }
  p = wave_sum(p);
  if (lane == 0) pout[i] = p;
}

// 1 / q to working precision (the hardware estimate and two Newton steps).
__device__ __forceinline__ double fast_rcp(double q) {
  double r = __builtin_amdgcn_rcp(q);
  r = __builtin_fma(__builtin_fma(-q, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-q, r, 1.0), r, r);
}

// Eigenpair m of the tridiagonal matrix (d, e), m-th from the top, on one wave.
// Eigenvalue: an interval that holds it shrinks 65-fold a pass, the 64 lanes
// counting the eigenvalues below 64 inner points.  Vector: forward and
// backward pivots s, p of T - lambda (lanes 0 and 1), the twist at the
// smallest |s_i + p_i - (d_i - lambda)|, then the two products outward from it.
// A lane's chain of n dependent steps bounds it (about 110 clocks a step).
constexpr int kEigPasses = 11;
__global__ __launch_bounds__(64)
void k_tri_eig(const double* __restrict__ dg, const double* __restrict__ eg, int n,
               double* __restrict__ evals, double* __restrict__ Z) {
  __shared__ double d[kEigMax], e[kEigMax], s[kEigMax], p[kEigMax];
  const int lane = threadIdx.x, m = blockIdx.x, want = n - 1 - m;  // ascending index
  double lo = INFINITY, hi = -INFINITY;
  for (int i = lane; i < n; i += 64) {
    d[i] = dg[i];
    e[i] = i < n - 1 ? eg[i] : 0.0;
    const double r = fabs(e[i]) + (i > 0 ? fabs(eg[i - 1]) : 0.0);
    lo = fmin(lo, d[i] - r);
    hi = fmax(hi, d[i] + r);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o));
    hi = fmax(hi, __shfl_xor(hi, o));
  }
  __syncthreads();
  const double norm = fmax(fabs(lo), fabs(hi));
  const double tiny = fmax(norm * 1e-30, 1e-290);  // smallest pivot
  lo -= 1e-14 * norm + tiny;
  hi += 1e-14 * norm + tiny;
#pragma unroll 1
  for (int pass = 0; pass < kEigPasses; ++pass) {
    const double step = (hi - lo) / 65.0, x = lo + step * (lane + 1);
    int below = 0;
    double q = 1.0, e2 = 0.0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) {
      q = (d[i] - x) - e2 * fast_rcp(q);
      if (fabs(q) < tiny) q = -tiny;
      below += q < 0.0;
      e2 = e[i] * e[i];
    }
    // points [0, c) have at most `want` eigenvalues below them
    const uint64_t over = __builtin_amdgcn_ballot_w64(below > want);
    const int c = over ? __builtin_ctzll(over) : 64;
    const double base = lo;
    lo = base + step * c;
    if (c < 64) hi = base + step * (c + 1);
  }
  const double lam = 0.5 * (lo + hi);
  if (lane == 0) evals[m] = lam;
  // ---- twisted factorization
  if (lane < 2) {
    double q = 1.0, e2 = 0.0;
    double* dst = lane == 0 ? s : p;
#pragma unroll 8
    for (int j = 0; j < n; ++j) {
      const int i = lane == 0 ? j : n - 1 - j;
      q = (d[i] - lam) - e2 * fast_rcp(q);
      if (fabs(q) < tiny) q = -tiny;
      dst[i] = q;
      const double ei = lane == 0 ? e[i] : i > 0 ? e[i - 1] : 0.0;
      e2 = ei * ei;
    }
  }
  __syncthreads();
  double best = INFINITY;
  int at = 0;
  for (int i = lane; i < n; i += 64) {
    const double g = fabs(s[i] + p[i] - (d[i] - lam));
    if (g < best) {
      best = g;
      at = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double g = __shfl_xor(best, o);
    const int a = __shfl_xor(at, o);
    if (g < best || (g == best && a < at)) {
      best = g;
      at = a;
    }
  }
  __syncthreads();
  // ratios: z_i = -(e_i / s_i) z_{i+1} below the twist, -(e_{i-1} / p_i) z_{i-1} above it
  for (int i = lane; i < n; i += 64) {
    s[i] = -e[i] / s[i];
    p[i] = i > 0 ? -e[i - 1] / p[i] : 0.0;
  }
  __syncthreads();
  if (lane < 2) {
    double z = 1.0;
    if (lane == 0) {
#pragma unroll 8
      for (int i = at - 1; i >= 0; --i) d[i] = z = s[i] * z;
    } else {
#pragma unroll 8
      for (int i = at + 1; i < n; ++i) d[i] = z = p[i] * z;
      d[at] = 1.0;
    }
  }
  __syncthreads();
  double sq = 0.0;
  for (int i = lane; i < n; i += 64) sq += d[i] * d[i];
  const double inv = 1.0 / sqrt(wave_sum(sq));
  for (int i = lane; i < n; i += 64) Z[(int64_t)m * n + i] = d[i] * inv;
}

// Row m of Z (an eigenvector of the tridiagonal matrix) times the reflectors,
// last column's first: z -= tau_k (v_k . z) v_k.  One wave per vector, the
// vector in registers, the next reflector's loads in flight.
__global__ __launch_bounds__(64)
void k_back(const double* __restrict__ V, const double* __restrict__ tau, int n,
            double* __restrict__ Z) {
  const int lane = threadIdx.x;
  double* zr = Z + (int64_t)blockIdx.x * n;
  double z[kEigE];
#pragma unroll
  for (int m = 0; m < kEigE; ++m) z[m] = lane + 64 * m < n ? zr[lane + 64 * m] : 0.0;
  constexpr int RB = 2;
  double v[RB][kEigE], t[RB];
  auto load = [&](int k, double (&x)[kEigE], double& tk) {
    const int kk = max(k, 0);
    tk = k >= 0 ? tau[kk] : 0.0;
#pragma unroll
    for (int m = 0; m < kEigE; ++m) {
      const int j = lane + 64 * m;
      x[m] = j < n ? V[(int64_t)kk * n + j] : 0.0;
    }
  };
  auto apply = [&](const double (&x)[kEigE], double tk) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int m = 0; m < kEigE; m += 2) {
      a += x[m] * z[m];
      b += x[m + 1] * z[m + 1];
    }
    const double c = tk * wave_sum(a + b);
#pragma unroll
    for (int m = 0; m < kEigE; ++m) z[m] -= c * x[m];
  };
  load(n - 2, v[0], t[0]);
#pragma unroll 1
  for (int k = n - 2; k >= 0; k -= 2) {
    load(k - 1, v[1], t[1]);
    apply(v[0], t[0]);
    load(k - 2, v[0], t[0]);
    apply(v[1], t[1]);
  }
#pragma unroll
  for (int m = 0; m < kEigE; ++m)
    if (lane + 64 * m < n) zr[lane + 64 * m] = z[m];
}

}  // namespace shard

using namespace shard;

extern "C" {

// V (n - 1 reflectors of n), two p vectors, d, e, tau
size_t shard_eigh_top_workspace(int32_t n) {
  return n < 2 || n > kEigMax ? 0 : ((size_t)n * n + 5 * (size_t)n) * sizeof(double);
}

int shard_eigh_top(double* a, int32_t n, int32_t top, double* evals, double* evecs,
                   void* workspace, size_t workspace_bytes, void* stream) {
  if (!a || !evals || !evecs || !workspace || top <= 0) return SHARD_ERR_ARG;
  if (n < 2 || n > kEigMax || top > n) return SHARD_ERR_SHAPE;
  if (workspace_bytes < shard_eigh_top_workspace(n)) return SHARD_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  double* V = (double*)workspace;
  double* p[2] = {V + (size_t)n * n, V + (size_t)n * n + n};
  double *d = p[1] + n, *e = d + n, *tau = e + n;
  const dim3 grid((unsigned)((n + 3) / 4));
  for (int k = 0; k < n - 1; ++k)
    hipLaunchKernelGGL(k_tridiag, grid, dim3(256), 0, s, a, n, k, p[k & 1], p[(k + 1) & 1], V, d, e, tau);
  hipLaunchKernelGGL(k_tri_eig, dim3((unsigned)top), dim3(64), 0, s, d, e, n, evals, evecs);
  hipLaunchKernelGGL(k_back, dim3((unsigned)top), dim3(64), 0, s, V, tau, n, evecs);
  SHARD_LAUNCH_CHECK("shard_eigh_top");
  return SHARD_OK;
}

}  // extern "C"
