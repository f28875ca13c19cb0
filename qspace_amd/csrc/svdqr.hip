// svdqr.hip -- QR preconditioning of the block SVD (after Drmac and Veselic,
// SIAM J. Matrix Anal. Appl. 29 (2008) 1322): the columns of a group matrix A
// (m x n, m >= n) in order of falling norm, A P = Q1 R1, then R1^T = Q2 R2
// (Householder, compact WY form of panels of 16 columns; Golub and Van Loan,
// Matrix Computations, 5.1-5.2), and the Jacobi sweeps (svd.hip) run on the
// n x n matrix X = R2^T instead of A.  With X W = U S:
//   A = (Q1 U) S (P Q2 W)^T.
// Sweeps until nothing rotates (numpy model of the round-robin order, entries
// falling over six decades / random), A itself: 27 / 11 at 246 x 187, 21 / 9 at
// 128 x 64; R1^T of the sorted columns: 11 / 11, 9 / 9; R2^T: 8 / 10, 7 / 9.
#include <cfloat>

#include "qsx_internal.hpp"
#include "lanes.hpp"

namespace qsx {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int QR_NT = 1024;  // one wave per panel column
constexpr int APPLY_NT = 256;

// C(r0.., c0..c0+15) <- (I - V op(T) V^T) C on one wave; V (16 columns, LDS,
// leading dim ldv) is zero above row r0, T is upper triangular (row-major
// 16 x 16, LDS), op(T) = T^T for TRANS (the factor Q^T of a factorisation).
// C is column-major with ldc a multiple of 16.  Lane l holds rows
// r + 4(l/16) .. +3 of column l%16 of each 16-row chunk: one 32-byte load
// per chunk, used as B operand of W = V^T C with k = 4(l/16) + j in MFMA j,
// and as the accumulator of C -= V Y with the MFMA's row i taken as matrix
// row 4(i%4) + i/4.  W's and Y's result layout (element v of lane l: row
// l/16 + 4v) is the B layout of the next product.
template <bool TRANS>
__device__ __forceinline__ void wy_tile(const double* vs, int ldv, const double* T, int r0, int rows,
                                        double* __restrict__ C, int ldc) {
  const int lane = threadIdx.x & 63, lc = lane & 15, kq = lane >> 4;
  double* c = C + (int64_t)lc * ldc + 4 * kq;
  d4 w = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int r = r0; r < rows; r += 16) {
    const d4 x = *(const d4*)(c + r);
    const double* v = vs + lc * ldv + r + 4 * kq;
#pragma unroll
    for (int j = 0; j < 4; ++j) w = __builtin_amdgcn_mfma_f64_16x16x4f64(v[j], x[j], w, 0, 0, 0);
  }
  d4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int k = kq + 4 * s;
    const double t = TRANS ? T[k * 16 + lc] : T[lc * 16 + k];
    y = __builtin_amdgcn_mfma_f64_16x16x4f64(t, w[s], y, 0, 0, 0);
  }
  const int row = 4 * (lc & 3) + (lc >> 2);
#pragma unroll 4
  for (int r = r0; r < rows; r += 16) {
    d4 x = *(const d4*)(c + r);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      x = __builtin_amdgcn_mfma_f64_16x16x4f64(-vs[(kq + 4 * s) * ldv + r + row], y[s], x, 0, 0, 0);
    *(d4*)(c + r) = x;
  }
}

// Householder QR of one matrix per workgroup.  F (ldf x n16 column-major, zero
// padded to multiples of 16) receives the reflectors below and R on and
// above the diagonal, T the panels' triangular factors, X = R^T (n x n).
// With it.perm >= 0 the columns are taken in order of falling norm (stable)
// and scaled by 2^-e, e the exponent of the largest entry (exact; expo).
//
// Bound: the chain of n dependent reflectors (norm, scaling, one dot and
// update per remaining panel column: one barrier each, every wave holding
// its panel column in registers), not the MFMA trailing update: 0.36 ms for
// groups of up to 246 x 187, 1.9 us a column with the trailing update.
template <int RM>
__global__ __launch_bounds__(QR_NT) void k_svd_qr(const SvdQr* __restrict__ items, double* __restrict__ work,
                                                  int32_t* __restrict__ perm, int32_t* __restrict__ expo) {
  constexpr int LD = 64 * RM + 4;
  __shared__ double vs[16 * LD];
  __shared__ double S[16][17], T[256], tau_s[16];
  __shared__ double key[SVD_QR_MAX_N];
  __shared__ int lperm[SVD_QR_MAX_N];
  __shared__ double wmax[QR_NT / 64];
  const SvdQr it = items[blockIdx.x];
  const int m = it.m, n = it.n, ldf = it.ldf, n16 = (n + 15) & ~15;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double* src = work + it.src;
  double* F = work + it.f;

  int e = 0;
  if (it.perm >= 0) {
    double mx = 0.0;
    const int64_t mn = (int64_t)m * n;  // src is contiguous (leading dim m)
    for (int64_t i = tid; i < mn; i += QR_NT) mx = fmax(mx, fabs(src[i]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) wmax[wave] = mx;
    __syncthreads();
    for (int w = 0; w < QR_NT / 64; ++w) mx = fmax(mx, wmax[w]);
    e = mx > 0.0 && mx <= DBL_MAX ? ilogb(mx) : 0;
    if (tid == 0) expo[it.grp] = e;
    for (int c = wave; c < n; c += QR_NT / 64) {
      double s = 0.0;
      for (int i = lane; i < m; i += 64) {
        const double x = ldexp(src[(int64_t)c * m + i], -e);
        s += x * x;
      }
      s = wave_sum(s);
      if (lane == 0) key[c] = s == s ? s : DBL_MAX;  // NaN first: the ranks stay a permutation
    }
    __syncthreads();
    if (tid < n) {
      const double k = key[tid];
      int r = 0;
      for (int c = 0; c < n; ++c) r += key[c] > k || (key[c] == k && c < tid);
      lperm[r] = tid;
      perm[it.perm + r] = tid;
    }
    __syncthreads();
  }
  for (int c = wave; c < n; c += QR_NT / 64) {
    const double* sc = src + (int64_t)(it.perm >= 0 ? lperm[c] : c) * m;
    for (int i = lane; i < m; i += 64) F[(int64_t)c * ldf + i] = ldexp(sc[i], -e);
  }
  __syncthreads();

  for (int k0 = 0; k0 < n; k0 += 16) {
    double* fc = F + (int64_t)(k0 + wave) * ldf;  // this wave's panel column (zero beyond n)
    double a[RM], v[RM];
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      const int i = lane + 64 * r;
      a[r] = i < ldf ? fc[i] : 0.0;
      v[r] = 0.0;
    }
    for (int t = 0; t < 16; ++t) {
      const int k = k0 + t;
      if (wave == t) {
        double s2 = 0.0, al = 0.0;
#pragma unroll
        for (int r = 0; r < RM; ++r) {
          const int i = lane + 64 * r;
          s2 += i > k ? a[r] * a[r] : 0.0;
          al += i == k ? a[r] : 0.0;
        }
        s2 = wave_sum(s2);
        al = read_lane(al, k & 63);
        double tau = 0.0, beta = al, inv = 0.0;
        if (s2 != 0.0) {
          const double h2 = al * al + s2, rn = rsqrt_d(h2), nrm = h2 * rn;
          beta = al >= 0.0 ? -nrm : nrm;
          tau = fma(fabs(al), rn, 1.0);  // (beta - al) / beta
          inv = 1.0 / (al - beta);
        }
#pragma unroll
        for (int r = 0; r < RM; ++r) {
          const int i = lane + 64 * r;
          v[r] = i > k ? a[r] * inv : (i == k ? 1.0 : 0.0);
          vs[t * LD + i] = v[r];
          if (i < ldf) fc[i] = i > k ? v[r] : (i == k ? beta : a[r]);
        }
        if (lane == 0) tau_s[t] = tau;
      }
      __syncthreads();
      const double tau = tau_s[t];
      double d = 0.0;
      if (wave > t) {
        double x[RM];
#pragma unroll
        for (int r = 0; r < RM; ++r) {
          x[r] = vs[t * LD + lane + 64 * r];
          d += x[r] * a[r];
        }
        d = tau * wave_sum(d);
#pragma unroll
        for (int r = 0; r < RM; ++r) a[r] -= d * x[r];
      } else if (wave < t) {  // V^T V, for the panel's triangular factor
#pragma unroll
        for (int r = 0; r < RM; ++r) d += vs[t * LD + lane + 64 * r] * v[r];
        d = wave_sum(d);
        if (lane == 0) S[wave][t] = d;
      }
    }
    __syncthreads();
    if (tid < 16) {  // row tid of T: T(i,j) = -tau_j sum_{i<=l<j} T(i,l) S(l,j)
      double tr[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        double s = 0.0;
#pragma unroll
        for (int l = 0; l < j; ++l) s += tr[l] * S[l][j];
        tr[j] = tid == j ? tau_s[j] : (tid < j ? -tau_s[j] * s : 0.0);
        T[tid * 16 + j] = tr[j];
        work[it.t + (int64_t)(k0 >> 4) * 256 + tid * 16 + j] = tr[j];
      }
    }
    __syncthreads();
    const int c0 = k0 + 16 + 16 * wave;
    if (c0 < n16) wy_tile<true>(vs, LD, T, k0, ldf, F + (int64_t)c0 * ldf, ldf);
    __syncthreads();
  }
  // X = R^T
  for (int j = wave; j < n; j += QR_NT / 64)
    for (int i = lane; i < n; i += 64)
      work[it.x + (int64_t)j * n + i] = i >= j ? F[(int64_t)i * ldf + j] : 0.0;
}

// C <- Q C for up to 4 column tiles of 16 (one per wave), Q the reflectors of
// a k_svd_qr factorisation, panels from the last to the first; the first
// it.m rows then go to the destination, row i to row perm[i] if it.perm >= 0
template <int RM>
__global__ __launch_bounds__(APPLY_NT) void k_svd_applyq(const SvdApply* __restrict__ items,
                                                         double* __restrict__ work,
                                                         const int32_t* __restrict__ perm) {
  constexpr int LD = 64 * RM + 4;
  __shared__ double vs[16 * LD];
  __shared__ double T[256];
  const SvdApply it = items[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ldf = it.ldf, n = it.n;
  const double* F = work + it.f;
  const int c0 = it.col0 + 16 * wave;
  double* C = work + it.c + (int64_t)c0 * ldf;
  const bool own = c0 < n;
  for (int k0 = (n - 1) & ~15; k0 >= 0; k0 -= 16) {
    for (int t = wave; t < 16; t += APPLY_NT / 64) {
      const double* fc = F + (int64_t)(k0 + t) * ldf;
#pragma unroll 4
      for (int i = k0 + lane; i < ldf; i += 64) {
        const double x = fc[i];
        vs[t * LD + i] = i > k0 + t ? x : (i == k0 + t ? 1.0 : 0.0);
      }
    }
    T[tid] = work[it.t + (int64_t)(k0 >> 4) * 256 + tid];
    __syncthreads();
    if (own) wy_tile<false>(vs, LD, T, k0, ldf, C, ldf);
    __syncthreads();
  }
  if (!own) return;
  for (int c = 0; c < 16 && c0 + c < n; ++c) {
    double* d = work + it.dst + (int64_t)(c0 + c) * it.m;
    for (int i = lane; i < it.m; i += 64)
      d[it.perm >= 0 ? perm[it.perm + i] : i] = C[(int64_t)c * ldf + i];
  }
}

// after the sweeps, one wave per column j: sigma_j = |x_j| 2^e and the matrices
// the reflectors act on, C1 = U (u_j = x_j / |x_j|) and C2 = W
__global__ __launch_bounds__(256) void k_svd_vectors(const SvdGroup* __restrict__ groups, double* __restrict__ work,
                                                     double* __restrict__ sig,
                                                     const int32_t* __restrict__ expo) {
  const SvdGroup g = groups[blockIdx.x];
  const int n = g.n, lane = threadIdx.x & 63;
  for (int j = blockIdx.y * 4 + (threadIdx.x >> 6); j < n; j += gridDim.y * 4) {
    const double* x = work + g.x + (int64_t)j * n;
    const double* w = work + g.w + (int64_t)j * n;
    double s2 = 0.0;
    for (int i = lane; i < n; i += 64) s2 += x[i] * x[i];
    s2 = wave_sum(s2);
    const double sg = sqrt(s2), inv = sg > 0.0 ? 1.0 / sg : 0.0;
    if (lane == 0) sig[g.s + j] = ldexp(sg, expo[blockIdx.x]);
    for (int i = lane; i < n; i += 64) {
      work[g.c1 + (int64_t)j * g.ldf + i] = x[i] * inv;
      work[g.c2 + (int64_t)j * g.n16 + i] = w[i];
    }
  }
}

}  // namespace

void launch_svd_qr(const SvdQr* ditems, int nitems, int maxrows, double* work, int32_t* perm, int32_t* expo,
                   hipStream_t s) {
  if (nitems <= 0) return;
  if (maxrows <= 256)
    hipLaunchKernelGGL(k_svd_qr<4>, dim3(nitems), dim3(QR_NT), 0, s, ditems, work, perm, expo);
  else if (maxrows <= 512)
    hipLaunchKernelGGL(k_svd_qr<8>, dim3(nitems), dim3(QR_NT), 0, s, ditems, work, perm, expo);
  else if (maxrows <= SVD_QR_MAX_M)
    hipLaunchKernelGGL(k_svd_qr<16>, dim3(nitems), dim3(QR_NT), 0, s, ditems, work, perm, expo);
  else
    fail(QSX_ERR_STRUCT, "QR of a group matrix of %d rows", maxrows);
  QSX_HIP(hipGetLastError());
}

void launch_svd_applyq(const SvdApply* ditems, int nitems, int maxrows, double* work, const int32_t* perm,
                       hipStream_t s) {
  if (nitems <= 0) return;
  if (maxrows <= 256)
    hipLaunchKernelGGL(k_svd_applyq<4>, dim3(nitems), dim3(APPLY_NT), 0, s, ditems, work, perm);
  else if (maxrows <= 512)
    hipLaunchKernelGGL(k_svd_applyq<8>, dim3(nitems), dim3(APPLY_NT), 0, s, ditems, work, perm);
  else if (maxrows <= SVD_QR_MAX_M)
    hipLaunchKernelGGL(k_svd_applyq<16>, dim3(nitems), dim3(APPLY_NT), 0, s, ditems, work, perm);
  else
    fail(QSX_ERR_STRUCT, "reflectors of a group matrix of %d rows", maxrows);
  QSX_HIP(hipGetLastError());
}

void launch_svd_vectors(const SvdGroup* dgroups, int ngroups, int maxn, double* work, double* sig,
                        const int32_t* expo, hipStream_t s) {
  if (ngroups <= 0) return;
  hipLaunchKernelGGL(k_svd_vectors, dim3(ngroups, (maxn + 15) / 16), dim3(256), 0, s, dgroups, work, sig, expo);
  QSX_HIP(hipGetLastError());
}

}  // namespace qsx
