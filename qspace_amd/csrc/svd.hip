// svd.hip -- the block SVD of the truncation (orthoQS): the group
// matrices are assembled from the blocks on the device, each is decomposed
// by a one-sided Jacobi SVD, and the kept singular vectors are scattered
// into the blocks of the two result tensors.
//
// One-sided Jacobi (Hestenes, J. SIAM 6 (1958); the rotation and stopping
// rule of Demmel and Veselic, SIAM J. Matrix Anal. Appl. 13 (1992)): the
// columns of a matrix are orthogonalised by plane rotations of column
// pairs; a sweep visits every pair once, in steps of disjoint pairs that run
// in parallel.  At the end x_j = sigma_j u_j and the accumulated rotations
// are W.  Matrices of up to SVD_QR_MAX_M x SVD_QR_MAX_N are reduced to an
// n x n triangle first (svdqr.hip) unless small; k_jacobi_lds runs all sweeps of
// one with n <= SVD_LDS_N in a workgroup's LDS, k_jacobi_cross one round of
// column blocks of a larger one.  Other matrices are swept as they are: in a
// workgroup's LDS where they fit (k_jacobi_whole: small ones, and few columns
// of more than SVD_QR_MAX_M rows), by k_jacobi_block where they do not.
#include <cfloat>

#include "qsx_internal.hpp"
#include "lanes.hpp"

namespace qsx {
namespace {

constexpr int SVD_NT = 1024;          // threads per workgroup of k_svd_finalize and k_jacobi_whole
constexpr int SVD_NT_LDS = 512;       // threads per workgroup of k_jacobi_lds
constexpr int SVD_NT_CROSS = 256;     // threads per workgroup of k_jacobi_cross
constexpr int SVD_NT_BLOCK = 512;     // threads per workgroup of the block steps
constexpr int SVD_SEG = 16;           // lanes per column pair
constexpr int SVD_SEG_CROSS = 32;     // lanes per block of columns in k_jacobi_cross
constexpr int SVD_MAX_SWEEPS = 60;
// Orthogonality target of a column pair: sqrt(m) eps (as LAPACK's dgesvj)
// for the first kTightSweeps sweeps, then m eps, the rounding bound of the
// length-m dot products that decide a rotation -- a pair whose computed
// cosine stays above the tight target only through that rounding (e.g.
// columns of nearly equal norm) would otherwise rotate forever.
constexpr int kTightSweeps = 20;
__host__ __device__ inline double jacobi_tol(int m, int sweep) {
  return (sweep < kTightSweeps ? sqrt((double)m) : (double)m) * DBL_EPSILON;
}

// the rotation of the Gram matrix [al ga; ga be] that zeroes ga (smaller
// angle); false when |ga| <= tol sqrt(al be): the pair is orthogonal.  A
// pair whose smaller column is below tol times the larger (norms) is left
// alone as well: such a column is rounding noise of a rank-deficient matrix
// (its singular value is below what FP64 resolves against the larger one),
// and rotating it against the larger column only makes new noise of the
// same size, so the sweeps would never end.
__device__ __forceinline__ bool jacobi_cs(double al, double be, double ga, double tol, double& c, double& s) {
  if (!(fabs(ga) > tol * sqrt(al) * sqrt(be))) return false;
  if (fmin(al, be) <= tol * tol * fmax(al, be)) return false;
  const double zeta = (be - al) / (2.0 * ga);
  const double az = fabs(zeta);
  const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (az + (az > 1e150 ? az : sqrt(1.0 + zeta * zeta)));
  c = 1.0 / sqrt(1.0 + t * t);
  s = c * t;
  return true;
}

// rotation of the column pair (ap, aq) of A (m rows) and (vp, vq) of V
// (n rows) by the 16 lanes of a segment; with R > 0 a lane holds its R
// elements of each column in registers (8 R < m <= 16 R, or m <= 16 with R = 1;
// with FULLV n > 8 R too: the first half of the rows needs no mask), R = 0 runs
// over the rows in chunks of 4 per lane.  True if the pair was rotated.
template <int R, bool FULLV>
__device__ __forceinline__ bool rotate_pair(double* ap, double* aq, double* vp, double* vq, int m, int n, int lane,
                                            double tol) {
  constexpr int L = SVD_SEG;
  double c, s;
  if constexpr (R > 0) {
    auto in_a = [&](int r) { return r < R / 2 || lane + L * r < m; };
    auto in_v = [&](int r) { return (FULLV && r < R / 2) || lane + L * r < n; };
    double x[R], y[R], u[R], z[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      x[r] = in_a(r) ? ap[i] : 0.0;
      y[r] = in_a(r) ? aq[i] : 0.0;
    }
    double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      al += x[r] * x[r];
      be += y[r] * y[r];
      ga += x[r] * y[r];
    }
    al = seg_sum(al);
    be = seg_sum(be);
    ga = seg_sum(ga);
    if (!jacobi_cs(al, be, ga, tol, c, s)) return false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      if (in_a(r)) {
        ap[i] = c * x[r] - s * y[r];
        aq[i] = s * x[r] + c * y[r];
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      u[r] = in_v(r) ? vp[i] : 0.0;
      z[r] = in_v(r) ? vq[i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      if (in_v(r)) {
        vp[i] = c * u[r] - s * z[r];
        vq[i] = s * u[r] + c * z[r];
      }
    }
    return true;
  } else {
    double al = 0.0, be = 0.0, ga = 0.0;
    for (int i0 = lane; i0 < m; i0 += 4 * L) {
      double x[4], y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + L * r;
        x[r] = i < m ? ap[i] : 0.0;
        y[r] = i < m ? aq[i] : 0.0;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        al += x[r] * x[r];
        be += y[r] * y[r];
        ga += x[r] * y[r];
      }
    }
    al = seg_sum(al);
    be = seg_sum(be);
    ga = seg_sum(ga);
    if (!jacobi_cs(al, be, ga, tol, c, s)) return false;
    for (int pass = 0; pass < 2; ++pass) {
      double* xp = pass ? vp : ap;
      double* yp = pass ? vq : aq;
      const int len = pass ? n : m;
      for (int i0 = lane; i0 < len; i0 += 4 * L) {
        double x[4], y[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = i0 + L * r;
          x[r] = i < len ? xp[i] : 0.0;
          y[r] = i < len ? yp[i] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = i0 + L * r;
          if (i < len) {
            xp[i] = c * x[r] - s * y[r];
            yp[i] = s * x[r] + c * y[r];
          }
        }
      }
    }
    return true;
  }
}

// Pair schedules over columns of A (leading dim m) and V (leading dim n),
// run by NT threads in segments of 16 lanes, one pair per segment at a
// time; every step's pairs are disjoint, steps are separated by barriers.
// Return true (in every thread) if any pair rotated; flag is LDS.
//  * sweep: all pairs of w columns in the round-robin order (w-1 steps of
//    w/2 pairs; column w is a dummy when w is odd);
//  * cross: all pairs (i, np + j), i < np, j < nq: step t pairs i with
//    (i + t) mod max(np, nq).
template <int NT, int R, bool CROSS, bool FULLV>
__device__ __forceinline__ bool jacobi_pairs(double* A, double* V, int np, int nq, int m, int n, double tol,
                                             int* flag) {
  constexpr int L = SVD_SEG;
  constexpr int nseg = NT / L;
  const int tid = threadIdx.x;
  const int seg = tid / L, lane = tid % L;
  const int w = np + nq;
  const int wp = w + (w & 1);
  const int cmax = np > nq ? np : nq;
  const int nsteps = CROSS ? cmax : wp - 1;
  const int npairs = CROSS ? cmax : wp / 2;
  if (tid == 0) *flag = 0;
  __syncthreads();
  for (int step = 0; step < nsteps; ++step) {
    for (int k = seg; k < npairs; k += nseg) {
      int p, q;
      if (CROSS) {
        const int j = (k + step) % cmax;
        if (k >= np || j >= nq) continue;
        p = k;
        q = np + j;
      } else {
        if (k == 0) {
          p = wp - 1;
          q = step;
        } else {
          p = (step + k) % (wp - 1);
          q = (step - k + wp - 1) % (wp - 1);
        }
        if (p >= w || q >= w) continue;  // the dummy column (whole segment)
      }
      if (rotate_pair<R, FULLV>(A + (int64_t)p * m, A + (int64_t)q * m, V + (int64_t)p * n, V + (int64_t)q * n, m, n,
                         lane, tol) &&
          lane == 0)
        *flag = 1;
    }
    __syncthreads();
  }
  const bool any = *flag != 0;
  __syncthreads();  // every thread has read the flag before it is reused
  return any;
}

// the variant for the column lengths: k_jacobi_whole's few columns in registers
// up to 256 rows, k_jacobi_block's in the registers of its 512 threads for 256 < n
// <= m <= 512 (masks for all 32 rows of a lane spill scalar registers: orthoQS of
// one 300 x 257 matrix 19.4 ms, 16.7 with masks for the second half only)
template <int NT, bool CROSS>
__device__ __forceinline__ bool jacobi_pairs_m(double* A, double* V, int np, int nq, int m, int n, double tol,
                                               int* flag) {
  if constexpr (NT == SVD_NT) {
    if (m <= 16) return jacobi_pairs<NT, 1, CROSS, false>(A, V, np, nq, m, n, tol, flag);
    if (m <= 32) return jacobi_pairs<NT, 2, CROSS, false>(A, V, np, nq, m, n, tol, flag);
    if (m <= 64) return jacobi_pairs<NT, 4, CROSS, false>(A, V, np, nq, m, n, tol, flag);
    if (m <= 128) return jacobi_pairs<NT, 8, CROSS, false>(A, V, np, nq, m, n, tol, flag);
    if (m <= 256) return jacobi_pairs<NT, 16, CROSS, false>(A, V, np, nq, m, n, tol, flag);
  } else {
    if (n > 256 && m <= 512) return jacobi_pairs<NT, 32, CROSS, true>(A, V, np, nq, m, n, tol, flag);
  }
  return jacobi_pairs<NT, 0, CROSS, false>(A, V, np, nq, m, n, tol, flag);
}

// one-wave workgroups a block is dealt to (gather, scatter): whole columns, or
// parts of columns where there are fewer columns (orthoQS of one 20223 x 1
// matrix with its rows on one wave / on 16: 0.65 / 0.40 ms)
constexpr int kColSplit = 16;
__device__ __forceinline__ int col_parts(int ncols) { return max(1, (int)gridDim.y / max(1, ncols)); }

// zero-padded group matrices: block e (d1 x d2, column-major) goes to
// row i0, column j0 of its matrix (leading dim ld), transposed when trans
__global__ __launch_bounds__(64) void k_svd_gather(const SvdGather* __restrict__ items, const double* __restrict__ src,
                                                    double* __restrict__ work) {
  const SvdGather it = items[blockIdx.x];
  const int parts = col_parts(it.d2);
  for (int c = blockIdx.y; c < it.d2 * parts; c += gridDim.y) {
    const int j = c / parts;
    for (int i = 64 * (c % parts) + threadIdx.x; i < it.d1; i += 64 * parts) {
      const int64_t d = it.trans ? it.dst_off + j + (int64_t)i * it.ld : it.dst_off + i + (int64_t)j * it.ld;
      work[d] = src[it.src_off + (int64_t)j * it.d1 + i] * it.scale;
    }
  }
}

// ---------------------------------------------------------------- n x n Jacobi
// A segment of L = 16 or 32 lanes rotates the columns of one 2-column block P against
// those of another, Q: the pairs (P0,Q0), (P1,Q1), then (P0,Q1), (P1,Q0),
// with all four columns of X and of W in registers (R elements per lane and
// column).  Two independent pairs per step share one chain of scalar work:
// after the first level of the dot products' reduction even lanes carry the
// first pair and odd lanes the second, so the rotation angles of both come
// out of one instruction stream and go back to the row by DPP broadcasts.
// The columns' squared norms are kept beside them and follow a rotation by
// |x|^2 -/+ t ga; they are summed anew when a rotation cancels most of one,
// and at the start of every sweep.
//
// Bound: the dependent chain of a step (dot, reduction, angle, update,
// barrier).  Against one pair per segment with both columns and all three
// sums through LDS, and the angle from three divisions and three square
// roots (1.7 us a step at n = 64, m = 128): 0.8 us a step at n = 64.  17
// groups of an SU(2) MPS tensor (up to 128 x 64): 2.1 ms in 20 sweeps, now
// 0.37 ms in 7 on their R2^T.  Measured no faster: 32 lanes a segment in LDS
// (0.47 against 0.43 ms), W's rotation beside the next angles (0.55 ms).
template <int R>
struct Cols2 {
  double x[2][R], w[2][R], nn[2];
};

// The rotation of the Gram matrix [al ga; ga be] that zeroes ga (smaller
// angle): x' = c x - s y, y' = s x + c y; with h^2 = (be-al)^2 + 4 ga^2,
// cos 2t = |be-al| / h, c^2 = (1 + cos 2t) / 2, s = ga / (h c).  The three
// are scaled by the larger norm's power of two first, so no square leaves the
// range.  No rotation (c = 1, s = 0) when |ga| <= tol sqrt(al be), or when a
// column is below tol times the other (norms): such a column is rounding
// noise of a rank-deficient matrix (its singular value is below what FP64
// resolves against the larger one), and rotating it against the larger
// column only makes new noise of the same size.  al, be become the new
// squared norms; cancel: one of them lost most of its digits.
__device__ __forceinline__ bool jacobi_angle(double& al, double& be, double ga, double tol2, double& c, double& s,
                                             bool& cancel) {
  const int e = __builtin_amdgcn_frexp_exp(fmax(al, be));
  const double a = ldexp(al, -e), b = ldexp(be, -e), g = ldexp(ga, -e);
  const bool rot = g * g > tol2 * a * b && fmin(a, b) > tol2 * fmax(a, b);
  const double d = b - a;
  const double r = rsqrt_d(fma(d, d, 4.0 * g * g));
  const double q = fma(0.5 * fabs(d), r, 0.5);
  const double rc = rsqrt_d(q);
  const double sn = (d >= 0.0 ? g : -g) * r * rc;
  const double t = sn * rc;
  const double an = fmax(fma(-t, g, a), 0.0), bn = fmax(fma(t, g, b), 0.0);
  c = rot ? q * rc : 1.0;
  s = rot ? sn : 0.0;
  cancel = rot && (an < 0x1p-10 * a || bn < 0x1p-10 * b);
  al = rot ? ldexp(an, e) : al;
  be = rot ? ldexp(bn, e) : be;
  return rot;
}

// the other half's value added, for segments of two rows (L = 32)
template <int L>
__device__ __forceinline__ double add_row(double v) {
  if constexpr (L == 16) return v;
  else return row_pair_sum(v);
}

template <int L, int R>
__device__ __forceinline__ double norm2(const double (&x)[R]) {
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) s += x[r] * x[r];
  return add_row<L>(seg_sum(s));
}

template <int R>
__device__ __forceinline__ void rotate_cols(double (&x)[R], double (&y)[R], double c, double s) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double a = x[r], b = y[r];
    x[r] = c * a - s * b;
    y[r] = s * a + c * b;
  }
}

// the pairs (P0, Q[CR]) and (P1, Q[1-CR]); true (for the wave's active
// segments) if any of them rotated
template <int L, int R, int CR>
__device__ __forceinline__ bool rotate_pairs(Cols2<R>& P, Cols2<R>& Q, double tol2, int lane) {
  double g0 = 0.0, g1 = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    g0 += P.x[0][r] * Q.x[CR][r];
    g1 += P.x[1][r] * Q.x[1 - CR][r];
  }
  const bool odd = lane & 1;
  double ga = odd ? g1 : g0;
  ga += dpp_mov<DPP_XOR1>(odd ? g0 : g1);
  ga += dpp_mov<DPP_XOR2>(ga);
  ga += dpp_mov<DPP_ROR4>(ga);
  ga += dpp_mov<DPP_ROR8>(ga);
  ga = add_row<L>(ga);
  double al = odd ? P.nn[1] : P.nn[0], be = odd ? Q.nn[1 - CR] : Q.nn[CR];
  double c, s;
  bool cancel;
  const bool rot = jacobi_angle(al, be, ga, tol2, c, s, cancel);
  // a row's lanes may differ in the last bit of ga: its lanes 0 and 1 decide
  // (both rows of a segment hold the same sums there)
  if (!__any(rot && (lane & 15) < 2)) return false;
  const double c0 = dpp_mov<DPP_BCAST<0>>(c), s0 = dpp_mov<DPP_BCAST<0>>(s);
  const double c1 = dpp_mov<DPP_BCAST<1>>(c), s1 = dpp_mov<DPP_BCAST<1>>(s);
  P.nn[0] = dpp_mov<DPP_BCAST<0>>(al);
  P.nn[1] = dpp_mov<DPP_BCAST<1>>(al);
  Q.nn[CR] = dpp_mov<DPP_BCAST<0>>(be);
  Q.nn[1 - CR] = dpp_mov<DPP_BCAST<1>>(be);
  rotate_cols(P.x[0], Q.x[CR], c0, s0);
  rotate_cols(P.x[1], Q.x[1 - CR], c1, s1);
  rotate_cols(P.w[0], Q.w[CR], c0, s0);
  rotate_cols(P.w[1], Q.w[1 - CR], c1, s1);
  if (__any(cancel && (lane & 15) < 2)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      P.nn[h] = norm2<L>(P.x[h]);
      Q.nn[h] = norm2<L>(Q.x[h]);
    }
  }
  return true;
}

// all pairs of P and Q
template <int L, int R>
__device__ __forceinline__ bool rotate_blocks(Cols2<R>& P, Cols2<R>& Q, double tol2, int lane) {
  bool any = rotate_pairs<L, R, 0>(P, Q, tol2, lane);
  any |= rotate_pairs<L, R, 1>(P, Q, tol2, lane);
  return any;
}

// columns c0, c0+1 of nc columns of n rows (L (R-2) < n <= L R); an absent
// second column is zero
template <int L, int R>
__device__ __forceinline__ void load_cols(Cols2<R>& b, const double* X, const double* W, int c0, int nc, int n,
                                          int ld, int lane) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool ok = c0 + h < nc;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      const bool in = ok && (r < R - 2 || i < n);
      b.x[h][r] = in ? X[(c0 + h) * ld + i] : 0.0;
      b.w[h][r] = in ? W[(c0 + h) * ld + i] : 0.0;
    }
  }
}

template <int L, int R>
__device__ __forceinline__ void store_cols(const Cols2<R>& b, double* X, double* W, int c0, int nc, int n, int ld,
                                           int lane) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (c0 + h >= nc) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + L * r;
      if (r < R - 2 || i < n) {
        X[(c0 + h) * ld + i] = b.x[h][r];
        W[(c0 + h) * ld + i] = b.w[h][r];
      }
    }
  }
}

// one sweep over all pairs of the nc columns in LDS (X, W: n rows each; nn:
// the columns' squared norms), NT threads: the pairs within the 2-column
// blocks (which also sums the norms), then blocks against blocks by halving:
// at depth d each of 2^d ranges of blocks is split into P and Q, every
// segment keeps one P block in registers and meets the Q blocks of its range
// one round at a time.  ceil(B/2) + ceil(B/4) + ... rounds of two steps, B
// blocks.  True (in every thread) if any pair rotated.
template <int NT, int L, int R>
__device__ __forceinline__ bool sweep_lds(double* X, double* W, double* nn, int nc, int n, int ld, double tol,
                                          int* flag) {
  constexpr int nseg = NT / L;
  const int seg = threadIdx.x / L, lane = threadIdx.x % L;
  const int B = (nc + 1) / 2;
  const double tol2 = tol * tol;
  if (threadIdx.x == 0) *flag = 0;
  __syncthreads();
  bool rotated = false;
  for (int k = seg; k < B; k += nseg) {
    Cols2<R> b;
    load_cols<L>(b, X, W, 2 * k, nc, n, ld, lane);
    double al = norm2<L>(b.x[0]), be = norm2<L>(b.x[1]), ga = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) ga += b.x[0][r] * b.x[1][r];
    ga = add_row<L>(seg_sum(ga));
    double c, s;
    bool cancel;
    if (jacobi_angle(al, be, ga, tol2, c, s, cancel)) {  // the same bits in the whole segment
      rotate_cols(b.x[0], b.x[1], c, s);
      rotate_cols(b.w[0], b.w[1], c, s);
      if (cancel) {
        al = norm2<L>(b.x[0]);
        be = norm2<L>(b.x[1]);
      }
      store_cols<L>(b, X, W, 2 * k, nc, n, ld, lane);
      rotated = true;
    }
    if (lane == 0) {
      nn[2 * k] = al;
      nn[2 * k + 1] = be;
    }
  }
  __syncthreads();
  for (int d = 0; (1 << d) < B; ++d) {
    const int hmax = (B + (2 << d) - 1) >> (d + 1);
    for (int base = 0; base < (hmax << d); base += nseg) {
      const int k = base + seg, rg = k / hmax, idx = k % hmax;
      int lo = 0, hi = B;
      for (int b = d - 1; b >= 0; --b) {
        const int mid = lo + (hi - lo + 1) / 2;
        if ((rg >> b) & 1) lo = mid;
        else hi = mid;
      }
      const int mid = lo + (hi - lo + 1) / 2, hp = mid - lo, hq = hi - mid;
      const bool act = rg < (1 << d) && idx < hp && hq > 0;
      Cols2<R> P;
      const int pc = 2 * (lo + idx);
      if (act) {
        load_cols<L>(P, X, W, pc, nc, n, ld, lane);
        P.nn[0] = nn[pc];
        P.nn[1] = nn[pc + 1];
      }
      bool any = false;
      for (int t = 0; t < hmax; ++t) {
        if (act && t < hp) {
          int j = idx + t;
          if (j >= hp) j -= hp;
          if (j < hq) {
            const int qc = 2 * (mid + j);
            Cols2<R> Q;
            load_cols<L>(Q, X, W, qc, nc, n, ld, lane);
            Q.nn[0] = nn[qc];
            Q.nn[1] = nn[qc + 1];
            if (rotate_blocks<L>(P, Q, tol2, lane)) {
              store_cols<L>(Q, X, W, qc, nc, n, ld, lane);
              if (lane < 2) nn[qc + lane] = lane ? Q.nn[1] : Q.nn[0];
              any = true;
            }
          }
        }
        __syncthreads();
      }
      if (act && any) {
        store_cols<L>(P, X, W, pc, nc, n, ld, lane);
        if (lane < 2) nn[pc + lane] = lane ? P.nn[1] : P.nn[0];
        rotated = true;
      }
      __syncthreads();
    }
  }
  if (rotated) *flag = 1;
  __syncthreads();
  const bool ret = *flag != 0;
  __syncthreads();  // every thread has read the flag before it is reused
  return ret;
}

// all sweeps of an n x n matrix (n <= SVD_LDS_N) in one workgroup, X and W in LDS
__global__ __launch_bounds__(SVD_NT_LDS) void k_jacobi_lds(const SvdGroup* __restrict__ groups,
                                                           const int32_t* __restrict__ which,
                                                           double* __restrict__ work, int32_t* __restrict__ sweeps) {
  __shared__ double lds[2 * SVD_LDS_N * (SVD_LDS_N + 8)];
  __shared__ double nn[SVD_LDS_N + 2];
  __shared__ int flag;
  const SvdGroup g = groups[which[blockIdx.x]];
  const int n = g.n, tid = threadIdx.x;
  // leading dimension 8 mod 16: the 16-lane segments of a wave read 2-column
  // blocks that start in different halves of the banks
  const int ld = ((n + 7) & ~15) + 8;
  double* X = lds;
  double* W = lds + n * ld;
  const int wave = tid >> 6, wl = tid & 63;
  for (int j = wave; j < n; j += SVD_NT_LDS / 64)
    for (int i = wl; i < n; i += 64) {
      X[j * ld + i] = work[g.x + j * n + i];
      W[j * ld + i] = i == j ? 1.0 : 0.0;
    }
  __syncthreads();
  int sw = 0;
  for (; sw < SVD_MAX_SWEEPS; ++sw) {
    const double tol = jacobi_tol(n, sw);
    bool any;
    switch ((n + 15) / 16) {
      case 1: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 1>(X, W, nn, n, n, ld, tol, &flag); break;
      case 2: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 2>(X, W, nn, n, n, ld, tol, &flag); break;
      case 3: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 3>(X, W, nn, n, n, ld, tol, &flag); break;
      case 4: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 4>(X, W, nn, n, n, ld, tol, &flag); break;
      case 5: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 5>(X, W, nn, n, n, ld, tol, &flag); break;
      default: any = sweep_lds<SVD_NT_LDS, SVD_SEG, 6>(X, W, nn, n, n, ld, tol, &flag); break;
    }
    if (!any) break;
  }
  for (int j = wave; j < n; j += SVD_NT_LDS / 64)
    for (int i = wl; i < n; i += 64) {
      work[g.x + j * n + i] = X[j * ld + i];
      work[g.w + j * n + i] = W[j * ld + i];
    }
  if (tid == 0) sweeps[blockIdx.x] = sw;
}

// contiguous columns of X and W between memory and LDS, up to 16 loads in
// flight per thread
template <int NT>
__device__ __forceinline__ void copy_cols(double* __restrict__ dx, double* __restrict__ dw,
                                          const double* __restrict__ sx, const double* __restrict__ sw, int n) {
  for (int e0 = threadIdx.x; e0 < n; e0 += 8 * NT) {
    double v[8], w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool in = e0 + u * NT < n;
      v[u] = in ? sx[e0 + u * NT] : 0.0;
      w[u] = in ? sw[e0 + u * NT] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (e0 + u * NT < n) {
        dx[e0 + u * NT] = v[u];
        dw[e0 + u * NT] = w[u];
      }
  }
}

// the column blocks P (registers, one 2-column block per segment) against Q (LDS)
template <int L, int R>
__device__ __forceinline__ bool cross_blocks(double* __restrict__ Xp, double* __restrict__ Wp, int np,
                                             const double* __restrict__ gx, const double* __restrict__ gw, double* Xq,
                                             double* Wq, double* nn, int nq, int n, double tol) {
  const int seg = threadIdx.x / L, lane = threadIdx.x % L;
  const int hp = (np + 1) / 2, hq = (nq + 1) / 2, h = hp > hq ? hp : hq;
  const double tol2 = tol * tol;
  Cols2<R> P{};
  if (seg < hp) {  // hp <= NT / L, checked by the host
    load_cols<L>(P, Xp, Wp, 2 * seg, np, n, n, lane);
  }
  copy_cols<SVD_NT_CROSS>(Xq, Wq, gx, gw, nq * n);
  P.nn[0] = norm2<L>(P.x[0]);
  P.nn[1] = norm2<L>(P.x[1]);
  __syncthreads();
  if (seg < hq) {
    for (int c = 2 * seg; c < 2 * seg + 2; ++c) {
      double s = 0.0;
      for (int i = lane; i < n && c < nq; i += L) s += Xq[c * n + i] * Xq[c * n + i];
      s = add_row<L>(seg_sum(s));
      if (lane == 0) nn[c] = s;
    }
  }
  __syncthreads();
  bool any = false;
  for (int t = 0; t < h; ++t) {
    int j = seg + t;
    if (j >= h) j -= h;
    if (seg < hp && j < hq) {
      Cols2<R> Q;
      load_cols<L>(Q, Xq, Wq, 2 * j, nq, n, n, lane);
      Q.nn[0] = nn[2 * j];
      Q.nn[1] = nn[2 * j + 1];
      if (rotate_blocks<L>(P, Q, tol2, lane)) {
        store_cols<L>(Q, Xq, Wq, 2 * j, nq, n, n, lane);
        if (lane < 2) nn[2 * j + lane] = lane ? Q.nn[1] : Q.nn[0];
        any = true;
      }
    }
    __syncthreads();
  }
  if (any) store_cols<L>(P, Xp, Wp, 2 * seg, np, n, n, lane);
  return any;
}

// one round of a sweep of a matrix with SVD_LDS_N < n <= SVD_QR_MAX_N: the
// pairs within column block P (q0 == q1) or the pairs of P against Q;
// rot[sweep * ngroups + grp] is set when one rotated.  A group that rotated
// nothing in the sweep before is done.  Blocks of 16 columns with 32 lanes a
// segment (21 us a launch, n = 187) against 32 columns with 16 lanes (51 us, half
// as many launches): one wave per SIMD either way, so the issue of a step's
// updates bounds a round, and smaller blocks spread it over more CUs.
__global__ __launch_bounds__(SVD_NT_CROSS) void k_jacobi_cross(const SvdGroup* __restrict__ groups, int ngroups,
                                                               const SvdBlockStep* __restrict__ steps,
                                                               double* __restrict__ work, int32_t* __restrict__ rot,
                                                               int sweep) {
  __shared__ double lds[2 * SVD_CROSS_COLS * SVD_QR_MAX_N];
  __shared__ double nn[SVD_CROSS_COLS + 2];
  __shared__ int flag;
  const SvdBlockStep st = steps[blockIdx.x];
  if (sweep > 0 && rot[(sweep - 1) * ngroups + st.grp] == 0) return;
  const SvdGroup g = groups[st.grp];
  const int n = g.n;
  const bool cross = st.q1 > st.q0;
  const int c0 = cross ? st.q0 : st.p0, nc = cross ? st.q1 - st.q0 : st.p1 - st.p0;
  double* X = lds;
  double* W = lds + nc * n;
  double* gx = work + g.x + (int64_t)c0 * n;
  double* gw = work + g.w + (int64_t)c0 * n;
  double* px = work + g.x + (int64_t)st.p0 * n;
  double* pw = work + g.w + (int64_t)st.p0 * n;
  const int np = st.p1 - st.p0;
  const double tol = jacobi_tol(n, sweep);
  bool any;
#define QSX_CROSS(R)                                                                              \
  any = cross ? cross_blocks<SVD_SEG_CROSS, R>(px, pw, np, gx, gw, X, W, nn, nc, n, tol)          \
              : (copy_cols<SVD_NT_CROSS>(X, W, gx, gw, nc * n), __syncthreads(), false) ||        \
                    sweep_lds<SVD_NT_CROSS, SVD_SEG_CROSS, R>(X, W, nn, nc, n, n, tol, &flag)
  if (n <= 128) QSX_CROSS(4);
  else if (n <= 160) QSX_CROSS(5);
  else if (n <= 192) QSX_CROSS(6);
  else if (n <= 224) QSX_CROSS(7);
  else QSX_CROSS(8);
#undef QSX_CROSS
  any = __syncthreads_or(any);
  if (!any) return;
  copy_cols<SVD_NT_CROSS>(gx, gw, X, W, nc * n);
  if (threadIdx.x == 0) rot[sweep * ngroups + st.grp] = 1;
}

// all sweeps of an m x n matrix with m n + n^2 <= SVD_LDS_DOUBLES (checked by
// the host) in one workgroup's LDS: a launch, where k_jacobi_block takes an
// upload, n block steps and a wait per sweep, and at least four columns' room
// (a single column of 10112 .. 20223 rows fits only here).  orthoQS of one
// 2000 x 8 matrix, this kernel / column blocks: 0.76 / 1.12 ms.
__global__ __launch_bounds__(SVD_NT) void k_jacobi_whole(const SvdItem* __restrict__ items,
                                                         const int32_t* __restrict__ which,
                                                         double* __restrict__ work, double* __restrict__ sig,
                                                         int32_t* __restrict__ sweeps) {
  __shared__ double lds[SVD_LDS_DOUBLES];
  __shared__ int rotated;
  const SvdItem it = items[which[blockIdx.x]];
  const int m = it.m, n = it.n;  // m >= n >= 1
  const int tid = threadIdx.x;
  double* A = lds;
  double* V = lds + m * n;
  for (int e = tid; e < m * n; e += SVD_NT) A[e] = work[it.a_off + e];
  for (int e = tid; e < n * n; e += SVD_NT) V[e] = e % (n + 1) == 0 ? 1.0 : 0.0;
  __syncthreads();
  int sw = 0;
  for (; sw < SVD_MAX_SWEEPS; ++sw)
    if (!jacobi_pairs_m<SVD_NT, false>(A, V, n, 0, m, n, jacobi_tol(m, sw), &rotated)) break;
  // sigma_j = |a_j|, u_j = a_j / sigma_j (a zero column stays zero)
  const int seg = tid / SVD_SEG, lane = tid % SVD_SEG;
  for (int j = seg; j < n; j += SVD_NT / SVD_SEG) {
    double* aj = A + j * m;
    double s2 = 0.0;
    for (int i = lane; i < m; i += SVD_SEG) s2 += aj[i] * aj[i];
    s2 = seg_sum(s2);
    const double sg = sqrt(s2);
    const double inv = sg > 0.0 ? 1.0 / sg : 0.0;
    for (int i = lane; i < m; i += SVD_SEG) aj[i] *= inv;
    if (lane == 0) sig[it.s_off + j] = sg;
  }
  __syncthreads();
  for (int e = tid; e < m * n; e += SVD_NT) work[it.a_off + e] = A[e];
  for (int e = tid; e < n * n; e += SVD_NT) work[it.v_off + e] = V[e];
  if (tid == 0) sweeps[blockIdx.x] = sw;
}

// one step of the block one-sided Jacobi of a group matrix too large for
// LDS: the columns of block P = [p0,p1) (and of block Q = [q0,q1)) and
// their columns of V are staged in LDS; the pairs within P (q0 == q1) or
// the pairs across P and Q are rotated, the columns go back; rot[group] = 1
// if anything rotated
__global__ __launch_bounds__(SVD_NT_BLOCK) void k_jacobi_block(const SvdItem* __restrict__ groups,
                                                         const SvdBlockStep* __restrict__ steps,
                                                         double* __restrict__ work, int32_t* __restrict__ rot,
                                                         int sweep) {
  __shared__ double lds[SVD_LDS_DOUBLES];
  __shared__ int rotated;
  const SvdBlockStep st = steps[blockIdx.x];
  const SvdItem g = groups[st.grp];
  const int m = g.m, n = g.n;
  const int np_ = st.p1 - st.p0, w = np_ + (st.q1 - st.q0);
  const int tid = threadIdx.x;
  double* A = lds;                       // w columns of m
  double* V = lds + (int64_t)w * m;      // w columns of n
  for (int64_t e = tid; e < (int64_t)w * m; e += SVD_NT_BLOCK) {
    const int c = (int)(e / m), i = (int)(e % m);
    const int gc = c < np_ ? st.p0 + c : st.q0 + (c - np_);
    A[e] = work[g.a_off + (int64_t)gc * m + i];
  }
  for (int64_t e = tid; e < (int64_t)w * n; e += SVD_NT_BLOCK) {
    const int c = (int)(e / n), i = (int)(e % n);
    const int gc = c < np_ ? st.p0 + c : st.q0 + (c - np_);
    V[e] = work[g.v_off + (int64_t)gc * n + i];
  }
  __syncthreads();
  // one block (q0 == q1): all its pairs; two blocks: the pairs across them
  const double tol = jacobi_tol(m, sweep);
  const bool any = w == np_ ? jacobi_pairs_m<SVD_NT_BLOCK, false>(A, V, w, 0, m, n, tol, &rotated)
                            : jacobi_pairs_m<SVD_NT_BLOCK, true>(A, V, np_, w - np_, m, n, tol, &rotated);
  for (int64_t e = tid; e < (int64_t)w * m; e += SVD_NT_BLOCK) {
    const int c = (int)(e / m), i = (int)(e % m);
    const int gc = c < np_ ? st.p0 + c : st.q0 + (c - np_);
    work[g.a_off + (int64_t)gc * m + i] = A[e];
  }
  for (int64_t e = tid; e < (int64_t)w * n; e += SVD_NT_BLOCK) {
    const int c = (int)(e / n), i = (int)(e % n);
    const int gc = c < np_ ? st.p0 + c : st.q0 + (c - np_);
    work[g.v_off + (int64_t)gc * n + i] = V[e];
  }
  if (tid == 0 && any) rot[st.grp] = 1;
}

// sigma_j = |a_j| and u_j = a_j / sigma_j of a group matrix in the work buffer
__global__ __launch_bounds__(SVD_NT) void k_svd_finalize(const SvdItem* __restrict__ groups,
                                                         const int32_t* __restrict__ which,
                                                         double* __restrict__ work, double* __restrict__ sig) {
  const SvdItem g = groups[which[blockIdx.x]];
  const int m = g.m, n = g.n;
  const int seg = threadIdx.x / SVD_SEG, lane = threadIdx.x % SVD_SEG;
  constexpr int nseg = SVD_NT / SVD_SEG;
  for (int j = seg; j < n; j += nseg) {
    double* aj = work + g.a_off + (int64_t)j * m;
    double s2 = 0.0;
    for (int i = lane; i < m; i += SVD_SEG) s2 += aj[i] * aj[i];
    s2 = seg_sum(s2);
    const double sg = sqrt(s2);
    const double inv = sg > 0.0 ? 1.0 / sg : 0.0;
    for (int i = lane; i < m; i += SVD_SEG) aj[i] *= inv;
    if (lane == 0) sig[g.s_off + j] = sg;
  }
}

// V = identity for the groups listed
__global__ __launch_bounds__(256) void k_svd_init_v(const SvdItem* __restrict__ groups,
                                                    const int32_t* __restrict__ which, double* __restrict__ work) {
  const SvdItem g = groups[which[blockIdx.x]];
  const int64_t nn = (int64_t)g.n * g.n;
  for (int64_t e = threadIdx.x; e < nn; e += 256) work[g.v_off + e] = (e % (g.n + 1)) == 0 ? 1.0 : 0.0;
}

// result block: dst[r + c * rows] = src[src_off + r + col_c * ld] * scale_c
// over the kept columns (col_c, scale_c) = cols[col0 + c]
__global__ __launch_bounds__(64) void k_svd_scatter(const SvdScatter* __restrict__ items,
                                                    const SvdCol* __restrict__ cols, const double* __restrict__ work,
                                                    double* __restrict__ out) {
  const SvdScatter it = items[blockIdx.x];
  const int parts = col_parts(it.ncols);
  for (int k = blockIdx.y; k < it.ncols * parts; k += gridDim.y) {
    const int c = k / parts;
    const SvdCol col = cols[it.col0 + c];
    const double* x = work + it.src_off + (int64_t)col.col * it.ld;
    for (int r = 64 * (k % parts) + threadIdx.x; r < it.rows; r += 64 * parts)
      out[it.dst_off + r + (int64_t)c * it.rows] = x[r] * col.scale * it.scale;
  }
}

}  // namespace

void launch_svd_gather(const SvdGather* ditems, int nitems, const double* src, double* work, hipStream_t s) {
  if (nitems <= 0) return;
  hipLaunchKernelGGL(k_svd_gather, dim3(nitems, kColSplit), dim3(64), 0, s, ditems, src, work);
  QSX_HIP(hipGetLastError());
}

void launch_jacobi_lds(const SvdGroup* dgroups, const int32_t* dwhich, int n, double* work, int32_t* sweeps,
                       hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_jacobi_lds, dim3(n), dim3(SVD_NT_LDS), 0, s, dgroups, dwhich, work, sweeps);
  QSX_HIP(hipGetLastError());
}

void launch_jacobi_cross(const SvdGroup* dgroups, int ngroups, const SvdBlockStep* dsteps, int nsteps, double* work,
                         int32_t* rot, int sweep, hipStream_t s) {
  if (nsteps <= 0) return;
  hipLaunchKernelGGL(k_jacobi_cross, dim3(nsteps), dim3(SVD_NT_CROSS), 0, s, dgroups, ngroups, dsteps, work, rot,
                     sweep);
  QSX_HIP(hipGetLastError());
}

void launch_jacobi_whole(const SvdItem* ditems, const int32_t* dwhich, int n, double* work, double* sig,
                         int32_t* sweeps, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_jacobi_whole, dim3(n), dim3(SVD_NT), 0, s, ditems, dwhich, work, sig, sweeps);
  QSX_HIP(hipGetLastError());
}

int jacobi_max_sweeps() { return SVD_MAX_SWEEPS; }

void launch_jacobi_block(const SvdItem* dgroups, const SvdBlockStep* dsteps, int nsteps, double* work, int32_t* rot,
                         int sweep, hipStream_t s) {
  if (nsteps <= 0) return;
  hipLaunchKernelGGL(k_jacobi_block, dim3(nsteps), dim3(SVD_NT_BLOCK), 0, s, dgroups, dsteps, work, rot, sweep);
  QSX_HIP(hipGetLastError());
}

void launch_svd_finalize(const SvdItem* dgroups, const int32_t* dwhich, int n, double* work, double* sig,
                         hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_svd_finalize, dim3(n), dim3(SVD_NT), 0, s, dgroups, dwhich, work, sig);
  QSX_HIP(hipGetLastError());
}

void launch_svd_init_v(const SvdItem* dgroups, const int32_t* dwhich, int n, double* work, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_svd_init_v, dim3(n), dim3(256), 0, s, dgroups, dwhich, work);
  QSX_HIP(hipGetLastError());
}

void launch_svd_scatter(const SvdScatter* ditems, int nitems, const SvdCol* dcols, const double* work, double* out,
                        hipStream_t s) {
  if (nitems <= 0) return;
  hipLaunchKernelGGL(k_svd_scatter, dim3(nitems, kColSplit), dim3(64), 0, s, ditems, dcols, work, out);
  QSX_HIP(hipGetLastError());
}

}  // namespace qsx
