// split.hip -- split-precision H*psi data half: FP64 operands as S BF16
// slices, products on the BF16 matrix cores with FP32 accumulation that is
// exact by construction, recombined in FP64.
//
// Method (Ozaki-type error-free splitting, restated from the published
// scheme; no reference counterpart -- moondg/qspace has no GPU path):
//  * each contraction line of an operand block (a row of A over its k-range,
//    a column of B over its k-range) is scaled by a power of two 2^-e with
//    max |x| < 2^e, so every scaled element lies in (-1, 1);
//  * the scaled value r_0 = x 2^-e is cut into slices of 7 bits:
//    q_s = rint(r_s 2^{7(s+1)}) (|q_s| <= 128, exact in BF16),
//    sigma_s = q_s 2^{-7(s+1)}, r_{s+1} = r_s - sigma_s (exact in FP64),
//    so x = 2^e (sum_s sigma_s + r_S) with |r_S| <= 2^{-7S-1};
//  * products sigma^A_s sigma^B_t with s + t = u are integers times
//    2^{-7(u+2)} of at most 14 bits; a sum of at most (u+1) * 128 of them
//    fits the 24-bit FP32 significand, so accumulating one u-group over at
//    most 128 k (8 MFMAs of k = 16) in FP32 is exact (the slices are stored
//    with their scale, so acc_u holds the group's value itself);
//  * groups u = 0..S-1 are kept (S(S+1)/2 MFMAs per k-step of 16); every
//    128 k and at each pair end the FP32 accumulators are flushed into FP64:
//    C += afac 2^{e_row + f_col} sum_u acc_u.
// The truncation of the slice expansion and of the dropped groups u >= S
// leaves a relative error of about 2^{-7S} of |row| |col| per term: S = 6
// gives ~1e-13 relative to the operand scale; S <= 5 does not reach 1e-12.
//
// Layout: the lines of an operand block in groups of 16, k in blocks of 16, the S
// slices of a (group, k block) one after the other, each slice as its 64 quads
// of 4 consecutive k in the MFMA's lane order (quad (k%16)/4 of line l%16 at
// place 16 (k%16)/4 + l%16), zero beyond the block: one slice of an operand
// fragment is one contiguous load of the wave (512 bytes; 1 KB in FP32).
// (Each line's own quads in a row instead, 56 bytes per quad, scattered every
// load over 64 cache lines and every store over as many: 36.8 us per GEMM at
// D* = 4000, 20.7 us now, with the next k block's loads behind the MFMAs.)  Exponents are int32
// per line.  One wave computes one 16x16 output tile
// (v_mfma_f32_16x16x16bf16_1k: A lane l holds row l%16, k 4(l/16)..+3;
// B lane l holds k 4(l/16)..+3, col l%16; result element v of lane l is
// row 4(l/16)+v, col l%16 -- checked on the device with exact integers), or
// a k-chunk of it whose partial tile the wave engine's reduction sums.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "qsx_internal.hpp"

namespace qsx {

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int NT = 256;
constexpr int kFlushK = 128;   // k per exact FP32 accumulation window
constexpr int kSlot = 64 * 64; // scratch doubles per partial tile (the wave engine's reduce reads them)
constexpr int kGroupElems = kSplitGroupElems;

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// position of slice s of quad q of a line (pbase: its place in its group's
// first k block)
__device__ __forceinline__ int64_t packed_at(const SplitLine& L, int q, int s, int S) {
  return L.pbase + ((int64_t)(q >> 2) * S + s) * kGroupElems + (q & 3) * 64;
}

// the slices of a quad of elements, scaled by 2^-e.  BF16: with t_s = r_s 2^(7s),
// q_s = rint(128 t_s), t_{s+1} = 128 t_s - q_s (exact) and sigma_s = q_s 2^-7(s+1)
// (at most 8 significant bits, exact in FP32 and BF16).  FP32 x 3: sigma_0 on
// the 2^-11 grid, sigma_1 and sigma_2 the FP32 roundings of the remainders.
template <typename T, bool F32>
__device__ __forceinline__ void slice_quad(const double (&x)[4], int e, int S, const SplitLine& L, int q,
                                           T* __restrict__ P) {
  if constexpr (F32) {
    f4 o[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double r = ldexp(x[j], -e);
      const double s0 = rint(r * 2048.0) * (1.0 / 2048.0);
      r -= s0;
      const float s1 = (float)r;
      r -= (double)s1;
      o[0][j] = (float)s0;
      o[1][j] = s1;
      o[2][j] = (float)r;
    }
#pragma unroll
    for (int s = 0; s < 3; ++s) *(f4*)((float*)P + packed_at(L, q, s, 3)) = o[s];
  } else {
    double t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = ldexp(x[j], -e);
    float scale = 1.0f;
    for (int s = 0; s < S; ++s) {
      scale *= 1.0f / 128.0f;
      s4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double u = t[j] * 128.0, n = rint(u);
        t[j] = u - n;
        o[j] = (short)(__float_as_uint((float)n * scale) >> 16);
      }
      *(s4*)((uint16_t*)P + packed_at(L, q, s, S)) = o;
    }
  }
}

__device__ __forceinline__ void load_quad(const SplitLine& L, const double* __restrict__ X, int q, double (&x)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = 4 * q + j;
    x[j] = k < L.K ? X[L.off + (int64_t)k * L.sk] : 0.0;
  }
}

__device__ __forceinline__ double quad_max(const double (&x)[4]) {
  return fmax(fmax(fabs(x[0]), fabs(x[1])), fmax(fabs(x[2]), fabs(x[3])));
}

// one wave per contraction line (lines contiguous along k), a quad per lane:
// exponent (max |x| < 2^e), then the slices
template <typename T, bool F32>
__global__ __launch_bounds__(NT) void k_split_lines(const SplitLine* __restrict__ lines, int nlines,
                                                    const double* __restrict__ X, T* __restrict__ P, int S,
                                                    int32_t* __restrict__ exps) {
  const int li = uniform(blockIdx.x * (NT / 64) + (threadIdx.x >> 6));
  if (li >= nlines) return;
  const int lane = threadIdx.x & 63;
  const SplitLine L = lines[li];
  const int nq = (L.K + 3) >> 2;
  double x[4] = {0.0, 0.0, 0.0, 0.0}, mx = 0.0;
  for (int q = lane; q < nq; q += 64) {
    load_quad(L, X, q, x);
    mx = fmax(mx, quad_max(x));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  const int e = mx > 0.0 ? ilogb(mx) + 1 : 0;
  if (lane == 0) exps[L.eidx] = e;
  for (int q = lane; q < nq; q += 64) {
    if (nq > 64) load_quad(L, X, q, x);
    slice_quad<T, F32>(x, e, S, L, q, P);
  }
}

// lines whose elements are strided while neighbouring lines are adjacent (e.g.
// the rows of a column-major block): one workgroup per 16 lines, lane l taking
// line l%16 and every 16th quad, so that each load reads 16 adjacent elements
// and each store 16 adjacent quads; the waves' maxima meet in LDS.  A lane's
// first two quads stay in registers between the maximum and the slices (k <=
// 128: one read).  One launch where the exponents took a fill, an integer
// atomic maximum over a 2-D grid and a second read (three launches, 3.4 + 8.7 +
// 22 us at D* = 4000, intermediate and operators; 23 us now).  Whole H*psi with
// 7 slices, D* = 4000: 136 -> 90 us.
template <typename T, bool F32>
__global__ __launch_bounds__(NT) void k_split_groups(const SplitLine* __restrict__ lines, int nlines,
                                                     const double* __restrict__ X, T* __restrict__ P, int S,
                                                     int32_t* __restrict__ exps) {
  constexpr int NQ = NT / 16;  // quads per round
  __shared__ double wm[NT / 64][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = blockIdx.x * 16 + (lane & 15), q0 = wave * 4 + (lane >> 4);
  SplitLine L{};
  if (li < nlines) L = lines[li];
  const int nq = (L.K + 3) >> 2;
  double x[4], y[4];
  load_quad(L, X, q0, x);
  load_quad(L, X, q0 + NQ, y);
  double mx = fmax(quad_max(x), quad_max(y));
  for (int q = q0 + 2 * NQ; q < nq; q += NQ) {
    double z[4];
    load_quad(L, X, q, z);
    mx = fmax(mx, quad_max(z));
  }
  mx = fmax(mx, __shfl_xor(mx, 16, 64));
  mx = fmax(mx, __shfl_xor(mx, 32, 64));
  if (lane < 16) wm[wave][lane] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) mx = fmax(mx, wm[w][lane & 15]);
  const int e = mx > 0.0 ? ilogb(mx) + 1 : 0;
  if (threadIdx.x < 16 && li < nlines) exps[L.eidx] = e;
  if (q0 < nq) slice_quad<T, F32>(x, e, S, L, q0, P);
  if (q0 + NQ < nq) slice_quad<T, F32>(y, e, S, L, q0 + NQ, P);
  for (int q = q0 + 2 * NQ; q < nq; q += NQ) {
    load_quad(L, X, q, x);
    slice_quad<T, F32>(x, e, S, L, q, P);
  }
}

// the 16 x 16 tile of a wave (lane l holds rows 4(l/16)+v, column l%16):
// into C, or as a k-chunk's partial tile (column-major 16 x 16) into its
// scratch slot for the wave engine's reduction
__device__ __forceinline__ void store_tile(const WorkItem& w, const double (&c64)[4], double* __restrict__ C,
                                           double* __restrict__ scratch) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  if (w.slot >= 0) {
    double* sp = scratch + (int64_t)w.slot * kSlot;
#pragma unroll
    for (int v = 0; v < 4; ++v) sp[(4 * lq + v) + 16 * lr] = c64[v];
    return;
  }
  const int col = w.n0 + lr;
  if (col >= w.N) return;
  double* c = C + w.c_off;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int r = w.m0 + 4 * lq + v;
    if (r < w.M) c[r + (int64_t)w.M * col] = c64[v];
  }
}

// The lanes' quads of the k block at k that lie in the chunk [kb, ke) of a pair
// of depth K; every other quad of the block is zeroed (the padding beyond K
// is stored as zeros)
template <int S, typename V>
__device__ __forceinline__ void mask_chunk(V (&a)[S], int k, int kb, int ke, int K) {
  if (k >= kb && (k + 16 <= ke || ke == K)) return;  // uniform
  const int kq = k + 4 * ((threadIdx.x & 63) >> 4);
  if (kq >= kb && kq < ke) return;
#pragma unroll
  for (int s = 0; s < S; ++s) a[s] = V{0, 0, 0, 0};
}

// BF16 slices: per k block of 16 a lane's 8 bytes of every slice of both
// fragments (v_mfma_f32_16x16x16bf16_1k: A lane l holds row l%16, k
// 4(l/16)..+3; B lane l holds k 4(l/16)..+3, column l%16); the next block's are
// in flight behind the MFMAs
template <int S>
__global__ __launch_bounds__(NT) void k_split_gemm(const WorkItem* __restrict__ items, int nitems,
                                                   const SplitPair* __restrict__ pairs,
                                                   const uint16_t* __restrict__ Ap, const int32_t* __restrict__ expA,
                                                   const uint16_t* __restrict__ Bp, const int32_t* __restrict__ expB,
                                                   double* __restrict__ C, double* __restrict__ scratch) {
  const int wid = uniform(blockIdx.x * (NT / 64) + (threadIdx.x >> 6));
  if (wid >= nitems) return;
  const WorkItem w = items[wid];
  if (w.slot == -2) return;
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  const int col = w.n0 + lr;
  const bool colok = col < w.N;
  double c64[4] = {0.0, 0.0, 0.0, 0.0};
  for (int p = w.p0; p <= w.p1; ++p) {
    const SplitPair pd = pairs[p];
    const int kb = p == w.p0 ? w.k0 : 0, ke = p == w.p1 ? w.k1 : pd.K;
    const int64_t grp = (int64_t)((pd.K + 15) >> 4) * (S * kGroupElems);  // a group of 16 lines
    const s4* pa = (const s4*)(Ap + pd.pa + (w.m0 >> 4) * grp) + lane;
    const s4* pb = (const s4*)(Bp + pd.pb + (w.n0 >> 4) * grp) + lane;
    const int kf = kb & ~15;
    s4 a[S], b[S], an[S], bn[S];
    auto fetch = [&](int k, s4(&u)[S], s4(&v)[S]) {
      const int o = (k >> 4) * (S * kGroupElems / 4);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        u[s] = pa[o + s * (kGroupElems / 4)];
        v[s] = pb[o + s * (kGroupElems / 4)];
      }
    };
    if (kf < ke) fetch(kf, a, b);
    int er[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = w.m0 + 4 * lq + v;
      er[v] = r < w.M ? expA[pd.ea + r] : 0;
    }
    const int fc = colok ? expB[pd.eb + col] : 0;
    f4 acc[S];
#pragma unroll
    for (int u = 0; u < S; ++u) acc[u] = f4{0.f, 0.f, 0.f, 0.f};
    int win = 0;
    for (int k = kf; k < ke; k += 16) {
      if (k + 16 < ke) fetch(k + 16, an, bn);
      mask_chunk<S>(a, k, kb, ke, pd.K);  // a zero operand suffices
#pragma unroll
      for (int u = 0; u < S; ++u)
#pragma unroll
        for (int s = 0; s <= u; ++s)
          acc[u] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[s], b[u - s], acc[u], 0, 0, 0);
      win += 16;
      if (win >= kFlushK || k + 16 >= ke) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          double t = 0.0;
#pragma unroll
          for (int u = S - 1; u >= 0; --u) t += (double)acc[u][v];
          c64[v] += pd.afac * ldexp(t, er[v] + fc);
        }
#pragma unroll
        for (int u = 0; u < S; ++u) acc[u] = f4{0.f, 0.f, 0.f, 0.f};
        win = 0;
      }
#pragma unroll
      for (int s = 0; s < S; ++s) {
        a[s] = an[s];
        b[s] = bn[s];
      }
    }
  }
  store_tile(w, c64, C, scratch);
}

// ---------------------------------------------------------------- FP32 x 3
// Three FP32 slices per element, products on the FP32 matrix cores
// (v_mfma_f32_16x16x4f32: A lane l holds row l%16 at one k, B lane l holds
// that k at column l%16, the four lane groups the four k of the MFMA;
// result element v of lane l is row 4(l/16)+v, column l%16), FP32
// accumulation, FP64 recombination:
//  * a line's scaled value r = x 2^-e in (-1, 1) is cut as sigma_0 =
//    rint(r 2^11) 2^-11 (at most 12 significant bits), sigma_1 =
//    fl32(r - sigma_0), sigma_2 = fl32(r - sigma_0 - sigma_1); the remainder
//    is below 2^-60;
//  * sigma_0 products are integers times 2^-22 below 2^22 in magnitude, so one
//    MFMA's sum of four is exact in FP32 and is added to FP64 after every
//    MFMA (u = 0);
//  * the groups u = 1 (sigma_0 sigma_1 + sigma_1 sigma_0, |.| < 2^-11) and
//    u = 2 (sigma_1 sigma_1 + sigma_0 sigma_2 + sigma_2 sigma_0) accumulate in
//    FP32 over a window of 32 k and are rounded at 2^-24 of their size: about
//    2^-35 of |row| |col| per term, the bound of this variant (the sigma_1
//    sigma_2 and sigma_2 sigma_2 products, below 2^-58, are dropped).
// Per k-step of 16 lane group g takes the quad k + 4g..+3 for the 4 MFMAs
// (MFMA j uses element j of every group's quad: the k order inside the step
// is permuted, which the sum does not see), so each lane loads its 3 slices
// as 16 bytes of 3 contiguous 1 KB runs.
constexpr int kF32Win = 32;  // k per FP32 accumulation window of u = 1, 2

__global__ __launch_bounds__(NT) void k_split_gemm_f32(const WorkItem* __restrict__ items, int nitems,
                                                       const SplitPair* __restrict__ pairs,
                                                       const float* __restrict__ Ap, const int32_t* __restrict__ expA,
                                                       const float* __restrict__ Bp, const int32_t* __restrict__ expB,
                                                       double* __restrict__ C, double* __restrict__ scratch) {
  const int wid = uniform(blockIdx.x * (NT / 64) + (threadIdx.x >> 6));
  if (wid >= nitems) return;
  const WorkItem w = items[wid];
  if (w.slot == -2) return;
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  const int col = w.n0 + lr;
  const bool colok = col < w.N;
  double c64[4] = {0.0, 0.0, 0.0, 0.0};
  for (int p = w.p0; p <= w.p1; ++p) {
    const SplitPair pd = pairs[p];
    const int kb = p == w.p0 ? w.k0 : 0, ke = p == w.p1 ? w.k1 : pd.K;
    const int64_t grp = (int64_t)((pd.K + 15) >> 4) * (3 * kGroupElems);  // a group of 16 lines
    const f4* pa = (const f4*)(Ap + pd.pa + (w.m0 >> 4) * grp) + lane;
    const f4* pb = (const f4*)(Bp + pd.pb + (w.n0 >> 4) * grp) + lane;
    double sc[4];
    const int fc = colok ? expB[pd.eb + col] : 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = w.m0 + 4 * lq + v;
      sc[v] = pd.afac * ldexp(1.0, (r < w.M ? expA[pd.ea + r] : 0) + fc);
    }
    f4 acc1 = f4{0.f, 0.f, 0.f, 0.f}, acc2 = f4{0.f, 0.f, 0.f, 0.f};
    int win = 0;
    const f4 z = f4{0.f, 0.f, 0.f, 0.f};
    const int kf = kb & ~15;
    f4 a[3] = {z, z, z}, b[3] = {z, z, z}, an[3], bn[3];
    auto fetch = [&](int k, f4(&u)[3], f4(&v)[3]) {
      const int o = (k >> 4) * (3 * kGroupElems / 4);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        u[s] = pa[o + s * (kGroupElems / 4)];
        v[s] = pb[o + s * (kGroupElems / 4)];
      }
    };
    if (kf < ke) fetch(kf, a, b);
    for (int k = kf; k < ke; k += 16) {
      if (k + 16 < ke) fetch(k + 16, an, bn);
      mask_chunk<3>(a, k, kb, ke, pd.K);  // a zero operand suffices
      const f4 a0 = a[0], a1 = a[1], a2 = a[2], b0 = b[0], b1 = b[1], b2 = b[2];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f4 acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[j], b0[j], z, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[j], b1[j], acc1, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[j], b0[j], acc1, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[j], b1[j], acc2, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[j], b2[j], acc2, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[j], b0[j], acc2, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) c64[v] += sc[v] * (double)acc0[v];
      }
      win += 16;
      if (win >= kF32Win || k + 16 >= ke) {
#pragma unroll
        for (int v = 0; v < 4; ++v) c64[v] += sc[v] * ((double)acc2[v] + (double)acc1[v]);
        acc1 = z;
        acc2 = z;
        win = 0;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        a[s] = an[s];
        b[s] = bn[s];
      }
    }
  }
  store_tile(w, c64, C, scratch);
}

template <typename T, bool F32>
void lines_launch(const SplitLine* dlines, int nlines, bool grouped, const double* X, T* P, int S,
                  int32_t* exps, hipStream_t s) {
  if (nlines <= 0) return;
  if (grouped) {
    hipLaunchKernelGGL((k_split_groups<T, F32>), dim3((nlines + 15) / 16), dim3(NT), 0, s, dlines, nlines, X, P, S,
                       exps);
  } else {
    const int nb = (nlines + NT / 64 - 1) / (NT / 64);
    hipLaunchKernelGGL((k_split_lines<T, F32>), dim3(nb), dim3(NT), 0, s, dlines, nlines, X, P, S, exps);
  }
  QSX_HIP(hipGetLastError());
}

}  // namespace

void launch_split_lines(const SplitLine* dlines, int nlines, bool per_lane, const double* X,
                        uint16_t* planes, int S, int32_t* exps, hipStream_t s) {
  lines_launch<uint16_t, false>(dlines, nlines, per_lane, X, planes, S, exps, s);
}

void launch_split_lines_f32(const SplitLine* dlines, int nlines, bool per_lane, const double* X,
                            float* planes, int32_t* exps, hipStream_t s) {
  lines_launch<float, true>(dlines, nlines, per_lane, X, planes, 3, exps, s);
}

void launch_split_gemm(int S, const WorkItem* ditems, int nitems, const SplitPair* dpairs, const uint16_t* Ap,
                       const int32_t* expA, const uint16_t* Bp, const int32_t* expB, double* C, double* scratch,
                       hipStream_t s) {
  if (nitems <= 0) return;
  const int nb = (nitems + NT / 64 - 1) / (NT / 64);
  switch (S) {
#define QSX_SPLIT_CASE(n)                                                                                     \
  case n:                                                                                                     \
    hipLaunchKernelGGL(k_split_gemm<n>, dim3(nb), dim3(NT), 0, s, ditems, nitems, dpairs, Ap, expA, Bp, expB, C, \
                       scratch);                                                                              \
    break;
    QSX_SPLIT_CASE(3) QSX_SPLIT_CASE(4) QSX_SPLIT_CASE(5) QSX_SPLIT_CASE(6) QSX_SPLIT_CASE(7) QSX_SPLIT_CASE(8)
#undef QSX_SPLIT_CASE
    default: fail(QSX_ERR_ARG, "split precision: %d slices (3..8 supported)", S);
  }
  QSX_HIP(hipGetLastError());
}

void launch_split_gemm_f32(const WorkItem* ditems, int nitems, const SplitPair* dpairs, const float* Ap,
                           const int32_t* expA, const float* Bp, const int32_t* expB, double* C, double* scratch,
                           hipStream_t s) {
  if (nitems <= 0) return;
  const int nb = (nitems + NT / 64 - 1) / (NT / 64);
  hipLaunchKernelGGL(k_split_gemm_f32, dim3(nb), dim3(NT), 0, s, ditems, nitems, dpairs, Ap, expA, Bp, expB, C,
                     scratch);
  QSX_HIP(hipGetLastError());
}

}  // namespace qsx
