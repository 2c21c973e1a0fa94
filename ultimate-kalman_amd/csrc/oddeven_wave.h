/*
 * oddeven_wave.h -- Householder QR of a stacked pair of blocks on one wave
 * (n <= 32), shared by oddeven_small.hip (n <= 16, the three phases of a step
 * pair in one kernel), oddeven_mid{20,24,28,32}.hip (16 < n <= 32, a kernel per
 * phase or per short level) and filter_small.hip; and a Cholesky factorization
 * of matrix-core tiles (n <= 64), shared by associative.hip and the dense
 * whitening of oddeven.hip.
 *
 * Layout: 16 matrix columns are a tile; lane (li, lk) = (lane % 16, lane / 16)
 * holds rows 4 g + lk, g = 0 .. NK - 1, of the tile's column li in NK = ceil(n
 * / 4) registers per block. The two stacked blocks of a QR (the pivot rows and
 * the rows below them) are registers [0, NK) and [NK, 2 NK). Then
 *   - the pivot column reaches every lane by a DPP row broadcast (a row of 16
 *     lanes shares lk, so lane k % 16 of each row has the rows its lanes need);
 *   - a dot product is one multiply-add per row granule and lane and one sum
 *     over the four lane rows, which a small matrix-core product with ones
 *     forms and hands to all lanes in one instruction.
 * A Householder step uses no LDS and no barrier. The steps are unrolled, each
 * with the granules that can hold a nonzero of its vector.
 */
#ifndef UKHIP_ODDEVEN_WAVE_H
#define UKHIP_ODDEVEN_WAVE_H

#include <hip/hip_runtime.h>

#include <utility>

#include "oddeven_qr.h"

namespace {

typedef float sm_f4 __attribute__((ext_vector_type(4)));

/* v of lane K (0 .. 15) of each row of 16 lanes, on all of its lanes */
template <int K>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xf, 0xf, true));
}
template <int K>
__device__ __forceinline__ double row_lane(double v) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + K, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + K, 0xf, 0xf, true));
}
/* v of lane `lane` (a constant), uniform */
__device__ __forceinline__ float one_lane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double one_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
/* the sum of v over lanes li, li + 16, li + 32, li + 48, on all four: the
 * product of a matrix of ones with v on the matrix cores (27 cycles measured,
 * against 68 for two cross-row swaps and additions in FP64; 43 against 52 in
 * FP32) */
__device__ __forceinline__ double rows_sum(double v) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, v, 0.0, 0, 0, 0);
}
__device__ __forceinline__ float rows_sum(float v) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(1.0f, v, sm_f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0)[0];
}

/* which registers can hold a nonzero of the Householder vector of pivot row
 * granule G (the structure flags of oddeven_qr.h, by granules of four rows) */
__host__ __device__ constexpr bool sm_need(int l, int NK, int G, int QF) {
  const int hg = (NK + 1) / 2;
  if (l < NK) return l >= G && (!(QF & QF_HALF0) || l < hg || l == G) && (!(QF & QF_DIAG0) || l == G);
  const int g = l - NK;
  return (!(QF & QF_TRI1) || g <= G) && (!(QF & QF_HALF1) || g < hg);
}
/* rows of a block that QF_HALF0 / QF_HALF1 keep */
__host__ __device__ constexpr int sm_half_rows(int NK) { return 4 * ((NK + 1) / 2); }

/* The scalars of a Householder step whose vector stays unscaled (the pivot
 * column with ukk on its pivot row): H = I - f1 f2^2 x x^T. FP32 as FP64:
 * rounded like exact operations, and 1 / (u^T u / 2) in one piece: with the
 * product of tau and two rounded reciprocals of ukk the mixed path's estimates
 * were further off, 1.40 times at n = 4 and 1.30 at n = 32 (k = 3000, one
 * refinement). f2 is a power of two that keeps squares in range. */
__device__ __forceinline__ void wave_scalars(double alpha, double s, double& ukk, double& f1, double& f2) {
  house_scalars(alpha, s, ukk, f1, f2);
}
__device__ __forceinline__ void wave_scalars(float alpha, float s, float& ukk, float& f1, float& f2) {
  const float t2 = fmaf(alpha, alpha, s);
  const bool tiny = t2 < 1e-28f, big = t2 > 1e28f;
  f2 = tiny ? 0x1p32f : big ? 0x1p-32f : 1.0f;
  const float a = alpha * f2, t = t2 * f2 * f2, aa = fabsf(a);
  const float y = __builtin_amdgcn_rsqf(t), h = 0.5f * y;
  float g = t * y;
  float w = __builtin_amdgcn_rcpf(fmaf(aa, g, t));
  g = fmaf(fmaf(-g, g, t), h, g); /* sqrt(t) */
  const float v = fmaf(aa, g, t);
  w = fmaf(fmaf(-v, w, 1.0f), w, w);
  ukk = alpha + copysignf(g * (tiny ? 0x1p-32f : big ? 0x1p32f : 1.0f), alpha);
  f1 = s != 0.0f ? w : 0.0f;
}

/* One Householder step: pivot column K (tile K / 16, lane K % 16), target row
 * K, applied to tiles K / 16 .. TILES - 1 and, on the first step of a pivot
 * tile, to the right-hand side where it is (e before step 0, lane li = 0 of
 * the finished tile before step 16). A zero column changes nothing: the
 * scalars of a column that counts as zero are zeros. Finished columns of the pivot tile are computed on below their pivots, where
 * they are never stored. */
template <int K, int NK, int TILES, int QF, class T>
__device__ __forceinline__ void sm_step(T (&a)[TILES][2 * NK], T (&e)[2 * NK], int lk) {
  constexpr int G = K / 4, KR = K % 4, PT = K / 16, NT = TILES - PT; /* tiles at work */
  constexpr bool EXTRA = K % 16 == 0;
  T(&ex)[2 * NK] = PT == 0 ? e : a[PT == 0 ? 0 : PT - 1];
  T x[2 * NK];
#pragma unroll
  for (int l = 0; l < 2 * NK; ++l)
    if (sm_need(l, NK, G, QF)) x[l] = row_lane<K % 16>(a[PT][l]);
  const T alpha = one_lane(x[G], 16 * KR);
  x[G] = lk > KR ? T(x[G]) : T(0);
  T q[2] = {T(0), T(0)}, d[NT + 1][2];
#pragma unroll
  for (int l = 0; l < 2 * NK; ++l)
    if (sm_need(l, NK, G, QF)) q[l & 1] = fma(x[l], x[l], q[l & 1]);
  const T s = rows_sum(q[0] + q[1]);
#pragma unroll
  for (int t = 0; t < NT + (EXTRA ? 1 : 0); ++t) {
    T(&c)[2 * NK] = t < NT ? a[t < NT ? PT + t : 0] : ex;
    d[t][0] = d[t][1] = T(0);
#pragma unroll
    for (int l = 0; l < 2 * NK; ++l)
      if (l != G && sm_need(l, NK, G, QF)) d[t][l & 1] = fma(x[l], c[l], d[t][l & 1]);
  }
  T ukk, f1, f2;
  wave_scalars(alpha, s, ukk, f1, f2);
  const bool none = f1 == T(0);
  ukk = none ? T(0) : T(ukk);
  if (sizeof(T) == 4) f2 = none ? T(0) : T(f2);
  const T ff = sizeof(T) == 4 ? T(-f1 * f2) : T(-f1);
  x[G] = lk == KR ? T(ukk) : T(x[G]);
#pragma unroll
  for (int t = 0; t < NT + (EXTRA ? 1 : 0); ++t) {
    T(&c)[2 * NK] = t < NT ? a[t < NT ? PT + t : 0] : ex;
    T v = fma(x[G], c[G], d[t][0] + d[t][1]);
    v = rows_sum(v);
    if (sizeof(T) == 4) v *= f2;
    const T tw = ff * v;
#pragma unroll
    for (int l = 0; l < 2 * NK; ++l)
      if (sm_need(l, NK, G, QF)) c[l] = fma(tw, x[l], c[l]);
  }
}

template <int K0, int NK, int TILES, int QF, class T, int... K>
__device__ __forceinline__ void sm_steps(T (&a)[TILES][2 * NK], T (&e)[2 * NK], int lk, int n,
                                         std::integer_sequence<int, K...>) {
  auto one = [&](auto k) { /* only the last granule can hold columns that are no pivots */
    if (k.value <= 4 * NK - 4 || k.value < n) sm_step<k.value, NK, TILES, QF, T>(a, e, lk);
  };
  (one(std::integral_constant<int, K0 + K>{}), ...);
}
/* What the right-hand side's travel leaves of the columns whose lanes it
 * takes: column 0 is final after step 0 (its one nonzero, in lane 0), column
 * 16 after step 16 (rows 0 .. 16, in lanes li = 0). */
template <int NK, class T>
struct SmKept {
  T r00;
  T c16[NK > 4 ? 5 : 1];
};
/* QR of columns 0 .. n - 1 applied to the columns after them and to the
 * right-hand side e (lanes li = 0). The right-hand side has no tile of its
 * own (at n = 16 or 32 it would open one for a single column): after the first
 * step of a pivot tile it moves into the lanes of that tile's first column.
 * Afterwards it is in lanes li = 0 of the last pivot tile. */
template <int NK, int TILES, int QF, class T>
__device__ __forceinline__ void sm_qr(T (&a)[TILES][2 * NK], T (&e)[2 * NK], SmKept<NK, T>& kept, int n, int li, int lk) {
  sm_step<0, NK, TILES, QF, T>(a, e, lk);
  kept.r00 = a[0][0];
#pragma unroll
  for (int l = 0; l < 2 * NK; ++l) a[0][l] = li == 0 ? T(e[l]) : T(a[0][l]);
  sm_steps<1, NK, TILES, QF, T>(a, e, lk, n, std::make_integer_sequence<int, (NK > 4 ? 16 : 4 * NK) - 1>{});
  if constexpr (NK > 4) {
    sm_step<16, NK, TILES, QF, T>(a, e, lk);
#pragma unroll
    for (int g = 0; g < 5; ++g) kept.c16[g] = a[1][g];
#pragma unroll
    for (int l = 0; l < 2 * NK; ++l) a[1][l] = li == 0 ? T(a[0][l]) : T(a[1][l]);
    sm_steps<17, NK, TILES, QF, T>(a, e, lk, n, std::make_integer_sequence<int, 4 * NK - 17>{});
  }
}

/* loads: register g <- element (4 g + lk, li) of a block with `rows` rows, ld
 * `ld`, `cols` columns, zero outside it; without a branch (src readable at its
 * first entry), so that all of a pair's loads are under way together */
template <int NK, class T>
__device__ __forceinline__ void sm_load(T* v, const T* __restrict__ src, int ld, int rows, int cols, int li, int lk) {
#pragma unroll
  for (int g = 0; g < NK; ++g) {
    const int r = 4 * g + lk;
    const bool in = r < rows && li < cols;
    const T x = src[in ? r + li * ld : 0];
    v[g] = in ? x : T(0);
  }
}
/* the same for sign * diag(w) M with M in double, each product rounded to T */
template <int NK, class T>
__device__ __forceinline__ void sm_load_scaled(T* v, const double* __restrict__ w, const double* __restrict__ M, int ld,
                                               int rows, int cols, double sign, int li, int lk) {
#pragma unroll
  for (int g = 0; g < NK; ++g) {
    const int r = 4 * g + lk;
    const bool in = r < rows && li < cols;
    const T x = T(sign * w[in ? r : 0] * M[in ? r + li * ld : 0]);
    v[g] = in ? x : T(0);
  }
}
/* a vector (the right-hand side; the same on every li) */
template <int NK, class T>
__device__ __forceinline__ void sm_load_vec(T* v, const T* __restrict__ src, int rows, int lk) {
#pragma unroll
  for (int g = 0; g < NK; ++g) {
    const int r = 4 * g + lk;
    const T x = src[r < rows ? r : 0];
    v[g] = r < rows ? x : T(0);
  }
}
template <int NK, class T>
__device__ __forceinline__ void sm_store(T* __restrict__ dst, const T* v, int ld, int rows, int cols, int li, int lk) {
  if (li < cols) {
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      const int r = 4 * g + lk;
      if (r < rows) dst[r + (int64_t)li * ld] = v[g];
    }
  }
}
/* tile 0 after sm_qr as its upper triangle (column 0: r00), n x n */
template <int NK, class T>
__device__ __forceinline__ void sm_store_triu(T* __restrict__ dst, const T* v, T r00, int n, int li, int lk) {
  if (li < n) {
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      const int r = 4 * g + lk;
      const T x = li == 0 ? (r == 0 ? T(r00) : T(0)) : (r <= li ? T(v[g]) : T(0));
      if (r < n) dst[r + (int64_t)li * n] = x;
    }
  }
}
/* the right-hand side out of lanes li = 0 */
template <int NK, class T>
__device__ __forceinline__ void sm_store_vec(T* __restrict__ dst, const T* v, int rows, int li, int lk) {
  if (li == 0) {
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      const int r = 4 * g + lk;
      if (r < rows) dst[r] = v[g];
    }
  }
}

/* ------------------------------------------------------------------------ */
/* Cholesky factorization on the matrix cores' tiles (n <= 64)               */
/* ------------------------------------------------------------------------ */

typedef double as_d4 __attribute__((ext_vector_type(4)));
/* D = A B + C on 16 x 16 x 4: lane (li, lk) supplies A[li][lk] and B[lk][li];
 * element r of the accumulator is D[4 r + lk][li]. So an accumulator is the
 * next product's B as it stands, and its transpose's A. */
__device__ __forceinline__ as_d4 as_mfma(double a, double b, as_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

/* Lets the matrix products before it finish. The compiler places the wait
 * states between a product and the first read of its result, but where
 * branches follow the product it counts them along one of the paths to the
 * read, another can be too short, and the read gets the sum without its last
 * term. So a group of products ends with this, in the same block. */
__device__ __forceinline__ void mfma_drain() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15\n\ts_nop 3");
  __builtin_amdgcn_sched_barrier(0);
}

/*
 * One step of the Cholesky factorization of a symmetric positive definite 16 x
 * 16 tile on one wave (accumulator layout): a is reduced to D L^T (row K final
 * at step K), wt becomes the transposed inverse of the unit lower factor. The
 * pivots are kept by row (pr) and by column (pc). FLOOR: a pivot below fl (lane
 * li: of row li), the rounding error of its original diagonal entry, counts as
 * that error, so that a semidefinite matrix has a factor too (a perturbation
 * of the size of the matrix's own rounding); NaN stays NaN.
 */
template <int K, bool FLOOR>
__device__ __forceinline__ void chol_step(double (&a)[4], double (&wt)[4], double (&pr)[4], double& pc, double fl,
                                          int li, int lk) {
  constexpr int G = K / 4, KR = K % 4;
  double x[4];
#pragma unroll
  for (int g = G; g < 4; ++g) x[g] = row_lane<K>(a[g]);
  double p = one_lane(x[G], 16 * KR);
  if (FLOOR) {
    const double f = one_lane(fl, K);
    p = p < f ? f : p;
  }
  double rp = __builtin_amdgcn_rcp(p);
  rp = fma(fma(-p, rp, 1.0), rp, rp);
  rp = fma(fma(-p, rp, 1.0), rp, rp);
  const double row = rows_sum(lk == KR ? a[G] : 0.0) * rp; /* row K over the pivot, on every lane row */
  x[G] = lk > KR ? x[G] : 0.0;
#pragma unroll
  for (int g = G; g < 4; ++g) a[g] = fma(-x[g], row, a[g]);
  const double m = li > K ? row : 0.0;
#pragma unroll
  for (int g = 0; g <= G; ++g) wt[g] = fma(-row_lane<K>(wt[g]), m, wt[g]);
  pr[G] = lk == KR ? p : pr[G];
  pc = li == K ? p : pc;
}
template <bool FLOOR, int... K>
__device__ __forceinline__ void chol_steps(double (&a)[4], double (&wt)[4], double (&pr)[4], double& pc,
                                           double fl, int lim, int li, int lk,
                                           std::integer_sequence<int, K...>) {
  auto one = [&](auto k) {
    if (k.value < lim) chol_step<k.value, FLOOR>(a, wt, pr, pc, fl, li, lk);
  };
  (one(std::integral_constant<int, K>{}), ...);
}
__device__ __forceinline__ double rsqrt_ulp(double p) {
  const double y = __builtin_amdgcn_rsq(p);
  const double y1 = fma(0.5 * y, fma(-p * y, y, 1.0), y);
  return fma(0.5 * y1, fma(-p * y1, y1, 1.0), y1);
}

}  // namespace

#endif /* UKHIP_ODDEVEN_WAVE_H */
