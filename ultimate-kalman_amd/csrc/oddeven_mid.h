/*
 * oddeven_mid.h -- the odd-even elimination's three phases for 16 < n <= 32,
 * one wave per step pair (or even step) and launch, on the layout and the
 * Householder steps of oddeven_wave.h; NK = ceil(n / 4) is compiled in
 * oddeven_mid{20,24,28,32}.hip.
 *
 * Reference: c/kalman_oddeven_smoother.c (phases :379-560, fix-last
 * :1452-1476, renaming :563-597).
 *
 * The phases' matrices are those of k_phase1..3 (oddeven_qr.h), their columns
 * packed into tiles of 16 in the order P, Q, Bl; the right-hand side travels
 * in the pivots' freed lanes. A phase is a kernel of its own: its unrolled
 * steps take 25 to 50 KB of code, and the three together would not stay in the
 * instruction cache.
 */
#ifndef UKHIP_ODDEVEN_MID_H
#define UKHIP_ODDEVEN_MID_H

#include <hip/hip_runtime.h>

#include "oddeven_wave.h"

namespace {

constexpr int MID_WAVES = 4; /* waves (work items) per workgroup */
/* Waves per SIMD asked of the register allocator. The steps' chains and the
 * fetching of their straight-line code leave a lone wave's SIMD idle more than
 * half of the time, so a second or third wave is worth a few spilled
 * registers. */
__host__ __device__ constexpr int mid_occ(int NK, int phase, bool fp32) {
  if (phase == 2) return fp32 ? (NK <= 6 ? 4 : 3) : 2;
  return fp32 ? (phase == 1 ? 4 : 5) : 2;
}

/* a tile's registers of one block <- rows [0, rows) of each lane's own column
 * at p, zero where !on. FULL: rows is n, so only the last granule can end
 * inside. The registers start as zeros and are loaded under one branch: no
 * register is written again while its load is under way. */
template <int NK, bool FULL, class T>
__device__ __forceinline__ void mid_load(T* v, const T* __restrict__ p, bool on, int rows, int lk) {
#pragma unroll
  for (int g = 0; g < NK; ++g) v[g] = T(0);
  if (on) {
#pragma unroll
    for (int g = 0; g < NK; ++g)
      if ((FULL && g < NK - 1) || 4 * g + lk < rows) v[g] = p[4 * g + lk];
  }
}
/* the same for sign * diag(w) times the column, in double, each product
 * rounded to T; w the same for every column. rows <= the readable rows of w. */
template <int NK, class T>
__device__ __forceinline__ void mid_load_scaled(T* v, const double* __restrict__ w, const double* __restrict__ p,
                                                bool on, int rows, double sign, int lk) {
  const int last = rows > 0 ? rows - 1 : 0;
  double x[NK], f[NK];
#pragma unroll
  for (int g = 0; g < NK; ++g) {
    const int r = 4 * g + lk, rr = r < last ? r : last;
    f[g] = w[rr];
    x[g] = on ? p[rr] : 0.0;
  }
#pragma unroll
  for (int g = 0; g < NK; ++g) v[g] = on && 4 * g + lk < rows ? T(sign * f[g] * x[g]) : T(0);
}
template <int NK, bool FULL, class T>
__device__ __forceinline__ void mid_store(T* __restrict__ p, const T* v, bool on, int rows, int lk) {
  if (on) {
#pragma unroll
    for (int g = 0; g < NK; ++g)
      if ((FULL && g < NK - 1) || 4 * g + lk < rows) p[4 * g + lk] = v[g];
  }
}
/* register g of pivot tile i after sm_qr as an entry of the upper triangle:
 * columns 0 and 16 from where the right-hand side left them, zero below the
 * diagonal */
template <int NK, int TILES, class T>
__device__ __forceinline__ T mid_pivot(const T (&a)[TILES][2 * NK], const SmKept<NK, T>& kept, int i, int g, int li, int lk) {
  const T own = li != 0 ? T(a[i][g]) : i == 0 ? (g == 0 ? T(kept.r00) : T(0)) : (g < 5 ? T(kept.c16[g < 5 ? g : 0]) : T(0));
  return 4 * g + lk <= 16 * i + li ? T(own) : T(0);
}
/* the pivot tiles after sm_qr as an upper triangle (ld n) */
template <int NK, int TILES, class T>
__device__ __forceinline__ void mid_store_triu(T* __restrict__ dst, const T (&a)[TILES][2 * NK], const SmKept<NK, T>& kept,
                                               int n, int li, int lk) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = 16 * t + li;
    T x[NK];
#pragma unroll
    for (int g = 0; g < NK; ++g) x[g] = mid_pivot<NK>(a, kept, t, g, li, lk);
    mid_store<NK, true>(dst + (int64_t)c * n, x, c < n, n, lk);
  }
}

/* LV: the level's stacked rows (C): 0 dense, 1 at most sm_half_rows(NK) rows, 2
 * upper triangular n x n (the levels above 0; B and D stored in full) */
template <int NK, class T, int LV>
__global__ void __launch_bounds__(64 * MID_WAVES, (mid_occ(NK, 1, sizeof(T) == 4)))
    k_mid1(uk_level_t lv, ChainT<T> in, ChainT<T> out, FactorsT<T> fac, int n) {
  constexpr int TILES = (NK + 1) / 2;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int64_t e = (int64_t)blockIdx.x * MID_WAVES + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (e >= lv.evens) return; /* whole waves; no barrier below */
  const int p = (int)find_problem(lv.even_start, lv.nprob, e);
  const int64_t u0 = lv.even_start[p], L = lv.L[p], s0 = lv.step_start[p], t0 = lv.next_start[p];
  const int64_t u = e - u0, j = 2 * u, t = t0 + u, sj = s0 + j, sp = sj + 1, nn = (int64_t)n * n;
  const int mr = LV == 2 ? n : in.mr;
  const bool lone = j + 1 == L;
  const bool b_synth = LV != 2 && in.b_synth, c_synth = LV != 2 && sizeof(T) == 4 && in.c_synth;
  const bool d_diag = LV != 2 && in.d_diag;
  T a[TILES][2 * NK], re[2 * NK];
  SmKept<NK, T> kept;
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int c = 16 * i + li;
    const bool isP = c < n, isQ = !lone && c >= n && c < 2 * n;
    const int qc = isP ? c : c - n;
    const T* p0 = isP ? in.B + sp * nn + qc * n : in.D + sp * nn + (d_diag ? 0 : qc * n);
    mid_load<NK, true>(a[i], p0, !lone && (isP ? !b_synth : isQ), n, lk);
    mid_load<NK, LV == 2>(a[i] + NK, in.C + sj * nn + qc * mr, isP && !c_synth, mr, lk);
  }
  mid_load<NK, true>(re, in.c + sp * n, !lone, n, lk);
  mid_load<NK, LV == 2>(re + NK, in.o + sj * n, true, mr, lk);
  if (d_diag) {
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      const int c = 16 * i + li;
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][g] = (c < n || 4 * g + lk == c - n) ? T(a[i][g]) : T(0);
    }
  }
  if (b_synth && !lone) {
    const double* F = in.wF + (in.wFidx ? in.wFidx[sp] * nn : 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = 16 * i + li;
      T v[NK];
      mid_load_scaled<NK>(v, in.wk + sp * n, F + c * n, c < n, n, -1.0, lk);
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][g] = c < n ? T(v[g]) : T(a[i][g]);
    }
  }
  if (c_synth) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = 16 * i + li;
      mid_load_scaled<NK>(a[i] + NK, in.rC + sj * mr, in.rG + sj * (int64_t)mr * n + c * mr, c < n, min(mr, in.rm[sj]), 1.0, lk);
    }
  }
  constexpr int QF = (LV == 1 ? QF_HALF1 : 0) | (LV == 2 ? QF_TRI1 : 0);
  sm_qr<NK, TILES, QF, T>(a, re, kept, n, li, lk);
  mid_store_triu<NK>(fac.R + e * nn, a, kept, n, li, lk);
#pragma unroll
  for (int i = 1; i < TILES; ++i) {
    const int c = 16 * i + li;
    const bool isQ = !lone && c >= n && c < 2 * n;
    mid_store<NK, true>(fac.Y + e * nn + (int64_t)(c - n) * n, a[i], isQ, n, lk);                  /* X_j */
    mid_store<NK, LV == 2>(out.C + t * nn + (int64_t)(c - n) * mr, a[i] + NK, isQ, mr, lk);        /* D~_{j+1} */
  }
  mid_store<NK, true>(fac.cf + e * n, a[1], li == 0, n, lk);                                        /* o_j */
  mid_store<NK, LV == 2>(out.o + t * n, a[1] + NK, li == 0 && !lone, mr, lk);                       /* c~_{j+1} */
  if (lone)
    for (int i = lane; i < nn; i += 64) fac.Y[e * nn + i] = T(0);
  if (j == 0)
    for (int i = lane; i < nn; i += 64) fac.Bt[e * nn + i] = T(0);
}

/* DV: the level's D and B blocks: 0 both stored in full, 1 D diagonal and B
 * formed on load, 2 D in full and B formed on load */
template <int NK, class T, int DV>
__global__ void __launch_bounds__(64 * MID_WAVES, (mid_occ(NK, 2, sizeof(T) == 4)))
    k_mid2(uk_level_t lv, ChainT<T> in, ChainT<T> out, FactorsT<T> fac, T* __restrict__ fix, int n) {
  constexpr int TILES = (3 * NK + 3) / 4;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int64_t e = (int64_t)blockIdx.x * MID_WAVES + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (e >= lv.evens) return; /* whole waves; no barrier below */
  const int p = (int)find_problem(lv.even_start, lv.nprob, e);
  const int64_t u0 = lv.even_start[p], L = lv.L[p], s0 = lv.step_start[p], t0 = lv.next_start[p];
  const int64_t u = e - u0, j = 2 * u, t = t0 + u, sj = s0 + j, nn = (int64_t)n * n;
  if (j == 0) return; /* the chain's first step has no [D; R~] */
  const bool lone = j + 1 == L;
  T a[TILES][2 * NK], re[2 * NK];
  SmKept<NK, T> kept;
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int c = 16 * i + li;
    const bool isP = c < n, isQ = c >= n && c < 2 * n, isB = c >= 2 * n && c < 3 * n;
    const int qc = isP ? c : (isQ ? c - n : c - 2 * n);
    const T* p0 = isP ? in.D + sj * nn + (DV == 1 ? 0 : qc * n) : in.B + sj * nn + qc * n;
    const T* p1 = (isP ? fac.R : fac.Y) + e * nn + qc * n; /* R~_j, X_j (zero for a lone step) */
    mid_load<NK, true>(a[i], p0, isP || (isB && DV == 0), n, lk);
    mid_load<NK, true>(a[i] + NK, p1, isP || isQ, n, lk);
  }
  mid_load<NK, true>(re, in.c + sj * n, true, n, lk);
  mid_load<NK, true>(re + NK, fac.cf + e * n, true, n, lk); /* o_j */
  if (DV == 1) { /* stored as its diagonal */
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][g] = (16 * i + li >= n || 4 * g + lk == 16 * i + li) ? T(a[i][g]) : T(0);
  }
  if (DV != 0) {
    const double* F = in.wF + (in.wFidx ? in.wFidx[sj] * nn : 0);
#pragma unroll
    for (int i = 2; i < TILES; ++i) { /* Bl starts at 2 n > 32 */
      const int c = 16 * i + li;
      const bool isB = c >= 2 * n && c < 3 * n;
      T v[NK];
      mid_load_scaled<NK>(v, in.wk + sj * n, F + (c - 2 * n) * n, isB, n, -1.0, lk);
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][g] = isB ? T(v[g]) : T(a[i][g]);
    }
  }
  constexpr int QF = QF_TRI1 | (DV == 1 ? QF_DIAG0 : 0); /* R~_j is upper triangular */
  sm_qr<NK, TILES, QF, T>(a, re, kept, n, li, lk);
  mid_store_triu<NK>(fac.R + e * nn, a, kept, n, li, lk);
  T* const Z = lone ? fix + (int64_t)p * (nn + n) : out.B + t * nn;
#pragma unroll
  for (int i = 1; i < TILES; ++i) {
    const int c = 16 * i + li;
    const bool isQ = c >= n && c < 2 * n, isB = c >= 2 * n && c < 3 * n;
    const int64_t qc = isQ ? c - n : c - 2 * n;
    mid_store<NK, true>((isQ ? fac.Y : fac.Bt) + e * nn + qc * n, a[i], isQ || isB, n, lk);
    mid_store<NK, true>((isQ ? out.D + t * nn : Z) + qc * n, a[i] + NK, isB || (isQ && !lone), n, lk); /* X~_j, Z_j */
  }
  mid_store<NK, true>(fac.cf + e * n, a[1], li == 0, n, lk);
  mid_store<NK, true>(lone ? Z + nn : out.c + t * n, a[1] + NK, li == 0, n, lk); /* o_j */
}

template <int NK, class T, int LV>
__global__ void __launch_bounds__(64 * MID_WAVES, (mid_occ(NK, 3, sizeof(T) == 4)))
    k_mid3(uk_level_t lv, ChainT<T> in, ChainT<T> out, const T* __restrict__ fix, int n) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int64_t unit = (int64_t)blockIdx.x * MID_WAVES + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (unit >= lv.units) return; /* whole waves; no barrier below */
  const int p = (int)find_problem(lv.unit_start, lv.nprob, unit);
  const int64_t u0 = lv.unit_start[p], L = lv.L[p], s0 = lv.step_start[p], t0 = lv.next_start[p];
  if (L == 1) return;
  const int64_t u = unit - u0, t = t0 + u, sp = s0 + 2 * u + 1, nn = (int64_t)n * n;
  const int mr = LV == 2 ? n : in.mr;
  const bool c_synth = LV != 2 && sizeof(T) == 4 && in.c_synth;
  T a[2][2 * NK], re[2 * NK];
  SmKept<NK, T> kept;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = 16 * i + li;
    mid_load<NK, LV == 2>(a[i], out.C + t * nn + (int64_t)c * mr, c < n, mr, lk); /* D~_{j+1} */
    mid_load<NK, LV == 2>(a[i] + NK, in.C + sp * nn + (int64_t)c * mr, c < n && !c_synth, mr, lk);
  }
  mid_load<NK, LV == 2>(re, out.o + t * n, true, mr, lk); /* c~_{j+1} */
  mid_load<NK, LV == 2>(re + NK, in.o + sp * n, true, mr, lk);
  if (c_synth) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = 16 * i + li;
      mid_load_scaled<NK>(a[i] + NK, in.rC + sp * mr, in.rG + sp * (int64_t)mr * n + c * mr, c < n, min(mr, in.rm[sp]), 1.0, lk);
    }
  }
  constexpr int QF = (LV == 1 ? QF_HALF0 | QF_HALF1 : 0) | (LV == 2 ? QF_TRI1 : 0);
  sm_qr<NK, 2, QF, T>(a, re, kept, n, li, lk);
  if ((L & 1) && u == L / 2 - 1) { /* [G~; Z] and [c; o_Z], Z and o_Z from the lone step's scratch */
    const T* fz = fix + (int64_t)p * (nn + n);
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      re[g] = a[1][g]; /* the right-hand side, in lanes li = 0 */
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i][g] = mid_pivot<NK>(a, kept, i, g, li, lk);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) mid_load<NK, true>(a[i] + NK, fz + (16 * i + li) * n, 16 * i + li < n, n, lk);
    mid_load<NK, true>(re + NK, fz + nn, true, n, lk);
    sm_qr<NK, 2, 0, T>(a, re, kept, n, li, lk);
  }
  mid_store_triu<NK>(out.C + t * nn, a, kept, n, li, lk); /* G~ */
  mid_store<NK, true>(out.o + t * n, a[1], li == 0, n, lk);
}

/*
 * The three phases of one level in one launch, for levels with few pairs (above
 * level 0: C upper triangular, B and D stored in full): a workgroup per pair,
 * whose waves share its columns. A lone wave's steps wait for the fetching of
 * their own code as much as for their operands (phase 2 at n = 32: 37 KB, 32 us
 * on an idle chip, about half of it instruction fetch), so each wave takes the
 * two pivot tiles and one more: 3 tiles instead of 6, half the code.
 *   waves 0 .. W2 - 1: phase 1, then phase 2, on tiles 0, 1 and 2 + wave (the
 *     tiles of phase 2; wave 0 owns what tiles 0 and 1 hold besides pivots);
 *   wave W2: phase 3, on D~ and c~ handed over in LDS after phase 1;
 *   waves W2 + 1 ..: an odd chain's last step, as waves 0 .. W2 - 1 do a pair's
 *     even step; its Z and o_Z go through LDS into phase 3's fold.
 * Level of 100 pairs, n = 32, FP64: 78 us in three launches.
 */
template <int NK>
struct MidLevel {
  static constexpr int W2 = (3 * NK + 3) / 4 - 2, WAVES = 2 * W2 + 1;
};

template <int NK, class T>
__global__ void __launch_bounds__(64 * MidLevel<NK>::WAVES)
    k_mid_level(uk_level_t lv, ChainT<T> in, ChainT<T> out, FactorsT<T> fac, int n) {
  constexpr int W2 = MidLevel<NK>::W2;
  __shared__ T sD[2][NK][64], sZ[2][NK][64]; /* D~, Z as tiles: [tile][granule][lane] */
  __shared__ T sc[NK][4], so[NK][4];         /* c~, o_Z: [granule][lk] */
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t item = blockIdx.x;
  const int p = (int)find_problem(lv.unit_start, lv.nprob, item);
  const int64_t u0 = lv.unit_start[p], e0 = lv.even_start[p], L = lv.L[p], s0 = lv.step_start[p], t0 = lv.next_start[p];
  const int64_t u = item - u0, t = t0 + u, nn = (int64_t)n * n;
  const bool single = L == 1, has_lone = !single && (L & 1) && u == L / 2 - 1;
  if (wave >= W2 && (single || (wave > W2 && !has_lone))) return; /* ended waves take no part in the barriers */
  SmKept<NK, T> kept;
  T re[2 * NK];

  if (wave == W2) { /* phase 3 */
    const int64_t sp = s0 + 2 * u + 1;
    T a[2][2 * NK];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      mid_load<NK, true>(a[i] + NK, in.C + sp * nn + (int64_t)(16 * i + li) * n, 16 * i + li < n, n, lk);
    mid_load<NK, true>(re + NK, in.o + sp * n, true, n, lk);
    __syncthreads(); /* D~ and c~ are in LDS */
#pragma unroll
    for (int g = 0; g < NK; ++g) {
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i][g] = 16 * i + li < n ? T(sD[i][g][lane]) : T(0);
      re[g] = sc[g][lk];
    }
    sm_qr<NK, 2, QF_TRI1, T>(a, re, kept, n, li, lk);
    if (has_lone) {
      __syncthreads(); /* Z and o_Z are in LDS */
#pragma unroll
      for (int g = 0; g < NK; ++g) {
        re[g] = a[1][g]; /* the right-hand side, in lanes li = 0 */
        re[NK + g] = so[g][lk];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a[i][g] = mid_pivot<NK>(a, kept, i, g, li, lk);
          a[i][NK + g] = 16 * i + li < n ? T(sZ[i][g][lane]) : T(0);
        }
      }
      sm_qr<NK, 2, 0, T>(a, re, kept, n, li, lk);
    }
    mid_store_triu<NK>(out.C + t * nn, a, kept, n, li, lk);
    mid_store<NK, true>(out.o + t * n, a[1], li == 0, n, lk);
    return;
  }

  const bool lone = wave > W2 || single; /* no right neighbour */
  const int w = wave > W2 ? wave - W2 - 1 : wave;
  const int64_t j = wave > W2 ? L - 1 : 2 * u, sj = s0 + j, sp = lone ? sj : sj + 1, e = e0 + (j >> 1);
  T a[3][2 * NK];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int c = 16 * (i < 2 ? i : 2 + w) + li;
    const bool isP = c < n, isQ = c >= n && c < 2 * n;
    mid_load<NK, true>(a[i], isP ? in.B + sp * nn + c * n : in.D + sp * nn + (int64_t)(c - n) * n, !lone && (isP || isQ), n, lk);
    mid_load<NK, true>(a[i] + NK, in.C + sj * nn + c * n, isP, n, lk);
  }
  mid_load<NK, true>(re, in.c + sp * n, !lone, n, lk);
  mid_load<NK, true>(re + NK, in.o + sj * n, true, n, lk);
  sm_qr<NK, 3, QF_TRI1, T>(a, re, kept, n, li, lk);

  if (!single) {
    if (wave < W2) { /* D~_{j+1}, c~_{j+1} to phase 3 */
#pragma unroll
      for (int i = 1; i < 3; ++i) {
        const int q = 16 * (i < 2 ? 1 : 2 + w) + li - n; /* column of D~ */
        if (q >= 0 && q < n && (i == 2 || w == 0)) {
#pragma unroll
          for (int g = 0; g < NK; ++g) sD[q >> 4][g][lk * 16 + (q & 15)] = a[i][NK + g];
        }
      }
      if (w == 0 && li == 0) {
#pragma unroll
        for (int g = 0; g < NK; ++g) sc[g][lk] = a[1][NK + g];
      }
    }
    __syncthreads();
  }

  if (j > 0) { /* phase 2: block 1 <- [R~_j | X_j | 0], block 0 <- [D_j | 0 | B_j] */
#pragma unroll
    for (int g = 0; g < NK; ++g) re[NK + g] = a[1][g]; /* o_j, in lanes li = 0 */
    T rt[2][NK];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < NK; ++g) rt[i][g] = 16 * i + li < n ? mid_pivot<NK>(a, kept, i, g, li, lk) : T(a[i][g]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int c = 16 * (i < 2 ? i : 2 + w) + li;
      const bool isP = c < n, isB = c >= 2 * n && c < 3 * n;
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][NK + g] = i < 2 ? T(rt[i < 2 ? i : 0][g]) : (isB ? T(0) : T(a[i][g]));
      mid_load<NK, true>(a[i], isP ? in.D + sj * nn + c * n : in.B + sj * nn + (int64_t)(c - 2 * n) * n, isP || isB, n, lk);
    }
    mid_load<NK, true>(re, in.c + sj * n, true, n, lk);
    sm_qr<NK, 3, QF_TRI1, T>(a, re, kept, n, li, lk);
  }
  if (w == 0) {
    mid_store_triu<NK>(fac.R + e * nn, a, kept, n, li, lk);
    mid_store<NK, true>(fac.cf + e * n, a[1], li == 0, n, lk);
    if (wave > W2) {
      if (li == 0) {
#pragma unroll
        for (int g = 0; g < NK; ++g) so[g][lk] = a[1][NK + g]; /* o_Z */
      }
    } else if (j > 0 && !lone) {
      mid_store<NK, true>(out.c + t * n, a[1] + NK, li == 0, n, lk);
    }
  }
#pragma unroll
  for (int i = 1; i < 3; ++i) {
    const int c = 16 * (i < 2 ? 1 : 2 + w) + li;
    const bool mine = i == 2 || w == 0, isQ = mine && c >= n && c < 2 * n, isB = mine && c >= 2 * n && c < 3 * n;
    const int64_t qc = isQ ? c - n : c - 2 * n;
    if (j == 0 && isB) {
#pragma unroll
      for (int g = 0; g < NK; ++g) a[i][g] = T(0); /* the chain's first step: no B~ */
    }
    mid_store<NK, true>((isQ ? fac.Y : fac.Bt) + e * nn + qc * n, a[i], isQ || isB, n, lk);
    if (j > 0 && wave < W2) mid_store<NK, true>((isQ ? out.D : out.B) + t * nn + qc * n, a[i] + NK, !lone && (isQ || isB), n, lk);
    if (wave > W2 && isB) { /* Z */
#pragma unroll
      for (int g = 0; g < NK; ++g) sZ[qc >> 4][g][lk * 16 + (qc & 15)] = a[i][NK + g];
    }
  }
  if (has_lone) __syncthreads();
}

/* Levels of at most this many pairs take k_mid_level: two workgroups per CU.
 * Smoothing n = 32 without covariances, never / up to this line / always: k =
 * 500 679 / 501 / 499 us, k = 4000 1011 / 768 / 804, k = 16000 1804 / 1557 / 1962
 * (FP32 elimination 1529 / 1290 / 1686); n = 24: k = 500 375 / 290 / 290, k =
 * 16000 959 / 836 / 938. */
constexpr int64_t MID_SPLIT = 512;

template <class T>
bool mid_one_launch(const uk_level_t* lv, const ChainT<T>& in) {
  return in.c_tri && !in.b_synth && !in.d_diag && lv->units <= MID_SPLIT;
}
/* phase 0: the whole level (where mid_one_launch says so), else phase 1 .. 3 */
template <int NK, class T>
bool mid_launch(const uk_level_t* lv, const ChainT<T>& in, const ChainT<T>& out, const FactorsT<T>& fac, T* fix, int n,
                hipStream_t st, int phase) {
  const int lvk = in.c_tri && !in.b_synth && !in.d_diag ? 2 : (in.mr <= sm_half_rows(NK) ? 1 : 0);
  const dim3 b(64 * MID_WAVES), g((unsigned)((lv->evens + MID_WAVES - 1) / MID_WAVES)),
      g3((unsigned)((lv->units + MID_WAVES - 1) / MID_WAVES));
  if (phase == 0) {
    if (!mid_one_launch(lv, in)) return false;
    k_mid_level<NK, T><<<dim3((unsigned)lv->units), dim3(64 * MidLevel<NK>::WAVES), 0, st>>>(*lv, in, out, fac, n);
  } else if (phase == 1) {
    if (lvk == 2) k_mid1<NK, T, 2><<<g, b, 0, st>>>(*lv, in, out, fac, n);
    else if (lvk == 1) k_mid1<NK, T, 1><<<g, b, 0, st>>>(*lv, in, out, fac, n);
    else k_mid1<NK, T, 0><<<g, b, 0, st>>>(*lv, in, out, fac, n);
  } else if (phase == 2) {
    if (in.d_diag && in.b_synth) k_mid2<NK, T, 1><<<g, b, 0, st>>>(*lv, in, out, fac, fix, n);
    else if (in.b_synth) k_mid2<NK, T, 2><<<g, b, 0, st>>>(*lv, in, out, fac, fix, n);
    else k_mid2<NK, T, 0><<<g, b, 0, st>>>(*lv, in, out, fac, fix, n);
  } else {
    if (lvk == 2) k_mid3<NK, T, 2><<<g3, b, 0, st>>>(*lv, in, out, fix, n);
    else if (lvk == 1) k_mid3<NK, T, 1><<<g3, b, 0, st>>>(*lv, in, out, fix, n);
    else k_mid3<NK, T, 0><<<g3, b, 0, st>>>(*lv, in, out, fix, n);
  }
  return true;
}
}  // namespace

/* The launchers of NK = NKV, for its translation unit. */
#define UKMID_DEFINE(NKV)                                                                                            \
  bool ukqr::mid_phase_##NKV(const uk_level_t* lv, const ChainT<double>& in, const ChainT<double>& out,               \
                             const FactorsT<double>& fac, double* fix, int n, hipStream_t st, int phase) {            \
    return mid_launch<NKV, double>(lv, in, out, fac, fix, n, st, phase);                                              \
  }                                                                                                                   \
  bool ukqr::mid_phase_##NKV(const uk_level_t* lv, const ChainT<float>& in, const ChainT<float>& out,                 \
                             const FactorsT<float>& fac, float* fix, int n, hipStream_t st, int phase) {              \
    return mid_launch<NKV, float>(lv, in, out, fac, fix, n, st, phase);                                               \
  }

#endif /* UKHIP_ODDEVEN_MID_H */
