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
#ifndef UK_MID_D2
#define UK_MID_D2 2
#endif
__host__ __device__ constexpr int mid_occ(int NK, int phase, bool fp32) {
  if (phase == 2) return fp32 ? (NK <= 6 ? 4 : 3) : (NK <= 6 ? 2 : UK_MID_D2);
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
/* the pivot tiles after sm_qr as an upper triangle (ld n) */
template <int NK, class T>
__device__ __forceinline__ void mid_store_triu(T* __restrict__ dst, const T (*a)[2 * NK], const SmKept<NK, T>& kept,
                                               int n, int li, int lk) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = 16 * t + li;
    T x[NK];
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      const T own = li != 0 ? T(a[t][g]) : t == 0 ? (g == 0 ? T(kept.r00) : T(0)) : (g < 5 ? T(kept.c16[g < 5 ? g : 0]) : T(0));
      x[g] = 4 * g + lk <= c ? T(own) : T(0);
    }
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
      a[0][g] = li == 0 ? (g == 0 && lk == 0 ? T(kept.r00) : T(0)) : T(a[0][g]);
      a[1][g] = li == 0 ? (g < 5 && 4 * g + lk <= 16 ? T(kept.c16[g < 5 ? g : 0]) : T(0)) : T(a[1][g]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) mid_load<NK, true>(a[i] + NK, fz + (16 * i + li) * n, 16 * i + li < n, n, lk);
    mid_load<NK, true>(re + NK, fz + nn, true, n, lk);
    sm_qr<NK, 2, 0, T>(a, re, kept, n, li, lk);
  }
  mid_store_triu<NK>(out.C + t * nn, a, kept, n, li, lk); /* G~ */
  mid_store<NK, true>(out.o + t * n, a[1], li == 0, n, lk);
}

template <int NK, class T>
void mid_launch(const uk_level_t* lv, const ChainT<T>& in, const ChainT<T>& out, const FactorsT<T>& fac, T* fix, int n,
                hipStream_t st, int phase) {
  const int lvk = in.c_tri && !in.b_synth && !in.d_diag ? 2 : (in.mr <= sm_half_rows(NK) ? 1 : 0);
  const dim3 b(64 * MID_WAVES), g((unsigned)((lv->evens + MID_WAVES - 1) / MID_WAVES)),
      g3((unsigned)((lv->units + MID_WAVES - 1) / MID_WAVES));
  if (phase == 1) {
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
}
}  // namespace

/* The launchers of NK = NKV, for its translation unit. */
#define UKMID_DEFINE(NKV)                                                                                            \
  void ukqr::mid_phase_##NKV(const uk_level_t* lv, const ChainT<double>& in, const ChainT<double>& out,               \
                             const FactorsT<double>& fac, double* fix, int n, hipStream_t st, int phase) {            \
    mid_launch<NKV, double>(lv, in, out, fac, fix, n, st, phase);                                                     \
  }                                                                                                                   \
  void ukqr::mid_phase_##NKV(const uk_level_t* lv, const ChainT<float>& in, const ChainT<float>& out,                 \
                             const FactorsT<float>& fac, float* fix, int n, hipStream_t st, int phase) {              \
    mid_launch<NKV, float>(lv, in, out, fac, fix, n, st, phase);                                                      \
  }

#endif /* UKHIP_ODDEVEN_MID_H */
