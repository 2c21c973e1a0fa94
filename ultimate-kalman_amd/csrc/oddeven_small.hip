/*
 * oddeven_small.hip -- the odd-even elimination for n <= 16: one launch per
 * level, one wave per step pair.
 *
 * Reference: c/kalman_oddeven_smoother.c (phases :379-560, fix-last
 * :1452-1476, renaming :563-597).
 *
 * The layout and the Householder steps are those of oddeven_wave.h, with one
 * tile per block. A step pair's three phases follow one another in the
 * registers: phase 1's R~, X, D~ are never stored.
 *
 * Most levels of a smoothing have few pairs, and there the time of a level is
 * one pair's chain. Such a level splits the pair's work over three waves:
 * phases 1 and 2, phases 1 and 3 (phase 1 is done twice, which costs nothing
 * there), and phases 1 and 2 of an odd chain's last step, whose rest rows join
 * the last pair's phase 3. A level with many pairs takes one wave per pair.
 */
#include <hip/hip_runtime.h>

#include "oddeven_wave.h"

namespace {

constexpr int SM_WAVES = 4; /* pairs (waves) per workgroup where a wave does a whole pair */

/*
 * One level. Work item: the step pair (j, j + 1), j = 2 u, with an odd chain's
 * last pair also the lone step L - 1; or a one-step chain. Phases (even step j
 * with its pair; the reference's):
 *   1: QR of [B_{j+1}; C_j] applied to [D_{j+1}; 0], [c_{j+1}; o_j]: R~_j, X_j,
 *      o_j and D~_{j+1}, c~_{j+1} (a lone or single step: B, D, c absent)
 *   3: QR of [D~_{j+1}; C_{j+1}] applied to [c~_{j+1}; o_{j+1}]; then, for an odd
 *      chain's last pair, of [G~; Z] applied to [c; o_Z]: the new step's C, o
 *   2: QR of [D_j; R~_j] applied to [0; X_j], [B_j; 0], [c_j; o_j]: the factors R,
 *      Y, B~, cf and the new step's B, D, c (a lone step: Z, o_Z)
 * LV, DV: as for k_phase1..3 (LV: C's structure; DV 1: D diagonal and B formed
 * on load; LV 0 with DV 0 takes every form at run time).
 */
template <int NK, class T, int LV, int DV>
__global__ void __launch_bounds__(256)
    k_level_small(uk_level_t lv, ChainT<T> in, ChainT<T> out, FactorsT<T> fac, int n, int split) {
  __shared__ T zbuf[SM_WAVES][2 * NK][64]; /* a lone step's Z and o_Z, per item */
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t item = split ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * SM_WAVES + wave;
  if (item >= lv.units) return; /* one wave per item: no barrier below; split: one item per workgroup, all in range */
  const int p = (int)find_problem(lv.unit_start, lv.nprob, item);
  const int64_t u0 = lv.unit_start[p], e0 = lv.even_start[p], L = lv.L[p], s0 = lv.step_start[p], t0 = lv.next_start[p];
  const int64_t u = item - u0, t = t0 + u;
  const int64_t nn = (int64_t)n * n;
  const int mr = in.mr;
  const bool single = L == 1, has_lone = !single && (L & 1) && u == L / 2 - 1;
  /* this wave's part: [the lone step,] then the pair's phases 3 and 2 */
  const bool do_lone = has_lone && (!split || wave == 2), do_main = !split || wave < 2;
  const bool do3 = !single && (!split || wave == 1), do2 = !split || wave == 0;
  if (split && !has_lone && (wave == 2 || (single && wave == 1))) return; /* no barrier for this item */
  T(&z)[2 * NK][64] = zbuf[split ? 0 : wave];
  const bool c_synth = LV != 2 && sizeof(T) == 4 && in.c_synth;
  const bool b_synth = DV == 1 || (LV == 0 && DV == 0 && in.b_synth);
  const bool d_diag = DV == 1 || (LV == 0 && DV == 0 && in.d_diag);

  for (int pass = do_lone ? 0 : 1; pass < (do_main ? 2 : 1); ++pass) {
    const bool lone = pass == 0 || single; /* no right neighbour */
    const int64_t j = pass == 0 ? L - 1 : 2 * u, sj = s0 + j, sp = lone ? sj : sj + 1, e = e0 + (j >> 1);
    const int nr = lone ? 0 : n; /* rows of the blocks of step j + 1 */
    T w[3][2 * NK], re[2 * NK];
    SmKept<NK, T> kept;
    /* loads of phase 1 */
    if (b_synth) sm_load_scaled<NK>(w[0], in.wk + sp * n, in.wF + (in.wFidx ? in.wFidx[sp] * nn : 0), n, nr, n, -1.0, li, lk);
    else sm_load<NK>(w[0], in.B + sp * nn, n, nr, n, li, lk);
    if (c_synth) sm_load_scaled<NK>(w[0] + NK, in.rC + sj * mr, in.rG + sj * (int64_t)mr * n, mr, min(mr, in.rm[sj]), n, 1.0, li, lk);
    else sm_load<NK>(w[0] + NK, in.C + sj * nn, mr, mr, n, li, lk);
    if (d_diag) {
      sm_load_vec<NK>(w[1], in.D + sp * nn, nr, lk);
#pragma unroll
      for (int g = 0; g < NK; ++g) w[1][g] = 4 * g + lk == li ? T(w[1][g]) : T(0);
    } else {
      sm_load<NK>(w[1], in.D + sp * nn, n, nr, n, li, lk);
    }
    sm_load_vec<NK>(re, in.c + sp * n, nr, lk);
    sm_load_vec<NK>(re + NK, in.o + sj * n, mr, lk);
#pragma unroll
    for (int g = 0; g < NK; ++g) w[1][NK + g] = T(0);
    /* and of the phase after it, in flight meanwhile: C_{j+1}, o_{j+1}; D_j, B_j, c_j */
    T c3[NK], o3[NK], d2[NK], b2[NK], v2[NK];
    const bool f3 = do3 && pass == 1, f2 = j > 0 && (do2 || pass == 0);
    if (f3) {
      if (c_synth) sm_load_scaled<NK>(c3, in.rC + sp * mr, in.rG + sp * (int64_t)mr * n, mr, min(mr, in.rm[sp]), n, 1.0, li, lk);
      else sm_load<NK>(c3, in.C + sp * nn, mr, mr, n, li, lk);
      sm_load_vec<NK>(o3, in.o + sp * n, mr, lk);
    }
    if (f2) {
      if (d_diag) {
        sm_load_vec<NK>(d2, in.D + sj * nn, n, lk);
#pragma unroll
        for (int g = 0; g < NK; ++g) d2[g] = 4 * g + lk == li ? T(d2[g]) : T(0);
      } else {
        sm_load<NK>(d2, in.D + sj * nn, n, n, n, li, lk);
      }
      if (b_synth) sm_load_scaled<NK>(b2, in.wk + sj * n, in.wF + (in.wFidx ? in.wFidx[sj] * nn : 0), n, n, n, -1.0, li, lk);
      else sm_load<NK>(b2, in.B + sj * nn, n, n, n, li, lk);
      sm_load_vec<NK>(v2, in.c + sj * n, n, lk);
    }

    /* phase 1 on tiles P, Q */
    constexpr int QF1 = (LV == 1 ? QF_HALF1 : 0) | (LV == 2 ? QF_TRI1 : 0);
    sm_qr<NK, 2, QF1, T>(reinterpret_cast<T(&)[2][2 * NK]>(w), re, kept, n, li, lk);

    /* phase 3 on D~ (the pivots) over C_{j+1}; the fold of a lone step's Z */
    if (f3) {
      T g3[1][2 * NK], e3[2 * NK];
      SmKept<NK, T> kept3;
#pragma unroll
      for (int g = 0; g < NK; ++g) {
        g3[0][g] = w[1][NK + g];
        g3[0][NK + g] = c3[g];
        e3[g] = w[0][NK + g]; /* c~, in the lanes li = 0 */
        e3[NK + g] = o3[g];
      }
      constexpr int QF3 = (LV == 1 ? QF_HALF0 | QF_HALF1 : 0) | (LV == 2 ? QF_TRI1 : 0);
      sm_qr<NK, 1, QF3, T>(g3, e3, kept3, n, li, lk);
      if (has_lone) {
        if (split) __syncthreads(); /* every wave of the item: Z is in LDS */
        else wave_lds_sync();
#pragma unroll
        for (int g = 0; g < NK; ++g) {
          e3[g] = g3[0][g];
          e3[NK + g] = z[NK + g][lane];
          g3[0][g] = li == 0 ? (g == 0 && lk == 0 ? T(kept3.r00) : T(0)) : (4 * g + lk <= li ? T(g3[0][g]) : T(0));
          g3[0][NK + g] = z[g][lane];
        }
        sm_qr<NK, 1, 0, T>(g3, e3, kept3, n, li, lk);
      }
      sm_store_triu<NK>(out.C + t * nn, g3[0], kept3.r00, n, li, lk);
      sm_store_vec<NK>(out.o + t * n, g3[0], n, li, lk);
    }

    /* phase 2 on tiles P (the pivots [D_j; R~_j]), Q ([0; X_j]), Bl ([B_j; 0]) */
    if (f2) {
#pragma unroll
      for (int g = 0; g < NK; ++g) {
        const T rt = li == 0 ? (g == 0 && lk == 0 ? T(kept.r00) : T(0)) : (4 * g + lk <= li ? T(w[0][g]) : T(0));
        re[NK + g] = w[0][g]; /* o_j, in the lanes li = 0 */
        re[g] = v2[g];
        w[0][NK + g] = rt;
        w[0][g] = d2[g];
        w[1][NK + g] = w[1][g];
        w[1][g] = T(0);
        w[2][g] = b2[g];
        w[2][NK + g] = T(0);
      }
      constexpr int QF2 = QF_TRI1 | (DV == 1 ? QF_DIAG0 : 0);
      sm_qr<NK, 3, QF2, T>(w, re, kept, n, li, lk);
      if (pass == 0) {
#pragma unroll
        for (int g = 0; g < NK; ++g) {
          z[g][lane] = w[2][NK + g];      /* Z */
          z[NK + g][lane] = w[0][NK + g]; /* o_Z, in the lanes li = 0 */
        }
      } else if (!lone) {
        sm_store<NK>(out.B + t * nn, w[2] + NK, n, n, n, li, lk);
        sm_store<NK>(out.D + t * nn, w[1] + NK, n, n, n, li, lk);
        sm_store_vec<NK>(out.c + t * n, w[0] + NK, n, li, lk);
      }
    }
    if (do2 || pass == 0) {
      if (!f2) { /* the chain's first step: no B~ */
#pragma unroll
        for (int g = 0; g < NK; ++g) w[2][g] = T(0);
      }
      sm_store_triu<NK>(fac.R + e * nn, w[0], kept.r00, n, li, lk);
      sm_store<NK>(fac.Bt + e * nn, w[2], n, n, n, li, lk);
      sm_store<NK>(fac.Y + e * nn, w[1], n, n, n, li, lk);
      sm_store_vec<NK>(fac.cf + e * n, w[0], n, li, lk);
    }
  }
  if (split && has_lone && wave != 1) __syncthreads(); /* wave 1 waits for it in phase 3 */
}

/* A level of at most this many pairs gives each pair three waves: beyond, the
 * pairs alone give every SIMD of the chip (1,024) a wave. Smoothing n = 16
 * without covariances, never / up to this line / always three waves: k = 500
 * 226 / 155 / 155 us, k = 4000 324 / 260 / 270, k = 16000 485 / 421 / 495 (FP32
 * elimination 469 / 399 / 453). */
constexpr int64_t SM_SPLIT = 1024;

template <int NK, class T>
void launch_nk(const uk_level_t* lv, const ChainT<T>& in, const ChainT<T>& out, const FactorsT<T>& fac, int n,
               hipStream_t st) {
  const int split = lv->units <= SM_SPLIT;
  const dim3 g((unsigned)(split ? lv->units : (lv->units + SM_WAVES - 1) / SM_WAVES)), b(split ? 192 : 64 * SM_WAVES);
  if (in.c_tri && !in.b_synth && !in.d_diag) k_level_small<NK, T, 2, 0><<<g, b, 0, st>>>(*lv, in, out, fac, n, split);
  else if (in.mr <= sm_half_rows(NK) && in.b_synth && in.d_diag)
    k_level_small<NK, T, 1, 1><<<g, b, 0, st>>>(*lv, in, out, fac, n, split);
  else if (in.b_synth && in.d_diag) k_level_small<NK, T, 0, 1><<<g, b, 0, st>>>(*lv, in, out, fac, n, split);
  else k_level_small<NK, T, 0, 0><<<g, b, 0, st>>>(*lv, in, out, fac, n, split);
}
template <class T>
void launch(const uk_level_t* lv, const ChainT<T>& in, const ChainT<T>& out, const FactorsT<T>& fac, int n,
            hipStream_t st) {
  switch ((n + 3) / 4) {
    case 1: launch_nk<1, T>(lv, in, out, fac, n, st); break;
    case 2: launch_nk<2, T>(lv, in, out, fac, n, st); break;
    case 3: launch_nk<3, T>(lv, in, out, fac, n, st); break;
    default: launch_nk<4, T>(lv, in, out, fac, n, st); break;
  }
}
}  // namespace

void ukqr::level_small(const uk_level_t* lv, const ChainT<double>& in, const ChainT<double>& out,
                       const FactorsT<double>& fac, int n, hipStream_t st) {
  launch<double>(lv, in, out, fac, n, st);
}
void ukqr::level_small(const uk_level_t* lv, const ChainT<float>& in, const ChainT<float>& out,
                       const FactorsT<float>& fac, int n, hipStream_t st) {
  launch<float>(lv, in, out, fac, n, st);
}
