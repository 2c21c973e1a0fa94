/*
 * filter_small.hip -- one step (evolve + observe) of every filter of a batch
 * of sequential UltimateKalman filters with n <= 16, one wave per filter
 * (c/kalman_ultimate.c:140-470); the same step as k_filter_step (oddeven.hip),
 * on the layout and the Householder steps of oddeven_wave.h:
 *   evolve:  QR of [R_{i-1}; -V F_i] (tile 0) applied to [0; V H_i] (tile 1) and
 *            [y_{i-1}; V c_i]; tile 1's lower block and the right-hand side's
 *            are the prediction (R~, y~), already in place for
 *   observe: QR of [R~; W G_i] applied to [y~; W o_i] -> (R_i, y_i);
 *   x_i = R_i^{-1} y_i by substitution in the same registers.
 * R_{i-1} is upper triangular, so a reflector reaches the upper block at its
 * pivot row alone (QF_DIAG0). Every load is issued before the first QR.
 */
#include <hip/hip_runtime.h>

#include "oddeven_wave.h"

namespace {

constexpr int FS_WAVES = 4; /* filters (waves) per workgroup */

/* x = R^{-1} y: R an upper triangular tile (identity beyond n), y the same on
 * every li; column by column, the solved entry uniform */
template <int NK, int... Q>
__device__ __forceinline__ void fs_solve(const double (&R)[NK], double (&y)[NK], double rinv,
                                         std::integer_sequence<int, Q...>) {
  auto one = [&](auto qq) {
    constexpr int q = 4 * NK - 1 - qq.value, G = q / 4;
    const double xq = one_lane(y[G] * rinv, 16 * (q % 4) + q); /* lane li = q, lk = q % 4 holds row q and 1 / R_qq */
#pragma unroll
    for (int g = 0; g <= G; ++g) y[g] = fma(-row_lane<q>(R[g]), xq, y[g]); /* rows above q; row q is set below */
    const int lk = (int)(threadIdx.x & 63) >> 4;
    y[G] = lk == q % 4 ? xq : y[G];
  };
  (one(std::integral_constant<int, Q>{}), ...);
}

/* HALF: at most sm_half_rows(NK) observation rows */
template <int NK, bool HALF>
__global__ void __launch_bounds__(64 * FS_WAVES) k_filter_small(uk_filter_t st, uk_filter_in_t in, int nf, int n, int first) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int64_t f = (int64_t)blockIdx.x * FS_WAVES + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (f >= nf) return; /* whole waves; no barrier below */
  const int64_t nn = (int64_t)n * n;
  const int mr = in.mr;
  const int mi = in.m_i ? in.m_i[f] : mr;
  const int m = mi < 0 ? 0 : (mi > mr ? mr : mi); /* device-resident counts are not checked on the host */
  const int zprev = first ? 0 : st.z[f];
  const double* kw = in.K + f * n;
  double w[2][2 * NK], e[2 * NK], t[1][2 * NK], et[2 * NK];
  SmKept<NK, double> kept;
  /* observation block and right-hand side: rows m .. are zero */
  if (in.pre) {
    sm_load<NK>(t[0] + NK, in.wC + f * nn, mr, m, n, li, lk); /* W G, ld mr in an n*n slot */
    sm_load_vec<NK>(et + NK, in.wo + f * n, m, lk);           /* W o */
  } else {
    sm_load_scaled<NK>(t[0] + NK, in.C + f * mr, in.G + f * (int64_t)mr * n, mr, m, n, 1.0, li, lk);
    double cw[NK];
    sm_load_vec<NK>(cw, in.C + f * mr, m, lk);
    sm_load_vec<NK>(et + NK, in.o + f * mr, m, lk);
#pragma unroll
    for (int g = 0; g < NK; ++g) et[NK + g] *= cw[g];
  }
  if (!first) {
    sm_load<NK>(w[0], st.R + f * nn, n, n, n, li, lk);
    sm_load_vec<NK>(e, st.y + f * n, n, lk);
    if (in.pre) {
      sm_load<NK>(w[0] + NK, in.wB + f * nn, n, n, n, li, lk); /* -V F */
      sm_load<NK>(w[1] + NK, in.wD + f * nn, n, n, n, li, lk); /* V H */
      sm_load_vec<NK>(e + NK, in.wc + f * n, n, lk);           /* V c */
    } else {
      double kv[NK];
      sm_load_vec<NK>(kv, kw, n, lk);
      sm_load_scaled<NK>(w[0] + NK, kw, in.F + (in.F_shared ? 0 : f * nn), n, n, n, -1.0, li, lk);
      if (in.H) sm_load_scaled<NK>(w[1] + NK, kw, in.H + f * nn, n, n, n, 1.0, li, lk);
      sm_load_vec<NK>(e + NK, in.c ? in.c + f * n : kw, in.c ? n : 0, lk);
#pragma unroll
      for (int g = 0; g < NK; ++g) {
        e[NK + g] *= kv[g];
        if (!in.H) w[1][NK + g] = 4 * g + lk == li ? kv[g] : 0.0; /* H = I */
      }
    }
#pragma unroll
    for (int g = 0; g < NK; ++g) w[1][g] = 0.0;
    sm_qr<NK, 2, QF_DIAG0, double>(w, e, kept, n, li, lk);
    if (st.hist) { /* the previous step's final rows: Rdiag, Rsupdiag, y (c/kalman_ultimate.c:140-260) */
      const int64_t hs = st.hslot * st.nf + f;
      sm_store_triu<NK>(st.hRd + hs * nn, w[0], kept.r00, n, li, lk);
      sm_store<NK>(st.hRs + hs * nn, w[1], n, n, n, li, lk);
      sm_store_vec<NK>(st.hy + hs * n, w[0], n, li, lk);
    }
#pragma unroll
    for (int g = 0; g < NK; ++g) {
      t[0][g] = w[1][NK + g];
      et[g] = w[0][NK + g]; /* in the lanes li = 0 */
    }
  } else {
#pragma unroll
    for (int g = 0; g < NK; ++g) t[0][g] = et[g] = 0.0;
  }
  sm_qr<NK, 1, HALF ? QF_HALF1 : 0, double>(t, et, kept, n, li, lk);
  sm_store_triu<NK>(st.R + f * nn, t[0], kept.r00, n, li, lk);
  sm_store_vec<NK>(st.y + f * n, t[0], n, li, lk);

  const int z = min(n, zprev + m);
  double R[NK], y[NK], diag = 1.0;
#pragma unroll
  for (int g = 0; g < NK; ++g) {
    const int r = 4 * g + lk;
    y[g] = r < n ? row_lane<0>(t[0][g]) : 0.0;
    const double v = li == 0 ? (g == 0 && lk == 0 ? kept.r00 : 0.0) : t[0][g];
    R[g] = (r < n && li < n && r <= li) ? v : (r == li ? 1.0 : 0.0);
    diag = r == li ? R[g] : diag;
  }
  fs_solve<NK>(R, y, 1.0 / diag, std::make_integer_sequence<int, 4 * NK>{});
  if (z < n) { /* the state is not yet determined */
#pragma unroll
    for (int g = 0; g < NK; ++g) y[g] = __builtin_nan("");
  }
  sm_store_vec<NK>(st.x + f * n, y, n, li, lk);
  if (lane == 0) st.z[f] = z;
}

template <int NK>
void launch_nk(const uk_filter_t* st, const uk_filter_in_t* in, int nf, int n, int first, hipStream_t s) {
  const dim3 g((unsigned)((nf + FS_WAVES - 1) / FS_WAVES)), b(64 * FS_WAVES);
  if (in->mr <= sm_half_rows(NK)) k_filter_small<NK, true><<<g, b, 0, s>>>(*st, *in, nf, n, first);
  else k_filter_small<NK, false><<<g, b, 0, s>>>(*st, *in, nf, n, first);
}
}  // namespace

/* One step of every filter, n <= 16 and at most n observation rows. */
extern "C" hipError_t uk_launch_filter_small(const uk_filter_t* st, const uk_filter_in_t* in, int nf, int n, int first,
                                             hipStream_t s) {
  if (n < 1 || n > 16 || in->mr > n) return hipErrorInvalidValue;
  switch ((n + 3) / 4) {
    case 1: launch_nk<1>(st, in, nf, n, first, s); break;
    case 2: launch_nk<2>(st, in, nf, n, first, s); break;
    case 3: launch_nk<3>(st, in, nf, n, first, s); break;
    default: launch_nk<4>(st, in, nf, n, first, s); break;
  }
  return hipGetLastError();
}
