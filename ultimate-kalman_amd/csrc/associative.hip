/*
 * associative.hip -- gfx950 kernels of the associative-scan smoother
 * (Saerkkae and Garcia-Fernandez), reference c/kalman_associative_smoother.c:
 * filtering elements :309-505, smoothing elements :697-753, combines
 * :889-1016, driver :1199-1240; matlab/KalmanAssociativeSmoother.m:20-262.
 *
 * Pipeline over a batch (all problems of one state dimension at once):
 *   k_weigh (shared with odd-even) -> whitened B = -V F, D = V H, c, C = W G, o
 *   ka_model     per step: F = -D^{-1} B, c = D^{-1} c_w, Q = (D^T D)^{-1}
 *                (the covariance-form model with H folded in: H^{-1} F,
 *                H^{-1} c, H^{-1} K H^{-T})
 *   ka_prior     per problem: information filter over steps 0..p, p the first
 *                step whose observations can determine the state (sum of m_t
 *                over t <= p reaches n), giving the filtered (x_p, P_p); the
 *                reference needs p = 0
 *   ka_felem     filtering elements (A, b, Z, e, J) of steps p+1 .. k-1
 *                (unobserved steps: e = 0, J = 0)
 *   filtering scan: chunk reduce, Hillis-Steele rounds over chunk totals,
 *                chunk down-sweep writing every prefix in place
 *   ka_selem     smoothing elements (E, g, L); steps before p from the
 *                information form
 *   smoothing scan (same scheme, last step first) -> estimates, covariances
 *
 * Every element build and every combine runs in one workgroup (256 threads, one
 * wave for n <= 16). Its blocks live in LDS with the odd leading dimension NB +
 * 1; products run on the FP64 matrix cores straight from there. (The filtering
 * work blocks of the 64 bucket go to a per-workgroup global slice: seven 64 x
 * 65 blocks exceed the 160 KiB of LDS.)
 * Wherever a symmetric positive definite matrix M is inverted in a formula, its
 * factor takes part instead: with M = G G^T, one forward elimination turns B
 * into G^{-1} B, and every result is a product of two such blocks
 * (chol_forward). The filtering combine's (I + Z J)^{-1}, which is not
 * symmetric, takes two factors: Z = L L^T and N = I + L^T J L (its eigenvalues
 * are at least 1). Observations are used whitened (noise covariance I), which
 * is the reference's S = G K G^T + C after the congruence with the whitening W.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/kalman.h"
#include "../../include/ukhip.h"
#include "oddeven_wave.h"
#include "ukhip_internal.h"

extern "C" void uk_set_error(const char* fmt, ...);
extern "C" int uk_bucket(int n);
extern "C" void* ukhip_stream(void);

namespace {

/* threads of the kernels of bucket NB */
template <int NB>
constexpr int AT = NB <= 16 ? 64 : 256;
constexpr int LDS_BYTES = 160 * 1024; /* gfx950 LDS per workgroup */

/* ------------------------------------------------------------------------ */
/* workgroup-level dense algebra on blocks of order <= NB                    */
/* ------------------------------------------------------------------------ */

/* element (i, k) of op(A) for a column-major A with leading dimension ld */
__device__ __forceinline__ double at(const double* A, int ld, bool t, int i, int k) {
  return t ? A[k + (int64_t)i * ld] : A[i + (int64_t)k * ld];
}

typedef double as_d4 __attribute__((ext_vector_type(4)));
/* D = A B + C on 16 x 16 x 4: lane (li, lk) supplies A[li][lk] and B[lk][li];
 * element r of the accumulator is D[4 r + lk][li]. So an accumulator is the
 * next product's B as it stands, and its transpose's A. */
__device__ __forceinline__ as_d4 as_mfma(double a, double b, as_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

/* C (m x q, ld ldc) = alpha op(A) op(B) + beta C with op(A) m x kk and
 * op(B) kk x q, on the matrix cores: the waves deal the 16 x 16 tiles of C
 * between them. Indices are clamped into range (rows and columns beyond C are
 * not stored) and the terms from kk on zeroed in A and B. Every thread has
 * read its inputs before any output is written, so C may alias A or B. Ends
 * with a barrier. */
template <int NB>
__device__ void mm(double* C, int ldc, const double* A, int lda, bool tA, const double* B, int ldb, bool tB, int m,
                   int q, int kk, double alpha, double beta) {
  constexpr int TB = (NB + 15) / 16, NW = AT<NB> / 64, PER = (TB * TB + NW - 1) / NW;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4, w = threadIdx.x >> 6;
  as_d4 acc[PER];
  int ia[PER], jb[PER];
#pragma unroll
  for (int s = 0; s < PER; ++s) {
    const int t = w + s * NW, i = (t % TB) * 16 + li, j = (t / TB) * 16 + li;
    acc[s] = as_d4{0.0, 0.0, 0.0, 0.0};
    ia[s] = i < m ? i : m - 1;
    jb[s] = j < q ? j : q - 1;
  }
#pragma unroll 2
  for (int k0 = 0; k0 < kk; k0 += 4) {
    const int k = k0 + lk, kc = k < kk ? k : kk - 1;
    double av[PER], bv[PER];
#pragma unroll
    for (int s = 0; s < PER; ++s) {
      av[s] = at(A, lda, tA, ia[s], kc);
      bv[s] = at(B, ldb, tB, kc, jb[s]);
    }
#pragma unroll
    for (int s = 0; s < PER; ++s) acc[s] = as_mfma(k < kk ? av[s] : 0.0, k < kk ? bv[s] : 0.0, acc[s]);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < PER; ++s) {
    const int t = w + s * NW;
    if (t < TB * TB) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = (t % TB) * 16 + 4 * r + lk, j = (t / TB) * 16 + li;
        if (i < m && j < q) {
          double* c = &C[i + (int64_t)j * ldc];
          *c = beta == 0.0 ? alpha * acc[s][r] : fma(beta, *c, alpha * acc[s][r]);
        }
      }
    }
  }
  __syncthreads();
}

/* y (m) = alpha op(A) x + beta y, one thread per row, the k loop in groups
 * of 8 loads with two partial sums; y may alias x. */
template <int NB>
__device__ void mv(double* y, const double* A, int lda, bool tA, const double* x, int m, int kk, double alpha,
                   double beta) {
  double r0 = 0.0, r1 = 0.0;
  const int i = threadIdx.x;
  if (i < m) {
    for (int k0 = 0; k0 < kk; k0 += 8) {
      double av[8], xv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = k0 + u < kk ? k0 + u : kk - 1;
        av[u] = at(A, lda, tA, i, k);
        xv[u] = k0 + u < kk ? x[k] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 8; u += 2) {
        r0 = fma(av[u], xv[u], r0);
        r1 = fma(av[u + 1], xv[u + 1], r1);
      }
    }
  }
  const double r = r0 + r1;
  __syncthreads();
  if (i < m) y[i] = beta == 0.0 ? alpha * r : fma(beta, y[i], alpha * r);
  __syncthreads();
}

/* D = op(S) (m x q; op(S) transposed when t). Threads walk an NB x NB grid
 * (compile-time strides) so that S is read along its columns; all of a
 * thread's loads are issued before its stores. */
template <int NB>
__device__ void copy_mat(double* D, int ldd, const double* S, int lds, bool t, int m, int q) {
  constexpr int PER = (NB * NB + AT<NB> - 1) / AT<NB>;
  double v[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int idx = (int)threadIdx.x + u * AT<NB>;
    const int r = idx % NB, c = idx / NB;
    int i = t ? c : r, j = t ? r : c;
    i = i < m ? i : m - 1;
    j = j < q ? j : q - 1;
    v[u] = at(S, lds, t, i, j);
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int idx = (int)threadIdx.x + u * AT<NB>;
    const int r = idx % NB, c = idx / NB;
    const int i = t ? c : r, j = t ? r : c;
    if (idx < NB * NB && i < m && j < q) D[i + (int64_t)j * ldd] = v[u];
  }
  __syncthreads();
}

/* D = d I on the leading n x n block; the padding rows and columns
 * [n, NB) of the NB x NB block become the identity. */
template <int NB>
__device__ void set_identity(double* D, int ld, int n, double d) {
  constexpr int PER = (NB * NB + AT<NB> - 1) / AT<NB>;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int idx = (int)threadIdx.x + u * AT<NB>;
    const int i = idx % NB, j = idx / NB;
    if (idx < NB * NB) D[i + (int64_t)j * ld] = (i == j) ? (i < n ? d : 1.0) : 0.0;
  }
  __syncthreads();
}

/* y (m) = a x + y */
template <int NB>
__device__ void axpy(double* y, const double* x, int m, double a) {
  for (int i = threadIdx.x; i < m; i += AT<NB>) y[i] = fma(a, x[i], y[i]);
  __syncthreads();
}

/* y (m) = x */
template <int NB>
__device__ void copy_vec(double* y, const double* x, int m) {
  for (int i = threadIdx.x; i < m; i += AT<NB>) y[i] = x[i];
  __syncthreads();
}

/* Pivot keys: |v| with its low 7 mantissa bits replaced by (127 - row), so
 * that an unsigned 64-bit maximum picks the largest magnitude and, among
 * (near-)equal magnitudes, the first row. NaN sorts above every number. */
__device__ __forceinline__ unsigned long long pivot_key(double v, int row) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(v));
  return (b & ~127ull) | (unsigned long long)(127 - row);
}
__device__ __forceinline__ int pivot_row(unsigned long long key) { return 127 - (int)(key & 127ull); }

/* Workgroup scratch of gj_inverse: pivot keys, pivot rows, column order. */
template <int NB>
struct GJScratch {
  unsigned long long key[NB + 1];
  int piv[NB];
  int col[NB];
};

/*
 * Inverse of the leading n x n block of A (ld) by Gauss-Jordan elimination
 * with partial pivoting (row interchanges, undone on the columns at the
 * end). Each step maps the whole matrix from one buffer into the other
 * (A <-> W, both ld) in one pass:
 *   new row k  = (row p, with 1 in column k) / a_pk,
 *   new row r  = (row r', with 0 in column k) - a_r'k * new row k,
 * r' being row r after the interchange of rows k and p. The pivot of the
 * next column is found in the same pass with LDS atomic maxima over the
 * candidates' keys, so a step costs one barrier. Returns the buffer (A or
 * W) holding the inverse; the other one is free. n <= NB <= 127.
 */
template <int NB>
__device__ double* gj_inverse(double* A, double* W, int ld, int n, GJScratch<NB>& g) {
  for (int i = threadIdx.x; i <= NB; i += AT<NB>) g.key[i] = 0ull;
  __syncthreads();
  for (int r = threadIdx.x; r < n; r += AT<NB>) atomicMax(&g.key[0], pivot_key(A[r], r));
  __syncthreads();
  double* cur = A;
  double* nxt = W;
  constexpr int PER = (NB * NB + AT<NB> - 1) / AT<NB>;
  for (int k = 0; k < n; ++k) {
    const int p = pivot_row(g.key[k]);
    if (threadIdx.x == 0) g.piv[k] = p;
    const double rp = 1.0 / cur[p + k * ld];
    double pj[PER], fk[PER], aj[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) { /* all loads first, indices clamped into the block */
      const int idx = (int)threadIdx.x + u * AT<NB>;
      const int r = idx < NB * NB ? idx % NB : 0, j = idx < NB * NB ? idx / NB : 0;
      const int sr = (r == p) ? k : (r == k ? p : r);
      pj[u] = cur[p + j * ld];
      fk[u] = cur[sr + k * ld];
      aj[u] = cur[sr + j * ld];
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int idx = (int)threadIdx.x + u * AT<NB>;
      const int r = idx % NB, j = idx / NB;
      if (idx < NB * NB && r < n && j < n) {
        const double rowk = (j == k ? 1.0 : pj[u]) * rp;
        const double v = r == k ? rowk : fma(-fk[u], rowk, j == k ? 0.0 : aj[u]);
        nxt[r + j * ld] = v;
        if (j == k + 1 && r > k) atomicMax(&g.key[k + 1], pivot_key(v, r));
      }
    }
    __syncthreads();
    double* t = cur;
    cur = nxt;
    nxt = t;
  }
  /* undo the interchanges on the columns, last first */
  if (threadIdx.x == 0) {
    for (int j = 0; j < n; ++j) g.col[j] = j;
    for (int k = n - 1; k >= 0; --k) {
      const int t = g.col[k];
      g.col[k] = g.col[g.piv[k]];
      g.col[g.piv[k]] = t;
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < NB * NB; idx += AT<NB>) {
    const int r = idx % NB, j = idx / NB;
    if (r < n && j < n) nxt[r + j * ld] = cur[r + g.col[j] * ld];
  }
  __syncthreads();
  return nxt;
}

/* X = A^{-1} for the leading n x n block of A (ld), A left unchanged (the
 * Gauss-Jordan inverse of a copy). W1 and W2 are scratch blocks; the
 * result is in one of them (returned), the other is free afterwards. */
template <int NB>
__device__ double* inverse(const double* A, double* W1, double* W2, int ld, int n, GJScratch<NB>& g) {
  copy_mat<NB>(W1, ld, A, ld, false, n, n);
  return gj_inverse<NB>(W1, W2, ld, n, g);
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

/*
 * Forward elimination with a symmetric positive definite M = G G^T (n x n, ld,
 * both triangles given): every block B[i] (n x q, ldb) and every vector (nv of
 * them at v, NB apart) becomes G^{-1} times itself. KEEP: M becomes G (lower
 * triangular, zeros above), else it is left half reduced.
 * Panels of 16: each wave factors the panel's diagonal tile in its registers
 * (the same work on every wave, instead of a barrier), takes T_r = G_pp^{-1}
 * M_pr for the block rows r below, and then 16 columns at a time of what is
 * dealt to it: T = G_pp^{-1} X_p, X_r -= T_r^T T. One barrier per panel.
 * A pivoted Gauss-Jordan inverse in LDS, one barrier per column, took this
 * place: 138 us a filtering combine at n = 48 with it.
 */
template <int NB, bool KEEP, bool FLOOR, int NBLK>
__device__ void chol_forward(double* M, int ld, int n, double* const (&B)[NBLK], int q, int ldb, double* v, int nv) {
  constexpr int TB = (NB + 15) / 16, NW = AT<NB> / 64;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tn = (n + 15) >> 4, tq = (q + 15) >> 4;
  double diag[TB];
  if (FLOOR) {
#pragma unroll
    for (int p = 0; p < TB; ++p) diag[p] = 16 * p + li < n ? fmax(2.2e-16 * M[(16 * p + li) * (ld + 1)], 1e-290) : 0.0;
    __syncthreads();
  }
#pragma unroll 1
  for (int p = 0; p < tn; ++p) {
    const int p0 = 16 * p;
    double a[4], wt[4], pr[4], pc = 1.0, fl = 0.0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int r = 4 * g + lk;
      const bool in = p0 + r < n && p0 + li < n;
      const double x = M[in ? p0 + r + (p0 + li) * ld : 0];
      a[g] = in ? x : (r == li ? 1.0 : 0.0);
      wt[g] = r == li ? 1.0 : 0.0;
      pr[g] = 1.0;
    }
    if (FLOOR) {
#pragma unroll
      for (int i = 0; i < TB; ++i) fl = p == i ? diag[i] : fl;
    }
    chol_steps<FLOOR>(a, wt, pr, pc, fl, n - p0, li, lk, std::make_integer_sequence<int, 16>{});
    const double sc = rsqrt_ulp(pc);
#pragma unroll
    for (int g = 0; g < 4; ++g) wt[g] *= sc; /* G_pp^{-T}: A operand of G_pp^{-1} */
    auto row_tile = [&](const double* X, int ldx, int cols, double (&t)[4]) { /* t = G_pp^{-1} X_p, 16 columns at X */
      double b[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int r = p0 + 4 * g + lk;
        const bool in = r < n && li < cols;
        const double x = X[in ? r + (int64_t)li * ldx : 0];
        b[g] = in ? x : 0.0;
      }
      as_d4 acc = as_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int g = 0; g < 4; ++g) acc = as_mfma(wt[g], b[g], acc);
#pragma unroll
      for (int g = 0; g < 4; ++g) t[g] = acc[g];
    };
    double tr[TB > 1 ? TB - 1 : 1][4];
#pragma unroll
    for (int i = 0; i < TB - 1; ++i)
      if (p + 1 + i < tn) row_tile(M + (p0 + 16 * (1 + i)) * ld, ld, n - (p0 + 16 * (1 + i)), tr[i]);
    const int trail = tn - 1 - p, tot = trail + NBLK * tq + (nv > 0 ? 1 : 0);
    for (int t = w; t < tot; t += NW) {
      double* X;
      int ldx, cols;
      if (t < trail) {
        X = M + (p0 + 16 * (1 + t)) * ld;
        ldx = ld;
        cols = n - (p0 + 16 * (1 + t));
      } else if (t < trail + NBLK * tq) {
        const int u = t - trail, blk = u / tq, c0 = 16 * (u - blk * tq);
        double* Bb = B[0];
#pragma unroll
        for (int i = 1; i < NBLK; ++i) Bb = blk == i ? B[i] : Bb;
        X = Bb + (int64_t)c0 * ldb;
        ldx = ldb;
        cols = q - c0;
      } else {
        X = v;
        ldx = NB;
        cols = nv;
      }
      double tc[4];
      row_tile(X, ldx, cols, tc);
      if (t >= trail && li < cols) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (p0 + 4 * g + lk < n) X[p0 + 4 * g + lk + (int64_t)li * ldx] = tc[g];
      }
#pragma unroll
      for (int i = 0; i < TB - 1; ++i) {
        const int r0 = p0 + 16 * (1 + i);
        if (r0 < n) {
          as_d4 acc;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const bool in = r0 + 4 * g + lk < n && li < cols;
            const double x = X[in ? r0 + 4 * g + lk + (int64_t)li * ldx : 0];
            acc[g] = in ? x : 0.0;
          }
#pragma unroll
          for (int g = 0; g < 4; ++g) acc = as_mfma(-tr[i][g], tc[g], acc);
#pragma unroll
          for (int g = 0; g < 4; ++g)
            if (r0 + 4 * g + lk < n && li < cols) X[r0 + 4 * g + lk + (int64_t)li * ldx] = acc[g];
        }
      }
    }
    if (KEEP) { /* G_rp = T_r^T, below the diagonal, where this panel reads nothing */
#pragma unroll
      for (int i = 0; i < TB - 1; ++i) {
        const int r = p0 + 16 * (1 + i) + li;
        if (i % NW == w && r < n) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            if (p0 + 4 * g + lk < n) M[r + (p0 + 4 * g + lk) * ld] = tr[i][g];
        }
      }
    }
    __syncthreads();
    if (KEEP && w == 0) { /* G_pp = (D^{-1/2} a)^T; no later panel reads this block */
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int k = 4 * g + lk;
        if (p0 + k < n && p0 + li < n) M[p0 + li + (p0 + k) * ld] = li >= k ? a[g] * rsqrt_ulp(pr[g]) : 0.0;
      }
    }
  }
  if (KEEP) {
    for (int idx = threadIdx.x; idx < NB * NB; idx += AT<NB>) {
      const int i = idx % NB, j = idx / NB;
      if (i < n && j < n && (i >> 4) < (j >> 4)) M[i + j * ld] = 0.0;
    }
    __syncthreads();
  }
}

/* W (ld) <- G^{-1} of M = G G^T (M is consumed); M^{-1} = W^T W */
template <int NB>
__device__ void chol_inverse_factor(double* M, double* W, int ld, int n) {
  set_identity<NB>(W, ld, n, 1.0);
  double* const B[1] = {W};
  chol_forward<NB, false, false>(M, ld, n, B, n, ld, nullptr, 0);
}

/* Per-thread registers holding an n x n global block (ld n) distributed over
 * the NB x NB grid: entry idx = threadIdx.x + u * AT<NB>. */
template <int NB>
struct RegBlk {
  static constexpr int PER = (NB * NB + AT<NB> - 1) / AT<NB>;
  double v[PER];
  __device__ void load(const double* G, int n) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int idx = (int)threadIdx.x + u * AT<NB>;
      const int i = idx % NB, j = idx / NB;
      v[u] = (idx < NB * NB && i < n && j < n) ? G[i + (int64_t)j * n] : 0.0;
    }
  }
  /* D (ld) <- the block, or its transpose; no barrier */
  __device__ void store(double* D, int ld, int n, bool t) const {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int idx = (int)threadIdx.x + u * AT<NB>;
      const int i = idx % NB, j = idx / NB;
      if (idx < NB * NB && i < n && j < n) D[t ? j + i * ld : i + j * ld] = v[u];
    }
  }
};

/* ------------------------------------------------------------------------ */
/* batch data                                                                */
/* ------------------------------------------------------------------------ */

struct AsProb {
  int64_t s0; /* first step (batch-global index) */
  int64_t k;  /* steps */
  int64_t p;  /* first step with a proper filtered distribution */
  int64_t e0; /* first filtering element (elements of steps p+1 .. k-1) */
};

/* covariance-form model and filtered distributions, one slot per step (ld n) */
struct AsModel {
  double* F;   /* n x n (unused on a problem's first step) */
  double* c;   /* n */
  double* Q;   /* n x n */
  double* xf;  /* filtered mean, steps >= p */
  double* Pf;  /* filtered covariance, steps >= p */
  double* Lam; /* filtered information matrix, steps < p */
  double* eta; /* filtered information vector, steps < p */
};

/* Element arrays (ld n): filtering (A, b, Z, e, J) or smoothing (E = A, g = b, L = Z). */
struct AsElems {
  double* A;
  double* b;
  double* Z;
  double* e;
  double* J;
};

template <int NB>
struct Ld {
  static constexpr int L = NB + 1; /* LDS leading dimension of an NB x NB block */
  static constexpr int SZ = NB * L;
};

/* ------------------------------------------------------------------------ */
/* model                                                                     */
/* ------------------------------------------------------------------------ */

template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_model(uk_chain_t wch, const int8_t* first, AsModel md, int n) {
  constexpr int L = Ld<NB>::L;
  __shared__ double B0[Ld<NB>::SZ], B1[Ld<NB>::SZ], B2[Ld<NB>::SZ];
  __shared__ GJScratch<NB> g;
  const int64_t s = blockIdx.x;
  if (first[s]) return;
  const int64_t nn = (int64_t)n * n;
  copy_mat<NB>(B0, L, wch.D + s * nn, n, false, n, n);
  double* Di = inverse<NB>(B0, B1, B2, L, n, g);                              /* D^{-1} */
  double* Bw = B0;
  copy_mat<NB>(Bw, L, wch.B + s * nn, n, false, n, n);
  mm<NB>(md.F + s * nn, n, Di, L, false, Bw, L, false, n, n, n, -1.0, 0.0);   /* F = -D^{-1} B */
  mv<NB>(md.c + s * n, Di, L, false, wch.c + s * n, n, n, 1.0, 0.0);             /* c = D^{-1} c_w */
  mm<NB>(md.Q + s * nn, n, Di, L, false, Di, L, true, n, n, n, 1.0, 0.0);     /* Q = D^{-1} D^{-T} */
}

/* The same where every H is the identity and every K given as 'w': the model is
 * the input's, Q = diag(1 / k^2). Consecutive threads, consecutive elements. */
__global__ void __launch_bounds__(256) ka_model_diag(uk_raw_t raw, AsModel md, int n) {
  const int64_t s = blockIdx.x;
  if (raw.first[s]) return;
  const int nn = n * n;
  const double* F = raw.F + raw.Fidx[s] * nn;
  for (int i = threadIdx.x; i < nn; i += 256) {
    const int c = i / n, r = i - c * n;
    const double k = raw.K[s * n + c];
    md.F[s * nn + i] = F[i];
    md.Q[s * nn + i] = r == c ? 1.0 / (k * k) : 0.0;
  }
  for (int i = threadIdx.x; i < n; i += 256) md.c[s * n + i] = raw.c[s * n + i];
}

/* ------------------------------------------------------------------------ */
/* prior: information filter over steps 0..p, one workgroup per problem      */
/* ------------------------------------------------------------------------ */

template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_prior(const AsProb* probs, uk_chain_t wch, const int32_t* m_obs, AsModel md,
                                                   int n, int mr) {
  constexpr int L = Ld<NB>::L;
  __shared__ double Lm[Ld<NB>::SZ], Mx[Ld<NB>::SZ], Qi[Ld<NB>::SZ], T2[Ld<NB>::SZ];
  __shared__ double et[NB], v1[NB], v2[NB];
  const AsProb pr = probs[blockIdx.x];
  const int64_t nn = (int64_t)n * n;
  set_identity<NB>(Lm, L, n, 0.0);
  for (int i = threadIdx.x; i < n; i += AT<NB>) et[i] = 0.0;
  __syncthreads();
  for (int64_t t = 0; t <= pr.p; ++t) {
    const int64_t s = pr.s0 + t;
    if (t > 0) {
      /* predict: with Mx = Lam + F^T Q^{-1} F = G G^T and r = eta - F^T Q^{-1} c,
       * Lam <- Q^{-1} - Y^T Y, eta <- Q^{-1} c + Y^T y,
       * Y = G^{-1} F^T Q^{-1}, y = G^{-1} r */
      const double* F = md.F + s * nn;
      copy_mat<NB>(Mx, L, md.Q + s * nn, n, false, n, n);
      chol_inverse_factor<NB>(Mx, Qi, L, n);
      mm<NB>(Qi, L, Qi, L, true, Qi, L, false, n, n, n, 1.0, 0.0);            /* Qi = Q^{-1} */
      mm<NB>(T2, L, Qi, L, false, F, n, false, n, n, n, 1.0, 0.0);            /* T2 = Q^{-1} F */
      copy_mat<NB>(Mx, L, Lm, L, false, n, n);
      mm<NB>(Mx, L, F, n, true, T2, L, false, n, n, n, 1.0, 1.0);             /* Mx = Lam + F^T T2 */
      mv<NB>(v1, Qi, L, false, md.c + s * n, n, n, 1.0, 0.0);                /* v1 = Q^{-1} c */
      mv<NB>(v2, F, n, true, v1, n, n, -1.0, 0.0);
      axpy<NB>(v2, et, n, 1.0);                                              /* v2 = r */
      copy_mat<NB>(Lm, L, T2, L, true, n, n);                                /* Lm = T2^T */
      double* const B[1] = {Lm};
      chol_forward<NB, false, false>(Mx, L, n, B, n, L, v2, 1);              /* Lm = Y, v2 = y */
      mm<NB>(Qi, L, Lm, L, true, Lm, L, false, n, n, n, -1.0, 1.0);           /* Lam- */
      mv<NB>(et, Lm, L, true, v2, n, n, 1.0, 0.0);
      axpy<NB>(et, v1, n, 1.0);                                              /* eta- */
      copy_mat<NB>(Lm, L, Qi, L, false, n, n);
    }
    const int m = m_obs[s];
    if (m > 0) { /* update: Lam += C^T C, eta += C^T o (whitened) */
      const double* Cw = wch.C + s * nn;
      mm<NB>(Lm, L, Cw, mr, true, Cw, mr, false, n, n, m, 1.0, 1.0);
      mv<NB>(et, Cw, mr, true, wch.o + s * n, n, m, 1.0, 1.0);
    }
    if (t < pr.p) {
      copy_mat<NB>(md.Lam + s * nn, n, Lm, L, false, n, n);
      for (int i = threadIdx.x; i < n; i += AT<NB>) md.eta[s * n + i] = et[i];
      __syncthreads();
    }
  }
  /* P_p = Lam^{-1}, x_p = P_p eta */
  const int64_t sp = pr.s0 + pr.p;
  copy_mat<NB>(Mx, L, Lm, L, false, n, n);
  chol_inverse_factor<NB>(Mx, Qi, L, n);
  mm<NB>(Qi, L, Qi, L, true, Qi, L, false, n, n, n, 1.0, 0.0);
  copy_mat<NB>(md.Pf + sp * nn, n, Qi, L, false, n, n);
  mv<NB>(md.xf + sp * n, Qi, L, false, et, n, n, 1.0, 0.0);
}

/* ------------------------------------------------------------------------ */
/* filtering elements (c :370-505, matlab :49-91)                            */
/* ------------------------------------------------------------------------ */

/*
 * Step s with model (F, c, Q) and whitened observation (C, o), noise I: with
 * S = C Q C^T + I = G G^T, Y_1 = G^{-1} C Q, Y_2 = G^{-1} C F,
 *   A = F - Y_1^T Y_2,  b = c + Y_1^T G^{-1} (o - C c),  Z = Q - Y_1^T Y_1,
 *   e = Y_2^T G^{-1} (o - C c),  J = Y_2^T Y_2.
 * The first element after the prior (x_p, P_p) uses Q1 = Q + F P_p F^T in
 * place of Q, A = 0, and b = m1 + Y_1^T G^{-1} (o - C m1) with m1 = F x_p + c.
 * Unobserved: A = F (0 if first), b = c
 * (m1 if first), Z = Q (Q1), e = 0, J = 0.
 */
template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_felem(const AsProb* probs, const int32_t* elem_prob, uk_chain_t wch,
                                               const int32_t* m_obs, AsModel md, AsElems el, int n, int mr) {
  constexpr int L = Ld<NB>::L;
  __shared__ double Qs[Ld<NB>::SZ], CQ[Ld<NB>::SZ], S[Ld<NB>::SZ], T[Ld<NB>::SZ];
  __shared__ double w1[NB], rr[2 * NB];
  double *const r = rr, *const rc = rr + NB;
  const int64_t ge = blockIdx.x;
  const AsProb pr = probs[elem_prob[ge]];
  const int64_t t = ge - pr.e0 + pr.p + 1;
  const int64_t s = pr.s0 + t;
  const bool firstel = t == pr.p + 1;
  const int64_t nn = (int64_t)n * n;
  const double* F = md.F + s * nn;
  const double* c = md.c + s * n;
  double* A = el.A + ge * nn;
  double* b = el.b + ge * n;
  double* Z = el.Z + ge * nn;
  double* e = el.e + ge * n;
  double* J = el.J + ge * nn;
  const int64_t spv = pr.s0 + pr.p;

  copy_mat<NB>(Qs, L, md.Q + s * nn, n, false, n, n);                       /* Qs = Q */
  copy_vec<NB>(w1, c, n);
  if (firstel) { /* Q1 = Q + F P F^T, m1 = F x + c */
    mm<NB>(T, L, F, n, false, md.Pf + spv * nn, n, false, n, n, n, 1.0, 0.0);
    mm<NB>(Qs, L, T, L, false, F, n, true, n, n, n, 1.0, 1.0);
    mv<NB>(w1, F, n, false, md.xf + spv * n, n, n, 1.0, 1.0);
  }
  const int m = m_obs[s];
  if (m == 0) {
    for (int idx = threadIdx.x; idx < NB * NB; idx += AT<NB>) {
      const int i = idx % NB, j = idx / NB;
      if (i < n && j < n) {
        A[i + j * n] = firstel ? 0.0 : F[i + j * n];
        Z[i + j * n] = Qs[i + j * L];
        J[i + j * n] = 0.0;
      }
    }
    for (int i = threadIdx.x; i < n; i += AT<NB>) {
      b[i] = w1[i];
      e[i] = 0.0;
    }
    return;
  }
  const double* ow = wch.o + s * n;
  copy_mat<NB>(T, L, wch.C + s * nn, mr, false, m, n);                       /* T = C (m x n) */
  mm<NB>(CQ, L, T, L, false, Qs, L, false, m, n, n, 1.0, 0.0);               /* CQ = C Q */
  set_identity<NB>(S, L, m, 1.0);
  mm<NB>(S, L, CQ, L, false, T, L, true, m, m, n, 1.0, 1.0);                 /* S = C Q C^T + I */
  mv<NB>(r, T, L, false, w1, m, n, -1.0, 0.0);
  axpy<NB>(r, ow, m, 1.0);                                                       /* r = o - C w1 */
  mv<NB>(rc, T, L, false, c, m, n, -1.0, 0.0);
  axpy<NB>(rc, ow, m, 1.0);                                                      /* rc = o - C c */
  copy_mat<NB>(Z, n, Qs, L, false, n, n);                                    /* Z = Q (Qs is free now) */
  mm<NB>(Qs, L, T, L, false, F, n, false, m, n, n, 1.0, 0.0);                /* Qs = C F */
  double* const B[2] = {CQ, Qs};
  chol_forward<NB, false, false>(S, L, m, B, n, L, rr, 2);                   /* CQ = Y_1, Qs = Y_2, r, rc = G^{-1} of them */
  mv<NB>(b, CQ, L, true, r, n, m, 1.0, 0.0);
  axpy<NB>(b, w1, n, 1.0);                                                   /* b = w1 + Y_1^T r */
  mm<NB>(Z, n, CQ, L, true, CQ, L, false, n, n, m, -1.0, 1.0);               /* Z = Q - Y_1^T Y_1 */
  if (firstel) {
    for (int idx = threadIdx.x; idx < NB * NB; idx += AT<NB>) {
      const int i = idx % NB, j = idx / NB;
      if (i < n && j < n) A[i + j * n] = 0.0;
    }
    __syncthreads();
  } else {
    copy_mat<NB>(A, n, F, n, false, n, n);
    mm<NB>(A, n, CQ, L, true, Qs, L, false, n, n, m, -1.0, 1.0);             /* A = F - Y_1^T Y_2 */
  }
  mv<NB>(e, Qs, L, true, rc, n, m, 1.0, 0.0);                                /* e = Y_2^T rc */
  mm<NB>(J, n, Qs, L, true, Qs, L, false, n, n, m, 1.0, 0.0);                /* J = Y_2^T Y_2 */
}

/* ------------------------------------------------------------------------ */
/* combines (c :889-1016, matlab :240-262)                                   */
/* ------------------------------------------------------------------------ */

/* blocks of an accumulator or of the work area (LDS, or global for the
 * filtering work of the 64 bucket), leading dimension Ld<NB>::L */
struct Blk {
  double *A, *b, *Z, *e, *J;
};
template <int NB>
struct Work {
  double *W1, *T, *T2, *Aj; /* W1: J_j, or E_j of the smoothing combine */
  double *v, *t0;           /* two vectors, NB apart; one */
};

/* a <- a (x) element g, filtering (A, b, Z, e, J of the reference's combine):
 *   A = A_j (I + Z_i J_j)^{-1} A_i,       b = A_j (I + Z_i J_j)^{-1} (b_i + Z_i e_j) + b_j,
 *   Z = A_j (I + Z_i J_j)^{-1} Z_i A_j^T + Z_j,
 *   e = A_i^T (I + J_j Z_i)^{-1} (e_j - J_j b_i) + e_i,
 *   J = A_i^T (I + J_j Z_i)^{-1} J_j A_i + J_i.
 * With Z_i = L L^T and N = I + L^T J_j L = G G^T: (I + Z_i J_j)^{-1} = L N^{-1}
 * L^{-1}, so that with Y_1 = G^{-1} L^{-1} A_i, Y_2 = G^{-1} L^T J_j A_i, Y_b =
 * G^{-1} L^T A_j^T, y_0 = G^{-1} (L^{-1} b_i + L^T e_j), y_1 = G^{-1} L^T (e_j -
 * J_j b_i):
 *   A = Y_b^T Y_1, b = Y_b^T y_0 + b_j, Z = Y_b^T Y_b + Z_j, e = Y_1^T y_1 + e_i,
 *   J = Y_1^T Y_2 + J_i.
 * Element g's blocks are read from HBM into registers first (all loads in
 * flight together) and written into LDS where they are needed. */
template <int NB>
__device__ void filt_combine(const Blk& a, const Work<NB>& w, const AsElems& el, int64_t g, int n) {
  constexpr int L = Ld<NB>::L;
  const int64_t nn = (int64_t)n * n;
  const double *bj = el.b + g * n, *ej = el.e + g * n;
  /* Up to NB = 48 Z_j is requested with the others; the 64 bucket fetches it
   * where it is used, to stay within its registers. */
  constexpr bool EARLY = NB <= 48;
  RegBlk<NB> rA, rZ, rJ;
  rJ.load(el.J + g * nn, n);
  rA.load(el.A + g * nn, n);
  if (EARLY) rZ.load(el.Z + g * nn, n);
  rJ.store(w.W1, L, n, false);
  rA.store(w.Aj, L, n, false);
  for (int i = threadIdx.x; i < n; i += AT<NB>) {
    w.v[i] = a.b[i];
    w.t0[i] = ej[i];
  }
  __syncthreads();
  mm<NB>(w.T2, L, w.W1, L, false, a.A, L, false, n, n, n, 1.0, 0.0);         /* T2 = J_j A_i */
  {
    double* const B[1] = {a.A};
    chol_forward<NB, true, true>(a.Z, L, n, B, n, L, w.v, 1);                /* Z = L, A = L^{-1} A_i, v = L^{-1} b_i */
  }
  mv<NB>(w.v, a.Z, L, true, w.t0, n, n, 1.0, 1.0);                           /* v = L^{-1} b_i + L^T e_j */
  mv<NB>(w.t0, w.W1, L, false, a.b, n, n, -1.0, 1.0);                        /* t0 = e_j - J_j b_i */
  mv<NB>(w.v + NB, a.Z, L, true, w.t0, n, n, 1.0, 0.0);
  mm<NB>(w.T, L, w.W1, L, false, a.Z, L, false, n, n, n, 1.0, 0.0);          /* T = J_j L */
  mm<NB>(w.T, L, a.Z, L, true, w.T, L, false, n, n, n, 1.0, 0.0);
  for (int i = threadIdx.x; i < n; i += AT<NB>) w.T[i * (L + 1)] += 1.0;     /* T = N (read after the next barrier) */
  mm<NB>(w.T2, L, a.Z, L, true, w.T2, L, false, n, n, n, 1.0, 0.0);
  mm<NB>(w.Aj, L, a.Z, L, true, w.Aj, L, true, n, n, n, 1.0, 0.0);           /* L^T A_j^T */
  {
    double* const B[3] = {a.A, w.T2, w.Aj};
    chol_forward<NB, false, false>(w.T, L, n, B, n, L, w.v, 2);              /* Y_1, Y_2, Y_b, y_0, y_1 */
  }
  mv<NB>(a.b, w.Aj, L, true, w.v, n, n, 1.0, 0.0);
  axpy<NB>(a.b, bj, n, 1.0);                                                 /* b */
  mv<NB>(a.e, a.A, L, true, w.v + NB, n, n, 1.0, 1.0);                       /* e */
  mm<NB>(a.J, L, a.A, L, true, w.T2, L, false, n, n, n, 1.0, 1.0);           /* J */
  if (!EARLY) rZ.load(el.Z + g * nn, n);
  rZ.store(a.Z, L, n, false);                                                /* Z = Z_j */
  __syncthreads();
  mm<NB>(a.Z, L, w.Aj, L, true, w.Aj, L, false, n, n, n, 1.0, 1.0);          /* Z */
  mm<NB>(a.A, L, w.Aj, L, true, a.A, L, false, n, n, n, 1.0, 0.0);           /* A */
}

/* a <- a (x) element g, smoothing; a is the running suffix and g the next
 * earlier step: E = E_j E_i, g = E_j g_i + g_j, L = E_j L_i E_j^T + L_j. */
template <int NB>
__device__ void smooth_combine(const Blk& a, const Work<NB>& w, const AsElems& el, int64_t g, int n) {
  constexpr int L = Ld<NB>::L;
  const int64_t nn = (int64_t)n * n;
  const double* gj = el.b + g * n;
  RegBlk<NB> rE, rL;
  rE.load(el.A + g * nn, n);
  rL.load(el.Z + g * nn, n);
  rE.store(w.W1, L, n, false);                                               /* W1 = E_j */
  __syncthreads();
  mm<NB>(a.A, L, w.W1, L, false, a.A, L, false, n, n, n, 1.0, 0.0);
  mv<NB>(a.b, w.W1, L, false, a.b, n, n, 1.0, 0.0);
  axpy<NB>(a.b, gj, n, 1.0);
  mm<NB>(w.T, L, w.W1, L, false, a.Z, L, false, n, n, n, 1.0, 0.0);
  rL.store(a.Z, L, n, false);
  __syncthreads();
  mm<NB>(a.Z, L, w.T, L, false, w.W1, L, true, n, n, n, 1.0, 1.0);
}

template <int NB>
__device__ void blk_load(const Blk& a, int ld, const AsElems& el, int64_t g, int n, bool filt) {
  const int64_t nn = (int64_t)n * n;
  RegBlk<NB> r;
  r.load(el.A + g * nn, n);
  r.store(a.A, ld, n, false);
  r.load(el.Z + g * nn, n);
  r.store(a.Z, ld, n, false);
  if (filt) {
    r.load(el.J + g * nn, n);
    r.store(a.J, ld, n, false);
  }
  for (int i = threadIdx.x; i < n; i += AT<NB>) {
    a.b[i] = el.b[g * n + i];
    if (filt) a.e[i] = el.e[g * n + i];
  }
  __syncthreads();
}

template <int NB>
__device__ void blk_store(const Blk& a, int ld, const AsElems& el, int64_t g, int n, bool filt) {
  const int64_t nn = (int64_t)n * n;
  for (int idx = threadIdx.x; idx < NB * NB; idx += AT<NB>) {
    const int i = idx % NB, j = idx / NB;
    if (i < n && j < n) {
      el.A[g * nn + i + j * n] = a.A[i + j * ld];
      el.Z[g * nn + i + j * n] = a.Z[i + j * ld];
      if (filt) el.J[g * nn + i + j * n] = a.J[i + j * ld];
    }
  }
  for (int i = threadIdx.x; i < n; i += AT<NB>) {
    el.b[g * n + i] = a.b[i];
    if (filt) el.e[g * n + i] = a.e[i];
  }
  __syncthreads();
}

/* LDS plan of a scan kernel: accumulator, then the work area when it fits */
template <int NB, bool FILT>
struct ScanPlan {
  static constexpr int SZ = Ld<NB>::SZ;
  static constexpr int ACC = FILT ? 3 * SZ + 2 * NB : 2 * SZ + NB;
  static constexpr int WORK = FILT ? 4 * SZ + 3 * NB : 2 * SZ;             /* W1, T, T2, Aj, v, t0 | W1, T */
  static constexpr bool WORK_GLOBAL = (ACC + WORK) * 8 > LDS_BYTES;
  static constexpr int LDS = ACC + (WORK_GLOBAL ? 0 : WORK);
};

template <int NB, bool FILT>
__device__ void scan_setup(double* lds, double* gwork, Blk& a, Work<NB>& w) {
  using SP = ScanPlan<NB, FILT>;
  constexpr int SZ = SP::SZ;
  double* q = lds;
  a.A = q; q += SZ;
  a.Z = q; q += SZ;
  a.J = nullptr;
  a.e = nullptr;
  if (FILT) { a.J = q; q += SZ; }
  a.b = q; q += NB;
  if (FILT) { a.e = q; q += NB; }
  double* p = SP::WORK_GLOBAL ? gwork + (int64_t)blockIdx.x * SP::WORK : q;
  w.W1 = p; p += SZ;
  w.T = p; p += SZ;
  w.T2 = w.Aj = w.v = w.t0 = nullptr;
  if (FILT) {
    w.T2 = p; p += SZ;
    w.Aj = p; p += SZ;
    w.v = p; p += 2 * NB;
    w.t0 = p;
  }
}

template <int NB, bool FILT>
__device__ __forceinline__ void combine(const Blk& a, const Work<NB>& w, const AsElems& el, int64_t g, int n) {
  if (FILT) filt_combine<NB>(a, w, el, g, n);
  else smooth_combine<NB>(a, w, el, g, n);
}

/* ------------------------------------------------------------------------ */
/* chunked scans                                                             */
/* ------------------------------------------------------------------------ */

/* A chunk: `len` elements of one problem in processing order, from `first`
 * in direction `dir` (+1 filtering, -1 smoothing); `tot` is its slot in the
 * chunk-total arrays and `rank` its index within its problem. */
struct Chunk {
  int64_t first;
  int64_t tot;
  int32_t len;
  int32_t dir;
  int32_t rank;
  int32_t pad;
};

/* pass 1: the total of every chunk */
template <int NB, bool FILT>
__global__ void __launch_bounds__(AT<NB>) ka_scan_reduce(const Chunk* ch, AsElems el, AsElems tot, int n, double* gwork) {
  using SP = ScanPlan<NB, FILT>;
  __shared__ double lds[SP::LDS];
  Blk a;
  Work<NB> w;
  scan_setup<NB, FILT>(lds, gwork, a, w);
  const Chunk c = ch[blockIdx.x];
  blk_load<NB>(a, Ld<NB>::L, el, c.first, n, FILT);
  for (int i = 1; i < c.len; ++i) combine<NB, FILT>(a, w, el, c.first + (int64_t)i * c.dir, n);
  blk_store<NB>(a, Ld<NB>::L, tot, c.tot, n, FILT);
}

/* pass 2, one Hillis-Steele round over the chunk totals of every problem:
 * out[t] = in[t - d] (x) in[t] when rank >= d, else in[t]. */
template <int NB, bool FILT>
__global__ void __launch_bounds__(AT<NB>) ka_scan_round(const Chunk* ch, AsElems in, AsElems out, int d, int n,
                                                    double* gwork) {
  using SP = ScanPlan<NB, FILT>;
  __shared__ double lds[SP::LDS];
  Blk a;
  Work<NB> w;
  scan_setup<NB, FILT>(lds, gwork, a, w);
  const Chunk c = ch[blockIdx.x];
  if (c.rank >= d) {
    blk_load<NB>(a, Ld<NB>::L, in, c.tot - d, n, FILT);
    combine<NB, FILT>(a, w, in, c.tot, n);
  } else {
    blk_load<NB>(a, Ld<NB>::L, in, c.tot, n, FILT);
  }
  blk_store<NB>(a, Ld<NB>::L, out, c.tot, n, FILT);
}

/* pass 3: every prefix within a chunk, seeded with the inclusive total of
 * the chunk before it; results overwrite the elements in place. */
template <int NB, bool FILT>
__global__ void __launch_bounds__(AT<NB>) ka_scan_down(const Chunk* ch, AsElems el, AsElems tot, int n, double* gwork) {
  using SP = ScanPlan<NB, FILT>;
  __shared__ double lds[SP::LDS];
  Blk a;
  Work<NB> w;
  scan_setup<NB, FILT>(lds, gwork, a, w);
  const Chunk c = ch[blockIdx.x];
  int i0 = 0;
  if (c.rank == 0) {
    blk_load<NB>(a, Ld<NB>::L, el, c.first, n, FILT);
    i0 = 1;
  } else {
    blk_load<NB>(a, Ld<NB>::L, tot, c.tot - 1, n, FILT);
  }
  for (int i = i0; i < c.len; ++i) {
    const int64_t g = c.first + (int64_t)i * c.dir;
    combine<NB, FILT>(a, w, el, g, n);
    blk_store<NB>(a, Ld<NB>::L, el, g, n, FILT);
  }
}

/* ------------------------------------------------------------------------ */
/* filtered distributions, smoothing elements, results                       */
/* ------------------------------------------------------------------------ */

/* filtered (x, P) of steps p+1 .. k-1: (b, Z) of the filtering prefixes */
template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_filtered(const AsProb* probs, const int32_t* elem_prob, AsElems el,
                                                  AsModel md, int n) {
  const int64_t g = blockIdx.x;
  const AsProb pr = probs[elem_prob[g]];
  const int64_t s = pr.s0 + (g - pr.e0) + pr.p + 1;
  const int64_t nn = (int64_t)n * n;
  for (int idx = threadIdx.x; idx < n * n; idx += AT<NB>) md.Pf[s * nn + idx] = el.Z[g * nn + idx];
  for (int i = threadIdx.x; i < n; i += AT<NB>) md.xf[s * n + i] = el.b[g * n + i];
}

/*
 * Smoothing element of step s, stored at slot s (c :697-753, matlab :94-114):
 *   last step: E = 0, g = x, L = P;
 *   t >= p: with (F, c, Q) of step s + 1,
 *           E = P F^T (F P F^T + Q)^{-1}, g = x - E (F x + c), L = P - E F P;
 *   t < p:  from the information form (Lam, eta),
 *           L = (Lam + F^T Q^{-1} F)^{-1}, E = L F^T Q^{-1}, g = L (eta - F^T Q^{-1} c).
 */
template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_selem(const AsProb* probs, const int32_t* step_prob, AsModel md, AsElems el,
                                               int n) {
  constexpr int L = Ld<NB>::L;
  __shared__ double M[Ld<NB>::SZ], T[Ld<NB>::SZ], U[Ld<NB>::SZ];
  __shared__ double v1[NB], v2[NB];
  const int64_t s = blockIdx.x;
  const AsProb pr = probs[step_prob[s]];
  const int64_t t = s - pr.s0;
  const int64_t nn = (int64_t)n * n;
  double* E = el.A + s * nn;
  double* gv = el.b + s * n;
  double* Lo = el.Z + s * nn;
  if (t == pr.k - 1) {
    for (int idx = threadIdx.x; idx < n * n; idx += AT<NB>) {
      E[idx] = 0.0;
      Lo[idx] = md.Pf[s * nn + idx];
    }
    for (int i = threadIdx.x; i < n; i += AT<NB>) gv[i] = md.xf[s * n + i];
    return;
  }
  const double* F = md.F + (s + 1) * nn;
  const double* c = md.c + (s + 1) * n;
  const double* Q = md.Q + (s + 1) * nn;
  if (t >= pr.p) {
    const double* P = md.Pf + s * nn;
    const double* x = md.xf + s * n;
    copy_mat<NB>(U, L, P, n, false, n, n);                                   /* U = P */
    copy_mat<NB>(M, L, F, n, false, n, n);                                   /* M = F */
    mm<NB>(T, L, M, L, false, U, L, false, n, n, n, 1.0, 0.0);               /* T = F P */
    mv<NB>(v1, M, L, false, x, n, n, 1.0, 0.0);
    axpy<NB>(v1, c, n, 1.0);                                                 /* v1 = F x + c */
    copy_mat<NB>(U, L, Q, n, false, n, n);
    mm<NB>(U, L, T, L, false, M, L, true, n, n, n, 1.0, 1.0);                /* U = F P F^T + Q = G G^T */
    set_identity<NB>(M, L, n, 1.0);
    double* const B[2] = {T, M};
    chol_forward<NB, false, false>(U, L, n, B, n, L, nullptr, 0);            /* T = Y = G^{-1} F P, M = G^{-1} */
    mm<NB>(E, n, T, L, true, M, L, false, n, n, n, 1.0, 0.0);                /* E = Y^T G^{-1} */
    mv<NB>(v2, M, L, false, v1, n, n, 1.0, 0.0);
    mv<NB>(gv, T, L, true, v2, n, n, -1.0, 0.0);
    axpy<NB>(gv, x, n, 1.0);                                                 /* g = x - E (F x + c) */
    copy_mat<NB>(Lo, n, P, n, false, n, n);
    mm<NB>(Lo, n, T, L, true, T, L, false, n, n, n, -1.0, 1.0);              /* L = P - Y^T Y */
  } else {
    copy_mat<NB>(U, L, Q, n, false, n, n);
    copy_mat<NB>(T, L, F, n, false, n, n);
    copy_vec<NB>(v1, c, n);
    set_identity<NB>(M, L, n, 1.0);
    double* const B[2] = {T, M};
    chol_forward<NB, false, false>(U, L, n, B, n, L, v1, 1);                 /* Q = G G^T: T = Y = G^{-1} F, M = G^{-1}, v1 = G^{-1} c */
    mm<NB>(M, L, M, L, true, T, L, false, n, n, n, 1.0, 0.0);                /* M = Q^{-1} F */
    copy_mat<NB>(U, L, md.Lam + s * nn, n, false, n, n);
    mm<NB>(U, L, T, L, true, T, L, false, n, n, n, 1.0, 1.0);                /* U = Lam + F^T Q^{-1} F */
    mv<NB>(v2, T, L, true, v1, n, n, -1.0, 0.0);
    axpy<NB>(v2, md.eta + s * n, n, 1.0);                                    /* v2 = eta - F^T Q^{-1} c */
    chol_inverse_factor<NB>(U, T, L, n);
    mm<NB>(T, L, T, L, true, T, L, false, n, n, n, 1.0, 0.0);                /* T = L */
    copy_mat<NB>(Lo, n, T, L, false, n, n);
    mm<NB>(E, n, T, L, false, M, L, true, n, n, n, 1.0, 0.0);                /* E = L (Q^{-1} F)^T */
    mv<NB>(gv, T, L, false, v2, n, n, 1.0, 0.0);                             /* g = L (eta - F^T Q^{-1} c) */
  }
}

/* the smoothing prefix of step s (taken from the last step) is (E, g, L):
 * estimate g, covariance L */
template <int NB>
__global__ void __launch_bounds__(AT<NB>) ka_results(AsElems el, double* xout, double* Sout, int n) {
  const int64_t s = blockIdx.x;
  const int64_t nn = (int64_t)n * n;
  for (int idx = threadIdx.x; idx < n * n; idx += AT<NB>) Sout[s * nn + idx] = el.Z[s * nn + idx];
  for (int i = threadIdx.x; i < n; i += AT<NB>) xout[s * n + i] = el.b[s * n + i];
}

} /* namespace */
/* ------------------------------------------------------------------------ */
/* host driver                                                               */
/* ------------------------------------------------------------------------ */

struct ukhip_batch;
extern "C" void uk_batch_view(ukhip_batch* b, const uk_raw_t** raw, double** xout, double** Sout, int64_t* steps,
                              int* nprob, const int64_t** k, void** assoc_ws, size_t* assoc_bytes);
extern "C" void uk_batch_set_assoc_ws(ukhip_batch* b, void* p, size_t bytes);
extern "C" void uk_batch_chain0(ukhip_batch* b, uk_chain_t* ch, const int32_t** m0);
extern "C" hipError_t uk_batch_weigh_dense0(ukhip_batch* b, hipStream_t st);
extern "C" hipError_t uk_batch_weigh_level0(ukhip_batch* b, hipStream_t st);

namespace {

bool ok(hipError_t e, const char* what) {
  if (e == hipSuccess) return true;
  uk_set_error("%s: %s", what, hipGetErrorString(e));
  return false;
}

/* Event timing of one associative smoothing (ukhip_batch_smooth_associative_timed):
 * an event after each kernel class, in launch order; slot i's time is
 * ev[i] -> ev[i + 1]. Set for the duration of one timed call on this thread. */
struct AsTimer {
  hipEvent_t ev[UKHIP_AS_SLOTS + 1]{};
  int32_t launches[UKHIP_AS_SLOTS]{};
  double ms[UKHIP_AS_SLOTS]{};
};
thread_local AsTimer* t_timer = nullptr;

/* chunks of at most `chunk` elements over `len` elements of one problem;
 * dir = +1 starts at `base`, dir = -1 at base + len - 1. */
int64_t make_chunks(std::vector<Chunk>& out, int64_t base, int64_t len, int dir, int64_t chunk, int64_t& tot0) {
  const int64_t nch = (len + chunk - 1) / chunk;
  for (int64_t r = 0; r < nch; ++r) {
    Chunk c{};
    const int64_t lo = r * chunk;
    c.first = dir > 0 ? base + lo : base + len - 1 - lo;
    c.len = (int32_t)std::min(chunk, len - lo);
    c.dir = dir;
    c.tot = tot0 + r;
    c.rank = (int32_t)r;
    out.push_back(c);
  }
  tot0 += nch;
  return nch;
}

/* Chunks aimed at over a batch: as many as the filtering scan's workgroups
 * that are resident at once (by its LDS: one per CU in buckets 48 and 64, two
 * in 32, ten single waves in 16). More would only add to the rounds over the
 * chunk totals. Chunks have at least 4 elements. */
template <int NB>
constexpr int64_t CHUNKS_TARGET = NB <= 16 ? 2560 : (NB <= 32 ? 512 : 256);

template <int NB>
int run_assoc(ukhip_batch* b) {
  hipStream_t st = (hipStream_t)ukhip_stream();
  const uk_raw_t* raw;
  double *xout, *Sout;
  int64_t S;
  int nprob;
  const int64_t* kk;
  void* ws;
  size_t ws_bytes;
  uk_batch_view(b, &raw, &xout, &Sout, &S, &nprob, &kk, &ws, &ws_bytes);
  if (!xout || !Sout) return -1;
  const int n = raw->n;
  uk_chain_t wch;
  const int32_t* m_obs = nullptr;
  uk_batch_chain0(b, &wch, &m_obs);
  const int mr = wch.mr;

  /* plan: p of every problem from the observation counts */
  std::vector<int32_t> m_h(S);
  if (!ok(hipMemcpy(m_h.data(), m_obs, S * sizeof(int32_t), hipMemcpyDeviceToHost), "download m")) return -1;
  std::vector<AsProb> probs(nprob);
  std::vector<int32_t> elem_prob, step_prob(S);
  int64_t s0 = 0, ne = 0;
  for (int p = 0; p < nprob; ++p) {
    AsProb pr{};
    pr.s0 = s0;
    pr.k = kk[p];
    int64_t acc = 0, pp = 0;
    for (pp = 0; pp < pr.k; ++pp) {
      acc += m_h[s0 + pp];
      if (acc >= n) break;
    }
    if (pp == pr.k) {
      uk_set_error("kalman_smooth_associative: problem %d: the observations do not determine the states", p);
      return -1;
    }
    pr.p = pp;
    pr.e0 = ne;
    for (int64_t t = pr.p + 1; t < pr.k; ++t) elem_prob.push_back(p);
    ne += pr.k - pr.p - 1;
    for (int64_t t = 0; t < pr.k; ++t) step_prob[s0 + t] = p;
    probs[p] = pr;
    s0 += pr.k;
  }
  const int64_t fchunk = std::max<int64_t>(4, (ne + CHUNKS_TARGET<NB> - 1) / CHUNKS_TARGET<NB>);
  const int64_t schunk = std::max<int64_t>(4, (S + CHUNKS_TARGET<NB> - 1) / CHUNKS_TARGET<NB>);
  std::vector<Chunk> fch, sch;
  int64_t ftot = 0, stot = 0, maxr_f = 0, maxr_s = 0;
  for (int p = 0; p < nprob; ++p) {
    const int64_t len = probs[p].k - probs[p].p - 1;
    if (len > 0) maxr_f = std::max(maxr_f, make_chunks(fch, probs[p].e0, len, +1, fchunk, ftot));
    maxr_s = std::max(maxr_s, make_chunks(sch, probs[p].s0, probs[p].k, -1, schunk, stot));
  }

  /* workspace */
  const size_t nn = (size_t)n * n;
  size_t need = 0;
  auto take = [&](size_t bytes) {
    const size_t r = need;
    need += (bytes + 255) & ~(size_t)255;
    return r;
  };
  auto elem_bytes = [&](int64_t cnt, bool filt) { return (size_t)std::max<int64_t>(cnt, 1) * ((filt ? 3 : 2) * nn + (filt ? 2 : 1) * n) * 8; };
  const size_t o_model = take((size_t)S * (4 * nn + 4 * n) * 8);
  const size_t o_fe = take(elem_bytes(ne, true));
  const size_t o_ft0 = take(elem_bytes(ftot, true)), o_ft1 = take(elem_bytes(ftot, true));
  const size_t o_se = take(elem_bytes(S, false));
  const size_t o_st0 = take(elem_bytes(stot, false)), o_st1 = take(elem_bytes(stot, false));
  const int64_t maxch = std::max<int64_t>((int64_t)std::max(fch.size(), sch.size()), 1);
  const size_t o_gw = take((size_t)maxch * ScanPlan<NB, true>::WORK * 8);
  const size_t tab_bytes = probs.size() * sizeof(AsProb) + (elem_prob.size() + step_prob.size()) * 4 +
                           (fch.size() + sch.size()) * sizeof(Chunk) + 6 * 256;
  const size_t o_tab = take(tab_bytes);
  if (ws_bytes < need) {
    if (ws) (void)hipFree(ws);
    uk_batch_set_assoc_ws(b, nullptr, 0);
    ws = nullptr;
    if (!ok(hipMalloc(&ws, need), "hipMalloc(associative workspace)")) return -1;
    uk_batch_set_assoc_ws(b, ws, need);
  }
  char* W = (char*)ws;
  AsModel md;
  {
    double* q = (double*)(W + o_model);
    md.F = q; q += S * nn;
    md.Q = q; q += S * nn;
    md.Pf = q; q += S * nn;
    md.Lam = q; q += S * nn;
    md.c = q; q += S * n;
    md.xf = q; q += S * n;
    md.eta = q;
  }
  auto elems_at = [&](size_t off, int64_t cnt, bool filt) {
    cnt = std::max<int64_t>(cnt, 1);
    AsElems e{};
    double* q = (double*)(W + off);
    e.A = q; q += cnt * nn;
    e.Z = q; q += cnt * nn;
    if (filt) { e.J = q; q += cnt * nn; }
    e.b = q; q += cnt * n;
    if (filt) e.e = q;
    return e;
  };
  const AsElems fe = elems_at(o_fe, ne, true);
  const AsElems ft[2] = {elems_at(o_ft0, ftot, true), elems_at(o_ft1, ftot, true)};
  const AsElems se = elems_at(o_se, S, false);
  const AsElems stt[2] = {elems_at(o_st0, stot, false), elems_at(o_st1, stot, false)};
  double* gw = (double*)(W + o_gw);

  /* tables */
  std::vector<char> tab(tab_bytes, 0);
  size_t to = 0;
  auto put = [&](const void* src, size_t bytes) {
    const size_t at_ = to;
    if (bytes) std::memcpy(tab.data() + to, src, bytes);
    to += (bytes + 255) & ~(size_t)255;
    return W + o_tab + at_;
  };
  const AsProb* d_probs = (const AsProb*)put(probs.data(), probs.size() * sizeof(AsProb));
  const int32_t* d_elem_prob = (const int32_t*)put(elem_prob.data(), elem_prob.size() * 4);
  const int32_t* d_step_prob = (const int32_t*)put(step_prob.data(), step_prob.size() * 4);
  const Chunk* d_fch = (const Chunk*)put(fch.data(), fch.size() * sizeof(Chunk));
  const Chunk* d_sch = (const Chunk*)put(sch.data(), sch.size() * sizeof(Chunk));
  if (!ok(hipMemcpyAsync(W + o_tab, tab.data(), to, hipMemcpyHostToDevice, st), "upload scan tables")) return -1;

  const dim3 blk(AT<NB>);
  AsTimer* tm = t_timer;
  auto mark = [&](int slot, int launches) { /* slot's launches are done: its closing event */
    if (!tm) return;
    tm->launches[slot] += launches;
    (void)hipEventRecord(tm->ev[slot + 1], st);
  };
  if (tm) (void)hipEventRecord(tm->ev[0], st);
  /* with every K and C given as 'w' and H = I only the observations need
   * whitening, and the model is the input's */
  const bool diag = raw->H_ident && !raw->K_full && !raw->C_full && mr == raw->mr;
  if (!ok(diag ? uk_batch_weigh_level0(b, st) : uk_batch_weigh_dense0(b, st), "k_weigh")) return -1;
  mark(UKHIP_AS_WEIGH, 1);
  if (diag) ka_model_diag<<<dim3((unsigned)S), dim3(256), 0, st>>>(*raw, md, n);
  else ka_model<NB><<<dim3((unsigned)S), blk, 0, st>>>(wch, raw->first, md, n);
  mark(UKHIP_AS_MODEL, 1);
  ka_prior<NB><<<dim3((unsigned)nprob), blk, 0, st>>>(d_probs, wch, m_obs, md, n, mr);
  mark(UKHIP_AS_PRIOR, 1);
  if (ne > 0) {
    const unsigned nc = (unsigned)fch.size();
    ka_felem<NB><<<dim3((unsigned)ne), blk, 0, st>>>(d_probs, d_elem_prob, wch, m_obs, md, fe, n, mr);
    mark(UKHIP_AS_FELEM, 1);
    ka_scan_reduce<NB, true><<<dim3(nc), blk, 0, st>>>(d_fch, fe, ft[0], n, gw);
    int cur = 0, rounds = 0;
    for (int64_t d = 1; d < maxr_f; d <<= 1) {
      ka_scan_round<NB, true><<<dim3(nc), blk, 0, st>>>(d_fch, ft[cur], ft[cur ^ 1], (int)d, n, gw);
      cur ^= 1;
      ++rounds;
    }
    ka_scan_down<NB, true><<<dim3(nc), blk, 0, st>>>(d_fch, fe, ft[cur], n, gw);
    mark(UKHIP_AS_FSCAN, 2 + rounds);
    ka_filtered<NB><<<dim3((unsigned)ne), blk, 0, st>>>(d_probs, d_elem_prob, fe, md, n);
    mark(UKHIP_AS_FILTERED, 1);
  } else {
    mark(UKHIP_AS_FELEM, 0);
    mark(UKHIP_AS_FSCAN, 0);
    mark(UKHIP_AS_FILTERED, 0);
  }
  {
    const unsigned nc = (unsigned)sch.size();
    ka_selem<NB><<<dim3((unsigned)S), blk, 0, st>>>(d_probs, d_step_prob, md, se, n);
    mark(UKHIP_AS_SELEM, 1);
    ka_scan_reduce<NB, false><<<dim3(nc), blk, 0, st>>>(d_sch, se, stt[0], n, gw);
    int cur = 0, rounds = 0;
    for (int64_t d = 1; d < maxr_s; d <<= 1) {
      ka_scan_round<NB, false><<<dim3(nc), blk, 0, st>>>(d_sch, stt[cur], stt[cur ^ 1], (int)d, n, gw);
      cur ^= 1;
      ++rounds;
    }
    ka_scan_down<NB, false><<<dim3(nc), blk, 0, st>>>(d_sch, se, stt[cur], n, gw);
    mark(UKHIP_AS_SSCAN, 2 + rounds);
    ka_results<NB><<<dim3((unsigned)S), blk, 0, st>>>(se, xout, Sout, n);
    mark(UKHIP_AS_RESULTS, 1);
  }
  if (!ok(hipGetLastError(), "associative launches")) return -1;
  /* the host tables above must outlive the asynchronous upload */
  if (!ok(hipStreamSynchronize(st), "associative smoothing")) return -1;
  if (tm) {
    for (int i = 0; i < UKHIP_AS_TOTAL; ++i) {
      float f = 0.f;
      if (!ok(hipEventElapsedTime(&f, tm->ev[i], tm->ev[i + 1]), "associative timing")) return -1;
      tm->ms[i] += f;
    }
    float f = 0.f;
    if (!ok(hipEventElapsedTime(&f, tm->ev[0], tm->ev[UKHIP_AS_TOTAL]), "associative timing")) return -1;
    tm->ms[UKHIP_AS_TOTAL] += f;
  }
  return 0;
}

}  // namespace

/* The associative smoother over a batch (c/kalman_associative_smoother.c:
 * 1199-1240). Covariances are always produced, as in the reference, whose
 * associative path does not read KALMAN_NO_COVARIANCE. */
extern "C" int uk_assoc_smooth(struct ukhip_batch* b, uint32_t options) {
  (void)options;
  const uk_raw_t* raw;
  double *xout, *Sout;
  int64_t S;
  int nprob;
  const int64_t* k;
  void* ws;
  size_t wsb;
  uk_batch_view(b, &raw, &xout, &Sout, &S, &nprob, &k, &ws, &wsb);
  if (!xout || !Sout) return -1; /* the output storage could not be allocated (error recorded) */
  uk_chain_t ch0;
  const int32_t* m0;
  uk_batch_chain0(b, &ch0, &m0);
  switch (uk_bucket(raw->n > ch0.mr ? raw->n : ch0.mr)) {
    case 8:
    case 16: return run_assoc<16>(b);
    case 32: return run_assoc<32>(b);
    case 48: return run_assoc<48>(b);
    case 64: return run_assoc<64>(b);
    default: uk_set_error("associative: state dimension %d is above 64", raw->n); return -1;
  }
}

/* ukhip_batch_smooth_associative_timed (include/ukhip.h): parts one after
 * another, each with its events; the slot sums are returned. */
extern "C" int uk_assoc_smooth_timed(struct ukhip_batch* b, uint32_t options, double* ms, int32_t* launches) {
  AsTimer tm;
  for (auto& e : tm.ev)
    if (!ok(hipEventCreate(&e), "hipEventCreate")) {
      for (auto& x : tm.ev)
        if (x) (void)hipEventDestroy(x);
      return -1;
    }
  t_timer = &tm;
  const int rc = uk_assoc_smooth(b, options);
  t_timer = nullptr;
  for (auto& e : tm.ev) (void)hipEventDestroy(e);
  if (rc != 0) return rc;
  for (int i = 0; i < UKHIP_AS_SLOTS; ++i) {
    if (ms) ms[i] += tm.ms[i];
    if (launches) launches[i] += tm.launches[i];
  }
  return 0;
}
