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
 * Every element build and every combine runs in one workgroup, on the FP64
 * matrix cores, with the matrices in registers (see Geo): one wave for n <= 16,
 * three to four waves above.
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
#include <memory>
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

/* ------------------------------------------------------------------------ */
/* workgroup-level dense algebra on blocks of order <= NB                    */
/* ------------------------------------------------------------------------ */

/* element (i, k) of op(A) for a column-major A with leading dimension ld */
__device__ __forceinline__ double at(const double* A, int ld, bool t, int i, int k) {
  return t ? A[k + (int64_t)i * ld] : A[i + (int64_t)k * ld];
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

/* ------------------------------------------------------------------------ */
/* tile columns                                                              */
/* ------------------------------------------------------------------------ */

/*
 * The layout of the element builds, the prior and the scans: a matrix of order
 * n <= 16 NT is NT x NT tiles in the accumulator layout, wave w holds tile
 * column w in NT registers quads, and vectors are a tile column too (on a wave
 * of their own for NT = 2 and 3; on wave 0 next to its matrix columns for NT =
 * 1 and for NT = 4, where a fifth wave would halve the registers of all).
 * All products have the form Y = P^T X (tmul): X and Y stay in the registers
 * of their waves and only P goes through LDS, where a tile is stored as it
 * lies in the lanes (for NT = 1 it does not leave the registers, and the kernel
 * uses no LDS and no barrier). Rows and columns from n on are zeros.
 * Against blocks of whole workgroups in LDS (products and eliminations on the
 * matrix cores as here) a filtering combine takes 41 us instead of 72 at n = 48,
 * with two workgroups on a CU instead of one, and 12 us instead of 25 for n <=
 * 16, launch included.
 */
template <int NT>
struct Geo {
  static constexpr bool SEP = NT == 2 || NT == 3; /* the vectors have a wave of their own */
  static constexpr int WAVES = NT + (SEP ? 1 : 0);
  static constexpr int THREADS = 64 * WAVES;
};
/* waves per SIMD the kernels over many elements are compiled for: two workgroups of four waves on a
 * CU at NT = 3; all registers for one wave at NT = 4. (The
 * element builds at n = 48, k = 10000: 855 -> 551 us and 840 -> 722 us with two,
 * a few registers spilled included.) */
template <int NT>
constexpr int SCAN_OCC = NT == 4 ? 1 : 2;

template <int NT>
struct Who { /* of this lane */
  int li, lk, lane, w;
  bool mat, vec;
  __device__ Who() {
    lane = threadIdx.x & 63;
    li = lane & 15;
    lk = lane >> 4;
    w = NT == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    mat = !Geo<NT>::SEP || w < NT;
    vec = w == (Geo<NT>::SEP ? NT : 0);
  }
};
template <int NT>
__device__ __forceinline__ void sync() {
  if (NT > 1) __syncthreads();
}

/* a matrix shared by the waves: tile (r, c) as it lies in the lanes */
template <int NT>
struct Sh {
  double* p;
  __device__ __forceinline__ void put(const as_d4 (&X)[NT], const Who<NT>& me) {
    if (!me.mat) return;
#pragma unroll
    for (int r = 0; r < NT; ++r)
#pragma unroll
      for (int g = 0; g < 4; ++g) p[((me.w * NT + r) * 4 + g) * 64 + me.lane] = X[r][g];
  }
  /* the transpose of an upper triangular matrix */
  __device__ __forceinline__ void put_upper_t(const as_d4 (&X)[NT], const Who<NT>& me) {
    if (!me.mat) return;
#pragma unroll
    for (int r = 0; r < NT; ++r)
      if (r <= me.w) {
#pragma unroll
        for (int g = 0; g < 4; ++g) p[(r * NT + me.w) * 256 + me.li * 16 + 4 * g + me.lk] = X[r][g];
      }
  }
  __device__ __forceinline__ as_d4 tile(int r, int c, const Who<NT>& me) const {
    as_d4 t;
#pragma unroll
    for (int g = 0; g < 4; ++g) t[g] = p[((c * NT + r) * 4 + g) * 64 + me.lane];
    return t;
  }
};
template <>
struct Sh<1> {
  as_d4 v;
  __device__ __forceinline__ void put(const as_d4 (&X)[1], const Who<1>&) { v = X[0]; }
  __device__ __forceinline__ void put_upper_t(const as_d4 (&X)[1], const Who<1>& me) { /* the product with I is exact */
    as_d4 y = as_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int g = 0; g < 4; ++g) y = as_mfma(X[0][g], 4 * g + me.lk == me.li ? 1.0 : 0.0, y);
    v = y;
  }
  __device__ __forceinline__ as_d4 tile(int, int, const Who<1>&) const { return v; }
};
template <int NT>
struct Lds {
  double b0[NT * NT * 256], b1[NT * NT * 256], wt[256], tr[NT * 256];
};
template <>
struct Lds<1> {
  double b0[1], b1[1], wt[1], tr[1];
};
template <int NT>
__device__ __forceinline__ Sh<NT> sh(double* p) {
  Sh<NT> s;
  if constexpr (NT > 1) s.p = p;
  return s;
}

/* Y += SGN P^T X; LOWER: P is lower triangular. Over the whole order, or with
 * kk >= 0 over the first kk rows of P and X (the rest is zeros) */
template <int NT, int SGN = 1, bool LOWER = false>
__device__ __forceinline__ void tmul(const Sh<NT>& P, const as_d4 (&X)[NT], as_d4 (&Y)[NT], const Who<NT>& me,
                                     int kk = -1) {
  auto rows = [&](int r) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      if (!LOWER || r >= i) {
        const as_d4 p = P.tile(r, i, me);
#pragma unroll
        for (int g = 0; g < 4; ++g) Y[i] = as_mfma(SGN < 0 ? -p[g] : p[g], X[r][g], Y[i]);
      }
    }
  };
  if (kk < 0) {
#pragma unroll
    for (int r = 0; r < NT; ++r) rows(r);
    mfma_drain();
  } else {
#pragma unroll
    for (int r = 0; r < NT; ++r)
      if (16 * r < kk) {
        rows(r);
        mfma_drain();
      }
  }
}
/* The same for one tile: as many of the four products as rows of P and X are
 * not zeros (they are n here where the whole order is asked for) */
template <int G, int SGN>
__device__ __forceinline__ void tmul_rows(const as_d4& p, const as_d4& x, as_d4& y) {
#pragma unroll
  for (int g = 0; g < G; ++g) y = as_mfma(SGN < 0 ? -p[g] : p[g], x[g], y);
  mfma_drain();
}
template <int SGN>
__device__ __forceinline__ void tmul_tile(const as_d4& p, const as_d4& x, as_d4& y, int kk) {
  if (kk > 12) tmul_rows<4, SGN>(p, x, y);
  else if (kk > 8) tmul_rows<3, SGN>(p, x, y);
  else if (kk > 4) tmul_rows<2, SGN>(p, x, y);
  else tmul_rows<1, SGN>(p, x, y);
}
template <int NT, int SGN = 1, bool LOWER = false>
__device__ __forceinline__ void tmul_n(const Sh<NT>& P, const as_d4 (&X)[NT], as_d4 (&Y)[NT], int n, const Who<NT>& me) {
  if constexpr (NT == 1) tmul_tile<SGN>(P.v, X[0], Y[0], n);
  else tmul<NT, SGN, LOWER>(P, X, Y, me);
}
template <int NT, int SGN = 1>
__device__ __forceinline__ void tmul_m(const Sh<NT>& P, const as_d4 (&X)[NT], as_d4 (&Y)[NT], int m, const Who<NT>& me) {
  if constexpr (NT == 1) tmul_tile<SGN>(P.v, X[0], Y[0], m);
  else tmul<NT, SGN>(P, X, Y, me, m);
}
template <int NT>
__device__ __forceinline__ void zero(as_d4 (&X)[NT]) {
#pragma unroll
  for (int r = 0; r < NT; ++r) X[r] = as_d4{0.0, 0.0, 0.0, 0.0};
}
/* X += 1 on the diagonal from row `lo` to below row `hi` */
template <int NT>
__device__ __forceinline__ void add_diag(as_d4 (&X)[NT], int lo, int hi, const Who<NT>& me) {
  const int col = 16 * me.w + me.li;
#pragma unroll
  for (int r = 0; r < NT; ++r) {
#pragma unroll
    for (int g = 0; g < 4; ++g) X[r][g] += 16 * r + 4 * g + me.lk == col && col >= lo && col < hi ? 1.0 : 0.0;
  }
}
/* this wave's column of G (rows x cols, ld); T: of its transpose, whose loads
 * are the contiguous ones (taken for symmetric matrices too) */
template <int NT, bool T>
__device__ __forceinline__ void load(as_d4 (&X)[NT], const double* G, int rows, int cols, int ld, const Who<NT>& me) {
  const int col = 16 * me.w + me.li, lr = T ? cols : rows, lc = T ? rows : cols;
  double v[NT][4];
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 16 * r + 4 * g + me.lk;
      v[r][g] = G[row < lr && col < lc ? (T ? col + row * ld : row + col * ld) : 0];
    }
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 16 * r + 4 * g + me.lk;
      X[r][g] = row < lr && col < lc ? v[r][g] : 0.0;
    }
}
template <int NT, bool T>
__device__ __forceinline__ void store(const as_d4 (&X)[NT], double* G, int n, const Who<NT>& me) {
  const int col = 16 * me.w + me.li;
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 16 * r + 4 * g + me.lk;
      if (row < n && col < n) G[T ? col + row * n : row + col * n] = X[r][g];
    }
}
/* a vector, the same in every column of its tiles */
template <int NT>
__device__ __forceinline__ void load_vec(as_d4 (&X)[NT], const double* v, int n, const Who<NT>& me) {
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 16 * r + 4 * g + me.lk;
      const double x = v[row < n ? row : 0];
      X[r][g] = row < n ? x : 0.0;
    }
}
template <int NT>
__device__ __forceinline__ void store_vec(const as_d4 (&X)[NT], double* v, int n, const Who<NT>& me) {
  if (me.li != 0) return;
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 16 * r + 4 * g + me.lk;
      if (row < n) v[row] = X[r][g];
    }
}
/* column K of the tiles in all columns */
template <int K, int NT>
__device__ __forceinline__ void spread(as_d4 (&X)[NT]) {
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int g = 0; g < 4; ++g) X[r][g] = row_lane<K>(X[r][g]);
}

/* row tile p of X through G_pp^{-1}, whose transpose is wt */
template <int NT>
__device__ __forceinline__ void panel_solve(as_d4& x, const as_d4& wt) {
  as_d4 y = as_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int g = 0; g < 4; ++g) y = as_mfma(wt[g], x[g], y);
  x = y;
}

/*
 * Forward elimination with a symmetric positive definite M = G G^T (tile rows
 * <= w of column w are used): M becomes G^T (rows <= w) and every R becomes
 * G^{-1} R; R1 of all waves, the others of those that hold matrix columns.
 * Rows of M from lim on are the identity's. Wave p factors diagonal tile p in its
 * registers and hands out the inverse of its factor, the waves solve row tile
 * p, hand out M's, and update the rows below: two barriers a panel.
 * A pivoted Gauss-Jordan inverse in LDS, one barrier per column, took this
 * place: 138 us a filtering combine at n = 48 with it.
 */
template <int NT, bool FLOOR, class... R>
__device__ __forceinline__ void chol_forward(Lds<NT>& s, as_d4 (&M)[NT], int lim, const Who<NT>& me, as_d4 (&R1)[NT],
                                             R&... Rs) {
  double fl = 0.0;
  if (FLOOR) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
      if (me.w == i) {
        double d = 0.0;
#pragma unroll
        for (int g = 0; g < 4; ++g) d = 4 * g + me.lk == me.li ? M[i][g] : d;
        fl = fmax(2.2e-16 * rows_sum(d), 1e-290);
      }
  }
  auto each = [&](auto f) {
    f(R1);
    if constexpr (!Geo<NT>::SEP || sizeof...(Rs) == 0) {
      (f(Rs), ...);
      mfma_drain();
    } else {
      mfma_drain();
      if (me.mat) {
        (f(Rs), ...);
        mfma_drain();
      }
    }
  };
#pragma unroll
  for (int p = 0; p < NT; ++p) {
    as_d4 wt;
    if (me.w == p) {
      double a[4], t[4], pr[4], pc = 1.0;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        a[g] = M[p][g];
        t[g] = 4 * g + me.lk == me.li ? 1.0 : 0.0;
        pr[g] = 1.0;
      }
      chol_steps<FLOOR>(a, t, pr, pc, fl, lim - 16 * p, me.li, me.lk, std::make_integer_sequence<int, 16>{});
      const double sc = rsqrt_ulp(pc);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        wt[g] = t[g] * sc;
        M[p][g] = me.li >= 4 * g + me.lk ? a[g] * rsqrt_ulp(pr[g]) : 0.0;
        if (NT > 1) s.wt[g * 64 + me.lane] = wt[g];
      }
    }
    if (NT > 1) {
      sync<NT>();
#pragma unroll
      for (int g = 0; g < 4; ++g) wt[g] = s.wt[g * 64 + me.lane];
    }
    each([&](as_d4(&X)[NT]) { panel_solve<NT>(X[p], wt); });
    if (p + 1 < NT) {
      if (me.mat && me.w > p) {
        panel_solve<NT>(M[p], wt);
        mfma_drain();
#pragma unroll
        for (int g = 0; g < 4; ++g) s.tr[(me.w * 4 + g) * 64 + me.lane] = M[p][g];
      }
      sync<NT>();
#pragma unroll
      for (int r = p + 1; r < NT; ++r) {
        as_d4 t;
#pragma unroll
        for (int g = 0; g < 4; ++g) t[g] = -s.tr[(r * 4 + g) * 64 + me.lane];
        auto update = [&](as_d4(&X)[NT]) {
#pragma unroll
          for (int g = 0; g < 4; ++g) X[r] = as_mfma(t[g], X[p][g], X[r]);
        };
        each(update);
        if (me.mat && me.w >= r) {
          update(M);
          mfma_drain();
        }
      }
    }
  }
}

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

template <int NT>
__global__ void __launch_bounds__(Geo<NT>::THREADS) ka_prior(const AsProb* probs, uk_chain_t wch, const int32_t* m_obs,
                                                             AsModel md, int n, int mr) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Sh<NT> b0 = sh<NT>(s.b0), b1 = sh<NT>(s.b1);
  const AsProb pr = probs[blockIdx.x];
  const int64_t nn = (int64_t)n * n;
  as_d4 Lm[NT], et[NT]; /* information matrix; vector (vector waves) */
  zero<NT>(Lm);
  zero<NT>(et);
  for (int64_t t = 0; t <= pr.p; ++t) {
    const int64_t st = pr.s0 + t;
    if (t > 0) {
      /* predict: with Q = G G^T, W = G^{-1}, Y = W F, y = W c and Lam + Y^T Y =
       * H H^T, V = H^{-1} Y^T W, v = H^{-1} (eta - Y^T y):
       * Lam <- W^T W - V^T V, eta <- W^T y + V^T v */
      as_d4 M[NT], Y[NT], W[NT], y[NT], D[NT];
      load<NT, true>(M, md.Q + st * nn, n, n, n, me);
      add_diag<NT>(M, n, 16 * NT, me);
      load<NT, false>(Y, md.F + st * nn, n, n, n, me);
      zero<NT>(W);
      add_diag<NT>(W, 0, n, me);
      load_vec<NT>(y, md.c + st * n, n, me);
      chol_forward<NT, false>(s, M, n, me, y, Y, W);
      b0.put(Y, me);
      b1.put(W, me);
      sync<NT>();
      zero<NT>(D);
      if (me.mat) {
        tmul_n<NT>(b0, W, D, n, me); /* Y^T W */
        tmul_n<NT>(b0, Y, Lm, n, me);
        zero<NT>(M);
        tmul_n<NT>(b1, W, M, n, me); /* Q^{-1} */
      }
      as_d4 ey[NT];
      zero<NT>(ey);
      if (me.vec) {
        tmul_n<NT, -1>(b0, y, et, n, me);
        tmul_n<NT>(b1, y, ey, n, me);
      }
      add_diag<NT>(Lm, n, 16 * NT, me);
      chol_forward<NT, false>(s, Lm, n, me, et, D);
      b0.put(D, me);
      sync<NT>();
      if (me.mat) {
        tmul_n<NT, -1>(b0, D, M, n, me);
#pragma unroll
        for (int r = 0; r < NT; ++r) Lm[r] = M[r];
      }
      if (me.vec) {
        tmul_n<NT>(b0, et, ey, n, me);
#pragma unroll
        for (int r = 0; r < NT; ++r) et[r] = ey[r];
      }
      sync<NT>();
    }
    const int m = m_obs[st];
    if (m > 0) { /* update: Lam += C^T C, eta += C^T o (whitened) */
      as_d4 C[NT], o[NT];
      load<NT, false>(C, wch.C + st * nn, m, n, mr, me);
      load_vec<NT>(o, wch.o + st * n, m, me);
      b0.put(C, me);
      sync<NT>();
      if (me.mat) tmul_m<NT>(b0, C, Lm, m, me);
      if (me.vec) tmul_m<NT>(b0, o, et, m, me);
      sync<NT>();
    }
    if (t < pr.p) {
      if (me.mat) store<NT, true>(Lm, md.Lam + st * nn, n, me);
      if (me.vec) store_vec<NT>(et, md.eta + st * n, n, me);
    }
  }
  /* P_p = Lam^{-1} = W^T W, x_p = P_p eta = W^T (W eta) */
  const int64_t sp = pr.s0 + pr.p;
  as_d4 W[NT], P[NT], x[NT];
  zero<NT>(W);
  add_diag<NT>(W, 0, n, me);
  add_diag<NT>(Lm, n, 16 * NT, me);
  chol_forward<NT, false>(s, Lm, n, me, et, W);
  b0.put(W, me);
  sync<NT>();
  if (me.mat) {
    zero<NT>(P);
    tmul_n<NT>(b0, W, P, n, me);
    store<NT, true>(P, md.Pf + sp * nn, n, me);
  }
  if (me.vec) {
    zero<NT>(x);
    tmul_n<NT>(b0, et, x, n, me);
    store_vec<NT>(x, md.xf + sp * n, n, me);
  }
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
template <int NT>
__global__ void __launch_bounds__(Geo<NT>::THREADS, SCAN_OCC<NT>) ka_felem(const AsProb* probs, const int32_t* elem_prob, uk_chain_t wch,
                                                             const int32_t* m_obs, AsModel md, AsElems el, int n, int mr) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Sh<NT> b0 = sh<NT>(s.b0), b1 = sh<NT>(s.b1);
  const int64_t ge = blockIdx.x;
  const AsProb pr = probs[elem_prob[ge]];
  const int64_t t = ge - pr.e0 + pr.p + 1;
  const int64_t st = pr.s0 + t;
  const bool firstel = t == pr.p + 1;
  const int64_t nn = (int64_t)n * n;
  const int64_t spv = pr.s0 + pr.p;
  const int m = m_obs[st];

  as_d4 Q[NT], F[NT], c[NT], w1[NT];
  load<NT, true>(Q, md.Q + st * nn, n, n, n, me);
  load<NT, false>(F, md.F + st * nn, n, n, n, me);
  load_vec<NT>(c, md.c + st * n, n, me);
#pragma unroll
  for (int r = 0; r < NT; ++r) w1[r] = c[r];
  if (firstel) { /* Q1 = Q + F P F^T, m1 = F x + c */
    as_d4 Ft[NT], P[NT], x[NT], U[NT];
    load<NT, true>(Ft, md.F + st * nn, n, n, n, me);
    load<NT, true>(P, md.Pf + spv * nn, n, n, n, me);
    load_vec<NT>(x, md.xf + spv * n, n, me);
    b0.put(Ft, me);
    b1.put(P, me);
    sync<NT>();
    if (me.mat) {
      zero<NT>(U);
      tmul_n<NT>(b1, Ft, U, n, me);
      tmul_n<NT>(b0, U, Q, n, me);
    }
    if (me.vec) tmul_n<NT>(b0, x, w1, n, me);
    sync<NT>();
  }
  as_d4 J[NT], e[NT];
  zero<NT>(J);
  zero<NT>(e);
  if (m > 0) {
    as_d4 Ct[NT], S[NT], CQ[NT], CF[NT], y[NT];
    load<NT, true>(Ct, wch.C + st * nn, m, n, mr, me);
    load_vec<NT>(y, wch.o + st * n, m, me);
    b0.put(Ct, me);
    b1.put(Q, me);
    sync<NT>();
    zero<NT>(CQ);
    zero<NT>(CF);
    zero<NT>(S);
    if (me.mat) {
      tmul_n<NT>(b0, Q, CQ, n, me);
      tmul_n<NT>(b0, F, CF, n, me);
      as_d4 U[NT];
      zero<NT>(U);
      tmul_n<NT>(b1, Ct, U, n, me);               /* Q C^T */
      tmul_n<NT>(b0, U, S, n, me);       /* S = C Q C^T + I */
      add_diag<NT>(S, 0, 16 * NT, me);
    }
    if (me.vec) { /* column 0: o - C w1, the others: o - C c */
      as_d4 x[NT];
#pragma unroll
      for (int r = 0; r < NT; ++r)
#pragma unroll
        for (int g = 0; g < 4; ++g) x[r][g] = me.li == 0 ? double(w1[r][g]) : double(c[r][g]);
      tmul_n<NT, -1>(b0, x, y, n, me);
    }
    chol_forward<NT, false>(s, S, m, me, y, CQ, CF); /* CQ = Y_1, CF = Y_2 */
    b0.put(CQ, me);
    b1.put(CF, me);
    sync<NT>();
    if (me.mat) {
      tmul_m<NT, -1>(b0, CQ, Q, m, me);           /* Z = Q - Y_1^T Y_1 */
      if (!firstel) tmul_m<NT, -1>(b0, CF, F, m, me); /* A = F - Y_1^T Y_2 */
      tmul_m<NT>(b1, CF, J, m, me);               /* J = Y_2^T Y_2 */
    }
    if (me.vec) {
      tmul_m<NT>(b0, y, w1, m, me);               /* b = w1 + Y_1^T r (column 0) */
      tmul_m<NT>(b1, y, e, m, me);                /* e = Y_2^T rc (column 1) */
      spread<1>(e);
    }
  }
  if (me.mat) {
    if (firstel) zero<NT>(F);
    store<NT, false>(F, el.A + ge * nn, n, me);
    store<NT, true>(Q, el.Z + ge * nn, n, me);
    store<NT, true>(J, el.J + ge * nn, n, me);
  }
  if (me.vec) {
    store_vec<NT>(w1, el.b + ge * n, n, me);
    store_vec<NT>(e, el.e + ge * n, n, me);
  }
}

/* ------------------------------------------------------------------------ */
/* combines (c :889-1016, matlab :240-262)                                   */
/* ------------------------------------------------------------------------ */

/* The accumulator of a scan: its blocks' columns, and on the vector wave b and
 * e, which lie in A's and Z's registers where that wave holds no matrix. */
template <int NT, bool SEP = Geo<NT>::SEP>
struct Acc {
  as_d4 A[NT], Z[NT], J[NT], vb[NT], ve[NT];
  __device__ __forceinline__ as_d4 (&b())[NT] { return vb; }
  __device__ __forceinline__ as_d4 (&e())[NT] { return ve; }
};
template <int NT>
struct Acc<NT, true> {
  as_d4 A[NT], Z[NT], J[NT];
  __device__ __forceinline__ as_d4 (&b())[NT] { return A; }
  __device__ __forceinline__ as_d4 (&e())[NT] { return Z; }
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
 *   J = Y_1^T Y_2 + J_i. */
template <int NT>
__device__ __forceinline__ void filt_combine(Acc<NT>& a, Lds<NT>& s, const AsElems& el, int64_t g, int n,
                                             const Who<NT>& me) {
  constexpr bool SEP = Geo<NT>::SEP;
  const int64_t nn = (int64_t)n * n;
  Sh<NT> b0 = sh<NT>(s.b0), b1 = sh<NT>(s.b1);
  as_d4 B1[NT], T2[NT], x[NT]; /* x: vector wave */
  {
    as_d4 Jj[NT];
    if (me.mat) {
      load<NT, true>(Jj, el.J + g * nn, n, n, n, me);
      load<NT, true>(B1, el.A + g * nn, n, n, n, me); /* A_j^T */
    }
    if (me.vec) load_vec<NT>(x, el.e + g * n, n, me);
    b0.put(Jj, me);
  }
  sync<NT>();
  if (me.mat) {
    zero<NT>(T2);
    tmul_n<NT>(b0, a.A, T2, n, me); /* J_j A_i */
  }
  if (me.vec) { /* column 0: e_j; the others: e_j - J_j b_i */
    as_d4 u[NT];
#pragma unroll
    for (int r = 0; r < NT; ++r) u[r] = x[r];
    tmul_n<NT, -1>(b0, a.b(), u, n, me);
#pragma unroll
    for (int r = 0; r < NT; ++r)
#pragma unroll
      for (int h = 0; h < 4; ++h) x[r][h] = me.li == 0 ? double(x[r][h]) : double(u[r][h]);
  }
  if (me.mat) add_diag<NT>(a.Z, n, 16 * NT, me);
  as_d4 M[NT]; /* Z = L L^T, then N = G G^T (e is the vector wave's Z) */
#pragma unroll
  for (int r = 0; r < NT; ++r) M[r] = a.Z[r];
  if constexpr (SEP) chol_forward<NT, true>(s, M, n, me, a.A);
  else chol_forward<NT, true>(s, M, n, me, a.b(), a.A); /* L^{-1} A_i, L^{-1} b_i */
  b1.put_upper_t(M, me);
  sync<NT>();
  if (me.mat) {
    as_d4 Lc[NT], T[NT], C2[NT];
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      Lc[r] = as_d4{0.0, 0.0, 0.0, 0.0};
      if (r >= me.w) Lc[r] = b1.tile(r, me.w, me);
    }
    zero<NT>(T);
    tmul_n<NT>(b0, Lc, T, n, me); /* J_j L */
    zero<NT>(M);
    tmul_n<NT, 1, true>(b1, T, M, n, me);
    add_diag<NT>(M, 0, 16 * NT, me);  /* N */
    zero<NT>(C2);
    tmul_n<NT, 1, true>(b1, T2, C2, n, me);
    zero<NT>(T);
    tmul_n<NT, 1, true>(b1, B1, T, n, me);
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      T2[r] = C2[r]; /* L^T J_j A_i */
      B1[r] = T[r];  /* L^T A_j^T */
    }
  }
  if (me.vec) { /* column 0: L^{-1} b_i + L^T e_j; the others: L^T (e_j - J_j b_i) */
#pragma unroll
    for (int r = 0; r < NT; ++r)
#pragma unroll
      for (int h = 0; h < 4; ++h) a.b()[r][h] = me.li == 0 ? double(a.b()[r][h]) : 0.0;
    tmul_n<NT, 1, true>(b1, x, a.b(), n, me);
  }
  if constexpr (SEP) chol_forward<NT, false>(s, M, n, me, a.A, T2, B1); /* y_0 | y_1 and Y_1, Y_2, Y_b */
  else chol_forward<NT, false>(s, M, n, me, a.b(), a.A, T2, B1);
  if (me.mat) load<NT, true>(a.Z, el.Z + g * nn, n, n, n, me);
  as_d4 bn[NT];
  if (me.vec) load_vec<NT>(bn, el.b + g * n, n, me);
  b0.put(B1, me);
  b1.put(a.A, me);
  sync<NT>();
  if (me.mat) {
    tmul_n<NT>(b1, T2, a.J, n, me);
    tmul_n<NT>(b0, B1, a.Z, n, me);
#pragma unroll
    for (int r = 0; r < NT; ++r) T2[r] = a.A[r];
  }
  if (me.vec) {
    tmul_n<NT>(b0, a.b(), bn, n, me);
    spread<0>(bn);
    as_d4 y1[NT];
    zero<NT>(y1);
    tmul_n<NT>(b1, a.b(), y1, n, me);
    spread<1>(y1);
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      a.e()[r] += y1[r];
      a.b()[r] = bn[r];
    }
  }
  if (me.mat) {
    zero<NT>(a.A);
    tmul_n<NT>(b0, T2, a.A, n, me);
  }
  sync<NT>();
}

/* a <- a (x) element g, smoothing; a is the running suffix and g the next
 * earlier step: E = E_j E_i, g = E_j g_i + g_j, L = E_j L_i E_j^T + L_j. */
template <int NT>
__device__ __forceinline__ void smooth_combine(Acc<NT>& a, Lds<NT>& s, const AsElems& el, int64_t g, int n,
                                               const Who<NT>& me) {
  const int64_t nn = (int64_t)n * n;
  Sh<NT> b0 = sh<NT>(s.b0), b1 = sh<NT>(s.b1);
  as_d4 Et[NT], Lj[NT], gj[NT];
  if (me.mat) {
    load<NT, true>(Et, el.A + g * nn, n, n, n, me); /* E_j^T */
    load<NT, true>(Lj, el.Z + g * nn, n, n, n, me);
  }
  if (me.vec) load_vec<NT>(gj, el.b + g * n, n, me);
  b0.put(Et, me);
  b1.put(a.Z, me);
  sync<NT>();
  if (me.mat) {
    as_d4 U[NT];
    zero<NT>(U);
    tmul_n<NT>(b1, Et, U, n, me); /* L_i E_j^T */
    tmul_n<NT>(b0, U, Lj, n, me);
    zero<NT>(U);
    tmul_n<NT>(b0, a.A, U, n, me);
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      a.Z[r] = Lj[r];
      a.A[r] = U[r];
    }
  }
  if (me.vec) {
    tmul_n<NT>(b0, a.b(), gj, n, me);
#pragma unroll
    for (int r = 0; r < NT; ++r) a.b()[r] = gj[r];
  }
  sync<NT>();
}

template <int NT, bool FILT>
__device__ __forceinline__ void acc_load(Acc<NT>& a, const AsElems& el, int64_t g, int n, const Who<NT>& me) {
  const int64_t nn = (int64_t)n * n;
  if (me.mat) {
    load<NT, false>(a.A, el.A + g * nn, n, n, n, me);
    load<NT, true>(a.Z, el.Z + g * nn, n, n, n, me);
    if (FILT) load<NT, true>(a.J, el.J + g * nn, n, n, n, me);
  }
  if (me.vec) {
    load_vec<NT>(a.b(), el.b + g * n, n, me);
    if (FILT) load_vec<NT>(a.e(), el.e + g * n, n, me);
  }
}
template <int NT, bool FILT>
__device__ __forceinline__ void acc_store(const Acc<NT>& ac, const AsElems& el, int64_t g, int n, Who<NT> me) {
  Acc<NT>& a = const_cast<Acc<NT>&>(ac);
  asm volatile("" : "+s"(n), "+v"(me.li), "+v"(me.lk));
  const int64_t nn = (int64_t)n * n;
  if (me.mat) {
    store<NT, false>(a.A, el.A + g * nn, n, me);
    store<NT, true>(a.Z, el.Z + g * nn, n, me);
    if (FILT) store<NT, true>(a.J, el.J + g * nn, n, me);
  }
  if (me.vec) {
    store_vec<NT>(a.b(), el.b + g * n, n, me);
    if (FILT) store_vec<NT>(a.e(), el.e + g * n, n, me);
  }
}
/* n and the lane are opaque, so that the addresses and masks made from them are
 * made in each combine: kept over a chunk's loop they took a fifth of the
 * registers */
template <int NT, bool FILT>
__device__ __forceinline__ void combine(Acc<NT>& a, Lds<NT>& s, const AsElems& el, int64_t g, int n, Who<NT> me) {
  asm volatile("" : "+s"(n), "+v"(me.li), "+v"(me.lk), "+v"(me.lane));
  if constexpr (FILT) filt_combine<NT>(a, s, el, g, n, me);
  else smooth_combine<NT>(a, s, el, g, n, me);
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
template <int NT, bool FILT>
__global__ void __launch_bounds__(Geo<NT>::THREADS, SCAN_OCC<NT>) ka_scan_reduce(const Chunk* ch, AsElems el, AsElems tot,
                                                                               int n) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Acc<NT> a;
  const Chunk c = ch[blockIdx.x];
  acc_load<NT, FILT>(a, el, c.first, n, me);
#pragma unroll 1
  for (int i = 1; i < c.len; ++i) combine<NT, FILT>(a, s, el, c.first + (int64_t)i * c.dir, n, me);
  acc_store<NT, FILT>(a, tot, c.tot, n, me);
}

/* pass 2, one Hillis-Steele round over the chunk totals of every problem:
 * out[t] = in[t - d] (x) in[t] when rank >= d, else in[t]. */
template <int NT, bool FILT>
__global__ void __launch_bounds__(Geo<NT>::THREADS, SCAN_OCC<NT>) ka_scan_round(const Chunk* ch, AsElems in, AsElems out,
                                                                              int d, int n) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Acc<NT> a;
  const Chunk c = ch[blockIdx.x];
  const bool join = c.rank >= d;
  acc_load<NT, FILT>(a, in, join ? c.tot - d : c.tot, n, me);
  if (join) combine<NT, FILT>(a, s, in, c.tot, n, me);
  acc_store<NT, FILT>(a, out, c.tot, n, me);
}

/* pass 3: every prefix within a chunk, seeded with the inclusive total of
 * the chunk before it; results overwrite the elements in place. */
template <int NT, bool FILT>
__global__ void __launch_bounds__(Geo<NT>::THREADS, SCAN_OCC<NT>) ka_scan_down(const Chunk* ch, AsElems el, AsElems tot,
                                                                             int n) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Acc<NT> a;
  const Chunk c = ch[blockIdx.x];
  const int i0 = c.rank == 0 ? 1 : 0;
  if (i0) acc_load<NT, FILT>(a, el, c.first, n, me);
  else acc_load<NT, FILT>(a, tot, c.tot - 1, n, me);
#pragma unroll 1
  for (int i = i0; i < c.len; ++i) {
    const int64_t g = c.first + (int64_t)i * c.dir;
    combine<NT, FILT>(a, s, el, g, n, me);
    acc_store<NT, FILT>(a, el, g, n, me);
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
template <int NT>
__global__ void __launch_bounds__(Geo<NT>::THREADS, SCAN_OCC<NT>) ka_selem(const AsProb* probs, const int32_t* step_prob, AsModel md,
                                                             AsElems el, int n) {
  __shared__ Lds<NT> s;
  const Who<NT> me;
  Sh<NT> b0 = sh<NT>(s.b0), b1 = sh<NT>(s.b1);
  const int64_t st = blockIdx.x;
  const AsProb pr = probs[step_prob[st]];
  const int64_t t = st - pr.s0;
  const int64_t nn = (int64_t)n * n;
  double* E = el.A + st * nn;
  double* gv = el.b + st * n;
  double* Lo = el.Z + st * nn;
  if (t == pr.k - 1) {
    for (int idx = threadIdx.x; idx < n * n; idx += Geo<NT>::THREADS) {
      E[idx] = 0.0;
      Lo[idx] = md.Pf[st * nn + idx];
    }
    for (int i = threadIdx.x; i < n; i += Geo<NT>::THREADS) gv[i] = md.xf[st * n + i];
    return;
  }
  const double* F = md.F + (st + 1) * nn;
  as_d4 M[NT], Y[NT], W[NT], y[NT], D[NT], P[NT], x[NT];
  load<NT, true>(M, md.Q + (st + 1) * nn, n, n, n, me);
  load_vec<NT>(y, md.c + (st + 1) * n, n, me);
  zero<NT>(W);
  add_diag<NT>(W, 0, n, me);
  zero<NT>(D);
  if (t >= pr.p) {
    load<NT, true>(P, md.Pf + st * nn, n, n, n, me);
    load<NT, true>(D, F, n, n, n, me); /* F^T */
    load_vec<NT>(x, md.xf + st * n, n, me);
    b0.put(D, me);
    b1.put(P, me);
    sync<NT>();
    zero<NT>(Y);
    if (me.mat) {
      tmul_n<NT>(b0, P, Y, n, me);              /* Y = F P */
      as_d4 U[NT];
      zero<NT>(U);
      tmul_n<NT>(b1, D, U, n, me);              /* U = P F^T */
      tmul_n<NT>(b0, U, M, n, me);     /* M = F P F^T + Q = G G^T */
    }
    if (me.vec) tmul_n<NT>(b0, x, y, n, me);    /* y = F x + c */
    add_diag<NT>(M, n, 16 * NT, me);
    chol_forward<NT, false>(s, M, n, me, y, Y, W); /* Y = G^{-1} F P, W = G^{-1}, y = G^{-1} (F x + c) */
    b0.put(Y, me);
    sync<NT>();
    if (me.mat) {
      zero<NT>(D);
      tmul_n<NT>(b0, W, D, n, me);
      store<NT, false>(D, E, n, me);          /* E = Y^T W */
      tmul_n<NT, -1>(b0, Y, P, n, me);
      store<NT, true>(P, Lo, n, me);          /* L = P - Y^T Y */
    }
    if (me.vec) {
      tmul_n<NT, -1>(b0, y, x, n, me);
      store_vec<NT>(x, gv, n, me);            /* g = x - E (F x + c) */
    }
  } else {
    load<NT, false>(Y, F, n, n, n, me);
    load<NT, true>(P, md.Lam + st * nn, n, n, n, me);
    load_vec<NT>(x, md.eta + st * n, n, me);
    add_diag<NT>(M, n, 16 * NT, me);
    chol_forward<NT, false>(s, M, n, me, y, Y, W); /* Q = G G^T: Y = G^{-1} F, W = G^{-1}, y = G^{-1} c */
    b0.put(Y, me);
    sync<NT>();
    if (me.mat) {
      tmul_n<NT>(b0, W, D, n, me);              /* D = F^T Q^{-1} */
      tmul_n<NT>(b0, Y, P, n, me);              /* P = Lam + F^T Q^{-1} F = H H^T */
    }
    if (me.vec) tmul_n<NT, -1>(b0, y, x, n, me); /* x = eta - F^T Q^{-1} c */
    add_diag<NT>(P, n, 16 * NT, me);
    zero<NT>(W);
    add_diag<NT>(W, 0, n, me);
    chol_forward<NT, false>(s, P, n, me, x, W, D); /* W = H^{-1}, D = H^{-1} F^T Q^{-1}, x = H^{-1} x */
    b0.put(W, me);
    sync<NT>();
    if (me.mat) {
      zero<NT>(M);
      tmul_n<NT>(b0, W, M, n, me);
      store<NT, true>(M, Lo, n, me);          /* L = W^T W */
      zero<NT>(M);
      tmul_n<NT>(b0, D, M, n, me);
      store<NT, false>(M, E, n, me);          /* E = L F^T Q^{-1} */
    }
    if (me.vec) {
      zero<NT>(y);
      tmul_n<NT>(b0, x, y, n, me);
      store_vec<NT>(y, gv, n, me);            /* g = L x */
    }
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
extern "C" std::shared_ptr<void>* uk_batch_assoc_plan(ukhip_batch* b);
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

/* Chunks aimed at over a batch: as many as the scan's workgroups that are
 * resident at once (two per CU at n = 33 .. 48, one above, ten single waves for
 * n <= 16). More would only add to the rounds over the chunk totals. Chunks
 * have at least 4 elements. */
template <int NB>
constexpr int64_t CHUNKS_TARGET = NB <= 16 ? 2560 : (NB <= 32 ? 768 : (NB <= 48 ? 512 : 256));

/* What a smoothing needs to know besides the inputs' values: fixed by a batch's
 * lengths and observation counts, made by its first associative smoothing and
 * kept with it, like the level tables of the odd-even path, so that a smoothing
 * is launches only and the parts of a composite batch overlap. (Eight problems
 * with n = 3 .. 16 in five parts: 2.70 ms when every smoothing downloaded the
 * counts, made and uploaded the tables and waited for them, 1.97 ms now.) */
struct AsPlan {
  std::vector<AsProb> probs;
  std::vector<int32_t> elem_prob, step_prob;
  std::vector<Chunk> fch, sch;
  std::vector<char> tab;  /* the tables as uploaded */
  int64_t ne = 0, ftot = 0, stot = 0, maxr_f = 0, maxr_s = 0;
  size_t o_model = 0, o_fe = 0, o_ft[2] = {0, 0}, o_se = 0, o_st[2] = {0, 0}, o_tab = 0, need = 0;
  size_t t_elem = 0, t_step = 0, t_fch = 0, t_sch = 0; /* offsets in tab */
};

template <int NB>
bool make_plan(AsPlan& pl, int64_t S, int nprob, const int64_t* kk, int n, const int32_t* m_obs) {
  /* p of every problem from the observation counts */
  std::vector<int32_t> m_h(S);
  if (!ok(hipMemcpy(m_h.data(), m_obs, S * sizeof(int32_t), hipMemcpyDeviceToHost), "download m")) return false;
  pl.probs.resize(nprob);
  pl.step_prob.resize(S);
  int64_t s0 = 0;
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
      return false;
    }
    pr.p = pp;
    pr.e0 = pl.ne;
    for (int64_t t = pr.p + 1; t < pr.k; ++t) pl.elem_prob.push_back(p);
    pl.ne += pr.k - pr.p - 1;
    for (int64_t t = 0; t < pr.k; ++t) pl.step_prob[s0 + t] = p;
    pl.probs[p] = pr;
    s0 += pr.k;
  }
  const int64_t fchunk = std::max<int64_t>(4, (pl.ne + CHUNKS_TARGET<NB> - 1) / CHUNKS_TARGET<NB>);
  const int64_t schunk = std::max<int64_t>(4, (S + CHUNKS_TARGET<NB> - 1) / CHUNKS_TARGET<NB>);
  for (int p = 0; p < nprob; ++p) {
    const int64_t len = pl.probs[p].k - pl.probs[p].p - 1;
    if (len > 0) pl.maxr_f = std::max(pl.maxr_f, make_chunks(pl.fch, pl.probs[p].e0, len, +1, fchunk, pl.ftot));
    pl.maxr_s = std::max(pl.maxr_s, make_chunks(pl.sch, pl.probs[p].s0, pl.probs[p].k, -1, schunk, pl.stot));
  }

  /* workspace */
  const size_t nn = (size_t)n * n;
  auto take = [&](size_t bytes) {
    const size_t r = pl.need;
    pl.need += (bytes + 255) & ~(size_t)255;
    return r;
  };
  auto elem_bytes = [&](int64_t cnt, bool filt) { return (size_t)std::max<int64_t>(cnt, 1) * ((filt ? 3 : 2) * nn + (filt ? 2 : 1) * n) * 8; };
  pl.o_model = take((size_t)S * (4 * nn + 4 * n) * 8);
  pl.o_fe = take(elem_bytes(pl.ne, true));
  for (auto& o : pl.o_ft) o = take(elem_bytes(pl.ftot, true));
  pl.o_se = take(elem_bytes(S, false));
  for (auto& o : pl.o_st) o = take(elem_bytes(pl.stot, false));

  /* tables */
  auto put = [&](const void* src, size_t bytes) {
    const size_t at_ = pl.tab.size();
    pl.tab.resize(at_ + ((bytes + 255) & ~(size_t)255), 0);
    if (bytes) std::memcpy(pl.tab.data() + at_, src, bytes);
    return at_;
  };
  put(pl.probs.data(), pl.probs.size() * sizeof(AsProb));
  pl.t_elem = put(pl.elem_prob.data(), pl.elem_prob.size() * 4);
  pl.t_step = put(pl.step_prob.data(), pl.step_prob.size() * 4);
  pl.t_fch = put(pl.fch.data(), pl.fch.size() * sizeof(Chunk));
  pl.t_sch = put(pl.sch.data(), pl.sch.size() * sizeof(Chunk));
  pl.o_tab = take(pl.tab.size());
  return true;
}

/* Enqueues the associative smoothing of one batch on st. */
template <int NB>
int run_assoc(ukhip_batch* b, hipStream_t st) {
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
  const size_t nn = (size_t)n * n;

  std::shared_ptr<void>& kept = *uk_batch_assoc_plan(b);
  if (!kept) {
    auto made = std::make_shared<AsPlan>();
    if (!make_plan<NB>(*made, S, nprob, kk, n, m_obs)) return -1;
    if (!ok(hipMalloc(&ws, made->need), "hipMalloc(associative workspace)")) return -1;
    uk_batch_set_assoc_ws(b, ws, made->need);
    kept = made; /* its host tables outlive the upload */
    if (!ok(hipMemcpyAsync((char*)ws + made->o_tab, made->tab.data(), made->tab.size(), hipMemcpyHostToDevice, st),
            "upload scan tables")) {
      kept.reset();
      (void)hipFree(ws);
      uk_batch_set_assoc_ws(b, nullptr, 0);
      return -1;
    }
  }
  const AsPlan& pl = *std::static_pointer_cast<AsPlan>(kept);
  char* W = (char*)ws;
  AsModel md;
  {
    double* q = (double*)(W + pl.o_model);
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
  const int64_t ne = pl.ne, maxr_f = pl.maxr_f, maxr_s = pl.maxr_s;
  const AsElems fe = elems_at(pl.o_fe, ne, true);
  const AsElems ft[2] = {elems_at(pl.o_ft[0], pl.ftot, true), elems_at(pl.o_ft[1], pl.ftot, true)};
  const AsElems se = elems_at(pl.o_se, S, false);
  const AsElems stt[2] = {elems_at(pl.o_st[0], pl.stot, false), elems_at(pl.o_st[1], pl.stot, false)};
  const char* T = W + pl.o_tab;
  const AsProb* d_probs = (const AsProb*)T;
  const int32_t* d_elem_prob = (const int32_t*)(T + pl.t_elem);
  const int32_t* d_step_prob = (const int32_t*)(T + pl.t_step);
  const Chunk* d_fch = (const Chunk*)(T + pl.t_fch);
  const Chunk* d_sch = (const Chunk*)(T + pl.t_sch);

  constexpr int NT = NB / 16;
  const dim3 blk(AT<NB>), tblk(Geo<NT>::THREADS);
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
  ka_prior<NT><<<dim3((unsigned)nprob), tblk, 0, st>>>(d_probs, wch, m_obs, md, n, mr);
  mark(UKHIP_AS_PRIOR, 1);
  if (ne > 0) {
    const unsigned nc = (unsigned)pl.fch.size();
    ka_felem<NT><<<dim3((unsigned)ne), tblk, 0, st>>>(d_probs, d_elem_prob, wch, m_obs, md, fe, n, mr);
    mark(UKHIP_AS_FELEM, 1);
    ka_scan_reduce<NT, true><<<dim3(nc), tblk, 0, st>>>(d_fch, fe, ft[0], n);
    int cur = 0, rounds = 0;
    for (int64_t d = 1; d < maxr_f; d <<= 1) {
      ka_scan_round<NT, true><<<dim3(nc), tblk, 0, st>>>(d_fch, ft[cur], ft[cur ^ 1], (int)d, n);
      cur ^= 1;
      ++rounds;
    }
    ka_scan_down<NT, true><<<dim3(nc), tblk, 0, st>>>(d_fch, fe, ft[cur], n);
    mark(UKHIP_AS_FSCAN, 2 + rounds);
    ka_filtered<NB><<<dim3((unsigned)ne), blk, 0, st>>>(d_probs, d_elem_prob, fe, md, n);
    mark(UKHIP_AS_FILTERED, 1);
  } else {
    mark(UKHIP_AS_FELEM, 0);
    mark(UKHIP_AS_FSCAN, 0);
    mark(UKHIP_AS_FILTERED, 0);
  }
  {
    const unsigned nc = (unsigned)pl.sch.size();
    ka_selem<NT><<<dim3((unsigned)S), tblk, 0, st>>>(d_probs, d_step_prob, md, se, n);
    mark(UKHIP_AS_SELEM, 1);
    ka_scan_reduce<NT, false><<<dim3(nc), tblk, 0, st>>>(d_sch, se, stt[0], n);
    int cur = 0, rounds = 0;
    for (int64_t d = 1; d < maxr_s; d <<= 1) {
      ka_scan_round<NT, false><<<dim3(nc), tblk, 0, st>>>(d_sch, stt[cur], stt[cur ^ 1], (int)d, n);
      cur ^= 1;
      ++rounds;
    }
    ka_scan_down<NT, false><<<dim3(nc), tblk, 0, st>>>(d_sch, se, stt[cur], n);
    mark(UKHIP_AS_SSCAN, 2 + rounds);
    ka_results<NB><<<dim3((unsigned)S), blk, 0, st>>>(se, xout, Sout, n);
    mark(UKHIP_AS_RESULTS, 1);
  }
  if (!ok(hipGetLastError(), "associative launches")) return -1;
  if (tm) {
    if (!ok(hipStreamSynchronize(st), "associative smoothing")) return -1;
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
extern "C" int uk_assoc_smooth(struct ukhip_batch* b, uint32_t options, hipStream_t st) {
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
    case 16: return run_assoc<16>(b, st);
    case 32: return run_assoc<32>(b, st);
    case 48: return run_assoc<48>(b, st);
    case 64: return run_assoc<64>(b, st);
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
  const int rc = uk_assoc_smooth(b, options, (hipStream_t)ukhip_stream());
  t_timer = nullptr;
  for (auto& e : tm.ev) (void)hipEventDestroy(e);
  if (rc != 0) return rc;
  for (int i = 0; i < UKHIP_AS_SLOTS; ++i) {
    if (ms) ms[i] += tm.ms[i];
    if (launches) launches[i] += tm.launches[i];
  }
  return 0;
}
