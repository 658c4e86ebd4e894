// Walker re-orthogonalisation (FP64): phi_s = Q_s R_s with diag(R_s) > 0.
//
// ipie's CPU path (ipie/walkers/uhf_walkers.py:108-143) takes LAPACK's
// economic QR and multiplies Q by sign(diag R), i.e. it returns the unique Q
// whose R has a positive real diagonal.  Here the same Q is produced by
// Cholesky-QR, which maps onto per-row independent work:
//   G = X^H X (+ shift),  G = R^H R,  X <- X R^{-1},
// as sweeps over the rows of X on FP64 MFMA: the Gram matrix of pass p + 1 is
// formed from the rows of X R_p^{-1} while they are written.
// Walkers with at most 48 columns that take the first branch below, that is all but
// ill-conditioned ones, run in reortho_fast_kernel, the others in reortho_kernel.  In
// mixed precision the walkers are rounded to pairs of BF16 values next, so that another
// order of the sums, which moves their last bits, would move a walker by 1e-6 now and
// then (k_greens_lu.hip): there the fast kernel factors in reortho_kernel's order.
//   - CholeskyQR2 (two passes, three sweeps; Yamamoto, Nakatsukasa, Yanagisawa,
//     Fukaya, ETNA 44 (2015) 306) when the unshifted Cholesky of X^H X succeeds
//     and 8 kappa sqrt(N n u + n (n + 1) u) <= 1/2 with kappa bounded by
//     ||R||_F ||R^-1||_F >= kappa_2(X): then Q is orthogonal to O(u).  Walkers
//     re-orthogonalised every few steps are far inside this bound.
//   - otherwise shifted CholeskyQR3 (a shifted pass, then CholeskyQR2; Fukaya,
//     Kannan, Nakatsukasa, Yamamoto, Yanagisawa, SIAM J. Sci. Comput. 42
//     (2020) A477), as accurate as Householder QR for any numerically
//     full-rank walker: the Gram matrix is formed again (the unshifted
//     attempt overwrote it), then three passes and four sweeps.
// log det R = sum over passes of sum_i log R_ii, and
//   detR = exp(log det R_a + log det R_b - detR_shift),
//   log_detR += log detR,  ovlp /= detR.
#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

constexpr int QR_THREADS = 256;
constexpr int QR_WAVES = QR_THREADS / 64;

__device__ double2 qr_zero;  // source of values past a matrix

// Row stride of G and Ri for at most 16 NT columns.
__host__ __device__ inline int qr_ld(int nt) { return 16 * nt + 1; }

// One sweep over the rows of X [N][n] (n <= 16 NT) in 16-row tiles, tile t on
// wave t % 4, on FP64 MFMA (16 x 16 x 4).  With Ri (upper triangular, zero
// rows and columns from n to 16 NT, row stride ldr) the rows are replaced by
// Y = X Ri in place; with G the Gram matrix Y^H Y (Y = X without Ri) is formed
// in G's upper triangle (row stride ldg) and its trace returned.  The
// accumulator register r of a Y tile holds row 4 r + lane / 16, column
// lane % 16, which is the A / B operand layout of K step r over those rows, so
// the Gram product takes Y straight from the registers.  The waves' partial
// Gram matrices are added into G in wave order (reproducible sums).
template <int NT>
__device__ double qr_sweep(double* __restrict__ X, int N, int n, const cplx* Ri, int ldr, cplx* G, int ldg) {
  constexpr int NPAIR = NT * (NT + 1) / 2;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  v4d gr[NPAIR], gi[NPAIR];
#pragma unroll
  for (int p = 0; p < NPAIR; ++p) {
    gr[p] = zero4d();
    gi[p] = zero4d();
  }
  const int ntile = (N + 15) / 16;
  for (int t = wave; t < ntile; t += QR_WAVES) {
    const int m0 = 16 * t;
    v4d yr[NT], yi[NT];
    if (Ri) {
#pragma unroll
      for (int J = 0; J < NT; ++J) {
        yr[J] = zero4d();
        yi[J] = zero4d();
      }
      const int mrow = m0 + l16;  // A operand: X[mrow][k0 + q]
#pragma unroll
      for (int k0 = 0; k0 < 16 * NT; k0 += 4) {
        const int k = k0 + q;
        const cplx x = (mrow < N && k < n) ? ld(X, (int64_t)mrow * n + k) : cmake(0.0, 0.0);
#pragma unroll
        for (int J = 0; J < NT; ++J) {
          if (k0 < 16 * (J + 1)) {  // Ri is upper triangular
            const cplx r = Ri[k * ldr + 16 * J + l16];
            yr[J] = mfma64(x.re, r.re, yr[J]);
            yr[J] = mfma64(-x.im, r.im, yr[J]);
            yi[J] = mfma64(x.re, r.im, yi[J]);
            yi[J] = mfma64(x.im, r.re, yi[J]);
          }
        }
      }
#pragma unroll
      for (int J = 0; J < NT; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + 4 * r + q, col = 16 * J + l16;
          if (row < N && col < n) st(X, (int64_t)row * n + col, cmake(yr[J][r], yi[J][r]));
        }
    } else {
#pragma unroll
      for (int J = 0; J < NT; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + 4 * r + q, col = 16 * J + l16;
          const cplx v = (row < N && col < n) ? ld(X, (int64_t)row * n + col) : cmake(0.0, 0.0);
          yr[J][r] = v.re;
          yi[J][r] = v.im;
        }
    }
    if (G) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int p = 0;
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int J = I; J < NT; ++J, ++p) {
            // G_IJ += conj(Y_I)^T Y_J over rows 4 r .. 4 r + 3 of the tile
            gr[p] = mfma64(yr[I][r], yr[J][r], gr[p]);
            gr[p] = mfma64(yi[I][r], yi[J][r], gr[p]);
            gi[p] = mfma64(yr[I][r], yi[J][r], gi[p]);
            gi[p] = mfma64(-yi[I][r], yr[J][r], gi[p]);
          }
      }
    }
  }
  if (!G) {
    __syncthreads();
    return 0.0;
  }
  for (int w = 0; w < QR_WAVES; ++w) {
    if (wave == w) {
      int p = 0;
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = I; J < NT; ++J, ++p)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * r + q, j = 16 * J + l16;
            if (i < n && j < n && j >= i) {
              const cplx v = cmake(gr[p][r], gi[p][r]);
              G[i * ldg + j] = w == 0 ? v : cadd(G[i * ldg + j], v);
            }
          }
    }
    __syncthreads();
  }
  double tr = 0.0;
  for (int i = 0; i < n; ++i) tr += G[i * ldg + i].re;
  return tr;
}

// In-place upper Cholesky G = R^H R (R in the upper triangle of G), one barrier
// per step: step k updates the trailing block with the unscaled row k
// (G_ij -= conj(G_ki) G_kj / G_kk) while row k - 1 is scaled by 1 / R_{k-1,k-1}.
// Returns sum_i log R_ii, or NaN if G is not numerically positive definite.
__device__ double qr_cholesky(cplx* G, int ldg, int n) {
  const int tid = threadIdx.x;
  double logdet = 0.0, dprev = 0.0;
  for (int k = 0; k <= n; ++k) {
    if (k > 0) {
      const double inv = 1.0 / dprev;
      for (int j = k + tid; j < n; j += QR_THREADS) G[(k - 1) * ldg + j] = cscale(G[(k - 1) * ldg + j], inv);
      if (tid == 0) G[(k - 1) * ldg + k - 1] = cmake(dprev, 0.0);
    }
    if (k == n) break;
    const double dkk = G[k * ldg + k].re;  // the same value in every thread
    if (!(dkk > 0.0)) {
      __syncthreads();
      return NAN;
    }
    const double d = sqrt(dkk), idkk = 1.0 / dkk;
    logdet += log(d);
    // trailing block: thread (tid / 16, tid % 16) takes rows k + 1 + tid / 16 + 16 a, columns
    // k + 1 + tid % 16 + 16 b (no integer division)
    for (int i = k + 1 + (tid >> 4); i < n; i += QR_THREADS / 16) {
      const cplx gki = G[k * ldg + i];
      int j = k + 1 + (tid & 15);
      if (j < i) j += (i - j + 15) / 16 * 16;  // first column >= i of this thread's residue class
      for (; j < n; j += 16) {
        const cplx gkj = G[k * ldg + j];
        cplx g = G[i * ldg + j];
        g.re -= (gki.re * gkj.re + gki.im * gkj.im) * idkk;
        g.im -= (gki.re * gkj.im - gki.im * gkj.re) * idkk;
        G[i * ldg + j] = g;
      }
    }
    dprev = d;
    __syncthreads();
  }
  __syncthreads();
  return logdet;
}

// ||R||_F ||R^{-1}||_F from the upper triangles (an upper bound of kappa_2(R)),
// the same value in every thread (fixed-order sums).
__device__ double qr_kappa_f(const cplx* R, const cplx* Ri, int ld, int n) {
  __shared__ double part[2][QR_WAVES];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double a = 0.0, b = 0.0;
  for (int e = threadIdx.x; e < n * n; e += QR_THREADS) {
    const int i = e / n, j = e % n;
    if (j >= i) {
      const cplx r = R[i * ld + j], x = Ri[i * ld + j];
      a += r.re * r.re + r.im * r.im;
      b += x.re * x.re + x.im * x.im;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_down(a, off, 64);
    b += __shfl_down(b, off, 64);
  }
  if (lane == 0) {
    part[0][wave] = a;
    part[1][wave] = b;
  }
  __syncthreads();
  double sa = 0.0, sb = 0.0;
  for (int w = 0; w < QR_WAVES; ++w) {
    sa += part[0][w];
    sb += part[1][w];
  }
  __syncthreads();  // part is rewritten by the next call
  return sqrt(sa * sb);
}

// Ri = R^{-1} (upper triangular, zero below and in the padding rows and
// columns up to np), one column per thread.
__device__ void qr_upper_inverse(const cplx* R, int ldr, int n, int np, cplx* Ri, int ldi) {
  const int j = threadIdx.x;
  if (j < np) {
    for (int i = np - 1; i > j || (j >= n && i >= 0); --i) Ri[i * ldi + j] = cmake(0.0, 0.0);
  }
  if (j < n) {
    for (int i = j; i >= 0; --i) {
      // four independent partial sums, loads issued four at a time
      cplx s4[4] = {cmake(i == j ? 1.0 : 0.0, 0.0), cmake(0.0, 0.0), cmake(0.0, 0.0), cmake(0.0, 0.0)};
      int k = i + 1;
      for (; k + 3 <= j; k += 4) {
        cplx r[4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          r[u] = R[i * ldr + k + u];
          x[u] = Ri[(k + u) * ldi + j];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          s4[u].re -= r[u].re * x[u].re - r[u].im * x[u].im;
          s4[u].im -= r[u].re * x[u].im + r[u].im * x[u].re;
        }
      }
      for (; k <= j; ++k) {
        const cplx r = R[i * ldr + k], x = Ri[k * ldi + j];
        s4[0].re -= r.re * x.re - r.im * x.im;
        s4[0].im -= r.re * x.im + r.im * x.re;
      }
      const cplx t = cadd(cadd(s4[0], s4[1]), cadd(s4[2], s4[3]));
      Ri[i * ldi + j] = cscale(t, 1.0 / R[i * ldr + i].re);
    }
  }
  __syncthreads();
}

// detR and what follows from it, from log det R of walker w.
__device__ void qr_finish(const ReorthoArgs& a, int w, double logdet) {
  const double shift = a.detR_shift ? a.detR_shift[w] : 0.0;
  const double detR = exp(logdet - shift);
  a.detR[w] = detR;
  if (a.log_detR) a.log_detR[w] += log(detR);
  if (a.ovlp) {
    const cplx o = ld(a.ovlp, w);
    st(a.ovlp, w, cmake(o.re / detR, o.im / detR));
  }
}

// ---------------------------------------------------------------- well-conditioned walkers
// CholeskyQR2 of both spins in one workgroup of four waves, the same sweeps as
// above with 256 registers a wave, so that two workgroups share a CU: one is in
// its sweeps (bound by the FP64 matrix pipe: 19200 MFMAs a walker at N = 400,
// n = 40, 131 us on a CU) while the other factors.  The factorisation, a serial chain
// that took most of the time column by column with a barrier each, is blocked by
// 16: a diagonal block is factored and inverted in one wave's registers (lane =
// column), the rest is 16 x 16 MFMA products, and the two spins' matrices run side
// by side on two waves each.  S holds one matrix per spin: the Gram matrix,
// then R, then R^-1, all in place, identity in the padding.
//   N = 400, n = 40, 1024 walkers: 0.91 ms against 2.54 ms in reortho_kernel; 12 walkers 278 us
//   against 557 us.
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Upper Cholesky D = R^H R of a 16 x 16 block and D <- R^-1 (zero below the
// diagonal); lane % 16 owns a column.  Adds this lane's log R_jj to logd; false
// (the same in every lane) if D is not numerically positive definite.
__device__ __forceinline__ bool qr_block_factor(cplx* D, int ld, double& logd) {
  const int l16 = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
  cplx c[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) c[i] = D[i * ld + l16];
  double diag = 1.0, inv = 1.0;  // R_jj and 1 / R_jj of this lane's column
  bool ok = true;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const double dkk = lane_value(c[k].re, k);
    ok = ok && dkk > 0.0;
    const double r = rsqrt(dkk);
    double d = dkk * r;
    d = fma(fma(-d, d, dkk), 0.5 * r, d);
    const cplx scaled = cscale(c[k], r);
    c[k].re = l16 == k ? d : scaled.re;
    c[k].im = l16 == k ? 0.0 : scaled.im;
    diag = l16 == k ? d : diag;
    inv = l16 == k ? r : inv;
#pragma unroll
    for (int i = k + 1; i < 16; ++i) {  // c_ij -= conj(R_ki) R_kj
      const double br = lane_value(c[k].re, i), bi = lane_value(c[k].im, i);
      c[i].re = fma(-br, c[k].re, c[i].re);
      c[i].re = fma(-bi, c[k].im, c[i].re);
      c[i].im = fma(-br, c[k].im, c[i].im);
      c[i].im = fma(bi, c[k].re, c[i].im);
    }
    // (the updates of a step before the next: the compiler would delay them and
    // keep every broadcast value)
    __builtin_amdgcn_sched_barrier(0);
  }
  logd += log(diag);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    c[i].re = l16 < i ? 0.0 : c[i].re;
    c[i].im = l16 < i ? 0.0 : c[i].im;
  }
  // X = R^-1 by rows from the last: X_ij = (delta_ij - sum_{k > i} R_ik X_kj) / R_ii
#pragma unroll
  for (int i = 15; i >= 0; --i) {
    cplx s0 = cmake(l16 == i ? 1.0 : 0.0, 0.0), s1 = cmake(0.0, 0.0);
#pragma unroll
    for (int k = i + 1; k < 16; ++k) {
      const double br = lane_value(c[i].re, k), bi = lane_value(c[i].im, k);
      cplx& t = (k & 1) ? s1 : s0;
      t.re = fma(-br, c[k].re, t.re);
      t.re = fma(bi, c[k].im, t.re);
      t.im = fma(-br, c[k].im, t.im);
      t.im = fma(-bi, c[k].re, t.im);
    }
    c[i] = cscale(cadd(s0, s1), lane_value(inv, i));
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if ((i & 3) == q) D[i * ld + l16] = c[i];
  return ok;
}

// acc += A B for 16 x 16 blocks in LDS; A read as stored, or conjugate transposed
// (HA); the result's register r of lane (q, l16) is element (4 r + q, l16), which is also
// the B operand of K step r.
struct QrAcc {
  v4d re, im;
};
template <bool HA>
__device__ __forceinline__ void qr_mma(const cplx* A, int ld, const cplx (&b)[4], QrAcc& acc) {
  const int l16 = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = 4 * r + q;
    cplx x = HA ? A[k * ld + l16] : A[l16 * ld + k];
    if (HA) x.im = -x.im;
    acc.re = mfma64(x.re, b[r].re, acc.re);
    acc.re = mfma64(-x.im, b[r].im, acc.re);
    acc.im = mfma64(x.re, b[r].im, acc.im);
    acc.im = mfma64(x.im, b[r].re, acc.im);
  }
}
__device__ __forceinline__ void qr_block_load(const cplx* B, int ld, cplx (&b)[4]) {
  const int l16 = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) b[r] = B[(4 * r + q) * ld + l16];
}
__device__ __forceinline__ void qr_block_store(cplx* B, int ld, const QrAcc& v, double scale) {
  const int l16 = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) B[(4 * r + q) * ld + l16] = cmake(scale * v.re[r], scale * v.im[r]);
}

// S_s <- R_s^-1 for every spin s < nspin (wave pair s), G = R^H R; log det R_s and
// whether the factorisation went through into logdet and ok.
template <int NT>
__device__ __forceinline__ void qr_factor(cplx* S, int nspin, double* logdet, int* ok) {
  constexpr int LD = 16 * NT + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), spin = wave >> 1, part = wave & 1;
  const int l16 = threadIdx.x & 15, q = (threadIdx.x & 63) >> 4;
  const bool mine = spin < nspin;
  cplx* G = S + spin * 16 * NT * LD;
  auto block = [&](int I, int J) { return G + 16 * I * LD + 16 * J; };
  double logd = 0.0;
  bool good = true;
#pragma unroll 1
  for (int b = 0; b < NT; ++b) {
    if (mine && part == 0) {
      const bool g = qr_block_factor(block(b, b), LD, logd);
      good = good && g;
    }
    __syncthreads();
    // the block row: R_bJ = (R_bb^-1)^H G_bJ
    for (int J = b + 1 + part; mine && J < NT; J += 2) {
      cplx x[4];
      qr_block_load(block(b, J), LD, x);
      QrAcc v{zero4d(), zero4d()};
      qr_mma<true>(block(b, b), LD, x, v);
      qr_block_store(block(b, J), LD, v, 1.0);
    }
    __syncthreads();
    // G_IJ -= R_bI^H R_bJ
    int t = 0;
    for (int I = b + 1; mine && I < NT; ++I)
      for (int J = I; J < NT; ++J, ++t) {
        if ((t & 1) != part) continue;
        cplx x[4];
        qr_block_load(block(b, J), LD, x);
        QrAcc v{zero4d(), zero4d()};
        qr_mma<true>(block(b, I), LD, x, v);
        cplx g[4];
        qr_block_load(block(I, J), LD, g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v.re[r] = g[r].re - v.re[r];
          v.im[r] = g[r].im - v.im[r];
        }
        qr_block_store(block(I, J), LD, v, 1.0);
      }
    __syncthreads();
  }
  // the inverse's block columns from the left, in place: T_K = R_KJ X_JJ, X_IJ = - sum_K X_IK T_K
#pragma unroll 1
  for (int J = 1; J < NT; ++J) {
    for (int K = part; mine && K < J; K += 2) {
      cplx x[4];
      qr_block_load(block(J, J), LD, x);
      QrAcc v{zero4d(), zero4d()};
      qr_mma<false>(block(K, J), LD, x, v);
      qr_block_store(block(K, J), LD, v, 1.0);
    }
    __syncthreads();
    QrAcc v[2] = {{zero4d(), zero4d()}, {zero4d(), zero4d()}};  // I = part, part + 2
#pragma unroll
    for (int u = 0; u < 2; ++u)
      for (int K = part + 2 * u; mine && K < J; ++K) {
        cplx x[4];
        qr_block_load(block(K, J), LD, x);
        qr_mma<false>(block(part + 2 * u, K), LD, x, v[u]);
      }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (mine && part + 2 * u < J) qr_block_store(block(part + 2 * u, J), LD, v[u], -1.0);
    __syncthreads();
  }
  if (mine && part == 0) {
    if (q != 0) logd = 0.0;
    for (int off = 8; off > 0; off >>= 1) logd += __shfl_xor(logd, off, 64);
    if (l16 == 0 && q == 0) {
      logdet[spin] = logd;
      ok[spin] = good;
    }
  }
  __syncthreads();
}

// The same in the order of the general kernel: every entry takes the operations of
// qr_cholesky and qr_upper_inverse one after the other (fused as the compiled code of
// those has them), log det R sums in the same order, so that a walker's bits are those of
// reortho_kernel.  A wave pair per spin side by side, rows through LDS; diag [nspin][16 NT]
// scratch.  Bound by the chain of n steps: N = 400, n = 40, 1024 walkers 1.11 ms and 12
// walkers 396 us, where the blocked form takes 0.91 and 278 and reortho_kernel 2.54 and 557.
// (Cholesky entries kept in registers and 16 columns x four partial sums a wave in the
// inverse: 1.07 ms and 344 us, in three times the code.)
template <int NT>
__device__ __forceinline__ void qr_factor_ordered(cplx* S, int nspin, int n0, int n1, double* diag, double* logdet,
                                                  int* ok) {
  constexpr int LD = 16 * NT + 1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), spin = wave >> 1, part = wave & 1;
  const int lane = threadIdx.x & 63, t = threadIdx.x & 127, ti = t >> 4, tj = t & 15;
  const int n = spin >= nspin ? 0 : spin == 0 ? n0 : n1, steps = nspin > 1 ? max(n0, n1) : n0;
  cplx* G = S + spin * 16 * NT * LD;
  diag += spin * 16 * NT;
  bool good = true;
  double dprev = 0.0;
#pragma unroll 1
  for (int k = 0; k <= steps; ++k) {
    if (k > 0 && k <= n && good) {  // row k - 1 is not read any more
      const double inv = 1.0 / dprev;
      if (k + t < n) G[(k - 1) * LD + k + t] = cscale(G[(k - 1) * LD + k + t], inv);
      if (t == 0) {
        G[(k - 1) * LD + k - 1] = cmake(dprev, 0.0);
        diag[k - 1] = dprev;
      }
    }
    if (k < n && good) {
      const double dkk = G[k * LD + k].re;  // the same value in every thread
      good = dkk > 0.0;
      if (good) {
        const double idkk = 1.0 / dkk;
        dprev = sqrt(dkk);
        for (int i = k + 1 + ti; i < n; i += 8) {
          const cplx gki = G[k * LD + i];
          int j = k + 1 + tj;
          if (j < i) j += (i - j + 15) / 16 * 16;  // first column >= i of this thread's residue class
          for (; j < n; j += 16) {
            const cplx gkj = G[k * LD + j], g = G[i * LD + j];
            const double re = fma(gki.re, gkj.re, gki.im * gkj.im), im = fma(gki.re, gkj.im, -(gki.im * gkj.re));
            G[i * LD + j] = cmake(fma(-idkk, re, g.re), fma(-idkk, im, g.im));
          }
        }
      }
    }
    __syncthreads();
  }
  if (good && part == 1) {
    const double lg = lane < n ? log(diag[lane]) : 0.0;
    double sum = 0.0;
    for (int k = 0; k < n; ++k) sum += lane_value(lg, k);
    if (lane == 0) logdet[spin] = sum;
  }
  // the inverse in place, rows from the last, lane = column: row i takes row i of R (read by
  // every lane of the wave before any writes) and the rows below of its own column
  if (good && part == 0) {
#pragma unroll 1
    for (int i = n - 1; i >= 0; --i) {
      const cplx* R = G + i * LD;
      const double rinv = 1.0 / R[i].re;
      if (lane >= i && lane < n) {
        cplx s[4] = {cmake(lane == i ? 1.0 : 0.0, 0.0), cmake(0.0, 0.0), cmake(0.0, 0.0), cmake(0.0, 0.0)};
        const auto less = [](cplx& v, cplx r, cplx x) {
          v.re -= fma(r.re, x.re, -(r.im * x.im));
          v.im -= fma(r.im, x.re, r.re * x.im);
        };
        int k = i + 1;
        for (; k + 3 <= lane; k += 4) {
          cplx r[4], x[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            r[u] = R[k + u];
            x[u] = G[(k + u) * LD + lane];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) less(s[u], r[u], x[u]);
        }
        for (; k <= lane; ++k) less(s[0], R[k], G[k * LD + lane]);
        G[i * LD + lane] = cscale(cadd(cadd(s[0], s[1]), cadd(s[2], s[3])), rinv);
      } else if (lane < i && lane / 16 == i / 16) {
        G[i * LD + lane] = cmake(0.0, 0.0);  // below the diagonal in its block
      }
    }
  }
  if (t == 0 && spin < nspin) ok[spin] = good;
  __syncthreads();
}

// The sweep of one matrix (as qr_sweep): APPLY replaces the rows by X S, GRAM leaves
// the Gram matrix of the (new) rows in S with identity padding and returns its
// trace.  A tile's 4 NT loads are in flight under the MFMAs before it; values past
// the matrix come from a zero line, so that nothing branches around a load.
template <int NT, bool APPLY, bool GRAM>
__device__ __forceinline__ double qr_fast_sweep(double* __restrict__ X, int N, int n, cplx* S, double* sums) {
  constexpr int LD = 16 * NT + 1, NPAIR = NT * (NT + 1) / 2;
  typedef double v2d __attribute__((ext_vector_type(2)));
  typedef const __attribute__((address_space(1))) v2d* gptr;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int ntile = (N + 15) / 16;
  const gptr zero = (gptr)(const void*)&qr_zero, base = (gptr)(const void*)X;
  v4d gr[GRAM ? NPAIR : 1], gi[GRAM ? NPAIR : 1], yr[NT], yi[NT];
  if (GRAM) {
#pragma unroll
    for (int p = 0; p < NPAIR; ++p) gr[p] = gi[p] = zero4d();
  }
  v2d x[4 * NT];
  // tile t: as the A operand of the product (row l16, column 4 u + q), or without it in
  // the accumulators' layout (row 4 r + q, column 16 J + l16; u = 4 J + r)
  auto fetch = [&](int t) {
#pragma unroll
    for (int u = 0; u < 4 * NT; ++u) {
      const int row = 16 * t + (APPLY ? l16 : 4 * (u & 3) + q), col = APPLY ? 4 * u + q : 16 * (u >> 2) + l16;
      const gptr p = base + (int64_t)row * n + col;
      x[u] = *(row < N && col < n ? p : zero);
    }
  };
  if (wave < ntile) fetch(wave);
#pragma unroll 1
  for (int t = wave; t < ntile; t += QR_WAVES) {
    if constexpr (APPLY) {
#pragma unroll
      for (int J = 0; J < NT; ++J) yr[J] = yi[J] = zero4d();
      int off = l16;  // (opaque: S would be held in registers over the tiles)
      asm volatile("" : "+v"(off));
#pragma unroll
      for (int u = 0; u < 4 * NT; ++u) {
        if (u % 4 == 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int J = u / 4; J < NT; ++J) {  // R^-1 is upper triangular
          const cplx r = S[(4 * u + q) * LD + 16 * J + off];
          yr[J] = mfma64(x[u][0], r.re, yr[J]);
          yr[J] = mfma64(-x[u][1], r.im, yr[J]);
          yi[J] = mfma64(x[u][0], r.im, yi[J]);
          yi[J] = mfma64(x[u][1], r.re, yi[J]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int J = 0; J < NT; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * t + 4 * r + q, col = 16 * J + l16;
          if (row < N && col < n) st(X, (int64_t)row * n + col, cmake(yr[J][r], yi[J][r]));
        }
    } else {
#pragma unroll
      for (int u = 0; u < 4 * NT; ++u) {
        yr[u >> 2][u & 3] = x[u][0];
        yi[u >> 2][u & 3] = x[u][1];
      }
    }
    if (t + QR_WAVES < ntile) fetch(t + QR_WAVES);
    if constexpr (GRAM) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int p = 0;
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int J = I; J < NT; ++J, ++p) {
            gr[p] = mfma64(yr[I][r], yr[J][r], gr[p]);
            gr[p] = mfma64(yi[I][r], yi[J][r], gr[p]);
            gi[p] = mfma64(yr[I][r], yi[J][r], gi[p]);
            gi[p] = mfma64(-yi[I][r], yr[J][r], gi[p]);
          }
      }
    }
  }
  __syncthreads();  // S has been read
  if constexpr (!GRAM) return 0.0;
  // the waves' sums in wave order; identity in the padding
#pragma unroll 1
  for (int w = 0; w < QR_WAVES; ++w) {
    if (wave == w) {
      int p = 0;
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = I; J < NT; ++J, ++p)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * r + q, j = 16 * J + l16;
            cplx v = cmake(gr[p][r], gi[p][r]);
            if (w > 0) v = cadd(v, S[i * LD + j]);
            if (w == QR_WAVES - 1 && i == j && i >= n) v = cmake(1.0, 0.0);
            S[i * LD + j] = v;
          }
    }
    __syncthreads();
  }
  return block_sum((int)threadIdx.x < n ? S[threadIdx.x * (LD + 1)].re : 0.0, sums);
}

template <int NT, bool ORDERED>
__global__ void __launch_bounds__(QR_THREADS, 2) reortho_fast_kernel(ReorthoArgs a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  constexpr int LD = 16 * NT + 1;
  extern __shared__ cplx smem[];
  __shared__ double logdet[2], sums[QR_WAVES], diag[ORDERED ? 2 * 16 * NT : 1];
  __shared__ int ok[2];
  cplx* S = smem;  // per spin [16 NT][LD]
  const int w = blockIdx.x, N = a.nbasis, nspin = a.nbeta > 0 ? 2 : 1;
  constexpr double u = 1.1102230246251565e-16;  // 2^-53
  double tr0 = 0.0, tr1 = 0.0;
#pragma unroll 1
  for (int s = 0; s < nspin; ++s) {
    const int n = s == 0 ? a.nalpha : a.nbeta;
    double* X = (s == 0 ? a.phia : a.phib) + 2 * (int64_t)w * N * n;
    (s == 0 ? tr0 : tr1) = qr_fast_sweep<NT, false, true>(X, N, n, S + s * 16 * NT * LD, sums);
  }
  double first[2] = {0.0, 0.0};  // log det R of the first pass
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {  // (one call site: the factorisation is inlined once)
    if constexpr (ORDERED) qr_factor_ordered<NT>(S, nspin, a.nalpha, a.nbeta, diag, logdet, ok);
    else qr_factor<NT>(S, nspin, logdet, ok);
    if (pass == 1) break;
    first[0] = logdet[0];
    if (nspin > 1) first[1] = logdet[1];
    bool slow = false;
    for (int s = 0; s < nspin; ++s) {
      const int n = s == 0 ? a.nalpha : a.nbeta;
      const double mn = (double)N * n + (double)n * (n + 1);
      // ||R^-1||_F^2 (||R||_F^2 is the Gram matrix's trace)
      double x2 = 0.0;
      for (int e = threadIdx.x; e < n * n; e += QR_THREADS) {
        const int i = e / n, j = e % n;
        if (j >= i) {
          const cplx x = S[s * 16 * NT * LD + i * LD + j];
          x2 += x.re * x.re + x.im * x.im;
        }
      }
      x2 = block_sum(x2, sums);
      slow = slow || !ok[s] || !(8.0 * sqrt((s == 0 ? tr0 : tr1) * x2) * sqrt(mn * u) <= 0.5);
    }
    if (threadIdx.x == 0) a.slow[w] = slow ? 1 : 0;
    if (slow) return;  // nothing written yet: reortho_kernel takes this walker
    __syncthreads();
#pragma unroll 1
    for (int s = 0; s < nspin; ++s) {
      const int n = s == 0 ? a.nalpha : a.nbeta;
      double* X = (s == 0 ? a.phia : a.phib) + 2 * (int64_t)w * N * n;
      qr_fast_sweep<NT, true, true>(X, N, n, S + s * 16 * NT * LD, sums);
    }
  }
  if (!ok[0] || (nspin > 1 && !ok[1])) {
    if (threadIdx.x == 0) {
      if (a.flags) atomicOr(a.flags, AFQMC_FLAG_CHOLESKY);
      if (a.wflags) atomicOr(a.wflags + w, AFQMC_FLAG_CHOLESKY);
      a.detR[w] = NAN;
    }
    return;
  }
#pragma unroll 1
  for (int s = 0; s < nspin; ++s) {
    const int n = s == 0 ? a.nalpha : a.nbeta;
    double* X = (s == 0 ? a.phia : a.phib) + 2 * (int64_t)w * N * n;
    qr_fast_sweep<NT, true, false>(X, N, n, S + s * 16 * NT * LD, sums);
  }
  if (threadIdx.x == 0) {
    double ld = first[0] + logdet[0];
    if (nspin > 1) ld = ORDERED ? ld + first[1] + logdet[1] : first[0] + first[1] + (logdet[0] + logdet[1]);
    qr_finish(a, w, ld);
  }
}

template <int NT>
__global__ void __launch_bounds__(QR_THREADS) reortho_kernel(ReorthoArgs a) {
  extern __shared__ cplx smem[];
  const int w = blockIdx.x;
  if (a.slow && !a.slow[w]) return;  // done by reortho_fast_kernel
  const int N = a.nbasis;
  const int ldg = qr_ld(NT);
  cplx* G = smem;                  // [16 NT][ldg]: Gram matrix, then R
  cplx* Ri = G + 16 * NT * ldg;    // [16 NT][ldg]: R^{-1}, zero padded
  const int nspin = a.nbeta > 0 ? 2 : 1;
  double logdet = 0.0;
  bool bad = false;
  constexpr double u = 1.1102230246251565e-16;  // 2^-53
  for (int s = 0; s < nspin; ++s) {
    const int n = s == 0 ? a.nalpha : a.nbeta;
    double* phi = (s == 0 ? a.phia : a.phib) + 2 * (int64_t)w * N * n;
    const double mn = (double)N * n + (double)n * (n + 1);
    // One loop, one call site per stage (the sweep is inlined once):
    //   apply: X <- X Ri in this sweep;  gram: form G = X^H X in it.
    // The first Gram pass is unshifted; if its Cholesky fails or R fails the
    // CholeskyQR2 bound, the Gram matrix is formed again and shifted.  Then
    // `left` apply + Gram passes (1 for CholeskyQR2, 2 after a shifted pass)
    // and a final apply.
    bool apply = false, gram = true, shifted = false;
    int left = 0;
    for (;;) {
      const double tr = qr_sweep<NT>(phi, N, n, apply ? Ri : nullptr, ldg, gram ? G : nullptr, ldg);
      if (!gram) break;
      if (shifted && !apply) {
        // shift = 11 (N n + n (n + 1)) u ||X||_F^2
        if (threadIdx.x == 0)
          for (int i = 0; i < n; ++i) G[i * ldg + i].re += 11.0 * mn * u * tr;
        __syncthreads();
      }
      const double ldr = qr_cholesky(G, ldg, n);
      const bool ok = ldr == ldr;  // the same in every thread
      if (ok) qr_upper_inverse(G, ldg, n, 16 * NT, Ri, ldg);
      if (!apply && !shifted && !(ok && 8.0 * qr_kappa_f(G, Ri, ldg, n) * sqrt(mn * u) <= 0.5)) {
        shifted = true;
        continue;
      }
      if (!ok) {
        bad = true;
        break;
      }
      logdet += ldr;
      left = apply ? left - 1 : (shifted ? 2 : 1);
      apply = true;
      gram = left > 0;
    }
    if (bad) break;
  }
  if (threadIdx.x == 0) {
    if (bad) {
      if (a.flags) atomicOr(a.flags, AFQMC_FLAG_CHOLESKY);
      if (a.wflags) atomicOr(a.wflags + w, AFQMC_FLAG_CHOLESKY);
      a.detR[w] = NAN;
      return;
    }
    qr_finish(a, w, logdet);
  }
}

}  // namespace

namespace {

template <int NT>
hipError_t launch_qr_nt(const ReorthoArgs& a, hipStream_t stream) {
  const size_t matrix = sizeof(cplx) * 16 * (size_t)NT * qr_ld(NT);
  hipError_t e = allow_lds((const void*)reortho_kernel<NT>, 2 * matrix);
  if (e != hipSuccess) return e;
  ReorthoArgs b = a;
  if constexpr (NT <= 3) {  // (64 columns do not fit the fast kernel's registers)
    const size_t lds = matrix * (a.nbeta > 0 ? 2 : 1);
    e = allow_lds(a.ordered ? (const void*)reortho_fast_kernel<NT, true> : (const void*)reortho_fast_kernel<NT, false>, lds);
    if (e != hipSuccess) return e;
    if (a.ordered)
      hipLaunchKernelGGL((reortho_fast_kernel<NT, true>), dim3(a.nwalkers), dim3(QR_THREADS), lds, stream, a);
    else
      hipLaunchKernelGGL((reortho_fast_kernel<NT, false>), dim3(a.nwalkers), dim3(QR_THREADS), lds, stream, a);
  } else {
    b.slow = nullptr;
    if (a.mark.acc && (e = launch_phase_mark(a.mark, stream)) != hipSuccess) return e;
  }
  hipLaunchKernelGGL(reortho_kernel<NT>, dim3(a.nwalkers), dim3(QR_THREADS), 2 * matrix, stream, b);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_reortho(const ReorthoArgs& a, hipStream_t stream) {
  const int nmax = a.nalpha > a.nbeta ? a.nalpha : a.nbeta;
  if (!a.slow) return hipErrorInvalidValue;
  switch ((nmax + 15) / 16) {
    case 1: return launch_qr_nt<1>(a, stream);
    case 2: return launch_qr_nt<2>(a, stream);
    case 3: return launch_qr_nt<3>(a, stream);
    case 4: return launch_qr_nt<4>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace afqmc
