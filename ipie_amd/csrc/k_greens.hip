// Batched single-determinant Green's function and overlap (FP64), one workgroup per
// walker, both spins side by side (each its own waves), no intermediate in memory:
//   O_s = phi_s^T conj(psi_s)    [n, n], v_mfma_f64_16x16x4f64 into LDS: a wave per
//                                16-row tile and K part, the parts added in order
//   det O_s, O_s^{-1}            columns dealt to the spin's waves (registers, lane =
//                                row), pivot rows chosen without moving them
//   ovlp                         phase_a phase_b exp(logdet_a + logdet_b - log_shift)
//   Ghalf_s = O_s^{-1} phi_s^T   [n, N], FP64 MFMA, a wave per 16 columns
// (Ghalf of the mixed step: k_greens_lu.hip.)
// Restates ipie/estimators/greens_function_single_det.py:62-154 and
// ipie/propagation/overlap.py:29-59.  All reductions are in a fixed order, so
// the result is bitwise reproducible run to run.
//
// Elimination: at step k the pivot row p is the unused row of the largest
// |re| + |im| of column k (to its high word, 20 bits; the first such row on ties) and
// every other row i has B[i][j] -= (B[i][k] / d) B[p][j], d = B[p][k].  For the overlap
// that is an LU: log|det| = sum log|d_k|, phase = prod d_k / |d_k| times the sign of
// the permutation k -> p_k, and only the columns after k are updated.  For the inverse
// (Gauss-Jordan) the used rows take part and column k becomes (B[i][k] / d, -1 in row p):
// row p_k then holds -d_k times row k of the inverse, its column j that of row p_j of O.
// Errors against 80-bit sums (n = 40, N = 400, trial orbitals with noise, rms): Ghalf
// 6.3e-16, overlap 1.9e-15 (LU and inverse from its factors: 6.7e-16 and 4.4e-15).
//
// What bounds it, by walkers: few (one workgroup a CU) the chain of n pivot steps, 0.6 us
// each (LDS hand-over of the pivot column, maximum over the rows, reciprocal, the
// updates of the owner's next column), and the MFMAs of one CU; many, VALU and MFMA
// work in turn, phi read once from HBM and once from the caches.  The owner of step
// k + 1 brings only its next column up to date before the step's barrier and the others
// after it.  Green's function + overlap of both spins, against separate kernels for O,
// the LU and inverse (a wave per matrix in LDS), the overlap and Ghalf, the matrices
// between them in memory:
//   N = 24, n = 5, W = 10        36 us ->  17      N = 200, n = 20, W = 512    183 us -> 122
//   N = 101, n = 10, 9, W = 137  72 us ->  26      N = 400, n = 40, W = 12     362 us -> 185
//   N = 255, n = 25 RHF, W = 71 184 us ->  58      N = 400, n = 40, W = 1024  1230 us -> 890
// One copy of a step's code instead of CW, or the step without branches, measured the same
// or slower; three waves a spin, two workgroups a CU, 1130 us at W = 1024.
#include <algorithm>

#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

__device__ __forceinline__ int gf_nspin(const GfArgs& a) { return (a.nbeta > 0 && !a.rhf) ? 2 : 1; }

// Waves of a spin for n <= 16 NT: NT row tiles times K parts of O; 16 NT / SW columns
// a wave in the elimination.
template <int NT>
struct GfPlan {
  static constexpr int SW = NT == 3 ? 6 : NT == 4 ? 8 : 4;
  static constexpr int PARTS = SW / NT;
  static constexpr int CW = 16 * NT / SW;
  static constexpr int KU = NT == 4 ? 2 : NT == 3 ? 3 : 4;  // K steps of O whose loads are in flight together
};

__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Largest v of the lanes < 16 NT (every lane active), wave-uniform: DPP maxima within the
// rows of 16 lanes (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror pair each lane with one of another group), then one lane of each row.
template <int NT>
__device__ __forceinline__ unsigned rows_max(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
  unsigned m = (unsigned)__builtin_amdgcn_readlane((int)v, 0);
#pragma unroll
  for (int t = 1; t < NT; ++t) m = max(m, (unsigned)__builtin_amdgcn_readlane((int)v, 16 * t));
  return m;
}

// 1 / d: conj(d') / |d'|^2 of d' = d 2^-e, larger part in [1/2, 1), so that no square
// leaves the exponent range; the reciprocal instruction (2^-23) and a third-order step.
__device__ __forceinline__ cplx crecip(cplx d) {
  const int e = -__builtin_amdgcn_frexp_exp(fmax(fabs(d.re), fabs(d.im)));
  const double x = ldexp(d.re, e), y = ldexp(d.im, e);
  const double q = fma(x, x, y * y);
  double r = __builtin_amdgcn_rcp(q);
  const double h = fma(-q, r, 1.0);
  r = fma(r, fma(h, h, h), r);
  return cmake(ldexp(x * r, e), ldexp(-y * r, e));
}

// a -= m u, u wave-uniform
__device__ __forceinline__ void sub_product(cplx& a, cplx m, cplx u) {
  a.re = fma(-m.re, u.re, a.re);
  a.im = fma(-m.re, u.im, a.im);
  a.re = fma(m.im, u.im, a.re);
  a.im = fma(-m.im, u.re, a.im);
}

template <int NT>
constexpr size_t gf_lds() {  // per spin: O, two pivot columns, the pivots
  return sizeof(cplx) * (16 * NT * (16 * NT + 1) + 3 * 16 * NT);
}

template <int NT, bool REAL, bool GHALF>
__global__ void __launch_bounds__(128 * GfPlan<NT>::SW) gf_kernel(GfArgs a) {
  using P = GfPlan<NT>;
  constexpr int SW = P::SW, CW = P::CW, R = 16 * NT, LD = R + 1, KU = P::KU;
  extern __shared__ cplx smem[];
  __shared__ int prow[2][R];  // pivot row of each step
  __shared__ int odd[2];      // parity of the pivot rows' permutation
  phase_mark(a.mark, blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int s = wave / SW, sw = wave % SW, w = blockIdx.y * gridDim.x + blockIdx.x, N = a.nbasis;
  if (w >= a.nwalkers) return;
  const int n = s == 0 ? a.nalpha : a.nbeta;
  const double* phi = (s == 0 ? a.phia : a.phib) + 2 * (int64_t)w * N * n;
  const double* psi = s == 0 ? a.psia : a.psib;
  cplx* O = smem + s * (R * LD + 3 * R);
  cplx* col = O + R * LD;    // [2][R]: pivot column of the even / odd steps over d
  cplx* dpiv = col + 2 * R;  // [R]: pivot of each row

  // ---- O[i][j] = sum_m phi[m][i] conj(psi[m][j])
  {
    const int it = sw % NT, part = sw / NT;
    const int i = it * 16 + r16;
    v4d re[NT], im[NT];
#pragma unroll
    for (int jt = 0; jt < NT; ++jt) {
      re[jt] = zero4d();
      im[jt] = zero4d();
    }
    if (it * 16 < n) {
      // rows i and columns j past n repeat the last one (no O entry of theirs is kept)
      const double* pa = phi + 2 * ((int64_t)kq * n + min(i, n - 1));
      const double* pb[NT];
#pragma unroll
      for (int jt = 0; jt < NT; ++jt) pb[jt] = psi + 2 * ((int64_t)kq * n + min(jt * 16 + r16, n - 1));
      const auto chunk = [&](int m0, bool tail) {
        cplx av[KU], bv[KU][NT];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int m = m0 + 4 * u;
          const int64_t o = (int64_t)(tail ? min(m, N - 1 - kq) : m) * n;  // (row m + kq)
          av[u] = ld(pa, o);
#pragma unroll
          for (int jt = 0; jt < NT; ++jt)
            bv[u][jt] = REAL ? cmake(pb[jt][2 * o], 0.0) : cconj(ld(pb[jt], o));
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          if (tail && m0 + 4 * u + kq >= N) av[u] = cmake(0.0, 0.0);
#pragma unroll
          for (int jt = 0; jt < NT; ++jt) {
            if (tail && m0 + 4 * u + kq >= N) bv[u][jt] = cmake(0.0, 0.0);
            re[jt] = mfma64(av[u].re, bv[u][jt].re, re[jt]);
            if (!REAL) re[jt] = mfma64(-av[u].im, bv[u][jt].im, re[jt]);
            if (!REAL) im[jt] = mfma64(av[u].re, bv[u][jt].im, im[jt]);
            im[jt] = mfma64(av[u].im, bv[u][jt].re, im[jt]);
          }
        }
      };
      int m0 = 4 * KU * part;
      for (; m0 + 4 * KU <= N; m0 += 4 * KU * P::PARTS) chunk(m0, false);
      if (m0 < N) chunk(m0, true);
    }
#pragma unroll
    for (int q = 0; q < P::PARTS; ++q) {  // parts added one after the other
      if (part == q)
#pragma unroll
        for (int jt = 0; jt < NT; ++jt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            cplx* o = O + (it * 16 + 4 * r + kq) * LD + jt * 16 + r16;
            const bool in = it * 16 + 4 * r + kq < n && jt * 16 + r16 < n;
            const cplx v = cmake(in ? re[jt][r] : 0.0, in ? im[jt][r] : 0.0);
            *o = q == 0 ? v : cadd(*o, v);
          }
      __syncthreads();
    }
  }

  // ---- elimination; this wave's columns are t SW + sw
  cplx b[CW];
#pragma unroll
  for (int t = 0; t < CW; ++t) b[t] = lane < R ? O[lane * LD + t * SW + sw] : cmake(0.0, 0.0);
  const int steps = max(a.nalpha, gf_nspin(a) == 2 ? a.nbeta : 0);
  const unsigned long long rows = n < 64 ? ~(~0ull << n) : ~0ull;
  unsigned long long open = rows;  // rows that no step has used
  int sign = 0, step_of = 0;       // parity of the permutation; this row's step
  // the previous step: this row's factor (zero when there is none) and its pivot row
  cplx m = cmake(0.0, 0.0);
  int p = 0;
  const auto update = [&](cplx& x) { sub_product(x, m, cmake(lane_value(x.re, p), lane_value(x.im, p))); };
#pragma unroll
  for (int t = 0; t < CW; ++t) {
    const int c0 = GHALF ? 0 : t;  // the overlap leaves finished columns alone
#pragma unroll 1
    for (int o = 0; o < SW; ++o) {
      const int k = t * SW + o;
      if (k >= steps) break;
      const bool mine = sw == o && k < n;
      if (mine) {
        update(b[t]);
        const bool cand = (open >> lane) & 1;
        const unsigned key = cand ? (unsigned)__double2hiint(fabs(b[t].re) + fabs(b[t].im)) : 0u;
        const unsigned most = rows_max<NT>(key);
        const int pk = __builtin_ctzll(__ballot(key == most) & open);  // (all zero: the first open row)
        const cplx d = cmake(lane_value(b[t].re, pk), lane_value(b[t].im, pk));
        const bool pivot = lane == pk;
        // (a zero pivot leaves the other rows as they are)
        const cplx f = (d.re == 0.0 && d.im == 0.0) || pivot ? cmake(0.0, 0.0) : cmul(b[t], crecip(d));
        if (lane < R) col[(k & 1) * R + lane] = f;
        if (lane == 0) prow[s][k] = pk;
        if (pivot) dpiv[lane] = d;
        // so that this step's update leaves f in the other rows
        b[t] = cmake(pivot ? -1.0 : 0.0, 0.0);
      } else {
#pragma unroll
        for (int c = c0; c < CW; ++c) update(b[c]);
      }
      __syncthreads();
      if (mine)
#pragma unroll
        for (int c = c0; c < CW; ++c)
          if (c != t) update(b[c]);
      m = cmake(0.0, 0.0);
      if (k < n) {
        m = col[(k & 1) * R + (lane < R ? lane : 0)];
        p = __builtin_amdgcn_readfirstlane(prow[s][k]);
        open &= ~(1ull << p);
        sign ^= __popcll((rows & ~open) >> p >> 1) & 1;
        if (lane == p) step_of = k;
      }
    }
  }
  if (sw == 0 && lane == 0) odd[s] = sign;
  if (GHALF) {
#pragma unroll
    for (int c = 0; c < CW; ++c) update(b[c]);
    if (lane < n) {
      const cplx rd = crecip(dpiv[lane]);
      const cplx sc = cmake(-rd.re, -rd.im);
#pragma unroll
      for (int t = 0; t < CW; ++t) {
        const int j = t * SW + sw;
        if (j < n) O[step_of * LD + prow[s][j]] = cmul(b[t], sc);
      }
    }
  }
  __syncthreads();

  // ---- overlap: the first wave, both spins
  if (wave == 0) {
    double lg = 0.0;
    cplx ph = cmake(1.0, 0.0);
    bool singular = false;
    const int ns = gf_nspin(a);
    for (int q = 0; q < ns; ++q) {
      const int nq = q == 0 ? a.nalpha : a.nbeta;
      const cplx* dq = smem + q * (R * LD + 3 * R) + R * LD + 2 * R;
      if (lane < nq) {
        // lane i takes log|d| and d / |d| of row i; a butterfly over the rows sums and
        // multiplies them
        const cplx d = dq[lane];
        const double ab = cabs(d);
        lg += log(ab);
        ph = cmul(ph, ab > 0.0 ? cmake(d.re / ab, d.im / ab) : cmake(0.0, 0.0));
        singular = singular || (d.re == 0.0 && d.im == 0.0);
      }
    }
    for (int off = 1; off < R; off <<= 1) {
      lg += __shfl_xor(lg, off, 64);
      const cplx o = cmake(__shfl_xor(ph.re, off, 64), __shfl_xor(ph.im, off, 64));
      ph = cmul(ph, o);
    }
    if (ns == 2 ? odd[0] ^ odd[1] : odd[0]) ph = cmake(-ph.re, -ph.im);
    if (a.nbeta > 0 && a.rhf) {
      ph = cmul(ph, ph);
      lg += lg;
    }
    singular = __ballot(singular) != 0;
    if (lane == 0) {
      const double e = exp(lg - (a.log_shift ? a.log_shift[w] : 0.0));
      st(a.ovlp, w, cmake(ph.re * e, ph.im * e));
      if (singular && a.flags) atomicOr(a.flags, AFQMC_FLAG_SINGULAR);
      if (singular && a.wflags) atomicOr(a.wflags + w, AFQMC_FLAG_SINGULAR);
    }
  }
  if (!GHALF) return;

  // ---- Ghalf[i][m] = sum_j Oinv[i][j] phi[m][j], all row tiles of 16 columns m a wave
  double* gh = (s == 0 ? a.ghalfa : a.ghalfb) + 2 * (int64_t)w * n * N;
  constexpr int G = 4;  // K steps per group; a group's loads are issued before the MFMAs of the one before
  const int nmt = (int)ceil_div(N, 16);
  for (int mt = SW - 1 - sw; mt < nmt; mt += SW) {  // (the first wave, busy with the overlap, comes last)
    const int mm = mt * 16 + r16;
    const double* row = phi + 2 * (int64_t)mm * n;
    v4d re[NT], im[NT];
#pragma unroll
    for (int it = 0; it < NT; ++it) {
      re[it] = zero4d();
      im[it] = zero4d();
    }
    cplx bv[2][G];
    const auto load = [&](int g, cplx (&v)[G]) {
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int k = 4 * (G * g + u) + kq;
        v[u] = (mm < N && k < n) ? ld(row, k) : cmake(0.0, 0.0);
      }
    };
    load(0, bv[0]);
#pragma unroll
    for (int g = 0; g < NT; ++g) {
      if (g + 1 < NT) load(g + 1, bv[(g + 1) & 1]);
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int ks = G * g + u;
        if (ks * 4 < n) {  // K steps past n have zero operands; a branch keeps the unroll
          const cplx v = bv[g & 1][u];
#pragma unroll
          for (int it = 0; it < NT; ++it) {
            const cplx f = O[(it * 16 + r16) * LD + 4 * ks + kq];
            re[it] = mfma64(f.re, v.re, re[it]);
            re[it] = mfma64(-f.im, v.im, re[it]);
            im[it] = mfma64(f.re, v.im, im[it]);
            im[it] = mfma64(f.im, v.re, im[it]);
          }
        }
      }
    }
#pragma unroll
    for (int it = 0; it < NT; ++it)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = it * 16 + 4 * r + kq;  // accumulator row = 4 r + lane / 16
        if (i < n && mm < N) st(gh, (int64_t)i * N + mm, cmake(re[it][r], im[it][r]));
      }
  }
}

__global__ void __launch_bounds__(256) imag_any_kernel(const double* __restrict__ z, int64_t n, int* flag) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n && z[2 * i + 1] != 0.0) *flag = 1;
}

}  // namespace

hipError_t launch_imag_any(const double* z, int64_t n, int* flag, hipStream_t stream) {
  if (n < 1) return hipSuccess;
  hipLaunchKernelGGL(imag_any_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream, z, n, flag);
  return hipGetLastError();
}

namespace {

template <int NT, bool REAL, bool GHALF>
hipError_t launch_gf_as(const GfArgs& a, hipStream_t stream) {
  const int nspin = (a.nbeta > 0 && !a.rhf) ? 2 : 1;
  const size_t lds = nspin * gf_lds<NT>();
  const hipError_t e = allow_lds((const void*)gf_kernel<NT, REAL, GHALF>, lds);
  if (e != hipSuccess) return e;
  // (a grid dimension takes less than 2^32 threads)
  const int64_t gx = std::min(a.nwalkers, 1 << 20);
  hipLaunchKernelGGL((gf_kernel<NT, REAL, GHALF>), dim3((unsigned)gx, (unsigned)ceil_div(a.nwalkers, gx)),
                     dim3(64 * GfPlan<NT>::SW * nspin), lds, stream, a);
  return hipGetLastError();
}

template <int NT>
hipError_t launch_gf_nt(const GfArgs& a, bool want_ghalf, hipStream_t stream) {
  if (!want_ghalf)
    return a.psi_real ? launch_gf_as<NT, true, false>(a, stream) : launch_gf_as<NT, false, false>(a, stream);
  return a.psi_real ? launch_gf_as<NT, true, true>(a, stream) : launch_gf_as<NT, false, true>(a, stream);
}

}  // namespace

hipError_t launch_gf(const GfArgs& a, bool want_ghalf, hipStream_t stream) {
  const int nmax = (a.nbeta > 0 && !a.rhf && a.nbeta > a.nalpha) ? a.nbeta : a.nalpha;
  if (nmax < 1 || nmax > 64 || a.nwalkers < 1 || a.gplanes[0]) return hipErrorInvalidValue;
  switch ((nmax + 15) / 16) {
    case 1: return launch_gf_nt<1>(a, want_ghalf, stream);
    case 2: return launch_gf_nt<2>(a, want_ghalf, stream);
    case 3: return launch_gf_nt<3>(a, want_ghalf, stream);
    default: return launch_gf_nt<4>(a, want_ghalf, stream);
  }
}

}  // namespace afqmc
