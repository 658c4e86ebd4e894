// Exchange as a quadratic form in the walker's half-rotated Green's function.
//
// With T_x = L_x G^T (L_x the [n, N] half-rotated Cholesky vector x, G = Ghalf
// [n, N]),
//   sum_x tr(T_x T_x) = sum_{i,j,m,m'} G[i][m'] G[j][m] sum_x L_x[i][m] L_x[j][m']
//                     = g^T Wq g,   g = vec(G),  Wq[(i,m'),(j,m)] = sum_x L_x[i][m] L_x[j][m'],
// i.e. Wq = R^T R (R = rchol as [X, n N]) with every N x N block transposed; Wq is
// real symmetric and walker-independent.  Per step the exchange of all walkers
// is one GEMM Y = G Wq (M = W, N = K = n N) and a dot product per walker, about
// X / N times fewer flops than forming every T_x (and no n x n trace epilogue).
// Same value as ipie/estimators/local_energy_sd.py:263-303 (exx_kernel_batch_real_rchol).
// Wq's symmetry halves it: with column tiles of T (QUAD64_TILE in FP64, QUAD_TILE in
// BF16), W' = Wq on the diagonal tiles, 2 Wq above them and 0 below, and column
// tile b of Y = G W' sums K over the tiles up to b only (g^T W' g = g^T Wq g).
//   quad_w_kernel       W' from rchol, FP64 accumulation, written in FP64 or as
//                       split-BF16 planes [2][n Kp][n Kp] (zero padding)
//   quad_sum_kernel     E_w = sum of the per-unit dot products written by the
//                       products' epilogues
#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

constexpr int QW_T = 128;          // tile edge of G = R^T R
constexpr int QW_XC = 16;          // Cholesky vectors per chunk
constexpr int QW_LD = QW_T + 16;   // LDS row, doubles: the four rows of a K step 128 bytes apart in the banks
constexpr size_t QW_LDS = 2 * 2 * 8 * (size_t)QW_XC * QW_LD;  // two stages of both operands

__device__ __forceinline__ uint16_t qf2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float qbf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// One 128 x 128 tile of G[P][Q] = sum_x R[x][P] R[x][Q], P = (j, p) and Q = (i, q) over the
// n N columns of R; G is symmetric, and only the tiles P <= Q are computed.  G[P][Q]
// is Wq[(i, p)][(j, q)] and, transposed, Wq[(j, q)][(i, p)]: each goes to its place in W'
// where that is kept (b's column tile at most a's).  Np is the column stride per
// orbital of the output (N for FP64, Kp for the padded planes, zero beforehand).
// What bounds it: the matrix units (v_mfma_f64_16x16x4f64, four waves of 64 x 64); the
// next chunk's loads are in flight under a chunk's products.  n N = 16000, 2400 vectors, per
// spin: 64 x 64 tiles per orbital pair on the vector units, 188 GB through L2, took
// 22.7 ms in FP64 and 44 ms as planes (every tile); now 12.0 and 11.7 ms (51 TFLOP/s).
__global__ void __launch_bounds__(256, 2) quad_w_kernel(const double* __restrict__ R, int X, int n, int N, int Np,
                                                       double* __restrict__ w64, int64_t ld64,
                                                       uint16_t* __restrict__ wplanes) {
  extern __shared__ double qw_lds[];
  const int tp = blockIdx.x, tq = blockIdx.y;
  if (tp > tq) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int wr = wave & 1, wc = wave >> 1;
  const int64_t nN = (int64_t)n * N;
  // this thread loads columns col, col + 64 of rows row, row + 4, ..
  const int row = threadIdx.x >> 6, col = lane;
  double va[QW_XC / 4][2], vb[QW_XC / 4][2];
  const auto fetch = [&](int x0) {
#pragma unroll
    for (int r = 0; r < QW_XC / 4; ++r) {
      const int x = x0 + row + 4 * r;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t P = (int64_t)tp * QW_T + col + 64 * h, Q = (int64_t)tq * QW_T + col + 64 * h;
        va[r][h] = x < X && P < nN ? R[x * nN + P] : 0.0;
        vb[r][h] = x < X && Q < nN ? R[x * nN + Q] : 0.0;
      }
    }
  };
  const auto stash = [&](int buf) {
    double* a = qw_lds + buf * 2 * QW_XC * QW_LD;
    double* b = a + QW_XC * QW_LD;
#pragma unroll
    for (int r = 0; r < QW_XC / 4; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[(row + 4 * r) * QW_LD + col + 64 * h] = va[r][h];
        b[(row + 4 * r) * QW_LD + col + 64 * h] = vb[r][h];
      }
  };
  v4d acc[4][4];
#pragma unroll
  for (int it = 0; it < 4; ++it)
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) acc[it][jt] = zero4d();
  fetch(0);
  stash(0);
  __syncthreads();
  int buf = 0;
  for (int x0 = 0; x0 < X; x0 += QW_XC) {
    const bool more = x0 + QW_XC < X;
    if (more) fetch(x0 + QW_XC);
    const double* a = qw_lds + buf * 2 * QW_XC * QW_LD + 64 * wr;
    const double* b = qw_lds + buf * 2 * QW_XC * QW_LD + QW_XC * QW_LD + 64 * wc;
#pragma unroll
    for (int k = 0; k < QW_XC / 4; ++k) {
      double fa[4], fb[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        fa[t] = a[(4 * k + kq) * QW_LD + 16 * t + r16];
        fb[t] = b[(4 * k + kq) * QW_LD + 16 * t + r16];
      }
#pragma unroll
      for (int it = 0; it < 4; ++it)
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) acc[it][jt] = mfma64(fa[it], fb[jt], acc[it][jt]);
    }
    if (more) stash(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  const int64_t ldo = (int64_t)n * Np;  // row length of the planes
  const int64_t plane = ldo * ldo;
  const auto put = [&](uint32_t a, uint32_t b, double g) {
    if (w64) {
      const uint32_t ta = a / QUAD64_TILE, tb = b / QUAD64_TILE;
      if (tb <= ta) w64[(int64_t)a * ld64 + b] = tb < ta ? 2.0 * g : g;
    } else {
      // plane row a is the output column, b the K index: W'_{b a}
      const uint32_t ta = a / QUAD_TILE, tb = b / QUAD_TILE;
      if (tb > ta) return;
      const double v = tb < ta ? 2.0 * g : g;
      const uint16_t hi = qf2bf((float)v);
      wplanes[a * ldo + b] = hi;
      wplanes[plane + a * ldo + b] = qf2bf((float)(v - (double)qbf2f(hi)));
    }
  };
  const uint32_t cols = (uint32_t)nN, uN = (uint32_t)N;
  uint32_t Q[4], oi[4], q[4];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    Q[jt] = tq * QW_T + 64 * wc + 16 * jt + r16;
    oi[jt] = Q[jt] / uN * Np;
    q[jt] = Q[jt] % uN;
  }
#pragma unroll
  for (int it = 0; it < 4; ++it)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t P = tp * QW_T + 64 * wr + 16 * it + 4 * r + kq;
      if (P >= cols) continue;
      const uint32_t oj = P / uN * Np, pp = P % uN;
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        if (Q[jt] >= cols) continue;
        put(oi[jt] + pp, oj + q[jt], acc[it][jt][r]);
        if (tp != tq) put(oj + q[jt], oi[jt] + pp, acc[it][jt][r]);
      }
    }
}

// out[w] = sum_s part[s][w]: WL walkers x 256 / WL slot lanes per workgroup, the
// slot lanes combined in a fixed order (few walkers, many slots: more lanes
// per walker keep the serial chain of each lane short).
template <int WL>
__global__ void __launch_bounds__(256) quad_sum_kernel(const double* __restrict__ part, int nslots, int nwalkers,
                                                      double* __restrict__ out) {
  constexpr int SL = 256 / WL;
  __shared__ double sr[SL][WL + 1], si[SL][WL + 1];
  const int wl = threadIdx.x % WL, sl = threadIdx.x / WL;
  const int w = blockIdx.x * WL + wl;
  double re = 0.0, im = 0.0;
  if (w < nwalkers) {
    for (int s = sl; s < nslots; s += SL) {
      const cplx v = ld(part, (int64_t)s * nwalkers + w);
      re += v.re;
      im += v.im;
    }
  }
  sr[sl][wl] = re;
  si[sl][wl] = im;
  __syncthreads();
  if (sl == 0 && w < nwalkers) {
    double tr = 0.0, ti = 0.0;
    for (int k = 0; k < SL; ++k) {
      tr += sr[k][wl];
      ti += si[k][wl];
    }
    st(out, w, cmake(tr, ti));
  }
}

// ---------------------------------------------------------------- FP8 operands
// FP8 (E4M3, round to nearest even) of four values, packed little-endian
__device__ __forceinline__ uint32_t pack_fp8x4(float v0, float v1, float v2, float v3) {
  int p = 0;
  p = __builtin_amdgcn_cvt_pk_fp8_f32(v0, v1, p, false);
  p = __builtin_amdgcn_cvt_pk_fp8_f32(v2, v3, p, true);
  return (uint32_t)p;
}

// power-of-two scale putting the largest magnitude at most at 224 (half the
// E4M3 maximum: the lo part of a split value and rounding stay in range)
__device__ __forceinline__ double fp8_scale(double amax) {
  return amax > 0.0 ? exp2(floor(log2(224.0 / amax))) : 1.0;
}

// max |x| over n BF16 values into *absmax (FP32 bits; non-negative floats
// order like their bit patterns, so the result does not depend on timing)
__global__ void __launch_bounds__(256) quad_absmax_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                        unsigned int* __restrict__ absmax) {
  float m = 0.0f;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
    m = fmaxf(m, fabsf(qbf2f(x[e])));
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(absmax, __float_as_uint(m));
}

__global__ void quad_w8_scale_kernel(const unsigned int* __restrict__ absmax, float* __restrict__ scale) {
  if (threadIdx.x == 0) scale[0] = (float)fp8_scale((double)__uint_as_float(absmax[0]));
}

// w8[r][k], 4 consecutive k per thread, zero outside ldn x ldn
__global__ void __launch_bounds__(256) quad_w8_kernel(const uint16_t* __restrict__ wp, int64_t ldn, int64_t ld8,
                                                    uint8_t* __restrict__ w8, const float* __restrict__ scale) {
  const int64_t q4 = ld8 / 4;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ld8 * q4) return;
  const int64_t r = idx / q4, k0 = (idx % q4) * 4;
  const float s = scale[0];
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t k = k0 + j;
    v[j] = (r < ldn && k < ldn) ? (qbf2f(wp[r * ldn + k]) + qbf2f(wp[ldn * ldn + r * ldn + k])) * s : 0.0f;
  }
  *reinterpret_cast<uint32_t*>(w8 + r * ld8 + k0) = pack_fp8x4(v[0], v[1], v[2], v[3]);
}

// one workgroup per walker: the largest |re|, |im| of d_w, then its scaled FP8 planes
__global__ void __launch_bounds__(256) split_fp8_rows_kernel(const double* __restrict__ g,
                                                           const double* __restrict__ gref, int nwalkers, int n,
                                                           int N, int Kp, int64_t ld8, uint8_t* __restrict__ a8,
                                                           const float* __restrict__ wscale,
                                                           double* __restrict__ row_inv) {
  __shared__ double red[256 / 64];
  const int w = blockIdx.x, tid = threadIdx.x;
  const double* gw = g + 2 * (int64_t)w * n * N;
  double m = 0.0;
  for (int e = tid; e < n * N; e += 256) {
    cplx d = ld(gw, e);
    if (gref) d = csub(d, ld(gref, e));
    m = fmax(m, fmax(fabs(d.re), fabs(d.im)));
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  const double s = fp8_scale(m);
  uint8_t* pre = a8 + (int64_t)w * ld8;
  uint8_t* pim = a8 + ((int64_t)nwalkers + w) * ld8;
  for (int64_t k0 = (int64_t)tid * 4; k0 < ld8; k0 += 4 * 256) {
    float vr[4], vi[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // a walker row holds n Kp < 2^31 values: 32-bit row and column
      const int k = (int)(k0 + j);
      const int i = k / Kp, mm = k - i * Kp;
      vr[j] = vi[j] = 0.0f;
      if (i < n && mm < N) {
        cplx d = ld(gw, (int64_t)i * N + mm);
        if (gref) d = csub(d, ld(gref, (int64_t)i * N + mm));
        vr[j] = (float)(d.re * s);
        vi[j] = (float)(d.im * s);
      }
    }
    *reinterpret_cast<uint32_t*>(pre + k0) = pack_fp8x4(vr[0], vr[1], vr[2], vr[3]);
    *reinterpret_cast<uint32_t*>(pim + k0) = pack_fp8x4(vi[0], vi[1], vi[2], vi[3]);
  }
  if (tid == 0) row_inv[w] = 1.0 / (s * (double)wscale[0]);
}

// The same planes with the walker's dG held in registers between the maximum
// and the conversion (G read once): one walker per workgroup of 1024 threads,
// J chunks of 4 consecutive padded K positions per thread (ld8 <= 4096 J;
// Kp a multiple of 4, so a chunk never crosses a row of Kp).
template <int J>
__global__ void __launch_bounds__(1024) split_fp8_rows_reg_kernel(const double* __restrict__ g,
                                                                 const double* __restrict__ gref, int nwalkers,
                                                                 int n, int N, int Kp, int ld8,
                                                                 uint8_t* __restrict__ a8,
                                                                 const float* __restrict__ wscale,
                                                                 double* __restrict__ row_inv) {
  __shared__ double red[16];
  const int w = blockIdx.x, tid = threadIdx.x;
  const double* gw = g + 2 * (int64_t)w * n * N;
  cplx v[J][4];
  double m = 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k0 = 4 * (tid + 1024 * j);
    const int i = k0 / Kp, m0 = k0 - i * Kp;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[j][r] = cplx{0.0, 0.0};
      if (k0 < ld8 && i < n && m0 + r < N) {
        cplx d = ld(gw, i * N + m0 + r);
        if (gref) d = csub(d, ld(gref, i * N + m0 + r));
        v[j][r] = d;
        m = fmax(m, fmax(fabs(d.re), fabs(d.im)));
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 16; ++t) m = fmax(m, red[t]);
  const double s = fp8_scale(m);
  uint8_t* pre = a8 + (int64_t)w * ld8;
  uint8_t* pim = a8 + ((int64_t)nwalkers + w) * ld8;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k0 = 4 * (tid + 1024 * j);
    if (k0 < ld8) {
      *reinterpret_cast<uint32_t*>(pre + k0) =
          pack_fp8x4((float)(v[j][0].re * s), (float)(v[j][1].re * s), (float)(v[j][2].re * s), (float)(v[j][3].re * s));
      *reinterpret_cast<uint32_t*>(pim + k0) =
          pack_fp8x4((float)(v[j][0].im * s), (float)(v[j][1].im * s), (float)(v[j][2].im * s), (float)(v[j][3].im * s));
    }
  }
  if (tid == 0) row_inv[w] = 1.0 / (s * (double)wscale[0]);
}

}  // namespace

hipError_t launch_quad_w8(const uint16_t* wplanes, int64_t ldn, int64_t ld8, uint8_t* w8, float* scale,
                          unsigned int* absmax, hipStream_t stream) {
  if (ldn < 1 || ld8 < ldn || ld8 % 64 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(quad_absmax_kernel, dim3(2048), dim3(256), 0, stream, wplanes, ldn * ldn, absmax);
  hipLaunchKernelGGL(quad_w8_scale_kernel, dim3(1), dim3(64), 0, stream, absmax, scale);
  const int64_t total = ld8 * (ld8 / 4);
  hipLaunchKernelGGL(quad_w8_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, stream, wplanes, ldn, ld8,
                     w8, scale);
  return hipGetLastError();
}

hipError_t launch_split_fp8_rows(const double* g, const double* gref, int nwalkers, int n, int N, int Kp,
                                 int64_t ld8, uint8_t* a8, const float* wscale, double* row_inv, hipStream_t stream) {
  if (nwalkers < 1 || n < 1 || Kp < N || ld8 < (int64_t)n * Kp || ld8 % 64 != 0 || ld8 > INT32_MAX)
    return hipErrorInvalidValue;
  if (Kp % 4 == 0 && ld8 <= 5 * 4096) {
    const int l = (int)ld8;
    if (ld8 <= 2 * 4096)
      hipLaunchKernelGGL(split_fp8_rows_reg_kernel<2>, dim3((unsigned)nwalkers), dim3(1024), 0, stream, g, gref,
                         nwalkers, n, N, Kp, l, a8, wscale, row_inv);
    else if (ld8 <= 3 * 4096)
      hipLaunchKernelGGL(split_fp8_rows_reg_kernel<3>, dim3((unsigned)nwalkers), dim3(1024), 0, stream, g, gref,
                         nwalkers, n, N, Kp, l, a8, wscale, row_inv);
    else
      hipLaunchKernelGGL(split_fp8_rows_reg_kernel<5>, dim3((unsigned)nwalkers), dim3(1024), 0, stream, g, gref,
                         nwalkers, n, N, Kp, l, a8, wscale, row_inv);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(split_fp8_rows_kernel, dim3((unsigned)nwalkers), dim3(256), 0, stream, g, gref, nwalkers, n, N,
                     Kp, ld8, a8, wscale, row_inv);
  return hipGetLastError();
}

hipError_t launch_quad_sum(const double* part, int nslots, int nwalkers, double* out, hipStream_t stream) {
  if (nslots < 1 || nwalkers < 1) return hipErrorInvalidValue;
  if (nwalkers >= 512)
    hipLaunchKernelGGL(quad_sum_kernel<16>, dim3((unsigned)ceil_div(nwalkers, 16)), dim3(256), 0, stream, part,
                       nslots, nwalkers, out);
  else
    hipLaunchKernelGGL(quad_sum_kernel<4>, dim3((unsigned)ceil_div(nwalkers, 4)), dim3(256), 0, stream, part,
                       nslots, nwalkers, out);
  return hipGetLastError();
}

hipError_t launch_quad_w(const double* rchol, int X, int n, int N, int Np, double* w64, int64_t ld64,
                         uint16_t* wplanes, hipStream_t stream) {
  if ((w64 == nullptr) == (wplanes == nullptr) || Np < N || X < 1 || (int64_t)n * Np >= INT32_MAX)
    return hipErrorInvalidValue;
  if (w64 && (Np != N || ld64 < (int64_t)n * N)) return hipErrorInvalidValue;
  if (wplanes) {  // the padding and what is past a row's column tile stay zero: [2][n Kp][n Kp] in doubles
    const int64_t ldo = (int64_t)n * Np;
    if (ldo % 2 != 0) return hipErrorInvalidValue;
    const hipError_t e = launch_setup_fill(reinterpret_cast<double*>(wplanes), ldo * ldo / 2, 0.0, stream);
    if (e != hipSuccess) return e;
  }
  const unsigned tiles = (unsigned)ceil_div((int64_t)n * N, QW_T);
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(quad_w_kernel), QW_LDS);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(quad_w_kernel, dim3(tiles, tiles), dim3(256), QW_LDS, stream, rchol, X, n, N, Np, w64, ld64,
                     wplanes);
  return hipGetLastError();
}

}  // namespace afqmc
