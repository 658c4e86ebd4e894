// FP64 MFMA products of the propagation step: C[w] = alpha A[w] B[w] for the
// one-body propagator (ipie/propagation/operations.py:26-55) and every Taylor
// term (operations.py:85-117).
//
// v_mfma_f64_16x16x4f64, operands loaded straight from global memory into the
// fragment registers (each lane reads a contiguous 4-element k range).  A real
// operand times a complex operand is two real MFMAs (re, im); complex times
// complex is four.
#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

// ---------------------------------------------------------------- batched NN
constexpr int NN_WAVES = 4;  // 64 rows per workgroup

template <int RN, bool ACPLX, bool FAST>
__global__ void __launch_bounds__(64 * NN_WAVES) batched_nn_kernel(BatchedNNArgs a) {
  const int nrb = (int)ceil_div(a.nrows, 16 * NN_WAVES);
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int w = lin / nrb, rb = lin % nrb;
  if (w >= a.nwalkers) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int l16 = lane & 15, q = lane >> 4;
  const int row0 = rb * 16 * NN_WAVES + wave * 16;
  if (row0 >= a.nrows) return;
  const int K = a.nrows;
  const int arow = row0 + l16;
  const bool okr = arow < a.nrows;
  const double* Ab = a.A + (ACPLX ? 2 : 1) * ((int64_t)w * a.a_stride + (int64_t)arow * K);
  const double* Bb = a.B + 2 * (int64_t)w * a.b_stride;
  v4d re[RN], im[RN];
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    re[j] = zero4d();
    im[j] = zero4d();
  }
  const int nch = (int)ceil_div(K, 16);
  for (int c = 0; c < nch; ++c) {
    const int kk = 16 * c + 4 * q;
    cplx af[4];
    if (FAST) {
      if (okr && kk < K) {
        if (ACPLX) {
          const double2* p = reinterpret_cast<const double2*>(Ab + 2 * kk);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const double2 v = p[s];
            af[s] = cplx{v.x, v.y};
          }
        } else {
          const double2* p = reinterpret_cast<const double2*>(Ab + kk);
          const double2 v0 = p[0], v1 = p[1];
          af[0] = cplx{v0.x, 0.0};
          af[1] = cplx{v0.y, 0.0};
          af[2] = cplx{v1.x, 0.0};
          af[3] = cplx{v1.y, 0.0};
        }
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) af[s] = cplx{0.0, 0.0};
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (okr && kk + s < K) {
          if (ACPLX) af[s] = cplx{Ab[2 * (kk + s)], Ab[2 * (kk + s) + 1]};
          else af[s] = cplx{Ab[kk + s], 0.0};
        } else {
          af[s] = cplx{0.0, 0.0};
        }
      }
    }
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      const int col = 16 * j + l16;
      cplx bf[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = kk + s;
        if (col < a.ncol && k < K) bf[s] = ld(Bb, (int64_t)k * a.ldb + col);
        else bf[s] = cplx{0.0, 0.0};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        re[j] = mfma64(af[s].re, bf[s].re, re[j]);
        im[j] = mfma64(af[s].re, bf[s].im, im[j]);
        if (ACPLX) {
          re[j] = mfma64(-af[s].im, bf[s].im, re[j]);
          im[j] = mfma64(af[s].im, bf[s].re, im[j]);
        }
      }
    }
  }
  double* Cb = a.C + 2 * (int64_t)w * a.c_stride;
  double* Sb = a.accum ? a.accum + 2 * (int64_t)w * a.c_stride : nullptr;
  const double* Ib = a.accum_init ? a.accum_init + 2 * (int64_t)w * a.c_stride : nullptr;
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int col = 16 * j + l16;
    if (col >= a.ncol) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 4 * r + q;
      if (row >= a.nrows) continue;
      const int64_t off = (int64_t)row * a.ldc + col;
      const cplx v = cmake(a.alpha * re[j][r], a.alpha * im[j][r]);
      st(Cb, off, v);
      if (Sb) {
        const cplx base = Ib ? ld(Ib, off) : ld(Sb, off);
        st(Sb, off, cadd(base, v));
      }
    }
  }
}

template <int RN, bool ACPLX>
hipError_t launch_nn_rn(const BatchedNNArgs& a, bool fast, hipStream_t stream) {
  const int nrb = (int)ceil_div(a.nrows, 16 * NN_WAVES);
  const dim3 grid(a.nwalkers * nrb);
  if (fast)
    hipLaunchKernelGGL((batched_nn_kernel<RN, ACPLX, true>), grid, dim3(64 * NN_WAVES), 0, stream, a);
  else
    hipLaunchKernelGGL((batched_nn_kernel<RN, ACPLX, false>), grid, dim3(64 * NN_WAVES), 0, stream, a);
  return hipGetLastError();
}

template <bool ACPLX>
hipError_t launch_nn(const BatchedNNArgs& a, bool fast, hipStream_t stream) {
  const int rn = (int)ceil_div(a.ncol, 16);
  switch (rn) {
    case 1: return launch_nn_rn<1, ACPLX>(a, fast, stream);
    case 2: return launch_nn_rn<2, ACPLX>(a, fast, stream);
    case 3: return launch_nn_rn<3, ACPLX>(a, fast, stream);
    case 4: return launch_nn_rn<4, ACPLX>(a, fast, stream);
    case 5: return launch_nn_rn<5, ACPLX>(a, fast, stream);
    case 6: return launch_nn_rn<6, ACPLX>(a, fast, stream);
    case 7: return launch_nn_rn<7, ACPLX>(a, fast, stream);
    case 8: return launch_nn_rn<8, ACPLX>(a, fast, stream);
    default: return hipErrorInvalidValue;
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

hipError_t launch_batched_nn(const BatchedNNArgs& a, hipStream_t stream) {
  const bool fast = (a.nrows % 4 == 0) && aligned16(a.A) && (a.a_complex || (a.nrows % 2 == 0));
  if (a.a_complex) return launch_nn<true>(a, fast, stream);
  return launch_nn<false>(a, fast, stream);
}

}  // namespace afqmc
