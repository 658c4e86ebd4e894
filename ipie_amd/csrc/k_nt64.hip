// FP64 contractions of complex rows with real rows, C[r, c] = sum_k A[r, k] B[c, k]
// (K contiguous in both), on v_mfma_f64_16x16x4f64:
//   * force bias   vbias[w, x] = sum_s sum_k Ghalf_s[w, k] rchol_s[x, k]
//                  (ipie/propagation/force_bias.py:79-121)
//   * VHS          VHS[w] = i sqrt(dt) sum_x xshifted[w, x] L_x from the packed upper
//                  triangle, written to both triangles
//                  (ipie/propagation/phaseless_generic.py:67-97,
//                   ipie/utils/pack_numba.py:22-33)
//   * the exchange's Y = G Wq
//
// What bounds it: one 16x16x4 FP64 MFMA takes 64 cycles on gfx950, so the matrix
// pipe is the limit as soon as a wave always has its operands in registers.
// Fragments loaded straight from memory did not give that: each lane group read
// 16 rows at the row pitch (32 cache lines per load instruction), one K chunk
// ahead, with one wave per SIMD (296 VGPRs), and ran at 59% of the FP64 MFMA
// peak.  Here a workgroup of four waves stages K chunks of 16 through LDS with
// direct global-to-LDS loads (two stages; the next chunk's loads run under the
// current chunk's MFMAs, one barrier per chunk); a row's piece of a chunk is
// 256 B (complex) or 128 B (real), so every load instruction covers whole
// cache lines.  The waves share the rows and each takes 32 of the tile's 128
// columns, which keeps the kernel within 256 registers (two workgroups per CU:
// one computes while the other waits at its barrier or writes its tile).
// Rows come in tiles of 16, 32, 48 or 64 (nt_rows below).
//
// LDS (16-byte slots): row r of A holds its 16 complex values with value k in
// slot r 16 + (k ^ (r % 16)); column c of B holds its 16 values in pairs, pair p
// in slot c 8 + (p ^ (c % 8)).  The XOR is applied to the source address, so
// a load fills 64 consecutive slots, and the eight lanes that read LDS together
// (eight rows, one k) hit eight different 16-byte bank groups.
#include <algorithm>
#include <cmath>

#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

constexpr int NT_KC = 16;                // K per LDS stage
constexpr int NT_RN = 2, NT_WAVES = 4;   // 16-column tiles per wave, waves side by side
constexpr int NT_TN = 16 * NT_RN * NT_WAVES;
constexpr int NT_THREADS = 64 * NT_WAVES;

__device__ double2 nt_zero;  // source of the slots past K

enum { NT_EPI_PART = 0, NT_EPI_VHS = 1 };

__device__ __forceinline__ void nt_load16(const char* src, double2* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// How the operands reach LDS: NT_DIRECT both by direct loads (16-byte aligned
// rows, K even); NT_BREG B's values one by one through registers (odd K or row
// pitch), stored after the current chunk's MFMAs are issued; NT_REG both.
enum { NT_DIRECT = 0, NT_BREG = 1, NT_REG = 2 };

template <int RM, int MODE, int EPI>
__global__ void __launch_bounds__(NT_THREADS, 2) nt64_kernel(NtArgs a) {
  constexpr int TM = 16 * RM;
  constexpr int A_SLOTS = TM * NT_KC, B_SLOTS = NT_TN * NT_KC / 2, STAGE = A_SLOTS + B_SLOTS;
  __shared__ double2 lds[2 * STAGE];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int nbm = (int)ceil_div(a.m, TM);
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int bm = lin % nbm, bn = lin / nbm, z = blockIdx.y;
  const int row0 = bm * TM;
  const int64_t col0 = (int64_t)bn * NT_TN;

  v4d re[RM][NT_RN], im[RM][NT_RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < NT_RN; ++j) {
      re[i][j] = zero4d();
      im[i][j] = zero4d();
    }

  // the chunks of all segments in order; this workgroup's range of them
  const int nch0 = (int)ceil_div(a.seg[0].K, NT_KC);
  const int nch = nch0 + (a.nseg > 1 ? (int)ceil_div(a.seg[1].K, NT_KC) : 0);
  const int z0 = (int)((int64_t)nch * z / a.ksplit), z1 = (int)((int64_t)nch * (z + 1) / a.ksplit);
  for (int s = 0; s < a.nseg; ++s) {
    const NtSegment sg = s == 0 ? a.seg[0] : a.seg[1];
    const int c_begin = s == 0 ? z0 : max(z0, nch0) - nch0, c_end = s == 0 ? min(z1, nch0) : z1 - nch0;
    if (c_begin >= c_end) continue;
    // this lane's slots: byte offsets from the tile's first row and column (rows
    // and columns past the end read the last one; their results are not written)
    const char* abase = reinterpret_cast<const char*>(sg.A + 2 * (int64_t)row0 * sg.lda);
    const char* bbase = reinterpret_cast<const char*>(sg.B + col0 * sg.ldb);
    const int last_r = (int)min((int64_t)TM, a.m - row0) - 1, last_c = (int)min((int64_t)NT_TN, a.n - col0) - 1;
    auto a_k = [&](int j) { return (lane & 15) ^ ((4 * (wave * RM + j) + (lane >> 4)) & 15); };
    auto b_k = [&](int) { return 2 * ((lane & 7) ^ (lane >> 3)); };  // column % 8 = lane / 8
    uint32_t ao[RM], bo[4];
#pragma unroll
    for (int j = 0; j < RM; ++j)
      ao[j] = 16u * ((uint32_t)min(4 * (wave * RM + j) + (lane >> 4), last_r) * (uint32_t)sg.lda + a_k(j));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      bo[j] = 8u * ((uint32_t)min(8 * (wave * 4 + j) + (lane >> 3), last_c) * (uint32_t)sg.ldb + b_k(j));
    double2 areg[RM], breg[4];
    // starts the loads of chunk c, into the LDS stage or the registers
    auto fetch = [&](int c, double2* stage) {
      const int k0 = NT_KC * c, left = sg.K - k0;
      const char* ac = abase + 16 * (int64_t)k0;
      const char* bc = bbase + 8 * (int64_t)k0;
      double2* As = stage + wave * RM * 64;
      double2* Bs = stage + A_SLOTS + wave * 4 * 64;
      const bool full = left >= NT_KC;
      const char* zero = reinterpret_cast<const char*>(&nt_zero);
#pragma unroll
      for (int j = 0; j < RM; ++j) {
        const char* p = full || a_k(j) < left ? ac + ao[j] : zero;
        if (MODE != NT_REG) nt_load16(p, As + 64 * j);
        else areg[j] = make_double2(reinterpret_cast<const double*>(p)[0], reinterpret_cast<const double*>(p)[1]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (MODE == NT_DIRECT) {
          nt_load16(full || b_k(j) < left ? bc + bo[j] : zero, Bs + 64 * j);
        } else {
          const double* p = reinterpret_cast<const double*>(bc + bo[j]);
          breg[j].x = b_k(j) < left ? p[0] : 0.0;
          breg[j].y = b_k(j) + 1 < left ? p[1] : 0.0;
        }
      }
    };
    auto stash = [&](double2* stage) {
      if (MODE == NT_REG) {
#pragma unroll
        for (int j = 0; j < RM; ++j) stage[(wave * RM + j) * 64 + lane] = areg[j];
      }
      if (MODE != NT_DIRECT) {
#pragma unroll
        for (int j = 0; j < 4; ++j) stage[A_SLOTS + (wave * 4 + j) * 64 + lane] = breg[j];
      }
    };
    if (s > 0) __syncthreads();  // the last chunk of the segment before has been read
    fetch(c_begin, lds);
    stash(lds);
    int buf = 0;
    for (int c = c_begin; c < c_end; ++c) {
      // chunk c has landed for every wave, and every wave is done reading the other stage
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const double2* As = lds + buf * STAGE;
      const double2* Bs = As + A_SLOTS;
      buf ^= 1;
      // all fragments of the chunk before the next loads start: an LDS read after
      // them would wait for them
      double2 bf[NT_RN][2], af[RM][4];
#pragma unroll
      for (int j = 0; j < NT_RN; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          bf[j][h] = Bs[(wave * 16 * NT_RN + 16 * j + l16) * 8 + ((2 * q + h) ^ (l16 & 7))];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < RM; ++i) af[i][k] = As[(16 * i + l16) * 16 + ((4 * q + k) ^ l16)];
      if (c + 1 < c_end) fetch(c + 1, lds + buf * STAGE);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < NT_RN; ++j) {
            const double b = (k & 1) ? bf[j][k >> 1].y : bf[j][k >> 1].x;
            re[i][j] = mfma64(af[i][k].x, b, re[i][j]);
            im[i][j] = mfma64(af[i][k].y, b, im[i][j]);
          }
      if (c + 1 < c_end) stash(lds + buf * STAGE);
    }
  }

#pragma unroll
  for (int j = 0; j < NT_RN; ++j) {
    const int64_t c = col0 + wave * 16 * NT_RN + 16 * j + l16;
    if (c >= a.n) continue;
    int ti = 0, tj = 0;
    if (EPI == NT_EPI_VHS) {
      ti = a.tri_i[c];
      tj = a.tri_j[c];
    }
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t w = row0 + 16 * i + 4 * r + q;
        if (w >= a.m) continue;
        if (EPI == NT_EPI_PART) {
          st(a.out, ((int64_t)z * a.m + w) * a.n + c, cmake(a.scale * re[i][j][r], a.scale * im[i][j][r]));
        } else {
          // i scale (re + i im), to both triangles
          const cplx v = cmake(-a.scale * im[i][j][r], a.scale * re[i][j][r]);
          double* base = a.out + 2 * w * a.nbasis * a.nbasis;
          st(base, (int64_t)ti * a.nbasis + tj, v);
          if (ti != tj) st(base, (int64_t)tj * a.nbasis + ti, v);
        }
      }
  }
}

// Cost of a launch in units of one 16-row tile's MFMA time per K chunk (1024
// cycles): the workgroups of the fullest CU (a fraction of one once there are
// many rounds), each its chunks and about two chunks' worth of start and
// epilogue, a tenth of a tile per chunk for the B columns each row tile reads again.
double nt_cost(int64_t m, int64_t colblocks, int rm, double chunks) {
  const double rounds = (double)(ceil_div(m, 16 * rm) * colblocks) / 256.0;
  return (rounds < 4.0 ? std::ceil(rounds) : rounds) * (chunks + 2.0) * (rm + 0.1);
}

// Rows per workgroup tile, in 16s (1 .. most): the least padding of m on a full
// GPU; smaller tiles where larger ones would leave CUs idle.
int nt_rows(int64_t m, int64_t colblocks, double chunks, int most) {
  int best = 1;
  for (int rm = 2; rm <= most; ++rm)
    if (nt_cost(m, colblocks, rm, chunks) < 0.999 * nt_cost(m, colblocks, best, chunks)) best = rm;
  return best;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int RM, int EPI>
hipError_t launch_nt_rm(const NtArgs& a, bool direct, dim3 grid, hipStream_t stream) {
  if (direct) hipLaunchKernelGGL((nt64_kernel<RM, NT_DIRECT, EPI>), grid, dim3(NT_THREADS), 0, stream, a);
  else hipLaunchKernelGGL((nt64_kernel<RM, NT_BREG, EPI>), grid, dim3(NT_THREADS), 0, stream, a);
  return hipGetLastError();
}

template <int EPI>
hipError_t launch_nt(const NtArgs& a, hipStream_t stream) {
  if (a.m < 1 || a.n < 1 || a.nseg < 1 || a.nseg > 2 || a.ksplit < 1) return hipErrorInvalidValue;
  bool a_vec = true, b_vec = true;
  for (int s = 0; s < a.nseg; ++s) {
    const NtSegment& g = a.seg[s];
    // 32-bit byte offsets within a tile (64 complex rows, 128 real columns)
    if (g.K < 1 || g.lda < g.K || g.ldb < g.K || g.lda > (1 << 22) || g.ldb > (1 << 22)) return hipErrorInvalidValue;
    a_vec = a_vec && aligned16(g.A);
    b_vec = b_vec && g.K % 2 == 0 && g.ldb % 2 == 0 && aligned16(g.B);
  }
  const int64_t nbn = ceil_div(a.n, NT_TN);
  int64_t chunks = 0;
  for (int s = 0; s < a.nseg; ++s) chunks += ceil_div(a.seg[s].K, NT_KC);
  // (64 rows do not fit the registers beside B's)
  const int rm = a_vec ? nt_rows(a.m, nbn * a.ksplit, (double)chunks / a.ksplit, b_vec ? 4 : 3) : 1;
  const int64_t blocks = nbn * ceil_div(a.m, 16 * rm);
  if (blocks > INT32_MAX || a.ksplit > 65535) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks, a.ksplit);
  if (!a_vec) {
    hipLaunchKernelGGL((nt64_kernel<1, NT_REG, EPI>), grid, dim3(NT_THREADS), 0, stream, a);
    return hipGetLastError();
  }
  switch (rm) {
    case 1: return launch_nt_rm<1, EPI>(a, b_vec, grid, stream);
    case 2: return launch_nt_rm<2, EPI>(a, b_vec, grid, stream);
    case 3: return launch_nt_rm<3, EPI>(a, b_vec, grid, stream);
    default:
      hipLaunchKernelGGL((nt64_kernel<4, NT_DIRECT, EPI>), grid, dim3(NT_THREADS), 0, stream, a);
      return hipGetLastError();
  }
}

}  // namespace

int nt64_ksplit(int64_t m, int64_t n, int64_t chunks, int most) {
  const int64_t nbn = ceil_div(n, NT_TN);
  // a further range writes and reads m n partial sums: 32 bytes each at 4.4 TB/s, in units of 0.43 us
  const double part = (double)m * n * 32.0 / 4.4e12 / 0.43e-6;
  int best = 1;
  double least = 0.0;
  for (int ks = 1; ks <= most && 2 * ks <= std::max<int64_t>(chunks, 2); ++ks) {
    const double each = (double)ceil_div(chunks, ks);
    const double t = nt_cost(m, nbn * ks, nt_rows(m, nbn * ks, each, 4), each) + part * ks;
    if (ks == 1 || t < 0.98 * least) {
      best = ks;
      least = t;
    }
  }
  return best;
}

hipError_t launch_nt64(const NtArgs& a, hipStream_t stream) {
  return a.tri_i ? launch_nt<NT_EPI_VHS>(a, stream) : launch_nt<NT_EPI_PART>(a, stream);
}

}  // namespace afqmc
