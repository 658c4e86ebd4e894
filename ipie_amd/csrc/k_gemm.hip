// FP64 products that propagate the walkers, on v_mfma_f64_16x16x4f64:
//   * one body   out[w] = expH1_s phi_s[w], both spins in one launch
//                (ipie/propagation/operations.py:26-55)
//   * Taylor     exp(V) P by Horner's rule, T <- P + (V T) / k for k = n .. 1
//                (operations.py:85-117 sums the same terms), V = VHS[w] symmetric and
//                held as its packed upper triangle; one launch per k, or for N <= 256
//                one for the series
//
// Both are bound by the FP64 matrix pipe (one 16x16x4 MFMA takes 64 cycles); the
// fragments come from LDS, staged in K chunks of 16 by direct global-to-LDS
// loads, each read under the MFMAs of the step before, one barrier per chunk
// (as in k_nt64.hip; unlike fragments loaded straight from memory by every wave,
// whose accumulators the compiler also moved between register files every chunk).
// Columns are real columns: a complex value takes two neighbouring ones, so a
// 16-column tile holds 8 complex columns and at most 15 real columns of padding
// are multiplied.

#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

// LDS is read through vector types: the compiler makes other reads wait for every
// direct load in flight
typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v1d __attribute__((ext_vector_type(1)));

constexpr int PG_KC = 16;       // K per LDS stage
constexpr int PG_THREADS = 256;  // four waves

__device__ double2 pg_zero;  // source of values past K

__device__ __forceinline__ void pg_load16(const char* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

__device__ __forceinline__ void pg_load4(const char* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}

// address of 16 zero bytes, kept in scalar registers
__device__ __forceinline__ const char* pg_zeros() {
  const char* z = reinterpret_cast<const char*>(&pg_zero);
  asm volatile("" : "+s"(z));
  return z;
}

// workgroup barrier: this wave's LDS reads are done, at most N of its loads in flight
template <int N>
__device__ __forceinline__ void pg_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// ends a block of up to N LDS reads and the MFMAs that run over them: the reads go first
template <int N>
__device__ __forceinline__ void pg_reads_first() {
  __builtin_amdgcn_sched_group_barrier(0x100, N, 0);
  __builtin_amdgcn_sched_group_barrier(0x008, 100, 0);
  __builtin_amdgcn_sched_barrier(0);
}

// ---------------------------------------------------------------- one body
// Workgroup tile: 16 RM rows of expH1 x 128 real columns (64 walker columns of
// one spin, over the walkers), 32 of them per wave.  LDS: row r of A keeps its
// pair p of K values in slot r 8 + (p ^ (r % 8)); B is K rows of 64 complex values.
// expH1 is read where the caller keeps it, in every call.  Its rows are 16-byte aligned
// for even N; for odd N they are loaded 4 bytes a lane, and so are walkers off 16 bytes
// (a caller of the C entry points), with 16-row tiles.
enum { OB_16 = 0, OB_A4 = 1, OB_AB4 = 2 };
template <int RM, int MODE>
struct ObPlan {
  static constexpr int A_LOADS = MODE == OB_16 ? (2 * RM + 3) / 4 : 2 * RM, B_LOADS = MODE == OB_AB4 ? 16 : 4;  // per wave
  static constexpr int LOADS = A_LOADS + B_LOADS;
  static constexpr int A_SLOTS = MODE == OB_16 ? 256 * A_LOADS : 128 * RM, STAGE = A_SLOTS + 1024;
  static constexpr int STAGES = RM == 1 ? 4 : RM <= 4 ? 3 : 2;
  static constexpr int LDS_BYTES = 16 * STAGE * STAGES;
  static_assert(2 * LDS_BYTES <= 160 * 1024 && (STAGES - 1) * LOADS <= 63, "two workgroups per CU, vmcnt");
};

template <int RM, int MODE>
__global__ void __launch_bounds__(PG_THREADS, 2) one_body64_kernel(OneBody64Args a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  using P = ObPlan<RM, MODE>;
  constexpr int ST = P::STAGES, TM = 16 * RM;
  extern __shared__ uint4 pg_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int N = a.nbasis, nrb = (int)ceil_div(N, TM);
  // row blocks fastest: the workgroups that run together share their columns in L2
  int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t blocks0 = ceil_div((int64_t)a.nwalkers * a.spin[0].n, 64);
  const int rb = lin % nrb;
  int64_t cb = lin / nrb;
  const int s = cb < blocks0 ? 0 : 1;
  if (s) cb -= blocks0;
  const OneBody64Spin sp = s == 0 ? a.spin[0] : a.spin[1];
  const int row0 = rb * TM;
  const int64_t ncols = (int64_t)a.nwalkers * sp.n;  // complex columns (w, c)

  // this lane's staged rows (byte offset, first K value) and column
  uint32_t ao[P::A_LOADS];
  int ak[P::A_LOADS];
#pragma unroll
  for (int j = 0; j < P::A_LOADS; ++j) {
    const int t = MODE == OB_16 ? (wave * P::A_LOADS + j) * 64 + lane : (wave * P::A_LOADS + j) * 16 + (lane >> 2);
    const int r = t >> 3, p = (t & 7) ^ (r & 7), part = MODE == OB_16 ? 0 : lane & 3;  // part: 4 bytes of a pair
    ak[j] = 2 * p + (part >> 1);
    ao[j] = 8u * ((uint32_t)min(r, N - 1 - row0) * (uint32_t)N + 2 * p) + 4 * part;
  }
  const char* abase = reinterpret_cast<const char*>(sp.exp + (int64_t)row0 * N);
  const char* zero = pg_zeros();
  constexpr int BC = MODE == OB_AB4 ? 4 : 1;  // loads of a K row: 64 columns, or 16 of 4 x 4 bytes
  const char* bcol[BC];
#pragma unroll
  for (int h = 0; h < BC; ++h) {
    const int64_t col = min(64 * cb + (MODE == OB_AB4 ? 16 * h + (lane >> 2) : lane), ncols - 1);
    bcol[h] = reinterpret_cast<const char*>(sp.src + 2 * (col / sp.n * sp.src_ws + sp.src_off + col % sp.n)) +
              (MODE == OB_AB4 ? 4 * (lane & 3) : 0);
  }
  const int nch = (int)ceil_div(N, PG_KC);
  auto fetch = [&](int c) {  // (zeros past N)
    const int cc = min(c, nch - 1);
    uint4* As = pg_lds + c % ST * P::STAGE;
    uint4* Bs = As + P::A_SLOTS;
#pragma unroll
    for (int j = 0; j < P::A_LOADS; ++j) {
      const char* p = PG_KC * cc + ak[j] < N ? abase + ao[j] + 8 * PG_KC * cc : zero;
      if constexpr (MODE == OB_16) pg_load16(p, As + (wave * P::A_LOADS + j) * 64);
      else pg_load4(p, As + (wave * P::A_LOADS + j) * 16);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = PG_KC * cc + 4 * wave + j;
#pragma unroll
      for (int h = 0; h < BC; ++h) {
        const char* p = bcol[h] + 16 * (int64_t)k * sp.src_ld;
        if constexpr (MODE == OB_AB4) pg_load4(k < N ? p : zero, Bs + (4 * wave + j) * 64 + 16 * h);
        else pg_load16(k < N ? p : zero, Bs + (4 * wave + j) * 64);
      }
    }
  };
  auto read = [&](int c, int h, v2d (&af)[RM], double (&bf)[2][2]) {
    const v2d* As = reinterpret_cast<const v2d*>(pg_lds + c % ST * P::STAGE);
    const double* Bs = reinterpret_cast<const double*>(pg_lds + c % ST * P::STAGE + P::A_SLOTS);
#pragma unroll
    for (int i = 0; i < RM; ++i) af[i] = As[(16 * i + l16) * 8 + ((2 * q + h) ^ (l16 & 7))];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bf[j][k] = reinterpret_cast<const v1d*>(Bs + (4 * q + 2 * h + k) * 128 + 32 * wave + 16 * j + l16)[0][0];
  };
  v4d acc[RM][2];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero4d();
  auto multiply = [&](const v2d (&af)[RM], const double (&bf)[2][2]) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma64(af[i][k], bf[j][k], acc[i][j]);
  };
  v2d af0[RM], af1[RM];
  double bf0[2][2], bf1[2][2];
  for (int t = 0; t < ST; ++t) fetch(t);
  pg_barrier<(ST - 1) * P::LOADS>();
  read(0, 0, af0, bf0);
  for (int c = 0; c < nch; ++c) {
    read(c, 1, af1, bf1);
    multiply(af0, bf0);
    pg_reads_first<RM + 4>();
    pg_barrier<(ST - 2) * P::LOADS>();
    __builtin_amdgcn_sched_barrier(0);
    read(c + 1, 0, af0, bf0);
    fetch(c + ST);
    multiply(af1, bf1);
    __builtin_amdgcn_sched_group_barrier(0x100, RM + 4, 0);
#pragma unroll
    for (int t = 0; t < P::LOADS; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x006, 10, 0);
      __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  pg_barrier<0>();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int rc = 32 * wave + 16 * j + l16;  // real column
    const int64_t cc = 64 * cb + (rc >> 1);
    if (cc >= ncols) continue;
    double* o = sp.out + 2 * (cc / sp.n * sp.out_ws + sp.out_off + cc % sp.n) + (rc & 1);
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + 16 * i + 4 * r + q;
        if (row < N) o[2 * (int64_t)row * sp.out_ld] = acc[i][j][r];
      }
  }
}

// ---------------------------------------------------------------- Taylor
// out[w] = base[w] + alpha V[w] prev[w]: workgroup tile 64 rows x 8 RN complex
// columns of one walker, 16 rows per wave.
//
// A wave stages its own 16 x 16 block of V per chunk.  Left of the diagonal the
// block is read as the mirror of the stored one (K rows of 16 values of r), on it
// value by value, right of it as stored, so that a load always takes runs of 256
// bytes: slot u 16 + (v ^ u), u the stored row, v the stored column.
// B is 16 K rows of 8 RN complex values.  Real column 2 c of the result is
// V_re B_re - V_im B_im and column 2 c + 1 is V_re B_im + V_im B_re: each lane reads
// its own and the other part of its complex column, the other one's sign
// flipped in the even lanes.
template <int RN>
struct TyPlan {
  static constexpr int B_LOADS = (RN + 1) / 2, LOADS = 4 + B_LOADS;  // per wave
  static constexpr int A_SLOTS = 1024, STAGE = A_SLOTS + 256 * B_LOADS;
  static constexpr int STAGES = RN <= 4 ? 3 : 2;
  static constexpr int LDS_BYTES = 16 * STAGE * STAGES;
  static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per CU");
};

template <int RN>
__global__ void __launch_bounds__(PG_THREADS, 2) taylor64_kernel(Taylor64Args a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  using P = TyPlan<RN>;
  constexpr int ST = P::STAGES;
  extern __shared__ uint4 pg_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int N = a.nbasis, nrb = (int)ceil_div(N, 64);
  // column blocks, then row blocks of a walker together: they share V in L2
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int cb = lin % a.colblocks, rb = lin / a.colblocks % nrb;
  const int64_t w = lin / a.colblocks / nrb;
  const int c0 = cb * a.colwidth, cw = min(a.colwidth, a.ncol - c0);
  const int row0 = 64 * rb + 16 * wave;
  const bool active = row0 < N;
  const char* V = reinterpret_cast<const char*>(a.vhs + w * ((int64_t)N * (N + 1)));  // complex [N (N + 1) / 2]
  const char* zero = pg_zeros();

  // B's slots of this lane: byte offsets from a chunk's first row, and its K row
  // (none for the columns past the block)
  const char* prev = reinterpret_cast<const char*>(a.prev + 2 * (w * N * a.ncol + c0));
  uint32_t bo[P::B_LOADS];
  int bk[P::B_LOADS];
#pragma unroll
  for (int j = 0; j < P::B_LOADS; ++j) {
    const int t = (wave * P::B_LOADS + j) * 64 + lane, k = t / (8 * RN), col = t % (8 * RN);
    bk[j] = t < 128 * RN && col < cw ? k : PG_KC;
    bo[j] = 16u * ((uint32_t)k * (uint32_t)a.ncol + col);
  }
  const int nch = (int)ceil_div(N, PG_KC);
  // starts the loads of chunk c (zeros past K; straight-line, so that the addresses
  // are computed between MFMAs)
  auto fetch = [&](int c) {
    const int k0 = PG_KC * c, left = N - k0;
    uint4* As = pg_lds + c % ST * P::STAGE + wave * 256;
    uint4* Bs = pg_lds + c % ST * P::STAGE + P::A_SLOTS + wave * P::B_LOADS * 64;
    const bool mirror = row0 > k0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = 4 * j + (lane >> 4), v = (lane & 15) ^ u;
      const int r = min(row0 + (mirror ? v : u), N - 1), k = k0 + (mirror ? u : v);
      const int lo = min(r, k), hi = max(r, k);
      uint32_t at = __umul24(lo, 2 * N - lo - 1) / 2 + hi;  // packed index
      asm volatile("" : "+v"(at));
      const char* p = V + ((uint64_t)at << 4);
      pg_load16(k < N ? p : zero, As + 64 * j);
    }
    const char* row = prev + (int64_t)k0 * a.ncol * 16;
#pragma unroll
    for (int j = 0; j < P::B_LOADS; ++j) {
      const char* p = row + bo[j];
      pg_load16(bk[j] < min(left, PG_KC) ? p : zero, Bs + j * 64);
    }
  };
  // K step s of chunk c: V (re, im), own and other part of the columns
  auto read = [&](int c, int s, v2d& af, double (&own)[RN], double (&other)[RN]) {
    const v2d* As = reinterpret_cast<const v2d*>(pg_lds + c % ST * P::STAGE + wave * 256);
    const v1d* Bs = reinterpret_cast<const v1d*>(pg_lds + c % ST * P::STAGE + P::A_SLOTS) + (4 * q + s) * 16 * RN;
    const int k = 4 * q + s;
    af = As[row0 > PG_KC * c ? 16 * k + (l16 ^ k) : 16 * l16 + (k ^ l16)];
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      own[j] = Bs[16 * j + l16][0];
      other[j] = Bs[16 * j + (l16 ^ 1)][0];
    }
  };
  const uint32_t flip = (l16 & 1) ? 0u : 0x80000000u;
  v4d acc[RN];
#pragma unroll
  for (int j = 0; j < RN; ++j) acc[j] = zero4d();
  auto multiply = [&](const v2d& af, const double (&own)[RN], const double (&other)[RN]) {
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      const double o = __hiloint2double(__double2hiint(other[j]) ^ flip, __double2loint(other[j]));
      acc[j] = mfma64(af[0], own[j], acc[j]);
      acc[j] = mfma64(af[1], o, acc[j]);
    }
  };
  v2d af0, af1;
  double own0[RN], own1[RN], other0[RN], other1[RN];
  for (int t = 0; t < ST; ++t) fetch(t);
  pg_barrier<(ST - 1) * P::LOADS>();
  if (!active) {  // rows past the matrix: only this wave's share of B
    for (int c = 0; c < nch; ++c) {
      pg_barrier<(ST - 2) * P::LOADS>();
      fetch(c + ST);
    }
    pg_barrier<0>();
    return;
  }
  read(0, 0, af0, own0, other0);
  for (int c = 0; c < nch; ++c) {
    read(c, 1, af1, own1, other1);
    multiply(af0, own0, other0);
    pg_reads_first<2 * RN + 1>();
    read(c, 2, af0, own0, other0);
    multiply(af1, own1, other1);
    pg_reads_first<2 * RN + 1>();
    read(c, 3, af1, own1, other1);
    multiply(af0, own0, other0);
    pg_reads_first<2 * RN + 1>();
    pg_barrier<(ST - 2) * P::LOADS>();
    __builtin_amdgcn_sched_barrier(0);
    read(c + 1, 0, af0, own0, other0);
    fetch(c + ST);
    multiply(af1, own1, other1);
    __builtin_amdgcn_sched_group_barrier(0x100, RN + 1, 0);
#pragma unroll
    for (int t = 0; t < P::LOADS; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * RN >= P::LOADS + 4 ? 2 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x006, 16, 0);
      __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  pg_barrier<0>();
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int rc = 16 * j + l16;
    if (rc >= 2 * cw) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 4 * r + q;
      if (row >= N) continue;
      const int64_t off = 2 * (w * N * a.ncol + (int64_t)row * a.ncol + c0) + rc;
      a.out[off] = a.base[off] + a.alpha * acc[j][r];
    }
  }
}

// The whole series for one walker's block of 8 RN complex columns: T stays in LDS and
// each wave owns 16 rows (at most 16 waves).  A launch per term costs more than a
// small matrix's products, and reads and writes T and pays its start and end six
// times.  NCH > 0: N is at most 16 NCH <= 128 and the wave keeps its rows of V in
// registers over the series (a chunk's products are shorter than a load from
// L2); NCH = 0: V is read straight into fragments, a chunk ahead, once per term.  The lane
// group q takes K = 4 s + q of MFMA step s, so that a load takes four neighbouring
// values of a row (or, mirrored, 16 of a stored row).
template <int NCH, int RN>
__global__ void __launch_bounds__(NCH > 0 ? 512 : 1024) taylor64_series_kernel(Taylor64Args a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  extern __shared__ uint4 pg_lds[];
  constexpr bool KEEP = NCH > 0 || RN <= 2;  // the base in registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int N = a.nbasis, nch = NCH > 0 ? NCH : (int)ceil_div(N, 16);
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int cb = lin % a.colblocks;
  const int64_t w = lin / a.colblocks;
  const int c0 = cb * a.colwidth, cw = min(a.colwidth, a.ncol - c0);
  const char* V = reinterpret_cast<const char*>(a.vhs + w * ((int64_t)N * (N + 1)));
  const double* base = a.base + 2 * (w * N * a.ncol + c0);
  double* out = a.out + 2 * (w * N * a.ncol + c0);
  v1d* T = reinterpret_cast<v1d*>(pg_lds);  // [16 nch][16 RN] real columns
  const char* zero = pg_zeros();

  // V[r][k] of this lane's row for the chunks 0, 1, .. in turn.  Left of the
  // diagonal block the mirrored element V[k][r]: its packed index grows by
  // 16 N + 120 - 16 k to the chunk of k; right of it the four steps are at fixed
  // distances in the row.
  typedef const __attribute__((address_space(1))) v2d* gv2d;
  const int r = min(16 * wave + l16, N - 1);
  uint32_t left[4];
  auto packed = [&](int k) {
    const int lo = min(r, k), hi = max(r, k);
    return __umul24(lo, 2 * N - lo - 1) / 2 + hi;
  };
  auto fetch = [&](int c, v2d (&af)[4]) {
    if (c < wave) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = 16 * c + 4 * s + q;
        left[s] = c == 0 ? packed(k) : left[s] + (16 * N + 120 - 16 * k);
        af[s] = *(gv2d)(V + ((uint64_t)left[s] << 4));
      }
    } else if (c > wave && 16 * c + 16 <= N) {
      const char* p = V + ((uint64_t)(packed(r) + 16 * c + q - r) << 4);
#pragma unroll
      for (int s = 0; s < 4; ++s) af[s] = *(gv2d)(p + 64 * s);
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int k = 16 * c + 4 * s + q;
        const char* p = V + ((uint64_t)packed(min(k, N - 1)) << 4);
        af[s] = *(gv2d)(k < N ? p : zero);
      }
    }
  };
  v2d vf[NCH > 0 ? NCH : 2][4];
#pragma unroll
  for (int c = 0; c < (NCH > 0 ? NCH : 1); ++c) fetch(c, vf[c]);

  for (int e = threadIdx.x; e < 16 * nch * 16 * RN; e += blockDim.x) {
    const int k = e / (16 * RN), rc = e % (16 * RN);
    T[e][0] = k < N && rc < 2 * cw ? base[2 * (int64_t)k * a.ncol + rc] : 0.0;
  }
  const uint32_t flip = (l16 & 1) ? 0u : 0x80000000u;
  v4d acc[RN], keep[KEEP ? RN : 1];
  // one chunk's products, each step's columns read under the step before
  auto chunk = [&](int c, const v2d (&af)[4]) {
    double own[2][RN], other[2][RN];
    auto read = [&](int s) {
      const v1d* row = T + (16 * c + 4 * s + q) * 16 * RN;
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        own[s & 1][j] = row[16 * j + l16][0];
        other[s & 1][j] = row[16 * j + (l16 ^ 1)][0];
      }
    };
    read(0);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s < 3) read(s + 1);
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        const double ot = other[s & 1][j];
        const double o = __hiloint2double(__double2hiint(ot) ^ flip, __double2loint(ot));
        acc[j] = mfma64(af[s][0], own[s & 1][j], acc[j]);
        acc[j] = mfma64(af[s][1], o, acc[j]);
      }
    }
  };
  const int row0 = 16 * wave + q;  // this lane's results: rows row0 + 4 r, real columns 16 j + l16
  auto base_at = [&](int j, int i) {
    const int row = row0 + 4 * i, rc = 16 * j + l16;
    return row < N && rc < 2 * cw ? base[2 * (int64_t)row * a.ncol + rc] : 0.0;
  };
  if (KEEP) {
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) keep[KEEP ? j : 0][i] = base_at(j, i);
  }
  __syncthreads();
  for (int n = a.terms; n >= 1; --n) {
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[j] = zero4d();
    if constexpr (NCH > 0) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) chunk(c, vf[c]);
    } else {
      // the next chunk's loads (at the end the next term's first) go first
      for (int c = 0; c < nch; c += 2) {
        fetch(c + 1 < nch ? c + 1 : 0, vf[1]);
        chunk(c, vf[0]);
        if (c + 1 >= nch) {
#pragma unroll
          for (int s = 0; s < 4; ++s) vf[0][s] = vf[1][s];
          break;
        }
        fetch(c + 2 < nch ? c + 2 : 0, vf[0]);
        chunk(c + 1, vf[1]);
      }
    }
    const double alpha = 1.0 / n;
    __syncthreads();  // every wave has read T
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + 4 * i, rc = 16 * j + l16;
        const double t = (KEEP ? keep[KEEP ? j : 0][i] : base_at(j, i)) + alpha * acc[j][i];
        if (n > 1) {
          if (row < N) T[row * 16 * RN + rc][0] = t;
        } else if (row < N && rc < 2 * cw) {
          out[2 * (int64_t)row * a.ncol + rc] = t;
        }
      }
    __syncthreads();
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int RM, int MODE>
hipError_t launch_ob_as(const OneBody64Args& a, int64_t colblocks, hipStream_t stream) {
  const int64_t blocks = colblocks * ceil_div(a.nbasis, 16 * RM);
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  constexpr int lds = ObPlan<RM, MODE>::LDS_BYTES;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(one_body64_kernel<RM, MODE>), lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((one_body64_kernel<RM, MODE>), dim3((unsigned)blocks), dim3(PG_THREADS), lds, stream, a);
  return hipGetLastError();
}

template <int RM>
hipError_t launch_ob_rm(const OneBody64Args& a, int64_t colblocks, hipStream_t stream) {
  bool aligned = a.nbasis % 2 == 0;
  for (int s = 0; s < a.nspin; ++s) aligned = aligned && aligned16(a.spin[s].exp);
  return aligned ? launch_ob_as<RM, OB_16>(a, colblocks, stream) : launch_ob_as<RM, OB_A4>(a, colblocks, stream);
}

template <int RN>
hipError_t launch_ty_rn(const Taylor64Args& a, hipStream_t stream) {
  const int64_t blocks = (int64_t)a.nwalkers * ceil_div(a.nbasis, 64) * a.colblocks;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(taylor64_kernel<RN>), TyPlan<RN>::LDS_BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(taylor64_kernel<RN>, dim3((unsigned)blocks), dim3(PG_THREADS), TyPlan<RN>::LDS_BYTES, stream, a);
  return hipGetLastError();
}

template <int NCH, int RN>
hipError_t launch_ty_series(const Taylor64Args& a, hipStream_t stream) {
  const int64_t blocks = (int64_t)a.nwalkers * a.colblocks;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  const unsigned tiles = (unsigned)ceil_div(a.nbasis, 16);
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(taylor64_series_kernel<NCH, RN>), tiles * 2048 * RN);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((taylor64_series_kernel<NCH, RN>), dim3((unsigned)blocks), dim3(64 * tiles), tiles * 2048 * RN,
                     stream, a);
  return hipGetLastError();
}

template <int NCH>
hipError_t launch_ty_series_rn(const Taylor64Args& a, hipStream_t stream) {
  switch (a.colwidth / 8) {
    case 1: return launch_ty_series<NCH, 1>(a, stream);
    case 2: return launch_ty_series<NCH, 2>(a, stream);
    default: return launch_ty_series<NCH, 3>(a, stream);
  }
}

}  // namespace

hipError_t launch_one_body64(const OneBody64Args& a, hipStream_t stream) {
  if (a.nwalkers < 1 || a.nspin < 1 || a.nspin > 2 || a.nbasis < 1 || a.nbasis > (1 << 20)) return hipErrorInvalidValue;
  int64_t colblocks = 0;
  for (int s = 0; s < a.nspin; ++s) {
    if (a.spin[s].n < 1) return hipErrorInvalidValue;
    colblocks += ceil_div((int64_t)a.nwalkers * a.spin[s].n, 64);
  }
  for (int s = 0; s < a.nspin; ++s)
    if (!aligned16(a.spin[s].src)) return launch_ob_as<1, OB_AB4>(a, colblocks, stream);
  // Row tiles of 16 RM: the least padding of N, against half a 16-row tile per
  // workgroup for the columns it reads again; smaller ones while CUs would idle.
  int best = 1;
  double cost = 0.0;
  for (int rm = 1; rm <= 5; ++rm) {
    const double rounds = (double)(colblocks * ceil_div(a.nbasis, 16 * rm)) / 256.0;
    const double t = (rounds < 1.0 ? 1.0 : rounds) * (rm + 0.5);
    if (rm == 1 || t < 0.999 * cost) {
      best = rm;
      cost = t;
    }
  }
  switch (best) {
    case 1: return launch_ob_rm<1>(a, colblocks, stream);
    case 2: return launch_ob_rm<2>(a, colblocks, stream);
    case 3: return launch_ob_rm<3>(a, colblocks, stream);
    case 4: return launch_ob_rm<4>(a, colblocks, stream);
    default: return launch_ob_rm<5>(a, colblocks, stream);
  }
}

// The series in one launch: at most 16 row tiles, T in LDS.  Column blocks of 8, 16 or
// 24: the least time of the fullest CU.  One workgroup a CU takes (us for 8, 16, 24
// columns, 6 terms) 13, 22, 32 at N = 64, 35, 62, 91 at N = 128, 120, 194, 290 at N = 200 and
// 183, 250, 371 at N = 255: a time for every 8 columns and a fixed part, 0.1 to 0.4 of it up
// to N = 200 and as much at N = 255.  The rule takes 0.14.
bool taylor64_in_one(int nbasis) { return nbasis <= 256; }

hipError_t launch_taylor64_series(Taylor64Args a, hipStream_t stream) {
  if (a.nwalkers < 1 || a.ncol < 1 || a.nbasis < 1 || !taylor64_in_one(a.nbasis) || a.terms < 1)
    return hipErrorInvalidValue;
  const int tiles = (int)ceil_div(a.nbasis, 16);
  int best = 1;
  double least = 0.0;
  for (int rn = 1; rn <= 3; ++rn) {
    const int64_t blocks = (int64_t)a.nwalkers * ceil_div(a.ncol, 8 * rn);
    const double rounds = blocks < 1024 ? (double)ceil_div(blocks, 256) : blocks / 256.0;
    const double t = rounds * (rn + 0.138);
    if (rn == 1 || t < 0.99 * least) {
      best = rn;
      least = t;
    }
  }
  // (blocks of equal width)
  a.colblocks = (int)ceil_div(a.ncol, 8 * best);
  a.colwidth = (int)ceil_div(ceil_div(a.ncol, a.colblocks), 8) * 8;
  a.colblocks = (int)ceil_div(a.ncol, a.colwidth);
  switch (tiles) {
    case 1: return launch_ty_series_rn<1>(a, stream);
    case 2: return launch_ty_series_rn<2>(a, stream);
    case 3: return launch_ty_series_rn<3>(a, stream);
    case 4: return launch_ty_series_rn<4>(a, stream);
    case 5: return launch_ty_series_rn<5>(a, stream);
    case 6: return launch_ty_series_rn<6>(a, stream);
    case 7: return launch_ty_series_rn<7>(a, stream);
    case 8: return launch_ty_series_rn<8>(a, stream);
    default: return launch_ty_series_rn<0>(a, stream);
  }
}

hipError_t launch_taylor64(Taylor64Args a, hipStream_t stream) {
  if (a.nwalkers < 1 || a.ncol < 1 || a.nbasis < 1 || a.nbasis > 65535) return hipErrorInvalidValue;
  // Columns in blocks of at most 80: as few as hold them, more while the grid
  // would leave CUs idle and a block keeps 16 columns.
  const int64_t rows = (int64_t)a.nwalkers * ceil_div(a.nbasis, 64);
  int nb = (int)ceil_div(a.ncol, 80);
  while (rows * nb < 512 && ceil_div(a.ncol, nb + 1) >= 16) ++nb;
  a.colwidth = (int)ceil_div(ceil_div(a.ncol, nb), 8) * 8;
  a.colblocks = (int)ceil_div(a.ncol, a.colwidth);
  switch (a.colwidth / 8) {
    case 1: return launch_ty_rn<1>(a, stream);
    case 2: return launch_ty_rn<2>(a, stream);
    case 3: return launch_ty_rn<3>(a, stream);
    case 4: return launch_ty_rn<4>(a, stream);
    case 5: return launch_ty_rn<5>(a, stream);
    case 6: return launch_ty_rn<6>(a, stream);
    case 7: return launch_ty_rn<7>(a, stream);
    case 8: return launch_ty_rn<8>(a, stream);
    case 9: return launch_ty_rn<9>(a, stream);
    default: return launch_ty_rn<10>(a, stream);
  }
}

}  // namespace afqmc
