// FP64 contractions of complex rows with real rows, C[r, c] = sum_k A[r, k] B[c, k]
// (K contiguous in both), on v_mfma_f64_16x16x4f64:
//   * force bias   vbias[w, x] = sum_s sum_k Ghalf_s[w, k] rchol_s[x, k]
//                  (ipie/propagation/force_bias.py:79-121)
//   * VHS          VHS[w] = i sqrt(dt) sum_x xshifted[w, x] L_x, its packed upper
//                  triangle (ipie/propagation/phaseless_generic.py:67-97; not unpacked:
//                  the Taylor kernel reads the triangle)
//   * the exchange as a quadratic form, sum_b g_b (G W')_b over the block-triangular
//     W' (k_quad.hip), the dot products in the epilogue
//
// What bounds it: one 16x16x4 FP64 MFMA takes 64 cycles on gfx950, so the matrix
// pipe is the limit as soon as a wave always has its operands in registers.
// Fragments loaded straight from memory did not give that: each lane group read
// 16 rows at the row pitch (32 cache lines per load instruction), one K chunk
// ahead, with one wave per SIMD (296 VGPRs), and ran at 59% of the FP64 MFMA
// peak.  Here a workgroup of four waves stages K chunks of 16 through LDS with
// direct global-to-LDS loads (two to four stages, by the row tile; the next chunks'
// loads run under the current chunk's MFMAs, one barrier per chunk); a row's piece of a chunk is
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
#include <type_traits>

#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

// LDS is read through this vector type: a read through double2 makes the compiler
// wait for every direct load in flight before it
typedef double v2d __attribute__((ext_vector_type(2)));

constexpr int NT_KC = 16;                // K per LDS stage
constexpr int NT_RN = 2, NT_WAVES = 4;   // 16-column tiles per wave, waves side by side
constexpr int NT_TN = 16 * NT_RN * NT_WAVES;
static_assert(NT_TN == QUAD64_TILE, "column tile of W'");
constexpr int NT_THREADS = 64 * NT_WAVES;

__device__ double2 nt_zero;  // source of the slots past K

enum { NT_EPI_PART = 0, NT_EPI_QDOT = 1 };

// Direct global-to-LDS loads: lane l's 16 (4) bytes go to dst + 16 l (4 l).
__device__ __forceinline__ void nt_load16(const char* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void nt_load4(const char* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src, (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}

// Loads of 16 bytes a lane where the operand's rows are 16-byte aligned (and B's
// K even, so that a pair is whole or absent), of 4 bytes otherwise.  Byte offsets within
// a tile take 32 bits, but for NT_AB4, which also takes rows of more than 2^22 values.
enum { NT_16 = 0, NT_B4 = 1, NT_AB4 = 2 };

template <int RM, int MODE>
struct NtPlan {
  static constexpr int TM = 16 * RM;
  static constexpr int A_SLOTS = TM * NT_KC, B_SLOTS = NT_TN * NT_KC / 2, STAGE = A_SLOTS + B_SLOTS;
  static constexpr int A_LOADS = MODE == NT_AB4 ? 4 * RM : RM, B_LOADS = MODE == NT_16 ? 4 : 16;  // per wave
  static constexpr int LOADS = A_LOADS + B_LOADS;
  // LDS stages: a chunk of a small row tile is multiplied in less time than a
  // load takes, so more of them are in flight (two workgroups still fit a CU)
  static constexpr int STAGES = RM == 1 ? 4 : RM == 2 ? 3 : 2;
  static constexpr int LDS_BYTES = 16 * STAGE * STAGES;
  static_assert(2 * LDS_BYTES <= 160 * 1024 && STAGES * LOADS <= 63 + LOADS, "LDS and vmcnt");
};

template <int N>
__device__ __forceinline__ void nt_barrier() {
  // (this wave's LDS reads are waited for where the compiler sees it, or it waits
  // for the next ones too before their use)
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int RM, int MODE, int EPI>
__global__ void __launch_bounds__(NT_THREADS, 2) nt64_kernel(NtArgs a) {
  phase_mark(a.mark, blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0);
  using P = NtPlan<RM, MODE>;
  constexpr int TM = P::TM, ST = P::STAGES;
  extern __shared__ uint4 nt_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int nbm = (int)ceil_div(a.m, TM);
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  // (QDOT: row blocks x column units, otherwise x column tiles, with K ranges in y)
  const int bm = lin % nbm, bu = lin / nbm, z = blockIdx.y;
  int4 unit = make_int4(bu, 0, 0, 0);
  if (EPI == NT_EPI_QDOT) unit = a.units[bu];
  const int bn = unit.x;
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
    int c_begin = s == 0 ? z0 : max(z0, nch0) - nch0, c_end = s == 0 ? min(z1, nch0) : z1 - nch0;
    if (EPI == NT_EPI_QDOT) {
      c_begin = unit.y;
      c_end = unit.z;
    }
    if (c_begin >= c_end) continue;
    // sources of this lane: byte offsets from the tile's first row and column
    // (rows and columns past the end read the last one; their results are not
    // written) and first K index of each load
    const char* abase = reinterpret_cast<const char*>(sg.A + 2 * (int64_t)row0 * sg.lda);
    const char* bbase = reinterpret_cast<const char*>(sg.B + col0 * sg.ldb);
    const uint32_t last_r = (uint32_t)min((int64_t)TM, a.m - row0) - 1, last_c = (uint32_t)min((int64_t)NT_TN, a.n - col0) - 1;
    using offset = std::conditional_t<MODE == NT_AB4, uint64_t, uint32_t>;
    const offset apitch = 16u * (offset)sg.lda, bpitch = 8u * (offset)sg.ldb;
    auto a_row = [&](int j) { return MODE == NT_AB4 ? 4 * RM * wave + j : 4 * (RM * wave + j) + (lane >> 4); };
    auto a_k = [&](int j) { return (MODE == NT_AB4 ? lane >> 2 : lane & 15) ^ (a_row(j) & 15); };
    auto a_off = [&](int j) {
      return min((uint32_t)a_row(j), last_r) * apitch + 16u * a_k(j) + (MODE == NT_AB4 ? 4u * (lane & 3) : 0u);
    };
    auto b_col = [&](int j) { return MODE == NT_16 ? 8 * (4 * wave + j) + (lane >> 3) : 2 * (16 * wave + j) + (lane >> 5); };
    auto b_pair = [&](int j) { return (MODE == NT_16 ? lane & 7 : (lane & 31) >> 2) ^ (b_col(j) & 7); };
    auto b_k = [&](int j) { return 2 * b_pair(j) + (MODE == NT_16 ? 0 : (lane & 3) >> 1); };
    auto b_off = [&](int j) {
      return min((offset)b_col(j) * bpitch, last_c * bpitch) + 16u * b_pair(j) + (MODE == NT_16 ? 0u : 4u * (lane & 3));
    };
    offset ao[RM], bo[4];  // of the 16-byte loads
#pragma unroll
    for (int j = 0; j < RM; ++j) ao[j] = a_off(j);
#pragma unroll
    for (int j = 0; j < 4; ++j) bo[j] = b_off(j);
    // starts the loads of chunk c into its stage (zeros past K, and all zeros past
    // c_end: every iteration issues the same number of loads, so that a wait can
    // name the ones that may stay in flight, and has no branch, so that their
    // addresses are computed between MFMAs)
    auto fetch = [&](int c) {
      const int k0 = NT_KC * c, left = c < c_end ? sg.K - k0 : 0;
      uint4* As = nt_lds + (c - c_begin) % ST * P::STAGE;
      uint4* Bs = As + P::A_SLOTS;
      const char* ac = abase + 16 * (int64_t)k0;
      const char* bc = bbase + 8 * (int64_t)k0;
      const char* zero = reinterpret_cast<const char*>(&nt_zero);
#pragma unroll
      for (int j = 0; j < P::A_LOADS; ++j) {
        if constexpr (MODE == NT_AB4) nt_load4(a_k(j) < left ? ac + a_off(j) : zero, As + (4 * RM * wave + j) * 16);
        else nt_load16(a_k(j) < left ? ac + ao[j] : zero, As + (RM * wave + j) * 64);
      }
#pragma unroll
      for (int j = 0; j < P::B_LOADS; ++j) {
        if constexpr (MODE == NT_16) nt_load16(b_k(j) < left ? bc + bo[j] : zero, Bs + (4 * wave + j) * 64);
        else nt_load4(b_k(j) < left ? bc + b_off(j) : zero, Bs + (16 * wave + j) * 16);
      }
    };
    // fragments of half h (K pairs h of every lane group) of chunk c
    auto read = [&](int c, int h, v2d (&af)[RM][2], v2d (&bf)[NT_RN]) {
      const v2d* As = reinterpret_cast<const v2d*>(nt_lds + (c - c_begin) % ST * P::STAGE);
      const v2d* Bs = As + P::A_SLOTS;
#pragma unroll
      for (int j = 0; j < NT_RN; ++j) bf[j] = Bs[(wave * 16 * NT_RN + 16 * j + l16) * 8 + ((2 * q + h) ^ (l16 & 7))];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < RM; ++i) af[i][k] = As[(16 * i + l16) * 16 + ((4 * q + 2 * h + k) ^ l16)];
    };
    auto multiply = [&](const v2d (&af)[RM][2], const v2d (&bf)[NT_RN]) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < NT_RN; ++j) {
            re[i][j] = mfma64(af[i][k][0], bf[j][k], re[i][j]);
            im[i][j] = mfma64(af[i][k][1], bf[j][k], im[i][j]);
          }
    };
    // Each half's fragments are read while the other half is multiplied.  Between
    // the halves of chunk c: chunk c + 1 has landed for every wave (the later
    // ones stay in flight) and every wave has read all of chunk c, whose stage
    // takes chunk c + ST.
    v2d af0[RM][2], bf0[NT_RN], af1[RM][2], bf1[NT_RN];
    for (int t = 0; t < ST; ++t) fetch(c_begin + t);
    nt_barrier<(ST - 1) * P::LOADS>();
    read(c_begin, 0, af0, bf0);
    for (int c = c_begin; c < c_end; ++c) {
      read(c, 1, af1, bf1);
      multiply(af0, bf0);
      __builtin_amdgcn_sched_barrier(0);
      nt_barrier<(ST - 2) * P::LOADS>();
      __builtin_amdgcn_sched_barrier(0);
      read(c + 1, 0, af0, bf0);
      fetch(c + ST);
      multiply(af1, bf1);
      // the reads, then the loads with their address arithmetic spread over the MFMAs
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * RM + NT_RN, 0);
      constexpr int MF = 4 * RM * NT_RN, PER = P::LOADS > MF ? 2 : 1;
#pragma unroll
      for (int t = 0; t < (P::LOADS + PER - 1) / PER; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x006, 12 * PER, 0);
        __builtin_amdgcn_sched_group_barrier(0x010, PER, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    nt_barrier<0>();
  }

  if (EPI == NT_EPI_QDOT) {
    // per row: the dot of this wave's 32 columns with d, summed over the 16 lanes
    // of the row, then over the waves (LDS is free: every wave passed the last barrier)
    double2* part = reinterpret_cast<double2*>(nt_lds);  // [wave][row]
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + 4 * r + q;
        const int64_t w = min((int64_t)row0 + row, a.m - 1);
        cplx e = cmake(0.0, 0.0);
#pragma unroll
        for (int j = 0; j < NT_RN; ++j) {
          const int64_t c = col0 + wave * 16 * NT_RN + 16 * j + l16;
          if (c < a.n) cfma(e, ld(a.dg, w * a.n + c), cmake(re[i][j][r], im[i][j][r]));
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
          e.re += __shfl_xor(e.re, off, 64);
          e.im += __shfl_xor(e.im, off, 64);
        }
        if (l16 == 0) part[wave * TM + row] = make_double2(e.re, e.im);
      }
    __syncthreads();
    if (threadIdx.x < TM && row0 + (int64_t)threadIdx.x < a.m) {
      cplx e = cmake(0.0, 0.0);
      for (int v = 0; v < NT_WAVES; ++v) e = cadd(e, ld(reinterpret_cast<const double*>(part), v * TM + threadIdx.x));
      st(a.out, (int64_t)bu * a.m + row0 + threadIdx.x, e);
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < NT_RN; ++j) {
    const int64_t c = col0 + wave * 16 * NT_RN + 16 * j + l16;
    if (c >= a.n) continue;
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t w = row0 + 16 * i + 4 * r + q;
        if (w >= a.m) continue;
        const cplx v = cmake(a.scale * re[i][j][r], a.scale * im[i][j][r]);
        st(a.out, ((int64_t)z * a.m + w) * a.n + c, a.times_i ? cmake(-v.im, v.re) : v);
      }
  }
}

// The form that B's loads allow: the tallest row tile in 16s (4-byte loads' addresses
// and 64 rows do not fit the registers together), and what a chunk costs beside its products,
// in 16-row tiles: the B columns each row tile reads again, and with 4-byte loads four
// times the load instructions (N = 255, 71 walkers, VHS of 1275 vectors: 48 rows 263 us,
// 16 rows 308).  The plans (K ranges, units) and the launch take it from here.
// Up to `whole` rounds the fullest CU's last one counts whole (N = 301, 600 walkers, force
// bias of 1000 vectors with 4-byte loads: 10 K ranges in 4.06 rounds 920 us, 5 in 2.97 807).
struct NtForm {
  int tallest;
  double over, whole;
};
constexpr NtForm nt_form(bool wide) { return wide ? NtForm{4, 0.25, 4.0} : NtForm{3, 0.75, 6.0}; }

// Cost of a launch in units of one 16-row tile's MFMA time per K chunk (1024
// cycles): the workgroups of the fullest CU (a fraction of one once there are
// many rounds), each its chunks and about two chunks' worth of start and
// epilogue.
double nt_cost(int64_t m, int64_t colblocks, int rm, double chunks, const NtForm& form) {
  const double rounds = (double)(ceil_div(m, 16 * rm) * colblocks) / 256.0;
  return (rounds < form.whole ? std::ceil(rounds) : rounds) * (chunks + 2.0) * (rm + form.over);
}

// Rows per workgroup tile, in 16s: the least padding of m on a full
// GPU; smaller tiles where larger ones would leave CUs idle.
int nt_rows(int64_t m, int64_t colblocks, double chunks, const NtForm& form) {
  int best = 1;
  for (int rm = 2; rm <= form.tallest; ++rm)
    if (nt_cost(m, colblocks, rm, chunks, form) < 0.999 * nt_cost(m, colblocks, best, chunks, form)) best = rm;
  return best;
}

// what the dot products of a unit add to its start and end, in chunks
constexpr double NT_QDOT_CHUNKS = 3.0;

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int RM, int MODE, int EPI>
hipError_t launch_nt_mode(const NtArgs& a, hipStream_t stream) {
  using P = NtPlan<RM, MODE>;
  const int64_t blocks = (EPI == NT_EPI_QDOT ? a.nunits : ceil_div(a.n, NT_TN)) * ceil_div(a.m, P::TM);
  if (blocks > INT32_MAX || a.ksplit > 65535) return hipErrorInvalidValue;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(nt64_kernel<RM, MODE, EPI>), P::LDS_BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((nt64_kernel<RM, MODE, EPI>), dim3((unsigned)blocks, a.ksplit), dim3(NT_THREADS), P::LDS_BYTES,
                     stream, a);
  return hipGetLastError();
}

template <int RM, int EPI>
hipError_t launch_nt_rm(const NtArgs& a, bool direct, hipStream_t stream) {
  return direct ? launch_nt_mode<RM, NT_16, EPI>(a, stream) : launch_nt_mode<RM, NT_B4, EPI>(a, stream);
}

template <int EPI>
hipError_t launch_nt(const NtArgs& a, hipStream_t stream) {
  if (a.m < 1 || a.n < 1 || a.nseg < 1 || a.nseg > 2 || a.ksplit < 1) return hipErrorInvalidValue;
  bool a_vec = true, b_vec = true, far = false;
  int64_t chunks = 0;
  for (int s = 0; s < a.nseg; ++s) {
    const NtSegment& g = a.seg[s];
    if (g.K < 1 || g.lda < g.K || g.ldb < g.K) return hipErrorInvalidValue;
    far = far || g.lda > (1 << 22) || g.ldb > (1 << 22);  // 64 complex rows, 128 real columns in 32 bits
    a_vec = a_vec && aligned16(g.A);
    b_vec = b_vec && g.K % 2 == 0 && g.ldb % 2 == 0 && aligned16(g.B);
    chunks += ceil_div(g.K, NT_KC);
  }
  if (!a_vec || far) return launch_nt_mode<1, NT_AB4, EPI>(a, stream);
  const int64_t colblocks = EPI == NT_EPI_QDOT ? a.nunits : ceil_div(a.n, NT_TN) * a.ksplit;
  const double each = EPI == NT_EPI_QDOT ? a.unit_chunks + NT_QDOT_CHUNKS : (double)chunks / a.ksplit;
  switch (nt_rows(a.m, colblocks, each, nt_form(b_vec))) {
    case 1: return launch_nt_rm<1, EPI>(a, b_vec, stream);
    case 2: return launch_nt_rm<2, EPI>(a, b_vec, stream);
    case 3: return launch_nt_rm<3, EPI>(a, b_vec, stream);
    default: return launch_nt_mode<4, NT_16, EPI>(a, stream);
  }
}

}  // namespace

int nt64_ksplit(int64_t m, int64_t n, int64_t chunks, bool even, int most) {
  const NtForm form = nt_form(even);
  const int64_t nbn = ceil_div(n, NT_TN);
  // a further range writes and reads m n partial sums: 32 bytes each at 4.4 TB/s, in units of 0.43 us
  const double part = (double)m * n * 32.0 / 4.4e12 / 0.43e-6;
  int best = 1;
  double least = 0.0;
  for (int ks = 1; ks <= most && 2 * ks <= std::max<int64_t>(chunks, 2); ++ks) {
    const double each = (double)ceil_div(chunks, ks);
    const double t = nt_cost(m, nbn * ks, nt_rows(m, nbn * ks, each, form), each, form) + part * ks;
    if (ks == 1 || t < 0.98 * least) {
      best = ks;
      least = t;
    }
  }
  return best;
}

int nt64_quad_units(int64_t m, int64_t n, std::vector<int4>& units) {
  const NtForm form = nt_form(n % 2 == 0);
  const int64_t kchunks = ceil_div(n, NT_KC), tiles = ceil_div(n, NT_TN);
  auto extent = [&](int64_t t) { return std::min<int64_t>((t + 1) * (NT_TN / NT_KC), kchunks); };
  auto list = [&](int T, std::vector<int4>& u) {
    u.clear();
    for (int64_t z = 0; z * T < kchunks; ++z)
      for (int64_t t = 0; t < tiles; ++t)
        if (z * T < extent(t))
          u.push_back(make_int4((int)t, (int)(z * T), (int)std::min<int64_t>((z + 1) * T, extent(t)), 0));
  };
  // When the last workgroup ends, in chunks, with the units handed in their order to the
  // first free of 512 places (two a CU): a unit shorter than T fills a round's end.
  // (N = 200, 512 walkers: T = 24 in 3 rounds 685 us, 32 in 2.25 755; N = 300, 512
  // walkers: 48 2600, 32 2670; N = 101, 137 walkers: 12 41, 16 46.)  Many rounds end
  // together whatever T.
  auto cost = [&](int T, const std::vector<int4>& u) {
    const double each = T + NT_QDOT_CHUNKS;
    const int rm = nt_rows(m, (int64_t)u.size(), each, form);
    const int64_t rows = ceil_div(m, 16 * rm);
    if (rows * (int64_t)u.size() > 8192) return nt_cost(m, (int64_t)u.size(), rm, each, form);
    // places that become free at each time, in chunks
    const int start = (int)NT_QDOT_CHUNKS;
    int64_t work = 0;
    for (const int4& e : u) work += rows * (e.z - e.y + start);
    std::vector<int> free((size_t)(work / 512 + 2 * (T + start) + 2), 0);
    free[0] = 512;
    size_t t = 0, end = 0;
    for (const int4& e : u) {
      const int d = e.z - e.y + start;
      for (int64_t left = rows; left > 0;) {
        while (free[t] == 0) ++t;
        const int k = (int)std::min<int64_t>(free[t], left);
        free[t] -= k;
        free[t + d] += k;
        left -= k;
        end = std::max(end, t + d);
      }
    }
    return 2.0 * (double)end * (rm + form.over);
  };
  int best = 0;
  double least = 0.0;
  std::vector<int4> u;
  // (a tile's own columns are 8 chunks: other lengths leave short units)
  for (int T : {64, 56, 48, 40, 32, 24, 16, 12, 8, 4}) {
    list(T, u);
    const double t = cost(T, u);
    if (best == 0 || t < 0.98 * least) {
      best = T;
      least = t;
    }
  }
  list(best, units);
  return best;
}

hipError_t launch_nt64(const NtArgs& a, hipStream_t stream) {
  if (a.units) {
    if (a.nseg != 1 || a.ksplit != 1 || a.nunits < 1 || a.seg[0].K != a.n) return hipErrorInvalidValue;
    return launch_nt<NT_EPI_QDOT>(a, stream);
  }
  return launch_nt<NT_EPI_PART>(a, stream);
}

}  // namespace afqmc
