// Per-walker elementwise / reduction kernels of the step:
//   fields      xbar, force-bias cap, xi, xshifted, cmf, cfb (+ Coulomb)
//               (ipie/propagation/phaseless_base.py:282-310, 360-368;
//                Coulomb: ipie/estimators/local_energy_sd.py:158-201)
//   weights     hybrid energy, phaseless importance weight
//               (phaseless_base.py:340-358, 370-380)
//   energy      e1b + Coulomb - exchange assembly
//               (ipie/estimators/local_energy_sd.py:358-403, 106-155)
//   normals     counter-based N(0, 1) fields (Philox4x32-10 + Box-Muller)
#include "afqmc_internal.hpp"

namespace afqmc {

namespace {

// Sums of v[0 .. S) and maxima of v[S .. S + M) over the workgroup's T threads, in thread 0:
// every value's steps side by side, one barrier.
template <int T, int S, int M>
__device__ __forceinline__ void reduce_all(double (&v)[S + M]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < S + M; ++i) {
      const double o = __shfl_xor(v[i], off, 64);
      v[i] = i < S ? v[i] + o : fmax(v[i], o);
    }
  if (T == 64) return;
  __shared__ double waves[T / 64][S + M];
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < S + M; ++i) waves[threadIdx.x >> 6][i] = v[i];
  __syncthreads();
  if (threadIdx.x == 0)
    for (int t = 1; t < T / 64; ++t)
#pragma unroll
      for (int i = 0; i < S + M; ++i) v[i] = i < S ? v[i] + waves[t][i] : fmax(v[i], waves[t][i]);
}

// Threads of a walker's workgroup for `items` items: a wave for at most 64, else 256, or
// more for at most `few` walkers, which leave CUs idle.
int walker_threads(int nwalkers, int64_t items, int few, int more) {
  return items <= 64 ? 64 : items > 256 && nwalkers <= few ? more : 256;
}

// Two standard normals (Philox key = seed, counter = (pair index, stream)) for pair index p of stream `counter`.
__device__ __forceinline__ double2 normal_pair(uint64_t seed, uint64_t counter, uint64_t p) {
  const uint4 c = make_uint4((uint32_t)p, (uint32_t)(p >> 32), (uint32_t)counter, (uint32_t)(counter >> 32));
  const uint4 r = philox4x32(c, make_uint2((uint32_t)seed, (uint32_t)(seed >> 32)));
  // 53-bit uniforms in (0, 1]
  const uint64_t a = ((uint64_t)r.x << 21) ^ ((uint64_t)r.y >> 11);
  const uint64_t b = ((uint64_t)r.z << 21) ^ ((uint64_t)r.w >> 11);
  const double u1 = ((double)(a & ((1ull << 53) - 1)) + 1.0) * (1.0 / 9007199254740992.0);
  const double u2 = (double)(b & ((1ull << 53) - 1)) * (1.0 / 9007199254740992.0);
  const double rad = sqrt(-2.0 * log(u1));
  double s, co;
  sincospi(2.0 * u2, &s, &co);
  return make_double2(rad * co, rad * s);
}

// A thread takes the pairs of entries that share a Philox draw (entries 2 p, 2 p + 1 of the
// [W, X] array; a pair may end in the next walker).  Latency-bound: the partial sums of
// 4 ranges are loaded together, the walker's sums reduced together.  (W, X, ranges)
// = (10, 72, 5): 7.8 -> 5.0 us; (12, 2400, 16): 46 -> 16; (300, 750, 16 in FP32): 23 -> 18;
// (1024, 2400, 16 in FP32): 117 -> 89, against one entry a thread, each range's load waited for,
// and six reductions of two barriers.
template <int T>
__global__ void __launch_bounds__(T) fields_kernel(FieldsArgs a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  const int w = blockIdx.x;
  const int X = a.nchol;
  const int64_t plane = (int64_t)a.nwalkers * X, first = (int64_t)w * X, end = first + X;
  // ecoul re, im, cmf re, im, cfb re, im, sum |xbar|; max |xbar|
  double sums[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  unsigned long long ncap = 0;
  const uint64_t counter = a.state ? a.state->counter : a.counter;
  for (int64_t p = (first >> 1) + threadIdx.x; 2 * p < end; p += T) {
    const int64_t i0 = max(2 * p, first), i1 = min(2 * p + 1, end - 1);  // (i0 == i1: one of them is the neighbour's)
    cplx vb[2] = {cmake(0.0, 0.0), cmake(0.0, 0.0)};
    for (int z0 = 0; z0 < a.ksplit; z0 += 4) {
      cplx v[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t at = min(z0 + u, a.ksplit - 1) * plane;
        if (a.part32) {  // split-BF16 partials, FP32 (their accumulation precision), summed in FP64
          const float2* p32 = reinterpret_cast<const float2*>(a.vbias_part) + at;
          const float2 f0 = p32[i0], f1 = p32[i1];
          v[u][0] = cmake((double)f0.x, (double)f0.y);
          v[u][1] = cmake((double)f1.x, (double)f1.y);
        } else {
          v[u][0] = ld(a.vbias_part, at + i0);
          v[u][1] = ld(a.vbias_part, at + i1);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (z0 + u < a.ksplit) {
          vb[0] = cadd(vb[0], v[u][0]);
          vb[1] = cadd(vb[1], v[u][1]);
        }
    }
    double2 normal = make_double2(0.0, 0.0);
    if (a.want_fields && !a.xi) normal = normal_pair(a.seed, counter, (uint64_t)p);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t idx = 2 * p + h;
      if (idx < first || idx >= end) continue;
      const cplx v = vb[h];
      if (a.vbias_out) st(a.vbias_out, idx, v);
      sums[0] += v.re * v.re - v.im * v.im;
      sums[1] += 2.0 * v.re * v.im;
      const cplx mf = ld(a.mf_shift, idx - first);
      // xbar = -sqrt(dt) (i vbias - mf_shift)
      cplx xb = cmake(a.sqrt_dt * (mf.re + v.im), a.sqrt_dt * (mf.im - v.re));
      const double axb = cabs(xb);
      if (axb > a.fbbound) {
        ++ncap;
        if (axb > 1e-13) xb = cmake(xb.re / axb, xb.im / axb);
      }
      const double axc = axb > a.fbbound ? 1.0 : axb;
      sums[6] += axc;
      sums[7] = fmax(sums[7], axc);
      if (!a.want_fields) continue;
      const double xi = a.xi ? a.xi[idx] : h ? normal.y : normal.x;
      if (a.xi_out) a.xi_out[idx] = xi;
      const cplx xs = cmake(xi - xb.re, -xb.im);
      st(a.xshifted, idx, xs);
      sums[2] += xs.re * mf.re - xs.im * mf.im;
      sums[3] += xs.re * mf.im + xs.im * mf.re;
      sums[4] += xi * xb.re - 0.5 * (xb.re * xb.re - xb.im * xb.im);
      sums[5] += xi * xb.im - xb.re * xb.im;
    }
  }
  if (a.want_fields && ncap && a.nfb) atomicAdd(a.nfb, ncap);
  reduce_all<T, 7, 1>(sums);
  if (threadIdx.x == 0) {
    if (a.xbar_mean) {
      a.xbar_mean[w] = sums[6] / X;
      a.xbar_max[w] = sums[7];
    }
    if (a.ecoul) st(a.ecoul, w, cmake(0.5 * sums[0], 0.5 * sums[1]));
    if (a.want_fields) {
      st(a.cmf, w, cmake(-a.sqrt_dt * sums[2], -a.sqrt_dt * sums[3]));
      st(a.cfb, w, cmake(sums[4], sums[5]));
    }
  }
}

__global__ void update_weight_kernel(WeightArgs a) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  phase_mark(a.mark, w == 0);
  if (w >= a.nwalkers) return;
  const cplx o_old = ld(a.ovlp_old, w), o_new = ld(a.ovlp_new, w);
  const cplx ratio = cdiv(o_new, o_old);
  const cplx lr = clog(ratio);
  const cplx cfb = ld(a.cfb, w), cmf = ld(a.cmf, w);
  const double eshift = a.state ? a.state->eshift : a.eshift;
  cplx eh = cmake(-(lr.re + cfb.re + cmf.re) / a.dt, -(lr.im + cfb.im + cmf.im) / a.dt);
  if (fabs(eshift) >= 1e-10) {
    const double emax = eshift + a.ebound, emin = eshift - a.ebound;
    eh.re = fmin(fmax(eh.re, emin), emax);
  }
  const cplx prev = ld(a.hybrid_energy, w);
  const cplx arg = cmake(-a.dt * (0.5 * (eh.re + prev.re) - eshift), -a.dt * 0.5 * (eh.im + prev.im));
  const double magn = exp(arg.re);  // |exp(arg)|
  const double dtheta = -a.dt * eh.im - cfb.im;
  double cosf = cos(dtheta);
  if (cosf < 0.0) cosf = 0.0;
  const double wnew = a.weight[w] * magn * cosf;
  a.weight[w] = wnew;
  st(a.hybrid_energy, w, eh);
  st(a.walker_ovlp, w, o_new);
  if (!isfinite(wnew) && a.flags) atomicOr(a.flags, AFQMC_FLAG_NONFINITE);
  if (!isfinite(wnew) && a.wflags) atomicOr(a.wflags + w, AFQMC_FLAG_NONFINITE);
  // the step's last phase is this kernel alone: walker 0's thread closes it
  phase_mark(PhaseMark{a.mark.acc, a.mark.phase, -1}, w == 0);
}

// (Four entries of both operands in flight a thread, four partial sums.)
template <int T>
__global__ void __launch_bounds__(T) energy_kernel(EnergyArgs a) {
  phase_mark(a.mark, blockIdx.x == 0 && threadIdx.x == 0);
  const int w = blockIdx.x;
  const int N = a.nbasis;
  double sums[2] = {0.0, 0.0};
  const int nspin = a.e1_in ? 0 : (a.rhf || a.nbeta == 0) ? 1 : 2;
  for (int s = 0; s < nspin; ++s) {
    const int n = s == 0 ? a.nalpha : a.nbeta, end = n * N;
    const double* g = (s == 0 ? a.ghalfa : a.ghalfb) + 2 * (int64_t)w * n * N;
    const double* h = s == 0 ? a.rH1a : a.rH1b;
    double er[4] = {0.0, 0.0, 0.0, 0.0}, ei[4] = {0.0, 0.0, 0.0, 0.0};
    for (int e0 = threadIdx.x; e0 < end; e0 += 4 * T) {
      cplx gv[4], hv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = min(e0 + u * T, end - 1);
        gv[u] = ld(g, e);
        hv[u] = ld(h, e);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + u * T < end) {
          er[u] += gv[u].re * hv[u].re - gv[u].im * hv[u].im;
          ei[u] += gv[u].re * hv[u].im + gv[u].im * hv[u].re;
        }
    }
    sums[0] += (er[0] + er[1]) + (er[2] + er[3]);
    sums[1] += (ei[0] + ei[1]) + (ei[2] + ei[3]);
  }
  reduce_all<T, 2, 0>(sums);
  const double er = sums[0], ei = sums[1];
  if (threadIdx.x == 0) {
    const double f = a.rhf ? 2.0 : 1.0;
    const cplx e1 = a.e1_in ? ld(a.e1_in, w) : cmake(f * er + a.ecore, f * ei);
    if (a.e1_out) st(a.e1_out, w, e1);
    cplx ex = cmake(0.0, 0.0);
    if (a.exx_est) {
      ex = ld(a.exx_est, w);
    } else {
      for (int z = 0; z < a.xs_a; ++z) ex = cadd(ex, ld(a.exx_part_a, (int64_t)z * a.nwalkers + w));
      if (a.exx_part_b)
        for (int z = 0; z < a.xs_b; ++z) ex = cadd(ex, ld(a.exx_part_b, (int64_t)z * a.nwalkers + w));
    }
    // UHF: exx = 1/2 (sum_a + sum_b); RHF: exx = 2 * 1/2 * sum_a
    const double fx = a.rhf ? 1.0 : 0.5;
    ex = cscale(ex, fx);
    const cplx e2 = csub(ld(a.ecoul, w), ex);
    st(a.energy, 3 * (int64_t)w + 0, cadd(e1, e2));
    st(a.energy, 3 * (int64_t)w + 1, e1);
    st(a.energy, 3 * (int64_t)w + 2, e2);
  }
}

__global__ void step_set_kernel(StepState* s, unsigned long long counter, double eshift) {
  if (threadIdx.x == 0) {
    s->counter = counter;
    s->eshift = eshift;
  }
}

__global__ void phase_mark_kernel(PhaseMark m) { phase_mark(m, threadIdx.x == 0); }

__global__ void phase_clear_kernel(unsigned long long* acc, int n) {
  if ((int)threadIdx.x < n) acc[threadIdx.x] = 0;
}

__global__ void step_advance_kernel(StepState* s, long long dcounter, long long dadam) {
  if (threadIdx.x == 0) {
    s->counter += (unsigned long long)dcounter;
    s->adam_t += dadam;
  }
}

__global__ void normals_kernel(double* out, int64_t n, uint64_t seed, uint64_t counter) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (2 * p >= n) return;
  const double2 v = normal_pair(seed, counter, (uint64_t)p);
  out[2 * p] = v.x;
  if (2 * p + 1 < n) out[2 * p + 1] = v.y;
}

}  // namespace

hipError_t launch_fields(const FieldsArgs& a, hipStream_t stream) {
  switch (walker_threads(a.nwalkers, a.nchol / 2 + 1, 256, 512)) {  // (129 registers: one workgroup of 512 a CU)
    case 64: hipLaunchKernelGGL(fields_kernel<64>, dim3(a.nwalkers), dim3(64), 0, stream, a); break;
    case 256: hipLaunchKernelGGL(fields_kernel<256>, dim3(a.nwalkers), dim3(256), 0, stream, a); break;
    default: hipLaunchKernelGGL(fields_kernel<512>, dim3(a.nwalkers), dim3(512), 0, stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_update_weight(const WeightArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL(update_weight_kernel, dim3((unsigned)ceil_div(a.nwalkers, 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_energy(const EnergyArgs& a, hipStream_t stream) {
  const int nmax = a.nalpha > a.nbeta ? a.nalpha : a.nbeta;
  switch (walker_threads(a.nwalkers, a.e1_in ? 1 : ceil_div((int64_t)nmax * a.nbasis, 4), 512, 1024)) {
    case 64: hipLaunchKernelGGL(energy_kernel<64>, dim3(a.nwalkers), dim3(64), 0, stream, a); break;
    case 256: hipLaunchKernelGGL(energy_kernel<256>, dim3(a.nwalkers), dim3(256), 0, stream, a); break;
    default: hipLaunchKernelGGL(energy_kernel<1024>, dim3(a.nwalkers), dim3(1024), 0, stream, a);
  }
  return hipGetLastError();
}

hipError_t launch_step_set(StepState* state, unsigned long long counter, double eshift, hipStream_t stream) {
  hipLaunchKernelGGL(step_set_kernel, dim3(1), dim3(64), 0, stream, state, counter, eshift);
  return hipGetLastError();
}

hipError_t launch_phase_mark(const PhaseMark& m, hipStream_t stream) {
  hipLaunchKernelGGL(phase_mark_kernel, dim3(1), dim3(64), 0, stream, m);
  return hipGetLastError();
}

hipError_t launch_phase_clear(unsigned long long* acc, int n, hipStream_t stream) {
  hipLaunchKernelGGL(phase_clear_kernel, dim3(1), dim3(64), 0, stream, acc, n);
  return hipGetLastError();
}

hipError_t launch_step_advance(StepState* state, long long dcounter, long long dadam, hipStream_t stream) {
  hipLaunchKernelGGL(step_advance_kernel, dim3(1), dim3(64), 0, stream, state, dcounter, dadam);
  return hipGetLastError();
}

// dst[i] = src[i] for i < n, then src[i] = 0 when clear (a kernel, not a
// memset, so that a captured graph replays it correctly).
__global__ void take_flags_kernel(int* src, int* dst, int n, int clear) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int v = src[i];
  if (dst) dst[i] = v;
  if (clear) src[i] = 0;
}

hipError_t launch_take_flags(int* src, int* dst, int n, int clear, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(take_flags_kernel, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream, src, dst, n, clear);
  return hipGetLastError();
}

hipError_t launch_draw_normals(double* out, int64_t n, uint64_t seed, uint64_t counter, hipStream_t stream) {
  const int64_t pairs = (n + 1) / 2;
  hipLaunchKernelGGL(normals_kernel, dim3((unsigned)ceil_div(pairs, 256)), dim3(256), 0, stream, out, n, seed,
                     counter);
  return hipGetLastError();
}

}  // namespace afqmc
