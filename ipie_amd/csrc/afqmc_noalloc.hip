// Green's function / overlap entry point that allocates nothing.
//
// afqmc_greens_function_noalloc is afqmc_greens_function without a context: the
// trial orbitals come in as arguments, and the kernel keeps the overlap matrices and
// their inverses in LDS.  The limit on a call, AFQMC_NOALLOC_SCRATCH_BYTES over
// the O matrices, their inverses and the per-walker partials of W walkers, is
// that of the static device array such a call once worked in.
#include <cstdio>

#include "afqmc_internal.hpp"
#include "../../include/afqmc_hip.h"

namespace {

constexpr size_t kScratchBytes = AFQMC_NOALLOC_SCRATCH_BYTES;
thread_local char g_err[256] = "";

int nerr(int code, const char* msg) {
  snprintf(g_err, sizeof(g_err), "%s", msg);
  return code;
}

// O matrices (or their inverses) [W, 2, nmax, nmax] complex and per-spin results [W, 2, 4]
size_t work_bytes(int nwalkers, int nalpha, int nbeta) {
  const int nmax = nalpha > nbeta ? nalpha : nbeta;
  return sizeof(afqmc::cplx) * (size_t)nwalkers * 2 * nmax * nmax + sizeof(double) * 8 * (size_t)nwalkers;
}

}  // namespace

extern "C" {

size_t afqmc_noalloc_scratch_bytes(int32_t nwalkers, int32_t nalpha, int32_t nbeta) {
  if (nwalkers < 1 || nalpha < 1 || nbeta < 0) return 0;
  return 2 * work_bytes(nwalkers, nalpha, nbeta);
}

const char* afqmc_noalloc_last_error(void) { return g_err; }

int afqmc_greens_function_noalloc(int32_t nwalkers, int32_t nbasis, int32_t nalpha, int32_t nbeta, int32_t rhf,
                                  const double* psia, const double* psib, const double* phia, const double* phib,
                                  double* ghalfa, double* ghalfb, double* ovlp, const double* log_shift,
                                  int32_t* walker_flags, void* stream) {
  g_err[0] = '\0';
  if (nwalkers < 1 || nbasis < 1 || nalpha < 1 || nbeta < 0)
    return nerr(AFQMC_ERR_SHAPE, "nwalkers, nbasis, nalpha must be positive and nbeta non-negative");
  if (nalpha > 64 || nbeta > 64 || nalpha > nbasis || nbeta > nbasis)
    return nerr(AFQMC_ERR_SHAPE, "nalpha and nbeta must be at most 64 and at most nbasis");
  const bool two = nbeta > 0 && !rhf;
  if (!psia || !phia || !ovlp || (two && (!psib || !phib)))
    return nerr(AFQMC_ERR_INVALID_ARG, "null trial, walker or overlap array");
  const bool want_ghalf = ghalfa != nullptr;
  if (want_ghalf && two && ghalfb == nullptr)
    return nerr(AFQMC_ERR_INVALID_ARG, "Ghalf of both spins, or of neither (overlap only)");
  const size_t half = work_bytes(nwalkers, nalpha, nbeta);
  if (half > kScratchBytes / 2) {
    snprintf(g_err, sizeof(g_err),
             "scratch of %zu bytes needed for %d walkers (nalpha %d, nbeta %d) exceeds the static %zu bytes",
             2 * half, nwalkers, nalpha, nbeta, kScratchBytes);
    return AFQMC_ERR_SHAPE;
  }
  afqmc::GfArgs a{};
  a.nwalkers = nwalkers;
  a.nbasis = nbasis;
  a.nalpha = nalpha;
  a.nbeta = nbeta;
  a.rhf = rhf ? 1 : 0;
  a.phia = phia;
  a.phib = two ? phib : nullptr;
  a.psia = psia;
  a.psib = two ? psib : nullptr;
  a.ghalfa = ghalfa;
  a.ghalfb = two ? ghalfb : nullptr;
  a.ovlp = ovlp;
  a.log_shift = log_shift;
  a.flags = nullptr;
  a.wflags = walker_flags;
  a.psi_real = 0;
  const hipError_t e = afqmc::launch_gf(a, want_ghalf, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "Green's function launch failed: %s", hipGetErrorString(e));
    return e == hipErrorInvalidValue ? AFQMC_ERR_SHAPE : AFQMC_ERR_HIP;
  }
  return AFQMC_OK;
}

}  // extern "C"
