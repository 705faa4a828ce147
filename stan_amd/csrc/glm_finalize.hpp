// Device helpers shared by the GLM passes: wave reductions and the final
// assembly of log density and gradient from the reduced statistics
// st[0] = sum of row terms, st[1] = sum of residuals, st[2..K+1] = X^T r,
// st[K+2] = count of non-finite linear predictors.
#ifndef STANX_GLM_FINALIZE_HPP
#define STANX_GLM_FINALIZE_HPP

#include <hip/hip_runtime.h>

#include "sx_internal.hpp"
#include "wave_ops.hpp"

namespace sx {
namespace {

constexpr double kHalfLog2Pi = 0.91893853320467274178032973640562;

__device__ __forceinline__ double wave_sum(double v) { return wave::sum(v); }

// Stores one output value.  HOST: `p` is pinned host memory that the host
// watches while the kernel runs, so the store goes through to it at once
// (system scope) instead of waiting in this XCD's L2 for the launch's end.
template <bool HOST>
__device__ __forceinline__ void put_out(double* p, double v) {
  if (HOST)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  else
    *p = v;
}

// The gradient of coefficient k: the reduced X^T r entry, scaled, plus the
// prior (each coefficient on its own, so any thread may do it).
template <int FAM, bool HOST>
__device__ __forceinline__ void finalize_beta(const pass_args& a, const double* th, double* out,
                                              int k, double xtr) {
  double scale = 1.0;
  if (FAM == SX_NORMAL) {
    const double sigma = exp(th[a.K + 1]);
    scale = 1.0 / (sigma * sigma);
  }
  double g = xtr * scale;
  if (a.beta_sd > 0) g += -th[1 + k] / (a.beta_sd * a.beta_sd);
  put_out<HOST>(out + 2 + k, g);
}

// Log density, intercept and scale gradients and the status word from the
// reduced sum of row terms, sum of residuals and non-finite count; one wave.
template <int FAM, bool HOST>
__device__ __forceinline__ void finalize_head(const pass_args& a, const double* th, double* out,
                                              double sum_term, double sum_r, double bad) {
  const int lane = threadIdx.x & 63;
  const int K = a.K;
  const double alpha = th[0];
  double lp_prior = 0.0;  // lane-partial of prior terms over beta
  double scale = 1.0;
  if (FAM == SX_NORMAL) {
    const double sigma = exp(th[K + 1]);
    scale = 1.0 / (sigma * sigma);
  }
  if (a.beta_sd > 0)
    for (int k = lane; k < K; k += 64) {
      const double z = th[1 + k] / a.beta_sd;
      lp_prior += -0.5 * z * z;
      if (!a.propto) lp_prior += a.beta_const;
    }
  lp_prior = wave_sum(lp_prior);
  if (lane != 0) return;
  double lp = 0.0;
  double ga = sum_r * scale;
  if (FAM == SX_LOGIT) {
    lp = sum_term;
  } else {
    const double u = th[K + 1];
    const double sigma = exp(u);
    if (!(sigma > 0) || !isfinite(sigma)) bad += 1.0;
    const double SS = sum_term;
    lp = -0.5 * SS * scale - static_cast<double>(a.N) * u;
    if (!a.propto) lp += -static_cast<double>(a.N) * kHalfLog2Pi;
    double gu = -static_cast<double>(a.N) + SS * scale;
    if (a.sigma_sd > 0) {
      // sigma ~ normal(sigma_mu, sigma_sd): d/du = -(sigma - mu) sigma / sd^2
      const double z = (sigma - a.sigma_mu) / a.sigma_sd;
      lp += -0.5 * z * z;
      if (!a.propto) lp += a.sigma_const;
      gu += -z * (sigma / a.sigma_sd);
    }
    if (a.jacobian) {
      lp += u;
      gu += 1.0;
    }
    put_out<HOST>(out + K + 2, gu);
  }
  if (a.alpha_sd > 0) {
    const double z = alpha / a.alpha_sd;
    lp += -0.5 * z * z;
    if (!a.propto) lp += a.alpha_const;
    ga += -alpha / (a.alpha_sd * a.alpha_sd);
  }
  lp += lp_prior;
  put_out<HOST>(out, lp);
  put_out<HOST>(out + 1, ga);
  if (!isfinite(lp)) bad += 1.0;
  put_out<HOST>(out + a.D + 1, bad > 0 ? 1.0 : 0.0);
}

}  // namespace
}  // namespace sx
#endif
