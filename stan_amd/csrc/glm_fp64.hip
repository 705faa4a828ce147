// Fused FP64 forward + adjoint pass of the GLM log density on gfx950.
//
// One launch evaluates, for theta = (alpha, beta[, u]):
//   logistic  (bernoulli_logit_glm):  eta = X beta + alpha,
//             lp_lik = sum_n -log1p(exp(-s_n eta_n)),  s_n = 2 y_n - 1,
//             r_n = s_n / (1 + exp(s_n eta_n)) = y_n - inv_logit(eta_n)
//   normal    (normal_id_glm):        d_n = y_n - (X beta + alpha)_n,
//             SS = sum d_n^2, r_n = d_n
// and the adjoint X^T r, sum r, reading every element of X exactly once:
// each wave loads a 64-row-block tile of X into registers (one 512-byte
// coalesced load per slot), forms eta with an L-lane reduction,
// evaluates the link, and accumulates x * r into per-lane FP64 registers.
// Block partials are summed in a fixed order by a second launch of a few
// blocks per chain, so results are bitwise reproducible, and that launch adds
// the priors and the log-Jacobian and writes lp and the gradient.  This
// replaces the two GEMV passes over X that the reference's CPU GLM performs
// per gradient (Stan Math bernoulli_logit_glm_lpmf / normal_id_glm_lpdf,
// reached through src/stan/model/gradient.hpp:21-35).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../include/stanx/sx_math.hpp"
#include "glm_finalize.hpp"
#include "glm_fp64_tile.hpp"
#include "sx_internal.hpp"

namespace sx {

namespace {

// Blocks of the cross-block reduction per chain: four waves each, wave 0
// for the log density, the others two columns.
__host__ __device__ constexpr int reduce_blocks(int K) { return (1 + (K + 1) / 2 + 3) / 4; }

template <int SMAX>
__device__ __forceinline__ void load_tile(const pass_args& a, int64_t t, int lane,
                                          double (&x)[SMAX]) {
  const __amdgpu_buffer_rsrc_t rs =
      make_rsrc(a.X + t * static_cast<int64_t>(a.S) * 64, static_cast<uint32_t>(a.S) * 512u);
#pragma unroll
  for (int j = 0; j < SMAX; ++j) x[j] = buf_f64(rs, lane * 8u, j * 512u);
}

// A single evaluation's theta travels in the kernel arguments (ARG; D <=
// kThetaArg): the launch itself carries it, where a host-to-device copy
// would be one more command in the stream with a gap after it.
struct theta_arg {
  double v[kThetaArg];
};
static_assert(sizeof(pass_args) + sizeof(theta_arg) + 16 <= 4096, "4 KB of kernel arguments");
struct no_theta {};
template <bool ARG>
using theta_of = std::conditional_t<ARG, theta_arg, no_theta>;

template <bool ARG>
__device__ __forceinline__ const double* theta_ptr(const pass_args& a, const theta_of<ARG>& t) {
  if constexpr (ARG)
    return t.v;
  else
    return a.theta;
}

template <int SMAX, int FAM, int PF, bool ARG>
__global__ __launch_bounds__(256) void glm_pass_f64(pass_args a, theta_of<ARG> ta) {
  extern __shared__ double lds[];
  // 1-D grid of chains x nb blocks.  With nb a multiple of 8 the blocks of
  // every chain that stream the same tiles sit on one XCD (block ids 8
  // apart), so a batched evaluation reads each tile of X from HBM about
  // once per XCD and the other chains find it in that XCD's L2; for one
  // chain the mapping is the identity.
  const int nb = static_cast<int>(gridDim.x) / a.chains;
  int blk, chain;
  {
    const int L = blockIdx.x;
    if ((nb & 7) == 0) {
      const int q = L >> 3;
      blk = (L & 7) + 8 * (q / a.chains);
      chain = q % a.chains;
    } else {
      blk = L % nb;
      chain = L / nb;
    }
    blk = __builtin_amdgcn_readfirstlane(blk);
    chain = __builtin_amdgcn_readfirstlane(chain);
  }
  const double* theta = theta_ptr<ARG>(a, ta);
  if constexpr (!ARG) theta += static_cast<int64_t>(chain) * a.theta_stride;
  a.partials += static_cast<int64_t>(chain) * a.E * nb;
  const int lane = threadIdx.x & 63;
  // the wave index is uniform across the wave: say so, so that tile
  // indices and buffer descriptors live in scalar registers
  const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int L = a.L;
  const int R = 64 >> a.lgL;
  const int q = lane >> (6 - a.lgL);
  const int r = lane & (R - 1);
  const int S = a.S;

  // the first tile's loads are issued before theta is staged: the two
  // latencies overlap
  const int64_t W = static_cast<int64_t>(nb) * nw;
  const int64_t first = static_cast<int64_t>(blk) * nw + wib;
  int64_t t = first;
  double xv[SMAX];
  double yv = 0.0;
  if (t < a.T) {
    yv = load_y<FAM>(a, t, R, r);
    load_tile<SMAX>(a, t, lane, xv);
  }
  // beta staged in LDS, padded to SMAX*L entries (zero beyond K)
  double* sbeta = lds + nw * a.E;
  for (int i = threadIdx.x; i < SMAX * L; i += blockDim.x)
    sbeta[i] = i < a.K ? theta[1 + i] : 0.0;
  __syncthreads();
  const double alpha = theta[0];
  double acc[SMAX];
#pragma unroll
  for (int j = 0; j < SMAX; ++j) acc[j] = 0.0;
  double s0 = 0.0, s1 = 0.0, bad = 0.0;

  for (; t < a.T; t += W) {
    double xn[SMAX];
    double yn = 0.0;
    if (PF) {
      // the next tile's loads are in flight during this tile's arithmetic
      const int64_t tn = t + W;
      if (tn < a.T) {
        yn = load_y<FAM>(a, tn, R, r);
        load_tile<SMAX>(a, tn, lane, xn);
      } else {
#pragma unroll
        for (int j = 0; j < SMAX; ++j) xn[j] = 0.0;
      }
    } else if (t != first) {
      yv = load_y<FAM>(a, t, R, r);
      load_tile<SMAX>(a, t, lane, xv);
    }
    // beta is re-read from LDS every tile: an opaque zero offset keeps the
    // compiler from hoisting SMAX loop-invariant values into registers
    int zoff = 0;
    asm volatile("" : "+s"(zoff));
    const double* sb = sbeta + zoff + q;
    double e = 0.0;
#pragma unroll
    for (int j = 0; j < SMAX; ++j) e = fma(xv[j], sb[j * L], e);
    e = wave::xor_sum(e, R, 64);
    const int64_t row = t * R + r;
    const bool valid = row < a.N;
    e += alpha;
    double rr = 0.0, term = 0.0;
    if (valid) {
      if (FAM == SX_LOGIT) {
        // with four slots the link is most of the work, and registers are free
        stanx::math::sx_logit_row<(SMAX > 4)>(e, yv != 0.0 ? 1.0 : -1.0, &term, &rr);
      } else {
        const double d = yv - e;
        rr = d;
        term = d * d;
      }
      if (!isfinite(e)) bad += 1.0;
    }
    if (q == 0) {
      s0 += term;
      s1 += rr;
    }
#pragma unroll
    for (int j = 0; j < SMAX; ++j) acc[j] = fma(xv[j], rr, acc[j]);
    if (PF) {
#pragma unroll
      for (int j = 0; j < SMAX; ++j) xv[j] = xn[j];
      yv = yn;
    }
  }

  // reduce the per-lane column partials over the R row-lanes of each column
  wave::xor_sum_n<SMAX>(acc, 1, R);
  s0 = wave_sum(s0);
  s1 = wave_sum(s1);
  bad = wave_sum(bad);
  const int E = a.E;
  if (r == 0) {
#pragma unroll
    for (int j = 0; j < SMAX; ++j) {
      const int c = j * L + q;
      if (j < S && c < a.K) lds[wib * E + 2 + c] = acc[j];
    }
  }
  if (lane == 0) {
    lds[wib * E + 0] = s0;
    lds[wib * E + 1] = s1;
    lds[wib * E + a.K + 2] = bad;
  }
  __syncthreads();
  // block partial, stored entry-major: partials[i * nb + block]
  for (int i = threadIdx.x; i < E; i += blockDim.x) {
    double v = 0.0;
    for (int w = 0; w < nw; ++w) v += lds[w * E + i];
    a.partials[static_cast<int64_t>(i) * nb + blk] = v;
  }
}

// Sum over the nb block partials of U entries (rows of nb doubles), in
// every lane: lane l adds blocks l, l + 64, ... in order, then a fixed
// shuffle tree.  Eight loads per entry are in flight before the first add;
// clamped indices and selects keep the loop free of branches.
template <int U>
__device__ __forceinline__ void sum_entries(const double* partials, const int (&e)[U], int nb,
                                            int lane, double (&w)[U]) {
#pragma unroll
  for (int u = 0; u < U; ++u) w[u] = 0.0;
  for (int b0 = 0; b0 < nb; b0 += 512) {
    double x[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < 8; ++k)
        x[u][k] = partials[static_cast<int64_t>(e[u]) * nb + min(b0 + lane + 64 * k, nb - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < 8; ++k) w[u] += (b0 + lane + 64 * k < nb) ? x[u][k] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) w[u] = wave_sum(w[u]);
}

// Cross-block reduction of the bulk pass's partials (fixed order, so the
// result is bitwise reproducible for a given launch shape) followed by the
// priors, Jacobian and output.  A separate launch: the kernel boundary
// makes every block's partials visible without per-block cache
// write-backs.  It is bound by latency (211 KB at N = 1e6, K = 100), so the
// entries are spread over ceil((1 + K / 2) / 4) blocks per chain instead of
// one (no entry needs another's sum).  Wave 0 takes the log density (row
// terms, residual sum, non-finite count), every other wave two columns.
// With theta in the launches and results stored to the host, an evaluation
// from a host theta takes 22 us at N = 3000, K = 37 (35 with one block and a
// copy at either end) and 131 us at N = 1e6, K = 100 (146), of which the
// pass 125.
template <int FAM, bool ARG, bool HOST>
__global__ __launch_bounds__(256) void glm_reduce_f64(pass_args a, int nb, theta_of<ARG> ta) {
  const int per = reduce_blocks(a.K);
  const int chain = static_cast<int>(blockIdx.x) / per;
  const double* theta = theta_ptr<ARG>(a, ta);
  if constexpr (!ARG) theta += static_cast<int64_t>(chain) * a.theta_stride;
  const double* partials = a.partials + static_cast<int64_t>(chain) * a.E * nb;
  double* out = a.out + static_cast<int64_t>(chain) * a.out_stride;
  const int lane = threadIdx.x & 63;
  const int w = (static_cast<int>(blockIdx.x) - chain * per) * 4 +
                __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (w == 0) {
    const int e[3] = {0, 1, a.K + 2};
    double v[3];
    sum_entries<3>(partials, e, nb, lane, v);
    finalize_head<FAM, HOST>(a, theta, out, v[0], v[1], v[2]);
    return;
  }
  const int k = 2 * (w - 1);
  if (k >= a.K) return;
  const int e[2] = {2 + k, min(3 + k, a.K + 1)};
  double v[2];
  sum_entries<2>(partials, e, nb, lane, v);
  if (lane < 2 && k + lane < a.K)
    finalize_beta<FAM, HOST>(a, theta, out, k + lane, lane == 0 ? v[0] : v[1]);
}

__global__ void tile_x_f64(const double* __restrict__ Xrm, double* __restrict__ Xt,
                           int64_t N, int64_t K, int L, int lgL, int S, int64_t total) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int lane = static_cast<int>(idx & 63);
  const int64_t js = idx >> 6;  // t * S + j
  const int64_t t = js / S;
  const int j = static_cast<int>(js - t * S);
  const int lgR = 6 - lgL;
  const int64_t row = (t << lgR) + (lane & ((1 << lgR) - 1));
  const int64_t col = static_cast<int64_t>(j) * L + (lane >> lgR);
  Xt[idx] = (row < N && col < K) ? Xrm[row * K + col] : 0.0;
}

template <int SMAX, int FAM, int PF, bool ARG>
void launch_one(const pass_args& a, const theta_of<ARG>& ta, int blocks, int threads,
                hipStream_t s) {
  const size_t lds =
      (static_cast<size_t>(threads / 64) * a.E + static_cast<size_t>(SMAX) * a.L) * sizeof(double);
  hipLaunchKernelGGL((glm_pass_f64<SMAX, FAM, PF, ARG>), dim3(blocks * a.chains), dim3(threads),
                     lds, s, a, ta);
}

template <int FAM, int PF, bool ARG>
hipError_t launch_fam(int smax, const pass_args& a, const theta_of<ARG>& ta, int blocks,
                      int threads, hipStream_t s) {
  switch (smax) {
    case 4: launch_one<4, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 8: launch_one<8, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 12: launch_one<12, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 16: launch_one<16, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 20: launch_one<20, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 24: launch_one<24, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 28: launch_one<28, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    case 32: launch_one<32, FAM, PF, ARG>(a, ta, blocks, threads, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int FAM, bool ARG>
hipError_t launch_pass(const tile_geom& g, const pass_args& a, const theta_of<ARG>& ta,
                       int blocks, int threads, hipStream_t s) {
  if constexpr (!ARG)
    if (chains_pass_fits(FAM, g, a, threads)) return launch_pass_f64_chains(FAM, g, a, blocks, s);
  return g.prefetch ? launch_fam<FAM, 1, ARG>(g.smax, a, ta, blocks, threads, s)
                    : launch_fam<FAM, 0, ARG>(g.smax, a, ta, blocks, threads, s);
}

template <int FAM, bool ARG, bool HOST>
hipError_t launch_reduce(const pass_args& a, const theta_of<ARG>& ta, int blocks, hipStream_t s) {
  hipLaunchKernelGGL((glm_reduce_f64<FAM, ARG, HOST>), dim3(a.chains * reduce_blocks(a.K)),
                     dim3(256), 0, s, a, blocks, ta);
  return hipGetLastError();
}

template <int FAM>
hipError_t launch_eval(const tile_geom& g, const pass_args& a, const double* h_theta, int blocks,
                       int threads, hipStream_t s) {
  hipError_t e;
  if (a.D <= kThetaArg) {
    theta_arg ta;
    for (int i = 0; i < kThetaArg; ++i) ta.v[i] = i < a.D ? h_theta[i] : 0.0;
    e = launch_pass<FAM, true>(g, a, ta, blocks, threads, s);
    if (e == hipSuccess) e = launch_reduce<FAM, true, true>(a, ta, blocks, s);
    return e;
  }
  e = hipMemcpyAsync(const_cast<double*>(a.theta), h_theta, sizeof(double) * a.D,
                     hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = launch_pass<FAM, false>(g, a, no_theta{}, blocks, threads, s);
  if (e == hipSuccess) e = launch_reduce<FAM, false, true>(a, no_theta{}, blocks, s);
  return e;
}

}  // namespace

tile_geom make_geom(int64_t N, int64_t K, int L, int smax) {
  tile_geom g;
  g.L = L;
  g.lgL = 0;
  while ((1 << g.lgL) < L) ++g.lgL;
  g.R = 64 / L;
  g.S = static_cast<int>((K + L - 1) / L);
  g.smax = smax;
  g.T = (N + g.R - 1) / g.R;
  return g;
}

hipError_t launch_pass_f64(int family, const tile_geom& g, const pass_args& a,
                           int blocks, int threads, hipStream_t s, bool reduce) {
  hipError_t e = hipErrorInvalidValue;
  if (family == SX_LOGIT)
    e = launch_pass<SX_LOGIT, false>(g, a, no_theta{}, blocks, threads, s);
  else if (family == SX_NORMAL)
    e = launch_pass<SX_NORMAL, false>(g, a, no_theta{}, blocks, threads, s);
  if (e != hipSuccess || !reduce) return e;
  return family == SX_LOGIT ? launch_reduce<SX_LOGIT, false, false>(a, no_theta{}, blocks, s)
                            : launch_reduce<SX_NORMAL, false, false>(a, no_theta{}, blocks, s);
}

hipError_t launch_eval_f64(int family, const tile_geom& g, const pass_args& a,
                           const double* h_theta, int blocks, int threads, hipStream_t s) {
  if (family == SX_LOGIT) return launch_eval<SX_LOGIT>(g, a, h_theta, blocks, threads, s);
  if (family == SX_NORMAL) return launch_eval<SX_NORMAL>(g, a, h_theta, blocks, threads, s);
  return hipErrorInvalidValue;
}

hipError_t launch_tile_x_f64(const double* Xrm, double* Xt, int64_t N, int64_t K,
                             const tile_geom& g, hipStream_t s) {
  const int64_t total = g.T * g.S * 64;
  if (total == 0) return hipSuccess;
  const int threads = 256;
  const int64_t blocks = (total + threads - 1) / threads;
  hipLaunchKernelGGL(tile_x_f64, dim3(static_cast<unsigned>(blocks)), dim3(threads), 0, s,
                     Xrm, Xt, N, K, g.L, g.lgL, g.S, total);
  return hipGetLastError();
}

}  // namespace sx
