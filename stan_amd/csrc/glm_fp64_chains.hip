// FP64 forward + adjoint pass of the GLM log density for several chains.
//
// The single-chain pass streams X once per chain.  Here a workgroup stages a
// tile of X in LDS once for 8 chains (two per wave), TT tiles at a time, and
// a lane's X values, read from LDS once, serve both of its wave's chains.
// What bounds it then is FP64 arithmetic, per (row, chain) 2 K FMAs and the
// link, at about half of its issue rate (two to three waves per SIMD, a
// barrier per step): N = 1e6, K = 100, 32 chains 848 us, of which the vector
// instructions issue for 460 (the single-chain pass over a grid of chains:
// 2678 us, X read from L2 for every chain).
//
// Lanes.  The L lanes of a row (L = 1, 2 or 4) lie 64 / L apart (lane =
// q R + r, R = 64 / L), so that every DPP row of 16 lanes holds rows of one
// column group q.  Its coefficients are then uniform in the DPP row: lane n
// of a row of 16 keeps beta of slots n and 16 + n, and the forward's FMA
// takes slot j's coefficient by row broadcast (row_newbcast, the one DPP
// control 64-bit instructions have), from two registers per chain instead of
// an LDS read per FMA.  All L lanes of a row hold its eta, so the links of
// the TT x 2 (tile, chain) pairs in flight are spread over them and the
// residuals exchanged by row swaps: no pair is evaluated twice.
//
// Every sum is formed in the single-chain pass's order, so a chain's result
// is bitwise its single evaluation: the workgroup of block b walks the tile
// sequences of that block's four waves (tiles 4 b + v, then every 4 nb-th)
// one after the other, reduces each over the row lanes, and adds the four
// in order.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../include/stanx/sx_math.hpp"
#include "glm_fp64_tile.hpp"
#include "sx_internal.hpp"
#include "wave_ops.hpp"

namespace sx {

namespace {

typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int kCB = 2;             // chains per wave
constexpr int kWG = 4 * kCB;       // chains per workgroup

// row term and residual of one (row, chain); zero past N
template <int FAM>
__device__ __forceinline__ void link_f64(double e, double yv, bool valid, double& term,
                                         double& rr) {
  term = 0.0;
  rr = 0.0;
  if (valid) {
    if (FAM == SX_LOGIT) {
      stanx::math::sx_logit_row(e, yv != 0.0 ? 1.0 : -1.0, &term, &rr);
    } else {
      const double d = yv - e;
      rr = d;
      term = d * d;
    }
  }
}

// e[2 tt + c] += beta_c(slot J0 + j) x_tt(slot J0 + j), j = 0 .. 3 in order:
// slot J0 + j's coefficient is lane (J0 + j) % 16 of b[c] in each row of 16
// lanes.  The s_nop covers a vector write of b just before (a DPP read of it
// needs two wait states, and the compiler does not look into the block).
#define SX_FMAC(E, B, X, N) \
  "v_fmac_f64_dpp " E ", " B ", " X " row_newbcast:" N " row_mask:0xf bank_mask:0xf\n\t"
template <int J0>
__device__ __forceinline__ void forward4(double (&e)[4], double b0, double b1, double x0, double x1,
                                         double x2, double x3, double y0, double y1, double y2,
                                         double y3) {
  asm("s_nop 1\n\t"
      SX_FMAC("%0", "%4", "%6", "%14") SX_FMAC("%1", "%5", "%6", "%14")
      SX_FMAC("%2", "%4", "%10", "%14") SX_FMAC("%3", "%5", "%10", "%14")
      SX_FMAC("%0", "%4", "%7", "%15") SX_FMAC("%1", "%5", "%7", "%15")
      SX_FMAC("%2", "%4", "%11", "%15") SX_FMAC("%3", "%5", "%11", "%15")
      SX_FMAC("%0", "%4", "%8", "%16") SX_FMAC("%1", "%5", "%8", "%16")
      SX_FMAC("%2", "%4", "%12", "%16") SX_FMAC("%3", "%5", "%12", "%16")
      SX_FMAC("%0", "%4", "%9", "%17") SX_FMAC("%1", "%5", "%9", "%17")
      SX_FMAC("%2", "%4", "%13", "%17") SX_FMAC("%3", "%5", "%13", "%17")
      : "+&v"(e[0]), "+&v"(e[1]), "+&v"(e[2]), "+&v"(e[3])
      : "v"(b0), "v"(b1), "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(y0), "v"(y1), "v"(y2), "v"(y3),
        "n"(J0 % 16), "n"(J0 % 16 + 1), "n"(J0 % 16 + 2), "n"(J0 % 16 + 3));
}
#undef SX_FMAC

// values of the NL lanes that share a row (NL = 1, 2, 4 of its L lanes), in
// all of them: out[i] is the value of the lane with q % NL = i
template <int LG, int NL>
__device__ __forceinline__ void spread(double v, double* out) {
  if constexpr (NL == 1) {
    out[0] = v;
  } else if constexpr (NL == 2 && LG == 1) {
    wave::both_halves(v, out[0], out[1]);
  } else if constexpr (NL == 2) {
    wave::both_rows(v, out[0], out[1]);
  } else {
    double a, b;
    wave::both_halves(v, a, b);  // a: q = 0, 1 by row; b: q = 2, 3
    wave::both_rows(a, out[0], out[1]);
    wave::both_rows(b, out[2], out[3]);
  }
}

template <int SMAX, int LG, int FAM>
__global__ __launch_bounds__(256, 2) void glm_pass_f64_chains(pass_args a, int nb) {
  constexpr int TT = 2;                   // tiles of a step
  // X values held from the forward to the adjoint; above 8 slots a second
  // LDS read of them costs less than the waves their registers would displace
  // (N = 200,003, K = 60, 16 slots: 153 us held, 137 us read again)
  constexpr bool HOLD = SMAX <= 8;
  constexpr int L = 1 << LG, R = 64 >> LG, LGR = 6 - LG;
  constexpr int XT = SMAX * 64;           // doubles of a staged tile
  constexpr int NC = TT * kCB;            // (tile, chain) pairs of a step: tt kCB + c
  constexpr int NL = L < NC ? L : NC;     // lanes of a row that share its links
  constexpr int NP = (SMAX + 7) / 8;      // 16-byte pieces of a tile per thread
  constexpr int N = SMAX + 3;             // sums of a sequence: slots, term, residual, flag
  __shared__ __attribute__((aligned(16))) double xs[2][TT * XT];
  extern __shared__ double tots[];        // block sums [wave][chain][E]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ngrp = (a.chains + kWG - 1) / kWG;
  // the chain groups of a block are 8 block ids apart where nb allows (one
  // XCD): the first brings the tiles into its L2
  int blk, grp;
  {
    const int id = blockIdx.x;
    if ((nb & 7) == 0) {
      const int u = id >> 3;
      blk = (id & 7) + 8 * (u / ngrp);
      grp = u % ngrp;
    } else {
      blk = id % nb;
      grp = id / nb;
    }
    blk = __builtin_amdgcn_readfirstlane(blk);
    grp = __builtin_amdgcn_readfirstlane(grp);
  }
  const int S = a.S, K = a.K, E = a.E;
  const int q = lane >> LGR, r = lane & (R - 1);
  const int c0 = grp * kWG + w * kCB;  // first chain of this wave
  const bool active = c0 < a.chains;   // else it only helps to stage
  double* const tot = tots + w * kCB * E;
  // slots past S and a step's missing second tile are never staged: finite
  // from the start (their products are with zeros)
  for (int i = threadIdx.x; i < TT * XT; i += 256) xs[0][i] = xs[1][i] = 0.0;
  double be[kCB][2], alpha[kCB];
#pragma unroll
  for (int c = 0; c < kCB; ++c) {
    const int ch = c0 + c < a.chains ? c0 + c : a.chains - 1;
    const double* th = a.theta + static_cast<int64_t>(ch) * a.theta_stride;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int col = (16 * i + (lane & 15)) * L + q;
      be[c][i] = col < K ? th[1 + col] : 0.0;
    }
    alpha[c] = th[0];
    for (int i = lane; i < E; i += 64) tot[c * E + i] = 0.0;
  }
  __syncthreads();
  double acc[kCB][SMAX], s0[kCB], s1[kCB], bad[kCB];
  const int64_t W = static_cast<int64_t>(nb) * 4;
  // a step's tiles t, t + W (those below T) and the wave's y values, into
  // registers, then into LDS (a tile past T: what was loaded before, finite)
  f64x2 stg[TT][NP];
  double yn[TT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
#pragma unroll
    for (int i = 0; i < NP; ++i) stg[tt][i] = f64x2{0.0, 0.0};
  const int pieces = S * 32;
  auto load = [&](int64_t t) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const int64_t tn = t + tt * W;
      yn[tt] = 0.0;
      if (tn < a.T) {
        yn[tt] = load_y<FAM>(a, tn, R, r);
        const f64x2* src =
            reinterpret_cast<const f64x2*>(a.X + tn * static_cast<int64_t>(S) * 64) + threadIdx.x;
#pragma unroll
        for (int i = 0; i < NP; ++i)
          if (static_cast<int>(threadIdx.x) + 256 * i < pieces) stg[tt][i] = src[256 * i];
      }
    }
  };
  auto store = [&](double* X) {
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      f64x2* dst = reinterpret_cast<f64x2*>(X + tt * XT) + threadIdx.x;
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (static_cast<int>(threadIdx.x) + 256 * i < pieces) dst[256 * i] = stg[tt][i];
    }
  };

  // one step: forward, link, adjoint on tiles t, t + W in X
  auto step = [&](const double* X, int64_t t, const double (&y)[TT]) {
    double e[NC], xv[TT][HOLD ? SMAX : 8];
#pragma unroll
    for (int i = 0; i < NC; ++i) e[i] = 0.0;
    // four slots at a time, the next four's reads in flight
    auto read = [&](int j0) {
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          xv[tt][HOLD ? j0 + j : (j0 & 4) + j] = X[tt * XT + (j0 + j) * 64 + lane];
    };
    auto fwd = [&](auto j0c) {
      constexpr int J0 = decltype(j0c)::value, O = HOLD ? J0 : J0 & 4;
      if (J0 + 4 < SMAX) read(J0 + 4);
      forward4<J0>(e, be[0][J0 / 16], be[1][J0 / 16], xv[0][O], xv[0][O + 1], xv[0][O + 2],
                   xv[0][O + 3], xv[1][O], xv[1][O + 1], xv[1][O + 2], xv[1][O + 3]);
    };
    read(0);
    fwd(std::integral_constant<int, 0>{});
    if constexpr (SMAX > 4) fwd(std::integral_constant<int, 4>{});
    if constexpr (SMAX > 8) fwd(std::integral_constant<int, 8>{});
    if constexpr (SMAX > 12) fwd(std::integral_constant<int, 12>{});
    if constexpr (SMAX > 16) fwd(std::integral_constant<int, 16>{});
    if constexpr (SMAX > 20) fwd(std::integral_constant<int, 20>{});
    if constexpr (SMAX > 24) fwd(std::integral_constant<int, 24>{});
    if constexpr (SMAX > 28) fwd(std::integral_constant<int, 28>{});
    wave::xor_sum_n<NC>(e, R, 64);
    int rows[TT];  // of the tile; <= 0: none
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      const int64_t left = a.N - (t + tt * W) * R;
      rows[tt] = left < R ? static_cast<int>(left < 0 ? 0 : left) : R;
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      e[i] += alpha[i % kCB];
      bad[i % kCB] = fma(e[i], 0.0, bad[i % kCB]);  // NaN once an eta is not finite
    }
    double term[NC], rr[NC];
#pragma unroll
    for (int k = 0; k < NC / NL; ++k) {
      double em = e[k * NL], ym = y[k * NL / kCB];
      int rm = rows[k * NL / kCB];
#pragma unroll
      for (int i = 1; i < NL; ++i)
        if ((q & (NL - 1)) == i) {
          em = e[k * NL + i];
          ym = y[(k * NL + i) / kCB];
          rm = rows[(k * NL + i) / kCB];
        }
      double tm, res;
      link_f64<FAM>(em, ym, r < rm, tm, res);
      spread<LG, NL>(tm, term + k * NL);
      spread<LG, NL>(res, rr + k * NL);
    }
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
      for (int c = 0; c < kCB; ++c) {
        s0[c] += term[tt * kCB + c];
        s1[c] += rr[tt * kCB + c];
      }
    if (!HOLD) asm volatile("" ::: "memory");  // X is read again, not held through the link
#pragma unroll
    for (int j = 0; j < SMAX; ++j)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        const double x = HOLD ? xv[tt][HOLD ? j : 0] : X[tt * XT + j * 64 + lane];
#pragma unroll
        for (int c = 0; c < kCB; ++c) acc[c][j] = fma(x, rr[tt * kCB + c], acc[c][j]);
      }
  };

  const int64_t first = static_cast<int64_t>(blk) * 4;
  int buf = 0;
  if (first < a.T) {
    load(first);
    store(xs[0]);
  }
  for (int v = 0; v < 4 && first + v < a.T; ++v) {
#pragma unroll
    for (int c = 0; c < kCB; ++c) {
#pragma unroll
      for (int j = 0; j < SMAX; ++j) acc[c][j] = 0.0;
      s0[c] = s1[c] = bad[c] = 0.0;
    }
    for (int64_t t = first + v; t < a.T; t += TT * W) {
      __syncthreads();
      double y[TT];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) y[tt] = yn[tt];
      // the next step, of this sequence or the next one, in flight
      int64_t tn = t + TT * W;
      if (tn >= a.T) tn = v < 3 ? first + v + 1 : a.T;
      if (tn < a.T) load(tn);
      if (active) step(xs[buf], t, y);
      buf ^= 1;
      if (tn < a.T) store(xs[buf]);  // its last readers passed this step's barrier
    }
    if (!active) continue;
    // the sequence's sums over the row lanes (slots, then the row terms,
    // residuals and non-finite flag of the lanes q = 0) join the block's
    int ln = lane; /* opaque: the addresses are formed here, not held */
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int c = 0; c < kCB; ++c) {
      double u[N];
#pragma unroll
      for (int j = 0; j < SMAX; ++j) u[j] = acc[c][j];
      u[SMAX] = s0[c];
      u[SMAX + 1] = s1[c];
      u[SMAX + 2] = bad[c] == bad[c] ? 0.0 : 1.0;
      wave::scatter_sum<0, LGR, N>(u);
#pragma unroll
      for (int i = 0; i < wave::scatter_left(0, LGR, N); ++i) {
        const int sl = wave::scatter_index<0, LGR, N>(ln, i), lq = ln >> LGR;
        int at = -1;
        if (sl >= SMAX) {
          if (lq == 0) at = sl == SMAX ? 0 : (sl == SMAX + 1 ? 1 : K + 2);
        } else if (sl >= 0 && sl * L + lq < K) {
          at = 2 + sl * L + lq;
        }
        if (at >= 0) tot[c * E + at] += u[i];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kCB; ++c)
    if (c0 + c < a.chains) {
      double* out = a.partials + static_cast<int64_t>(c0 + c) * E * nb + blk;
      for (int i = lane; i < E; i += 64) out[static_cast<int64_t>(i) * nb] = tot[c * E + i];
    }
}

template <int SMAX, int LG>
void launch_one(int family, const pass_args& a, int blocks, hipStream_t s) {
  const int ngrp = (a.chains + kWG - 1) / kWG;
  const size_t lds = static_cast<size_t>(kWG) * a.E * sizeof(double);
  if (family == SX_LOGIT)
    hipLaunchKernelGGL((glm_pass_f64_chains<SMAX, LG, SX_LOGIT>), dim3(blocks * ngrp), dim3(256),
                       lds, s, a, blocks);
  else
    hipLaunchKernelGGL((glm_pass_f64_chains<SMAX, LG, SX_NORMAL>), dim3(blocks * ngrp), dim3(256),
                       lds, s, a, blocks);
}

template <int LG>
hipError_t launch_lg(int family, int smax, const pass_args& a, int blocks, hipStream_t s) {
  switch (smax) {
    case 4: launch_one<4, LG>(family, a, blocks, s); break;
    case 8: launch_one<8, LG>(family, a, blocks, s); break;
    case 12: launch_one<12, LG>(family, a, blocks, s); break;
    case 16: launch_one<16, LG>(family, a, blocks, s); break;
    case 20: launch_one<20, LG>(family, a, blocks, s); break;
    case 24: launch_one<24, LG>(family, a, blocks, s); break;
    case 28: launch_one<28, LG>(family, a, blocks, s); break;
    case 32: launch_one<32, LG>(family, a, blocks, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pass_f64_chains(int family, const tile_geom& g, const pass_args& a, int blocks,
                                  hipStream_t s) {
  switch (g.L) {
    case 1: return launch_lg<0>(family, g.smax, a, blocks, s);
    case 2: return launch_lg<1>(family, g.smax, a, blocks, s);
    case 4: return launch_lg<2>(family, g.smax, a, blocks, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace sx
