// Cross-lane sums within a wave on the VALU (gfx950): DPP permutations for
// lane distances 1, 2, 4, 8 and the row-swapping permlane instructions for
// 16 and 32.  A shuffle through LDS (ds_bpermute) costs an LDS round trip
// per step and dword; these cost one or two VALU instructions, which is what
// the latency of a 64-lane sum of a double (six dependent steps) hangs on.
// Every step adds the same two values as the shuffle it replaces (a + b, or
// b + a), so sums are bitwise those of __shfl_xor.  Measured: a single
// evaluation at N = 3000, K = 37 24.2 -> 21.5 us, at N = 1e6, K = 100 134.7
// -> 131.5 us; 256 device chains (N = 20,000, K = 100) 5 % per run.
#ifndef STANX_WAVE_OPS_HPP
#define STANX_WAVE_OPS_HPP

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sx {
namespace wave {

// DPP controls
constexpr int kQuadXor1 = 0xb1;       // quad_perm [1, 0, 3, 2]
constexpr int kQuadXor2 = 0x4e;       // quad_perm [2, 3, 0, 1]
constexpr int kRowShl4 = 0x104;       // lane i reads lane i + 4 of its row
constexpr int kRowShr4 = 0x114;       // lane i reads lane i - 4 of its row
constexpr int kRowRor8 = 0x128;       // lane i reads lane i ^ 8 of its row of 16

// the dword of lane ^ OFF (OFF = 1, 2, 4, 8)
template <int OFF>
__device__ __forceinline__ int dpp_xor(int x) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8, "within a row of 16 lanes");
  if constexpr (OFF == 1) return __builtin_amdgcn_mov_dpp(x, kQuadXor1, 0xf, 0xf, true);
  if constexpr (OFF == 2) return __builtin_amdgcn_mov_dpp(x, kQuadXor2, 0xf, 0xf, true);
  if constexpr (OFF == 4) {
    // lanes 0-3 and 8-11 of a row read upwards, 4-7 and 12-15 downwards
    const int up = __builtin_amdgcn_update_dpp(x, x, kRowShl4, 0xf, 0x5, false);
    return __builtin_amdgcn_update_dpp(up, x, kRowShr4, 0xf, 0xa, false);
  }
  return __builtin_amdgcn_mov_dpp(x, kRowRor8, 0xf, 0xf, true);
}

// v + (v of lane ^ OFF), OFF = 1 .. 32
template <int OFF>
__device__ __forceinline__ double add_xor(double v) {
  const uint64_t b = __double_as_longlong(v);
  const unsigned lo = static_cast<unsigned>(b), hi = static_cast<unsigned>(b >> 32);
  if constexpr (OFF <= 8) {
    const unsigned l2 = dpp_xor<OFF>(static_cast<int>(lo)), h2 = dpp_xor<OFF>(static_cast<int>(hi));
    return v + __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(h2) << 32) | l2));
  } else {
    // the swap of a value with its own copy leaves the even rows (halves)
    // of both in one register and the odd ones in the other
    unsigned l0, l1, h0, h1;
    if constexpr (OFF == 16) {
      const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
      l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
    } else {
      const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
      const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
      l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
    }
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(h0) << 32) | l0)) +
           __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(h1) << 32) | l1));
  }
}

// v[0 .. N): sums over the lanes that differ in the bits from lo up to (not
// including) hi, powers of two, one distance after the other
template <int N>
__device__ __forceinline__ void xor_sum_n(double (&v)[N], int lo, int hi) {
#define SX_XOR_STEP(OFF)            \
  if (lo <= OFF && hi > OFF) {      \
    _Pragma("unroll") for (int i = 0; i < N; ++i) v[i] = add_xor<OFF>(v[i]); \
  }
  SX_XOR_STEP(1)
  SX_XOR_STEP(2)
  SX_XOR_STEP(4)
  SX_XOR_STEP(8)
  SX_XOR_STEP(16)
  SX_XOR_STEP(32)
#undef SX_XOR_STEP
}
__device__ __forceinline__ double xor_sum(double v, int lo, int hi) {
  double x[1] = {v};
  xor_sum_n<1>(x, lo, hi);
  return x[0];
}

// Scattered sums of N values over the lanes that differ in bits LG .. END-1:
// at each distance a lane keeps one half of its values and hands the other
// half to its partner, so the work halves from step to step (a full
// butterfly does all N at every distance).  The additions, and so the bits,
// are the butterfly's.  At the end a lane's v[i], i < scatter_left(LG, END,
// N), is the total of value scatter_index<..>(lane, i) (-1: none).
constexpr int scatter_left(int LG, int END, int N) {
  return LG >= END ? N : scatter_left(LG + 1, END, (N + 1) / 2);
}
template <int LG, int END, int N>
__device__ __forceinline__ int scatter_index(int lane, int i) {
  if constexpr (LG >= END) {
    return i;
  } else {
    constexpr int H = (N + 1) / 2;
    int j = scatter_index<LG + 1, END, H>(lane, i);
    if (j >= 0 && (lane & (1 << LG))) j += H;
    return j < N ? j : -1;
  }
}
// lanes with bit OFF clear: a + (a of lane ^ OFF); set: b + (b of lane ^ OFF)
template <int OFF>
__device__ __forceinline__ double keep_half(double a, double b) {
  const uint64_t ua = __double_as_longlong(a), ub = __double_as_longlong(b);
  unsigned aw[2] = {static_cast<unsigned>(ua), static_cast<unsigned>(ua >> 32)};
  unsigned bw[2] = {static_cast<unsigned>(ub), static_cast<unsigned>(ub >> 32)};
  unsigned x[2], y[2];  // own and partner's
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if constexpr (OFF == 16) {
      const auto w = __builtin_amdgcn_permlane16_swap(aw[i], bw[i], false, false);
      x[i] = w[0], y[i] = w[1];
    } else if constexpr (OFF == 32) {
      const auto w = __builtin_amdgcn_permlane32_swap(aw[i], bw[i], false, false);
      x[i] = w[0], y[i] = w[1];
    } else if constexpr (OFF >= 4) {
      // banks of 4 lanes: those with the bit set take b
      constexpr int set = OFF == 4 ? 0xa : 0xc, clear = 0xf ^ set;
      constexpr int up = OFF == 4 ? kRowShl4 : kRowRor8, down = OFF == 4 ? kRowShr4 : kRowRor8;
      x[i] = __builtin_amdgcn_update_dpp(aw[i], bw[i], 0xe4 /* same lane */, 0xf, set, false);
      const int t = __builtin_amdgcn_update_dpp(aw[i], aw[i], up, 0xf, clear, false);
      y[i] = __builtin_amdgcn_update_dpp(t, bw[i], down, 0xf, set, false);
    } else {
      const bool set = (__lane_id() & OFF) != 0;
      x[i] = set ? bw[i] : aw[i];
      const int pa = dpp_xor<OFF>(aw[i]), pb = dpp_xor<OFF>(bw[i]);
      y[i] = set ? pb : pa;
    }
  }
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(x[1]) << 32) | x[0])) +
         __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(y[1]) << 32) | y[0]));
}
template <int LG, int END, int N, int M>
__device__ __forceinline__ void scatter_sum(double (&v)[M]) {
  if constexpr (LG < END) {
    constexpr int H = (N + 1) / 2;
#pragma unroll
    for (int i = 0; i < H; ++i)
      v[i] = keep_half<(1 << LG)>(v[i], i + H < N ? v[i + H < N ? i + H : 0] : 0.0);
    scatter_sum<LG + 1, END, H>(v);
  }
}

// Both values of a pair of lanes, in each of the two: swaps of v with its
// own copy.
__device__ __forceinline__ void swap16(unsigned v, unsigned& even, unsigned& odd) {
  const auto w = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  even = w[0], odd = w[1];
}
__device__ __forceinline__ void swap32(unsigned v, unsigned& lo, unsigned& hi) {
  const auto w = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  lo = w[0], hi = w[1];
}
__device__ __forceinline__ double join(unsigned lo, unsigned hi) {
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
// lane bit 5: out[0] from the lower half's lane, out[1] from the upper's
__device__ __forceinline__ void both_halves(double v, double& a, double& b) {
  const uint64_t u = __double_as_longlong(v);
  unsigned l0, l1, h0, h1;
  swap32(static_cast<unsigned>(u), l0, l1);
  swap32(static_cast<unsigned>(u >> 32), h0, h1);
  a = join(l0, h0);
  b = join(l1, h1);
}
// lane bit 4
__device__ __forceinline__ void both_rows(double v, double& a, double& b) {
  const uint64_t u = __double_as_longlong(v);
  unsigned l0, l1, h0, h1;
  swap16(static_cast<unsigned>(u), l0, l1);
  swap16(static_cast<unsigned>(u >> 32), h0, h1);
  a = join(l0, h0);
  b = join(l1, h1);
}

// Sum of v over the 64 lanes (xor butterfly): every lane gets the total.
__device__ __forceinline__ double sum(double v) { return xor_sum(v, 1, 64); }

}  // namespace wave
}  // namespace sx
#endif
