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

// sum over the lanes that differ in the bits from lo up to (not including)
// hi, powers of two, one distance after the other
__device__ __forceinline__ double xor_sum(double v, int lo, int hi) {
  if (lo <= 1 && hi > 1) v = add_xor<1>(v);
  if (lo <= 2 && hi > 2) v = add_xor<2>(v);
  if (lo <= 4 && hi > 4) v = add_xor<4>(v);
  if (lo <= 8 && hi > 8) v = add_xor<8>(v);
  if (lo <= 16 && hi > 16) v = add_xor<16>(v);
  if (lo <= 32 && hi > 32) v = add_xor<32>(v);
  return v;
}

// Sum of v over the 64 lanes (xor butterfly): every lane gets the total.
__device__ __forceinline__ double sum(double v) { return xor_sum(v, 1, 64); }

}  // namespace wave
}  // namespace sx
#endif
