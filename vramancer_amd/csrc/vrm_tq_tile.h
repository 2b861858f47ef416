// A TurboQuant row on four lanes: what the 16-rows-per-wavefront kernels share.
// Lane (r, g) = lane % 16, lane / 16 holds the quarter of row r over dims
// PD / 4 * g .. PD / 4 * g + PD / 4 - 1.
#pragma once
#include "vrm_common.h"
#include "vrm_tq_layout.h"

namespace vrm {
namespace {

#pragma clang fp contract(off)

constexpr int kTile = 16;  // rows per wavefront

// One butterfly stage across lanes for two elements a, b: the lower lane
// keeps lower + upper, the upper lane lower - upper.  The swap gathers both
// lanes' operands of a in the lower lane and of b in the upper one.
template <int H>
__device__ __forceinline__ void cross_butterfly(float& a, float& b) {
  const auto r = H == 16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                         : __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const float lo = __uint_as_float(r[0]), hi = __uint_as_float(r[1]);
  const uint32_t s = __float_as_uint(__fadd_rn(lo, hi)), d = __float_as_uint(__fsub_rn(lo, hi));
  const auto t = H == 16 ? __builtin_amdgcn_permlane16_swap(s, d, false, false)
                         : __builtin_amdgcn_permlane32_swap(s, d, false, false);
  a = __uint_as_float(t[0]);
  b = __uint_as_float(t[1]);
}

// Walsh-Hadamard transform of the row in the reference's butterfly order.
template <int PD>
__device__ __forceinline__ void tile_fwht(float (&v)[PD / 4]) {
  constexpr int NQ = PD / 4;
#pragma unroll
  for (int h = 1; h < NQ; h <<= 1) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if (!(i & h)) {
        const float lo = v[i], hi = v[i + h];
        v[i] = __fadd_rn(lo, hi);
        v[i + h] = __fsub_rn(lo, hi);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NQ; i += 2) cross_butterfly<16>(v[i], v[i + 1]);
#pragma unroll
  for (int i = 0; i < NQ; i += 2) cross_butterfly<32>(v[i], v[i + 1]);
}

// Slot of angle a of level l of a quarter.
template <int PD, int BITS>
__device__ __forceinline__ int slot_in_quarter(int l, int a) {
  int q, s;
  tq::slot_of(PD, l, a, BITS, q, s);
  return s;
}

template <int PD, int BITS>
struct Quarter {
  static constexpr int NQ = PD / 4;                          // dims, and slots, of a lane
  static constexpr int LQ = PD == 128 ? 4 : 3;               // its top level
  static constexpr int WORDS = (NQ * BITS + 31) / 32;        // dwords of its record
  uint32_t w[WORDS];

  __device__ __forceinline__ void put(int slot, uint32_t bin) {
    const int pos = slot * BITS;
    w[pos / 32] |= bin << (pos % 32);
    if (pos % 32 + BITS > 32) w[pos / 32 + 1] |= bin >> (32 - pos % 32);
  }
  __device__ __forceinline__ uint32_t get(int slot) const {
    const int pos = slot * BITS;
    uint32_t x = w[pos / 32] >> (pos % 32);
    if (pos % 32 + BITS > 32) x |= w[pos / 32 + 1] << (32 - pos % 32);
    return x & ((1u << BITS) - 1);
  }
};

}  // namespace
}  // namespace vrm
