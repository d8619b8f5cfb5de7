// lane_ops.hpp -- exact moves of doubles between the lanes of a quad, and the
// butterfly sum of a wave.
#pragma once

#include <hip/hip_runtime.h>

namespace femdev {

// every lane of a quad (lanes 4j .. 4j + 3) receives lane L's value: a DPP
// quad broadcast of both 32-bit halves, so the bits move unchanged
template <int L>
__device__ inline double quad_bcast(double v) {
  typedef unsigned int qb_u32x2 __attribute__((ext_vector_type(2)));
  const qb_u32x2 x = __builtin_bit_cast(qb_u32x2, v);
  qb_u32x2 r;
  r.x = uint32_t(__builtin_amdgcn_mov_dpp(int(x.x), L * 0x55, 0xF, 0xF, false));
  r.y = uint32_t(__builtin_amdgcn_mov_dpp(int(x.y), L * 0x55, 0xF, 0xF, false));
  return __builtin_bit_cast(double, r);
}

// value of lane i ^ X, X = 1, 2, 4 or 8
template <int X>
__device__ inline double lane_xor(double v) {
  typedef unsigned int lx_u32x2 __attribute__((ext_vector_type(2)));
  const lx_u32x2 x = __builtin_bit_cast(lx_u32x2, v);
  auto move = [](uint32_t h) -> uint32_t {
    constexpr int CTRL = X == 1 ? 0xB1 : X == 2 ? 0x4E : 0x128;  // quad permutations, rotation of a row by 8
    if (X != 4) return uint32_t(__builtin_amdgcn_mov_dpp(int(h), CTRL, 0xF, 0xF, false));
    // even quads of a row from four lanes up, odd ones from four lanes down
    const int up = __builtin_amdgcn_update_dpp(0, int(h), 0x104, 0xF, 0x5, false);
    return uint32_t(__builtin_amdgcn_update_dpp(up, int(h), 0x114, 0xF, 0xA, false));
  };
  lx_u32x2 r;
  r.x = move(x.x);
  r.y = move(x.y);
  return __builtin_bit_cast(double, r);
}

// v + (v of lane i ^ X), X = 16 or 32: the swap leaves one of the two in each result
template <int X>
__device__ inline double half_sum(double v) {
  typedef unsigned int hs_u32x2 __attribute__((ext_vector_type(2)));
  const hs_u32x2 x = __builtin_bit_cast(hs_u32x2, v);
  auto swap = [](uint32_t h) {
    if (X == 16) return __builtin_amdgcn_permlane16_swap(h, h, false, false);
    return __builtin_amdgcn_permlane32_swap(h, h, false, false);
  };
  const auto lo = swap(x.x), hi = swap(x.y);
  hs_u32x2 a, b;
  a.x = lo[0];
  a.y = hi[0];
  b.x = lo[1];
  b.y = hi[1];
  return __builtin_bit_cast(double, a) + __builtin_bit_cast(double, b);
}

// sum over the wave in every lane: a butterfly of distances 32, 16, 8, 4, 2, 1.
// Register moves: a shuffle through LDS takes several times as long, and the
// six steps wait for each other.
__device__ inline double wave_sum(double v) {
  v = half_sum<32>(v);
  v = half_sum<16>(v);
  v += lane_xor<8>(v);
  v += lane_xor<4>(v);
  v += lane_xor<2>(v);
  v += lane_xor<1>(v);
  return v;
}

}  // namespace femdev
