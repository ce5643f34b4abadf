#pragma once
// What the kernels that run the B/C projections inside the SSM walk share (fused_bc.hip,
// fused_bc_short.hip).
#include "mfma_tile.hpp"
#include "ssm_chunk.hpp"

namespace mqc {

using namespace mfma;

// W rows of one K stage of a GEMM tile: rows [0, R) from W_B and [R, 2 R) from W_C, hs4 = 4
// times the unit's states of each (rows past them read the unit's first state: in a ragged
// last unit the 8-row groups of a DMA instruction are whole pairs of states, d_state being
// even).
template <int R>
struct WRowsOf {
  const uint16_t* wb;
  const uint16_t* wc;
  int64_t row0;
  int hs4, K;
  __device__ const void* operator()(int g, int k0, int i, uint32_t& voff,
                                    const DmaLane& dl) const {
    voff = (uint32_t)(dl.lrow * K * 2) + dl.cb(i);
    const int r = g & (R - 1);  // 8-row groups never straddle B and C
    const int rr = r < hs4 ? r : 0;
    return (g < R ? wb : wc) + ((row0 + rr) * K + k0);
  }
};

// The walk's and the epilogue's LDS addresses are the same for every tile; left to
// itself the compiler computes them once and holds them (tens of registers) through
// the K loop, which then spills. Passing a lane's base through this empty statement
// makes it opaque, so the addresses derived from it are recomputed where used.
template <typename V>
__device__ inline V opaque(V v) {
  asm volatile("" : "+v"(v));
  return v;
}

// The two 16-bit elements of a 32-bit word (low half first) in fp32.
template <typename T>
__device__ inline float lo16(uint32_t w) {
  if constexpr (std::is_same<T, bf16_t>::value) return __uint_as_float(w << 16);
  else return io<T>::bits_to_f32(w & 0xffffu);
}
template <typename T>
__device__ inline float hi16(uint32_t w) {
  if constexpr (std::is_same<T, bf16_t>::value) return __uint_as_float(w & 0xffff0000u);
  else return io<T>::bits_to_f32(w >> 16);
}

// Exchange x of the odd 16-lane rows with y of the even rows (v_permlane16_swap_b32):
// afterwards even-row lanes hold (own x, the odd neighbour's x) and odd-row lanes
// (the even neighbour's y, own y). Issued as assembly with both registers read-write,
// as the library's other row swaps (common.hpp), N pairs behind one pair of s_nops.
template <int N>
__device__ inline void row_swap16(float* x, float* y) {
  static_assert(N == 8, "eight pairs per statement");
  asm volatile(
      "s_nop 1\n\t"
      "v_permlane16_swap_b32 %0, %8\n\t"
      "v_permlane16_swap_b32 %1, %9\n\t"
      "v_permlane16_swap_b32 %2, %10\n\t"
      "v_permlane16_swap_b32 %3, %11\n\t"
      "v_permlane16_swap_b32 %4, %12\n\t"
      "v_permlane16_swap_b32 %5, %13\n\t"
      "v_permlane16_swap_b32 %6, %14\n\t"
      "v_permlane16_swap_b32 %7, %15\n\t"
      "s_nop 1"
      : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]),
        "+v"(x[7]), "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]),
        "+v"(y[6]), "+v"(y[7]));
}

__device__ inline float row_half_mirror(float v) { return dpp_mov<0x141>(v); }

}  // namespace mqc
