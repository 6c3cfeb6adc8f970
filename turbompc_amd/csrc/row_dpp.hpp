// Row products with the broadcast folded into the arithmetic, for kernels that
// keep a vector one element per lane of a 16-lane DPP row: lane k of the row is
// read by every lane of it (row_newbcast:k) inside v_fmac_*_dpp, one instruction
// per term and no LDS.  The compiler keeps such a broadcast as a separate move,
// so the blocks are written out.  Each block starts with the wait states a DPP
// read needs after a VALU write of its source; a result is last written by an
// ordinary instruction (the final add), or the block ends with wait states.
// Accumulators are early-clobber operands ("+&v"): later instructions of a block
// still read its sources, also where one holds an accumulator's starting value.
// Every lane of a 16-lane row that is active at all must be active.
#pragma once
#include "common.hpp"

namespace tmpc {

// acc + sum_k w[k] s(lane O + k), k < N: even and odd k in two chains (the odd
// one starts with a multiply in fp32; v_mul_f64 has no DPP form, so it starts
// at zero in fp64).

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[2], float s, float acc) {
  static_assert(O >= 0 && O + 2 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "n"(O + 0), "n"(O + 1));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[3], float s, float acc) {
  static_assert(O >= 0 && O + 3 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c8 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "n"(O + 0), "n"(O + 1), "n"(O + 2));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[4], float s, float acc) {
  static_assert(O >= 0 && O + 4 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c10 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[6], float s, float acc) {
  static_assert(O >= 0 && O + 6 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:%c14 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[12], float s, float acc) {
  static_assert(O >= 0 && O + 12 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c15 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c16 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c17 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c18 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:%c19 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:%c20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:%c21 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:%c22 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:%c23 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %12 row_newbcast:%c24 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:%c25 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %14 row_newbcast:%c26 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5), "n"(O + 6), "n"(O + 7), "n"(O + 8), "n"(O + 9), "n"(O + 10), "n"(O + 11));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ float row_fma(const float (&w)[13], float s, float acc) {
  static_assert(O >= 0 && O + 13 <= 16, "a 16-lane row");
  float odd;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c16 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %4 row_newbcast:%c17 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c18 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c19 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:%c20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:%c21 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:%c22 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:%c23 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:%c24 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %12 row_newbcast:%c25 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:%c26 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %14 row_newbcast:%c27 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %15 row_newbcast:%c28 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "=&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "v"(w[12]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5), "n"(O + 6), "n"(O + 7), "n"(O + 8), "n"(O + 9), "n"(O + 10), "n"(O + 11), "n"(O + 12));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[2], double s, double acc) {
  static_assert(O >= 0 && O + 2 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c6 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "n"(O + 0), "n"(O + 1));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[3], double s, double acc) {
  static_assert(O >= 0 && O + 3 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c8 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "n"(O + 0), "n"(O + 1), "n"(O + 2));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[4], double s, double acc) {
  static_assert(O >= 0 && O + 4 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c10 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[6], double s, double acc) {
  static_assert(O >= 0 && O + 6 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:%c14 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[12], double s, double acc) {
  static_assert(O >= 0 && O + 12 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c15 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c16 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c17 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c18 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:%c19 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:%c20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:%c21 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:%c22 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:%c23 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %12 row_newbcast:%c24 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:%c25 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %14 row_newbcast:%c26 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5), "n"(O + 6), "n"(O + 7), "n"(O + 8), "n"(O + 9), "n"(O + 10), "n"(O + 11));
  return acc + odd;
}

template <int O>
__device__ __forceinline__ double row_fma(const double (&w)[13], double s, double acc) {
  static_assert(O >= 0 && O + 13 <= 16, "a 16-lane row");
  double odd = 0.0;
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c16 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %4 row_newbcast:%c17 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c18 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c19 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:%c20 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:%c21 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:%c22 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:%c23 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:%c24 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %12 row_newbcast:%c25 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:%c26 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %14 row_newbcast:%c27 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:%c28 row_mask:0xf bank_mask:0xf"
      : "+&v"(acc), "+&v"(odd)
      : "v"(s), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "v"(w[12]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3), "n"(O + 4), "n"(O + 5), "n"(O + 6), "n"(O + 7), "n"(O + 8), "n"(O + 9), "n"(O + 10), "n"(O + 11), "n"(O + 12));
  return acc + odd;
}

// (g + h) + sum_k w[k] s(lane k), k < N.  The sum of g and h is formed in the block, in the
// place of a wait state: formed before it, the compiler waits for g and h ahead of the
// loads that the caller has in flight (a chain of fp64, T = 101, NX = 6 7270 cycles, 6810
// like this).

__device__ __forceinline__ float row_fma_sum(const float (&w)[4], float s, float g, float h) {
  float acc, odd;
  asm volatile(
      "s_nop 0\n"
      "v_add_f32 %0, %3, %4\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "=&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
  return acc + odd;
}

__device__ __forceinline__ float row_fma_sum(const float (&w)[6], float s, float g, float h) {
  float acc, odd;
  asm volatile(
      "s_nop 0\n"
      "v_add_f32 %0, %3, %4\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "=&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]));
  return acc + odd;
}

__device__ __forceinline__ float row_fma_sum(const float (&w)[12], float s, float g, float h) {
  float acc, odd;
  asm volatile(
      "s_nop 0\n"
      "v_add_f32 %0, %3, %4\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "=&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]));
  return acc + odd;
}

__device__ __forceinline__ float row_fma_sum(const float (&w)[13], float s, float g, float h) {
  float acc, odd;
  asm volatile(
      "s_nop 0\n"
      "v_add_f32 %0, %3, %4\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_mul_f32_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "=&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "v"(w[12]));
  return acc + odd;
}

__device__ __forceinline__ double row_fma_sum(const double (&w)[4], double s, double g, double h) {
  double acc, odd = 0.0;
  asm volatile(
      "s_nop 0\n"
      "v_add_f64 %0, %3, %4\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "+&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]));
  return acc + odd;
}

__device__ __forceinline__ double row_fma_sum(const double (&w)[6], double s, double g, double h) {
  double acc, odd = 0.0;
  asm volatile(
      "s_nop 0\n"
      "v_add_f64 %0, %3, %4\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "+&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]));
  return acc + odd;
}

__device__ __forceinline__ double row_fma_sum(const double (&w)[12], double s, double g, double h) {
  double acc, odd = 0.0;
  asm volatile(
      "s_nop 0\n"
      "v_add_f64 %0, %3, %4\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "+&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]));
  return acc + odd;
}

__device__ __forceinline__ double row_fma_sum(const double (&w)[13], double s, double g, double h) {
  double acc, odd = 0.0;
  asm volatile(
      "s_nop 0\n"
      "v_add_f64 %0, %3, %4\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf"
      : "=&v"(acc), "+&v"(odd)
      : "v"(s), "v"(g), "v"(h), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "v"(w[11]), "v"(w[12]));
  return acc + odd;
}

// Two or three such sums side by side, one chain each (in place): independent
// chains leave no stall between dependent instructions (one chain alone issues every
// 8.4 cycles, two every 6.5, three and more every 5.1).

__device__ __forceinline__ void row_fma_2(const float (&w0)[4], float s0, float& a0, const float (&w1)[4], float s1, float& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %8 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %9 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %10 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %11 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]));
}

__device__ __forceinline__ void row_fma_3(const float (&w0)[4], float s0, float& a0, const float (&w1)[4], float s1, float& a1, const float (&w2)[4], float s2, float& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %10 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %14 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %11 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %15 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %12 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %16 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %13 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %17 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]));
}

__device__ __forceinline__ void row_fma_2(const float (&w0)[6], float s0, float& a0, const float (&w1)[6], float s1, float& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %10 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %11 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %12 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %13 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %14 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %15 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]));
}

__device__ __forceinline__ void row_fma_3(const float (&w0)[6], float s0, float& a0, const float (&w1)[6], float s1, float& a1, const float (&w2)[6], float s2, float& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %12 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %18 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %13 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %19 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %14 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %20 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %15 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %21 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %16 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %17 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]));
}

__device__ __forceinline__ void row_fma_2(const float (&w0)[12], float s0, float& a0, const float (&w1)[12], float s1, float& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %16 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %17 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %18 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %19 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %20 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %21 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %22 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %23 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %24 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %25 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %26 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %27 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]));
}

__device__ __forceinline__ void row_fma_3(const float (&w0)[12], float s0, float& a0, const float (&w1)[12], float s1, float& a1, const float (&w2)[12], float s2, float& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %18 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %30 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %19 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %31 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %20 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %32 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %21 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %33 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %34 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %35 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %12 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %24 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %36 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %13 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %25 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %37 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %14 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %26 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %38 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %15 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %27 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %39 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %16 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %28 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %40 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %29 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %41 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]), "v"(w2[6]), "v"(w2[7]), "v"(w2[8]), "v"(w2[9]), "v"(w2[10]), "v"(w2[11]));
}

__device__ __forceinline__ void row_fma_2(const float (&w0)[13], float s0, float& a0, const float (&w1)[13], float s1, float& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %17 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %18 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %19 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %20 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %21 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %22 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %23 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %24 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %25 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %26 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %27 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %28 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %16 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %3, %29 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w0[12]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w1[12]));
}

__device__ __forceinline__ void row_fma_3(const float (&w0)[13], float s0, float& a0, const float (&w1)[13], float s1, float& a1, const float (&w2)[13], float s2, float& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %19 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %32 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %20 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %33 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %21 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %34 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %22 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %35 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %23 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %36 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %24 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %37 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %12 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %25 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %38 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %13 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %26 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %39 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %14 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %27 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %40 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %15 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %28 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %41 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %16 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %29 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %42 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %30 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %43 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %3, %18 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %4, %31 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %5, %44 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w0[12]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w1[12]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]), "v"(w2[6]), "v"(w2[7]), "v"(w2[8]), "v"(w2[9]), "v"(w2[10]), "v"(w2[11]), "v"(w2[12]));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(float s, const float (&w0)[2], float& a0, const float (&w1)[2], float& a1) {
  static_assert(O >= 0 && O + 2 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %5 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w1[0]), "v"(w1[1]), "n"(O + 0), "n"(O + 1));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(float s, const float (&w0)[3], float& a0, const float (&w1)[3], float& a1) {
  static_assert(O >= 0 && O + 3 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %6 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %7 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "n"(O + 0), "n"(O + 1), "n"(O + 2));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(float s, const float (&w0)[4], float& a0, const float (&w1)[4], float& a1) {
  static_assert(O >= 0 && O + 4 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f32_dpp %0, %2, %3 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %7 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %4 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %8 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %5 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %9 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %2, %10 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3));
}

__device__ __forceinline__ void row_fma_2(const double (&w0)[4], double s0, double& a0, const double (&w1)[4], double s1, double& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %8 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %9 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %10 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %11 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]));
}

__device__ __forceinline__ void row_fma_3(const double (&w0)[4], double s0, double& a0, const double (&w1)[4], double s1, double& a1, const double (&w2)[4], double s2, double& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %10 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %14 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %11 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %15 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %12 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %16 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %13 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %17 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]));
}

__device__ __forceinline__ void row_fma_2(const double (&w0)[6], double s0, double& a0, const double (&w1)[6], double s1, double& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %10 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %11 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %12 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %13 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %14 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %15 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]));
}

__device__ __forceinline__ void row_fma_3(const double (&w0)[6], double s0, double& a0, const double (&w1)[6], double s1, double& a1, const double (&w2)[6], double s2, double& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %12 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %18 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %13 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %19 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %14 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %20 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %15 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %21 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %16 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %17 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]));
}

__device__ __forceinline__ void row_fma_2(const double (&w0)[12], double s0, double& a0, const double (&w1)[12], double s1, double& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %16 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %17 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %18 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %19 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %20 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %21 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %22 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %23 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %24 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %25 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %26 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %27 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]));
}

__device__ __forceinline__ void row_fma_3(const double (&w0)[12], double s0, double& a0, const double (&w1)[12], double s1, double& a1, const double (&w2)[12], double s2, double& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %18 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %30 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %19 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %31 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %20 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %32 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %21 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %33 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %22 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %34 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %23 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %35 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %12 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %24 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %36 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %13 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %25 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %37 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %14 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %26 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %38 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %15 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %27 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %39 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %16 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %28 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %40 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %29 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %41 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]), "v"(w2[6]), "v"(w2[7]), "v"(w2[8]), "v"(w2[9]), "v"(w2[10]), "v"(w2[11]));
}

__device__ __forceinline__ void row_fma_2(const double (&w0)[13], double s0, double& a0, const double (&w1)[13], double s1, double& a1) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %17 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %18 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %19 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %20 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %21 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %22 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %23 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %24 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %25 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %26 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %27 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %28 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %16 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %3, %29 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s0), "v"(s1), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w0[12]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w1[12]));
}

__device__ __forceinline__ void row_fma_3(const double (&w0)[13], double s0, double& a0, const double (&w1)[13], double s1, double& a1, const double (&w2)[13], double s2, double& a2) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %3, %6 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %19 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %32 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %20 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %33 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %8 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %21 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %34 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %9 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %22 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %35 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %10 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %23 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %36 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %11 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %24 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %37 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %12 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %25 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %38 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %13 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %26 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %39 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %14 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %27 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %40 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %15 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %28 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %41 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %16 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %29 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %42 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %30 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %43 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %3, %18 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %31 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %5, %44 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1), "+&v"(a2)
      : "v"(s0), "v"(s1), "v"(s2), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w0[4]), "v"(w0[5]), "v"(w0[6]), "v"(w0[7]), "v"(w0[8]), "v"(w0[9]), "v"(w0[10]), "v"(w0[11]), "v"(w0[12]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "v"(w1[4]), "v"(w1[5]), "v"(w1[6]), "v"(w1[7]), "v"(w1[8]), "v"(w1[9]), "v"(w1[10]), "v"(w1[11]), "v"(w1[12]), "v"(w2[0]), "v"(w2[1]), "v"(w2[2]), "v"(w2[3]), "v"(w2[4]), "v"(w2[5]), "v"(w2[6]), "v"(w2[7]), "v"(w2[8]), "v"(w2[9]), "v"(w2[10]), "v"(w2[11]), "v"(w2[12]));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(double s, const double (&w0)[2], double& a0, const double (&w1)[2], double& a1) {
  static_assert(O >= 0 && O + 2 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %5 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c8 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w1[0]), "v"(w1[1]), "n"(O + 0), "n"(O + 1));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(double s, const double (&w0)[3], double& a0, const double (&w1)[3], double& a1) {
  static_assert(O >= 0 && O + 3 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %6 row_newbcast:%c9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %7 row_newbcast:%c10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "n"(O + 0), "n"(O + 1), "n"(O + 2));
}

template <int O>
__device__ __forceinline__ void row_fma_x2(double s, const double (&w0)[4], double& a0, const double (&w1)[4], double& a1) {
  static_assert(O >= 0 && O + 4 <= 16, "a 16-lane row");
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %2, %3 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %7 row_newbcast:%c11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %8 row_newbcast:%c12 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %9 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %2, %10 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a0), "+&v"(a1)
      : "v"(s), "v"(w0[0]), "v"(w0[1]), "v"(w0[2]), "v"(w0[3]), "v"(w1[0]), "v"(w1[1]), "v"(w1[2]), "v"(w1[3]), "n"(O + 0), "n"(O + 1), "n"(O + 2), "n"(O + 3));
}

// c[k] += s * src(lane k), k < N, in fp64.

__device__ __forceinline__ void row_axpy(double (&c)[4], double src, double s) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %4, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %4, %5 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %4, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3])
      : "v"(src), "v"(s));
}

__device__ __forceinline__ void row_axpy(double (&c)[6], double src, double s) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %6, %7 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %6, %7 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %6, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %6, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %6, %7 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %6, %7 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]), "+&v"(c[5])
      : "v"(src), "v"(s));
}

__device__ __forceinline__ void row_axpy(double (&c)[12], double src, double s) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %12, %13 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %12, %13 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %12, %13 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %12, %13 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %12, %13 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %12, %13 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %12, %13 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %12, %13 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %8, %12, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %9, %12, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %10, %12, %13 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %11, %12, %13 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]), "+&v"(c[5]), "+&v"(c[6]), "+&v"(c[7]), "+&v"(c[8]), "+&v"(c[9]), "+&v"(c[10]), "+&v"(c[11])
      : "v"(src), "v"(s));
}

__device__ __forceinline__ void row_axpy(double (&c)[13], double src, double s) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %13, %14 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %13, %14 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %13, %14 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %13, %14 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %13, %14 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %13, %14 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %13, %14 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %13, %14 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %8, %13, %14 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %9, %13, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %10, %13, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %11, %13, %14 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %12, %13, %14 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]), "+&v"(c[5]), "+&v"(c[6]), "+&v"(c[7]), "+&v"(c[8]), "+&v"(c[9]), "+&v"(c[10]), "+&v"(c[11]), "+&v"(c[12])
      : "v"(src), "v"(s));
}

// a[j] += g * a[j](lane KP), j < N, in fp64: the rows' step of the sweep with
// pivot row KP.

template <int KP>
__device__ __forceinline__ void row_sweep(double (&a)[4], double g) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %4 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%c5 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
      : "v"(g), "n"(KP));
}

template <int KP>
__device__ __forceinline__ void row_sweep(double (&a)[6], double g) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %4, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %5, %6 row_newbcast:%c7 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5])
      : "v"(g), "n"(KP));
}

template <int KP>
__device__ __forceinline__ void row_sweep(double (&a)[12], double g) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %4, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %5, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %6, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %7, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %8, %8, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %9, %9, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %10, %10, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %11, %11, %12 row_newbcast:%c13 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7]), "+&v"(a[8]), "+&v"(a[9]), "+&v"(a[10]), "+&v"(a[11])
      : "v"(g), "n"(KP));
}

template <int KP>
__device__ __forceinline__ void row_sweep(double (&a)[13], double g) {
  asm volatile(
      "s_nop 1\n"
      "v_fmac_f64_dpp %0, %0, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %1, %1, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %2, %2, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %3, %3, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %4, %4, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %5, %5, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %6, %6, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %7, %7, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %8, %8, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %9, %9, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %10, %10, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %11, %11, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f64_dpp %12, %12, %13 row_newbcast:%c14 row_mask:0xf bank_mask:0xf\n"
      "s_nop 1"
      : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7]), "+&v"(a[8]), "+&v"(a[9]), "+&v"(a[10]), "+&v"(a[11]), "+&v"(a[12])
      : "v"(g), "n"(KP));
}

}  // namespace tmpc
