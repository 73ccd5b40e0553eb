// fp32 products on the bf16 matrix cores: every operand split into three bf16 pieces, x = h + m + l, and six of the
// nine piece products summed in fp32.  What is left out of x y, m l' + l m' + l l', is below 2^-22.9 of it (2^-23.03 for
// both at 1 + 2^-8 - 2^-23) and 2^-26.0 in the root mean square of normal operands, a quarter of an fp32 rounding's.
// 6 v_mfma_f32_32x32x16_bf16 replace 8 v_mfma_f32_32x32x2_f32 of twice the cycles each, which round the accumulator
// every two terms: the sums are closer to 64 bits than theirs.  Relative error in norm: factors of 1024 1.36e-7 on the
// fp32 MFMA, 1.20e-7 here, 8192 2.33e-7, 1.87e-7; the feedback of a forced sweep of 256^2 8.7e-7, 7.5e-7, 3000 x 4095
// 1.388e-6, 1.295e-6.
#pragma once

#include "common.h"

#include <type_traits>

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

// x = h + m + l in bf16 pieces, exactly, eight values at once: h rounded to nearest, m the leading eight bits of the rest,
// l the last eight.  m and l have one sign, which for two different operands is random, so that the products left out
// cancel in a sum; a sum of squares (the diagonal of P P^T) lacks 2^-26.1 of itself.  Whole-register integer steps and
// byte permutes, 6.5 instructions a value.  m rounded to nearest takes 7.5 (at most 2^-24.2 left out, 2^-27.4 rms, no bias
// in squares): factors of 1000 to 3072 1.0-1.6 % slower for 1-3 % less error, the sweep's error the same to three digits.
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&p)[3]) {
  typedef unsigned uint4v __attribute__((ext_vector_type(4)));
  uint4v w[3];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    unsigned h[2], m[2], l[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float v = x[2 * s + e];
      h[e] = __builtin_bit_cast(unsigned, v) + 0x8000u;
      const float r = v - __builtin_bit_cast(float, h[e] & 0xffff0000u);
      m[e] = __builtin_bit_cast(unsigned, r);
      l[e] = __builtin_bit_cast(unsigned, r - __builtin_bit_cast(float, m[e] & 0xffff0000u));
    }
    w[0][s] = __builtin_amdgcn_perm(h[1], h[0], 0x07060302);
    w[1][s] = __builtin_amdgcn_perm(m[1], m[0], 0x07060302);
    w[2][s] = __builtin_amdgcn_perm(l[1], l[0], 0x07060302);
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) p[q] = __builtin_bit_cast(bf16x8, w[q]);
}

// The six piece products of a 16-deep half, smallest first.
constexpr int NPROD = 6;
__device__ constexpr int prod_a[NPROD] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int prod_b[NPROD] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ bool any_nonfinite(const floatx16& acc) {
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) s = __builtin_fmaf(acc[r], 0.f, s);
  return __builtin_amdgcn_ballot_w64(!(s == 0.f)) != 0;
}

// Product of a 128 x 128 block from fp32 panels, by 256 threads: four waves of 64 x 64 (2 x 2 accumulators).  The
// k loop walks k-tiles of 16.  Thread (wave, lane) stages the eight values of row (or column) 32 wave + lane % 32 at
// k = 8 (lane / 32) .. + 7 of either panel -- the operand lane of an MFMA -- so that splitting is done once per
// workgroup and value, between the MFMAs, and LDS reads and writes are 16 bytes a lane in lane order, without bank
// conflicts.  Two k-tiles are in LDS and the values of a third in registers on their way: one barrier per k-tile.
// A wave's k-tile is 24 MFMAs of 32 clocks beside some 130 other instructions and 18 KB of LDS traffic; a block of
// rank 1024 takes 48 us alone on its CU and two together 90.  Measured: the two factorisations of 8192 10.2 ms with
// fp32 MFMAs, 7.9 here, 14336 + 4096 22.7 -> 18.6; B A^-1 at 8192 x 8192 x 6144 3.9 -> 2.3 ms.  (Splitting with the
// conversions to bf16 18.9; four k-tiles in flight in registers instead of one: slower, 55 us a block.)
struct SplitLds {
  bf16x8 a[2][4][3][64];  // [buffer][32 rows][piece][lane]
  bf16x8 b[2][4][3][64];
};

// EXACT: the same product on the fp32 MFMA, for a block whose split sum is not finite (an infinity has no pieces, and
// the sum of fp32 products must tell infinities and NaN as it always did).
template <bool EXACT>
__device__ __forceinline__ void stage_lane(bf16x8 (&dst)[3][64], int lane, const float (&x)[8]) {
  if constexpr (EXACT) {
    float* d = reinterpret_cast<float*>(&dst[0][0]);
    *reinterpret_cast<float4*>(d + 4 * lane) = make_float4(x[0], x[1], x[2], x[3]);
    *reinterpret_cast<float4*>(d + 256 + 4 * lane) = make_float4(x[4], x[5], x[6], x[7]);
  } else {
    bf16x8 p[3];
    split8(x, p);
#pragma unroll
    for (int q = 0; q < 3; ++q) dst[q][lane] = p[q];
  }
}

// acc = sum over the k-tiles [t_lo, t_hi); load_a(t, x) and load_b(t, x) give this thread's eight values of a k-tile
// (zeros outside the panels).
template <bool EXACT, class LoadA, class LoadB>
__device__ __forceinline__ void block_product(SplitLds& sm, int t_lo, int t_hi, floatx16 (&acc)[2][2],
                                              LoadA load_a, LoadB load_b) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wy = wave >> 1, wx = wave & 1;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][d][r] = 0.f;
  if (t_lo >= t_hi) return;
  float xa[8], xb[8];
  auto step = [&](int t, auto cur_c) {
    constexpr int cur = decltype(cur_c)::value;
    __syncthreads();  // buffer cur is complete; buffer 1 - cur is no longer read
    bf16x8 fa[2][3], fb[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < (EXACT ? 2 : 3); ++q) {
        fa[h][q] = sm.a[cur][2 * wy + h][q][lane];
        fb[h][q] = sm.b[cur][2 * wx + h][q][lane];
      }
    // past the last k-tile: staged again and not multiplied, so that the step is free of branches
    const int next = t + 2 < t_hi ? t + 2 : t_hi - 1;
    stage_lane<EXACT>(sm.a[1 - cur][wave], lane, xa);
    load_a(next, xa);
    stage_lane<EXACT>(sm.b[1 - cur][wave], lane, xb);
    load_b(next, xb);
    if constexpr (EXACT) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int d = 0; d < 2; ++d)
              acc[a][d] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float4v, fa[a][q])[s],
                                                               __builtin_bit_cast(float4v, fb[d][q])[s], acc[a][d], 0,
                                                               0, 0);
    } else {
#pragma unroll
      for (int x = 0; x < NPROD; ++x)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int d = 0; d < 2; ++d)
            acc[a][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][prod_a[x]], fb[d][prod_b[x]], acc[a][d], 0, 0, 0);
      // the splitting of the next k-tile between the MFMAs of this one
#pragma unroll
      for (int x = 0; x < 4 * NPROD; ++x) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
    }
  };
  load_a(t_lo, xa);
  load_b(t_lo, xb);
  stage_lane<EXACT>(sm.a[0][wave], lane, xa);
  stage_lane<EXACT>(sm.b[0][wave], lane, xb);
  load_a(t_lo + 1 < t_hi ? t_lo + 1 : t_lo, xa);
  load_b(t_lo + 1 < t_hi ? t_lo + 1 : t_lo, xb);
  for (int t = t_lo; t < t_hi; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 < t_hi) step(t + 1, std::integral_constant<int, 1>{});
  }
}

// The block product on split operands, and where a sum of the workgroup is not finite once more in fp32.
template <class LoadA, class LoadB>
__device__ __forceinline__ void split_block_product(SplitLds& sm, int t_lo, int t_hi, floatx16 (&acc)[2][2],
                                                    LoadA load_a, LoadB load_b) {
  block_product<false>(sm, t_lo, t_hi, acc, load_a, load_b);
  bool odd = false;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int d = 0; d < 2; ++d) odd |= any_nonfinite(acc[a][d]);
  if (__syncthreads_or(odd)) block_product<true>(sm, t_lo, t_hi, acc, load_a, load_b);
}

// Eight consecutive floats of a row from byte offset `off` of buffer r, `soff` more in the scalar field: two 128-bit
// loads; an offset past the extent reads zeros (the scalar field is not part of the check).
__device__ __forceinline__ void load_row8(__amdgpu_buffer_rsrc_t r, int off0, int off1, int soff, float (&x)[8]) {
  const float4v lo = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(r, off0, soff, 0));
  const float4v hi = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(r, off1, soff, 0));
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    x[s] = lo[s];
    x[4 + s] = hi[s];
  }
}

// Workgroup lin of n renumbered so that each XCD (own L2) runs a contiguous share of the blocks: the
// hardware deals workgroup w to XCD w % 8.
__device__ __forceinline__ int64_t xcd_contiguous(int64_t lin, int64_t n) {
  const int64_t base = n / 8, extra = n % 8, xcd = lin % 8;
  return xcd * base + (xcd < extra ? xcd : extra) + lin / 8;
}

}  // namespace
