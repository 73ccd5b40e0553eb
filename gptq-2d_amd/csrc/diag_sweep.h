// The 63 antidiagonals of one 32 x 32 tile by eight waves taking turns (fp32, plain entries).
//
// An entry is rounded at y = (Y + D) + F, D = sum over r' < r of L[r, r'] E[r', c], F = sum over c' < c of C[r, c'] U[c', c],
// C = (Cin + D) + E.  Wave w rounds the antidiagonals t = w (mod 8), lane 32 h + r of it the entry (r, t - r).  In the
// seven steps between its turns a wave sums the feedback of its next antidiagonal from the errors already
// published: half h = 0 of its lanes D, half h = 1 F, both as a walk over the distance d = r - r' or c - c' (the
// factors' blocks stored by distance, E by columns and C by rows, so that both halves run the same instructions),
// a distance as soon as its errors exist; the last step before the turn exchanges the halves.  At its turn it
// adds the two terms of distance 1, rounds and publishes: two LDS reads, some 18 dependent operations and one write
// are all that lies between two barriers.
//
// What bounds it is that chain: one wave issues an instruction every 8 clocks or so whether or not it waits for
// the one before (measured, one wave per SIMD: 9 clocks for a v_add_f32, dependent or not; LDS write and read back 65,
// a barrier 10-18), so a step costs its instruction count on the wave that rounds.  sweep_tile, where every wave
// runs the quantizer and its share of the feedback in every step, has about 55 of them a step.
//
// The affine quantizer takes the IEEE quotient y / s from R = 1 / s rounded, q0 = y R and one FMA correction with
// the exact remainder y - q0 s (Markstein's method), for 2^-60 <= |s| <= 2^60: the remainder is exact unless |y| <
// 2^-60, where a last bit of the tiny quotient cannot change the code, or q0 overflows, |y| >= 2^68.  No step tests
// for that: a lane whose error reaches 2^61, or is infinite or NaN, marks the tile, and a marked tile is swept again with
// the division itself (EXACT), as is one with a scale outside the range, a NaN zero point or qmin > qmax from the start.
#pragma once

#include "tile_sweep.h"

namespace {

constexpr int DW = 8;             // waves of a workgroup, antidiagonals between a wave's turns
constexpr int DTHREADS = 64 * DW;
constexpr int DSTEPS = 2 * TR - 1;
constexpr int KP = TR + 4;        // pitch of the factors by distance: 128-bit reads of 16 rows on 16 bank groups
constexpr int XP = 2 * TR + 4;    // pitch of E and C: 32 zeros, then 32 entries

// (k, r and the padding first: lanes without an entry run past the ends of the runs, within the struct)
struct DiagLds {
  float k[2 * TR * KP];         // L[r, r - d] at r KP + d, then U[c - d, c] at (32 + c) KP + d; zeros at d = 0 and outside
  float r[TR * TR];             // entry (r, c): R
  float dump[64 + 2 + 62];      // written by lanes without an entry
  int zp[DW], odd[DW], bad[DW];  // the waves' votes: a zero point is not 0; a scale needs the division; an error is huge
  union {
    struct {
      float4 a[TR * TR];        // entry (r, c): Y, Cin, scale (forced: value), zero point; from its rounding on z in x, y in z
      float x[2 * TR * XP];     // E[r, c] at c XP + 32 + r, then C[r, c] at (32 + r) XP + 32 + c; zeros before each run
    };
    float red[DW][TR][TR + 1];  // before the image: the waves' partial sums of the pulled feedback
  };
};

// Entry t (row t / 32, column t % 32) of the tile's image: the factors' diagonal blocks and R, which need no feedback ...
// Whether its scale and zero point are outside what R serves.
template <int KIND>
__device__ __forceinline__ bool diag_coefs(DiagLds& dl, int t, float s, float z, float l, float u, bool q_ok) {
  const int r = t >> 5, c = t & 31;
  // each run of 32 distances: the entries below (above) the diagonal, and zeros for d = 0 and beyond the first row
  dl.k[r * KP + (c < r ? r - c : (c == r ? 0 : c))] = c < r ? l : 0.f;
  dl.k[(TR + c) * KP + (r < c ? c - r : (r == c ? 0 : r))] = r < c ? u : 0.f;
  if constexpr (KIND == Q_AFFINE) {
    const float as = __builtin_fabsf(s);
    dl.r[t] = 1.f / s;
    return !(q_ok && as >= 0x1p-60f && as <= 0x1p60f && z == z);
  }
  return false;
}

// ... and the values (the same memory as the partial sums); the zeros before E's and C's runs.
__device__ __forceinline__ void diag_entry(DiagLds& dl, int t, float y, float c, float s, float z) {
  dl.a[t] = make_float4(y, c, s, z);
}
__device__ __forceinline__ void diag_zeros(DiagLds& dl) {
  static_assert(DTHREADS == 2 * TR * 8, "eight 128-bit stores per run");
  *reinterpret_cast<float4*>(&dl.x[(threadIdx.x >> 3) * XP + 4 * (threadIdx.x & 7)]) = make_float4(0.f, 0.f, 0.f, 0.f);
}

// A vote of the workgroup: each wave writes its own before a barrier that is there anyway, and any() reads them after it.
__device__ __forceinline__ void vote(int (&v)[DW], bool mine, int wave) {
  const unsigned long long b = __builtin_amdgcn_ballot_w64(mine);
  if ((threadIdx.x & 63) == 0) v[wave] = b != 0;
}
__device__ __forceinline__ bool any(const int (&v)[DW]) {
  int x = 0;
#pragma unroll
  for (int k = 0; k < DW; ++k) x |= v[k];
  return __builtin_amdgcn_readfirstlane(x) != 0;
}

// v with its halves exchanged: lo gets the lower half's values in both halves, hi the upper half's.
__device__ __forceinline__ void both_halves(float v, float& lo, float& hi) {
  typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
  const unsigned x = __float_as_uint(v);
  const uintx2 s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  lo = __uint_as_float(s.x);
  hi = __uint_as_float(s.y);
}

// The sweep of the tile's image (complete, a barrier after it was written); leaves z, y, E and C in it, without a
// barrier after the last entries' z and y.  Whether an error of this lane reached 2^61.  ZP: some zero point is not 0.
template <int KIND, bool YPRE, bool EXACT, bool ZP>
__device__ __forceinline__ bool sweep_diag(DiagLds& dl, float qmin, float qmax, int wave) {
  const int lane = threadIdx.x & 63, r = lane & 31;
  const bool up = lane >= 32;  // half 1: F
  asm volatile("" : "+v"(qmin), "+v"(qmax));  // in registers (else re-read from the kernel arguments every step)
  // errors that only the values' own arithmetic makes infinite or NaN (round), or that mark the tile (affine)
  constexpr bool LAX = KIND == Q_ROUND || (KIND == Q_AFFINE && !EXACT);
  const float kl = dl.k[r * KP + 1], klx = up ? kl : 0.f;  // L[r, r - 1]
  // The lane's entry (r, c) of the wave's antidiagonal, c = t - r, and what belongs to it, each a pointer that moves by
  // a constant from antidiagonal to antidiagonal.  A lane without an entry (c outside 0 .. 31) reads whatever lies
  // there (all inside dl: c in [-31, 62]) and writes to the dump.
  int c = wave - r;
  const float* kp = up ? dl.k + (TR + c) * KP : dl.k + r * KP;  // this half's coefficients by distance
  const float* ku_p = dl.k + (TR + c) * KP + 1;                 // U[c - 1, c]
  const float* pe = dl.x + c * XP + TR + r - 1;                 // E[r - 1, c]
  const float* pc = dl.x + (TR + r) * XP + TR + c - 1;          // C[r, c - 1]
  const float* vp = (up ? pc : pe) - (TR - 2);                  // this half's values: distance d at vp[31 - d]
  const float4* ap = dl.a + (r * TR + c);
  const float* rp = dl.r + (r * TR + c);
  const int kstep = up ? DW * KP : 0, vstep = up ? DW : DW * XP;
  float* const dump = dl.dump + lane;

  // of the entry at its turn: the feedback up to distance 2; C without its newest term (half 0: -0)
  float ss = 0.f, base = 0.f, sticky = 0.f;
  float4 en, k4[2], v4[2];
  float ku, rcp = 0.f;
  bool on = false;
  float *out = dump, *zo = dump;  // where the error (half 0) or C (half 1) goes; z and y
  // distances 4 q .. 4 q + 3: their operands, and their terms
  auto read = [&](int x, int q) __attribute__((always_inline)) {
    k4[x] = *reinterpret_cast<const float4*>(kp + 4 * q);
    const float* v = vp + (TR - 4) - 4 * q;
    v4[x] = make_float4(v[0], v[1], v[2], v[3]);
  };
  auto add = [&](float& acc, int x) __attribute__((always_inline)) {
    acc = __builtin_fmaf(k4[x].w, v4[x].x, acc);
    acc = __builtin_fmaf(k4[x].z, v4[x].y, acc);
    acc = __builtin_fmaf(k4[x].y, v4[x].z, acc);
    acc = __builtin_fmaf(k4[x].x, v4[x].w, acc);
  };
  auto one = [&](float& acc, int d) __attribute__((always_inline)) {
    acc = __builtin_fmaf(kp[d], vp[TR - 1 - d], acc);
  };
  auto read_entry = [&]() __attribute__((always_inline)) {
    en = *ap;
    if constexpr (KIND == Q_AFFINE) rcp = *rp;
    ku = *ku_p;
    on = (unsigned)c < (unsigned)TR;
    out = on ? const_cast<float*>(up ? pc : pe) + 1 : dump;
    zo = on ? reinterpret_cast<float*>(const_cast<float4*>(ap)) : dump;
  };
  // the last step before the turn: the halves' sums, then the barrier after which distance 1 is published
  auto last = [&](float acc) __attribute__((always_inline)) {
    float dd, ff;
    both_halves(acc, dd, ff);
    ss = dd + ff;
    base = up || !LAX ? en.y + dd : -0.f;
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };
  // The wave's turn: distance 1, the rounding, the barrier that publishes it, and after that z (and y) to the image.
  // Every instruction before the barrier counts (see above): y = Y + (D + F), and half 1's C = (Cin + D) + e and half 0's
  // e = -0 + e are one sum with operands of their own (LAX: half 0 adds 0 times the error above, which is finite).
  auto turn = [&]() __attribute__((always_inline)) {
    const float ve = *pe, vc = *pc;
    const float yv = en.x + __builtin_fmaf(ku, vc, __builtin_fmaf(kl, ve, ss));
    float z;
    if constexpr (KIND == Q_AFFINE && EXACT) {
      z = quantize_entry_div(yv, en.z, en.w, qmin, qmax);
    } else if constexpr (KIND == Q_AFFINE) {
#pragma clang fp contract(off)
      const float q0 = yv * rcp;
      const float q = __builtin_fmaf(__builtin_fmaf(-q0, en.z, yv), rcp, q0);
      if constexpr (ZP)
        z = (__builtin_amdgcn_fmed3f(round_even(q + en.w), qmin, qmax) - en.w) * en.z;
      else
        z = __builtin_amdgcn_fmed3f(round_even(q), qmin, qmax) * en.z;
    } else if constexpr (KIND == Q_FORCED) {
      z = en.z;
    } else {
      z = round_even(yv);
    }
    const float e = z - yv;
    if constexpr (LAX)
      *out = __builtin_fmaf(klx, ve, base) + e;
    else
      *out = up ? __builtin_fmaf(kl, ve, base) + e : e;
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    zo[0] = z;
    if constexpr (YPRE) zo[2] = yv;
    if constexpr (KIND == Q_AFFINE && !EXACT) {
      sticky = __builtin_fmaf(on ? e : 0.f, 0x1p67f, sticky);  // infinite or NaN from |e| = 2^61 on
      asm volatile("" : "+v"(sticky));  // here, not in line before the next turn
    }
  };

  // the wave's first antidiagonal t = wave has distances up to 7
  read_entry();
  for (int t = 0; t + 1 < wave; ++t) __syncthreads();
  if (wave > 0) {
    float acc = 0.f;
    read(0, 1);
    add(acc, 0);
    one(acc, 3);
    one(acc, 2);
    last(acc);
  } else {
    base = up || !LAX ? en.y : -0.f;
  }
  turn();
  int t = wave;
  for (; t + DW < DSTEPS; t += DW) {
    c += DW, kp += kstep, ku_p += DW * KP, pe += DW * XP, pc += DW, vp += vstep, ap += DW, rp += DW;
    // at s steps before the turn the errors of distance s + 1 and beyond are published; operands are read a step
    // before their terms are added where that is so
    float acc = 0.f;
    read(0, 7);
    __syncthreads();  // s = 7
    read(1, 6);
    add(acc, 0);
    read(0, 5);
    __syncthreads();  // 6
    add(acc, 1);
    read(1, 4);
    add(acc, 0);
    read(0, 3);
    __syncthreads();  // 5
    add(acc, 1);
    read(1, 2);
    add(acc, 0);
    __syncthreads();  // 4
    read(0, 1);
    add(acc, 1);
    read_entry();
    __syncthreads();  // 3
    add(acc, 0);
    one(acc, 3);
    __syncthreads();  // 2
    one(acc, 2);
    last(acc);        // 1
    turn();
  }
  for (++t; t < DSTEPS; ++t) __syncthreads();
  return !(__builtin_fabsf(sticky) < __builtin_inff());
}

}  // namespace
