// In-tile part of the fused GPTQ-2D sweeps, shared by the sweep that reads fp32 and fp64 operands
// (sweep_tiles.hip) and the one that reads split operands (sweep_split.hip): quantizers, the LDS image of a
// tile, the sweep of a tile's antidiagonals (plain entries) or rows (1 x 32 super-entries), and the fp32 MFMA
// pull of a tile's feedback.
#pragma once

#include "common.h"
#include "lds_dma.h"

#include <type_traits>
#include <utility>

namespace {

constexpr int TR = 32;       // tile edge
constexpr int PARTS = 8;     // threads cooperating on one entry of an antidiagonal
constexpr int NTHREADS = TR * PARTS;

// Q_ABSMAX: the abs-max INT quantizer of a super-entry row (int_abs_max_quantizer, quantizer_int.py:120-134),
// only with 1 x TR super-entries.
enum QKind : int32_t { Q_ROUND = 0, Q_AFFINE = 1, Q_FORCED = 2, Q_ABSMAX = 3 };

template <typename T>
struct QSpec {
  int32_t kind;
  const T* scale;  // affine: full [*, m, n] scale; forced: the codes' values
  const T* zp;     // affine: full [*, m, n] zero point
  BatchMap smap, zmap;
  T qmin, qmax;
  T* ypre;          // optional [B, m, n]: Y of every entry just before it is rounded
  T* sout;          // abs-max, optional [B, m, n]: the scale each entry's row was rounded with
  int32_t dtype16;  // abs-max: the scale's 16-bit type (1 bf16, 2 fp16)
};

// f(integral_constant<int, I>) for I = 0, 1, ..., in order: a loop whose index is a compile-time constant in
// every iteration.
template <typename F, int... I>
__device__ __forceinline__ void static_for(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// The affine quantizer (clamp(round(y / s + z), qmin, qmax) - z) s by IEEE division, the dequantized value
// rounded on its own (as the reference's plug-in writes it), so that a caller's error z - y is exactly that
// difference: no contraction of the product into the caller's subtraction.
template <typename T>
__device__ __forceinline__ T quantize_entry_div(T yv, T sv, T zv, T qmin, T qmax) {
#pragma clang fp contract(off)
  const T code = clamp_val(round_even(yv / sv + zv), qmin, qmax);
  return (code - zv) * sv;
}

// The abs-max quantizer clamp(round(y / s), qmin, qmax) s of quantizer_int.py:134 (the product is exact for
// a 16-bit scale and a small code, and rounded on its own in any case).
template <typename T>
__device__ __forceinline__ T quantize_absmax_entry(T yv, T sv, T qmin, T qmax) {
#pragma clang fp contract(off)
  return clamp_val(round_even(yv / sv), qmin, qmax) * sv;
}

// ------------------------------------------------------------------------------------------------ 1 x TR super-entries
//
// With super-entries of one row and TR columns (gptq_2d_super_entry with super_entry_shape (1, TR), e.g. the
// three-factor layer's 1 x 32 abs-max groups) a tile holds the TR super-entries (i0 + r, J) of one coarse
// column, ordered by row; the tiles' coarse stages and the feedback between tiles (pulls, flushes) are
// those of plain entries, and U's TR x TR diagonal blocks -- identity by the super-entry convention -- are
// never read.  Inside a tile the sweep is TR steps, one per row: the row's entries are rounded jointly
// from y = Y + down (the in-tile feedback through L[I,I]), then their errors are pushed to the rows below.
// Thread (g, c) = (tid / 32, tid % 32) owns column c of rows 4g .. 4g + 3; a row is the 32 lanes of one
// half-wave, so the abs-max of a super-entry row is a half-wave reduction.

// Maximum over the 32 lanes of each half-wave (all of them receive it).  fp32: by exchanges of lanes in the vector
// registers (quad permutes, mirrors of 8 and 16 lanes, the swap of 16-lane rows), 10 instructions; five shuffles
// through LDS are 65 clocks each on the chain of every row.
template <typename T>
__device__ __forceinline__ T halfwave_max(T v) {
  if constexpr (sizeof(T) == 4) {
    auto with = [&](auto ctrl_c) {
      const T o = __builtin_bit_cast(
          T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(ctrl_c)::value, 0xf, 0xf, true));
      v = o > v ? o : v;
    };
    with(std::integral_constant<int, 0xB1>{});   // lane ^ 1
    with(std::integral_constant<int, 0x4E>{});   // lane ^ 2
    with(std::integral_constant<int, 0x141>{});  // the other quad of 8 lanes
    with(std::integral_constant<int, 0x140>{});  // the other half of 16
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto rows = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned r0 = rows[0], r1 = rows[1];
    const T a = __builtin_bit_cast(T, r0), b = __builtin_bit_cast(T, r1);
    return b > a ? b : a;
  } else {
#pragma unroll
    for (int k = 16; k >= 1; k >>= 1) {
      const T o = __shfl_xor(v, k, 32);
      v = o > v ? o : v;
    }
    return v;
  }
}

// The rows' quantizer inputs (affine: scale and zero point; forced: the values), read from global memory
// at the start of the kernel.
template <typename T, int KIND>
struct RowInputs {
  T s[4], z[4];

  __device__ __forceinline__ void load(const QSpec<T>& qs, int64_t b, int64_t m, int64_t n, int64_t i0, int64_t j0) {
    const int cc = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int rows_in = m - i0 < TR ? (int)(m - i0) : TR;
    const int64_t corner = i0 * n + j0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * g + i;
      const bool in = r < rows_in;
      const int64_t off = corner + (int64_t)r * n + cc;
      s[i] = z[i] = T(0);
      if constexpr (KIND == Q_AFFINE) {
        s[i] = in ? qs.scale[qs.smap.offset(b) + off] : T(1);
        z[i] = in ? qs.zp[qs.zmap.offset(b) + off] : T(0);
      } else if constexpr (KIND == Q_FORCED) {
        s[i] = in ? qs.scale[qs.smap.offset(b) + off] : T(0);
      }
    }
  }
};

// The TR row steps of one tile, then its Y, C and E to global memory (`image`, uniform over the workgroup: Y and C to ys
// and cs instead, beside the published errors in es, and a barrier).  ys / cs: the tile's Y and C with
// the pulled feedback (row pitches ysp, csp); lp[r lpp + k] = L[i0 + r, i0 + k] for k < r, zero
// elsewhere; es: TR x esp floats for the published errors.  Expects the image complete (a barrier after
// it was written).
template <typename T, int KIND, bool YPRE>
__device__ __forceinline__ void sweep_rows(T* ys, int ysp, T* cs, int csp, const T* lp, int lpp, T* es,
                                           int esp, const RowInputs<T, KIND>& in, T* __restrict__ y,
                                           T* __restrict__ c, T* __restrict__ e, const QSpec<T>& qs, int64_t m,
                                           int64_t n, int64_t i0, int64_t j0, int64_t mat, bool image = false) {
  const int cc = threadIdx.x & 31, g = threadIdx.x >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rows_in = m - i0 < TR ? (int)(m - i0) : TR;  // the super-entries span the tile's columns
  T Y[4], C[4], D[4], E[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    Y[i] = ys[(4 * g + i) * ysp + cc];
    C[i] = cs[(4 * g + i) * csp + cc];
    D[i] = E[i] = T(0);
  }
  const T qmin = qs.qmin, qmax = qs.qmax, half = (qs.qmax - qs.qmin) / T(2);
  auto step = [&](auto r_c) __attribute__((always_inline)) {
    constexpr int r = decltype(r_c)::value, slot = r & 3;
    // the wave that holds the row; the others wait for its errors (fp64, 512^2 affine: 697 us, 703 with the branch)
    if (sizeof(T) == 8 || wave == (r >> 3)) {
      const bool own = g == (r >> 2) && r < rows_in;
      const T yv = Y[slot] + D[slot];
      T z, sc = T(1);
      if constexpr (KIND == Q_ABSMAX) {
        // scale from the row's current abs max (a NaN entry counts as 0, as in the plug-in's comparison
        // loop), rounded to the 16-bit type through fp32, 0 -> 1; the reduction runs on every lane
        const T a = own ? __builtin_fmax(__builtin_fabs(yv), T(0)) : T(0);
        const T amax = halfwave_max(a);
        sc = round_scale16(amax / half, qs.dtype16);
        sc = sc == T(0) ? T(1) : sc;
        z = quantize_absmax_entry(yv, sc, qmin, qmax);
      } else if constexpr (KIND == Q_AFFINE) {
        // the dequantized value rounded on its own, before the error z - y (no contraction into it)
        z = quantize_entry_div(yv, in.s[slot], in.z[slot], qmin, qmax);
      } else if constexpr (KIND == Q_FORCED) {
        z = in.s[slot];
      } else {
        z = round_even(yv);
      }
      const T ev = z - yv;
      const T cf = (C[slot] + D[slot]) + ev;
      if (own) {
        Y[slot] = z;
        E[slot] = ev;
        C[slot] = cf;
        es[r * esp + cc] = ev;
        if constexpr (YPRE) qs.ypre[mat + (i0 + r) * n + j0 + cc] = yv;
        if constexpr (KIND == Q_ABSMAX) {
          if (qs.sout) qs.sout[mat + (i0 + r) * n + j0 + cc] = sc;
        }
      }
    }
    if constexpr (r + 1 < TR) {
      __syncthreads();  // the row's errors before the rows below read them
      const T er = es[r * esp + cc];
#pragma unroll
      for (int i = 0; i < 4; ++i) D[i] += lp[(4 * g + i) * lpp + r] * er;
    }
  };
  static_for(step, std::make_integer_sequence<int, TR>{});
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * g + i;
    if (image) {
      ys[r * ysp + cc] = Y[i];
      cs[r * csp + cc] = C[i];
    } else if (r < rows_in) {
      const int64_t off = mat + (i0 + r) * n + j0 + cc;
      y[off] = Y[i];
      c[off] = C[i];
      e[off] = E[i];
    }
  }
  if (image) __syncthreads();
}

// ------------------------------------------------------------------------------------------------ fp32: pull + sweep

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Quantizer of the fused sweeps, applied to one value.
template <int KIND>
__device__ __forceinline__ float quantize_entry(float yv, float sv, float zv, float qmin, float qmax) {
  if constexpr (KIND == Q_AFFINE) {
    const float code = clamp_val(round_even(yv / sv + zv), qmin, qmax);
    return (code - zv) * sv;
  } else if constexpr (KIND == Q_FORCED) {
    return sv;
  } else {
    return round_even(yv);
  }
}

// One wave's share of a band product on MFMA: acc += sum over the k-chunks ch in [c_lo, c_hi) with
// ch = c_lo + part (mod nparts) of A[i0 + 0..31, 8 ch + 0..7] B[8 ch + 0..7, j0 + 0..31], A and B
// row-major (lda, ldb), read straight from global memory into the MFMA operand layout: lane l
// supplies A(l % 32, 8 ch + 4 (l / 32) + s) and B(8 ch + 4 (l / 32) + s, l % 32) to MFMA s = 0..3 of
// the chunk.  Loads of G chunks are issued before their MFMAs.
template <bool VEC>
__device__ __forceinline__ void pull_chunks(floatx16& acc, const float* __restrict__ A, int64_t lda, int64_t a_rows,
                                            int64_t a_cols, const float* __restrict__ Bm, int64_t ldb,
                                            int64_t b_rows, int64_t b_cols, int64_t i0, int64_t j0, int64_t c_lo,
                                            int64_t c_hi, int part, int nparts, int li, int hh) {
  // this lane's row of A and column of B as pointers (64-bit arithmetic once); k offsets in 32 bits
  const int64_t ia = i0 + li, jb = j0 + li;
  const bool arow = ia < a_rows, bcol = jb < b_cols;
  const float* ap = A + (arow ? ia : 0) * lda;
  const float* bp = Bm + (bcol ? jb : 0);
  const int clo = (int)c_lo, chi = (int)c_hi, acols = (int)a_cols, brows = (int)b_rows;
  constexpr int G = 4;
  for (int base = clo + part; base < chi; base += nparts * G) {
    float av[G][4], bv[G][4];
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int ch = base + nparts * q;
      const int k0 = 8 * ch + 4 * hh;
      const bool ok = ch < chi;
      if (VEC) {
        const float4 f = (ok && arow && k0 < acols) ? *reinterpret_cast<const float4*>(ap + k0)
                                                    : make_float4(0.f, 0.f, 0.f, 0.f);
        av[q][0] = f.x, av[q][1] = f.y, av[q][2] = f.z, av[q][3] = f.w;
      } else {
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) av[q][s2] = (ok && arow && k0 + s2 < acols) ? ap[k0 + s2] : 0.f;
      }
      const float* bk = bp + (int64_t)k0 * ldb;
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2) bv[q][s2] = (ok && bcol && k0 + s2 < brows) ? bk[s2 * ldb] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if (base + nparts * q >= chi) break;
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q][s2], bv[q][s2], acc, 0, 0, 0);
    }
  }
}

// pull_chunks for the right product R = C U with U = P (x) Q given by its factors (nq % 16 == 0): B value (k, j)
// is Q[k % nq, j % nq] times P[k / nq, j / nq] -- one fp32 multiplication, the entry of the explicit product bit
// for bit.  A lane's column is fixed, and an 8-row chunk lies in one block of P, so each chunk takes one P entry
// per lane; the chunk's 16-row unit is split on the scalar unit.  Q is read through a buffer resource based at
// the chunk's first row (the lane's column in the vector offset, the row step in the scalar one, a lane past
// the matrix masked by an offset beyond the extent): no branches and no 64-bit address arithmetic per load.
// Every row a chunk reads lies below n (the right product's k-tiles are t < J <= nt - 1).
template <bool VEC>
__device__ __forceinline__ void pull_chunks_kron(floatx16& acc, const float* __restrict__ A, int64_t lda,
                                                 int64_t a_rows, int64_t a_cols, const KronU& kr, int64_t b_rows,
                                                 int64_t b_cols, int64_t i0, int64_t j0, int64_t c_lo, int64_t c_hi,
                                                 int part, int nparts, int li, int hh) {
  const int64_t ia = i0 + li, jb = j0 + li;
  const bool arow = ia < a_rows, bcol = jb < b_cols;
  const float* ap = A + (arow ? ia : 0) * lda;
  int pj = 0, qj = 0;  // the lane's column: block of P, column of Q
  if (bcol) kron_index(kr, (int)jb, pj, qj);
  // the tile's columns in one block of P (all but the tiles that straddle a block edge): the chunks' P entries
  // are read through the scalar cache
  int pu0, pu1, qu;
  kron_index(kr, (int)j0, pu0, qu);
  kron_index(kr, (int)(j0 + TR - 1 < b_cols - 1 ? j0 + TR - 1 : b_cols - 1), pu1, qu);
  const int nq = kr.nq;
  const int qoff = bcol ? (qj + 4 * hh * nq) * 4 : OOB;  // bytes: the lane's column of Q, its k slot
  const float* pp = kr.p + pj;
  const int clo = (int)c_lo, chi = (int)c_hi, acols = (int)a_cols;
  const int upart = __builtin_amdgcn_readfirstlane(part), unparts = __builtin_amdgcn_readfirstlane(nparts);
  constexpr int G = 4;
  auto run = [&](auto uniform_c) {
    constexpr bool UNI = decltype(uniform_c)::value;
    for (int base = clo + upart; base < chi; base += unparts * G) {
      float av[G][4], bv[G][4], pv[G];
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int ch = base + unparts * q;
        const int k0 = 8 * ch + 4 * hh;
        const bool ok = ch < chi;
        if (VEC) {
          const float4 f = (ok && arow && k0 < acols) ? *reinterpret_cast<const float4*>(ap + k0)
                                                      : make_float4(0.f, 0.f, 0.f, 0.f);
          av[q][0] = f.x, av[q][1] = f.y, av[q][2] = f.z, av[q][3] = f.w;
        } else {
#pragma unroll
          for (int s2 = 0; s2 < 4; ++s2) av[q][s2] = (ok && arow && k0 + s2 < acols) ? ap[k0 + s2] : 0.f;
        }
        int ub, ur;  // the chunk's rows: 16-row unit ch / 2 = block ub of P, rows 16 ur + 8 (ch % 2) + .. of Q
        kron_split(kr, (unsigned)(ok ? ch >> 1 : 0), ub, ur);
        if constexpr (UNI)
          pv[q] = kron_p_uniform(kr, ub * kr.np + pu0);
        else
          pv[q] = pp[ub * kr.np];
        const int row0 = 16 * ur + 8 * (ch & 1);
        const int64_t ext = ok ? (int64_t)(nq - row0) * nq : 0;  // elements from the chunk's first row
        const __amdgpu_buffer_rsrc_t qr =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kr.q + (int64_t)row0 * nq), (short)0,
                                              (int)(ext < OOB / 4 ? ext * 4 : OOB), 0x00020000);
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
          bv[q][s2] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(qr, qoff, s2 * nq * 4, 0));
      }
      // the products after all loads: a product inside a mask's branch would make each load wait for its data
      // before the next one issues
#pragma unroll
      for (int q = 0; q < G; ++q)
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) bv[q][s2] *= pv[q];
#pragma unroll
      for (int q = 0; q < G; ++q) {
        if (base + unparts * q >= chi) break;
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q][s2], bv[q][s2], acc, 0, 0, 0);
      }
    }
  };
  if (pu0 == pu1)
    run(std::true_type{});
  else
    run(std::false_type{});
}

// LDS row pitch of the tile's Y and E images: 40 = 8 (mod 32) keeps the column walks of the E reads
// (a row step of 39 = -7 mod 32 banks between neighbouring columns) and the final row-wise stores free
// of bank conflicts beyond 2-way.
constexpr int SP = 40;

// LDS image of one tile for the fp32 in-tile sweep.  L[I,I] and U[J,J] are stored with zero padding so
// that the sweep reads them at any offset in [-TR, 2 TR) without masks:
// Lp[r][TR + k] = L[i0+r, i0+k] for 0 <= k < r (zero elsewhere), Up[TR + k][c] = U[j0+k, j0+c] for
// k < c (zero elsewhere).  Ys: the tile's Y with the pulled feedback (on entry), the result (at the end).
// Cs[r][TR + c] and Es[TR + r][c]: the C and E images, padded by TR zero columns (C) and rows (E) on
// each side: C holds C + pulled D on entry and each entry's final C from its rounding on; E holds
// zeros on entry and each entry's error from its rounding on.  The sweep reads both at offsets that
// leave the tile (times zero coefficients), so the padding must hold finite values.
// Row pitches of the padded L, U and C images: with 103, 39 and 98 floats every per-step read of the
// sweep (L[r, t - c], U[t - r, c], C[r, t - r] over a half-wave's 4 rows x 8 parts) falls on 32 distinct
// banks; the natural pitches (97, 33, 97) put 4 rows on one bank in each of them.
constexpr int LPW = 3 * TR + 7;
constexpr int UPW = TR + 7;
constexpr int CPW = 3 * TR + 2;
constexpr int EROWS = 3 * TR;

// (T = double: the same image in fp64; every pitch gives the 32 lanes of a half-wave 32 distinct positions
// mod 32, so their 64-bit reads cover the 64 banks once)
template <typename T>
struct TileLdsT {
  T Ys[TR][SP];  // first: the sweep's base pointers below reach up to 23 rows / columns before Lp and Up
  T Lp[TR][LPW];
  T Up[3 * TR][UPW];
  T Cs[TR][CPW];
  T Es[EROWS][SP];
};
using TileLds = TileLdsT<float>;

// Affine / round / forced quantizer of the in-tile sweep, given the precomputed correctly rounded
// reciprocal rv = 1/sv and whether sv lies in [2^-60, 2^60] (affine only).  y / s is formed as
// q0 = y rv, then one FMA correction with the exact remainder y - q0 s (Markstein's method): the
// IEEE quotient whenever also 2^-60 <= |y| < 2^61 (then no product or remainder over- or
// underflows: |q0| lies in [2^-121, 2^121] and the remainder is a multiple of 2^-107).  `exact` says
// whether that holds -- the biased exponent of y in [67, 187], one bit-field test (zero, denormal,
// infinite and NaN y fail it) -- and otherwise quantize_entry_div (the division itself) gives the
// value.  This keeps the division's ten dependent operations off the per-antidiagonal critical path.
//
__device__ __forceinline__ float fma_of(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_of(double a, double b, double c) { return __builtin_fma(a, b, c); }

// fp64: the same with 2^-500 <= |s| <= 2^500 and 2^-500 <= |y| < 2^501 (biased exponent of y in [523, 1523]):
// |q0| lies in [2^-1001, 2^1001] and the remainder is a multiple of 2^-605, all normal.
template <int KIND, typename T>
__device__ __forceinline__ T quantize_entry_rcp(T yv, T sv, T zv, T rv, bool s_ok, T qmin, T qmax, bool& exact) {
  // the dequantized value is rounded on its own (as the reference's plug-in writes it), so that the
  // caller's error z - y is exactly that difference: no contraction into the caller's subtraction
#pragma clang fp contract(off)
  if constexpr (KIND == Q_AFFINE) {
    const T q0 = yv * rv;
    const T rem = fma_of(-q0, sv, yv);
    const T q = fma_of(rem, rv, q0);
    // s_ok also holds only when the zero point is not NaN and qmin <= qmax: then q is the IEEE
    // quotient, round(q + z) is not NaN, and the median of (x, qmin, qmax) is the clamp, in one
    // operation on the per-step critical path
    if constexpr (sizeof(T) == 4) {
      const unsigned ex = (__float_as_uint(yv) >> 23) & 0xffu;
      exact = s_ok && ex - 67u <= 120u;
      const T code = __builtin_amdgcn_fmed3f(round_even(q + zv), qmin, qmax);
      return (code - zv) * sv;
    } else {
      const unsigned ex = (unsigned)(__builtin_bit_cast(unsigned long long, yv) >> 52) & 0x7ffu;
      exact = s_ok && ex - 523u <= 1000u;
      const T code = clamp_val(round_even(q + zv), qmin, qmax);
      return (code - zv) * sv;
    }
  } else if constexpr (KIND == Q_FORCED) {
    exact = true;
    return sv;
  } else {
    exact = true;
    return round_even(yv);
  }
}


// Thread ownership of the in-tile sweep.  Thread (r, part) = (tid / 8, tid % 8) owns the four entries
// (r, c) of its row with (c + r) % 8 == part; slot j holds the one whose antidiagonal t_e = r + c has
// (t_e / 8) % 4 == j.  The entry rounded at step t is then slot (t / 8) % 4 of part t % 8 in every row: a
// compile-time register in the unrolled loop over t.
__device__ __forceinline__ void slot_columns(int r, int part, int (&cs)[4]) {
  const int qlo = (r - part + 7) >> 3;  // smallest q with 8 q + part >= r
#pragma unroll
  for (int j = 0; j < 4; ++j) cs[j] = 8 * (qlo + ((j - qlo) & 3)) + part - r;  // in [0, TR)
}

// Quantizer inputs of the sweep's entries in its own layout (slot order), read from global memory at
// the start of the kernel so that their latency overlaps the pull.
template <int KIND, typename T = float>
struct SweepInputs {
  T s[4], z[4];

  __device__ __forceinline__ void load(const QSpec<T>& qs, int64_t b, int64_t m, int64_t n, int64_t i0,
                                       int64_t j0) {
    const int tid = threadIdx.x, r = tid >> 3, part = tid & 7;
    int cs[4];
    slot_columns(r, part, cs);
    const int rows_in = m - i0 < TR ? (int)(m - i0) : TR, cols_in = n - j0 < TR ? (int)(n - j0) : TR;
    const int64_t corner = i0 * n + j0;
    const T* st = KIND != Q_ROUND ? qs.scale + qs.smap.offset(b) + corner : nullptr;
    const T* zt = KIND == Q_AFFINE ? qs.zp + qs.zmap.offset(b) + corner : nullptr;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = r < rows_in && cs[j] < cols_in;
      const int off = r * (int)n + cs[j];
      s[j] = z[j] = T(0);
      if constexpr (KIND == Q_AFFINE) {
        s[j] = in ? st[off] : T(1);
        z[j] = in ? zt[off] : T(0);
      } else if constexpr (KIND == Q_FORCED) {
        s[j] = in ? st[off] : T(0);
      }
    }
  }
};

// The tile's 63 antidiagonals, in push form.  A step: the rounding lanes quantize (their entries'
// feedback is complete) and write the error into the E image and the final C into the C image; one
// workgroup barrier; then every lane reads the step's error in each of its columns (E[t - c, c]) and
// the final C of its row (C[r, t - r]) and adds the step's feedback to its entries' sums -- down:
// L[r, t-c] E[t-c, c], right: C[r, t-r] U[t-r, c].  An entry is rounded at y = (Y + down) + right,
// and its C becomes (C + down) + error.  The zero-padded diagonal blocks make the terms vanish for
// entries already rounded, for sources below the entry (not yet written in the images: their zeros or
// values times zero) and for sources outside the tile.  Expects the tile image complete in LDS (a barrier
// after it was written) and leaves the swept tile in it (Ys, Cs, Es; a barrier after the last write).
//
// The step is bound by its chain (the quantizer's ~13 dependent operations, the LDS write, barrier
// and read-back, ~150 clocks measured for the exchange alone) and by the LDS reads of four waves
// (13 per lane); the image pitches keep every read free of bank conflicts.
template <int KIND, bool YPRE, typename T>
__device__ __forceinline__ void sweep_tile(TileLdsT<T>& tl, const SweepInputs<KIND, T>& in, const QSpec<T>& qs,
                                           int64_t m, int64_t n, int64_t i0, int64_t j0, int64_t mat) {
  const int tid = threadIdx.x;
  const int r = tid >> 3, part = tid & 7;
  const int rows_in = m - i0 < TR ? (int)(m - i0) : TR;  // tile rows / columns inside the matrix
  const int cols_in = n - j0 < TR ? (int)(n - j0) : TR;
  const bool row_in = r < rows_in;
  int cs[4];
  slot_columns(r, part, cs);
  // per entry: Y and C on entry, the in-tile down and right feedback sums D and F (kept apart from
  // Y, so that their rounding errors scale with the feedback, not with Y), the error E, the
  // quantizer inputs S, Z and the reciprocal R of S, and the step at which the entry is rounded (-1
  // for entries outside the matrix)
  T Y[4], C[4], D[4], F[4], E[4], S[4], Z[4], R[4];
  int tr[4];
  bool s_ok[4];
  const bool qmin_le_qmax = qs.qmin <= qs.qmax;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    tr[j] = row_in && cs[j] < cols_in ? r + cs[j] : -1;
    Y[j] = tl.Ys[r][cs[j]];
    C[j] = tl.Cs[r][TR + cs[j]];
    D[j] = F[j] = E[j] = T(0);
    S[j] = in.s[j];
    Z[j] = in.z[j];
    R[j] = T(0);
    s_ok[j] = false;
    if constexpr (KIND == Q_AFFINE) {
      R[j] = T(1) / S[j];
      T as;
      if constexpr (sizeof(T) == 4)
        as = __builtin_fabsf(S[j]);
      else
        as = __builtin_fabs(S[j]);
      // the range in which the quotient from the reciprocal is the IEEE one (quantize_entry_rcp)
      constexpr T s_lo = sizeof(T) == 4 ? T(0x1p-60) : T(0x1p-500), s_hi = sizeof(T) == 4 ? T(0x1p60) : T(0x1p500);
      s_ok[j] = as >= s_lo && as <= s_hi && Z[j] == Z[j] && qmin_le_qmax;
    }
  }
  T* ypre_row = YPRE ? qs.ypre + mat + (i0 + r) * n + j0 : nullptr;
  // clamp bounds pinned in registers (an empty asm makes them opaque): otherwise the compiler
  // re-reads them from the kernel arguments on every step
  T qmin = qs.qmin, qmax = qs.qmax;
  asm volatile("" : "+v"(qmin), "+v"(qmax));
  // what a thread reads and writes at step t, as pointers plus t or t times the row pitch (immediate
  // offsets): the C of its row's rounded entry C[r, t - r] (which the rounding lane writes), that
  // lane's E[r, t - r], and per slot the source E[t - c, c] and the coefficients L[r, t - c], U[t - r, c]
  T* const cp = &tl.Cs[r][TR] - r;
  T* const ewp = &tl.Es[TR + r][0] - r;
  const T* ep[4];
  const T* lp[4];
  const T* up[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ep[j] = &tl.Es[TR][0] + (cs[j] - cs[j] * SP);
    lp[j] = &tl.Lp[r][TR] - cs[j];
    up[j] = &tl.Up[TR][0] + (cs[j] - r * UPW);
  }
  constexpr int STEPS = 2 * TR - 1;
  // L and U coefficients of step t in LV[t & 1], UV[t & 1], read a step ahead (they do not depend on
  // the sweep), so that only the published errors and C are read between the barrier and the
  // feedback update, and no register copies are needed in the unrolled loop
  T LV[2][4], UV[2][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    LV[0][j] = lp[j][0];
    UV[0][j] = up[j][0];
  }
  // one step at compile-time index t (the loop is unrolled by a fold over the steps: the register slot,
  // the parity buffers and the LDS immediates are compile-time in every step)
  auto step = [&](auto t_c) __attribute__((always_inline)) {
    constexpr int t = decltype(t_c)::value;
    constexpr int cur = t & 1, ka = (t >> 3) & 3;
    // every lane evaluates its step's register; only the rounding lanes keep and publish it
    const bool rnd = tr[ka] == t;
    const T yv = (Y[ka] + D[ka]) + F[ka];
    {
      bool exact;
      T z = quantize_entry_rcp<KIND>(yv, S[ka], Z[ka], R[ka], s_ok[ka], qmin, qmax, exact);
      T ev = z - yv;
      const T cd = C[ka] + D[ka];
      T cf = cd + ev;
      if (rnd) {
        // published at once; a lane whose quotient needs the division writes again (same address:
        // the later write stands), behind a branch taken only when some lane of the wave needs it
        ewp[t] = ev;
        cp[t] = cf;
        if constexpr (KIND == Q_AFFINE) {
          if (__builtin_amdgcn_ballot_w64(!exact)) {
            asm volatile("");  // keeps the division behind the branch (no speculation into a select)
            if (!exact) {
              z = quantize_entry_div(yv, S[ka], Z[ka], qmin, qmax);
              ev = z - yv;
              cf = cd + ev;
              ewp[t] = ev;
              cp[t] = cf;
            }
          }
        }
        Y[ka] = z;
        E[ka] = ev;
        C[ka] = cf;
      }
    }
    if constexpr (t == STEPS - 1) {
      if constexpr (YPRE) {
        if (rnd) ypre_row[t - r] = yv;
      }
      return;  // nothing left to receive feedback
    }
    __syncthreads();  // every wave's writes of this step before any wave's reads
    const T cr = cp[t];
    T ev[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) ev[j] = ep[j][t * SP];
    if constexpr (t + 1 < STEPS - 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        LV[cur ^ 1][j] = lp[j][t + 1];
        UV[cur ^ 1][j] = up[j][(t + 1) * UPW];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      D[j] += LV[cur][j] * ev[j];
      F[j] += cr * UV[cur][j];
    }
    // the pre-quantization value out after the step's feedback is issued
    if constexpr (YPRE) {
      if (rnd) ypre_row[t - r] = yv;
    }
    // no second barrier: every image entry is written once (at its entry's step), so the next step's
    // writes never touch what this step reads
  };
  static_for(step, std::make_integer_sequence<int, STEPS>{});

#pragma unroll
  for (int j = 0; j < 4; ++j) tl.Ys[r][cs[j]] = Y[j];
  __syncthreads();
}

// The swept tile's Y, C and E from its LDS image to global memory.
template <typename T>
__device__ __forceinline__ void store_tile(const TileLdsT<T>& tl, T* __restrict__ y, T* __restrict__ c,
                                           T* __restrict__ e, int64_t m, int64_t n, int64_t i0, int64_t j0,
                                           int64_t mat) {
  const int rows_in = m - i0 < TR ? (int)(m - i0) : TR, cols_in = n - j0 < TR ? (int)(n - j0) : TR;
  T* yt = y + mat + i0 * n + j0;
  T* ct = c + mat + i0 * n + j0;
  T* et = e + mat + i0 * n + j0;
  for (int t = threadIdx.x; t < TR * TR; t += NTHREADS) {
    const int rr = t / TR, cc = t % TR;
    if (rr < rows_in && cc < cols_in) {
      const int off = rr * (int)n + cc;
      yt[off] = tl.Ys[rr][cc];
      ct[off] = tl.Cs[rr][TR + cc];
      et[off] = tl.Es[TR + rr][cc];
    }
  }
}

// The pulled feedback at (r, cc) from the four waves' partial sums (wave w's in red[w / 2][w % 2]):
// waves [0, wd) summed the down product D, the others the right product R (in wave order).
__device__ __forceinline__ void pulled_sums(const float (*red)[2][TR][TR + 1], int wd, int r, int cc, float& dd,
                                            float& rr) {
  const float s0 = red[0][0][r][cc], s1 = red[0][1][r][cc], s2 = red[1][0][r][cc], s3 = red[1][1][r][cc];
  dd = (wd > 0 ? s0 : 0.f) + (wd > 1 ? s1 : 0.f) + (wd > 2 ? s2 : 0.f) + (wd > 3 ? s3 : 0.f);
  rr = (wd > 0 ? 0.f : s0) + (wd > 1 ? 0.f : s1) + (wd > 2 ? 0.f : s2) + (wd > 3 ? 0.f : s3);
}

// Own tile data of the fp32 kernels, read before the tile's feedback is complete (it does not
// depend on it): entry q of this thread is (t / TR, t % TR) with t = threadIdx.x + NTHREADS q.
// ROWS: the tile image of the row-super-entry sweep (1 x TR super-entries): no U block (identity by the
// super-entry convention, never read), no padding and no E image.
template <bool ROWS, typename T = float>
struct TileRegs {
  static constexpr int NQ = TR * TR / NTHREADS;
  T y[NQ], c[NQ], l[NQ], u[NQ];

  // KR (fp32): U given by its Kronecker factors (ub unused), each entry of the diagonal tile (J, J) read as its
  // P entry times its Q entry.
  template <bool KR = false>
  __device__ __forceinline__ void load(const T* __restrict__ yg, const T* __restrict__ cg,
                                       const T* __restrict__ lb, const T* __restrict__ ub, int64_t m,
                                       int64_t n, int64_t i0, int64_t j0, int64_t mat, const KronU& kr = KronU{}) {
    static_assert(!KR || sizeof(T) == 4, "Kronecker U: fp32");
    // the tile's corner in every operand (64-bit arithmetic once, uniform), then 32-bit offsets in
    // the tile (32 rows of at most 2^26 elements)
    const int rows_in = m - i0 < TR ? (int)(m - i0) : TR, cols_in = n - j0 < TR ? (int)(n - j0) : TR;
    const int ni = (int)n, mi = (int)m;
    const int64_t corner = i0 * n + j0;
    const T* yt = yg + mat + corner;
    const T* ct = cg + mat + corner;
    const T* lt = lb + i0 * m + i0;  // L[i0 + r, i0 + cc] at r m + cc
    const T* ut = KR ? nullptr : ub + j0 * n + j0;  // U[j0 + r, j0 + cc] at r n + cc
    T pu[NQ];  // KR: the P entries of the u[q]
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int t = threadIdx.x + NTHREADS * q;
      const int r = t / TR, cc = t % TR;
      const bool in = r < rows_in && cc < cols_in;
      const int off = r * ni + cc;
      y[q] = in ? yt[off] : T(0);
      c[q] = in ? ct[off] : T(0);
      // L[i0+r, i0+cc] strictly below the diagonal; U[j0+r, j0+cc] strictly above it
      l[q] = (cc < r && r < rows_in) ? lt[r * mi + cc] : T(0);
      if constexpr (KR) {
        const bool on = !ROWS && r < cc && cc < cols_in;
        int ib = 0, iq = 0, jb = 0, jq = 0;
        if (on) {
          kron_index(kr, (int)j0 + r, ib, iq);
          kron_index(kr, (int)j0 + cc, jb, jq);
        }
        u[q] = on ? kr.q[(int64_t)iq * kr.nq + jq] : T(0);
        pu[q] = on ? kr.p[(int64_t)ib * kr.np + jb] : T(0);
      } else {
        u[q] = (!ROWS && r < cc && cc < cols_in) ? ut[off] : T(0);
      }
    }
    if constexpr (KR) {  // the products after all loads (masked entries: 0 times 0)
#pragma unroll
      for (int q = 0; q < NQ; ++q) u[q] *= pu[q];
    }
  }

  // LDS image of the tile with the pulled feedback D (down) and R (right) added: C + D, Y + (D + R),
  // the zero padding of the diagonal blocks and of the C image, and the zeroed E image.  fp32: red holds
  // the waves' partial sums when `pulled` (pulled_sums: the first wd waves' are D's).  fp64: red64, when
  // given, holds D (red64[0]) and R (red64[1]) whole.
  __device__ __forceinline__ void store(TileLdsT<T>& tl, const float (*red)[2][TR][TR + 1], bool pulled, int wd,
                                        const double (*red64)[TR][TR + 1] = nullptr) const {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int t = threadIdx.x + NTHREADS * q;
      const int r = t / TR, cc = t % TR;
      T dd = T(0), rr = T(0);
      if constexpr (sizeof(T) == 4) {
        if (pulled) pulled_sums(red, wd, r, cc, dd, rr);
      } else {
        if (red64) dd = red64[0][r][cc], rr = red64[1][r][cc];
      }
      tl.Ys[r][cc] = y[q] + (dd + rr);
      tl.Cs[r][TR + cc] = c[q] + dd;
      tl.Lp[r][TR + cc] = l[q];
      if constexpr (!ROWS) tl.Up[TR + r][cc] = u[q];
    }
    if constexpr (ROWS) return;
    // zero padding without divisions: 8 threads per row of Lp and of Cs (71 and 66 padding columns), 4 per
    // padding row of Up (39 columns each); a strided column walk per thread
    {
      static_assert(NTHREADS == 8 * TR && LPW - TR <= 72 && CPW - TR <= 72 && UPW <= 40, "padding walk shape");
      const int r = threadIdx.x >> 3, sub = threadIdx.x & 7;
#pragma unroll
      for (int i = 0; i < 9; ++i) {
        const int k = sub + 8 * i;
        if (k < LPW - TR) tl.Lp[r][k < TR ? k : k + TR] = T(0);
        if (k < CPW - TR) tl.Cs[r][k < TR ? k : k + TR] = T(0);
      }
      const int row = threadIdx.x >> 2, sub4 = threadIdx.x & 3;
      T* up_row = tl.Up[row < TR ? row : row + TR];
#pragma unroll
      for (int i = 0; i < 10; ++i) {
        const int col = sub4 + 4 * i;
        if (col < UPW) up_row[col] = T(0);
      }
    }
    // the E image: all zeros (read times zero coefficients before the entries' errors are written)
    {
      T* es = &tl.Es[0][0];
      constexpr int EN = EROWS * SP;
#pragma unroll
      for (int i = 0; i < (EN + NTHREADS - 1) / NTHREADS; ++i) {
        const int k = threadIdx.x + NTHREADS * i;
        if (k < EN) es[k] = T(0);
      }
    }
  }
};

// A wave's partial product into red[product][half] (layout of the 32 x 32 MFMA accumulator).
__device__ __forceinline__ void stash_partial(float (*red)[2][TR][TR + 1], const floatx16& acc, int product,
                                              int half) {
  const int lane = threadIdx.x & 63, li = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int r = 0; r < 16; ++r) red[product][half][8 * (r >> 2) + 4 * hh + (r & 3)][li] = acc[r];
}

}  // namespace
