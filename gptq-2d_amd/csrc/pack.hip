// Packed output formats of a quantized layer (no counterpart kernels in the reference, which returns only
// dequantized values; quantizer_trellis.py:11-16 states that the T*K-bit code is recoverable).
//
// INT codes.  Under the affine quantizer (quantizer_int.py:63-83) an entry's value is z = (q - zp) * s with an
// integer code q in [qmin, qmax].  Its packed code is u = q - qmin in `bits` = ceil(log2(qmax - qmin + 1))
// bits; the codes of a row of the [B, m, n] layer form one little-endian bit field: code j occupies bits
// [j*bits, (j+1)*bits) of the row, bit k of the row is bit (k % 32) of word k / 32 (for 4 bits: code j is
// nibble j % 8 of word j / 8, low nibble first).  Rows start on a word boundary (row_words words each, the
// unused tail zero).  The packer recovers q = rint(z / s + zp) and counts, per row, the entries whose
// value is not reproduced by (q - zp) * s with q in range (those are packed as code 0); the
// unpacker evaluates (q - zp) * s, the quantizer's own expression, so a counted-clean row round-trips
// exactly (as numbers; the sign of a zero is not kept).  Scale and zero point are read through element
// strides (0 broadcasts).
//
// Trellis streams.  A bitshift-trellis path (quantizer_trellis.py:82-143) of S = T / V states of L bits
// shifts K*V new bits into the low end of the state each step: s_{t+1} >> KV == s_t mod 2^(L - KV).  Its
// stream holds the top KV bits of every state in order, MSB first (stream bit k is bit 31 - k % 32 of word
// k / 32), so state t is the L-bit window starting at stream bit t*KV.  A tail-biting path is circular
// (s_0 >> KV == s_{S-1} mod 2^(L-KV)): exactly T*K bits, windows read modulo that length.  Without tail-biting
// the stream adds the low L - KV bits of the last state (T*K + L - KV bits).  The packer counts, per
// sequence, states out of range, breaks of the shift rule and copies of a state that disagree; the decoder
// writes the states and/or the values table[s, v] * scale, the quantizer's expression.
//
// Sequences are the p x q super-entries of a [B, m, n] layout read row by row (the layout of the trellis
// quantizer's super-entries); step t of sequence (b, I, J) holds entries e = t*V .. t*V + V - 1 of the block,
// entry e at (I*p + e / q, J*q + e % q).  A plain [R, T] array of sequences is the case B = 1, m = R,
// n = T, p = 1, q = T.  In the packer the per-entry state map may repeat each state over its V entries
// (copies = V) or list the states once per step (copies = 1, entry e = t).
#include "common.h"

namespace {

// Packed code of value zv under (s, zp); ok = the quantizer's output for that code equals zv (as numbers: the
// quantizer gives -0 for a code of -0, which rint returns for small negative inputs; a zero's sign is not kept).
template <typename T>
__device__ __forceinline__ uint32_t int_code(T zv, T s, T zp, T qmin, T qmax, bool& ok) {
  const T q = round_even(zv / s + zp);
  ok = q >= qmin && q <= qmax && (q - zp) * s == zv;
  return ok ? (uint32_t)(int64_t)(q - qmin) : 0u;
}

template <typename T>
struct IntLayout {
  const T* s;
  int64_t sb, sm, sn;
  const T* zp;
  int64_t zb, zm, zn;
};

// The INT kernels are bound by HBM (the values read or written once, 4 or 8 bytes an entry, and as many bytes again of
// every scale and zero point that varies along the row), so neighbouring threads read neighbouring 16 bytes of all of
// them (global memory needs only the element's own alignment for that); a scale or zero point that does not vary along
// the row is read once per row, and no thread divides a 64-bit index per value.
//
// Values j .. j + N - 1 of a row of n; past the row's end 0.
template <typename T, int N>
__device__ __forceinline__ void load_values(T (&v)[N], const T* __restrict__ row, int64_t j, int64_t n) {
  constexpr int VE = 16 / (int)sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(VE), aligned(sizeof(T))));
  if (j + N <= n) {
#pragma unroll
    for (int k = 0; k < N; k += VE) {
      const vec_t x = *reinterpret_cast<const vec_t*>(row + j + k);
#pragma unroll
      for (int e = 0; e < VE; ++e) v[k + e] = x[e];
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = j + k < n ? row[j + k] : T(0);
  }
}

// N consecutive values of a field (scale or zero point) of a row from column j on: `fixed` where the row has one.
template <typename T, int N>
__device__ __forceinline__ void load_field(T (&v)[N], const T* __restrict__ row, int64_t stride, T fixed, int64_t j,
                                           int64_t n) {
  if (stride == 1) {
    load_values<T, N>(v, row, j, n);
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = stride && j + k < n ? row[(j + k) * stride] : fixed;
  }
}

// A row's values, its words, and its scale and zero point (the fields' own values where they vary along it).
template <typename T>
struct IntRow {
  const T *s, *p;
  T s0, p0;
  int64_t sn, zn;

  __device__ __forceinline__ IntRow(const IntLayout<T>& lay, int64_t row, int64_t rows, int64_t m,
                                    int64_t n) {
    const int64_t b = rows == m ? 0 : row / m, i = rows == m ? row : row % m;
    s = lay.s + b * lay.sb + i * lay.sm;
    p = lay.zp ? lay.zp + b * lay.zb + i * lay.zm : nullptr;
    sn = lay.sn, zn = p ? lay.zn : 0;
    s0 = sn || n == 0 ? T(0) : *s;
    p0 = !p || zn || n == 0 ? T(0) : *p;
  }
  template <int N>
  __device__ __forceinline__ void load(T (&sv)[N], T (&pv)[N], int64_t j, int64_t n) const {
    load_field(sv, s, sn, s0, j, n);
    load_field(pv, p, zn, p0, j, n);
  }
};

// Sum over the TPR threads of a row (in its thread 0).
template <int TPR>
__device__ __forceinline__ int row_sum(int v, int (&sums)[4]) {
#pragma unroll
  for (int k = (TPR < 64 ? TPR : 64) / 2; k >= 1; k >>= 1) v += __shfl_xor(v, k, 64);
  if constexpr (TPR == 256) {
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sums[0] + sums[1] + sums[2] + sums[3];
  }
  return v;
}

// Codes of any width, TPR threads per row.  A thread packs four consecutive values of a chunk of 4 TPR (a whole number
// of words at any width) into one piece of 4 `bits` bits in LDS, and takes its words of the chunk from the pieces there;
// the next chunk's values are on their way meanwhile.  4096^2 fp32, 5 bits: one scale per row 23 us, a scale per entry 26,
// scale and zero point per entry 35 (41, 50 and 77 with a word a lane that gathers its codes, 27, 185 and 576 with 32
// consecutive values a thread, whose loads touch a cache line each); 16 bits 27, 29, 38; 100000 x 24 at 3 bits 7.7 (94, 133).
template <typename T, int TPR>
__global__ __launch_bounds__(256) void int_pack_kernel(const T* __restrict__ z, int64_t rows, int64_t m, int64_t n,
                                                       IntLayout<T> lay, T qmin, T qmax, int bits,
                                                       uint32_t* __restrict__ words, int64_t row_words,
                                                       int32_t* __restrict__ bad) {
  constexpr int N = 4, CH = N * TPR;
  __shared__ uint64_t pieces[2][256 / TPR][TPR];
  __shared__ int sums[4];
  const int t = threadIdx.x % TPR;
  const int64_t at = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  const bool live = at < rows;
  const int64_t row = live ? at : rows - 1;  // the others take part in the barriers only
  auto sync = [&]() {
    if constexpr (TPR > 64) {
      __syncthreads();
    } else {  // a row's threads are lanes of one wave
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  const IntRow<T> f(lay, row, rows, m, n);
  const T* zr = z + row * n;
  uint32_t* wr = words + row * row_words;
  const int cw = CH / 32 * bits, pw = N * bits;  // words of a chunk, bits of a piece
  T v[N], sv[N], pv[N];
  auto load = [&](int64_t j) {
    if (j >= n) return;
    load_values<T, N>(v, zr, j, n);
    f.load(sv, pv, j, n);
  };
  int nbad = 0, buf = 0;
  int64_t j = N * t;
  load(j);
  for (int64_t w0 = 0; w0 < row_words; w0 += cw, j += CH, buf ^= 1) {
    uint64_t u = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      if (j + k < n) {
        bool ok;
        u |= (uint64_t)int_code(v[k], sv[k], pv[k], qmin, qmax, ok) << (k * bits);
        nbad += ok ? 0 : 1;
      }
    }
    uint64_t* const mine = pieces[buf][threadIdx.x / TPR];
    mine[t] = u;
    load(j + CH);
    sync();  // one a chunk: the next chunk's pieces go to the other buffer
    for (int w = t; w < cw && w0 + w < row_words; w += TPR) {
      // the pieces that overlap the word, the first from its bit `skip` on
      int k = 32 * w / pw;
      const int skip = 32 * w - k * pw;
      uint32_t word = (uint32_t)(mine[k++] >> skip);
      for (int pos = pw - skip; pos < 32; pos += pw) word |= (uint32_t)mine[k++] << pos;
      if (live) wr[w0 + w] = word;
    }
  }
  nbad = row_sum<TPR>(nbad, sums);
  if (t == 0 && live && bad) bad[row] = nbad;
}

// 4 and 8 bits with one scale and zero point per row: a thread packs the 32 / BITS codes of a word, without LDS.
// 4096^2 at 4 bits 17.6 us, 8 bits 17.9; the kernel above 21.8 and 22.9.
template <typename T, int BITS, int TPR>
__global__ __launch_bounds__(256) void int_pack_words_kernel(const T* __restrict__ z, int64_t rows, int64_t m,
                                                             int64_t n, IntLayout<T> lay, T qmin, T qmax,
                                                             uint32_t* __restrict__ words, int64_t row_words,
                                                             int32_t* __restrict__ bad) {
  constexpr int N = 32 / BITS;
  __shared__ int sums[4];
  const int t = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (TPR == 64 && row >= rows) return;  // uniform over the wave
  const IntRow<T> f(lay, row, rows, m, n);
  const T* zr = z + row * n;
  uint32_t* wr = words + row * row_words;
  int nbad = 0;
  for (int64_t w = t; w < row_words; w += TPR) {
    const int64_t j = w * N;
    uint32_t word = 0;
    if (j < n) {
      T v[N];
      load_values<T, N>(v, zr, j, n);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (j + k < n) {
          bool ok;
          word |= int_code(v[k], f.s0, f.p0, qmin, qmax, ok) << (k * BITS);
          nbad += ok ? 0 : 1;
        }
      }
    }
    wr[w] = word;
  }
  nbad = row_sum<TPR>(nbad, sums);
  if (t == 0 && bad) bad[row] = nbad;
}

// A thread writes N consecutive values of a row (gpr groups of N per row).  BITS 4 or 8: N = 8 and one scale and zero
// point per row (fp32; 4096^2 at 4 bits 15.9 us, 20.5 with 16 bytes a thread); BITS 0: any width, N values of 16 bytes
// (5 bits: one scale per row 21 us, a scale per entry 23, with zero points 32; 8 values a thread 26, 50 and 74).
template <typename T, int BITS>
__global__ __launch_bounds__(256) void int_unpack_kernel(const uint32_t* __restrict__ words, int64_t rows, int64_t m,
                                                         int64_t n, int64_t gpr, int64_t row_words, IntLayout<T> lay,
                                                         T qmin, int bits, T* __restrict__ z) {
  constexpr int VE = 16 / (int)sizeof(T), N = BITS ? 8 : VE;
  typedef T vec_t __attribute__((ext_vector_type(VE), aligned(sizeof(T))));
  const uint32_t mask = (1u << bits) - 1u;
  const int64_t total = rows * gpr;
  const bool small = total <= 0xffffffffll;  // uniform: 32-bit index arithmetic
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int64_t row = small ? (int64_t)((uint32_t)idx / (uint32_t)gpr) : idx / gpr;
    const int64_t j = (idx - row * gpr) * N;
    const uint32_t* wr = words + row * row_words;
    // BITS 0: the N codes' bits lie in three words at most (N bits <= 64, from bit `off` of the first)
    uint32_t word[3] = {0u, 0u, 0u};
    int off = 0;
    if constexpr (BITS != 0) {
      const int64_t w = j * BITS >> 5;
      word[0] = wr[w];
      if (BITS == 8 && j + 4 < n) word[1] = wr[w + 1];
    } else {
      const int64_t start = j * bits, w = start >> 5;
      off = (int)(start & 31);
#pragma unroll
      for (int x = 0; x < 3; ++x)
        if ((x == 0 || off + N * bits > 32 * x) && w + x < row_words) word[x] = wr[w + x];
    }
    const IntRow<T> f(lay, row, rows, m, n);
    T v[N], sv[N], pv[N];
    if constexpr (BITS == 0) f.load(sv, pv, j, n);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      uint32_t u;
      if constexpr (BITS != 0) {
        u = word[k * BITS / 32] >> (k * BITS % 32);
        sv[k] = f.s0, pv[k] = f.p0;
      } else {
        const int pos = off + k * bits;
        const uint32_t lo = pos < 32 ? word[0] : (pos < 64 ? word[1] : word[2]), hi = pos < 32 ? word[1] : word[2];
        u = (uint32_t)((((uint64_t)hi << 32) | lo) >> (pos & 31));
      }
      const T q = T(u & mask) + qmin;
      v[k] = (q - pv[k]) * sv[k];
    }
    T* zr = z + row * n + j;
    if (j + N <= n) {
#pragma unroll
      for (int k = 0; k < N; k += VE) {
        vec_t x;
#pragma unroll
        for (int e = 0; e < VE; ++e) x[e] = v[k + e];
        *reinterpret_cast<vec_t*>(zr + k) = x;
      }
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k)
        if (j + k < n) zr[k] = v[k];
    }
  }
}

// ------------------------------------------------------------------------------------------------ trellis

struct SeqLayout {
  int64_t m, n, p, q;  // the [B, m, n] layout of p x q blocks
  int64_t ncol;        // n / q
  int64_t per_b;       // (m / p) * (n / q) sequences per batch matrix

  // Offset of entry e of sequence r.
  __device__ __forceinline__ int64_t at(int64_t r, int64_t e) const {
    const int64_t b = r / per_b, k = r % per_b;
    const int64_t I = k / ncol, J = k % ncol;
    return (b * m + I * p + e / q) * n + J * q + e % q;
  }
};

// MSB-first bit writer into one sequence's words.
struct StreamWriter {
  uint32_t* w;
  int64_t pos = 0;  // words written
  uint64_t acc = 0;
  int nacc = 0;

  __device__ __forceinline__ void put(uint32_t v, int k) {  // the low k <= 32 bits of v
    acc = (acc << k) | (k == 32 ? (uint64_t)v : ((uint64_t)v & ((1ull << k) - 1)));
    nacc += k;
    if (nacc >= 32) {
      w[pos++] = (uint32_t)(acc >> (nacc - 32));
      nacc -= 32;
    }
  }
  __device__ __forceinline__ void flush(int64_t row_words) {
    if (nacc > 0) w[pos++] = (uint32_t)(acc << (32 - nacc));
    nacc = 0;
    while (pos < row_words) w[pos++] = 0u;
  }
};

// One thread per sequence.
__global__ __launch_bounds__(256) void trellis_pack_kernel(const int64_t* __restrict__ st, int64_t seqs, SeqLayout lay,
                                                           int64_t steps, int copies, int L, int KV, int tail,
                                                           uint32_t* __restrict__ words, int64_t row_words,
                                                           int32_t* __restrict__ bad) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= seqs) return;
  const int64_t low_mask = ((int64_t)1 << (L - KV)) - 1;
  const int64_t limit = (int64_t)1 << L;
  StreamWriter out{words + r * row_words};
  int nbad = 0;
  int64_t first = 0, prev = 0;
  for (int64_t t = 0; t < steps; ++t) {
    int64_t s = st[lay.at(r, t * copies)];
    for (int c = 1; c < copies; ++c) nbad += st[lay.at(r, t * copies + c)] != s ? 1 : 0;
    if (s < 0 || s >= limit) {
      ++nbad;
      s = 0;
    }
    if (t == 0)
      first = s;
    else
      nbad += (s >> KV) != (prev & low_mask) ? 1 : 0;
    out.put((uint32_t)(s >> (L - KV)), KV);
    prev = s;
  }
  if (tail) {
    nbad += (first >> KV) != (prev & low_mask) ? 1 : 0;
  } else {
    for (int k = L - KV; k > 0; k -= 32 < k ? 32 : k) {
      const int c = k < 32 ? k : 32;
      out.put((uint32_t)(prev >> (k - c)), c);
    }
  }
  out.flush(row_words);
  if (bad) bad[r] = nbad;
}

__device__ __forceinline__ uint32_t stream_bit(const uint32_t* w, int64_t k) { return (w[k >> 5] >> (31 - (k & 31))) & 1u; }

// One thread per (sequence, step): the state is the L-bit window at bit t*KV (modulo the stream length for
// a tail-biting path); states [seqs, steps] and/or values in the block layout.
template <typename T>
__global__ __launch_bounds__(256) void trellis_unpack_kernel(const uint32_t* __restrict__ words, int64_t seqs,
                                                             SeqLayout lay, int64_t steps, int64_t row_words, int L,
                                                             int KV, int V, int tail, const T* __restrict__ table,
                                                             const T* __restrict__ scale, int64_t scale_stride,
                                                             T* __restrict__ values, int64_t* __restrict__ states) {
  const int64_t total = seqs * steps;
  const int64_t len = tail ? steps * KV : steps * KV + L - KV;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int64_t r = idx / steps, t = idx % steps;
    const uint32_t* w = words + r * row_words;
    const int64_t start = t * KV;
    int64_t s = 0;
    if (start + L <= len) {
      const int64_t wi = start >> 5;
      const int off = (int)(start & 31);
      uint64_t v = (uint64_t)w[wi] << 32;
      if (off + L > 32) v |= w[wi + 1];
      s = (int64_t)((v >> (64 - off - L)) & ((1ull << L) - 1));
    } else {  // a tail-biting window that wraps
      for (int i = 0; i < L; ++i) s = (s << 1) | stream_bit(w, (start + i) % len);
    }
    if (states) states[idx] = s;
    if (values) {
      const T sc = scale ? scale[r * scale_stride] : T(1);
      for (int v = 0; v < V; ++v) values[lay.at(r, t * V + v)] = table[s * V + v] * sc;
    }
  }
}

bool make_layout(SeqLayout& lay, int64_t B, int64_t m, int64_t n, int64_t p, int64_t q, int64_t& seqs) {
  if (B < 0 || m < 0 || n < 0 || p <= 0 || q <= 0 || m % p || n % q) return false;
  lay.m = m;
  lay.n = n;
  lay.p = p;
  lay.q = q;
  lay.ncol = n / q;
  lay.per_b = (m / p) * (n / q);
  seqs = B * lay.per_b;
  return true;
}

bool trellis_shape_ok(int L, int K, int V) { return K >= 1 && V >= 1 && K * V <= L && L <= 30; }

template <typename T>
bool int_layout(IntLayout<T>& lay, const T* s, const int64_t* ss, const T* zp, const int64_t* zs) {
  if (!s || !ss || (zp && !zs)) return false;
  lay.s = s;
  lay.sb = ss[0];
  lay.sm = ss[1];
  lay.sn = ss[2];
  lay.zp = zp;
  lay.zb = zp ? zs[0] : 0;
  lay.zm = zp ? zs[1] : 0;
  lay.zn = zp ? zs[2] : 0;
  return true;
}

unsigned grid_for(int64_t total) {
  const int64_t blocks = cdiv(total, 256);
  return (unsigned)(blocks < 65536 ? (blocks > 0 ? blocks : 1) : 65536);
}

template <typename T>
int pack_int(const T* z, int64_t B, int64_t m, int64_t n, const T* s, const int64_t* ss, const T* zp,
             const int64_t* zs, double qmin, double qmax, int32_t bits, uint32_t* words, int64_t row_words,
             int32_t* bad, hipStream_t stream) {
  IntLayout<T> lay;
  if (B < 0 || m < 0 || n < 0 || bits < 1 || bits > 16 || !(qmin <= qmax) || qmax - qmin >= (double)(1 << bits) ||
      row_words < cdiv(n * bits, 32))
    return GPTQ2D_EINVAL;
  const int64_t rows = B * m;
  if (rows == 0) return 0;
  if (!int_layout(lay, s, ss, zp, zs)) return GPTQ2D_EINVAL;
  // 4 and 8 bits, one scale and zero point per row, 256 columns and more (16384 x 256 at 8 bits 7.7 us against 9.5 with
  // the other kernel, 65536 x 64 at 4 bits 30 against 8): a workgroup per row from 256 words on, a wave below (a row too
  // short to feed four waves).  Otherwise threads by the row's length, fp32, one scale per row, 3 bits: 65536 x 100 in 14
  // us by 8 threads and 29 by a wave, 16384 x 256 11 and 9, 2048 x 2048 by a wave 11 and by a workgroup 9, 4096 x 1000 by
  // a wave 9.  A grid has fewer than 2^32 threads.
  const bool fixed = lay.sn == 0 && lay.zn == 0 && n >= 256, wide = rows < ((int64_t)1 << 24);
  auto words_of = [&](auto kernel, int rows_per_wg) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)cdiv(rows, rows_per_wg)), dim3(256), 0, stream, z, rows, m, n, lay, (T)qmin,
                       (T)qmax, words, row_words, bad);
  };
  auto any_width = [&](auto kernel, int rows_per_wg) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)cdiv(rows, rows_per_wg)), dim3(256), 0, stream, z, rows, m, n, lay, (T)qmin,
                       (T)qmax, bits, words, row_words, bad);
  };
  if (fixed && bits == 4)
    row_words >= 256 && wide ? words_of(int_pack_words_kernel<T, 4, 256>, 1) : words_of(int_pack_words_kernel<T, 4, 64>, 4);
  else if (fixed && bits == 8)
    row_words >= 256 && wide ? words_of(int_pack_words_kernel<T, 8, 256>, 1) : words_of(int_pack_words_kernel<T, 8, 64>, 4);
  else if (n <= 128)
    any_width(int_pack_kernel<T, 8>, 32);
  else if (n < 2048 || !wide)
    any_width(int_pack_kernel<T, 64>, 4);
  else
    any_width(int_pack_kernel<T, 256>, 1);
  return (int)hipGetLastError();
}

template <typename T>
int unpack_int(const uint32_t* words, int64_t B, int64_t m, int64_t n, int64_t row_words, const T* s,
               const int64_t* ss, const T* zp, const int64_t* zs, double qmin, int32_t bits, T* z,
               hipStream_t stream) {
  IntLayout<T> lay;
  if (B < 0 || m < 0 || n < 0 || bits < 1 || bits > 16 || row_words < cdiv(n * bits, 32)) return GPTQ2D_EINVAL;
  const int64_t total = B * m * n;
  if (total == 0) return 0;
  if (!int_layout(lay, s, ss, zp, zs)) return GPTQ2D_EINVAL;
  const bool fixed = sizeof(T) == 4 && lay.sn == 0 && lay.zn == 0;
  const int group = fixed && (bits == 4 || bits == 8) ? 8 : 16 / (int)sizeof(T);
  const int64_t gpr = cdiv(n, group);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid_for(B * m * gpr)), dim3(256), 0, stream, words, B * m, m, n, gpr, row_words, lay,
                       (T)qmin, bits, z);
  };
  if (fixed && bits == 4)
    go(int_unpack_kernel<T, 4>);
  else if (fixed && bits == 8)
    go(int_unpack_kernel<T, 8>);
  else
    go(int_unpack_kernel<T, 0>);
  return (int)hipGetLastError();
}

template <typename T>
int trellis_unpack(const uint32_t* words, int64_t B, int64_t m, int64_t n, int64_t p, int64_t q, int64_t row_words,
                   int32_t L, int32_t K, int32_t V, int32_t tail, const T* table, const T* scale, int64_t scale_stride,
                   T* values, int64_t* states, hipStream_t stream) {
  SeqLayout lay;
  int64_t seqs;
  if (!make_layout(lay, B, m, n, p, q, seqs) || !trellis_shape_ok(L, K, V) || (p * q) % V || (values && !table))
    return GPTQ2D_EINVAL;
  const int64_t steps = p * q / V, KV = K * V;
  const int64_t len = tail ? steps * KV : steps * KV + L - KV;
  if (row_words < cdiv(len, 32)) return GPTQ2D_EINVAL;
  const int64_t total = seqs * steps;
  if (total == 0) return 0;
  hipLaunchKernelGGL(trellis_unpack_kernel<T>, dim3(grid_for(total)), dim3(256), 0, stream, words, seqs, lay, steps,
                     row_words, L, K * V, V, tail ? 1 : 0, table, scale, scale_stride, values, states);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

int32_t gptq2d_int_code_bits(double qmin, double qmax) {
  if (!(qmin <= qmax) || qmin != (double)(int64_t)qmin || qmax != (double)(int64_t)qmax) return -1;
  const double range = qmax - qmin + 1;
  int bits = 1;
  while ((double)((int64_t)1 << bits) < range) ++bits;
  return bits <= 16 ? bits : -1;
}

int64_t gptq2d_trellis_stream_words(int64_t steps, int32_t L, int32_t K, int32_t V, int32_t tail_biting) {
  if (steps < 1 || !trellis_shape_ok(L, K, V)) return -1;
  const int64_t len = tail_biting ? steps * K * V : steps * K * V + L - K * V;
  return cdiv(len, 32);
}

int gptq2d_trellis_pack(const int64_t* states, int64_t B, int64_t m, int64_t n, int64_t p, int64_t q, int32_t copies,
                        int32_t L, int32_t K, int32_t V, int32_t tail_biting, uint32_t* words, int64_t row_words,
                        int32_t* bad, hipStream_t stream) {
  SeqLayout lay;
  int64_t seqs;
  if (!make_layout(lay, B, m, n, p, q, seqs) || !trellis_shape_ok(L, K, V) || copies < 1 || (p * q) % copies)
    return GPTQ2D_EINVAL;
  const int64_t steps = p * q / copies;
  if (row_words < gptq2d_trellis_stream_words(steps, L, K, V, tail_biting)) return GPTQ2D_EINVAL;
  if (seqs == 0) return 0;
  hipLaunchKernelGGL(trellis_pack_kernel, dim3((unsigned)cdiv(seqs, 256)), dim3(256), 0, stream, states, seqs, lay,
                     steps, copies, L, K * V, tail_biting ? 1 : 0, words, row_words, bad);
  return (int)hipGetLastError();
}

#define GPTQ2D_PACK_ABI(SUF, T)                                                                                      \
  int gptq2d_pack_int_##SUF(const T* z, int64_t B, int64_t m, int64_t n, const T* scale, const int64_t* sstride,     \
                            const T* zp, const int64_t* zstride, double qmin, double qmax, int32_t bits,             \
                            uint32_t* words, int64_t row_words, int32_t* bad, hipStream_t stream) {                  \
    return pack_int<T>(z, B, m, n, scale, sstride, zp, zstride, qmin, qmax, bits, words, row_words, bad, stream);   \
  }                                                                                                                   \
  int gptq2d_unpack_int_##SUF(const uint32_t* words, int64_t B, int64_t m, int64_t n, int64_t row_words,             \
                              const T* scale, const int64_t* sstride, const T* zp, const int64_t* zstride,           \
                              double qmin, int32_t bits, T* z, hipStream_t stream) {                                 \
    return unpack_int<T>(words, B, m, n, row_words, scale, sstride, zp, zstride, qmin, bits, z, stream);            \
  }                                                                                                                   \
  int gptq2d_trellis_unpack_##SUF(const uint32_t* words, int64_t B, int64_t m, int64_t n, int64_t p, int64_t q,       \
                                  int64_t row_words, int32_t L, int32_t K, int32_t V, int32_t tail_biting,           \
                                  const T* table, const T* scale, int64_t scale_stride, T* values, int64_t* states,  \
                                  hipStream_t stream) {                                                              \
    return trellis_unpack<T>(words, B, m, n, p, q, row_words, L, K, V, tail_biting, table, scale, scale_stride,      \
                             values, states, stream);                                                                \
  }

GPTQ2D_PACK_ABI(f32, float)
GPTQ2D_PACK_ABI(f64, double)

}  // extern "C"
