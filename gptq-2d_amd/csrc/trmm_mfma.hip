// Row-major fp32 products with one lower triangular operand, on split operands (split_mma.h): the
// levels of the LDL's triangular inverse (ldl.hip), where every product multiplies an inverted
// diagonal block, lower triangular with its upper triangle cleared to zeros.
//
//   D = alpha A B   for `batch` strided problems, A: M x K (row stride lda), B: K x N (ldb), D: M x N
//   tri = 1: B lower (B(k, j) = 0 for k < j)  -> block column J0.. needs only k >= J0
//   tri = 2: A lower (A(i, k) = 0 for k > i)  -> block row I0.. needs only k < I0 + 128
//
// A dense GEMM library multiplies the zero triangle too; skipping the k-tiles that only meet zeros
// halves the arithmetic of a triangular product.  The boundary k-tiles (where the triangle's edge
// crosses the block) are multiplied in full: the zeros stored there make the result exact.
//
// One workgroup per 128 x 128 block of D, four waves of 64 x 64.  A's k runs along a row: a thread's eight values
// of a k-tile are two 128-bit loads; B's runs down a column: eight loads, coalesced along the columns.
// Loads past the matrices return zeros (buffer range checks), so ragged edges need no branches.
#include "common.h"
#include "lds_dma.h"
#include "linalg.h"
#include "split_mma.h"

namespace {

constexpr int TB = 128;  // block edge
constexpr int KT = 16;   // k-tile depth
constexpr int BAND = 8;  // block rows whose blocks are numbered column by column: 64 blocks in flight on an XCD share
                         // 8 panels of either operand

__global__ __launch_bounds__(256, 2) void tri_gemm_kernel(TriGemm g, int64_t nbn) {
  __shared__ __align__(16) SplitLds sm;
  const int nbm = (int)((g.M + TB - 1) / TB);
  const int64_t lin = xcd_contiguous(blockIdx.x, gridDim.x);
  const int band0 = (int)(lin / (nbn * BAND)) * BAND, rows = nbm - band0 < BAND ? nbm - band0 : BAND;
  const int64_t at = lin - (int64_t)band0 * nbn;
  int bi = band0 + (int)(at % rows);
  const int bj = (int)(at / rows);
  if (g.tri == 2) {
    // a block row's k range grows with its index: rows taken as 0, last, 1, last - 1, ... so that
    // every XCD's contiguous share mixes long and short rows
    const int q = bi;
    bi = (q & 1) ? nbm - 1 - (q >> 1) : (q >> 1);
  }
  const int I0 = bi * TB, J0 = bj * TB;
  const int M = (int)g.M, N = (int)g.N, K = (int)g.K;
  const int lda = (int)g.lda, ldb = (int)g.ldb, ldd = (int)g.ldd;
  const float* A = g.A + (int64_t)blockIdx.y * g.sa + (int64_t)blockIdx.z * g.sa2;
  const float* B = g.B + (int64_t)blockIdx.y * g.sb + (int64_t)blockIdx.z * g.sb2;
  float* D = g.D + (int64_t)blockIdx.y * g.sd + (int64_t)blockIdx.z * g.sd2;

  const int nkt = (K + KT - 1) / KT;
  int t_lo = 0, t_hi = nkt;
  if (g.tri == 1) t_lo = J0 / KT;
  if (g.tri == 2) t_hi = (I0 + TB) / KT < nkt ? (I0 + TB) / KT : nkt;

  const int tid = threadIdx.x, lane = tid & 63, li = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // buffer resources based at the block's rows of A and, per k-tile, at the k-tile's rows of B, so that every
  // byte offset stays below 128 rows of lda (A) or 16 rows of ldb (B) floats at any operand size
  const int arows = M - I0 < TB ? M - I0 : TB;
  const __amdgpu_buffer_rsrc_t ra = matrix_rsrc(A + (int64_t)I0 * lda, (int64_t)(arows - 1) * lda + K);
  const int row = 32 * wave + li;  // A's row and B's column staged by this thread
  const bool arow = row < arows, bcol = J0 + row < N;
  const int aoff = (row * lda + 8 * hh) * 4;
  int boff[8];  // rows past K lie past the resource's extent (ldb >= N)
#pragma unroll
  for (int s = 0; s < 8; ++s) boff[s] = bcol ? ((8 * hh + s) * ldb + row) * 4 : OOB;
  auto load_a = [&](int t, float (&x)[8]) {
    const int k = t * KT + 8 * hh;
    load_row8(ra, arow && k < K ? aoff : OOB, arow && k + 4 < K ? aoff + 16 : OOB, 64 * t, x);
  };
  auto load_b = [&](int t, float (&x)[8]) {
    const int k0 = t * KT, krows = K - k0 < KT ? K - k0 : KT;
    const __amdgpu_buffer_rsrc_t rb = matrix_rsrc(B + (int64_t)k0 * ldb + J0, (int64_t)(krows - 1) * ldb + (N - J0));
#pragma unroll
    for (int s = 0; s < 8; ++s)
      x[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, boff[s], 0, 0));
  };
  const int wy = wave >> 1, wx = wave & 1;
  floatx16 acc[2][2];
  split_block_product(sm, t_lo, t_hi, acc, load_a, load_b);
  const float alpha = g.alpha;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int j = J0 + 64 * wx + 32 * d + li;
      if (j >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = I0 + 64 * wy + 32 * a + 8 * (r >> 2) + 4 * hh + (r & 3);
        if (i < M) D[(int64_t)i * ldd + j] = alpha * acc[a][d][r];
      }
    }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int gptq2d_tri_gemm_f32(const TriGemm& g, hipStream_t stream) {
  if (g.M < 0 || g.N < 0 || g.K < 0 || g.batch < 0 || g.tri < 0 || g.tri > 2 || g.batch2 < 0 || g.batch2 > 65535)
    return GPTQ2D_EINVAL;
  const unsigned nz = g.batch2 > 1 ? (unsigned)g.batch2 : 1u;
  if (g.M == 0 || g.N == 0 || g.batch == 0) return 0;
  if ((g.sa2 % 4 || g.sb2 % 4) && nz > 1) return GPTQ2D_EUNSUPPORTED;
  // 128-bit staging: rows and the block offsets of every operand on 16-byte boundaries
  if (g.K % 4 || g.N % 4 || g.lda % 4 || g.ldb % 4 || g.sa % 4 || g.sb % 4 || !aligned16(g.A) || !aligned16(g.B))
    return GPTQ2D_EUNSUPPORTED;
  // 32-bit byte offsets inside a block's 128 rows of A (plus K) and a k-tile's 32 rows of B (plus N)
  const int64_t lim = (int64_t)1 << 29;
  if (TB * g.lda + g.K >= lim || 32 * g.ldb + g.N >= lim || g.M >= lim || g.N >= lim || g.K >= lim || g.K == 0 || g.ldb < g.N)
    return GPTQ2D_EUNSUPPORTED;
  const int64_t nbm = (g.M + TB - 1) / TB, nbn = (g.N + TB - 1) / TB;
  if (nbm * nbn > 0x7fffffff) return GPTQ2D_EUNSUPPORTED;
  for (int64_t b0 = 0; b0 < g.batch; b0 += 65535) {
    TriGemm h = g;
    h.A += b0 * g.sa;
    h.B += b0 * g.sb;
    h.D += b0 * g.sd;
    const unsigned nb = (unsigned)(g.batch - b0 < 65535 ? g.batch - b0 : 65535);
    hipLaunchKernelGGL(tri_gemm_kernel, dim3((unsigned)(nbm * nbn), nb, nz), dim3(256), 0, stream, h, nbn);
    const int rc = (int)hipGetLastError();
    if (rc) return rc;
  }
  return 0;
}
