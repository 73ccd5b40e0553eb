// Fused GPTQ-2D sweep for per-entry quantizers (round, affine, teacher-forced codes).
//
// The matrix is cut into TR x TR tiles.  GPTQ-2D gives the same rounding for any order of the
// entries that respects the partial order (i' <= i, j' <= j), so the sweep runs over coarse
// stages T = I + J of tiles: the tiles of one coarse stage do not depend on each other, and each
// is swept by one workgroup entirely in LDS -- its 2*TR-1 antidiagonals one after another, every
// entry of an antidiagonal at once, the in-tile error feedback through the diagonal blocks
// L[I,I] and U[J,J], the quantizer applied in place.  Feedback between tiles: after each outer
// block of `outer_tiles` coarse stages, the block flush of flush.hip with P = Q = TR (on MFMA) into
// all later stages; inside an outer block, fp32 tiles pull the feedback of the block's earlier tiles
// on MFMA (tile_stage_kernel), fp64 stages are flushed into the rest of the block after each coarse
// stage (sweep_tile64_kernel then sweeps).  Both run the same push-form in-tile sweep (sweep_tile).
// The host loop below issues every launch of the sweep from C++ in one call, so a whole layer is one
// C-ABI call and one capturable stream of kernels.
//
// In exact arithmetic the result equals the reference's blocked sweep (gptq_2d.py:1295-1375) and
// Algorithm 1 on vec(X) (GPTQ-2D paper, Theorem 1); in floating point the sums are accumulated in
// a different order.  The in-tile value of entry (r, c) when it is rounded is
//   y = (Y[r,c] + sum_{r'<r} L[r,r'] E[r',c]) + sum_{c'<c} C[r,c'] U[c',c]
// where C[r,c'] is already complete (all rows above in the tile were rounded earlier).
#include "profile.h"
#include "tile_sweep.h"

#include <mutex>

template <typename T>
int gptq2d_flush(T* y, T* c, const T* e, const T* l, const T* u, int64_t m, int64_t n, int64_t P, int64_t Q,
                 int64_t s0, int64_t s1, int64_t s_end, const BatchMap& lmap, const BatchMap& umap, int64_t B,
                 hipStream_t stream);
template <typename T>
int gptq2d_fill(T* x, T v, int64_t count, hipStream_t stream);
int gptq2d_flush_kron(float* y, float* c, const float* e, const float* l, const KronU& kr, int64_t m, int64_t n,
                      int64_t s0, int64_t s1, int64_t s_end, hipStream_t stream);

namespace {

constexpr int64_t BAND64 = 4;  // fp64 fused sweep: tile stages per band flush inside an outer block

// One launch per coarse stage of the row-super-entry sweep on the generic (fp64) path: each workgroup
// loads its tile's Y, C and L[I,I] and sweeps it (the feedback of earlier tiles was flushed in).
template <typename T, int KIND, bool YPRE>
__global__ __launch_bounds__(NTHREADS) void sweep_rows_kernel(T* __restrict__ y, T* __restrict__ c,
                                                              T* __restrict__ e, const T* __restrict__ l, int64_t m,
                                                              int64_t n, int64_t stage, int64_t tile_lo,
                                                              BatchMap lmap, QSpec<T> qs, int64_t nx, int64_t ny) {
  __shared__ T Ys[TR][TR + 1];
  __shared__ T Cs[TR][TR + 1];
  __shared__ T Ls[TR][TR + 1];
  __shared__ T Es[TR][TR + 1];
  const GridIds id = grid_ids(nx, ny);
  const int64_t b = id.b;
  const int64_t I = tile_lo + id.x, J = stage - I;
  const int64_t i0 = I * TR, j0 = J * TR;
  const int64_t mat = b * m * n;
  const T* lb = l + lmap.offset(b);
  const int rows_in = m - i0 < TR ? (int)(m - i0) : TR;
  RowInputs<T, KIND> in;
  in.load(qs, b, m, n, i0, j0);
  for (int t = threadIdx.x; t < TR * TR; t += NTHREADS) {
    const int r = t / TR, cc = t % TR;
    const bool rin = r < rows_in;
    const int64_t off = mat + (i0 + r) * n + j0 + cc;
    Ys[r][cc] = rin ? y[off] : T(0);
    Cs[r][cc] = rin ? c[off] : T(0);
    Ls[r][cc] = (cc < r && rin) ? lb[(i0 + r) * m + i0 + cc] : T(0);  // strictly below the diagonal
  }
  __syncthreads();
  sweep_rows<T, KIND, YPRE>(&Ys[0][0], TR + 1, &Cs[0][0], TR + 1, &Ls[0][0], TR + 1, &Es[0][0], TR + 1, in, y, c, e, qs,
                            m, n, i0, j0, mat);
}


// One launch per coarse stage T of the fused fp32 sweep, inside the outer block of tile stages
// [S0, S1).  The feedback a tile (I, J) needs from the tiles of its outer block swept before it
// (no flush has delivered it yet) is D = sum L[I,t] E[t,J] over t in [max(0, S0-J), I) and
// R = sum C[I,t] U[t,J] over t in [max(0, S0-I), J).  It is pulled on MFMA in two parts:
//  * prep workgroups (blockIdx.x >= n_sweep) take the tiles of stage T+1 and add the part from
//    the k-tiles before the last one (t < I-1, resp. t < J-1: stages up to T-1, all final) to
//    their Y and C in global memory -- no tile of stage T touches those;
//  * sweep workgroups take the tiles of stage T, pull the last k-tile (the tiles (I-1, J) and
//    (I, J-1) of stage T-1) and sweep the tile's 63 antidiagonals in LDS (sweep_tile).
// So only one k-tile of each product is on the stage-to-stage critical path; the rest runs beside
// the previous stage's sweeps.  Waves 0-1 take the down product, waves 2-3 the right one, each
// every second 8-deep k-chunk; the two halves meet in LDS.
// KR: U = P (x) Q given by its factors (kr; u unused): the right products pull Q times P entries.
template <bool VEC, int KIND, bool YPRE, bool ROWS, bool KR = false>
__global__ __launch_bounds__(NTHREADS, 2) void tile_stage_kernel(float* __restrict__ y, float* __restrict__ c,
                                                                 float* __restrict__ e, const float* __restrict__ l,
                                                                 const float* __restrict__ u, int64_t m, int64_t n,
                                                                 int64_t stage, int64_t S0, int64_t tile_lo,
                                                                 int64_t n_sweep, int64_t prep_lo, BatchMap lmap,
                                                                 BatchMap umap, QSpec<float> qs, int64_t nx,
                                                                 int64_t ny, KronU kr) {
  __shared__ float red[2][2][TR][TR + 1];
  __shared__ TileLds tl;

  const GridIds id = grid_ids(nx, ny);
  const int64_t b = id.b;
  const bool sweep = id.x < n_sweep;
  const int64_t st = sweep ? stage : stage + 1;
  const int64_t I = sweep ? tile_lo + id.x : prep_lo + (id.x - n_sweep), J = st - I;
  const int64_t i0 = I * TR, j0 = J * TR;
  const int64_t mat = b * m * n;
  const float* lb = l + lmap.offset(b);
  const float* ub = KR ? nullptr : u + umap.offset(b);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, hh = lane >> 5;

  // k-chunk ranges (8 columns each) of this workgroup's part of the two products
  const int64_t dlo = S0 - J > 0 ? S0 - J : 0, rlo = S0 - I > 0 ? S0 - I : 0;
  int64_t d0, d1, r0, r1;
  if (sweep) {
    d0 = I - 1 >= dlo ? 4 * (I - 1) : 0, d1 = I - 1 >= dlo ? 4 * I : 0;
    r0 = J - 1 >= rlo ? 4 * (J - 1) : 0, r1 = J - 1 >= rlo ? 4 * J : 0;
  } else {
    d0 = 4 * dlo, d1 = I - 1 > dlo ? 4 * (I - 1) : d0;
    r0 = 4 * rlo, r1 = J - 1 > rlo ? 4 * (J - 1) : r0;
  }
  const bool pulled = d0 < d1 || r0 < r1;
  if (!sweep && !pulled) return;

  // own tile data first: it does not depend on the pull, so its loads overlap the pull's
  TileRegs<ROWS> own;
  SweepInputs<ROWS ? Q_ROUND : KIND> qin;
  RowInputs<float, ROWS ? KIND : Q_ROUND> rin;
  if (sweep) {
    own.template load<KR>(y, c, lb, ub, m, n, i0, j0, mat, kr);
    if constexpr (ROWS)
      rin.load(qs, b, m, n, i0, j0);
    else
      qin.load(qs, b, m, n, i0, j0);
  }

  // the four waves dealt to the two products in proportion to their chunk counts (a tile near its
  // outer block's edge has nearly all its history in one of them), each product's chunks
  // interleaved over its waves
  const int64_t nd = d1 - d0, nr = r1 - r0;
  int wd = nd == 0 ? 0 : (nr == 0 ? 4 : (int)((4 * nd + (nd + nr) / 2) / (nd + nr)));
  if (nd > 0 && nr > 0) wd = wd < 1 ? 1 : (wd > 3 ? 3 : wd);
  if (pulled) {
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (wave < wd)
      pull_chunks<VEC>(acc, lb, m, m, m, e + mat, n, m, n, i0, j0, d0, d1, wave, wd, li, hh);
    else if constexpr (KR)
      pull_chunks_kron<VEC>(acc, c + mat, n, m, n, kr, n, n, i0, j0, r0, r1, wave - wd, 4 - wd, li, hh);
    else
      pull_chunks<VEC>(acc, c + mat, n, m, n, ub, n, n, n, i0, j0, r0, r1, wave - wd, 4 - wd, li, hh);
    stash_partial(red, acc, wave >> 1, wave & 1);
  }
  __syncthreads();

  if (!sweep) {  // prep: Y += D + R, C += D in place
    const int rows_in = m - i0 < TR ? (int)(m - i0) : TR, cols_in = n - j0 < TR ? (int)(n - j0) : TR;
    float* yt = y + mat + i0 * n + j0;
    float* ct = c + mat + i0 * n + j0;
#pragma unroll
    for (int q = 0; q < TR * TR / NTHREADS; ++q) {
      const int t = tid + NTHREADS * q;
      const int r = t / TR, cc = t % TR;
      if (r < rows_in && cc < cols_in) {
        const int off = r * (int)n + cc;
        float dd, rr;
        pulled_sums(red, wd, r, cc, dd, rr);
        yt[off] = yt[off] + (dd + rr);
        ct[off] = ct[off] + dd;
      }
    }
    return;
  }

  // ---- the tile image in LDS, then the in-tile sweep
  own.store(tl, red, pulled, wd);
  __syncthreads();
  if constexpr (ROWS)
    sweep_rows<float, KIND, YPRE>(&tl.Ys[0][0], SP, &tl.Cs[0][TR], CPW, &tl.Lp[0][TR], LPW, &tl.Es[TR][0], SP, rin, y, c,
                                  e, qs, m, n, i0, j0, mat);
  else {
    sweep_tile<KIND, YPRE>(tl, qin, qs, m, n, i0, j0, mat);
    store_tile(tl, y, c, e, m, n, i0, j0, mat);
  }
}

// fp64 feedback of tile (I, J) from the k-tiles t in [d0, d1) (down: D = sum L[I,t] E[t,J]) and [r0, r1) (right:
// R = sum C[I,t] U[t,J]), on MFMA (v_mfma_f64_16x16x4_f64), into red[0] (D) and red[1] (R).  Wave w owns the
// 16 x 16 quadrant (w / 2, w % 2) of both products; lane l (q = l % 16, h = l / 16) supplies A(q, 8 h + s) and
// B(8 h + s, q) to MFMA s = 0..7 of a k-tile (which k a slot carries is free as long as A and B agree), and
// accumulator element r of lane l holds (h + 4 r, q) of the quadrant.  The k-tiles of both products form one
// list of jobs (D's first), loaded PJ jobs at a time, one chunk ahead of the chunk whose MFMAs run.
__device__ __forceinline__ void pull64(double (*red)[TR][TR + 1], const double* __restrict__ lb,
                                       const double* __restrict__ eb, const double* __restrict__ cb,
                                       const double* __restrict__ ub, int64_t m, int64_t n, int64_t i0, int64_t j0,
                                       int d0, int d1, int r0, int r1) {
  typedef double doublex4 __attribute__((ext_vector_type(4)));
  constexpr int PJ = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = lane & 15, h = lane >> 4;
  const int64_t i = i0 + 16 * (wave >> 1) + q, j = j0 + 16 * (wave & 1) + q;
  const bool iin = i < m, jin = j < n;
  // this lane's rows of L and C, columns of E and U (64-bit arithmetic once)
  const double* la = lb + (iin ? i : 0) * m;
  const double* ca = cb + (iin ? i : 0) * n;
  const double* ej = eb + (jin ? j : 0);
  const double* uj = ub + (jin ? j : 0);
  const int nd = d1 - d0, nj = nd + (r1 - r0);
  double a[2][PJ][8], bv[2][PJ][8];
  // job x's operands: k = 32 t + 8 h + s, inside k < m (L's columns, E's rows) or k < n (C's columns, U's rows)
  auto load = [&](int x, double (&av)[8], double (&bb)[8]) {
    const bool dn = x < nd;
    const int64_t k0 = (int64_t)(dn ? d0 + x : r0 + (x - nd)) * TR + 8 * h;
    const int64_t kmax = dn ? m : n;
    const double* ap = dn ? la : ca;
    const double* bp = dn ? ej : uj;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bool ok = x < nj && k0 + s < kmax;
      av[s] = ok && iin ? ap[k0 + s] : 0.;
      bb[s] = ok && jin ? bp[(k0 + s) * n] : 0.;
    }
  };
  doublex4 accd = {0., 0., 0., 0.}, accr = {0., 0., 0., 0.};
  auto chunk = [&](int c0, auto cur_c) {
    constexpr int cur = decltype(cur_c)::value;
    if (c0 + PJ < nj) {
#pragma unroll
      for (int x = 0; x < PJ; ++x) load(c0 + PJ + x, a[1 - cur][x], bv[1 - cur][x]);
    }
#pragma unroll
    for (int x = 0; x < PJ; ++x) {
      const int job = c0 + x;  // uniform
      if (job >= nj) break;
      if (job < nd) {
#pragma unroll
        for (int s = 0; s < 8; ++s) accd = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][x][s], bv[cur][x][s], accd, 0, 0, 0);
      } else {
#pragma unroll
        for (int s = 0; s < 8; ++s) accr = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][x][s], bv[cur][x][s], accr, 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int x = 0; x < PJ; ++x) load(x, a[0][x], bv[0][x]);
  for (int c0 = 0; c0 < nj; c0 += 2 * PJ) {
    chunk(c0, std::integral_constant<int, 0>{});
    if (c0 + PJ < nj) chunk(c0 + PJ, std::integral_constant<int, 1>{});
  }
  const int rq = 16 * (wave >> 1) + h, cq = 16 * (wave & 1) + q;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    red[0][rq + 4 * r][cq] = accd[r];
    red[1][rq + 4 * r][cq] = accr[r];
  }
}

// One launch per coarse stage of the fused fp64 sweep: each workgroup takes one tile of the stage.  Its
// feedback from the outer blocks before its own and from its own block's stages before `band_lo` has been
// flushed into its Y and C (outer flushes, then band flushes of `band` stages inside an outer block); the rest,
// from the tiles of stages [band_lo, stage), it pulls itself on MFMA (pull64).  Then it builds the fp32 sweep's
// LDS image in fp64 and runs the same push-form sweep of its 63 antidiagonals (sweep_tile).  The image and the
// pulled sums take 139 KB of LDS: one workgroup per CU, at most one per tile of the stage.
template <int KIND, bool YPRE>
__global__ __launch_bounds__(NTHREADS) void sweep_tile64_kernel(double* __restrict__ y, double* __restrict__ c,
                                                                double* __restrict__ e, const double* __restrict__ l,
                                                                const double* __restrict__ u, int64_t m, int64_t n,
                                                                int64_t stage, int64_t tile_lo, int64_t band_lo,
                                                                BatchMap lmap, BatchMap umap, QSpec<double> qs,
                                                                int64_t nx, int64_t ny) {
  __shared__ TileLdsT<double> tl;
  __shared__ double red[2][TR][TR + 1];
  const GridIds id = grid_ids(nx, ny);
  const int64_t b = id.b;
  const int64_t I = tile_lo + id.x, J = stage - I;
  const int64_t i0 = I * TR, j0 = J * TR;
  const int64_t mat = b * m * n;
  const double* lb = l + lmap.offset(b);
  const double* ub = u + umap.offset(b);
  // k-tiles of the pull: the tiles (t, J) and (I, t) of stages [band_lo, stage)
  const int64_t dlo = band_lo - J > 0 ? band_lo - J : 0, rlo = band_lo - I > 0 ? band_lo - I : 0;
  const int d0 = (int)dlo, d1 = (int)(I > dlo ? I : dlo), r0 = (int)rlo, r1 = (int)(J > rlo ? J : rlo);
  const bool pulled = d0 < d1 || r0 < r1;
  SweepInputs<KIND, double> in;
  in.load(qs, b, m, n, i0, j0);
  TileRegs<false, double> regs;
  regs.load(y, c, lb, ub, m, n, i0, j0, mat);  // own data first: its loads overlap the pull's
  if (pulled) {
    pull64(red, lb, e + mat, c + mat, ub, m, n, i0, j0, d0, d1, r0, r1);
    __syncthreads();
  }
  regs.store(tl, nullptr, false, 0, pulled ? red : nullptr);
  __syncthreads();
  sweep_tile<KIND, YPRE>(tl, in, qs, m, n, i0, j0, mat);
  store_tile(tl, y, c, e, m, n, i0, j0, mat);
}

template <int KIND>
void launch_tile64_k(dim3 grid, hipStream_t stream, double* y, double* c, double* e, const double* l, const double* u,
                     int64_t m, int64_t n, int64_t st, int64_t lo, int64_t band_lo, const BatchMap& lmap,
                     const BatchMap& umap, const QSpec<double>& qs, int64_t nx, int64_t ny) {
  if (qs.ypre)
    hipLaunchKernelGGL((sweep_tile64_kernel<KIND, true>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, u, m, n, st, lo,
                       band_lo, lmap, umap, qs, nx, ny);
  else
    hipLaunchKernelGGL((sweep_tile64_kernel<KIND, false>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, u, m, n, st,
                       lo, band_lo, lmap, umap, qs, nx, ny);
}

template <bool VEC, int KIND, bool ROWS, bool KR>
void launch_tile_stage_k(dim3 grid, hipStream_t stream, float* y, float* c, float* e, const float* l, const float* u,
                         int64_t m, int64_t n, int64_t st, int64_t S0, int64_t lo, int64_t n_sweep, int64_t prep_lo,
                         const BatchMap& lmap, const BatchMap& umap, const QSpec<float>& qs, int64_t nx, int64_t ny,
                         const KronU& kr) {
  if (qs.ypre)
    hipLaunchKernelGGL((tile_stage_kernel<VEC, KIND, true, ROWS, KR>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, u,
                       m, n, st, S0, lo, n_sweep, prep_lo, lmap, umap, qs, nx, ny, kr);
  else
    hipLaunchKernelGGL((tile_stage_kernel<VEC, KIND, false, ROWS, KR>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, u,
                       m, n, st, S0, lo, n_sweep, prep_lo, lmap, umap, qs, nx, ny, kr);
}

template <bool VEC, bool ROWS, bool KR = false>
void launch_tile_stage(int32_t kind, dim3 grid, hipStream_t stream, float* y, float* c, float* e, const float* l,
                       const float* u, int64_t m, int64_t n, int64_t st, int64_t S0, int64_t lo, int64_t n_sweep,
                       int64_t prep_lo, const BatchMap& lmap, const BatchMap& umap, const QSpec<float>& qs, int64_t nx,
                       int64_t ny, const KronU& kr = KronU{}) {
  if (kind == Q_AFFINE)
    launch_tile_stage_k<VEC, Q_AFFINE, ROWS, KR>(grid, stream, y, c, e, l, u, m, n, st, S0, lo, n_sweep, prep_lo, lmap,
                                                 umap, qs, nx, ny, kr);
  else if (kind == Q_FORCED)
    launch_tile_stage_k<VEC, Q_FORCED, ROWS, KR>(grid, stream, y, c, e, l, u, m, n, st, S0, lo, n_sweep, prep_lo, lmap,
                                                 umap, qs, nx, ny, kr);
  else if (ROWS && kind == Q_ABSMAX)
    launch_tile_stage_k<VEC, Q_ABSMAX, true, KR>(grid, stream, y, c, e, l, u, m, n, st, S0, lo, n_sweep, prep_lo, lmap,
                                                 umap, qs, nx, ny, kr);
  else
    launch_tile_stage_k<VEC, Q_ROUND, ROWS, KR>(grid, stream, y, c, e, l, u, m, n, st, S0, lo, n_sweep, prep_lo, lmap,
                                                umap, qs, nx, ny, kr);
}

template <typename T, int KIND>
void launch_rows_stage(dim3 grid, hipStream_t stream, T* y, T* c, T* e, const T* l, int64_t m, int64_t n, int64_t st,
                       int64_t lo, const BatchMap& lmap, const QSpec<T>& qs, int64_t nx, int64_t ny) {
  if (qs.ypre)
    hipLaunchKernelGGL((sweep_rows_kernel<T, KIND, true>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, m, n, st, lo,
                       lmap, qs, nx, ny);
  else
    hipLaunchKernelGGL((sweep_rows_kernel<T, KIND, false>), grid, dim3(NTHREADS), 0, stream, y, c, e, l, m, n, st, lo,
                       lmap, qs, nx, ny);
}

bool aligned16(const void* p) { return p == nullptr || ((uintptr_t)p & 15) == 0; }

bool strides_mult4(const BatchMap& bm) {
  for (int d = 0; d < bm.nd; ++d)
    if (bm.stride[d] % 4) return false;
  return true;
}

// rows: super-entries of 1 x TR (the row sweep); dtype16: the abs-max scale's 16-bit type; kron: U given by its
// Kronecker factors (u unused; fp32, one matrix, rows staged 128 bits at a time).
template <typename T>
int sweep_fused(T* y, T* c, T* e, const T* l, const T* u, int64_t m, int64_t n, int32_t bnd, const int64_t* bshape,
                const int64_t* lstride, const int64_t* ustride, int32_t qkind, const T* qa, const int64_t* qa_stride,
                const T* qb, const int64_t* qb_stride, double qmin, double qmax, T* ypre, int64_t outer_tiles,
                int64_t stage_begin, int64_t stage_end, hipStream_t stream, bool rows = false, int32_t dtype16 = 0,
                T* scale_out = nullptr, const KronU* kron = nullptr) {
  BatchMap lmap, umap;
  if (!make_batch_map(lmap, bnd, bshape, lstride) || !make_batch_map(umap, bnd, bshape, ustride)) return GPTQ2D_EINVAL;
  if (m <= 0 || n <= 0 || outer_tiles < 1) return GPTQ2D_EINVAL;
  // U from its factors: the outer flush that reads them is the tuned tile flush alone (m, n < 2^20), so sizes it
  // rejects are refused here, before any stage has written y
  if (kron && (sizeof(T) != 4 || bnd != 0 || n != (int64_t)kron->np * kron->nq || m >= ((int64_t)1 << 20) ||
               n >= ((int64_t)1 << 20)))
    return GPTQ2D_EUNSUPPORTED;
  // the tile kernels index inside a tile with 32-bit offsets (32 rows of a row length < 2^26)
  if (m >= ((int64_t)1 << 26) || n >= ((int64_t)1 << 26)) return GPTQ2D_EUNSUPPORTED;
  if (qkind != Q_ROUND && qkind != Q_AFFINE && qkind != Q_FORCED && !(rows && qkind == Q_ABSMAX)) return GPTQ2D_EINVAL;
  if ((qkind == Q_AFFINE && (!qa || !qb)) || (qkind == Q_FORCED && !qa)) return GPTQ2D_EINVAL;
  if (qkind == Q_ABSMAX && (!(qmin < qmax) || (dtype16 != 1 && dtype16 != 2))) return GPTQ2D_EINVAL;
  if (rows && n % TR) return GPTQ2D_EINVAL;  // the super-entries tile the rows
  QSpec<T> qs;
  qs.kind = qkind;
  qs.scale = qa;
  qs.zp = qb;
  if (!make_batch_map(qs.smap, bnd, bshape, qa_stride) || !make_batch_map(qs.zmap, bnd, bshape, qb_stride))
    return GPTQ2D_EINVAL;
  qs.qmin = (T)qmin;
  qs.qmax = (T)qmax;
  qs.ypre = ypre;
  qs.sout = qkind == Q_ABSMAX ? scale_out : nullptr;
  qs.dtype16 = dtype16;
  const int64_t B = batch_count(bnd, bshape);
  if (B == 0) return 0;
  const int64_t mt = cdiv(m, TR), nt = cdiv(n, TR), stages = mt + nt - 1;
  if (stage_end < 0 || stage_end > stages) stage_end = stages;
  // a call covers whole outer blocks: [stage_begin, stage_end) starts on an outer block's first stage and
  // ends after one's last (or at the end of the sweep), so that consecutive calls resume exactly
  if (stage_begin < 0 || stage_begin > stage_end || stage_begin % outer_tiles ||
      (stage_end % outer_tiles && stage_end != stages))
    return GPTQ2D_EINVAL;
  // 128-bit operand loads of the MFMA pull: rows, matrices and pointers 16-byte aligned
  const bool vec = m % 4 == 0 && n % 4 == 0 && aligned16(y) && aligned16(c) && aligned16(e) && aligned16(l) &&
                   aligned16(u) && strides_mult4(lmap) && strides_mult4(umap);
  if (kron && !(vec && aligned16(kron->q))) return GPTQ2D_EUNSUPPORTED;
  int rc;
  if (stage_begin == 0 && (rc = gptq2d_fill<T>(c, T(0), B * m * n, stream))) return rc;
  // fp64: stages per band flush inside an outer block (the tile sweeps pull the band's earlier stages); the row
  // sweep pulls nothing, so its every stage is flushed
  const int64_t band = rows ? 1 : BAND64;
  for (int64_t S0 = stage_begin; S0 < stage_end; S0 += outer_tiles) {
    const int64_t S1 = S0 + outer_tiles < stages ? S0 + outer_tiles : stages;
    for (int64_t st = S0; st < S1; ++st) {
      const int64_t lo = st - nt + 1 > 0 ? st - nt + 1 : 0;
      const int64_t hi = st < mt - 1 ? st : mt - 1;
      const bool prof = gptq2d_prof_on(PROF_TILE_SWEEP);
      if (prof) gptq2d_prof_begin(PROF_TILE_SWEEP, stream);
      if constexpr (sizeof(T) == 4) {
        // fp32: this stage's sweeps plus the prep of the next stage of the outer block
        int64_t plo = 0, pcount = 0;
        if (st + 1 < S1) {
          plo = st + 1 - nt + 1 > 0 ? st + 1 - nt + 1 : 0;
          pcount = (st + 1 < mt - 1 ? st + 1 : mt - 1) - plo + 1;
        }
        const Grid3 g = make_grid(hi - lo + 1 + pcount, 1, B);
        auto launch = [&](auto vec_c, auto rows_c) {
          launch_tile_stage<decltype(vec_c)::value, decltype(rows_c)::value>(
              qkind, g.grid, stream, y, c, e, l, u, m, n, st, S0, lo, hi - lo + 1, plo, lmap, umap, qs, g.nx, g.ny);
        };
        using True = std::true_type;
        using False = std::false_type;
        if (kron) {
          if (rows)
            launch_tile_stage<true, true, true>(qkind, g.grid, stream, y, c, e, l, nullptr, m, n, st, S0, lo,
                                                hi - lo + 1, plo, lmap, umap, qs, g.nx, g.ny, *kron);
          else
            launch_tile_stage<true, false, true>(qkind, g.grid, stream, y, c, e, l, nullptr, m, n, st, S0, lo,
                                                 hi - lo + 1, plo, lmap, umap, qs, g.nx, g.ny, *kron);
        } else if (vec)
          rows ? launch(True{}, True{}) : launch(True{}, False{});
        else
          rows ? launch(False{}, True{}) : launch(False{}, False{});
      } else {
        const Grid3 g = make_grid(hi - lo + 1, 1, B);
        if (rows) {
          if (qkind == Q_AFFINE)
            launch_rows_stage<T, Q_AFFINE>(g.grid, stream, y, c, e, l, m, n, st, lo, lmap, qs, g.nx, g.ny);
          else if (qkind == Q_FORCED)
            launch_rows_stage<T, Q_FORCED>(g.grid, stream, y, c, e, l, m, n, st, lo, lmap, qs, g.nx, g.ny);
          else if (qkind == Q_ABSMAX)
            launch_rows_stage<T, Q_ABSMAX>(g.grid, stream, y, c, e, l, m, n, st, lo, lmap, qs, g.nx, g.ny);
          else
            launch_rows_stage<T, Q_ROUND>(g.grid, stream, y, c, e, l, m, n, st, lo, lmap, qs, g.nx, g.ny);
        } else {
          // the push-form sweep of the fp32 engine, in fp64, pulling its band's earlier stages
          const int64_t blo = st - (st - S0) % band;
          if (qkind == Q_AFFINE)
            launch_tile64_k<Q_AFFINE>(g.grid, stream, y, c, e, l, u, m, n, st, lo, blo, lmap, umap, qs, g.nx, g.ny);
          else if (qkind == Q_FORCED)
            launch_tile64_k<Q_FORCED>(g.grid, stream, y, c, e, l, u, m, n, st, lo, blo, lmap, umap, qs, g.nx, g.ny);
          else
            launch_tile64_k<Q_ROUND>(g.grid, stream, y, c, e, l, u, m, n, st, lo, blo, lmap, umap, qs, g.nx, g.ny);
        }
      }
      // work of a tile sweep: its entries (the in-tile feedback is latency-, not throughput-bound)
      if (prof) gptq2d_prof_end(PROF_TILE_SWEEP, (double)B * (hi - lo + 1) * TR * TR, stream);
      if ((rc = (int)hipGetLastError())) return rc;
      if constexpr (sizeof(T) == 8) {
        // a band's stages into the rest of the outer block, after the band's last stage
        if (st + 1 < S1 && (st + 1 - S0) % band == 0 &&
            (rc = gptq2d_flush<T>(y, c, e, l, u, m, n, TR, TR, st + 1 - band, st + 1, S1, lmap, umap, B, stream)))
          return rc;
      }
    }
    if (S1 < stages) {
      if constexpr (sizeof(T) == 4) {
        if (kron) {
          if ((rc = gptq2d_flush_kron(y, c, e, l, *kron, m, n, S0, S1, stages, stream))) return rc;
          continue;
        }
      }
      if ((rc = gptq2d_flush<T>(y, c, e, l, u, m, n, TR, TR, S0, S1, stages, lmap, umap, B, stream))) return rc;
    }
  }
  return 0;
}

// ------------------------------------------------------------------------------------------------ no-alloc entry

// Scratch of gptq2d_sweep_fused_noalloc_*: the sweep's C and E buffers, each half of this array, in a
// fixed device array that the HIP runtime places on every GPU that loads the library (it stays there
// until the process ends).  Host code never uses the name `scratch` as an address (it is a host-side
// stand-in): the device address comes from hipGetSymbolAddress, once per device, on the first call
// made with that device current.
constexpr int64_t NOALLOC_SCRATCH_BYTES = (int64_t)128 << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex scratch_mutex;
void* scratch_ptr[NOALLOC_MAX_DEVICES];

// Device address of the current device's scratch array, or nullptr if it cannot be had.
void* scratch_address() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NOALLOC_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    scratch_ptr[dev] = p;
  }
  return scratch_ptr[dev];
}

template <typename T>
int sweep_fused_noalloc(T* y, const T* l, const T* u, int64_t m, int64_t n, int32_t bnd, const int64_t* bshape,
                        const int64_t* lstride, const int64_t* ustride, int32_t qkind, const T* qa,
                        const int64_t* qa_stride, const T* qb, const int64_t* qb_stride, double qmin, double qmax,
                        T* ypre, int64_t outer_tiles, hipStream_t stream) {
  if (m < 0 || n < 0 || bnd < 0 || bnd > GPTQ2D_MAX_BATCH_DIMS) return GPTQ2D_EINVAL;
  // each of C and E takes half the array: B m n elements of T at most (checked before any product can
  // overflow: every factor is below 2^31 once the first test passes)
  const int64_t cap = NOALLOC_SCRATCH_BYTES / 2 / (int64_t)sizeof(T);
  int64_t count = 1;
  for (int32_t d = 0; d < bnd; ++d) {
    if (bshape[d] < 0) return GPTQ2D_EINVAL;
    count = bshape[d] == 0 || count == 0 ? 0 : (bshape[d] > cap / count ? cap + 1 : count * bshape[d]);
  }
  if (m > 0 && n > 0 && count > 0 && (m > cap || n > cap / m || count > cap / (m * n))) return GPTQ2D_ESCRATCH;
  T* c = static_cast<T*>(scratch_address());
  if (!c) return GPTQ2D_EUNSUPPORTED;
  T* e = c + cap;
  return sweep_fused<T>(y, c, e, l, u, m, n, bnd, bshape, lstride, ustride, qkind, qa, qa_stride, qb, qb_stride, qmin,
                        qmax, ypre, outer_tiles, 0, -1, stream);
}

}  // namespace

extern "C" {

#define GPTQ2D_FUSED_ABI(SUF, T)                                                                                    \
  int gptq2d_sweep_fused_##SUF(T* y, T* c, T* e, const T* l, const T* u, int64_t m, int64_t n, int32_t bnd,        \
                               const int64_t* bshape, const int64_t* lstride, const int64_t* ustride, int32_t qkind, \
                               const T* qa, const int64_t* qa_stride, const T* qb, const int64_t* qb_stride,       \
                               double qmin, double qmax, T* ypre, int64_t outer_tiles, int64_t stage_begin,          \
                               int64_t stage_end, hipStream_t stream) {                                              \
    return sweep_fused<T>(y, c, e, l, u, m, n, bnd, bshape, lstride, ustride, qkind, qa, qa_stride, qb, qb_stride,   \
                          qmin, qmax, ypre, outer_tiles, stage_begin, stage_end, stream);                             \
  }                                                                                                                  \
  int64_t gptq2d_sweep_fused_tile_##SUF(void) { return TR; }                                                      \
  int gptq2d_sweep_fused_se_##SUF(T* y, T* c, T* e, const T* l, const T* u, int64_t m, int64_t n, int64_t p,         \
                                  int64_t q, int32_t bnd, const int64_t* bshape, const int64_t* lstride,             \
                                  const int64_t* ustride, int32_t qkind, const T* qa, const int64_t* qa_stride,     \
                                  const T* qb, const int64_t* qb_stride, double qmin, double qmax, int32_t dtype16, \
                                  T* ypre, T* scale_out, int64_t outer_tiles, int64_t stage_begin,                  \
                                  int64_t stage_end, hipStream_t stream) {                                           \
    if (p <= 0 || q <= 0 || m % p || n % q) return GPTQ2D_EINVAL;                                                  \
    if (p == 1 && q == 1 && qkind != Q_ABSMAX)                                                                       \
      return sweep_fused<T>(y, c, e, l, u, m, n, bnd, bshape, lstride, ustride, qkind, qa, qa_stride, qb, qb_stride, \
                            qmin, qmax, ypre, outer_tiles, stage_begin, stage_end, stream);                          \
    if (p != 1 || q != TR) return GPTQ2D_EUNSUPPORTED;                                                              \
    return sweep_fused<T>(y, c, e, l, u, m, n, bnd, bshape, lstride, ustride, qkind, qa, qa_stride, qb, qb_stride,   \
                          qmin, qmax, ypre, outer_tiles, stage_begin, stage_end, stream, true, dtype16, scale_out);  \
  }                                                                                                                  \
  int gptq2d_sweep_fused_noalloc_##SUF(T* y, const T* l, const T* u, int64_t m, int64_t n, int32_t bnd,              \
                                       const int64_t* bshape, const int64_t* lstride, const int64_t* ustride,       \
                                       int32_t qkind, const T* qa, const int64_t* qa_stride, const T* qb,           \
                                       const int64_t* qb_stride, double qmin, double qmax, T* ypre,                 \
                                       int64_t outer_tiles, hipStream_t stream) {                                    \
    return sweep_fused_noalloc<T>(y, l, u, m, n, bnd, bshape, lstride, ustride, qkind, qa, qa_stride, qb, qb_stride, \
                                  qmin, qmax, ypre, outer_tiles, stream);                                            \
  }

int64_t gptq2d_sweep_fused_noalloc_capacity(int32_t elem_bytes) {
  return elem_bytes == 4 || elem_bytes == 8 ? NOALLOC_SCRATCH_BYTES / 2 / elem_bytes : -1;
}

GPTQ2D_FUSED_ABI(f32, float)
GPTQ2D_FUSED_ABI(f64, double)

int gptq2d_sweep_fused_kron_f32(float* y, float* c, float* e, const float* l, const float* up, const float* uq,
                                int64_t m, int64_t np, int64_t nq, int64_t p, int64_t q, int32_t qkind,
                                const float* qa, const float* qb, double qmin, double qmax, int32_t dtype16,
                                float* ypre, float* scale_out, int64_t outer_tiles, int64_t stage_begin,
                                int64_t stage_end, hipStream_t stream) {
  if (!up || !uq || np <= 0 || nq <= 0 || p <= 0 || q <= 0) return GPTQ2D_EINVAL;
  KronU kr;
  if (!make_kron_u(kr, up, uq, np, nq)) return GPTQ2D_EUNSUPPORTED;
  const int64_t n = np * nq;
  if (m % p || n % q) return GPTQ2D_EINVAL;
  const bool rows = !(p == 1 && q == 1 && qkind != Q_ABSMAX);
  if (rows && (p != 1 || q != TR)) return GPTQ2D_EUNSUPPORTED;
  return sweep_fused<float>(y, c, e, l, nullptr, m, n, 0, nullptr, nullptr, nullptr, qkind, qa, nullptr, qb, nullptr,
                            qmin, qmax, ypre, outer_tiles, stage_begin, stage_end, stream, rows, dtype16, scale_out,
                            &kr);
}

}  // extern "C"
