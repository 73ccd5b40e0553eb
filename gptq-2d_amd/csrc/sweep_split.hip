// Fused fp32 GPTQ-2D sweep whose products between tiles run on the bf16 matrix cores from split operands.
//
// The schedule is that of sweep_tiles.hip: 32 x 32 tiles by coarse stages T = I + J, one launch per stage (the
// stage's tiles are swept in LDS while other workgroups pull the next stage's in-block feedback), and after each
// outer block one flush of its errors into all later stages.  What differs is how a product of two fp32 matrices
// is formed.  Each operand is held as three bf16 pieces, x = h + m + l (split_mma.h: h rounded to nearest, m truncated; 24
// bits together: exact but for pieces below 2^-133), and a product takes the six piece products of weight 2^-16 and
// above, each exact, on v_mfma_f32_32x32x16_bf16 with fp32 accumulation:
//   x y = hh' + hm' + mh' + mm' + hl' + lh'   (left out: ml', lm', below 2^-24 |x y| each, and ll', below 2^-32).
// Against 64 bits the sums are closer than v_mfma_f32_32x32x2_f32's, whose every two terms round the accumulator (the
// figures are in split_mma.h), and six bf16 instructions of 32 cycles replace eight fp32 ones of 64 (measured peaks on
// an MI355X: 1865 / 6 = 311 against 135 TFLOP/s).
//
// Split operands are stored as the instruction reads them, one 6 KB block per 32 x 32 tile in two 16-deep halves
// of three 1 KB pieces: [half][piece][lane][8], lane l holding k = 16 half + 8 (l / 32) + 0..7 of row (left
// operands L, C) or column (right operands E, U) l % 32.  A 1 KB piece is one coalesced 128-bit load per lane,
// straight into registers (pulls) or linearly into LDS (flush), and its LDS reads are free of bank conflicts with
// no swizzle.  The halves of one row of left tiles, and of one column of right tiles, lie consecutively along
// k, so a product walks both operands linearly.  L (tiles strictly below the diagonal), U (strictly above) are
// split once per sweep, E and C by the tile that has swept them.  Rows and columns past the matrix are zeros, so
// no product needs a mask, an alignment or a second form for ragged sizes.
//
// Infinities: x - h is NaN for an infinite x, so a sum with an infinite operand comes out NaN where fp32 may keep
// an infinity.  A sum that is not finite is therefore formed again by the fp32 pull of tile_sweep.h from the fp32
// matrices (rare; every finite sum has only finite operands).
#include "diag_sweep.h"
#include "flush_items.h"
#include "profile.h"
#include "split_mma.h"
#include "tile_sweep.h"

double gptq2d_flush_flops(int64_t m, int64_t n, int64_t P, int64_t Q, int64_t s0, int64_t s1, int64_t s_end);

namespace {


constexpr int64_t HB = 3 * 64 * 16;  // bytes of a 16-deep half block: three pieces of 64 lanes x 16 bytes

// Split operands of one sweep: base addresses, bytes between the batch's matrices (0: shared by the batch).
struct Split {
  char *l, *u, *e, *c;
  int64_t l_bs, u_bs, ec_bs;
  int mt, nt;

  // rows of left blocks and columns of right blocks: half `ch` of the row or column is at + HB ch
  __device__ __forceinline__ char* l_row(int64_t b, int64_t I) const { return l + b * l_bs + I * (I - 1) * HB; }
  __device__ __forceinline__ char* u_col(int64_t b, int64_t J) const { return u + b * u_bs + J * (J - 1) * HB; }
  __device__ __forceinline__ char* e_col(int64_t b, int64_t J) const { return e + b * ec_bs + J * mt * 2 * HB; }
  __device__ __forceinline__ char* c_row(int64_t b, int64_t I) const { return c + b * ec_bs + I * nt * 2 * HB; }
};

// Arguments of the stage and flush kernels, small (a launch's first instructions wait for them): the batch's element
// offsets into L, U, the scales and the zero points come from a table in device memory instead of four BatchMaps.
struct StageArgs {
  float *y, *c, *e;
  const float *l, *u, *scale, *zp;
  float *ypre, *sout;
  const int64_t* offsets;  // [B][4], null where every offset is 0
  Split sp;
  KronU kr;
  float qmin, qmax;
  int dtype16;
  int m, n;
};
struct Offsets {
  int64_t l, u, s, z;
  __device__ __forceinline__ Offsets(const int64_t* table, int64_t b) : l(0), u(0), s(0), z(0) {
    if (!table) return;
    typedef const __attribute__((address_space(4))) int64_t* cptr;  // the scalar cache: written by an earlier launch
    const cptr t = (cptr)(table + 4 * b);
    l = t[0], u = t[1], s = t[2], z = t[3];
  }
};

__global__ void batch_offsets_kernel(int64_t* table, int64_t B, BatchMap lmap, BatchMap umap, BatchMap smap,
                                     BatchMap zmap) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  table[4 * b] = lmap.offset(b);
  table[4 * b + 1] = umap.offset(b);
  table[4 * b + 2] = smap.offset(b);
  table[4 * b + 3] = zmap.offset(b);
}

__device__ __forceinline__ void store_half(char* half, int lane, const float (&x)[8]) {
  bf16x8 p[3];
  split8(x, p);
#pragma unroll
  for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(half + 1024 * k + 16 * lane) = p[k];
}

// Row I and column t < I of the k-th block in the packed order of a strict lower triangle (row I at I (I - 1) / 2).
__device__ __forceinline__ void triangle_index(int64_t k, int64_t& I, int64_t& t) {
  I = (int64_t)((1. + __builtin_sqrt(1. + 8. * (double)k)) * 0.5);
  while (I * (I - 1) / 2 > k) --I;
  while ((I + 1) * I / 2 <= k) ++I;
  t = k - I * (I - 1) / 2;
}

// L's and U's blocks, two tiles per workgroup: 128 threads write the 128 (half, lane) groups of 8 values of a tile.
// Workgroups from `groups` on clear C, nc values, in the same launch: a call of a few tiles is bound by the host's
// launches (4 x 128 with a Kronecker U 66 -> 62 us, 4 matrices of 16 x 16 42 -> 40).  Bound by HBM: 4 KB read and 6 KB
// written per tile of both triangles, 4 bytes of C.
template <bool KR>
__global__ __launch_bounds__(256) void split_factors_kernel(const float* __restrict__ l, const float* __restrict__ u,
                                                            int64_t m, int64_t n, int64_t nl, int64_t nu,
                                                            BatchMap lmap, BatchMap umap, Split sp, int64_t bl,
                                                            int64_t bu, KronU kr, int64_t groups, float* __restrict__ c,
                                                            int64_t nc) {
  if (blockIdx.x >= groups) {
    const int64_t wgs = gridDim.x - groups, wg = (blockIdx.x - groups) + wgs * blockIdx.y;
    for (int64_t i = wg * 256 + threadIdx.x; i < nc; i += wgs * gridDim.y * 256) c[i] = 0.f;
    return;
  }
  const int lane = threadIdx.x & 63, half = (threadIdx.x >> 6) & 1;
  const int li = lane & 31, kk = 16 * half + 8 * (lane >> 5);
  int64_t k = 2 * (int64_t)blockIdx.x + (threadIdx.x >> 7);
  const int64_t b = blockIdx.y;
  float v[8];
  int64_t I, t;
  if (k < nl) {
    if (b >= bl) return;
    triangle_index(k, I, t);  // L[I, t]: row li, columns kk ..
    const int64_t i = I * TR + li, c0 = t * TR + kk;  // every column of a tile left of the diagonal is inside
    const float* src = l + lmap.offset(b) + i * m + c0;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = i < m ? src[s] : 0.f;
    store_half(sp.l_row(b, I) + (2 * t + half) * HB, lane, v);
    return;
  }
  k -= nl;
  if (k >= nu || b >= bu) return;
  triangle_index(k, I, t);  // U[t, J = I]: column li, rows kk ..
  const int64_t j = I * TR + li, r0 = t * TR + kk;
  if constexpr (KR) {
    int jb = 0, jq = 0, rb, rq;
    if (j < n) kron_index(kr, (int)j, jb, jq);
    kron_index(kr, (int)r0, rb, rq);  // 8 aligned rows lie in one block of P
    const float p = j < n ? kr.p[(int64_t)rb * kr.np + jb] : 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = j < n ? p * kr.q[(int64_t)(rq + s) * kr.nq + jq] : 0.f;
  } else {
    const float* src = u + umap.offset(b) + r0 * n + j;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = j < n ? src[s * n] : 0.f;
  }
  store_half(sp.u_col(b, I) + (2 * t + half) * HB, lane, v);
}

// ------------------------------------------------------------------------------------------------ tile stage

// One wave's share of a band product: acc += sum over the 16-deep halves ch = c_lo + part (mod nparts) below c_hi of
// the row of left blocks at `a` times the column of right blocks at `b`, straight from global memory.  The loads of G
// halves are issued before their products; FULL: G of them always, the last half again past c_hi (not multiplied), so
// that no branch lies between them.  FULL suits the plain tiles' two halves at a time (4096^2 at 512 antidiagonals 4.371 ms,
// 4.395 without; at 768 it is the other way, 3000^2 2.89, 2.82), not the rows' six.
template <int G, bool FULL>
__device__ __forceinline__ void pull_split(floatx16& acc, const char* __restrict__ a, const char* __restrict__ b,
                                           int c_lo, int c_hi, int part, int nparts, int lane) {
  for (int base = c_lo + part; base < c_hi; base += nparts * G) {
    bf16x8 av[G][3], bv[G][3];
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int ch = base + nparts * q;
      if (!FULL && ch >= c_hi) break;
      const int at = ch < c_hi ? ch : c_hi - 1;
      const char* ap = a + at * HB + 16 * lane;
      const char* bp = b + at * HB + 16 * lane;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        av[q][p] = *reinterpret_cast<const bf16x8*>(ap + 1024 * p);
        bv[q][p] = *reinterpret_cast<const bf16x8*>(bp + 1024 * p);
      }
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if (base + nparts * q >= c_hi) break;
#pragma unroll
      for (int x = 0; x < NPROD; ++x)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[q][prod_a[x]], bv[q][prod_b[x]], acc, 0, 0, 0);
    }
  }
}

// What a workgroup pulls for tile (I, J): the 16-deep halves [d0, d1) of the down product and [r0, r1) of the right
// one, dealt to `waves` waves (the first wd to the down product) in proportion to their lengths.
struct PullRange {
  int d0, d1, r0, r1, wd;
  bool any;

  // a sweep's newest k-tile, or a prep's k-tiles of the outer block before it
  __device__ __forceinline__ PullRange(bool sweep, int64_t S0, int64_t I, int64_t J, int waves) {
    const int dlo = S0 - J > 0 ? (int)(S0 - J) : 0, rlo = S0 - I > 0 ? (int)(S0 - I) : 0;
    if (sweep) {
      d0 = I - 1 >= dlo ? 2 * ((int)I - 1) : 0, d1 = I - 1 >= dlo ? 2 * (int)I : 0;
      r0 = J - 1 >= rlo ? 2 * ((int)J - 1) : 0, r1 = J - 1 >= rlo ? 2 * (int)J : 0;
    } else {
      d0 = 2 * dlo, d1 = I - 1 > dlo ? 2 * ((int)I - 1) : d0;
      r0 = 2 * rlo, r1 = J - 1 > rlo ? 2 * ((int)J - 1) : r0;
    }
    const int nd = d1 - d0, nr = r1 - r0;
    any = nd > 0 || nr > 0;
    wd = nd == 0 ? 0 : (nr == 0 ? waves : (waves * nd + (nd + nr) / 2) / (nd + nr));
    if (nd > 0 && nr > 0) wd = wd < 1 ? 1 : (wd > waves - 1 ? waves - 1 : wd);
  }
};

// The fp32 sum of the halves that pull_split takes for this wave (a sum that is not finite, see above).
template <bool KR>
__device__ __forceinline__ void pull_exact(floatx16& acc, bool down, const float* __restrict__ lb,
                                           const float* __restrict__ eb, const float* __restrict__ cb,
                                           const float* __restrict__ ub, const KronU& kr, int64_t m, int64_t n,
                                           int64_t i0, int64_t j0, int c_lo, int c_hi, int part, int nparts, int lane) {
  const int li = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int ch = c_lo + part; ch < c_hi; ch += nparts) {
    if (down)
      pull_chunks<false>(acc, lb, m, m, m, eb, n, m, n, i0, j0, 2 * ch, 2 * ch + 2, 0, 1, li, hh);
    else if constexpr (KR)
      pull_chunks_kron<false>(acc, cb, n, m, n, kr, n, n, i0, j0, 2 * ch, 2 * ch + 2, 0, 1, li, hh);
    else
      pull_chunks<false>(acc, cb, n, m, n, ub, n, n, n, i0, j0, 2 * ch, 2 * ch + 2, 0, 1, li, hh);
  }
}

// The split E and C of a swept tile of 1 x 32 rows, from its LDS image: threads 0-127 the 128 (half, lane) groups of
// E's block (column l % 32, rows 16 half + 8 (l / 32) ..), threads 128-255 those of C's (row l % 32, columns ..).  A block
// that is null is not written.
__device__ __forceinline__ void store_split(const TileLds& tl, char* eblk, char* cblk, int rows_in, int cols_in) {
  const int lane = threadIdx.x & 63, half = (threadIdx.x >> 6) & 1;
  const int li = lane & 31, kk = 16 * half + 8 * (lane >> 5);
  float v[8];
  if (threadIdx.x < 128) {
    if (!eblk) return;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = kk + s < rows_in && li < cols_in ? tl.Es[TR + kk + s][li] : 0.f;
    store_half(eblk + half * HB, lane, v);
  } else {
    if (!cblk) return;
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = li < rows_in && kk + s < cols_in ? tl.Cs[li][TR + kk + s] : 0.f;
    store_half(cblk + half * HB, lane, v);
  }
}

// One launch per coarse stage T inside the outer block of tile stages [S0, S1): prep workgroups pull the feedback of
// the tiles of stage T + 1 from the block's tiles up to stage T - 1, sweep workgroups pull the newest k-tile of
// the tiles of stage T and sweep them (as tile_stage_kernel of sweep_tiles.hip, on split operands).
//
// Latency-bound: of a sweep workgroup's 24 thousand clocks at 4096^2, 4 go by until its operands have arrived, 2.5 on
// the image, 16 in sweep_diag and 1.3 on the stores.  Per launch 17.5 us with the 256-thread sweep that has every wave
// in every step, 12.5 us here (4096^2); 8192^2 19.4 -> 14.9 us, 256^2 13.9 -> 10.7.
template <int KIND, bool YPRE, bool KR>
__global__ __launch_bounds__(DTHREADS, 2) void tile_stage_split_kernel(StageArgs g, int stage, int S0, int tile_lo,
                                                                       int n_sweep, int prep_lo) {
  __shared__ __align__(16) DiagLds dl;
  constexpr int NQ = TR * TR / DTHREADS;

  const int b = blockIdx.y;
  const bool sweep = (int)blockIdx.x < n_sweep;
  const int I = sweep ? tile_lo + (int)blockIdx.x : prep_lo + ((int)blockIdx.x - n_sweep);
  const int J = (sweep ? stage : stage + 1) - I;
  const int m = g.m, n = g.n, i0 = I * TR, j0 = J * TR;
  const int64_t mat = (int64_t)b * m * n, at = mat + (int64_t)i0 * n + j0;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a sweep has four halves at most: four waves pull them, one each
  const int waves = sweep ? 4 : DW;
  const PullRange pr(sweep, S0, I, J, waves);
  if (!sweep && !pr.any) return;
  const Offsets off(g.offsets, b);

  const bool down = wave < pr.wd, pulls = pr.any && wave < waves;
  const int c_lo = down ? pr.d0 : pr.r0, c_hi = down ? pr.d1 : pr.r1, part = down ? wave : wave - pr.wd,
            np = down ? pr.wd : waves - pr.wd;
  const char* pa = down ? g.sp.l_row(b, I) : g.sp.c_row(b, I);
  const char* pb = down ? g.sp.e_col(b, J) : g.sp.u_col(b, J);
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto stash = [&]() {
    if (!pulls) return;
    if (any_nonfinite(acc))
      pull_exact<KR>(acc, down, g.l + off.l, g.e + mat, g.c + mat, KR ? nullptr : g.u + off.u, g.kr, m, n, i0, j0, c_lo,
                     c_hi, part, np, lane);
    const int li = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int r = 0; r < 16; ++r) dl.red[wave][8 * (r >> 2) + 4 * hh + (r & 3)][li] = acc[r];
  };
  // the sums at entry k of this thread (row tid / 32 + 16 k, column tid % 32)
  const int cc = tid & 31, r0 = tid >> 5;
  auto sums = [&](int k, float& dd, float& rr) {
    dd = rr = 0.f;
#pragma unroll
    for (int w = 0; w < DW; ++w) {
      if (w >= waves) break;
      const float v = dl.red[w][r0 + 16 * k][cc];
      dd += w < pr.wd ? v : 0.f;
      rr += w < pr.wd ? 0.f : v;
    }
  };
  const int rows_in = m - i0 < TR ? m - i0 : TR, cols_in = n - j0 < TR ? n - j0 : TR;

  if (!sweep) {  // Y += D + R, C += D in place
    pull_split<2, true>(acc, pa, pb, c_lo, c_hi, part, np, lane);
    stash();
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int r = r0 + 16 * k;
      if (r < rows_in && cc < cols_in) {
        float dd, rr;
        sums(k, dd, rr);
        float* yt = g.y + at + r * n + cc;
        float* ct = g.c + at + r * n + cc;
        *yt += dd + rr;
        *ct += dd;
      }
    }
    return;
  }

  // the pull's operands first (what it waits for is in flight when the rest is asked for), then the tile's own: all
  // through buffer resources with masked offsets, no branch between them, so that each wait is for its own loads
  bf16x8 av[3], bv[3];
  const int ch = c_lo + part;
  const bool mine = pulls && ch < c_hi;
  if (mine) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      av[p] = *reinterpret_cast<const bf16x8*>(pa + ch * HB + 1024 * p + 16 * lane);
      bv[p] = *reinterpret_cast<const bf16x8*>(pb + ch * HB + 1024 * p + 16 * lane);
    }
  }
  static_assert(DTHREADS / TR == 16, "entry k of a thread lies in the tile's rows 16 k .. 16 k + 15");
  float yo[NQ], co[NQ], so[NQ], zo[NQ], lo[NQ], uo[NQ], pu[NQ];
  {
    auto rsrc = [](const float* p) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, OOB, 0x00020000);
    };
    auto load = [](__amdgpu_buffer_rsrc_t r, int o) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
    };
    const int64_t corner = (int64_t)i0 * n + j0;
    const __amdgpu_buffer_rsrc_t ry = rsrc(g.y + at), rc = rsrc(g.c + at);
    const __amdgpu_buffer_rsrc_t rl = rsrc(g.l + off.l + (int64_t)i0 * m + i0);
    const __amdgpu_buffer_rsrc_t rt = rsrc(KR ? nullptr : g.u + off.u + (int64_t)j0 * n + j0);
    const __amdgpu_buffer_rsrc_t rs = rsrc(KIND == Q_ROUND ? nullptr : g.scale + off.s + corner);
    const __amdgpu_buffer_rsrc_t rz = rsrc(KIND == Q_AFFINE ? g.zp + off.z + corner : nullptr);
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int r = r0 + 16 * k;
      const int o = r < rows_in && cc < cols_in ? (r * n + cc) * 4 : OOB;
      const int ol = cc < r && r < rows_in ? (r * m + cc) * 4 : OOB;
      int ou = r < cc && cc < cols_in ? (r * n + cc) * 4 : OOB;
      yo[k] = load(ry, o);
      co[k] = load(rc, o);
      lo[k] = load(rl, ol);
      if constexpr (KR) {
        // the P entry times the Q entry.  U's rows j0 + 16 k .. + 15 are 16 rows of Q in one block of P: the resources
        // are based there, so that no offset exceeds 16 rows of Q (an offset from Q's first entry would not fit 32
        // bits from nq = 23171 on)
        int ib, i16, jb = 0, jq = 0;
        kron_split(g.kr, (unsigned)(j0 / 16 + k), ib, i16);
        if (ou != OOB) {
          kron_index(g.kr, j0 + cc, jb, jq);
          ou = (r0 * g.kr.nq + jq) * 4;
        }
        pu[k] = load(rsrc(g.kr.p + (int64_t)ib * g.kr.np), ou != OOB ? jb * 4 : OOB);
        uo[k] = load(rsrc(g.kr.q + (int64_t)i16 * 16 * g.kr.nq), ou);
      } else {
        uo[k] = load(rt, ou);
      }
      so[k] = KIND == Q_ROUND ? 0.f : load(rs, o);
      zo[k] = KIND == Q_AFFINE ? load(rz, o) : 0.f;
    }
  }
  if (mine) {
#pragma unroll
    for (int x = 0; x < NPROD; ++x)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[prod_a[x]], bv[prod_b[x]], acc, 0, 0, 0);
  }
  stash();
  const bool q_ok = g.qmin <= g.qmax;
  bool nonzero = false, odd = false;
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    if constexpr (KR) uo[k] *= pu[k];
    if (KIND == Q_AFFINE && !(r0 + 16 * k < rows_in && cc < cols_in)) so[k] = 1.f;
    nonzero |= !(zo[k] == 0.f);
    odd |= diag_coefs<KIND>(dl, tid + DTHREADS * k, so[k], zo[k], lo[k], uo[k], q_ok);
  }
  vote(dl.zp, nonzero, wave);
  vote(dl.odd, odd, wave);
  if (pr.any) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      float dd, rr;
      sums(k, dd, rr);
      yo[k] += dd + rr;
      co[k] += dd;
    }
    __syncthreads();  // the partial sums are read: their memory holds the image from here on
  }
  auto image = [&]() {
#pragma unroll
    for (int k = 0; k < NQ; ++k) diag_entry(dl, tid + DTHREADS * k, yo[k], co[k], so[k], zo[k]);
    diag_zeros(dl);
    __syncthreads();
  };
  image();
  if constexpr (KIND == Q_AFFINE) {
    bool exact = any(dl.odd);
    if (!exact) {
      const bool bad = any(dl.zp) ? sweep_diag<KIND, YPRE, false, true>(dl, g.qmin, g.qmax, wave)
                                  : sweep_diag<KIND, YPRE, false, false>(dl, g.qmin, g.qmax, wave);
      vote(dl.bad, bad, wave);
      __syncthreads();
      exact = any(dl.bad);
      if (exact) image();
    }
    if (exact) {
      sweep_diag<KIND, YPRE, true, true>(dl, g.qmin, g.qmax, wave);
      __syncthreads();
    }
  } else {
    sweep_diag<KIND, YPRE, false, false>(dl, g.qmin, g.qmax, wave);
    __syncthreads();
  }

  // the swept tile: threads 0-255 the split E and C (128 (half, lane) groups of 8 values each: E's column lane % 32,
  // rows 16 half + 8 (lane / 32) .., C's row lane % 32, columns ..), the others Y, C and E in fp32
  if (tid < 256) {
    const int half = wave & 1, li = lane & 31, kk = 16 * half + 8 * (lane >> 5);
    const bool ec = wave < 2;
    const float* run = dl.x + (ec ? li : TR + li) * XP + TR + kk;
    const int in = ec ? (li < cols_in ? rows_in : 0) : (li < rows_in ? cols_in : 0);
    float v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = kk + s < in ? run[s] : 0.f;
    store_half((ec ? g.sp.e_col(b, J) + I * 2 * HB : g.sp.c_row(b, I) + J * 2 * HB) + half * HB, lane, v);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = ((tid - 256) >> 5) + 8 * k;
      if (r < rows_in && cc < cols_in) {
        const int64_t o = at + r * n + cc;
        const float4 v = dl.a[r * TR + cc];
        g.y[o] = v.x;
        g.c[o] = dl.x[(TR + r) * XP + TR + cc];
        g.e[o] = dl.x[cc * XP + TR + r];
        if constexpr (YPRE) g.ypre[o] = v.z;
      }
    }
  }
}

// The same for 1 x 32 super-entries (sweep_rows), 256 threads.
template <int KIND, bool YPRE, bool KR>
__global__ __launch_bounds__(NTHREADS, 2) void row_stage_split_kernel(StageArgs g, int stage, int S0, int tile_lo,
                                                                      int n_sweep, int prep_lo) {
  __shared__ float red[2][2][TR][TR + 1];
  __shared__ TileLds tl;

  const int b = blockIdx.y;
  const bool sweep = (int)blockIdx.x < n_sweep;
  const int I = sweep ? tile_lo + (int)blockIdx.x : prep_lo + ((int)blockIdx.x - n_sweep);
  const int J = (sweep ? stage : stage + 1) - I;
  const int64_t m = g.m, n = g.n, i0 = (int64_t)I * TR, j0 = (int64_t)J * TR;
  const int64_t mat = b * m * n;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const PullRange pr(sweep, S0, I, J, 4);
  if (!sweep && !pr.any) return;
  const Offsets off(g.offsets, b);
  const float* lb = g.l + off.l;
  float* const y = g.y;
  float* const c = g.c;
  float* const e = g.e;
  const Split& sp = g.sp;
  const KronU& kr = g.kr;
  QSpec<float> qs;  // of this matrix: no batch offsets left
  qs.scale = g.scale ? g.scale + off.s : nullptr;
  qs.zp = g.zp ? g.zp + off.z : nullptr;
  qs.smap.nd = qs.zmap.nd = 0;
  qs.qmin = g.qmin, qs.qmax = g.qmax;
  qs.ypre = g.ypre, qs.sout = g.sout, qs.dtype16 = g.dtype16;

  TileRegs<true> own;
  RowInputs<float, KIND> rin;
  if (sweep) {
    own.load(y, c, lb, static_cast<const float*>(nullptr), m, n, i0, j0, mat);  // U's diagonal blocks are not read
    rin.load(qs, b, m, n, i0, j0);
  }
  if (pr.any) {
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const bool down = wave < pr.wd;
    const int c_lo = down ? pr.d0 : pr.r0, c_hi = down ? pr.d1 : pr.r1, part = down ? wave : wave - pr.wd,
              np = down ? pr.wd : 4 - pr.wd;
    const char* pa = down ? sp.l_row(b, I) : sp.c_row(b, I);
    const char* pb = down ? sp.e_col(b, J) : sp.u_col(b, J);
    // a sweep has two halves of a product at most; a prep's path is its loads, and no later launch hides it (1024^2 round
    // at 512 antidiagonals 702 us with four halves at a time, read again past the last, 604 with six)
    if (sweep)
      pull_split<1, false>(acc, pa, pb, c_lo, c_hi, part, np, lane);
    else
      pull_split<6, false>(acc, pa, pb, c_lo, c_hi, part, np, lane);
    if (any_nonfinite(acc))
      pull_exact<KR>(acc, down, lb, e + mat, c + mat, KR ? nullptr : g.u + off.u, kr, m, n, i0, j0, c_lo, c_hi,
                     part, np, lane);
    stash_partial(red, acc, wave >> 1, wave & 1);
  }
  __syncthreads();

  const int rows_in = m - i0 < TR ? (int)(m - i0) : TR, cols_in = n - j0 < TR ? (int)(n - j0) : TR;
  if (!sweep) {  // prep: Y += D + R, C += D in place
    float* yt = y + mat + i0 * n + j0;
    float* ct = c + mat + i0 * n + j0;
#pragma unroll
    for (int q = 0; q < TR * TR / NTHREADS; ++q) {
      const int t = tid + NTHREADS * q;
      const int r = t / TR, cc = t % TR;
      if (r < rows_in && cc < cols_in) {
        const int off = r * (int)n + cc;
        float dd, rr;
        pulled_sums(red, pr.wd, r, cc, dd, rr);
        yt[off] = yt[off] + (dd + rr);
        ct[off] = ct[off] + dd;
      }
    }
    return;
  }
  own.store(tl, red, pr.any, pr.wd);
  __syncthreads();
  // the split blocks that a later tile reads (the last tile row's E and the last tile column's C have none)
  char* const eblk = I + 1 < sp.mt ? sp.e_col(b, J) + I * 2 * HB : nullptr;
  char* const cblk = J + 1 < sp.nt ? sp.c_row(b, I) + J * 2 * HB : nullptr;
  const bool image = eblk || cblk;
  sweep_rows<float, KIND, YPRE>(&tl.Ys[0][0], SP, &tl.Cs[0][TR], CPW, &tl.Lp[0][TR], LPW, &tl.Es[TR][0], SP, rin, y, c, e,
                                qs, m, n, i0, j0, mat, image);
  if (!image) return;
  store_split(tl, eblk, cblk, rows_in, cols_in);
  store_tile(tl, y, c, e, m, n, i0, j0, mat);
}

// ------------------------------------------------------------------------------------------------ outer flush

// D += acc over a 32 x 32 tile whose rows start at `base` (row pitch n, columns from j0; `rows` rows inside the
// matrix): all 16 reads of a lane in flight before its first write, lanes past the matrix masked by their offset.
__device__ __forceinline__ void add_tile(float* base, const floatx16& acc, int64_t rows, int64_t n, int64_t j0, int li,
                                         int hh) {
  const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(base, (short)0, OOB, 0x00020000);
  int off[16];
  float cur[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int ri = 8 * (r >> 2) + 4 * hh + (r & 3);
    off[r] = (ri < rows && j0 + li < n) ? (ri * (int)n + (int)j0 + li) * 4 : OOB;
    cur[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, off[r], 0, 0));
  }
#pragma unroll
  for (int r = 0; r < 16; ++r)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, cur[r] + acc[r]), rd, off[r], 0, 0);
}

// C += D, Y += D + R over the target tiles of a band (flush_mfma.hip), on split operands.  A workgroup owns WT x WT
// target tiles, four waves of (WT / 2)^2; each 16-deep half of its operands (WT left and WT right blocks, 3 KB
// each) is staged one half ahead straight into LDS, double-buffered.  Halves outside a tile row's or column's band
// or triangle are staged as zeros, so every wave runs its whole MFMA block on any half where one of its tiles is
// active.
//
// WT = 4: a wave reads 12 KB of LDS per 24 MFMAs of 32 cycles, half of the LDS rate, where one tile per wave
// (WT = 2) would read at all of it; WT = 2 only where 4 x 4 blocks are fewer than two per compute unit.  Three
// workgroups of 48 KB share a compute unit.  Bound by the matrix cores (56% busy over 8192^2's launches) and, before
// the k-tiles were walked in cyclic order, by the caches behind them (6 TB/s of L2 misses, 37% hits): 8192^2 at 768
// antidiagonals, 21 launches, 1000 GFLOP: 8.9-9.0 ms on the fp32 instruction (112 TFLOP/s), 6.4 ms here, 5.7-5.8 ms
// in cyclic order (175); 8192 x 28672, 35 launches: 68.0, 42.8, 38.1 ms (216 TFLOP/s); 4096^2 at 512: 1.48 -> 1.09.
template <int WT, bool KR>
__global__ __launch_bounds__(256, WT == 4 ? 3 : 4) void flush_split_kernel(StageArgs ga, int S0, int S1, int S_end) {
  constexpr int H = WT / 2;
  constexpr int LOADS = WT / 2;  // blocks staged by one wave per half: blocks LOADS w .. of the 2 WT
  __shared__ __align__(16) char sm[2][2 * WT][HB];

  // runs of XG consecutive items go to one XCD (flush_tiles_mfma_kernel)
  constexpr int XG = 16;
  const int nwg = (int)gridDim.x, w = (int)blockIdx.x;
  const int full = nwg / (8 * XG) * (8 * XG);
  int item = w;
  if (w < full) {
    const int within = w % (8 * XG);
    item = w - within + (within % 8) * XG + within / 8;
  }
  const int64_t b = blockIdx.y;
  const Split& sp = ga.sp;
  const int64_t m = ga.m, n = ga.n;
  const TileGeo32 q{sp.mt, sp.nt, S0, S1, S_end};
  int by = 0, bx = 0;
  if (!item_block<WT, 8>(q, item, by, bx)) return;
  const int I0 = by * WT, J0 = bx * WT;
  if (J0 >= q.nt || I0 + J0 >= q.S_end || I0 + J0 + 2 * WT - 2 < q.S1) return;

  // workgroup-wide k-tile ranges of the two products
  int lo[2] = {INT32_MAX, INT32_MAX}, hi[2] = {0, 0};
  for (int a = 0; a < WT; ++a)
    for (int d = 0; d < WT; ++d) {
      if (!is_target(q, I0 + a, J0 + d)) continue;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        int x, z;
        tile_range(q, p, I0 + a, J0 + d, x, z);
        if (x < z) {
          lo[p] = x < lo[p] ? x : lo[p];
          hi[p] = z > hi[p] ? z : hi[p];
        }
      }
    }
  if (lo[0] >= hi[0] && lo[1] >= hi[1]) return;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, hh = lane >> 5;
  const int wi = (wave >> 1) * H, wj = (wave & 1) * H;
  const int64_t mat = b * m * n;

  // k-tile ranges of this wave's tiles (empty where not a target) and their union
  int tlo[2][H][H], thi[2][H][H], wlo[2] = {INT32_MAX, INT32_MAX}, whi[2] = {0, 0};
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int a = 0; a < H; ++a)
#pragma unroll
      for (int d = 0; d < H; ++d) {
        int x, z;
        tile_range(q, p, I0 + wi + a, J0 + wj + d, x, z);
        if (!is_target(q, I0 + wi + a, J0 + wj + d) || z < x) z = x;
        tlo[p][a][d] = x;
        thi[p][a][d] = z;
        if (x < z) {
          wlo[p] = x < wlo[p] ? x : wlo[p];
          whi[p] = z > whi[p] ? z : whi[p];
        }
      }

  floatx16 acc[H][H];
#pragma unroll
  for (int a = 0; a < H; ++a)
#pragma unroll
    for (int d = 0; d < H; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][d][r] = 0.f;

  int redo[2] = {0, 0};  // tiles whose sums are not finite
  const int voff = 16 * lane;
#pragma unroll
  for (int ph = 0; ph < 2; ++ph) {
    if (lo[ph] < hi[ph]) {
      // the blocks this wave stages: x < WT the row I0 + x of left blocks, else the column J0 + x - WT of right
      // ones; half ch is staged while ch lies in [vlo, vhi), zeros otherwise
      __amdgpu_buffer_rsrc_t src[LOADS];
      int vlo[LOADS], vhi[LOADS];
#pragma unroll
      for (int x = 0; x < LOADS; ++x) {
        const int blk = LOADS * wave + x;
        const bool left = blk < WT;
        const int idx = left ? I0 + blk : J0 + blk - WT;
        const bool in = idx < (left ? q.mt : q.nt);
        const bool tri = left == (ph == 0);  // L and U: k-tiles t < idx; C and E: the band's, S0 <= t + idx < S1
        int v0 = tri ? 0 : q.S0 - idx, v1 = tri ? idx : q.S1 - idx;
        const int kt = ph == 0 ? q.mt : q.nt;
        v0 = v0 < 0 ? 0 : v0;
        v1 = v1 > kt ? kt : v1;
        vlo[x] = 2 * v0;
        vhi[x] = in ? 2 * v1 : 0;
        const char* base = left ? (ph == 0 ? sp.l_row(b, idx) : sp.c_row(b, idx))
                                : (ph == 0 ? sp.e_col(b, idx) : sp.u_col(b, idx));
        src[x] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), (short)0, OOB, 0x00020000);
      }
      auto issue = [&](int ch, int buf) {
#pragma unroll
        for (int x = 0; x < LOADS; ++x) {
          char* dst = sm[buf][LOADS * wave + x];
          if (ch >= vlo[x] && ch < vhi[x])
            dma_load_3k(src[x], dst, voff, ch * (int)HB);
          else
            dma_load_3k(src[x], dst, OOB, 0);
        }
      };
      auto step = [&](int ch, int next, int buf) {
        __syncthreads();  // half ch is complete; the other buffer is no longer read
        if (next >= 0) issue(next, 1 - buf);
        const int t = ch >> 1;
        if (t >= wlo[ph] && t < whi[ph]) {
          bf16x8 fa[H][3], fb[H][3];
#pragma unroll
          for (int x = 0; x < H; ++x)
#pragma unroll
            for (int p = 0; p < 3; ++p) {
              fa[x][p] = *reinterpret_cast<const bf16x8*>(&sm[buf][wi + x][1024 * p + voff]);
              fb[x][p] = *reinterpret_cast<const bf16x8*>(&sm[buf][WT + wj + x][1024 * p + voff]);
            }
#pragma unroll
          for (int x = 0; x < NPROD; ++x)
#pragma unroll
            for (int a = 0; a < H; ++a)
#pragma unroll
              for (int d = 0; d < H; ++d)
                acc[a][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][prod_a[x]], fb[d][prod_b[x]], acc[a][d], 0, 0,
                                                                     0);
        }
        wait_dma();
      };
      // k-tiles in cyclic order from the first multiple of the band's length: a tile's range starts at S0 - J (or
      // S0 - I), so from their first k-tiles on, workgroups of neighbouring columns (rows) would walk the row
      // panels they share out of step
      const int len = hi[ph] - lo[ph], period = q.S1 - q.S0;
      int t0 = (lo[ph] + period - 1) / period * period;
      if (t0 >= hi[ph]) t0 = lo[ph];
      __syncthreads();  // the previous product's last reads are done
      issue(2 * t0, 0);
      wait_dma();
      for (int s = 0, t = t0; s < len; ++s) {
        const int tn = t + 1 < hi[ph] ? t + 1 : lo[ph];
        step(2 * t, 2 * t + 1, 0);
        step(2 * t + 1, s + 1 < len ? 2 * tn : -1, 1);
        t = tn;
      }
    }
    // C += D after the down product, Y += D + R after the right one
#pragma unroll
    for (int a = 0; a < H; ++a)
#pragma unroll
      for (int d = 0; d < H; ++d) {
        const bool has = ph == 0 ? tlo[0][a][d] < thi[0][a][d]
                                 : (tlo[0][a][d] < thi[0][a][d] || tlo[1][a][d] < thi[1][a][d]);
        if (!has) continue;
        const int64_t I = I0 + wi + a, J = J0 + wj + d;
        if (any_nonfinite(acc[a][d])) {  // formed again in fp32 below
          redo[ph] |= 1 << (a * H + d);
          continue;
        }
        add_tile((ph == 0 ? ga.c : ga.y) + mat + I * TR * n, acc[a][d], m - I * TR, n, J * TR, li, hh);
      }
  }
  if ((redo[0] | redo[1]) == 0) return;
  const Offsets off(ga.offsets, b);
  for (int x = 0; x < H * H; ++x) {
    if (!(((redo[0] | redo[1]) >> x) & 1)) continue;
    const int64_t I = I0 + wi + x / H, J = J0 + wj + x % H;
    int x0, x1;
    floatx16 f;
#pragma unroll
    for (int r = 0; r < 16; ++r) f[r] = 0.f;
    tile_range(q, 0, (int)I, (int)J, x0, x1);
    pull_chunks<false>(f, ga.l + off.l, m, m, m, ga.e + mat, n, m, n, I * TR, J * TR, 4 * x0, 4 * x1, 0,
                       1, li, hh);
    if ((redo[0] >> x) & 1) add_tile(ga.c + mat + I * TR * n, f, m - I * TR, n, J * TR, li, hh);
    tile_range(q, 1, (int)I, (int)J, x0, x1);
    if constexpr (KR)
      pull_chunks_kron<false>(f, ga.c + mat, n, m, n, ga.kr, n, n, I * TR, J * TR, 4 * x0, 4 * x1, 0, 1, li, hh);
    else
      pull_chunks<false>(f, ga.c + mat, n, m, n, ga.u + off.u, n, n, n, I * TR, J * TR, 4 * x0, 4 * x1, 0,
                         1, li, hh);
    add_tile(ga.y + mat + I * TR * n, f, m - I * TR, n, J * TR, li, hh);
  }
}

// ------------------------------------------------------------------------------------------------ host

struct Args {
  StageArgs g;
  int64_t m, n, B;
  int32_t kind;
  BatchMap lmap, umap, smap, zmap;
  int64_t* offsets;
  hipStream_t stream;
};

template <int WT, bool KR>
int launch_flush(const Args& a, const TileFlush& g) {
  const int64_t items = count_items<WT>(g);
  if (items == 0) return 0;
  if (items > 0x7fffffff) return GPTQ2D_EUNSUPPORTED;
  hipLaunchKernelGGL((flush_split_kernel<WT, KR>), dim3((unsigned)items, (unsigned)a.B), dim3(256), 0, a.stream, a.g,
                     (int)g.S0, (int)g.S1, (int)g.S_end);
  return (int)hipGetLastError();
}

struct Stage {
  int st, S0, lo, n_sweep, prep_lo, n_prep;
};

template <int KIND, bool ROWS, bool KR>
void launch_stage_k(const Args& a, const Stage& s) {
  auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(s.n_sweep + s.n_prep), (unsigned)a.B), dim3(threads), 0, a.stream, a.g,
                       s.st, s.S0, s.lo, s.n_sweep, s.prep_lo);
  };
  if constexpr (ROWS)
    a.g.ypre ? go(row_stage_split_kernel<KIND, true, KR>, NTHREADS)
             : go(row_stage_split_kernel<KIND, false, KR>, NTHREADS);
  else
    a.g.ypre ? go(tile_stage_split_kernel<KIND, true, KR>, DTHREADS)
             : go(tile_stage_split_kernel<KIND, false, KR>, DTHREADS);
}

template <bool ROWS, bool KR>
void launch_stage(const Args& a, const Stage& s) {
  if (a.kind == Q_AFFINE)
    launch_stage_k<Q_AFFINE, ROWS, KR>(a, s);
  else if (a.kind == Q_FORCED)
    launch_stage_k<Q_FORCED, ROWS, KR>(a, s);
  else if constexpr (ROWS) {
    if (a.kind == Q_ABSMAX)
      launch_stage_k<Q_ABSMAX, true, KR>(a, s);
    else
      launch_stage_k<Q_ROUND, true, KR>(a, s);
  } else
    launch_stage_k<Q_ROUND, false, KR>(a, s);
}

bool shared_over_batch(const BatchMap& bm) {
  for (int d = 0; d < bm.nd; ++d)
    if (bm.shape[d] > 1 && bm.stride[d] != 0) return false;
  return true;
}

int64_t triangle_bytes(int64_t tiles) { return tiles * (tiles - 1) * HB; }

// The workspace: split E and C, then L and U (one copy where the batch shares the factor), then the table of offsets.
int64_t split_bytes(int64_t m, int64_t n, int64_t B, int64_t bl, int64_t bu, Split* sp, char* work) {
  const int64_t mt = cdiv(m, TR), nt = cdiv(n, TR), ec = mt * nt * 2 * HB;
  const int64_t lt = triangle_bytes(mt), ut = triangle_bytes(nt);
  if (sp) {
    sp->e = work;
    sp->c = sp->e + B * ec;
    sp->l = sp->c + B * ec;
    sp->u = sp->l + bl * lt;
    sp->ec_bs = ec;
    sp->l_bs = bl > 1 ? lt : 0;
    sp->u_bs = bu > 1 ? ut : 0;
    sp->mt = (int)mt;
    sp->nt = (int)nt;
  }
  return 2 * B * ec + bl * lt + bu * ut + B * 4 * (int64_t)sizeof(int64_t);
}

// Workgroups of split_factors_kernel that split a matrix's factors.
int64_t factor_groups(int64_t mt, int64_t nt) { return cdiv(mt * (mt - 1) / 2 + nt * (nt - 1) / 2, 2); }

template <bool KR>
int run(Args& a, int64_t bl, int64_t bu, bool rows, int64_t outer_tiles, int64_t stage_begin, int64_t stage_end) {
  const Split& sp = a.g.sp;
  const int64_t mt = sp.mt, nt = sp.nt, stages = mt + nt - 1;
  int rc;
  const int64_t nl = mt * (mt - 1) / 2, nu = nt * (nt - 1) / 2, groups = factor_groups(mt, nt);
  const int64_t nc = stage_begin == 0 ? a.B * a.m * a.n : 0, ny = bl > bu ? bl : bu;
  // C by at most 4096 workgroups, of 256 values a pass
  const int64_t clear = cdiv(cdiv(nc, 256) < 4096 ? cdiv(nc, 256) : 4096, ny);
  if (a.g.offsets)
    hipLaunchKernelGGL(batch_offsets_kernel, dim3((unsigned)cdiv(a.B, 256)), dim3(256), 0, a.stream, a.offsets, a.B, a.lmap,
                       a.umap, a.smap, a.zmap);
  if (groups + clear > 0)
    hipLaunchKernelGGL((split_factors_kernel<KR>), dim3((unsigned)(groups + clear), (unsigned)ny), dim3(256), 0, a.stream,
                       a.g.l, a.g.u, a.m, a.n, nl, nu, a.lmap, a.umap, sp, bl, bu, a.g.kr, groups, a.g.c, nc);
  if ((rc = (int)hipGetLastError())) return rc;
  for (int64_t S0 = stage_begin; S0 < stage_end; S0 += outer_tiles) {
    const int64_t S1 = S0 + outer_tiles < stages ? S0 + outer_tiles : stages;
    for (int64_t st = S0; st < S1; ++st) {
      const int64_t lo = st - nt + 1 > 0 ? st - nt + 1 : 0;
      const int64_t hi = st < mt - 1 ? st : mt - 1;
      int64_t plo = 0, pcount = 0;
      if (st + 1 < S1) {
        plo = st + 1 - nt + 1 > 0 ? st + 1 - nt + 1 : 0;
        pcount = (st + 1 < mt - 1 ? st + 1 : mt - 1) - plo + 1;
      }
      const Stage s{(int)st, (int)S0, (int)lo, (int)(hi - lo + 1), (int)plo, (int)pcount};
      const bool prof = gptq2d_prof_on(PROF_TILE_SWEEP);
      if (prof) gptq2d_prof_begin(PROF_TILE_SWEEP, a.stream);
      rows ? launch_stage<true, KR>(a, s) : launch_stage<false, KR>(a, s);
      if (prof) gptq2d_prof_end(PROF_TILE_SWEEP, (double)a.B * (hi - lo + 1) * TR * TR, a.stream);
      if ((rc = (int)hipGetLastError())) return rc;
    }
    if (S1 < stages) {
      const TileFlush g{a.m, a.n, mt, nt, S0, S1, stages};
      const bool prof = gptq2d_prof_on(PROF_FLUSH);
      if (prof) gptq2d_prof_begin(PROF_FLUSH, a.stream);
      rc = count_items<4>(g) * a.B >= 2 * device_cus() ? launch_flush<4, KR>(a, g) : launch_flush<2, KR>(a, g);
      if (prof)
        gptq2d_prof_end(PROF_FLUSH, (double)a.B * gptq2d_flush_flops(a.m, a.n, TR, TR, S0, S1, stages), a.stream);
      if (rc) return rc;
    }
  }
  return 0;
}

}  // namespace

extern "C" {

int64_t gptq2d_sweep_split_workspace(int64_t m, int64_t n, int32_t bnd, const int64_t* bshape, const int64_t* lstride,
                                     const int64_t* ustride) {
  BatchMap lmap, umap;
  if (m <= 0 || n <= 0 || m >= ((int64_t)1 << 20) || n >= ((int64_t)1 << 20) ||
      !make_batch_map(lmap, bnd, bshape, lstride) || !make_batch_map(umap, bnd, bshape, ustride))
    return -1;
  const int64_t B = batch_count(bnd, bshape);
  return split_bytes(m, n, B, shared_over_batch(lmap) ? 1 : B, shared_over_batch(umap) ? 1 : B, nullptr, nullptr);
}

int gptq2d_sweep_split_f32(float* y, float* c, float* e, const float* l, const float* u, const float* up,
                           const float* uq, int64_t np, int64_t nq, int64_t m, int64_t n, int64_t p, int64_t q,
                           int32_t bnd, const int64_t* bshape, const int64_t* lstride, const int64_t* ustride,
                           int32_t qkind, const float* qa, const int64_t* qa_stride, const float* qb,
                           const int64_t* qb_stride, double qmin, double qmax, int32_t dtype16, float* ypre,
                           float* scale_out, int64_t outer_tiles, int64_t stage_begin, int64_t stage_end, void* work,
                           int64_t work_bytes, hipStream_t stream) {
  Args a{};
  if (m <= 0 || n <= 0 || p <= 0 || q <= 0 || m % p || n % q || outer_tiles < 1) return GPTQ2D_EINVAL;
  if (!make_batch_map(a.lmap, bnd, bshape, lstride) || !make_batch_map(a.umap, bnd, bshape, ustride) ||
      !make_batch_map(a.smap, bnd, bshape, qa_stride) || !make_batch_map(a.zmap, bnd, bshape, qb_stride))
    return GPTQ2D_EINVAL;
  const bool rows = !(p == 1 && q == 1 && qkind != Q_ABSMAX), kron = up != nullptr;
  if (rows && (p != 1 || q != TR)) return GPTQ2D_EUNSUPPORTED;
  // 32-bit offsets: 32 rows of a matrix, a row or column of blocks (n / 32 blocks of 6 KB)
  if (m >= ((int64_t)1 << 20) || n >= ((int64_t)1 << 20)) return GPTQ2D_EUNSUPPORTED;
  if (qkind != Q_ROUND && qkind != Q_AFFINE && qkind != Q_FORCED && !(rows && qkind == Q_ABSMAX)) return GPTQ2D_EINVAL;
  if ((qkind == Q_AFFINE && (!qa || !qb)) || (qkind == Q_FORCED && !qa)) return GPTQ2D_EINVAL;
  if (qkind == Q_ABSMAX && (!(qmin < qmax) || (dtype16 != 1 && dtype16 != 2))) return GPTQ2D_EINVAL;
  if (kron) {
    if (!make_kron_u(a.g.kr, up, uq, np, nq)) return GPTQ2D_EUNSUPPORTED;
    if (bnd != 0 || n != np * nq) return GPTQ2D_EINVAL;
  } else if (!u) {
    return GPTQ2D_EINVAL;
  }
  a.B = batch_count(bnd, bshape);
  if (a.B == 0) return 0;
  // the grids: matrices along y, and below 2^32 threads along x for the factors' blocks and C's
  if (a.B > 65535 || factor_groups(cdiv(m, TR), cdiv(n, TR)) > ((int64_t)1 << 24) - 4097) return GPTQ2D_EUNSUPPORTED;
  const int64_t bl = shared_over_batch(a.lmap) ? 1 : a.B, bu = shared_over_batch(a.umap) ? 1 : a.B;
  if (!work || ((uintptr_t)work & 15) || work_bytes < split_bytes(m, n, a.B, bl, bu, &a.g.sp, (char*)work))
    return GPTQ2D_EINVAL;
  a.m = m, a.n = n, a.stream = stream, a.kind = qkind;
  a.g.y = y, a.g.c = c, a.g.e = e, a.g.l = l, a.g.u = u, a.g.m = (int)m, a.g.n = (int)n;
  a.g.scale = qa, a.g.zp = qb, a.g.qmin = (float)qmin, a.g.qmax = (float)qmax;
  a.g.ypre = ypre, a.g.sout = qkind == Q_ABSMAX ? scale_out : nullptr, a.g.dtype16 = dtype16;
  a.offsets = (int64_t*)((char*)a.g.sp.u + bu * triangle_bytes(a.g.sp.nt));
  const bool zero = bl == 1 && bu == 1 && (!qa || shared_over_batch(a.smap)) && (!qb || shared_over_batch(a.zmap));
  a.g.offsets = zero ? nullptr : a.offsets;  // no table, and no launch for it, where every offset is 0
  const int64_t stages = a.g.sp.mt + a.g.sp.nt - 1;
  if (stage_end < 0 || stage_end > stages) stage_end = stages;
  if (stage_begin < 0 || stage_begin > stage_end || stage_begin % outer_tiles ||
      (stage_end % outer_tiles && stage_end != stages))
    return GPTQ2D_EINVAL;
  return kron ? run<true>(a, bl, bu, rows, outer_tiles, stage_begin, stage_end)
              : run<false>(a, bl, bu, rows, outer_tiles, stage_begin, stage_end);
}

}  // extern "C"
