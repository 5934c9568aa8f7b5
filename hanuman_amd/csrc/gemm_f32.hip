// Float32 expert path (compute dtype float32, moe.py:70-74 and the shared
// expert's swiglu, moe.py:23-29) and its backward: grouped GEMMs on the
// float32 matrix cores, v_mfma_f32_32x32x2_f32 (exact float32 products,
// float32 sums), on the masters as they are (w_gate/w_up [N, D, F], w_down
// [N, F, D], row-major float32).
//
// grouped_gemm_f32_kernel: C[r][n] = sum_k A[r][k] * B_e(k, n) over the rows r
// of expert e's segment [offsets[e], offsets[e+1]), A [rows, K] row-major.
// B_e(k, n) is B_e[k][n] (a master [K, ncols]) or, transposed (BT), B_e[n][k]
// (a master [ncols, K] read as its transpose: the data gradients d_ys Wd^T
// and dg Wg^T + du Wu^T).  Epilogues:
//   plain    C = the sums;
//   SwiGLU   the GEMM runs against w_gate and w_up and writes
//            h = silu(g) * u (moe.py:72);
//   dSwiGLU  the same two GEMMs (g, u recomputed) and, with the cotangent dh
//            [rows, F], writes dg to columns [0, F) and du to [F, 2F) of C
//            (the VJP of moe.py:72);
// and, without a second accumulator, a two-phase K: for k >= ksplit the B
// operand is the second matrix at k - ksplit, so that dg Wg^T + du Wu^T is
// one GEMM over [dg | du] (K = 2F).
//
// Tiles of 64 rows x 64 columns, one per workgroup of 4 waves (wave (wm, wn)
// owns a 32 x 32 block); K runs in steps of 16 through LDS.  A single-matrix
// GEMM sums in two interleaved accumulator chains through two LDS stages,
// each step's loads issued two steps ahead; the g/u GEMMs (two chains
// already) load each step at its start through one stage, which keeps more
// workgroups on a CU.  Row tiles are
// numbered per expert segment (ceil(rows / 64) each), found from offsets by
// each workgroup (an LDS scan over the experts); workgroups past the last
// tile exit.  Rows past a segment are never stored.
//
// grouped_wgrad_f32_kernel: the weight gradients, C_e[m][n] = sum over the
// rows r of expert e's segment of A[r][m] * B[r][n] (dWd[e] = h^T d_ys,
// dWg|dWu[e] = xs^T dg|du), one 64 x 64 tile of one expert per workgroup,
// the segment's rows 16 at a time (rows past it load as zero; an empty
// segment writes zeros).  Columns at or past nsplit go to a second output
// (dWu beside dWg).
#include <algorithm>
#include <atomic>

#include "hmoe_common.h"

namespace hmoe {
namespace {

constexpr int kF32Tile = 64;
constexpr int kF32K = 16;
constexpr int kF32MaxExperts = 1024;

enum F32Epilogue { kEpiPlain = 0, kEpiSwiglu = 1, kEpiDSwiglu = 2 };

__device__ __forceinline__ f32x16 mfma32x2(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int EPI, bool BT>
__global__ __launch_bounds__(256) void grouped_gemm_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B0, const float* __restrict__ B1,
    const int32_t* __restrict__ offsets, int n_experts, int kdim, int ksplit, int ncols,
    const float* __restrict__ dh, float* __restrict__ C, int64_t ldc) {
  constexpr bool kDual = EPI != kEpiPlain;  // two accumulators (g and u)
  __shared__ int32_t mstart[kF32MaxExperts + 1];
  __shared__ int32_t scan[256];
  // A tile [64 rows][16 k] and B tiles [16 k][64 n], +1 float of padding per
  // row so that the operand reads below hit distinct banks; two stages for a
  // single matrix, one for g and u (whose kernels keep more workgroups per CU)
  constexpr int kStages = kDual ? 1 : 2;
  __shared__ float sa[kStages][kF32Tile][kF32K + 1];
  __shared__ float sb0[kStages][kF32K][kF32Tile + 1];
  __shared__ float sb1[1][kDual ? kF32K : 1][kF32Tile + 1];
  const int tid = threadIdx.x;
  // per-expert row-tile starts (exclusive scan of ceil(rows_e / 64))
  const int per = (n_experts + 255) / 256;
  int local = 0;
  for (int j = 0; j < per; ++j) {
    const int e = tid * per + j;
    if (e < n_experts) local += (offsets[e + 1] - offsets[e] + kF32Tile - 1) / kF32Tile;
  }
  scan[tid] = local;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int v = tid >= off ? scan[tid - off] : 0;
    __syncthreads();
    scan[tid] += v;
    __syncthreads();
  }
  int run = scan[tid] - local;
  for (int j = 0; j < per; ++j) {
    const int e = tid * per + j;
    if (e < n_experts) {
      mstart[e] = run;
      run += (offsets[e + 1] - offsets[e] + kF32Tile - 1) / kF32Tile;
    }
  }
  if (tid == 255) mstart[n_experts] = scan[255];
  __syncthreads();
  const int n_tiles_n = ncols / kF32Tile;
  const int m_tile = blockIdx.x / n_tiles_n;
  const int n0 = (blockIdx.x - m_tile * n_tiles_n) * kF32Tile;
  if (m_tile >= mstart[n_experts]) return;  // uniform per workgroup
  int lo = 0, hi = n_experts;  // largest e with mstart[e] <= m_tile
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (mstart[mid] <= m_tile) lo = mid; else hi = mid;
  }
  const int e = lo;
  const int64_t row0 = offsets[e] + static_cast<int64_t>(m_tile - mstart[e]) * kF32Tile;
  const int64_t row_end = offsets[e + 1];
  // each B matrix is ksplit long along K; expert stride ksplit * ncols
  const int64_t bstride = static_cast<int64_t>(ksplit) * ncols;
  const float* be0 = B0 + e * bstride;
  const float* be1 = B1 != nullptr ? B1 + e * bstride : nullptr;

  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31, hi2 = lane >> 5;
  // A single matrix sums in two accumulator chains (the K pairs of a step
  // alternate between them), added before the epilogue.
  f32x16 acc0, acc1, acc0b;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    acc0[r] = 0.0f;
    acc1[r] = 0.0f;
    acc0b[r] = 0.0f;
  }
  // loader: A 64 x 16 = 1024 floats, 4 per thread (row tid / 4, k 4 (tid % 4)
  // .. +4); B 16 x 64, 4 per thread: k tid / 16, n 4 (tid % 16) .. +4, or,
  // transposed, n tid / 4, k 4 (tid % 4) .. +4 (4 consecutive k of a row)
  const int a_r = tid >> 2, a_k = (tid & 3) * 4;
  const int b_k = BT ? (tid & 3) * 4 : tid >> 4;
  const int b_n = BT ? tid >> 2 : (tid & 15) * 4;
  const int64_t ar = row0 + a_r < row_end ? row0 + a_r : row_end - 1;  // rows past: any row
  auto load_b = [&](const float* be, int kk0) __attribute__((always_inline)) {
    return BT ? *reinterpret_cast<const f32x4*>(be + static_cast<int64_t>(n0 + b_n) * ksplit + kk0 + b_k)
              : *reinterpret_cast<const f32x4*>(be + static_cast<int64_t>(kk0 + b_k) * ncols + n0 + b_n);
  };
  f32x4 av, bv0, bv1 = {0.0f, 0.0f, 0.0f, 0.0f};
  auto fetch = [&](int k0) __attribute__((always_inline)) {
    av = *reinterpret_cast<const f32x4*>(A + ar * kdim + k0 + a_k);
    if (kDual) {
      bv0 = load_b(be0, k0);
      bv1 = load_b(be1, k0);
    } else {
      bv0 = k0 < ksplit ? load_b(be0, k0) : load_b(be1, k0 - ksplit);  // uniform branch
    }
  };
  auto park = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      sa[buf][a_r][a_k + q] = av[q];
      if (BT) {
        sb0[buf][b_k + q][b_n] = bv0[q];
        if (kDual) sb1[buf][b_k + q][b_n] = bv1[q];
      } else {
        sb0[buf][b_k][b_n + q] = bv0[q];
        if (kDual) sb1[buf][b_k][b_n + q] = bv1[q];
      }
    }
  };
  const int nsteps = kdim / kF32K;
  if constexpr (kDual) {
    // g and u: one stage, each step's loads at its start; two chains already
    for (int st = 0; st < nsteps; ++st) {
      fetch(st * kF32K);
      __syncthreads();
      park(0);
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < kF32K; kk += 2) {
        const float x = sa[0][wm * 32 + l32][kk + hi2];
        acc0 = mfma32x2(sb0[0][kk + hi2][wn * 32 + l32], x, acc0);
        acc1 = mfma32x2(sb1[0][kk + hi2][wn * 32 + l32], x, acc1);
      }
    }
  } else {
    // K step s goes global -> registers during step s - 2 and registers ->
    // LDS stage s & 1 at the end of step s - 1.
    fetch(0);
    park(0);
    if (nsteps > 1) fetch(kF32K);
    __syncthreads();
    for (int st = 0; st < nsteps; ++st) {
      const int buf = st & 1;
      // D[m][n] += A[m][k] B[k][n]: lane supplies A[m = l32][k = hi2] (here the
      // weights, so that a lane ends with one token row) and B[k = hi2][n = l32]
#pragma unroll
      for (int kk = 0; kk < kF32K; kk += 4) {
        const float x0 = sa[buf][wm * 32 + l32][kk + hi2];
        const float x1 = sa[buf][wm * 32 + l32][kk + 2 + hi2];
        acc0 = mfma32x2(sb0[buf][kk + hi2][wn * 32 + l32], x0, acc0);
        acc0b = mfma32x2(sb0[buf][kk + 2 + hi2][wn * 32 + l32], x1, acc0b);
      }
      if (st + 1 < nsteps) park(buf ^ 1);
      if (st + 2 < nsteps) fetch((st + 2) * kF32K);
      __syncthreads();
    }
  }
  if (!kDual) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc0[r] += acc0b[r];
  }
  // lane holds row wm*32 + l32 and columns wn*32 + 8 (r/4) + 4 hi2 + r%4
  const int64_t row = row0 + wm * 32 + l32;
  if (row >= row_end) return;
  const int col = n0 + wn * 32 + hi2 * 4;
  float* crow = C + row * ldc + col;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 v, w;
    f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
    if (EPI == kEpiDSwiglu) d = *reinterpret_cast<const f32x4*>(dh + row * ncols + col + q * 8);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float g = acc0[4 * q + r];
      if (EPI == kEpiSwiglu) {
        v[r] = (g / (1.0f + expf(-g))) * acc1[4 * q + r];
      } else if (EPI == kEpiDSwiglu) {
#pragma clang fp contract(off)
        const float u = acc1[4 * q + r];
        const float s = 1.0f / (1.0f + expf(-g));
        v[r] = d[r] * u * (s * (1.0f + g * (1.0f - s)));
        w[r] = d[r] * (g * s);
      } else {
        v[r] = g;
      }
    }
    *reinterpret_cast<f32x4*>(crow + q * 8) = v;
    if (EPI == kEpiDSwiglu) *reinterpret_cast<f32x4*>(crow + ncols + q * 8) = w;
  }
}

struct WgradTile {
  int e, m0, n0;
};
// S x S tile t of the experts' [mdim][ncols] gradients.
template <int S>
__device__ __forceinline__ WgradTile wgrad_f32_tile(int t, int mdim, int ncols) {
  const int tm = mdim / S, tn = ncols / S;
  const int e = t / (tm * tn);
  const int rem = t - e * tm * tn;
  return {e, (rem / tn) * S, (rem - (rem / tn) * tn) * S};
}

// The 64 x 64 tile at (m0, n0) of expert e, summed over the rows r_lo .. r_hi.
__device__ __forceinline__ void wgrad_f32_sum(float (&sa)[kF32K][kF32Tile + 1],
                                              float (&sb)[kF32K][kF32Tile + 1],
                                              const float* __restrict__ A, int64_t lda,
                                              const float* __restrict__ B, int64_t ldb, int e, int m0,
                                              int n0, int64_t r_lo, int64_t r_hi, int mdim, int ncols,
                                              int nsplit, float* __restrict__ C0,
                                              float* __restrict__ C1) {
  const int tid = threadIdx.x;
  const int lr = tid >> 4, lc = (tid & 15) * 4;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31, hi2 = lane >> 5;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  for (int64_t r0 = r_lo; r0 < r_hi; r0 += kF32K) {
    const int64_t r = r0 + lr;
    f32x4 av = {0.0f, 0.0f, 0.0f, 0.0f}, bv = {0.0f, 0.0f, 0.0f, 0.0f};
    if (r < r_hi) {
      av = *reinterpret_cast<const f32x4*>(A + r * lda + m0 + lc);
      bv = *reinterpret_cast<const f32x4*>(B + r * ldb + n0 + lc);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      sa[lr][lc + q] = av[q];
      sb[lr][lc + q] = bv[q];
    }
    __syncthreads();
    // D[n][m] += B^T[n][k] A[k][m]: lane supplies B[k = hi2][n = l32] and
    // A[k = hi2][m = l32], so that a lane ends with one output row m
#pragma unroll
    for (int kk = 0; kk < kF32K; kk += 2)
      acc = mfma32x2(sb[kk + hi2][wn * 32 + l32], sa[kk + hi2][wm * 32 + l32], acc);
  }
  // lane holds row m0 + wm*32 + l32 and columns wn*32 + 8 (r/4) + 4 hi2 + r%4
  const int64_t m = m0 + wm * 32 + l32;
  const int col = n0 + wn * 32 + hi2 * 4;
  float* dst;
  if (n0 < nsplit)
    dst = C0 + (static_cast<int64_t>(e) * mdim + m) * nsplit + col;
  else
    dst = C1 + (static_cast<int64_t>(e) * mdim + m) * (ncols - nsplit) + (col - nsplit);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = acc[4 * q + r];
    *reinterpret_cast<f32x4*>(dst + q * 8) = v;
  }
}

__global__ __launch_bounds__(256) void grouped_wgrad_f32_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    const int32_t* __restrict__ offsets, int mdim, int ncols, int nsplit, float* __restrict__ C0,
    float* __restrict__ C1) {
  __shared__ float sa[kF32K][kF32Tile + 1];
  __shared__ float sb[kF32K][kF32Tile + 1];
  const WgradTile t = wgrad_f32_tile<kF32Tile>(static_cast<int>(blockIdx.x), mdim, ncols);
  wgrad_f32_sum(sa, sb, A, lda, B, ldb, t.e, t.m0, t.n0, offsets[t.e], offsets[t.e + 1], mdim, ncols,
                nsplit, C0, C1);
}

// ---- few tiles: K split over the waves ----------------------------------------
// Where 64 x 64 tiles are fewer than the CUs (a short prompt, one shared expert,
// a weight gradient of few experts), the kernels above are bound by the latency
// of their K steps.  Here a workgroup's 4 waves share one 32 x 32 tile and split
// K: wave w takes the 32-long K chunks w, w + 4, ..., its operands going from
// global memory straight into registers in the MFMA's layout, a chunk (16
// MFMAs) ahead, with no LDS and no barrier in the loop; the four partial tiles
// are added through LDS in wave order and each wave finishes a quarter of the
// columns.  An MFMA sums k and k + 4 of a chunk's groups of 8 (any order serves
// both operands alike), so a row-major A is read 16 bytes a lane; the waves'
// chunks of a row share its lines.  Four times the tiles and four waves in K:
// 16 times the chains.  Measured, us (64 x 64 -> split; d_model 256, d_ff 512):
// one 2048-row segment, down 18.3 -> 13.2 (128 tiles), its weight gradients 62.4
// -> 14.6 and 63.4 -> 16.4 (32, 64 tiles); 80 rows on 8 experts, gate/up 16.3 ->
// 7.6, down 17.8 -> 7.3; 8 experts' weight gradients over 4096 rows 26.3 -> 18.3
// (256 tiles) and 32.2 -> 27.8 (512).  Past the lines below the operands' traffic
// (twice that of a 64 x 64 tile) loses: gate/up of 2048 rows 17.1 against 22.4
// (256 tiles), 16 experts' weight gradients (1536 tiles) 30.2 against 38.8.
// Short sums lose too, for their four times as many workgroups: a segment's
// weight gradient gains from about 40 rows up where these are one round over the
// chip (128 tiles, 32 rows 3.9 against 3.6, 128 rows 6.7 / 4.4), 120 where they
// are two (256 tiles, 32 rows 4.1 / 5.5, 128 rows 6.9 / 6.6, 256 rows 10.8 / 11.0,
// 512 rows 25 / 17) and 360 for three (512 tiles, 96 rows 8.3 / 11.0, 512 rows
// 31 / 27).
constexpr int kF32Split = 32;

// A lane's f32x4 groups of the four waves' partial fragments, added in wave
// order: part[wave][fragment][q][lane].
__device__ __forceinline__ f32x4 sum_parts(const f32x4* part, int frags, int f, int q, int lane) {
  f32x4 v = part[(f * 4 + q) * 64 + lane];
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    const f32x4 t = part[((w * frags + f) * 4 + q) * 64 + lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] += t[r];
  }
  return v;
}

template <int EPI, bool BT>
__global__ __launch_bounds__(256) void grouped_gemm_f32_split_kernel(
    const float* __restrict__ A, const float* __restrict__ B0, const float* __restrict__ B1,
    const int32_t* __restrict__ offsets, int n_experts, int kdim, int ksplit, int ncols,
    const float* __restrict__ dh, float* __restrict__ C, int64_t ldc) {
  constexpr bool kDual = EPI != kEpiPlain;  // two accumulators (g and u)
  constexpr int kMats = kDual ? 2 : 1;
  __shared__ int32_t mstart[kF32MaxExperts + 1];
  __shared__ int32_t scan[256];
  __shared__ f32x4 part[4 * kMats * 4 * 64];
  const int tid = threadIdx.x;
  // per-expert row-tile starts (exclusive scan of ceil(rows_e / kF32Split))
  const int per = (n_experts + 255) / 256;
  int local = 0;
  for (int j = 0; j < per; ++j) {
    const int e = tid * per + j;
    if (e < n_experts) local += (offsets[e + 1] - offsets[e] + kF32Split - 1) / kF32Split;
  }
  scan[tid] = local;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int v = tid >= off ? scan[tid - off] : 0;
    __syncthreads();
    scan[tid] += v;
    __syncthreads();
  }
  int run = scan[tid] - local;
  for (int j = 0; j < per; ++j) {
    const int e = tid * per + j;
    if (e < n_experts) {
      mstart[e] = run;
      run += (offsets[e + 1] - offsets[e] + kF32Split - 1) / kF32Split;
    }
  }
  if (tid == 255) mstart[n_experts] = scan[255];
  __syncthreads();
  const int n_tiles_n = ncols / kF32Split;
  const int m_tile = blockIdx.x / n_tiles_n;
  const int n0 = (blockIdx.x - m_tile * n_tiles_n) * kF32Split;
  if (m_tile >= mstart[n_experts]) return;  // uniform per workgroup
  int lo = 0, hi = n_experts;  // largest e with mstart[e] <= m_tile
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (mstart[mid] <= m_tile) lo = mid; else hi = mid;
  }
  const int e = __builtin_amdgcn_readfirstlane(lo);
  const int64_t row0 = offsets[e] + static_cast<int64_t>(m_tile - mstart[e]) * kF32Split;
  const int64_t row_end = offsets[e + 1];
  // each B matrix is ksplit long along K; expert stride ksplit * ncols
  const int64_t bstride = static_cast<int64_t>(ksplit) * ncols;
  const float* be0 = B0 + e * bstride;
  const float* be1 = B1 != nullptr ? B1 + e * bstride : be0;

  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi2 = lane >> 5;
  // this lane's row (past the segment: its last one)
  const float* arow = A + (row0 + l32 < row_end ? row0 + l32 : row_end - 1) * kdim;
  const int n = n0 + l32;
  // One chunk of 32 k: group g of 8 k, lane half hi2 holds k = 8 g + 4 hi2 + 0..3.
  struct Chunk {
    f32x4 a[4];
    f32x4 b[kMats][4];
  };
  auto load = [&](Chunk& c, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k = k0 + 8 * g + 4 * hi2;
      c.a[g] = *reinterpret_cast<const f32x4*>(arow + k);
#pragma unroll
      for (int m = 0; m < kMats; ++m) {
        // (a single matrix changes to the second one at ksplit, a multiple of 32)
        const float* be = m == 1 || (!kDual && k0 >= ksplit) ? be1 : be0;
        const int kb = !kDual && k0 >= ksplit ? k - ksplit : k;
        f32x4& v = c.b[m][g];
        if constexpr (BT) {
          v = *reinterpret_cast<const f32x4*>(be + static_cast<int64_t>(n) * ksplit + kb);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = be[static_cast<int64_t>(kb + r) * ncols + n];
        }
      }
    }
  };
  // The last 16 k of a K that is an odd multiple of 16 (a single matrix, or g
  // and u: a two-phase K is a multiple of 128): zeros past it.
  auto load_tail = [&](Chunk& c, int k0) __attribute__((always_inline)) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k = k0 + 8 * g + 4 * hi2;
      c.a[g] = g < 2 ? *reinterpret_cast<const f32x4*>(arow + k) : zero;
#pragma unroll
      for (int m = 0; m < kMats; ++m) {
        const float* be = m == 1 ? be1 : be0;
        f32x4 v = zero;
        if (g < 2) {
          if (BT) {
            v = *reinterpret_cast<const f32x4*>(be + static_cast<int64_t>(n) * ksplit + k);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = be[static_cast<int64_t>(k + r) * ncols + n];
          }
        }
        c.b[m][g] = v;
      }
    }
  };
  f32x16 acc[kMats];
#pragma unroll
  for (int m = 0; m < kMats; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.0f;
  // D[n][m] += B^T[n][k] A^T[k][m]: the weights are the first operand, so that
  // a lane ends with one token row and groups of 4 columns
  auto compute = [&](const Chunk& c) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < kMats; ++m) acc[m] = mfma32x2(c.b[m][g][r], c.a[g][r], acc[m]);
  };
  const int nfull = kdim / 32;
  Chunk c0, c1;
  int ch = wave;
  if (ch < nfull) load(c0, ch * 32);
  for (; ch < nfull; ch += 8) {
    if (ch + 4 < nfull) load(c1, (ch + 4) * 32);
    compute(c0);
    if (ch + 4 >= nfull) break;
    if (ch + 8 < nfull) load(c0, (ch + 8) * 32);
    compute(c1);
  }
  if (kdim % 32 != 0 && (nfull & 3) == wave) {
    load_tail(c0, nfull * 32);
    compute(c0);
  }
#pragma unroll
  for (int m = 0; m < kMats; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[m][4 * q + r];
      part[((wave * kMats + m) * 4 + q) * 64 + lane] = v;
    }
  __syncthreads();
  // Wave w finishes group q = w: lane row l32, columns 8 w + 4 hi2 + 0..3.
  const int64_t row = row0 + l32;
  if (row >= row_end) return;
  const int col = n0 + 8 * wave + 4 * hi2;
  const f32x4 g4 = sum_parts(part, kMats, 0, wave, lane);
  f32x4 v = g4;
  if constexpr (kDual) {
    const f32x4 u4 = sum_parts(part, kMats, 1, wave, lane);
    if constexpr (EPI == kEpiSwiglu) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (g4[r] / (1.0f + expf(-g4[r]))) * u4[r];
    } else {
#pragma clang fp contract(off)
      const f32x4 d = *reinterpret_cast<const f32x4*>(dh + row * ncols + col);
      f32x4 w;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float sg = 1.0f / (1.0f + expf(-g4[r]));
        v[r] = d[r] * u4[r] * (sg * (1.0f + g4[r] * (1.0f - sg)));
        w[r] = d[r] * (g4[r] * sg);
      }
      *reinterpret_cast<f32x4*>(C + row * ldc + ncols + col) = w;
    }
  }
  *reinterpret_cast<f32x4*>(C + row * ldc + col) = v;
}

// Four workgroups a 64 x 64 tile.  The lengths of the segments are known only
// here: one of fewer than min_rows is summed as above, by the first quarter of
// the workgroups, beside their parts of the others.
__global__ __launch_bounds__(256) void grouped_wgrad_f32_split_kernel(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    const int32_t* __restrict__ offsets, int mdim, int ncols, int nsplit, int min_rows,
    float* __restrict__ C0, float* __restrict__ C1) {
  union Lds {
    f32x4 part[4 * 4 * 64];
    float ab[2][kF32K][kF32Tile + 1];
  };
  __shared__ Lds lds;
  f32x4* const part = lds.part;
  const int tid = threadIdx.x;
  const WgradTile t = wgrad_f32_tile<kF32Split>(static_cast<int>(blockIdx.x), mdim, ncols);
  const int e = t.e, m0 = t.m0, n0 = t.n0;
  const int64_t r_lo = __builtin_amdgcn_readfirstlane(offsets[e]);
  const int rows = __builtin_amdgcn_readfirstlane(offsets[e + 1]) - static_cast<int>(r_lo);
  if (blockIdx.x < gridDim.x / 4) {
    const WgradTile w = wgrad_f32_tile<kF32Tile>(static_cast<int>(blockIdx.x), mdim, ncols);
    const int64_t r0 = offsets[w.e], r1 = offsets[w.e + 1];
    if (r1 - r0 < min_rows) {
      wgrad_f32_sum(lds.ab[0], lds.ab[1], A, lda, B, ldb, w.e, w.m0, w.n0, r0, r1, mdim, ncols, nsplit,
                    C0, C1);
      __syncthreads();
    }
  }
  if (rows < min_rows) return;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi2 = lane >> 5;
  // One chunk of 32 rows: MFMA s takes rows 2 s + hi2.  The resources start at
  // the chunk and end at the segment, so later rows read as zeros.
  struct Chunk {
    float a[16];
    float b[16];
  };
  const int a_voff = (hi2 * static_cast<int>(lda) + m0 + l32) * 4;
  const int b_voff = (hi2 * static_cast<int>(ldb) + n0 + l32) * 4;
  auto load = [&](Chunk& c, int r0) __attribute__((always_inline)) {
    const int left = rows - r0 < 32 ? rows - r0 : 32;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(A + (r_lo + r0) * lda), 0, left * static_cast<int>(lda) * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(B + (r_lo + r0) * ldb), 0, left * static_cast<int>(ldb) * 4, 0x00020000);
    // (the row offset is in the range-checked vector offset)
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      c.a[s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          ra, a_voff + 2 * s * static_cast<int>(lda) * 4, 0, 0));
      c.b[s] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          rb, b_voff + 2 * s * static_cast<int>(ldb) * 4, 0, 0));
    }
  };
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  // D[n][m] += B^T[n][k] A[k][m], so that a lane ends with one output row m
  auto compute = [&](const Chunk& c) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 16; ++s) acc = mfma32x2(c.b[s], c.a[s], acc);
  };
  const int n_ch = (rows + 31) / 32;
  Chunk c0, c1;
  int ch = wave;
  if (ch < n_ch) load(c0, ch * 32);
  for (; ch < n_ch; ch += 8) {
    if (ch + 4 < n_ch) load(c1, (ch + 4) * 32);
    compute(c0);
    if (ch + 4 >= n_ch) break;
    if (ch + 8 < n_ch) load(c0, (ch + 8) * 32);
    compute(c1);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = acc[4 * q + r];
    part[(wave * 4 + q) * 64 + lane] = v;
  }
  __syncthreads();
  // wave w finishes group q = w: row m0 + l32, columns 8 w + 4 hi2 + 0..3
  const int64_t m = static_cast<int64_t>(e) * mdim + m0 + l32;
  const f32x4 v = sum_parts(part, 1, 0, wave, lane);
  const int col = n0 + 8 * wave + 4 * hi2;
  float* dst = n0 < nsplit ? C0 + m * nsplit + col : C1 + m * (ncols - nsplit) + (col - nsplit);
  *reinterpret_cast<f32x4*>(dst) = v;
}

// CUs of the stream's device (256 if it cannot be queried), cached per device.
int f32_cus(hipStream_t s) {
  int dev = 0;
  if (hipStreamGetDevice(s, &dev) != hipSuccess && hipGetDevice(&dev) != hipSuccess) return 256;
  static std::atomic<int> cached[64];
  int cus = dev >= 0 && dev < 64 ? cached[dev].load(std::memory_order_relaxed) : 0;
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return 256;
    if (dev >= 0 && dev < 64) cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

template <int EPI, bool BT>
int launch_f32(const float* A, const float* B0, const float* B1, const int32_t* offsets,
               int n_experts, int64_t rows_cap, int kdim, int ksplit, int ncols, const float* dh,
               float* C, int64_t ldc, hipStream_t s, const char* what) {
  const int64_t m_tiles = ceil_div(rows_cap, kF32Tile) + n_experts;
  const int64_t grid = m_tiles * (ncols / kF32Tile);
  HMOE_REQUIRE(grid < (int64_t(1) << 31), "%s: too many tiles", what);
  // fewer 64 x 64 tiles than three quarters of the CUs (rows_cap rows at most)
  if (ceil_div(rows_cap, kF32Tile) * (ncols / kF32Tile) * 4 < int64_t(3) * f32_cus(s)) {
    const int64_t split = (ceil_div(rows_cap, kF32Split) + std::min<int64_t>(n_experts, rows_cap)) *
                          (ncols / kF32Split);
    hipLaunchKernelGGL((grouped_gemm_f32_split_kernel<EPI, BT>), dim3(static_cast<unsigned>(split)),
                       dim3(256), 0, s, A, B0, B1, offsets, n_experts, kdim, ksplit, ncols, dh, C, ldc);
    return check_launch(what);
  }
  hipLaunchKernelGGL((grouped_gemm_f32_kernel<EPI, BT>), dim3(static_cast<unsigned>(grid)), dim3(256),
                     0, s, A, B0, B1, offsets, n_experts, kdim, ksplit, ncols, dh, C, ldc);
  return check_launch(what);
}

int launch_wgrad_f32(const float* A, int64_t lda, const float* B, int64_t ldb,
                     const int32_t* offsets, int n_experts, int mdim, int ncols, int nsplit,
                     float* C0, float* C1, hipStream_t s, const char* what) {
  const int64_t grid = static_cast<int64_t>(n_experts) * (mdim / kF32Tile) * (ncols / kF32Tile);
  HMOE_REQUIRE(grid < (int64_t(1) << 31), "%s: too many tiles", what);
  const int64_t cus = f32_cus(s);
  if (grid <= 2 * cus) {
    // Three workgroups fit a CU (their registers): the more rounds of them, the
    // longer a sum has to be to gain, see above.
    const int64_t rounds = ceil_div(4 * grid, 3 * cus);
    const int min_rows = rounds == 1 ? 40 : rounds == 2 ? 120 : 360;
    hipLaunchKernelGGL(grouped_wgrad_f32_split_kernel, dim3(static_cast<unsigned>(4 * grid)), dim3(256),
                       0, s, A, lda, B, ldb, offsets, mdim, ncols, nsplit, min_rows, C0, C1);
    return check_launch(what);
  }
  hipLaunchKernelGGL(grouped_wgrad_f32_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, s, A,
                     lda, B, ldb, offsets, mdim, ncols, nsplit, C0, C1);
  return check_launch(what);
}

}  // namespace
}  // namespace hmoe

#define HMOE_F32_CHECK_EXPERTS(what)                                                            \
  HMOE_REQUIRE(n_experts >= 1 && n_experts <= kF32MaxExperts,                                   \
               what ": n_experts must be in [1, %d] (got %d)", kF32MaxExperts, n_experts)

extern "C" int hmoe_grouped_gate_up_f32(const float* xs, const int32_t* offsets, int n_experts,
                                        int64_t rows_cap, int d_model, int d_ff,
                                        const float* w_gate, const float* w_up, float* h,
                                        hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_gate_up_f32");
  HMOE_REQUIRE(rows_cap >= 0, "grouped_gate_up_f32: rows_cap must be >= 0");
  HMOE_REQUIRE_CODE(d_model % kF32K == 0 && d_model > 0 && d_ff % kF32Tile == 0 && d_ff > 0,
                    HMOE_ERR_UNSUPPORTED,
                    "grouped_gate_up_f32: d_model must be a multiple of %d and d_ff of %d "
                    "(got %d, %d)", kF32K, kF32Tile, d_model, d_ff);
  if (rows_cap == 0) return HMOE_OK;
  HMOE_REQUIRE(xs && offsets && w_gate && w_up && h, "grouped_gate_up_f32: null pointer argument");
  return launch_f32<kEpiSwiglu, false>(xs, w_gate, w_up, offsets, n_experts, rows_cap, d_model,
                                       d_model, d_ff, nullptr, h, d_ff,
                                       static_cast<hipStream_t>(stream), "hmoe_grouped_gate_up_f32");
}

extern "C" int hmoe_grouped_down_f32(const float* h, const int32_t* offsets, int n_experts,
                                     int64_t rows_cap, int d_ff, int d_model, const float* w_down,
                                     float* ys, hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_down_f32");
  HMOE_REQUIRE(rows_cap >= 0, "grouped_down_f32: rows_cap must be >= 0");
  HMOE_REQUIRE_CODE(d_ff % kF32K == 0 && d_ff > 0 && d_model % kF32Tile == 0 && d_model > 0,
                    HMOE_ERR_UNSUPPORTED,
                    "grouped_down_f32: d_ff must be a multiple of %d and d_model of %d "
                    "(got %d, %d)", kF32K, kF32Tile, d_ff, d_model);
  if (rows_cap == 0) return HMOE_OK;
  HMOE_REQUIRE(h && offsets && w_down && ys, "grouped_down_f32: null pointer argument");
  return launch_f32<kEpiPlain, false>(h, w_down, nullptr, offsets, n_experts, rows_cap, d_ff, d_ff,
                                      d_model, nullptr, ys, d_model,
                                      static_cast<hipStream_t>(stream), "hmoe_grouped_down_f32");
}

// ---- backward -----------------------------------------------------------------

// Both dims of the backward GEMMs run as K in one of them and as 64-wide
// column tiles in another, so d_model and d_ff are multiples of 64.
#define HMOE_F32_CHECK_DIMS(what)                                                               \
  HMOE_REQUIRE_CODE(d_model % kF32Tile == 0 && d_model > 0 && d_ff % kF32Tile == 0 && d_ff > 0, \
                    HMOE_ERR_UNSUPPORTED,                                                       \
                    what ": d_model and d_ff must be multiples of %d (got %d, %d)", kF32Tile,   \
                    d_model, d_ff)

extern "C" int hmoe_grouped_dgrad_down_f32(const float* d_ys, const int32_t* offsets,
                                           int n_experts, int64_t rows_cap, int d_model, int d_ff,
                                           const float* w_down, float* dh, hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_dgrad_down_f32");
  HMOE_REQUIRE(rows_cap >= 0, "grouped_dgrad_down_f32: rows_cap must be >= 0");
  HMOE_F32_CHECK_DIMS("grouped_dgrad_down_f32");
  if (rows_cap == 0) return HMOE_OK;
  HMOE_REQUIRE(d_ys && offsets && w_down && dh, "grouped_dgrad_down_f32: null pointer argument");
  // dh[r][f] = sum_d d_ys[r][d] Wd[e][f][d]: Wd read transposed
  return launch_f32<kEpiPlain, true>(d_ys, w_down, nullptr, offsets, n_experts, rows_cap, d_model,
                                     d_model, d_ff, nullptr, dh, d_ff,
                                     static_cast<hipStream_t>(stream), "hmoe_grouped_dgrad_down_f32");
}

extern "C" int hmoe_grouped_gate_up_swiglu_bwd_f32(const float* xs, const int32_t* offsets,
                                                   int n_experts, int64_t rows_cap, int d_model,
                                                   int d_ff, const float* w_gate, const float* w_up,
                                                   const float* dh, float* dgu,
                                                   hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_gate_up_swiglu_bwd_f32");
  HMOE_REQUIRE(rows_cap >= 0, "grouped_gate_up_swiglu_bwd_f32: rows_cap must be >= 0");
  HMOE_F32_CHECK_DIMS("grouped_gate_up_swiglu_bwd_f32");
  if (rows_cap == 0) return HMOE_OK;
  HMOE_REQUIRE(xs && offsets && w_gate && w_up && dh && dgu,
               "grouped_gate_up_swiglu_bwd_f32: null pointer argument");
  return launch_f32<kEpiDSwiglu, false>(xs, w_gate, w_up, offsets, n_experts, rows_cap, d_model,
                                        d_model, d_ff, dh, dgu, 2 * static_cast<int64_t>(d_ff),
                                        static_cast<hipStream_t>(stream),
                                        "hmoe_grouped_gate_up_swiglu_bwd_f32");
}

extern "C" int hmoe_grouped_dgrad_gate_up_f32(const float* dgu, const int32_t* offsets,
                                              int n_experts, int64_t rows_cap, int d_model,
                                              int d_ff, const float* w_gate, const float* w_up,
                                              float* d_xs, hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_dgrad_gate_up_f32");
  HMOE_REQUIRE(rows_cap >= 0, "grouped_dgrad_gate_up_f32: rows_cap must be >= 0");
  HMOE_F32_CHECK_DIMS("grouped_dgrad_gate_up_f32");
  if (rows_cap == 0) return HMOE_OK;
  HMOE_REQUIRE(dgu && offsets && w_gate && w_up && d_xs,
               "grouped_dgrad_gate_up_f32: null pointer argument");
  // d_xs[r][d] = sum_f dg[r][f] Wg[e][d][f] + du[r][f] Wu[e][d][f]: K = 2F in
  // two phases, both masters read transposed
  return launch_f32<kEpiPlain, true>(dgu, w_gate, w_up, offsets, n_experts, rows_cap, 2 * d_ff,
                                     d_ff, d_model, nullptr, d_xs, d_model,
                                     static_cast<hipStream_t>(stream),
                                     "hmoe_grouped_dgrad_gate_up_f32");
}

extern "C" int hmoe_grouped_wgrad_gate_up_f32(const float* xs, const float* dgu,
                                              const int32_t* offsets, int n_experts, int d_model,
                                              int d_ff, float* dw_gate, float* dw_up,
                                              hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_wgrad_gate_up_f32");
  HMOE_F32_CHECK_DIMS("grouped_wgrad_gate_up_f32");
  HMOE_REQUIRE(xs && dgu && offsets && dw_gate && dw_up,
               "grouped_wgrad_gate_up_f32: null pointer argument");
  return launch_wgrad_f32(xs, d_model, dgu, 2 * static_cast<int64_t>(d_ff), offsets, n_experts,
                          d_model, 2 * d_ff, d_ff, dw_gate, dw_up, static_cast<hipStream_t>(stream),
                          "hmoe_grouped_wgrad_gate_up_f32");
}

extern "C" int hmoe_grouped_wgrad_down_f32(const float* h, const float* d_ys,
                                           const int32_t* offsets, int n_experts, int d_ff,
                                           int d_model, float* dw_down, hmoe_stream_t stream) {
  using namespace hmoe;
  HMOE_F32_CHECK_EXPERTS("grouped_wgrad_down_f32");
  HMOE_F32_CHECK_DIMS("grouped_wgrad_down_f32");
  HMOE_REQUIRE(h && d_ys && offsets && dw_down, "grouped_wgrad_down_f32: null pointer argument");
  return launch_wgrad_f32(h, d_ff, d_ys, d_model, offsets, n_experts, d_ff, d_model, d_model,
                          dw_down, nullptr, static_cast<hipStream_t>(stream),
                          "hmoe_grouped_wgrad_down_f32");
}
