// Router: fp32 logits, top-k selection and gate weights (model/moe.py:175-192).
//
// Logits are float32 roundings of float64 sums taken in ascending d from +0.0
// (see router_kernel for how the float64 matrix cores keep that order).
// Top-k is K rounds of a max over the totalOrder keys that resolves equal
// keys to the lower expert index: up to 64 experts eight tokens per wave (8
// lanes per token, 64-bit (key, expert) composites, select_group8); beyond,
// one token per wave (a wave-wide max, then a ballot of the lanes at the
// maximum whose lowest expert wins, select_and_gate).
#include <atomic>

#include "hmoe_common.h"
#include "quant_e4m3.h"

namespace hmoe {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// max(v, v of the lane DPP control CTRL names), in the rows ROW_MASK enables
// (other lanes keep v).
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int32_t dpp_max_i32(int32_t v) {
  const int32_t t = ROW_MASK == 0xF ? __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false)
                                    : __builtin_amdgcn_update_dpp(v, v, CTRL, ROW_MASK, 0xF, false);
  return t > v ? t : v;
}

// Wave-wide maxima of NTOK independent values, returned in every lane, on
// the VALU (data-parallel-primitive moves instead of LDS permutes): within
// each row of 16 lanes quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror
// and row_mirror leave the row's maximum in all its lanes; row_bcast15 into
// rows 1 and 3 and row_bcast31 into rows 2 and 3 bring the wave's maximum to
// lane 63, which is read out.
template <int NTOK>
__device__ __forceinline__ void wave_max_i32(int32_t (&v)[NTOK]) {
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0xB1>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0x4E>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0x141>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0x140>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0x142, 0xA>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = dpp_max_i32<0x143, 0xC>(v[q]);
#pragma unroll
  for (int q = 0; q < NTOK; ++q) v[q] = __builtin_amdgcn_readlane(v[q], 63);
}

// Selection + gates for NTOK tokens whose logits are spread over the wave
// (lane owns experts lane + 64*j); the tokens' reduction chains interleave.
// Round k takes the wave maximum of the live totalOrder keys, then the
// lowest expert holding it: the first j (ascending) whose ballot of live
// entries at the maximum is non-empty, and that ballot's lowest lane -- the
// lower-index tie-break of lax.top_k.  The winner's value is read from its
// lane, and the gate denominators are summed from those values in k order.
// Lane k < K writes slot k of every token q with store[q].  bias holds the
// lane's experts' selection biases (load_bias).
//
// load_bias: a lane's N selection biases, expert e0 + j step, 0 without a bias
// or past n_experts; unconditional loads from clamped addresses, so they are
// in flight together (loaded one by one under their conditions they cost the
// selection a serial chain of N memory latencies).
template <int N>
__device__ __forceinline__ void load_bias(float (&b)[N], const float* __restrict__ bias, int e0,
                                          int step, int n_experts) {
#pragma unroll
  for (int j = 0; j < N; ++j) b[j] = 0.0f;
  if (bias == nullptr) return;  // uniform
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int e = e0 + j * step;
    b[j] = bias[e < n_experts ? e : n_experts - 1];
  }
#pragma unroll
  for (int j = 0; j < N; ++j) b[j] = e0 + j * step < n_experts ? b[j] : 0.0f;
}

template <int EPL, int NTOK>
__device__ __forceinline__ void select_and_gate(const float (&logit)[NTOK][EPL],
                                                const bool (&store)[NTOK],
                                                const float (&bias)[EPL], int n_experts,
                                                int top_k, int mode, float rsf,
                                                int32_t* const (&top_idx_row)[NTOK],
                                                float* const (&gates_row)[NTOK]) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  constexpr int32_t kDead = INT32_MIN;
  float val[NTOK][EPL];  // value the gate is built from: sigmoid score or logit
  int32_t key[NTOK][EPL];
  uint64_t dead[NTOK][EPL];  // lanes whose entry j is retired or past n_experts (uniform)
#pragma unroll
  for (int q = 0; q < NTOK; ++q)
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int e = lane + 64 * j;
      float kf = logit[q][j];
      if (mode == HMOE_ROUTE_SIGMOID_BIAS) {
        const float sg = sigmoid_det(logit[q][j]);
        val[q][j] = sg;
        kf = sg + bias[j];
      } else {
        val[q][j] = logit[q][j];
      }
      key[q][j] = e < n_experts ? total_order_key(kf) : kDead;
      dead[q][j] = __builtin_amdgcn_ballot_w64(e >= n_experts);
    }
  int my_e[NTOK];
  float my_v[NTOK], denom[NTOK], vmax[NTOK];
#pragma unroll
  for (int q = 0; q < NTOK; ++q) {
    my_e[q] = 0;
    my_v[q] = 0.0f;
    denom[q] = 0.0f;
    vmax[q] = 0.0f;
  }
  for (int k = 0; k < top_k; ++k) {
    int32_t best[NTOK];
#pragma unroll
    for (int q = 0; q < NTOK; ++q) {
      best[q] = key[q][0];
#pragma unroll
      for (int j = 1; j < EPL; ++j) best[q] = key[q][j] > best[q] ? key[q][j] : best[q];
    }
    wave_max_i32<NTOK>(best);
#pragma unroll
    for (int q = 0; q < NTOK; ++q) {
      uint64_t mask = 0;
      int jw = 0;
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        const uint64_t mj = __builtin_amdgcn_ballot_w64(key[q][j] == best[q]) & ~dead[q][j];
        if (mask == 0 && mj != 0) {
          mask = mj;
          jw = j;
        }
      }
      // mask is non-empty: top_k <= n_experts keeps a live entry at the maximum
      const int lw = __builtin_ctzll(mask);
      float v_win = 0.0f;
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        if (j == jw) {
          v_win = lane_bcast(val[q][j], lw);
          if (lane == lw) key[q][j] = kDead;
          dead[q][j] |= 1ull << lw;
        }
      }
      if (lane == k) {
        my_e[q] = lw + 64 * jw;
        my_v[q] = v_win;
      }
      if (mode == HMOE_ROUTE_SIGMOID_BIAS) denom[q] = denom[q] + v_win;
      else if (k == 0) vmax[q] = v_win;
    }
  }
#pragma unroll
  for (int q = 0; q < NTOK; ++q) {
    float w;
    if (mode == HMOE_ROUTE_SIGMOID_BIAS) {
      w = (my_v[q] / (denom[q] + 1e-9f)) * rsf;
    } else {
      // exp of each slot in its lane, summed in k order
      const float ex = exp_det(my_v[q] - vmax[q]);
      for (int k = 0; k < top_k; ++k) denom[q] = denom[q] + lane_bcast(ex, k);
      w = ex / denom[q];
    }
    if (store[q] && lane < top_k) {
      top_idx_row[q][lane] = my_e[q];
      gates_row[q][lane] = w;
    }
  }
}

// One stage of a max over each aligned group of 8 lanes of a (64-bit key,
// value) pair: the pair of the lane the DPP control CTRL names replaces this
// lane's if its key is larger.  quad_perm [1,0,3,2], then [2,3,0,1], then
// row_half_mirror leave the group's largest pair in all 8 lanes.
template <int CTRL>
__device__ __forceinline__ void dpp_max_kv(int64_t& k, float& v) {
  const int32_t lo = __builtin_amdgcn_mov_dpp(static_cast<int32_t>(k), CTRL, 0xF, 0xF, false);
  const int32_t hi = __builtin_amdgcn_mov_dpp(static_cast<int32_t>(k >> 32), CTRL, 0xF, 0xF, false);
  const int32_t vv = __builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, false);
  const int64_t t = static_cast<int64_t>((static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) |
                                         static_cast<uint32_t>(lo));
  if (t > k) {
    k = t;
    v = __int_as_float(vv);
  }
}

// Selection + gates for 8 tokens per wave: lane group g = lane / 8 takes one
// token, lane p = lane % 8 of the group its experts p*E .. p*E + E - 1.  Every
// entry is a 64-bit composite, the totalOrder key in the high bits above
// 0xFFFF - expert, so the larger composite is the larger key and on equal
// keys the lower expert (the lax.top_k order); retired entries and those past
// n_experts hold INT64_MIN, below every live one.  Round k: each lane's
// largest entry, then the group's largest (three DPP stages, carrying the
// entry's value); the lane that holds it retires it.  Lane p records slots
// p, p + 8, p + 16, p + 24; the gate denominators are summed in k order.
template <int E>
__device__ __forceinline__ void select_group8(const float (&logit)[E], bool store,
                                              const float (&bias)[E], int n_experts,
                                              int top_k, int mode, float rsf,
                                              int32_t* __restrict__ top_idx_row,
                                              float* __restrict__ gates_row) {
#pragma clang fp contract(off)
  const int p = threadIdx.x & 7;
  constexpr int64_t kGone = INT64_MIN;
  int64_t ck[E];
  float val[E];  // value the gate is built from: sigmoid score or logit
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int e = p * E + j;
    float kf = logit[j];
    if (mode == HMOE_ROUTE_SIGMOID_BIAS) {
      const float sg = sigmoid_det(logit[j]);
      val[j] = sg;
      kf = sg + bias[j];
    } else {
      val[j] = logit[j];
    }
    const uint64_t key = static_cast<uint64_t>(static_cast<int64_t>(total_order_key(kf)));
    ck[j] = e < n_experts ? static_cast<int64_t>((key << 16) | static_cast<uint64_t>(0xFFFF - e)) : kGone;
  }
  int my_e[4] = {0, 0, 0, 0};
  float my_v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  float denom = 0.0f, vmax = 0.0f;
  for (int k = 0; k < top_k; ++k) {
    int64_t best = ck[0];
    float bv = val[0];
    int barg = 0;
#pragma unroll
    for (int j = 1; j < E; ++j) {
      if (ck[j] > best) {
        best = ck[j];
        bv = val[j];
        barg = j;
      }
    }
    int64_t gb = best;
    float gv = bv;
    dpp_max_kv<0xB1>(gb, gv);
    dpp_max_kv<0x4E>(gb, gv);
    dpp_max_kv<0x141>(gb, gv);
    // composites are unique, so exactly one lane of the group holds gb
    const bool owner = gb == best;
#pragma unroll
    for (int j = 0; j < E; ++j)
      if (owner && barg == j) ck[j] = kGone;
    const int w = 0xFFFF - static_cast<int>(gb & 0xFFFF);
    float rec = gv;
    if (mode == HMOE_ROUTE_SIGMOID_BIAS) {
      denom = denom + gv;
    } else {
      if (k == 0) vmax = gv;
      rec = exp_det(gv - vmax);
      denom = denom + rec;
    }
    if ((k & 7) == p) {
      const int r = k >> 3;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q == r) {
          my_e[q] = w;
          my_v[q] = rec;
        }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = 8 * q + p;
    if (store && k < top_k) {
      top_idx_row[k] = my_e[q];
      gates_row[k] = mode == HMOE_ROUTE_SIGMOID_BIAS ? (my_v[q] / (denom + 1e-9f)) * rsf
                                                     : my_v[q] / denom;
    }
  }
}

// Eight consecutive activations as raw bits (one or two 16-byte loads; the
// address must be 16-byte aligned), widened to float32 later.
template <typename XT>
struct X8;
template <>
struct X8<float> {
  f32x4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const f32x4*>(p);
    b = *reinterpret_cast<const f32x4*>(p + 4);
  }
  __device__ __forceinline__ float get(int i) const { return i < 4 ? a[i] : b[i - 4]; }
};
template <>
struct X8<uint16_t> {
  u32x4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const u32x4*>(p); }
  __device__ __forceinline__ float get(int i) const {
    const uint32_t u = v[i >> 1];
    return __uint_as_float((i & 1) ? (u & 0xffff0000u) : (u << 16));
  }
};
// Rows n_waves block .. + n_waves of x to e4m3, one per wave.
template <typename XT>
__device__ __forceinline__ void router_quant_rows(const XT* __restrict__ x, int block, int n_waves,
                                                  int64_t tokens, int d_model,
                                                  uint8_t* __restrict__ x_q,
                                                  float* __restrict__ x_scale) {
  static_assert(sizeof(XT) == 2, "x is quantised from bf16");
  const int64_t r = static_cast<int64_t>(block) * n_waves + (threadIdx.x >> 6);
  if (r >= tokens) return;
  const uint16_t* xr = reinterpret_cast<const uint16_t*>(x) + r * d_model;
  if (d_model <= 64 * kRowRegs * 8)
    quant_row_e4m3<true>(xr, d_model, x_q + r * d_model, x_scale + r);
  else
    quant_row_e4m3<false>(xr, d_model, x_q + r * d_model, x_scale + r);
}

// Selection of a workgroup's n_tok tokens (t0 ..) from their logits in LDS
// ([token][NP]), eight tokens per wave (lane group lane / 8 one token, lane p
// of it experts p NP / 8 ..); the logits go to memory on the way.
template <int NP>
__device__ __forceinline__ void router_select8(const float* lg, int n_tok, int wave, int n_waves,
                                               int64_t t0, int64_t tokens, const float (&bv)[NP / 8],
                                               int n_experts, int top_k, int mode, float rsf,
                                               float* __restrict__ logits,
                                               int32_t* __restrict__ top_idx,
                                               float* __restrict__ gates) {
  constexpr int kE8 = NP / 8;
  const int lane = threadIdx.x & 63;
  const int p8 = lane & 7;
#pragma unroll 1
  for (int i = wave * 8; i < n_tok; i += n_waves * 8) {
    if (t0 + i >= tokens) break;
    const int row = i + (lane >> 3);
    const int64_t tok = t0 + row;
    const bool st = row < n_tok && tok < tokens;
    const int64_t tq = st ? tok : tokens - 1;
    float l[kE8];
#pragma unroll
    for (int j = 0; j < kE8; ++j) {
      const int e = p8 * kE8 + j;
      l[j] = st && e < n_experts ? lg[row * NP + e] : 0.0f;
      if (st && e < n_experts) logits[tq * n_experts + e] = l[j];
    }
    select_group8<kE8>(l, st, bv, n_experts, top_k, mode, rsf, top_idx + tq * top_k,
                       gates + tq * top_k);
  }
}

// Logits on the float64 matrix cores.  v_mfma_f64_16x16x4f64 (and its 4 x 4 x
// 4, four-block form) computes D = C + A[:,0]B[0,:] + ... + A[:,3]B[3,:] with
// the additions done one after another in k order, each rounded to float64 (C
// first); the products of bf16/fp32 activations and fp32/bf16 weights are
// exact in float64.  Walking d upwards four at a time from C = +0.0 therefore
// reproduces the sequential d-ascending float64 sum bit for bit.
//
// One wave owns one tile of 16 experts: a single accumulator chain of
// d_model / 4 dependent MFMAs for a group of TOK tokens.  One chain
// alone keeps its SIMD's float64 pipe full (measured: a dependent 16x16x4
// chain issues every 64 cycles, as fast as independent ones; 4x4x4 every 22),
// so the kernel is paced by the chains a SIMD holds and by the float64
// conversions, which share that pipe (8.7 cycles each):
//   * x is widened once per workgroup, when a chunk of it is parked in LDS as
//     float64 ([d][token], so that a wave's operand is 64 consecutive
//     doubles), instead of by every wave for every expert tile;
//   * W goes from global memory straight into the registers of the one wave
//     that owns its columns, a chunk ahead, zeros past d_model.  (Through LDS,
//     by DMA, its reads and those of x together are more than the LDS delivers:
//     29 against 16 us at one token, 64 experts, d_model 2048);
//   * a wave widens the W values of a group of MFMAs before the group: between
//     two MFMAs of the chain a conversion costs 21 cycles (it waits for the
//     first and the second waits for it).
// Operands: A[i][k] in lane i + 16k (16x16x4) or i + 4b + 16k for block b
// (4x4x4), B[k][j] in lane j + 16k (16 columns either way); D[i][j] in lane
// j + 16 (i % 4), register i / 4 (16x16x4), or lane j + 16 i (4x4x4).
// Workgroup barrier that waits for this wave's LDS operations only: the W and
// x loads of the next chunks stay in flight.
__device__ __forceinline__ void barrier_lds_only() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
}

// MFMA steps (of 4 d) per chunk.  Short chains (4 tokens) take 64 where the
// registers allow two chunks of W (32 took 19.4 instead of 16.9 us at one
// token, 64 experts, d_model 2048); 16-token ones 32, whose registers let more
// workgroups share a CU (16384 tokens: 83 against 91 us).
constexpr int router_steps(int mt, int tok) { return tok == 4 && mt <= 8 ? 64 : 32; }

// Waves per expert tile, each with tokens of its own: a workgroup has at least
// four waves, one per SIMD (two-wave workgroups two to a CU shared SIMDs: 79
// against 59 us at 8192 tokens, 32 experts, d_model 4096).
constexpr int router_groups(int mt) { return mt == 1 ? 4 : mt == 2 ? 2 : 1; }

// One W value as loaded, widened exactly.
template <typename WT>
__device__ __forceinline__ uint32_t load_w_bits(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <>
__device__ __forceinline__ uint32_t load_w_bits<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
template <>
__device__ __forceinline__ uint32_t load_w_bits<uint16_t>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
}
template <typename WT>
__device__ __forceinline__ double widen_w(uint32_t bits) {
  return static_cast<double>(__uint_as_float(sizeof(WT) == 4 ? bits : bits << 16));
}

// MT: the most expert tiles of a workgroup; the launch has ceil(n_experts /
// 16), more than MT / 2, and router_groups waves for each.  TOK tokens in a
// chain: 16, or 4 on the 4x4x4 form.
//
// QX: the launch also quantises x to e4m3 per token (the rule and code of
// hmoe_quantize_rows_fp8): workgroups past the first router_blocks take one
// row of x per wave.  They start once the router's workgroups are placed and
// run beside them, whose float64 MFMA chains leave the memory system and most
// of the VALU issue idle.
template <int MT, int TOK, bool TAIL, typename XT, typename WT, bool QX>
__global__ __launch_bounds__(64 * MT * router_groups(MT), MT > 8 || TOK == 16 ? 4 : 2) void router_kernel(
    const XT* __restrict__ x, const WT* __restrict__ w, const float* __restrict__ bias,
    int64_t tokens, int d_model, int n_experts, int top_k, int mode, float rsf,
    float* __restrict__ logits, int32_t* __restrict__ top_idx, float* __restrict__ gates,
    uint8_t* __restrict__ x_q, float* __restrict__ x_scale, int router_blocks) {
  static_assert(TOK == 16 || (TOK == 4 && !TAIL), "a chain holds 16 or 4 tokens");
  static_assert(!QX || sizeof(XT) == 2, "x is quantised from bf16");
  const int n_waves = static_cast<int>(blockDim.x) >> 6;
  if constexpr (QX) {
    if (static_cast<int>(blockIdx.x) >= router_blocks) {
      router_quant_rows(x, static_cast<int>(blockIdx.x) - router_blocks, n_waves, tokens, d_model,
                        x_q, x_scale);
      return;
    }
  }
  constexpr int kRSteps = router_steps(MT, TOK);
  constexpr int kRDc = 4 * kRSteps;                      // d per chunk
  constexpr int kGW = router_groups(MT);                 // waves per expert tile
  constexpr int kTB = TOK * kGW;                         // tokens per workgroup
  constexpr int kNP = 16 * MT;                           // columns of the logit staging
  constexpr int kMinThr = 64 * kGW * (MT == 1 ? 1 : MT / 2 + 1);  // fewest threads of a launch
  constexpr int kXG = kRDc / 8 * kTB;                    // groups of 8 d in a chunk of x
  constexpr int kXR = (kXG + kMinThr - 1) / kMinThr;     // groups per thread
  constexpr int kXBytes = 2 * kRDc * kTB * 8;
  constexpr int kLgBytes = kTB * kNP * 4;
  __shared__ __attribute__((aligned(16))) uint8_t smem[kXBytes > kLgBytes ? kXBytes : kLgBytes];
  // [2][kRDc][kTB]; row d lies at d ^ (d / 8 & kSwz), so that the rows 8 apart
  // which the lanes of one parking write take fall on different banks, while
  // the four rows of an operand read stay within one aligned group of 8
  double* xs = reinterpret_cast<double*>(smem);
  constexpr int kSwz = kTB <= 4 ? 7 : kTB <= 8 ? 3 : kTB <= 16 ? 1 : 0;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int threads = static_cast<int>(blockDim.x);
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kTB;
  const int nchunks = (d_model + kRDc - 1) / kRDc;

  // x: group g = tid + threads r is token g % kTB, d 8 (g / kTB) .. + 8 of the
  // chunk.  d_model is a multiple of 8, so a group is wholly inside or outside
  // a row; loads are unconditional from clamped addresses and masked when
  // parked.
  const XT* xrow[kXR];
  int xd[kXR];
#pragma unroll
  for (int r = 0; r < kXR; ++r) {
    const int g = tid + threads * r;
    const int64_t tok = t0 + g % kTB;
    xrow[r] = x + (tok < tokens ? tok : tokens - 1) * static_cast<int64_t>(d_model);
    xd[r] = g < kXG ? 8 * (g / kTB) : 0;
  }
  X8<XT> xr[kXR];
  auto fetch_x = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kXR; ++r) {
      const int d = c * kRDc + xd[r];
      xr[r].load(xrow[r] + (d < d_model ? d : 0));
    }
  };
  auto park_x = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kXR; ++r) {
      const int g = tid + threads * r;
      const bool ok = c * kRDc + xd[r] < d_model;
      double* dst = xs + (c & 1) * (kRDc * kTB) + g % kTB;
      const int sw = (xd[r] >> 3) & kSwz;
      if (g < kXG) {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          dst[(xd[r] + (q ^ sw)) * kTB] = ok ? static_cast<double>(xr[r].get(q)) : 0.0;
      }
    }
  };
  // W: lane (k, j) reads row 4 s + k, column n of its tile; columns past
  // n_experts repeat the last one (never stored).  The resource of a chunk
  // starts at its first row and ends with the matrix; rows past d_model are
  // zeros from the range check, which is relied on for the vector offset only.
  // Short chains have the step's row there (48 tokens, 64 experts, d_model 2048:
  // 16.7 us, 18.2 with it in the scalar offset).  In long ones that spills
  // registers (4096 tokens: 67 against 33 us), so theirs is the scalar offset:
  // all chunks are full, or (TAIL: d_model is no multiple of the chunk, 35 us) a
  // step past the end has an empty resource.
  const int kl = lane >> 4;
  const int tile = kGW == 1 ? wave : wave / kGW;
  const int tw = kGW == 1 ? 0 : (wave % kGW) * TOK;  // the wave's first token
  int n = tile * 16 + (lane & 15);
  n = n < n_experts ? n : n_experts - 1;
  constexpr int kWB = static_cast<int>(sizeof(WT));
  const int w_voff = (kl * n_experts + n) * kWB;
  const int w_step = 4 * n_experts * kWB;
  struct WChunk {
    const WT* first;
    int bytes, steps, step;  // left of the matrix; bytes from step to step
  };
  auto w_chunk = [&](int c) __attribute__((always_inline)) {
    const bool any = c < nchunks;
    const int64_t left = any ? (static_cast<int64_t>(d_model) - c * kRDc) * n_experts * kWB : 0;
    return WChunk{w + (any ? static_cast<int64_t>(c) * kRDc * n_experts : 0),
                  static_cast<int>(left < 0x7fffffff ? left : 0x7fffffff),
                  any ? (d_model - c * kRDc) / 4 : 0, any || TOK == 4 ? w_step : 0};
  };
  auto load_w = [&](const WChunk& k, int s) __attribute__((always_inline)) {
    const bool in = !TAIL || s < k.steps;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<WT*>(k.first), 0, in ? k.bytes : 0, 0x00020000);
    return TOK == 4 ? load_w_bits<WT>(r, w_voff + s * k.step, 0)
                    : load_w_bits<WT>(r, w_voff, in ? s * k.step : 0);
  };
  uint32_t wr0[kRSteps], wr1[kRSteps];
  {
    const WChunk k0 = w_chunk(0);
#pragma unroll
    for (int s = 0; s < kRSteps; ++s) wr0[s] = load_w(k0, s);
  }
  // the lane's selection biases, long before they are needed
  constexpr int kE8 = kNP / 8, kEPL = (kNP + 63) / 64;
  float bv[MT <= 4 ? kE8 : kEPL];
  load_bias(bv, mode == HMOE_ROUTE_SIGMOID_BIAS ? bias : nullptr, MT <= 4 ? (lane & 7) * kE8 : lane,
            MT <= 4 ? 1 : 64, n_experts);
  fetch_x(0);
  park_x(0);
  if (nchunks > 1) fetch_x(1);
  __syncthreads();

  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  double acc4 = 0.0;
  // operand row 4 s + kl lies at 8 (s / 2) + ((4 (s & 1) + kl) ^ sw), sw = s / 2
  // & kSwz: the lane part kl ^ (sw & 3) by sw & 3
  int a_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) a_off[q] = (kl ^ q) * kTB + tw + (TOK == 16 ? lane & 15 : lane & 3);
  auto a_at = [&](int s) __attribute__((always_inline)) {
    const int sw = (s >> 1) & kSwz;
    return a_off[sw & 3] + (8 * (s >> 1) + ((4 * (s & 1)) ^ (sw & 4))) * kTB;
  };
  // Per group of kRGroup steps: the next group's x operands are read and W
  // values widened, then this group's MFMAs run back to back.  The scheduling
  // barriers keep that order (left free, the compiler hoists every conversion
  // of a chunk, and with it the wait for the chunk's last W load, to the
  // chunk's start).
  constexpr int kRGroup = 4;
  // Chunk c on W registers wc, loading chunk c + 1's into wn.  Two register
  // sets and a pair of chunks per iteration: with one set, refilled in place,
  // the compiler joined the loop with copies that waited for every load.
  auto chunk = [&](const uint32_t (&wc)[kRSteps], uint32_t (&wn)[kRSteps], int c)
      __attribute__((always_inline)) {
    const double* xc = xs + (c & 1) * (kRDc * kTB);
    const WChunk kn = w_chunk(c + 1);
    double ac[kRGroup], an[kRGroup], bc[kRGroup], bn[kRGroup];
    auto operands = [&](int s0, double (&a)[kRGroup], double (&b)[kRGroup])
        __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < kRGroup; ++q) a[q] = xc[a_at(s0 + q)];
#pragma unroll
      for (int q = 0; q < kRGroup; ++q) b[q] = widen_w<WT>(wc[s0 + q]);
    };
    operands(0, ac, bc);
#pragma unroll
    for (int s0 = 0; s0 < kRSteps; s0 += kRGroup) {
#pragma unroll
      for (int q = 0; q < kRGroup; ++q) wn[s0 + q] = load_w(kn, s0 + q);
      if (s0 + kRGroup < kRSteps) operands(s0 + kRGroup, an, bn);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kRGroup; ++q) {
        if constexpr (TOK == 16)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ac[q], bc[q], acc, 0, 0, 0);
        else
          acc4 = __builtin_amdgcn_mfma_f64_4x4x4f64(ac[q], bc[q], acc4, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kRGroup; ++q) {
        bc[q] = bn[q];
        ac[q] = an[q];
      }
    }
    // (parked a part at a time between the MFMA groups instead, its conversions
    // stall the chain: 36 against 29 us at 48 tokens, 64 experts)
    if (c + 1 < nchunks) {
      park_x(c + 1);
      if (c + 2 < nchunks) fetch_x(c + 2);
    }
    barrier_lds_only();
  };
  for (int c = 0; c < nchunks; c += 2) {
    chunk(wr0, wr1, c);
    if (c + 1 >= nchunks) break;  // uniform
    chunk(wr1, wr0, c + 1);
  }

  // float32 logits into LDS, row = token of the workgroup, column = expert
  float* lg = reinterpret_cast<float*>(smem);
  if constexpr (TOK == 16) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      lg[(tw + kl + 4 * r) * kNP + tile * 16 + (lane & 15)] = static_cast<float>(acc[r]);
  } else {
    lg[(tw + kl) * kNP + tile * 16 + (lane & 15)] = static_cast<float>(acc4);
  }
  __syncthreads();

  if constexpr (MT <= 4) {
    router_select8<kNP>(lg, kTB, wave, n_waves, t0, tokens, bv, n_experts, top_k, mode, rsf, logits,
                        top_idx, gates);
  } else {
    // Selection: wave w takes the token pairs w, w + n_waves, ...
#pragma unroll 1
    for (int row = wave * 2; row < kTB; row += n_waves * 2) {
      const int64_t tok = t0 + row;
      if (tok >= tokens) break;
      float l[2][kEPL];
      bool st[2];
      int32_t* ti[2];
      float* gt[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        st[q] = tok + q < tokens;
        const int64_t tq = st[q] ? tok + q : tok;
        ti[q] = top_idx + tq * top_k;
        gt[q] = gates + tq * top_k;
#pragma unroll
        for (int j = 0; j < kEPL; ++j) {
          const int e = lane + 64 * j;
          l[q][j] = e < n_experts ? lg[(row + q) * kNP + e] : 0.0f;
          if (st[q] && e < n_experts) logits[tq * n_experts + e] = l[q][j];
        }
      }
      select_and_gate<kEPL, 2>(l, st, bv, n_experts, top_k, mode, rsf, ti, gt);
    }
  }
}

// NT = 1 or 2 expert tiles and more tokens than short chains fill the chip
// with: x and W staged in LDS as float32 through registers two chunks ahead,
// each wave (one chain) widening both operands.  Here W's rows are so short that
// the direct loads of router_kernel are mostly address work, and several waves
// would load the same ones.  This form against that one, us: 8192 tokens, d_model
// 4096, 32 experts with x's quantisation 59.5 / 69.9 (59.5 / 62.6 alone); d_model
// 2048, 8 experts 36.3 / 47.0, 16384 tokens 37.1 / 48.0; 16 experts, d_model 1024,
// 22.1 / 27.3 (40000 tokens 63.1 / 60.3, the one measured loss); 10 experts (by
// elements), 40000 tokens, d_model 2048 86 / 107.
//
// WV: W is 16-byte aligned and n_experts a multiple of the W elements in 16
// bytes, so a chunk of W is staged with 16-byte loads; else (one tile only: 18
// and 30 experts gain nothing) by elements, in chunks of half the length, whose
// registers would spill.
template <int V>
struct IntC {
  static constexpr int value = V;
};

template <int NT, bool WV>
struct alignas(16) RouterStagedLds {
  static constexpr int kDc = WV ? 128 : 64;  // d per chunk (one barrier per chunk)
  static constexpr int kTB = 64 / NT;        // tokens
  float x[2][kTB][kDc + 4];                  // 16-byte aligned rows
  float w[2][kDc][16 * NT + 8];
};

template <int NT, bool WV, typename XT, typename WT, bool QX>
__global__ __launch_bounds__(256) void router_staged_kernel(
    const XT* __restrict__ x, const WT* __restrict__ w, const float* __restrict__ bias,
    int64_t tokens, int d_model, int n_experts, int top_k, int mode, float rsf,
    float* __restrict__ logits, int32_t* __restrict__ top_idx, float* __restrict__ gates,
    uint8_t* __restrict__ x_q, float* __restrict__ x_scale, int router_blocks) {
  if constexpr (QX) {
    if (static_cast<int>(blockIdx.x) >= router_blocks) {
      router_quant_rows(x, static_cast<int>(blockIdx.x) - router_blocks, 4, tokens, d_model, x_q,
                        x_scale);
      return;
    }
  }
  constexpr int kThr = 256;
  constexpr int kNP = 16 * NT;
  constexpr int kTB = RouterStagedLds<NT, WV>::kTB;
  constexpr int kTG = kTB / 16;                               // token groups
  constexpr int kDc = RouterStagedLds<NT, WV>::kDc;
  constexpr int kE16 = 16 / static_cast<int>(sizeof(WT));     // W elements per 16-byte load
  constexpr int kWV = kDc * kNP / kE16 / kThr;                // 16-byte W loads per thread per chunk
  constexpr int kWPer = kDc * kNP / kThr;                     // W elements per thread per chunk
  __shared__ RouterStagedLds<NT, WV> lds;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int tg = wave % kTG;
  const int ep = wave / kTG;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kTB;

  // Staging assignment: x elements (tt, dd..dd+7) = (g / kXT, (g % kXT) * 8) for
  // the groups g = tid + kThr r < kXT*kTB (kXT = kDc / 8 groups per token
  // row).  d_model is a multiple of 8, so a group of 8 is wholly inside or
  // outside the row.  Every load is unconditional from an
  // in-range address (clamped token row, d or expert 0) and masked
  // afterwards, so the loads of a chunk stay in flight together until they
  // are parked in LDS.
  constexpr int kXT = kDc / 8;
  constexpr int kXR = kXT * kTB / kThr;  // x groups per thread
  int xs_tt[kXR], xs_dd[kXR];
  int64_t xs_row[kXR];
#pragma unroll
  for (int r = 0; r < kXR; ++r) {
    const int g = tid + kThr * r;
    xs_tt[r] = g / kXT;
    xs_dd[r] = (g % kXT) * 8;
    const int64_t tok = t0 + xs_tt[r];
    xs_row[r] = (tok < tokens ? tok : tokens - 1) * static_cast<int64_t>(d_model);
  }
  // Two register sets: the loads of chunk c + 2 are issued at the start of
  // chunk c, so a load has two chunks of MFMAs to arrive before it is parked.
  X8<XT> xr0[kXR], xr1[kXR];
  constexpr int kWRegs = WV ? 4 * kWV : kWPer;
  uint32_t wr0[kWRegs], wr1[kWRegs];
  // Element q of the staging by elements: row idx / kNP, expert idx % kNP, idx =
  // q * kThr + tid.
  auto w_ok = [&](int q, int d0) __attribute__((always_inline)) {
    const int idx = q * kThr + tid;
    return idx % kNP < n_experts && d0 + idx / kNP < d_model;
  };
  // Vector q covers elements idx .. idx + kE16 - 1 (idx = (q*kThr + tid) *
  // kE16) of the chunk, i.e. row idx / n_experts, experts idx % n_experts ...
  auto wv_idx = [&](int q) __attribute__((always_inline)) { return (q * kThr + tid) * kE16; };
  auto fetch = [&](X8<XT>* xr, uint32_t* wr, int d0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kXR; ++r) {
      const int dx = d0 + xs_dd[r];
      xr[r].load(x + xs_row[r] + (dx < d_model ? dx : 0));
    }
    if constexpr (WV) {
#pragma unroll
      for (int q = 0; q < kWV; ++q) {
        const int idx = wv_idx(q);
        const bool ok = idx < kDc * n_experts && d0 + idx / n_experts < d_model;
        const u32x4 v = *reinterpret_cast<const u32x4*>(
            w + (ok ? static_cast<int64_t>(d0) * n_experts + idx : 0));
#pragma unroll
        for (int j = 0; j < 4; ++j) wr[4 * q + j] = v[j];
      }
    } else {
#pragma unroll
      for (int q = 0; q < kWPer; ++q) {
        const int idx = q * kThr + tid;
        const int64_t off = static_cast<int64_t>(d0 + idx / kNP) * n_experts + idx % kNP;
        const WT v = w[w_ok(q, d0) ? off : 0];
        if constexpr (sizeof(WT) == 4)
          wr[q] = __float_as_uint(v);
        else
          wr[q] = static_cast<uint32_t>(v) << 16;
      }
    }
    // Keep the loads ahead of the MFMAs; the masking happens in park().
    __builtin_amdgcn_sched_barrier(0);
  };
  auto park = [&](const X8<XT>* xr, const uint32_t* wr, int buf, int d0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kXR; ++r) {
      const bool x_ok = d0 + xs_dd[r] < d_model;
      f32x4 lo, hi;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        lo[q] = x_ok ? xr[r].get(q) : 0.0f;
        hi[q] = x_ok ? xr[r].get(4 + q) : 0.0f;
      }
      *reinterpret_cast<f32x4*>(&lds.x[buf][xs_tt[r]][xs_dd[r]]) = lo;
      *reinterpret_cast<f32x4*>(&lds.x[buf][xs_tt[r]][xs_dd[r] + 4]) = hi;
    }
    if constexpr (WV) {
#pragma unroll
      for (int q = 0; q < kWV; ++q) {
        const int idx = wv_idx(q);
        if (idx < kDc * n_experts) {
          const int d = idx / n_experts;
          const int n = idx - d * n_experts;
          const bool ok = d0 + d < d_model;
          float* dst = &lds.w[buf][d][n];
          if (sizeof(WT) == 4) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = ok ? __uint_as_float(wr[4 * q + j]) : 0.0f;
            *reinterpret_cast<f32x4*>(dst) = v;
          } else {
            f32x4 lo, hi;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const uint32_t a = wr[4 * q + j], b = wr[4 * q + 2 + j];
              lo[2 * j] = ok ? __uint_as_float(a << 16) : 0.0f;
              lo[2 * j + 1] = ok ? __uint_as_float(a & 0xffff0000u) : 0.0f;
              hi[2 * j] = ok ? __uint_as_float(b << 16) : 0.0f;
              hi[2 * j + 1] = ok ? __uint_as_float(b & 0xffff0000u) : 0.0f;
            }
            *reinterpret_cast<f32x4*>(dst) = lo;
            *reinterpret_cast<f32x4*>(dst + 4) = hi;
          }
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < kWPer; ++q) {
        const int idx = q * kThr + tid;
        lds.w[buf][idx / kNP][idx % kNP] = w_ok(q, d0) ? __uint_as_float(wr[q]) : 0.0f;
      }
    }
  };
  if (WV && n_experts < kNP) {
    // Expert columns past n_experts are never written by the vector staging:
    // zero them once in both buffers.
    for (int i = tid; i < 2 * kDc * kNP; i += kThr) {
      const int n = i % kNP;
      if (n >= n_experts) lds.w[i / (kDc * kNP)][(i / kNP) % kDc][n] = 0.0f;
    }
  }

  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  const int a_row = tg * 16 + (lane & 15);
  const int k_of_lane = lane >> 4;
  const int col0 = ep * 16 + (lane & 15);
  const int nchunks = (d_model + kDc - 1) / kDc;
  // Chunk c (S = c % 2): prefetch chunk c + 2 into register set S, run the
  // MFMAs on LDS buffer S, park chunk c + 1 (register set S ^ 1) into buffer
  // S ^ 1.
  auto chunk = [&](auto Sc, int c) __attribute__((always_inline)) {
    constexpr int S = decltype(Sc)::value;
    X8<XT>* xs_ld = S == 0 ? xr0 : xr1;
    uint32_t* ws_ld = S == 0 ? wr0 : wr1;
    const X8<XT>* xs_pk = S == 0 ? xr1 : xr0;
    const uint32_t* ws_pk = S == 0 ? wr1 : wr0;
    if (c + 2 < nchunks) fetch(xs_ld, ws_ld, (c + 2) * kDc);
#pragma unroll
    for (int s = 0; s < kDc / 4; ++s) {
      const double a = static_cast<double>(lds.x[S][a_row][4 * s + k_of_lane]);
      const double b = static_cast<double>(lds.w[S][4 * s + k_of_lane][col0]);
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
    if (c + 1 < nchunks) park(xs_pk, ws_pk, S ^ 1, (c + 1) * kDc);
    __syncthreads();
  };
  fetch(xr0, wr0, 0);
  if (nchunks > 1) fetch(xr1, wr1, kDc);
  park(xr0, wr0, 0, 0);
  __syncthreads();
  for (int c = 0; c < nchunks; c += 2) {
    chunk(IntC<0>{}, c);
    if (c + 1 < nchunks) chunk(IntC<1>{}, c + 1);
  }

  // float32 logits into LDS, row = token of the workgroup, column = expert
  float* lg = &lds.w[0][0][0];
  static_assert(sizeof(float) * kTB * kNP <= sizeof(lds.w), "logit staging does not fit");
#pragma unroll
  for (int r = 0; r < 4; ++r) lg[(tg * 16 + k_of_lane + 4 * r) * kNP + col0] = static_cast<float>(acc[r]);
  __syncthreads();
  float bv[kNP / 8];
  load_bias(bv, mode == HMOE_ROUTE_SIGMOID_BIAS ? bias : nullptr, (lane & 7) * (kNP / 8), 1, n_experts);
  router_select8<kNP>(lg, kTB, wave, 4, t0, tokens, bv, n_experts, top_k, mode, rsf, logits,
                      top_idx, gates);
}

// One wave per token: selection and gates from given logits.
// Tokens per wave (their reduction chains would interleave); one measured
// fastest once the reductions moved off the LDS permutes (4: 24.5 against
// 22.8 us at 32768 tokens, 64 experts, top-8).
constexpr int kSelTok = 1;

template <int EPL>
__global__ __launch_bounds__(256) void select_kernel(const float* __restrict__ logits,
                                                     const float* __restrict__ bias, int64_t tokens,
                                                     int n_experts, int top_k, int mode, float rsf,
                                                     int32_t* __restrict__ top_idx,
                                                     float* __restrict__ gates) {
  const int lane = threadIdx.x & 63;
  const int64_t tok0 = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * kSelTok;
  if (tok0 >= tokens) return;
  float bv[EPL];
  load_bias(bv, mode == HMOE_ROUTE_SIGMOID_BIAS ? bias : nullptr, lane, 64, n_experts);
  float l[kSelTok][EPL];
  bool st[kSelTok];
  int32_t* ti[kSelTok];
  float* gt[kSelTok];
#pragma unroll
  for (int q = 0; q < kSelTok; ++q) {
    st[q] = tok0 + q < tokens;
    const int64_t tq = st[q] ? tok0 + q : tok0;  // a token past the end repeats the first
    ti[q] = top_idx + tq * top_k;
    gt[q] = gates + tq * top_k;
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int e = lane + 64 * j;
      l[q][j] = e < n_experts ? logits[tq * n_experts + e] : 0.0f;
    }
  }
  select_and_gate<EPL, kSelTok>(l, st, bv, n_experts, top_k, mode, rsf, ti, gt);
}

// Selection and gates from given logits for up to 64 experts, eight tokens
// per wave (lane group lane / 8 one token, lane p its experts 8p .. 8p + 7).
__global__ __launch_bounds__(256) void select_kernel_g8(const float* __restrict__ logits,
                                                        const float* __restrict__ bias,
                                                        int64_t tokens, int n_experts, int top_k,
                                                        int mode, float rsf,
                                                        int32_t* __restrict__ top_idx,
                                                        float* __restrict__ gates) {
  const int lane = threadIdx.x & 63;
  const int p = lane & 7;
  const int64_t tok0 = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * 8;
  if (tok0 >= tokens) return;  // uniform per wave
  const int64_t tok = tok0 + (lane >> 3);
  const bool st = tok < tokens;
  const int64_t tq = st ? tok : tokens - 1;
  float bv[8];
  load_bias(bv, mode == HMOE_ROUTE_SIGMOID_BIAS ? bias : nullptr, p * 8, 1, n_experts);
  float l[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int e = p * 8 + j;
    l[j] = e < n_experts ? logits[tq * n_experts + e] : 0.0f;
  }
  select_group8<8>(l, st, bv, n_experts, top_k, mode, rsf, top_idx + tq * top_k,
                   gates + tq * top_k);
}

// CU count of the stream's device (0 if it cannot be queried), cached per device.
int stream_cus(hipStream_t s) {
  int dev = 0;
  if (hipStreamGetDevice(s, &dev) != hipSuccess && hipGetDevice(&dev) != hipSuccess) return 0;
  static std::atomic<int> cached[64];
  int cus = dev >= 0 && dev < 64 ? cached[dev].load(std::memory_order_relaxed) : 0;
  if (cus == 0 && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
      cus > 0 && dev >= 0 && dev < 64)
    cached[dev].store(cus, std::memory_order_relaxed);
  return cus > 0 ? cus : 0;
}

// Optional e4m3 quantisation of x in the router's launch (router_kernel QX).
struct XQuant {
  uint8_t* q = nullptr;
  float* scale = nullptr;
};

template <int MT, int TOK, bool TAIL, typename XT, typename WT>
void launch_router_tok(const void* x, const void* w, const float* bias, int64_t tokens,
                       int d_model, int n_experts, int top_k, int mode, float rsf, float* logits,
                       int32_t* top_idx, float* gates, hipStream_t stream, XQuant xq) {
  const int waves = (n_experts + 15) / 16 * router_groups(MT);
  const int rblocks = static_cast<int>(ceil_div(tokens, TOK * router_groups(MT)));
  if constexpr (sizeof(XT) == 2) {
    if (xq.q != nullptr) {
      hipLaunchKernelGGL((router_kernel<MT, TOK, TAIL, XT, WT, true>),
                         dim3(static_cast<unsigned>(rblocks + ceil_div(tokens, waves))),
                         dim3(64 * waves), 0, stream, static_cast<const XT*>(x),
                         static_cast<const WT*>(w), bias, tokens, d_model, n_experts, top_k, mode,
                         rsf, logits, top_idx, gates, xq.q, xq.scale, rblocks);
      return;
    }
  }
  hipLaunchKernelGGL((router_kernel<MT, TOK, TAIL, XT, WT, false>), dim3(static_cast<unsigned>(rblocks)),
                     dim3(64 * waves), 0, stream, static_cast<const XT*>(x),
                     static_cast<const WT*>(w), bias, tokens, d_model, n_experts, top_k, mode, rsf,
                     logits, top_idx, gates, nullptr, nullptr, rblocks);
}

template <int NT, bool WV, typename XT, typename WT>
void launch_router_staged(const void* x, const void* w, const float* bias, int64_t tokens,
                          int d_model, int n_experts, int top_k, int mode, float rsf,
                          float* logits, int32_t* top_idx, float* gates, hipStream_t stream,
                          XQuant xq) {
  const int rblocks = static_cast<int>(ceil_div(tokens, RouterStagedLds<NT, WV>::kTB));
  if constexpr (sizeof(XT) == 2) {
    if (xq.q != nullptr) {
      hipLaunchKernelGGL((router_staged_kernel<NT, WV, XT, WT, true>),
                         dim3(static_cast<unsigned>(rblocks + ceil_div(tokens, 4))), dim3(256), 0,
                         stream, static_cast<const XT*>(x), static_cast<const WT*>(w), bias, tokens,
                         d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, xq.q,
                         xq.scale, rblocks);
      return;
    }
  }
  hipLaunchKernelGGL((router_staged_kernel<NT, WV, XT, WT, false>), dim3(static_cast<unsigned>(rblocks)),
                     dim3(256), 0, stream, static_cast<const XT*>(x), static_cast<const WT*>(w),
                     bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates,
                     nullptr, nullptr, rblocks);
}

// Chains of 4 tokens while they leave at most 1.5 waves per SIMD: they are
// three times as fast a chain as those of 16 (d_model / 4 MFMAs of 22 instead
// of 64 cycles) but do half the work per cycle of the float64 pipe.  Measured
// at d_model 2048, 64 experts: 1000 tokens 17.5 against 30.3 us, 2048 26.8 /
// 30.4, 4096 48 / 32; 32 experts (d_model 4096), 2000 tokens: 27 / 59.  A device
// whose CU count cannot be read takes 16.
template <int MT, typename XT, typename WT>
void launch_router(const void* x, const void* w, const float* bias, int64_t tokens, int d_model,
                   int n_experts, int top_k, int mode, float rsf, float* logits, int32_t* top_idx,
                   float* gates, hipStream_t stream, XQuant xq) {
  const int waves = (n_experts + 15) / 16 * router_groups(MT);
  if (ceil_div(tokens, 4 * router_groups(MT)) * waves <= int64_t(6) * stream_cus(stream)) {
    launch_router_tok<MT, 4, false, XT, WT>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf,
                                            logits, top_idx, gates, stream, xq);
    return;
  }
  const bool wv = n_experts % (16 / static_cast<int>(sizeof(WT))) == 0 &&
                  reinterpret_cast<uintptr_t>(w) % 16 == 0;
  if constexpr (MT <= 2) {
    if (wv) {
      launch_router_staged<MT, true, XT, WT>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf,
                                             logits, top_idx, gates, stream, xq);
      return;
    }
  }
  if constexpr (MT == 1) {
    launch_router_staged<1, false, XT, WT>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf,
                                           logits, top_idx, gates, stream, xq);
  } else if (d_model % (4 * router_steps(MT, 16)) == 0) {
    launch_router_tok<MT, 16, false, XT, WT>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf,
                                             logits, top_idx, gates, stream, xq);
  } else {
    launch_router_tok<MT, 16, true, XT, WT>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf,
                                            logits, top_idx, gates, stream, xq);
  }
}

template <int MT>
void dispatch_router(int x_dtype, int w_dtype, const void* x, const void* w, const float* bias,
                     int64_t tokens, int d_model, int n_experts, int top_k, int mode, float rsf,
                     float* logits, int32_t* top_idx, float* gates, hipStream_t s,
                     XQuant xq = XQuant()) {
  if (x_dtype == HMOE_BF16 && w_dtype == HMOE_F32)
    launch_router<MT, uint16_t, float>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else if (x_dtype == HMOE_F32 && w_dtype == HMOE_F32)
    launch_router<MT, float, float>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else if (x_dtype == HMOE_BF16 && w_dtype == HMOE_BF16)
    launch_router<MT, uint16_t, uint16_t>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else
    launch_router<MT, float, uint16_t>(x, w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
}

int validate_routing(int64_t tokens, int n_experts, int top_k, int mode) {
  HMOE_REQUIRE(tokens >= 0, "router: tokens must be >= 0 (got %lld)", (long long)tokens);
  HMOE_REQUIRE(n_experts >= 1 && n_experts <= 256, "router: n_experts must be in [1, 256] (got %d)",
               n_experts);
  HMOE_REQUIRE(top_k >= 1 && top_k <= n_experts && top_k <= 32,
               "router: top_k must be in [1, min(n_experts, 32)] (got %d, n_experts %d)", top_k,
               n_experts);
  HMOE_REQUIRE(mode == HMOE_ROUTE_SIGMOID_BIAS || mode == HMOE_ROUTE_SOFTMAX,
               "router: unknown routing mode %d", mode);
  return HMOE_OK;
}

}  // namespace
}  // namespace hmoe

extern "C" int hmoe_router(const void* x, int x_dtype, const void* router_w, int w_dtype,
                           const float* bias, int64_t tokens, int d_model, int n_experts,
                           int top_k, int mode, float routed_scaling_factor, float* logits,
                           int32_t* top_idx, float* gates, hmoe_stream_t stream) {
  using namespace hmoe;
  if (int rc = validate_routing(tokens, n_experts, top_k, mode)) return rc;
  HMOE_REQUIRE(d_model >= 8 && d_model % 8 == 0,
               "router: d_model must be a positive multiple of 8 (got %d)", d_model);
  HMOE_REQUIRE(x_dtype == HMOE_F32 || x_dtype == HMOE_BF16, "router: x dtype must be F32 or BF16");
  HMOE_REQUIRE(w_dtype == HMOE_F32 || w_dtype == HMOE_BF16, "router: weight dtype must be F32 or BF16");
  if (tokens == 0) return HMOE_OK;
  HMOE_REQUIRE(x && router_w && logits && top_idx && gates, "router: null pointer argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float rsf = routed_scaling_factor;
  if (n_experts <= 16)
    dispatch_router<1>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s);
  else if (n_experts <= 32)
    dispatch_router<2>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s);
  else if (n_experts <= 64)
    dispatch_router<4>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s);
  else if (n_experts <= 128)
    dispatch_router<8>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s);
  else
    dispatch_router<16>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s);
  return check_launch("hmoe_router");
}

extern "C" int hmoe_router_quant_fp8(const void* x, int x_dtype, const void* router_w, int w_dtype,
                                     const float* bias, int64_t tokens, int d_model, int n_experts,
                                     int top_k, int mode, float routed_scaling_factor,
                                     float* logits, int32_t* top_idx, float* gates, uint8_t* x_q,
                                     float* x_scale, hmoe_stream_t stream) {
  using namespace hmoe;
  if (int rc = validate_routing(tokens, n_experts, top_k, mode)) return rc;
  HMOE_REQUIRE(d_model >= 8 && d_model % 8 == 0,
               "router_quant_fp8: d_model must be a positive multiple of 8 (got %d)", d_model);
  HMOE_REQUIRE(x_dtype == HMOE_BF16, "router_quant_fp8: x dtype must be BF16");
  HMOE_REQUIRE(w_dtype == HMOE_F32 || w_dtype == HMOE_BF16,
               "router_quant_fp8: weight dtype must be F32 or BF16");
  if (tokens == 0) return HMOE_OK;
  HMOE_REQUIRE(x && router_w && logits && top_idx && gates && x_q && x_scale,
               "router_quant_fp8: null pointer argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float rsf = routed_scaling_factor;
  XQuant xq;
  xq.q = x_q;
  xq.scale = x_scale;
  if (n_experts <= 16)
    dispatch_router<1>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else if (n_experts <= 32)
    dispatch_router<2>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else if (n_experts <= 64)
    dispatch_router<4>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else if (n_experts <= 128)
    dispatch_router<8>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  else
    dispatch_router<16>(x_dtype, w_dtype, x, router_w, bias, tokens, d_model, n_experts, top_k, mode, rsf, logits, top_idx, gates, s, xq);
  return check_launch("hmoe_router_quant_fp8");
}

extern "C" int hmoe_router_from_logits(const float* logits, const float* bias, int64_t tokens,
                                       int n_experts, int top_k, int mode,
                                       float routed_scaling_factor, int32_t* top_idx,
                                       float* gates, hmoe_stream_t stream) {
  using namespace hmoe;
  if (int rc = validate_routing(tokens, n_experts, top_k, mode)) return rc;
  if (tokens == 0) return HMOE_OK;
  HMOE_REQUIRE(logits && top_idx && gates, "router_from_logits: null pointer argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(ceil_div(tokens, 4 * kSelTok)));
  if (n_experts <= 64)
    hipLaunchKernelGGL(select_kernel_g8, dim3(static_cast<unsigned>(ceil_div(tokens, 32))), dim3(256), 0, s,
                       logits, bias, tokens, n_experts, top_k, mode, routed_scaling_factor, top_idx, gates);
  else if (n_experts <= 128)
    hipLaunchKernelGGL(select_kernel<2>, grid, dim3(256), 0, s, logits, bias, tokens, n_experts, top_k, mode, routed_scaling_factor, top_idx, gates);
  else
    hipLaunchKernelGGL(select_kernel<4>, grid, dim3(256), 0, s, logits, bias, tokens, n_experts, top_k, mode, routed_scaling_factor, top_idx, gates);
  return check_launch("hmoe_router_from_logits");
}
