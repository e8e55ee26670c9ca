// gemv.hip -- fused weight-dequant x fp16 decode GEMM for gfx950 (ti_gemm_wq_a16).
//
// Replaces the decode projections of the reference: TensorEngine::matmul ->
// matmul_3d_2d (src/core/tensor_engine.cpp:594-640, scalar fp32, one core) with the
// int weights' convert_dtype (:2218-2284), plus the neighbouring element-wise ops of
// TransformerLayer::forward (src/model/inference_engine.cpp:203-233, 376-401).
//
// Shape of the work (M <= 16 decode rows, N outputs, K inputs), one launch per projection:
//   * one 8-wave workgroup per CU streams a contiguous run of 16-row tiles; wave w owns
//     k-tiles w, w+8, ... of every tile and keeps R items (1 KiB each for int4) of packed
//     weights in flight as dwordx4 loads straight into VGPRs, refilled R items ahead across
//     tile boundaries (weights are read once: no LDS round trip, cdna_hip_programming.md
//     "GEMV / M <= 16").
//   * everything small the workgroup needs (group scales, the activation rows, the
//     epilogue's residual / position inputs) is loaded BEFORE the weight ring is issued,
//     so waiting for it never drains the ring (vmcnt retires in issue order).
//   * the activation row(s) are staged in LDS as fp16 (rms_norm fused), read back as MFMA
//     A fragments; per item 4 x v_mfma_f32_16x16x32_f16 on (x, dequantized W) then one
//     fp32 FMA by the group scale; int4 nibbles -> fp16 with the 0x6400 magic (exact), int8
//     with v_perm_b32 + the same magic.
//   * the stream loop has no branches and no barriers: each item's running partial is
//     written to its tile's LDS slab (or a dummy slab), so the compiler schedules R items
//     as one block; after the stream the 8 waves' partials are summed in a fixed order
//     (deterministic) and the epilogue (residual add, SiLU*up, RoPE + KV append, logits +
//     argmax) runs on the 16 x M results of each tile.
#include <math.h>
#include <atomic>
#include <stdlib.h>

#include "attention_body.hpp"
#include "gemm_common.hpp"
#include "gemm_wide.hpp"

namespace ti {

#ifndef TI_GEMV_RING_VGPRS
// VGPRs per lane of packed weights in flight.  Deeper is slower: a CU accepts a bounded
// number of outstanding loads, and a wave whose refill cannot issue stalls before its next
// item's math (tools/probe_gemv.hip sweep: 16-24 best, 64 costs ~15 %).
#define TI_GEMV_RING_VGPRS 20
#endif
#ifndef TI_GEMV_SYNC
#define TI_GEMV_SYNC 0   // blocks of R items between workgroup barriers in the stream (0 = none)
#endif
#ifndef TI_GEMV_RING_DELAY
#define TI_GEMV_RING_DELAY 0
#endif
#if TI_GEMV_EXP & 4   // diagnostic: per-workgroup phase timestamps (s_memrealtime, 100 MHz)
__device__ unsigned long long g_gemv_ts[4096 * 8];
#define GEMV_TS(k) \
  do { if (threadIdx.x == 0) g_gemv_ts[blockIdx.x * 8 + (k)] = __builtin_amdgcn_s_memrealtime(); } while (0)
__device__ unsigned long long g_gemv_wts[4096 * 8];   // per-wave end of stream
#define GEMV_WTS() \
  do { if ((threadIdx.x & 63) == 0) g_gemv_wts[blockIdx.x * 8 + (threadIdx.x >> 6)] = __builtin_amdgcn_s_memrealtime(); } while (0)
__device__ unsigned long long g_rows_ts[4096 * 8 * 8];   // [wg][wave][phase] (gemm_rows_kernel)
#define ROWS_TS(k)                                                                                     \
  do {                                                                                                 \
    if ((threadIdx.x & 63) == 0)                                                                       \
      g_rows_ts[(blockIdx.x * 8 + (threadIdx.x >> 6)) * 8 + (k)] = __builtin_amdgcn_s_memrealtime();   \
  } while (0)
#else
#define GEMV_WTS() do { } while (0)
#define GEMV_TS(k) do { } while (0)
#define ROWS_TS(k) do { } while (0)
#endif

// Workgroups per launch: one 8-wave workgroup per CU (a second workgroup per CU measured slower),
// never more than there are 16-row tiles.

__host__ __device__ inline int gemv_lds_bytes_tiles(int M, int K, int tiles_per_wg, bool g32 = false, bool aff = false);

// Tiles per workgroup are bounded by the LDS image (partial slabs and scales grow with
// them): very wide outputs (a 128k vocabulary) get more workgroups than CUs.
__host__ inline int gemv_grid(int M, int N, int K, int num_cus, bool g32 = false, bool aff = false) {
  const int NT = N >> 4;
  const int g = num_cus > 0 ? num_cus : 256;
  int grid = NT < g ? NT : g;
  while (grid < NT && gemv_lds_bytes_tiles(M, K, (NT + grid - 1) / grid, g32, aff) > 160 * 1024) grid += grid / 8 + 1;
  return grid < NT ? grid : NT;
}

// LDS image of one workgroup (bytes, each region 16-aligned):
//   x      [M][K + 8] fp16            activation rows (row pad breaks bank aliasing)
//   scales [ntl][K/128][16] fp16      group scales of the workgroup's tiles ([ntl][K/128][4][16]
//                                     with group-32 weights, TI_BITS_G32)
//   corr   [K/128][16] f32            int4: per (group, row) offset correction (see deq_int4_raw)
//                                     ([K/32][16] with group-32 weights)
//   slab   [ntl + 1][8][64] f32x4     per-wave partial tiles (+ one dummy slab)
//   es     epilogue inputs: residual [ntl][M][16] f32 (+ the fold weights of the same
//          outputs, TI_EPI_RESID_F32 with fold_x), or RoPE (cos, sin) [M][hd] + pos [M]
//   best   [16] u64                   argmax keys of the workgroup
//   (affine group-32, TI_BITS_AFF: + the block minimums [ntl][K/128][4][16] fp16 after the scales
//    and the blocks' sums of x [K/32][16] f32 after corr)
struct GemvLds {
  int x, sc, corr, slab, es, best, total, mins, bsum;
};
__host__ __device__ inline GemvLds gemv_lds_layout(int M, int K, int ntl, bool g32 = false, bool aff = false) {
  GemvLds l;
  const int gm = g32 ? 4 : 1;                  // scale / correction groups per 128 k
  l.x = 0;
  l.sc = l.x + align16(M * (K + 8) * 2);
  l.mins = l.sc + align16(ntl * (K >> 7) * 32 * gm);
  l.corr = l.mins + (aff ? align16(ntl * (K >> 7) * 32 * gm) : 0);
  l.bsum = l.corr + (K >> 7) * 16 * 4 * gm;
  l.slab = l.bsum + (aff ? (K >> 7) * 16 * 4 * gm : 0);   // int4 offset correction [K/128 (x4)][16 rows] f32
  l.es = l.slab + (ntl + 1) * kGemvWaves * kWave * 16;
  const int es_bytes = 2 * ntl * M * 16 * 4 > M * 128 * 4 + 64 ? 2 * ntl * M * 16 * 4 : M * 128 * 4 + 64;
  l.best = l.es + align16(es_bytes);
  l.total = l.best + 16 * 8;
  return l;
}
__host__ __device__ inline int gemv_lds_bytes_tiles(int M, int K, int tiles_per_wg, bool g32, bool aff) {
  return gemv_lds_layout(M, K, tiles_per_wg, g32, aff).total;
}

// ------------------------------------------------------------- x staging (LDS)
// x staging modes (chosen on the host): fp16 rows prefetched into registers; fp32 rows;
// rms_norm of ONE row of K <= 4096 held in registers; rms_norm of several / longer rows.
// XM_F16F: fp16 rows of h * nw (TI_X_F16_FOLDED, one row) staged like XM_F16; the rms comes
// from the producer's partial sums of squares and divides the outputs before the epilogue.
// XM_ATTN: the attention's split partials (TI_X_ATTN_SPLITS, one row), merged while staging.
enum { XM_F16 = 0, XM_F32 = 1, XM_NORM1 = 2, XM_NORM = 3, XM_F16F = 4, XM_ATTN = 5 };

// Generic staging (M > 1 with rms_norm, f32 rows, or rows longer than the register
// prefetch covers).  Runs after the ring is issued, so its loads wait behind the ring.
template <int XM>
__device__ __forceinline__ void stage_x_generic(const GemvArgs& a, f16* xl, float* red, int k8_from) {
  const int tid = threadIdx.x, K = a.K, xs = K + 8, K8 = K >> 3;
  if constexpr (XM == XM_NORM || XM == XM_NORM1) {
    // rms_norm (tensor_engine.cpp:1488-1505): y = (x / sqrt(sum(x^2)/K + eps)) * w.
    for (int m = 0; m < a.M; ++m) {
      const float* xr = (const float*)a.x + (size_t)m * a.ldx;
      float ss = 0.0f;
      for (int k8 = tid; k8 < K8; k8 += kGemvThreads) {
        const float4 v0 = *(const float4*)(xr + 8 * k8), v1 = *(const float4*)(xr + 8 * k8 + 4);
        ss = fmaf(v0.x, v0.x, ss); ss = fmaf(v0.y, v0.y, ss); ss = fmaf(v0.z, v0.z, ss); ss = fmaf(v0.w, v0.w, ss);
        ss = fmaf(v1.x, v1.x, ss); ss = fmaf(v1.y, v1.y, ss); ss = fmaf(v1.z, v1.z, ss); ss = fmaf(v1.w, v1.w, ss);
      }
      ss = group_sum<kWave>(ss);
      if ((tid & 63) == 0) red[tid >> 6] = ss;
      __syncthreads();
      float tot = 0.0f;
#pragma unroll
      for (int w = 0; w < kGemvWaves; ++w) tot += red[w];
      const float rms = sqrtf(tot / (float)K + a.eps);
      for (int k8 = tid; k8 < K8; k8 += kGemvThreads) {
        const float4 v0 = *(const float4*)(xr + 8 * k8), v1 = *(const float4*)(xr + 8 * k8 + 4);
        const float4 w0 = *(const float4*)(a.norm_w + 8 * k8), w1 = *(const float4*)(a.norm_w + 8 * k8 + 4);
        f16x8 h;
        h[0] = mul_f16(v0.x / rms, w0.x); h[1] = mul_f16(v0.y / rms, w0.y);
        h[2] = mul_f16(v0.z / rms, w0.z); h[3] = mul_f16(v0.w / rms, w0.w);
        h[4] = mul_f16(v1.x / rms, w1.x); h[5] = mul_f16(v1.y / rms, w1.y);
        h[6] = mul_f16(v1.z / rms, w1.z); h[7] = mul_f16(v1.w / rms, w1.w);
        *(f16x8*)(xl + m * xs + 8 * k8) = h;
      }
      __syncthreads();   // red reused by the next row
    }
  } else if constexpr (XM == XM_F32) {
    for (int i = tid; i < a.M * K8; i += kGemvThreads) {
      const int m = i / K8, k8 = i - m * K8;
      const float* xr = (const float*)a.x + (size_t)m * a.ldx + 8 * k8;
      const float4 v0 = *(const float4*)xr, v1 = *(const float4*)(xr + 4);
      f16x8 h;
      h[0] = (f16)v0.x; h[1] = (f16)v0.y; h[2] = (f16)v0.z; h[3] = (f16)v0.w;
      h[4] = (f16)v1.x; h[5] = (f16)v1.y; h[6] = (f16)v1.z; h[7] = (f16)v1.w;
      *(f16x8*)(xl + m * xs + 8 * k8) = h;
    }
  } else {
    for (int i = tid + k8_from; i < a.M * K8; i += kGemvThreads) {
      const int m = i / K8, k8 = i - m * K8;
      *(u32x4*)(xl + m * xs + 8 * k8) = *(const u32x4*)((const f16*)a.x + (size_t)m * a.ldx + 8 * k8);
    }
  }
}

// ------------------------------------------------------------------ epilogue
// Thread (l, i) holds y[m][n] of tile nt with m = 4*(l>>4) + i, n = l & 15 (the
// v_mfma_f32_16x16x32 C layout, reduced over the 8 waves); l is the lane or, for M <= 4,
// n alone.  Partners of the shuffles below (n ^ 1, n + 8) sit in the same 16-lane group.  `best` is the
// thread's running argmax key for LOGITS_ARGMAX.
// RESID with fold_x (M == 1): also the fp16 h * nw of the next projection's TI_X_F16_FOLDED input
// (fold weights pre-staged at fw) and this thread's running sum of h^2 (ssacc).
__device__ __forceinline__ void epilogue(const GemvArgs& a, int nt, int tl, int l, int i, float v, const float* es,
                                         unsigned long long& best, bool ok, const float* fw, float& ssacc) {
  const ti_epilogue& e = a.epi;
  const int m = 4 * (l >> 4) + i, n = l & 15, ng = nt * 16 + n;
  const bool live = ok && m < a.M;
  switch (e.kind) {
    case TI_EPI_STORE_F32:
      if (live) ((float*)e.out)[(size_t)m * e.ldo + ng] = v;
      break;
    case TI_EPI_STORE_F16:
      if (live) ((uint16_t*)e.out)[(size_t)m * e.ldo + ng] = f2h(v);
      break;
    case TI_EPI_RESID_F32:   // add(residual, y), tensor_engine.cpp:1626-1678; residual pre-staged in LDS
      if (live) {
        const float r = es[(tl * a.M + m) * 16 + n] + v;
        ((float*)e.out)[(size_t)m * e.ldo + ng] = r;
        if (e.fold_x) {
          e.fold_x[ng] = f2h(r * fw[tl * 16 + n]);
          ssacc = fmaf(r, r, ssacc);
        }
      }
      break;
    case TI_EPI_SILU_MUL_F16: {
      // compute_ffn (inference_engine.cpp:386-391): multiply(up, silu(gate)).
      const float up = lane_xor<8>(v);   // lanes n < 8: the up row n + 8 of the same tile
      const float s = v / (1.0f + expf(-v));
      if (live && n < 8) ((uint16_t*)e.out)[(size_t)m * e.ldo + nt * 8 + n] = f2h(up * s);
      break;
    }
    case TI_EPI_QKV_ROPE_KV: {
      const float partner = lane_xor<1>(v);
      const int hd = e.head_dim;
      const bool qk = ng < e.q_dim + e.kv_dim;
      float r = v;
      int p = 0;
      if (live) {
        p = ((const int*)(es + a.M * hd))[m];
        if (qk) {
          const int base = ng < e.q_dim ? 0 : e.q_dim;
          const int d = (ng - base) % hd;
          const float2 cs = *(const float2*)(es + m * hd + (d & ~1));   // (cos, sin) of pos[m], staged
          // apply_rope (tensor_engine.cpp:1602-1612): even = x*c - y*s, odd = x*s + y*c,
          // evaluated with the reference build's contraction pattern.
          r = (d & 1) == 0 ? fmaf(-partner, cs.y, v * cs.x) : fmaf(v, cs.x, partner * cs.y);
        }
      }
      if (!live) break;
      if (ng < e.q_dim) {
        ((float*)e.out)[(size_t)m * e.ldo + ng] = r;
      } else {
        const bool is_k = qk;
        const int c = ng - e.q_dim - (is_k ? 0 : e.kv_dim);
        const int kvh = c / hd, d = c - kvh * hd;
        uint16_t* cache = is_k ? e.k_cache : e.v_cache;
        cache[(size_t)m * e.kv_stream_stride + ((size_t)kvh * e.max_seq + p) * hd + d] = f2h(r);
      }
      break;
    }
    case TI_EPI_LOGITS_ARGMAX: {
      if (live) {
        ((float*)e.out)[(size_t)m * e.ldo + ng] = v;
        const unsigned long long key = ((unsigned long long)float_order_key(v) << 32) |
                                       (unsigned long long)(0xFFFFFFFFu - (uint32_t)ng);
        best = key > best ? key : best;
      }
      break;
    }
    default:
      break;
  }
}

// Offset-folded int4 input prep of one staged x piece (deq_int4_raw): the high-nibble slots scaled
// by 1/16 (exact in fp16) and the piece's share of corr[g][m] = 1032 * sum_lo x + 1152 * sum_hi x.
__device__ __forceinline__ float int4_x_prep(f16x8& h) {
  const f16 s16 = (f16)0.0625f;
  h[2] *= s16; h[3] *= s16; h[6] *= s16; h[7] *= s16;
  const float lo = ((float)h[0] + (float)h[1]) + ((float)h[4] + (float)h[5]);
  const float hi = ((float)h[2] + (float)h[3]) + ((float)h[6] + (float)h[7]);
  return 1032.0f * lo + 1152.0f * hi;
}

// --------------------------------------------------------------------- kernel
// The fields on the prologue's critical path come first as separate arguments: gfx950 can
// preload leading kernel arguments into SGPRs before the waves start (compiled with
// -mllvm -amdgpu-kernarg-preload-count, see Makefile), so the first x / weight / epilogue-input
// loads do not wait for a kernarg s_load round trip (the grid size is passed too: gridDim
// comes from the hidden kernargs).  Everything read before the weight ring is issued sits in
// the 14 dwords the hardware preloads (s[2:15]; packed below); the struct carries the rest.
//   p_aux: the rms_norm weight (XM_NORM*), the producer's ss partials (XM_F16F), the splits'
//          (max, sum) pairs (XM_ATTN), else NULL
//   p_mgk: M | grid << 6 | epilogue kind << 18 | head_dim / 64 << 21 (XM_ATTN)
//   p_kx:  K | (ldx, or n_ss for XM_F16F, or splits for XM_ATTN) << 16
// Workgroup blockIdx.x runs over its contiguous tile range.
// G32: group-32 weights (TI_BITS_G32, GGUF Q4_0 / Q8_0 blocks): within a tile, lane l holds for
// MFMA step s4 the 8 k = 32 s4 + 8 (l >> 4) + e, so each v_mfma_f32_16x16x32 reduces exactly one
// 32-weight block; its scale (and, int4, its offset correction) is applied per step.
template <int BITS, int XM, bool G32 = false, bool AFF = false>
__global__ __launch_bounds__(kGemvThreads, 1) void gemv_wq_kernel(const u32x4* p_tiles, const uint16_t* p_scales,
                                                                   const void* p_x, const float* p_aux, int p_mgk,
                                                                   int p_N, int p_kx, int p_ldo, const float* p_pre,
                                                                   GemvArgs a) {
  const unsigned long long t_entry = stamp_now();
  const unsigned bid = blockIdx.x;
  a.tiles = p_tiles;
  a.scales = p_scales;
  a.x = p_x;
  a.norm_w = p_aux;
  a.M = p_mgk & 63;
  // p_N = q | r << 8: NT = q * grid + r 16-row tiles, workgroup b takes q (+1 for b < r) of them from
  // t0 = b q + min(b, r) (scalar arithmetic only; launch_gemv packs it)
  const int nt_q = p_N & 0xff, nt_r = (int)((unsigned)p_N >> 8);
  a.K = p_kx & 0xffff;
  a.ldx = XM == XM_F16F || XM == XM_ATTN ? a.K : (int)((unsigned)p_kx >> 16);
  const int p_grid = (p_mgk >> 6) & 0xfff;
  a.N = 16 * (nt_q * p_grid + nt_r);
  constexpr int C = TileFmt<BITS>::kChunks;
  constexpr int R = TI_GEMV_RING_VGPRS / (4 * C) > 2 ? TI_GEMV_RING_VGPRS / (4 * C) : 2;   // ring depth (items)
  constexpr int XPF = 3;                           // fp16 x: 16-byte pieces prefetched per thread
  extern __shared__ __attribute__((aligned(16))) char smem[];
  GEMV_TS(0);
  const int KT = a.K >> 7, xs = a.K + 8, NT = a.N >> 4, K8 = a.K >> 3;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: counters live in SGPRs
  const int t0 = (int)bid * nt_q + ((int)bid < nt_r ? (int)bid : nt_r);
  const int ntl = nt_q + ((int)bid < nt_r ? 1 : 0);
  constexpr bool kOneRow = XM == XM_F16F || XM == XM_ATTN || XM == XM_NORM1;   // (M == 1 by construction)
  const int KW = wave < KT ? (KT - wave + kGemvWaves - 1) / kGemvWaves : 0;   // k-tiles per tile, this wave
  const int total = ntl * KW;
  static_assert(!G32 || BITS != 16, "group-32 weights: int4 / int8");
  static_assert(!AFF || (G32 && BITS == 4), "affine blocks: group-32 int4");
  const GemvLds L = gemv_lds_layout(a.M, a.K, ntl, G32, AFF);
  uint16_t* ml = (uint16_t*)(smem + L.mins);       // AFF: block minimums, as sl
  float* bsum = (float*)(smem + L.bsum);           // AFF: [K/32][16] sums of x per block and row
  f16* xl = (f16*)(smem + L.x);
  uint16_t* sl = (uint16_t*)(smem + L.sc);
  float* corr = (float*)(smem + L.corr);           // [K/128][16] (int4 only)
  f32x4* slab = (f32x4*)(smem + L.slab);           // [ntl + 1][8][64]
  float* es = (float*)(smem + L.es);
  unsigned long long* best_l = (unsigned long long*)(smem + L.best);
  float* red = (float*)(smem + L.slab);            // norm reduction scratch (before the stream)

  // ---- 1. small inputs into registers, ahead of the ring
  const int n_sc = BITS == 16 ? 0 : ntl * KT * (G32 ? 8 : 2);  // u32x4 pieces of scales
  const u32x4* sg = (const u32x4*)(a.scales + (size_t)t0 * KT * (G32 ? 64 : 16));
  u32x4 sc_reg = {0u, 0u, 0u, 0u};
#if TI_GEMV_EXP & 8   // diagnostic: no dependency on x / scales (constants instead of loads)
  const int nx16 = a.M * K8;
  float4 v0 = {1.0f, 1.0f, 1.0f, 1.0f}, v1 = v0, w0 = v0, w1 = v0;
  u32x4 xr16[XPF];
  for (int q = 0; q < XPF; ++q) xr16[q] = (u32x4){0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
  sc_reg = xr16[0];
  auto load_x = [&]() {};
  if (false) {
#else
  if constexpr (BITS != 16) sc_reg = ld_w(sg + (tid < n_sc ? tid : 0));

  const int nx16 = a.M * K8;
  float4 v0, v1, w0, w1;
  u32x4 xr16[XPF];
  // x rows and the epilogue input depend on the previous launch
  // XM_ATTN: this thread's 8 dims (one head) of every split, and the splits' (max, sum)
  constexpr int kPS = TI_ATTN_MAX_PART_SPLITS;
  u32x4 po[XM == XM_ATTN ? kPS : 1];
  float2 pml[XM == XM_ATTN ? kPS : 1];
  auto load_x = [&]() {
    if constexpr (XM == XM_ATTN) {
      const int S = (int)((unsigned)p_kx >> 16), hsh = ((p_mgk >> 21) & 3) == 2 ? 7 : 6;
      const int i = tid < K8 ? tid : K8 - 1, h = (8 * i) >> hsh, d = (8 * i) & ((1 << hsh) - 1);
#pragma unroll
      for (int sp = 0; sp < kPS; ++sp) {
        const int r = h * S + (sp < S ? sp : S - 1);
        po[sp] = *(const u32x4*)((const f16*)a.x + ((size_t)r << hsh) + d);
        pml[sp] = *(const float2*)(p_aux + 2 * r);
      }
    } else if constexpr (XM == XM_NORM1) {
      const int k8 = tid < K8 ? tid : K8 - 1;
      const float* xr = (const float*)a.x;
      v0 = *(const float4*)(xr + 8 * k8);
      v1 = *(const float4*)(xr + 8 * k8 + 4);
    } else if constexpr (XM == XM_F16 || XM == XM_F16F) {
#pragma unroll
      for (int q = 0; q < XPF; ++q) {
        const int i = tid + q * kGemvThreads < nx16 ? tid + q * kGemvThreads : nx16 - 1;
        const int m = kOneRow ? 0 : i / K8, k8 = i - m * K8;
        xr16[q] = *(const u32x4*)((const f16*)a.x + (size_t)m * a.ldx + 8 * k8);
      }
    }
  };
  if constexpr (XM == XM_NORM1) {
#endif
    const int k8 = tid < K8 ? tid : K8 - 1;
    w0 = *(const float4*)(a.norm_w + 8 * k8);
    w1 = *(const float4*)(a.norm_w + 8 * k8 + 4);
  }
  load_x();
  // Epilogue input, one word per thread, loaded unconditionally (a branch here would make
  // the compiler wait at the join): a residual element of our tiles, this step's position
  // of row tid, or a dummy word of x.
  // (p_pre / kind / ldo are preloaded: epi.out for RESID, epi.pos for QKV, else x)
  const int kind = (p_mgk >> 18) & 7, ldo = p_ldo;
  const int n_res = kind == TI_EPI_RESID_F32 ? ntl * a.M * 16 : 0;
  const float* pre_p;
  {
    const int idx = tid < n_res ? tid : 0;
    const int tl = kOneRow ? idx >> 4 : idx / (a.M * 16), rem = idx - tl * a.M * 16, m = rem >> 4, n = rem & 15;
    pre_p = kind == TI_EPI_RESID_F32 ? p_pre + (size_t)m * ldo + (t0 + tl) * 16 + n
            : kind == TI_EPI_QKV_ROPE_KV ? p_pre + (tid < a.M ? tid : 0) : p_pre;
  }
  const float pre = *pre_p;
  // RESID with fold_x: the fold weight of the same output (one row), consumed by the epilogue
  // (its pointer comes from the kernarg struct: loaded after the ring is issued, below)
  float fw_pre = 0.0f;
  // XM_F16F: this lane's share of the producer's partial sums of squares (up to 256 of them),
  // clamped loads; masked and summed after the stream
  float ss4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const int n_ss = (int)((unsigned)p_kx >> 16);
  if constexpr (XM == XM_F16F) {
#pragma unroll
    for (int j = 0; j < 4; ++j) ss4[j] = p_aux[lane + 64 * j < n_ss ? lane + 64 * j : 0];
  }

  // ---- 2. the weight ring.  Item j of this wave = (tile j / KW, k-tile wave + 8 * (j % KW));
  // items past the end re-load the last item (no branch around loads); coordinates advance
  // by counters (no integer division in the stream).
  const u32x4* tb = a.tiles + (size_t)t0 * KT * (kWave * C) + lane;
  const size_t last_off = total > 0 ? ((size_t)(ntl - 1) * KT + wave + kGemvWaves * (KW - 1)) * (kWave * C) : 0;
  int rt = 0, rk = 0, rj = 0;                      // refill cursor: tile, k index, item
  auto refill_off = [&]() -> size_t {
    const size_t o = rj < total ? ((size_t)rt * KT + wave + kGemvWaves * rk) * (kWave * C) : last_off;
    ++rj;
    if (++rk == KW) { rk = 0; ++rt; }
    return o;
  };
  // Only the first R0 slots go out before the staging barrier: a CU's memory pipe accepts a
  // limited number of outstanding loads, so a wave issuing all R slots blocks in issue for
  // microseconds, and the barrier (hence the first MFMA) would wait for the slowest wave's
  // whole burst.  The rest of the ring is issued right after the barrier.
  constexpr int R0 = R >= 8 ? 4 : R;
  u32x4 ring[R][C];
#if TI_GEMV_RING_DELAY > 0   // A/B knob: hold the ring back (x 64 clocks) behind the small loads
  __builtin_amdgcn_s_sleep(TI_GEMV_RING_DELAY);
#endif
#pragma unroll
  for (int s = 0; s < R0; ++s) {
    const size_t o = refill_off();
#pragma unroll
    for (int c = 0; c < C; ++c) ring[s][c] = ld_w(tb + o + c * kWave);
  }
  const bool fold = (XM == XM_F16 || XM == XM_ATTN) && kind == TI_EPI_RESID_F32 && a.epi.fold_x != nullptr;
  if constexpr (XM == XM_F16 || XM == XM_ATTN) {   // fold weight (consumed by the epilogue)
    const float* fw_p = fold ? a.epi.fold_w + (size_t)t0 * 16 + (tid < n_res ? tid : 0) : pre_p;
    fw_pre = *fw_p;
  }

  GEMV_TS(1);
  STAMP_MARK(ph_issued);
  // ---- 3. stage scales and x in LDS (waits only for the loads of step 1)
  if constexpr (BITS != 16) {
    if (tid < n_sc) ((u32x4*)sl)[tid] = sc_reg;
  }
  // int4 (group 128): the x pieces staged from registers get their 1/16 scaling and offset correction
  // here, before the staging barrier (no second LDS pass and barrier in front of the stream); every
  // piece of x must come from registers for that (rare long shapes take the pass below)
  constexpr bool kRegPrep = BITS == 4 && !G32 && (XM == XM_NORM1 || XM == XM_ATTN || XM == XM_F16 || XM == XM_F16F);
  const bool reg_prep = kRegPrep && (XM == XM_NORM1 || XM == XM_ATTN || nx16 <= XPF * kGemvThreads);
  if constexpr (XM == XM_NORM1) {
    // rms_norm (tensor_engine.cpp:1488-1505) of the single row, x and w held in registers.
    float ss = 0.0f;
    if (tid < K8) {
      ss = fmaf(v0.x, v0.x, ss); ss = fmaf(v0.y, v0.y, ss); ss = fmaf(v0.z, v0.z, ss); ss = fmaf(v0.w, v0.w, ss);
      ss = fmaf(v1.x, v1.x, ss); ss = fmaf(v1.y, v1.y, ss); ss = fmaf(v1.z, v1.z, ss); ss = fmaf(v1.w, v1.w, ss);
    }
    ss = group_sum<kWave>(ss);
    if (lane == 0) red[wave] = ss;
    lds_barrier();
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < kGemvWaves; ++w) tot += red[w];
    const float rms = sqrtf(tot / (float)a.K + a.eps);
    float part = 0.0f;
    if (tid < K8) {
      f16x8 h;
      h[0] = mul_f16(v0.x / rms, w0.x); h[1] = mul_f16(v0.y / rms, w0.y);
      h[2] = mul_f16(v0.z / rms, w0.z); h[3] = mul_f16(v0.w / rms, w0.w);
      h[4] = mul_f16(v1.x / rms, w1.x); h[5] = mul_f16(v1.y / rms, w1.y);
      h[6] = mul_f16(v1.z / rms, w1.z); h[7] = mul_f16(v1.w / rms, w1.w);
      if constexpr (kRegPrep) part = int4_x_prep(h);
      *(f16x8*)(xl + 8 * tid) = h;
    }
    if constexpr (kRegPrep) {
      part = group_sum<16>(part);
      if (tid < K8 && (lane & 15) == 0) corr[(tid >> 4) * 16] = part;
    }
  } else if constexpr (XM == XM_ATTN) {
    // the attention's split merge (attention.hip last-arriver merge): weights
    // l_s * exp(m_s - max), normalised rows o_s, empty splits (m = -inf) weigh 0
    const int S = (int)((unsigned)p_kx >> 16);
    float mx = -INFINITY;
#pragma unroll
    for (int sp = 0; sp < kPS; ++sp) mx = sp < S ? fmaxf(mx, pml[sp].x) : mx;
    float num[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, den = 0.0f;
#pragma unroll
    for (int sp = 0; sp < kPS; ++sp) {
      const float f = sp < S && pml[sp].x != -INFINITY ? pml[sp].y * __expf(pml[sp].x - mx) : 0.0f;
      den += f;
      const f16x8 o = __builtin_bit_cast(f16x8, po[sp]);
#pragma unroll
      for (int e = 0; e < 8; ++e) num[e] = fmaf(f, (float)o[e], num[e]);
    }
    float part = 0.0f;
    if (tid < K8) {
      f16x8 hx;
#pragma unroll
      for (int e = 0; e < 8; ++e) hx[e] = (f16)(den > 0.0f ? num[e] / den : 0.0f);
      if constexpr (kRegPrep) part = int4_x_prep(hx);
      *(f16x8*)(xl + 8 * tid) = hx;
    }
    if constexpr (kRegPrep) {
      part = group_sum<16>(part);
      if (tid < K8 && (lane & 15) == 0) corr[(tid >> 4) * 16] = part;
    }
  } else if constexpr (XM == XM_F16 || XM == XM_F16F) {
#pragma unroll
    for (int q = 0; q < XPF; ++q) {
      const int i = tid + q * kGemvThreads;
      const int m = kOneRow || i >= nx16 ? 0 : i / K8, k8 = i - m * K8;
      float part = 0.0f;
      if (i < nx16) {
        if (kRegPrep && reg_prep) {
          f16x8 h = __builtin_bit_cast(f16x8, xr16[q]);
          part = int4_x_prep(h);
          *(f16x8*)(xl + m * xs + 8 * k8) = h;
        } else {
          *(u32x4*)(xl + m * xs + 8 * k8) = xr16[q];
        }
      }
      if (kRegPrep && reg_prep) {   // (uniform: every lane of a 16-lane group has the same q)
        part = group_sum<16>(part);
        if (i < nx16 && (lane & 15) == 0) corr[(k8 >> 4) * 16 + m] = part;
      }
    }
  }
  // rare shapes: what the register prefetch did not cover (these loads wait behind the ring)
  if constexpr (BITS != 16) {
    for (int i = tid + kGemvThreads; i < n_sc; i += kGemvThreads) ((u32x4*)sl)[i] = sg[i];
  }
  if constexpr (AFF) {   // the minimums follow all N/16 tiles' scales in the same buffer
    const u32x4* mg = (const u32x4*)(a.scales + (size_t)NT * KT * 64 + (size_t)t0 * KT * 64);
    for (int i = tid; i < n_sc; i += kGemvThreads) ((u32x4*)ml)[i] = mg[i];
  }
  if constexpr (XM == XM_F16 || XM == XM_F16F) {
    if (nx16 > XPF * kGemvThreads) stage_x_generic<XM>(a, xl, red, XPF * kGemvThreads);
  } else if constexpr (XM != XM_NORM1 && XM != XM_ATTN) {
    stage_x_generic<XM>(a, xl, red, 0);
  }
  if (a.epi.kind == TI_EPI_QKV_ROPE_KV && tid < a.M) ((int*)(es + a.M * a.epi.head_dim))[tid] = __builtin_bit_cast(int, pre);
  if (tid < 16) best_l[tid] = 0ull;
  lds_barrier();
  STAMP_MARK(ph_staged);
#pragma unroll
  for (int s = R0; s < R; ++s) {
    const size_t o = refill_off();
#pragma unroll
    for (int c = 0; c < C; ++c) ring[s][c] = ld_w(tb + o + c * kWave);
  }
  if constexpr (BITS == 4) if (!reg_prep) {
    // Offset-folded int4 (deq_int4_raw): scale the high-nibble slots of x by 1/16 (exact in
    // fp16) and build corr[g][m] = 1032 * sum_lo a + 1152 * sum_hi a per 128-k group.  A
    // group is 16 consecutive k8 pieces, i.e. 16 consecutive lanes (K8 % 16 == 0).
    const f16 s16 = (f16)0.0625f;
    for (int i0 = 0; i0 < a.M * K8; i0 += kGemvThreads) {
      const int idx = i0 + tid;
      float part = 0.0f, sx = 0.0f;
      int m = 0, k8 = 0;
      if (idx < a.M * K8) {
        m = idx / K8;
        k8 = idx - m * K8;
        f16x8 h = *(const f16x8*)(xl + m * xs + 8 * k8);
        h[2] *= s16; h[3] *= s16; h[6] *= s16; h[7] *= s16;
        *(f16x8*)(xl + m * xs + 8 * k8) = h;
        const float lo = ((float)h[0] + (float)h[1]) + ((float)h[4] + (float)h[5]);
        const float hi = ((float)h[2] + (float)h[3]) + ((float)h[6] + (float)h[7]);
        part = 1032.0f * lo + 1152.0f * hi;
        if constexpr (AFF) sx = lo + 16.0f * hi;   // the piece's sum of x (high slots were scaled by 1/16)
      }
      if constexpr (G32) {   // one 32-k block = 4 consecutive pieces
        part = group_sum<4>(part);
        if (idx < a.M * K8 && (lane & 3) == 0) corr[(k8 >> 2) * 16 + m] = part;
        if constexpr (AFF) {
          sx = group_sum<4>(sx);
          if (idx < a.M * K8 && (lane & 3) == 0) bsum[(k8 >> 2) * 16 + m] = sx;
        }
      } else {
        part = group_sum<16>(part);
        if (idx < a.M * K8 && (lane & 15) == 0) corr[(k8 >> 4) * 16 + m] = part;
      }
    }
    lds_barrier();
  }

  // RoPE (cos, sin) of each row's position: issued now, consumed after the stream.
  float cs_reg = 0.0f;
  const int n_cs = a.epi.kind == TI_EPI_QKV_ROPE_KV ? a.M * a.epi.head_dim : 0;
  if (n_cs > 0) {
    const int hd = a.epi.head_dim, idx = tid < n_cs ? tid : 0, m = idx / hd, j = idx - m * hd;
    cs_reg = a.epi.rope_cs[(size_t)((const int*)(es + a.M * hd))[m] * hd + j];
  }

  GEMV_TS(2);
  STAMP_MARK(ph_stream);
  // ---- 4. the stream: branch-free, R items per block
  const int r = lane & 15, kq = lane >> 4;
  const f16* xrow = xl + (r < a.M ? r : a.M - 1) * xs + kq * 32;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t magic;   // 0x64006400 in a VGPR (see deq_int4_raw)
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  f32x4* my_slab = slab + wave * kWave + lane;     // + tile * 8 * 64
  constexpr int kSlabStride = kGemvWaves * kWave;
  int ct = 0, ck = 0;                              // compute cursor: tile, k index
  auto item = [&](const u32x4 (&w)[C]) {
    const int kt = wave + kGemvWaves * ck;
    f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (BITS == 16) t = acc;
    if constexpr (G32) {
      const f16* xr32 = xrow - kq * 32 + kq * 8;   // this lane's 8 k of each 32-k block
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const f16x8 bf = dequant_step<BITS>(w, s4, magic);
        const f16x8 af = *(const f16x8*)(xr32 + kt * 128 + s4 * 32);
        f32x4 tb = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf, (f32x4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        if constexpr (BITS == 4) tb -= *(const f32x4*)(corr + (kt * 4 + s4) * 16 + 4 * kq);
        const float sc = h2f(sl[((ct * KT + kt) * 4 + s4) * 16 + r]);
        acc[0] = fmaf(sc, tb[0], acc[0]);
        acc[1] = fmaf(sc, tb[1], acc[1]);
        acc[2] = fmaf(sc, tb[2], acc[2]);
        acc[3] = fmaf(sc, tb[3], acc[3]);
        if constexpr (AFF) {   // weight = d (q - 8) + (8 d + m): the offset term times the block's sum of x
          const float mt = fmaf(8.0f, sc, h2f(ml[((ct * KT + kt) * 4 + s4) * 16 + r]));
          const f32x4 bs = *(const f32x4*)(bsum + (kt * 4 + s4) * 16 + 4 * kq);
          acc[0] = fmaf(mt, bs[0], acc[0]);
          acc[1] = fmaf(mt, bs[1], acc[1]);
          acc[2] = fmaf(mt, bs[2], acc[2]);
          acc[3] = fmaf(mt, bs[3], acc[3]);
        }
      }
    } else {
#if TI_GEMV_EXP & 1   // diagnostic build (tools/probe_gemv.hip): stream only, no dequant / MFMA
    t[0] += __builtin_bit_cast(float, w[0][0] ^ w[0][1] ^ w[0][2] ^ w[0][3]) + (float)xrow[kt];
#else
    (void)t;
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const f16x8 bf = dequant_step<BITS>(w, s4, magic);
      const f16x8 af = *(const f16x8*)(xrow + kt * 128 + s4 * 8);
      t = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf, t, 0, 0, 0);
    }
#endif
    if constexpr (BITS == 16) {
      acc = t;
    } else {
      if constexpr (BITS == 4) {   // remove the folded offsets of this group (deq_int4_raw)
        const f32x4 cr = *(const f32x4*)(corr + kt * 16 + 4 * kq);
        t -= cr;
      }
      const float sc = h2f(sl[(ct * KT + kt) * 16 + r]);
      acc[0] = fmaf(sc, t[0], acc[0]);
      acc[1] = fmaf(sc, t[1], acc[1]);
      acc[2] = fmaf(sc, t[2], acc[2]);
      acc[3] = fmaf(sc, t[3], acc[3]);
    }
    }   // !G32
    // the tile's last item lands in its slab, every other item in the dummy slab
    const bool last = ++ck == KW;
    my_slab[(last ? ct : ntl) * kSlabStride] = acc;
    if (last) acc = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    ck = last ? 0 : ck;
    ct += last ? 1 : 0;
  };
  int j0 = 0;
#if TI_GEMV_SYNC > 0
  // Waves of a CU drift apart (the oldest wins issue arbitration); a workgroup barrier every
  // TI_GEMV_SYNC blocks keeps them together while every wave still has blocks left (the
  // count of barriers is the same for all waves: blocks below the smallest wave total).
  const int common = ntl * (KT / kGemvWaves);
  int blk = 0;
  for (; j0 + R <= common; j0 += R) {
#pragma unroll
    for (int s = 0; s < R; ++s) {
      item(ring[s]);
      const size_t o = refill_off();
#pragma unroll
      for (int c = 0; c < C; ++c) ring[s][c] = ld_w(tb + o + c * kWave);
    }
    if (++blk == TI_GEMV_SYNC) {
      blk = 0;
      __builtin_amdgcn_s_barrier();
    }
  }
#endif
  for (; j0 + R <= total; j0 += R) {   // full blocks: no branches, R items scheduled together
#pragma unroll
    for (int s = 0; s < R; ++s) {
      item(ring[s]);
      const size_t o = refill_off();   // refill this slot R items ahead (clamped past the end)
#pragma unroll
      for (int c = 0; c < C; ++c) ring[s][c] = ld_w(tb + o + c * kWave);
    }
  }
#pragma unroll
  for (int s = 0; s < R; ++s)          // tail: the last total % R items, nothing refilled
    if (j0 + s < total) item(ring[s]);
  if (KW == 0)   // K < 8*128: this wave owns no k-tiles; its partials are zero
    for (int tl = 0; tl < ntl; ++tl) my_slab[tl * kSlabStride] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

  GEMV_TS(3);
  GEMV_WTS();
  STAMP_MARK(ph_streamed);
  // ---- 5. epilogue inputs into LDS, reduce the 8 partials per tile, epilogue
  if (tid < n_res) es[tid] = pre;
  if (fold && tid < n_res) es[n_res + tid] = fw_pre;
  if (tid < n_cs) es[tid] = cs_reg;
  // inputs past the one-per-thread prefetch (ntl * M * 16 or M * head_dim > 512): loaded now
  for (int i = tid + kGemvThreads; i < n_res; i += kGemvThreads) {
    const int tl = i / (a.M * 16), rem = i - tl * a.M * 16, m = rem >> 4, n = rem & 15;
    es[i] = p_pre[(size_t)m * ldo + (t0 + tl) * 16 + n];
    if (fold) es[n_res + i] = a.epi.fold_w[(size_t)t0 * 16 + i];
  }
  // XM_F16F: rms of the row from the producer's partials, the same fixed-order sum in every
  // wave (rms_norm, tensor_engine.cpp:1488-1505, with the division moved behind the GEMM)
  float rms = 1.0f;
  if constexpr (XM == XM_F16F) {
    float t = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) t += lane + 64 * j < n_ss ? ss4[j] : 0.0f;
    t = group_sum<kWave>(t);
    rms = sqrtf(t / (float)a.K + a.eps);
  }
  float ssacc = 0.0f;
  const float* fw_l = es + n_res;
  for (int i = tid + kGemvThreads; i < n_cs; i += kGemvThreads) {
    const int hd = a.epi.head_dim, m = i / hd, j = i - m * hd;
    es[i] = a.epi.rope_cs[(size_t)((const int*)(es + a.M * hd))[m] * hd + j];
  }
  lds_barrier();
  GEMV_TS(5);
  STAMP_MARK(ph_reduce);
  unsigned long long best[4] = {0ull, 0ull, 0ull, 0ull};
  if (a.M <= 4) {
    // rows m < 4 live in lanes 0-15 of each partial (C layout m = 4*(l>>4) + i): one thread per
    // (tile, n), all tiles in one pass over the workgroup, the M components of its f32x4.
    for (int tb0 = wave * kWave; tb0 < ntl * 16; tb0 += kGemvThreads) {
      const int t = tb0 + lane, ok = t < ntl * 16, tl = ok ? t >> 4 : 0, n = lane & 15;
      const f32x4* sp = slab + tl * kSlabStride + n;
      f32x4 v = sp[0];
#pragma unroll
      for (int w = 1; w < kGemvWaves; ++w) v += sp[w * kWave];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < a.M) epilogue(a, t0 + tl, tl, n, i, XM == XM_F16F ? v[i] / rms : v[i], es, best[i], ok, fw_l, ssacc);
    }
  } else {
    const int i4 = wave & 3;
    for (int tl = wave >> 2; tl < ntl; tl += 2) {
      const float* sp = (const float*)(slab + tl * kSlabStride + lane) + i4;
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < kGemvWaves; ++w) v += sp[w * kWave * 4];
      epilogue(a, t0 + tl, tl, lane, i4, v, es, best[0], true, fw_l, ssacc);
    }
  }
  STAMP_MARK(ph_epi);
  if (a.epi.kind == TI_EPI_LOGITS_ARGMAX) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const unsigned long long other = __shfl_xor(best[i], o, kWave);
        best[i] = other > best[i] ? other : best[i];
      }
    }
    if (a.M <= 4) {
      if ((lane & 15) == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i)   // constant bounds: best[] stays in registers
          if (i < a.M && best[i]) atomicMax(best_l + i, best[i]);
    } else {
      const int m = 4 * (lane >> 4) + (wave & 3);
      if ((lane & 15) == 0 && m < a.M && best[0]) atomicMax(best_l + m, best[0]);
    }
    lds_barrier();
    if (tid < a.M && best_l[tid])
      atomicMax(a.epi.argmax + (size_t)tid * TI_ARGMAX_SLOTS + (bid & (TI_ARGMAX_SLOTS - 1)), best_l[tid]);
    if (a.epi.step_ctr && bid == 0 && tid == 0) *a.epi.step_ctr += a.epi.advance;
  }
  if (fold && a.M <= 4 && ntl * 16 <= kWave) {
    // every output of the workgroup was wave 0's (the M <= 4 epilogue above): its sum alone, no
    // barrier -- the same value as the general form below, whose other terms are exact zeros
    if (wave == 0) {
      const float sw = group_sum<kWave>(ssacc);
      if (lane == 0) a.epi.fold_ss[bid] = sw;
    }
  } else if (fold) {   // this workgroup's sum of h^2, waves in a fixed order (best_l: unused by RESID)
    float* red2 = (float*)best_l;
    const float sw = group_sum<kWave>(ssacc);
    if (lane == 0) red2[wave] = sw;
    lds_barrier();
    if (tid == 0) {
      float t = 0.0f;
#pragma unroll
      for (int w = 0; w < kGemvWaves; ++w) t += red2[w];
      a.epi.fold_ss[bid] = t;
    }
  }
  GEMV_TS(4);
  stamp_end(a.stamp, t_entry, ph_issued, ph_staged, ph_stream, ph_streamed, ph_reduce, ph_epi, ph_streamed);
}

// ================================================================= batched rows
// gemv_mbr_kernel<MB, NTL>: int4 weights x 3..16 fp16 rows (a batch of a few streams, and long-K projections whose
// rows no longer fit gemv_wq_kernel's LDS image): direct calls of ti_gemm_wq_a16, and engines with a weight of 4 GiB or more
// (others run ti_gemm_rows from 3 rows on).  Weights are read once per launch, straight into registers, in
// chunks of 1024 k (8 k-tiles, one per wave), one chunk ahead.
__host__ __device__ inline int mbr_slab_bytes(int MB, int ntl) { return align16(ntl * MB * kGemvWaves * kWave * 16); }
__host__ __device__ inline int mbr_lds_bytes(int MB, int ntl, int K) {
  return mbr_slab_bytes(MB, ntl) + align16(ntl * (K >> 7) * 32);
}

template <int MB, int NTL>
struct MbrChunk {       // one chunk's operands of one wave
  u32x4 w[NTL];        // packed int4 weights of (tile tl, this wave's k-tile)
  f16x8 x[MB][4];      // A fragments: rows 16 b + (lane & 15), k = kt*128 + 32 (lane >> 4) + 8 s4
};

// Each wave loads the A fragments of its own
// k-tile straight into registers, one chunk ahead, so no barrier is needed until the end;
// at <= 16 rows this beats the LDS-staged kernel (bench.py --batch 8/16).
template <int MB, int NTL>
__device__ __forceinline__ void gemv_mbr_body(const GemvArgs a, int grid);
template <int MB, int NTL>
__global__ __launch_bounds__(kGemvThreads, 1) void gemv_mbr_kernel(const GemvArgs a, int grid) {
  const unsigned long long t_entry = stamp_now();
  gemv_mbr_body<MB, NTL>(a, grid);
  stamp_end(a.stamp, t_entry);
}
template <int MB, int NTL>
__device__ __forceinline__ void gemv_mbr_body(const GemvArgs a, int grid) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int KT = a.K >> 7, NT = a.N >> 4, NC = (KT + kGemvWaves - 1) / kGemvWaves;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t0 = (int)(blockIdx.x * (unsigned)NT / (unsigned)grid);
  const int t1 = (int)((blockIdx.x + 1) * (unsigned)NT / (unsigned)grid);
  const int ntl = t1 - t0;                           // NTL or NTL - 1
  f32x4* slab = (f32x4*)smem;                        // after the stream: [NTL][MB][8][64]
  uint16_t* sl = (uint16_t*)(smem + mbr_slab_bytes(MB, NTL));   // [ntl][KT][16]

  // scales of our tiles: loaded first (two pieces per thread cover ntl * KT <= 512 groups)
  const int n_sc = ntl * KT * 2;
  const u32x4* sg = (const u32x4*)(a.scales + (size_t)t0 * KT * 16);
  const u32x4 sc0 = ld_w(sg + (tid < n_sc ? tid : 0));
  const u32x4 sc1 = ld_w(sg + (tid + kGemvThreads < n_sc ? tid + kGemvThreads : 0));

  const f16* xg = (const f16*)a.x;
  const u32x4* tb = a.tiles + lane;
  auto load = [&](MbrChunk<MB, NTL>& ch, int c) {
    const int kt = min(c * kGemvWaves + wave, KT - 1);
#pragma unroll
    for (int tl = 0; tl < NTL; ++tl) ch.w[tl] = ld_w(tb + ((size_t)(t0 + min(tl, ntl - 1)) * KT + kt) * kWave);
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int m = min(b * 16 + r, a.M - 1);
      const f16* xr = xg + (size_t)m * a.ldx + kt * 128 + kq * 32;   // the tile's k order (B fragments)
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) ch.x[b][s4] = *(const f16x8*)(xr + s4 * 8);
    }
  };
  MbrChunk<MB, NTL> B0, B1;
  load(B0, 0);
  if (tid < n_sc) ((u32x4*)sl)[tid] = sc0;
  if (tid + kGemvThreads < n_sc) ((u32x4*)sl)[tid + kGemvThreads] = sc1;
  lds_barrier();

  f32x4 acc[NTL][MB];
#pragma unroll
  for (int t = 0; t < NTL; ++t)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[t][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t magic;
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  auto compute = [&](const MbrChunk<MB, NTL>& ch, int c) {
    const int kt = c * kGemvWaves + wave;
    const bool kvalid = kt < KT;
#pragma unroll
    for (int tl = 0; tl < NTL; ++tl) {
      f32x4 t[MB];
#pragma unroll
      for (int b = 0; b < MB; ++b) t[b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const f16x8 bf = deq_int4_signed(ch.w[tl][s4], magic);
#pragma unroll
        for (int b = 0; b < MB; ++b) t[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ch.x[b][s4], bf, t[b], 0, 0, 0);
      }
      const float sc = kvalid ? h2f(sl[(min(tl, ntl - 1) * KT + kt) * 16 + r]) : 0.0f;
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        acc[tl][b][0] = fmaf(sc, t[b][0], acc[tl][b][0]);
        acc[tl][b][1] = fmaf(sc, t[b][1], acc[tl][b][1]);
        acc[tl][b][2] = fmaf(sc, t[b][2], acc[tl][b][2]);
        acc[tl][b][3] = fmaf(sc, t[b][3], acc[tl][b][3]);
      }
    }
  };
  // chunks two at a time, each loaded one chunk ahead (the reload past the end is harmless)
  int c = 0;
  for (; c + 1 < NC; c += 2) {
    load(B1, c + 1);
    compute(B0, c);
    load(B0, c + 2 < NC ? c + 2 : NC - 1);
    compute(B1, c + 1);
  }
  if (c < NC) compute(B0, c);

  // ---- sum the 8 waves' blocks in a fixed order, then the epilogue
#pragma unroll
  for (int tl = 0; tl < NTL; ++tl)
#pragma unroll
    for (int b = 0; b < MB; ++b) slab[((tl * MB + b) * kGemvWaves + wave) * kWave + lane] = acc[tl][b];
  lds_barrier();
  const int n = lane & 15, nblk = ntl * MB * 4;
  const int nblk_pad = (nblk + kGemvWaves - 1) / kGemvWaves * kGemvWaves;
  for (int cb = wave; cb < nblk_pad; cb += kGemvWaves) {   // wave-uniform trip count (shuffles inside)
    const bool ok = cb < nblk;
    const int cbc = ok ? cb : 0, tl = cbc / (MB * 4), b = (cbc >> 2) % MB, i = cbc & 3;
    const float* sp = (const float*)(slab + (tl * MB + b) * kGemvWaves * kWave + lane) + i;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kGemvWaves; ++w) v += sp[w * kWave * 4];
    const int m = b * 16 + 4 * (lane >> 4) + i;
    epilogue_mb(a, t0 + tl, m, n, v, ok && m < a.M);
  }
  if (a.epi.kind == TI_EPI_LOGITS_ARGMAX && a.epi.step_ctr && blockIdx.x == 0 && tid == 0)
    *a.epi.step_ctr += a.epi.advance;
}

// ------------------------------------------------------------- rows kernel (17..64 rows)
// Batched decode at configs[3] / [4] scale (64 / 32 streams): the weights are still read once
// per launch, but every weight fragment now meets up to 64 rows.  Register operands, no LDS in
// the stream: the 8 waves form RG row groups of 8 / RG waves; a group owns MB 16-row blocks
// and splits the k-tiles over its waves (k-tile w, w + 8 / RG, ...).  Per item a wave holds
// the packed weights of the workgroup's NTL tiles at that k-tile (a WD-slot ring, issued
// WD - 1 items ahead: HBM latency) and its rows' x fragments (two slots, one item ahead: L2
// latency).  The item count is padded to a multiple of WD with zero-scale clamped items, so
// the loop body has no branches (no vmcnt(0) at a join).  After the stream the partial blocks
// of the group's waves are summed in a fixed order through LDS and the epilogue runs.
template <int MB, int NTL, int RG, bool XP = false>
struct RowsCfg {
  static constexpr int kGroupWaves = kGemvWaves / RG;
  static constexpr int kWD = MB * NTL <= 3 ? 4 : 3;   // ring slots (VGPR budget: no spills)
};
__host__ __device__ inline int rows_slab_bytes(int mb_total, int ntl) {
  return align16(ntl * mb_total * kGemvWaves * kWave * 16);
}
// batched fold (ti_hip.h TI_FOLD_SS_ROWS): per-thread partial sums [512] | 1 / rms per row [64] |
// per-tile sums of h^2 per row [4][64], behind the slab and the scales
constexpr int kFoldLdsBytes = 4096;
__host__ __device__ inline int rows_fold_offset(int mb_total, int ntl, int K) {
  return rows_slab_bytes(mb_total, ntl) + align16(ntl * (K >> 7) * 32);
}
__host__ __device__ inline int rows_lds_bytes(int mb_total, int ntl, int K) {
  return rows_fold_offset(mb_total, ntl, K) + kFoldLdsBytes;
}

// Workgroups: n_cg column groups x n_rb row blocks of 16 RG MB rows (narrow outputs split the
// rows: a workgroup's activation bytes shrink with its rows, and its column group's weights are
// re-read by the other row blocks from the same XCD's L2 -- blockIdx % 8 is the column group's
// low bits, a speed placement only).
template <int MB, int NTL, int RG, bool XP>
__device__ __forceinline__ void gemm_rows_body(const GemvArgs a, int n_cg, int n_rb);
template <int MB, int NTL, int RG, bool XP>
__global__ __launch_bounds__(kGemvThreads, 1) void gemm_rows_kernel(const GemvArgs a, int n_cg, int n_rb) {
  const unsigned long long t_entry = stamp_now();
  gemm_rows_body<MB, NTL, RG, XP>(a, n_cg, n_rb);
  stamp_end(a.stamp, t_entry);
}
template <int MB, int NTL, int RG, bool XP>
__device__ __forceinline__ void gemm_rows_body(const GemvArgs a, int n_cg, int n_rb) {
  constexpr int GW = RowsCfg<MB, NTL, RG>::kGroupWaves, WD = RowsCfg<MB, NTL, RG>::kWD;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int KT = a.K >> 7, NT = a.N >> 4;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / GW, gw = wave % GW;
  const int rest = blockIdx.x >> 3, rb = rest % n_rb, cg = (rest / n_rb) * 8 + (blockIdx.x & 7);
  if (cg >= n_cg) return;
  const int b0 = rb * RG * MB;                       // first 16-row block of this workgroup
  const int t0 = (int)(cg * (unsigned)NT / (unsigned)n_cg);
  const int t1 = (int)((cg + 1) * (unsigned)NT / (unsigned)n_cg);
  const int ntl = t1 - t0;                           // NTL or NTL - 1
  const int NI = (KT + GW - 1) / GW, NIP = (NI + WD - 1) / WD * WD;
  ROWS_TS(0);
  f32x4* slab = (f32x4*)smem;                        // after the stream: [NTL][RG * MB][8][64]
  uint16_t* sl = (uint16_t*)(smem + rows_slab_bytes(RG * MB, NTL));   // [ntl][KT][16]

  // the workgroup's group scales (ntl * KT <= 512: two 16-byte pieces per thread), first
  const int n_sc = ntl * KT * 2;
  const u32x4* sg = (const u32x4*)(a.scales + (size_t)t0 * KT * 16);
  u32x4 scr[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) scr[j] = ld_w(sg + (tid + j * kGemvThreads < n_sc ? tid + j * kGemvThreads : 0));

  const f16* xg = (const f16*)a.x;
  const u32x4* tb = a.tiles + lane;
  auto kt_of = [&](int it) { return min(gw + GW * it, KT - 1); };
  auto load_w = [&](u32x4 (&w)[NTL], int it) {
#if TI_GEMV_EXP & 128   // diagnostic: no weight traffic after the first ring
    it = it < WD ? it : it % WD;
#endif
    const int kt = kt_of(it);
#pragma unroll
    for (int tl = 0; tl < NTL; ++tl) w[tl] = ld_w(tb + ((size_t)(t0 + min(tl, ntl - 1)) * KT + kt) * kWave);
  };
  auto load_x = [&](f16x8 (&x)[MB][4], int it) {
#if TI_GEMV_EXP & 256   // diagnostic: no activation traffic after the first ring
    it = it < WD ? it : it % WD;
#endif
    const int kt = kt_of(it);
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      if constexpr (XP) {   // TI_X_F16_PACKED: one contiguous KiB per (block, s4)
        const int bb = min(b0 + grp * MB + b, (a.M - 1) >> 4);
        const f16* xp = xg + ((size_t)(bb * KT + kt) * 4) * 512 + lane * 8;
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) x[b][s4] = *(const f16x8*)(xp + s4 * 512);
      } else {
        const int m = min((b0 + grp * MB + b) * 16 + r, a.M - 1);
        // the tile's k order (A fragments): k = 128 kt + 32 kq + 8 s4 (+ e)
        const f16* xr = xg + (size_t)m * a.ldx + kt * 128 + kq * 32;
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) x[b][s4] = *(const f16x8*)(xr + s4 * 8);
      }
    }
  };
  u32x4 W[WD][NTL];
  f16x8 X[WD][MB][4];
#pragma unroll
  for (int u = 0; u < WD - 1; ++u) {
    load_w(W[u], u);
    load_x(X[u], u);
  }
  // batched fold: the consumer's per-row rms shares (after the first ring loads: their wait
  // costs nothing the first item would not wait for), the producer's per-tile h^2 sums
  constexpr int R = 16 * RG * MB;
  float* fold_l = (float*)(smem + rows_fold_offset(RG * MB, NTL, a.K));
  const bool fold_in = a.epi.ss_in != nullptr, fold_out = a.epi.kind == TI_EPI_RESID_F32 && a.epi.fold_x != nullptr;
  const float share = fold_in ? fold_share(a, b0 * 16 + tid % R, tid / R, kGemvThreads / R) : 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (tid + j * kGemvThreads < n_sc) ((u32x4*)sl)[tid + j * kGemvThreads] = scr[j];
  lds_barrier();
  ROWS_TS(1);

  f32x4 acc[NTL][MB];
#pragma unroll
  for (int t = 0; t < NTL; ++t)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[t][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t magic;
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  auto compute = [&](const u32x4 (&w)[NTL], const f16x8 (&x)[MB][4], int it) {
    const int kt = gw + GW * it;
    const bool kvalid = kt < KT;
    const int ktc = kvalid ? kt : KT - 1;
#pragma unroll
    for (int tl = 0; tl < NTL; ++tl) {
      f32x4 t[MB];
#pragma unroll
      for (int b = 0; b < MB; ++b) t[b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const f16x8 bf = deq_int4_signed(w[tl][s4], magic);
#pragma unroll
        for (int b = 0; b < MB; ++b) t[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[b][s4], bf, t[b], 0, 0, 0);
      }
      const float sc = kvalid ? h2f(sl[(min(tl, ntl - 1) * KT + ktc) * 16 + r]) : 0.0f;
#pragma unroll
      for (int b = 0; b < MB; ++b) acc[tl][b] = fma_scale4(sc, t[b], acc[tl][b]);
    }
  };
  for (int i = 0; i < NIP; i += WD) {
#pragma unroll
    for (int u = 0; u < WD; ++u) {
      load_w(W[(u + WD - 1) % WD], i + u + WD - 1);  // WD - 1 items ahead (clamped past the end)
      load_x(X[(u + WD - 1) % WD], i + u + WD - 1);
      compute(W[u], X[u], i + u);
#if TI_GEMV_EXP & 4
      if (i + u == 0) ROWS_TS(2);
#endif
    }
  }
  ROWS_TS(3);

  // ---- sum each group's waves in a fixed order, then the epilogue
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  ROWS_TS(4);
#pragma unroll
  for (int tl = 0; tl < NTL; ++tl)
#pragma unroll
    for (int b = 0; b < MB; ++b) slab[((tl * RG * MB + grp * MB + b) * kGemvWaves + wave) * kWave + lane] = acc[tl][b];
  if (fold_in) fold_l[tid] = share;
  lds_barrier();
  if (fold_in) {
    fold_rms_finish(a, fold_l, fold_l + kGemvThreads, R, tid);
    lds_barrier();
  }
  const int n = lane & 15, nblk = ntl * RG * MB * 4;
  const int nblk_pad = (nblk + kGemvWaves - 1) / kGemvWaves * kGemvWaves;
  for (int cb = wave; cb < nblk_pad; cb += kGemvWaves) {   // wave-uniform trip count (shuffles inside)
    const bool ok = cb < nblk;
    const int cbc = ok ? cb : 0, tl = cbc / (RG * MB * 4), bb = (cbc >> 2) % (RG * MB), i = cbc & 3;
    const int g = bb / MB;
    const float* sp = (const float*)(slab + (tl * RG * MB + bb) * kGemvWaves * kWave + lane) + i;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < GW; ++w) v += sp[(g * GW + w) * kWave * 4];
    const int rl = bb * 16 + 4 * (lane >> 4) + i, m = b0 * 16 + rl;
    if (fold_in) v = v / fold_l[kGemvThreads + rl];
    if (fold_out) {   // residual add + the next call's folded input (fp16(h * w), sum of h^2 per row)
      const ti_epilogue& e = a.epi;
      const int ng = (t0 + tl) * 16 + n;
      float hn = 0.0f;
      if (ok && m < a.M) {
        float* o = (float*)e.out + (size_t)m * e.ldo + ng;
        hn = *o + v;
        *o = hn;
        float p = hn * e.fold_w[ng];
        asm volatile("" : "+v"(p));   // fp16(fp32 product): no fused multiply-convert (one rounding less)
        e.fold_x[e.fold_packed ? TI_PACKED_INDEX(m, ng, e.ldo >> 7) : (size_t)m * e.ldo + ng] = f2h(p);
      }
      const float sq = group_sum<16>(hn * hn);
      if (ok && n == 0) fold_l[kGemvThreads + 64 + tl * 64 + rl] = sq;
      continue;
    }
    epilogue_mb(a, t0 + tl, m, n, v, ok && m < a.M);
  }
  if (fold_out) {   // this column group's sum of h^2 per row, tiles in order
    lds_barrier();
    if (tid < R && b0 * 16 + tid < a.M) {
      float t = 0.0f;
      for (int tl = 0; tl < ntl; ++tl) t += fold_l[kGemvThreads + 64 + tl * 64 + tid];
      a.epi.fold_ss[(size_t)cg * TI_FOLD_SS_ROWS + b0 * 16 + tid] = t;
    }
  }
  ROWS_TS(5);
  if (a.epi.kind == TI_EPI_LOGITS_ARGMAX && a.epi.step_ctr && blockIdx.x == 0 && tid == 0)
    *a.epi.step_ctr += a.epi.advance;
}

static std::atomic<int> g_num_cus{0};   // (a racing first query stores the same value)

__host__ inline int gemv_xmode(int x_kind, int M, int K) {
  if (x_kind == TI_X_F16) return XM_F16;
  if (x_kind == TI_X_F16_FOLDED) return XM_F16F;
  if (x_kind == TI_X_ATTN_SPLITS) return XM_ATTN;
  if (x_kind == TI_X_F32) return XM_F32;
  return M == 1 && (K >> 3) <= kGemvThreads ? XM_NORM1 : XM_NORM;
}

template <int BITS, bool G32 = false, bool AFF = false>
static int launch_gemv(const GemvArgs& a, int lds, hipStream_t s, int grid) {
  const float* pre = a.epi.kind == TI_EPI_RESID_F32 ? (const float*)a.epi.out
                     : a.epi.kind == TI_EPI_QKV_ROPE_KV ? (const float*)a.epi.pos : (const float*)a.x;
  const int xm = gemv_xmode(a.x_kind, a.M, a.K);
  // packed preloaded arguments (see gemv_wq_kernel)
  const float* aux = xm == XM_F16F || xm == XM_ATTN ? a.epi.ss_in : xm == XM_F16 ? nullptr : a.norm_w;
  const int mgk = a.M | (grid << 6) | (a.epi.kind << 18) | (xm == XM_ATTN ? (a.epi.head_dim / 64) << 21 : 0);
  const int kx = a.K | ((xm == XM_F16F || xm == XM_ATTN ? a.epi.n_ss : a.ldx) << 16);
  const int ldo = a.epi.ldo;
  const int NT = a.N >> 4, nt_q = NT / grid, nt_r = NT % grid;   // the kernel's tile split (gemv_wq_kernel)
  if (nt_q > 255 || nt_r >= (1 << 23))
    return ti_set_error(TI_ERR_UNSUPPORTED, "gemv_wq_kernel: %d tiles over %d workgroups", NT, grid);
  const int pn = nt_q | (nt_r << 8);
  switch (xm) {
    case XM_F16: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_F16, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
    case XM_F32: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_F32, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
    case XM_ATTN: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_ATTN, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
    case XM_F16F: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_F16F, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
    case XM_NORM1: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_NORM1, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
    default: hipLaunchKernelGGL((gemv_wq_kernel<BITS, XM_NORM, G32, AFF>), dim3(grid), dim3(kGemvThreads), lds, s, a.tiles, a.scales, a.x, aux, mgk, pn, kx, ldo, pre, a); break;
  }
  TI_LAUNCH_CHECK("gemv_wq_kernel");
  return TI_OK;
}

// rms_norm rows into fp16 (the batched path's activation prep): the same arithmetic as the
// fused XM_NORM staging above (per-thread k8 pieces, wave sums, 8 waves in order).
__global__ __launch_bounds__(kGemvThreads) void rmsnorm_f16_kernel(const float* x, int ldx, const float* w, float eps,
                                                                    uint16_t* y, int ldy, int K, int pk_kt) {
  __shared__ float red[kGemvWaves];
  const int m = blockIdx.x, tid = threadIdx.x, K8 = K >> 3;
  const float* xr = x + (size_t)m * ldx;
  float ss = 0.0f;
  for (int k8 = tid; k8 < K8; k8 += kGemvThreads) {
    const float4 v0 = *(const float4*)(xr + 8 * k8), v1 = *(const float4*)(xr + 8 * k8 + 4);
    ss = fmaf(v0.x, v0.x, ss); ss = fmaf(v0.y, v0.y, ss); ss = fmaf(v0.z, v0.z, ss); ss = fmaf(v0.w, v0.w, ss);
    ss = fmaf(v1.x, v1.x, ss); ss = fmaf(v1.y, v1.y, ss); ss = fmaf(v1.z, v1.z, ss); ss = fmaf(v1.w, v1.w, ss);
  }
  ss = group_sum<kWave>(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int i = 0; i < kGemvWaves; ++i) tot += red[i];
  const float rms = sqrtf(tot / (float)K + eps);
  for (int k8 = tid; k8 < K8; k8 += kGemvThreads) {
    const float4 v0 = *(const float4*)(xr + 8 * k8), v1 = *(const float4*)(xr + 8 * k8 + 4);
    const float4 w0 = *(const float4*)(w + 8 * k8), w1 = *(const float4*)(w + 8 * k8 + 4);
    f16x8 h;
    h[0] = mul_f16(v0.x / rms, w0.x); h[1] = mul_f16(v0.y / rms, w0.y);
    h[2] = mul_f16(v0.z / rms, w0.z); h[3] = mul_f16(v0.w / rms, w0.w);
    h[4] = mul_f16(v1.x / rms, w1.x); h[5] = mul_f16(v1.y / rms, w1.y);
    h[6] = mul_f16(v1.z / rms, w1.z); h[7] = mul_f16(v1.w / rms, w1.w);
    *(f16x8*)(y + (pk_kt > 0 ? TI_PACKED_INDEX(m, 8 * k8, pk_kt) : (size_t)m * ldy + 8 * k8)) = h;
  }
}

// Batched-rows geometry: at most 8 tiles per workgroup (register accumulators), and the
// workgroup's scales in two 16-byte pieces per thread.
__host__ inline int mb_tiles_cap(int MB, int K) {
  const int lim = MB == 2 ? 6 : 8, cap = 512 / (K >> 7);   // (register budget: no spills)
  return cap < 1 ? 1 : (cap > lim ? lim : cap);
}
__host__ inline int mb_grid(int MB, int N, int K, int num_cus, int* ntl_out) {
  const int NT = N >> 4, cap = mb_tiles_cap(MB, K);
  int grid = NT < num_cus ? NT : num_cus;
  if ((NT + grid - 1) / grid > cap) grid = (NT + cap - 1) / cap;
  *ntl_out = (NT + grid - 1) / grid;
  return grid;
}

static int launch_mb(const GemvArgs& a, int grid, int ntl, int lds, hipStream_t s) {
#define TI_MB_CASE(n) \
  case n: hipLaunchKernelGGL((gemv_mbr_kernel<1, n>), dim3(grid), dim3(kGemvThreads), lds, s, a, grid); break
  switch (ntl) {
    TI_MB_CASE(1); TI_MB_CASE(2); TI_MB_CASE(3); TI_MB_CASE(4); TI_MB_CASE(5); TI_MB_CASE(6); TI_MB_CASE(7);
    default: hipLaunchKernelGGL((gemv_mbr_kernel<1, 8>), dim3(grid), dim3(kGemvThreads), lds, s, a, grid);
  }
#undef TI_MB_CASE
  TI_LAUNCH_CHECK("gemv_mbr_kernel");
  return TI_OK;
}
// Rows kernel (M > 16): RG row groups x MB blocks per group, NTL tiles per workgroup.
__host__ inline void rows_shape(int M, int* MB, int* RG) {
  const int rg = M > 32 ? 2 : 1;   // 64 rows: two groups of 32
  const int mb = (M + 16 * rg - 1) / (16 * rg);
  *MB = mb;
  *RG = rg;
}
// Tile kernel from this many rows on (the rows kernel takes at most 64 rows).
static int tile_rows() { return 65; }
__host__ inline int rows_tiles_cap(int MB, int K) {
  const int lim = MB >= 2 ? 3 : 4, cap = 512 / (K >> 7);   // VGPR budget / scale pieces
  return cap < 1 ? 1 : (cap > lim ? lim : cap);
}
// Column groups for row blocks of MB blocks per group (one round of workgroups where the VGPR
// cap on tiles per workgroup allows).
// The launch is ceil(n_cg / 8) * 8 * n_rb workgroups spread round-robin over the 8 XCDs, so with
// row blocks the column groups per block are a multiple of 8 (3 row blocks x 85 groups = 264
// workgroups put 33 on an XCD of 32 CUs: a second round, 1.7x the time, tools/rows_m_sweep.py).
__host__ inline int rows_grid(int MB, int N, int K, int num_cus, int* ntl_out, int n_rb = 1) {
  const int NT = N >> 4, cap = rows_tiles_cap(MB, K);
  const int per = n_rb > 1 ? (num_cus / n_rb / 8 * 8 > 0 ? num_cus / n_rb / 8 * 8 : 8) : num_cus;
  int n_cg = NT < per ? NT : per;
  if ((NT + n_cg - 1) / n_cg > cap) n_cg = (NT + cap - 1) / cap;
  *ntl_out = (NT + n_cg - 1) / n_cg;
  return n_cg;
}
// Rows per workgroup (16 RG MB): the fewest activation + weight bytes per workgroup over the
// launch's rounds -- a workgroup streams its rows' activations (R K 2 bytes, L2) and its tiles'
// weights (ntl 8 K bytes); narrow outputs (O, down) take 16-row blocks, wide ones all the rows.
// TI_GEMM_ROWS_SPLIT=0 keeps all rows in one workgroup (A/B knob).
__host__ inline void rows_plan(int M, int N, int K, int cus, int* MB, int* RG, int* n_rb, int* n_cg, int* ntl) {
  rows_shape(M, MB, RG);   // all rows in one workgroup
  *n_rb = 1;
  *n_cg = rows_grid(*MB, N, K, cus, ntl, 1);
  if (!gemm_knobs().rows_split) return;
  const int NT = N >> 4;
  auto cost = [&](int mb, int rg, int nrb, int ncg, int nt) {
    const long rounds = ((long)(ncg + 7) / 8 * 8 * nrb + cus - 1) / cus;
    return rounds * ((long)16 * rg * mb * K * 2 + (long)nt * 8 * K);
  };
  long best = cost(*MB, *RG, 1, *n_cg, *ntl);
  const int shapes[2][2] = {{1, 1}, {2, 1}};   // 16 and 32 rows per workgroup
  for (const auto& sh : shapes) {
    const int mb = sh[0], rg = sh[1], rows = 16 * mb * rg;
    if (rows >= M) continue;
    const int nrb = (M + rows - 1) / rows;
    int nt = 0;
    const int ncg = rows_grid(mb, N, K, cus, &nt, nrb);
    const long c = cost(mb, rg, nrb, ncg, nt);
    if (c * 20 < best * 17 && nt <= NT) {   // a clear (15 %) win only: the model ignores round overlap
      best = c;
      *MB = mb;
      *RG = rg;
      *n_rb = nrb;
      *n_cg = ncg;
      *ntl = nt;
    }
  }
}
template <int MB, int RG, bool XP>
static int launch_rows_t(const GemvArgs& a, int ntl, int n_cg, int n_rb, int lds, hipStream_t s) {
  const dim3 grid((unsigned)((n_cg + 7) / 8 * 8 * n_rb));
  if (ntl == 1) hipLaunchKernelGGL((gemm_rows_kernel<MB, 1, RG, XP>), grid, dim3(kGemvThreads), lds, s, a, n_cg, n_rb);
  else if (ntl == 2) hipLaunchKernelGGL((gemm_rows_kernel<MB, 2, RG, XP>), grid, dim3(kGemvThreads), lds, s, a, n_cg, n_rb);
  else if (ntl == 3) hipLaunchKernelGGL((gemm_rows_kernel<MB, 3, RG, XP>), grid, dim3(kGemvThreads), lds, s, a, n_cg, n_rb);
  else if constexpr (MB < 2) hipLaunchKernelGGL((gemm_rows_kernel<MB, 4, RG, XP>), grid, dim3(kGemvThreads), lds, s, a, n_cg, n_rb);
  else return ti_set_error(TI_ERR_ARG, "gemm_rows_kernel: %d tiles per workgroup at MB %d", ntl, MB);
  TI_LAUNCH_CHECK("gemm_rows_kernel");
  return TI_OK;
}
template <bool XP>
static int launch_rows_x(const GemvArgs& a, int MB, int RG, int ntl, int n_cg, int n_rb, int lds, hipStream_t s) {
  if (RG == 2)
    return MB == 1 ? launch_rows_t<1, 2, XP>(a, ntl, n_cg, n_rb, lds, s) : launch_rows_t<2, 2, XP>(a, ntl, n_cg, n_rb, lds, s);
  return MB == 1 ? launch_rows_t<1, 1, XP>(a, ntl, n_cg, n_rb, lds, s) : launch_rows_t<2, 1, XP>(a, ntl, n_cg, n_rb, lds, s);
}
static int launch_rows(const GemvArgs& a, int MB, int RG, int ntl, int n_cg, int n_rb, int lds, hipStream_t s) {
  return a.x_kind == TI_X_F16_PACKED ? launch_rows_x<true>(a, MB, RG, ntl, n_cg, n_rb, lds, s)
                                     : launch_rows_x<false>(a, MB, RG, ntl, n_cg, n_rb, lds, s);
}
#define TI_ROWS_FNS1(MB, RG, XP)                                                                      \
  (const void*)gemm_rows_kernel<MB, 1, RG, XP>, (const void*)gemm_rows_kernel<MB, 2, RG, XP>,            \
      (const void*)gemm_rows_kernel<MB, 3, RG, XP>
#define TI_ROWS_FNS2(XP)                                                                              \
  TI_ROWS_FNS1(1, 1, XP), TI_ROWS_FNS1(2, 1, XP), TI_ROWS_FNS1(1, 2, XP), TI_ROWS_FNS1(2, 2, XP),        \
      (const void*)gemm_rows_kernel<1, 4, 1, XP>, (const void*)gemm_rows_kernel<1, 4, 2, XP>
#define TI_ROWS_FNS TI_ROWS_FNS2(false), TI_ROWS_FNS2(true)

#define TI_MB_FNS1(K)                                                                                \
  (const void*)K<1, 1>, (const void*)K<1, 2>, (const void*)K<1, 3>, (const void*)K<1, 4>, (const void*)K<1, 5>, \
      (const void*)K<1, 6>, (const void*)K<1, 7>, (const void*)K<1, 8>
#define TI_MB_FNS TI_MB_FNS1(gemv_mbr_kernel)

// devices (bit per ordinal) whose attributes are set; engines may be driven from several threads
// (test_gpu_threads.py): fetch_or, and a repeated setup by a racing first call is harmless
static std::atomic<unsigned long long> g_prepared{0};

}  // namespace ti

// Raise the dynamic-LDS cap of the GEMM instantiations (call before any stream capture).
static int query_cus() {
  int n = ti::g_num_cus.load(std::memory_order_relaxed);
  if (n <= 0) {
    int dev = 0;
    if (!(hipGetDevice(&dev) == hipSuccess &&
          hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0))
      n = 256;
    ti::g_num_cus.store(n, std::memory_order_relaxed);
  }
  return n;
}

int ti::gemm_cus() { return query_cus(); }

extern "C" int ti_gemm_prepare(void) {
  using namespace ti;
  query_cus();
  int dev = 0;
  TI_HIP_CHECK(hipGetDevice(&dev), "hipGetDevice");
  const unsigned long long bit = 1ull << (dev & 63);
  if (g_prepared.load(std::memory_order_acquire) & bit) return TI_OK;
  const void* fns[] = {
      (const void*)gemv_wq_kernel<4, XM_F16>,  (const void*)gemv_wq_kernel<4, XM_F32>,
      (const void*)gemv_wq_kernel<4, XM_NORM1>, (const void*)gemv_wq_kernel<4, XM_NORM>,
      (const void*)gemv_wq_kernel<8, XM_F16>,  (const void*)gemv_wq_kernel<8, XM_F32>,
      (const void*)gemv_wq_kernel<8, XM_NORM1>, (const void*)gemv_wq_kernel<8, XM_NORM>,
      (const void*)gemv_wq_kernel<16, XM_F16>, (const void*)gemv_wq_kernel<16, XM_F32>,
      (const void*)gemv_wq_kernel<16, XM_NORM1>, (const void*)gemv_wq_kernel<16, XM_NORM>,
      (const void*)gemv_wq_kernel<4, XM_F16F>, (const void*)gemv_wq_kernel<8, XM_F16F>,
      (const void*)gemv_wq_kernel<16, XM_F16F>, (const void*)gemv_wq_kernel<4, XM_ATTN>,
      (const void*)gemv_wq_kernel<8, XM_ATTN>, (const void*)gemv_wq_kernel<16, XM_ATTN>, TI_MB_FNS, TI_ROWS_FNS};
  for (const void* f : fns)
    TI_HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                 "hipFuncSetAttribute(gemv_wq_kernel)");
  int rc = wide_prepare();
  if (rc == TI_OK) rc = few_prepare();
  if (rc == TI_OK) rc = block_prepare();
  if (rc != TI_OK) return rc;
  g_prepared.fetch_or(bit, std::memory_order_acq_rel);
  return TI_OK;
}

extern "C" int ti_gemm_lds_bytes(int M, int N, int K) {
  if (M < 1 || N < 16 || K < 128) return 0;
  const int NT = N >> 4, grid = ti::gemv_grid(M, N, K, query_cus());
  return ti::gemv_lds_bytes_tiles(M, K, (NT + grid - 1) / grid);
}

// The fused kernel takes the rows while its LDS image fits; int4 with fp16 activations
// also has the batched-rows kernel (up to TI_GEMM_MAX_ROWS rows, any K).
// int4 with more than 2 rows goes to the batched-rows kernel: from 4 rows on it is faster at
// every 7B projection (bench.py --batch 2..16, rocprof), at 2 rows the two tie.
static int fused_rows_pref(int bits) { return bits == 4 ? 2 : 16; }
static bool fused_fits(int M, int N, int K, bool g32 = false, bool aff = false) {
  if (M > 16) return false;
  const int NT = N >> 4, grid = ti::gemv_grid(M, N, K, query_cus(), g32, aff);
  return ti::gemv_lds_bytes_tiles(M, K, (NT + grid - 1) / grid, g32, aff) <= 160 * 1024;
}
static bool use_batched(int bits, int x_kind, int M, int N, int K) {
  const bool mb_ok = bits == 4 && x_kind == TI_X_F16;
  return !fused_fits(M, N, K) || (mb_ok && M > fused_rows_pref(bits));
}

// 17..64 int4 rows of a WIDE output take the many-rows kernel, whose workgroups copy a row's activations once per
// 64 columns or more, instead of the batched-rows kernel, which moves every row's activations per workgroup: from
// rows x N = 850000 on, and at 17..32 rows from N = 16384 on (measured, us, batched-rows / many-rows: 64 x 12288
// 19.0 / 18.4, 32 x 28672 36.5 / 19.6, 64 x 22016 35.5 / 27.3, 24 x 22016 25.2 / 19.2).
static bool wide_tile(int bits, int M, int N) {
  constexpr long kWideMN = 850000, kWideN32 = 16384;
  if (bits != 4 || M <= 16 || M >= ti::tile_rows()) return false;
  if (M <= 32 && N >= kWideN32) return true;
  return (long)M * N >= kWideMN;
}
extern "C" int ti_gemm_packed_rows(int bits, int M) { return bits == 4 && M > 16 && M < ti::tile_rows() ? 1 : 0; }
extern "C" int ti_gemm_packed_rows_for(int bits, int M, int N, int K) {
  (void)K;
  return ti_gemm_packed_rows(bits, M) && !wide_tile(bits, M, N) ? 1 : 0;
}

extern "C" int ti_gemm_fold_partials(int bits, int M, int N, int K) {
  if (bits != 4 || M <= 16 || M >= ti::tile_rows() || M > TI_FOLD_SS_ROWS || N < 16 || (N & 15) || K < 128 || (K & 127))
    return 0;
  int MB = 0, RG = 0, n_rb = 0, n_cg = 0, ntl = 0;
  ti::rows_plan(M, N, K, query_cus(), &MB, &RG, &n_rb, &n_cg, &ntl);
  return n_cg;
}

extern "C" int ti_gemm_tile_plan(int bits, int M, int N, int K, int64_t ws_bytes, int* wmr, int* tpw, int* n_ks) {
  if (!wmr || !tpw || !n_ks) return ti_set_error(TI_ERR_ARG, "ti_gemm_tile_plan: null pointer");
  if ((bits & ~TI_BITS_G32) != 4 || M < ti::tile_rows() || M > TI_GEMM_MAX_ROWS || N < 16 || (N & 15) || K < 128 ||
      (K & 127))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_tile_plan: M=%d N=%d K=%d bits %d is not a tile-kernel call", M, N,
                        K, bits);
  ti::WidePlan p;
  if (!ti::wide_plan(bits, M, N, K, query_cus(), ws_bytes, false, &p))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_tile_plan: M=%d N=%d K=%d bits %d", M, N, K, bits);
  // eight waves: one 64 x 384 workgroup, or two of four waves (64 x 128 or 64 x 64 each) on neighbouring row blocks
  *wmr = p.tiles == 24 ? 1 : 2;
  *tpw = p.tiles == 24 ? 3 : p.tiles / 4;
  *n_ks = p.n_ks;
  return TI_OK;
}

extern "C" int ti_gemm_max_rows(int bits, int x_kind, int N, int K) {
  if (N < 16 || K < 128) return 0;
  if (bits & TI_BITS_G32) {   // group-32 weights: the fused kernel; int4 fp16 rows also the tile kernel
    const bool aff = (bits & TI_BITS_AFF) != 0;   // (affine blocks: fused pieces only)
    if (x_kind == TI_X_F16_PACKED) return 0;
    if ((bits & ~(TI_BITS_G32 | TI_BITS_AFF)) == 4 && x_kind == TI_X_F16) return TI_GEMM_MAX_ROWS;   // 16-row pieces
    int m = 16;
    while (m > 1 && !fused_fits(m, N, K, true, aff)) --m;
    return fused_fits(m, N, K, true, aff) ? m : 0;
  }
  if (bits == 4 && (x_kind == TI_X_F16 || x_kind == TI_X_F16_PACKED)) return TI_GEMM_MAX_ROWS;
  if (x_kind == TI_X_F16_PACKED) return 0;
  int m = fused_rows_pref(bits);
  while (m > 1 && !fused_fits(m, N, K)) --m;
  return fused_fits(m, N, K) ? m : 0;
}

extern "C" int ti_rmsnorm_f16(const float* x, int ldx, const float* w, float eps, uint16_t* y, int ldy, int M, int K,
                              ti_stream_t stream) {
  if (!x || !w || !y) return ti_set_error(TI_ERR_ARG, "ti_rmsnorm_f16: null pointer");
  if (M < 1 || K < 8 || (K & 7) || ldx < K || ldy < K)
    return ti_set_error(TI_ERR_ARG, "ti_rmsnorm_f16: bad shape (M=%d K=%d ldx=%d ldy=%d)", M, K, ldx, ldy);
  ti_stamp_next(ti::STAMP_RMSNORM, 0);   // (unstamped; keeps the stamped step's launch list whole)
  hipLaunchKernelGGL(ti::rmsnorm_f16_kernel, dim3(M), dim3(ti::kGemvThreads), 0, (hipStream_t)stream, x, ldx, w, eps,
                     y, ldy, K, 0);
  TI_LAUNCH_CHECK("rmsnorm_f16_kernel");
  return TI_OK;
}

extern "C" int ti_rmsnorm_f16_packed(const float* x, int ldx, const float* w, float eps, uint16_t* y, int M, int K,
                                     ti_stream_t stream) {
  if (!x || !w || !y) return ti_set_error(TI_ERR_ARG, "ti_rmsnorm_f16_packed: null pointer");
  if (M < 1 || K < 128 || (K & 127) || ldx < K)
    return ti_set_error(TI_ERR_ARG, "ti_rmsnorm_f16_packed: bad shape (M=%d K=%d ldx=%d)", M, K, ldx);
  ti_stamp_next(ti::STAMP_RMSNORM, 0);   // (unstamped; keeps the stamped step's launch list whole)
  hipLaunchKernelGGL(ti::rmsnorm_f16_kernel, dim3(M), dim3(ti::kGemvThreads), 0, (hipStream_t)stream, x, ldx, w, eps,
                     y, K, K, K >> 7);
  TI_LAUNCH_CHECK("rmsnorm_f16_kernel");
  return TI_OK;
}

static int gemm_impl(const void* tiles, const uint16_t* scales, int bits, const void* x, int x_kind, int ldx,
                     const float* norm_w, float eps, int M, int N, int K, const ti_epilogue* epi,
                     ti_stream_t stream) {
  using namespace ti;
  if (!tiles || !x || !epi || !epi->out) return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: null pointer");
  const bool g32 = (bits & TI_BITS_G32) != 0, aff = (bits & TI_BITS_AFF) != 0;
  bits &= ~(TI_BITS_G32 | TI_BITS_AFF);
  if ((bits != 4 && bits != 8 && bits != 16) || (g32 && bits == 16) || (aff && (!g32 || bits != 4)))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: bits must be 4, 8 or 16 (+ TI_BITS_G32 for 4 / 8, + TI_BITS_AFF "
                        "for 4 | G32; got %d)", bits);
  // int4 fp16 rows, row-major: the many-rows kernel (gemm_wide.hip) from 65 rows on and for wide outputs from 17 (the
  // batched-rows kernel below that: the packed and the row-major form of a call give the same bits), group-32 from 17,
  // where its 16-byte row pieces are aligned; affine blocks, int8 and fp16 weights run the fused kernel here
  // (ti_gemm_rows: any format).  Blocks of 32 write no packed output
  const int64_t ws_bytes = epi->splitk_ws ? epi->splitk_bytes : 0;
  WidePlan wp;
  const bool wide = bits == 4 && !aff && x_kind == TI_X_F16 && M > 16 && (g32 ? !epi->out_packed : M >= tile_rows() || wide_tile(bits, M, N)) &&
                    rows_aligned(x, ldx) && wide_plan(bits | (g32 ? TI_BITS_G32 : 0), M, N, K, query_cus(), ws_bytes, epi->ss_in, &wp);
  int g32_rows = 16;   // rows per fused launch (its LDS image holds the x rows)
  while (g32 && g32_rows > 1 && !fused_fits(g32_rows, N, K, true, aff)) --g32_rows;
  if (g32 && (x_kind == TI_X_F16_PACKED || (!wide && !fused_fits(std::min(M, g32_rows), N, K, true, aff))))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: group-32 weights: fused kernel rows (M=%d N=%d K=%d) "
                        "or int4 fp16 rows >= %d; no packed rows", M, N, K, tile_rows());
  if (bits != 16 && !scales) return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: scales required for bits %d", bits);
  if (M < 1 || M > TI_GEMM_MAX_ROWS)
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: M must be in [1,%d] (got %d)", TI_GEMM_MAX_ROWS, M);
  if (K <= 0 || (K & 127) || N <= 0 || (N & 15))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: K %% 128 and N %% 16 must be 0 (K=%d N=%d)", K, N);
  if (x_kind < TI_X_F16 || x_kind > TI_X_F16_PACKED)
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: bad x_kind %d", x_kind);
  if (x_kind == TI_X_F16_PACKED && bits != 4)
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: TI_X_F16_PACKED needs bits 4 (batched-rows kernel)");
  if (x_kind == TI_X_ATTN_SPLITS &&
      (M != 1 || !epi->ss_in || epi->n_ss < 1 || epi->n_ss > TI_ATTN_MAX_PART_SPLITS ||
       (epi->head_dim != 64 && epi->head_dim != 128) || K % epi->head_dim || K > 4096))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: TI_X_ATTN_SPLITS needs M == 1, ss_in, 1 <= n_ss <= %d, head_dim "
                        "64/128 and K <= 4096", TI_ATTN_MAX_PART_SPLITS);
  if (x_kind == TI_X_F16_FOLDED && (M != 1 || !epi->ss_in || epi->n_ss < 1 || epi->n_ss > 256))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: TI_X_F16_FOLDED needs M == 1, ss_in and 1 <= n_ss <= 256");
  const bool fold_out = epi->kind == TI_EPI_RESID_F32 && epi->fold_x;
  if (fold_out && M == 1 && (!epi->fold_w || !epi->fold_ss || (x_kind != TI_X_F16 && x_kind != TI_X_ATTN_SPLITS)))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: fold_x needs M == 1, fp16 x, fold_w and fold_ss");
  if (fold_out && M > 1 && (!epi->fold_w || !epi->fold_ss || x_kind != TI_X_F16_PACKED || M > TI_FOLD_SS_ROWS ||
                            (N & 127)))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: a batched fold_x needs TI_X_F16_PACKED x, M <= %d, fold_w, "
                        "fold_ss and N %% 128 == 0", TI_FOLD_SS_ROWS);
  // batched fold consumer: fp16(h * nw) rows normalised behind the GEMM (rows / tile kernels)
  const bool fold_in = M > 1 && epi->ss_in && (x_kind == TI_X_F16 || x_kind == TI_X_F16_PACKED);
  if (fold_in && (M > TI_FOLD_SS_ROWS || epi->n_ss < 1 || epi->n_ss > 4096))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: a batched folded input needs M <= %d and 1 <= n_ss <= 4096",
                        TI_FOLD_SS_ROWS);
  if (K > 0xffff || ldx > 0xffff)
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: K %d / ldx %d above 65535", K, ldx);
  if (x_kind == TI_X_F32_RMSNORM && !norm_w) return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: norm_w required");
  if (ldx < K) return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: ldx %d < K %d", ldx, K);
  {
    const int rc = check_epilogue(*epi, N, "ti_gemm_wq_a16");
    if (rc != TI_OK) return rc;
  }
  // pieces of rows: group-32 through the fused kernel; int4 rows past the batched-rows kernel that are not aligned
  const int piece = wide ? 0 : g32 && M > g32_rows ? g32_rows : !g32 && bits == 4 && x_kind == TI_X_F16 && M >= tile_rows() ? tile_rows() - 1 : 0;
  if (piece) {
    if (x_kind == TI_X_ATTN_SPLITS || x_kind == TI_X_F16_FOLDED || (epi->out_packed && g32))
      return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: rows in pieces need plain x rows");
    const size_t x_elem = x_kind == TI_X_F16 ? 2 : 4;
    const size_t out_elem = epi->kind == TI_EPI_STORE_F16 || epi->kind == TI_EPI_SILU_MUL_F16 ? 2 : 4;
    for (int m0 = 0, mm; m0 < M; m0 += mm) {
      mm = std::min(piece, M - m0);
      if (epi->out_packed && M - m0 > piece && M - m0 <= piece + 16) mm = piece - 16;   // (packed outputs need more than 16 rows)
      ti_epilogue ep = *epi;
      ep.out = static_cast<char*>(epi->out) + (size_t)m0 * epi->ldo * out_elem;
      if (ep.pos) ep.pos += m0;
      if (ep.k_cache) ep.k_cache += (size_t)m0 * ep.kv_stream_stride;
      if (ep.v_cache) ep.v_cache += (size_t)m0 * ep.kv_stream_stride;
      if (ep.argmax) ep.argmax += (size_t)m0 * TI_ARGMAX_SLOTS;
      if (m0 + mm < M) ep.step_ctr = nullptr;
      const int rc = gemm_impl(tiles, scales, bits | (g32 ? TI_BITS_G32 : 0) | (aff ? TI_BITS_AFF : 0),
                               static_cast<const char*>(x) + (size_t)m0 * ldx * x_elem,
                               x_kind, ldx, norm_w, eps, mm, N, K, &ep, stream);
      if (rc != TI_OK) return rc;
    }
    return TI_OK;
  }
  const bool packed_x = x_kind == TI_X_F16_PACKED;
  const bool batched = wide || (!g32 && (packed_x || use_batched(bits, x_kind, M, N, K)));
  if (epi->out_packed && (!batched || (epi->kind != TI_EPI_STORE_F16 && epi->kind != TI_EPI_SILU_MUL_F16) ||
                          (epi->ldo & 127)))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_wq_a16: out_packed needs the batched-rows kernel, a fp16 store / SiLU "
                        "epilogue and ldo %% 128 == 0");
  if (batched && fold_out && M == 1)
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: fold_x needs the fused kernel");
  if (batched && !(bits == 4 && (x_kind == TI_X_F16 || packed_x)))
    return ti_set_error(TI_ERR_UNSUPPORTED,
                        "ti_gemm_wq_a16: M=%d K=%d exceeds the fused kernel (ti_gemm_max_rows); the batched-rows "
                        "kernel needs bits 4 and fp16 rows (normalise with ti_rmsnorm_f16)", M, K);
  int grid = 0, lds = 0, ntl = 0, rMB = 0, rRG = 0, r_rb = 1;
  const bool rows = !wide && batched && M > 16;
  if (wide) {
    // (its plan has the grid)
  } else if (rows) {
    rows_plan(M, N, K, query_cus(), &rMB, &rRG, &r_rb, &grid, &ntl);   // grid: column groups
    lds = rows_lds_bytes(rRG * rMB, ntl, K);
  } else if (batched) {
    grid = mb_grid(1, N, K, query_cus(), &ntl);
    lds = mbr_lds_bytes(1, ntl, K);
  } else {
    grid = gemv_grid(M, N, K, query_cus(), g32, aff);
    lds = gemv_lds_bytes_tiles(M, K, ((N >> 4) + grid - 1) / grid, g32, aff);
  }
  if ((fold_out && M > 1 && !rows) || (fold_in && !rows && !wide))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: the batched fold runs on the batched-rows (fold_x) / "
                        "rows or many-rows (folded input) kernels (M=%d N=%d K=%d)", M, N, K);
  if (lds > 160 * 1024)
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: LDS image %d B too large (M=%d N=%d K=%d)", lds, M, N, K);
  if (!batched && grid > 0xfff)
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_wq_a16: %d workgroups (N=%d) above 4095", grid, N);
  if (wide || lds > 64 * 1024) {   // no-op once this device is prepared
    const int rc = ti_gemm_prepare();
    if (rc != TI_OK) return rc;
  }
  GemvArgs a;
  a.tiles = (const u32x4*)tiles;
  a.scales = scales;
  a.x = x;
  a.norm_w = norm_w;
  a.eps = eps;
  a.x_kind = x_kind;
  a.ldx = ldx;
  a.M = M;
  a.N = N;
  a.K = K;
  a.epi = *epi;
  a.vec = epilogue_vec(*epi);
  {   // workgroups of the launch below (stamp buffer sizing)
    const long wgs = wide ? wide_workgroups(wp) : rows ? (long)((grid + 7) / 8 * 8) * r_rb : grid;
    a.stamp = ti_stamp_next(wide ? STAMP_TILE : rows ? STAMP_ROWS : batched ? STAMP_MB : STAMP_GEMV, wgs);
  }
  hipStream_t s = (hipStream_t)stream;
  if (wide) a.norm_w = nullptr;
  if (wide) return wide_launch(bits | (g32 ? TI_BITS_G32 : 0), wp, a, s);
  if (rows) return launch_rows(a, rMB, rRG, ntl, grid, r_rb, lds, s);
  if (batched) return launch_mb(a, grid, ntl, lds, s);
  if (aff) return launch_gemv<4, true, true>(a, lds, s, grid);
  if (g32) return bits == 4 ? launch_gemv<4, true>(a, lds, s, grid) : launch_gemv<8, true>(a, lds, s, grid);
  if (bits == 4) return launch_gemv<4>(a, lds, s, grid);
  if (bits == 8) return launch_gemv<8>(a, lds, s, grid);
  return launch_gemv<16>(a, lds, s, grid);
}

extern "C" int ti_epilogue_bytes(void) { return (int)sizeof(ti_epilogue); }

// The kernel ti_gemm_wq_a16 launches for plain (not group-32) weights: the same predicates as
// gemm_impl (use_batched, wide_tile, tile_rows, rows_on).  For bench / profile labels.
extern "C" int ti_gemm_kernel_name(int bits, int x_kind, int M, int N, int K, char* buf, int len) {
  using namespace ti;
  if (!buf || len < 1) return ti_set_error(TI_ERR_ARG, "ti_gemm_kernel_name: null buffer");
  if ((bits != 4 && bits != 8 && bits != 16) || M < 1 || M > TI_GEMM_MAX_ROWS || N < 16 || K < 128)
    return ti_set_error(TI_ERR_ARG, "ti_gemm_kernel_name: bits %d M %d N %d K %d", bits, M, N, K);
  const bool packed_x = x_kind == TI_X_F16_PACKED;
  const bool batched = packed_x || use_batched(bits, x_kind, M, N, K);
  const bool wide = batched && x_kind == TI_X_F16 && (M >= tile_rows() || wide_tile(bits, M, N)), rows = !wide && batched && M > 16;
  const char* name = wide ? "gemm_wide_kernel" : rows ? "gemm_rows_kernel" : batched ? "gemv_mbr_kernel" : nullptr;
  if (name) snprintf(buf, (size_t)len, "%s", name);
  else snprintf(buf, (size_t)len, "gemv_wq_kernel<%d,%d>", bits, gemv_xmode(x_kind, M, K));
  return TI_OK;
}

extern "C" int ti_gemm_grid(int M, int N, int K) {
  if (M < 1 || M > 16 || N < 16 || K < 128 || (N & 15) || (K & 127) || !fused_fits(M, N, K)) return 0;
  return ti::gemv_grid(M, N, K, query_cus());
}

extern "C" int ti_gemm_wq_a16(const void* tiles, const uint16_t* scales, int bits, const void* x,
                              int x_kind, int ldx, const float* norm_w, float eps, int M, int N, int K,
                              const ti_epilogue* epi, ti_stream_t stream) {
  return gemm_impl(tiles, scales, bits, x, x_kind, ldx, norm_w, eps, M, N, K, epi, stream);
}

