// gemm_wide.hpp -- the many-rows GEMM (gemm_wide.hip): row-major fp16 x against packed weights of every format.
#pragma once
#include "gemm_common.hpp"

namespace ti {

// Formats by their bits value (ti_hip.h): 4, 8, 16, 4 | 32, 8 | 32, 4 | 32 | 64.
template <int F>
struct WideFmt {
  static constexpr int kBits = F & 31;
  static constexpr bool kG32 = (F & TI_BITS_G32) != 0, kAff = (F & TI_BITS_AFF) != 0;
  static constexpr int kTile = kBits * 256;                               // bytes of a 16 x 128 weight tile
  static constexpr int kScale = kBits == 16 ? 0 : kG32 ? 128 : 32;        // bytes of its scales
};

// Batched fold: a column block's sum of h^2 of a row is negative where fp16 does not hold its h w, the lowest bit of the
// mantissa 0 where one of them passes 65504, 1 where they are small (wide_fold_store; an infinite sum counts as the former).
// A row is normalised before it is rounded if one block of it is past 65504 or more than half of them are small: small ones
// beside others are within the row's rounding, and what is done does not hang on the blocks' width.
__device__ __forceinline__ float fold_mark(float t, bool over, bool small) {
  const uint32_t b = __builtin_bit_cast(uint32_t, t);
  if (over) return __builtin_bit_cast(float, (b & ~1u) | 0x80000000u);
  return small ? __builtin_bit_cast(float, b | (t < INFINITY ? 0x80000001u : 0x80000000u)) : t;
}
// Consumer side: this thread's share of row m's partial sums (part, part + P, ...), summed in order; negative if one of them is.
__device__ __forceinline__ float wide_fold_share(const GemvArgs& a, int m, int part, int P) {
  float t = 0.0f;
  uint32_t any = 0;
  if (m >= a.M) return t;
  const float* ss = a.epi.ss_in + m;
  for (int b0 = part; b0 < a.epi.n_ss; b0 += 16 * P) {
    float v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = b0 + j * P < a.epi.n_ss ? ss[(size_t)(b0 + j * P) * TI_FOLD_SS_ROWS] : 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      t += fabsf(v[j]);
      any |= __builtin_bit_cast(uint32_t, v[j]);
    }
  }
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, t) | (any & 0x80000000u));
}
// The threads' shares to the rms of every row, negative as they are (behind a barrier; one follows).
template <int ROWS, int NW>
__device__ __forceinline__ void wide_fold_rms(const GemvArgs& a, float share, int tid, float* rmsv) {
  rmsv[ROWS + tid] = share;
  lds_barrier();
  if (tid < ROWS) {
    float t = 0.0f;
    uint32_t any = 0;
    for (int p = 0; p < 64 * NW / ROWS; ++p) {
      const float v = rmsv[ROWS + p * ROWS + tid];
      t += fabsf(v);
      any |= __builtin_bit_cast(uint32_t, v);
    }
    rmsv[tid] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, sqrtf(t / (float)a.K + a.eps)) | (any & 0x80000000u));
  }
  lds_barrier();
}
// Where a row's rms is negative: the marks counted, the rms of rows that are taken as they are made positive (behind a barrier; one
// follows).  Apart, so that calls without a mark do not pay for it (0.1 us each).
template <int ROWS, int NW>
__device__ __forceinline__ void wide_fold_settle(const GemvArgs& a, int m0, int tid, float* rmsv) {
  constexpr int P = 64 * NW / ROWS;
  uint32_t* marks = (uint32_t*)rmsv + ROWS;   // small blocks; the top bit: one is past 65504
  const int m = m0 + tid % ROWS, part = tid / ROWS;
  uint32_t n = 0, over = 0;
  for (int b0 = m < a.M && part < P ? part : a.epi.n_ss; b0 < a.epi.n_ss; b0 += 16 * P) {
    uint32_t v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      v[j] = b0 + j * P < a.epi.n_ss ? __builtin_bit_cast(uint32_t, a.epi.ss_in[(size_t)(b0 + j * P) * TI_FOLD_SS_ROWS + m]) : 0u;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      n += v[j] & (v[j] >> 31);
      over |= v[j] & ~(v[j] << 31);
    }
  }
  marks[tid] = n | (over & 0x80000000u);
  lds_barrier();
  if (tid < ROWS && rmsv[tid] < 0.0f) {
    n = over = 0;
#pragma unroll 8
    for (int p = 0; p < P; ++p) {
      n += marks[p * ROWS + tid] & 0xffffu;
      over |= marks[p * ROWS + tid];
    }
    if ((int32_t)over >= 0 && 2 * (int)n <= a.epi.n_ss) rmsv[tid] = -rmsv[tid];
  }
  lds_barrier();
}
// The rows (from m0) whose rms is negative as ti_rmsnorm_f16 gives them.  Every workgroup rewrites them whole, with the same values,
// before it reads them: a chain of loads per piece, so a row's pieces fly 4 at a time (Llama-2-7B int4 with every row like this, us,
// one at a time -> this: steps of 3 rows 2807 -> 2710, of 24 5713 -> 4950, prompts of 20 5049 -> 4420, of 64 10400 -> 7941;
// none of them 1650, 2340, 2070 and 2760).
template <int ROWS, int NW>
__device__ __forceinline__ void wide_refold(const GemvArgs& a, int m0, int wave, int lane, const float* rmsv) {
  typedef f16 f16x4 __attribute__((ext_vector_type(4)));
  constexpr int U = 4;
#pragma unroll 1
  for (int m = wave; m < ROWS; m += NW) {   // (rows past M have a positive one)
    const float rms = -rmsv[m];
    if (__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, rms)) < 0) continue;
#pragma unroll 1
    for (int k0 = 0; k0 < a.K; k0 += 4 * kWave * U) {   // (K is a multiple of 128: past it, lanes repeat the last piece)
      f32x4 v[U], w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = min(k0 + 4 * (kWave * u + lane), a.K - 4);
        v[u] = *(const f32x4*)(a.epi.fold_w + (size_t)(m0 + m) * a.K + k);
        w[u] = *(const f32x4*)(a.norm_w + k);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        f16x4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = mul_f16(v[u][i] / rms, w[u][i]);
        *(f16x4*)((f16*)a.x + (size_t)(m0 + m) * a.ldx + min(k0 + 4 * (kWave * u + lane), a.K - 4)) = y;
        __builtin_amdgcn_sched_barrier(0);   // (one piece's divisions at a time: registers)
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
}

// One weight tile's outputs (16 columns from tn) for the 16 TM rows from mb, from the wave's staging block and what tile_pre
// fetched.  fold_out: the residual add and the next call's folded input; hsq, psq: the lane's sums of h^2 and of (h w)^2, the latter infinite where an
// |h w| passes 65504 (wide_fold_part).
template <int TM>
__device__ __forceinline__ void wide_tile_out(const GemvArgs& a, int tn, int mb, const float* stg, int lane, int r, int kq, bool fold_out,
                                              const TilePre<TM>& pre, float (&hsq)[TM], float (&psq)[TM]) {
  const ti_epilogue& e = a.epi;
  if (fold_out) {   // residual add + the next call's folded input (fp16(h * w), sum of h^2 per row)
    const int c4 = 4 * (lane & 3), ng = tn * 16 + c4;
    const float4 w = *(const float4*)(e.fold_w + ng);
#pragma unroll
    for (int it = 0; it < TM; ++it) {
      const int row = 16 * it + (lane >> 2), m = mb + row;
      const float4 v = *(const float4*)(stg + row * kTileEpiStride + c4);
      float q = 0.0f;
      if (m < a.M) {
        float4* o = (float4*)((float*)e.out + (size_t)m * e.ldo + ng);
        const float4 h0 = pre.v[it], h = make_float4(h0.x + v.x, h0.y + v.y, h0.z + v.z, h0.w + v.w);
        *o = h;
        float p[4] = {h.x * w.x, h.y * w.y, h.z * w.z, h.w * w.w};
        // (largest |p|; as outputs the products are rounded on their own, as in mul_f16)
        float top = 0.0f;
        asm("v_max3_f32 %0, %0, |%1|, |%2|\n\tv_max3_f32 %0, %0, |%3|, |%4|" : "+v"(top), "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
        auto f = [](float v) { return (uint32_t)f2h(v); };
        *(uint2*)(e.fold_x + (size_t)m * e.ldo + ng) = make_uint2(f(p[0]) | (f(p[1]) << 16), f(p[2]) | (f(p[3]) << 16));
        q = (h.x * h.x + h.y * h.y) + (h.z * h.z + h.w * h.w);
        psq[it] = top > 65504.0f ? INFINITY : fmaf(p[0], p[0], fmaf(p[1], p[1], fmaf(p[2], p[2], fmaf(p[3], p[3], psq[it]))));
      }
      q += lane_xor<1>(q);
      hsq[it] += q + lane_xor<2>(q);
    }
  } else if (a.vec) {
    tile_epilogue_lds<TM>(a, tn, mb, stg, lane, pre);
  } else {
#pragma unroll 1
    for (int q = 0; q < TM * 4; ++q) {
      const int row = q * 4 + kq, m = mb + row;
      epilogue_mb(a, tn, min(m, a.M - 1), r, stg[row * kTileEpiStride + r], m < a.M);
    }
  }
}
// The wave's sums of its 16 TM rows to part.
template <int TM>
__device__ __forceinline__ void wide_fold_part(float2* part, const float (&hsq)[TM], const float (&psq)[TM], int lane) {
#pragma unroll
  for (int it = 0; it < TM; ++it) {
    const float p2 = psq[it] + lane_xor<1>(psq[it]), p4 = p2 + lane_xor<2>(p2);
    if ((lane & 3) == 0) part[16 * it + (lane >> 2)] = make_float2(hsq[it], p4);
  }
}
// The W parts of a block of TILES weight tiles (behind a barrier), in order, to fold_ss.  Small: their mean square below 2^-23.
// fp16's steps of 2^-24 raise its rounding error, 2.08e-4 of a row of normal deviates, by 0.1 % at an rms of 2^-11.5, 1 % at
// 2^-12 and 7 % at 2^-13; a model of norm weights of 0.02 .. 0.05 on embeddings of up to 0.02 starts at 2^-11.2.
template <int ROWS, int W, int TILES>
__device__ __forceinline__ void wide_fold_store(const GemvArgs& a, const float2* part, int cb, int m0, int tid) {
  if (tid >= ROWS || m0 + tid >= a.M) return;
  float t = 0.0f, p = 0.0f;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float2 v = part[w * ROWS + tid];
    t += v.x;
    p += v.y;
  }
  const int cols = min(16 * TILES, a.N - cb * 16 * TILES);
  a.epi.fold_ss[(size_t)cb * TI_FOLD_SS_ROWS + m0 + tid] = fold_mark(t, p == INFINITY, p < (float)cols * 0x1p-23f);
}

struct WidePlan {
  int shape;             // workgroup shape (gemm_wide.hip), -1: none
  int n_cb, n_rb, n_ks;  // column blocks x row blocks x k-slices
  int rows, tiles;       // of a block
  float us, whole;       // estimate; the same with a split's seam as it is beside other launches (for the choice between kernels)
};
// fmt: the bits of ti_gemm_wq_a16.  fold: a call with a folded input or output.  only: the one shape to consider (-1: all).  False: not a
// call of this kernel (shape or format).
bool wide_plan(int fmt, int M, int N, int K, int cus, int64_t ws_bytes, bool fold, WidePlan* p, int only = -1);
long wide_workgroups(const WidePlan& p);
int wide_launch(int fmt, const WidePlan& p, const GemvArgs& a, hipStream_t s);
int gemm_cus();       // CUs of the current device (gemv.hip)
int wide_prepare();   // dynamic-LDS limits on the current device


// gemm_few.hip: up to 48 rows, a workgroup's waves split K
struct FewPlan {
  int shape, n_cb;   // workgroup shape, column blocks
  float us;          // estimate
};
bool few_plan(int fmt, int M, int N, int K, int cus, FewPlan* p, int only = -1);
long few_workgroups(const FewPlan& p);
int few_launch(int fmt, const FewPlan& p, const GemvArgs& a, hipStream_t s);
int few_prepare();

// gemm_block.hip: 17 rows and more (fp16: 33) (outputs of whole 16-byte pieces, a.vec).  fold: a call with a folded input or output.
struct BlockPlan {
  int shape, n_cb, n_rb;   // workgroup shape, column blocks x row blocks
  bool fold;
  float us;                // estimate
};
bool block_plan(int fmt, int M, int N, int K, int cus, bool fold, BlockPlan* p, int only = -1);
long block_workgroups(const BlockPlan& p);
int block_launch(int fmt, const BlockPlan& p, const GemvArgs& a, hipStream_t s);
int block_prepare();

}  // namespace ti
