// gemm_common.hpp -- what the weight x fp16 GEMM kernels share (gemv.hip, gemm_wide.hip): launch arguments,
// weight loads, the barrier that leaves loads in flight, the epilogues of ti_gemm_wq_a16 and the batched fold.
#pragma once
#include <math.h>
#include <stdlib.h>

#include "common.hpp"
#include "dequant.hpp"

#ifndef TI_GEMV_EXP
#define TI_GEMV_EXP 0   // product build; tools/probe_gemv.hip compiles diagnostic variants
#endif

namespace ti {

constexpr int kGemvWaves = 8;
constexpr int kGemvThreads = kGemvWaves * kWave;

struct GemvArgs {
  const u32x4* tiles;
  const uint16_t* scales;
  const void* x;
  const float* norm_w;         // (gemm_wide_kernel: of a folded input whose rows are at hand as epi.fold_w, or NULL)
  float eps;
  int32_t x_kind, ldx, M, N, K;
  ti_epilogue epi;
  int32_t vec;                 // the epilogue's outputs and inputs may be accessed four columns at a time (epilogue_vec)
  unsigned long long* stamp;   // in-step launch stamps (common.hpp stamp_end), NULL in product launches
};

// 16-byte pieces of fp16 rows
__host__ inline bool rows_aligned(const void* x, int ldx) { return ((uintptr_t)x & 15) == 0 && (ldx & 7) == 0; }

// Whether four columns of an output row (and of what the epilogue reads beside it) are one aligned access: 16 bytes of
// fp32, 8 of fp16; a rotary head is whole 16-column tiles.
__host__ inline int epilogue_vec(const ti_epilogue& e) {
  auto al = [](const void* p, unsigned n) { return ((uintptr_t)p & (n - 1)) == 0; };
  switch (e.kind) {
    case TI_EPI_STORE_F32: case TI_EPI_LOGITS_ARGMAX: return al(e.out, 16) && (e.ldo & 3) == 0;
    case TI_EPI_RESID_F32: return al(e.out, 16) && (e.ldo & 3) == 0 && (!e.fold_x || (al(e.fold_x, 8) && al(e.fold_w, 16)));
    case TI_EPI_SILU_MUL_F16: return !e.out_packed && al(e.out, 8) && (e.ldo & 3) == 0;
    case TI_EPI_QKV_ROPE_KV:
      return al(e.out, 16) && (e.ldo & 3) == 0 && (e.head_dim & 15) == 0 && al(e.rope_cs, 16) && al(e.k_cache, 8) && al(e.v_cache, 8) &&
             (e.kv_stream_stride & 3) == 0;
    default: return 0;
  }
}

__host__ inline int check_epilogue(const ti_epilogue& e, int N, const char* who) {
  switch (e.kind) {
    case TI_EPI_STORE_F32: case TI_EPI_STORE_F16: case TI_EPI_RESID_F32:
      if (e.ldo < N) return ti_set_error(TI_ERR_ARG, "%s: ldo %d < N %d", who, e.ldo, N);
      return TI_OK;
    case TI_EPI_SILU_MUL_F16:
      if (e.ldo < N / 2) return ti_set_error(TI_ERR_ARG, "%s: ldo < N/2", who);
      return TI_OK;
    case TI_EPI_QKV_ROPE_KV:
      if (!e.pos || !e.rope_cs || !e.k_cache || !e.v_cache || e.head_dim <= 0 || e.head_dim > 128 || (e.head_dim & 1) ||
          e.q_dim + 2 * e.kv_dim != N || e.q_dim % e.head_dim || e.kv_dim % e.head_dim || e.ldo < e.q_dim)
        return ti_set_error(TI_ERR_ARG, "%s: inconsistent QKV epilogue", who);
      return TI_OK;
    case TI_EPI_LOGITS_ARGMAX:
      if (!e.argmax || e.ldo < N) return ti_set_error(TI_ERR_ARG, "%s: argmax/ldo", who);
      return TI_OK;
    default:
      return ti_set_error(TI_ERR_ARG, "%s: unknown epilogue %d", who, e.kind);
  }
}

__host__ __device__ constexpr int align16(int b) { return (b + 15) & ~15; }

// The GEMM's two remaining A/B knobs, read once per process (thread-safe static init).
struct GemmKnobs {
  bool splitk = true;       // TI_GEMM_SPLITK=0: no split-K for under-filled tile grids
  bool rows_split = true;   // TI_GEMM_ROWS_SPLIT=0: all rows in one batched-rows workgroup
};
__host__ inline const GemmKnobs& gemm_knobs() {
  static const GemmKnobs k = [] {
    GemmKnobs v;
    if (const char* e = getenv("TI_GEMM_SPLITK")) v.splitk = atoi(e) != 0;
    if (const char* e = getenv("TI_GEMM_ROWS_SPLIT")) v.rows_split = atoi(e) != 0;
    return v;
  }();
  return k;
}

// Weight stream load: read once per launch, so non-temporal where that pays (TI_GEMV_NT).
#ifndef TI_GEMV_NT
#define TI_GEMV_NT 1
#endif
__device__ __forceinline__ u32x4 ld_w(const u32x4* p) {
#if TI_GEMV_NT || (TI_GEMV_EXP & 16)
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}

// LDS barrier that leaves the wave's outstanding global loads in flight (a plain
// __syncthreads() may drain vmcnt): LDS writes retired, then s_barrier.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ f16x8 deq_int4_signed(uint32_t w, uint32_t magic) {
  const f16x8 r = deq_int4_raw(w, magic);   // lanes (1024 + n) and (1024 + 16 n)
  const f16x2 lo_off = {(f16)-1032.0f, (f16)-1032.0f}, hi_mul = {(f16)0.0625f, (f16)0.0625f},
              hi_off = {(f16)-72.0f, (f16)-72.0f};
  // (1024 + 16 n) / 16 - 72 = n - 8 exactly: one v_pk_fma_f16 (the build's -ffp-contract=off
  // would otherwise split it into a multiply and an add)
  const f16x2 a = (f16x2){r[0], r[1]} + lo_off, b = __builtin_elementwise_fma((f16x2){r[2], r[3]}, hi_mul, hi_off);
  const f16x2 c = (f16x2){r[4], r[5]} + lo_off, d = __builtin_elementwise_fma((f16x2){r[6], r[7]}, hi_mul, hi_off);
  return (f16x8){a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// Epilogue of one output y[m][nt*16 + n]; the inputs gemv_wq_kernel stages in LDS are read
// from global.  Shuffle partners (n ^ 1, n + 8) are lanes of the same 16-lane group.
__device__ __forceinline__ void epilogue_mb(const GemvArgs& a, int nt, int m, int n, float v, bool live) {
  const ti_epilogue& e = a.epi;
  const int ng = nt * 16 + n;
  switch (e.kind) {
    case TI_EPI_STORE_F32:
      if (live) ((float*)e.out)[(size_t)m * e.ldo + ng] = v;
      break;
    case TI_EPI_STORE_F16:
      if (live)
        ((uint16_t*)e.out)[e.out_packed ? TI_PACKED_INDEX(m, ng, e.ldo >> 7) : (size_t)m * e.ldo + ng] = f2h(v);
      break;
    case TI_EPI_RESID_F32:
      if (live) {
        float* o = (float*)e.out + (size_t)m * e.ldo + ng;
        *o = *o + v;
      }
      break;
    case TI_EPI_SILU_MUL_F16: {
      const float up = __shfl_down(v, 8, kWave);
      if (live && n < 8) {
        const float s = v / (1.0f + expf(-v));
        const int j = nt * 8 + n;
        ((uint16_t*)e.out)[e.out_packed ? TI_PACKED_INDEX(m, j, e.ldo >> 7) : (size_t)m * e.ldo + j] = f2h(up * s);
      }
      break;
    }
    case TI_EPI_QKV_ROPE_KV: {
      const float partner = __shfl_xor(v, 1, kWave);
      if (!live) break;
      const int hd = e.head_dim, p = e.pos[m];
      if (ng < e.q_dim + e.kv_dim) {
        const int base = ng < e.q_dim ? 0 : e.q_dim;
        const int d = (ng - base) % hd;
        const float2 cs = *(const float2*)(e.rope_cs + (size_t)p * hd + (d & ~1));
        const float r = (d & 1) == 0 ? fmaf(-partner, cs.y, v * cs.x) : fmaf(v, cs.x, partner * cs.y);
        if (ng < e.q_dim) {
          ((float*)e.out)[(size_t)m * e.ldo + ng] = r;
        } else {
          const int kvh = (ng - e.q_dim) / hd;
          e.k_cache[(size_t)m * e.kv_stream_stride + ((size_t)kvh * e.max_seq + p) * hd + d] = f2h(r);
        }
      } else {
        const int c = ng - e.q_dim - e.kv_dim;
        const int kvh = c / hd, d = c - kvh * hd;
        e.v_cache[(size_t)m * e.kv_stream_stride + ((size_t)kvh * e.max_seq + p) * hd + d] = f2h(v);
      }
      break;
    }
    case TI_EPI_LOGITS_ARGMAX: {
      unsigned long long key = 0ull;
      if (live) {
        ((float*)e.out)[(size_t)m * e.ldo + ng] = v;
        key = ((unsigned long long)float_order_key(v) << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)ng);
      }
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const unsigned long long other = __shfl_xor(key, o, kWave);
        key = other > key ? other : key;
      }
      if (n == 0 && key) atomicMax(e.argmax + (size_t)m * TI_ARGMAX_SLOTS + (blockIdx.x & (TI_ARGMAX_SLOTS - 1)), key);
      break;
    }
    default:
      break;
  }
}

// Batched fold, consumer side: this thread's share of row `row`'s partial sums of h^2 (rows
// of R per workgroup, 512 / R threads per row taking partials part, part + P, ...; loads issued
// 8 at a time, summed in partial order).  fold_rms_finish turns the shares into rms per row.
__device__ __forceinline__ float fold_share(const GemvArgs& a, int m, int part, int P) {
  float t = 0.0f;
  if (m >= a.M) return t;
  const float* ss = a.epi.ss_in + m;
  for (int b0 = part; b0 < a.epi.n_ss; b0 += 8 * P) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = b0 + j * P < a.epi.n_ss ? ss[(size_t)(b0 + j * P) * TI_FOLD_SS_ROWS] : 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) t += fabsf(v[j]);   // (negative: ti_gemm_rows_folded; x is taken as it is here)
  }
  return t;
}
// part[512] holds every thread's share (thread = part * R + row); rms[row] = sqrt(sum / K + eps)
// (the M == 1 fold's formula, gemv_wq_kernel XM_F16F).  Call between two workgroup barriers.
__device__ __forceinline__ void fold_rms_finish(const GemvArgs& a, const float* part, float* rms, int R, int tid) {
  if (tid < R) {
    float t = 0.0f;
    for (int p = 0; p < kGemvThreads / R; ++p) t += part[p * R + tid];
    rms[tid] = sqrtf(t / (float)a.K + a.eps);
  }
}

constexpr int kTileEpiStride = 20;   // floats per row of a wave's 64 x 16 staging block (padded: no bank conflicts)

// What the epilogue of weight tile tn reads beside the products, for rows mb .. mb + 16 RB - 1 of one wave (a.vec): the residual,
// or the positions and their (cos, sin) pairs -- two dependent loads.  Fetched for all rows at once, beside the tile's products or
// ahead of its staging: read row by row where they are used, each row waits for its own (a 7B
// int4 prompt of 512 whose products all end here: 8684 -> 8579 us).
template <int RB>
struct TilePre {
  float4 v[RB];
  int32_t pos[RB];
};
struct TileQkv {   // a tile lies in one of q / k / v and in one head (head_dim % 16 == 0)
  bool q, k;
  int head, d;   // of its first column
};
__device__ __forceinline__ TileQkv tile_qkv(const ti_epilogue& e, int tn) {
  const int n = tn * 16;
  const bool q = n < e.q_dim, k = !q && n < e.q_dim + e.kv_dim;
  const int c = q ? n : k ? n - e.q_dim : n - e.q_dim - e.kv_dim, head = c / e.head_dim;
  return {q, k, head, c - head * e.head_dim};
}
template <int RB>
__device__ __forceinline__ void tile_pos(const GemvArgs& a, int mb, int lane, TilePre<RB>& p) {   // (any time before the others)
  if (a.epi.kind == TI_EPI_QKV_ROPE_KV)
#pragma unroll
    for (int it = 0; it < RB; ++it) p.pos[it] = a.epi.pos[min(mb + (lane >> 2) + 16 * it, a.M - 1)];
}
template <int RB>
__device__ __forceinline__ void tile_pre(const GemvArgs& a, int tn, int mb, int lane, TilePre<RB>& p) {
  const ti_epilogue& e = a.epi;
  const int c4 = 4 * (lane & 3), m0 = mb + (lane >> 2);
  if (!a.vec) return;
  if (e.kind == TI_EPI_RESID_F32) {
#pragma unroll
    for (int it = 0; it < RB; ++it) p.v[it] = *(const float4*)((const float*)e.out + (size_t)min(m0 + 16 * it, a.M - 1) * e.ldo + tn * 16 + c4);
  } else if (e.kind == TI_EPI_QKV_ROPE_KV) {
    const TileQkv t = tile_qkv(e, tn);
    if (t.q || t.k)
#pragma unroll
      for (int it = 0; it < RB; ++it) p.v[it] = *(const float4*)(e.rope_cs + (size_t)p.pos[it] * e.head_dim + t.d + c4);
  }
}

// Epilogue of weight tile tn (16 outputs) for rows mb .. mb + 16 RB - 1 of one wave, from its LDS block
// stg[row][col] (row stride kTileEpiStride).  Same arithmetic as epilogue_mb, element for element.
//   STORE_F32 / RESID_F32 / QKV_ROPE_KV / LOGITS_ARGMAX: lane l owns columns 4 (l & 3) .. + 3 of rows 16 it + l / 4
//   SILU_MUL_F16: lane l owns outputs 4 (l & 1) .. + 3 (gate columns, up = column + 8) of rows 32 it + l / 2
template <int RB>
__device__ __forceinline__ void tile_epilogue_lds(const GemvArgs& a, int tn, int mb, const float* stg, int lane, const TilePre<RB>& p) {
  const ti_epilogue& e = a.epi;
  if (e.kind == TI_EPI_SILU_MUL_F16) {
    const int h = 4 * (lane & 1);
#pragma unroll
    for (int it = 0; it < (RB + 1) / 2; ++it) {
      const int row = 32 * it + (lane >> 1), m = mb + row;
      if (row >= 16 * RB) continue;
      const float4 g = *(const float4*)(stg + row * kTileEpiStride + h);
      const float4 u = *(const float4*)(stg + row * kTileEpiStride + 8 + h);
      if (m >= a.M) continue;
      auto sm = [](float v, float up) { return f2h(up * (v / (1.0f + expf(-v)))); };
      const uint32_t lo = sm(g.x, u.x) | ((uint32_t)sm(g.y, u.y) << 16), hi = sm(g.z, u.z) | ((uint32_t)sm(g.w, u.w) << 16);
      *(uint2*)((uint16_t*)e.out + (size_t)m * e.ldo + tn * 8 + h) = make_uint2(lo, hi);
    }
    return;
  }
  const int c4 = 4 * (lane & 3), ng = tn * 16 + c4, m0 = mb + (lane >> 2);
  float4 v[RB];
#pragma unroll
  for (int it = 0; it < RB; ++it) v[it] = *(const float4*)(stg + (16 * it + (lane >> 2)) * kTileEpiStride + c4);
  if (e.kind == TI_EPI_STORE_F32) {
#pragma unroll
    for (int it = 0; it < RB; ++it)
      if (m0 + 16 * it < a.M) *(float4*)((float*)e.out + (size_t)(m0 + 16 * it) * e.ldo + ng) = v[it];
  } else if (e.kind == TI_EPI_RESID_F32) {
#pragma unroll
    for (int it = 0; it < RB; ++it) {
      const float4 h = p.v[it];
      if (m0 + 16 * it < a.M)
        *(float4*)((float*)e.out + (size_t)(m0 + 16 * it) * e.ldo + ng) = make_float4(h.x + v[it].x, h.y + v[it].y, h.z + v[it].z, h.w + v[it].w);
    }
  } else if (e.kind == TI_EPI_LOGITS_ARGMAX) {
    // A row's 16 columns are 4 lanes: keys by register moves, all rows' at once (epilogue_mb's 16 lanes exchange 64-bit keys through
    // LDS four times a row, one row after another: us, 32000 columns, int4 K 4096 at 64 rows 43.1 -> 34.6, int8 K 2048 at 24 26.2 -> 23.4).
#pragma unroll
    for (int it = 0; it < RB; ++it) {
      const int m = m0 + 16 * it;
      const float x[4] = {v[it].x, v[it].y, v[it].z, v[it].w};
      unsigned long long key = 0ull;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned long long k = ((unsigned long long)float_order_key(x[i]) << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)(ng + i));
        key = k > key ? k : key;
      }
      auto meet = [&](uint32_t hi, uint32_t lo) {
        const unsigned long long k = ((unsigned long long)hi << 32) | lo;
        key = k > key ? k : key;
      };
      meet(lane_xor_u32<1>((uint32_t)(key >> 32)), lane_xor_u32<1>((uint32_t)key));
      meet(lane_xor_u32<2>((uint32_t)(key >> 32)), lane_xor_u32<2>((uint32_t)key));
      if (m >= a.M) continue;
      *(float4*)((float*)e.out + (size_t)m * e.ldo + ng) = v[it];
      if ((lane & 3) == 0) atomicMax(e.argmax + (size_t)m * TI_ARGMAX_SLOTS + (blockIdx.x & (TI_ARGMAX_SLOTS - 1)), key);
    }
  } else {   // TI_EPI_QKV_ROPE_KV
    const TileQkv t = tile_qkv(e, tn);
    const int hd = e.head_dim, d = t.d + c4;
    if (t.q || t.k)
      // (cos, sin) of pairs d / 2 and d / 2 + 1: even output fmaf(-odd, sin, even * cos), odd
      // output fmaf(odd, cos, even * sin) (epilogue_mb with partner = the other of the pair)
#pragma unroll
      for (int it = 0; it < RB; ++it) {
        const float4 cs = p.v[it], x = v[it];
        v[it] = make_float4(fmaf(-x.y, cs.y, x.x * cs.x), fmaf(x.y, cs.x, x.x * cs.y), fmaf(-x.w, cs.w, x.z * cs.z), fmaf(x.w, cs.z, x.z * cs.w));
      }
    uint16_t *kc = e.k_cache, *vc = e.v_cache;
    asm("" : "+s"(kc), "+s"(vc));   // (values: a choice between the argument's fields would copy it to scratch)
    uint16_t* cache = t.k ? kc : vc;
#pragma unroll
    for (int it = 0; it < RB; ++it) {
      const int m = m0 + 16 * it;
      if (m >= a.M) continue;
      if (t.q)
        *(float4*)((float*)e.out + (size_t)m * e.ldo + ng) = v[it];
      else
        *(uint2*)(cache + (size_t)m * e.kv_stream_stride + ((size_t)t.head * e.max_seq + p.pos[it]) * hd + d) =
            make_uint2(f2h(v[it].x) | ((uint32_t)f2h(v[it].y) << 16), f2h(v[it].z) | ((uint32_t)f2h(v[it].w) << 16));
    }
  }
}

// Physical 16-byte chunk of logical chunk c in activation row `row` of the many-rows kernel's LDS image:
// c ^ tile_swz(row).  An A-fragment read (ds_read_b128, lane l: row l & 15, chunk 4 (l >> 4) + s, or
// 4 s + (l >> 4) with group-32 weights) is serviced in the lane groups {0-3,12-15,20-27},
// {4-11,16-19,28-31}, {32-35,44-47,52-59}, {36-43,48-51,60-63}; each
// holds the 16 rows once, rows {0-3,12-15} at one chunk column and rows {4-11} at the next.  With
// (row + 4) & 15 the first set lands in chunks 0-7 and the second in 8-15 of a row, so the 16 lanes
// of a group hit 16 different chunks (64 banks): conflict-free.  (row & 15 put both sets on the
// same 8 chunks: 2-way conflicts in every group, SQ_LDS_BANK_CONFLICT 3.3 cycles per read.)
__device__ __forceinline__ int tile_swz(int row) { return (row + 4) & 15; }


}  // namespace ti
