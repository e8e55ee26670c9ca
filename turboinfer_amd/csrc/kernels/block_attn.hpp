// block_attn.hpp -- prompt attention on keys and values that the waves of a workgroup share in LDS (latent_attn.hip, gqa_attn.hip):
// 16-bit heads whose keys lie as NKT, values as NV MFMA fragments of 16 dims (keys: 32) a 64-key block.
//
// A wave that streams its own 64-key blocks from L2 loads 32 .. 40 KiB per 2048 .. 2560 cycles of products of 32 rows: all that a
// CU can load.  Here eight waves hold four blocks of 16 MQ rows in two parts of the keys; 128 keys at a time are copied to LDS
// once for all of them, the next 128 while these are multiplied.  What bounds it now: LDS (MQ 2: 64 bytes a cycle of operand
// reads) beside the products and the softmax's chain.
#pragma once

#include "elem.hpp"

namespace ti {

constexpr float kBlockLog2e = 1.44269504088896341f;

// Row block of wave group q = 0 .. 3 of workgroup j of QG: j, 2 QG - 1 - j, 2 QG + j, 4 QG - 1 - j, as many keys in every workgroup
// where a row's keys grow with its number.
__device__ __forceinline__ int block_of(int q, int j, int QG) { return (q + 1) / 2 * 2 * QG + (q & 1 ? -1 - j : j); }
// Wave w's group and part: waves w and w + 4, one SIMD's, are a part of one block and of its mirror.
__device__ __forceinline__ int block_group(int wave) { return wave < 4 ? wave : 7 - wave; }

// LDS bytes: 2 iterations of 2 blocks.
template <int NKT, int NV>
constexpr int block_lds() { return 4 * (4 * NKT + 2 * NV) * 1024; }

// All waves of the workgroup.  live: this wave has rows; low / last: the lowest of their positions and the highest (last -1:
// none); end: the last 64-key block of any of the workgroup's waves.
//   query(kt, q): operand of 32 dims kt of row tile q;  limit(q): position of this lane's row (column lane & 15)
//   source(e, blk, off): where fragment e of 64-key block blk is: [4 key tiles][NKT] keys (as tile(t, kt) numbers them), then [NV][2] values;
//     off: the lane's bytes behind it (16 lane on entry)
//   sink(q): the row's score without a value, or -1e30 / scale ..; counted(q): whether it counts
//   out(q, v, l): value fragment v of row tile q, not yet divided by l
template <int MQ, int NKT, int NV, class Query, class Tile, class Source, class Limit, class Sink, class Out>
__device__ __forceinline__ void block_attention(char* lds, float scale2, bool live, int low, int last, int end, Query query, Tile tile, Source source,
                                                Limit limit, Sink sink, Out out) {
  typedef bf16x8 V;
  constexpr int NF = 4 * NKT + 2 * NV, NC = 2 * NF / 8;   // 1-KiB fragments of 64 keys; copies of a wave
  static_assert(2 * NF % 8 == 0 && 4 * MQ * (4 * NV + 2) * 256 <= block_lds<NKT, NV>());
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4;
  const int part = wave >> 2, iters = (end >> 1) + 1;
  V qf[NKT][MQ];
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
    for (int q = 0; q < MQ; ++q) qf[kt][q] = query(kt, q);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  auto issue = [&](int it) {   // an iteration's two blocks (past the last key: the last block again)
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int f = i * 8 + wave, b = f >= NF;
      uint32_t off = (uint32_t)lane * 16;
      const void* src = source(b ? f - NF : f, min(2 * it + b, end), off);
      dma_1k_asm(src, off, lds0 + (uint32_t)((it & 1) * 2 * NF + f) * 1024);
    }
  };
  f32x4 o[MQ][NV];
  float mr[MQ], lr[MQ], top[MQ];   // o, lr: relative to 2^mr; the largest score, the sink among them
#pragma unroll
  for (int q = 0; q < MQ; ++q) {
    bool counts;
    top[q] = mr[q] = sink(q, counts);   // weight 2^(sink - max), no value; counted by one part
    lr[q] = counts && part == 0 && g == 0 ? 1.0f : 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) o[q][v] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (only copies are counted below)
  issue(0);
  for (int it = 0; it < iters; ++it) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_sync();   // everyone's copies are here, and everyone has done with the other half
    if (it + 1 < iters) issue(it + 1);
    const int k0 = (2 * it + part) * 64;
    if (k0 > last) continue;
    const V* st = (const V*)lds + ((it & 1) * 2 + part) * NF * 64 + lane;
    f32x4 s[MQ][4];
#pragma unroll
    for (int q = 0; q < MQ; ++q)
#pragma unroll
      for (int t = 0; t < 4; ++t) s[q][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      V k[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) k[t] = st[tile(t, kt) * 64];
#pragma unroll
      for (int q = 0; q < MQ; ++q)
#pragma unroll
        for (int t = 0; t < 4; ++t) s[q][t] = mma(k[t], qf[kt][q], s[q][t]);
    }
    const bool ragged = k0 + 63 > low;   // (uniform: a row of these does not see all of the block)
#pragma unroll
    for (int q = 0; q < MQ; ++q) {
      float mx = -INFINITY;
      const int p = limit(q) - k0 - 4 * g;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (ragged) s[q][t][r] = t * 16 + r <= p ? s[q][t][r] : -INFINITY;
          mx = fmaxf(mx, s[q][t][r]);
        }
      // Weights are taken against the block's own maximum times the power of 2 that brings it to the running one or less than twice that: in
      // every block the largest weight is a power of 2, which bf16 holds exactly, and those just below it have the smallest roundings.
      // Output errors against float64: this 2.04e-3, sharp rows 1.66e-3; weights against the running maximum 2.07e-3 and 1.68e-3; sums
      // moved only to maxima > 8 away 2.34e-3 and 2.02e-3.
      mx = fmaxf(xor32_max(xor16_max(mx)) * scale2, top[q] - 64.0f);
      top[q] = fmaxf(top[q], mx);
      mx += fmaxf(ceilf(top[q] - mx), 0.0f);
      if (MQ > 1 || __builtin_amdgcn_ballot_w64(mx != mr[q]) != 0) {   // (hardly ever not; one tile a wave: the branch keeps its loads ahead, 42 -> 37 us)
        const float alpha = mr[q] == mx ? 1.0f : __builtin_amdgcn_exp2f(mr[q] - mx);
        mr[q] = mx;
        lr[q] *= alpha;
#pragma unroll
        for (int v = 0; v < NV; ++v) o[q][v] *= alpha;
      }
      const float off = mr[q] == -INFINITY ? 0.0f : mr[q];   // (a sink of -inf and no key yet: weights 0)
      float l = 0.0f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[q][t][r] = __builtin_amdgcn_exp2f(fmaf(s[q][t][r], scale2, -off));
          l += s[q][t][r];
        }
      lr[q] += l;
    }
    bf16x8 pf[MQ][2];
#pragma unroll
    for (int q = 0; q < MQ; ++q)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pf[q][b][r] = (bf16)s[q][2 * b][r];
          pf[q][b][4 + r] = (bf16)s[q][2 * b + 1][r];
        }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      V vv[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) vv[b] = st[(4 * NKT + v * 2 + b) * 64];
#pragma unroll
      for (int q = 0; q < MQ; ++q)
#pragma unroll
        for (int b = 0; b < 2; ++b) o[q][v] = mma(vv[b], pf[q][b], o[q][v]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_sync();   // part 1 hands its sums to part 0 where the keys were
  float* x = (float*)lds + (size_t)block_group(wave) * MQ * (4 * NV + 2) * 64;
  if (part) {
#pragma unroll
    for (int q = 0; q < MQ; ++q) {
      float* d = x + q * (4 * NV + 2) * 64;
#pragma unroll
      for (int v = 0; v < NV; ++v) *(f32x4*)(d + v * 256 + lane * 4) = o[q][v];
      d[NV * 256 + lane] = mr[q];
      d[NV * 256 + 64 + lane] = lr[q];
    }
  }
  lds_sync();
  if (part || !live) return;
#pragma unroll
  for (int q = 0; q < MQ; ++q) {
    const float* d = x + q * (4 * NV + 2) * 64;
    const float m1 = d[NV * 256 + lane], l1 = d[NV * 256 + 64 + lane], mx = fmaxf(mr[q], m1);
    const float f0 = __builtin_amdgcn_exp2f(mr[q] - mx), f1 = __builtin_amdgcn_exp2f(m1 - mx);
    float l = lr[q] * f0 + l1 * f1;
    l += lane_xor<16>(l);
    l += lane_xor<32>(l);
#pragma unroll
    for (int v = 0; v < NV; ++v) o[q][v] = o[q][v] * f0 + *(const f32x4*)(d + v * 256 + lane * 4) * f1;
    out(q, o[q], l);
  }
}

}  // namespace ti
