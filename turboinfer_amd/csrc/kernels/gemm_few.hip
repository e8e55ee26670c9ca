// gemm_few.hip -- packed weights x fp16 rows for few rows (decode batches, short prompts), every weight format of
// ti_gemm_rows: int4 / int8 per group of 128, blocks of 32 (GGUF Q4_0, Q8_0, Q4_1), fp16.
#include "gemm_wide.hpp"

namespace ti {

constexpr int kFewWaves = 8;

template <int F, int TM, int TN>
struct FewCfg {
  static constexpr int kRows = 16 * TM;
  // rms per row and its shares | every wave's rows of a group | partial sums of every wave | each tile's staging block
  static constexpr int kX = (kRows + kFewWaves * kWave) * 4, kRed = kX + kFewWaves * kRows * 256;
  static constexpr int kStg = kRed + kFewWaves * TN * TM * 1024, kSs = kStg + TN * kRows * kTileEpiStride * 4;
  static constexpr int kLds = kSs + TN * kRows * 8;
  static_assert(TN <= kFewWaves && kLds <= 160 * 1024);
};

// Bound: the launch (~ 3 us from the first workgroup's entry to the last one's end without any work), one memory latency and
// what a CU takes in (~ 100 KB/us; reads of 2 MB that the L2 holds reach 110 on every CU at once, 140 on one): the rows, once
// per workgroup, and its weights.  So a workgroup owns 16 TN whole columns and its 8 waves split K and meet in LDS (a split over
// workgroups meets in memory: ~ 3 us); a wave has two groups of 128 k in flight in registers, rows as whole 256-byte pieces that
// it turns into fragments in its own part of the LDS (fragment-shaped loads, 16 bytes of 16 rows, take four times as long: 2048
// columns, K 5632, 24 rows 13.6 -> 9.8 us).  Against the many-rows
// kernel (gemm_wide.hip), us, many-rows -> this: int8 2048 -> 2560 at 8 rows 7.3 -> 5.7, 24 rows 8.3 -> 6.9; 2048 -> 2048 6.6 ->
// 5.0; 5632 -> 2048 8.6 -> 7.5; int4 4096 -> 12288 at 16 rows 12.2 -> 10.4, 11008 -> 4096 12.2 -> 10.9; blocks of 32 bytes'
// 1024 -> 5632 at 24 rows 8.3 -> 6.3.  Wide outputs that take several rounds of workgroups stay with the
// many-rows kernel (its workgroups share a row's copy among 64 columns).
template <int F, int TM, int TN>
__global__ __launch_bounds__(64 * kFewWaves, 2) void gemm_few_kernel(const GemvArgs a) {
  typedef FewCfg<F, TM, TN> C;
  typedef WideFmt<F> Fm;
  constexpr int NW = kFewWaves, kWr = Fm::kBits / 4, kSr = Fm::kG32 ? 4 : 1;
  const unsigned long long t_entry = stamp_now();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int KT = a.K >> 7, NT = a.N >> 4;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cb = blockIdx.x, t0 = cb * TN;
  const int n = (KT - wave + NW - 1) / NW;   // this wave's groups: wave, wave + NW, ..

  // a load of rows takes 256 bytes of four each
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (uint32_t)(((size_t)(a.M - 1) * a.ldx + a.K) * 2), 0x00020000);
  uint32_t vx[4 * TM];
#pragma unroll
  for (int q = 0; q < 4 * TM; ++q) vx[q] = (uint32_t)min(4 * q + (lane >> 4), a.M - 1) * (uint32_t)a.ldx * 2u + (uint32_t)(lane & 15) * 16u;
  char* xl = smem + C::kX + wave * (C::kRows * 256);
  const __amdgpu_buffer_rsrc_t rs_s = __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, 0, (uint32_t)((size_t)NT * KT * Fm::kScale * (Fm::kAff ? 2 : 1)), 0x00020000);
  const u32x4* wp[TN];   // (uniform)
  uint32_t so[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const size_t g = (size_t)min(t0 + t, NT - 1) * KT + wave;
    wp[t] = a.tiles + g * (Fm::kTile / 16);
    so[t] = (uint32_t)g * Fm::kScale;
  }
  const uint32_t mins = (uint32_t)NT * (uint32_t)KT * Fm::kScale;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TN][TM];
  uint32_t magic;
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  struct Group {
    f16x8 x[4 * TM];
    u32x4 w[TN][kWr];
    uint16_t sc[TN][kSr], mn[Fm::kAff ? TN : 1][kSr];
  };
  auto load = [&](Group& d, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
#pragma unroll
      for (int c = 0; c < kWr; ++c) d.w[t][c] = ld_w(wp[t] + (size_t)i * NW * (Fm::kTile / 16) + c * 64 + lane);
      if constexpr (Fm::kBits != 16)
#pragma unroll
        for (int j = 0; j < kSr; ++j) {
          const uint32_t o = so[t] + (uint32_t)i * NW * Fm::kScale + j * 32;
          d.sc[t][j] = __builtin_amdgcn_raw_buffer_load_b16(rs_s, r * 2, o, 0);
          if constexpr (Fm::kAff) d.mn[t][j] = __builtin_amdgcn_raw_buffer_load_b16(rs_s, r * 2, mins + o, 0);
        }
    }
#pragma unroll
    for (int q = 0; q < 4 * TM; ++q) d.x[q] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rs_x, vx[q], (uint32_t)(i * NW + wave) * 256u, 0));
  };
  auto compute = [&](const Group& g) __attribute__((always_inline)) {
    // the rows turn into fragments in the wave's own part of the LDS (no barrier; chunks XOR-swizzled by row, tile_swz)
#pragma unroll
    for (int q = 0; q < 4 * TM; ++q) {
      const int row = 4 * q + (lane >> 4);
      *(f16x8*)(xl + row * 256 + ((lane & 15) ^ tile_swz(row)) * 16) = g.x[q];
    }
    f16x8 x[4][TM];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
      for (int b = 0; b < TM; ++b)
        x[s4][b] = *(const f16x8*)(xl + (16 * b + r) * 256 + ((Fm::kG32 ? s4 * 4 + kq : kq * 4 + s4) ^ tile_swz(r)) * 16);
    if constexpr (Fm::kBits == 16) {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int b = 0; b < TM; ++b)
            acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[s4][b], __builtin_bit_cast(f16x8, g.w[t][s4]), acc[t][b], 0, 0, 0);
      return;
    }
    auto deq = [&](int t, int s4) -> f16x8 {
      if constexpr (Fm::kBits == 8) return dequant_step<8>(g.w[t], s4, magic);
      else return deq_int4_signed(g.w[t][0][s4], magic);
    };
    if constexpr (!Fm::kG32) {
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        f32x4 part[TM];
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          const f16x8 bf = deq(t, s4);
#pragma unroll
          for (int b = 0; b < TM; ++b)
            part[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[s4][b], bf, s4 == 0 ? zero : part[b], 0, 0, 0);
        }
        const float s = h2f(g.sc[t][0]);
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[t][b] = fma_scale4(s, part[b], acc[t][b]);
      }
    } else {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        f32x4 xs[TM];   // the block's sum of x per row, in every column
        if constexpr (Fm::kAff) {
          const f16x8 ones = {(f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1};
#pragma unroll
          for (int b = 0; b < TM; ++b) xs[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[s4][b], ones, zero, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          const f16x8 bf = deq(t, s4);
          const float s = h2f(g.sc[t][s4]);
#pragma unroll
          for (int b = 0; b < TM; ++b) {
            const f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[s4][b], bf, zero, 0, 0, 0);
            acc[t][b] = fma_scale4(s, p, acc[t][b]);
            if constexpr (Fm::kAff) acc[t][b] = fma_scale4(fmaf(8.0f, s, h2f(g.mn[t][s4])), xs[b], acc[t][b]);   // d (q - 8) + (8 d + m)
          }
        }
      }
    }
  };
  // The wave's groups, two in flight: no branch between a group's loads and its products, so that the products wait for
  // their own loads only.
  auto product = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int b = 0; b < TM; ++b) acc[t][b] = zero;
    Group g[2];
    if (n >= 2) {
      load(g[0], 0);
      load(g[1], 1);
      int i = 0;
      for (; n - i >= 4; i += 2) {
        compute(g[0]);
        load(g[0], i + 2);
        compute(g[1]);
        load(g[1], i + 3);
      }
      compute(g[0]);
      if (n - i == 3) {
        load(g[0], i + 2);
        compute(g[1]);
        compute(g[0]);
      } else {
        compute(g[1]);
      }
    } else if (n == 1) {
      load(g[0], 0);
      compute(g[0]);
    }
    f32x4* red = (f32x4*)(smem + C::kRed) + lane;
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int b = 0; b < TM; ++b) red[((wave * TN + t) * TM + b) * 64] = acc[t][b];
  };
  const bool fold_in = a.epi.ss_in != nullptr;
  float* rmsv = (float*)smem;
  const float share = fold_in ? wide_fold_share(a, tid % C::kRows, tid / C::kRows, 64 * NW / C::kRows) : 0.0f;
  TilePre<TM> pre;   // (of the tile that this wave finishes)
  tile_pos<TM>(a, 0, lane, pre);
  product();
  if (wave < TN) tile_pre<TM>(a, min(t0 + wave, NT - 1), 0, lane, pre);
  if (fold_in) {
    wide_fold_rms<C::kRows, NW>(a, share, tid, rmsv);
    auto marked = [&]() __attribute__((always_inline)) {   // (a row's rms is negative)
      return __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int32_t, rmsv[lane % C::kRows]) < 0) != 0;
    };
    if (__builtin_expect(a.norm_w && marked(), 0)) {
      wide_fold_settle<C::kRows, NW>(a, 0, tid, rmsv);
      if (marked()) {   // rows that fp16 did not hold: again, behind their rewriting
        wide_refold<C::kRows, NW>(a, 0, wave, lane, rmsv);
        lds_barrier();
        product();
        lds_barrier();
        if (tid < C::kRows && rmsv[tid] < 0.0f) rmsv[tid] = 1.0f;
      }
    }
  }
  lds_barrier();
  const ti_epilogue& e = a.epi;
  const bool fold_out = e.kind == TI_EPI_RESID_F32 && e.fold_x != nullptr;
  if (wave < TN) {
    const int t = wave, tn = t0 + t;
    float hsq[TM], psq[TM];
#pragma unroll
    for (int b = 0; b < TM; ++b) hsq[b] = psq[b] = 0.0f;
    if (tn < NT) {
      f32x4 av[TM];
      const f32x4* red = (const f32x4*)(smem + C::kRed) + t * TM * 64 + lane;
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        av[b] = red[b * 64];
#pragma unroll
        for (int w = 1; w < NW; ++w) av[b] += red[(w * TN * TM + b) * 64];
      }
      float* stg = (float*)(smem + C::kStg) + t * C::kRows * kTileEpiStride;
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = b * 16 + 4 * kq + i;
          stg[row * kTileEpiStride + r] = fold_in ? av[b][i] / fabsf(rmsv[row]) : av[b][i];
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      wide_tile_out<TM>(a, tn, 0, stg, lane, r, kq, fold_out, pre, hsq, psq);
    }
    if (fold_out) wide_fold_part<TM>((float2*)(smem + C::kSs) + t * C::kRows, hsq, psq, lane);
  }
  if (fold_out) {
    lds_barrier();
    wide_fold_store<C::kRows, TN, TN>(a, (const float2*)(smem + C::kSs), cb, 0, tid);
  }
  if (e.kind == TI_EPI_LOGITS_ARGMAX && e.step_ctr && cb == 0 && tid == 0) *e.step_ctr += e.advance;
  stamp_end(a.stamp, t_entry);
}

// ------------------------------------------------------------------ host: shapes, plan, launch
// us of a launch, of a round over the 256 CUs and of a group per wave in it: fitted to measured points (int4, int8 and blocks of 32:
// 8 numbers of rows from 5 to 48 by 15 .. 18 (columns, K) from 1024 x 1024 to 32000 x 4096; where a shape is within 1/3 of the best).
// Blocks of 3 tiles and more, and 2 at 48 rows, keep 5632 .. 22016 columns in one round, where the many-rows kernel took them or a
// second round began.  us, before -> this: int4 2048 -> 11264 at 24 rows 8.8 -> 7.1, 4096 -> 12288 at 16 rows 9.1 -> 8.3, 32 rows 14.0 ->
// 10.7, 4096 -> 6144 at 48 rows 13.9 -> 12.3; int8 2048 -> 11264 at 24 rows 9.7 -> 8.7; blocks of 32 bytes' 1024 -> 5632 at 40 rows
// 9.7 -> 6.0.  (fp16: 16 x 48 spills and gains 0 .. 10 %; int4's 48 x 32 keeps three addresses in scratch, once, ahead of its
// main loop, and gains 22 .. 32 % at 36 .. 48 rows.)
struct FewShape {
  const void* fn;
  int rows, tiles, lds;
  float fix, round, group;
};
template <int F, int TM, int TN>
static FewShape few_shape(float fix, float round, float group) {
  typedef FewCfg<F, TM, TN> C;
  return {(const void*)gemm_few_kernel<F, TM, TN>, C::kRows, TN, C::kLds, fix, round, group};
}
constexpr int kFewShapes = 11;
template <int F>
static const FewShape* few_shapes() {   // rows x columns: 16 x 16, 32, 48, 64, 96 | 32 x 16, 32 (fp16: its weights spill), 48, 64 | 48 x 16, 32
  if constexpr (F == 4) {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.155f, 0.744f, 0.627f), few_shape<F, 1, 2>(2.503f, 0.708f, 0.733f),
                                           few_shape<F, 1, 3>(1.689f, 1.425f, 1.122f), few_shape<F, 1, 4>(0.775f, 2.378f, 1.356f),
                                           few_shape<F, 1, 6>(1.618f, 1.482f, 2.109f), few_shape<F, 2, 1>(1.705f, 1.705f, 1.004f),
                                           few_shape<F, 2, 2>(1.211f, 2.443f, 1.144f), few_shape<F, 2, 3>(0.75f, 3.18f, 1.384f),
                                           few_shape<F, 2, 4>(-0.074f, 3.974f, 1.665f), few_shape<F, 3, 1>(1.944f, 1.944f, 1.335f),
                                           few_shape<F, 3, 2>(0.957f, 2.992f, 1.707f)};
    return s;
  } else if constexpr (F == 8) {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.393f, 0.354f, 0.861f), few_shape<F, 1, 2>(2.024f, 0.93f, 1.172f),
                                           few_shape<F, 1, 3>(1.131f, 1.238f, 2.023f), few_shape<F, 2, 1>(1.721f, 1.721f, 1.175f),
                                           few_shape<F, 2, 2>(0.553f, 3.222f, 1.425f), few_shape<F, 2, 3>(0.737f, 2.437f, 2.25f),
                                           few_shape<F, 3, 1>(1.877f, 1.877f, 1.6f), few_shape<F, 3, 2>(0.485f, 3.656f, 1.912f)};
    return s;
  } else if constexpr (F == 16) {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.40f, 1.08f, 1.110f), few_shape<F, 1, 2>(-1.83f, 5.58f, 1.634f),
                                           few_shape<F, 2, 1>(0.84f, 3.03f, 1.531f), few_shape<F, 3, 1>(0.60f, 3.68f, 1.936f)};
    return s;
  } else if constexpr (F == (4 | TI_BITS_G32)) {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.769f, 0.207f, 0.687f), few_shape<F, 1, 2>(2.626f, 0.44f, 0.902f),
                                           few_shape<F, 1, 3>(1.89f, 0.783f, 1.613f), few_shape<F, 2, 1>(1.675f, 1.675f, 1.054f),
                                           few_shape<F, 2, 2>(1.103f, 2.339f, 1.357f), few_shape<F, 2, 3>(1.512f, 1.689f, 2.06f),
                                           few_shape<F, 3, 1>(0.879f, 2.81f, 1.464f), few_shape<F, 3, 2>(0.428f, 3.366f, 1.85f)};
    return s;
  } else if constexpr (F == (8 | TI_BITS_G32)) {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.451f, 0.298f, 0.915f), few_shape<F, 1, 2>(1.465f, 1.245f, 1.437f),
                                           few_shape<F, 1, 3>(1.376f, 0.674f, 2.549f), few_shape<F, 2, 1>(-2.158f, 5.345f, 1.246f),
                                           few_shape<F, 2, 2>(0.277f, 2.838f, 1.76f), few_shape<F, 2, 3>(0.914f, 1.589f, 2.866f),
                                           few_shape<F, 3, 1>(0.763f, 2.694f, 1.695f), few_shape<F, 3, 2>(-0.171f, 3.767f, 2.15f)};
    return s;
  } else {
    static const FewShape s[kFewShapes] = {few_shape<F, 1, 1>(2.92f, 0.96f, 0.721f), few_shape<F, 1, 2>(-0.34f, 4.37f, 1.038f),
                                           few_shape<F, 2, 1>(1.21f, 3.09f, 1.199f), few_shape<F, 2, 2>(-0.32f, 4.74f, 1.656f),
                                           few_shape<F, 3, 1>(0.86f, 3.91f, 1.661f)};
    return s;
  }
}
static const FewShape* few_shapes_of(int fmt) {
  switch (fmt) {
    case 4: return few_shapes<4>();
    case 8: return few_shapes<8>();
    case 16: return few_shapes<16>();
    case 4 | TI_BITS_G32: return few_shapes<4 | TI_BITS_G32>();
    case 8 | TI_BITS_G32: return few_shapes<8 | TI_BITS_G32>();
    case 4 | TI_BITS_G32 | TI_BITS_AFF: return few_shapes<4 | TI_BITS_G32 | TI_BITS_AFF>();
    default: return nullptr;
  }
}

// The shape whose rounds cost least, one row block (more rows than 48 read the weights twice: the many-rows kernel).
bool few_plan(int fmt, int M, int N, int K, int cus, FewPlan* p, int only) {
  const FewShape* sh = few_shapes_of(fmt);
  if (!sh || M < 1 || M > 48 || N < 16 || (N & 15) || K < 128 || (K & 127)) return false;
  // (the kernel's byte offsets into rows and scales are 32 bits)
  if ((uint64_t)(N >> 4) * (K >> 7) * ((fmt & 31) * 256u) >= 0xfff00000ull) return false;
  p->shape = -1;
  for (int i = 0; i < kFewShapes; ++i) {
    const FewShape& s = sh[i];
    if (!s.fn || (only >= 0 && i != only) || M > s.rows) continue;
    const int n_cb = ((N >> 4) + s.tiles - 1) / s.tiles;
    const float us = s.fix + (float)((n_cb + cus - 1) / cus) * (s.round + s.group * (float)(((K >> 7) + kFewWaves - 1) / kFewWaves));
    if (p->shape < 0 || us < p->us) *p = {i, n_cb, us};
  }
  return p->shape >= 0;
}

int few_prepare() {
  for (int f : {4, 8, 16, 4 | TI_BITS_G32, 8 | TI_BITS_G32, 4 | TI_BITS_G32 | TI_BITS_AFF}) {
    const FewShape* sh = few_shapes_of(f);
    for (int i = 0; i < kFewShapes; ++i)
      if (sh[i].fn && sh[i].lds > 64 * 1024)
        TI_HIP_CHECK(hipFuncSetAttribute(sh[i].fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024), "hipFuncSetAttribute(gemm_few_kernel)");
  }
  return TI_OK;
}

long few_workgroups(const FewPlan& p) { return p.n_cb; }

int few_launch(int fmt, const FewPlan& p, const GemvArgs& a, hipStream_t stream) {
  const FewShape& s = few_shapes_of(fmt)[p.shape];
  GemvArgs arg = a;
  void* args[] = {&arg};
  TI_HIP_CHECK(hipLaunchKernel(s.fn, dim3((unsigned)few_workgroups(p)), dim3(64 * kFewWaves), args, s.lds, stream),
               "hipLaunchKernel(gemm_few_kernel)");
  TI_LAUNCH_CHECK("gemm_few_kernel");
  return TI_OK;
}

}  // namespace ti
