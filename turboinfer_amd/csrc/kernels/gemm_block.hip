// gemm_block.hip -- packed weights x fp16 rows for prompt chunks and large batches: int4 and int8 per group of 128, and fp16.
#include "gemm_wide.hpp"

namespace ti {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// N (1, 2 or 4) copies of 64 lanes x 16 bytes from rs + v[i] + soff + 1024 i to LDS byte address lds + 1024 i.  Issued from
// asm, so hipcc does not count them: the caller waits with a counted s_waitcnt vmcnt and a barrier.
template <int N>
__device__ __forceinline__ void rows_dma(__amdgpu_buffer_rsrc_t rs, const uint32_t* v, uint32_t soff, uint32_t lds) {
  uint32_t keep;
#define TI_ROWS_DMA "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %1, %2 offen lds\n\t"
  if constexpr (N == 1)
    asm volatile(TI_ROWS_DMA "s_mov_b32 m0, %0" : "=&s"(keep) : "s"(rs), "s"(soff), "s"(lds), "v"(v[0]) : "memory");
  else if constexpr (N == 2)
    asm volatile(TI_ROWS_DMA "buffer_load_dwordx4 %5, %1, %2 offen offset:1024 lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(rs), "s"(soff), "s"(lds), "v"(v[0]), "v"(v[1]) : "memory");
  else
    asm volatile(TI_ROWS_DMA "buffer_load_dwordx4 %5, %1, %2 offen offset:1024 lds\n\tbuffer_load_dwordx4 %6, %1, %2 offen offset:2048 lds\n\t"
                 "buffer_load_dwordx4 %7, %1, %2 offen offset:3072 lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(rs), "s"(soff), "s"(lds), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]) : "memory");
#undef TI_ROWS_DMA
}

constexpr int kTurnRow = 36, kTurn = 32 * kTurnRow + 32;   // floats: a wave's 32 x 32 block on its way from columns to rows

template <int F, int WN, int KG, int RT, int CT, int NS>
struct BlockGemm {
  typedef WideFmt<F> W;
  static constexpr int kWaves = WN * KG, kRows = 32 * RT, kCols = 32 * CT * WN;
  static constexpr int kA = KG * kRows * 256;                             // LDS bytes of a stage's rows
  static constexpr int kDma = kRows / 4 / WN;                             // row copies of a wave and stage
  static constexpr int kWl = W::kBits == 16 ? 8 : W::kBits / 2;           // 1 KiB weight loads of 32 columns and 128 k
  static constexpr int kSets = W::kBits == 16 ? 2 : 3;
  static constexpr int kLoads = CT * (kWl + (W::kBits == 16 ? 0 : 1));    // with the scales'
  static constexpr int kFin = KG < RT ? KG : RT, kRf = RT / kFin;         // groups that finish row tiles, and how many each
  static constexpr int kPart = (KG - 1) * WN * CT * RT * 4096;            // the other groups' sums (behind the rows, once read)
  static constexpr int kEpi = kPart + kFin * WN * kTurn * 4, kLds = NS * kA > kEpi ? NS * kA : kEpi;
  // folds: the column-waves' sums of the next one, the threads' shares (kP a row) of this one's and the waves' marks
  static constexpr int kRed = kEpi, kSums = NS * kA > kRed + WN * kRows * 8 ? NS * kA : kRed + WN * kRows * 8, kMarks = kSums + kWaves * 256;
  static constexpr int kFoldLds = kMarks + kWaves * 4, kP = 64 * kWaves / kRows;
  static_assert(kRows / 4 % WN == 0 && (kDma % 4 == 0 || kDma <= 2) && RT % kFin == 0 && kFoldLds <= 160 * 1024);
  static constexpr int vm(int n) { return n > 63 ? 63 : n; }
};

// The epilogue (a.vec; same arithmetic as epilogue_mb): acc[t][b] are columns 0 .. 15 of weight tile n + 2 t in row m + 32 b.  A
// lane's 16 columns are 64 bytes (SiLU's 8 outputs 16) of one row, and what a row tile reads beside its products is in
// flight together.
// FOLD: a folded output also takes the next call's input, fp16(h w), and the lanes' sums of h^2 and (h w)^2 (wide_tile_out's) to hsq, psq.
template <bool FOLD, int CT, int RT>
__device__ __forceinline__ void block_out(const GemvArgs& a, f32x16 (&acc)[CT][RT], int n, int m, int NT, float (&hsq)[RT], float (&psq)[RT]) {
  typedef uint32_t u32x4a8 __attribute__((ext_vector_type(4), aligned(8)));
  const ti_epilogue& e = a.epi;
  auto pair = [](float lo, float hi) { return f2h(lo) | ((uint32_t)f2h(hi) << 16); };
  if (e.kind == TI_EPI_SILU_MUL_F16) {
    auto sm = [](float v, float up) { return up * (v / (1.0f + expf(-v))); };
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        const f32x16 v = acc[t][b];
        u32x4a8 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = pair(sm(v[2 * i], v[8 + 2 * i]), sm(v[2 * i + 1], v[9 + 2 * i]));
        if (m + 32 * b < a.M && n + 2 * t < NT) *(u32x4a8*)((uint16_t*)e.out + (size_t)(m + 32 * b) * e.ldo + (n + 2 * t) * 8) = o;
      }
    return;
  }
  auto store = [&](const f32x16& v, float* o) {
#pragma unroll
    for (int q = 0; q < 4; ++q) ((f32x4*)o)[q] = (f32x4){v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  };
  if (e.kind == TI_EPI_STORE_F32) {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int b = 0; b < RT; ++b)
        if (m + 32 * b < a.M && n + 2 * t < NT) store(acc[t][b], (float*)e.out + (size_t)(m + 32 * b) * e.ldo + (n + 2 * t) * 16);
  } else if (e.kind == TI_EPI_RESID_F32) {
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      f32x4 h[RT][4], w[4];
      if (FOLD && e.fold_x)
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = *(const f32x4*)(e.fold_w + min(n + 2 * t, NT - 1) * 16 + 4 * q);
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        const f32x4* o = (const f32x4*)((const float*)e.out + (size_t)min(m + 32 * b, a.M - 1) * e.ldo + min(n + 2 * t, NT - 1) * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) h[b][q] = o[q];
      }
#pragma unroll
      for (int b = 0; b < RT; ++b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][b][i] = h[b][i >> 2][i & 3] + acc[t][b][i];
        if (m + 32 * b < a.M && n + 2 * t < NT) store(acc[t][b], (float*)e.out + (size_t)(m + 32 * b) * e.ldo + (n + 2 * t) * 16);
      }
      if (FOLD && e.fold_x)
#pragma unroll
        for (int b = 0; b < RT; ++b) {
          const f32x16& v = acc[t][b];
          float p[16], top = 0.0f, hs = 0.0f, ps = 0.0f;
#pragma unroll
          for (int i = 0; i < 16; ++i) p[i] = v[i] * w[i >> 2][i & 3];
#pragma unroll
          for (int i = 0; i < 16; i += 4) {   // (as outputs the products are rounded on their own, as in mul_f16)
            asm("v_max3_f32 %0, %0, |%1|, |%2|\n\tv_max3_f32 %0, %0, |%3|, |%4|" : "+v"(top), "+v"(p[i]), "+v"(p[i + 1]), "+v"(p[i + 2]), "+v"(p[i + 3]));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              hs = fmaf(v[i + j], v[i + j], hs);
              ps = fmaf(p[i + j], p[i + j], ps);
            }
          }
          if (m + 32 * b < a.M && n + 2 * t < NT) {
            uint16_t* o = e.fold_x + (size_t)(m + 32 * b) * e.ldo + (n + 2 * t) * 16;
#pragma unroll
            for (int i = 0; i < 16; i += 8)
              *(u32x4a8*)(o + i) = (u32x4a8){pair(p[i], p[i + 1]), pair(p[i + 2], p[i + 3]), pair(p[i + 4], p[i + 5]), pair(p[i + 6], p[i + 7])};
            hsq[b] += hs;
            psq[b] += top > 65504.0f ? INFINITY : ps;
          }
        }
    }
  } else {   // TI_EPI_QKV_ROPE_KV: a tile lies in one of q / k / v and in one head (head_dim % 16 == 0)
    const int hd = e.head_dim;
    int pos[RT];
#pragma unroll
    for (int b = 0; b < RT; ++b) pos[b] = e.pos[min(m + 32 * b, a.M - 1)];
    uint16_t *kc = e.k_cache, *vc = e.v_cache;
    asm("" : "+s"(kc), "+s"(vc));   // (values: a choice between the argument's fields would copy it to scratch)
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int c0 = min(n + 2 * t, NT - 1) * 16;
      const bool in_q = c0 < e.q_dim, in_k = !in_q && c0 < e.q_dim + e.kv_dim;
      const int c = in_q ? c0 : in_k ? c0 - e.q_dim : c0 - e.q_dim - e.kv_dim, head = c / hd, d = c - head * hd;
      f32x4 cs[RT][4];
      if (in_q || in_k)
#pragma unroll
        for (int b = 0; b < RT; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) cs[b][q] = *(const f32x4*)(e.rope_cs + (size_t)pos[b] * hd + d + 4 * q);
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        f32x16& v = acc[t][b];
        if (in_q || in_k)   // (cos, sin) of column pairs
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            const float x0 = v[i], x1 = v[i + 1], co = cs[b][i >> 2][i & 3], si = cs[b][i >> 2][(i & 3) + 1];
            v[i] = fmaf(-x1, si, x0 * co);
            v[i + 1] = fmaf(x1, co, x0 * si);
          }
        if (m + 32 * b >= a.M || n + 2 * t >= NT) continue;
        if (in_q) {
          store(v, (float*)e.out + (size_t)(m + 32 * b) * e.ldo + c0);
        } else {
          uint16_t* cache = (in_k ? kc : vc) + (size_t)(m + 32 * b) * e.kv_stream_stride + ((size_t)head * e.max_seq + pos[b]) * hd + d;
#pragma unroll
          for (int q = 0; q < 2; ++q)
            *(u32x4a8*)(cache + 8 * q) = (u32x4a8){pair(v[8 * q], v[8 * q + 1]), pair(v[8 * q + 2], v[8 * q + 3]), pair(v[8 * q + 4], v[8 * q + 5]),
                                                   pair(v[8 * q + 6], v[8 * q + 7])};
        }
      }
    }
  }
}

// A fold's sums (wide_fold_share), 8 of a thread's in flight: the first ones beside the first rows.
__device__ __forceinline__ void block_share_load(const GemvArgs& a, int m, int b, int P, float (&v)[8]) {   // partials b, b + P, ..
  constexpr uint32_t pitch = TI_FOLD_SS_ROWS * 4u;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)a.epi.ss_in, 0, (uint32_t)a.epi.n_ss * pitch, 0x00020000);
  const uint32_t o = m < a.M ? (uint32_t)b * pitch + (uint32_t)m * 4u : 0x80000000u;   // (past the end: 0)
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o + (uint32_t)(j * P) * pitch, 0, 0));
}
__device__ __forceinline__ float block_share(const GemvArgs& a, int m, int part, int P, float (&v)[8]) {
  float t = 0.0f;
  uint32_t any = 0;
  for (int b = part;;) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      t += fabsf(v[j]);
      any |= __builtin_bit_cast(uint32_t, v[j]);
    }
    b += 8 * P;
    if (b - part >= a.epi.n_ss) break;   // (uniform)
    block_share_load(a, m, b, P, v);
  }
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, t) | (any & 0x80000000u));
}

// Bound: the vector unit beside the matrix cores (7 .. 9 vector instructions an MFMA; the matrix cores are busy 44 .. 58 % of a
// launch of a 7B int4 prompt of 512) and the clock, ~ 2.0 GHz while prompts run.  A 32x32x16 MFMA
// holds the vector issue for ~ 8 cycles of its 32 and does twice a 16x16x32's work (7.5 of 16): as many scale FMAs per product
// leave time for the unpacking.  The weights pass LDS by (each is read by one wave only): half the DMA, whose bursts with the
// barriers' skew were half of a stage in gemm_wide_kernel (int4, cycles of the main loop per 64 x 256 columns and 128 k: 64 x 384
// blocks 2130, 48 % MFMA -> 64 x 256 blocks here 1440 at 71 %).  Copies of the rows are issued four to an M0 setting, the weights' loads
// spread over the steps of a stage.  us, gemm_wide_kernel -> here: int4 512 rows 4096 -> 22016 114 -> 100, 11008 -> 4096 64 ->
// 56, 4096 -> 4096 30 -> 23.5, 4096 -> 12288 63 -> 60; int8 1000 rows 2048 -> 11264 75 -> 60.5, 5632 -> 2048 43.5 -> 35, 2048 ->
// 2560 25.7 -> 22.5; fp16 333 rows 33.5 -> 25.4, 30.7 -> 23.5, 12.1 -> 11.2.  Whole prompts: 7B int4 of 512 rows 9159 -> 8184,
// TinyLlama int8 of 1000 4346 -> 3807, fp16 of 333 2358 -> 2152.
// Slices of K by workgroups, as gemm_wide_kernel has them, were no gain here beyond what it keeps.
// FOLD: a batched fold's input or output.  The sums come in beside the first rows and are kept in LDS; rows that must be normalised
// first are found before the products, not behind them (a loop around the products cost 27 registers), in calls of their own, as the
// code costs the others 0 .. 2 us.  Steps of 64 streams of the 7B model, int4: 13 241 -> 12 943 us; prompts of 44 rows of TinyLlama
// int8 1132 -> 1091, of 43 of Llama-3-8B int4 2719 -> 2608.
//
// Block of 32 RT rows x 32 CT WN columns per workgroup; wave (g, wn) owns all rows of 32 CT columns and the 128-k groups g, g +
// KG, .. of the workgroup's (KG > 1: the groups meet in LDS at the end).  A stage is KG groups: their rows come to LDS by DMA, NS
// stages in flight (chunks XOR-swizzled by row, tile_swz); a wave's packed weights and scales, which no other wave reads, come
// straight to registers two groups ahead (fp16: one).  v_mfma_f32_32x32x16: lane l holds 8 k of row (column) l & 31; its k octet
// s of the packed layout's quarter 2 j + (l >> 5) makes step u = 4 j + s, so a 32-column operand is two 16-column tiles' words as
// they are packed.
template <int F, int WN, int KG, int RT, int CT, int NS, bool FOLD>
__global__ __launch_bounds__(64 * WN * KG, 2) void gemm_block_kernel(const GemvArgs a, int n_cb, int n_rb) {
  typedef BlockGemm<F, WN, KG, RT, CT, NS> C;
  typedef WideFmt<F> Fm;
  constexpr int B = Fm::kBits;
  const unsigned long long t_entry = stamp_now();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int KT = a.K >> 7, NT = a.N >> 4;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = KG == 1 ? 0 : wave / WN, wn = wave % WN;
  // the row blocks of a column block share an XCD (its L2 holds their weights once)
  const int rest = blockIdx.x >> 3, cb8 = rest / n_rb, rb = rest - cb8 * n_rb, cb = cb8 * 8 + (blockIdx.x & 7);
  if (cb >= n_cb) return;
  const int m0 = rb * C::kRows, t0 = cb * (C::kCols / 16) + wn * 2 * CT;
  const int nk = (KT - g + KG - 1) / KG, ns = (KT + KG - 1) / KG;   // this wave's groups, the workgroup's stages

  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, (uint32_t)(((size_t)(a.M - 1) * a.ldx + a.K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)a.tiles, 0, (uint32_t)((size_t)NT * KT * Fm::kTile), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_s = __builtin_amdgcn_make_buffer_rsrc((void*)a.scales, 0, (uint32_t)((size_t)NT * KT * Fm::kScale), 0x00020000);
  uint32_t vx[C::kDma];
#pragma unroll
  for (int q = 0; q < C::kDma; ++q) {   // (wave (g, wn) copies a share of group g's rows)
    const int row = 4 * (wn * C::kDma + q) + (lane >> 4), c = (lane & 15) ^ tile_swz(row);
    // (rows_dma adds 1024 (q & 3): not more than the row's own offset, as a row is 256 bytes or more and M > 12)
    vx[q] = (uint32_t)min(m0 + row, a.M - 1) * (uint32_t)a.ldx * 2u + (uint32_t)c * 16u - (uint32_t)(q & 3) * 1024u;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem + (uint32_t)(g * WN + wn) * (C::kDma * 1024u);
  auto group = [&](int s) { return min(s * KG + g, KT - 1); };   // (past the end: the last one again)
  auto issue = [&](int s, int buf) __attribute__((always_inline)) {
    const uint32_t st = lds0 + (uint32_t)buf * C::kA, k = (uint32_t)group(s) * 256u;
#pragma unroll
    for (int q = 0; q < C::kDma; q += C::kDma % 4 ? C::kDma : 4)
      rows_dma<C::kDma % 4 ? C::kDma : 4>(rs_x, vx + q, k, __builtin_amdgcn_readfirstlane(st + q * 1024u));
  };
  // operand column r of 32: a column of the first or second tile.  fp16 products come as rows per lane (the operands change
  // places), of 16 columns as block_out takes them where r is column 4 (r >> 3) + (r & 3) of tile (r >> 2) & 1.  (Scaled ones
  // would need 16 scales per lane and step: 64 x 256 blocks of int4 81 k -> 92 k cycles.)
  const int col = B == 16 ? 4 * (r >> 3) + (r & 3) : r & 15, second = B == 16 ? r >> 2 & 1 : r >> 4;
  uint32_t vw[CT], vs[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const uint32_t tile = (uint32_t)min(t0 + 2 * t + second, NT - 1) * (uint32_t)KT;
    vw[t] = tile * Fm::kTile + (uint32_t)(h * 16 + col) * 16u;
    vs[t] = tile * Fm::kScale + (uint32_t)col * 2u;
  }
  struct Set {
    u32x4 w[CT][C::kWl];
    uint16_t sc[CT];
  };
  auto load_part = [&](Set& d, int s, int u) __attribute__((always_inline)) {   // u: of 7 (the scales: 0)
    const uint32_t k = (uint32_t)group(s);
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      if constexpr (B != 16)
        if (u == 0) d.sc[t] = __builtin_amdgcn_raw_buffer_load_b16(rs_s, vs[t], k * Fm::kScale, 0);
#pragma unroll
      for (int l = 0; l < C::kWl; ++l)   // j = l & 1 of the tile's KiB l >> 1
        if ((t * C::kWl + l) * 7 / (CT * C::kWl) == u)
          d.w[t][l] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_w, vw[t] + (l >> 1) * 1024 + (l & 1) * 512, k * Fm::kTile, 0));
    }
  };
  auto load_set = [&](Set& d, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 7; ++u) load_part(d, s, u);
  };
  uint32_t magic;
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  auto weights = [&](const Set& d, int t, int u) __attribute__((always_inline)) -> f16x8 {
    const int j = u >> 2, s = u & 3;
    if constexpr (B == 4) {
      return deq_int4_signed(d.w[t][j][s], magic);
    } else if constexpr (B == 8) {
      f16x8 q;
      deq_int8_word(d.w[t][j + 2 * (s >> 1)][(s & 1) * 2], q, 0);
      deq_int8_word(d.w[t][j + 2 * (s >> 1)][(s & 1) * 2 + 1], q, 4);
      return q;
    } else {
      return __builtin_bit_cast(f16x8, d.w[t][j + 2 * s]);
    }
  };
  // chunk 4 (2 j + h) + s of row r lies at (4 h ^ tile_swz(r)) ^ (8 j + s)
  const uint32_t x0 = (uint32_t)(g * C::kRows * 256 + r * 256 + ((4 * h) ^ tile_swz(r)) * 16);
  auto read_x = [&](f16x8 (&d)[RT], int buf, int u) __attribute__((always_inline)) {
    const char* p = smem + ((x0 + (uint32_t)buf * C::kA) ^ (uint32_t)((8 * (u >> 2) + (u & 3)) * 16));
#pragma unroll
    for (int b = 0; b < RT; ++b) d[b] = *(const f16x8*)(p + b * 32 * 256);
  };
  const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  f32x16 acc[CT][RT], part[B == 16 ? 1 : CT][RT];   // part: a group's sum, scaled during the next group's first step
  float pend[CT];                                   // its scale
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    pend[t] = 0.0f;
#pragma unroll
    for (int b = 0; b < RT; ++b) {
      acc[t][b] = zero;
      if constexpr (B != 16) part[t][b] = zero;
    }
  }
  auto scale = [&](int t, int b) __attribute__((always_inline)) {
    if constexpr (B != 16)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][b][i] = fmaf(pend[t], part[t][b][i], acc[t][b][i]);
  };
  f16x8 x[2][RT], wq[CT];
  auto mul = [&](const f16x8 (&xs)[RT], const Set& d, const Set& dn, auto u_) __attribute__((always_inline)) {
    constexpr int u = decltype(u_)::value;
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const f16x8 w = wq[t];
      wq[t] = u < 7 ? weights(d, t, u + 1) : weights(dn, t, 0);
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        if constexpr (B == 16) {
          acc[t][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, xs[b], acc[t][b], 0, 0, 0);
        } else {
          if constexpr (u == 0) {
            scale(t, b);
            __builtin_amdgcn_sched_barrier(0);
          }
          part[t][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs[b], w, u == 0 ? zero : part[t][b], 0, 0, 0);
        }
      }
      if constexpr (u == 7 && B != 16) {
        pend[t] = h2f(d.sc[t]);
        asm("" : "+v"(pend[t]));   // (the converted value: v_fma_mix is slower)
      }
#pragma unroll
      for (int b = 0; b < RT; ++b) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);         // one product,
        __builtin_amdgcn_sched_group_barrier(0x002, 12 / RT, 0);   // then vector arithmetic
      }
    }
  };

  const bool fold_in = FOLD && a.epi.ss_in != nullptr;
  float* sums = (float*)(smem + C::kSums);
  int* marks = (int*)(smem + C::kMarks);
  Set set[C::kSets];
#pragma unroll 1
  for (bool again = false;;) {   // (once, unless a fold's rows must be normalised first)
    float fs[8];
    const bool look = fold_in && !again;
    if (look) block_share_load(a, m0 + tid % C::kRows, tid / C::kRows, C::kP, fs);
#pragma unroll
    for (int q = 0; q < NS; ++q) issue(q, q);
#pragma unroll
    for (int q = 0; q < C::kSets - 1; ++q) load_set(set[q], q);
    if (look) {
      const float share = block_share(a, m0 + tid % C::kRows, tid / C::kRows, C::kP, fs);
      sums[tid] = share;
      if (a.norm_w) marks[wave] = __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int32_t, share) < 0) != 0;
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::vm((NS - 1) * C::kDma + (C::kSets - 1) * C::kLoads)) : "memory");
    lds_barrier();
    if (!look || !a.norm_w) break;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(lane < C::kWaves && marks[lane < C::kWaves ? lane : 0]) == 0, 1)) break;
    // a row has a mark: the marks counted, the rows that fp16 does not hold rewritten (every workgroup that reads them writes the same)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    const float share = sums[tid];
    float* rmsv = (float*)smem;
    wide_fold_rms<C::kRows, C::kWaves>(a, share, tid, rmsv);
    wide_fold_settle<C::kRows, C::kWaves>(a, m0, tid, rmsv);
    sums[tid] = rmsv[tid % C::kRows] < 0.0f ? -fabsf(share) : fabsf(share);
    wide_refold<C::kRows, C::kWaves>(a, m0, wave, lane, rmsv);
    again = true;
  }
  read_x(x[0], 0, 0);
#pragma unroll
  for (int t = 0; t < CT; ++t) wq[t] = weights(set[0], t, 0);
  int buf = 0;
  // Stage s in slot s % NS.  Rows are read from LDS one step ahead; the last step waits for the next stage's rows, meets the
  // other waves (whose reads of this stage are done: its slot takes stage s + NS) and reads the next stage's first operands.
  // live: this wave has a group in it; tail: of the last stages.
  auto stage = [&](int s, Set& cur, Set& next, Set& fill, bool live, bool tail) __attribute__((always_inline)) {
    if (live)
      [&]<int... U>(std::integer_sequence<int, U...>) __attribute__((always_inline)) {
        ((read_x(x[(U + 1) & 1], buf, U + 1), load_part(fill, s + C::kSets - 1, U), __builtin_amdgcn_sched_barrier(0), mul(x[U & 1], cur, next, std::integral_constant<int, U>()),
          __builtin_amdgcn_sched_barrier(0)),
         ...);
      }(std::make_integer_sequence<int, 7>());
    // this wave's share of stage s + 1 is there (the last stages' loads of weights that no stage takes are not made)
    if (!live) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (tail) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::vm((NS - 2) * C::kDma)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::vm((NS - 2) * C::kDma + C::kLoads)) : "memory");
    lds_barrier();
    issue(s + NS, buf);
    buf = buf + 1 == NS ? 0 : buf + 1;
    if (live) {
      read_x(x[0], buf, 0);
      __builtin_amdgcn_sched_barrier(0);
      mul(x[1], cur, next, std::integral_constant<int, 7>());
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int s = 0;
  const int whole = KT / KG;   // stages in which every wave has a group
  if constexpr (C::kSets == 3) {
    for (; s + 3 <= whole; s += 3) {
      stage(s, set[0], set[1], set[2], true, false);
      stage(s + 1, set[1], set[2], set[0], true, false);
      stage(s + 2, set[2], set[0], set[1], true, false);
    }
    if (s < ns) stage(s, set[0], set[1], set[2], s < nk, true);
    if (s + 1 < ns) stage(s + 1, set[1], set[2], set[0], s + 1 < nk, true);
    if (s + 2 < ns) stage(s + 2, set[2], set[0], set[1], s + 2 < nk, true);
  } else {
    for (; s + 2 <= whole; s += 2) {
      stage(s, set[0], set[1], set[1], true, false);
      stage(s + 1, set[1], set[0], set[0], true, false);
    }
    if (s < ns) stage(s, set[0], set[1], set[1], s < nk, true);
    if (s + 1 < ns) stage(s + 1, set[1], set[0], set[0], s + 1 < nk, true);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the clamped stages past the end
  lds_barrier();
#pragma unroll
  for (int t = 0; t < CT; ++t)
#pragma unroll
    for (int b = 0; b < RT; ++b) scale(t, b);

  if constexpr (KG > 1) {   // row tiles b / kRf are finished by group b / kRf: the others leave theirs, summed in order of the groups
    f32x4* px = (f32x4*)smem + lane;
    auto at = [&](int o, int t, int b, int q) { return ((((o * WN + wn) * CT + t) * RT + b) * 4 + q) * 64; };
#pragma unroll
    for (int b = 0; b < RT; ++b)
      if (b / C::kRf != g)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            px[at(g > b / C::kRf ? g - 1 : g, t, b, q)] = (f32x4){acc[t][b][4 * q], acc[t][b][4 * q + 1], acc[t][b][4 * q + 2], acc[t][b][4 * q + 3]};
    lds_barrier();
#pragma unroll
    for (int b = 0; b < RT; ++b)
      if (b / C::kRf == g)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int o = 0; o < KG; ++o) {
              const f32x4 own = {acc[t][b][4 * q], acc[t][b][4 * q + 1], acc[t][b][4 * q + 2], acc[t][b][4 * q + 3]};
              if (o == b / C::kRf) v += own;
              else v += px[at(o > b / C::kRf ? o - 1 : o, t, b, q)];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][b][4 * q + i] = v[i];
          }
  }
  const bool fold_out = FOLD && a.epi.kind == TI_EPI_RESID_F32 && a.epi.fold_x != nullptr;
  float2* red = (float2*)(smem + C::kRed);
  if (g < C::kFin)
#pragma unroll
    for (int f = 0; f < C::kFin; ++f)
      if (f == g) {   // scaled sums: from a column's rows per lane to 16 columns of a row, by the wave's own block of LDS
        float* turn = (float*)(smem + C::kPart) + (g * WN + wn) * kTurn;
        f32x16 v[CT][C::kRf];
        float hsq[C::kRf], psq[C::kRf];
#pragma unroll
        for (int b = 0; b < C::kRf; ++b) {
          const int row = (f * C::kRf + b) * 32 + r;   // of the block
          hsq[b] = psq[b] = 0.0f;
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            const f32x16& c = acc[t][f * C::kRf + b];
            if constexpr (B == 16) {
              v[t][b] = c;
              continue;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
              *(f32x4*)(turn + r * kTurnRow + (r >> 4) * 32 + 8 * q + 4 * h) = (f32x4){c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < 16; ++i) v[t][b][i] = turn[(16 * h + i) * kTurnRow + h * 32 + r];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (read before the next block is written)
          }
          if (fold_in) {
            float t2 = 0.0f;
            uint32_t any = 0;
#pragma unroll
            for (int p = 0; p < C::kP; ++p) {
              t2 += fabsf(sums[p * C::kRows + row]);
              any |= __builtin_bit_cast(uint32_t, sums[p * C::kRows + row]);
            }
            const float rms = (int32_t)any < 0 && a.norm_w ? 1.0f : sqrtf(t2 / (float)a.K + a.eps);   // (negative: normalised)
            // divided, as by the other kernels: v / rms ~ q = v (1 / rms), one correction by its remainder, which is exact, and infinities,
            // zeros and NaN as a division gives them.  A plain division's ~ 10 instructions for each of up to 32 sums cost a call 2 .. 5 %
            // (us, 64 rows, int4 4096 -> 22016 22.3 -> 22.9), these four 0.3 .. 1 %; the product with 1 / rms alone rounds twice (a call's
            // error, 40 rows 4096 -> 4096: 8.4e-8 of the result, these 7.9e-8).
            const float inv = 1.0f / rms;
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const float y = v[t][b][i], q = y * inv;
                v[t][b][i] = __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, rms, y), inv, q), rms, y);
              }
          }
        }
        block_out<FOLD, CT, C::kRf>(a, v, t0 + h, m0 + f * 32 * C::kRf + r, NT, hsq, psq);
        if (fold_out)
#pragma unroll
          for (int b = 0; b < C::kRf; ++b) {
            const float2 p = make_float2(hsq[b] + lane_xor<32>(hsq[b]), psq[b] + lane_xor<32>(psq[b]));
            if (h == 0) red[wn * C::kRows + (f * C::kRf + b) * 32 + r] = p;
          }
      }
  if (fold_out) {
    lds_barrier();
    wide_fold_store<C::kRows, WN, C::kCols / 16>(a, red, cb, m0, tid);
  }
  stamp_end(a.stamp, t_entry);
}

// ------------------------------------------------------------------ host: shapes, plan, launch
// Estimated us: fix + stages * max(alone, full * rounds) + round * rounds, a round being one workgroup on each CU (fitted, per
// shape and format, to 10 .. 13 numbers of rows from 65 to 1024 by 14 (columns, K) from 1024 x 2048 to 22016 x 4096 and 4096 x 11008
// with the epilogues a model has there, weights from HBM).  Fewer rows are taken by the same numbers: of 17 to 64 rows a launch takes 0.9 ..
// 1.1 (int4), 1.0 .. 1.4 (int8) and 1.0 .. 1.5 (fp16) of its estimate, by shape, the more the more its weights fill the time.
// Blocks of 32 rows and of 4 groups of waves are for grids that would leave
// CUs idle or a wave a SIMD (us, without -> with, int4: 2048 -> 2048 at 128 rows 9.9 -> 7.3, 5632 -> 2048 at 333 22.4 -> 17.5, 4096 -> 12288 at
// 150 30.8 -> 23.7; int8: 11008 -> 4096 at 150 38.8 -> 31.9, 5632 -> 2048 at 333 22.6 -> 19.4; fp16: 2048 -> 2560 at 128 11.3 -> 9.8; the
// mean up to 640 rows 9 %, 6 % and 4 %).
struct BlockShape {
  const void* fn[2];   // [fold]
  int rows, cols, groups, threads, lds[2];   // (lds: [fold])
  float fix, alone, full, round;
};
template <int F, int WN, int KG, int RT, int CT, int NS>
static BlockShape block_shape(float fix, float alone, float full, float round) {
  typedef BlockGemm<F, WN, KG, RT, CT, NS> C;
  const void* fold = nullptr;
  // (a fold's calls have up to 64 rows; int4's 64 x 256 is the fastest of none of them, and spills)
  if constexpr (RT <= 2 && CT == 1) fold = (const void*)gemm_block_kernel<F, WN, KG, RT, CT, NS, true>;
  return {{(const void*)gemm_block_kernel<F, WN, KG, RT, CT, NS, false>, fold}, C::kRows, C::kCols, KG, 64 * C::kWaves, {C::kLds, C::kFoldLds}, fix, alone, full, round};
}
struct BlockShapes {
  const BlockShape* s;
  int n;
};
static BlockShapes block_shapes_of(int fmt) {   // rows x columns (by groups of waves)
  if (fmt == 4) {
    static const BlockShape s[] = {
        block_shape<4, 8, 1, 4, 1, 2>(0.0f, 0.368f, 1.432f, 7.200f),     // 128 x 256
        block_shape<4, 4, 1, 2, 2, 4>(1.294f, 0.946f, 0.803f, 3.204f),   // 64 x 256
        block_shape<4, 6, 1, 3, 1, 3>(0.855f, 1.039f, 1.029f, 4.991f),   // 96 x 192
        block_shape<4, 4, 2, 2, 1, 3>(1.227f, 0.604f, 1.016f, 3.220f),   // 64 x 128 (2)
        block_shape<4, 4, 1, 2, 1, 3>(1.882f, 0.683f, 0.469f, 1.334f),   // 64 x 128
        block_shape<4, 4, 2, 1, 1, 3>(3.245f, 0.602f, 0.557f, 0.939f),   // 32 x 128 (2)
        block_shape<4, 2, 4, 1, 1, 2>(2.771f, 0.801f, 0.688f, 1.218f),   // 32 x 64 (4)
        block_shape<4, 2, 2, 1, 1, 3>(3.256f, 0.475f, 0.354f, 0.521f),   // 32 x 64 (2)
        block_shape<4, 1, 4, 1, 1, 2>(2.905f, 0.654f, 0.503f, 0.789f)};  // 32 x 32 (4)
    return {s, (int)(sizeof(s) / sizeof(s[0]))};
  }
  if (fmt == 8) {
    static const BlockShape s[] = {
        block_shape<8, 8, 1, 4, 1, 2>(0.0f, 1.171f, 1.539f, 7.474f),     // 128 x 256
        block_shape<8, 4, 2, 4, 1, 2>(2.693f, 1.358f, 2.026f, 3.539f),   // 128 x 128 (2)
        block_shape<8, 4, 1, 4, 1, 2>(2.800f, 1.168f, 0.972f, 1.691f),   // 128 x 128
        block_shape<8, 6, 1, 3, 1, 3>(1.304f, 1.119f, 1.106f, 4.927f),   // 96 x 192
        block_shape<8, 4, 2, 2, 1, 3>(0.571f, 0.379f, 1.097f, 4.039f),   // 64 x 128 (2)
        block_shape<8, 4, 1, 2, 1, 3>(3.613f, 0.597f, 0.550f, 0.396f),   // 64 x 128
        block_shape<8, 2, 4, 2, 1, 2>(1.490f, 1.272f, 1.335f, 3.557f),   // 64 x 64 (4)
        block_shape<8, 2, 2, 2, 1, 2>(2.422f, 0.834f, 0.711f, 1.151f),   // 64 x 64 (2)
        block_shape<8, 4, 2, 1, 1, 3>(2.706f, 0.771f, 0.758f, 1.251f),   // 32 x 128 (2)
        block_shape<8, 2, 4, 1, 1, 2>(2.734f, 0.920f, 0.877f, 1.168f),   // 32 x 64 (4)
        block_shape<8, 2, 2, 1, 1, 3>(2.489f, 0.539f, 0.445f, 0.716f),   // 32 x 64 (2)
        block_shape<8, 1, 4, 1, 1, 2>(3.013f, 0.705f, 0.635f, 0.583f)};  // 32 x 32 (4)
    return {s, (int)(sizeof(s) / sizeof(s[0]))};
  }
  if (fmt == 16) {
    static const BlockShape s[] = {
        block_shape<16, 8, 1, 4, 1, 2>(1.278f, 1.734f, 1.703f, 2.529f),   // 128 x 256
        block_shape<16, 4, 2, 4, 1, 2>(1.963f, 1.301f, 2.077f, 2.948f),   // 128 x 128 (2)
        block_shape<16, 4, 1, 4, 1, 2>(3.563f, 1.155f, 1.016f, 0.0f),     // 128 x 128
        block_shape<16, 6, 1, 3, 1, 3>(3.988f, 1.243f, 1.228f, 0.279f),   // 96 x 192
        block_shape<16, 4, 1, 2, 1, 3>(2.426f, 0.835f, 0.702f, 0.0f),     // 64 x 128
        block_shape<16, 2, 2, 2, 1, 2>(2.637f, 0.996f, 0.903f, 0.078f),   // 64 x 64 (2)
        block_shape<16, 2, 2, 1, 1, 3>(2.225f, 0.807f, 0.709f, 0.0f),     // 32 x 64 (2)
        block_shape<16, 1, 4, 1, 1, 2>(3.066f, 0.913f, 0.886f, 0.186f)};  // 32 x 32 (4)
    return {s, (int)(sizeof(s) / sizeof(s[0]))};
  }
  return {nullptr, 0};
}

// The shape whose busiest CU is done first.  A fold's sums and marks cost its calls ~ 1.5 us.
bool block_plan(int fmt, int M, int N, int K, int cus, bool fold, BlockPlan* p, int only) {
  const BlockShapes sh = block_shapes_of(fmt);
  if (M <= (fmt == 16 ? 32 : 16) || M > (fold ? TI_FOLD_SS_ROWS : TI_GEMM_MAX_ROWS) || N < 16 || (N & 15) || K < 128 || (K & 127)) return false;
  const int NT = N >> 4, KT = K >> 7;
  // (the kernel's byte offsets into the weights and their scales are 32 bits)
  if ((uint64_t)NT * KT * (fmt * 256u) >= 0xfff00000ull) return false;
  p->shape = -1;
  for (int i = 0; i < sh.n; ++i) {
    const BlockShape& s = sh.s[i];
    if ((only >= 0 && i != only) || (fold && !s.fn[1])) continue;
    const int n_cb = (N + s.cols - 1) / s.cols, n_rb = (M + s.rows - 1) / s.rows;
    const long n = ((long)((n_cb + 7) / 8) * n_rb + cus / 8 - 1) / (cus / 8);   // (launched: whole XCD rows)
    const float one = (float)n * s.full;
    const float us = (fold ? 1.5f : 0.0f) + s.fix + (float)((KT + s.groups - 1) / s.groups) * (one > s.alone ? one : s.alone) + (float)n * s.round;
    if (p->shape < 0 || us < p->us) *p = {i, n_cb, n_rb, fold, us};
  }
  return p->shape >= 0;
}

int block_prepare() {
  for (int f : {4, 8, 16}) {
    const BlockShapes sh = block_shapes_of(f);
    for (int i = 0; i < sh.n; ++i)
      for (int f2 = 0; f2 < 2; ++f2)
        if (sh.s[i].fn[f2] && sh.s[i].lds[f2] > 64 * 1024)
          TI_HIP_CHECK(hipFuncSetAttribute(sh.s[i].fn[f2], hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                       "hipFuncSetAttribute(gemm_block_kernel)");
  }
  return TI_OK;
}

long block_workgroups(const BlockPlan& p) { return (long)((p.n_cb + 7) / 8) * 8 * p.n_rb; }

int block_launch(int fmt, const BlockPlan& p, const GemvArgs& a, hipStream_t stream) {
  const BlockShape& s = block_shapes_of(fmt).s[p.shape];
  GemvArgs arg = a;
  int n_cb = p.n_cb, n_rb = p.n_rb;
  void* args[] = {&arg, &n_cb, &n_rb};
  TI_HIP_CHECK(hipLaunchKernel(s.fn[p.fold], dim3((unsigned)block_workgroups(p)), dim3(s.threads), args, s.lds[p.fold], stream),
               "hipLaunchKernel(gemm_block_kernel)");
  TI_LAUNCH_CHECK("gemm_block_kernel");
  return TI_OK;
}

}  // namespace ti
