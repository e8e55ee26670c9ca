// gemm_wide.hip -- packed weights x fp16 rows for many rows (prompt chunks, large batches), every weight
// format of ti_gemm_wq_a16: int4 / int8 per group of 128, blocks of 32 (GGUF Q4_0, Q8_0, Q4_1), fp16.
#include <type_traits>

#include "gemm_common.hpp"
#include "gemm_wide.hpp"

namespace ti {

typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32x4s raw_rsrc(const void* p, uint32_t bytes) {
  const uint64_t a = (uint64_t)p;
  u32x4s r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}
// 64 lanes x 16 (4) bytes from rsrc + lane offset + wave offset to LDS byte address lds.  Issued from asm, so
// hipcc does not count it: the caller waits with a counted s_waitcnt vmcnt and a barrier.
__device__ __forceinline__ void dma16(u32x4s rs, uint32_t voff, uint32_t soff, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(voff), "s"(rs), "s"(soff), "s"(lds) : "memory");
}
__device__ __forceinline__ void dma4(u32x4s rs, uint32_t voff, uint32_t soff, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(voff), "s"(rs), "s"(soff), "s"(lds) : "memory");
}

template <int F, int WM, int WN, int TM, int TN, int NS>
struct WideCfg {
  typedef WideFmt<F> W;
  static constexpr int kWaves = WM * WN, kRows = 16 * TM * WM, kTiles = TN * WN;
  static constexpr int kA = kRows * 256, kW = kTiles * W::kTile;
  static constexpr int kScaleDma = W::kScale == 0 ? 0 : (TN * W::kScale + 255) / 256 * (W::kAff ? 2 : 1);   // dword DMAs per wave
  static constexpr int kS = kWaves * kScaleDma * 256;
  static constexpr int kStage = kA + kW + kS;
  // after the stream: rms per row | each wave's staging block | (sum of h^2, of (h w)^2) per column-wave and row | ticket
  static constexpr int kEpiStg = kRows * 4, kEpiRed = kEpiStg + kWaves * 16 * TM * kTileEpiStride * 4;
  static constexpr int kEpiFlag = kEpiRed + 2 * WN * kRows * 4, kEpi = kEpiFlag + 16;
  static constexpr int kLds = NS * kStage > kEpi ? NS * kStage : kEpi;
  static constexpr bool kFold = kRows <= TI_FOLD_SS_ROWS;   // (every wave of these has all rows)
  static_assert(!kFold || WM == 1, "a wave sees every row's rms");
  static constexpr int kDmaA = kRows / 4 / kWaves, kDmaW = kTiles * (W::kTile / 1024) / kWaves;
  static constexpr int kDma = kDmaA + kDmaW + kScaleDma;
  static_assert(kRows / 4 % kWaves == 0 && kTiles * (W::kTile / 1024) % kWaves == 0, "equal DMA counts per wave");
};

// Split-K merge of a workgroup's block: every k-slice's workgroup stores its fp32 partial block write-through into
// the workspace and, its stores drained, adds to the block's ticket; the last arriver reads the other slices back
// (sc1 loads), sums the n_ks slices in slice order (deterministic whatever the arrival order), re-arms the ticket
// and runs the epilogue (true).  Every wave of the workgroup calls it.
template <int TN, int TM>
__device__ __forceinline__ bool wide_merge(const GemvArgs& a, f32x4 (&acc)[TN][TM], int block, int n_blocks, int waves, int wave,
                                           int ks, int n_ks, int lane, int* flag) {
  char* ws = (char*)a.epi.splitk_ws;
  int32_t* ticket = (int32_t*)ws + block;
  const __amdgpu_buffer_rsrc_t rs = sc1_rsrc(ws + TI_SPLITK_TICKET_BYTES);
  constexpr int kSlab = TN * TM * kWave * 16;   // bytes per wave and slice
  auto off = [&](int sl, int t, int b) {
    return (uint32_t)((((size_t)sl * n_blocks + block) * waves + wave) * kSlab + (size_t)((t * TM + b) * kWave + lane) * 16);
  };
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int b = 0; b < TM; ++b) __builtin_amdgcn_raw_buffer_store_b128(acc[t][b], rs, off(ks, t, b), 0, kAuxSc1Load);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  lds_barrier();
  if (*flag != n_ks - 1) return false;
  f32x4 sum[TN][TM];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int b = 0; b < TM; ++b) sum[t][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  constexpr int CH = TN * TM >= 8 ? 1 : TN * TM >= 4 ? 2 : 4;   // slices per round trip (registers)
  for (int s0 = 0; s0 < n_ks; s0 += CH) {
    f32x4 ld[CH][TN][TM];
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int b = 0; b < TM; ++b)
          ld[c][t][b] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off(min(s0 + c, n_ks - 1), t, b), 0, kAuxSc1Load));
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (s0 + c < n_ks)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int b = 0; b < TM; ++b) sum[t][b] += s0 + c == ks ? acc[t][b] : ld[c][t][b];
  }
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[t][b] = sum[t][b];
  if (threadIdx.x == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-arm
  return true;
}

// Bound: int4 and int8 by the vector unit beside the matrix cores (a 16x16x32 MFMA and its share of dequant and scale
// FMAs take ~ 0.87 (16 + 4 V) cycles with V vector instructions per MFMA: V 3 at 64 rows a wave, more with fewer rows
// to share a dequantised tile), small row counts and fp16 by the copies into a CU (~ 45 KB/us with the
// hand-overs of the stages; plain reads reach 110), so a block
// keeps 64 rows as soon as the call has them.  DMA straight to LDS leaves the registers to the accumulators; the
// next stage's unpacking is interleaved with this one's MFMAs.  Measured inside a pass, us (tile and batched-rows
// kernels -> this one): int4 64 rows 4096 -> 12288 24.0 -> 23.1, 4096 -> 22016 32.6 -> 29.0, the mean of 4096 -> 4096 and
// 11008 -> 4096 18.1 -> 17.2.  (Prompt chunks: gemm_block.hip.)
//
// Block of 16 TM WM rows x 16 TN WN columns per workgroup; wave (wm, wn) owns 16 TM rows x TN weight tiles.  A
// stage is one 128-k group of the block: the rows' activations (chunks XOR-swizzled by row, tile_swz), the packed
// weight tiles and their scales, all copied to LDS by DMA, NS stages in flight.
template <int F, int WM, int WN, int TM, int TN, int NS>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_wide_kernel(const GemvArgs a, int n_cb, int n_rb, int n_ks) {
  typedef WideCfg<F, WM, WN, TM, TN, NS> C;
  typedef WideFmt<F> Fm;
  constexpr int NW = C::kWaves;
  const unsigned long long t_entry = stamp_now();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int KT = a.K >> 7, NT = a.N >> 4;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
  // the row blocks and k-slices of a column block share an XCD (its L2 holds their weights once)
  const int rest = blockIdx.x >> 3, rb = rest % n_rb, r2 = rest / n_rb, ks = r2 % n_ks, cb = r2 / n_ks * 8 + (blockIdx.x & 7);
  if (cb >= n_cb) return;
  const int m0 = rb * C::kRows, t0 = cb * C::kTiles;
  const int kb = ks * KT / n_ks, ke = (ks + 1) * KT / n_ks, nk = ke - kb;

  const u32x4s rs_x = raw_rsrc(a.x, (uint32_t)(((size_t)(a.M - 1) * a.ldx + a.K) * 2));
  const u32x4s rs_w = raw_rsrc(a.tiles, (uint32_t)((size_t)NT * KT * Fm::kTile));
  const u32x4s rs_s = raw_rsrc(a.scales, (uint32_t)((size_t)NT * KT * Fm::kScale * (Fm::kAff ? 2 : 1)));
  uint32_t vx[C::kDmaA];
#pragma unroll
  for (int q = 0; q < C::kDmaA; ++q) {
    const int row = 4 * (wave * C::kDmaA + q) + (lane >> 4), c = (lane & 15) ^ tile_swz(row);
    vx[q] = (uint32_t)min(m0 + row, a.M - 1) * (uint32_t)a.ldx * 2u + (uint32_t)c * 16u;
  }
  const uint32_t vl = (uint32_t)lane * 16u;
  uint32_t vs[C::kScaleDma > 0 ? C::kScaleDma : 1];
  if constexpr (C::kScaleDma > 0) {
    constexpr int kPerTile = Fm::kScale / 4, kHalf = Fm::kAff ? C::kScaleDma / 2 : C::kScaleDma;   // dwords per tile
#pragma unroll
    for (int q = 0; q < C::kScaleDma; ++q) {
      const int d = (q % kHalf) * 64 + lane, t = min(d / kPerTile, TN - 1);
      vs[q] = (uint32_t)min(t0 + wn * TN + t, NT - 1) * (uint32_t)KT * Fm::kScale + (uint32_t)(d % kPerTile) * 4u +
              (q >= kHalf ? (uint32_t)NT * (uint32_t)KT * Fm::kScale : 0u);
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  auto issue = [&](int kg, int buf) __attribute__((always_inline)) {   // C::kDma loads per wave, always
    const uint32_t st = lds0 + (uint32_t)buf * C::kStage;
#pragma unroll
    for (int q = 0; q < C::kDmaA; ++q)
      dma16(rs_x, vx[q], (uint32_t)kg * 256u, __builtin_amdgcn_readfirstlane(st + (uint32_t)(wave * C::kDmaA + q) * 1024u));
#pragma unroll
    for (int q = 0; q < C::kDmaW; ++q) {
      const int i = wave * C::kDmaW + q, t = i / (Fm::kTile / 1024), ch = i % (Fm::kTile / 1024);
      const uint32_t so = ((uint32_t)min(t0 + t, NT - 1) * (uint32_t)KT + (uint32_t)kg) * Fm::kTile + (uint32_t)ch * 1024u;
      dma16(rs_w, vl, __builtin_amdgcn_readfirstlane(so), __builtin_amdgcn_readfirstlane(st + C::kA + (uint32_t)i * 1024u));
    }
#pragma unroll
    for (int q = 0; q < C::kScaleDma; ++q)
      dma4(rs_s, vs[q], (uint32_t)kg * (uint32_t)Fm::kScale,
           __builtin_amdgcn_readfirstlane(st + C::kA + C::kW + (uint32_t)(wave * C::kScaleDma + q) * 256u));
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TN][TM];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[t][b] = zero;
  uint32_t magic;
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));

  // Operands of k-step s4 (activation fragments, fp16 also the weights), and of a stage (packed weights, scales,
  // block minimums).
  constexpr int kWr = Fm::kBits == 16 ? 1 : Fm::kBits / 4, kSr = Fm::kG32 ? 4 : 1;
  struct Step {
    f16x8 x[TM];
    u32x4 w[Fm::kBits == 16 ? TN : 1];
  };
  struct Stage {
    u32x4 w[TN][kWr];
    uint16_t sc[TN][kSr], mn[Fm::kAff ? TN : 1][kSr];
  };
  auto read_step = [&](Step& d, int buf, int s4) __attribute__((always_inline)) {
    const char* st = smem + buf * C::kStage;
    const f16* xr = (const f16*)st + (wm * 16 * TM + r) * 128 + (((Fm::kG32 ? s4 * 4 + kq : kq * 4 + s4) ^ tile_swz(r)) * 8);
#pragma unroll
    for (int b = 0; b < TM; ++b) d.x[b] = *(const f16x8*)(xr + b * 16 * 128);
    if constexpr (Fm::kBits == 16)
#pragma unroll
      for (int t = 0; t < TN; ++t)
        d.w[t] = ((const u32x4*)(st + C::kA))[(wn * TN + t) * (Fm::kTile / 16) + s4 * 64 + lane];
  };
  auto read_stage = [&](Stage& d, int buf) __attribute__((always_inline)) {
    if constexpr (Fm::kBits != 16) {
      const char* st = smem + buf * C::kStage;
      const u32x4* wl = (const u32x4*)(st + C::kA) + wn * TN * (Fm::kTile / 16) + lane;
      const uint16_t* sl = (const uint16_t*)(st + C::kA + C::kW + wave * C::kScaleDma * 256) + r;
#pragma unroll
      for (int t = 0; t < TN; ++t) {
#pragma unroll
        for (int c = 0; c < kWr; ++c) d.w[t][c] = wl[t * (Fm::kTile / 16) + c * 64];
#pragma unroll
        for (int j = 0; j < kSr; ++j) {
          d.sc[t][j] = sl[(t * kSr + j) * 16];
          if constexpr (Fm::kAff) d.mn[t][j] = sl[C::kScaleDma / 2 * 128 + (t * kSr + j) * 16];
        }
      }
    }
  };
  auto deq = [&](const Stage& g, int s4, int t) __attribute__((always_inline)) -> f16x8 {
    if constexpr (Fm::kBits == 8) return dequant_step<8>(g.w[t], s4, magic);
    else return deq_int4_signed(g.w[t][0][s4], magic);
  };
  // A unit is (k-step, tile): TM products.  Among them go the dequantization of the next unit's weights (bfn) and the
  // scaling of a finished partial sum: group-128 a tile's four steps sum into part[t], scaled one unit later; blocks
  // of 32 one unit's products, in alternating halves of part.  `pend` (`pm`): the scale (offset) of the partial sums
  // that the last unit left unscaled.
  f32x4 part[Fm::kBits == 16 ? 1 : Fm::kG32 ? 2 : TN][TM];
  f32x4 xs[Fm::kAff ? 2 : 1][TM];
  f16x8 bfn;
  float pend = 0.0f, pm = 0.0f;
  if constexpr (Fm::kBits != 16)
#pragma unroll
    for (int b = 0; b < TM; ++b) part[Fm::kG32 ? 1 : TN - 1][b] = xs[Fm::kAff ? 1 : 0][b] = zero;
  auto mul = [&](const Step& d, const Stage& g, const Stage& gn, auto sc_) __attribute__((always_inline)) {
    constexpr int s4 = decltype(sc_)::value;
    if constexpr (Fm::kBits == 16) {
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const f16x8 bf = __builtin_bit_cast(f16x8, d.w[t]);
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.x[b], bf, acc[t][b], 0, 0, 0);
      }
      return;
    }
    if constexpr (Fm::kAff) {   // the block's sum of x per row, in every column
      const f16x8 ones = {(f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1, (f16)1};
#pragma unroll
      for (int b = 0; b < TM; ++b) xs[s4 & 1][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.x[b], ones, zero, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      constexpr int kUnits = 4 * TN;
      const int p = Fm::kG32 ? (s4 * TN + t) & 1 : t, tp = t > 0 ? t - 1 : TN - 1;   // slot of this unit, tile before it
      const f16x8 bf = bfn;
      bfn = t + 1 < TN ? deq(g, s4, t + 1) : s4 < 3 ? deq(g, (s4 + 1) & 3, 0) : deq(gn, 0, 0);
      const bool scale = Fm::kG32 || (s4 == 0 && t == 0) || (s4 == 3 && t > 0);
      if (scale) {
        const f32x4* q = part[Fm::kG32 ? p ^ 1 : tp];
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[tp][b] = fma_scale4(pend, q[b], acc[tp][b]);
        if constexpr (Fm::kAff) {   // weight = d (q - 8) + (8 d + m)
          const f32x4* x1 = xs[t > 0 ? s4 & 1 : (s4 & 1) ^ 1];
#pragma unroll
          for (int b = 0; b < TM; ++b) acc[tp][b] = fma_scale4(pm, x1[b], acc[tp][b]);
        }
      }
#pragma unroll
      for (int b = 0; b < TM; ++b)
        part[p][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(d.x[b], bf, Fm::kG32 || s4 == 0 ? zero : part[p][b], 0, 0, 0);
      if (Fm::kG32 || s4 == 3) pend = h2f(g.sc[t][Fm::kG32 ? s4 : 0]);
      if constexpr (Fm::kAff) pm = fmaf(8.0f, pend, h2f(g.mn[t][s4]));
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                     // one product,
        if (scale) __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);          // then vector arithmetic
        else __builtin_amdgcn_sched_group_barrier(0x002, 12 / TM, 0);
      }
      static_assert(!Fm::kG32 || kUnits % 2 == 0, "alternating halves");
    }
  };

  // Stage kg lives in buffer kg % NS.  Each k-step's operands are read from LDS one step ahead; the last step of
  // a stage waits for the next stage's DMA, meets the other waves (whose reads of this stage are done, so its
  // buffer takes stage kg + NS) and reads the next stage's first operands before its own products.
#pragma unroll
  for (int s = 0; s < NS; ++s) issue(min(kb + s, ke - 1), s);
  // batched fold (decode rows, ti_hip.h TI_FOLD_SS_ROWS): this thread's share of its row's sum of squares
  const bool fold_in = C::kFold && a.epi.ss_in != nullptr;
  const float share = fold_in ? wide_fold_share(a, m0 + tid % C::kRows, tid / C::kRows, 64 * NW / C::kRows) : 0.0f;
  // What the epilogue reads: blocks of 64 x 64 (one tile a wave) ask for it beside their products, the others behind the main loop, a
  // tile at a time (us, 16 x 64 blocks of int4, early -> late: 512 -> 256 4.4 -> 4.0, 1024 -> 1024 split over K 5.9 -> 5.5; early, 16 and 32 rows
  // take 10 .. 17 registers more, a wave a SIMD).
  constexpr bool kEarly = TN == 1 && TM == 4;
  TilePre<TM> pre;
  if constexpr (kEarly) tile_pos<TM>(a, m0 + wm * 16 * TM, lane, pre);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * C::kDma) : "memory");
  lds_barrier();
  Step st[2];
  Stage sg[2];
  read_stage(sg[0], 0);
  read_step(st[0], 0, 0);
  if constexpr (Fm::kBits != 16) bfn = deq(sg[0], 0, 0);
  int buf = 0;
  auto stage = [&](int kg, Stage& cur, Stage& next) __attribute__((always_inline)) {
    read_step(st[1], buf, 1);
    __builtin_amdgcn_sched_barrier(0);
    mul(st[0], cur, next, std::integral_constant<int, 0>());
    __builtin_amdgcn_sched_barrier(0);
    read_step(st[0], buf, 2);
    __builtin_amdgcn_sched_barrier(0);
    mul(st[1], cur, next, std::integral_constant<int, 1>());
    __builtin_amdgcn_sched_barrier(0);
    read_step(st[1], buf, 3);
    __builtin_amdgcn_sched_barrier(0);
    mul(st[0], cur, next, std::integral_constant<int, 2>());
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * C::kDma) : "memory");   // this wave's part of stage kg + 1
    lds_barrier();
    issue(min(kb + kg + NS, ke - 1), buf);
    buf = buf + 1 == NS ? 0 : buf + 1;
    read_stage(next, buf);
    read_step(st[0], buf, 0);
    __builtin_amdgcn_sched_barrier(0);
    mul(st[1], cur, next, std::integral_constant<int, 3>());
    __builtin_amdgcn_sched_barrier(0);
  };
  int kg = 0;
  for (; kg + 2 <= nk; kg += 2) {
    stage(kg, sg[0], sg[1]);
    stage(kg + 1, sg[1], sg[0]);
  }
  if (kg < nk) stage(kg, sg[0], sg[1]);
  auto last = [&]() __attribute__((always_inline)) {   // what the last unit left
    if constexpr (Fm::kBits != 16)
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        acc[TN - 1][b] = fma_scale4(pend, part[Fm::kG32 ? 1 : TN - 1][b], acc[TN - 1][b]);
        if constexpr (Fm::kAff) acc[TN - 1][b] = fma_scale4(pm, xs[1][b], acc[TN - 1][b]);
      }
  };
  last();
  if constexpr (kEarly) tile_pre<TM>(a, min(t0 + wn * TN, NT - 1), m0 + wm * 16 * TM, lane, pre);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the clamped stages past the end
  lds_barrier();

  float* rmsv = (float*)smem;
  float rms[TM][4];
#pragma unroll
  for (int b = 0; b < TM; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) rms[b][i] = 1.0f;
  if (fold_in) {
    wide_fold_rms<C::kRows, NW>(a, share, tid, rmsv);
    auto marked = [&]() __attribute__((always_inline)) {   // (reads the rows' rms; one of them is negative)
      uint32_t any = 0;
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          rms[b][i] = rmsv[wm * 16 * TM + b * 16 + 4 * kq + i];
          any |= __builtin_bit_cast(uint32_t, rms[b][i]);
        }
      return __builtin_amdgcn_ballot_w64((int32_t)any < 0) != 0;
    };
    if (__builtin_expect(marked(), 0)) {
      if (a.norm_w) wide_fold_settle<C::kRows, NW>(a, m0, tid, rmsv);
      if (a.norm_w && marked()) {   // rows that fp16 did not hold: again, behind their rewriting, a stage at a time
        wide_refold<C::kRows, NW>(a, m0, wave, lane, rmsv);
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int b = 0; b < TM; ++b) acc[t][b] = zero;
        pend = pm = 0.0f;
        if constexpr (Fm::kBits != 16)
#pragma unroll
          for (int b = 0; b < TM; ++b) part[Fm::kG32 ? 1 : TN - 1][b] = xs[Fm::kAff ? 1 : 0][b] = zero;
#pragma unroll 1
        for (int kg = kb; kg < ke; ++kg) {
          issue(kg, 0);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          lds_barrier();
          read_stage(sg[0], 0);
          if constexpr (Fm::kBits != 16) bfn = deq(sg[0], 0, 0);
          [&]<int... S>(std::integer_sequence<int, S...>) __attribute__((always_inline)) {
            ((read_step(st[0], 0, S), mul(st[0], sg[0], sg[0], std::integral_constant<int, S>())), ...);
          }(std::make_integer_sequence<int, 4>());
          lds_barrier();
        }
        last();
      }
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) rms[b][i] = rms[b][i] < 0.0f && a.norm_w ? 1.0f : fabsf(rms[b][i]);
    }
  }
  if (n_ks > 1 && !wide_merge<TN, TM>(a, acc, cb * n_rb + rb, n_cb * n_rb, NW, wave, ks, n_ks, lane, (int*)(smem + C::kEpiFlag))) {
    stamp_end(a.stamp, t_entry);
    return;
  }
  const ti_epilogue& e = a.epi;
  const bool fold_out = C::kFold && e.kind == TI_EPI_RESID_F32 && e.fold_x != nullptr;
  float* stg = (float*)(smem + C::kEpiStg) + wave * (16 * TM * kTileEpiStride);
  const int mb = m0 + wm * 16 * TM;
  float hsq[TM], psq[TM];
#pragma unroll
  for (int b = 0; b < TM; ++b) hsq[b] = psq[b] = 0.0f;
  if constexpr (!kEarly) tile_pos<TM>(a, mb, lane, pre);
#pragma unroll 1
  for (int t = 0; t < TN; ++t) {   // (rolled: the tile's accumulators by static selects, so acc stays in registers)
    const int tn = t0 + wn * TN + t;
    f32x4 av[TM];
#pragma unroll
    for (int tt = 0; tt < TN; ++tt)
      if (tt == t)
#pragma unroll
        for (int b = 0; b < TM; ++b) av[b] = acc[tt][b];
    if (tn >= NT) continue;
    // (values of this tile: the rows' addresses of every epilogue, taken out of the loop, are up to 56 registers, and int4's 64 x 128
    // blocks run 3 a CU: 4096 -> 22016 at 1024 rows 215 -> 194 us)
    int ln = lane;
    if constexpr (TN > 1) {
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int b = 0; b < TM; ++b) asm volatile("" : "+v"(pre.pos[b]));
    }
    if constexpr (!kEarly) tile_pre<TM>(a, tn, mb, ln, pre);
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        stg[(b * 16 + 4 * kq + i) * kTileEpiStride + r] = fold_in ? av[b][i] / rms[b][i] : av[b][i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wide_tile_out<TM>(a, tn, mb, stg, ln, r, kq, fold_out, pre, hsq, psq);
  }
  if (fold_out) {   // this column block's sum of h^2 per row, column-waves in order
    float2* red = (float2*)(smem + C::kEpiRed);
    wide_fold_part<TM>(red + wn * C::kRows + wm * 16 * TM, hsq, psq, lane);
    lds_barrier();
    wide_fold_store<C::kRows, WN, C::kTiles>(a, red, cb, m0, tid);
  }
  if (e.kind == TI_EPI_LOGITS_ARGMAX && e.step_ctr && cb == 0 && rb == 0 && tid == 0) *e.step_ctr += e.advance;
  stamp_end(a.stamp, t_entry);
}

// ------------------------------------------------------------------ host: shapes, plan, launch
// Workgroup shapes.  us: one 128-k stage of a workgroup alone on its CU, and per workgroup of a full CU (measured,
// K 2048 .. 11008, weights from HBM; the launch's own ~ 4.5 us and a split's seam come on top, wide_plan).
struct WideShape {
  const void* fn;
  int rows, tiles, threads, lds, slab;   // slab: bytes of a split-K slice of one block
  float alone, full;
};
template <int F, int WM, int WN, int TM, int TN, int NS>
static WideShape wide_shape(float alone, float full) {
  typedef WideCfg<F, WM, WN, TM, TN, NS> C;
  static_assert(C::kLds <= 160 * 1024, "LDS");
  return {(const void*)gemm_wide_kernel<F, WM, WN, TM, TN, NS>, C::kRows, C::kTiles, 64 * C::kWaves, C::kLds,
          C::kWaves * TN * TM * kWave * 16, alone, full};
}
constexpr int kWideShapes = 5;
template <int F>
static const WideShape* wide_shapes() {   // 64 x 384 (fp16: 128 x 192, blocks of 32: none) | 64 x 128 (fp16: 128 x 128) | 64 x 64 | 32 x 64 | 16 x 64
  if constexpr (F == 4) {
    static const WideShape s[kWideShapes] = {wide_shape<F, 1, 8, 4, 3, 2>(1.25f, 1.53f), wide_shape<F, 1, 4, 4, 2, 2>(1.00f, 0.51f),
                                             wide_shape<F, 1, 4, 4, 1, 3>(0.42f, 0.345f), wide_shape<F, 1, 4, 2, 1, 3>(0.30f, 0.22f),
                                             wide_shape<F, 1, 4, 1, 1, 3>(0.23f, 0.18f)};
    return s;
  } else if constexpr (F == 8) {
    static const WideShape s[kWideShapes] = {wide_shape<F, 1, 8, 4, 3, 2>(1.25f, 1.81f), wide_shape<F, 1, 4, 4, 2, 2>(1.17f, 0.61f),
                                             wide_shape<F, 1, 4, 4, 1, 3>(0.46f, 0.41f), wide_shape<F, 1, 4, 2, 1, 3>(0.36f, 0.36f),
                                             wide_shape<F, 1, 4, 1, 1, 3>(0.32f, 0.32f)};
    return s;
  } else if constexpr (F == 16) {
    // (128 x 128 -> 128 x 192, us: 333 rows 2048 -> 11264 49 -> 33, one round instead of two; 1000 rows 81 -> 68)
    static const WideShape s[kWideShapes] = {wide_shape<F, 2, 4, 4, 3, 2>(1.62f, 1.62f), wide_shape<F, 2, 4, 4, 2, 2>(1.30f, 1.30f),
                                             wide_shape<F, 1, 4, 4, 1, 3>(0.57f, 0.56f), wide_shape<F, 1, 4, 2, 1, 3>(0.60f, 0.64f),
                                             wide_shape<F, 1, 4, 1, 1, 3>(0.55f, 0.60f)};
    return s;
  } else {
    constexpr float u = F & TI_BITS_AFF ? 1.3f : 1.0f;
    static const WideShape s[kWideShapes] = {{nullptr}, wide_shape<F, 1, 4, 4, 2, 2>(1.15f * u, 0.72f * u),
                                             wide_shape<F, 1, 4, 4, 1, 2>(0.51f * u, 0.42f * u), wide_shape<F, 1, 4, 2, 1, 3>(0.36f * u, 0.32f * u),
                                             wide_shape<F, 1, 4, 1, 1, 3>(0.30f * u, 0.24f * u)};
    return s;
  }
}
static const WideShape* wide_shapes_of(int fmt) {
  switch (fmt) {
    case 4: return wide_shapes<4>();
    case 8: return wide_shapes<8>();
    case 16: return wide_shapes<16>();
    case 4 | TI_BITS_G32: return wide_shapes<4 | TI_BITS_G32>();
    case 8 | TI_BITS_G32: return wide_shapes<8 | TI_BITS_G32>();
    case 4 | TI_BITS_G32 | TI_BITS_AFF: return wide_shapes<4 | TI_BITS_G32 | TI_BITS_AFF>();
    default: return nullptr;
  }
}

// The shape and split whose busiest CU is done first.  Rows per block: 16, 32 and 64 (128; a fold's block has all rows in
// every wave) as the call's rows need;
// splits only into slices of at least 4 stages, whose blocks fit the workspace, and of at most two workgroups a CU
// (the seam, measured: ~ 0.5 us + 0.65 us per MB of partial blocks).
bool wide_plan(int fmt, int M, int N, int K, int cus, int64_t ws_bytes, bool fold, WidePlan* p, int only) {
  const WideShape* sh = wide_shapes_of(fmt);
  if (!sh || M < 1 || M > TI_GEMM_MAX_ROWS || N < 16 || (N & 15) || K < 128 || (K & 127)) return false;
  const int NT = N >> 4, KT = K >> 7;
  // (the kernel's byte offsets into the weights and their scales are 32 bits)
  if ((uint64_t)NT * KT * ((fmt & 31) * 256u) >= 0xfff00000ull) return false;
  float best = 0.0f;
  p->shape = -1;
  for (int i = 0; i < kWideShapes; ++i) {
    const WideShape& s = sh[i];
    if (!s.fn || (only >= 0 && i != only) || (s.rows < 64 && M > s.rows) || (s.rows >= 64 && M <= 32) || (fold && s.rows > TI_FOLD_SS_ROWS)) continue;
    const int n_cb = (NT + s.tiles - 1) / s.tiles, n_rb = (M + s.rows - 1) / s.rows;
    const long per_xcd = (long)((n_cb + 7) / 8) * n_rb;   // (launched: whole XCD rows)
    for (int ks = 1; ks <= 8; ks += ks < 4 ? 1 : 2) {
      if (ks > 1 && (KT / ks < 4 || per_xcd * ks > cus / 4 || !gemm_knobs().splitk || (size_t)n_cb * n_rb * 4 > TI_SPLITK_TICKET_BYTES ||
                     (int64_t)((size_t)ks * n_cb * n_rb * s.slab + TI_SPLITK_TICKET_BYTES) > ws_bytes))
        break;
      const int nk = (KT + ks - 1) / ks;
      const long n = (per_xcd * ks + cus / 8 - 1) / (cus / 8);
      const float one = (float)n * s.full, mb = 1e-6f * (float)ks * (float)n_cb * (float)n_rb * (float)s.slab;
      const float alone = 4.5f + (float)nk * (one > s.alone ? one : s.alone), us = ks > 1 ? alone + 0.5f + 0.65f * mb : alone;
      if (p->shape < 0 || us < best) {
        best = us;
        *p = {i, n_cb, n_rb, ks, s.rows, s.tiles, us, ks > 1 ? alone + 0.8f + 0.3f * (float)ks + 0.35f * mb : us};
      }
    }
  }
  return p->shape >= 0;
}

int wide_prepare() {
  for (int f : {4, 8, 16, 4 | TI_BITS_G32, 8 | TI_BITS_G32, 4 | TI_BITS_G32 | TI_BITS_AFF}) {
    const WideShape* sh = wide_shapes_of(f);
    for (int i = 0; i < kWideShapes; ++i)
      if (sh[i].fn && sh[i].lds > 64 * 1024)
        TI_HIP_CHECK(hipFuncSetAttribute(sh[i].fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                     "hipFuncSetAttribute(gemm_wide_kernel)");
  }
  return TI_OK;
}

long wide_workgroups(const WidePlan& p) { return (long)((p.n_cb + 7) / 8) * 8 * p.n_rb * p.n_ks; }

int wide_launch(int fmt, const WidePlan& p, const GemvArgs& a, hipStream_t stream) {
  const WideShape& s = wide_shapes_of(fmt)[p.shape];
  GemvArgs arg = a;
  int n_cb = p.n_cb, n_rb = p.n_rb, n_ks = p.n_ks;
  void* args[] = {&arg, &n_cb, &n_rb, &n_ks};
  TI_HIP_CHECK(hipLaunchKernel(s.fn, dim3((unsigned)wide_workgroups(p)), dim3(s.threads), args, s.lds, stream),
               "hipLaunchKernel(gemm_wide_kernel)");
  TI_LAUNCH_CHECK("gemm_wide_kernel");
  return TI_OK;
}

}  // namespace ti

// Which kernel a call of ti_gemm_rows takes, by their estimates (the many-rows kernel's is 4 % (int4, also in blocks of 32), 12 % (int8 in
// blocks of 32) or 8 % low for calls of up to 48 rows).
//   Few rows: more than one round of workgroups over the CUs only up to 16 rows, int4 only for logits (us, few / many rows: int4 4096 ->
//   28672 at 16 rows 18.8 / 17.5, 32000 logits 21.8 / 23.5; blocks of 32 bytes' 4096 -> 22016 at 31 rows 24.3 / 22.1).
//   Block: an output that it writes (not logits), 33 rows and more (us, before / block at 64 rows: int4 4096 -> 4096 11.9 / 9.4, 4096 -> 22016
//   26 / 21, 2048 -> 2560 9.8 / 6.4, int8 2048 -> 2048 9.4 / 6.0; at 48 rows int4 4096 -> 12288 19.0 / 14.9, int8 4096 -> 22016 31.4 / 27.2);
//   17 to 32 of int4 (32 rows, folded, 4096 -> 28672 22.3 / 20.1, 4096 -> 22016 19.0 / 16.3), and 25 to 32 of int8 up to 24576 columns (4096 ->
//   22016 at 32 rows 27.9 / 27.0, at 17 25.8 / 26.8), as wider weights fill the time (int8 4096 -> 28672 at 17 rows 28.3 / 31.0, at 32 29.9 /
//   30.7; prompts of 22 of the 7B model in fp16 3472 / 3749).
//   Against it a split costs 0.8 us, 0.3 a slice and 0.35 a MB of partial blocks (fitted to 700
//   calls; the split itself is chosen by 0.5 and 0.65 a MB, and with it the order of its sums): the many-rows kernel keeps long K of few rows
//   or narrow outputs (int4 11008 -> 4096 at 64 rows 17.9 / 18.7; 14336 -> 4096 at 96 26.3 / 27.3, fp16 5632 -> 2048 at 700 34.5 / 37.8),
//   and short K, where the blocks' ends weigh.  fp16 folds: by 0.95 of the others' (as often slower
//   as faster from there up: 4096 -> 12288 at 60 rows 27.8 / 28.8, 2048 -> 11264 15.7 / 14.6).
// 6000 calls (3 .. 1024 rows, 21 (columns, K) of five formats, outputs and folds of a model): the choice costs 0.3 .. 0.9 % more than the best
// of the three in the mean, by format.
struct RowsPlan {
  int kernel;   // TI_ROWS_FEW, _MANY or _BLOCK
  ti::FewPlan f;
  ti::WidePlan w;
  ti::BlockPlan b;
  int n_cb() const { return kernel == TI_ROWS_FEW ? f.n_cb : kernel == TI_ROWS_MANY ? w.n_cb : b.n_cb; }
};
// kind: of the epilogue; vec: its rows are whole 16-byte pieces (epilogue_vec)
static bool rows_plan_of(int kernel, int bits, int M, int N, int K, int64_t ws_bytes, bool fold, int kind, bool vec, RowsPlan* p) {
  const int cus = ti::gemm_cus(), only = kernel / TI_ROWS_SHAPE - 1;
  kernel %= TI_ROWS_SHAPE;
  auto asked = [&](int k) { return kernel == TI_ROWS_AUTO || kernel == k; };
  p->kernel = TI_ROWS_AUTO;
  float us = 0.0f, whole = 0.0f;   // of the kernel chosen, by the many-rows kernel's measure
  if (asked(TI_ROWS_MANY) && ti::wide_plan(bits, M, N, K, cus, ws_bytes, fold, &p->w, only)) {
    p->kernel = TI_ROWS_MANY;
    us = p->w.us;
    whole = p->w.whole;
  }
  const float low = (bits & ~TI_BITS_G32) == 4 ? 1.04f : bits == (8 | TI_BITS_G32) ? 1.12f : 1.08f;
  if (asked(TI_ROWS_FEW) && ti::few_plan(bits, M, N, K, cus, &p->f, only) &&
      (p->kernel == TI_ROWS_AUTO ||
       (p->f.us < low * us && (p->f.n_cb <= cus || (M <= 16 && (bits != 4 || kind == TI_EPI_LOGITS_ARGMAX)))))) {
    p->kernel = TI_ROWS_FEW;
    whole = p->f.us / low;
  }
  if (asked(TI_ROWS_BLOCK) && vec && kind != TI_EPI_LOGITS_ARGMAX && (kernel != TI_ROWS_AUTO || M > 32 || bits == 4 || (bits == 8 && M > 24 && N <= 24576)) &&
      ti::block_plan(bits, M, N, K, cus, fold, &p->b, only) &&
      (p->kernel == TI_ROWS_AUTO || p->b.us < (bits == 16 && fold ? 0.95f : 1.0f) * whole))
    p->kernel = TI_ROWS_BLOCK;
  return p->kernel != TI_ROWS_AUTO;
}

static bool rows_kernel_ok(int kernel) {   // (a shape is one kernel's)
  return kernel >= 0 && kernel % TI_ROWS_SHAPE <= TI_ROWS_BLOCK && (kernel < TI_ROWS_SHAPE || kernel % TI_ROWS_SHAPE != TI_ROWS_AUTO);
}

extern "C" int ti_gemm_rows_fold_partials_on(int kernel, int bits, int M, int N, int K, int64_t ws_bytes) {
  RowsPlan p;
  if (M > TI_FOLD_SS_ROWS || !rows_kernel_ok(kernel) || !rows_plan_of(kernel, bits, M, N, K, ws_bytes, true, TI_EPI_RESID_F32, true, &p))
    return 0;
  return p.n_cb();
}
extern "C" int ti_gemm_rows_fold_partials(int bits, int M, int N, int K, int64_t ws_bytes) {
  return ti_gemm_rows_fold_partials_on(TI_ROWS_AUTO, bits, M, N, K, ws_bytes);
}

extern "C" int ti_gemm_rows_kernel(int bits, int M, int N, int K, int64_t ws_bytes, int kind, int fold) {
  RowsPlan p;
  if (M < 1 || M > (fold ? TI_FOLD_SS_ROWS : TI_GEMM_MAX_ROWS)) return 0;
  return rows_plan_of(TI_ROWS_AUTO, bits, M, N, K, ws_bytes, fold != 0, kind, kind != TI_EPI_STORE_F16, &p) ? p.kernel : 0;
}

static int rows_impl(int kernel, const void* tiles, const uint16_t* scales, int bits, const void* x, int ldx, const float* h, const float* norm_w,
                     float eps, int M, int N, int K, const ti_epilogue* epi, ti_stream_t stream) {
  using namespace ti;
  if (!tiles || !x || !epi || !epi->out) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: null pointer");
  if (!rows_kernel_ok(kernel)) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: kernel %d", kernel);
  if (bits != 16 && !scales) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: scales required for bits %d", bits);
  if (M < 1 || M > TI_GEMM_MAX_ROWS || K <= 0 || (K & 127) || N <= 0 || (N & 15) || ldx < K || K > 0xffff || ldx > 0xffff)
    return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: M=%d N=%d K=%d ldx=%d", M, N, K, ldx);
  if (!rows_aligned(x, ldx)) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: x must be 16-byte aligned rows (ldx %d)", ldx);
  const int rc = check_epilogue(*epi, N, "ti_gemm_rows");
  if (rc != TI_OK) return rc;
  if (epi->out_packed) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: row-major outputs only");
  if (epi->ss_in && (M > TI_FOLD_SS_ROWS || epi->n_ss < 1 || epi->n_ss > 4096))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: a folded input needs M <= %d and 1 <= n_ss <= 4096", TI_FOLD_SS_ROWS);
  GemvArgs a{};
  a.tiles = (const u32x4*)tiles;
  a.scales = scales;
  a.x = x;
  a.eps = eps;
  a.x_kind = TI_X_F16;
  a.ldx = ldx;
  a.M = M;
  a.N = N;
  a.K = K;
  a.epi = *epi;
  a.vec = epilogue_vec(*epi);
  const bool fold_out = epi->kind == TI_EPI_RESID_F32 && epi->fold_x;
  if (fold_out &&
      (M > TI_FOLD_SS_ROWS || !epi->fold_w || !epi->fold_ss || epi->fold_packed || !a.vec))
    return ti_set_error(TI_ERR_ARG, "ti_gemm_rows: fold_x needs M <= %d, fold_w, fold_ss and 16-byte aligned rows", TI_FOLD_SS_ROWS);
  RowsPlan p;
  if (h) {
    if (!epi->ss_in || fold_out || !norm_w || (((uintptr_t)h | (uintptr_t)norm_w) & 15))
      return ti_set_error(TI_ERR_ARG, "ti_gemm_rows_folded: ss_in, no fold_x, and 16-byte aligned h and norm_w");
    a.norm_w = norm_w;
    a.epi.fold_w = h;
  }
  if (!rows_plan_of(kernel, bits, M, N, K, epi->splitk_ws ? epi->splitk_bytes : 0, epi->ss_in || fold_out, epi->kind, a.vec != 0, &p))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_gemm_rows: bits %d, M=%d N=%d K=%d", bits, M, N, K);
  const int rp = ti_gemm_prepare();   // no-op once this device is prepared
  if (rp != TI_OK) return rp;
  const hipStream_t s = (hipStream_t)stream;
  switch (p.kernel) {
    case TI_ROWS_FEW: a.stamp = ti_stamp_next(STAMP_TILE, few_workgroups(p.f)); return few_launch(bits, p.f, a, s);
    case TI_ROWS_MANY: a.stamp = ti_stamp_next(STAMP_TILE, wide_workgroups(p.w)); return wide_launch(bits, p.w, a, s);
    default: a.stamp = ti_stamp_next(STAMP_TILE, block_workgroups(p.b)); return block_launch(bits, p.b, a, s);
  }
}

extern "C" int ti_gemm_rows(const void* tiles, const uint16_t* scales, int bits, const void* x, int ldx, float eps, int M, int N,
                            int K, const ti_epilogue* epi, ti_stream_t stream) {
  return rows_impl(TI_ROWS_AUTO, tiles, scales, bits, x, ldx, nullptr, nullptr, eps, M, N, K, epi, stream);
}

extern "C" int ti_gemm_rows_folded(const void* tiles, const uint16_t* scales, int bits, uint16_t* x, int ldx, const float* h,
                                   const float* norm_w, float eps, int M, int N, int K, const ti_epilogue* epi, ti_stream_t stream) {
  if (!h) return ti_set_error(TI_ERR_ARG, "ti_gemm_rows_folded: null pointer");
  return rows_impl(TI_ROWS_AUTO, tiles, scales, bits, x, ldx, h, norm_w, eps, M, N, K, epi, stream);
}

extern "C" int ti_gemm_rows_on(int kernel, const void* tiles, const uint16_t* scales, int bits, uint16_t* x, int ldx, const float* h,
                               const float* norm_w, float eps, int M, int N, int K, const ti_epilogue* epi, ti_stream_t stream) {
  return rows_impl(kernel, tiles, scales, bits, x, ldx, h, norm_w, eps, M, N, K, epi, stream);
}
