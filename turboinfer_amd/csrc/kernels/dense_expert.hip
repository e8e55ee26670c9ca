// dense_expert.hip -- grouped products (experts) of many rows: tiles of up to 256 rows of one expert's list x 256 columns.
#include "dense.hpp"

namespace ti {

// Bound: experts of few rows, the weights (64 experts, gate/up 2816 x 2048: 738 MB in 127 us, 5.8 TB/s); of many, LDS beside the
// matrix cores (a k-tile of 256 x 256: 96 KiB of operand reads and 32 of copies in the 1024 cycles of its products; alone, products
// and reads take 0.49 us, products and copies 0.50, all three 0.66).  So, against dense_block_kernel's 256-row form:
//   * 256 workgroups stay and take one block after the other: the next one's first k-tiles are on their way through the last
//     products and the outputs of this one (a block of its own: ~ 10 us of launch, first loads and outputs per 45 us);
//   * rows are copied in 128-byte pieces, two k-tiles at a time (64-byte ones: 14 ns a KiB and CU, these 8), chunks XOR-swizzled by
//     row pair against bank conflicts;
//   * outputs leave as 16 bytes a lane (SiLU * up had 2).
// us, gate/up + down (2048 x 1408), 64 experts, 2048 rows spread evenly / as a trained router does: 207 + 115 / 225 + 132 -> 181 + 104 /
// 199 + 116; 900 rows 153 + 90 -> 147 + 85.  No gain: blocks of the last round cut into 128 or 64 columns (the others leave the
// memory to them), copies of rows and weights by different waves, four waves of 128 x 128 (fewer reads, but every one shows).
template <int EPI>
__global__ __launch_bounds__(512, 2) void dense_expert_kernel(const ti_dense_args a, int n_cols) {
  typedef El<bf16>::V V;
  constexpr int KT = El<bf16>::KT, WN = 4, FN = 4, NW = 8, P = 2, ND = 2 * P;   // waves 2 x 4; copies a wave makes of each operand a k-tile
  constexpr int kW = 16 * 1024, kA = 2 * kW, kW0 = 3 * kA;             // ring: 3 pairs of k-tiles of rows, 4 k-tiles of weights
  extern __shared__ __attribute__((aligned(1024))) char ring[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
  const int nk = a.K / KT, NT = (a.N + 15) >> 4, n_tiles = __builtin_amdgcn_readfirstlane(min(*a.n_tiles, a.max_tiles));
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;

  struct Item {   // one block of products: an expert, rows of the list, column tiles from n on
    int e, first, rows, n;
  };
  // the workgroup's j-th: an XCD's tiles with all their columns, dealt to its workgroups there and back
  const int xcd = (int)(blockIdx.x & 7), per = (int)(gridDim.x >> 3), at = (int)(blockIdx.x >> 3);
  auto item = [&](int j, Item& t) {
    const int i = j * per + (j & 1 ? per - 1 - at : at), k = i / n_cols, y = k * 8 + (k & 1 ? 7 - xcd : xcd);
    if (y >= n_tiles) return false;
    t.e = __builtin_amdgcn_readfirstlane(a.tiles[4 * y]);
    t.first = __builtin_amdgcn_readfirstlane(a.tiles[4 * y + 1]);
    t.rows = __builtin_amdgcn_readfirstlane(a.tiles[4 * y + 2]);
    t.n = (i - k * n_cols) * 16;
    return true;
  };
  // this wave's copies: column tiles wave and wave + 8 of a k-tile; 8-row groups 2 (wave + 8 i) + h of a pair's half h
  const char *w[P], *xa = (const char*)a.a;
  uint32_t row[2 * P], off[2 * P];   // byte offsets of the next item's rows, this one's
  auto rows_of = [&](const Item& t) {
#pragma unroll
    for (int i = 0; i < 2 * P; ++i) {
      const int m = 16 * ((i >> 1) * NW + wave) + 8 * (i & 1) + (lane >> 3);
      row[i] = (uint32_t)row_in(a, t.first + min(m, t.rows - 1)) * (uint32_t)a.lda * 2u + (uint32_t)((lane & 7) ^ (m >> 1 & 7)) * 16;
    }
  };
  auto aim_a = [&] {
    xa = (const char*)a.a;
#pragma unroll
    for (int i = 0; i < 2 * P; ++i) off[i] = row[i];
  };
  auto aim_w = [&](const Item& t) {
#pragma unroll
    for (int i = 0; i < P; ++i)
      w[i] = (const char*)a.w + ((size_t)t.e * a.w_batch * 2 + (size_t)min(t.n + i * NW + wave, NT - 1) * nk * 1024);
  };
  Item cur, nxt;
  if (!item(0, cur)) return;
  rows_of(cur);
  aim_a();
  aim_w(cur);
  bool last = !item(1, nxt);
  if (!last) rows_of(nxt);
  int f = 0;   // the k-tile to copy next
  uint32_t fill_a = lds0 + wave * 2048, fill_w = lds0 + kW0 + wave * 1024;
  auto dma_a = [&](int h, int i) __attribute__((always_inline)) {
    dma_1k_asm(xa, off[2 * i + h], fill_a + i * (NW * 2048) + h * 1024);
    if (h == 1 && i == P - 1) {
      xa += 128;
      fill_a = fill_a - lds0 >= 2 * kA ? fill_a - 2 * kA : fill_a + kA;
    }
  };
  auto dma_w = [&](int i) __attribute__((always_inline)) {
    dma_1k_asm(w[i], (uint32_t)lane * 16, fill_w + i * (NW * 1024));
    w[i] += 1024;
    if (i == P - 1) fill_w = fill_w - lds0 >= kW0 + 3 * kW ? fill_w - 3 * kW : fill_w + kW;
  };
  // k-tile f's weights, and of the rows what is due with them: an even one's pair's second half, behind an odd one the next
  // pair's first
#pragma unroll
  for (int i = 0; i < P; ++i) dma_a(0, i);
#pragma unroll
  for (; f < 4; ++f)
#pragma unroll
    for (int i = 0; i < P; ++i) {
      dma_w(i);
      dma_a(f & 1 ? 0 : 1, i);
    }

  const int at_a = (wm * 16 + (lane & 15)) * 128, at_w = kW0 + wn * FN * 1024 + lane * 16, sw = lane >> 1 & 7;
  int slot_a = 0, slot_w = 0;   // ring bytes of the pair / weights being multiplied
  int j = 0;
  auto block = [&]<int R>() __attribute__((always_inline)) {
    f32x4 acc[R][FN];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int c = 0; c < FN; ++c) acc[i][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    V af[R - 1], al[2], wf[2][FN];
    auto read_a = [&](V& d, int pair, int h, int i) { d = *(const V*)(ring + pair + at_a + (((h * 4 + (lane >> 4)) ^ sw) * 16) + i * 4096); };
    auto read_w = [&](int k, V (&d)[FN], int c) { d[c] = *(const V*)(ring + k + at_w + c * 1024); };
    wait_dma<3 * ND>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int c = 0; c < FN; ++c) read_w(slot_w, wf[0], c);
#pragma unroll
    for (int i = 0; i < R - 1; ++i) read_a(af[i], slot_a, 0, i);
    read_a(al[0], slot_a, 0, R - 1);
    // k-tile s, s & 1 == B: its operands were read a stage ago; each register takes the next k-tile's as soon as its products
    // are issued (the last row tile has two, so that no read is issued late).  The reads are waited for ahead of the barrier:
    // the k-tile's own ring slot is free behind it.
    auto stage = [&]<int B>() __attribute__((always_inline)) {
      const int nw = slot_w == 3 * kW ? 0 : slot_w + kW, na = B == 0 ? slot_a : slot_a == 2 * kA ? 0 : slot_a + kA;
      if (f == nk && !last) {
        aim_w(nxt);
        f = 0;
      }
      if (B == 1 && f == nk - 1) {   // (no next item: the last pair again, which nothing reads)
        if (last) xa -= 128;
        else aim_a();
      }
      const bool more = f < nk;
      if (more) wait_dma<2 * ND>();
      else wait_dma<0>();
      lds_sync();
#pragma unroll
      for (int i = 0; i < R; ++i) {
#pragma unroll
        for (int c = 0; c < FN; ++c) acc[i][c] = mma(wf[B][c], i < R - 1 ? af[i < R - 1 ? i : 0] : al[B], acc[i][c]);
        __builtin_amdgcn_sched_barrier(0);
        if (i < R - 1) {
          read_a(af[i], na, B ^ 1, i);
          if (i == 0) read_a(al[B ^ 1], na, B ^ 1, R - 1);
#pragma unroll
          for (int c = i * FN / (R - 1); c < (i + 1) * FN / (R - 1); ++c) read_w(nw, wf[B ^ 1], c);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
#pragma unroll
          for (int d = 0; d < P; ++d)
            if (d * R / P == i) {
              dma_w(d);
              dma_a(B ? 0 : 1, d);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      ++f;
      slot_w = nw;
      slot_a = na;
    };
    for (int s = 0; s < nk; s += 2) {
      stage.template operator()<0>();
      stage.template operator()<1>();
    }
    // the rows of the item after the next one, beside the outputs
    const Item done = cur;
    const bool none = last;
    if (!none) {
      cur = nxt;
      last = !item(++j + 1, nxt);
      if (!last) rows_of(nxt);
    }
    const int c0 = done.n + wn * FN;
    const bool whole = (c0 + 4) * 16 <= a.N && a.ldo % 8 == 0 && ((uintptr_t)a.out & 15) == 0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int mt = (i * 2 + wm) * 16, m = mt + (lane & 15);
      if (mt >= done.rows) break;
      const int mo = m < done.rows ? row_out(a, done.first + m) : 0;
      if (whole) {
        if constexpr (EPI == TI_DE_SWIGLU) store_swiglu64(a, m < done.rows, mo, c0, acc[i], lane);
        else store64(a, m < done.rows, mo, c0, acc[i], lane);
        continue;
      }
      const DenseSpan sp = {done.rows, done.first, 0, nullptr};
#pragma unroll
      for (int c = 0; c < FN; ++c)
        if (c0 + c < NT) dense_out<bf16, EPI>(a, sp, m, mo, mt, c0 + c, acc[i][c], lane);
    }
    return none;
  };
  for (;;) {
    const int live = (cur.rows + 31) / 32;   // row tiles a wave
    bool none;
    if (live > 7) none = block.template operator()<8>();
    else if (live > 6) none = block.template operator()<7>();
    else if (live > 5) none = block.template operator()<6>();
    else if (live > 4) none = block.template operator()<5>();
    else if (live > 2) none = block.template operator()<4>();
    else none = block.template operator()<2>();
    if (none) return;
  }
}

// 16-bit tiles of 256 rows whose K is long enough for the ring, rows in reach of 32-bit offsets.
bool expert_takes(const ti_dense_args& a) {
  const int64_t rows = std::max<int64_t>(a.M, (int64_t)a.max_tiles * a.tile_rows);
  return a.tile_rows == 256 && a.K >= 6 * El<bf16>::KT && rows * a.lda * 2 <= 0x7fffffff;
}
template <int EPI>
int launch_expert(const ti_dense_args& a, hipStream_t s) {
  constexpr int kLds = 160 * 1024;
  auto* fn = dense_expert_kernel<EPI>;
  TI_HIP_CHECK(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLds),
               "hipFuncSetAttribute(dense_expert_kernel)");
  hipLaunchKernelGGL(fn, dim3(256), dim3(512), kLds, s, a, (a.N + 255) / 256);
  TI_LAUNCH_CHECK("dense_expert_kernel");
  return TI_OK;
}
template int launch_expert<TI_DE_T>(const ti_dense_args&, hipStream_t);
template int launch_expert<TI_DE_SWIGLU>(const ti_dense_args&, hipStream_t);

}  // namespace ti
