// dense.hip -- matrix products of the layer-stack models (ti_stack.h ti_dense): fragment-ordered
// weights x row-major activations on MFMA, bf16 or fp32, with the consumer's first step fused into
// the epilogue (SiLU * up, rotary pairs, head gates, logits + argmax, key / value fragments).
//
// Four kernels share the epilogue (dense_expert.hip has a fifth, for experts of many rows):
//   * dense_half_kernel (M <= 16, N <= 2048, plain outputs): weight streaming by 8 columns a workgroup.
//   * dense_skinny_kernel (M <= 64, or few tiles of outputs): HBM-bound weight streaming.  One workgroup per 16 output columns,
//     its waves split k; each weight fragment is one contiguous KiB read once and multiplied with up
//     to 4 row tiles; the waves' partial sums meet in LDS.
//   * dense_block_kernel (more rows: tiles of 32 x 64 up to 256 x 256): both operands copied to an LDS ring by DMA,
//     4 to 12 stages ahead, waves in a WM x WN grid, for the smaller tiles one such grid per half of k.
//   * dense_tile_kernel (its 64-row tiles for grouped products and the epilogues of short or narrow products): 4 waves
//     side by side over a BM x BN tile, activations staged through double-buffered LDS in fragment order, each wave's
//     weight fragments straight from L2 into registers; both 2 or 4 k-stages (128 bytes each) ahead of their use.
// All take independent batches (per-head products) or grouped tiles (experts: a tile is up to
// tile_rows entries of one expert's list, rows gathered and scattered through the list).
#include "dense.hpp"

namespace ti {

template <class T, int MT, int W, int EPI>
__global__ __launch_bounds__(64 * W) void dense_skinny_kernel(const ti_dense_args a) {
  typedef typename El<T>::V V;
  constexpr int KT = El<T>::KT, VEC = El<T>::VEC, U = 8;
  __shared__ f32x4 red[W][MT][64];
  DenseSpan sp;
  if (!dense_span(a, blockIdx.y, sp, sizeof(T))) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockIdx.x, nk = a.K / KT, z0 = blockIdx.z * MT * 16;
  const V* wp = (const V*)sp.w + (size_t)nt * nk * 64 + lane;
  const V* ap[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int p = sp.first + min(z0 + mt * 16 + (lane & 15), sp.rows - 1);
    ap[mt] = (const V*)((const T*)a.a + (size_t)sp.batch * a.a_batch + (size_t)row_in(a, p) * a.lda) + (lane >> 4);
  }
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // n k-tiles of this wave: their weight fragments in flight together (kept to ~64 VGPRs: workgroups
  // per CU hide more latency than a deeper wave)
  auto batch = [&]<int N>(int kt) {
    V wf[N];
#pragma unroll
    for (int u = 0; u < N; ++u) wf[u] = wp[(size_t)(kt + u * W) * 64];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      V af[N];
#pragma unroll
      for (int u = 0; u < N; ++u) af[u] = ap[mt][(kt + u * W) * (KT / VEC)];
#pragma unroll
      for (int u = 0; u < N; ++u) acc[mt] = mma(wf[u], af[u], acc[mt]);
    }
  };
  int kt = wave;
  for (; kt + (U - 1) * W < nk; kt += U * W) batch.template operator()<U>(kt);
  if (kt + 3 * W < nk) {
    batch.template operator()<4>(kt);
    kt += 4 * W;
  }
  if (kt + W < nk) {
    batch.template operator()<2>(kt);
    kt += 2 * W;
  }
  if (kt < nk) batch.template operator()<1>(kt);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) red[wave][mt][lane] = acc[mt];
  __syncthreads();
  for (int mt = wave; mt < MT; mt += W) {
    f32x4 v = red[0][mt][lane];
#pragma unroll
    for (int w = 1; w < W; ++w) v += red[w][mt][lane];
    const int m = z0 + mt * 16 + (lane & 15), n0 = nt * 16 + 4 * (lane >> 4);
    if constexpr (EPI == TI_DE_LOGITS)
      dense_argmax(a, m, sp.rows, n0, v, lane, nt);
    else
      dense_store<T, EPI>(a, sp.batch, m, m < sp.rows ? row_out(a, sp.first + m) : 0, sp.rows, n0, v);
  }
  if (EPI == TI_DE_LOGITS && a.step_ctr && nt == 0 && blockIdx.z == 0 && tid == 0) *a.step_ctr += a.advance;
}

// Up to 16 rows of a product of at most 2048 columns: the skinny kernel's 16-column workgroups leave half of the CUs idle, so
// these take 8.  A product's 16 x 16 tile holds two k-tiles: its weight rows 0 .. 7 and rows of a 0 .. 7 are the first's, 8 ..
// 15 the second's, and the diagonal blocks are summed at the end (the other two mean nothing); rows 8 .. 15 of a are a
// second product.  2048 columns, K 8192 (33.5 MB), 8 rows: 13.6 -> 10.4 us; a step of Nogitar 2k (15 of them) of 8 streams 477 ->
// 450 us, of 16 550 -> 529, fp32 of one 710 -> 609.  Up to 2048 columns these workgroups fit the CUs at once; beyond, a
// second round starts.  us at 1 / 8 / 16 rows, skinny -> this, N x K: bf16 256 x 2048 4.1 / 4.7 / 5.2 -> 3.4 / 3.8 / 4.6, 2048 x
// 1024 3.6 / 3.9 / 4.1 -> 3.2 / 3.4 / 3.9, 2048 x 8192 11.2 / 13.1 / 16.5 -> 8.7 / 9.8 / 13.6, 2176 x 8192 11.2 / 13.2 / 16.2 -> 11.0 /
// 14.7 / 20.6, 4096 x 2048 5.4 / 5.7 / 6.3 -> 5.2 / 5.6 / 7.0; fp32 2048 x 8192 29.2 / 29.7 / 31.1 -> 18.0 / 18.0 / 22.8, 2176 x 8192 29.6 /
// 29.9 / 31.4 -> 20.5 / 27.5 / 39.0.
template <class T, int MT, int W, int EPI>
__global__ __launch_bounds__(64 * W) void dense_half_kernel(const ti_dense_args a) {
  typedef typename El<T>::V V;
  constexpr int KT = El<T>::KT, VEC = El<T>::VEC, U = 8;
  __shared__ f32x4 red[W][MT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockIdx.x >> 1, half = blockIdx.x & 1;
  const int nk = a.K / KT, np = nk >> 1, second = lane >> 3 & 1;   // (K is padded to two k-tiles)
  const V* wp = (const V*)a.w + ((size_t)nt * nk + second) * 64 + (lane >> 4) * 16 + half * 8 + (lane & 7);
  const V* ap[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    ap[mt] = (const V*)((const T*)a.a + (size_t)min(mt * 8 + (lane & 7), a.M - 1) * a.lda + second * KT) + (lane >> 4);
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto batch = [&]<int N>(int p) {   // N k-tile pairs of this wave, their weights in flight together
    V wf[N];
#pragma unroll
    for (int u = 0; u < N; ++u) wf[u] = wp[(size_t)(p + u * W) * 128];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      V af[N];
#pragma unroll
      for (int u = 0; u < N; ++u) af[u] = ap[mt][(p + u * W) * (2 * KT / VEC)];
#pragma unroll
      for (int u = 0; u < N; ++u) acc[mt] = mma(wf[u], af[u], acc[mt]);
    }
  };
  int p = wave;
  for (; p + (U - 1) * W < np; p += U * W) batch.template operator()<U>(p);
  if (p + 3 * W < np) {
    batch.template operator()<4>(p);
    p += 4 * W;
  }
  if (p + W < np) {
    batch.template operator()<2>(p);
    p += 2 * W;
  }
  if (p < np) batch.template operator()<1>(p);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) red[wave][mt][lane] = acc[mt];
  __syncthreads();
  // lane 16 g + j, g < 2, j < 8: columns 4 g .. of row j; the second k-tile's 40 lanes on
  if (wave >= MT || lane >= 32 || (lane & 15) >= 8) return;
  f32x4 v = red[0][wave][lane] + red[0][wave][lane + 40];
#pragma unroll
  for (int w = 1; w < W; ++w) v += red[w][wave][lane] + red[w][wave][lane + 40];
  const int m = wave * 8 + (lane & 7);
  dense_store<T, EPI>(a, 0, m, m, a.M, nt * 16 + half * 8 + 4 * (lane >> 4), v);
}

// Consecutive workgroups go to the 8 XCDs in turn.  An XCD gets a contiguous run of the work list, ordered so that
// neighbours share weight columns (its L2 holds them once): row tiles fastest, for grouped products 4 tiles (mostly one
// expert's) fastest, then the columns.  Grouped tiles of 128 rows and more are dealt to the XCDs, there and back, each with
// all its columns (its rows are read into one L2): lists come with the large tiles first, so the XCDs' loads match and
// the small tiles fill the last round (2048 rows of trained-like routing, 64 experts, 75 tiles, us: a run per XCD by expert 275 / -, 4
// tiles by expert in turn 249 / 147 (gate/up 2816 x 2048 / down 2048 x 1408), this 231 / 129; 863 MB of weights, 5.4 TB/s at
// best, are 160 of the 231).
struct TileAt {
  int id, m, n, y;   // work item, row tile, column tile, batch / grouped tile
};
__host__ __device__ inline bool tiles_dealt(const ti_dense_args& a) { return a.tile_rows >= 128; }
inline int tile_grid(const ti_dense_args& a, int m_tiles, int n_tiles) {
  if (tiles_dealt(a)) return (a.max_tiles + 7) / 8 * 8 * n_tiles;
  return ((a.tile_rows ? (a.max_tiles + 3) / 4 * 4 : m_tiles) * n_tiles + 7) / 8 * 8;
}
__device__ __forceinline__ bool tile_at(const ti_dense_args& a, int m_tiles, int n_tiles, TileAt& t) {
  if (tiles_dealt(a)) {
    const int x = (int)(blockIdx.x & 7), i = (int)(blockIdx.x >> 3) / n_tiles;
    t = {(int)blockIdx.x, 0, (int)(blockIdx.x >> 3) - i * n_tiles, i * 8 + (i & 1 ? 7 - x : x)};
    return t.y < *a.n_tiles;
  }
  const int list = a.tile_rows ? (*a.n_tiles + 3) / 4 * 4 * n_tiles : m_tiles * n_tiles, per = (list + 7) >> 3;
  t.id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t.id >= list) return false;
  if (a.tile_rows) {
    const int b = t.id / (4 * n_tiles), r = t.id - b * 4 * n_tiles;
    t.m = 0;
    t.n = r >> 2;
    t.y = b * 4 + (r & 3);
  } else {
    t.m = t.id % m_tiles;
    t.n = t.id / m_tiles;
    t.y = blockIdx.y;
  }
  return true;
}

template <class T, int BM, int BN, int D, int EPI>
__global__ __launch_bounds__(256, BM * BN > 16384 ? 1 : 2) void dense_tile_kernel(const ti_dense_args a, int m_tiles, int n_tiles) {
  typedef typename El<T>::V V;
  constexpr int KT = El<T>::KT, VEC = El<T>::VEC, FM = BM / 16, FN = BN / 64, NA = BM / 32;
  constexpr bool VF = EPI == TI_DE_VFRAG;
  __shared__ V as[2][FM * 2][64];
  TileAt at;
  DenseSpan sp;
  if (!tile_at(a, m_tiles, n_tiles, at) || !dense_span(a, at.y, sp, sizeof(T))) return;
  const int m_base = at.m * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nk = a.K / KT, nst = nk >> 1, NT = (a.N + 15) >> 4;
  const V* ap[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int f = i * 4 + wave;   // fragment (row tile f >> 1, k-tile f & 1) of the stage
    const int p = sp.first + min(m_base + (f >> 1) * 16 + (lane & 15), sp.rows - 1);
    ap[i] = (const V*)((const T*)a.a + (size_t)sp.batch * a.a_batch + (size_t)row_in(a, p) * a.lda) + (f & 1) * (KT / VEC) +
            (lane >> 4);
  }
  const V* wp[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
    wp[j] = (const V*)sp.w + (size_t)min(at.n * (BN / 16) + wave * FN + j, NT - 1) * nk * 64 + lane;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // TI_DE_LRU: what its outputs take beside the products, on its way through them.  (Read behind them it was waited for tile by tile, as
  // the outputs stored in between might overlap it; with 16-byte outputs, 1500 rows, 10 blocks of 256 channels: 35.5 -> 28.1 us.)
  constexpr bool LRU = EPI == TI_DE_LRU;
  typedef T T2 __attribute__((ext_vector_type(2)));
  T2 lu[LRU ? FM : 1][LRU ? FN : 1];
  float lb[LRU ? FN : 1][4], lr[LRU ? FN : 1][2];
  if constexpr (LRU) {
    const int per = a.N >> 1;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n0 = (at.n * (BN / 16) + wave * FN + j) * 16 + 4 * (lane >> 4), c = min(n0 >> 1, per - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) lb[j][i] = a.add[(size_t)sp.batch * a.N + min(n0 + i, a.N - 1)];
#pragma unroll
      for (int i = 0; i < 2; ++i) lr[j][i] = a.lru_rate[sp.batch * per + min(c + i, per - 1)];
#pragma unroll
      for (int i = 0; i < FM; ++i)   // (an odd last channel's pair ends in the row's padding: K is even)
        lu[i][j] = *(const T2*)((const T*)a.a + (size_t)min(m_base + i * 16 + (lane & 15), sp.rows - 1) * a.lda + (size_t)sp.batch * a.a_batch + (c & ~1));
    }
  }
  // rings of D stages in registers: weights of stage s in set s % D, activations likewise until they
  // move to LDS one stage before their use
  V ar[D][NA], w[D][FN][2];
  auto load_a = [&](V (&d)[NA], int s) {
#pragma unroll
    for (int i = 0; i < NA; ++i) d[i] = ap[i][min(s, nst - 1) * 2 * (KT / VEC)];
  };
  auto load_w = [&](V (&d)[FN][2], int s) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      d[j][0] = wp[j][(size_t)min(s, nst - 1) * 128];
      d[j][1] = wp[j][(size_t)min(s, nst - 1) * 128 + 64];
    }
  };
  auto store_a = [&](int buf, const V (&d)[NA]) {
#pragma unroll
    for (int i = 0; i < NA; ++i) as[buf][i * 4 + wave][lane] = d[i];
  };
  // s % 4 == B.  A stage's operand reads all go out first (left alone, the scheduler keeps two in
  // flight and waits for LDS between products), the hand-over of the next stage's activations next.
  auto stage = [&]<int B>(int s) {
    V af[2][FM];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < FM; ++i) af[kk][i] = as[B & 1][i * 2 + kk][lane];
    __builtin_amdgcn_sched_barrier(0);
    store_a((B + 1) & 1, ar[(B + 1) % D]);
    load_a(ar[(B + 1) % D], s + 1 + D);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = VF ? mma(af[kk][i], w[B % D][j][kk], acc[i][j]) : mma(w[B % D][j][kk], af[kk][i], acc[i][j]);
    load_w(w[B % D], s + D);
    lds_sync();
  };
  load_a(ar[0], 0);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load_w(w[d], d);
    if (d == 0) {
      store_a(0, ar[0]);
      load_a(ar[0], D);
    } else {
      load_a(ar[d], d);
    }
  }
  lds_sync();
  for (int s = 0; s < nst; s += 4) {
    stage.template operator()<0>(s);
    if (s + 1 < nst) stage.template operator()<1>(s + 1);
    if (s + 2 < nst) stage.template operator()<2>(s + 2);
    if (s + 3 < nst) stage.template operator()<3>(s + 3);
  }
  if constexpr (LRU) {
    const int per = a.N >> 1, channels = per * a.batch;
    const bool quads = per % 2 == 0 && ((uintptr_t)a.out & 15) == 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m_base + i * 16 + (lane & 15);
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int c = ((at.n * (BN / 16) + wave * FN + j) * 16 + 4 * (lane >> 4)) >> 1;
        const float2 p = lru_coef(acc[i][j][0] + lb[j][0], acc[i][j][1] + lb[j][1], lr[j][0], (float)lu[i][j][0]);
        const float2 q = lru_coef(acc[i][j][2] + lb[j][2], acc[i][j][3] + lb[j][3], lr[j][1], (float)lu[i][j][1]);
        if (m >= sp.rows || c >= per) continue;
        float* o = (float*)a.out + ((size_t)m * channels + sp.batch * per + c) * 2;
        if (quads) {
          *(f32x4*)o = (f32x4){p.x, p.y, q.x, q.y};
        } else {
          *(float2*)o = p;
          if (c + 1 < per) *(float2*)(o + 2) = q;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int mt = m_base + i * 16;
    const int m = mt + (lane & 15);
    const int mo = m < sp.rows ? row_out(a, sp.first + m) : 0;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int nt = at.n * (BN / 16) + wave * FN + j;
      if (nt < NT) dense_out<T, EPI>(a, sp, m, mo, mt, nt, acc[i][j], lane);
    }
  }
  if (EPI == TI_DE_LOGITS && a.step_ctr && at.id == 0 && tid == 0) *a.step_ctr += a.advance;
}

template <int KG, int WM, int WN, int FM, int FN, int NS>
struct BlockCfg {
  static constexpr int kWaves = KG * WM * WN, BM = 16 * FM * WM, BN = 16 * FN * WN;
  static constexpr int kLds = NS * KG * (FM * WM + FN * WN) * 1024;
  static constexpr bool kBig = FM * FN > 16;
  static_assert(kLds <= 160 * 1024 && NS >= 4 && KG <= 2 && (KG == 1 || kLds >= WM * WN * FM * FN * 1024));
};

// Bound: with every CU at it the products (~ 1340 TFLOP/s is what the chip's power leaves a bf16 product of random data);
// a block alone on its CU, LDS traffic and the hand-over of a stage.  So waves take tiles of up to 128 x 64 (LDS reads
// 12 KiB per 32 products), fragments are read a stage ahead into the registers just used, and blocks of at most 128 x 128
// run two groups of waves (KG 2) that take alternate k-tiles and meet in LDS at the end: a barrier and its skew per two
// k-tiles, fewer LDS reads per product than tiles of half the size.  Deeper rings than NS give nothing.  A row of a stage
// is 64 bytes: four lanes fetch it (chunks XOR-swizzled by row against LDS bank conflicts), 2 - 10 % over a lane per row; with two
// k-tiles a stage 128 bytes, eight lanes (us a launch inside a prompt: 1500 rows, K 2048 .. 8192, 2048 columns 45.6 -> 39.8, 2048 rows
// 31.1 -> 29.1; means over 245 products of 512 .. 4096 columns, 100 .. 2048 rows, K 512 .. 8192, weights in the caches and not: bf16 32 x 64 0 - 4 %
// faster, 64 x 64 3 - 9, 64 x 128 3 - 5, 128 x 128 1 - 5; fp32 0 - 3).
// Measured, us, bf16, dense_tile_kernel and blocks without KG -> this: 2048 x 2048 at 100 rows 10.8 -> 8.6, 333 11.4 ->
// 9.2, 1000 18.4 -> 15.0; 2048 x 8192 (N x K) at 333 46.5 -> 29, 1500 85.5 -> 64; 5120 x 2048 at 700 29.8 -> 22; fp32
// 2048 x 2048 at 100 rows 45 -> 24.
//
// One tile: `step` rows at most (ungrouped calls: rows a row tile covers, tile_plan), BN columns.  A wave multiplies R row
// tiles, R the fewest of FM, 3/4 and 1/2 of it that hold the tile's rows: a ragged last tile, a small expert's and calls that
// spread over the CUs better by 3/4-high tiles leave the rest out, copies included.
template <class T, int KG, int WM, int WN, int FM, int FN, int NS, int EPI>
__global__ __launch_bounds__(64 * KG * WM * WN, 2) void dense_block_kernel(const ti_dense_args a, int m_tiles, int n_tiles, int step_rows) {
  typedef typename El<T>::V V;
  typedef BlockCfg<KG, WM, WN, FM, FN, NS> C;
  constexpr int KT = El<T>::KT, VEC = El<T>::VEC, NW = C::kWaves;
  constexpr bool VF = EPI == TI_DE_VFRAG;
  extern __shared__ __attribute__((aligned(1024))) char ring[];
  TileAt at;
  DenseSpan sp;
  if (!tile_at(a, m_tiles, n_tiles, at) || !dense_span(a, at.y, sp, sizeof(T))) return;
  const int m_base = at.m * step_rows, m_end = min(sp.rows, m_base + step_rows);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
  const int nk = a.K / KT, NT = (a.N + 15) >> 4, ns = nk / KG;   // (K is padded to two k-tiles)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  const int live = EPI == TI_DE_KFRAG || EPI == TI_DE_VFRAG ? FM : ((m_end - m_base + 15) / 16 + WM - 1) / WM;

  auto tile = [&]<int R>() __attribute__((always_inline)) {
    constexpr int NA = KG * R * WM, NF = NA + KG * FN * WN, ND = (NF + NW - 1) / NW, REST = NF % NW;
    static_assert(NS * ND < 64, "vmcnt");
    const bool whole = REST == 0 || wave < REST;   // this wave copies ND fragments a stage, else one less
    // this wave's KiB of a stage (KG k-tiles of the block): rows, then weight tiles by k-tile
    const V* src[ND];
    uint32_t dst[ND], step[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int f = min(i * NW + wave, NF - 1);
      dst[i] = lds0 + (uint32_t)f * 1024;
      if (f < NA) {   // 16 rows x 64 bytes, or with two k-tiles a stage 8 x 128
        const int m = KG == 2 ? f * 8 + (lane >> 3) : f * 16 + (lane >> 2);
        const int p = sp.first + min(m_base + m, sp.rows - 1);
        src[i] = (const V*)((const T*)a.a + (size_t)sp.batch * a.a_batch + (size_t)row_in(a, p) * a.lda) +
                 (KG == 2 ? (lane & 7) ^ (m >> 1 & 7) : (lane & 3) ^ (lane >> 3 & 3));
        step[i] = KG * KT / VEC;
      } else {
        const int g = (f - NA) / (FN * WN), ct = (f - NA) % (FN * WN);
        src[i] = (const V*)sp.w + ((size_t)min(at.n * (FN * WN) + ct, NT - 1) * nk + g) * 64 + lane;
        step[i] = KG * 64;
      }
    }
    uint32_t fill = 0;   // ring byte the next stage is copied to
    auto dma1 = [&](int i) __attribute__((always_inline)) {
      if (i == ND - 1 && !whole) return;
      dma_1k_asm(src[i], dst[i] + fill);
      src[i] += step[i];
    };
    auto filled = [&] { fill = fill == (NS - 1) * NF * 1024 ? 0 : fill + NF * 1024; };
    auto wait = [&]<int STAGES>() __attribute__((always_inline)) {   // all but this wave's copies of the newest STAGES stages
      if (whole) wait_dma<STAGES * ND>();
      else wait_dma<STAGES * (ND - 1)>();
    };
    f32x4 acc[R][FN];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    V af[R], w[2][FN];
    const V* const first = (const V*)ring;
    const V* cur = first;   // the stage being multiplied
    // wave (kg, wm, wn): k-tile kg of a stage, row tiles wm, wm + WM, .., weight tiles wn * FN ..
    const int at_a = KG == 2 ? wm * 128 + (lane & 15) * 8 + ((kg * 4 + (lane >> 4)) ^ (lane >> 1 & 7))
                             : wm * 64 + (lane & 15) * 4 + (lane >> 4 ^ (lane >> 1 & 3));
    const int at_w = (NA + kg * FN * WN + wn * FN) * 64 + lane;
    auto read_a = [&](const V* st, int i) { af[i] = st[i * KG * WM * 64 + at_a]; };
    auto read_w = [&](const V* st, V (&d)[FN], int j) { d[j] = st[j * 64 + at_w]; };
    // One stage.  Its weights and all but its last R / 4 row tiles were read a stage ago; each register takes the next
    // stage's fragment as soon as its products are issued.  The last ones are read here, so that reads of a ring slot end
    // with its stage and the slot is free once every wave has passed the next barrier.  MORE: another stage is copied
    // (2: found out here).
    auto stage = [&]<int B, int MORE>(int s) __attribute__((always_inline)) {
      constexpr int EARLY = R - R / 4;
      const bool more = MORE == 2 ? s + NS - 1 < ns : MORE;
      if (MORE == 2 && s + NS - 2 >= ns) wait_dma<0>();   // stage s + 1 is here (the last ones: everything)
      else wait.template operator()<NS - 3>();
      __builtin_amdgcn_s_barrier();
      const V* nxt = cur == first + (NS - 1) * NF * 64 ? first : cur + NF * 64;
#pragma unroll
      for (int i = EARLY; i < R; ++i) read_a(cur, i);
#pragma unroll
      for (int i = 0; i < R; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = VF ? mma(af[i], w[B][j], acc[i][j]) : mma(w[B][j], af[i], acc[i][j]);
        if (i < EARLY) read_a(nxt, i);
#pragma unroll
        for (int j = i * FN / R; j < (i + 1) * FN / R; ++j) read_w(nxt, w[B ^ 1], j);
        __builtin_amdgcn_sched_barrier(0);
        if (more) {   // the copies spread over the products: a bunch of them blocks the wave's issue
#pragma unroll
          for (int d = 0; d < ND; ++d)
            if (min(1 + d, R - 1) == i) dma1(d);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) filled();
      cur = nxt;
    };
#pragma unroll
    for (int d = 0; d < NS - 1; ++d)
      if (d < ns) {
#pragma unroll
        for (int i = 0; i < ND; ++i) dma1(i);
        filled();
      }
    if (NS - 1 > ns) wait_dma<0>();
    else wait.template operator()<NS - 2>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int j = 0; j < FN; ++j) read_w(cur, w[0], j);
#pragma unroll
    for (int i = 0; i < R - R / 4; ++i) read_a(cur, i);
    int s = 0;
    if constexpr (!C::kBig)   // (a second copy of the largest tiles' loop spills)
      for (; s + NS < ns; s += 2) {
        stage.template operator()<0, 1>(s);
        stage.template operator()<1, 1>(s + 1);
      }
    for (; s < ns; s += 2) {
      stage.template operator()<0, 2>(s);
      if (KG == 1 || s + 1 < ns) stage.template operator()<1, 2>(s + 1);
    }
    constexpr int H = KG == 1 ? R : (R + 1) / 2;
    if constexpr (KG == 2) {   // the halves of k meet: a wave of the first finishes row tiles < H, its partner the others
      __builtin_amdgcn_s_barrier();   // (every wave's reads of the ring are done)
      f32x4* x = (f32x4*)ring + (size_t)(wm * WN + wn) * R * FN * 64 + lane;
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          if ((i >= H) == (kg == 0)) x[(i * FN + j) * 64] = acc[i][j];
      lds_sync();
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          if ((i >= H) != (kg == 0)) acc[i][j] += x[(i * FN + j) * 64];
    }
    const int c0 = at.n * (FN * WN) + wn * FN;
    auto rows = [&](auto&& put) __attribute__((always_inline)) {   // put(i, m, mo, mt): row tiles that this wave finishes
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int mt = m_base + (i * WM + wm) * 16;
        if (i >= live) break;
        if (KG == 2 && (i >= H) == (kg == 0)) continue;
        const int m = mt + (lane & 15);
        put(i, m, m < m_end ? row_out(a, sp.first + m) : 0, mt);
      }
    };
    if constexpr (FN == 4)
      if (wave64<T, EPI>(a, c0)) {
        Wave64<EPI> w64(a, c0, lane);
        rows([&](int i, int m, int mo, int) __attribute__((always_inline)) { w64.out(a, m < m_end, m, mo, c0, acc[i], lane); });
        return;
      }
    rows([&](int i, int m, int mo, int mt) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
        if (c0 + j < NT) dense_out<T, EPI>(a, sp, m, mo, mt, c0 + j, acc[i][j], lane);
    });
  };
  if constexpr (FM == 8) {
    if (live > 7) tile.template operator()<8>();
    else if (live > 6) tile.template operator()<7>();
    else if (live > 5) tile.template operator()<6>();
    else if (live > 4) tile.template operator()<5>();
    else if (live > 2) tile.template operator()<4>();
    else tile.template operator()<2>();
  } else {
    constexpr int R2 = FM / 2, R1 = FM * 3 / 4;
    if (live > R1) tile.template operator()<FM>();
    else if (R1 != R2 && live > R2) tile.template operator()<R1>();
    else tile.template operator()<R2>();
  }
}

template <class T, int MT, int EPI>
int launch_skinny(const ti_dense_args& a, hipStream_t s) {
  const int NT = (a.N + 15) / 16, y = a.tile_rows ? a.max_tiles : a.batch, nk = a.K / El<T>::KT;
  const int z = a.tile_rows ? 1 : (a.M + 16 * MT - 1) / (16 * MT);
  if (nk >= 32)
    hipLaunchKernelGGL((dense_skinny_kernel<T, MT, 8, EPI>), dim3(NT, y, z), dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((dense_skinny_kernel<T, MT, 4, EPI>), dim3(NT, y, z), dim3(256), 0, s, a);
  TI_LAUNCH_CHECK("dense_skinny_kernel");
  return TI_OK;
}

template <class T, int BM, int BN, int D, int EPI>
int launch_tile(const ti_dense_args& a, hipStream_t s) {
  const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN;
  hipLaunchKernelGGL((dense_tile_kernel<T, BM, BN, D, EPI>), dim3(tile_grid(a, mt, nt), a.tile_rows ? 1 : a.batch), dim3(256), 0,
                     s, a, mt, nt);
  TI_LAUNCH_CHECK("dense_tile_kernel");
  return TI_OK;
}

template <class T, int KG, int WM, int WN, int FM, int FN, int NS, int EPI>
int launch_block(const ti_dense_args& a, int step_rows, hipStream_t s) {
  typedef BlockCfg<KG, WM, WN, FM, FN, NS> C;
  const int rows = EPI == TI_DE_KFRAG || EPI == TI_DE_VFRAG ? (a.M + 127) / 128 * 128 : a.M;   // (fragments: whole blocks of 128 keys)
  const int mt = (rows + step_rows - 1) / step_rows, nt = (a.N + C::BN - 1) / C::BN;
  auto* fn = dense_block_kernel<T, KG, WM, WN, FM, FN, NS, EPI>;
  TI_HIP_CHECK(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds),
               "hipFuncSetAttribute(dense_block_kernel)");
  hipLaunchKernelGGL(fn, dim3(tile_grid(a, mt, nt), a.tile_rows ? 1 : a.batch), dim3(64 * C::kWaves), C::kLds, s, a, mt, nt, step_rows);
  TI_LAUNCH_CHECK("dense_block_kernel");
  return TI_OK;
}

template <class T, int EPI>
int launch_half(const ti_dense_args& a, hipStream_t s) {
  const dim3 grid((a.N + 15) / 16 * 2);
  const bool long_k = a.K / El<T>::KT >= 32;
  if (a.M <= 8 && long_k) hipLaunchKernelGGL((dense_half_kernel<T, 1, 8, EPI>), grid, dim3(512), 0, s, a);
  else if (a.M <= 8) hipLaunchKernelGGL((dense_half_kernel<T, 1, 4, EPI>), grid, dim3(256), 0, s, a);
  else if (long_k) hipLaunchKernelGGL((dense_half_kernel<T, 2, 8, EPI>), grid, dim3(512), 0, s, a);
  else hipLaunchKernelGGL((dense_half_kernel<T, 2, 4, EPI>), grid, dim3(256), 0, s, a);
  TI_LAUNCH_CHECK("dense_half_kernel");
  return TI_OK;
}

// up to 64 rows: as many row tiles per workgroup as still leave two workgroups per CU
template <class T, int EPI>
int skinny(const ti_dense_args& a, hipStream_t s) {
  const long g = (long)((a.N + 15) / 16) * a.batch;
  const int mt = (a.M + 15) / 16;
  if constexpr (EPI == TI_DE_F32)
    // (row_div: its check in the kernel costs steps of small models 1 - 3 %)
    if (!a.tile_rows && mt == 1 && a.batch == 1 && a.N <= 2048 && a.row_div <= 1) return launch_half<T, EPI>(a, s);
  if (a.tile_rows || mt == 1 || g < 256) return launch_skinny<T, 1, EPI>(a, s);
  if (mt == 2 || g < 512) return launch_skinny<T, 2, EPI>(a, s);
  return launch_skinny<T, 4, EPI>(a, s);
}

// More rows: the tile whose rounds over the 256 CUs cost least: us of a launch, of a round and of 2048 k in it, fitted to
// measurements (bf16: M 70 .. 2048, N 512 .. 14336, K 256 .. 8192, fp32 M 70 .. 700; the choice costs 0.4 % more than the best
// tile of each point, in the mean).  rows: how many of the block's a tile takes.
struct BlockTile {
  int m, n, rows;
  float fix[2], round[2], k2048[2];   // bf16, fp32
};
constexpr int kTiles = 11;
constexpr BlockTile kTile[kTiles] = {
    {256, 256, 256, {-2.41f, 4.2f}, {13.0f, 4.2f}, {40.8f, 349.3f}}, {256, 256, 192, {-1.68f, 4.8f}, {11.36f, 4.8f}, {34.07f, 275.6f}},
    {128, 256, 128, {-0.74f, 7.4f}, {7.51f, 7.4f}, {26.02f, 232.9f}}, {128, 256, 96, {-0.75f, 6.8f}, {6.83f, 6.8f}, {22.84f, 195.5f}},
    {128, 128, 128, {2.40f, 4.6f}, {2.35f, 3.8f}, {16.59f, 128.8f}}, {128, 128, 128, {-0.97f, -2.3f}, {6.58f, 11.9f}, {14.30f, 132.9f}},
    {128, 128, 96, {0.49f, 0.4f}, {4.73f, 8.8f}, {13.01f, 99.2f}}, {64, 128, 64, {-0.16f, 1.4f}, {4.73f, 5.0f}, {9.26f, 69.0f}},
    {64, 128, 48, {0.39f, -0.5f}, {4.03f, 5.7f}, {8.37f, 54.0f}}, {64, 64, 64, {0.73f, -0.2f}, {3.40f, 4.4f}, {6.13f, 36.7f}},
    {32, 64, 32, {1.57f, 0.3f}, {2.27f, 3.9f}, {5.34f, 20.6f}}};
inline int tile_of(const ti_dense_args& a) {
  const int f = a.dtype == TI_DT_F32;
  int best = 0;
  float least = 0.0f;
  for (int i = 0; i < kTiles; ++i) {
    const BlockTile& t = kTile[i];
    const long wgs = (long)((a.M + t.rows - 1) / t.rows) * ((a.N + t.n - 1) / t.n) * a.batch;
    const float us = t.fix[f] + (float)((wgs + 255) / 256) * (t.round[f] + t.k2048[f] * (float)a.K * (1.f / 2048));
    if (i == 0 || us < least) {
      least = us;
      best = i;
    }
  }
  return best;
}
// Few 16 x 16 tiles of outputs (short prompts' narrower products, routers): a workgroup each (dense_skinny_kernel), its waves over k, where
// blocks would leave most CUs idle.  The line is where a second round of workgroups begins, with fp32's a third.  Measured, us, blocks -> this,
// bf16: 66 x 1024 (K 2048) 8.5 -> 5.7, 100 x 512 (1024) 6.2 -> 3.9, 1000 x 64 (2048) 8.5 -> 4.8, 2048 x 64 8.4 -> 7.8; at 512 tiles 250 x 512 (4096) 12.9 ->
// 11.2, at 576 and 640 8.4 -> 7.8 and 13.2 -> 15.9; fp32: 100 x 1024 (2048) 22.8 -> 12.0, 2048 x 64 23.0 -> 13.3, at 1024 tiles 23.0 -> 20.6, at
// 1216 13.2 -> 13.7.  Short k leaves the waves nothing to share (300 x 64, bf16: K 256 3.86 / 3.87, K 512 x 384 4.76 -> 3.88).  Few columns of long k have
// more rows at as many tiles, which every column tile reads again and which fit no L2: half as many (bf16: 1000 x 64 (8192) 22.0 -> 15.0, 1200 22.0 ->
// 23.6, 2048 x 64 (4096) 13.0 -> 14.6, 1000 x 128 (4096) 12.9 -> 14.6, 700 x 128 (3072) 10.6 -> 10.1, 500 x 256 (8192) 22.9 -> 21.4; fp32: 2048 x 64 (8192)
// 78.5 -> 44.4, 2048 x 128 (8192) 79.0 -> 83.7, (4096) 43.0 -> 43.5, 1000 x 256 (8192) 79.5 -> 74.9).
inline bool few_tiles(const ti_dense_args& a) {
  const int f = a.dtype == TI_DT_F32;
  const bool narrow = a.N < 256 && a.K > (f ? 4096 : 3072);
  return a.K >= (f ? 256 : 512) && (long)((a.M + 15) / 16) * ((a.N + 15) / 16) * a.batch <= (f ? 1024 : 512) >> narrow;
}
template <class T, int EPI>
int tiled(const ti_dense_args& a, hipStream_t s) {
  if (few_tiles(a)) return launch_skinny<T, 1, EPI>(a, s);
  const int i = tile_of(a), rows = kTile[i].rows;
  switch (i) {
    case 0: case 1: return launch_block<T, 1, 2, 4, 8, 4, 5, EPI>(a, rows, s);
    case 2: case 3: return launch_block<T, 1, 2, 4, 4, 4, 5, EPI>(a, rows, s);
    case 4: return launch_block<T, 1, 2, 2, 4, 4, 5, EPI>(a, rows, s);
    case 5: case 6: return launch_block<T, 2, 2, 2, 4, 4, 5, EPI>(a, rows, s);
    case 7: case 8: return launch_block<T, 2, 1, 4, 4, 2, 6, EPI>(a, rows, s);
    case 9: return launch_block<T, 2, 2, 2, 2, 2, 9, EPI>(a, rows, s);
    default: return launch_block<T, 2, 1, 4, 2, 1, 13, EPI>(a, rows, s);
  }
}
// Grouped products: the tile of the list's rows.
template <class T, int EPI>
int grouped(const ti_dense_args& a, hipStream_t s) {
  if constexpr (sizeof(T) == 2)
    if (expert_takes(a)) return launch_expert<EPI>(a, s);
  if (a.tile_rows == 256) return launch_block<T, 1, 2, 4, 8, 4, 5, EPI>(a, 256, s);
  if (a.tile_rows == 128) return launch_block<T, 1, 2, 4, 4, 4, 5, EPI>(a, 128, s);
  return launch_tile<T, 64, 256, 2, EPI>(a, s);
}

// Key and value fragments: blocks of 64 x 64 with two groups of waves while they are one round of workgroups (fp32: two), else of
// 128 x 128.  us, 128 x 128 -> 64 x 64, bf16: 130 rows of 512 columns (K 256) 7.5 -> 4.3, 300 of 2048 (K 512) 9.2 -> 5.6, 500 9.2 -> 6.0, 700
// 9.5 -> 9.8, 2048 10.4 -> 18.6; fp32 20.7 -> 8.0, 36 -> 13, 36 -> 13.3, 700 36 -> 23.4.
template <class T, int EPI>
int fragments(const ti_dense_args& a, hipStream_t s) {
  if ((long)((a.M + 127) / 128) * ((a.N + 127) / 128) <= (sizeof(T) == 4 ? 128 : 64)) return launch_block<T, 2, 2, 2, 2, 2, 9, EPI>(a, 64, s);
  return launch_block<T, 1, 2, 2, 4, 4, 5, EPI>(a, 128, s);
}

inline bool few_rows(const ti_dense_args& a) { return a.tile_rows == 1 || a.tile_rows == 16 || (!a.tile_rows && a.M <= 64); }
template <class T>
int dispatch_dense(const ti_dense_args& a, hipStream_t s) {
  const bool few = few_rows(a);
  switch (a.epi) {
    case TI_DE_F32: return few ? skinny<T, TI_DE_F32>(a, s) : tiled<T, TI_DE_F32>(a, s);
    case TI_DE_ROPE: return few ? skinny<T, TI_DE_ROPE>(a, s) : tiled<T, TI_DE_ROPE>(a, s);
    case TI_DE_ACT: return few ? skinny<T, TI_DE_ACT>(a, s) : tiled<T, TI_DE_ACT>(a, s);
    case TI_DE_LRU: return few ? skinny<T, TI_DE_LRU>(a, s) : launch_tile<T, 64, 128, 4, TI_DE_LRU>(a, s);   // (short k: the epilogue decides)
    case TI_DE_LOGITS: return few ? skinny<T, TI_DE_LOGITS>(a, s) : launch_tile<T, 64, 64, 4, TI_DE_LOGITS>(a, s);
    case TI_DE_GATE: return few ? skinny<T, TI_DE_GATE>(a, s) : launch_tile<T, 64, 64, 4, TI_DE_GATE>(a, s);
    case TI_DE_SWIGLU:
      if (few) return skinny<T, TI_DE_SWIGLU>(a, s);
      return a.tile_rows ? grouped<T, TI_DE_SWIGLU>(a, s) : tiled<T, TI_DE_SWIGLU>(a, s);
    case TI_DE_T:
      if (few) return skinny<T, TI_DE_T>(a, s);
      return a.tile_rows ? grouped<T, TI_DE_T>(a, s) : launch_tile<T, 64, 64, 4, TI_DE_T>(a, s);
    // (every row of a 128-row tile is written by the fragment epilogues; 2048 x 2048, K 512: 15.0 -> 14.4 us by blocks)
    case TI_DE_KFRAG: return fragments<T, TI_DE_KFRAG>(a, s);
    default: return fragments<T, TI_DE_VFRAG>(a, s);
  }
}

template <class T>
__global__ __launch_bounds__(256) void stack_fill_kernel(uint64_t stream, uint64_t n, float scale, T* out) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
    out[i] = (T)(scale * synth_unit(stream, i));
}

// fp32 source elements into fragment order (ti_stack_pack)
template <class T>
__global__ __launch_bounds__(256) void stack_pack_kernel(const float* src, int64_t rs, int64_t ks, int rows, int K, int nk,
                                                         const int32_t* map, T* dst) {
  constexpr int VEC = El<T>::VEC, KT = El<T>::KT;
  const int64_t n = (int64_t)rows * K;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int r = (int)(i / K), k = (int)(i - (int64_t)r * K), d = map ? map[r] : r;
    dst[(((int64_t)(d >> 4) * nk + k / KT) * 64 + ((k % KT) / VEC) * 16 + (d & 15)) * VEC + k % VEC] = (T)src[r * rs + k * ks];
  }
}
template <class T>
__global__ __launch_bounds__(256) void stack_convert_kernel(const float* src, uint64_t n, T* dst) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) dst[i] = (T)src[i];
}

}  // namespace ti

extern "C" int ti_stack_kpad(int dtype, int K) {
  const int u = dtype == TI_DT_BF16 ? 64 : 32;
  return (K + u - 1) / u * u;
}

extern "C" size_t ti_stack_weight_bytes(int dtype, int N, int K) {
  if (N < 1 || K < 1) return 0;
  return (size_t)((N + 15) / 16 * 16) * ti_stack_kpad(dtype, K) * (dtype == TI_DT_BF16 ? 2 : 4);
}

extern "C" int ti_stack_pack(const float* src, int64_t rs, int64_t ks, int rows, int K, const int32_t* map, int dtype,
                             void* dst, ti_stream_t stream) {
  using namespace ti;
  if (!src || !dst || rows < 1 || K < 1 || (dtype != TI_DT_BF16 && dtype != TI_DT_F32))
    return ti_set_error(TI_ERR_ARG, "ti_stack_pack: bad arguments");
  const unsigned g = (unsigned)std::min<int64_t>(((int64_t)rows * K + 255) / 256, 8192);
  const int kp = ti_stack_kpad(dtype, K);
  if (dtype == TI_DT_BF16)
    hipLaunchKernelGGL(stack_pack_kernel<bf16>, dim3(g), dim3(256), 0, (hipStream_t)stream, src, rs, ks, rows, K,
                       kp / El<bf16>::KT, map, (bf16*)dst);
  else
    hipLaunchKernelGGL(stack_pack_kernel<float>, dim3(g), dim3(256), 0, (hipStream_t)stream, src, rs, ks, rows, K,
                       kp / El<float>::KT, map, (float*)dst);
  TI_LAUNCH_CHECK("stack_pack_kernel");
  return TI_OK;
}

extern "C" int ti_stack_convert(const float* src, uint64_t n, int dtype, void* dst, ti_stream_t stream) {
  using namespace ti;
  if (!src || !dst || (dtype != TI_DT_BF16 && dtype != TI_DT_F32)) return ti_set_error(TI_ERR_ARG, "ti_stack_convert: bad arguments");
  if (n == 0) return TI_OK;
  const unsigned g = (unsigned)std::min<uint64_t>((n + 255) / 256, 4096);
  if (dtype == TI_DT_BF16)
    hipLaunchKernelGGL(stack_convert_kernel<bf16>, dim3(g), dim3(256), 0, (hipStream_t)stream, src, n, (bf16*)dst);
  else
    hipLaunchKernelGGL(stack_convert_kernel<float>, dim3(g), dim3(256), 0, (hipStream_t)stream, src, n, (float*)dst);
  TI_LAUNCH_CHECK("stack_convert_kernel");
  return TI_OK;
}

extern "C" size_t ti_dense_args_bytes(void) { return sizeof(ti_dense_args); }

extern "C" int ti_dense_tile(const ti_dense_args* a, int* rows, int* cols) {
  using namespace ti;
  if (!a || !rows || !cols || a->M < 1 || a->N < 1 || a->K < 1 || a->batch < 1 ||
      (a->epi != TI_DE_F32 && a->epi != TI_DE_SWIGLU && a->epi != TI_DE_ROPE && a->epi != TI_DE_ACT) || a->tile_rows)
    return ti_set_error(TI_ERR_ARG, "ti_dense_tile: bad arguments");
  const bool none = few_rows(*a) || few_tiles(*a);
  *rows = none ? 0 : kTile[tile_of(*a)].m;
  *cols = none ? 0 : kTile[tile_of(*a)].n;
  return TI_OK;
}

extern "C" int ti_dense(const ti_dense_args* a, ti_stream_t stream) {
  using namespace ti;
  if (!a || !a->w || !a->a || !a->out || a->M < 1 || a->N < 1 || a->K < 1 || a->batch < 1)
    return ti_set_error(TI_ERR_ARG, "ti_dense: bad arguments");
  if (a->dtype != TI_DT_BF16 && a->dtype != TI_DT_F32) return ti_set_error(TI_ERR_ARG, "ti_dense: dtype %d", a->dtype);
  const int vec = a->dtype == TI_DT_BF16 ? 8 : 4;
  if (a->K != ti_stack_kpad(a->dtype, a->K) || a->lda % vec || a->a_batch % vec)
    return ti_set_error(TI_ERR_ARG, "ti_dense: K %d / lda %d not padded", a->K, a->lda);
  if ((!a->tile_rows && !a->rows_in && a->lda < a->K) || a->batch > 65535)
    return ti_set_error(TI_ERR_ARG, "ti_dense: lda %d < K %d or batch %d", a->lda, a->K, a->batch);
  const bool rows_ok = a->tile_rows == 1 || a->tile_rows == 16 || a->tile_rows == 64 || a->tile_rows == 128 ||
                       a->tile_rows == 256;
  if (a->tile_rows && (a->epi == TI_DE_F32 || a->epi > TI_DE_SWIGLU || !rows_ok || a->max_tiles < 1 || a->max_tiles > 65535 ||
                       a->batch != 1 || (a->rows_in && a->row_div < 1) || !a->tiles ||
                       (a->tile_rows == 1 ? a->rows_in || a->rows_out : !a->n_tiles)))
    return ti_set_error(TI_ERR_ARG, "ti_dense: grouped arguments");
  if (!a->tile_rows && (a->rows_in || a->rows_out)) return ti_set_error(TI_ERR_ARG, "ti_dense: row lists need grouped tiles");
  switch (a->epi) {
    case TI_DE_F32: case TI_DE_T: break;
    case TI_DE_SWIGLU:
      if (a->N % 2 || a->batch != 1) return ti_set_error(TI_ERR_ARG, "ti_dense: SWIGLU N %d", a->N);
      break;
    case TI_DE_ROPE:
      if (!a->rope_cs || !a->pos || a->head_w < 1 || a->N % a->head_w || a->head_w % 4 || a->rot_off % 4 || a->ldo % 4 ||
          a->rot_off > a->head_w || a->batch != 1)
        return ti_set_error(TI_ERR_ARG, "ti_dense: ROPE arguments");
      break;
    case TI_DE_GATE:
      if (!a->gate || a->gate_ld < a->batch) return ti_set_error(TI_ERR_ARG, "ti_dense: GATE arguments");
      break;
    case TI_DE_LOGITS:
      if (!a->argmax || a->batch != 1) return ti_set_error(TI_ERR_ARG, "ti_dense: LOGITS arguments");
      break;
    case TI_DE_KFRAG: case TI_DE_VFRAG: {
      const int unit = a->epi == TI_DE_KFRAG ? 4 * vec : 16;
      if (a->head_w < 1 || a->N % a->head_w || a->head_w % unit || a->batch != 1 || a->key_blocks % 8 ||
          (long)a->key_blocks * 16 < ((long)a->M + 127) / 128 * 128)
        return ti_set_error(TI_ERR_ARG, "ti_dense: key / value fragments: head_w %d, key_blocks %d, M %d", a->head_w,
                            a->key_blocks, a->M);
      break;
    }
    case TI_DE_ACT:
      if (a->batch != 1 || a->t_cols < 0 || a->t_cols > a->N || (a->t_cols < a->N && !a->out2) || a->ldo < a->t_cols ||
          a->act < TI_ACT_NONE || a->act > TI_ACT_GELU_ERF)
        return ti_set_error(TI_ERR_ARG, "ti_dense: ACT arguments");
      break;
    case TI_DE_LRU:
      if (a->N % 2 || !a->add || !a->lru_rate)
        return ti_set_error(TI_ERR_ARG, "ti_dense: LRU arguments");
      break;
    default: return ti_set_error(TI_ERR_ARG, "ti_dense: epilogue %d", a->epi);
  }
  return a->dtype == TI_DT_BF16 ? dispatch_dense<bf16>(*a, (hipStream_t)stream) : dispatch_dense<float>(*a, (hipStream_t)stream);
}

extern "C" int ti_stack_fill(uint64_t seed, uint32_t tid, uint64_t n, float scale, int dtype, void* out, ti_stream_t stream) {
  using namespace ti;
  if (!out || (dtype != TI_DT_BF16 && dtype != TI_DT_F32)) return ti_set_error(TI_ERR_ARG, "ti_stack_fill: bad arguments");
  if (n == 0) return TI_OK;
  const unsigned g = (unsigned)std::min<uint64_t>((n + 255) / 256, 4096);
  const uint64_t st = synth_stream(seed, tid);
  if (dtype == TI_DT_BF16)
    hipLaunchKernelGGL(stack_fill_kernel<bf16>, dim3(g), dim3(256), 0, (hipStream_t)stream, st, n, scale, (bf16*)out);
  else
    hipLaunchKernelGGL(stack_fill_kernel<float>, dim3(g), dim3(256), 0, (hipStream_t)stream, st, n, scale, (float*)out);
  TI_LAUNCH_CHECK("stack_fill_kernel");
  return TI_OK;
}
