// attn_spread.hip -- decode attention of a GQA batch (4 or 8 q-heads per kv-head, head_dim 64 or 128) on MFMA, the
// streams' keys dealt evenly over the workgroups whatever their lengths (ti_attn_decode_spread).
//
// attn_split_kernel gives every (stream, kv-head) the same number of workgroups, so a ragged batch lasts as long as
// its longest stream, and does the products of all q-heads of a group on the vector unit, which at 4 and more heads
// takes about as long as the stream of keys (4 heads, head_dim 128: ~ 44 instructions per key and wave; 8192 keys take
// a CU 150 us or more).  Here:
//   * A stream's keys, in units of 32, are cut into segments of about the same length for all streams -- the units of
//     all streams over `parts` -- one workgroup each.  Every wave derives its workgroup's
//     segment from pos.  The last of a stream's segments to arrive merges them, as in attn_split_kernel.
//   * A wave takes every 4th unit of a segment: S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_16x16x32_f16, layouts as
//     in attn_prefill_kernel.  q and p are fp32, split into fp16 hi + lo: columns 0 .. 7 of the product hold hi,
//     columns 8 .. 15 lo (column c: q-head c & (G - 1)), so one product does both and a lane adds its partner's, column
//     c ^ 8, scores at once and outputs at the end.
//   * A column of q carries a power of two that takes its largest value to 2^14, p a factor 2^9 (both cancel), so that the
//     lo halves keep 2^-39 of the column's largest q and 2^-34 of the row's largest p; the running maximum moves when a
//     score passes it by 4 (p below 2^9 e^4 = 27955 fits fp16).  Scores are sums of 32 dims added pairwise.  Error of the
//     fp32 rows against float64 over that of attn_split_kernel's, queries of 0.03 .. 6, 400 .. 5000 keys, both head_dims and
//     group sizes: 0.99 in the mean (0.87 at small queries, 1.09 at the largest); without the three 1.2 .. 3.6.
// 4-wave workgroups, up to two a CU.  Workgroups come segment by segment, the kv-heads of a segment side by side: those
// the grid has past the last segment are the last, and the ones at work go to CUs of their own (kv-head by kv-head, 24
// streams: 18.4 us instead of 13.0).  Bound by HBM and, for short batches, by the chain of first loads, arrival and
// merge; measured, us per layer (attn_split_kernel -> this one): 32 streams of 4096 .. 8192 keys, 8 kv-heads x 4,
// head_dim 128: 178 -> 136 (820 MB); 24 streams of 700 .. 1400 keys, 4 kv-heads x 8, head_dim 64: 25.9 -> 13.0.
#include <math.h>

#include "common.hpp"

namespace ti {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct SpreadArgs {
  const float* q;
  const uint16_t* kc;
  const uint16_t* vc;
  const int32_t* pos;
  int32_t* tickets;   // [M][kv_heads], zero between calls
  float* part;        // [segment][heads][head_dim + 4]
  uint16_t* out;
  int64_t stride;
  int32_t max_seq, M, heads, kv_heads, parts;
  float scale;
  unsigned long long* stamp;
};

constexpr int kSpreadWaves = 4, kSpreadUnit = 32, kSpreadMaxSeg = 256;
constexpr int kAuxNt = 2;   // buffer aux: non-temporal (V's whole lines; K's come in halves, the second from L2)
constexpr float kSpreadUp = 512.0f, kSpreadSlack = 4.0f;

__device__ __forceinline__ void spread_split(float x, _Float16& hi, _Float16& lo) {   // hi + lo = x to ~ 2^-22
  asm("" : "+v"(x));   // one value for both roundings
  hi = (_Float16)x;
  lo = (_Float16)(x - (float)hi);
}

template <int HD, int G, int R>   // R: units in flight per wave
__global__ __launch_bounds__(64 * kSpreadWaves, 2) void attn_spread_kernel(const SpreadArgs a) {
  constexpr int DV = HD / 16, KW = HD / 32, NW = kSpreadWaves, ROW = HD + 4;
  const unsigned long long t_entry = stamp_now();
  __shared__ float s_m[NW][G], s_l[NW][G];
  __shared__ __attribute__((aligned(16))) float s_acc[NW][G][HD];
  __shared__ __attribute__((aligned(16))) float s_row[G][ROW];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, kvh = blockIdx.x, item = blockIdx.y;
  // this workgroup's segment: stream m, units [a0, a1), the stream's segment seg of n_seg; row: segments before the
  // stream's first (a stream has one at least)
  auto units = [&](int b) { return b + lane < a.M ? max(1, (a.pos[b + lane] + kSpreadUnit) / kSpreadUnit) : 0; };
  const int un0 = units(0);
  int total = 0;
  for (int b = 0; b < a.M; b += 64) {
    int u = b == 0 ? un0 : units(b);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) u += __shfl_xor(u, o, kWave);
    total += u;
  }
  // units a segment, 3 a wave at least
  const int chunk = max(3 * NW, (total + a.parts - 1) / a.parts);
  int m = -1, n_seg = 0, un = 0, row0 = 0;
  for (int b = 0, carry = 0; b < a.M; b += 64) {
    const int u = b == 0 ? un0 : units(b), n = (u + chunk - 1) / chunk;
    int incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o, kWave);
      incl += lane >= o ? t : 0;
    }
    const unsigned long long past = __builtin_amdgcn_ballot_w64(carry + incl > item);
    if (past) {
      const int l = __builtin_ctzll(past);
      m = b + l;
      n_seg = __builtin_amdgcn_readlane(n, l);
      un = __builtin_amdgcn_readlane(u, l);
      row0 = carry + __builtin_amdgcn_readlane(incl, l) - n_seg;
      break;
    }
    carry += __builtin_amdgcn_readlane(incl, 63);
  }
  // fewer segments than the grid allows for (the last workgroups, so that those at work are dealt to CUs of their own)
  if (m < 0) {
    stamp_end(a.stamp, t_entry);
    return;
  }
  const int seg = item - row0, a0 = un * seg / n_seg, a1 = un * (seg + 1) / n_seg, L = a.pos[m] + 1;
  {
    const int mine = L > 0 && a0 + wave < a1 ? (a1 - a0 - wave + NW - 1) / NW : 0;   // this wave's units
    f32x4 acc[DV];
#pragma unroll
    for (int t = 0; t < DV; ++t) acc[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -INFINITY, l_run = 0.0f;
    if (mine > 0) {
      const int64_t base = (int64_t)m * a.stride + (int64_t)kvh * a.max_seq * HD;
      const auto krs = buffer_rsrc(a.kc + base), vrs = buffer_rsrc(a.vc + base);
      // B operand: dims 32 c + 8 g + e of this lane's column; q's loads and the ring's go out before either is waited for
      const float* qr = a.q + ((size_t)m * a.heads + kvh * G + (r & (G - 1))) * HD + 8 * g;
      float4 qv[KW][2];
#pragma unroll
      for (int c = 0; c < KW; ++c) qv[c][0] = *(const float4*)(qr + 32 * c), qv[c][1] = *(const float4*)(qr + 32 * c + 4);
      typedef uint32_t vw_t __attribute__((ext_vector_type(DV / 2)));
      u32x4 kr[R][2][KW];
      vw_t vr[R][2][4];
      // unit i of this wave (one past its last: its last again, not consumed); rows past the stream's keys may be
      // unwritten and read its last key, which p = 0 multiplies away
      auto load = [&](int i, u32x4 (&k)[2][KW], vw_t (&v)[2][4]) {
        const int kb = (a0 + wave + NW * min(i, mine - 1)) * kSpreadUnit;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int key = min(kb + 16 * b + r, L - 1);
#pragma unroll
          for (int c = 0; c < KW; ++c)
            k[b][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, (key * HD + 8 * g + 32 * c) * 2, 0, 0));
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int off = (min(kb + 16 * b + 4 * g + j, L - 1) * HD + r * DV) * 2;
            if constexpr (HD == 128) v[b][j] = __builtin_bit_cast(vw_t, __builtin_amdgcn_raw_buffer_load_b128(vrs, off, 0, kAuxNt));
            else v[b][j] = __builtin_bit_cast(vw_t, __builtin_amdgcn_raw_buffer_load_b64(vrs, off, 0, kAuxNt));
          }
      };
#pragma unroll
      for (int u = 0; u < R; ++u) load(u, kr[u], vr[u]);
      __builtin_amdgcn_sched_barrier(0);   // (q is not waited for before the ring's loads are out)
      // a column of q times a power of two, its largest value to 2^14 .. 2^15, so that the lo halves are no subnormals;
      // scores and their maximum stay in these units (up to 2^38), `unit` of them are 1
      f16x8 qf[KW];
      float unit = 1.0f, back = 1.0f;
      {
        float mx = 0.0f;
#pragma unroll
        for (int c = 0; c < KW; ++c)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(qv[c][j].x), fabsf(qv[c][j].y))), fmaxf(fabsf(qv[c][j].z), fabsf(qv[c][j].w)));
        mx = xor32_max(xor16_max(mx)) * a.scale;
        const int e = mx < INFINITY ? max((int)(__builtin_bit_cast(uint32_t, mx) >> 23) - 141, -100) : 0;
        unit = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
        back = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
        const float f = a.scale * unit;
#pragma unroll
        for (int c = 0; c < KW; ++c) {
          const float v[8] = {qv[c][0].x, qv[c][0].y, qv[c][0].z, qv[c][0].w, qv[c][1].x, qv[c][1].y, qv[c][1].z, qv[c][1].w};
#pragma unroll
          for (int e2 = 0; e2 < 8; ++e2) {
            _Float16 hi, lo;
            spread_split(v[e2] * f, hi, lo);
            qf[c][e2] = r < 8 ? hi : lo;
          }
        }
      }
      const float log2e = back * 1.44269504088896341f, slack = unit * kSpreadSlack;
      for (int i0 = 0; i0 < mine; i0 += R) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
          const int i = i0 + u, kb = i < mine ? (a0 + wave + NW * i) * kSpreadUnit : L;
          // this unit's K passes through an empty asm behind the previous unit's softmax, so that its products are not
          // hoisted to where they would wait for the loads issued last
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int c = 0; c < KW; ++c) asm volatile("" : "+v"(kr[u][b][c]));
          // 32 dims a sum, added pairwise: one chain over the dims rounds its whole sum at every step
          f32x4 sc[KW][2], s[2];
#pragma unroll
          for (int c = 0; c < KW; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b)
              sc[c][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kr[u][b][c]), qf[c], (f32x4){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
          for (int b = 0; b < 2; ++b) s[b] = KW == 2 ? sc[0][b] + sc[1][b] : (sc[0][b] + sc[1][b]) + (sc[KW - 2][b] + sc[KW - 1][b]);
          float pv[2][4], bm = -INFINITY;
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) pv[b][e] = s[b][e] + lane_xor<8>(s[b][e]);
          if (kb + kSpreadUnit > L) {   // the stream's last unit, or none
            const int lim = L - 1 - kb - 4 * g;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (16 * b + e > lim) pv[b][e] = -INFINITY;
          }
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) bm = fmaxf(bm, pv[b][e]);
          bm = xor32_max(xor16_max(bm));
          const float mn = fmaxf(m_run, bm);
          if (__builtin_amdgcn_ballot_w64(mn > m_run + slack) != 0) {   // wave-uniform; the first unit
            const float alpha = m_run == mn ? 1.0f : __builtin_amdgcn_exp2f((m_run - mn) * log2e);
            l_run *= alpha;
            m_run = mn;
#pragma unroll
            for (int t = 0; t < DV; ++t)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[t][e] *= alpha;
          }
          f16x8 pf;   // k-slot 4 b + e: key 16 b + 4 g + e of the unit
          float ps = 0.0f;
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float p = __builtin_amdgcn_exp2f((pv[b][e] - m_run) * log2e) * kSpreadUp;
              ps += p;
              _Float16 hi, lo;
              spread_split(p, hi, lo);
              pf[4 * b + e] = r < 8 ? hi : lo;
            }
          l_run += ps;
          asm volatile("" : "+v"(l_run));
#pragma unroll
          for (int t = 0; t < DV; ++t) {
            const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
            u32x4 vf;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              vf[2 * b] = __builtin_amdgcn_perm(vr[u][b][1][t >> 1], vr[u][b][0][t >> 1], sel);
              vf[2 * b + 1] = __builtin_amdgcn_perm(vr[u][b][3][t >> 1], vr[u][b][2][t >> 1], sel);
            }
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, vf), pf, acc[t], 0, 0, 0);
          }
          load(i + R, kr[u], vr[u]);
        }
      }
      m_run *= back;
      l_run += lane_xor<16>(l_run);
      l_run += lane_xor<32>(l_run);
#pragma unroll
      for (int t = 0; t < DV; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] += lane_xor<8>(acc[t][e]);
    }
    // lane (r, g): O^T[dim DV (4 g + e) + t][column r] in acc[t][e]
    if (r < G) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < DV; t += 4)
          *(f32x4*)&s_acc[wave][r][DV * (4 * g + e) + t] = (f32x4){acc[t][e], acc[t + 1][e], acc[t + 2][e], acc[t + 3][e]};
      if (g == 0) {
        s_m[wave][r] = m_run;
        s_l[wave][r] = l_run;
      }
    }
    __syncthreads();
    for (int idx = tid; idx < G * HD; idx += 64 * NW) {
      const int h = idx / HD, d = idx - h * HD;
      float mx = s_m[0][h];
#pragma unroll
      for (int w = 1; w < NW; ++w) mx = fmaxf(mx, s_m[w][h]);
      float o = 0.0f, l = 0.0f;
      if (mx != -INFINITY) {
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const float f = s_m[w][h] == -INFINITY ? 0.0f : __expf(s_m[w][h] - mx);
          o = fmaf(f, s_acc[w][h][d], o);
          l = fmaf(f, s_l[w][h], l);
        }
      }
      if (n_seg == 1) {
        a.out[((size_t)m * a.heads + kvh * G + h) * HD + d] = f2h(l > 0.0f ? o / l : 0.0f);
        continue;
      }
      s_row[h][d] = o;
      if (d < 4) s_row[h][HD + d] = d == 0 ? mx : d == 1 ? l : 0.0f;
    }
  }
  if (n_seg == 1) {
    stamp_end(a.stamp, t_entry);
    return;
  }
  __syncthreads();
  // publish the G rows write-through, drain, arrive; the last arriver merges (attn_split_body's hand-off)
  const __amdgpu_buffer_rsrc_t wsr = sc1_rsrc(a.part);
  auto at = [&](int s) { return (uint32_t)(((row0 + s) * a.heads + kvh * G) * ROW); };
  for (int i = tid; i < G * ROW / 4; i += 64 * NW)
    __builtin_amdgcn_raw_buffer_store_b128(*(const f32x4*)(&s_row[0][0] + 4 * i), wsr, (at(seg) + 4 * i) * 4, 0, kAuxSc1Load);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int32_t* ticket = a.tickets + (size_t)m * a.kv_heads + kvh;
  if (tid == 0) s_last = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n_seg - 1;
  __syncthreads();
  if (s_last) {
    // CAP segments' rows at a time through LDS, one round trip each, in segment order (the sum does not depend on who
    // merges)
    constexpr int CAP = 12 * 64 * NW * 4 / (G * ROW), OUT = G * HD / (64 * NW);
    __shared__ __attribute__((aligned(16))) float s_seg[CAP][G][ROW];
    float mx[OUT], num[OUT], den[OUT];
#pragma unroll
    for (int k = 0; k < OUT; ++k) mx[k] = -INFINITY, num[k] = 0.0f, den[k] = 0.0f;
    for (int s0 = 0; s0 < n_seg; s0 += CAP) {
      const int n = min(CAP, n_seg - s0), nv = n * G * (ROW / 4);
      f32x4 v[12];
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        const int i = min(tid + k * 64 * NW, nv - 1), s = i / (G * (ROW / 4));
        v[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wsr, (at(s0 + s) + 4 * (i - s * (G * (ROW / 4)))) * 4, 0,
                                                                              kAuxSc1Load));
      }
#pragma unroll
      for (int k = 0; k < 12; ++k)
        if (tid + k * 64 * NW < nv) *(f32x4*)(&s_seg[0][0][0] + 4 * (tid + k * 64 * NW)) = v[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < OUT; ++k) {
        const int idx = tid + k * 64 * NW, h = idx / HD, d = idx - h * HD;
        float top = mx[k];
        for (int s = 0; s < n; ++s) top = fmaxf(top, s_seg[s][h][HD]);
        const float fa = __expf(mx[k] - top);   // (a segment holds a key at least: top is above -inf)
        num[k] *= fa;
        den[k] *= fa;
        mx[k] = top;
        for (int s = 0; s < n; ++s) {
          const float f = __expf(s_seg[s][h][HD] - top);
          num[k] = fmaf(f, s_seg[s][h][d], num[k]);
          den[k] = fmaf(f, s_seg[s][h][HD + 1], den[k]);
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < OUT; ++k) {
      const int idx = tid + k * 64 * NW, h = idx / HD, d = idx - h * HD;
      a.out[((size_t)m * a.heads + kvh * G + h) * HD + d] = f2h(num[k] / den[k]);
    }
    if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-arm
  }
  stamp_end(a.stamp, t_entry);
}

template <int HD, int G, int R>
static int launch_spread(const SpreadArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((attn_spread_kernel<HD, G, R>), dim3(a.kv_heads, a.parts + a.M), dim3(64 * kSpreadWaves), 0, s, a);
  TI_LAUNCH_CHECK("attn_spread_kernel");
  return TI_OK;
}

}  // namespace ti

static size_t spread_tickets(int heads) { return ((size_t)TI_ATTN_MAX_M * heads * sizeof(int32_t) + 255) & ~(size_t)255; }

extern "C" size_t ti_attn_spread_workspace_bytes(int M, int heads, int head_dim, int parts) {
  return spread_tickets(heads) + (size_t)(parts + M) * heads * (head_dim + 4) * sizeof(float);
}

extern "C" int ti_attn_decode_spread(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, int64_t kv_stream_stride,
                                     int max_seq, const int32_t* pos, int M, int heads, int kv_heads, int head_dim, int parts,
                                     float* workspace, uint16_t* out, ti_stream_t stream) {
  using namespace ti;
  if (!q || !k_cache || !v_cache || !pos || !workspace || !out)
    return ti_set_error(TI_ERR_ARG, "ti_attn_decode_spread: null pointer");
  if (M < 1 || M > TI_ATTN_MAX_M || heads < 1 || kv_heads < 1 || kv_heads > 65535 || heads % kv_heads || parts < 1 || parts > kSpreadMaxSeg ||
      max_seq < 1 || (int64_t)max_seq * head_dim * 2 > 0x7fffffff)
    return ti_set_error(TI_ERR_ARG, "ti_attn_decode_spread: bad sizes M=%d heads=%d kv_heads=%d parts=%d max_seq=%d", M, heads,
                        kv_heads, parts, max_seq);
  const int G = heads / kv_heads;
  if ((head_dim != 64 && head_dim != 128) || (G != 4 && G != 8))
    return ti_set_error(TI_ERR_UNSUPPORTED, "ti_attn_decode_spread: head_dim %d, heads/kv_heads %d (64 or 128, 4 or 8)", head_dim, G);
  if (kv_stream_stride < (int64_t)kv_heads * max_seq * head_dim)
    return ti_set_error(TI_ERR_ARG, "ti_attn_decode_spread: kv_stream_stride too small");
  if (ti_attn_spread_workspace_bytes(M, heads, head_dim, parts) - spread_tickets(heads) > 0x7fffffff)
    return ti_set_error(TI_ERR_ARG, "ti_attn_decode_spread: M=%d parts=%d: the partial rows pass 2 GiB", M, parts);
  SpreadArgs a;
  a.q = q;
  a.kc = k_cache;
  a.vc = v_cache;
  a.pos = pos;
  a.tickets = (int32_t*)workspace;
  a.part = (float*)((char*)workspace + spread_tickets(heads));
  a.out = out;
  a.stride = kv_stream_stride;
  a.max_seq = max_seq;
  a.M = M;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.parts = parts;
  a.scale = 1.0f / sqrtf((float)head_dim);
  a.stamp = ti_stamp_next(STAMP_ATTN, (long)(parts + M) * kv_heads);
  hipStream_t s = (hipStream_t)stream;
  if (head_dim == 128) return G == 4 ? launch_spread<128, 4, 2>(a, s) : launch_spread<128, 8, 2>(a, s);
  return G == 4 ? launch_spread<64, 4, 2>(a, s) : launch_spread<64, 8, 2>(a, s);
}
