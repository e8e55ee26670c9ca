// dense.hpp -- what the kernels of layer-stack products share (dense.hip, dense_expert.hip): epilogues, grouped tiles.
#pragma once

#include <algorithm>

#include "elem.hpp"

namespace ti {

__device__ __forceinline__ unsigned long long logit_key(float v, int n) {
  return ((unsigned long long)float_order_key(v) << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)n);
}

// GELU for 16-bit outputs, h = z / 2: |z| < 1: h + h erf, erf(z / sqrt 2) = z Q(z^2); beyond: max(z, 0) - |h| E with E =
// erfc(|z| / sqrt 2) = t 2^(P(t) - x^2 log2 e), t = 1 / (1 + x / 2) (the form of erfcc in Numerical Recipes, Press,
// Teukolsky, Vetterling, Flannery), P fitted to log2(erfcx(x) / t) over x 0.7 .. 16 and Q over its range (Chebyshev bases,
// reweighted towards equal errors).  Against float64 no further off than 0.5 z (1 + erff) in any part of the range
// (relative, rms): |z| < 0.3 2.8e-8 against 4.2e-8, 0.3 .. 6 2.9e-8 against 4.0e-8, -1.4 .. -1 1.0e-7 against 1.4e-7,
// -5 .. -3 3.5e-7 against 6.6e-3 (its cancellation).  ~ 28 instructions; erff's two branches, ~ 60 (1500 x 8192, K 2048, us:
// 88 -> 78).
__device__ __forceinline__ float gelu_erf(float z) {
  const float h = 0.5f * z, w = z * z;
  float q = 1.84936216e-04f;
  q = fmaf(q, w, -2.33070040e-03f);
  q = fmaf(q, w, 1.99283324e-02f);
  q = fmaf(q, w, -1.32977456e-01f);
  q = fmaf(q, w, 7.97884405e-01f);
  const float t = __builtin_amdgcn_rcpf(fmaf(fabsf(z), 0.35355339059327376f, 1.0f));
  float p = -3.10784221e-01f;
  p = fmaf(p, t, 1.23818982e+00f);
  p = fmaf(p, t, -1.68483531e+00f);
  p = fmaf(p, t, 7.01514661e-01f);
  p = fmaf(p, t, -1.47596598e-01f);
  p = fmaf(p, t, 5.91505647e-01f);
  p = fmaf(p, t, 1.43761384e+00f);
  p = fmaf(p, t, -1.82553995e+00f);
  const float e = t * __builtin_amdgcn_exp2f(fmaf(w, -0.72134752044448170f, p));
  const float far = fmaf(-fminf(fabsf(h), 1e38f), e, fmaxf(z, 0.0f));   // (inf - inf * 0)
  return w < 1.0f ? fmaf(h, z * q, h) : far;
}

template <class T>
__device__ __forceinline__ float activate(int act, float z) {
  if (act == TI_ACT_GELU_ERF) {
    if constexpr (sizeof(T) == 2) return gelu_erf(z);
    else return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
  }
  // (1 + tanh x) / 2 is the logistic function of 2 x
  if (act == TI_ACT_GELU_TANH) return z * fast_sigmoid(1.59576912160573072f * fmaf(0.044715f * z * z, z, z));
  return z;
}

// Four consecutive output columns n0.. of row m (out row mo); rows >= rows are padding.
template <class T, int EPI>
__device__ __forceinline__ void dense_store(const ti_dense_args& a, int batch, int m, int mo, int rows, int n0, f32x4 v) {
  constexpr int VEC = El<T>::VEC, KT = El<T>::KT;
  const bool live = m < rows;
  switch (EPI) {
    case TI_DE_F32: {
      if (!live) return;
      float* o = (float*)a.out + (size_t)batch * a.o_batch + (size_t)mo * a.ldo + n0;
      if (a.add)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += a.add[min(n0 + i, a.N - 1)];
      if (n0 + 4 <= a.N && ((a.ldo | a.o_batch) & 3) == 0) {
        *(f32x4*)o = v;
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + i < a.N) o[i] = v[i];
      return;
    }
    case TI_DE_T: {
      if (!live) return;
      T* o = (T*)a.out + (size_t)batch * a.o_batch + (size_t)mo * a.ldo + n0;
      if (n0 + 4 <= a.N && ((a.ldo | a.o_batch) & 3) == 0) {
        *(typename El<T>::Q*)o = quad<T>(v);
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + i < a.N) o[i] = (T)v[i];
      return;
    }
    case TI_DE_SWIGLU: {
      if (!live) return;
      T* o = (T*)a.out + (size_t)mo * a.ldo + (n0 >> 1);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (n0 + 2 * i < a.N) o[i] = (T)(v[2 * i] * sigmoidf(v[2 * i]) * v[2 * i + 1]);
      return;
    }
    case TI_DE_ROPE: {
      if (!live || n0 >= a.N) return;
      const int r = n0 % a.head_w - a.rot_off;
      if (r >= 0) {
        const int pairs = (a.head_w - a.rot_off) >> 1;
        const float* cs = a.rope_cs + ((size_t)a.pos[m] * pairs + (r >> 1)) * 2;
        const f32x4 t = *(const f32x4*)cs;
        v = (f32x4){v[0] * t[0] - v[1] * t[1], v[1] * t[0] + v[0] * t[1], v[2] * t[2] - v[3] * t[3],
                    v[3] * t[2] + v[2] * t[3]};
      }
      *(typename El<T>::Q*)((T*)a.out + (size_t)mo * a.ldo + n0) = quad<T>(v);
      return;
    }
    case TI_DE_GATE: {
      if (!live) return;
      const float g = a.gate[(size_t)m * a.gate_ld + batch];
      T* o = (T*)a.out + (size_t)mo * a.ldo + (size_t)batch * a.N + n0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n0 + i < a.N) o[i] = (T)(v[i] * g);
      return;
    }
    case TI_DE_KFRAG: {   // every row of the tile is written (padding rows repeat the last key)
      if (n0 >= a.N) return;
      const int h = n0 / a.head_w, d = n0 - h * a.head_w, dt = a.head_w / KT;
      T* o = (T*)a.out + ((((size_t)h * a.key_blocks + (m >> 4)) * dt + d / KT) * 64 + ((d % KT) / VEC) * 16 + (m & 15)) * VEC +
             d % VEC;
      *(typename El<T>::Q*)o = quad<T>(v);
      return;
    }
    case TI_DE_ACT: {
      if (!live) return;
      if (n0 + 4 <= a.N && (n0 >= a.act_cols || n0 + 4 <= a.act_cols)) {
        if (a.add)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] += a.add[n0 + i];
        if (n0 < a.act_cols)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = activate<T>(a.act, v[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (a.add) v[i] += a.add[min(n0 + i, a.N - 1)];
          if (n0 + i < a.act_cols) v[i] = activate<T>(a.act, v[i]);
        }
      }
      T* o = (T*)a.out + (size_t)mo * a.ldo + n0;
      if (n0 + 4 <= a.t_cols && (a.ldo & 3) == 0) {
        *(typename El<T>::Q*)o = quad<T>(v);
        return;
      }
      float* o2 = a.out2 + (size_t)mo * a.ld2 + n0 - a.t_cols;
      if (n0 >= a.t_cols && n0 + 4 <= a.N && ((a.t_cols | a.ld2) & 3) == 0 && ((uintptr_t)a.out2 & 15) == 0) {
        *(f32x4*)o2 = v;
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + i;
        if (n < a.t_cols) o[i] = (T)v[i];
        else if (n < a.N) o2[i] = v[i];
      }
      return;
    }
    case TI_DE_LRU: {
      if (!live || n0 >= a.N) return;
      const int per = a.N >> 1, channels = per * a.batch;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int j = (n0 >> 1) + i, c = batch * per + j;
        if (j >= per) return;
        const float* gb = a.add + (size_t)batch * a.N + n0 + 2 * i;
        const float u = (float)((const T*)a.a)[(size_t)m * a.lda + (size_t)batch * a.a_batch + j];
        *(float2*)((float*)a.out + ((size_t)m * channels + c) * 2) = lru_coef(v[2 * i] + gb[0], v[2 * i + 1] + gb[1], a.lru_rate[c], u);
      }
      return;
    }
    default: return;
  }
}

// TI_DE_VFRAG: four consecutive keys m0.. of column n.
template <class T>
__device__ __forceinline__ void dense_store_v(const ti_dense_args& a, int m0, int n, f32x4 v) {
  constexpr int VEC = El<T>::VEC, KT = El<T>::KT;
  if (n >= a.N) return;
  const int h = n / a.head_w, d = n - h * a.head_w;
  const int kb = m0 / KT, t = (m0 % KT) >> 4, g = (m0 & 15) >> 2, nkb = a.key_blocks * 16 / KT;
  T* o = (T*)a.out + ((((size_t)h * (a.head_w >> 4) + (d >> 4)) * nkb + kb) * 64 + g * 16 + (d & 15)) * VEC + t * 4;
  *(typename El<T>::Q*)o = quad<T>(v);
}

// Greedy argmax keys of a 16-column tile: lane l holds columns n0.. of row m = its (l & 15).
__device__ __forceinline__ void dense_argmax(const ti_dense_args& a, int m, int rows, int n0, f32x4 v, int lane, int slot) {
  unsigned long long key = 0ull;
  if (m < rows) {
    float* o = (float*)a.out + (size_t)m * a.ldo + n0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n0 + i < a.N) {
        o[i] = v[i];
        const unsigned long long k = logit_key(v[i], n0 + i);
        key = k > key ? k : key;
      }
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    const unsigned long long other = __shfl_xor(key, o, kWave);
    key = other > key ? other : key;
  }
  if (lane < 16 && key) atomicMax(a.argmax + (size_t)m * TI_ARGMAX_SLOTS + (slot & (TI_ARGMAX_SLOTS - 1)), key);
}

struct DenseSpan {   // what a workgroup works on
  int rows, first, batch;
  const void* w;
};

__device__ __forceinline__ bool dense_span(const ti_dense_args& a, int y, DenseSpan& s, size_t esize) {
  s.batch = 0;
  int e = 0;
  if (a.tile_rows == 1) {
    s.first = y;
    s.rows = 1;
    e = a.tiles[y];
    e = __builtin_amdgcn_readfirstlane(e);
  } else if (a.tile_rows) {
    if (y >= *a.n_tiles) return false;
    e = a.tiles[4 * y];
    s.first = a.tiles[4 * y + 1];
    s.rows = a.tiles[4 * y + 2];
  } else {
    s.first = 0;
    s.rows = a.M;
    s.batch = e = y;
  }
  s.w = (const char*)a.w + (size_t)e * a.w_batch * esize;
  return true;
}
__device__ __forceinline__ int row_in(const ti_dense_args& a, int p) {
  const int r = a.rows_in ? a.rows_in[p] : p;
  return a.row_div > 1 ? r / a.row_div : r;
}
__device__ __forceinline__ int row_out(const ti_dense_args& a, int p) { return a.rows_out ? a.rows_out[p] : p; }

// One 16 x 16 block of products: row tile mt.. (row m, out row mo of this lane), column tile nt.
template <class T, int EPI>
__device__ __forceinline__ void dense_out(const ti_dense_args& a, const DenseSpan& sp, int m, int mo, int mt, int nt, f32x4 v, int lane) {
  if constexpr (EPI == TI_DE_VFRAG)
    dense_store_v<T>(a, mt + 4 * (lane >> 4), nt * 16 + (lane & 15), v);
  else if constexpr (EPI == TI_DE_LOGITS)
    dense_argmax(a, m, sp.rows, nt * 16 + 4 * (lane >> 4), v, lane, nt);
  else
    dense_store<T, EPI>(a, sp.batch, m, mo, sp.rows, nt * 16 + 4 * (lane >> 4), v);
}

template <int N>
__device__ __forceinline__ void wait_dma() {   // all but the wave's N newest vector memory operations done
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 4 x 4 dwords turned over between four registers and the four 16-lane groups: d[k] of group g becomes d[g] of group k.
__device__ __forceinline__ void turn_groups(uint32_t (&d)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto t = __builtin_amdgcn_permlane32_swap(d[i], d[i + 2], false, false);
    d[i] = t[0];
    d[i + 2] = t[1];
  }
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const auto t = __builtin_amdgcn_permlane16_swap(d[i], d[i + 1], false, false);
    d[i] = t[0];
    d[i + 1] = t[1];
  }
}

// Rows of 16-bit outputs that take 16 bytes at any multiple of 8 columns.
__host__ __device__ inline bool rows16(const ti_dense_args& a) { return a.ldo % 8 == 0 && ((uintptr_t)a.out & 15) == 0; }

// A row tile of four column tiles nt.. (lane: row lane & 15, out row mo), 16-bit outputs: a lane takes 16 consecutive columns of
// its row (SiLU * up: 8), where the products gave it 4 of each tile.
__device__ __forceinline__ void store64(const ti_dense_args& a, bool live, int mo, int nt, const f32x4 (&v)[4], int lane) {
  uint32_t d[2][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u32x2 q = __builtin_bit_cast(u32x2, quad<bf16>(v[j]));
    d[0][j] = q[0];
    d[1][j] = q[1];
  }
  turn_groups(d[0]);
  turn_groups(d[1]);
  if (live) {
    u32x4* o = (u32x4*)((bf16*)a.out + (size_t)mo * a.ldo + nt * 16 + (lane >> 4) * 16);
    o[0] = (u32x4){d[0][0], d[1][0], d[0][1], d[1][1]};
    o[1] = (u32x4){d[0][2], d[1][2], d[0][3], d[1][3]};
  }
}
__device__ __forceinline__ void store_swiglu64(const ti_dense_args& a, bool live, int mo, int nt, const f32x4 (&v)[4], int lane) {
  uint32_t d[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16x2 q = {(bf16)(v[j][0] * sigmoidf(v[j][0]) * v[j][1]), (bf16)(v[j][2] * sigmoidf(v[j][2]) * v[j][3])};
    d[j] = __builtin_bit_cast(uint32_t, q);
  }
  turn_groups(d);
  if (live) *(u32x4*)((bf16*)a.out + (size_t)mo * a.ldo + nt * 8 + (lane >> 4) * 8) = (u32x4){d[0], d[1], d[2], d[3]};
}

// A block's epilogue on whole 64-column pieces: what the columns need (bias, activation, place in the head) is found once for
// a wave's rows, outputs leave as 16 bytes a lane.  wave64: column tiles nt .. nt + 3 take it.  (dense_store decides and checks
// per element and stores 2 .. 8 bytes; unrolled for a wave's 32 tiles of 4, ~ 72 KB of code.  1500 rows, K 2048, 256 x 256 blocks, us:
// 8192 columns plain 58.6 -> 49.8, GELU 69.2 -> 61.3, SiLU * up 53.9 -> 48.9; 5120 with GELU (tanh) and biases 45.1 -> 33.9; 3072
// rotary, K 1536, 26.7 -> 23.8.)
template <class T, int EPI>
__device__ __forceinline__ bool wave64(const ti_dense_args& a, int nt) {
  if constexpr (sizeof(T) != 2 || (EPI != TI_DE_SWIGLU && EPI != TI_DE_ROPE && EPI != TI_DE_ACT)) return false;
  const int n0 = nt * 16, n1 = n0 + 64;
  if (n1 > a.N || !rows16(a)) return false;
  return EPI != TI_DE_ACT || (n1 <= a.t_cols && (n1 <= a.act_cols || n0 >= a.act_cols));
}
template <int EPI>
struct Wave64 {   // column tiles nt .. nt + 3
  f32x4 add[4];
  int rot[4], act;   // ROPE: the first of the lane's columns within the head's rotated part, or negative
  bool any;
  __device__ __forceinline__ Wave64(const ti_dense_args& a, int nt, int lane) {
    if constexpr (EPI == TI_DE_ACT) {
      act = nt * 16 < a.act_cols ? a.act : TI_ACT_NONE;
      if (a.add)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) add[j][i] = a.add[(nt + j) * 16 + 4 * (lane >> 4) + i];
    }
    if constexpr (EPI == TI_DE_ROPE) {
#pragma unroll
      for (int j = 0; j < 4; ++j) rot[j] = ((nt + j) * 16 + 4 * (lane >> 4)) % a.head_w - a.rot_off;
      any = __builtin_amdgcn_ballot_w64(max(max(rot[0], rot[1]), max(rot[2], rot[3])) >= 0) != 0;
    }
  }
  __device__ __forceinline__ void out(const ti_dense_args& a, bool live, int m, int mo, int nt, f32x4 (&v)[4], int lane) {
    if constexpr (EPI == TI_DE_SWIGLU) {
      store_swiglu64(a, live, mo, nt, v, lane);
    } else {
      if constexpr (EPI == TI_DE_ROPE) {
        if (any) {
          const int pairs = (a.head_w - a.rot_off) >> 1;
          const float* cs = a.rope_cs + (size_t)a.pos[live ? m : 0] * pairs * 2;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 t = *(const f32x4*)(cs + max(rot[j], 0));   // (columns in front of the rotated part are left as they are)
            const f32x4 u = {v[j][0] * t[0] - v[j][1] * t[1], v[j][1] * t[0] + v[j][0] * t[1], v[j][2] * t[2] - v[j][3] * t[3],
                             v[j][3] * t[2] + v[j][2] * t[3]};
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = rot[j] >= 0 ? u[i] : v[j][i];
          }
        }
      } else {
        if (a.add)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] += add[j];
        if (act == TI_ACT_GELU_ERF) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = activate<bf16>(TI_ACT_GELU_ERF, v[j][i]);
        } else if (act == TI_ACT_GELU_TANH) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = activate<bf16>(TI_ACT_GELU_TANH, v[j][i]);
        }
      }
      store64(a, live, mo, nt, v, lane);
    }
  }
};

// dense_expert.hip
bool expert_takes(const ti_dense_args& a);
template <int EPI>
int launch_expert(const ti_dense_args& a, hipStream_t s);

}  // namespace ti
