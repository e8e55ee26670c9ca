// dense.hpp -- what the kernels of layer-stack products share (dense.hip, dense_expert.hip): epilogues, grouped tiles.
#pragma once

#include <algorithm>

#include "elem.hpp"

namespace ti {

__device__ __forceinline__ unsigned long long logit_key(float v, int n) {
  return ((unsigned long long)float_order_key(v) << 32) | (unsigned long long)(0xFFFFFFFFu - (uint32_t)n);
}

// GELU for 16-bit outputs, h = z / 2: |z| < 1: h + h erf, erf(z / sqrt 2) = z Q(z^2); beyond: z - h E or h E with E =
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
  const float far = z >= 0.0f ? fmaf(-fminf(h, 1e38f), e, z) : h * e;   // (inf - inf * 0)
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
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (a.add) v[i] += a.add[min(n0 + i, a.N - 1)];
        if (n0 + i < a.act_cols) v[i] = activate<T>(a.act, v[i]);
      }
      T* o = (T*)a.out + (size_t)mo * a.ldo + n0;
      if (n0 + 4 <= a.t_cols && (a.ldo & 3) == 0) {
        *(typename El<T>::Q*)o = quad<T>(v);
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = n0 + i;
        if (n < a.t_cols) o[i] = (T)v[i];
        else if (n < a.N) a.out2[(size_t)mo * a.ld2 + n - a.t_cols] = v[i];
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

// dense_expert.hip
bool expert_takes(const ti_dense_args& a);
template <int EPI>
int launch_expert(const ti_dense_args& a, hipStream_t s);

}  // namespace ti
