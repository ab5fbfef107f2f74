// A token's rotation and its write into the cache, by one workgroup: in a launch of its own (rope_kv_store) and beside the
// state-space mixer's first launch (ssd.hip).  The cache's layout is the one that attention.hip describes.
#pragma once
#include "common.h"

// ---------------------------------------------------------------- rope + cache write
// For token t at absolute position p:
//   q[t, h, :] is rotated in place; k[t, h, :] is rotated and stored; v[t, h, :] is stored.
//   Rotation (half-split, first rotary_dim dims): angle = (float)p * inv_freq[j];
//   out[j] = x[j] cos - x[j+half] sin;  out[j+half] = x[j+half] cos + x[j] sin.
//   (reference: src/decoder.rs:186-195, 226-229; K is cached after rotation, :953-962)
// slot_mapping[t] = page*page_size + offset of the token's cache cell; null = nothing is stored.
template <typename T>
__device__ __forceinline__ void rope_kv_store_row(const long token, T* __restrict__ qkv, long ld, int Hq, int Hkv, int dh, int dv,
                                                  const int* __restrict__ positions, const float* __restrict__ inv_freq,
                                                  int rotary_dim, const int* __restrict__ slot_mapping,
                                                  T* __restrict__ k_base, T* __restrict__ v_base, long page_stride,
                                                  int page_size) {
  T* row = qkv + token * ld;
  const float position = (float)positions[token];
  const int half = rotary_dim / 2;
  long cell = -1;
  long page = 0;
  int offset = 0;
  if (slot_mapping) {
    cell = slot_mapping[token];
    page = cell / page_size;
    offset = (int)(cell - page * page_size);
  }
  // q heads then k heads: (head, pair) items
  const int rotary_heads = Hq + Hkv;
  const int pairs = rotary_heads * (dh / 2);   // items cover dh/2 "columns": rotated pairs and pass-through pairs
  for (int item = threadIdx.x; item < pairs; item += blockDim.x) {
    const int head = item / (dh / 2);
    const int j = item - head * (dh / 2);
    T* x = row + (long)head * dh;
    // column j pairs with j+half when j < half; columns >= rotary_dim pass through.
    // Enumerate so that every element of the head is visited exactly once:
    //   j in [0, half): rotated pair (j, j+half)
    //   j in [half, dh/2): pass-through elements (rotary_dim + 2*(j-half)) and the next one
    float a, b;
    int ia, ib;
    if (j < half) {
      ia = j;
      ib = j + half;
      const float x0 = to_float(x[ia]);
      const float x1 = to_float(x[ib]);
      float s = 0.f, c = 1.f;
      if (inv_freq) {
        const float angle = position * inv_freq[j];
        s = sinf(angle);
        c = cosf(angle);
      }
      a = x0 * c - x1 * s;
      b = x1 * c + x0 * s;
    } else {
      ia = rotary_dim + 2 * (j - half);
      ib = ia + 1;
      a = to_float(x[ia]);
      b = to_float(x[ib]);
    }
    if (head < Hq) {
      x[ia] = from_float<T>(a);
      x[ib] = from_float<T>(b);
    } else if (cell >= 0) {
      const int kvh = head - Hq;
      T* dst = k_base + page * page_stride + ((long)kvh * page_size + offset) * dh;
      dst[ia] = from_float<T>(a);
      dst[ib] = from_float<T>(b);
    }
  }
  if (cell >= 0) {
    const T* v = row + (long)(Hq + Hkv) * dh;
    for (int item = threadIdx.x; item < Hkv * dv; item += blockDim.x) {
      const int kvh = item / dv;
      const int i = item - kvh * dv;
      v_base[page * page_stride + ((long)kvh * dv + i) * page_size + offset] = v[item];
    }
  }
}
