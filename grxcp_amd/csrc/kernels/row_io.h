// Element access for the grxDNN row kernels (norms, softmax, GELU): 16-byte
// chunks of bf16 / fp16 / fp32 unpacked to fp32 and packed back with round
// to nearest even, from rows on 16-byte boundaries (AL) or of any element
// alignment and length.
#ifndef GRXCP_ROW_IO_H
#define GRXCP_ROW_IO_H

#include "../launch.h"
#include "device_common.h"

namespace grxk {

template <NormType T> struct Io;  // NormType doubles as the row element type
template <> struct Io<NormType::BF16> {
  static constexpr int kVec = 8;
  __device__ static float ld(const uint8_t* p, int64_t i) { return bf16_to_f32(((const uint16_t*)p)[i]); }
  __device__ static void st(uint8_t* p, int64_t i, float v) { ((uint16_t*)p)[i] = f32_to_bf16(v); }
  __device__ static void unpack(const u32x4 w, float* f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f[2 * q] = __uint_as_float(w[q] << 16);
      f[2 * q + 1] = __uint_as_float(w[q] & 0xffff0000u);
    }
  }
  __device__ static u32x4 pack(const float* f) {
    // v_cvt_pk_bf16_f32: round to nearest even, NaN quieted -- the same
    // bits as f32_to_bf16.
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    u32x4 w;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bf16x2 v = {(__bf16)f[2 * q], (__bf16)f[2 * q + 1]};
      w[q] = __builtin_bit_cast(uint32_t, v);
    }
    return w;
  }
};
template <> struct Io<NormType::F16> {
  static constexpr int kVec = 8;
  __device__ static float ld(const uint8_t* p, int64_t i) { return f16_to_f32(((const uint16_t*)p)[i]); }
  __device__ static void st(uint8_t* p, int64_t i, float v) { ((uint16_t*)p)[i] = f32_to_f16(v); }
  __device__ static void unpack(const u32x4 w, float* f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f[2 * q] = f16_to_f32((uint16_t)(w[q] & 0xffffu));
      f[2 * q + 1] = f16_to_f32((uint16_t)(w[q] >> 16));
    }
  }
  __device__ static u32x4 pack(const float* f) {
    u32x4 w;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      w[q] = (uint32_t)f32_to_f16(f[2 * q]) | ((uint32_t)f32_to_f16(f[2 * q + 1]) << 16);
    return w;
  }
};
template <> struct Io<NormType::F32> {
  static constexpr int kVec = 4;
  __device__ static float ld(const uint8_t* p, int64_t i) { return ((const float*)p)[i]; }
  __device__ static void st(uint8_t* p, int64_t i, float v) { ((float*)p)[i] = v; }
  __device__ static void unpack(const u32x4 w, float* f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) f[q] = __uint_as_float(w[q]);
  }
  __device__ static u32x4 pack(const float* f) {
    u32x4 w;
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = __float_as_uint(f[q]);
    return w;
  }
};

// A chunk at element alignment: one global_load / store_dwordx4, which gfx950
// takes at any address (unaligned access mode, the amdhsa default), at the
// rate of the address's own alignment: softmax of 16384 x 8191 bf16 took 105
// us with unaligned chunks, 16384 x 8001 89 us with its chunks on memory's
// 16-byte boundaries. Plain stores in place of the non-temporal ones: 100.
typedef uint32_t u32x4e __attribute__((ext_vector_type(4), aligned(2)));

// How a row of `hidden` elements falls into chunks. An aligned row (AL)
// starts on 16 bytes and hidden is a multiple of the chunk. Any other row has
// its chunks on the 16-byte boundaries of memory as far as its start allows:
// chunk c holds elements c*V - head .. c*V - head + V - 1, of which the first
// and last chunk may lie partly outside the row. head = elements between the
// boundary before the row and its start (0 where the launch has no room for
// one chunk more, which costs rate, not correctness).
template <NormType T, bool AL>
struct RowChunks {
  static constexpr int V = Io<T>::kVec;
  static constexpr bool kRepeats = false;
  int hidden, head = 0;
  __device__ __forceinline__ RowChunks(const uint8_t* row, int hidden_, int align_mask) : hidden(hidden_) {
    if constexpr (!AL) head = (int)((uintptr_t)row / (16 / V)) & align_mask;
  }
  __device__ __forceinline__ int first(int c) const { return c * V - (AL ? 0 : head); }
  __device__ __forceinline__ bool any(int c) const { return AL ? c < hidden / V : first(c) < hidden; }
  __device__ __forceinline__ bool whole(int c) const {
    return AL ? any(c) : first(c) >= 0 && first(c) + V <= hidden;
  }
  __device__ __forceinline__ bool has(int c, int e) const {
    return AL || (first(c) + e >= 0 && first(c) + e < hidden);
  }

  // Chunk c of a row, `none` in place of the elements outside it. STREAM:
  // non-temporal.
  template <bool STREAM = true>
  __device__ __forceinline__ u32x4 load(const uint8_t* row, int c, u32x4 none) const {
    if (whole(c)) {
      const uint8_t* q = row + (int64_t)first(c) * (16 / V);
      if constexpr (AL && STREAM) return __builtin_nontemporal_load((const u32x4*)q);
      else if constexpr (AL) return *(const u32x4*)q;
      else if constexpr (STREAM) return __builtin_nontemporal_load((const u32x4e*)q);
      else return *(const u32x4e*)q;
    }
    u32x4 w = none;
    if constexpr (!AL) {
      if (any(c)) {
        // Every element's load is issued before the first is used (those
        // outside the row repeat its ends): one latency, where a branch per
        // element would be V (softmax of 16384 x 8001 bf16: 121 us).
        uint32_t u[V];
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const int i = min(max(first(c) + e, 0), hidden - 1);
          if constexpr (V == 4) u[e] = ((const uint32_t*)row)[i];
          else u[e] = ((const uint16_t*)row)[i];
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
          if constexpr (V == 4) w[e] = has(c, e) ? u[e] : none[e];
          else u[e] = has(c, e) ? u[e] : (e & 1) ? none[e >> 1] >> 16 : none[e >> 1] & 0xffffu;
        }
        if constexpr (V == 8)
#pragma unroll
          for (int h = 0; h < 4; ++h) w[h] = u[2 * h] | (u[2 * h + 1] << 16);
      }
    }
    return w;
  }

  // The elements of w that lie in the row, to chunk c.
  __device__ __forceinline__ void store(uint8_t* row, int c, u32x4 w) const {
    if (whole(c)) {
      uint8_t* q = row + (int64_t)first(c) * (16 / V);
      if constexpr (AL) __builtin_nontemporal_store(w, (u32x4*)q);
      else __builtin_nontemporal_store((u32x4e)w, (u32x4e*)q);
    } else if constexpr (!AL) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        if (!has(c, e)) continue;
        if constexpr (V == 4) ((uint32_t*)row)[first(c) + e] = w[e];
        else ((uint16_t*)row)[first(c) + e] = (uint16_t)((e & 1) ? w[e >> 1] >> 16 : w[e >> 1]);
      }
    }
  }
};

// A row of at least V elements at any element alignment as whole chunks: chunk
// c starts at element c*V, but the last one ends with the row and repeats
// elements of the one before it, which `has` leaves to that one (both store the
// same values). Every load and store is one instruction without a branch.
template <NormType T>
struct WholeChunks {
  static constexpr int V = Io<T>::kVec;
  static constexpr bool kRepeats = true;
  int hidden;
  __device__ __forceinline__ WholeChunks(const uint8_t*, int hidden_, int) : hidden(hidden_) {}
  __device__ __forceinline__ int first(int c) const { return min(c * V, hidden - V); }
  __device__ __forceinline__ bool any(int c) const { return c * V < hidden; }
  __device__ __forceinline__ bool whole(int c) const { return c * V + V <= hidden; }
  __device__ __forceinline__ bool has(int c, int e) const { return first(c) + e >= c * V; }
  template <bool STREAM = true>
  __device__ __forceinline__ u32x4 load(const uint8_t* row, int c, u32x4 none) const {
    const u32x4e* q = (const u32x4e*)(row + (int64_t)first(c) * (16 / V));
    if (!any(c)) return none;
    return STREAM ? __builtin_nontemporal_load(q) : *q;
  }
  __device__ __forceinline__ void store(uint8_t* row, int c, u32x4 w) const {
    if (any(c)) __builtin_nontemporal_store((u32x4e)w, (u32x4e*)(row + (int64_t)first(c) * (16 / V)));
  }
};

}  // namespace grxk

#endif  // GRXCP_ROW_IO_H
