// What the attention kernels share (attention.hip: decode and few query rows; attention_tile.hip:
// prefill): operand types, the call's arguments, output rows and the softmax-state merge.
#pragma once

#include <type_traits>

#include "lr_common.hpp"

namespace lr {

typedef __bf16 attn_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 attn_f16x8 __attribute__((ext_vector_type(8)));
typedef float attn_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned attn_u32x4 __attribute__((ext_vector_type(4)));

constexpr int kAttnWaves = 4;
constexpr int kAttnThreads = 64 * kAttnWaves;
constexpr float kAttnLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();

template <typename T> struct AttnVec;
template <> struct AttnVec<__bf16> {
  using x8 = attn_bf16x8;
  static __device__ __forceinline__ attn_f32x4 mfma(x8 a, x8 b, attn_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct AttnVec<_Float16> {
  using x8 = attn_f16x8;
  static __device__ __forceinline__ attn_f32x4 mfma(x8 a, x8 b, attn_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

struct AttnArgs {
  const void* queries;      // element strides below; the last dimension is contiguous
  int64_t q_batch, q_head, q_query;
  const void* keys;         // [key_rows, D]
  const void* values;       // [key_rows, D]
  int64_t key_rows;
  const int32_t* cu;        // [segments + 1]
  int64_t kv_heads, groups, length;
  int64_t tiles;            // query-row tiles per segment: ceil(L*G / R)
  int64_t splits;           // key chunks per (segment, tile) in the grid
  float scale;
  void* out;                // [B, L, kv_heads * G, D]
  float* part_o;            // [units * splits, R, D]
  float* part_ml;           // [units * splits, R, 2]
  const void* pending_keys;    // NULL, or [segments, D]: a row after each segment's cached rows
  const void* pending_values;  // with pending_keys
};

template <typename T>
__device__ __forceinline__ void unpack8(attn_u32x4 raw, float (&v)[8]) {
  if constexpr (std::is_same<T, __bf16>::value) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = __builtin_bit_cast(float, raw[e] << 16);
      v[2 * e + 1] = __builtin_bit_cast(float, raw[e] & 0xffff0000u);
    }
  } else {
    const attn_f16x8 h = __builtin_bit_cast(attn_f16x8, raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(h[e]);
  }
}

template <typename T>
__device__ __forceinline__ attn_u32x4 pack8(const float (&v)[8]) {
  typename AttnVec<T>::x8 h;
#pragma unroll
  for (int e = 0; e < 8; ++e) h[e] = static_cast<T>(v[e]);  // round to nearest even
  return __builtin_bit_cast(attn_u32x4, h);
}

__device__ __forceinline__ attn_u32x4 load16(const void* p) {
  return *(const __attribute__((address_space(1))) attn_u32x4*)p;
}

// Index arithmetic is unsigned 32-bit (a call has fewer than 2^31 query rows and blocks): the 64-bit
// divisions of a tile's coordinates took over a thousand instructions ahead of the first load.

// Query of row `row` (row = query * G + group).
__device__ __forceinline__ unsigned query_of(const AttnArgs& a, unsigned row) {
  return a.length == 1 ? 0u : row / static_cast<unsigned>(a.groups);
}

// Output row `row` of segment `seg` (query i = row / G, query head h*G + row % G).
template <typename T, int D>
__device__ __forceinline__ T* output_row(const AttnArgs& a, unsigned seg, unsigned row) {
  const unsigned groups = static_cast<unsigned>(a.groups), kv_heads = static_cast<unsigned>(a.kv_heads);
  const unsigned b = seg / kv_heads, h = seg - b * kv_heads;
  const unsigned i = query_of(a, row), g = row - i * groups;
  return static_cast<T*>(a.out) +
         ((static_cast<int64_t>(b) * a.length + i) * (a.kv_heads * a.groups) + h * groups + g) * D;
}

// A value and its copy in the lane 16 (32) away, in both lanes: the row swap of two registers that
// hold it, no LDS round trip. (Inline assembly: with the builtin, a bit cast of its second result as
// a vector element takes the first one in this compiler. The wait states cover a vector instruction
// that has just written the operands.)
struct LanePair {
  float first, second;
};
template <int DISTANCE>
__device__ __forceinline__ LanePair lane_pair(float x) {
  static_assert(DISTANCE == 16 || DISTANCE == 32, "row swaps");
  float a = x, b = x;
  if constexpr (DISTANCE == 16)
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  else
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return {a, b};
}

// A (max, exp-sum, unnormalised output slice) softmax state; merge_into folds another in.
struct MergeState {
  float m, l, o[8];
};

__device__ __forceinline__ void merge_into(MergeState& s, float m, float l, const float (&o)[8]) {
  if (m == kNegInf) return;
  const float mx = fmaxf(s.m, m);
  const float ws = s.m == kNegInf ? 0.f : __builtin_amdgcn_exp2f((s.m - mx) * kAttnLog2e);
  const float wo = __builtin_amdgcn_exp2f((m - mx) * kAttnLog2e);
  s.l = __builtin_fmaf(wo, l, s.l * ws);
#pragma unroll
  for (int e = 0; e < 8; ++e) s.o[e] = __builtin_fmaf(wo, o[e], s.o[e] * ws);
  s.m = mx;
}

}  // namespace lr
