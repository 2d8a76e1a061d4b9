// Shared by the gated attention kernels: geometry, the argument block and small helpers.
#pragma once

#include "common.h"

namespace lollm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;

constexpr int AT_D = 256;            // head dim
constexpr int AT_ROWS = 32;          // MFMA rows per pair (n_rep x QB)

struct AttnArgs {
  const uint16_t* q;       // (B, T, Hq, D)
  const uint16_t* kc;      // K cache
  const uint16_t* vc;      // V cache
  const int32_t* kv_len;   // (B) keys per sequence, the T new ones included
  const uint16_t* gate;    // (B, T, Hq * D) or null
  uint16_t* out;           // (B, T, Hq * D)
  float* ws;               // partials: (nw + pairs) x AT_PART, then the combine table
  long long seq_stride, head_stride;  // cache strides in elements
  int B, T, Hq, Hkv, n_rep, QB, qblocks, max_len, nw;
  float cl2;               // scale * log2(e)
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }

// Row groups per wave of the long-call kernel (attn_prefill.hip) for this geometry on a device
// with `cus` CUs, or 0 where the split-K kernels are the faster ones.
int attn_prefill_groups(int B, int T, int Hkv, int n_rep, int cus);
int attn_prefill_launch(const AttnArgs& a, int groups, hipStream_t st);

}  // namespace lollm
