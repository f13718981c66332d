// Shared declarations for the MI355X (gfx950) vision-tower kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/mi355_vit.h"

typedef __bf16 bf16_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

#define MVIT_WAVE 64

// Work-groups of 256 threads that one launch can have: the runtime takes fewer than 2^32 threads per grid dimension.
constexpr int64_t MVIT_MAX_GROUPS_256 = (1ll << 24) - 1;

// Records a formatted message for mvit_last_error() and returns `code`.
int mvit_set_error(int code, const char* fmt, ...);

#define MVIT_REQUIRE(cond, ...)                                   \
  do {                                                            \
    if (!(cond)) return mvit_set_error(MVIT_ERR_ARG, __VA_ARGS__); \
  } while (0)

// Checks the launch of the kernel just enqueued (configuration errors only; no sync).
#define MVIT_CHECK_LAUNCH(name)                                                        \
  do {                                                                                 \
    hipError_t e__ = hipGetLastError();                                                \
    if (e__ != hipSuccess)                                                             \
      return mvit_set_error(MVIT_ERR_LAUNCH, "%s launch: %s", name, hipGetErrorString(e__)); \
  } while (0)

static inline bool mvit_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Launches that several steps of a block share (block.cpp).
// Attention over windows of at most 64 tokens with the rotary embedding of q and k inside (bf16, head_dim 80; qkv [S, 3 * nheads * 80]).  The rotated
// q and k replace the others in qkv where `keep` is set, so every window is taken once, in its own place: an order of segments (windows are about
// alike) is not looked at, since one that names a window twice would have it rotated twice.  `mvit_window_rope_takes`: whether a block's tensors suit it.
struct mvit_window_rope {
  void *qkv, *o;
  float* lse;
  const int32_t* cu;
  const float *cos, *sin;
  int n_seg, nheads;
  int64_t S;
  float q_gain, attn_scale;
  bool keep;
};
bool mvit_window_rope_takes(const mvit_window_rope& w, int head_dim, int max_seqlen, int dtype);  // attention.hip
int mvit_attn_fwd_window_rope(const mvit_window_rope& w, hipStream_t stream);                     // attention.hip
// its backward: d_o [S, nheads * 80] -> dqkv [S, 3 * nheads * 80], from the rotated q and k; delta [nheads, S]
int mvit_attn_bwd_window_rope(const mvit_window_rope& w, const void* d_o, void* dqkv, float* delta, hipStream_t stream);
int mvit_gemm_wgrad_group(const mvit_gemm_args* list, int n, hipStream_t stream);  // gemm.hip
struct mvit_partials {  // out[c] = the sum of n_partial rows of `cols` floats, in the order of mvit_reduce_partials
  const float* partial;
  int n_partial;
  int64_t cols;
  void* out;
};
int mvit_reduce_partials_group(const mvit_partials* list, int n, int out_dtype, hipStream_t stream);  // bandwidth.hip

// Per-device host state (function attributes set, compute-unit counts, symbol addresses) is kept in arrays of this
// many slots indexed by the current device's ordinal.
#define MVIT_MAX_DEVICES 64
// Ordinal of the current device, or -1 (with the error recorded) when it cannot be told or has no slot.
static inline int mvit_current_device(const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MVIT_MAX_DEVICES) {
    mvit_set_error(MVIT_ERR_LAUNCH, "%s: hipGetDevice: %s (device %d, %d slots)", who, hipGetErrorString(e), dev, MVIT_MAX_DEVICES);
    return -1;
  }
  return dev;
}

template <typename T>
struct mvit_elem;
template <>
struct mvit_elem<float> {
  static constexpr int vec = 4;  // elements per 16-byte vector
};
template <>
struct mvit_elem<bf16_t> {
  static constexpr int vec = 8;
};

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }
template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) {
  return v;
}
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) {
  return (bf16_t)v;  // round-to-nearest-even
}

// One pair of a rotary embedding, with the roundings spelled out: the passes of their own and the attention that rotates give the same bits
__device__ __forceinline__ void rope_pair(float a, float b, float c0, float c1, float s0, float s1, int backward, float& oa, float& ob) {
  if (!backward) {
    oa = __builtin_fmaf(a, c0, -(b * s0));
    ob = __builtin_fmaf(b, c1, a * s1);
  } else {
    oa = __builtin_fmaf(a, c0, b * s1);
    ob = __builtin_fmaf(b, c1, -(a * s0));
  }
}

// A vector that is not read again before it has left the caches anyway: it does not push out what is
template <typename V>
__device__ __forceinline__ V load_once(const V* p) {
  return __builtin_nontemporal_load(p);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
