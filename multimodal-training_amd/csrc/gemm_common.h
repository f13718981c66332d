// What the GEMM kernels share: launch parameters, tile order, and the epilogue arithmetic on eight consecutive columns.
// Included by gemm.hip inside its anonymous namespace's translation unit only.
#pragma once
#include "mvit_common.h"
#include <type_traits>

struct GemmParams {
  int64_t M, N, K;
  const void* A;
  int64_t lda;
  const void* B;
  const void* B2;
  int64_t ldb;
  const void* bias;
  const void* bias2;
  void* C;
  int64_t ldc;
  const void* R;
  int64_t ldr;
  void* aux;
  int64_t ldaux;
  int64_t aux_off;
  int reduce_epi;  // split_k > 1: the epilogue that the reduction over the K slices applies (none, bias, bias + residual)
  int tiles_m, tiles_n;
  int split_k;        // K slices (1 = none)
  int64_t k_chunk;    // K extent of one slice (multiple of BK)
  float* workspace;   // [split_k][M][N] fp32 partial sums when split_k > 1
  int vec_ok;         // every epilogue pointer / stride allows 16-byte accesses
  int half_vec_ok;    // the output allows 8-byte stores of bf16 (a row pitch that is a multiple of 4 elements only)
  float* colsum;      // SWIGLU_BWD: column sums of the output before rounding, one row per tile row, [tiles_m][ldc] (null: not wanted)
  void* row_sums;     // TT_NONE(_F32), optional: [M] sums of op(A) over k, in the type of C (a bias gradient beside its weight gradient)
  float* row_ws;      // split_k > 1: their partial sums, [split_k][M]
  int group_m, panel_w;  // tiles are walked in groups of this many tile rows, and a group in panels of this many tile columns
  // A operand made from decoded frames (gemm_dl_kernel<..., PIX = true>): image table and the affine form of the
  // rescale / normalise step, value = byte * px_a[channel] + px_c[channel]
  const mvit_image* px_images;
  int px_n_images;
  float px_a[3], px_c[3];
};

// The bf16 products' tile order, for tiles of bm rows (tile_coords): groups of 2,048 rows, 8 x 4 tiles of 256 x 256 per XCD at a time, once
// A is too large to stay in the memory-side cache (256 MB) beside the output from one panel to the next.  us, whole panels -> groups
// (K = 1280): 3840 columns with bias 32,768 rows (A is 84 MB) 257 / 247 -> 258 / 247, 36,864 (94 MB) 299 -> 288, 40,960 333 -> 318, 65,536 557 -> 507;
// SwiGLU 32,768 rows 525 / 511 -> 530 / 528, 36,864 619 -> 587, 40,960 717 -> 628, 65,536 1,143 -> 1,050; SwiGLU backward 394 -> 393, 453 -> 441, 505 -> 489,
// 788 -> 775.  Groups of 1,024, 4,096 and 8,192 rows at 65,536: 552, 535, 549 and 1,040, 1,074, 1,153; panels of eight columns 544, 1,067.
constexpr int64_t TILE_GROUP_BYTES = 88ll << 20;
inline void set_tile_order(GemmParams& p, int bm) {
  p.panel_w = p.tiles_n <= 6 ? p.tiles_n : 4;
  p.group_m = p.tiles_n > p.panel_w && p.M * p.K * 2 > TILE_GROUP_BYTES && 2048 / bm < p.tiles_m ? 2048 / bm : p.tiles_m;
}

// bf16 kernels behind mvit_gemm that live in translation units of their own; gemm.hip chooses (the K slices of a split
// product are reduced there too).  They cover the products of the vision tower, see mvit_gemm_tiled_kind.
enum GemmTiledKind { TILED_NONE = -1, NN_NONE, NN_BIAS, NN_BIAS_RES, NN_BIAS_GELU, NN_SWIGLU, NT_NONE, NT_GELU_BWD, NT_SWIGLU_BWD, TT_NONE, TT_NONE_F32 };
int mvit_gemm_pp(GemmTiledKind kind, const GemmParams& p, int n_cu, hipStream_t stream);                  // gemm_pingpong.hip
// Whether a launch of tiles of bm rows has a wave read B ahead of the main loops (touch_b, gemm_small.hip): a work-group has one of `own_units`
// compute units, which no other stream's work fills, to itself, and there are tile rows enough to share the reading.
inline bool gemm_reads_ahead(GemmTiledKind kind, int bm, int64_t tiles_m, int64_t tiles, int64_t slices, int64_t own_units) {
  return kind != NN_SWIGLU && kind != NT_SWIGLU_BWD && kind != TT_NONE && kind != TT_NONE_F32 && bm < 192 && slices == 1 && tiles_m >= 4 && tiles <= own_units;
}
int mvit_gemm_small(GemmTiledKind kind, int bm, int bn, bool lone, const GemmParams& p, int own_units, hipStream_t stream);  // gemm_small.hip; own_units: compute units that no other stream's work fills

constexpr int GEMM_GROUP_MAX = 4;
struct GemmGroup {
  int n;
  unsigned first_block[GEMM_GROUP_MAX];
  GemmParams p[GEMM_GROUP_MAX];
};
int mvit_gemm_small_group(int bm, int bn, GemmGroup& group, hipStream_t stream);                                // gemm_small.hip

int mvit_gemm_f32(int ta, int tb, int epi, const GemmParams& p, int n_cu, hipStream_t stream);              // gemm_f32.hip

namespace {

// Tile order inside one K slice: groups of group_m tile rows; within a group panels of panel_w tile columns, row by row.  Work-groups
// that run at the same time on one XCD (consecutive tile indices) then cover a compact block of the output, e.g. 8 x 4 tiles, so the
// A and B panels they stream through that XCD's L2 are shared as widely as possible; and a group's rows of A are in the memory-side
// cache when its next panel reads them, where whole panels of tall products read all of A from HBM once per panel.
__device__ __forceinline__ void tile_coords(const GemmParams& p, int tile, int& tm, int& tn) {
  const int pw = p.panel_w;
  int row0 = 0, rows = p.tiles_m;
  if (p.group_m < p.tiles_m) {
    row0 = tile / (p.group_m * p.tiles_n) * p.group_m;
    rows = p.tiles_m - row0 < p.group_m ? p.tiles_m - row0 : p.group_m;
    tile -= row0 * p.tiles_n;
  }
  const int full_panels = p.tiles_n / pw, per_panel = rows * pw;
  if (tile < full_panels * per_panel) {
    const int r = tile % per_panel;
    tm = row0 + r / pw;
    tn = (tile / per_panel) * pw + r % pw;
  } else {
    const int r = tile - full_panels * per_panel, w = p.tiles_n - full_panels * pw;
    tm = row0 + r / w;
    tn = full_panels * pw + r % w;
  }
}

__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752440f)); }
__device__ __forceinline__ float gelu_erf_grad(float z) {
  const float cdf = 0.5f * (1.f + erff(z * 0.70710678118654752440f));
  const float pdf = 0.39894228040143267794f * __expf(-0.5f * z * z);
  return cdf + z * pdf;
}
// 1 / (1 + e^-z) with the hardware reciprocal (1 ulp) instead of the IEEE division sequence
__device__ __forceinline__ float sigmoidf_(float z) { return __builtin_amdgcn_rcpf(1.f + __expf(-z)); }

// 8 consecutive elements <-> fp32 registers
__device__ __forceinline__ void load8(const bf16_t* p, float* v) {
  const bf16x8 x = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (float)x[e];
}
__device__ __forceinline__ void load8(const float* p, float* v) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = a[e];
    v[4 + e] = b[e];
  }
}
template <typename T>
__device__ __forceinline__ void unpack8(const T __attribute__((ext_vector_type(8))) & x, float* v) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (float)x[e];
}
// Epilogue outputs are stored plainly: the two stores that make a 128-byte line meet in the L2, and the next kernels find what fits
// the memory-side cache there.  With the non-temporal hint a launch alone is the faster one where its output does not fit (us plain /
// hinted, 3840 columns with bias of 65,536 rows, 503 MB, 561 / 506, of 14,336 rows 124 / 128; SwiGLU of 25,524 rows 390 / 399), but
// steps are not, whichever outputs take it (65,536 rows: 639 ms either way), and shorter ones lose: ms per step hinted -> plain
// 4,360 rows without gradients 8.56 -> 8.17, 4,096 with checkpointing 30.1 -> 29.4, 14,336 65.9 -> 64.9, 25,524 112.4 -> 111.4.
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store8(bf16_t* p, const float* v) {
  bf16x8 x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (bf16_t)v[e];
  *reinterpret_cast<u32x4_t*>(p) = __builtin_bit_cast(u32x4_t, x);
}
__device__ __forceinline__ void store8(float* p, const float* v) {
  *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<f32x4*>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}
template <typename T>
__device__ __forceinline__ T __attribute__((ext_vector_type(8))) load8_stream(const void* p) {
  typedef T raw8 __attribute__((ext_vector_type(8)));
  if constexpr (sizeof(T) == 2) {
    return __builtin_bit_cast(raw8, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p)));
  } else {
    raw8 r;
    const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
    const f32x4 b = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p) + 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] = a[e];
      r[4 + e] = b[e];
    }
    return r;
  }
}

// Epilogue on 8 consecutive output columns n..n+7 of row m.  v: accumulators (gate half for SWIGLU), u: up half.
// FULL: all 8 columns exist and every pointer allows 16-byte accesses (compile-time trip counts, vector memory
// operations); otherwise a scalar path bounded by the matrix edge.
// PRE: the epilogue's per-element inputs (residual / saved activations) were fetched earlier into pre[0..1].
// hb / hb2: the 8 bias values of columns n .. n+7, already in registers (null: loaded here)
template <typename T, typename TO, int EPI, bool FULL, bool PRE = false>
__device__ __forceinline__ void emit8_impl(const GemmParams& p, int64_t m, int64_t n, float* v, const float* u,
                                           const T __attribute__((ext_vector_type(8))) * pre, float (&cs)[16], bool do_cs,
                                           const float* hb = nullptr, const float* hb2 = nullptr) {
  TO* Cp = static_cast<TO*>(p.C);
  const T* Rp = static_cast<const T*>(p.R);
  T* auxp = static_cast<T*>(p.aux);
  const T* bias = static_cast<const T*>(p.bias);
  const T* bias2 = static_cast<const T*>(p.bias2);
  const int cnt = FULL ? 8 : ((p.N - n) < 8 ? (int)(p.N - n) : 8);
  constexpr bool vec = FULL;

  if constexpr (EPI == MVIT_EPI_BIAS || EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_BIAS_GELU || EPI == MVIT_EPI_SWIGLU) {
    if (hb) {
      for (int e = 0; e < 8; ++e) v[e] += hb[e];
    } else if (bias) {
      float b[8];
      if (vec) load8(bias + n, b);
      else
        for (int e = 0; e < cnt; ++e) b[e] = to_f32(bias[n + e]);
      for (int e = 0; e < cnt; ++e) v[e] += b[e];
    }
  }
  if constexpr (EPI == MVIT_EPI_SWIGLU) {
    float uu[8], h[8];
    for (int e = 0; e < 8; ++e) uu[e] = u[e];
    if (hb2) {
      for (int e = 0; e < 8; ++e) uu[e] += hb2[e];
    } else if (bias2) {
      float b[8];
      if (vec) load8(bias2 + n, b);
      else
        for (int e = 0; e < cnt; ++e) b[e] = to_f32(bias2[n + e]);
      for (int e = 0; e < cnt; ++e) uu[e] += b[e];
    }
    // round g and u to the storage type first: the backward recomputes from those stored values
    for (int e = 0; e < 8; ++e) {
      v[e] = to_f32(from_f32<T>(v[e]));
      uu[e] = to_f32(from_f32<T>(uu[e]));
      h[e] = v[e] * sigmoidf_(v[e]) * uu[e];
    }
    TO* h_out = Cp + m * p.ldc + n;
    if (auxp) {  // a caller that will not differentiate passes no aux and gets the product alone
      T* g_out = auxp + m * p.ldaux + n;
      T* u_out = g_out + p.aux_off;
      if (vec) {
        store8(g_out, v);
        store8(u_out, uu);
      } else {
        for (int e = 0; e < cnt; ++e) {
          g_out[e] = from_f32<T>(v[e]);
          u_out[e] = from_f32<T>(uu[e]);
        }
      }
    }
    if (vec) store8(h_out, h);
    else
      for (int e = 0; e < cnt; ++e) h_out[e] = from_f32<TO>(h[e]);
    return;
  }
  if constexpr (EPI == MVIT_EPI_SWIGLU_BWD) {
    const T* g_in = Rp + m * p.ldr + n;
    const T* u_in = g_in + p.aux_off;
    float g[8], uu[8], dg[8], du[8];
    if (PRE) {
      unpack8<T>(pre[0], g);
      unpack8<T>(pre[1], uu);
    } else if (vec) {
      load8(g_in, g);
      load8(u_in, uu);
    } else {
      for (int e = 0; e < 8; ++e) {
        g[e] = e < cnt ? to_f32(g_in[e]) : 0.f;
        uu[e] = e < cnt ? to_f32(u_in[e]) : 0.f;
      }
    }
    for (int e = 0; e < 8; ++e) {
      const float sg = sigmoidf_(g[e]);
      const float silu = g[e] * sg;
      dg[e] = v[e] * uu[e] * (sg + silu * (1.f - sg));
      du[e] = v[e] * silu;
    }
    if (do_cs) {  // running column sums of this thread's 8 columns (the gate / up bias gradient)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (e < cnt) {
          cs[e] += dg[e];
          cs[8 + e] += du[e];
        }
      }
    }
    TO* dg_out = Cp + m * p.ldc + n;
    TO* du_out = dg_out + p.aux_off;
    if (vec) {
      store8(dg_out, dg);
      store8(du_out, du);
    } else {
      for (int e = 0; e < cnt; ++e) {
        dg_out[e] = from_f32<TO>(dg[e]);
        du_out[e] = from_f32<TO>(du[e]);
      }
    }
    return;
  }
  if constexpr (EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_GELU_BWD) {
    float r[8];
    if (PRE) unpack8<T>(pre[0], r);
    else if (vec) load8(Rp + m * p.ldr + n, r);
    else
      for (int e = 0; e < 8; ++e) r[e] = e < cnt ? to_f32(Rp[m * p.ldr + n + e]) : 0.f;
    for (int e = 0; e < 8; ++e) {
      if constexpr (EPI == MVIT_EPI_BIAS_RES) v[e] += r[e];
      else v[e] *= gelu_erf_grad(r[e]);
    }
  }
  if constexpr (EPI == MVIT_EPI_BIAS_GELU) {
    T* z_out = auxp + m * p.ldaux + n;
    for (int e = 0; e < 8; ++e) v[e] = to_f32(from_f32<T>(v[e]));  // gelu of the stored pre-activation
    if (vec) store8(z_out, v);
    else
      for (int e = 0; e < cnt; ++e) z_out[e] = from_f32<T>(v[e]);
    for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
  }
  TO* c_out = Cp + m * p.ldc + n;
  if constexpr (EPI == MVIT_EPI_ACCUM) {
    float c[8];
    if (vec) load8(c_out, c);
    else
      for (int e = 0; e < 8; ++e) c[e] = e < cnt ? to_f32(c_out[e]) : 0.f;
    for (int e = 0; e < 8; ++e) v[e] += c[e];
  }
  if (vec) store8(c_out, v);
  else
    for (int e = 0; e < cnt; ++e) c_out[e] = from_f32<TO>(v[e]);
}

template <typename T, typename TO, int EPI>
__device__ __forceinline__ void emit8(const GemmParams& p, int64_t m, int64_t n, float* v, const float* u, bool vec,
                                      float (&cs)[16], bool do_cs) {
  if (vec && n + 8 <= p.N) emit8_impl<T, TO, EPI, true>(p, m, n, v, u, nullptr, cs, do_cs);
  else if (EPI == MVIT_EPI_NONE && sizeof(TO) == 2 && p.half_vec_ok && n + 4 <= p.N) {
    TO* c = static_cast<TO*>(p.C) + m * p.ldc + n;
    *reinterpret_cast<bf16x4*>(c) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
    if (n + 8 <= p.N) *reinterpret_cast<bf16x4*>(c + 4) = bf16x4{(bf16_t)v[4], (bf16_t)v[5], (bf16_t)v[6], (bf16_t)v[7]};
    else
      for (int e = 4; n + e < p.N; ++e) c[e] = from_f32<TO>(v[e]);
  }
  else emit8_impl<T, TO, EPI, false>(p, m, n, v, u, nullptr, cs, do_cs);
}

}  // namespace
