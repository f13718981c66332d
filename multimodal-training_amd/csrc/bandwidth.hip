// HBM-bound kernels of the vision tower: RMSNorm fwd/bwd, rotary embedding, row gather, segment copy,
// pad, cast, column sums.  One wave (64 lanes) owns a row where a row reduction is needed; all global
// accesses are 16-byte vectors along the contiguous dimension whenever shapes allow it.
#include "mvit_common.h"

#include <chrono>

// ------------------------------------------------------------------------------------------------
// RMSNorm forward.  One wave per row, 4 rows per 256-thread block; grid-stride over rows.
// Algorithmic bytes per row: read cols*e, write cols*e (+ the weight once, + 4 B rstd).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rmsnorm_fwd_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                          T* __restrict__ y, float* __restrict__ rstd,
                                                          int64_t rows, int cols, float eps) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  for (int64_t r = wave; r < rows; r += nwaves) {
    const T* xr = x + r * cols;
    T* yr = y + r * cols;
    float ss = 0.f;
    if (VEC) {
      for (int c = lane * V; c < cols; c += 64 * V) {
        vec_t v = *reinterpret_cast<const vec_t*>(xr + c);
#pragma unroll
        for (int j = 0; j < V; ++j) {
          float f = to_f32(v[j]);
          ss += f * f;
        }
      }
    } else {
      for (int c = lane; c < cols; c += 64) {
        float f = to_f32(xr[c]);
        ss += f * f;
      }
    }
    ss = wave_sum(ss);
    const float rs = rsqrtf(ss / (float)cols + eps);
    if (lane == 0) rstd[r] = rs;
    if (VEC) {
      for (int c = lane * V; c < cols; c += 64 * V) {
        vec_t v = *reinterpret_cast<const vec_t*>(xr + c);
        vec_t g = *reinterpret_cast<const vec_t*>(w + c);
        vec_t o;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          // normalise in fp32, round to the storage type, then scale (two roundings, like the reference)
          T n = from_f32<T>(to_f32(v[j]) * rs);
          o[j] = from_f32<T>(to_f32(g[j]) * to_f32(n));
        }
        *reinterpret_cast<vec_t*>(yr + c) = o;
      }
    } else {
      for (int c = lane; c < cols; c += 64) {
        T n = from_f32<T>(to_f32(xr[c]) * rs);
        yr[c] = from_f32<T>(to_f32(w[c]) * to_f32(n));
      }
    }
  }
}

// The same for rows of at most NCH vectors per lane: a row is read once, all its loads in flight at a time, and stays in registers; the next
// row's loads are under way before this one's result is stored.  us for 1280 columns in bf16, before (a second pass over the row) / now: 1,024 rows
// 4.2 / 3.7, 4,096 6.5 / 5.6, 14,336 17.4 / 15.3, 25,524 23.2 / 20.4, 65,536 68 / 59 (5.6 TB/s).
template <typename T, int NCH>
__global__ __launch_bounds__(256) void rmsnorm_fwd_row_kernel(const T* __restrict__ x, const T* __restrict__ w, T* __restrict__ y,
                                                              float* __restrict__ rstd, int64_t rows, int cols, float eps) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  vec_t v[NCH], g[NCH];
  auto load = [&](int64_t row, vec_t (&to)[NCH], const T* from) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (i * 64 + lane) * V;
      if (i < NCH - 1 || c < cols) to[i] = *reinterpret_cast<const vec_t*>(from + row * cols + c);
    }
  };
  load(r, v, x);
  load(0, g, w);
  while (true) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (i < NCH - 1 || (i * 64 + lane) * V < cols) {
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float f = to_f32(v[i][j]);
          ss += f * f;
        }
      }
    ss = wave_sum(ss);
    const float rs = rsqrtf(ss / (float)cols + eps);
    if (lane == 0) rstd[r] = rs;
    vec_t o[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int j = 0; j < V; ++j) {
        // normalise in fp32, round to the storage type, then scale (two roundings, like the reference)
        const T n = from_f32<T>(to_f32(v[i][j]) * rs);
        o[i][j] = from_f32<T>(to_f32(g[i][j]) * to_f32(n));
      }
    const int64_t next = r + nwaves;
    if (next < rows) load(next, v, x);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (i * 64 + lane) * V;
      if (i < NCH - 1 || c < cols) *reinterpret_cast<vec_t*>(y + r * cols + c) = o[i];
    }
    if (next >= rows) return;
    r = next;
  }
}

// RMSNorm backward.  Same row ownership; each block keeps its weight-gradient partial in LDS (fp32 [cols])
// and writes it to dw_partial[blockIdx.x, :] at the end, so the result does not depend on atomics order.
// Algorithmic bytes per row: read dy, x (2*cols*e) [+ dx_add], write dx (cols*e).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void rmsnorm_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ x,
                                                          const T* __restrict__ w, const float* __restrict__ rstd,
                                                          const T* dx_add, T* dx, float* __restrict__ dw_partial,
                                                          int64_t rows, int cols) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  extern __shared__ float dw_lds[];  // [4][cols]
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  float* my_dw = dw_lds + (size_t)wv * cols;
  for (int c = lane; c < cols; c += 64) my_dw[c] = 0.f;
  const int64_t wave = (int64_t)blockIdx.x * 4 + wv;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  const float inv_cols = 1.f / (float)cols;
  for (int64_t r = wave; r < rows; r += nwaves) {
    const T* xr = x + r * cols;
    const T* gr = dy + r * cols;
    const float rs = rstd[r];
    float dot = 0.f;
    if (VEC) {
      for (int c = lane * V; c < cols; c += 64 * V) {
        vec_t xv = *reinterpret_cast<const vec_t*>(xr + c);
        vec_t gv = *reinterpret_cast<const vec_t*>(gr + c);
        vec_t wv_ = *reinterpret_cast<const vec_t*>(w + c);
#pragma unroll
        for (int j = 0; j < V; ++j) dot += to_f32(gv[j]) * to_f32(wv_[j]) * to_f32(xv[j]);
      }
    } else {
      for (int c = lane; c < cols; c += 64) dot += to_f32(gr[c]) * to_f32(w[c]) * to_f32(xr[c]);
    }
    dot = wave_sum(dot) * rs * inv_cols;  // mean(dy*w*xhat)
    if (VEC) {
      for (int c = lane * V; c < cols; c += 64 * V) {
        vec_t xv = *reinterpret_cast<const vec_t*>(xr + c);
        vec_t gv = *reinterpret_cast<const vec_t*>(gr + c);
        vec_t wv_ = *reinterpret_cast<const vec_t*>(w + c);
        vec_t av;
        if (dx_add) av = *reinterpret_cast<const vec_t*>(dx_add + r * cols + c);
        vec_t o;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float xhat = to_f32(xv[j]) * rs;
          const float g = to_f32(gv[j]);
          float d = rs * (g * to_f32(wv_[j]) - xhat * dot);
          if (dx_add) d += to_f32(av[j]);
          o[j] = from_f32<T>(d);
          my_dw[c + j] += g * xhat;
        }
        *reinterpret_cast<vec_t*>(dx + r * cols + c) = o;
      }
    } else {
      for (int c = lane; c < cols; c += 64) {
        const float xhat = to_f32(xr[c]) * rs;
        const float g = to_f32(gr[c]);
        float d = rs * (g * to_f32(w[c]) - xhat * dot);
        if (dx_add) d += to_f32(dx_add[r * cols + c]);
        dx[r * cols + c] = from_f32<T>(d);
        my_dw[c] += g * xhat;
      }
    }
  }
  __syncthreads();
  float* out = dw_partial + (size_t)blockIdx.x * cols;
  for (int c = threadIdx.x; c < cols; c += 256)
    out[c] = dw_lds[c] + dw_lds[cols + c] + dw_lds[2 * (size_t)cols + c] + dw_lds[3 * (size_t)cols + c];
}

// The same for rows of at most NCH vectors per lane: a row's operands are read once, all loads in flight at a time, and a lane's part of the
// weight gradient stays in registers.  Bound by HBM from some thousand rows on; us for 1280 columns with dx_add, before (two passes over the row,
// the weight gradient in LDS) / now: 1,024 rows 7.0 / 5.4, 4,096 14.4 / 13.6, 14,336 34.3 / 30.5, 25,524 55.1 / 52.3, 65,536 130 / 130; with the next row's
// loads under way as well 5.7 / 14.2 / 30.3 / 51.4 / 129, in twice the registers.
// ONCE: the two operands that nothing reads after this pass, dy and x, go past the caches where each is ONCE_BYTES and more, and leave them to what the
// next launches read.  ms per step with / without, paired passes: 14,336 rows -0.29 (0.44 %), 25,524 -0.11, 16,384 checkpointed -0.2; at 4,096 rows, where they are
// in the caches, +0.05.
constexpr int64_t ONCE_BYTES = 24ll << 20;
template <typename T, int NCH, bool ADD, bool ONCE>
__global__ __launch_bounds__(256) void rmsnorm_bwd_row_kernel(const T* __restrict__ dy, const T* __restrict__ x, const T* __restrict__ w,
                                                              const float* __restrict__ rstd, const T* dx_add, T* dx,
                                                              float* __restrict__ dw_partial, int64_t rows, int cols) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  extern __shared__ __attribute__((aligned(16))) float dw_lds[];  // [4][cols]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  const float inv_cols = 1.f / (float)cols;
  float dw[NCH][V];
#pragma unroll
  for (int i = 0; i < NCH; ++i)
#pragma unroll
    for (int j = 0; j < V; ++j) dw[i][j] = 0.f;
  auto mine = [&](int i) { return i < NCH - 1 || (i * 64 + lane) * V < cols; };
  struct Row {
    vec_t x[NCH], g[NCH], a[NCH];
    float rs;
  };
  auto load = [&](int64_t r, Row& to) {
    to.rs = rstd[r];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int64_t at = r * cols + (i * 64 + lane) * V;
      if (mine(i)) {
        to.x[i] = ONCE ? load_once(reinterpret_cast<const vec_t*>(x + at)) : *reinterpret_cast<const vec_t*>(x + at);
        to.g[i] = ONCE ? load_once(reinterpret_cast<const vec_t*>(dy + at)) : *reinterpret_cast<const vec_t*>(dy + at);
        if (ADD) to.a[i] = *reinterpret_cast<const vec_t*>(dx_add + at);
      }
    }
  };
  int64_t r = (int64_t)blockIdx.x * 4 + wv;
  if (r < rows) {
    Row now;
    load(r, now);
    vec_t wt[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      if (mine(i)) wt[i] = *reinterpret_cast<const vec_t*>(w + (i * 64 + lane) * V);
    while (true) {
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (mine(i)) {
#pragma unroll
          for (int j = 0; j < V; ++j) dot += to_f32(now.g[i][j]) * to_f32(wt[i][j]) * to_f32(now.x[i][j]);
        }
      const float rs = now.rs;
      dot = wave_sum(dot) * rs * inv_cols;  // mean(dy*w*xhat)
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (mine(i)) {
          vec_t o;
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const float xhat = to_f32(now.x[i][j]) * rs;
            const float g = to_f32(now.g[i][j]);
            float d = rs * (g * to_f32(wt[i][j]) - xhat * dot);
            if (ADD) d += to_f32(now.a[i][j]);
            o[j] = from_f32<T>(d);
            dw[i][j] += g * xhat;
          }
          *reinterpret_cast<vec_t*>(dx + r * cols + (i * 64 + lane) * V) = o;
        }
      r += nwaves;
      if (r >= rows) break;
      load(r, now);
    }
  }
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (mine(i)) {
#pragma unroll
      for (int q = 0; q < V; q += 4)
        *reinterpret_cast<f32x4*>(dw_lds + (size_t)wv * cols + (i * 64 + lane) * V + q) = f32x4{dw[i][q], dw[i][q + 1], dw[i][q + 2], dw[i][q + 3]};
    }
  __syncthreads();
  float* out = dw_partial + (size_t)blockIdx.x * cols;
  for (int c = threadIdx.x; c < cols; c += 256)
    out[c] = dw_lds[c] + dw_lds[cols + c] + dw_lds[2 * (size_t)cols + c] + dw_lds[3 * (size_t)cols + c];
}

// out[c] = sum_b partial[b, c].  A block owns 32 columns; its 8 row groups each add every 8th partial row
// (fixed order, so the sum is reproducible), then combine through LDS.
template <typename T>
__global__ __launch_bounds__(256) void reduce_partials_kernel(const float* __restrict__ partial, int n_partial,
                                                              int64_t cols, T* __restrict__ out) {
  __shared__ float red[8][33];
  const int cx = threadIdx.x & 31, ry = threadIdx.x >> 5;
  const int64_t c = (int64_t)blockIdx.x * 32 + cx;
  float s = 0.f;
  if (c < cols)
    for (int b = ry; b < n_partial; b += 8) s += partial[(size_t)b * cols + c];
  red[ry][cx] = s;
  __syncthreads();
  if (ry == 0 && c < cols) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) t += red[k][cx];
    out[c] = from_f32<T>(t);
  }
}

// The same sum for cols % 4 == 0: a block owns 16 columns (4 lanes x float4) and 64 row groups, so that a tall
// partial array (1024 rows from the RMSNorm backward) is walked by many short, independent load chains.
template <typename T>
__device__ __forceinline__ void reduce_partials_16(const float* __restrict__ partial, int n_partial, int64_t cols, T* __restrict__ out, int64_t c0) {
  __shared__ float red[64][17];
  const int cx = threadIdx.x & 3, ry = threadIdx.x >> 2;
  const int64_t c = c0 + cx * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (c < cols) {
#pragma unroll 4
    for (int b = ry; b < n_partial; b += 64) s += *reinterpret_cast<const f32x4*>(partial + (size_t)b * cols + c);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[ry][cx * 4 + e] = s[e];
  __syncthreads();
  if (threadIdx.x < 16 && c0 + threadIdx.x < cols) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 64; ++k) t += red[k][threadIdx.x];
    out[c0 + threadIdx.x] = from_f32<T>(t);
  }
}
template <typename T>
__global__ __launch_bounds__(256) void reduce_partials_vec_kernel(const float* __restrict__ partial, int n_partial, int64_t cols, T* __restrict__ out) {
  reduce_partials_16(partial, n_partial, cols, out, (int64_t)blockIdx.x * 16);
}
// several such sums in one launch
constexpr int PARTIALS_GROUP_MAX = 4;
struct PartialsGroup {
  int n, first_block[PARTIALS_GROUP_MAX];
  mvit_partials p[PARTIALS_GROUP_MAX];
};
template <typename T>
__global__ __launch_bounds__(256) void reduce_partials_group_kernel(const PartialsGroup g) {
  int i = 0;
  while (i + 1 < g.n && (int)blockIdx.x >= g.first_block[i + 1]) ++i;
  const mvit_partials& p = g.p[i];
  reduce_partials_16(p.partial, p.n_partial, p.cols, static_cast<T*>(p.out), (int64_t)(blockIdx.x - g.first_block[i]) * 16);
}

// Column sums with 16-byte loads: a block owns 128 columns (16 lanes x 8/4 elements) and 16 row phases.
template <typename T>
__global__ __launch_bounds__(256) void colsum_vec_kernel(const T* __restrict__ x, int64_t ld, int64_t rows, int64_t cols,
                                                         float* __restrict__ partial) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  __shared__ float red[16][16 * V + 1];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t c0 = ((int64_t)blockIdx.x * 16 + tx) * V;
  float acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) acc[j] = 0.f;
  if (c0 < cols) {
    for (int64_t r = (int64_t)blockIdx.y * 16 + ty; r < rows; r += (int64_t)gridDim.y * 16) {
      const vec_t v = *reinterpret_cast<const vec_t*>(x + r * ld + c0);
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] += to_f32(v[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) red[ty][tx * V + j] = acc[j];
  __syncthreads();
  if (threadIdx.x < 16 * V) {
    const int64_t c = (int64_t)blockIdx.x * 16 * V + threadIdx.x;
    if (c < cols) {
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < 16; ++k) t += red[k][threadIdx.x];
      partial[(size_t)blockIdx.y * cols + c] = t;
    }
  }
}

// Column sums: block b accumulates rows b, b+grid, ... ; thread owns columns.  Partials [grid, cols].
template <typename T>
__global__ __launch_bounds__(256) void colsum_kernel(const T* __restrict__ x, int64_t ld, int64_t rows, int64_t cols,
                                                     float* __restrict__ partial) {
  // blockIdx.x: column chunk of 256*2 columns; blockIdx.y: row slice
  const int64_t c0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 2;
  if (c0 >= cols) return;
  const bool two = (c0 + 1 < cols);
  float s0 = 0.f, s1 = 0.f;
  for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
    const T* p = x + r * ld + c0;
    s0 += to_f32(p[0]);
    if (two) s1 += to_f32(p[1]);
  }
  partial[(size_t)blockIdx.y * cols + c0] = s0;
  if (two) partial[(size_t)blockIdx.y * cols + c0 + 1] = s1;
}

// ------------------------------------------------------------------------------------------------
// Rotary embedding in place.  A thread owns V consecutive elements of the first half of one head and
// the matching V of the second half.  Algorithmic bytes per (row, head): 2*head_dim*e + table share.
// The first `lead_heads` heads are multiplied by `lead_scale` before the one rounding to the storage type (the
// queries of an attention layer take the softmax scale here, so that no later pass rounds them a second time).
template <typename T>
__global__ __launch_bounds__(256) void rope_kernel(T* __restrict__ x, const float* __restrict__ cosb, const float* __restrict__ sinb, int64_t rows,
                                                   int nheads, int head_dim, int64_t row_stride, int backward, int lead_heads, float lead_scale) {
  const int half = head_dim / 2;
  const int64_t total = rows * nheads * half;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int j = (int)(i % half);
    const int64_t rh = i / half;
    const int h = (int)(rh % nheads);
    const int64_t r = rh / nheads;
    T* p = x + r * row_stride + (int64_t)h * head_dim + j;
    const float* c = cosb + r * head_dim + j;
    const float* s = sinb + r * head_dim + j;
    float oa, ob;
    rope_pair(to_f32(p[0]), to_f32(p[half]), c[0], c[half], s[0], s[half], backward, oa, ob);
    const float gain = h < lead_heads ? lead_scale : 1.f;
    p[0] = from_f32<T>(oa * gain);
    p[half] = from_f32<T>(ob * gain);
  }
}

// The same on vectors: a thread takes one chunk of V pairs of every `groups`-th head of a row, whose angles it reads once, with the loads
// of ROPE_HEADS heads in flight.  Bound by HBM (bytes of x twice, angles once); a thread per chunk of a head, which read its angles for one head
// each and found its place by 64-bit divisions, took, us at 1,024 / 4,096 / 25,524 / 65,536 rows of 32 heads of 80 (row pitch 3840), 5.0 / 12.2 /
// 60.6 / 145; this 4.5 / 11.5 / 54.1 / 139, with four heads in flight 4.5 / 11.3 / 53.1 / 140, with eight 4.5 / 12.5 / 56 / 142.
constexpr int ROPE_HEADS = 2;
template <typename T>
__global__ __launch_bounds__(256) void rope_vec_kernel(T* __restrict__ x, const float* __restrict__ cosb, const float* __restrict__ sinb, int64_t rows,
                                                       int nheads, int head_dim, int64_t row_stride, int backward, int lead_heads, float lead_scale,
                                                       int chunks, int groups) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int half = head_dim / 2, per_row = chunks * groups, rows_here = 256 / per_row;
  const int row = threadIdx.x / per_row, at = threadIdx.x - row * per_row, first = at / chunks, ch = at - first * chunks;
  if (row >= rows_here) return;
  for (int64_t r = (int64_t)blockIdx.x * rows_here + row; r < rows; r += (int64_t)gridDim.x * rows_here) {
    const float* c = cosb + r * head_dim + ch * V;
    const float* s = sinb + r * head_dim + ch * V;
    float c0[V], c1[V], s0[V], s1[V];
#pragma unroll
    for (int j = 0; j < V; ++j) c0[j] = c[j], c1[j] = c[j + half], s0[j] = s[j], s1[j] = s[j + half];
    for (int h0 = first; h0 < nheads; h0 += ROPE_HEADS * groups) {
      T* p = x + r * row_stride + (int64_t)h0 * head_dim + ch * V;
      const int64_t step = (int64_t)groups * head_dim;
      vec_t lo[ROPE_HEADS], hi[ROPE_HEADS];
#pragma unroll
      for (int k = 0; k < ROPE_HEADS; ++k)
        if (h0 + k * groups < nheads) {
          lo[k] = *reinterpret_cast<const vec_t*>(p + k * step);
          hi[k] = *reinterpret_cast<const vec_t*>(p + k * step + half);
        }
#pragma unroll
      for (int k = 0; k < ROPE_HEADS; ++k)
        if (h0 + k * groups < nheads) {
          const float gain = h0 + k * groups < lead_heads ? lead_scale : 1.f;
          vec_t olo, ohi;
#pragma unroll
          for (int j = 0; j < V; ++j) {
            float oa, ob;
            rope_pair(to_f32(lo[k][j]), to_f32(hi[k][j]), c0[j], c1[j], s0[j], s1[j], backward, oa, ob);
            olo[j] = from_f32<T>(oa * gain);
            ohi[j] = from_f32<T>(ob * gain);
          }
          *reinterpret_cast<vec_t*>(p + k * step) = olo;
          *reinterpret_cast<vec_t*>(p + k * step + half) = ohi;
        }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Row gather / segment copy: pure byte movement in 16-byte (or 4-byte) words.
template <typename W>
__global__ __launch_bounds__(256) void gather_rows_kernel(const W* __restrict__ src, const int64_t* __restrict__ index,
                                                          W* __restrict__ dst, int64_t n_rows, int64_t row_words) {
  // blockIdx.y strides over rows; threads over words
  for (int64_t r = blockIdx.y; r < n_rows; r += gridDim.y) {
    const W* s = src + index[r] * row_words;
    W* d = dst + r * row_words;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < row_words; c += (int64_t)gridDim.x * 256) d[c] = s[c];
  }
}

template <typename W>
__global__ __launch_bounds__(256) void segment_copy_kernel(const W* __restrict__ src, W* __restrict__ dst,
                                                           const int64_t* __restrict__ desc, int64_t row_words) {
  // blockIdx.z: segment; blockIdx.y strides over the segment's rows
  const int64_t* d3 = desc + 3 * (int64_t)blockIdx.z;
  const int64_t s0 = d3[0], d0 = d3[1], n = d3[2];
  for (int64_t r = blockIdx.y; r < n; r += gridDim.y) {
    const W* s = src + (s0 + r) * row_words;
    W* d = dst + (d0 + r) * row_words;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < row_words; c += (int64_t)gridDim.x * 256) d[c] = s[c];
  }
}

// Copies of contiguous byte ranges, the list being a kernel argument: nothing has to reach the device in front of the launch.
// A work-group moves one 32 KiB piece; every thread has eight independent 16-byte loads in flight.  HBM-bound.
// A launch's loads and stores carry the non-temporal hint by what it moves in all (COPY_NT_LOADS, COPY_NT_STORES): a source that
// is read once only pushes the destination out of the 256 MB memory-side cache, and a destination that fills most of it is gone
// before its reader comes.  us of a copy and a copy of the result, 16 ranges, plain / hinted loads / both hints: 64 MiB 48.6 / 46.6 / -, 72 57.2 / 51.4 / -,
// 96 75.1 / 69.3 / 70.3, 128 107 / 87.8 / 90.5, 144 115 / 102 / 100, 160 121 / 113 / 110, 192 144 / 133 / 131, 256 190 / 170 / 172, 320 239 / 227 / 213.  Below 64 MiB hinted loads gain or lose
// with the pattern, so there they are plain: these pairs 48 MiB 42.1 / 37.5, split over ranks and put together again 39 MiB 33.4 / 36.6, 40 MiB a rank 51.6 / 56.
constexpr int COPY_MAX_RANGES = 96, COPY_STEPS = 8, COPY_PIECE = 256 * COPY_STEPS;  // words per piece
constexpr int64_t COPY_NT_LOADS = 64ll << 20, COPY_NT_STORES = 160ll << 20;         // bytes of a launch
struct CopyRanges {
  int n;
  int first_piece[COPY_MAX_RANGES];
  const void* src[COPY_MAX_RANGES];
  void* dst[COPY_MAX_RANGES];
  int64_t words[COPY_MAX_RANGES];
};
template <typename W, bool NT_LOADS, bool NT_STORES>
__global__ __launch_bounds__(256) void copy_ranges_kernel(const CopyRanges a) {
  int lo = 0, hi = a.n;  // invariant: first_piece[lo] <= blockIdx.x < first_piece[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((int)blockIdx.x >= a.first_piece[mid]) lo = mid;
    else hi = mid;
  }
  const int64_t begin = (int64_t)(blockIdx.x - a.first_piece[lo]) * COPY_PIECE + threadIdx.x, words = a.words[lo];
  const W* s = static_cast<const W*>(a.src[lo]) + begin;
  W* d = static_cast<W*>(a.dst[lo]) + begin;
  auto load = [&](int i) { return NT_LOADS ? __builtin_nontemporal_load(s + i * 256) : s[i * 256]; };
  auto store = [&](int i, W v) {
    if (NT_STORES) __builtin_nontemporal_store(v, d + i * 256);
    else d[i * 256] = v;
  };
  if (begin - (int64_t)threadIdx.x + COPY_PIECE <= words) {
    W v[COPY_STEPS];
#pragma unroll
    for (int i = 0; i < COPY_STEPS; ++i) v[i] = load(i);
#pragma unroll
    for (int i = 0; i < COPY_STEPS; ++i) store(i, v[i]);
  } else {
#pragma unroll
    for (int i = 0; i < COPY_STEPS; ++i)
      if (begin + i * 256 < words) store(i, load(i));
  }
}

template <typename E>
__global__ __launch_bounds__(256) void pad_pack_kernel(const E* __restrict__ pack, E* __restrict__ padded,
                                                       uint8_t* __restrict__ mask, const int64_t* __restrict__ lens,
                                                       const int64_t* __restrict__ offsets, int64_t pad_len,
                                                       int64_t row_elems, E pad_value) {
  const int64_t b = blockIdx.z;
  const int64_t len = lens[b], off = offsets[b];
  for (int64_t r = blockIdx.y; r < pad_len; r += gridDim.y) {
    E* d = padded + (b * pad_len + r) * row_elems;
    const bool real = r < len;
    const E* s = pack + (off + (real ? r : 0)) * row_elems;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < row_elems; c += (int64_t)gridDim.x * 256)
      d[c] = real ? s[c] : pad_value;
    if (blockIdx.x == 0 && threadIdx.x == 0) mask[b * pad_len + r] = real ? 1 : 0;
  }
}

template <typename S, typename D>
__global__ __launch_bounds__(256) void cast2d_kernel(const S* __restrict__ src, int64_t src_ld, D* __restrict__ dst,
                                                     int64_t dst_ld, int64_t rows, int64_t cols) {
  for (int64_t r = blockIdx.y; r < rows; r += gridDim.y)
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < cols; c += (int64_t)gridDim.x * 256)
      dst[r * dst_ld + c] = from_f32<D>(to_f32(src[r * src_ld + c]));
}

// ------------------------------------------------------------------------------------------------
static inline hipStream_t S_(mvit_stream_t s) { return reinterpret_cast<hipStream_t>(s); }
// ------------------------------------------------------------------------------------------------
// Vision -> text hand-off: where the token ids equal the image placeholder, the rows of the text embedding are
// replaced by the vision rows, the k-th placeholder taking vision row k (masked_scatter with a row mask).
// One work-group ranks the placeholders, 8,192 tokens at a time, each of its 16 waves a contiguous 512 of them: all eight loads of a
// lane are in flight at once, the placeholders among 64 tokens are a ballot kept in registers, and the waves' counts are scanned
// through LDS.  The row merge is then a pure byte copy.  Bound by the latency of the loads (cold in place) and of the counts' way to
// host memory: 7,405 tokens 7.8 us in place, 12.4 with a contiguous slice of all tokens per wave walked twice, 6.6 either way with the
// ids in the cache; 20,480 there 11.2 / 13.2.
constexpr int RANK_STEPS = 8;
__global__ __launch_bounds__(1024) void image_token_ranks_kernel(const int64_t* __restrict__ ids, const int64_t* __restrict__ labels,
                                                                 int64_t n, int64_t image_id, int64_t ignore_label,
                                                                 int32_t* __restrict__ rank, int64_t* __restrict__ positions,
                                                                 int64_t* __restrict__ counts) {
  __shared__ int found[2][16], wrong[16];  // found: of this span and of the one before, which slower waves may still read
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int before = 0, bad = 0, buf = 0;
  for (int64_t base = 0; base < n; base += 1024 * RANK_STEPS, buf ^= 1) {
    const int64_t first = base + wave * (64 * RANK_STEPS) + lane;
    int64_t id[RANK_STEPS], label[RANK_STEPS];
#pragma unroll
    for (int s = 0; s < RANK_STEPS; ++s) {
      const int64_t i = first + s * 64, at = i < n ? i : n - 1;
      id[s] = ids[at];
      label[s] = labels != nullptr ? labels[at] : ignore_label;
    }
    unsigned long long is_image[RANK_STEPS];
    int cnt = 0;
#pragma unroll
    for (int s = 0; s < RANK_STEPS; ++s) {
      const bool img = first + s * 64 < n && id[s] == image_id;
      is_image[s] = __ballot(img);
      cnt += __popcll(is_image[s]);
      bad += __popcll(__ballot(img && label[s] != ignore_label));
    }
    if (lane == 0) found[buf][wave] = cnt;
    __syncthreads();
    int k = before;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int f = found[buf][w];
      if (w < wave) k += f;
      before += f;
    }
#pragma unroll
    for (int s = 0; s < RANK_STEPS; ++s) {
      const int64_t i = first + s * 64;
      const bool img = (is_image[s] >> lane) & 1;
      const int mine = k + __popcll(is_image[s] & ((1ull << lane) - 1));
      if (i < n) rank[i] = img ? mine : -1;
      if (img && positions != nullptr) positions[mine] = i;
      k += __popcll(is_image[s]);
    }
  }
  if (lane == 0) wrong[wave] = bad;
  __syncthreads();
  if (threadIdx.x == 0) {
    int all_bad = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) all_bad += wrong[w];
    counts[0] = before;
    counts[1] = all_bad;
  }
}

// Backward of the merge in one pass over the gradient: a placeholder's row goes to its vision row and leaves zeros in the text
// gradient, any other row stays text gradient.
template <typename W>
__global__ __launch_bounds__(256) void split_rows_kernel(const W* __restrict__ grad, const int32_t* __restrict__ rank, W* __restrict__ text,
                                                         W* __restrict__ vision, int64_t n_rows, int64_t n_vision, int64_t row_words) {
  for (int64_t r = blockIdx.y; r < n_rows; r += gridDim.y) {
    const int k = rank[r];
    const bool img = k >= 0 && k < n_vision;
    if (img ? vision == nullptr && text == nullptr : text == nullptr) continue;
    const W* g = grad + r * row_words;
    W *v = img && vision ? vision + (int64_t)k * row_words : nullptr, *t = text ? text + r * row_words : nullptr;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < row_words; c += (int64_t)gridDim.x * 256) {
      if (img) {
        if (v) v[c] = g[c];
        if (t) t[c] = W{};
      } else {
        t[c] = g[c];
      }
    }
  }
}

template <typename W>
__global__ __launch_bounds__(256) void merge_rows_kernel(const W* __restrict__ embeds, const W* __restrict__ vision,
                                                         const int32_t* __restrict__ rank, W* __restrict__ merged, int64_t n_rows,
                                                         int64_t n_vision, int64_t row_words) {
  for (int64_t r = blockIdx.y; r < n_rows; r += gridDim.y) {
    const int k = rank[r];
    const bool img = k >= 0 && k < n_vision;  // a rank beyond the vision rows keeps the text row (the caller has refused that case)
    const W* s = img ? (vision ? vision + (int64_t)k * row_words : nullptr) : embeds + r * row_words;
    W* d = merged + r * row_words;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < row_words; c += (int64_t)gridDim.x * 256) d[c] = s ? s[c] : W{};
  }
}

static inline int clamp_grid(int64_t v, int64_t hi) { return (int)(v < 1 ? 1 : (v > hi ? hi : v)); }

template <typename T>
static void launch_rope(T* x, const float* cosb, const float* sinb, int64_t rows, int nheads, int head_dim, int64_t row_stride, int backward,
                        int lead_heads, float lead_scale, hipStream_t stream) {
  constexpr int V = mvit_elem<T>::vec;
  const int half = head_dim / 2, chunks = half / V;
  if (half % V == 0 && chunks <= 256 && row_stride % V == 0 && mvit_aligned16(x)) {
    const int want = (nheads + ROPE_HEADS - 1) / ROPE_HEADS, groups = want * chunks <= 256 ? want : 256 / chunks, rows_here = 256 / (chunks * groups);
    const int grid = clamp_grid((rows + rows_here - 1) / rows_here, MVIT_MAX_GROUPS_256);
    hipLaunchKernelGGL((rope_vec_kernel<T>), grid, 256, 0, stream, x, cosb, sinb, rows, nheads, head_dim, row_stride, backward, lead_heads, lead_scale, chunks, groups);
  } else {
    const int grid = clamp_grid((rows * nheads * half + 255) / 256, 65535 * 16);
    hipLaunchKernelGGL((rope_kernel<T>), grid, 256, 0, stream, x, cosb, sinb, rows, nheads, head_dim, row_stride, backward, lead_heads, lead_scale);
  }
}

// A row in registers: the kernel of that many vectors per lane, null where a row is longer
template <typename T>
static auto rms_fwd_row(int64_t cols) -> decltype(&rmsnorm_fwd_row_kernel<T, 1>) {
  switch ((cols + 64 * mvit_elem<T>::vec - 1) / (64 * mvit_elem<T>::vec)) {
    case 1: return rmsnorm_fwd_row_kernel<T, 1>;
    case 2: return rmsnorm_fwd_row_kernel<T, 2>;
    case 3: return rmsnorm_fwd_row_kernel<T, 3>;
    case 4: return rmsnorm_fwd_row_kernel<T, 4>;
    case 5: return rmsnorm_fwd_row_kernel<T, 5>;
    default: return nullptr;
  }
}
template <typename T, bool ADD, bool ONCE>
static auto rms_bwd_row(int64_t cols) -> decltype(&rmsnorm_bwd_row_kernel<T, 1, ADD, ONCE>) {
  switch ((cols + 64 * mvit_elem<T>::vec - 1) / (64 * mvit_elem<T>::vec)) {
    case 1: return rmsnorm_bwd_row_kernel<T, 1, ADD, ONCE>;
    case 2: return rmsnorm_bwd_row_kernel<T, 2, ADD, ONCE>;
    case 3: return rmsnorm_bwd_row_kernel<T, 3, ADD, ONCE>;
    case 4: return rmsnorm_bwd_row_kernel<T, 4, ADD, ONCE>;
    case 5: return rmsnorm_bwd_row_kernel<T, 5, ADD, ONCE>;
    default: return nullptr;
  }
}

int mvit_reduce_partials_group(const mvit_partials* list, int n, int out_dtype, hipStream_t stream) {
  bool together = n >= 2 && n <= PARTIALS_GROUP_MAX && (out_dtype == MVIT_BF16 || out_dtype == MVIT_F32);
  for (int i = 0; i < n; ++i) together = together && list[i].partial && list[i].out && list[i].n_partial > 0 && list[i].cols > 0 && list[i].cols % 4 == 0 && mvit_aligned16(list[i].partial);
  if (!together) {
    for (int i = 0; i < n; ++i)
      if (int rc = mvit_reduce_partials(list[i].partial, list[i].n_partial, list[i].cols, list[i].out, out_dtype, stream)) return rc;
    return MVIT_OK;
  }
  PartialsGroup g = {};
  g.n = n;
  int blocks = 0;
  for (int i = 0; i < n; ++i) {
    g.p[i] = list[i];
    g.first_block[i] = blocks;
    blocks += (int)((list[i].cols + 15) / 16);
  }
  if (out_dtype == MVIT_BF16) hipLaunchKernelGGL((reduce_partials_group_kernel<bf16_t>), blocks, 256, 0, stream, g);
  else hipLaunchKernelGGL((reduce_partials_group_kernel<float>), blocks, 256, 0, stream, g);
  MVIT_CHECK_LAUNCH("reduce_partials");
  return MVIT_OK;
}

extern "C" {

int mvit_rmsnorm_fwd(const void* x, const void* w, void* y, float* rstd, int64_t rows, int64_t cols, float eps,
                     int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(rows >= 0 && cols > 0 && cols < (1 << 24), "rmsnorm_fwd: bad shape %lld x %lld", (long long)rows, (long long)cols);
  if (rows == 0) return MVIT_OK;
  MVIT_REQUIRE(x && w && y && rstd, "rmsnorm_fwd: null pointer");
  auto go = [&](auto zero) -> void {
    using T = decltype(zero);
    const bool vec = cols % mvit_elem<T>::vec == 0 && mvit_aligned16(x) && mvit_aligned16(y) && mvit_aligned16(w);
    auto kern = rms_fwd_row<T>(cols);
    if (!vec) kern = rmsnorm_fwd_kernel<T, false>;
    else if (kern == nullptr) kern = rmsnorm_fwd_kernel<T, true>;
    hipLaunchKernelGGL(kern, clamp_grid((rows + 3) / 4, 8192), 256, 0, S_(stream), (const T*)x, (const T*)w, (T*)y, rstd, rows, (int)cols, eps);
  };
  if (dtype == MVIT_BF16) go(bf16_t{});
  else if (dtype == MVIT_F32) go(float{});
  else return mvit_set_error(MVIT_ERR_UNSUPPORTED, "rmsnorm_fwd: dtype %d", dtype);
  MVIT_CHECK_LAUNCH("rmsnorm_fwd");
  return MVIT_OK;
}

int mvit_rmsnorm_bwd(const void* dy, const void* x, const void* w, const float* rstd, const void* dx_add, void* dx,
                     float* dw_partial, int n_partial, int64_t rows, int64_t cols, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(dw_partial && w && (rows == 0 || (dy && x && rstd && dx)), "rmsnorm_bwd: null pointer");  // no rows: only the partial sums are written (zeros)
  MVIT_REQUIRE(rows >= 0 && cols > 0 && n_partial > 0, "rmsnorm_bwd: bad shape");
  const size_t lds = 4 * (size_t)cols * sizeof(float);
  MVIT_REQUIRE(lds <= 160 * 1024, "rmsnorm_bwd: cols %lld needs %zu B of LDS (> 160 KiB)", (long long)cols, lds);
  const int grid = n_partial;  // every block writes its partial row, rows or not
  bool al = mvit_aligned16(dy) && mvit_aligned16(x) && mvit_aligned16(w) && mvit_aligned16(dx) && (!dx_add || mvit_aligned16(dx_add));
  auto go = [&](auto zero) -> void {
    using T = decltype(zero);
    const bool vec = cols % mvit_elem<T>::vec == 0 && al;
    const bool once = rows * cols * (int64_t)sizeof(T) >= ONCE_BYTES;
    auto kern = !dx_add ? rms_bwd_row<T, false, false>(cols) : once ? rms_bwd_row<T, true, true>(cols) : rms_bwd_row<T, true, false>(cols);
    if (!vec) kern = rmsnorm_bwd_kernel<T, false>;
    else if (kern == nullptr) kern = rmsnorm_bwd_kernel<T, true>;
    hipLaunchKernelGGL(kern, grid, 256, lds, S_(stream), (const T*)dy, (const T*)x, (const T*)w, rstd, (const T*)dx_add, (T*)dx, dw_partial, rows, (int)cols);
  };
  if (dtype == MVIT_BF16) go(bf16_t{});
  else if (dtype == MVIT_F32) go(float{});
  else return mvit_set_error(MVIT_ERR_UNSUPPORTED, "rmsnorm_bwd: dtype %d", dtype);
  MVIT_CHECK_LAUNCH("rmsnorm_bwd");
  return MVIT_OK;
}

int mvit_reduce_partials(const float* partial, int n_partial, int64_t cols, void* out, int out_dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(partial && out && n_partial > 0 && cols > 0, "reduce_partials: bad arguments");
  if (cols % 4 == 0 && mvit_aligned16(partial) && (out_dtype == MVIT_BF16 || out_dtype == MVIT_F32)) {
    const int vgrid = (int)((cols + 15) / 16);
    if (out_dtype == MVIT_BF16)
      hipLaunchKernelGGL((reduce_partials_vec_kernel<bf16_t>), vgrid, 256, 0, S_(stream), partial, n_partial, cols, (bf16_t*)out);
    else
      hipLaunchKernelGGL((reduce_partials_vec_kernel<float>), vgrid, 256, 0, S_(stream), partial, n_partial, cols, (float*)out);
    MVIT_CHECK_LAUNCH("reduce_partials");
    return MVIT_OK;
  }
  const int grid = (int)((cols + 31) / 32);
  if (out_dtype == MVIT_BF16)
    hipLaunchKernelGGL((reduce_partials_kernel<bf16_t>), grid, 256, 0, S_(stream), partial, n_partial, cols, (bf16_t*)out);
  else if (out_dtype == MVIT_F32)
    hipLaunchKernelGGL((reduce_partials_kernel<float>), grid, 256, 0, S_(stream), partial, n_partial, cols, (float*)out);
  else
    return mvit_set_error(MVIT_ERR_UNSUPPORTED, "reduce_partials: dtype %d", out_dtype);
  MVIT_CHECK_LAUNCH("reduce_partials");
  return MVIT_OK;
}

int mvit_colsum(const void* x, int64_t ld, int64_t rows, int64_t cols, float* partial, int n_partial, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE((x || rows == 0) && partial && n_partial > 0 && n_partial <= 65535 && cols > 0 && rows >= 0 && ld >= cols, "colsum: bad arguments");
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "colsum: dtype %d", dtype);
  const int vec = dtype == MVIT_BF16 ? 8 : 4;
  if (cols % vec == 0 && ld % vec == 0 && mvit_aligned16(x)) {
    dim3 grid((unsigned)((cols + 16 * vec - 1) / (16 * vec)), (unsigned)n_partial);
    if (dtype == MVIT_BF16)
      hipLaunchKernelGGL((colsum_vec_kernel<bf16_t>), grid, 256, 0, S_(stream), (const bf16_t*)x, ld, rows, cols, partial);
    else
      hipLaunchKernelGGL((colsum_vec_kernel<float>), grid, 256, 0, S_(stream), (const float*)x, ld, rows, cols, partial);
  } else {
    dim3 grid((unsigned)((cols + 511) / 512), (unsigned)n_partial);
    if (dtype == MVIT_BF16)
      hipLaunchKernelGGL((colsum_kernel<bf16_t>), grid, 256, 0, S_(stream), (const bf16_t*)x, ld, rows, cols, partial);
    else
      hipLaunchKernelGGL((colsum_kernel<float>), grid, 256, 0, S_(stream), (const float*)x, ld, rows, cols, partial);
  }
  MVIT_CHECK_LAUNCH("colsum");
  return MVIT_OK;
}

int mvit_rope(void* x, const float* cosb, const float* sinb, int64_t rows, int nheads, int head_dim, int64_t row_stride,
              int backward, int dtype, mvit_stream_t stream) {
  return mvit_rope_scaled(x, cosb, sinb, rows, nheads, head_dim, row_stride, backward, 0, 1.f, dtype, stream);
}

int mvit_rope_scaled(void* x, const float* cosb, const float* sinb, int64_t rows, int nheads, int head_dim, int64_t row_stride,
                     int backward, int lead_heads, float lead_scale, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(lead_heads >= 0 && lead_heads <= nheads, "rope: lead_heads=%d of %d heads", lead_heads, nheads);
  MVIT_REQUIRE(rows >= 0 && nheads > 0 && head_dim > 0 && head_dim % 2 == 0 && row_stride >= (int64_t)nheads * head_dim,
               "rope: bad shape rows=%lld heads=%d head_dim=%d stride=%lld", (long long)rows, nheads, head_dim, (long long)row_stride);
  if (rows == 0) return MVIT_OK;
  MVIT_REQUIRE(x && cosb && sinb, "rope: null pointer");
  if (dtype == MVIT_BF16) launch_rope((bf16_t*)x, cosb, sinb, rows, nheads, head_dim, row_stride, backward, lead_heads, lead_scale, S_(stream));
  else if (dtype == MVIT_F32) launch_rope((float*)x, cosb, sinb, rows, nheads, head_dim, row_stride, backward, lead_heads, lead_scale, S_(stream));
  else return mvit_set_error(MVIT_ERR_UNSUPPORTED, "rope: dtype %d", dtype);
  MVIT_CHECK_LAUNCH("rope");
  return MVIT_OK;
}

int mvit_gather_rows(const void* src, const int64_t* index, void* dst, int64_t n_rows, int64_t row_bytes, mvit_stream_t stream) {
  MVIT_REQUIRE(n_rows >= 0 && row_bytes > 0 && row_bytes % 2 == 0, "gather_rows: row_bytes %lld must be a positive multiple of 2", (long long)row_bytes);
  if (n_rows == 0) return MVIT_OK;
  MVIT_REQUIRE(src && index && dst, "gather_rows: null pointer");
  const unsigned gy = (unsigned)clamp_grid(n_rows, 65535);
  if (row_bytes % 16 == 0 && mvit_aligned16(src) && mvit_aligned16(dst)) {
    const int64_t words = row_bytes / 16;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((gather_rows_kernel<u32x4>), grid, 256, 0, S_(stream), (const u32x4*)src, index, (u32x4*)dst, n_rows, words);
  } else if (row_bytes % 4 == 0) {
    const int64_t words = row_bytes / 4;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((gather_rows_kernel<uint32_t>), grid, 256, 0, S_(stream), (const uint32_t*)src, index, (uint32_t*)dst, n_rows, words);
  } else {
    const int64_t words = row_bytes / 2;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((gather_rows_kernel<uint16_t>), grid, 256, 0, S_(stream), (const uint16_t*)src, index, (uint16_t*)dst, n_rows, words);
  }
  MVIT_CHECK_LAUNCH("gather_rows");
  return MVIT_OK;
}

int mvit_segment_copy(const void* src, void* dst, const int64_t* desc, int64_t nseg, int64_t max_seg_rows, int64_t row_bytes, mvit_stream_t stream) {
  MVIT_REQUIRE(nseg >= 0 && nseg <= 65535 && row_bytes > 0 && row_bytes % 2 == 0, "segment_copy: bad nseg/row_bytes");
  if (nseg == 0 || max_seg_rows <= 0) return MVIT_OK;
  MVIT_REQUIRE(src && dst && desc, "segment_copy: null pointer");
  const unsigned gy = (unsigned)clamp_grid(max_seg_rows, 4096);
  if (row_bytes % 16 == 0 && mvit_aligned16(src) && mvit_aligned16(dst)) {
    const int64_t words = row_bytes / 16;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy, (unsigned)nseg);
    hipLaunchKernelGGL((segment_copy_kernel<u32x4>), grid, 256, 0, S_(stream), (const u32x4*)src, (u32x4*)dst, desc, words);
  } else if (row_bytes % 4 == 0) {
    const int64_t words = row_bytes / 4;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy, (unsigned)nseg);
    hipLaunchKernelGGL((segment_copy_kernel<uint32_t>), grid, 256, 0, S_(stream), (const uint32_t*)src, (uint32_t*)dst, desc, words);
  } else {
    const int64_t words = row_bytes / 2;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy, (unsigned)nseg);
    hipLaunchKernelGGL((segment_copy_kernel<uint16_t>), grid, 256, 0, S_(stream), (const uint16_t*)src, (uint16_t*)dst, desc, words);
  }
  MVIT_CHECK_LAUNCH("segment_copy");
  return MVIT_OK;
}

int mvit_pad_pack(const void* pack, void* padded, uint8_t* mask, const int64_t* lens, const int64_t* offsets, int64_t batch,
                  int64_t pad_len, int64_t row_elems, int elem_size, uint32_t pad_bits, mvit_stream_t stream) {
  MVIT_REQUIRE(batch >= 0 && batch <= 65535 && pad_len >= 0 && row_elems > 0, "pad_pack: bad shape");
  MVIT_REQUIRE(elem_size == 2 || elem_size == 4, "pad_pack: elem_size %d", elem_size);
  if (batch == 0 || pad_len == 0) return MVIT_OK;
  MVIT_REQUIRE(padded && mask && lens && offsets, "pad_pack: null pointer");
  dim3 grid((unsigned)clamp_grid((row_elems + 255) / 256, 64), (unsigned)clamp_grid(pad_len, 4096), (unsigned)batch);
  if (elem_size == 2)
    hipLaunchKernelGGL((pad_pack_kernel<uint16_t>), grid, 256, 0, S_(stream), (const uint16_t*)pack, (uint16_t*)padded, mask, lens, offsets, pad_len, row_elems, (uint16_t)pad_bits);
  else
    hipLaunchKernelGGL((pad_pack_kernel<uint32_t>), grid, 256, 0, S_(stream), (const uint32_t*)pack, (uint32_t*)padded, mask, lens, offsets, pad_len, row_elems, pad_bits);
  MVIT_CHECK_LAUNCH("pad_pack");
  return MVIT_OK;
}

int mvit_cast2d(const void* src, int64_t src_ld, int src_dtype, void* dst, int64_t dst_ld, int dst_dtype, int64_t rows,
                int64_t cols, mvit_stream_t stream) {
  MVIT_REQUIRE(rows >= 0 && cols >= 0 && src_ld >= cols && dst_ld >= cols, "cast2d: bad arguments");
  if (rows == 0 || cols == 0) return MVIT_OK;
  MVIT_REQUIRE(src && dst, "cast2d: null pointer");
  dim3 grid((unsigned)clamp_grid((cols + 255) / 256, 256), (unsigned)clamp_grid(rows, 16384));
  hipStream_t s = S_(stream);
  if (src_dtype == MVIT_F32 && dst_dtype == MVIT_BF16)
    hipLaunchKernelGGL((cast2d_kernel<float, bf16_t>), grid, 256, 0, s, (const float*)src, src_ld, (bf16_t*)dst, dst_ld, rows, cols);
  else if (src_dtype == MVIT_BF16 && dst_dtype == MVIT_F32)
    hipLaunchKernelGGL((cast2d_kernel<bf16_t, float>), grid, 256, 0, s, (const bf16_t*)src, src_ld, (float*)dst, dst_ld, rows, cols);
  else if (src_dtype == MVIT_F32 && dst_dtype == MVIT_F32)
    hipLaunchKernelGGL((cast2d_kernel<float, float>), grid, 256, 0, s, (const float*)src, src_ld, (float*)dst, dst_ld, rows, cols);
  else if (src_dtype == MVIT_BF16 && dst_dtype == MVIT_BF16)
    hipLaunchKernelGGL((cast2d_kernel<bf16_t, bf16_t>), grid, 256, 0, s, (const bf16_t*)src, src_ld, (bf16_t*)dst, dst_ld, rows, cols);
  else
    return mvit_set_error(MVIT_ERR_UNSUPPORTED, "cast2d: dtypes %d -> %d", src_dtype, dst_dtype);
  MVIT_CHECK_LAUNCH("cast2d");
  return MVIT_OK;
}

int mvit_image_token_ranks(const int64_t* input_ids, const int64_t* labels, int64_t n_tokens, int64_t image_token_id,
                           int64_t ignore_label, int32_t* rank, int64_t* positions, int64_t* counts, mvit_stream_t stream) {
  MVIT_REQUIRE(counts && (n_tokens == 0 || (input_ids && rank)), "image_token_ranks: null pointer");  // no tokens: only the counts are written (zeros)
  MVIT_REQUIRE(n_tokens >= 0 && n_tokens <= 0x7fffffffLL, "image_token_ranks: n_tokens %lld out of range", (long long)n_tokens);
  hipLaunchKernelGGL(image_token_ranks_kernel, dim3(1), 1024, 0, S_(stream), input_ids, labels, n_tokens, image_token_id, ignore_label,
                     rank, positions, counts);
  MVIT_CHECK_LAUNCH("image_token_ranks");
  return MVIT_OK;
}

int mvit_wait_host_values(const int64_t* values, int n, int64_t timeout_us) {
  MVIT_REQUIRE(values != nullptr && n > 0 && timeout_us >= 0, "wait_host_values: null pointer or bad count");
  const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(timeout_us);
  for (int i = 0; i < n;) {
    if (__atomic_load_n(values + i, __ATOMIC_ACQUIRE) >= 0) ++i;
    else if (std::chrono::steady_clock::now() >= end) return 1;
  }
  return MVIT_OK;
}

int mvit_await_host_values(const int64_t* values, int n, mvit_stream_t stream) {
  // Asking the stream is for those that fail; once asked, the GPU starts what is queued next some 10 us later, hence so seldom.  The wait is
  // a spin as that for an event is.  us from the beginning of 7 ms of queued work to the end of a kernel launched after the wait: for
  // an event behind the kernel 7,023 - 7,029, in polls with sleeps between them 7,108 - 7,143, this 7,024 - 7,026; on an idle stream 39 / 36 / 35.
  for (;;) {
    if (const int rc = mvit_wait_host_values(values, n, 100 * 1000); rc != 1) return rc;
    const hipError_t e = hipStreamQuery(S_(stream));
    (void)hipGetLastError();  // reported here, not by the next launch
    if (e != hipErrorNotReady) {
      if (mvit_wait_host_values(values, n, 0) == MVIT_OK) return MVIT_OK;
      return mvit_set_error(MVIT_ERR_LAUNCH, "await_host_values: %s", e == hipSuccess ? "the stream has ended without them" : hipGetErrorString(e));
    }
  }
}

int mvit_merge_rows(const void* embeds, const void* vision, const int32_t* rank, void* merged, int64_t n_tokens, int64_t n_vision,
                    int64_t row_bytes, mvit_stream_t stream) {
  MVIT_REQUIRE(n_tokens >= 0 && n_vision >= 0 && row_bytes > 0 && row_bytes % 2 == 0, "merge_rows: bad sizes (row_bytes %lld)", (long long)row_bytes);
  if (n_tokens == 0) return MVIT_OK;
  MVIT_REQUIRE(embeds && rank && merged, "merge_rows: null pointer");
  const unsigned gy = (unsigned)clamp_grid(n_tokens, 65535);
  const bool al = mvit_aligned16(embeds) && mvit_aligned16(merged) && (vision == nullptr || mvit_aligned16(vision));
  if (row_bytes % 16 == 0 && al) {
    const int64_t words = row_bytes / 16;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((merge_rows_kernel<u32x4>), grid, 256, 0, S_(stream), (const u32x4*)embeds, (const u32x4*)vision, rank, (u32x4*)merged, n_tokens, n_vision, words);
  } else if (row_bytes % 4 == 0) {
    const int64_t words = row_bytes / 4;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((merge_rows_kernel<uint32_t>), grid, 256, 0, S_(stream), (const uint32_t*)embeds, (const uint32_t*)vision, rank, (uint32_t*)merged, n_tokens, n_vision, words);
  } else {
    const int64_t words = row_bytes / 2;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((merge_rows_kernel<uint16_t>), grid, 256, 0, S_(stream), (const uint16_t*)embeds, (const uint16_t*)vision, rank, (uint16_t*)merged, n_tokens, n_vision, words);
  }
  MVIT_CHECK_LAUNCH("merge_rows");
  return MVIT_OK;
}

int mvit_split_rows(const void* grad, const int32_t* rank, void* text, void* vision, int64_t n_tokens, int64_t n_vision,
                    int64_t row_bytes, mvit_stream_t stream) {
  MVIT_REQUIRE(n_tokens >= 0 && n_vision >= 0 && row_bytes > 0 && row_bytes % 2 == 0, "split_rows: bad sizes (row_bytes %lld)", (long long)row_bytes);
  if (n_tokens == 0 || (!text && !vision)) return MVIT_OK;
  MVIT_REQUIRE(grad && rank, "split_rows: null pointer");
  const unsigned gy = (unsigned)clamp_grid(n_tokens, 65535);
  const bool al = mvit_aligned16(grad) && (!text || mvit_aligned16(text)) && (!vision || mvit_aligned16(vision));
  if (row_bytes % 16 == 0 && al) {
    const int64_t words = row_bytes / 16;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((split_rows_kernel<u32x4>), grid, 256, 0, S_(stream), (const u32x4*)grad, rank, (u32x4*)text, (u32x4*)vision, n_tokens, n_vision, words);
  } else if (row_bytes % 4 == 0) {
    const int64_t words = row_bytes / 4;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((split_rows_kernel<uint32_t>), grid, 256, 0, S_(stream), (const uint32_t*)grad, rank, (uint32_t*)text, (uint32_t*)vision, n_tokens, n_vision, words);
  } else {
    const int64_t words = row_bytes / 2;
    dim3 grid((unsigned)clamp_grid((words + 255) / 256, 64), gy);
    hipLaunchKernelGGL((split_rows_kernel<uint16_t>), grid, 256, 0, S_(stream), (const uint16_t*)grad, rank, (uint16_t*)text, (uint16_t*)vision, n_tokens, n_vision, words);
  }
  MVIT_CHECK_LAUNCH("split_rows");
  return MVIT_OK;
}

int mvit_copy_ranges(const mvit_copy_range* ranges, int n_ranges, mvit_stream_t stream) {
  MVIT_REQUIRE(n_ranges >= 0 && (n_ranges == 0 || ranges), "copy_ranges: null list");
  uintptr_t bits = 0;
  for (int i = 0; i < n_ranges; ++i) {
    MVIT_REQUIRE(ranges[i].bytes >= 0 && (ranges[i].bytes == 0 || (ranges[i].src && ranges[i].dst)), "copy_ranges: range %d", i);
    bits |= reinterpret_cast<uintptr_t>(ranges[i].src) | reinterpret_cast<uintptr_t>(ranges[i].dst) | (uintptr_t)ranges[i].bytes;
  }
  const int64_t word = bits % 16 == 0 ? 16 : (bits % 4 == 0 ? 4 : (bits % 2 == 0 ? 2 : 1));  // the widest that suits every range
  CopyRanges a;
  int64_t pieces = 0, bytes = 0;
  a.n = 0;
  auto flush = [&]() -> int {
    if (a.n == 0) return MVIT_OK;
    const dim3 grid((unsigned)pieces);
    if (word == 16 && bytes >= COPY_NT_STORES) hipLaunchKernelGGL((copy_ranges_kernel<u32x4, true, true>), grid, 256, 0, S_(stream), a);
    else if (word == 16 && bytes >= COPY_NT_LOADS) hipLaunchKernelGGL((copy_ranges_kernel<u32x4, true, false>), grid, 256, 0, S_(stream), a);
    else if (word == 16) hipLaunchKernelGGL((copy_ranges_kernel<u32x4, false, false>), grid, 256, 0, S_(stream), a);
    else if (word == 4) hipLaunchKernelGGL((copy_ranges_kernel<uint32_t, false, false>), grid, 256, 0, S_(stream), a);
    else if (word == 2) hipLaunchKernelGGL((copy_ranges_kernel<uint16_t, false, false>), grid, 256, 0, S_(stream), a);
    else hipLaunchKernelGGL((copy_ranges_kernel<uint8_t, false, false>), grid, 256, 0, S_(stream), a);
    MVIT_CHECK_LAUNCH("copy_ranges");
    a.n = 0;
    pieces = bytes = 0;
    return MVIT_OK;
  };
  for (int i = 0; i < n_ranges; ++i) {
    const char* src = static_cast<const char*>(ranges[i].src);
    char* dst = static_cast<char*>(ranges[i].dst);
    for (int64_t left = ranges[i].bytes / word; left > 0;) {  // a range longer than a launch is cut
      if (a.n == COPY_MAX_RANGES || pieces == MVIT_MAX_GROUPS_256)
        if (int rc = flush()) return rc;
      const int64_t room = (MVIT_MAX_GROUPS_256 - pieces) * COPY_PIECE, words = left < room ? left : room;
      a.first_piece[a.n] = (int)pieces;
      a.src[a.n] = src;
      a.dst[a.n] = dst;
      a.words[a.n++] = words;
      pieces += (words + COPY_PIECE - 1) / COPY_PIECE;
      bytes += words * word;
      src += words * word;
      dst += words * word;
      left -= words;
    }
  }
  return flush();
}

}  // extern "C"
