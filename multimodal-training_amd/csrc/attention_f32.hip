// fp32 attention, forward and backward (the parity path), on v_mfma_f32_16x16x4_f32.
//
// Each wave owns 16 rows of one side (queries in the forward and for dQ, keys for dK / dV) with all of head_dim in registers;
// 32-row tiles of the other side pass through LDS and serve the four waves of the work-group.  Every product is oriented so
// that the accumulator layout of the scores is the operand layout of the product that follows:
//   forward, dQ: S^T = K Q^T (lane: query l % 16, keys 4 (l / 16) + r)  ->  O^T += V^T P^T, dQ^T += K^T dS^T
//   dK, dV:      S = Q K^T   (lane: key l % 16, queries 4 (l / 16) + r) ->  dV^T += dO^T P, dK^T += Q^T dS
// An MFMA contracts four values, one per 16-lane group.  Score MFMA (s, j) takes head_dim index 16 s + 4 g + j from group g, so
// one 16-byte LDS read feeds four of them; MFMA r of the second product takes row 4 g + r, which is where the scores lie.
// LDS rows are padded by four floats: 16-byte reads of 16 rows and 4-byte reads of rows 4 apart are both conflict-free.
// Bound by the fp32 matrix rate where a launch has enough segments and heads to fill the chip.
#include "attention_common.h"

namespace {

constexpr int TILE = 32;  // rows of the other side per step

template <int HD>
struct F32Attn {
  static constexpr int PITCH = HD + 4, NS = HD / 16, CHUNKS = TILE * HD / 4, PER = (CHUNKS + 255) / 256;

  // rows [row0, row0 + TILE) of X (zeros from row `limit` on), 16 bytes per thread and step, requested ahead of their use
  struct Tile {
    f32x4 v[PER];
    __device__ __forceinline__ void fetch(const float* X, int64_t stride, int row0, int limit) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + 256 * i, row = c / (HD / 4), col = c % (HD / 4) * 4;
        v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (c < CHUNKS && row0 + row < limit) v[i] = *reinterpret_cast<const f32x4*>(X + (int64_t)(row0 + row) * stride + col);
      }
    }
    __device__ __forceinline__ void put(float* lds) const {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + 256 * i, row = c / (HD / 4), col = c % (HD / 4) * 4;
        if (c < CHUNKS) *reinterpret_cast<f32x4*>(lds + row * PITCH + col) = v[i];
      }
    }
  };
  // this wave's own 16 rows as score operand: lane holds row l % 16, values 16 s + 4 (l / 16) + j
  static __device__ __forceinline__ void own(const float* X, int64_t stride, int row, bool valid, f32x4 (&f)[NS]) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      f[s] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (valid) f[s] = *reinterpret_cast<const f32x4*>(X + (int64_t)row * stride + 16 * s + 4 * g);
    }
  }
  // scores of LDS rows [blk * 16, +16) against the own rows
  static __device__ __forceinline__ f32x4 scores(const float* lds, int blk, const f32x4 (&f)[NS]) {
    const int l = threadIdx.x & 63;
    const float* at = lds + (blk * 16 + (l & 15)) * PITCH + 4 * (l >> 4);
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(at + 16 * s);
#pragma unroll
      for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], f[s][j], c, 0, 0, 0);
    }
    return c;
  }
  // acc^T[d][own row] += lds^T[d][row] w[row][own row] over LDS rows [blk * 16, +16)
  static __device__ __forceinline__ void accumulate(const float* lds, int blk, const f32x4 w, f32x4 (&acc)[NS]) {
    const int l = threadIdx.x & 63;
    const float* at = lds + (blk * 16 + 4 * (l >> 4)) * PITCH + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int d = 0; d < NS; ++d) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(at[r * PITCH + 16 * d], w[r], acc[d], 0, 0, 0);
  }
  static __device__ __forceinline__ void store(float* X, int64_t stride, int row, const f32x4 (&acc)[NS], float factor) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int d = 0; d < NS; ++d)
      *reinterpret_cast<f32x4*>(X + (int64_t)row * stride + 16 * d + 4 * g) = f32x4{acc[d][0] * factor, acc[d][1] * factor, acc[d][2] * factor, acc[d][3] * factor};
  }
};

template <int HD>
__global__ __launch_bounds__(256) void attn_fwd_f32(const AttnParams p) {
  using A = F32Attn<HD>;
  __shared__ __attribute__((aligned(16))) float sk[TILE * A::PITCH], sv[TILE * A::PITCH];
  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  if ((int)blockIdx.x * 64 >= L) return;
  const int l = threadIdx.x & 63, g = l >> 4, qi = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + (l & 15);
  const bool valid = qi < L;
  const float* K = static_cast<const float*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const float* V = static_cast<const float*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  f32x4 q[A::NS], acc[A::NS];
  A::own(static_cast<const float*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD, p.q_stride, qi, valid, q);
#pragma unroll
  for (int d = 0; d < A::NS; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  typename A::Tile tk, tv;
  tk.fetch(K, p.k_stride, 0, L);
  tv.fetch(V, p.v_stride, 0, L);
  for (int k0 = 0; k0 < L; k0 += TILE) {
    __syncthreads();
    tk.put(sk);
    tv.put(sv);
    __syncthreads();
    if (k0 + TILE < L) {
      tk.fetch(K, p.k_stride, k0 + TILE, L);
      tv.fetch(V, p.v_stride, k0 + TILE, L);
    }
    f32x4 s[2];
    float mx = m;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      s[b] = A::scores(sk, b, q);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[b][r] = k0 + b * 16 + 4 * g + r < L ? s[b][r] * p.scale : -INFINITY;
        mx = fmaxf(mx, s[b][r]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));  // the four lane groups hold different keys of the same query
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float alpha = expf(m - mx);
    m = mx;
    lsum *= alpha;
#pragma unroll
    for (int d = 0; d < A::NS; ++d) acc[d] = f32x4{acc[d][0] * alpha, acc[d][1] * alpha, acc[d][2] * alpha, acc[d][3] * alpha};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[b][r] = expf(s[b][r] - mx);
        lsum += s[b][r];
      }
      A::accumulate(sv, b, s[b], acc);
    }
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (valid) {
    A::store(static_cast<float*>(p.out) + (int64_t)s0 * p.o_stride + (int64_t)h * HD, p.o_stride, qi, acc, 1.f / lsum);
    if (g == 0) p.lse[(int64_t)h * p.total + s0 + qi] = m + logf(lsum);
  }
}

template <int HD>
__global__ __launch_bounds__(256) void attn_bwd_dq_f32(const AttnParams p) {
  using A = F32Attn<HD>;
  __shared__ __attribute__((aligned(16))) float sk[TILE * A::PITCH], sv[TILE * A::PITCH];
  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  if ((int)blockIdx.x * 64 >= L) return;
  const int l = threadIdx.x & 63, g = l >> 4, qi = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + (l & 15);
  const bool valid = qi < L;
  const float* K = static_cast<const float*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const float* V = static_cast<const float*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  f32x4 q[A::NS], go[A::NS], acc[A::NS];
  A::own(static_cast<const float*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD, p.q_stride, qi, valid, q);
  A::own(static_cast<const float*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD, p.do_stride, qi, valid, go);
#pragma unroll
  for (int d = 0; d < A::NS; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float lse = valid ? p.lse[(int64_t)h * p.total + s0 + qi] : INFINITY;
  const float dl = valid ? p.delta[(int64_t)h * p.total + s0 + qi] : 0.f;
  typename A::Tile tk, tv;
  tk.fetch(K, p.k_stride, 0, L);
  tv.fetch(V, p.v_stride, 0, L);
  for (int k0 = 0; k0 < L; k0 += TILE) {
    __syncthreads();
    tk.put(sk);
    tv.put(sv);
    __syncthreads();
    if (k0 + TILE < L) {
      tk.fetch(K, p.k_stride, k0 + TILE, L);
      tv.fetch(V, p.v_stride, k0 + TILE, L);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const f32x4 s = A::scores(sk, b, q), dp = A::scores(sv, b, go);
      f32x4 ds;
#pragma unroll
      for (int r = 0; r < 4; ++r) ds[r] = k0 + b * 16 + 4 * g + r < L ? expf(s[r] * p.scale - lse) * (dp[r] - dl) : 0.f;
      A::accumulate(sk, b, ds, acc);
    }
  }
  if (valid) A::store(static_cast<float*>(p.dq) + (int64_t)s0 * p.dq_stride + (int64_t)h * HD, p.dq_stride, qi, acc, p.scale);
}

template <int HD>
__global__ __launch_bounds__(256) void attn_bwd_dkdv_f32(const AttnParams p) {
  using A = F32Attn<HD>;
  __shared__ __attribute__((aligned(16))) float sq[TILE * A::PITCH], sdo[TILE * A::PITCH], slse[TILE], sdl[TILE];
  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  if ((int)blockIdx.x * 64 >= L) return;
  const int l = threadIdx.x & 63, g = l >> 4, ki = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + (l & 15);
  const bool valid = ki < L;
  const float* Q = static_cast<const float*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD;
  const float* DO = static_cast<const float*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD;
  f32x4 k[A::NS], v[A::NS], dk[A::NS], dv[A::NS];
  A::own(static_cast<const float*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD, p.k_stride, ki, valid, k);
  A::own(static_cast<const float*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD, p.v_stride, ki, valid, v);
#pragma unroll
  for (int d = 0; d < A::NS; ++d) dk[d] = dv[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  typename A::Tile tq, tdo;
  tq.fetch(Q, p.q_stride, 0, L);
  tdo.fetch(DO, p.do_stride, 0, L);
  for (int q0 = 0; q0 < L; q0 += TILE) {
    __syncthreads();
    tq.put(sq);
    tdo.put(sdo);
    if (threadIdx.x < TILE) {  // queries past the end: exp(s - inf) = 0
      const bool ok = q0 + (int)threadIdx.x < L;
      slse[threadIdx.x] = ok ? p.lse[(int64_t)h * p.total + s0 + q0 + threadIdx.x] : INFINITY;
      sdl[threadIdx.x] = ok ? p.delta[(int64_t)h * p.total + s0 + q0 + threadIdx.x] : 0.f;
    }
    __syncthreads();
    if (q0 + TILE < L) {
      tq.fetch(Q, p.q_stride, q0 + TILE, L);
      tdo.fetch(DO, p.do_stride, q0 + TILE, L);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const f32x4 s = A::scores(sq, b, k), dp = A::scores(sdo, b, v);
      const f32x4 lse = *reinterpret_cast<const f32x4*>(slse + b * 16 + 4 * g), dl = *reinterpret_cast<const f32x4*>(sdl + b * 16 + 4 * g);
      f32x4 e, ds;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        e[r] = expf(s[r] * p.scale - lse[r]);
        ds[r] = e[r] * (dp[r] - dl[r]);
      }
      A::accumulate(sdo, b, e, dv);
      A::accumulate(sq, b, ds, dk);
    }
  }
  if (valid) {
    A::store(static_cast<float*>(p.dk) + (int64_t)s0 * p.dk_stride + (int64_t)h * HD, p.dk_stride, ki, dk, p.scale);
    A::store(static_cast<float*>(p.dv) + (int64_t)s0 * p.dv_stride + (int64_t)h * HD, p.dv_stride, ki, dv, 1.f);
  }
}

template <int HD>
int launch(const AttnParams& p, int n_seg, int max_seqlen, bool bwd, hipStream_t s) {
  const dim3 grid((unsigned)((max_seqlen + 63) / 64), (unsigned)n_seg, (unsigned)p.nheads);
  if (!bwd) {
    hipLaunchKernelGGL((attn_fwd_f32<HD>), grid, 256, 0, s, p);
  } else {
    hipLaunchKernelGGL((attn_bwd_dkdv_f32<HD>), grid, 256, 0, s, p);
    hipLaunchKernelGGL((attn_bwd_dq_f32<HD>), grid, 256, 0, s, p);
  }
  MVIT_CHECK_LAUNCH("attn_f32");
  return MVIT_OK;
}

}  // namespace

int mvit_attn_f32(const AttnParams& p, int head_dim, int n_seg, int max_seqlen, bool bwd, hipStream_t s) {
  switch (head_dim) {
    case 32: return launch<32>(p, n_seg, max_seqlen, bwd, s);
    case 64: return launch<64>(p, n_seg, max_seqlen, bwd, s);
    case 80: return launch<80>(p, n_seg, max_seqlen, bwd, s);
    default: return launch<128>(p, n_seg, max_seqlen, bwd, s);
  }
}
