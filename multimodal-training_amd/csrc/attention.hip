// Variable-length (cu_seqlens) non-causal attention, forward and backward, for gfx950.
//
// bf16 path: flash-style kernels on v_mfma_f32_16x16x32_bf16; head_dim = 16*ND is contracted in 32-wide steps
// plus, for odd ND (head_dim 80 = 5 x 16), one half-filled 32-wide step.  All products are oriented so that the
// accumulator layout of one MFMA is directly the B-operand layout of the next:
//   forward : S^T = K Q^T   (lane: query l%16, keys 4*(l/16)+i)  ->  O^T += V^T P^T
//   dK/dV   : S = Q K^T, dP = dO V^T (lane: key l%16, queries 4*(l/16)+i)  ->  dV^T += dO^T P, dK^T += Q^T dS
//   dQ      : S^T, dP^T as in the forward  ->  dQ^T += K^T dS^T
// Operands that are needed "transposed" (V, dO, Q, K as the left factor of the second product) are read
// from their natural [row][head_dim] LDS tiles with ds_read_b64_tr_b16.  Softmax statistics live in
// registers; row reductions are two cross-lane exchanges (lanes l, l^16, l^32, l^48 share a query).
// The backward is split in two kernels (dK/dV, then dQ), which keeps it free of atomics and bit-reproducible.
//
// fp32 path (parity mode): attention_f32.hip.
#include "attention_common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;


typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
typedef short s16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 tr_pair(const bf16_t* p0, const bf16_t* p1) {
  s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p0);
  s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p1);
  s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, both);
}
__device__ __forceinline__ bf16x8 pack8(const f32x4& a, const f32x4& b) {
  bf16x8 r;
  r[0] = (bf16_t)a[0]; r[1] = (bf16_t)a[1]; r[2] = (bf16_t)a[2]; r[3] = (bf16_t)a[3];
  r[4] = (bf16_t)b[0]; r[5] = (bf16_t)b[1]; r[6] = (bf16_t)b[2]; r[7] = (bf16_t)b[3];
  return r;
}
__device__ __forceinline__ f32x4 mfma32(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

template <int ND>
struct Geo {
  static constexpr int HD = 16 * ND;
  static constexpr int NK32 = ND / 2;         // 32-wide contraction steps over head_dim
  static constexpr bool TAIL16 = (ND & 1);    // plus one 16-wide step
  static constexpr int PK = HD + 8;           // pitch of tiles read with 16-byte row loads
  static constexpr int PV = (HD % 32 == 0) ? HD + 16 : HD;  // pitch of tiles read only through transposing loads
  static constexpr int CH = 2 * ND;           // 16-byte chunks per row
};

// Bank-rotated LDS tile layout for tiles that are read both row-wise (16-byte fragments of 16 consecutive rows)
// and through the transposing load (8 consecutive rows x 32 bytes): chunk c (16 bytes) of row r lives at byte
// r * 512 + 16 * (c + rot(r)), rot(r) = 2 * (r & 7) + ((r >> 3) & 1).  Modulo the 256 bytes of one pass over the
// banks, sixteen consecutive rows put one chunk index into sixteen different 16-byte slots, and eight consecutive
// rows put one pair of chunks into eight disjoint 32-byte windows, so neither access pattern has bank conflicts
// (a plain pitch cannot satisfy both: the first needs pitch/16 odd, the second pitch/32 odd).  The rotation is
// additive, so every access is a per-lane base plus a compile-time offset; rows are 512 bytes so that it never
// wraps (10 chunks of data + rotation <= 25 slots; head_dim 128: 31).
constexpr int SWZ = 256;  // pitch in elements; used as the PITCH argument to select this layout
__device__ __forceinline__ int swz_off(int row, int chunk) {
  return row * SWZ + ((chunk + (((row & 7) << 1) | ((row >> 3) & 1))) << 3);
}
// Transposed operand of the 16 x 16 block (rows row0.., head-dim 16*d..) : two transposing loads 16 rows apart.
template <int PITCH>
__device__ __forceinline__ bf16x8 tr_block(const bf16_t* tile, int row0, int d, int g, int r) {
  const int row = row0 + 4 * g + (r >> 2);
  if (PITCH == SWZ) {
    const int chunk = 2 * d + ((r & 3) >> 1), sub = 4 * (r & 1);
    return tr_pair(tile + swz_off(row, chunk) + sub, tile + swz_off(row + 16, chunk) + sub);
  }
  const bf16_t* a = tile + row * PITCH + 16 * d + 4 * (r & 3);
  return tr_pair(a, a + 16 * PITCH);
}

// Operand fragments of 16 rows x head_dim for one lane, in the "row l%16, contraction 8*(l/16)+j" layout
// (serves as MFMA A for rows, or as MFMA B for columns).
template <int ND>
struct RowFrag {
  bf16x8 k32[Geo<ND>::NK32 > 0 ? Geo<ND>::NK32 : 1];
  bf16x4 k16;
};

template <int ND>
__device__ __forceinline__ void load_rowfrag_global(RowFrag<ND>& f, const bf16_t* row_ptr, bool valid, int g) {
  using G = Geo<ND>;
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
    if (valid) v = *reinterpret_cast<const bf16x8*>(row_ptr + 32 * ks + 8 * g);
    f.k32[ks] = v;
  }
  if (G::TAIL16) {
    bf16x4 v = {(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
    if (valid) v = *reinterpret_cast<const bf16x4*>(row_ptr + 32 * G::NK32 + 4 * g);
    f.k16 = v;
  }
}
template <int ND, int PITCH>
__device__ __forceinline__ void load_rowfrag_lds(RowFrag<ND>& f, const bf16_t* tile, int row, int g) {
  using G = Geo<ND>;
  if (PITCH == SWZ) {
#pragma unroll
    for (int ks = 0; ks < G::NK32; ++ks) f.k32[ks] = *reinterpret_cast<const bf16x8*>(tile + swz_off(row, 4 * ks + g));
    if (G::TAIL16) f.k16 = *reinterpret_cast<const bf16x4*>(tile + swz_off(row, 4 * G::NK32 + (g >> 1)) + 4 * (g & 1));
    return;
  }
  const bf16_t* p = tile + row * PITCH;
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks) f.k32[ks] = *reinterpret_cast<const bf16x8*>(p + 32 * ks + 8 * g);
  if (G::TAIL16) f.k16 = *reinterpret_cast<const bf16x4*>(p + 32 * G::NK32 + 4 * g);
}
// acc = rows(a) . rows(b)^T over head_dim  (16x16 tile).
// The 16-wide remainder of head_dim (odd ND) is issued as a 32-wide MFMA whose upper four contraction slots
// are zero: a v_mfma_f32_16x16x16_bf16 chained onto the accumulator of the 32-wide steps returned wrong sums
// on gfx950 (also with an all-zero remainder), so that instruction is not used here.
template <int ND>
__device__ __forceinline__ f32x4 dot_frag(const RowFrag<ND>& a, const RowFrag<ND>& b) {
  using G = Geo<ND>;
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks) c = mfma32(a.k32[ks], b.k32[ks], c);
  if (G::TAIL16) {
    const bf16_t z = (bf16_t)0.f;
    const bf16x8 ax = {a.k16[0], a.k16[1], a.k16[2], a.k16[3], z, z, z, z};
    const bf16x8 bx = {b.k16[0], b.k16[1], b.k16[2], b.k16[3], z, z, z, z};
    c = mfma32(ax, bx, c);
  }
  return c;
}

// Cooperative global -> LDS copy of `rows` x head_dim (zero-filled past `valid_rows`).
template <int ND, int PITCH, int NTHREADS>
__device__ __forceinline__ void stage_tile(bf16_t* tile, const bf16_t* src, int64_t stride, int rows, int valid_rows) {
  using G = Geo<ND>;
  const int nchunks = rows * G::CH;
  for (int c = threadIdx.x; c < nchunks; c += NTHREADS) {
    const int r = c / G::CH, dc = c % G::CH;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
    if (r < valid_rows) v = *reinterpret_cast<const bf16x8*>(src + (int64_t)r * stride + dc * 8);
    *reinterpret_cast<bf16x8*>(tile + r * PITCH + dc * 8) = v;
  }
}

// The same copy split in two halves (global -> registers, registers -> LDS) with the per-thread chunk
// coordinates computed once, so that the loads of the next tile can be in flight while the current one is used.
template <int ND, int ROWS, int PITCH, int NTHREADS>
struct TileStager {
  using G = Geo<ND>;
  static constexpr int CHUNKS = ROWS * G::CH;
  static constexpr int PER = (CHUNKS + NTHREADS - 1) / NTHREADS;
  int row[PER];      // tile row of chunk i (ROWS = "no chunk")
  int lds_off[PER];  // element offset in the LDS tile
  int64_t goff[PER]; // element offset from the tile's first row in global memory
  bf16x8 regs[PER];

  __device__ __forceinline__ void init(int64_t stride) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = threadIdx.x + NTHREADS * i;
      const int r = c / G::CH, dc = c % G::CH;
      row[i] = c < CHUNKS ? r : ROWS;
      lds_off[i] = PITCH == SWZ ? swz_off(r, dc) : r * PITCH + dc * 8;
      goff[i] = (int64_t)r * stride + dc * 8;
    }
  }
  __device__ __forceinline__ void load(const bf16_t* src, int valid_rows) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
      if (row[i] < valid_rows) v = *reinterpret_cast<const bf16x8*>(src + goff[i]);
      regs[i] = v;
    }
  }
  __device__ __forceinline__ void scale(float c) {  // the loaded chunks times c, rounded back to bf16
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) regs[i][j] = (bf16_t)((float)regs[i][j] * c);
  }
  __device__ __forceinline__ void store(bf16_t* tile) const {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (row[i] < ROWS) *reinterpret_cast<bf16x8*>(tile + lds_off[i]) = regs[i];
  }
};

// Reductions over the four lanes l, l^16, l^32, l^48 (the lanes that share one query / key column) with the
// VALU lane-swap instructions of gfx950 instead of LDS permutes: v_permlane32_swap exchanges the upper half of its
// first operand with the lower half of its second, v_permlane16_swap does the same for the odd / even rows of 16.
__device__ __forceinline__ float quad_max(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  x = fmaxf(a, b);
  a = x;
  b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

// dot_frag with one extra contraction slot (odd ND only: the 16-wide remainder leaves half of its 32-wide MFMA
// empty): adds a_x * b_x from lane group 0, which is how the forward folds "- running maximum" into the scores.
template <int ND>
__device__ __forceinline__ f32x4 dot_frag_plus(const RowFrag<ND>& a, const RowFrag<ND>& b, bf16_t a_x, bf16_t b_x) {
  using G = Geo<ND>;
  static_assert(G::TAIL16, "needs the spare slots of the padded remainder");
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks) c = mfma32(a.k32[ks], b.k32[ks], c);
  const bf16_t z = (bf16_t)0.f;
  const bf16x8 ax = {a.k16[0], a.k16[1], a.k16[2], a.k16[3], a_x, z, z, z};
  const bf16x8 bx = {b.k16[0], b.k16[1], b.k16[2], b.k16[3], b_x, z, z, z};
  return mfma32(ax, bx, c);
}

// A float as the sum of two bf16 numbers (16 bits of mantissa): for values that ride in spare contraction slots.
struct HiLo {
  bf16_t hi, lo;
};
__device__ __forceinline__ HiLo split_hilo(float x) {
  HiLo r;
  r.hi = (bf16_t)x;
  r.lo = (bf16_t)(x - (float)r.hi);
  return r;
}
// dot_frag with two extra contraction slots: adds a0*b0 + a1*b1 (operands given per lane; lane groups other than
// 0 must pass zeros on at least one side).  The backward uses it for "- lse" and "- delta", split as hi + lo.
template <int ND>
__device__ __forceinline__ f32x4 dot_frag_plus2(const RowFrag<ND>& a, const RowFrag<ND>& b, bf16_t a0, bf16_t a1, bf16_t b0, bf16_t b1) {
  using G = Geo<ND>;
  static_assert(G::TAIL16, "needs the spare slots of the padded remainder");
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks) c = mfma32(a.k32[ks], b.k32[ks], c);
  const bf16_t z = (bf16_t)0.f;
  const bf16x8 ax = {a.k16[0], a.k16[1], a.k16[2], a.k16[3], a0, a1, z, z};
  const bf16x8 bx = {b.k16[0], b.k16[1], b.k16[2], b.k16[3], b0, b1, z, z};
  return mfma32(ax, bx, c);
}
// Multiply a fragment by a scalar (rounded back to bf16): Q enters every score product as Q * scale * log2(e).
template <int ND>
__device__ __forceinline__ void scale_rowfrag(RowFrag<ND>& f, float c) {
  using G = Geo<ND>;
#pragma unroll
  for (int ks = 0; ks < G::NK32; ++ks)
#pragma unroll
    for (int j = 0; j < 8; ++j) f.k32[ks][j] = (bf16_t)((float)f.k32[ks][j] * c);
  if (G::TAIL16) {
#pragma unroll
    for (int j = 0; j < 4; ++j) f.k16[j] = (bf16_t)((float)f.k16[j] * c);
  }
}

__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// ================================================================================================
// Forward.  Block = NWAVES waves x 16*QB queries of one (segment, head); BNK keys per iteration.
// At least two work-groups share a CU, K/V tiles are double buffered in LDS and the next tile is
// fetched while the current one is used; key masking only runs on a segment's last, partial tile; the output
// accumulators are rescaled only in iterations where some row maximum of the wave actually grew.
template <int ND, int NWAVES, int BNK, bool PIPE, int QB = 4, int MINW = 2>
__global__ __launch_bounds__(64 * NWAVES, MINW) void attn_fwd_mfma(const AttnParams p) {
  using G = Geo<ND>;
  constexpr int HD = G::HD, NT = 64 * NWAVES, KT = BNK / 16, KK = BNK / 32, NBUF = PIPE ? 2 : 1;
  __shared__ __attribute__((aligned(16))) bf16_t lds_k[NBUF][BNK * G::PK];
  __shared__ __attribute__((aligned(16))) bf16_t lds_v[NBUF][BNK * G::PV];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_q0 = blockIdx.x * (16 * QB * NWAVES);
  if (blk_q0 >= L) return;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, g = l >> 4, r = l & 15;
  const int q0 = blk_q0 + wv * (16 * QB);

  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;

  // Q is scaled by softmax_scale * log2(e) once (rounded to bf16), so the MFMA hands out scores in log2 units.
  // With an odd ND the spare contraction slot of the padded remainder also subtracts the row's running
  // stabiliser m_run (kept as a bf16-representable number): exp2 is then applied to the MFMA result directly.
  constexpr bool FOLD = G::TAIL16;
  constexpr float TAU = 2.f;  // the stabiliser only moves when a score exceeds it by more than TAU (log2 units)
  const float c = p.scale * LOG2E;
  RowFrag<ND> qf[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q0 + qb * 16 + r;
    load_rowfrag_global<ND>(qf[qb], Q + (int64_t)qi * p.q_stride, qi < L, g);
    scale_rowfrag<ND>(qf[qb], c);
  }
  const bf16_t one_x = (bf16_t)(g == 0 ? 1.f : 0.f);  // key side of the extra slot
  bf16_t negm_x[QB];                                    // query side: -m_run in lane group 0

  f32x4 o[QB][ND], lacc[QB];  // lacc: row sums of P, accumulated by the MFMA against a tile of ones
  float m_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = 0.f;
    negm_x[qb] = (bf16_t)0.f;
    lacc[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) o[qb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (bf16_t)1.f;

  constexpr bool STAGED = PIPE || QB == 1;  // through registers, all of a tile's loads in flight at once
  TileStager<ND, BNK, G::PK, STAGED ? NT : BNK * G::CH> sk;  // (degenerate when not)
  TileStager<ND, BNK, G::PV, STAGED ? NT : BNK * G::CH> sv;
  if (STAGED) {
    sk.init(p.k_stride);
    sv.init(p.v_stride);
  }
  if (PIPE) {
    sk.load(K, min(BNK, L));
    sv.load(V, min(BNK, L));
    sk.store(lds_k[0]);
    sv.store(lds_v[0]);
    __syncthreads();
  }

  int buf = 0;
  for (int k0 = 0; k0 < L; k0 += BNK) {
    const int valid = min(BNK, L - k0);
    const bool has_next = k0 + BNK < L;
    if (PIPE) {
      if (has_next) {
        const int nv = min(BNK, L - k0 - BNK);
        sk.load(K + (int64_t)(k0 + BNK) * p.k_stride, nv);
        sv.load(V + (int64_t)(k0 + BNK) * p.v_stride, nv);
      }
    } else {
      if constexpr (STAGED) {
        sk.load(K + (int64_t)k0 * p.k_stride, valid);
        sv.load(V + (int64_t)k0 * p.v_stride, valid);
        if (k0 > 0) __syncthreads();
        sk.store(lds_k[0]);
        sv.store(lds_v[0]);
      } else {
        if (k0 > 0) __syncthreads();
        stage_tile<ND, G::PK, NT>(lds_k[0], K + (int64_t)k0 * p.k_stride, p.k_stride, BNK, valid);
        stage_tile<ND, G::PV, NT>(lds_v[0], V + (int64_t)k0 * p.v_stride, p.v_stride, BNK, valid);
      }
      __syncthreads();
    }
    const bf16_t* tk = lds_k[PIPE ? buf : 0];
    const bf16_t* tv = lds_v[PIPE ? buf : 0];

    // raw scores: s[qb][kt][i] = S[query qb*16 + r][key kt*16 + 4g + i]
    f32x4 s[QB][KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      RowFrag<ND> kf;
      load_rowfrag_lds<ND, G::PK>(kf, tk, kt * 16 + r, g);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        if constexpr (FOLD) s[qb][kt] = dot_frag_plus<ND>(kf, qf[qb], one_x, negm_x[qb]);  // log2-scaled score - m_run
        else s[qb][kt] = dot_frag<ND>(kf, qf[qb]);
      }
    }
    if (valid < BNK) {  // last, partial tile of the segment
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kt * 16 + 4 * g + i >= valid) s[qb][kt][i] = -INFINITY;
    }
    bf16x8 pb[QB][KK];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float mx = fmaxf(s[qb][0][0], s[qb][0][1]);
      mx = max3(mx, s[qb][0][2], s[qb][0][3]);
#pragma unroll
      for (int kt = 1; kt < KT; ++kt) {
        mx = max3(mx, s[qb][kt][0], s[qb][kt][1]);
        mx = max3(mx, s[qb][kt][2], s[qb][kt][3]);
      }
      mx = quad_max(mx);
      if (!FOLD) mx -= m_run[qb];  // excess over the current stabiliser
      const bool grow = k0 == 0 || mx > TAU;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        float m_new = grow ? m_run[qb] + mx : m_run[qb];
        if (FOLD) m_new = (float)(bf16_t)m_new;
        const float delta = m_new - m_run[qb];
        const float alpha = k0 == 0 ? 1.f : __builtin_amdgcn_exp2f(-delta);
        m_run[qb] = m_new;
        lacc[qb] *= alpha;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) o[qb][dt] *= alpha;
        if (FOLD) {  // this tile's scores were taken against the old stabiliser
          negm_x[qb] = (bf16_t)(g == 0 ? -m_new : 0.f);
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[qb][kt][i] -= delta;
        }
      }
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[qb][kt][i] = __builtin_amdgcn_exp2f(FOLD ? s[qb][kt][i] : s[qb][kt][i] - m_run[qb]);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) pb[qb][kk] = pack8(s[qb][2 * kk], s[qb][2 * kk + 1]);
    }
    // O^T[d][q] += sum_key V[key][d] P[q][key]; contraction slots (g, j): keys t0*16+4g+j | t1*16+4g+j-4
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        const bf16_t* a0 = tv + ((2 * kk) * 16 + 4 * g + (r >> 2)) * G::PV + 16 * dt + 4 * (r & 3);
        const bf16x8 vf = tr_pair(a0, a0 + 16 * G::PV);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) o[qb][dt] = mfma32(vf, pb[qb][kk], o[qb][dt]);
      }
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) lacc[qb] = mfma32(ones, pb[qb][kk], lacc[qb]);
    if (PIPE) {
      if (has_next) {
        sk.store(lds_k[buf ^ 1]);
        sv.store(lds_v[buf ^ 1]);
      }
      __syncthreads();
      buf ^= 1;
    }
  }

  bf16_t* O = static_cast<bf16_t*>(p.out) + (int64_t)s0 * p.o_stride + (int64_t)h * HD;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float lt = lacc[qb][0];  // every row of the ones tile holds the row sum
    const int qi = q0 + qb * 16 + r;
    if (qi < L) {
      const float inv = 1.f / lt;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        bf16x4 ov;
#pragma unroll
        for (int i = 0; i < 4; ++i) ov[i] = (bf16_t)(o[qb][dt][i] * inv);
        *reinterpret_cast<bf16x4*>(O + (int64_t)qi * p.o_stride + 16 * dt + 4 * g) = ov;
      }
      if (g == 0) p.lse[(int64_t)h * p.total + s0 + qi] = (m_run[qb] + __builtin_amdgcn_logf(lt)) * LN2;
    }
  }
}

// ================================================================================================
// Windows (at most 64 tokens), forward, with the rotary embedding of q and k inside: the pass of its own reads and writes both once more.
// A thread owns eight columns of the first half of a head and the matching eight of the second in one row, so ND waves rotate and four of
// them compute.  Rounded where the separate passes round (rotation to bf16, then the attention of attn_fwd_mfma): the same bits.
// Bound by the chain load -> rotation -> products -> store, i.e. by the work-groups that a unit holds, where q, k and v come from the memory-side
// cache, and by memory beyond (1,006 MB at 65,536 rows x 16 heads where the rotated values are kept for a backward, else 671).  So two forms:
// * one head to a work-group, 72 registers and 32 KiB, five of them to a unit;
// * LOOP: `heads` heads of a window one after the other, the tables' part of a thread in registers for all of them, the next head's q, k and v
//   travelling while the four waves multiply: 136 registers, two work-groups to a unit.
// us, rotation in a pass of its own (rope_vec_kernel, attn_fwd_mfma) / one head, kept, not kept / LOOP, two heads, kept, four, not kept.  Operands from HBM:
// 4,096 rows 23.8 / 19.8, 15.3 / 21.3, 14.6; 14,336 66.5 / 65.8, 44.4 / 60.6, 43.7; 25,524 116 / 115, 75.5 / 108, 75.3; 65,536 301 / 293, 192 / 259, 175.  In the caches:
// 1,024 rows 7.8, 7.3 / 7.4, 9.8; 2,304 9.8, 7.7 / 12.5, 10.3; 4,360 15.8, 12.7 / 20.0, 19.9; 14,336 40.5, 31.4 / 47.0, 37.1.
// Measured and not kept: half of the table registers (the tables' halves are alike as a rule, but the caller need not give such) 262 and 169 at
// 65,536; three work-groups of LOOP by spilling 286 and 199.
struct WindowRope {
  const float *cos, *sin;
  float q_gain;
  int heads, keep, n_seg, parts;
};
template <int ND, bool LOOP>
__global__ __launch_bounds__(64 * ND, LOOP ? 3 : 5) void attn_fwd_window_rope(const AttnParams p, const WindowRope w) {
  using G = Geo<ND>;
  static_assert(G::TAIL16 && ND >= 4, "four computing waves; the stabiliser in the spare slots");
  constexpr int HD = G::HD, NT = 64 * ND, KT = 4, KK = 2, HALF = HD / 2;
  __shared__ __attribute__((aligned(16))) bf16_t lds_q[64 * G::PK], lds_k[64 * G::PK], lds_v[64 * G::PV];

  // grid (parts, windows): in one dimension 65,535 windows of 205 heads would be 2^32 threads.  Work items are dealt so that all heads of a window meet on one XCD (seg_and_head)
  int seg = blockIdx.y, part = blockIdx.x;
  const unsigned items = (unsigned)w.n_seg * (unsigned)w.parts;
  if (items % 8 == 0) {
    const unsigned at = blockIdx.y * (unsigned)w.parts + blockIdx.x, item = (at & 7) * (items >> 3) + (at >> 3);
    seg = item / (unsigned)w.parts;
    part = item % (unsigned)w.parts;
  }
  const int s0 = p.cu[seg], L = min(p.cu[seg + 1] - s0, 64);
  if (L <= 0) return;
  const int t = threadIdx.x, l = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), g = l >> 4, r = l & 15;
  const int row = t / ND, ch = t % ND;  // this thread's pair of chunks of q and k
  const int vrow = t / G::CH, vch = t % G::CH;  // and its chunks of v: rows vrow and vrow + 32
  const bool valid = row < L;
  // one row pitch for q, k and v; 32-bit byte offsets of the lane from uniform addresses
  const int64_t first = (int64_t)s0 * p.q_stride + (int64_t)part * w.heads * HD;
  char* const Q = static_cast<char*>(const_cast<void*>(p.q)) + 2 * first;
  char* const K = static_cast<char*>(const_cast<void*>(p.k)) + 2 * first;
  const char* const V = static_cast<const char*>(p.v) + 2 * first;
  const unsigned at_qk = (unsigned)((row * p.q_stride + ch * 8) * 2), at_v = (unsigned)((vrow * p.q_stride + vch * 8) * 2);
  auto vec = [](char* base, unsigned at) -> bf16x8& { return *reinterpret_cast<bf16x8*>(base + at); };
  bf16x8 q0, q1, k0, k1, v0, v1;
  const bf16x8 zero = {};
  auto load = [&](int j) {
    q0 = q1 = k0 = k1 = v0 = v1 = zero;
    if (valid) {
      q0 = vec(Q + j * 2 * HD, at_qk);
      q1 = vec(Q + j * 2 * HD + 2 * HALF, at_qk);
      k0 = vec(K + j * 2 * HD, at_qk);
      k1 = vec(K + j * 2 * HD + 2 * HALF, at_qk);
    }
    if (vrow < L) v0 = vec(const_cast<char*>(V) + j * 2 * HD, at_v);
    if (vrow + 32 < L) v1 = vec(const_cast<char*>(V) + 64 * p.q_stride + j * 2 * HD, at_v);
  };
  load(0);
  float c0[8], c1[8], sn0[8], sn1[8];
  {
    const int64_t at = (int64_t)(s0 + (valid ? row : 0)) * HD + ch * 8;
    auto fetch = [&](const float* table, float (&to)[8]) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(table + at), b = *reinterpret_cast<const f32x4*>(table + at + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) to[j] = a[j], to[4 + j] = b[j];
    };
    fetch(w.cos, c0);
    fetch(w.cos + HALF, c1);
    fetch(w.sin, sn0);
    fetch(w.sin + HALF, sn1);
  }
  auto rotate = [&](bf16x8& a, bf16x8& b, float gain) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float oa, ob;
      rope_pair((float)a[j], (float)b[j], c0[j], c1[j], sn0[j], sn1[j], 0, oa, ob);
      a[j] = (bf16_t)(oa * gain);
      b[j] = (bf16_t)(ob * gain);
    }
  };
  const float c = p.scale * LOG2E;
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (bf16_t)1.f;
  const bf16_t one_x = (bf16_t)(g == 0 ? 1.f : 0.f);
  const int q_first = wv * 16, qi = q_first + r;

  for (int j = 0; j < (LOOP ? w.heads : 1); ++j) {
    rotate(q0, q1, w.q_gain);
    rotate(k0, k1, 1.f);
    if (j > 0) __syncthreads();  // the previous head's tiles have been used
    *reinterpret_cast<bf16x8*>(lds_q + row * G::PK + ch * 8) = q0;
    *reinterpret_cast<bf16x8*>(lds_q + row * G::PK + HALF + ch * 8) = q1;
    *reinterpret_cast<bf16x8*>(lds_k + row * G::PK + ch * 8) = k0;
    *reinterpret_cast<bf16x8*>(lds_k + row * G::PK + HALF + ch * 8) = k1;
    *reinterpret_cast<bf16x8*>(lds_v + vrow * G::PV + vch * 8) = v0;
    *reinterpret_cast<bf16x8*>(lds_v + (vrow + 32) * G::PV + vch * 8) = v1;
    if (w.keep && valid) {
      vec(Q + j * 2 * HD, at_qk) = q0;
      vec(Q + j * 2 * HD + 2 * HALF, at_qk) = q1;
      vec(K + j * 2 * HD, at_qk) = k0;
      vec(K + j * 2 * HD + 2 * HALF, at_qk) = k1;
    }
    if (LOOP && j + 1 < w.heads) load(j + 1);
    __syncthreads();
    if (wv >= 4 || q_first >= L) {
      if (!LOOP) return;
      continue;
    }  // for the whole wave; it meets the others at the barriers

    RowFrag<ND> qf;
    load_rowfrag_lds<ND, G::PK>(qf, lds_q, qi, g);
    scale_rowfrag<ND>(qf, c);
    f32x4 s[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      RowFrag<ND> kf;
      load_rowfrag_lds<ND, G::PK>(kf, lds_k, kt * 16 + r, g);
      s[kt] = dot_frag_plus<ND>(kf, qf, one_x, (bf16_t)0.f);
    }
    if (L < 64) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kt * 16 + 4 * g + i >= L) s[kt][i] = -INFINITY;
    }
    float mx = fmaxf(s[0][0], s[0][1]);
    mx = max3(mx, s[0][2], s[0][3]);
#pragma unroll
    for (int kt = 1; kt < KT; ++kt) {
      mx = max3(mx, s[kt][0], s[kt][1]);
      mx = max3(mx, s[kt][2], s[kt][3]);
    }
    const float m = (float)(bf16_t)quad_max(mx);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - m);
    bf16x8 pb[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) pb[kk] = pack8(s[2 * kk], s[2 * kk + 1]);
    f32x4 o[ND], sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        const bf16_t* a0 = lds_v + ((2 * kk) * 16 + 4 * g + (r >> 2)) * G::PV + 16 * dt + 4 * (r & 3);
        o[dt] = mfma32(tr_pair(a0, a0 + 16 * G::PV), pb[kk], o[dt]);
      }
      sum = mfma32(ones, pb[kk], sum);
    }
    // the wave's own rows of the q tile, which no other wave reads, turn the results into whole chunks of rows
    const float inv = 1.f / sum[0];
    bf16_t* turn = lds_q + q_first * G::PK;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      bf16x4 ov;
#pragma unroll
      for (int i = 0; i < 4; ++i) ov[i] = (bf16_t)(o[dt][i] * inv);
      *reinterpret_cast<bf16x4*>(turn + r * G::PK + 16 * dt + 4 * g) = ov;
    }
    const int h = part * w.heads + j;
    if (g == 0 && qi < L) p.lse[(int64_t)h * p.total + s0 + qi] = (m + __builtin_amdgcn_logf(sum[0])) * LN2;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    bf16_t* O = static_cast<bf16_t*>(p.out) + (int64_t)(s0 + q_first) * p.o_stride + (int64_t)h * HD;
#pragma unroll
    for (int i = 0; i < (16 * G::CH + 63) / 64; ++i) {
      const int at = l + 64 * i, rr = at / G::CH, cc = at % G::CH;
      if (rr < 16 && q_first + rr < L) *reinterpret_cast<bf16x8*>(O + (int64_t)rr * p.o_stride + cc * 8) = *reinterpret_cast<const bf16x8*>(turn + rr * G::PK + cc * 8);
    }
  }
}

// ================================================================================================
// Long segments, "wide" kernels: a wave owns 64 rows (two 32-row blocks), four waves per work-group, one
// work-group per CU (up to 512 registers per lane).  Products whose contraction runs over head_dim use
// v_mfma_f32_32x32x16_bf16, so head_dim = 16 * ND is contracted exactly (80 = 5 x 16, no padding); products whose
// contraction runs over rows (keys or queries) use v_mfma_f32_16x16x32_bf16 with head_dim as the 16-wide M dimension.
// A 32x32 accumulator tile (lane: column l%32; register i: row 8*(i/4) + 4*(l/32) + i%4) becomes the B operand of the
// 16x16x32 product after packing to bf16 pairs and four v_permlane16_swap: lanes l and l^16 exchange halves, after
// which lane l holds, for columns l%16 (words 0-3) and 16 + l%16 (words 4-7), the rows
//     base(G) + {0..3}  and  base(G) + 8 + {0..3},   G = l / 16,  base = {0, 16, 4, 20}[G]
// in its eight contraction slots; the transposed left factor is read from LDS with the same row mapping.
// Row statistics ride in the accumulator input of the first MFMA of a chain (a tile of "- statistic" values), so
// exp2 is applied to the MFMA result directly.
// A wave that is alone on its SIMD issues about one instruction per seven cycles and hides no latency by itself:
// matrix and vector instructions are therefore interleaved by hand (__builtin_amdgcn_sched_barrier pins the order),
// LDS fragments are requested a phase before their use, and tiles reach LDS by direct loads three tiles ahead.
// d = a . b + c and d += a . b on v_mfma_f32_32x32x16_bf16 with the result in ordinary vector registers (the compiler's
// own MFMA selection would, in a kernel that uses accumulation registers, place results there and copy them back for
// the vector ALU).  The compiler does not see an MFMA here and inserts no wait states: ordinary instructions may read
// d only after mfma_drain() or after eleven or more other issue slots (every use below sits behind at least two
// further MFMAs).  The B operand `b` sits in accumulation registers (see to_acc_regs): an operand that never changes
// costs no ordinary register that way.
__device__ __forceinline__ void mfma32x32_init(f32x16& d, const bf16x8& a, const u32x4& b, const f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(__builtin_bit_cast(u32x4, a)), "a"(b), "v"(c));
}
__device__ __forceinline__ void mfma32x32_acc(f32x16& d, const bf16x8& a, const u32x4& b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(__builtin_bit_cast(u32x4, a)), "a"(b));
}
// the same two with both operands in ordinary vector registers
__device__ __forceinline__ void mfma32x32_init_v(f32x16& d, const bf16x8& a, const bf16x8& b, const f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(__builtin_bit_cast(u32x4, a)), "v"(__builtin_bit_cast(u32x4, b)), "v"(c));
}
__device__ __forceinline__ void mfma32x32_acc_v(f32x16& d, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(__builtin_bit_cast(u32x4, a)), "v"(__builtin_bit_cast(u32x4, b)));
}
// Moves a fragment into accumulation registers through the lane's own 16-byte LDS slot (a DS load can target them).
__device__ __forceinline__ u32x4 to_acc_regs(const bf16x8& v, float* slot) {
  const unsigned addr = (unsigned)(uintptr_t)slot;
  *reinterpret_cast<volatile bf16x8*>(slot) = v;
  u32x4 r;
  asm volatile("s_waitcnt lgkmcnt(0)\n\tds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=a"(r) : "v"(addr) : "memory");
  return r;
}
__device__ __forceinline__ void mfma_drain() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ f32x16 splat16(float x) {
  f32x16 r;
#pragma unroll
  for (int i = 0; i < 16; ++i) r[i] = x;
  return r;
}
__device__ __forceinline__ unsigned pack2(float a, float b) {
  bf16x2 v = {(bf16_t)a, (bf16_t)b};
  return __builtin_bit_cast(unsigned, v);
}
// lanes l and l^16 trade: afterwards a = the pair's value for the lower lane's column, b = for the upper lane's
__device__ __forceinline__ void swap16(unsigned& a, unsigned& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);  // the compiler spaces it from the writes of a and b
  a = r[0];
  b = r[1];
}
struct BOps {
  bf16x8 lo, hi;  // B operands of the 16x16x32 product for columns l%16 and 16 + l%16 of the 32-column tile
};
__device__ __forceinline__ BOps to_b_operands(unsigned (&w)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) swap16(w[j], w[j + 4]);
  const u32x4 a = {w[0], w[1], w[2], w[3]}, b = {w[4], w[5], w[6], w[7]};
  BOps r;
  r.lo = __builtin_bit_cast(bf16x8, a);
  r.hi = __builtin_bit_cast(bf16x8, b);
  return r;
}
__device__ __forceinline__ bf16x8 scale_frag(bf16x8 v, float c) {
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (bf16_t)((float)v[j] * c);
  return v;
}
__device__ __forceinline__ bf16x8 load_frag_global(const bf16_t* p, bool valid) {
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
  if (valid) v = *reinterpret_cast<const bf16x8*>(p);
  return v;
}
// delta[h, s] = sum_d O[s,h,d] * dO[s,h,d].  One lane per (row, head), 16-byte loads; neighbouring lanes take
// neighbouring heads of the same row, so a wave sweeps contiguous memory.
template <typename T>
__global__ __launch_bounds__(256) void attn_delta_kernel(const T* __restrict__ o, const T* __restrict__ d_o,
                                                         float* __restrict__ delta, int64_t total, int nheads, int hd,
                                                         int64_t o_stride, int64_t do_stride) {
  constexpr int V = mvit_elem<T>::vec;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total * nheads) return;
  const int64_t s = i / nheads;
  const int h = (int)(i % nheads);
  const T* a = o + s * o_stride + (int64_t)h * hd;
  const T* b = d_o + s * do_stride + (int64_t)h * hd;
  float acc = 0.f;
  if (hd % V == 0 && (o_stride % V) == 0 && (do_stride % V) == 0) {
    for (int j = 0; j < hd; j += V) {
      const vec_t x = *reinterpret_cast<const vec_t*>(a + j);
      const vec_t y = *reinterpret_cast<const vec_t*>(b + j);
#pragma unroll
      for (int e = 0; e < V; ++e) acc += to_f32(x[e]) * to_f32(y[e]);
    }
  } else {
    for (int j = 0; j < hd; ++j) acc += to_f32(a[j]) * to_f32(b[j]);
  }
  delta[(int64_t)h * total + s] = acc;
}

// Same result with coalesced traffic: a block takes 16 consecutive rows; every thread multiplies 16-byte chunks
// (consecutive threads, consecutive chunks of a row), parks the chunk sums in LDS, and thread (h, r) then adds the
// chunks of its head in a fixed order and writes delta[h][s0 + r], 16 consecutive floats per head.
template <typename T>
__global__ __launch_bounds__(256) void attn_delta_rows_kernel(const T* __restrict__ o, const T* __restrict__ d_o,
                                                              float* __restrict__ delta, int64_t total, int nheads, int hd,
                                                              int64_t o_stride, int64_t do_stride) {
  constexpr int V = mvit_elem<T>::vec, R = 16;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  extern __shared__ float part[];  // [R][nheads * hd / V]
  const int cph = hd / V, cpr = nheads * cph;
  const int64_t s0 = (int64_t)blockIdx.x * R;
  const int rows = total - s0 < R ? (int)(total - s0) : R;
  for (int q = threadIdx.x; q < rows * cpr; q += 256) {
    const int r = q / cpr, c = q % cpr;
    const vec_t x = *reinterpret_cast<const vec_t*>(o + (s0 + r) * o_stride + (int64_t)c * V);
    const vec_t y = *reinterpret_cast<const vec_t*>(d_o + (s0 + r) * do_stride + (int64_t)c * V);
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < V; ++e) acc += to_f32(x[e]) * to_f32(y[e]);
    part[q] = acc;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nheads * R; t += 256) {
    const int h = t / R, r = t % R;
    if (r >= rows) continue;
    const float* src = part + r * cpr + h * cph;
    float acc = 0.f;
    for (int j = 0; j < cph; ++j) acc += src[j];
    delta[(int64_t)h * total + s0 + r] = acc;
  }
}

// ================================================================================================
// dK, dV.  Block = 64*NWAVES keys of one (segment, head); 32 queries per iteration, Q / dO tiles (and the
// rows' lse, delta) double buffered in LDS with the next tile's loads in flight during the MFMAs.
template <int ND, int NWAVES, int RB>
__global__ __launch_bounds__(64 * NWAVES) void attn_bwd_dkdv_mfma(const AttnParams p) {
  using G = Geo<ND>;
  constexpr int HD = G::HD, BQ = 32, NT = 64 * NWAVES, SPAN = 16 * RB * NWAVES;  // RB 16-row blocks per wave
  constexpr int P = SWZ;  // Q / dO tiles are read as row fragments and through the transposing load
  __shared__ __attribute__((aligned(16))) bf16_t lds_q[2][BQ * P];
  __shared__ __attribute__((aligned(16))) bf16_t lds_do[2][BQ * P];
  __shared__ __attribute__((aligned(16))) float lds_lse[2][BQ];
  __shared__ __attribute__((aligned(16))) float lds_delta[2][BQ];
  __shared__ __attribute__((aligned(8))) bf16_t lds_fold[2][BQ][4];  // -lse2 and -delta per row, each as hi + lo
  constexpr bool FOLD = G::TAIL16;

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_k0 = blockIdx.x * SPAN;
  if (blk_k0 >= L) return;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, g = l >> 4, r = l & 15;
  const int key0 = blk_k0 + wv * 16 * RB;

  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  const bf16_t* DO = static_cast<const bf16_t*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD;
  const float* LSE = p.lse + (int64_t)h * p.total + s0;
  const float* DELTA = p.delta + (int64_t)h * p.total + s0;

  RowFrag<ND> kf[RB], vf[RB];
#pragma unroll
  for (int kb = 0; kb < RB; ++kb) {
    const int ki = key0 + kb * 16 + r;
    load_rowfrag_global<ND>(kf[kb], K + (int64_t)ki * p.k_stride, ki < L, g);
    load_rowfrag_global<ND>(vf[kb], V + (int64_t)ki * p.v_stride, ki < L, g);
  }
  f32x4 dk[RB][ND], dv[RB][ND];
#pragma unroll
  for (int kb = 0; kb < RB; ++kb)
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      dk[kb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
      dv[kb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  const float c = p.scale * LOG2E;
  const bf16_t one_x = (bf16_t)(g == 0 ? 1.f : 0.f);

  TileStager<ND, BQ, P, NT> sq, sdo;
  sq.init(p.q_stride);
  sdo.init(p.do_stride);
  float r_lse = 0.f, r_delta = 0.f;  // threads 0..31 carry one row's statistics
  auto load_stats = [&](int qs, int valid) {
    if (threadIdx.x < BQ) {
      const bool ok = (int)threadIdx.x < valid;
      r_lse = ok ? LSE[qs + threadIdx.x] * LOG2E : 1e30f;  // huge => p = 0 for padded queries
      r_delta = ok ? DELTA[qs + threadIdx.x] : 0.f;
    }
  };
  auto store_stats = [&](int b) {
    if (threadIdx.x < BQ) {
      lds_lse[b][threadIdx.x] = r_lse;
      lds_delta[b][threadIdx.x] = r_delta;
      const HiLo nl = split_hilo(-r_lse), nd = split_hilo(-r_delta);
      lds_fold[b][threadIdx.x][0] = nl.hi;
      lds_fold[b][threadIdx.x][1] = nl.lo;
      lds_fold[b][threadIdx.x][2] = nd.hi;
      lds_fold[b][threadIdx.x][3] = nd.lo;
    }
  };
  sq.load(Q, min(BQ, L));
  sdo.load(DO, min(BQ, L));
  load_stats(0, min(BQ, L));
  sq.scale(c);  // the Q tile holds Q * scale * log2(e): scores leave the MFMA in log2 units
  sq.store(lds_q[0]);
  sdo.store(lds_do[0]);
  store_stats(0);
  __syncthreads();

  int buf = 0;
  for (int qs = 0; qs < L; qs += BQ) {
    const bool has_next = qs + BQ < L;
    if (has_next) {
      const int nv = min(BQ, L - qs - BQ);
      sq.load(Q + (int64_t)(qs + BQ) * p.q_stride, nv);
      sdo.load(DO + (int64_t)(qs + BQ) * p.do_stride, nv);
      load_stats(qs + BQ, nv);
    }
    const bf16_t* tq = lds_q[buf];
    const bf16_t* tdo = lds_do[buf];

    RowFrag<ND> qa[2], da[2];  // natural-layout A operands: row = query t*16 + r
    bf16x8 qt[ND], dt_[ND];    // transposed A operands: row = head-dim 16*dt + r, slots = queries
    f32x4 lse2[2], dl[2];
    bf16x4 fold[2];  // FOLD: (-lse2 hi, lo, -delta hi, lo) of query t*16 + r, riding in the padded MFMA's spare slots
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      load_rowfrag_lds<ND, P>(qa[t], tq, t * 16 + r, g);
      load_rowfrag_lds<ND, P>(da[t], tdo, t * 16 + r, g);
      if (FOLD) {
        fold[t] = *reinterpret_cast<const bf16x4*>(lds_fold[buf][t * 16 + r]);
        if (g != 0) fold[t] = bf16x4{(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
      } else {
        lse2[t] = *reinterpret_cast<const f32x4*>(lds_lse[buf] + t * 16 + 4 * g);
        dl[t] = *reinterpret_cast<const f32x4*>(lds_delta[buf] + t * 16 + 4 * g);
      }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      qt[d] = tr_block<P>(tq, 0, d, g, r);
      dt_[d] = tr_block<P>(tdo, 0, d, g, r);
    }
#pragma unroll
    for (int kb = 0; kb < RB; ++kb) {
      f32x4 pv[2], ds[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        // S[q = t*16+4g+i][key = kb*16+r] in log2 units, and dP in the same layout
        if constexpr (FOLD) {
          const f32x4 s = dot_frag_plus2<ND>(qa[t], kf[kb], fold[t][0], fold[t][1], one_x, one_x);   // - lse2
          const f32x4 dp = dot_frag_plus2<ND>(da[t], vf[kb], fold[t][2], fold[t][3], one_x, one_x);  // - delta
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float e = __builtin_amdgcn_exp2f(s[i]);
            pv[t][i] = e;
            ds[t][i] = e * dp[i];
          }
        } else {
          const f32x4 s = dot_frag<ND>(qa[t], kf[kb]);
          const f32x4 dp = dot_frag<ND>(da[t], vf[kb]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float e = __builtin_amdgcn_exp2f(s[i] - lse2[t][i]);
            pv[t][i] = e;
            ds[t][i] = e * (dp[i] - dl[t][i]);
          }
        }
      }
      const bf16x8 pb = pack8(pv[0], pv[1]);
      const bf16x8 dsb = pack8(ds[0], ds[1]);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        dv[kb][d] = mfma32(dt_[d], pb, dv[kb][d]);
        dk[kb][d] = mfma32(qt[d], dsb, dk[kb][d]);
      }
    }
    if (has_next) {
      sq.scale(c);
      sq.store(lds_q[buf ^ 1]);
      sdo.store(lds_do[buf ^ 1]);
      store_stats(buf ^ 1);
    }
    __syncthreads();
    buf ^= 1;
  }

  bf16_t* DK = static_cast<bf16_t*>(p.dk) + (int64_t)s0 * p.dk_stride + (int64_t)h * HD;
  bf16_t* DV = static_cast<bf16_t*>(p.dv) + (int64_t)s0 * p.dv_stride + (int64_t)h * HD;
#pragma unroll
  for (int kb = 0; kb < RB; ++kb) {
    const int ki = key0 + kb * 16 + r;
    if (ki < L) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        bf16x4 a, b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] = (bf16_t)(dk[kb][d][i] * LN2);  // dS^T (Q scale log2e) / log2e
          b[i] = (bf16_t)dv[kb][d][i];
        }
        *reinterpret_cast<bf16x4*>(DK + (int64_t)ki * p.dk_stride + 16 * d + 4 * g) = a;
        *reinterpret_cast<bf16x4*>(DV + (int64_t)ki * p.dv_stride + 16 * d + 4 * g) = b;
      }
    }
  }
}

// ================================================================================================
// LDS tile layout of the wide backward kernels: 32 rows of 256 bytes (16 slots of 16 bytes, 10 of them used at head_dim
// 80); chunk c of row r lives in slot c ^ xs(r), xs(r) = 2*(r & 3) + ((r >> 2) & 1).  Eight consecutive rows put one
// chunk index into eight different slots (16-byte row-fragment reads), four consecutive rows put one pair of chunks
// into four different 32-byte windows (transposing reads): neither pattern has bank conflicts.  The tile is filled by
// global_load_lds_dwordx4 (16 bytes per lane straight into LDS at M0 + 16 * lane, no staging registers): lane i of
// instruction j fills slot 64*j + i, i.e. it fetches chunk (i & 15) ^ xs(row) of row 4*j + i/16.
constexpr int XS_PITCH = 128;                 // elements per LDS row
constexpr int XS_TILE = 32 * XS_PITCH;        // elements per 32-row tile (8 KiB)
__device__ __forceinline__ int xs(int row) { return ((row & 3) << 1) | ((row >> 2) & 1); }
__device__ __forceinline__ bf16x8 xs_row_frag(const bf16_t* tile, int row, int s, int h) {
  return *reinterpret_cast<const bf16x8*>(tile + row * XS_PITCH + (((2 * s + h) ^ xs(row)) << 3));
}
// transposed A operand (see tr_block_wide) of head-dim block d from rows base(G) + (r >> 2) and + 8
__device__ __forceinline__ bf16x8 xs_tr_block(const bf16_t* tile, int d, int G, int r) {
  const int row = 16 * (G & 1) + 4 * (G >> 1) + (r >> 2);
  const bf16_t* a = tile + row * XS_PITCH + (((2 * d + ((r & 3) >> 1)) ^ xs(row)) << 3) + 4 * (r & 1);
  return tr_pair(a, a + 8 * XS_PITCH);  // xs(row + 8) == xs(row)
}
// wave-uniform values as scalars (the compiler cannot prove uniformity of values derived from the wave index)
__device__ __forceinline__ unsigned uniform_u32(unsigned x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ const void* uniform_ptr(const void* q) {
  const uint64_t v = (uint64_t)(uintptr_t)q;
  const uint64_t u = (uint64_t)uniform_u32((unsigned)v) | ((uint64_t)uniform_u32((unsigned)(v >> 32)) << 32);
  return (const void*)(uintptr_t)u;
}
// lds_addr and base must be wave-uniform (scalar registers)
__device__ __forceinline__ void lds_direct_16(unsigned lds_addr, unsigned voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory");
}
__device__ __forceinline__ void lds_direct_4(unsigned lds_addr, unsigned voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// q_scaled[s, h, :] = bf16(q[s, h, :] * c) for the wide backward kernels (the forward rounds Q * scale * log2(e) to
// bf16 the same way, so the recomputed probabilities match the forward's), and the row statistics in the form the
// MFMA accumulators are initialised with: nlse2 = - lse * log2(e), ndelta = - delta.
__global__ __launch_bounds__(256) void attn_bwd_prepare_kernel(const bf16_t* __restrict__ q, int64_t q_stride, bf16_t* __restrict__ qs,
                                                               int64_t qs_stride, int64_t total, int cols, float c,
                                                               const float* __restrict__ lse, const float* __restrict__ delta,
                                                               float* __restrict__ nlse2, float* __restrict__ ndelta, int64_t nstat) {
  const int cpr = cols / 8;
  const int64_t nchunk = total * cpr;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nchunk; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / cpr;
    const int ch = (int)(i % cpr);
    bf16x8 v = *reinterpret_cast<const bf16x8*>(q + row * q_stride + ch * 8);
    *reinterpret_cast<bf16x8*>(qs + row * qs_stride + ch * 8) = scale_frag(v, c);
  }
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nstat; i += (int64_t)gridDim.x * 256) {
    nlse2[i] = -lse[i] * LOG2E;
    ndelta[i] = -delta[i];
  }
}

// ================================================================================================
// dK, dV for long segments, "wide" form: a wave owns 64 keys (two groups of 32), four waves = 256 keys per work-group,
// one work-group per CU.  K / V fragments of the wave's keys and the 2 x 80 accumulators live in accumulation
// registers; pre-scaled Q / dO tiles of 32 queries and their statistics stream through an LDS ring of four tiles,
// written by direct global -> LDS loads three tiles ahead.  Per tile and key group:
//   S = Q K^T - lse2, dP = dO V^T - delta   (v_mfma_f32_32x32x16_bf16, head_dim contracted exactly; the first MFMA of
//                                            a chain takes the tile of "- statistic" values as its accumulator input)
//   P = exp2(S), dS = P * dP                 (vector ALU), packed to bf16 and turned into B operands by lane swaps
//   dV^T += dO^T P, dK^T += Q^T dS           (v_mfma_f32_16x16x32_bf16, transposed left factors read from LDS)
// A wave is alone on its SIMD, so matrix and vector instructions are interleaved by hand: the second key group's
// score MFMAs run under the first group's exp / pack, the first group's dV / dK MFMAs under the second group's.
template <int ND>
__global__ __launch_bounds__(256, 1) void attn_bwd_dkdv_wide(const AttnParams p) {
  static_assert(ND == 5, "the hand-placed instruction order below is laid out for head_dim 80");
  using G = Geo<ND>;
  constexpr int HD = G::HD, BQ = 32, NT = 256, RING = 4;
  __shared__ __attribute__((aligned(1024))) bf16_t lds_q[RING][XS_TILE];
  __shared__ __attribute__((aligned(1024))) bf16_t lds_do[RING][XS_TILE];
  __shared__ __attribute__((aligned(256))) float lds_nlse[RING][64];  // - lse * log2(e) per query of the tile (32 used)
  __shared__ __attribute__((aligned(256))) float lds_ndel[RING][64];  // - delta
  __shared__ __attribute__((aligned(16))) float lds_fix[NT * 4];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_k0 = blockIdx.x * 256;
  if (blk_k0 >= L) return;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hh = l >> 5, c32 = l & 31, G4 = l >> 4, r = l & 15;
  const int key0 = blk_k0 + wv * 64;

  const bf16_t* QS = static_cast<const bf16_t*>(p.q_scaled) + (int64_t)s0 * p.qs_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  const bf16_t* DO = static_cast<const bf16_t*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD;
  const float* NLSE = p.nlse2 + (int64_t)h * p.total + s0;
  const float* NDEL = p.ndelta + (int64_t)h * p.total + s0;

  // B operands of the score products (column = key 32*kg + l%32, contraction = head-dim 16*s + 8*(l/32) ..)
  u32x4 kf[2][ND], vf[2][ND];
#pragma unroll
  for (int kg = 0; kg < 2; ++kg) {
    const int ki = key0 + 32 * kg + c32;
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      kf[kg][s] = to_acc_regs(load_frag_global(K + (int64_t)ki * p.k_stride + 16 * s + 8 * hh, ki < L), lds_fix + threadIdx.x * 4);
      vf[kg][s] = to_acc_regs(load_frag_global(V + (int64_t)ki * p.v_stride + 16 * s + 8 * hh, ki < L), lds_fix + threadIdx.x * 4);
    }
  }
  f32x4 dk[4][ND], dv[4][ND];  // [16-key block][16-wide head-dim block]: lane = key l%16, registers = head-dim 4*(l/16) + i
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dk[kb][d] = f32x4{0.f, 0.f, 0.f, 0.f};
      dv[kb][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  // Direct global -> LDS loads: per tile and tensor eight 1 KiB instructions, two of them this wave's; wave 0 and 1 also
  // fetch one array of statistics each.  Rows past the segment end are read from the segment's last row (they stay
  // finite and meet a probability of exactly zero: their statistics are overwritten before use).
  int trow[2], tchunk[2];
  unsigned voff_q[2], voff_do[2];  // byte offsets of this lane's chunks from the tile's first row (tiles without a tail)
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int slot = 64 * (2 * wv + j) + l;
    trow[j] = slot >> 4;
    tchunk[j] = min(((slot & 15) ^ xs(trow[j])), 2 * ND - 1);  // padding slots re-fetch the last chunk
    voff_q[j] = (unsigned)(trow[j] * (int)p.qs_stride * 2 + tchunk[j] * 16);
    voff_do[j] = (unsigned)(trow[j] * (int)p.do_stride * 2 + tchunk[j] * 16);
  }
  const unsigned lds_q0 = (unsigned)(uintptr_t)&lds_q[0][0], lds_do0 = (unsigned)(uintptr_t)&lds_do[0][0];
  const unsigned lds_nl0 = (unsigned)(uintptr_t)&lds_nlse[0][0], lds_nd0 = (unsigned)(uintptr_t)&lds_ndel[0][0];
  auto request_tile = [&](int qs, int slot) {  // 5 (waves 0, 1) or 4 load instructions
    if (qs >= L) return;
    const int last = L - 1 - qs;  // last valid row of the tile (>= 0)
    const bool tail = last < BQ - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      unsigned vq = voff_q[j], vd = voff_do[j];
      if (tail) {
        const int row = min(trow[j], last);
        vq = (unsigned)(row * (int)p.qs_stride * 2 + tchunk[j] * 16);
        vd = (unsigned)(row * (int)p.do_stride * 2 + tchunk[j] * 16);
      }
      lds_direct_16(lds_q0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, vq, QS + (int64_t)qs * p.qs_stride);
      lds_direct_16(lds_do0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, vd, DO + (int64_t)qs * p.do_stride);
    }
    if (wv < 2) lds_direct_4((wv == 0 ? lds_nl0 : lds_nd0) + slot * 256, (unsigned)(min(l, last) * 4), (wv == 0 ? NLSE : NDEL) + qs);
  };
  auto request_inner_tile = [&](int qs, int slot) {  // the same for a tile of 32 rows inside the segment
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      lds_direct_16(lds_q0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, voff_q[j], QS + (int64_t)qs * p.qs_stride);
      lds_direct_16(lds_do0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, voff_do[j], DO + (int64_t)qs * p.do_stride);
    }
    // every wave fetches one array of statistics (waves 2 and 3 the same bytes as 0 and 1): five loads per wave and
    // tile, so the wait at the end of the step is the same instruction for all of them
    lds_direct_4(((wv & 1) == 0 ? lds_nl0 : lds_nd0) + slot * 256, (unsigned)(l < BQ ? l * 4 : (BQ - 1) * 4), ((wv & 1) == 0 ? NLSE : NDEL) + qs);
  };
  // statistics of rows past the segment end: probability zero, no contribution
  auto fix_tail = [&](int qs, int slot) {
    if (qs < L && qs + BQ > L && threadIdx.x < BQ && qs + (int)threadIdx.x >= L) {
      lds_nlse[slot][threadIdx.x] = -1e30f;
      lds_ndel[slot][threadIdx.x] = 0.f;
    }
  };
  request_tile(0, 0);
  request_tile(BQ, 1);
  request_tile(2 * BQ, 2);
  wait_vmcnt<0>();
  fix_tail(0, 0);
  fix_tail(BQ, 1);
  fix_tail(2 * BQ, 2);
  __syncthreads();

  bf16x8 qa[ND], da[ND];  // A operands of the score products: row = query l%32 of the tile
  f32x16 nl, nd;          // - lse2 and - delta of the tile's queries in accumulator layout (register i: query 8*(i/4) + 4*(l/32) + i%4)
  f32x16 sc[2], dp[2];    // per key group: S - lse2 and dP - delta, lane = key l%32
  auto fetch_rows = [&](int slot) {
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      qa[s] = xs_row_frag(lds_q[slot], c32, s, hh);
      da[s] = xs_row_frag(lds_do[slot], c32, s, hh);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(&lds_nlse[slot][8 * j + 4 * hh]);
      const f32x4 b = *reinterpret_cast<const f32x4*>(&lds_ndel[slot][8 * j + 4 * hh]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        nl[4 * j + i] = a[i];
        nd[4 * j + i] = b[i];
      }
    }
  };
  fetch_rows(0);
  // the same reads in five parts (one per head-dim step), to sit between MFMAs
  auto fetch_rows_part = [&](int slot, int s) {
    qa[s] = xs_row_frag(lds_q[slot], c32, s, hh);
    da[s] = xs_row_frag(lds_do[slot], c32, s, hh);
    if (s < 4) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(&lds_nlse[slot][8 * s + 4 * hh]);
      const f32x4 b = *reinterpret_cast<const f32x4*>(&lds_ndel[slot][8 * s + 4 * hh]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        nl[4 * s + i] = a[i];
        nd[4 * s + i] = b[i];
      }
    }
  };

  // One step of the loop over tiles.  INNER: tile it+3 lies wholly inside the segment, so its request needs no bounds,
  // the wait at the end always leaves one tile in flight and no statistics need fixing: the steady state of a long
  // segment runs without the scalar bookkeeping of the general step, which only the last tiles take.
  int it = 0, qs = 0;
  auto step = [&](auto inner_tag) {
    constexpr bool INNER = decltype(inner_tag)::value;
    const int b0 = it & 3, b1 = (it + 1) & 3, b3 = (it + 3) & 3;
    // tile it+3 is requested into the slot that tile it-1 left (every wave is past the barrier that ended iteration it-1)
    if constexpr (INNER) request_inner_tile(qs + 3 * BQ, b3);
    else request_tile(qs + 3 * BQ, b3);
    // ---- phase 1: score products of key group 0; the transposed left factors that phase 3 needs are read from LDS
    // between the MFMAs
    bf16x8 qt[ND], dt_[ND];
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      if (s == 0) {
        mfma32x32_init(sc[0], qa[0], kf[0][0], nl);
        mfma32x32_init(dp[0], da[0], vf[0][0], nd);
      } else {
        mfma32x32_acc(sc[0], qa[s], kf[0][s]);
        mfma32x32_acc(dp[0], da[s], vf[0][s]);
      }
      qt[s] = xs_tr_block(lds_q[b0], s, G4, r);
      dt_[s] = xs_tr_block(lds_do[b0], s, G4, r);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 2: score products of key group 1 under the vector work of group 0
    unsigned pw[8], dw[8];
    auto words = [&](int j) {
      const float e0 = __builtin_amdgcn_exp2f(sc[0][2 * j]), e1 = __builtin_amdgcn_exp2f(sc[0][2 * j + 1]);
      pw[j] = pack2(e0, e1);
      dw[j] = pack2(e0 * dp[0][2 * j], e1 * dp[0][2 * j + 1]);
    };
    BOps pb, db;
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      // from the second step on the vector work is split between the two MFMAs: a wave issues in order, so whatever
      // stands behind a second MFMA waits with it for the pipe, and only work placed between the two fills the first
      // one's shadow.  (Step 0 keeps both MFMAs first: they separate group 0's last score MFMAs from the first read of
      // their results, which the compiler does not guard.)
      if (s == 0) {
        mfma32x32_init(sc[1], qa[0], kf[1][0], nl);
        mfma32x32_init(dp[1], da[0], vf[1][0], nd);
        words(0);
        words(1);
      } else if (s < 4) {
        mfma32x32_acc(sc[1], qa[s], kf[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        words(2 * s);
        __builtin_amdgcn_sched_barrier(0);
        mfma32x32_acc(dp[1], da[s], vf[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        words(2 * s + 1);
      } else {  // the lane swaps of group 0 under the last two score MFMAs
        mfma32x32_acc(sc[1], qa[s], kf[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        pb = to_b_operands(pw);
        __builtin_amdgcn_sched_barrier(0);
        mfma32x32_acc(dp[1], da[s], vf[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        db = to_b_operands(dw);
        asm volatile("s_nop 1");
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 3: dV / dK of key group 0 under the vector work of group 1
    unsigned pw1[8], dw1[8];
    auto words1 = [&](int j) {
      const float e0 = __builtin_amdgcn_exp2f(sc[1][2 * j]), e1 = __builtin_amdgcn_exp2f(sc[1][2 * j + 1]);
      pw1[j] = pack2(e0, e1);
      dw1[j] = pack2(e0 * dp[1][2 * j], e1 * dp[1][2 * j + 1]);
    };
    BOps pb1, db1;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dv[0][d] = mfma32(dt_[d], pb.lo, dv[0][d]);
      dk[0][d] = mfma32(qt[d], db.lo, dk[0][d]);
      dv[1][d] = mfma32(dt_[d], pb.hi, dv[1][d]);
      dk[1][d] = mfma32(qt[d], db.hi, dk[1][d]);
      if (d < 4) {
        words1(2 * d);
        words1(2 * d + 1);
      } else {
        pb1 = to_b_operands(pw1);
        db1 = to_b_operands(dw1);
        asm volatile("s_nop 1");
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 4: dV / dK of key group 1 under the fragment reads of the next tile; the barrier is waited for while
    // these MFMAs drain
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dv[2][d] = mfma32(dt_[d], pb1.lo, dv[2][d]);
      dk[2][d] = mfma32(qt[d], db1.lo, dk[2][d]);
      dv[3][d] = mfma32(dt_[d], pb1.hi, dv[3][d]);
      dk[3][d] = mfma32(qt[d], db1.hi, dk[3][d]);
      fetch_rows_part(b1, d);
      __builtin_amdgcn_sched_barrier(0);
    }
    // tile it+2 (requested in iteration it-1) must have landed before any wave reads it in the next iteration; the
    // loads requested in this iteration (five by waves 0 and 1, four by the others) may stay in flight
    if constexpr (INNER) {
      wait_vmcnt<5>();
    } else if (qs + 3 * BQ < L) {
      if (wv < 2) wait_vmcnt<5>();
      else wait_vmcnt<4>();
    } else {
      wait_vmcnt<0>();
    }
    if constexpr (!INNER) fix_tail(qs + 2 * BQ, (it + 2) & 3);
    __syncthreads();
  };
  for (; qs + 4 * BQ <= L; qs += BQ, ++it) step(std::true_type{});
  for (; qs < L; qs += BQ, ++it) step(std::false_type{});

  bf16_t* DK = static_cast<bf16_t*>(p.dk) + (int64_t)s0 * p.dk_stride + (int64_t)h * HD;
  bf16_t* DV = static_cast<bf16_t*>(p.dv) + (int64_t)s0 * p.dv_stride + (int64_t)h * HD;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int ki = key0 + kb * 16 + r;
    if (ki < L) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        bf16x4 a, b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] = (bf16_t)(dk[kb][d][i] * LN2);  // dS^T (Q scale log2e) / log2e
          b[i] = (bf16_t)dv[kb][d][i];
        }
        *reinterpret_cast<bf16x4*>(DK + (int64_t)ki * p.dk_stride + 16 * d + 4 * G4) = a;
        *reinterpret_cast<bf16x4*>(DV + (int64_t)ki * p.dv_stride + 16 * d + 4 * G4) = b;
      }
    }
  }
}

// ================================================================================================
// Forward for long segments on v_mfma_f32_32x32x16_bf16 only.  A wave owns two blocks of 32 queries (the N dimension of
// every product), eight waves = 512 queries per work-group, one work-group per CU (two waves per SIMD, ~250 registers).
// Per tile of 32 keys and query block:
//   S^T = K Q'^T          5 MFMAs, head_dim contracted exactly; A = a row fragment of the K tile, B = Q' in registers
//                         the accumulator input is a tile of -m (the running stabiliser), so scores arrive stabilised
//   P^T = exp2(S^T)       the accumulator layout (lane: query l%32; register i: key 8*(i/4) + 4*(l/32) + i%4) is, after
//                         packing pairs, already the B operand of the next product: registers 0-7 are contraction
//                         step 0 (keys 0-15), registers 8-15 step 1, with contraction slot j of lane half hh standing
//                         for key 16*ks + 4*hh + (j < 4 ? j : j + 4); no lane exchange is needed
//   O^T += V^T P^T        6 MFMAs: head_dim padded to 96 rows (three 32-row blocks).  Columns 80-95 of the V tile in LDS
//                         hold ones, so rows 80-95 of O^T accumulate the row sums of P for free.
// The transposed left factor V^T is read from the natural [key][head_dim] tile with the transposing LDS load using the
// same slot -> key map.  K / V tiles reach a four-slot LDS ring by direct global -> LDS loads three tiles ahead; lanes
// that would fill the padding chunks are switched off, so the ones written once at the start stay in place.
// 16-byte chunk c of row r of a tile sits in slot c ^ xs16(r): sixteen consecutive rows put one chunk index into sixteen
// different slots (row fragments), four consecutive rows put a pair of chunks into four different 32-byte windows
// (transposing reads).
__device__ __forceinline__ int xs16(int row) { return ((row & 3) << 1) | ((row >> 2) & 1) | (((row >> 3) & 1) << 3); }
__device__ __forceinline__ f32x16 mfma32x32(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// v_max3_f32 / v_max_f32 as they are: the compiler's fmaxf first quiets a possible signalling NaN in every operand
// (one more instruction each); scores are finite or -inf
__device__ __forceinline__ float raw_max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float raw_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// the full maximum of a value held by lanes l and l ^ 32 (the two halves hold different keys of the same query)
__device__ __forceinline__ float max_across_halves(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));  // a = low half's value, b = high half's, in every lane
  return raw_max(a, b);
}

template <int ND>
__global__ __launch_bounds__(512, 1) void attn_fwd_x32(const AttnParams p) {
  static_assert(ND == 5, "the padded third block of head_dim and its ones columns are laid out for head_dim 80");
  using G = Geo<ND>;
  constexpr int HD = G::HD, BK = 32, RING = 4, QB = 2, WQ = 32 * QB;  // QB blocks of 32 queries per wave
  constexpr float TAU = 2.f;  // the stabiliser only moves when a score exceeds it by more than TAU (log2 units)
  __shared__ __attribute__((aligned(1024))) bf16_t lds_k[RING][XS_TILE];
  __shared__ __attribute__((aligned(1024))) bf16_t lds_v[RING][XS_TILE];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_q0 = blockIdx.x * (8 * WQ);
  if (blk_q0 >= L) return;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hh = l >> 5, c32 = l & 31, G4 = l >> 4, r = l & 15;
  const int q_first = blk_q0 + wv * WQ + c32;  // block qb: query q_first + 32 * qb

  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;

  // ones in chunks 10 and 11 (head_dim 80 .. 95) of every row of every V slot
  for (int i = threadIdx.x; i < RING * 32 * 2; i += 512) {
    const int slot = i >> 6, row = (i >> 1) & 31, ch = 10 + (i & 1);  // i < RING * 64
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = (bf16_t)1.f;
    *reinterpret_cast<bf16x8*>(&lds_v[slot][row * XS_PITCH + ((ch ^ xs16(row)) << 3)]) = ones;
  }

  // B operand of the score product: Q * scale * log2(e), rounded to bf16 (scores then come out in log2 units)
  bf16x8 qf[QB][ND];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      const int qi = q_first + 32 * qb;
      qf[qb][s] = scale_frag(load_frag_global(Q + (int64_t)qi * p.q_stride + 16 * s + 8 * hh, qi < L), p.scale * LOG2E);
    }

  // direct global -> LDS loads: one 1 KiB instruction per wave, tensor and tile (rows 4*wv .. 4*wv + 3)
  const int trow = 4 * wv + (l >> 4);
  const int tchunk = (l & 15) ^ xs16(trow);
  const bool tactive = tchunk < 2 * ND;
  const unsigned lds_k0 = (unsigned)(uintptr_t)&lds_k[0][0], lds_v0 = (unsigned)(uintptr_t)&lds_v[0][0];
  auto request_tile = [&](int ks, int slot) {
    if (ks >= L) return;
    const int row = min(trow, L - 1 - ks);  // rows past the segment end repeat its last row; their scores are masked
    const unsigned vk = (unsigned)(row * (int)p.k_stride * 2 + tchunk * 16), vv = (unsigned)(row * (int)p.v_stride * 2 + tchunk * 16);
    if (tactive) {
      lds_direct_16(lds_k0 + slot * (XS_TILE * 2) + wv * 1024, vk, K + (int64_t)ks * p.k_stride);
      lds_direct_16(lds_v0 + slot * (XS_TILE * 2) + wv * 1024, vv, V + (int64_t)ks * p.v_stride);
    }
  };
  f32x16 o[QB][3];  // O^T: block mt, register i = head_dim 32*mt + 8*(i/4) + 4*hh + i%4 of query l%32; rows 80-95 = row sum of P
  float m_run[QB];
  f32x16 negm[QB];  // - m_run in every register: the accumulator input of the score product, so that scores arrive stabilised

  // V^T fragment (block mt of head_dim, contraction step ks): lane i of 16-lane group g4 supplies four consecutive
  // head-dim values of one key row; the transposing load hands lane j of the group head_dim 32*mt + 16*(g4 & 1) + j
  // for the four keys 16*ks + 4*(g4 >> 1) + {0..3}, a second load the keys 8 further on
  auto vt_frag = [&](const bf16_t* tile, int mt, int ks) {
    const int row = 16 * ks + 4 * (G4 >> 1) + (r >> 2);
    const int ch = 4 * mt + 2 * (G4 & 1) + ((r & 3) >> 1);
    const bf16_t* a0 = tile + row * XS_PITCH + ((ch ^ xs16(row)) << 3) + 4 * (r & 1);
    const bf16_t* a1 = tile + (row + 8) * XS_PITCH + ((ch ^ xs16(row + 8)) << 3) + 4 * (r & 1);
    return tr_pair(a0, a1);
  };

  // K row fragments (A operand of the score product) are fetched one tile ahead: tile it+1 is complete in LDS from the
  // start of iteration it on (see the wait before the barrier), so its fragments are requested under the last MFMAs of
  // tile it and no LDS latency opens the next iteration
  bf16x8 kf[ND];
  auto fetch_k = [&](int slot) {
#pragma unroll
    for (int s = 0; s < ND; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(lds_k[slot] + c32 * XS_PITCH + (((2 * s + hh) ^ xs16(c32)) << 3));
  };
  // One tile of 32 keys.  CHECK: the tile's row maxima are taken and the stabiliser follows them.  The first sweep over
  // the keys does that for the first tile only and then leaves the stabiliser where it is: exp2 of a bf16 / fp32 value has
  // 250 binary orders of range, so a later score may exceed the first tile's maximum by more than a hundred (base-2
  // units) before anything overflows, and scores far below it vanish exactly as they would against the true maximum.
  // A row whose sums did overflow is seen at the end (an infinity or NaN in its accumulators) and the work-group sweeps
  // again with the maxima taken on every tile.
  int it = 0;
  auto tile_step = [&](int k0, auto check_tag) {
    constexpr bool CHECK = decltype(check_tag)::value;
    const int b0 = it & (RING - 1), b1 = (it + 1) & (RING - 1), b3 = (it + 3) & (RING - 1);
    request_tile(k0 + 3 * BK, b3);
    const bf16_t* tv = lds_v[b0];
    f32x16 sc[QB];
    unsigned pw[QB][8];
    auto mask_tail = [&](int qb) {
      if (k0 + BK > L) {  // last, partial tile
        asm volatile("" ::: "memory");
        const int valid = L - k0;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (4 * hh >= valid - (8 * (i >> 2) + (i & 3))) sc[qb][i] = -INFINITY;  // key 8*(i/4) + 4*hh + i%4 >= valid
      }
    };
    auto row_max = [&](int qb) {
      float mx = raw_max3(sc[qb][0], sc[qb][1], sc[qb][2]);
#pragma unroll
      for (int i = 3; i < 15; i += 2) mx = raw_max3(mx, sc[qb][i], sc[qb][i + 1]);
      mx = raw_max(mx, sc[qb][15]);
      return max_across_halves(mx);
    };
    // mx = the largest score of the tile minus the current stabiliser; the stabiliser moves when that excess is above
    // TAU for some query of the wave (rare after the first tiles): accumulators and this tile's scores are rebased
    auto rescale = [&](int qb, float mx) {
      const bool grow = k0 == 0 || mx > TAU;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        asm volatile("" ::: "memory");
        const float delta = grow ? mx : 0.f;
        const float alpha = k0 == 0 ? 1.f : __builtin_amdgcn_exp2f(-delta);
        m_run[qb] += delta;
        negm[qb] = splat16(-m_run[qb]);
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[qb][i] -= delta;
#pragma unroll
        for (int mt = 0; mt < 3; ++mt) o[qb][mt] *= alpha;
      }
    };
    auto p_operand = [&](int qb, int ks) {
      const u32x4 w4 = {pw[qb][4 * ks], pw[qb][4 * ks + 1], pw[qb][4 * ks + 2], pw[qb][4 * ks + 3]};
      return __builtin_bit_cast(bf16x8, w4);
    };
    {
      // Two query blocks per wave, software-pipelined by hand: the second block's score MFMAs run under the first
      // block's softmax arithmetic, the first block's P.V MFMAs under the second block's; scheduling barriers pin the
      // order.  Only the first score MFMA of each block is inline assembly (its accumulator input is the stabiliser
      // tile, which the compiler's own MFMA selection would first copy into the result registers).  The compiler sees
      // no MFMA there and inserts no wait states for its result: the two are issued together, so that a whole MFMA
      // separates each from the accumulating MFMA that reads its result; all later dependencies are the compiler's.
      auto words = [&](int qb, int w0, int w1) {
#pragma unroll
        for (int w = w0; w < w1; ++w) pw[qb][w] = pack2(__builtin_amdgcn_exp2f(sc[qb][2 * w]), __builtin_amdgcn_exp2f(sc[qb][2 * w + 1]));
      };
      mfma32x32_init_v(sc[0], kf[0], qf[0][0], negm[0]);
      mfma32x32_init_v(sc[1], kf[0], qf[1][0], negm[1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 1; s < ND; ++s) sc[0] = mfma32x32(kf[s], qf[0][s], sc[0]);
      sc[1] = mfma32x32(kf[1], qf[1][1], sc[1]);
      __builtin_amdgcn_sched_barrier(0);
      mask_tail(0);
      if constexpr (CHECK) rescale(0, row_max(0));
      __builtin_amdgcn_sched_barrier(0);
      sc[1] = mfma32x32(kf[2], qf[1][2], sc[1]);
      __builtin_amdgcn_sched_barrier(0);
      words(0, 0, 3);
      __builtin_amdgcn_sched_barrier(0);
      sc[1] = mfma32x32(kf[3], qf[1][3], sc[1]);
      __builtin_amdgcn_sched_barrier(0);
      words(0, 3, 6);
      __builtin_amdgcn_sched_barrier(0);
      sc[1] = mfma32x32(kf[4], qf[1][4], sc[1]);
      __builtin_amdgcn_sched_barrier(0);
      words(0, 6, 8);
      // the V fragments (kept for both blocks) and the first two P.V MFMAs of block 0 separate the last score MFMA of
      // block 1 from the first read of its result
      bf16x8 vf[6];
#pragma unroll
      for (int n = 0; n < 6; ++n) vf[n] = vt_frag(tv, n % 3, n / 3);
      o[0][0] = mfma32x32(vf[0], p_operand(0, 0), o[0][0]);
      o[0][1] = mfma32x32(vf[1], p_operand(0, 0), o[0][1]);
      __builtin_amdgcn_sched_barrier(0);
      mask_tail(1);
      if constexpr (CHECK) rescale(1, row_max(1));
      __builtin_amdgcn_sched_barrier(0);
      o[0][2] = mfma32x32(vf[2], p_operand(0, 0), o[0][2]);
      __builtin_amdgcn_sched_barrier(0);
      words(1, 0, 2);
      __builtin_amdgcn_sched_barrier(0);
      o[0][0] = mfma32x32(vf[3], p_operand(0, 1), o[0][0]);
      __builtin_amdgcn_sched_barrier(0);
      words(1, 2, 4);
      __builtin_amdgcn_sched_barrier(0);
      o[0][1] = mfma32x32(vf[4], p_operand(0, 1), o[0][1]);
      __builtin_amdgcn_sched_barrier(0);
      words(1, 4, 6);
      __builtin_amdgcn_sched_barrier(0);
      o[0][2] = mfma32x32(vf[5], p_operand(0, 1), o[0][2]);
      __builtin_amdgcn_sched_barrier(0);
      words(1, 6, 8);
      __builtin_amdgcn_sched_barrier(0);
      fetch_k(b1);  // next tile's K fragments (garbage past the last tile, never used)
#pragma unroll
      for (int n = 0; n < 6; ++n) o[1][n % 3] = mfma32x32(vf[n], p_operand(1, n / 3), o[1][n % 3]);
    }
    // tile it+2 (requested one iteration ago) must have landed before any wave reads it; this iteration's own two
    // requests may stay in flight
    if (k0 + 3 * BK < L) wait_vmcnt<2>();
    else wait_vmcnt<0>();
    __syncthreads();
  };
  auto sweep = [&](auto every_tile_tag) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      m_run[qb] = 0.f;
      negm[qb] = splat16(0.f);
#pragma unroll
      for (int mt = 0; mt < 3; ++mt) o[qb][mt] = splat16(0.f);
    }
    request_tile(0, 0);
    request_tile(BK, 1);
    request_tile(2 * BK, 2);
    wait_vmcnt<0>();
    __syncthreads();
    fetch_k(0);
    it = 0;
    tile_step(0, std::true_type{});
    ++it;
    for (int k0 = BK; k0 < L; k0 += BK, ++it) tile_step(k0, every_tile_tag);
  };
  sweep(std::false_type{});
  {
    // x * 0 is NaN for an infinity or a NaN and 0 otherwise: one chain of multiply-adds over a block's accumulators
    float chk = 0.f;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int mt = 0; mt < 3; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) chk = __builtin_fmaf(o[qb][mt][i], 0.f, chk);
    if (__syncthreads_or(chk != chk)) sweep(std::true_type{});  // the ring is idle: every wave is past its last tile
  }

#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q_first + 32 * qb;
    if (qi < L) {
      const float lsum = o[qb][2][8];  // head_dim row 80 (or 84): the row sum of P
      const float inv = 1.f / lsum;
      bf16_t* O = static_cast<bf16_t*>(p.out) + (int64_t)(s0 + qi) * p.o_stride + (int64_t)h * HD;
#pragma unroll
      for (int mt = 0; mt < 3; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (32 * mt + 8 * j >= HD) continue;
          bf16x4 ov;
#pragma unroll
          for (int i = 0; i < 4; ++i) ov[i] = (bf16_t)(o[qb][mt][4 * j + i] * inv);
          *reinterpret_cast<bf16x4*>(O + 32 * mt + 8 * j + 4 * hh) = ov;
        }
      if (hh == 0) p.lse[(int64_t)h * p.total + s0 + qi] = (m_run[qb] + __builtin_amdgcn_logf(lsum)) * LN2;
    }
  }
}

// ================================================================================================
// dQ for long segments, "wide" form: a wave owns 64 queries (two blocks of 32), four waves = 256 queries per
// work-group, one work-group per CU.  Pre-scaled Q and dO fragments of the wave's queries, and the 80 accumulators,
// live in accumulation registers; K / V tiles of 32 keys stream through an LDS ring of four tiles (direct
// global -> LDS loads, three tiles ahead).  Per tile and query block:
//   S^T = K Q^T - lse2, dP^T = V dO^T - delta   (v_mfma_f32_32x32x16_bf16; lane = query, so the statistics are per-lane
//                                                constants kept as ready-made accumulator input tiles)
//   dS^T = exp2(S^T) * dP^T                      (vector ALU), packed to bf16, lane swaps
//   dQ^T += K^T dS^T                             (v_mfma_f32_16x16x32_bf16, K^T read from LDS with the transposing load)
template <int ND>
__global__ __launch_bounds__(256, 1) void attn_bwd_dq_wide(const AttnParams p) {
  static_assert(ND == 5, "the hand-placed instruction order below is laid out for head_dim 80");
  using G = Geo<ND>;
  constexpr int HD = G::HD, BK = 32, NT = 256, RING = 4;
  // one array for both streamed tensors: a fragment's address in the V tile is its address in the K tile plus a
  // constant that fits the instruction's offset field, so one address computation serves both
  __shared__ __attribute__((aligned(1024))) bf16_t lds_kv[2 * RING][XS_TILE];
  bf16_t (*const lds_k)[XS_TILE] = lds_kv;
  bf16_t (*const lds_v)[XS_TILE] = lds_kv + RING;
  __shared__ __attribute__((aligned(16))) float lds_fix[NT * 4];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_q0 = blockIdx.x * 256;
  if (blk_q0 >= L) return;
  const int l = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hh = l >> 5, c32 = l & 31, G4 = l >> 4, r = l & 15;
  const int q0 = blk_q0 + wv * 64;

  const bf16_t* QS = static_cast<const bf16_t*>(p.q_scaled) + (int64_t)s0 * p.qs_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  const bf16_t* DO = static_cast<const bf16_t*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD;
  const float* NLSE = p.nlse2 + (int64_t)h * p.total + s0;
  const float* NDEL = p.ndelta + (int64_t)h * p.total + s0;

  // B operands of the score products (column = query 32*qb + l%32, contraction = head-dim 16*s + 8*(l/32) ..) and the
  // accumulator input tiles holding the query's - lse2 / - delta in all sixteen registers
  u32x4 qf[2][ND], dof[2][ND];
  f32x16 nl[2], nd[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int qi = q0 + 32 * qb + c32;
    const bool ok = qi < L;
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      qf[qb][s] = to_acc_regs(load_frag_global(QS + (int64_t)qi * p.qs_stride + 16 * s + 8 * hh, ok), lds_fix + threadIdx.x * 4);
      dof[qb][s] = to_acc_regs(load_frag_global(DO + (int64_t)qi * p.do_stride + 16 * s + 8 * hh, ok), lds_fix + threadIdx.x * 4);
    }
    nl[qb] = splat16(ok ? NLSE[qi] : -1e30f);  // hugely negative => p = 0 for queries past the end
    nd[qb] = splat16(ok ? NDEL[qi] : 0.f);
  }
  f32x4 dq[2][2][ND];  // [query block][half][head-dim block]: lane = query l%16 of the half, registers = head-dim 4*(l/16) + i
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int d = 0; d < ND; ++d) dq[qb][hf][d] = f32x4{0.f, 0.f, 0.f, 0.f};

  // direct global -> LDS loads of the K / V tiles (see attn_bwd_dkdv_wide); rows past the segment end repeat its last row
  int trow[2], tchunk[2];
  unsigned voff_k[2], voff_v[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int slot = 64 * (2 * wv + j) + l;
    trow[j] = slot >> 4;
    tchunk[j] = min(((slot & 15) ^ xs(trow[j])), 2 * ND - 1);
    voff_k[j] = (unsigned)(trow[j] * (int)p.k_stride * 2 + tchunk[j] * 16);
    voff_v[j] = (unsigned)(trow[j] * (int)p.v_stride * 2 + tchunk[j] * 16);
  }
  const unsigned lds_k0 = (unsigned)(uintptr_t)&lds_k[0][0], lds_v0 = (unsigned)(uintptr_t)&lds_v[0][0];
  auto request_tile = [&](int k0, int slot) {  // 4 load instructions
    if (k0 >= L) return;
    const int last = L - 1 - k0;
    const bool tail = last < BK - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      unsigned vk = voff_k[j], vv = voff_v[j];
      if (tail) {
        const int row = min(trow[j], last);
        vk = (unsigned)(row * (int)p.k_stride * 2 + tchunk[j] * 16);
        vv = (unsigned)(row * (int)p.v_stride * 2 + tchunk[j] * 16);
      }
      lds_direct_16(lds_k0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, vk, K + (int64_t)k0 * p.k_stride);
      lds_direct_16(lds_v0 + slot * (XS_TILE * 2) + (2 * wv + j) * 1024, vv, V + (int64_t)k0 * p.v_stride);
    }
  };
  request_tile(0, 0);
  request_tile(BK, 1);
  request_tile(2 * BK, 2);
  wait_vmcnt<0>();
  __syncthreads();

  bf16x8 ka[ND], va[ND];  // A operands of the score products: row = key l%32 of the tile
  auto fetch_rows = [&](int slot) {
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      ka[s] = xs_row_frag(lds_k[slot], c32, s, hh);
      va[s] = xs_row_frag(lds_v[slot], c32, s, hh);
    }
  };
  fetch_rows(0);

  f32x16 sc[2], dp[2];  // per query block: S^T - lse2 and dP^T - delta, lane = query l%32, register i = key 8*(i/4) + 4*(l/32) + i%4
  int it = 0;
  for (int k0 = 0; k0 < L; k0 += BK, ++it) {
    const int b0 = it & 3, b1 = (it + 1) & 3, b3 = (it + 3) & 3;
    request_tile(k0 + 3 * BK, b3);
    const int valid = L - k0;  // keys of this tile inside the segment (>= 1)
    // ---- phase 1: score products of query block 0; K^T fragments for the dQ products are read between the MFMAs
    bf16x8 kt[ND];
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      if (s == 0) {
        mfma32x32_init(sc[0], ka[0], qf[0][0], nl[0]);
        mfma32x32_init(dp[0], va[0], dof[0][0], nd[0]);
      } else {
        mfma32x32_acc(sc[0], ka[s], qf[0][s]);
        mfma32x32_acc(dp[0], va[s], dof[0][s]);
      }
      kt[s] = xs_tr_block(lds_k[b0], s, G4, r);
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 2: score products of query block 1 under the vector work of block 0
    unsigned dw[2][8];
    auto word = [&](int qb, int j) {
      const float x0 = __builtin_amdgcn_exp2f(sc[qb][2 * j]) * dp[qb][2 * j], x1 = __builtin_amdgcn_exp2f(sc[qb][2 * j + 1]) * dp[qb][2 * j + 1];
      dw[qb][j] = pack2(x0, x1);
    };
    // keys past the segment end (last tile only) contribute nothing: their dP is zeroed before it is used
    auto mask_tail = [&](int qb) {
      if (valid < BK) {
        asm volatile("" ::: "memory");  // keeps this rare block a branch
        mfma_drain();
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + 4 * hh + (i & 3) >= valid) dp[qb][i] = 0.f;
      }
    };
    mask_tail(0);
    BOps d0;
#pragma unroll
    for (int s = 0; s < ND; ++s) {
      // vector work between the two MFMAs from the second step on (see attn_bwd_dkdv_wide)
      if (s == 0) {
        mfma32x32_init(sc[1], ka[0], qf[1][0], nl[1]);
        mfma32x32_init(dp[1], va[0], dof[1][0], nd[1]);
        word(0, 0);
        word(0, 1);
      } else if (s < 4) {
        mfma32x32_acc(sc[1], ka[s], qf[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        word(0, 2 * s);
        __builtin_amdgcn_sched_barrier(0);
        mfma32x32_acc(dp[1], va[s], dof[1][s]);
        __builtin_amdgcn_sched_barrier(0);
        word(0, 2 * s + 1);
      } else {  // the lane swaps of block 0 under the last two score MFMAs
        mfma32x32_acc(sc[1], ka[s], qf[1][s]);
        mfma32x32_acc(dp[1], va[s], dof[1][s]);
        d0 = to_b_operands(dw[0]);
        asm volatile("s_nop 1");
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 3: dQ of query block 0 under the vector work of block 1
    mask_tail(1);
    BOps d1;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dq[0][0][d] = mfma32(kt[d], d0.lo, dq[0][0][d]);
      dq[0][1][d] = mfma32(kt[d], d0.hi, dq[0][1][d]);
      if (d < 4) {
        word(1, 2 * d);
        word(1, 2 * d + 1);
      } else {
        d1 = to_b_operands(dw[1]);
        asm volatile("s_nop 1");
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- phase 4: dQ of query block 1 under the fragment reads of the next tile
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dq[1][0][d] = mfma32(kt[d], d1.lo, dq[1][0][d]);
      dq[1][1][d] = mfma32(kt[d], d1.hi, dq[1][1][d]);
      ka[d] = xs_row_frag(lds_k[b1], c32, d, hh);
      va[d] = xs_row_frag(lds_v[b1], c32, d, hh);
      __builtin_amdgcn_sched_barrier(0);
    }
    // tile it+2 (requested in iteration it-1) must have landed before any wave reads it in the next iteration
    if (k0 + 3 * BK < L) wait_vmcnt<4>();
    else wait_vmcnt<0>();
    __syncthreads();
  }

  bf16_t* DQ = static_cast<bf16_t*>(p.dq) + (int64_t)s0 * p.dq_stride + (int64_t)h * HD;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int qi = q0 + 32 * qb + 16 * hf + r;
      if (qi < L) {
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          bf16x4 a;
#pragma unroll
          for (int i = 0; i < 4; ++i) a[i] = (bf16_t)(dq[qb][hf][d][i] * p.scale);
          *reinterpret_cast<bf16x4*>(DQ + (int64_t)qi * p.dq_stride + 16 * d + 4 * G4) = a;
        }
      }
    }
}

// ================================================================================================
// dQ.  Block = 64*NWAVES queries of one (segment, head); 32 keys per iteration, K / V tiles double buffered.
template <int ND, int NWAVES, int RB>
__global__ __launch_bounds__(64 * NWAVES) void attn_bwd_dq_mfma(const AttnParams p) {
  using G = Geo<ND>;
  constexpr int HD = G::HD, BK = 32, NT = 64 * NWAVES, SPAN = 16 * RB * NWAVES;  // RB 16-row blocks per wave
  constexpr int P = SWZ;  // the K tile is read as row fragments and through the transposing load
  __shared__ __attribute__((aligned(16))) bf16_t lds_k[2][BK * P];
  __shared__ __attribute__((aligned(16))) bf16_t lds_v[2][BK * P];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg], L = p.cu[seg + 1] - s0;
  const int blk_q0 = blockIdx.x * SPAN;
  if (blk_q0 >= L) return;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, g = l >> 4, r = l & 15;
  const int q0 = blk_q0 + wv * 16 * RB;

  const bf16_t* Q = static_cast<const bf16_t*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD;
  const bf16_t* K = static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD;
  const bf16_t* V = static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD;
  const bf16_t* DO = static_cast<const bf16_t*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD;
  const float* LSE = p.lse + (int64_t)h * p.total + s0;
  const float* DELTA = p.delta + (int64_t)h * p.total + s0;

  constexpr bool FOLD = G::TAIL16;
  const float c = p.scale * LOG2E;
  const bf16_t one_x = (bf16_t)(g == 0 ? 1.f : 0.f);
  RowFrag<ND> qf[RB], dof[RB];
  float neg_lse2[RB], dl[RB];
  HiLo f_lse[RB], f_dl[RB];  // FOLD: -lse2 and -delta of the lane's query as hi + lo (lane group 0 only)
#pragma unroll
  for (int qb = 0; qb < RB; ++qb) {
    const int qi = q0 + qb * 16 + r;
    const bool ok = qi < L;
    load_rowfrag_global<ND>(qf[qb], Q + (int64_t)qi * p.q_stride, ok, g);
    scale_rowfrag<ND>(qf[qb], c);  // scores leave the MFMA in log2 units
    load_rowfrag_global<ND>(dof[qb], DO + (int64_t)qi * p.do_stride, ok, g);
    neg_lse2[qb] = ok ? -LSE[qi] * LOG2E : -1e30f;  // hugely negative => p = 0 for padded queries
    dl[qb] = ok ? DELTA[qi] : 0.f;
    f_lse[qb] = split_hilo(g == 0 ? neg_lse2[qb] : 0.f);
    f_dl[qb] = split_hilo(g == 0 ? -dl[qb] : 0.f);
  }
  f32x4 dq[RB][ND];
#pragma unroll
  for (int qb = 0; qb < RB; ++qb)
#pragma unroll
    for (int d = 0; d < ND; ++d) dq[qb][d] = f32x4{0.f, 0.f, 0.f, 0.f};

  TileStager<ND, BK, P, NT> sk, sv;
  sk.init(p.k_stride);
  sv.init(p.v_stride);
  sk.load(K, min(BK, L));
  sv.load(V, min(BK, L));
  sk.store(lds_k[0]);
  sv.store(lds_v[0]);
  __syncthreads();

  int buf = 0;
  for (int k0 = 0; k0 < L; k0 += BK) {
    const int valid = min(BK, L - k0);
    const bool has_next = k0 + BK < L;
    if (has_next) {
      const int nv = min(BK, L - k0 - BK);
      sk.load(K + (int64_t)(k0 + BK) * p.k_stride, nv);
      sv.load(V + (int64_t)(k0 + BK) * p.v_stride, nv);
    }
    const bf16_t* tk = lds_k[buf];
    const bf16_t* tv = lds_v[buf];

    RowFrag<ND> ka[2], va[2];
    bf16x8 kt[ND];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      load_rowfrag_lds<ND, P>(ka[t], tk, t * 16 + r, g);
      load_rowfrag_lds<ND, P>(va[t], tv, t * 16 + r, g);
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      kt[d] = tr_block<P>(tk, 0, d, g, r);
    }
#pragma unroll
    for (int qb = 0; qb < RB; ++qb) {
      f32x4 ds[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        // S[q = qb*16+r][key = t*16+4g+i] in log2 units, and dP in the same layout
        if constexpr (FOLD) {
          const f32x4 s = dot_frag_plus2<ND>(ka[t], qf[qb], one_x, one_x, f_lse[qb].hi, f_lse[qb].lo);   // - lse2
          const f32x4 dp = dot_frag_plus2<ND>(va[t], dof[qb], one_x, one_x, f_dl[qb].hi, f_dl[qb].lo);  // - delta
#pragma unroll
          for (int i = 0; i < 4; ++i) ds[t][i] = __builtin_amdgcn_exp2f(s[i]) * dp[i];
        } else {
          const f32x4 s = dot_frag<ND>(ka[t], qf[qb]);
          const f32x4 dp = dot_frag<ND>(va[t], dof[qb]);
#pragma unroll
          for (int i = 0; i < 4; ++i) ds[t][i] = __builtin_amdgcn_exp2f(s[i] + neg_lse2[qb]) * (dp[i] - dl[qb]);
        }
      }
      if (valid < BK) {  // keys past the segment end contribute nothing
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (t * 16 + 4 * g + i >= valid) ds[t][i] = 0.f;
      }
      const bf16x8 dsb = pack8(ds[0], ds[1]);
#pragma unroll
      for (int d = 0; d < ND; ++d) dq[qb][d] = mfma32(kt[d], dsb, dq[qb][d]);
    }
    if (has_next) {
      sk.store(lds_k[buf ^ 1]);
      sv.store(lds_v[buf ^ 1]);
    }
    __syncthreads();
    buf ^= 1;
  }

  bf16_t* DQ = static_cast<bf16_t*>(p.dq) + (int64_t)s0 * p.dq_stride + (int64_t)h * HD;
#pragma unroll
  for (int qb = 0; qb < RB; ++qb) {
    const int qi = q0 + qb * 16 + r;
    if (qi < L) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        bf16x4 a;
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = (bf16_t)(dq[qb][d][i] * p.scale);
        *reinterpret_cast<bf16x4*>(DQ + (int64_t)qi * p.dq_stride + 16 * d + 4 * g) = a;
      }
    }
  }
}

// ================================================================================================
// Whole backward of a short segment (<= 64 rows, the windowed layers) in one work-group: Q, K, V and dO of one
// (segment, head) are staged in LDS once.  Pass A works in the dQ orientation (a lane owns a query), where
// delta_q = sum_k P[q,k] * dP[q,k] (equal to dO_q . O_q, so O is never read) is a lane-local sum, and writes dQ;
// pass B repeats the dK/dV kernel's tile loop on the staged tiles.  HBM traffic: four tiles in, three out.
// Results are turned in LDS and leave as 16-byte chunks, a row's 160 bytes together: as 8-byte pieces of 32 bytes a row, straight from the accumulators,
// they took twice the write requests.  us before / now, operands from HBM: 4,096 rows x 16 heads 27.8 / 25.0, 14,336 80 / 68, 25,524 128 / 108, 65,536 307 / 259
// (4.5 TB/s).  Waves without rows leave before pass B; while they turned nothing but zeros, short windows were slower than with the pieces: 65,536 rows x 16 heads, pieces /
// all waves / this, windows of 16 tokens 506 / 515 / 491, of 4 1,592 / 1,710 / 1,541, head_dim 32 190 / 219 / 175, 627 / 738 / 558.
// ROPE: dQ and dK are turned back by the rotary embedding's angles on their way out (with the roundings of the pass of its own, which read and wrote both
// once more); dQ waits in LDS for the tables, which are fetched once for both and travel while dK and dV are rounded.  ms per step, pass of its own /
// inside: 1,024 rows 12.0 / 11.6, 4,096 checkpointed 27.9 / 27.6, 14,336 62.2 / 61.0, 25,524 104.9 / 104.3, 36,864 239.6 / 238.3.
template <int ND, bool ROPE = false>  // four waves share the staged tiles; wave w owns queries and keys [16 w, 16 w + 16)
__global__ __launch_bounds__(256, 2) void attn_bwd_window_mfma(const AttnParams p, const WindowRope rope) {
  using G = Geo<ND>;
  constexpr int HD = G::HD, R = 64, PK = G::PK;
  __shared__ __attribute__((aligned(16))) bf16_t lds_q[R * PK];
  __shared__ __attribute__((aligned(16))) bf16_t lds_k[R * PK];
  __shared__ __attribute__((aligned(16))) bf16_t lds_v[R * PK];
  __shared__ __attribute__((aligned(16))) bf16_t lds_do[R * PK];
  __shared__ __attribute__((aligned(16))) float lds_lse[R];
  __shared__ __attribute__((aligned(16))) float lds_delta[R];

  int seg, h;
  seg_and_head(p, seg, h);
  const int s0 = p.cu[seg];
  const int L = min(p.cu[seg + 1] - s0, R);
  if (L <= 0) return;
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, g = l >> 4, r = l & 15;
  const float c = p.scale * LOG2E;
  // lanes hand rows of LDS to each other within a wave, in both directions: what was read before the rows change, what was written before it is read
  auto lanes_meet = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // results leave as whole chunks of rows: turned in the wave's own sixteen rows of the k or v tile, which no other wave reads behind pass A
  auto turn_in = [&](bf16_t* tile, const bf16x4 (&v)[ND]) {
    lanes_meet();
#pragma unroll
    for (int d = 0; d < ND; ++d) *reinterpret_cast<bf16x4*>(tile + (wv * 16 + r) * PK + 16 * d + 4 * g) = v[d];
  };
  auto leave = [&](bf16_t* tile, const bf16x4 (&v)[ND], bf16_t* dst, int64_t stride) {
    const bf16_t* turn = tile + wv * 16 * PK;
    turn_in(tile, v);
    lanes_meet();
#pragma unroll
    for (int i = 0; i < (16 * G::CH + 63) / 64; ++i) {
      const int at = l + 64 * i, rr = at / G::CH, cc = at % G::CH;
      if (rr < 16 && wv * 16 + rr < L) *reinterpret_cast<bf16x8*>(dst + (int64_t)(wv * 16 + rr) * stride + cc * 8) = *reinterpret_cast<const bf16x8*>(turn + rr * PK + cc * 8);
    }
  };
  bf16x4 dq_out[ND];
  bf16_t* DQ = static_cast<bf16_t*>(p.dq) + (int64_t)s0 * p.dq_stride + (int64_t)h * HD;
  {
    TileStager<ND, R, PK, 256> sq, sk, sv, sdo;
    sq.init(p.q_stride);
    sk.init(p.k_stride);
    sv.init(p.v_stride);
    sdo.init(p.do_stride);
    sq.load(static_cast<const bf16_t*>(p.q) + (int64_t)s0 * p.q_stride + (int64_t)h * HD, L);
    sk.load(static_cast<const bf16_t*>(p.k) + (int64_t)s0 * p.k_stride + (int64_t)h * HD, L);
    sv.load(static_cast<const bf16_t*>(p.v) + (int64_t)s0 * p.v_stride + (int64_t)h * HD, L);
    sdo.load(static_cast<const bf16_t*>(p.d_o) + (int64_t)s0 * p.do_stride + (int64_t)h * HD, L);
    if (wv == 0) lds_lse[l] = l < L ? p.lse[(int64_t)h * p.total + s0 + l] * LOG2E : INFINITY;  // +inf => p = 0 for padded queries
    sq.scale(c);  // the Q tile holds Q * scale * log2(e): scores leave the MFMA in log2 units
    sq.store(lds_q);
    sk.store(lds_k);
    sv.store(lds_v);
    sdo.store(lds_do);
  }
  __syncthreads();

  // ---- pass A: dQ^T += K^T dS^T per 16-query block, keys in two chunks of 32
  {
    RowFrag<ND> ka[2][2], va[2][2];
    bf16x8 kt[2][ND];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        load_rowfrag_lds<ND, PK>(ka[kc][t], lds_k, kc * 32 + t * 16 + r, g);
        load_rowfrag_lds<ND, PK>(va[kc][t], lds_v, kc * 32 + t * 16 + r, g);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const int off = (kc * 32 + 4 * g + (r >> 2)) * PK + 16 * d + 4 * (r & 3);
        kt[kc][d] = tr_pair(lds_k + off, lds_k + off + 16 * PK);
      }
    }
    float* DELTA = p.delta + (int64_t)h * p.total + s0;
    if (wv * 16 < L) {
      const int qi = wv * 16 + r;
      RowFrag<ND> qf, dof;
      load_rowfrag_lds<ND, PK>(qf, lds_q, qi, g);
      load_rowfrag_lds<ND, PK>(dof, lds_do, qi, g);
      const float neg_lse2 = -lds_lse[qi];
      f32x4 e[2][2], dp[2][2];
      float part = 0.f;
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 sc = dot_frag<ND>(ka[kc][t], qf);  // S[q = wv*16+r][key = kc*32+t*16+4g+i]
          dp[kc][t] = dot_frag<ND>(va[kc][t], dof);      // dP, same layout
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float x = __builtin_amdgcn_exp2f(sc[i] + neg_lse2);
            if (kc * 32 + t * 16 + 4 * g + i >= L) x = 0.f;  // keys past the segment end
            e[kc][t][i] = x;
            part = __builtin_fmaf(x, dp[kc][t][i], part);
          }
        }
      part += __shfl_xor(part, 16);
      part += __shfl_xor(part, 32);  // lanes r, r+16, r+32, r+48 share query wv*16+r
      if (g == 0) {
        lds_delta[qi] = part;
        if (qi < L) DELTA[qi] = part;
      }
      f32x4 dq[ND];
#pragma unroll
      for (int d = 0; d < ND; ++d) dq[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        f32x4 ds[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) ds[t][i] = e[kc][t][i] * (dp[kc][t][i] - part);
        const bf16x8 dsb = pack8(ds[0], ds[1]);
#pragma unroll
        for (int d = 0; d < ND; ++d) dq[d] = mfma32(kt[kc][d], dsb, dq[d]);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) dq_out[d][i] = (bf16_t)(dq[d][i] * p.scale);
    }
    for (int q = 16 * ((L + 15) / 16) + (int)threadIdx.x; q < R; q += 256) lds_delta[q] = 0.f;  // query blocks that were skipped
  }
  __syncthreads();
  if (wv * 16 >= L) return;  // the waves meet no more

  // ---- pass B: dV^T += dO^T P, dK^T += Q^T dS per 16-key block, queries in two tiles of 32
  {
    RowFrag<ND> kf, vf;
    f32x4 dk[ND], dv[ND];
    load_rowfrag_lds<ND, PK>(kf, lds_k, wv * 16 + r, g);
    load_rowfrag_lds<ND, PK>(vf, lds_v, wv * 16 + r, g);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      dk[d] = f32x4{0.f, 0.f, 0.f, 0.f};
      dv[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (!ROPE) leave(lds_v, dq_out, DQ, p.dq_stride);
    if (ROPE) turn_in(lds_v, dq_out);  // stays there until the tables are fetched, once for both
#pragma unroll 1
    for (int qs = 0; qs < L; qs += 32) {
      const bf16_t* tq = lds_q + qs * PK;
      const bf16_t* tdo = lds_do + qs * PK;
      RowFrag<ND> qa[2], da[2];
      bf16x8 qt[ND], dt_[ND];
      f32x4 lse2[2], dl[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        load_rowfrag_lds<ND, PK>(qa[t], tq, t * 16 + r, g);
        load_rowfrag_lds<ND, PK>(da[t], tdo, t * 16 + r, g);
        lse2[t] = *reinterpret_cast<const f32x4*>(lds_lse + qs + t * 16 + 4 * g);
        dl[t] = *reinterpret_cast<const f32x4*>(lds_delta + qs + t * 16 + 4 * g);
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const int off = (4 * g + (r >> 2)) * PK + 16 * d + 4 * (r & 3);
        qt[d] = tr_pair(tq + off, tq + off + 16 * PK);
        dt_[d] = tr_pair(tdo + off, tdo + off + 16 * PK);
      }
      f32x4 pv[2], ds[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f32x4 sc = dot_frag<ND>(qa[t], kf);   // S[q = qs+t*16+4g+i][key = wv*16+r]
        const f32x4 dpp = dot_frag<ND>(da[t], vf);  // dP, same layout
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = __builtin_amdgcn_exp2f(sc[i] - lse2[t][i]);
          pv[t][i] = x;
          ds[t][i] = x * (dpp[i] - dl[t][i]);
        }
      }
      const bf16x8 pb = pack8(pv[0], pv[1]);
      const bf16x8 dsb = pack8(ds[0], ds[1]);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        dv[d] = mfma32(dt_[d], pb, dv[d]);
        dk[d] = mfma32(qt[d], dsb, dk[d]);
      }
    }
    bf16_t* DK = static_cast<bf16_t*>(p.dk) + (int64_t)s0 * p.dk_stride + (int64_t)h * HD;
    bf16_t* DV = static_cast<bf16_t*>(p.dv) + (int64_t)s0 * p.dv_stride + (int64_t)h * HD;
    // ROPE: a lane takes eight columns of the first half of a head and the matching eight of the second; sixteen rows are 16 * ND such pairs
    constexpr int HALF = HD / 2, PAIRS = ROPE ? (16 * ND + 63) / 64 : 0;
    float c0[8], c1[8], sn0[8], sn1[8];
    auto fetch = [&](int i) {
      const int at = l + 64 * i, rr = at / ND, row = wv * 16 + rr;
      const int64_t angle = (int64_t)(s0 + (rr < 16 && row < L ? row : 0)) * HD + at % ND * 8;
      auto eight = [&](const float* table, float (&to)[8]) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(table + angle), y = *reinterpret_cast<const f32x4*>(table + angle + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) to[j] = x[j], to[4 + j] = y[j];
      };
      eight(rope.cos, c0);
      eight(rope.cos + HALF, c1);
      eight(rope.sin, sn0);
      eight(rope.sin + HALF, sn1);
    };
    if (ROPE) fetch(0);
    bf16x4 a[ND], b[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[d][i] = (bf16_t)(dk[d][i] * LN2);  // dS^T (Q scale log2e) / log2e
        b[d][i] = (bf16_t)dv[d][i];
      }
    if constexpr (!ROPE) {
      leave(lds_k, a, DK, p.dk_stride);
    } else {
      turn_in(lds_k, a);
      lanes_meet();
#pragma unroll
      for (int i = 0; i < PAIRS; ++i) {
        const int at = l + 64 * i, rr = at / ND, cc = at % ND, row = wv * 16 + rr;
        if (i > 0) fetch(i);
        if (rr >= 16 || row >= L) continue;
        auto back = [&](const bf16_t* tile, bf16_t* dst, int64_t stride, float gain) {
          bf16x8 lo = *reinterpret_cast<const bf16x8*>(tile + row * PK + cc * 8), hi = *reinterpret_cast<const bf16x8*>(tile + row * PK + HALF + cc * 8);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float oa, ob;
            rope_pair((float)lo[j], (float)hi[j], c0[j], c1[j], sn0[j], sn1[j], 1, oa, ob);
            lo[j] = (bf16_t)(oa * gain);
            hi[j] = (bf16_t)(ob * gain);
          }
          *reinterpret_cast<bf16x8*>(dst + (int64_t)row * stride + cc * 8) = lo;
          *reinterpret_cast<bf16x8*>(dst + (int64_t)row * stride + HALF + cc * 8) = hi;
        };
        back(lds_v, DQ, p.dq_stride, rope.q_gain);
        back(lds_k, DK, p.dk_stride, 1.f);
      }
    }
    leave(lds_v, b, DV, p.dv_stride);
  }
}

// ------------------------------------------------------------------------------------------------
constexpr int WIDE_MIN_SEQLEN = 512;  // from here on the 64-rows-per-wave kernels fill their work-groups well enough
inline int pick_waves(int max_seqlen) { return max_seqlen <= 64 ? 1 : (max_seqlen <= 128 ? 2 : 4); }

template <int ND>
int launch_fwd_mfma(const AttnParams& p, int n_seg, int max_seqlen, hipStream_t s) {
  const int nw = pick_waves(max_seqlen);
  dim3 grid((unsigned)((max_seqlen + 64 * nw - 1) / (64 * nw)), (unsigned)n_seg, (unsigned)p.nheads);
  if (nw == 1 && ND <= 5) {
    // windows: four waves x 16 queries share the staged K / V tiles.  Bound by memory (671 MB at 65,536 rows x 16 heads) and by the
    // chain load -> products -> store, i.e. by how many waves a compute unit holds: 96 registers, five per SIMD.  Two waves of 32
    // queries (128 registers, a tile staged load by load) / this, us, operands from HBM: 16,384 rows 51 / 43, 25,524 in windows of
    // 4 ... 64 76 / 64, 65,536 179 / 152
    AttnParams pw = p;
    if (grid.x == 1 && ((int64_t)n_seg * p.nheads) % 8 == 0) pw.seg_major = 2;  // heads of a segment together on one XCD
    if constexpr (ND <= 5) hipLaunchKernelGGL((attn_fwd_mfma<ND, 4, 64, false, 1, 5>), grid, 256, 0, s, pw);
  } else if (nw == 1) hipLaunchKernelGGL((attn_fwd_mfma<ND, 1, 64, false>), grid, 64, 0, s, p);
  else if (nw == 2) hipLaunchKernelGGL((attn_fwd_mfma<ND, 2, 64, false>), grid, 128, 0, s, p);
  else if constexpr (ND <= 5) {
    // long segments: 8 waves x 32 queries, <= 128 registers, so that four waves share a SIMD and cover each
    // other's MFMA -> softmax -> MFMA dependency stalls
    // all heads of a segment are neighbours in the launch order: with the caller's longest-first segment order
    // the work-groups then start in order of decreasing run time
    AttnParams pl = p;
    pl.seg_major = 1;  // n_seg fits gridDim.z: checked at the entry point
    dim3 gl = pl.seg_major ? dim3(grid.x, grid.z, grid.y) : grid;
    if constexpr (ND == 5) {
      if (max_seqlen >= WIDE_MIN_SEQLEN) {  // 64 queries per wave, 512 per work-group
        hipLaunchKernelGGL((attn_fwd_x32<ND>), dim3((unsigned)((max_seqlen + 511) / 512), gl.y, gl.z), 512, 0, s, pl);
        MVIT_CHECK_LAUNCH("attn_fwd");
        return MVIT_OK;
      }
    }
    hipLaunchKernelGGL((attn_fwd_mfma<ND, 8, 32, true, 2, 4>), gl, 512, 0, s, pl);
  }
  else hipLaunchKernelGGL((attn_fwd_mfma<ND, 4, 32, true>), grid, 256, 0, s, p);  // head_dim 128: register budget
  MVIT_CHECK_LAUNCH("attn_fwd");
  return MVIT_OK;
}
using G5 = Geo<5>;
template <int ND>
int launch_bwd_mfma(const AttnParams& p, int n_seg, int max_seqlen, hipStream_t s) {
  // short segments (windows): one work-group does the whole backward of a (segment, head); long ones: 8 waves x 32 rows
  if (max_seqlen <= 64) {
    dim3 grid(1, (unsigned)n_seg, (unsigned)p.nheads);
    if constexpr (ND <= 5) {
      // four waves x 16 rows: ~160 registers, three work-groups (12 waves) per CU to cover the load -> MFMA -> store latency
      AttnParams pw = p;
      if (((int64_t)n_seg * p.nheads) % 8 == 0) pw.seg_major = 2;  // heads of a segment together on one XCD
      hipLaunchKernelGGL((attn_bwd_window_mfma<ND>), grid, 256, 0, s, pw, WindowRope{});  // computes delta itself
    } else {
      hipLaunchKernelGGL((attn_bwd_dkdv_mfma<ND, 1, 4>), grid, 64, 0, s, p);
      hipLaunchKernelGGL((attn_bwd_dq_mfma<ND, 1, 4>), grid, 64, 0, s, p);
    }
  } else if (max_seqlen <= 128) {
    dim3 grid(1, (unsigned)n_seg, (unsigned)p.nheads);
    hipLaunchKernelGGL((attn_bwd_dkdv_mfma<ND, 2, 4>), grid, 128, 0, s, p);
    hipLaunchKernelGGL((attn_bwd_dq_mfma<ND, 2, 4>), grid, 128, 0, s, p);
  } else {
    dim3 grid((unsigned)((max_seqlen + 255) / 256), (unsigned)n_seg, (unsigned)p.nheads);
    AttnParams pl = p;
    pl.seg_major = 1;  // as in the forward: segment-major launch order
    dim3 gl = pl.seg_major ? dim3(grid.x, grid.z, grid.y) : grid;
    if (ND == 5 && max_seqlen >= WIDE_MIN_SEQLEN) {
      if constexpr (ND == 5) {
        // the dq buffer holds the pre-scaled queries until the dQ kernel overwrites it with the result
        const int64_t nstat = (int64_t)p.nheads * p.total;
        pl.q_scaled = p.dq;
        pl.qs_stride = p.dq_stride;
        pl.nlse2 = p.delta + nstat;
        pl.ndelta = p.delta + 2 * nstat;
        const int cols = p.nheads * G5::HD;
        const int64_t nchunk = p.total * (cols / 8);
        const unsigned pgrid = (unsigned)std::min<int64_t>(8192, (std::max(nchunk, nstat) + 255) / 256);
        hipLaunchKernelGGL(attn_bwd_prepare_kernel, dim3(pgrid), 256, 0, s, static_cast<const bf16_t*>(p.q), p.q_stride,
                           static_cast<bf16_t*>(p.dq), p.dq_stride, p.total, cols, p.scale * LOG2E, (const float*)p.lse,
                           (const float*)p.delta, p.delta + nstat, p.delta + 2 * nstat, nstat);
        hipLaunchKernelGGL((attn_bwd_dkdv_wide<ND>), gl, 256, 0, s, pl);
        hipLaunchKernelGGL((attn_bwd_dq_wide<ND>), gl, 256, 0, s, pl);
      }
    } else {
      hipLaunchKernelGGL((attn_bwd_dkdv_mfma<ND, 8, 2>), gl, 512, 0, s, pl);
      hipLaunchKernelGGL((attn_bwd_dq_mfma<ND, 8, 2>), gl, 512, 0, s, pl);
    }
  }
  MVIT_CHECK_LAUNCH("attn_bwd");
  return MVIT_OK;
}
int check_common(const char* who, const int32_t* cu, int n_seg, int max_seqlen, int64_t total, int nheads, int head_dim,
                 int dtype, std::initializer_list<int64_t> strides, std::initializer_list<const void*> ptrs) {
  MVIT_REQUIRE(cu && n_seg >= 0 && max_seqlen >= 0 && total >= 0 && nheads > 0 && nheads <= 65535 && n_seg <= 65535,
               "%s: bad sizes (n_seg=%d max_seqlen=%d total=%lld nheads=%d)", who, n_seg, max_seqlen, (long long)total, nheads);
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "%s: dtype %d", who, dtype);
  MVIT_REQUIRE(head_dim == 32 || head_dim == 64 || head_dim == 80 || head_dim == 128, "%s: head_dim %d not built (32, 64, 80, 128)", who, head_dim);
  const int vec = dtype == MVIT_BF16 ? 8 : 1;
  for (int64_t st : strides)
    MVIT_REQUIRE(st >= (int64_t)nheads * head_dim && st % vec == 0, "%s: row stride %lld must cover %d heads and be a multiple of %d", who, (long long)st, nheads, vec);
  if (n_seg == 0 || max_seqlen == 0 || total == 0) return MVIT_OK;  // nothing to do: empty tensors have no address to check
  for (const void* q : ptrs) MVIT_REQUIRE(q && mvit_aligned16(q), "%s: null or unaligned pointer", who);
  return MVIT_OK;
}

// Do two sets of `rows` rows of `width` bytes, starting at a and b with row pitches pa and pb (bytes), share a byte?
// Exact when the pitches are equal (tensors interleaved in one buffer, like q | k | v, are told apart); otherwise the
// two address ranges are compared as wholes.
bool strided_rows_overlap(const void* a, int64_t pa, const void* b, int64_t pb, int64_t rows, int64_t width) {
  const int64_t x = (int64_t)reinterpret_cast<uintptr_t>(a), y = (int64_t)reinterpret_cast<uintptr_t>(b);
  const int64_t ea = x + (rows - 1) * pa + width, eb = y + (rows - 1) * pb + width;
  if (ea <= y || eb <= x) return false;
  if (pa != pb || pa < width) return true;
  // equal pitch: row i of a starts at x + i*pa; relative to b's rows the column offset is constant
  int64_t off = (x - y) % pa;
  if (off < 0) off += pa;
  // a's row covers [off, off + width) modulo the pitch; b's rows cover [0, width)
  return off < width || off + width > pa;
}

}  // namespace

// Not windows of fewer than ten tokens on average: a work-group costs the same for four tokens as for 64, and the two passes hold more of them.  us of a
// block's forward (kept), 65,536 rows x 16 heads, two passes / inside: windows of 4 tokens 1,840 / 1,945, 6 1,608 / 1,649, 8 1,489 / 1,509, 10 1,424 / 1,426,
// 12 1,377 / 1,366; 14,336 rows, 4 426 / 444, 8 361 / 356.  The backward goes the same way (65,536 rows, 12 2,451 / 2,349, 16 2,342 / 2,285).
bool mvit_window_rope_takes(const mvit_window_rope& w, int head_dim, int max_seqlen, int dtype) {
  return w.S >= 10 * (int64_t)w.n_seg && dtype == MVIT_BF16 && head_dim == 80 && max_seqlen > 0 && max_seqlen <= 64 && w.n_seg > 0 && w.n_seg <= 65535 && w.nheads > 0 && w.nheads <= 65535 && w.S > 0 &&
         mvit_aligned16(w.qkv) && mvit_aligned16(w.o) && mvit_aligned16(w.lse) && mvit_aligned16(w.cos) && mvit_aligned16(w.sin);
}
int mvit_attn_fwd_window_rope(const mvit_window_rope& w, hipStream_t stream) {
  const int64_t C = (int64_t)w.nheads * 80;
  AttnParams p = {};
  bf16_t* qkv = static_cast<bf16_t*>(w.qkv);
  p.q = qkv; p.k = qkv + C; p.v = qkv + 2 * C; p.out = w.o; p.lse = w.lse; p.cu = w.cu; p.total = w.S; p.nheads = w.nheads;
  p.q_stride = p.k_stride = p.v_stride = 3 * C; p.o_stride = C; p.scale = w.attn_scale;
  WindowRope r{w.cos, w.sin, w.q_gain, 1, w.keep ? 1 : 0, w.n_seg, w.nheads};
  // LOOP once q, k and v are more than stays in the memory-side cache (256 MB) between the product that writes them and this, and windows long
  // enough for two work-groups to keep a unit's loads coming: us of a block's forward, 65,536 rows x 16 heads, one head / LOOP, kept and not kept:
  // windows of 16 tokens 1,311 / 1,410, 1,234 / 1,359; 32 1,247 / 1,251, +31; 40 1,250 / 1,233, +4; 48 1,248 / 1,219, -10; 64 1,246 / 1,211, -12
  const bool loop = w.S * 3 * C * 2 > (160ll << 20) && w.S >= (w.keep ? 40 : 48) * (int64_t)w.n_seg;
  const int most = !loop ? 1 : w.keep ? 2 : 4;
  while (2 * r.heads <= most && w.nheads % (2 * r.heads) == 0) r.heads *= 2;
  r.parts = w.nheads / r.heads;
  const dim3 grid((unsigned)r.parts, (unsigned)w.n_seg);
  if (r.heads > 1) hipLaunchKernelGGL((attn_fwd_window_rope<5, true>), grid, 320, 0, stream, p, r);
  else hipLaunchKernelGGL((attn_fwd_window_rope<5, false>), grid, 320, 0, stream, p, r);
  MVIT_CHECK_LAUNCH("attn_fwd_window_rope");
  return MVIT_OK;
}

int mvit_attn_bwd_window_rope(const mvit_window_rope& w, const void* d_o, void* dqkv, float* delta, hipStream_t stream) {
  const int64_t C = (int64_t)w.nheads * 80;
  AttnParams p = {};
  const bf16_t* qkv = static_cast<const bf16_t*>(w.qkv);
  bf16_t* d = static_cast<bf16_t*>(dqkv);
  p.q = qkv; p.k = qkv + C; p.v = qkv + 2 * C; p.d_o = d_o; p.lse = w.lse; p.delta = delta; p.dq = d; p.dk = d + C; p.dv = d + 2 * C;
  p.cu = w.cu; p.total = w.S; p.nheads = w.nheads;
  p.q_stride = p.k_stride = p.v_stride = p.dq_stride = p.dk_stride = p.dv_stride = 3 * C; p.o_stride = p.do_stride = C; p.scale = w.attn_scale;
  if (((int64_t)w.n_seg * w.nheads) % 8 == 0) p.seg_major = 2;  // heads of a segment together on one XCD
  hipLaunchKernelGGL((attn_bwd_window_mfma<5, true>), dim3(1, (unsigned)w.n_seg, (unsigned)w.nheads), 256, 0, stream, p, WindowRope{w.cos, w.sin, w.q_gain, 1, 0, w.n_seg, w.nheads});
  MVIT_CHECK_LAUNCH("attn_bwd_window_rope");
  return MVIT_OK;
}

extern "C" {

int64_t mvit_attn_bwd_delta_elems(int max_seqlen, int64_t total, int nheads, int head_dim, int dtype) {
  const bool wide = dtype == MVIT_BF16 && head_dim == 80 && max_seqlen >= WIDE_MIN_SEQLEN;
  return (wide ? 3 : 1) * (int64_t)nheads * total;
}

int mvit_attn_fwd(const void* q, const void* k, const void* v, void* o, float* lse, const int32_t* cu_seqlens,
                  const int32_t* seg_order, int n_seg, int max_seqlen, int64_t total, int nheads, int head_dim, int64_t q_stride, int64_t k_stride,
                  int64_t v_stride, int64_t o_stride, float scale, int dtype, mvit_stream_t stream) {
  if (int rc = check_common("attn_fwd", cu_seqlens, n_seg, max_seqlen, total, nheads, head_dim, dtype,
                            {q_stride, k_stride, v_stride, o_stride}, {q, k, v, o, (const void*)lse}))
    return rc;
  if (n_seg == 0 || max_seqlen == 0 || total == 0) return MVIT_OK;
  AttnParams p = {};
  p.q = q; p.k = k; p.v = v; p.out = o; p.lse = lse; p.cu = cu_seqlens; p.order = seg_order; p.total = total; p.nheads = nheads;
  p.q_stride = q_stride; p.k_stride = k_stride; p.v_stride = v_stride; p.o_stride = o_stride; p.scale = scale;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == MVIT_BF16) {
    switch (head_dim) {
      case 32: return launch_fwd_mfma<2>(p, n_seg, max_seqlen, s);
      case 64: return launch_fwd_mfma<4>(p, n_seg, max_seqlen, s);
      case 80: return launch_fwd_mfma<5>(p, n_seg, max_seqlen, s);
      default: return launch_fwd_mfma<8>(p, n_seg, max_seqlen, s);
    }
  }
  return mvit_attn_f32(p, head_dim, n_seg, max_seqlen, false, s);
}

int mvit_attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o, const float* lse, void* dq,
                  void* dk, void* dv, float* delta, int64_t delta_elems, const int32_t* cu_seqlens, const int32_t* seg_order, int n_seg, int max_seqlen,
                  int64_t total, int nheads, int head_dim, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t o_stride,
                  int64_t do_stride, int64_t dq_stride, int64_t dk_stride, int64_t dv_stride, float scale, int dtype,
                  mvit_stream_t stream) {
  if (int rc = check_common("attn_bwd", cu_seqlens, n_seg, max_seqlen, total, nheads, head_dim, dtype,
                            {q_stride, k_stride, v_stride, o_stride, do_stride, dq_stride, dk_stride, dv_stride},
                            {q, k, v, o, d_o, (const void*)lse, dq, dk, dv, (const void*)delta}))
    return rc;
  if (total == 0) return MVIT_OK;
  // the long-segment kernels keep three arrays of row statistics in the workspace and park the pre-scaled queries in dq
  const bool wide = dtype == MVIT_BF16 && head_dim == 80 && max_seqlen >= WIDE_MIN_SEQLEN;
  const int64_t need = (wide ? 3 : 1) * (int64_t)nheads * total;
  MVIT_REQUIRE(delta_elems >= need, "attn_bwd: the delta workspace holds %lld floats, this call needs %lld (%d x nheads x total)",
               (long long)delta_elems, (long long)need, wide ? 3 : 1);
  {
    const int64_t e = dtype == MVIT_BF16 ? 2 : 4, width = (int64_t)nheads * head_dim * e;
    const struct { const void* ptr; int64_t stride; const char* name; } ins[] = {{q, q_stride, "q"}, {k, k_stride, "k"}, {v, v_stride, "v"}, {o, o_stride, "o"}, {d_o, do_stride, "d_o"}};
    const struct { const void* ptr; int64_t stride; const char* name; } outs[] = {{dq, dq_stride, "dq"}, {dk, dk_stride, "dk"}, {dv, dv_stride, "dv"}};
    for (const auto& w : outs)
      for (const auto& r : ins)
        MVIT_REQUIRE(!strided_rows_overlap(w.ptr, w.stride * e, r.ptr, r.stride * e, total, width),
                     "attn_bwd: %s overlaps %s (outputs are written, and dq is used as scratch, before all inputs have been read)", w.name, r.name);
  }
  if (n_seg == 0 || max_seqlen == 0 || total == 0) return MVIT_OK;
  AttnParams p = {};
  p.q = q; p.k = k; p.v = v; p.o = o; p.d_o = d_o; p.lse = const_cast<float*>(lse); p.delta = delta;
  p.dq = dq; p.dk = dk; p.dv = dv; p.cu = cu_seqlens; p.order = seg_order; p.total = total; p.nheads = nheads;
  p.q_stride = q_stride; p.k_stride = k_stride; p.v_stride = v_stride; p.o_stride = o_stride; p.do_stride = do_stride;
  p.dq_stride = dq_stride; p.dk_stride = dk_stride; p.dv_stride = dv_stride; p.scale = scale;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int vecw = dtype == MVIT_BF16 ? 8 : 4;
  const size_t part_bytes = (size_t)16 * nheads * (head_dim / vecw) * sizeof(float);
  if (dtype == MVIT_BF16 && max_seqlen <= 64 && head_dim <= 80) {
    // the window kernel derives delta from P and dP itself
  } else if (head_dim % vecw == 0 && o_stride % vecw == 0 && do_stride % vecw == 0 && part_bytes <= 48 * 1024 && mvit_aligned16(o) && mvit_aligned16(d_o)) {
    const int dgrid = (int)((total + 15) / 16);
    if (dtype == MVIT_BF16)
      hipLaunchKernelGGL((attn_delta_rows_kernel<bf16_t>), dgrid, 256, part_bytes, s, (const bf16_t*)o, (const bf16_t*)d_o, delta, total, nheads, head_dim, o_stride, do_stride);
    else
      hipLaunchKernelGGL((attn_delta_rows_kernel<float>), dgrid, 256, part_bytes, s, (const float*)o, (const float*)d_o, delta, total, nheads, head_dim, o_stride, do_stride);
  } else {
    const int64_t npairs = total * nheads;
    const int dgrid = (int)((npairs + 255) / 256);
    if (dtype == MVIT_BF16)
      hipLaunchKernelGGL((attn_delta_kernel<bf16_t>), dgrid, 256, 0, s, (const bf16_t*)o, (const bf16_t*)d_o, delta, total, nheads, head_dim, o_stride, do_stride);
    else
      hipLaunchKernelGGL((attn_delta_kernel<float>), dgrid, 256, 0, s, (const float*)o, (const float*)d_o, delta, total, nheads, head_dim, o_stride, do_stride);
  }
  MVIT_CHECK_LAUNCH("attn_delta");
  if (dtype == MVIT_BF16) {
    switch (head_dim) {
      case 32: return launch_bwd_mfma<2>(p, n_seg, max_seqlen, s);
      case 64: return launch_bwd_mfma<4>(p, n_seg, max_seqlen, s);
      case 80: return launch_bwd_mfma<5>(p, n_seg, max_seqlen, s);
      default: return launch_bwd_mfma<8>(p, n_seg, max_seqlen, s);
    }
  }
  return mvit_attn_f32(p, head_dim, n_seg, max_seqlen, true, s);
}

}  // extern "C"
