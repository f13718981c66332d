// MFMA GEMM for gfx950 with fused epilogues:  C[M,N] = epi( sum_k A[m,k] * B[n,k] ).
//
// Main loops:
//   bf16, the products of the vision tower: gemm_pp_kernel (gemm_pingpong.hip) and, where its 256x256 tiles are too few,
//      gemm_small_kernel (gemm_small.hip); choose_tile() below picks.
//   bf16, the rest (SwiGLU backward of many rows, patch embedding from frames, fp32 outputs, accumulation): 256x256 tile, 8
//      waves of 128x64 (4x2 blocks of 32x32 each), BK = 32, four LDS stages filled by direct global -> LDS loads (see
//      gemm_dl_kernel).
//   bf16 operands whose row pitch exceeds 2^22 elements (the direct loads use 32-bit lane offsets): 256x256 tile, 8 waves,
//      BK = 64, global -> registers -> LDS, double-buffered LDS, one barrier per K step (gemm_kernel).
//   fp32 (the parity path): gemm_f32_kernel (gemm_f32.hip).
// Operands whose contraction index is contiguous in memory are staged as [row][k] and read with 16-byte LDS
// loads; operands whose contraction index is the slow dimension (dgrad's weight, both operands of wgrad) are
// staged as [k][row] exactly as they lie in memory and read with ds_read_b64_tr_b16, which hands each lane 4
// consecutive k for its row.
// The epilogue stages the accumulators through LDS (fp32) so that bias / residual / activation inputs are
// read and results written as 16-byte vectors along N.
// Work-group ids are remapped so that the tiles a single XCD (one L2) works on are neighbours in N.
#include "gemm_common.h"
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>

namespace {


template <typename T>
struct Cfg;
template <>
struct Cfg<bf16_t> {
  static constexpr int BK = 64, VEC = 8;
  static constexpr int PITCH_K = BK + 8;  // [row][k] staging: 144-byte rows, conflict-free 16-byte reads
  static constexpr int PAD_T = 32;        // [k][row] staging: row pitch = rows + 32 elements
};

template <int VAR>
struct Waves;
template <>
struct Waves<1> {  // 256x256 tile, 8 waves of 128x64, double-buffered LDS, one work-group per CU
  static constexpr int BM = 256, BN = 256, WM = 128, WN = 64, NTHREADS = 512, MIN_WAVES = 2;
};

// Stage one operand tile (ROWS rows of the output dimension x BK of the contraction) global -> registers -> LDS.
// TR = false: memory is [row][k];  TR = true: memory is [k][row].
// A thread's chunks are a fixed distance apart (NTHREADS/8 rows, or NTHREADS/(ROWS/V) k-rows when TR), so one
// pointer, one remaining-K counter and a row mask describe the whole K loop.  Loads are unconditional (masked
// chunks read the operand's first element) and zeroed, if need be, when written to LDS.
// DUAL (SWIGLU's B operand): rows alternate between two matrices, so every chunk keeps its own pointer.
template <typename T, int ROWS, bool TR, int NTHREADS, int WN, bool DUAL>
struct TileLoader {
  using C = Cfg<T>;
  static constexpr int V = C::VEC;
  typedef T vec_t __attribute__((ext_vector_type(V)));
  static constexpr int CHUNKS = ROWS * C::BK / V;  // 16-byte chunks per tile
  static constexpr int PER_THREAD = CHUNKS / NTHREADS;
  static constexpr int LDS_ELEMS = TR ? C::BK * (ROWS + C::PAD_T) : ROWS * C::PITCH_K;
  static constexpr int ROW_STEP = TR ? 0 : NTHREADS / (C::BK / V);  // tile rows between consecutive chunks
  static constexpr int K_STEP = TR ? NTHREADS / (ROWS / V) : 0;     // k between consecutive chunks
  vec_t regs[PER_THREAD];
  const T* ptr[DUAL ? PER_THREAD : 1];
  const T* safe;      // always-valid address for masked chunks
  int64_t chunk_step; // elements between consecutive chunks of this thread
  int64_t step;       // pointer advance per K tile
  int k_left;         // K elements left from chunk 0's position (<= 0: exhausted)
  unsigned row_mask;  // bit i: chunk i lies on a valid row

  __device__ __forceinline__ void init(const T* __restrict__ base, const T* __restrict__ base2, int64_t ld,
                                       int64_t row0, int64_t row_limit, int64_t k_begin, int64_t k_end) {
    step = TR ? (int64_t)C::BK * ld : (int64_t)C::BK;
    chunk_step = TR ? (int64_t)K_STEP * ld : (int64_t)ROW_STEP * ld;
    safe = base;
    row_mask = 0;
    const int c0 = threadIdx.x;
    const int kk0 = TR ? c0 / (ROWS / V) : (c0 % (C::BK / V)) * V;
    const int64_t left = k_end - (k_begin + kk0);
    k_left = (int)(left > (1 << 30) ? (1 << 30) : left);
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int c = threadIdx.x + NTHREADS * i;
      const int r = TR ? (c % (ROWS / V)) * V : c / (C::BK / V);
      const int kk = TR ? c / (ROWS / V) : (c % (C::BK / V)) * V;
      const T* src = base;
      int64_t grow = row0 + r;
      if (DUAL) {  // tile row r = wn*WN + half*(WN/2) + j -> matrix `half`, row row0 + wn*(WN/2) + j
        const int wn = r / WN, w = r % WN, half = w / (WN / 2), j = w % (WN / 2);
        grow = row0 + wn * (WN / 2) + j;
        if (half) src = base2;
      }
      const bool row_ok = grow < row_limit;
      if (row_ok) row_mask |= 1u << i;
      const int64_t gk = k_begin + kk;
      const T* q = row_ok ? (TR ? src + gk * ld + grow : src + grow * ld + gk) : src;
      if (DUAL) ptr[i] = q;
      else if (i == 0) ptr[0] = TR ? src + gk * ld + grow : src + grow * ld + gk;  // may lie past the edge: never dereferenced then
    }
  }
  __device__ __forceinline__ bool live(int i, int kl) const { return ((row_mask >> i) & 1u) && (kl - i * K_STEP > 0); }
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const bool ok = live(i, k_left);
      const T* q = DUAL ? ptr[i] : ptr[0] + i * chunk_step;
      regs[i] = *reinterpret_cast<const vec_t*>(ok ? q : safe);
    }
    k_left -= C::BK;
    if (DUAL) {
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) ptr[i] += step;
    } else {
      ptr[0] += step;
    }
  }
  __device__ __forceinline__ void store(T* lds) const {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      vec_t v = regs[i];
      if (!live(i, k_left + C::BK)) {  // this chunk was outside the matrix / K range when it was loaded
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = from_f32<T>(0.f);
      }
      const int c = threadIdx.x + NTHREADS * i;
      int off;
      if (!TR) {
        const int r = c / (C::BK / V), kk = (c % (C::BK / V)) * V;
        off = r * C::PITCH_K + kk;
      } else {
        const int kk = c / (ROWS / V), r = (c % (ROWS / V)) * V;
        off = kk * (ROWS + C::PAD_T) + r;
      }
      *reinterpret_cast<vec_t*>(lds + off) = v;
    }
  }
};

// The A operand of the patch embedding made on the fly from decoded uint8 frames (no [rows, 1176] matrix in memory).
// The contraction index is re-ordered so that it runs along memory: k' = line * 48 + b with line = frame-of-the-pair *
// 14 + y and b = x * 3 + channel for b < 42 (the 42 bytes of one pixel line of a patch are contiguous in the frame);
// b = 42..47 pads the line to six 8-byte pieces and meets zero weights (mvit_patch_embed_pack_weight).
// 1344 = 28 lines * 48 = 42 K tiles of 32.  A lane fetches one 8-byte piece per row and K tile with a single vector load
// and turns it into a 16-byte bf16 chunk with eight conversions byte -> float -> a * x + c -> bf16.  Pieces advance by a
// fixed count per K tile, so (line, piece) and the channel of the piece's first byte are stepped, not recomputed.
constexpr int PX_LINE = 48, PX_LINES = 28, PX_K = PX_LINE * PX_LINES, PX_PATCH = 14;
__device__ __forceinline__ int px_find_image(const mvit_image* t, int n, int64_t row) {
  int lo = 0, hi = n;  // invariant: t[lo].first_row <= row < t[hi].first_row
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (t[mid].first_row <= row) lo = mid;
    else hi = mid;
  }
  return lo;
}
// Where patch `row` of the batch lies: first byte of its 14 x 14 pixel square in the first frame of its temporal pair,
// bytes per image line, distance to the pair's second frame (0 when
// the last frame of an odd count, or a still image, fills both halves).
__device__ __forceinline__ void px_locate(const GemmParams& p, int64_t row, const uint8_t*& base, int& line_bytes, int& frame_off) {
  if (row >= p.M) row = p.M - 1;  // rows past the edge repeat the last row; their results are never stored
  const mvit_image im = p.px_images[px_find_image(p.px_images, p.px_n_images, row)];
  const int gh = im.height / PX_PATCH, gw = im.width / PX_PATCH, per_t = gh * gw;
  const int64_t local = row - im.first_row;
  const int t = (int)(local / per_t), rem = (int)(local % per_t);
  // rem = ((block row * (gw / 2) + block column) * 2 + row in block) * 2 + column in block
  const int blk = rem >> 2, hb = blk / (gw >> 1), wb = blk % (gw >> 1);
  const int y0 = (2 * hb + ((rem >> 1) & 1)) * PX_PATCH, x0 = (2 * wb + (rem & 1)) * PX_PATCH;
  const int f0 = 2 * t, f1 = f0 + 1 < im.frames ? f0 + 1 : im.frames - 1;
  const int lb = im.width * 3;
  const int64_t fb = (int64_t)lb * im.height;
  const int64_t first = f0 * fb + (int64_t)y0 * lb + x0 * 3;
  line_bytes = lb;
  frame_off = (int)((f1 - f0) * fb);
  base = im.pixels + first;
}
// The 8 bytes at p (2-byte aligned when the frame buffer is 4-byte aligned; global memory takes unaligned vector loads),
// as one load whose result is not touched until px_convert8, so that it can stay in flight.
struct PxRaw {
  u32x2 w;
};
__device__ __forceinline__ void px_fetch8(const uint8_t* p, PxRaw& r) {
  typedef __attribute__((address_space(1))) const uint8_t* global_bytes;  // frames are in device memory: no generic-address load
  __builtin_memcpy(&r.w, (global_bytes)(uintptr_t)p, 8);
}
// the normalisation constants as six scalars (kernel arguments indexed by a lane-varying channel would be fetched from
// memory for every use)
struct PxNorm {
  float a0, a1, a2, c0, c1, c2;
  __device__ __forceinline__ explicit PxNorm(const GemmParams& p) : a0(p.px_a[0]), a1(p.px_a[1]), a2(p.px_a[2]), c0(p.px_c[0]), c1(p.px_c[1]), c2(p.px_c[2]) {}
};
// 8 bytes -> bf16(byte * a + c), the first byte belonging to channel ch0.  tail: the load was moved 6 bytes back so that
// it ends with the line (piece 5 holds bytes 40, 41 of the line and six padding columns): its last two bytes are the
// piece's first two, the rest of the piece is padding.
__device__ __forceinline__ bf16x8 px_convert8(const PxRaw& r, int ch0, bool tail, const PxNorm nm) {
  const unsigned raw[2] = {tail ? r.w[1] >> 16 : r.w[0], tail ? 0u : r.w[1]};
  // a, c of bytes 0, 1, 2 (mod 3) of the piece: the constants rotated by ch0
  const bool r1 = ch0 == 1, r2 = ch0 == 2;
  const float ar0 = r2 ? nm.a2 : (r1 ? nm.a1 : nm.a0), ar1 = r2 ? nm.a0 : (r1 ? nm.a2 : nm.a1), ar2 = r2 ? nm.a1 : (r1 ? nm.a0 : nm.a2);
  const float cr0 = r2 ? nm.c2 : (r1 ? nm.c1 : nm.c0), cr1 = r2 ? nm.c0 : (r1 ? nm.c2 : nm.c1), cr2 = r2 ? nm.c1 : (r1 ? nm.c0 : nm.c2);
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = (float)((raw[e >> 2] >> (8 * (e & 3))) & 0xffu);
    v[e] = (bf16_t)__builtin_fmaf(x, e % 3 == 0 ? ar0 : (e % 3 == 1 ? ar1 : ar2), e % 3 == 0 ? cr0 : (e % 3 == 1 ? cr1 : cr2));
  }
  return v;
}
// MFMA operand fetch from LDS for the 32-row sub-tile starting at `row`, contraction offset `k`.
template <bool TR, int ROWS>
__device__ __forceinline__ bf16x8 frag_bf16(const bf16_t* lds, int row, int k) {
  using C = Cfg<bf16_t>;
  const int l = threadIdx.x & 63;
  if (!TR) {
    return *reinterpret_cast<const bf16x8*>(lds + (row + (l & 31)) * C::PITCH_K + k + 8 * (l >> 5));
  } else {
    // lane i of 16-lane group G fetches 4 elements of k-row (k + 8*(G/2) + i/4) at column 16*(G%2) + 4*(i%4);
    // the transposing read returns to lane j of the group the 4 consecutive k of column 16*(G%2) + j.
    constexpr int P = ROWS + C::PAD_T;
    const int G = l >> 4, i = l & 15;
    const bf16_t* p = lds + (k + 8 * (G >> 1) + (i >> 2)) * P + row + 16 * (G & 1) + 4 * (i & 3);
    typedef s16x4 __attribute__((address_space(3))) * lds_ptr_t;
    s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
    s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + 4 * P));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, both);
  }
}

// Per-element epilogue inputs (residual / saved activations) of an interior tile, fetched ahead of their use.
// One pass of the epilogue covers (BM/WM)*32 rows; a thread owns ITEMS 8-column groups per pass.  Two passes are
// buffered (one when an element needs two inputs): the epilogue requests pass a+2 when pass a has been consumed.
template <typename T, int EPI, int BM, int BN, int WM, int NTHREADS>
struct EpiPre {
  static constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  static constexpr int PASS_ROWS = (BM / WM) * 32, GROUPS = (DUAL ? BN / 2 : BN) / 8;
  static constexpr bool HAS_IN = (EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_GELU_BWD || EPI == MVIT_EPI_SWIGLU_BWD) &&
                                 (PASS_ROWS * GROUPS) % NTHREADS == 0;
  static constexpr int ITEMS = HAS_IN ? PASS_ROWS * GROUPS / NTHREADS : 1, NLOAD = EPI == MVIT_EPI_SWIGLU_BWD ? 2 : 1;
  static constexpr int RPI = NTHREADS / GROUPS;  // rows between a thread's consecutive items
  static_assert(!HAS_IN || (NTHREADS % GROUPS == 0 && 32 % RPI == 0), "row mapping of the prefetched epilogue");
  typedef T raw8 __attribute__((ext_vector_type(8)));
  static constexpr int NBUF = NLOAD == 2 ? 1 : 2;  // passes buffered (two 16-byte inputs per element: one pass)
  raw8 pre[NBUF][ITEMS][NLOAD];
  const char* base;     // R + m0 * ldr + n0 (block-uniform)
  unsigned thread_off;  // this thread's byte offset inside a pass: row threadIdx / GROUPS, column group threadIdx % GROUPS
  bool active;          // block-uniform: this tile takes the prefetched path

  __device__ __forceinline__ void init(const GemmParams& p, int64_t m0, int64_t n0) {
    active = HAS_IN && p.vec_ok && m0 + BM <= p.M && n0 + GROUPS * 8 <= p.N && p.ldr * (int64_t)BM * sizeof(T) < (1ll << 31);
    base = reinterpret_cast<const char*>(static_cast<const T*>(p.R) + m0 * p.ldr + n0);
    thread_off = (unsigned)(((threadIdx.x / GROUPS) * p.ldr + (threadIdx.x % GROUPS) * 8) * sizeof(T));
  }
  // Item `it` of pass a is tile row (RPI*it/32)*WM + a*32 + (RPI*it)%32 + threadIdx/GROUPS: a uniform row offset
  // (scalar address arithmetic) plus the per-thread offset.
  __device__ __forceinline__ void load_item(const GemmParams& p, int a, int it, raw8 (&dst)[NLOAD]) const {
    const int rowoff = (RPI * it / 32) * WM + a * 32 + (RPI * it) % 32;
    const char* r = base + (int64_t)rowoff * p.ldr * (int64_t)sizeof(T);
    dst[0] = load8_stream<T>(r + thread_off);
    if (NLOAD == 2) dst[1] = load8_stream<T>(r + p.aux_off * (int64_t)sizeof(T) + thread_off);
  }
  template <int BUF>
  __device__ __forceinline__ void fetch(const GemmParams& p, int a) {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) load_item(p, a, it, pre[BUF][it]);
  }
};

// Epilogue shared by every main loop.  acc[a][b][4*j+i] is C[m0 + wm*WM + a*32 + 8*j + 4*(l/32) + i][wave column
// b*32 + l%32].  Pass a: every wave parks its a-th 32-row sub-tile in LDS (fp32, [(BM/WM)*32 rows][BN + 8]), then
// the block walks the pass in 8-column groups.  The caller guarantees that no wave still reads operands from LDS.
template <typename T, typename TO, int EPI, int BM, int BN, int WM, int WN, int NTHREADS, bool MI16 = false>
__device__ __forceinline__ void run_epilogue(const GemmParams& p, f32x16 (&acc)[WM / 32][WN / 32], unsigned char* smem_raw,
                                             int64_t m0, int64_t n0, int wm, int wn, int slice,
                                             EpiPre<T, EPI, BM, BN, WM, NTHREADS>& ep) {
  constexpr int MT = WM / 32, NT = WN / 32;
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  const int l = threadIdx.x & 63;
  // MI16: acc[a][b] holds the four 16x16 results of the 32x32 block, [(ra*2 + cb)*4 + i] = C[16*ra + 4*(l/16) + i][16*cb + l%16]
  // Staging rows are BN floats with no padding; 16-column chunks of a row are permuted by the row instead, so that the
  // rows one parking store touches (4 apart: four of them with the 16x16 results, two with the 32x32 ones) fall on
  // different banks.  Groups of 8 columns stay contiguous for the read-out.
  constexpr int SP = BN;
  auto swz = [](int row) { return MI16 ? ((row >> 2) & 3) << 4 : ((row >> 2) & 1) << 5; };
  constexpr int PASS_ROWS = (BM / WM) * 32;
  constexpr int NCOLS = DUAL ? BN / 2 : BN;
  constexpr int GROUPS = NCOLS / 8;
  float* stage = reinterpret_cast<float*>(smem_raw);
  const int lc = l & 31, lr = 4 * (l >> 5);
  const bool to_ws = (EPI == MVIT_EPI_NONE) && p.split_k > 1;
  float* ws = to_ws ? p.workspace + (int64_t)slice * p.M * p.N : nullptr;
  const bool ws_vec = (p.N % 4 == 0);
  // SWIGLU_BWD can hand back the column sums of dg | du (the bias gradient): a thread's items all lie in the same
  // 8 columns, so it keeps 2 x 8 running sums; after the last pass the rows-of-threads are added through LDS.
  constexpr bool CAN_CS = (EPI == MVIT_EPI_SWIGLU_BWD) && NTHREADS % GROUPS == 0 && NTHREADS == 2 * GROUPS * 8;
  float cs_acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) cs_acc[e] = 0.f;
  const bool do_cs = CAN_CS && p.colsum != nullptr;
  auto finish_colsum = [&]() {
    if constexpr (CAN_CS) {
      if (!do_cs) return;
      constexpr int TR_ = NTHREADS / GROUPS;  // thread rows sharing a column group
      __syncthreads();                        // the staging area is free
      float* red = stage;                     // [TR_][2][GROUPS * 8]
      const int trow = threadIdx.x / GROUPS, cgx = threadIdx.x % GROUPS;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        red[(trow * 2 + 0) * (GROUPS * 8) + cgx * 8 + e] = cs_acc[e];
        red[(trow * 2 + 1) * (GROUPS * 8) + cgx * 8 + e] = cs_acc[8 + e];
      }
      __syncthreads();
      const int half = threadIdx.x / (GROUPS * 8), col = threadIdx.x % (GROUPS * 8);  // NTHREADS == 2 * GROUPS * 8
      float t = 0.f;
#pragma unroll
      for (int k = 0; k < TR_; ++k) t += red[(k * 2 + half) * (GROUPS * 8) + col];
      if (n0 + col < p.N) p.colsum[(m0 / BM) * p.ldc + (half ? p.aux_off : 0) + n0 + col] = t;
    }
  };

  // Tiles inside the matrix: compile-time trip counts, no edge tests, 16-byte accesses only.  When the epilogue
  // reads one value per output element, those reads run up to two passes ahead, so their latency hides behind
  // the LDS staging and the previous passes' arithmetic and stores.
  using EP = EpiPre<T, EPI, BM, BN, WM, NTHREADS>;
  if constexpr ((PASS_ROWS * GROUPS) % NTHREADS == 0) {
    const bool interior = m0 + BM <= p.M && n0 + NCOLS <= p.N && (to_ws ? ws_vec : p.vec_ok != 0) && (!EP::HAS_IN || ep.active);
    if (interior) {
      constexpr int ITEMS = PASS_ROWS * GROUPS / NTHREADS;
      constexpr int NBUF = EP::NBUF;
      // a thread's items all lie in one 8-column group (NTHREADS is a multiple of GROUPS): its bias values are loaded
      // once per tile, before the accumulators are parked, instead of once per item behind the previous items' stores
      // (memory instructions of a wave complete in order, so a load issued after a store also waits for that store)
      constexpr bool HAS_BIAS = EPI == MVIT_EPI_BIAS || EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_BIAS_GELU || EPI == MVIT_EPI_SWIGLU;
      static_assert(NTHREADS % GROUPS == 0, "a thread's items share their column group");
      float hb[8], hb2[8];
      if constexpr (HAS_BIAS) {
        const int64_t nb = n0 + (threadIdx.x % GROUPS) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) hb[e] = hb2[e] = 0.f;
        if (p.bias) load8(static_cast<const T*>(p.bias) + nb, hb);
        if (DUAL && p.bias2) load8(static_cast<const T*>(p.bias2) + nb, hb2);
      }
      if constexpr (EP::HAS_IN) {
        ep.template fetch<0>(p, 0);
        if (NBUF == 2 && MT > 1) ep.template fetch<(NBUF - 1)>(p, 1);
      }
#pragma unroll
      for (int a = 0; a < MT; ++a) {
        if (a > 0) __syncthreads();
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          int col;
          if (DUAL) col = (b / (NT / 2)) * (BN / 2) + wn * (WN / 2) + (b % (NT / 2)) * 32 + lc;
          else col = wn * WN + b * 32 + lc;
          if constexpr (MI16) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                stage[(wm * 32 + 16 * (q >> 1) + 4 * (l >> 4) + i) * SP + (((col - lc) + 16 * (q & 1) + (l & 15)) ^ swz(4 * (l >> 4)))] = acc[a][b][4 * q + i];
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int i = 0; i < 4; ++i) stage[(wm * 32 + 8 * j + lr + i) * SP + (col ^ swz(lr))] = acc[a][b][4 * j + i];
          }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
          const int c = threadIdx.x + NTHREADS * it, row = c / GROUPS, cg = c % GROUPS;
          const int64_t m = m0 + (row / 32) * WM + a * 32 + (row % 32), n = n0 + cg * 8;
          const float* sp = stage + row * SP + ((cg * 8) ^ swz(row));
          const f32x4 v0 = *reinterpret_cast<const f32x4*>(sp), v1 = *reinterpret_cast<const f32x4*>(sp + 4);
          float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
          float u[8];
          if (DUAL) {
            const f32x4 u0 = *reinterpret_cast<const f32x4*>(sp + BN / 2), u1 = *reinterpret_cast<const f32x4*>(sp + BN / 2 + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              u[e] = u0[e];
              u[4 + e] = u1[e];
            }
          }
          if (to_ws) store8(ws + m * p.N + n, v);
          else if constexpr (EP::HAS_IN) {
            // the same item of pass a + NBUF is requested before this item's stores are issued: a wave's memory
            // instructions complete in order, so the wait for a load also waits for every store issued before it
            typename EP::raw8 nx[EP::NLOAD];
            if (a + NBUF < MT) ep.load_item(p, a + NBUF, it, nx);
            emit8_impl<T, TO, EPI, true, true>(p, m, n, v, u, ep.pre[a % NBUF][it], cs_acc, do_cs, HAS_BIAS ? hb : nullptr, nullptr);
            if (a + NBUF < MT) {
#pragma unroll
              for (int k = 0; k < EP::NLOAD; ++k) ep.pre[a % NBUF][it][k] = nx[k];
            }
            if constexpr (EP::NLOAD == 2) __builtin_amdgcn_sched_barrier(0);  // keeps the items apart: registers
          } else emit8_impl<T, TO, EPI, true, false>(p, m, n, v, u, nullptr, cs_acc, false, HAS_BIAS ? hb : nullptr, (HAS_BIAS && DUAL) ? hb2 : nullptr);
        }
      }
      finish_colsum();
      return;
    }
  }
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    if (a > 0) __syncthreads();
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      int col;
      if (DUAL) col = (b / (NT / 2)) * (BN / 2) + wn * (WN / 2) + (b % (NT / 2)) * 32 + lc;
      else col = wn * WN + b * 32 + lc;
      if constexpr (MI16) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            stage[(wm * 32 + 16 * (q >> 1) + 4 * (l >> 4) + i) * SP + (((col - lc) + 16 * (q & 1) + (l & 15)) ^ swz(4 * (l >> 4)))] = acc[a][b][4 * q + i];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) stage[(wm * 32 + 8 * j + lr + i) * SP + (col ^ swz(lr))] = acc[a][b][4 * j + i];
      }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < PASS_ROWS * GROUPS; c += NTHREADS) {
      const int row = c / GROUPS, cg = c % GROUPS;
      const int64_t m = m0 + (row / 32) * WM + a * 32 + (row % 32);
      const int64_t n = n0 + cg * 8;
      if (m >= p.M || n >= p.N) continue;
      float v[8], u[8];
      const float* sp = stage + row * SP + ((cg * 8) ^ swz(row));
      const f32x4 v0 = *reinterpret_cast<const f32x4*>(sp), v1 = *reinterpret_cast<const f32x4*>(sp + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = v0[e];
        v[4 + e] = v1[e];
      }
      if (DUAL) {
        const f32x4 u0 = *reinterpret_cast<const f32x4*>(sp + BN / 2), u1 = *reinterpret_cast<const f32x4*>(sp + BN / 2 + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[e] = u0[e];
          u[4 + e] = u1[e];
        }
      }
      if (to_ws) {
        float* w = ws + m * p.N + n;
        if (ws_vec && n + 8 <= p.N) store8(w, v);
        else
          for (int e = 0; e < 8 && n + e < p.N; ++e) w[e] = v[e];
      } else {
        emit8<T, TO, EPI>(p, m, n, v, u, p.vec_ok != 0, cs_acc, do_cs);
      }
    }
  }
  finish_colsum();
}

template <typename T, typename TO, bool TA, bool TB, int EPI, int VAR>
__global__ __launch_bounds__(Waves<VAR>::NTHREADS, Waves<VAR>::MIN_WAVES) void gemm_kernel(const GemmParams p) {
  using C = Cfg<T>;
  using W = Waves<VAR>;
  constexpr int BK = C::BK, BM = W::BM, BN = W::BN, WM = W::WM, WN = W::WN, NTHREADS = W::NTHREADS;
  constexpr int MT = WM / 32, NT = WN / 32, WGN = BN / WN;  // waves along N
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  using LoaderA = TileLoader<T, BM, TA, NTHREADS, WN, false>;
  using LoaderB = TileLoader<T, BN, TB, NTHREADS, WN, DUAL>;
  constexpr int STAGE_ELEMS = LoaderA::LDS_ELEMS + LoaderB::LDS_ELEMS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T* lds = reinterpret_cast<T*>(smem_raw);

  // XCD-aware tile order: hardware deals consecutive work-group ids round-robin to the 8 XCDs; give each
  // XCD a contiguous range of tiles (N fastest) so that its L2 sees one A panel at a time.
  // With split-K the slices are the slowest index: all tiles of one K slice share the same rows of A and B.
  const int tiles = p.tiles_m * p.tiles_n;
  const int total = tiles * p.split_k;
  const int per_xcd = (total + 7) / 8;
  const int work = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (work >= total) return;
  const int slice = work / tiles, tile = work % tiles;
  int tm, tn;
  tile_coords(p, tile, tm, tn);
  const int64_t k_begin = (int64_t)slice * p.k_chunk;
  const int64_t k_end = p.split_k > 1 ? (k_begin + p.k_chunk < p.K ? k_begin + p.k_chunk : p.K) : p.K;
  constexpr int N_PER_BLOCK = DUAL ? BN / 2 : BN;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * N_PER_BLOCK;

  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wm = wv / WGN, wn = wv % WGN;

  f32x16 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  LoaderA la;
  LoaderB lb;
  const T* A = static_cast<const T*>(p.A);
  const T* B = static_cast<const T*>(p.B);
  const T* B2 = static_cast<const T*>(p.B2);
  la.init(A, nullptr, p.lda, m0, p.M, k_begin, k_end);
  lb.init(B, B2, p.ldb, n0, p.N, k_begin, k_end);
  la.load();
  lb.load();
  la.store(lds);
  lb.store(lds + LoaderA::LDS_ELEMS);
  __syncthreads();

  int buf = 0;
  for (int64_t k0 = k_begin; k0 < k_end; k0 += BK) {
    const bool has_next = k0 + BK < k_end;
    if (has_next) {
      la.load();
      lb.load();
    }
    const T* lds_a = lds + buf * STAGE_ELEMS;
    const T* lds_b = lds_a + LoaderA::LDS_ELEMS;
    {
      // operand fragments are fetched one 16-wide step ahead of the MFMAs that consume them
      const bf16_t* la_ = reinterpret_cast<const bf16_t*>(lds_a);
      const bf16_t* lb_ = reinterpret_cast<const bf16_t*>(lds_b);
      bf16x8 fa[2][MT], fb[2][NT];
#pragma unroll
      for (int a = 0; a < MT; ++a) fa[0][a] = frag_bf16<TA, BM>(la_, wm * WM + a * 32, 0);
#pragma unroll
      for (int b = 0; b < NT; ++b) fb[0][b] = frag_bf16<TB, BN>(lb_, wn * WN + b * 32, 0);
#pragma unroll
      for (int s4 = 0; s4 < BK / 16; ++s4) {
        const int cur = s4 & 1, nxt = cur ^ 1;
        if (s4 + 1 < BK / 16) {
#pragma unroll
          for (int a = 0; a < MT; ++a) fa[nxt][a] = frag_bf16<TA, BM>(la_, wm * WM + a * 32, (s4 + 1) * 16);
#pragma unroll
          for (int b = 0; b < NT; ++b) fb[nxt][b] = frag_bf16<TB, BN>(lb_, wn * WN + b * 32, (s4 + 1) * 16);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the fetches of step s4+1 ahead of the MFMAs of step s4
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
          for (int b = 0; b < NT; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[cur][a], fb[cur][b], acc[a][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (has_next) {
      T* nxt = lds + (buf ^ 1) * STAGE_ELEMS;
      la.store(nxt);
      lb.store(nxt + LoaderA::LDS_ELEMS);
    }
    __syncthreads();  // also: operands fully consumed before LDS is reused by the epilogue
    buf ^= 1;
  }

  EpiPre<T, EPI, BM, BN, WM, NTHREADS> ep;
  ep.init(p, m0, n0);
  run_epilogue<T, TO, EPI, BM, BN, WM, WN, NTHREADS>(p, acc, smem_raw, m0, n0, wm, wn, slice, ep);
}

// ---- bf16 main loop with direct global -> LDS loads (no staging registers) ----------------------------------
// 256x256 tile, 8 waves of 128x64, BK = 32, NSTAGE LDS stages of 16 KiB per operand.  global_load_lds_dwordx4 moves
// 16 bytes per lane straight into LDS at M0 + 16*lane, so one wave instruction fills 1 KiB of contiguous LDS and
// NSTAGE-1 K tiles are in flight while one is consumed; addresses are a per-lane 32-bit offset (constant over the
// K loop) plus a wave-uniform 64-bit base that a scalar add advances.  Because the LDS image of one instruction
// is contiguous, bank conflicts are avoided by permuting which global chunk a lane fetches:
//   [row][k] operands: 64-byte rows of 4 chunks, chunk c of row r lives in slot c ^ ((r >> 2) & 3);
//   [k][row] operands: 512-byte k-rows of 32 chunks, chunk c of k-row k lives in slot c ^ ((k & 3) << 2).
// Rows past the matrix edge are clamped to valid rows (they only feed outputs that are never stored).  A partial
// last K tile (K not a multiple of 32) is loaded through registers with zeros past the end of K.
// The compiler does not see these loads: s_waitcnt vmcnt is placed by hand (loads return in order).
// waves per work-group: 8 -> each owns 128x64 (two waves per SIMD), 4 -> 128x128 (one per SIMD).
template <int NW>
struct DL {
  static constexpr int BM = 256, BN = 256, BK = 32, WM = 128, WN = NW == 8 ? 64 : 128, NTHREADS = 64 * NW;
  static constexpr int TILE_BYTES = 256 * BK * 2;
  static constexpr int CPT = 16 / NW;  // 1 KiB load instructions per wave and K tile and operand
};
constexpr int DL_BK = 32, DL_TILE_BYTES = 256 * DL_BK * 2;

__device__ __forceinline__ void dl_load(unsigned lds_addr, unsigned voff, const char* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

template <bool TR, bool DUAL, int NW, bool MI16 = false>
struct DlOperand {
  static constexpr int CPT = DL<NW>::CPT, WN = DL<NW>::WN;
  unsigned voff[CPT];  // byte offset of this lane's 16-byte chunks from `base`
  const char* base;    // wave-uniform, advanced by `step` every K tile (DUAL: odd waves read the second matrix)
  int64_t step;

  __device__ __forceinline__ void init(const bf16_t* X, const bf16_t* X2, int64_t ld, int64_t row0, int64_t limit,
                                       int64_t k_begin, int wv) {
    const int l = threadIdx.x & 63;
    step = TR ? 2 * DL_BK * ld : 2 * DL_BK;
    // DUAL: tile row r = wn*WN + half*(WN/2) + j -> matrix `half`, row row0 + wn*(WN/2) + j; a wave's rows
    // [wv * 16 * CPT, +16 * CPT) all have half = wv & 1.
    const bf16_t* src = (DUAL && (wv & 1)) ? X2 : X;
    base = reinterpret_cast<const char*>(TR ? src + k_begin * ld + row0 : src + row0 * ld + k_begin);
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int q = wv * CPT + i;  // which 1 KiB of the stage this instruction fills
      if (!TR) {
        const int r = q * 16 + (l >> 2), c = (l & 3) ^ ((r >> 2) & 3);
        int64_t grow = row0 + r;
        if (DUAL) grow = row0 + (r / WN) * (WN / 2) + (r % (WN / 2));
        if (grow >= limit) grow = limit - 1;
        voff[i] = (unsigned)(((grow - row0) * ld + c * 8) * 2);
      } else {
        const int kr = 2 * q + (l >> 5);
        // MI16: the four 16-lane groups of a transposing read sit 8 k-rows apart; odd multiples of 8 are moved
        // by two chunks so that two neighbouring groups never share banks
        int ch = (l & 31) ^ ((kr & 3) << 2) ^ (MI16 ? ((kr >> 3) & 1) << 1 : 0);
        if (row0 + ch * 8 >= limit) ch = 0;
        voff[i] = (unsigned)((kr * ld + ch * 8) * 2);
      }
    }
  }
  // lds_addr: LDS byte address of this wave's CPT KiB slice of the operand's stage
  __device__ __forceinline__ void issue(unsigned lds_addr) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) dl_load(lds_addr + i * 1024, voff[i], base);
    base += step;
  }
  __device__ __forceinline__ void issue_tail(unsigned char* lds_slice, int k_rem, int wv) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int q = wv * CPT + i;
      int k;  // first contraction index of the chunk
      if (!TR) {
        const int r = q * 16 + (l >> 2);
        k = ((l & 3) ^ ((r >> 2) & 3)) * 8;
      } else {
        k = 2 * q + (l >> 5);
      }
      bf16x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = from_f32<bf16_t>(0.f);
      if (k < k_rem) v = *reinterpret_cast<const bf16x8*>(base + voff[i]);
      *reinterpret_cast<bf16x8*>(lds_slice + i * 1024 + l * 16) = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // written before this wave's next barrier
  }
};

// The loader of that operand for the DL layout: this operand cannot travel global -> LDS directly, so a K tile takes two calls, a step of the main loop apart:
// request() loads this lane's 8 bytes of each of its CPT rows into registers, flush() converts them and writes the 16-byte
// chunk where the direct load of a [row][k] operand would have put it (slot l of the wave's 1 KiB slice holds chunk
// (l & 3) ^ ((row >> 2) & 3) of row 16 * slice + l / 4).  A K tile of 32 is 4 pieces, so pieces advance by 4 per tile.
template <int NW>
struct DlPixelOperand {
  static constexpr int CPT = DL<NW>::CPT;
  static_assert(PX_K % DL_BK == 0, "whole K tiles");
  const uint8_t* base[CPT];
  int line_bytes[CPT], frame_off[CPT];
  int line, piece;  // of the next request
  int ch0;          // channel of the first byte of the piece that the next flush converts
  PxRaw raw[CPT];

  __device__ __forceinline__ void init(const GemmParams& p, int64_t row0, int wv) {
    const int l = threadIdx.x & 63;
    line = 0;
    piece = (l & 3) ^ ((l >> 4) & 3);  // (row >> 2) & 3 = (l >> 4) & 3: slices start at multiples of 16 rows
    ch0 = (2 * piece) % 3;
#pragma unroll
    for (int i = 0; i < CPT; ++i) px_locate(p, row0 + (wv * CPT + i) * 16 + (l >> 2), base[i], line_bytes[i], frame_off[i]);
  }
  __device__ __forceinline__ void request() {
    const int second = line >= PX_PATCH ? 1 : 0, y = line - PX_PATCH * second;
    const int in_line = piece == 5 ? 8 * 5 - 6 : 8 * piece;  // the last piece is read as the last 8 bytes of the line
#pragma unroll
    for (int i = 0; i < CPT; ++i) px_fetch8(base[i] + ((second ? frame_off[i] : 0) + y * line_bytes[i] + in_line), raw[i]);
    piece += 4;
    if (piece >= 6) {
      piece -= 6;
      line += 1;
    }
  }
  // lds_slice: this wave's CPT KiB of the operand's stage.  The write is complete before the wave's next barrier
  // because the fragment reads that follow it in program order are (LDS operations of a wave complete in order).
  __device__ __forceinline__ void flush(unsigned char* lds_slice, const PxNorm nm) {
    const int l = threadIdx.x & 63;
    const bool tail = piece == 3;  // the piece in registers is 4 pieces (mod 6) before the next request's
#pragma unroll
    for (int i = 0; i < CPT; ++i) *reinterpret_cast<bf16x8*>(lds_slice + i * 1024 + l * 16) = px_convert8(raw[i], ch0, tail, nm);
    ch0 = ch0 == 0 ? 2 : ch0 - 1;  // 32 bytes further: + 2 mod 3 (a wrap to the next line moves by 48 = 0 mod 3)
  }
};

// MFMA operand fetch for the DL layout: sub-tile `a` (32 rows) of the wave, 16-wide contraction step ks, stage s.
template <bool TR, int NSUB, bool MI16 = false>
struct DlFrag {
  unsigned off[MI16 ? (TR ? 2 * NSUB : 1) : (TR ? NSUB : 2)];
  __device__ __forceinline__ void init(int rowbase, unsigned region) {
    const int l = threadIdx.x & 63;
    if constexpr (MI16) {
      // v_mfma_f32_16x16x32 operand: lane l holds row l%16 of a 16-row block, contraction 8*(l/16) .. +7 of the 32-wide stage
      if (!TR) {
        const int r = rowbase + (l & 15);  // blocks are 16 rows apart: (r >> 2) & 3 is the same for every block
        off[0] = region + r * 64 + (((l >> 4) ^ ((r >> 2) & 3)) << 4);
      } else {
        const int G = l >> 4, i = l & 15, k = 8 * G + (i >> 2);
#pragma unroll
        for (int a = 0; a < 2 * NSUB; ++a) {
          const int ch = (rowbase + a * 16) / 8 + ((i & 3) >> 1);
          off[a] = region + k * 512 + ((ch ^ ((k & 3) << 2) ^ (((k >> 3) & 1) << 1)) << 4) + (i & 1) * 8;
        }
      }
      return;
    }
    if (!TR) {
      const int x = ((l & 31) >> 2) & 3;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) off[ks] = region + (rowbase + (l & 31)) * 64 + (((ks * 2 + (l >> 5)) ^ x) << 4);
    } else {
      // lane i of 16-lane group G fetches 4 rows of k-row 8*(G/2) + i/4 at row 16*(G%2) + 4*(i%4); the transposing
      // read hands lane j of the group the 4 consecutive k of row 16*(G%2) + j.
      const int G = l >> 4, i = l & 15;
#pragma unroll
      for (int a = 0; a < NSUB; ++a) {
        const int ch = (rowbase + a * 32) / 8 + 2 * (G & 1) + ((i & 3) >> 1);
        off[a] = region + (8 * (G >> 1) + (i >> 2)) * 512 + ((ch ^ (((i >> 2) & 3) << 2)) << 4) + (i & 1) * 8;
      }
    }
  }
  // MI16: fragment of the 16-row block `blk` of the wave for the whole 32-wide stage s
  __device__ __forceinline__ bf16x8 read16(const unsigned char* smem, int blk, int s) const {
    if (!TR) {
      return *reinterpret_cast<const bf16x8*>(smem + off[0] + blk * 16 * 64 + s * DL_TILE_BYTES);
    } else {
      typedef s16x4 __attribute__((address_space(3))) * lds_ptr_t;
      const unsigned char* p = smem + off[blk] + s * DL_TILE_BYTES;
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + 4 * 512));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8, both);
    }
  }
  __device__ __forceinline__ bf16x8 read(const unsigned char* smem, int a, int ks, int s) const {
    if (!TR) {
      return *reinterpret_cast<const bf16x8*>(smem + off[ks] + a * 32 * 64 + s * DL_TILE_BYTES);
    } else {
      typedef s16x4 __attribute__((address_space(3))) * lds_ptr_t;
      const unsigned char* p = smem + off[a] + s * DL_TILE_BYTES + ks * 16 * 512;
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p));
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + 4 * 512));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      return __builtin_bit_cast(bf16x8, both);
    }
  }
};

// Wait until at most n K tiles' loads (PER per lane each) are still in flight.
template <int PER>
__device__ __forceinline__ void wait_tiles(int n) {
  if (n >= 3) wait_vm<3 * PER>();
  else if (n == 2) wait_vm<2 * PER>();
  else if (n == 1) wait_vm<PER>();
  else wait_vm<0>();
}

// PIX: the A operand is made from decoded frames (DlPixelOperand)
template <typename TO, bool TA, bool TB, int EPI, int NSTAGE, int NW, bool MI16 = false, bool PIX = false>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemm_dl_kernel(const GemmParams p) {
  static_assert(!PIX || (!TA && !MI16), "frames as the A operand: [row][k] layout, 32x32x16 fragments");
  using T = bf16_t;
  using D = DL<NW>;
  constexpr int BM = D::BM, BN = D::BN, WM = D::WM, WN = D::WN, TILE = D::TILE_BYTES, SLICE = D::CPT * 1024;
  constexpr int MT = WM / 32, NT = WN / 32, WGN = BN / WN;
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const int tiles = p.tiles_m * p.tiles_n;
  const int total = tiles * p.split_k;
  const int per_xcd = (total + 7) / 8;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / WGN, wn = wv % WGN;
  DlFrag<TA, MT, MI16> ra;
  DlFrag<TB, NT, MI16> rb;
  ra.init(wm * WM, 0);
  rb.init(wn * WN, NSTAGE * TILE);
  typedef __attribute__((address_space(3))) unsigned char lds_byte;
  const unsigned lds0 = (unsigned)(__UINTPTR_TYPE__)(lds_byte*)smem_raw + wv * SLICE;  // this wave's slice of a stage

  // Persistent work-groups: the grid has at most one work-group per CU; work-group (xcd, slot) walks that XCD's
  // tile range with stride slots-per-XCD, the order a one-tile-per-work-group grid would be dispatched in.
  typename std::conditional<PIX, DlPixelOperand<NW>, DlOperand<TA, false, NW, MI16>>::type la;
  DlOperand<TB, DUAL, NW, MI16> lb;
  int T_ = 0, k_tail = 0;  // of the tile whose operands are being loaded
  [[maybe_unused]] int px_pending = -1;  // PIX: stage whose A bytes are in registers, requested by the previous issue()
  [[maybe_unused]] const PxNorm px_norm(p);
  const bool px_late = PIX && wv >= NW / 2;
  auto issue = [&](int t, int s) {  // K tile t into stage s (both wave-uniform)
    if constexpr (PIX) {
      // the A bytes requested one call ago are converted and written now (their K tile is read two barriers from here),
      // then K tile t is requested: B straight into LDS, A into registers
      if (px_pending >= 0) la.flush(smem_raw + px_pending * TILE + wv * SLICE, px_norm);
      px_pending = -1;
      if (t >= T_) return;
      lb.issue(lds0 + (NSTAGE + s) * TILE);
      la.request();
      px_pending = s;
    } else {
      if (t >= T_) return;
      if (k_tail != 0 && t == T_ - 1) {
        la.issue_tail(smem_raw + s * TILE + wv * SLICE, k_tail, wv);
        lb.issue_tail(smem_raw + (NSTAGE + s) * TILE + wv * SLICE, k_tail, wv);
      } else {
        la.issue(lds0 + s * TILE);
        lb.issue(lds0 + (NSTAGE + s) * TILE);
      }
    }
  };
  constexpr int N_PER_BLOCK = DUAL ? BN / 2 : BN;
  int next_slice = 0;
  int64_t next_m0 = 0, next_n0 = 0;
  // decodes work item `idx` of this work-group's XCD and starts its first loads; false past the end
  auto start_tile = [&](int idx) -> bool {
    if (idx >= per_xcd) return false;
    const int work = (blockIdx.x & 7) * per_xcd + idx;
    if (work >= total) return false;
    next_slice = work / tiles;
    int tm, tn;
    tile_coords(p, work % tiles, tm, tn);
    const int64_t k_begin = (int64_t)next_slice * p.k_chunk;
    const int64_t k_end = p.split_k > 1 ? (k_begin + p.k_chunk < p.K ? k_begin + p.k_chunk : p.K) : p.K;
    next_m0 = (int64_t)tm * BM;
    next_n0 = (int64_t)tn * N_PER_BLOCK;
    if constexpr (PIX) la.init(p, next_m0, wv);
    else la.init(static_cast<const T*>(p.A), nullptr, p.lda, next_m0, p.M, k_begin, wv);
    lb.init(static_cast<const T*>(p.B), static_cast<const T*>(p.B2), p.ldb, next_n0, p.N, k_begin, wv);
    const int klen = (int)(k_end - k_begin);
    T_ = (klen + DL_BK - 1) / DL_BK;
    k_tail = klen % DL_BK;
#pragma unroll
    for (int t = 0; t < NSTAGE - 1; ++t) issue(t, t);
    return true;
  };
  int idx = blockIdx.x >> 3;
  while (start_tile(idx)) {
  const int slice = next_slice;
  const int64_t m0 = next_m0, n0 = next_n0;

  f32x16 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;

  EpiPre<T, EPI, BM, BN, WM, D::NTHREADS> ep;
  ep.init(p, m0, n0);

  [[maybe_unused]] bf16x8 fa[2][MT], fb[2][NT];
  for (int t0 = 0; t0 < T_; t0 += NSTAGE) {
#pragma unroll
    for (int s = 0; s < NSTAGE; ++s) {
      const int t = t0 + s;
      if (t >= T_) break;
      // tile t has landed once only the tiles issued after it are pending
      const int rem = T_ - 1 - t;
      constexpr int AHEAD = NSTAGE - 2;
      wait_tiles<2 * D::CPT>(rem < 0 ? 0 : (rem < AHEAD ? rem : AHEAD));
      __builtin_amdgcn_s_barrier();  // every wave's share of that tile is in LDS; stage (s-1) has been consumed
      // PIX: the conversion of the A bytes is vector work of about the length of a K tile's MFMAs.  The two waves of a
      // SIMD (w and w + NW/2) do it at opposite ends of the step, one before its MFMAs and one after, so that one
      // wave's conversions run under the other's MFMAs.
      if (!px_late) issue(t + NSTAGE - 1, (s + NSTAGE - 1) % NSTAGE);

      if constexpr (MI16) {
        // one 32-wide step per stage on v_mfma_f32_16x16x32_bf16: 2*MT x 2*NT blocks of 16x16
        bf16x8 ga[2 * MT], gb[2 * NT];
#pragma unroll
        for (int a = 0; a < 2 * MT; ++a) ga[a] = ra.read16(smem_raw, a, s);
#pragma unroll
        for (int b = 0; b < 2 * NT; ++b) gb[b] = rb.read16(smem_raw, b, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < 2 * MT; ++a)
#pragma unroll
          for (int b = 0; b < 2 * NT; ++b) {
            f32x16& blk = acc[a >> 1][b >> 1];
            const int q = (a & 1) * 2 + (b & 1);
            f32x4 c = {blk[4 * q], blk[4 * q + 1], blk[4 * q + 2], blk[4 * q + 3]};
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga[a], gb[b], c, 0, 0, 0);
            blk[4 * q] = c[0];
            blk[4 * q + 1] = c[1];
            blk[4 * q + 2] = c[2];
            blk[4 * q + 3] = c[3];
          }
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
      for (int a = 0; a < MT; ++a) fa[0][a] = ra.read(smem_raw, a, 0, s);
#pragma unroll
      for (int b = 0; b < NT; ++b) fb[0][b] = rb.read(smem_raw, b, 0, s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < MT; ++a) fa[1][a] = ra.read(smem_raw, a, 1, s);
#pragma unroll
      for (int b = 0; b < NT; ++b) fb[1][b] = rb.read(smem_raw, b, 1, s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0][a], fb[0][b], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1][a], fb[1][b], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (PIX) {
        if (px_late) {
          issue(t + NSTAGE - 1, (s + NSTAGE - 1) % NSTAGE);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // no LDS read follows the write before the barrier
        }
      }
    }
  }
  __syncthreads();  // operands fully consumed before the epilogue overwrites them
  idx += gridDim.x >> 3;
  run_epilogue<T, TO, EPI, BM, BN, WM, WN, D::NTHREADS, MI16>(p, acc, smem_raw, m0, n0, wm, wn, slice, ep);
  __syncthreads();  // the staging area is free again before operands land in it
  }
}

// C[m, n] = epilogue(sum over slices of the fp32 partial tiles) (fixed order, so the result is reproducible); the
// epilogue is none, + bias[n] or + bias[n] + R[m, n], in the order of the one-pass kernels' epilogue.
// VEC: four consecutive columns per thread (N, the pitches and the pointers allow vector accesses).  The partial tiles are not read again.
template <typename T, typename TO, bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int split_k, int64_t M, int64_t N,
                                                            TO* __restrict__ C, int64_t ldc, int epi, const T* __restrict__ bias,
                                                            const T* __restrict__ R, int64_t ldr, const float* __restrict__ row_ws,
                                                            TO* __restrict__ row_sums) {
  const int64_t total = M * N;
  if (row_ws != nullptr)
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < M; i += (int64_t)gridDim.x * 256) {
      float s = 0.f;
      for (int k = 0; k < split_k; ++k) s += row_ws[(int64_t)k * M + i];
      row_sums[i] = from_f32<TO>(s);
    }
  if constexpr (VEC) {
    const int64_t quads = total / 4, nq = N / 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < quads; i += (int64_t)gridDim.x * 256) {
      f32x4 s = {0.f, 0.f, 0.f, 0.f};  // the same sum, from the same zero, as the scalar form
      for (int k = 0; k < split_k; ++k) {
        const f32x4 v = load_once(reinterpret_cast<const f32x4*>(ws + (int64_t)k * total + 4 * i));
        s = f32x4{s[0] + v[0], s[1] + v[1], s[2] + v[2], s[3] + v[3]};
      }
      const int64_t m = i / nq, n = (i % nq) * 4;
      if (epi != MVIT_EPI_NONE) {
        const auto b = *reinterpret_cast<const T __attribute__((ext_vector_type(4)))*>(bias + n);
        s = f32x4{s[0] + to_f32(b[0]), s[1] + to_f32(b[1]), s[2] + to_f32(b[2]), s[3] + to_f32(b[3])};
      }
      if (epi == MVIT_EPI_BIAS_RES) {
        const auto r = *reinterpret_cast<const T __attribute__((ext_vector_type(4)))*>(R + m * ldr + n);
        s = f32x4{s[0] + to_f32(r[0]), s[1] + to_f32(r[1]), s[2] + to_f32(r[2]), s[3] + to_f32(r[3])};
      }
      TO* c = C + m * ldc + n;
      if constexpr (sizeof(TO) == 2) *reinterpret_cast<bf16x4*>(c) = bf16x4{(bf16_t)s[0], (bf16_t)s[1], (bf16_t)s[2], (bf16_t)s[3]};
      else *reinterpret_cast<f32x4*>(c) = s;
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
      float s = 0.f;
      for (int k = 0; k < split_k; ++k) s += ws[(int64_t)k * total + i];
      const int64_t m = i / N, n = i % N;
      if (epi != MVIT_EPI_NONE) s += to_f32(bias[n]);
      if (epi == MVIT_EPI_BIAS_RES) s += to_f32(R[m * ldr + n]);
      C[m * ldc + n] = from_f32<TO>(s);
    }
  }
}
template <typename T, typename TO>
void launch_splitk_reduce(const GemmParams& p, hipStream_t stream) {
  const int64_t elems = p.M * p.N;
  const int epi = p.reduce_epi;
  const T* bias = static_cast<const T*>(p.bias);
  const T* R = static_cast<const T*>(p.R);
  bool vec = p.N % 4 == 0 && p.ldc % 4 == 0 && mvit_aligned16(p.workspace) && (reinterpret_cast<uintptr_t>(p.C) % (4 * sizeof(TO))) == 0;
  if (epi != MVIT_EPI_NONE) vec = vec && reinterpret_cast<uintptr_t>(bias) % (4 * sizeof(T)) == 0;
  if (epi == MVIT_EPI_BIAS_RES) vec = vec && p.ldr % 4 == 0 && reinterpret_cast<uintptr_t>(R) % (4 * sizeof(T)) == 0;
  const int64_t items = vec ? elems / 4 : elems;
  const int rgrid = (int)((items + 255) / 256 < 8192 ? (items + 255) / 256 : 8192);
  if (vec) hipLaunchKernelGGL((splitk_reduce_kernel<T, TO, true>), rgrid, 256, 0, stream, p.workspace, p.split_k, p.M, p.N, static_cast<TO*>(p.C), p.ldc, epi, bias, R, p.ldr, p.row_ws, static_cast<TO*>(p.row_sums));
  else hipLaunchKernelGGL((splitk_reduce_kernel<T, TO, false>), rgrid, 256, 0, stream, p.workspace, p.split_k, p.M, p.N, static_cast<TO*>(p.C), p.ldc, epi, bias, R, p.ldr, p.row_ws, static_cast<TO*>(p.row_sums));
}

template <typename T, typename TO, bool TA, bool TB, int EPI, int VAR>
int launch(const GemmParams& p, hipStream_t stream) {
  using W = Waves<VAR>;
  constexpr int BM = W::BM, BN = W::BN;
  using LA = TileLoader<T, BM, TA, W::NTHREADS, W::WN, false>;
  using LB = TileLoader<T, BN, TB, W::NTHREADS, W::WN, false>;
  const size_t operands = 2 * (size_t)(LA::LDS_ELEMS + LB::LDS_ELEMS) * sizeof(T);
  const size_t staging = (size_t)(BM / W::WM) * 32 * (BN + 8) * sizeof(float);
  const size_t lds = operands > staging ? operands : staging;
  auto kern = gemm_kernel<T, TO, TA, TB, EPI, VAR>;
  static bool attr_set_on[MVIT_MAX_DEVICES] = {};  // dynamic LDS above 64 KiB needs opting in once per kernel and device
  const int dev = mvit_current_device("gemm");
  if (dev < 0) return MVIT_ERR_LAUNCH;
  bool& attr_set = attr_set_on[dev];
  if (!attr_set && lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return mvit_set_error(MVIT_ERR_LAUNCH, "gemm: hipFuncSetAttribute(%zu B LDS): %s", lds, hipGetErrorString(e));
    attr_set = true;
  }
  if (p.split_k > 1 && EPI != MVIT_EPI_NONE) return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: split_k needs EPI_NONE");
  const int total = p.tiles_m * p.tiles_n * p.split_k;
  const int grid = ((total + 7) / 8) * 8;
  hipLaunchKernelGGL(kern, grid, W::NTHREADS, lds, stream, p);
  MVIT_CHECK_LAUNCH("gemm");
  if (p.split_k > 1) {
    launch_splitk_reduce<T, TO>(p, stream);
    MVIT_CHECK_LAUNCH("gemm split-k reduce");
  }
  return MVIT_OK;
}

// Column sums of C per `rows` rows, columns [0, N) and [aux_off, aux_off + N): what the bf16 SwiGLU-backward epilogue hands back
// from its tiles, for the fp32 product.
__global__ __launch_bounds__(256) void tile_colsum_kernel(const float* __restrict__ C, int64_t ldc, int64_t M, int64_t N, int64_t aux_off, int rows, float* __restrict__ out) {
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x, m0 = (int64_t)blockIdx.y * rows, m1 = m0 + rows < M ? m0 + rows : M;
  if (n >= N) return;
  const int64_t col = n + blockIdx.z * aux_off;
  float s = 0.f;
  for (int64_t m = m0; m < m1; ++m) s += C[m * ldc + col];
  out[blockIdx.y * ldc + col] = s;
}

// Compute units of the device (rounded down to a multiple of the 8 XCDs): persistent GEMM work-groups run one per unit.
int device_cu_count(int dev) {
  static int n_cu_on[MVIT_MAX_DEVICES] = {};
  int& n_cu = n_cu_on[dev];
  if (n_cu == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    n_cu = v / 8 * 8 > 0 ? v / 8 * 8 : 8;
  }
  return n_cu;
}

template <typename TO, bool TA, bool TB, int EPI, int NSTAGE, int NW, bool MI16 = false, bool PIX = false>
int launch_dl(const GemmParams& p, hipStream_t stream) {
  using D = DL<NW>;
  constexpr size_t operands = 2 * (size_t)NSTAGE * D::TILE_BYTES;
  constexpr size_t staging = (size_t)(D::BM / D::WM) * 32 * D::BN * sizeof(float);
  constexpr size_t lds = staging > operands ? staging : operands;
  static_assert(lds <= 160 * 1024, "operand stages plus the epilogue staging area exceed the LDS of a CU");
  auto kern = gemm_dl_kernel<TO, TA, TB, EPI, NSTAGE, NW, MI16, PIX>;
  static bool attr_set_on[MVIT_MAX_DEVICES] = {};  // once per kernel and device
  const int dev = mvit_current_device("gemm");
  if (dev < 0) return MVIT_ERR_LAUNCH;
  bool& attr_set = attr_set_on[dev];
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return mvit_set_error(MVIT_ERR_LAUNCH, "gemm: hipFuncSetAttribute(%zu B LDS): %s", lds, hipGetErrorString(e));
    attr_set = true;
  }
  if (p.split_k > 1 && EPI != MVIT_EPI_NONE) return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: split_k needs EPI_NONE");
  const int total = p.tiles_m * p.tiles_n * p.split_k;
  const int n_cu = device_cu_count(dev);
  const int want = ((total + 7) / 8) * 8;
  const int grid = want < n_cu ? want : n_cu;
  hipLaunchKernelGGL(kern, grid, D::NTHREADS, lds, stream, p);
  MVIT_CHECK_LAUNCH("gemm");
  if (p.split_k > 1) {
    launch_splitk_reduce<bf16_t, TO>(p, stream);
    MVIT_CHECK_LAUNCH("gemm split-k reduce");
  }
  return MVIT_OK;
}

template <typename T, typename TO, bool TA, bool TB, int EPI>
int launch_var(int var, const GemmParams& p, hipStream_t s) {
  // always served by the tiles that choose_tile() picks from, unless a row pitch exceeds 32-bit lane offsets
  constexpr bool TILED = sizeof(TO) == 2 ? (EPI == MVIT_EPI_NONE || EPI == MVIT_EPI_GELU_BWD) : (TA && TB && EPI == MVIT_EPI_NONE);
  if constexpr (!TILED) {
    // direct-to-LDS main loop: v_mfma_f32_16x16x32_bf16 for the plain GEMMs with an operand behind the transposing
    // LDS read (input gradients +1 % on real data), v_mfma_f32_32x32x16_bf16 for the forward GEMMs (both operands
    // row-major: 3-5 % faster that way).  SwiGLU backward takes the form of the smaller tiles that serve few rows
    // (gemm_small.hip): a row's gradient has the same bits whatever batch it lies in
    constexpr bool MI16 = TB && (EPI == MVIT_EPI_NONE || EPI == MVIT_EPI_SWIGLU_BWD);
    if (var == 3) return launch_dl<TO, TA, TB, EPI, 4, 8, MI16>(p, s);
  } else if (var == 3) {
    return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: epilogue %d of trans_a=%d trans_b=%d is served by tiles", EPI, (int)TA, (int)TB);
  }
  return launch<T, TO, TA, TB, EPI, 1>(p, s);  // register-staged main loop: operands whose row pitch exceeds 32-bit lane offsets
}

template <typename T, typename TO, bool TA, bool TB>
int dispatch_epi(int epi, int var, const GemmParams& p, hipStream_t s) {
  switch (epi) {
    case MVIT_EPI_NONE: return launch_var<T, TO, TA, TB, MVIT_EPI_NONE>(var, p, s);
    case MVIT_EPI_BIAS: return launch_var<T, TO, TA, TB, MVIT_EPI_BIAS>(var, p, s);
    case MVIT_EPI_ACCUM: return launch_var<T, TO, TA, TB, MVIT_EPI_ACCUM>(var, p, s);
    default: break;
  }
  if constexpr (!TA && !TB) {
    // forward-only epilogues (both operands contraction-contiguous)
    switch (epi) {
      case MVIT_EPI_BIAS_RES: return launch_var<T, TO, false, false, MVIT_EPI_BIAS_RES>(var, p, s);
      case MVIT_EPI_BIAS_GELU: return launch_var<T, TO, false, false, MVIT_EPI_BIAS_GELU>(var, p, s);
      case MVIT_EPI_SWIGLU: return launch_var<T, TO, false, false, MVIT_EPI_SWIGLU>(var, p, s);
      default: break;
    }
  }
  if constexpr (!TA && TB) {
    // data-gradient epilogues
    switch (epi) {
      case MVIT_EPI_SWIGLU_BWD: return launch_var<T, TO, false, true, MVIT_EPI_SWIGLU_BWD>(var, p, s);
      case MVIT_EPI_GELU_BWD: return launch_var<T, TO, false, true, MVIT_EPI_GELU_BWD>(var, p, s);
      default: break;
    }
  }
  return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: epilogue %d not built for trans_a=%d trans_b=%d", epi, (int)TA, (int)TB);
}

template <typename T, typename TO>
int dispatch_trans(int ta, int tb, int epi, int var, const GemmParams& p, hipStream_t s) {
  if (!ta && !tb) return dispatch_epi<T, TO, false, false>(epi, var, p, s);
  if (!ta && tb) return dispatch_epi<T, TO, false, true>(epi, var, p, s);
  if (ta && tb) return dispatch_epi<T, TO, true, true>(epi, var, p, s);
  return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: trans_a=1, trans_b=0 is not built");
}

inline bool vec16(const void* ptr, int64_t ld, size_t esize) {
  return ptr == nullptr || (mvit_aligned16(ptr) && (ld * (int64_t)esize) % 16 == 0);
}

// ---- which bf16 kernel and tile
GemmTiledKind tiled_kind(int dtype, int out_dtype, int ta, int tb, int epi, const GemmParams& p) {
  if (dtype != MVIT_BF16) return TILED_NONE;
  if (out_dtype != MVIT_BF16) return ta && tb && epi == MVIT_EPI_NONE ? TT_NONE_F32 : TILED_NONE;
  const bool even = p.N % 2 == 0 && (reinterpret_cast<uintptr_t>(p.bias) | reinterpret_cast<uintptr_t>(p.bias2)) % 4 == 0;  // biases travel in pairs
  if (!ta && !tb) {
    switch (epi) {
      case MVIT_EPI_NONE: return NN_NONE;
      case MVIT_EPI_BIAS: return p.bias && even ? NN_BIAS : TILED_NONE;
      case MVIT_EPI_BIAS_RES: return p.bias && even ? NN_BIAS_RES : TILED_NONE;
      case MVIT_EPI_BIAS_GELU: return p.bias && even ? NN_BIAS_GELU : TILED_NONE;
      case MVIT_EPI_SWIGLU: return p.bias && p.bias2 && even ? NN_SWIGLU : TILED_NONE;
      default: return TILED_NONE;
    }
  }
  if (!ta && tb) return epi == MVIT_EPI_NONE ? NT_NONE : (epi == MVIT_EPI_GELU_BWD ? NT_GELU_BWD : (epi == MVIT_EPI_SWIGLU_BWD ? NT_SWIGLU_BWD : TILED_NONE));
  return ta && tb && epi == MVIT_EPI_NONE ? TT_NONE : TILED_NONE;
}

bool pp_takes(GemmTiledKind kind, int64_t k_chunk, int64_t k_last) {  // at least three K tiles of 64 in every slice
  return k_chunk > 128 && k_last > 128;
}

// Modelled times (us) of the tiles on one MI355X, fitted to every tile's time at 256 ... 16,384 rows of the tower's products: a
// step of 64 along K takes 1.15 us in a 256 x 256 tile (one work-group per compute unit; 1.2 with both operands behind the
// transposing LDS read; 2,392 cycles, so more when the clock falls under a long load, which lengthens every tile's steps alike), and in the smaller ones `one` us while every unit has at most one work-group and `two` us once it has
// two.  Tiles of one work-group per unit (`lone`) interleave loads, LDS reads and MFMAs, so their steps are shorter than those of a
// single work-group of the kind that shares its unit, and shorter again (`one_ahead`) where a wave reads B ahead of the main loops (gemm_reads_ahead).
// For 1280 columns that gives 32 x 64 up to 384 rows, 64 x 64 up to 768, 64 x 128 up to 1,600, 128 x 128 up to 3,200 and 192 x 128 from 3,265 to 4,800, one work-group
// per unit each.  us, input gradients of 1280 columns, weights from HBM, K = 6912, 3840, 3456, 1280: 384 rows, 32 x 64 / 64 x 64 25.0, 15.1, 13.9, 7.7 / 31.0, 19.1, 17.4, 8.9; 512,
// 32 x 64 in two rounds / 64 x 64 37.1, 21.9, 20.0, 9.7 / 29.1, 17.6, 15.9, 8.7; 784, 32 x 64 in two rounds / 64 x 128 44.4, 26.0, 23.4, 10.9 / 36.5, 23.1, 20.4, 10.6; 1,024, two 64 x 64
// to a unit / 64 x 128 43.7, 26.0, 23.6, 11.0 / 37.2, 22.5, 20.6, 10.8; 1,600 57.0, 33.3, 30.2, 13.5 / 38.6, 24.0, 22.1, 11.1.  Beside another stream nothing is read ahead (1,024 rows on
// 64 x 128 45.6, 27.2, 24.7, 11.7), but the same tiles are taken: two 64 x 64 to a unit compete with the other stream for the L2s.  ms per step, 8 blocks of 2560 columns,
// two 64 x 64 / 64 x 128: 440 rows 4.99 - 5.07 / 4.86 - 5.01, 576 5.42 - 5.49 / 5.12 - 5.27.
// (input gradient of 6912 x 1280, us, shared / 128 lone / 192 lone: 2,048 rows 70 / 48 / 61, 3,136 73 / 55 / 65, 4,096 78 / 95 / 68,
// 6,084 91 / 104 / 127; ms per step before -> with them: 3,136 rows 21.0 -> 19.9, 4,096 checkpointed 29.2 -> 28.0).  A fuller last round, a shorter step and more units at work all lower the estimate; the epilogue of a 256 x 256 tile is
// the longest.  The line between the tiles follows from these numbers and not from any shape: e.g. weight gradients of
// 3840 x 1280 over 4,096 rows take 49 us in one slice on 128 x 128 and 57 in three on 256 x 256, over 8,192 rows 93 and 87.
//
// What a launch costs is its time alone only where nothing runs beside it.  In a block's backward the input gradients and the weight
// gradients run on two streams, and the units that one launch's last round leaves idle work for the other: there (`overlapped`, which
// the caller says) the estimate is a mean of the time alone (weight `alone`) and of the units' time divided by the number of units,
// which favours the tile that wastes least over the one that ends its rounds best.  That holds where there is work for idle units, i.e. not for input
// gradients of so few rows that 256 x 256 tiles would give less than half of the units work.  ms per 32-block step, tiles by time
// alone -> by this mean: 14,336 rows 69.0 -> 66.7, 16,384 (checkpointed, optimizer included) 102.6 -> 100.4, 9,600 50.0 -> 49.0 (that
// one by the weight gradients' tiles), 4,096, 6,084 and 20,000 unchanged; with the mean at few rows too 1,760 rows 15.6 -> 16.2.
// An input gradient that has the GPU to itself takes the tile that is done first.  There the small tiles' steps grow with the length
// of the launch (clock, and operands that the L2s and the memory-side cache no longer hold): a launch of r rounds takes 5 % longer per round beyond the
// first on 128 x 128 tiles, 15 % on 64-row ones.  us, input gradients of 1280 columns, the mean above -> this: K = 6912 13,312 rows 268 -> 215,
// 14,336 267 -> 223, 16,384 282 -> 294 (4 % off the best), 18,432 and 27,648 284 and 432 (328 and 540 without the growth); K = 3840 13,312 rows
// 155 -> 129, 16,384 160 -> 148; 5120 columns, K = 5120 (the merger) 3,584 rows 202 -> 171.  (One launch each; rows_in_full_rounds then cuts some in two.)  Over 107 sizes from 1,024 to 65,536 rows the
// choice is 0.1 % off the fastest tile on average.
constexpr double PP_STEP_US = 1.15, PP_TILE_US = 7., PP_SWIGLU_TILE_US = 11.;
struct TileChoice {
  int bm, bn;
  double us;
  bool lone = false;  // the tile's kernel of one work-group per compute unit
};
// The 256-row SwiGLU-backward kernel: gemm_pp_kernel, or gemm_dl_kernel (bm = 0) for a contraction of fewer than three K tiles
TileChoice full_rows_tile(GemmTiledKind kind, int64_t k_chunk, int64_t k_last) {
  return pp_takes(kind, k_chunk, k_last) ? TileChoice{256, 256, 0.} : TileChoice{0, 0, 0.};
}
// The small tiles of weight gradients, two work-groups to a unit
struct TileTimes {
  int bm, bn;
  double one, two, per_tile;
};
constexpr TileTimes WGRAD_TILES[] = {{64, 64, 0.23, 0.36, 2.}, {64, 128, 0.37, 0.52, 2.}, {128, 128, 0.60, 0.72, 2.5}};
// `full_rows`: whether that kernel may be chosen
TileChoice choose_tile(GemmTiledKind kind, int64_t M, int64_t N, int64_t k_chunk, int64_t k_last, int64_t slices, int n_cu, bool overlapped, bool full_rows = true) {
  const bool tt = kind == TT_NONE || kind == TT_NONE_F32;
  const double steps = (double)((k_chunk + 63) / 64);
  const int64_t n_mul = kind == NN_SWIGLU ? 2 : 1;
  const bool input_grad = kind == NT_NONE || kind == NT_GELU_BWD, fills = 2 * ((M + 255) / 256) * ((N + 255) / 256) >= n_cu;
  const double alone = !overlapped ? 1. : tt ? 0.5 : (input_grad && fills ? 0.3 : 1.);
  TileChoice best{0, 0, 1e30};
  auto consider = [&](int bm, int bn, double one, double two, double per_tile, bool lone = false, double one_ahead = 0.) {
    const int64_t tiles_m = (M + bm - 1) / bm, items = tiles_m * ((N * n_mul + bn - 1) / bn) * slices;
    if (one_ahead > 0. && gemm_reads_ahead(kind, bm, tiles_m, items, slices, n_cu)) one = one_ahead;
    const int64_t slots = two > 0. ? 2 * (int64_t)n_cu : n_cu, full = items / slots, rest = items % slots;
    const double round = steps * (two > 0. ? two : one) + per_tile;
    double us = full * round;
    // nearly all units with two (SwiGLU backward, 64 x 64 / 64 x 128: 528 rows 16.2 / 16.4 us, 576 16.9 / 16.5); not weight gradients: 512 x 640 over 8,192 rows so in 12 slices of 64 x 128 24.3, without 6 of 64 x 64 20.3
    if (!tt && bm * bn == 64 * 64 && full == 0 && 4 * rest > 7 * n_cu) two *= 1.15;
    if (rest > 0) us += steps * (two > 0. && rest > n_cu ? two : one) + per_tile;
    if (input_grad && !overlapped && two > 0. && items > slots) us *= 1. + (bm == 128 ? 0.05 : 0.15) * (double)((items - 1) / slots);
    us = 4. + alone * us + (1. - alone) * round * (double)items / (double)slots;
    if (us < best.us) best = TileChoice{bm, bn, us, lone};
  };
  const bool swiglu = kind == NN_SWIGLU;
  if (pp_takes(kind, k_chunk, k_last) && kind != NT_SWIGLU_BWD) consider(256, 256, tt ? 1.2 : PP_STEP_US, 0., swiglu ? PP_SWIGLU_TILE_US : PP_TILE_US);
  if (kind == NT_SWIGLU_BWD) {  // two inputs, two outputs and the column sums lengthen its epilogue
    consider(64, 64, 0.28, 0., 2., true);
    consider(64, 64, 0.30, 0.43, 2.);
    consider(64, 128, 0.47, 0.70, 2.);
    consider(128, 128, 0.55, 0.90, 5.);
  } else if (tt) {
    for (const TileTimes& t : WGRAD_TILES) consider(t.bm, t.bn, t.one, t.two, t.per_tile);
  } else {
    if (!swiglu) consider(64, 64, 0.19, 0.36, 2.);
    consider(64, 128, 0.37, 0.52, 2.);
    consider(128, 128, 0.60, 0.72, swiglu ? 6. : 2.5);
    consider(128, 128, swiglu ? 0.45 : 0.44, 0., swiglu ? 2.5 : 3., true, 0.40);
    if (!swiglu) {
      consider(32, 64, 0.15, 0., 1.2, true, 0.13);
      consider(64, 64, 0.18, 0., 2., true, 0.155);
      consider(64, 128, 0.365, 0., 2., true, 0.30);
      consider(192, 128, 0.60, 0., 4., true);
    }
  }
  // SwiGLU backward: the 256-row kernel as soon as its tiles give half of the units work.  Its launch shares the GPU with
  // the down projection's weight gradient on the second stream, which fills the units it leaves idle, while two small tiles per
  // unit compete with it for the L2s.  ms per 32-block step, 64 x 64 / 64 x 128 / 128 x 128 / 256 x 256: 576 rows 9.56 / 9.53 / 9.87 / 10.48,
  // 1,600 14.8 / 14.6 / 14.4 / 14.8, 2,048 16.4 / 16.2 / 15.8 / 16.2, 2,304 18.0 / 17.8 / 18.0 / 17.5, 3,136 21.9 / 21.7 / 22.0 / 21.8,
  // 4,900 31.8 / 31.4 / 31.0 / 30.6, 6,084 37.2 / 36.7 / 36.2 / 35.8 (alone 128 x 128 is ahead up to 20,000 rows, 165 us against 185 at 14,336)
  // The line stays at one half, although 256 x 256 is ahead at 2,304 rows, just below it: the tile decides how many rows a partial
  // column sum has, so moving the line changes the rounding of the gate / up bias gradients.
  if (kind == NT_SWIGLU_BWD && full_rows && 2 * ((M + 255) / 256) * ((N + 255) / 256) >= n_cu) best = full_rows_tile(kind, k_chunk, k_last);
  return best;
}

// Rows of a forward product, or of an input gradient that has the units to itself, that fill whole rounds of 256 x 256 tiles, when the rest is better taken by a second launch of the
// tiles that suit it (0: one launch for all).  14,336 rows are 56 x 5 tiles of 1280 columns, 1.09 rounds of 256 units: a second
// round for 24 tiles, or 2.2 rounds of 128 x 128 tiles at two thirds of the rate.  255 tiles in one round and 1,280 rows on small
// tiles are faster than either (forward products of the tower, time alone of the step: 14,336 rows 71.6 -> 69.6 ms, 9,600 51.7 ->
// 50.2, 4,360 without gradients 8.92 -> 8.61).  Input gradients, us in one launch / head and rest: 14,336 x 1280, K = 6912 211 / 200, K = 3840
// 126 / 115; 16,384 x 1280, K = 6912, GELU backward 318 / 260; 3,584 x 5120, K = 3584, GELU backward 166 / 144; 4,096 x 5120, K = 5120 187 / 169.  Over 126 drawn sizes that it cuts
// (1,340 to 60,000 rows) 10 % less on average and nowhere more than 0.2 % more; 16,384 x 1280, K = 1280, GELU backward 88 / 89.  In the backward the second stream fills the last round, see choose_tile.
int64_t rows_in_full_rounds(GemmTiledKind kind, int64_t M, int64_t N, int64_t K, int n_cu, bool overlapped) {
  if (!(kind == NN_NONE || kind == NN_BIAS || kind == NN_BIAS_RES || kind == NN_BIAS_GELU || kind == NN_SWIGLU || ((kind == NT_NONE || kind == NT_GELU_BWD) && !overlapped)) || !pp_takes(kind, K, K)) return 0;
  const int64_t tn = (N * (kind == NN_SWIGLU ? 2 : 1) + 255) / 256, rounds = (M + 255) / 256 * tn / n_cu, rows = rounds * n_cu / tn * 256;
  if (rows == 0 || rows >= M) return 0;
  const double head = 4. + (double)rounds * ((double)((K + 63) / 64) * PP_STEP_US + (kind == NN_SWIGLU ? PP_SWIGLU_TILE_US : PP_TILE_US));
  return head + choose_tile(kind, M - rows, N, K, K, 1, n_cu, false).us + 1. < choose_tile(kind, M, N, K, K, 1, n_cu, false).us ? rows : 0;
}

// packed[n][line * 48 + b] = w[n][channel * 392 + frame * 196 + y * 14 + x] for b = x * 3 + channel < 42, else 0
// (line = frame * 14 + y): the patch-embedding weight in the contraction order of DlPixelOperand
template <typename T>
__global__ __launch_bounds__(256) void pack_patch_weight_kernel(const T* __restrict__ w, int64_t ldw, int64_t n_out, bf16_t* __restrict__ packed) {
  const int64_t total = n_out * PX_K;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t n = i / PX_K;
    const int k = (int)(i % PX_K), ln = k / PX_LINE, b = k % PX_LINE;
    float v = 0.f;
    if (b < PX_PATCH * 3) {
      const int x = b / 3, ch = b % 3, fr = ln / PX_PATCH, y = ln % PX_PATCH;
      v = to_f32(w[n * ldw + ch * (2 * PX_PATCH * PX_PATCH) + fr * (PX_PATCH * PX_PATCH) + y * PX_PATCH + x]);
    }
    packed[i] = from_f32<bf16_t>(v);
  }
}

// float -> bf16 bits, round to nearest even (finite inputs)
inline uint16_t host_bf16_bits(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

}  // namespace

extern "C" int mvit_patch_embed_pack_weight(const void* w, int dtype, int64_t ldw, int64_t n_out, void* packed, mvit_stream_t stream) {
  MVIT_REQUIRE(w && packed, "patch_embed_pack_weight: null pointer");
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "patch_embed_pack_weight: dtype %d", dtype);
  MVIT_REQUIRE(n_out > 0 && ldw >= MVIT_PIXEL_ROW, "patch_embed_pack_weight: n_out=%lld ldw=%lld", (long long)n_out, (long long)ldw);
  MVIT_REQUIRE(mvit_aligned16(packed), "patch_embed_pack_weight: packed must be 16-byte aligned");
  const int64_t total = n_out * PX_K;
  const int grid = (int)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == MVIT_BF16) hipLaunchKernelGGL((pack_patch_weight_kernel<bf16_t>), grid, 256, 0, s, static_cast<const bf16_t*>(w), ldw, n_out, static_cast<bf16_t*>(packed));
  else hipLaunchKernelGGL((pack_patch_weight_kernel<float>), grid, 256, 0, s, static_cast<const float*>(w), ldw, n_out, static_cast<bf16_t*>(packed));
  MVIT_CHECK_LAUNCH("patch_embed_pack_weight");
  return MVIT_OK;
}

extern "C" int mvit_patch_embed_frames(const mvit_image* images, int n_images, int64_t total_rows, const void* packed_w, int64_t n_out,
                                       void* out, int64_t ldo, int out_dtype, double rescale, float mean_r, float mean_g, float mean_b,
                                       float std_r, float std_g, float std_b, mvit_stream_t stream) {
  MVIT_REQUIRE(images && packed_w && out, "patch_embed_frames: null pointer");
  MVIT_REQUIRE(n_images > 0 && total_rows >= 0 && n_out > 0 && ldo >= n_out, "patch_embed_frames: n_images=%d total_rows=%lld n_out=%lld ldo=%lld",
               n_images, (long long)total_rows, (long long)n_out, (long long)ldo);
  MVIT_REQUIRE(out_dtype == MVIT_BF16 || out_dtype == MVIT_F32, "patch_embed_frames: out_dtype %d", out_dtype);
  MVIT_REQUIRE(mvit_aligned16(packed_w), "patch_embed_frames: packed_w must be 16-byte aligned");
  if (total_rows == 0) return MVIT_OK;
  GemmParams p;
  memset(&p, 0, sizeof(p));
  // the kernel computes byte * a + c in one fused multiply-add; that is only taken when, rounded to bf16, it gives
  // the table of mvit_patchify ((float)((double)byte * rescale) - mean) / std for all 256 bytes of every channel
  const float mean[3] = {mean_r, mean_g, mean_b}, stdv[3] = {std_r, std_g, std_b};
  for (int c = 0; c < 3; ++c) {
    MVIT_REQUIRE(stdv[c] != 0.f, "patch_embed_frames: std[%d] = 0", c);
    p.px_a[c] = (float)(rescale / (double)stdv[c]);
    p.px_c[c] = (float)(-(double)mean[c] / (double)stdv[c]);
    for (int b = 0; b < 256; ++b) {
      const float x = (float)((double)b * rescale);
      volatile float diff = x - mean[c];
      const float table = diff / stdv[c];
      const float affine = fmaf((float)b, p.px_a[c], p.px_c[c]);
      if (host_bf16_bits(table) != host_bf16_bits(affine))
        return mvit_set_error(MVIT_ERR_UNSUPPORTED, "patch_embed_frames: byte %d of channel %d: a * x + c does not round to the bf16 value of "
                              "(x * rescale - mean) / std for these constants; use mvit_patchify + mvit_gemm", b, c);
    }
  }
  p.M = total_rows; p.N = n_out; p.K = PX_K;
  p.B = packed_w; p.ldb = PX_K; p.C = out; p.ldc = ldo;
  p.px_images = images; p.px_n_images = n_images;
  p.vec_ok = vec16(out, ldo, out_dtype == MVIT_BF16 ? 2 : 4);
  const int64_t tm = (total_rows + 255) / 256, tn = (n_out + 255) / 256;
  MVIT_REQUIRE(tm * tn < (1ll << 30), "patch_embed_frames: too many tiles");
  p.tiles_m = (int)tm; p.tiles_n = (int)tn;
  set_tile_order(p, 256);
  p.split_k = 1; p.k_chunk = PX_K; p.reduce_epi = MVIT_EPI_NONE;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (out_dtype == MVIT_BF16) return launch_dl<bf16_t, false, false, MVIT_EPI_NONE, 4, 8, false, true>(p, s);
  return launch_dl<float, false, false, MVIT_EPI_NONE, 4, 8, false, true>(p, s);
}

extern "C" int mvit_gemm(const mvit_gemm_args* a, mvit_stream_t stream) {
  MVIT_REQUIRE(a, "gemm: null args");
  MVIT_REQUIRE(a->M >= 0 && a->N > 0 && a->K > 0, "gemm: bad shape M=%lld N=%lld K=%lld", (long long)a->M, (long long)a->N, (long long)a->K);
  if (a->M == 0) return MVIT_OK;
  MVIT_REQUIRE(a->A && a->B && a->C, "gemm: null operand");
  const int vec = a->dtype == MVIT_BF16 ? 8 : 4;
  MVIT_REQUIRE(a->dtype == MVIT_BF16 || a->dtype == MVIT_F32, "gemm: dtype %d", a->dtype);
  MVIT_REQUIRE(a->out_dtype == MVIT_BF16 || a->out_dtype == MVIT_F32, "gemm: out_dtype %d", a->out_dtype);
  MVIT_REQUIRE(mvit_aligned16(a->A) && mvit_aligned16(a->B) && (!a->B2 || mvit_aligned16(a->B2)), "gemm: operands must be 16-byte aligned");
  MVIT_REQUIRE(a->lda % vec == 0 && a->ldb % vec == 0, "gemm: lda=%lld ldb=%lld must be multiples of %d", (long long)a->lda, (long long)a->ldb, vec);
  // 16-byte vectors never straddle the edge of the contiguous dimension
  if (!a->trans_a) MVIT_REQUIRE(a->K % vec == 0 && a->lda >= a->K, "gemm: K=%lld must be a multiple of %d (lda=%lld)", (long long)a->K, vec, (long long)a->lda);
  else MVIT_REQUIRE(a->lda >= (a->M + vec - 1) / vec * vec, "gemm: transposed A needs lda=%lld >= M=%lld rounded up to %d", (long long)a->lda, (long long)a->M, vec);
  if (!a->trans_b) MVIT_REQUIRE(a->K % vec == 0 && a->ldb >= a->K, "gemm: K=%lld must be a multiple of %d (ldb=%lld)", (long long)a->K, vec, (long long)a->ldb);
  else MVIT_REQUIRE(a->ldb >= (a->N + vec - 1) / vec * vec, "gemm: transposed B needs ldb=%lld >= N=%lld rounded up to %d", (long long)a->ldb, (long long)a->N, vec);
  int epi = a->epilogue;
  if (epi == MVIT_EPI_BIAS_RES || epi == MVIT_EPI_GELU_BWD || epi == MVIT_EPI_SWIGLU_BWD) MVIT_REQUIRE(a->R, "gemm: epilogue %d needs R", epi);
  if (epi == MVIT_EPI_BIAS_GELU) MVIT_REQUIRE(a->aux, "gemm: epilogue %d needs aux", epi);
  if (epi == MVIT_EPI_SWIGLU) MVIT_REQUIRE(a->B2 && !a->trans_a && !a->trans_b, "gemm: SWIGLU needs B2 and untransposed operands");
  MVIT_REQUIRE(a->ldc >= a->N, "gemm: ldc=%lld < N=%lld", (long long)a->ldc, (long long)a->N);

  GemmParams p;
  p.M = a->M; p.N = a->N; p.K = a->K;
  p.A = a->A; p.lda = a->lda; p.B = a->B; p.B2 = a->B2; p.ldb = a->ldb;
  p.bias = a->bias; p.bias2 = a->bias2; p.C = a->C; p.ldc = a->ldc;
  p.R = a->R; p.ldr = a->ldr; p.aux = a->aux; p.ldaux = a->ldaux; p.aux_off = a->aux_off;
  const size_t es = a->dtype == MVIT_BF16 ? 2 : 4, eo = a->out_dtype == MVIT_BF16 ? 2 : 4;
  p.vec_ok = vec16(a->C, a->ldc, eo) && vec16(a->R, a->ldr, es) && vec16(a->aux, a->ldaux, es) && vec16(a->bias, 0, es) &&
             vec16(a->bias2, 0, es) && (a->aux_off * (int64_t)(es < eo ? es : eo)) % 16 == 0;
  p.half_vec_ok = a->ldc % 4 == 0 && reinterpret_cast<uintptr_t>(a->C) % 8 == 0;
  const int var = (a->lda > (1ll << 22) || a->ldb > (1ll << 22)) ? 1 : 3;  // 3: direct-to-LDS loads (32-bit lane offsets); 1: register-staged
  const int BM = 256, BN = 256;
  const int n_per_block = (epi == MVIT_EPI_SWIGLU) ? BN / 2 : BN;
  const int64_t tm = (a->M + BM - 1) / BM, tn = (a->N + n_per_block - 1) / n_per_block;
  MVIT_REQUIRE(tm * tn < (1ll << 30), "gemm: too many tiles");
  p.tiles_m = (int)tm; p.tiles_n = (int)tn;
  set_tile_order(p, BM);
  p.split_k = 1; p.k_chunk = a->K; p.workspace = nullptr; p.reduce_epi = MVIT_EPI_NONE;
  p.colsum = nullptr;
  const int colsum_rows = a->colsum_rows == 64 ? 64 : 256;
  p.row_sums = a->row_sums; p.row_ws = nullptr;
  if (a->row_sums)
    MVIT_REQUIRE(a->dtype == MVIT_BF16 && a->trans_a && a->trans_b && epi == MVIT_EPI_NONE && var == 3,
                 "gemm: row sums come with a plain bf16 product of two transposed operands");
  if (epi == MVIT_EPI_SWIGLU_BWD && a->workspace) {
    MVIT_REQUIRE(a->colsum_rows == 0 || a->colsum_rows == 256 || a->colsum_rows == 64, "gemm: colsum_rows %d is not 256 or 64", a->colsum_rows);
    const int64_t need = (int64_t)sizeof(float) * ((a->M + colsum_rows - 1) / colsum_rows) * a->ldc;
    MVIT_REQUIRE(mvit_aligned16(a->workspace) && a->workspace_bytes >= need, "gemm: SWIGLU_BWD column sums need a workspace of %lld bytes", (long long)need);
    p.colsum = static_cast<float*>(a->workspace);
  }
  if (a->split_k > 1) {
    const int bk = a->dtype == MVIT_BF16 ? 64 : 16;
    const int64_t chunk = ((a->K + a->split_k - 1) / a->split_k + bk - 1) / bk * bk;
    const int64_t slices = (a->K + chunk - 1) / chunk;  // never an empty slice
    MVIT_REQUIRE(epi == MVIT_EPI_NONE || epi == MVIT_EPI_BIAS || epi == MVIT_EPI_BIAS_RES,
                 "gemm: split_k is available with the plain, bias and bias + residual epilogues (got %d)", epi);
    if (epi != MVIT_EPI_NONE) MVIT_REQUIRE(a->bias, "gemm: split_k with epilogue %d needs bias", epi);
    MVIT_REQUIRE(a->workspace && mvit_aligned16(a->workspace) && a->workspace_bytes >= (int64_t)sizeof(float) * slices * a->M * (a->N + (a->row_sums ? 1 : 0)),
                 "gemm: split_k=%d needs a 16-byte aligned workspace of %lld bytes", a->split_k, (long long)(sizeof(float) * slices * a->M * (a->N + (a->row_sums ? 1 : 0))));
    MVIT_REQUIRE(tm * tn * slices < (1ll << 30), "gemm: too many tiles");
    if (slices > 1) {
      // the main kernel leaves fp32 partial tiles; the reduction over the slices applies the epilogue
      p.split_k = (int)slices; p.k_chunk = chunk; p.workspace = static_cast<float*>(a->workspace);
      p.reduce_epi = epi;
      if (a->row_sums) p.row_ws = p.workspace + slices * a->M * a->N;
      epi = MVIT_EPI_NONE;
    }
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const GemmTiledKind kind = var == 3 ? tiled_kind(a->dtype, a->out_dtype, a->trans_a, a->trans_b, epi, p) : TILED_NONE;
  if (kind != TILED_NONE) {
    const int dev = mvit_current_device("gemm");
    if (dev < 0) return MVIT_ERR_LAUNCH;
    const int n_cu = device_cu_count(dev);
    TileChoice c = choose_tile(kind, p.M, p.N, p.k_chunk, p.K - (p.split_k - 1) * p.k_chunk, p.split_k, n_cu, a->overlapped != 0);
    const bool all_256 = getenv("MVIT_GEMM_NO_HALF_TILES") != nullptr;
    if (all_256 && c.bm != 256 && pp_takes(kind, p.k_chunk, p.K - (p.split_k - 1) * p.k_chunk)) c = TileChoice{256, 256, 0.};
    // the column sums are per tile row: their granularity names the kernels (64 rows: a tile of 64 x 64, 64 x 128 or 128 x 128)
    if (kind == NT_SWIGLU_BWD && p.colsum != nullptr) c = colsum_rows == 64 ? choose_tile(kind, p.M, p.N, p.k_chunk, p.K, 1, n_cu, a->overlapped != 0, false) : full_rows_tile(kind, p.K, p.K);
    if (c.bm != 0) {
      auto run = [&](GemmParams q, const TileChoice& t) -> int {
        q.tiles_m = (int)((q.M + t.bm - 1) / t.bm);
        const int n_cols = kind == NN_SWIGLU ? t.bn / 2 : t.bn;
        q.tiles_n = (int)((q.N + n_cols - 1) / n_cols);
        MVIT_REQUIRE((int64_t)q.tiles_m * q.tiles_n * q.split_k < (1ll << 30), "gemm: too many tiles");
        set_tile_order(q, t.bm);
        return t.bm == 256 ? mvit_gemm_pp(kind, q, n_cu, s) : mvit_gemm_small(kind, t.bm, t.bn, t.lone, q, a->overlapped ? 0 : n_cu, s);
      };
      const int64_t head = all_256 || p.split_k > 1 ? 0 : rows_in_full_rounds(kind, p.M, p.N, p.K, n_cu, a->overlapped != 0);
      if (head > 0) {  // a row's result does not depend on the tile that computes it
        GemmParams q = p;
        q.M = head;
        if (int rc = run(q, TileChoice{256, 256, 0.})) return rc;
        q.M = p.M - head;
        q.A = static_cast<const bf16_t*>(p.A) + head * p.lda;
        q.C = static_cast<bf16_t*>(p.C) + head * p.ldc;
        if (p.R) q.R = static_cast<const bf16_t*>(p.R) + head * p.ldr;
        if (p.aux) q.aux = static_cast<bf16_t*>(p.aux) + head * p.ldaux;
        return run(q, choose_tile(kind, q.M, q.N, q.K, q.K, 1, n_cu, false));
      }
      const int rc = run(p, c);
      if (rc != MVIT_OK) return rc;
      if (p.split_k > 1) {
        if (kind == TT_NONE_F32) launch_splitk_reduce<bf16_t, float>(p, s);
        else launch_splitk_reduce<bf16_t, bf16_t>(p, s);
        MVIT_CHECK_LAUNCH("gemm split-k reduce");
      }
      return MVIT_OK;
    }
  }
  if (a->dtype == MVIT_BF16) {
    MVIT_REQUIRE(p.colsum == nullptr || colsum_rows == 256, "gemm: column sums per 64 rows need bf16 results and row pitches of at most 2^22 elements");
    if (a->out_dtype == MVIT_BF16) return dispatch_trans<bf16_t, bf16_t>(a->trans_a, a->trans_b, epi, var, p, s);
    return dispatch_trans<bf16_t, float>(a->trans_a, a->trans_b, epi, var, p, s);
  }
  MVIT_REQUIRE(a->out_dtype == MVIT_F32, "gemm: fp32 operands need fp32 output");
  const int dev = mvit_current_device("gemm");
  if (dev < 0) return MVIT_ERR_LAUNCH;
  const int rc = mvit_gemm_f32(a->trans_a, a->trans_b, epi, p, device_cu_count(dev), s);
  if (rc != MVIT_OK) return rc;
  if (p.split_k > 1) {
    launch_splitk_reduce<float, float>(p, s);
    MVIT_CHECK_LAUNCH("gemm split-k reduce");
  }
  if (p.colsum != nullptr) {
    hipLaunchKernelGGL(tile_colsum_kernel, dim3((unsigned)((p.N + 255) / 256), (unsigned)((p.M + colsum_rows - 1) / colsum_rows), 2), 256, 0, s,
                       static_cast<const float*>(p.C), p.ldc, p.M, p.N, p.aux_off, colsum_rows, p.colsum);
    MVIT_CHECK_LAUNCH("gemm column sums");
  }
  return MVIT_OK;
}

// Weight gradients of a few rows in one launch of small tiles, instead of a launch each (plain bf16 products of two transposed
// operands; anything else is done one by one).  A row's result does not depend on the tile, so the results are the same.
int mvit_gemm_wgrad_group(const mvit_gemm_args* list, int n, hipStream_t s) {
  bool together = n >= 2 && n <= GEMM_GROUP_MAX;
  for (int i = 0; i < n; ++i) {
    const mvit_gemm_args& a = list[i];
    together = together && a.dtype == MVIT_BF16 && a.out_dtype == MVIT_BF16 && a.trans_a && a.trans_b && a.epilogue == MVIT_EPI_NONE && a.split_k <= 1 &&
               a.M > 0 && a.N > 0 && a.K > 0 && a.A && a.B && a.C && mvit_aligned16(a.A) && mvit_aligned16(a.B) && a.lda % 8 == 0 && a.ldb % 8 == 0 &&
               a.lda >= (a.M + 7) / 8 * 8 && a.ldb >= (a.N + 7) / 8 * 8 && a.ldc >= a.N && a.lda <= (1ll << 22) && a.ldb <= (1ll << 22);
  }
  if (!together) {
    for (int i = 0; i < n; ++i)
      if (int rc = mvit_gemm(&list[i], s)) return rc;
    return MVIT_OK;
  }
  const int dev = mvit_current_device("gemm");
  if (dev < 0) return MVIT_ERR_LAUNCH;
  const int n_cu = device_cu_count(dev);
  // one tile shape for all of them: the model of choose_tile over the sum of their tiles
  int bm = 128, bn = 128;
  double best = 1e30;
  for (const TileTimes& t : WGRAD_TILES) {
    int64_t items = 0, k = 0;
    for (int i = 0; i < n; ++i) {
      items += ((list[i].M + t.bm - 1) / t.bm) * ((list[i].N + t.bn - 1) / t.bn);
      k = list[i].K > k ? list[i].K : k;
    }
    MVIT_REQUIRE(items < (1ll << 30), "gemm: too many tiles");
    const double steps = (double)((k + 63) / 64);
    const int64_t rest = items % (2 * n_cu);
    double us = (double)(items / (2 * n_cu)) * (steps * t.two + t.per_tile);
    if (rest > 0) us += steps * (rest > n_cu ? t.two : t.one) + t.per_tile;
    if (us < best) best = us, bm = t.bm, bn = t.bn;
  }
  GemmGroup g;
  memset(&g, 0, sizeof(g));
  g.n = n;
  for (int i = 0; i < n; ++i) {
    const mvit_gemm_args& a = list[i];
    GemmParams& p = g.p[i];
    p.M = a.M; p.N = a.N; p.K = a.K;
    p.A = a.A; p.lda = a.lda; p.B = a.B; p.ldb = a.ldb; p.C = a.C; p.ldc = a.ldc;
    p.row_sums = a.row_sums;
    p.vec_ok = vec16(a.C, a.ldc, 2);
    p.half_vec_ok = a.ldc % 4 == 0 && reinterpret_cast<uintptr_t>(a.C) % 8 == 0;
    p.split_k = 1; p.k_chunk = a.K; p.reduce_epi = MVIT_EPI_NONE;
    p.tiles_m = (int)((a.M + bm - 1) / bm);
    p.tiles_n = (int)((a.N + bn - 1) / bn);
    set_tile_order(p, bm);
  }
  return mvit_gemm_small_group(bm, bn, g, s);
}

// Slices along the contraction for a product with few output tiles and a long contraction (a weight gradient, contracted
// over the tokens): the count with the lowest modelled time.  Every slice costs an fp32 partial tile written and read back
// (3.5 TB/s) and one more launch sums them.
static int wgrad_split_k(int64_t out_rows, int64_t out_cols, int64_t k, bool overlapped) {
  if (out_rows <= 0 || out_cols <= 0 || k <= 0) return 1;
  int best = 1;
  double best_us = 1e30;
  for (int sk = 1; sk <= 16 && (sk == 1 || k / sk >= 512); ++sk) {
    const int64_t chunk = ((k + sk - 1) / sk + 63) / 64 * 64, slices = (k + chunk - 1) / chunk;
    double us = choose_tile(TT_NONE, out_rows, out_cols, chunk, k - (slices - 1) * chunk, slices, 256, overlapped).us;
    if (slices > 1) us += 5. + (double)slices * (double)out_rows * (double)out_cols * 4. / 3.5e6;
    if (us < best_us) {
      best_us = us;
      best = sk;
    }
  }
  return best;
}

static GemmTiledKind bf16_kind(int trans_a, int trans_b, int epilogue, int64_t N) {
  GemmParams p{};
  p.N = N;
  p.bias = p.bias2 = &p;  // as a product with biases has them
  return tiled_kind(MVIT_BF16, MVIT_BF16, trans_a, trans_b, epilogue, p);
}

extern "C" int64_t mvit_gemm_full_round_rows(int trans_a, int trans_b, int epilogue, int64_t M, int64_t N, int64_t K, int overlapped, int n_cu) {
  const GemmTiledKind kind = bf16_kind(trans_a, trans_b, epilogue, N);
  if (M <= 0 || N <= 0 || K <= 0 || n_cu <= 0 || kind == TILED_NONE) return -1;
  return rows_in_full_rounds(kind, M, N, K, n_cu, overlapped != 0);
}

extern "C" int mvit_gemm_tile(int trans_a, int trans_b, int epilogue, int64_t M, int64_t N, int64_t K, int overlapped, int n_cu, int32_t* tile) {
  MVIT_REQUIRE(tile && M > 0 && N > 0 && K > 0 && n_cu > 0, "gemm_tile: null pointer or bad shape");
  const GemmTiledKind kind = bf16_kind(trans_a, trans_b, epilogue, N);
  if (kind == TILED_NONE) return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm_tile: trans_a=%d trans_b=%d epilogue %d of %lld columns has no choice of tiles", trans_a, trans_b, epilogue, (long long)N);
  const TileChoice c = choose_tile(kind, M, N, K, K, 1, n_cu, overlapped != 0);
  tile[0] = c.bm; tile[1] = c.bn;
  tile[2] = c.bm == 0 || c.bm == 256 || c.lone ? 1 : 2;
  const int64_t tiles_m = c.bm ? (M + c.bm - 1) / c.bm : 0;
  tile[3] = c.bm != 0 && c.bm != 256 && gemm_reads_ahead(kind, c.bm, tiles_m, tiles_m * ((N + c.bn - 1) / c.bn), 1, overlapped ? 0 : n_cu);
  return MVIT_OK;
}

extern "C" int mvit_gemm_wgrad_split_k(int64_t out_rows, int64_t out_cols, int64_t k) { return wgrad_split_k(out_rows, out_cols, k, false); }

extern "C" int mvit_gemm_wgrad_split_k_overlapped(int64_t out_rows, int64_t out_cols, int64_t k) { return wgrad_split_k(out_rows, out_cols, k, true); }

extern "C" int mvit_gemm_swiglu_bwd_colsum_rows(int64_t M, int64_t N, int64_t K) {
  const int bm = choose_tile(NT_SWIGLU_BWD, M, N, K, K, 1, 256, false).bm;
  return bm == 0 || bm == 256 ? 256 : 64;
}
