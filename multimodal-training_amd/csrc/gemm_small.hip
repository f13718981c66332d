// bf16 GEMM for products with too few 256 x 256 tiles to fill the chip: one work-group per BM x BN tile, NW waves of
// WM x WN, K tiles of 64 in a ring of NST LDS stages filled by direct global -> LDS loads up to NST - 1 K tiles ahead.
// A wave reads the next fragments from LDS, and requests its share of a K tile further on, between the MFMAs of the present ones.
// Requesting the whole share at once stalls the wave's MFMAs until the address unit has taken it (16 clocks per KiB: half of the step).
// What bounds a step is the unit's way from L2 into LDS and out of it again: some 64 bytes per clock in, 200 out, one after the other, i.e.
// 0.18 us for a 64 x 64 tile's K tile of 64 whether one work-group has the unit or two share it, 0.27 for 64 x 128, 0.13 for 32 x 64.  So the
// tile that puts each unit to work once wins, and the fewer bytes per product the better.  Weights that come from HBM make a step 1.2 to 1.6 times
// as long, again by its bytes and whatever the ring's depth (a unit's requests in flight).  1280 columns, operands in the caches, us, 64 x 64 (two to
// a unit beyond 256 tiles) / 64 x 128 (one), K = 6912, 3840, 3456 and 1280: 1,024 rows 42.3, 25.0, 21.9, 11.2 / 34.8, 20.1, 18.0, 10.4; 1,600 rows
// 52.4, 27.5, 23.3, 12.0 / 41.7, 21.0, 19.0, 10.8; 64 x 64 / 32 x 64, 256 rows 24.6, 15.6, 13.5, 7.7 / 20.6, 12.9, 10.5, 6.5.  From HBM: choose_tile.
// Two forms of the loop:
// * `WHOLE`: the fragments of a whole K tile are read one K tile ahead, so a step has one barrier and one LDS latency, and the stage that a
//   step has read is free for the K tile a whole ring ahead: the tiles of 64 rows and fewer that have a unit to themselves.  As many stages as cover
//   the latency of L2 and no more, because the first K tile waits for the ring's first requests (64 x 64, us at K = 6912 / 1280: 4 stages 24.1 / 7.3,
//   6 24.6 / 7.8, 9 25.4 / 8.8; by halves and 6 stages 24.6 / 7.7).
// * by halves of a K tile: 128 x 128 and 192 x 128, whose halves have MFMAs enough to cover the LDS latency (whole K tiles: 192 x 128 66 -> 76 us at
//   4,096 rows and K = 6912; 128 x 128 with residual 13.3 -> 14.4 at K = 1280), and 64 x 64 where two share a unit (weights from HBM, 1,024 rows, input
//   gradients, whole K tiles / halves 46.6, 27.6, 11.7 / 43.4, 25.8, 11.3).  One step after the other -> by halves, 2,048 rows on 128 x 128 39.4 -> 28,
//   70 -> 52; MFMAs alone would take 21 and 33.  SwiGLU of 257 to 512 rows on 128 x 128, two work-groups of two stages / one of four: 18.3 / 14.5.
// Two stages of 128 x 128 and three of 64 x 128 (so that two work-groups share a compute unit): one multiplies while the other waits.  The same
// loop serves the weight gradients (A behind the transposing read) with every ring: interleaved they are no faster (1280 x 1280
// over 6,084 rows 44.9 / 44.4 us; ms per step 4,096 rows 29.0 / 29.2, 4,900 30.2 / 30.0, 6,084 35.4 / 35.6).  Their tiles that sum A's rows
// have a loop of their own: a branch in the loop made the others wait too (3840 x 1280 over 6,084 rows 80.7 -> 71.5, over 4,096 58.6 -> 52.7).
// A wave's tile is as square as its registers allow, because LDS reads are the next limit: 128 x 128 split in eight waves of
// 32 x 64 read 96 KiB per K tile, in four of 64 x 64 64 KiB (4,096 rows, two transposed-layout operands, K = 6848: 84 -> 77 us;
// K contiguous in both, K = 3424: 55 -> 52; weight gradient of 3840 x 1280 over 2,048 rows: 32 -> 27).
// Fragment layouts, K order, MFMA form and epilogue arithmetic are those of gemm_pp_kernel (gemm_pingpong.hip), so the results
// are the same bits whichever of the two computed them.
// SwiGLU backward, 128 x 128 (224 registers: two inputs per element beside the accumulators) / 64 x 128 alone, us at 2,048 rows: 27 / 34.
// A work-group computes one tile, so bias, residual and saved activations are fetched into registers before the main loop.
#include "gemm_direct.h"

#include <type_traits>

namespace {

template <int BM_, int BN_, int WGM_, int WGN_, int NST_, bool WHOLE_ = false>
struct SmallCfg {
  static constexpr bool WHOLE = WHOLE_;  // form of the main loop, see above
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, NST = NST_, BK = 64;
  static constexpr int NW = WGM * WGN, NTHREADS = 64 * NW, WM = BM / WGM, WN = BN / WGN;
  static constexpr int A_BYTES = BM * BK * 2, STAGE = (BM + BN) * BK * 2, LDS = NST * STAGE;
  static constexpr int PER_A = BM / 8 / NW, PER_B = BN / 8 / NW, PER = PER_A + PER_B;  // 1 KiB loads per wave and K tile
  static_assert(NST >= 2 && (NST - 1) * PER < 64 && (BM == 32 || BM == 64 || BM == 128 || BM == 192) && (BN == 64 || BN == 128), "ring depths and swizzles built");
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && WM % 16 == 0 && WN % 32 == 0, "whole load instructions and MFMA blocks per wave");
};

template <int PER, int MOST>
__device__ __forceinline__ void wait_tiles(int in_flight) {
  if constexpr (MOST > 0) {
    if (in_flight < MOST) return wait_tiles<PER, MOST - 1>(in_flight);
  }
  pp_wait_vm<MOST * PER>();
}

// chunk (16 bytes) swizzle of a staged operand: [row][k] tiles by row, [k][row] tiles of ROWS rows by k
template <bool TR, bool IS_A, int ROWS>
__device__ __forceinline__ int small_swizzle(int major) {
  if (!TR) return IS_A ? (major >> 1) & 7 : ((major >> 1) & 1) | (((major >> 3) & 3) << 1);
  static_assert(!TR || ROWS == 64 || ROWS == 128, "rows of a [k][row] tile");
  if (ROWS == 64) return (((major >> 1) & 1) << 1) | (((major >> 3) & 1) << 2);
  return ((major & 3) << 1) | (((major >> 3) & 1) << 3);
}

template <typename TO, bool TA, bool TB, int EPI, typename S>
__device__ __forceinline__ void gemm_small_tile(const GemmParams& p, const unsigned block) {
  using T = bf16_t;
  constexpr int BM = S::BM, BN = S::BN, BK = S::BK, NST = S::NST;
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  constexpr bool HAS_IN = EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_GELU_BWD || EPI == MVIT_EPI_SWIGLU_BWD;
  constexpr bool HAS_BIAS = EPI == MVIT_EPI_BIAS || EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_BIAS_GELU || EPI == MVIT_EPI_SWIGLU;
  constexpr int NA = S::WM / 16, NB = S::WN / 16, NGB = NB / 2;  // row blocks, column blocks, groups of 32 columns of a wave
  static_assert(!DUAL || (!TB && NGB == 2), "SWIGLU: a gate group and an up group per wave");
  constexpr int NG = DUAL ? 1 : NGB, NCOLS = DUAL ? BN / 2 : BN, ITEMS = NA * NG;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n), total = tiles * (unsigned)p.split_k, per_xcd = (total + 7) / 8;
  const unsigned work = (block & 7) * per_xcd + (block >> 3);
  if ((block >> 3) >= per_xcd || work >= total) return;
  const unsigned slice = p.split_k > 1 ? work / tiles : 0;
  int tm, tn;
  tile_coords(p, (int)(work - slice * tiles), tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * NCOLS;
  const int64_t k_begin = (int64_t)slice * p.k_chunk;
  const int64_t k_end = p.split_k > 1 ? (k_begin + p.k_chunk < p.K ? k_begin + p.k_chunk : p.K) : p.K;
  const int klen = (int)(k_end - k_begin), n_kt = (klen + BK - 1) / BK, k_tail = klen % BK;

  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / S::WGN, wn = wv % S::WGN;
  const int i16 = l & 15, g4 = l >> 4;
  typedef __attribute__((address_space(3))) unsigned char lds_byte;
  const unsigned lds_base = (unsigned)(__UINTPTR_TYPE__)(lds_byte*)smem_raw;

  // ---- loader
  constexpr int A_CH = BM / 8, B_CH = BN / 8;  // chunks of a [k][row] operand's k-row
  unsigned va[S::PER_A], vb[S::PER_B];
  const char *ba, *bb;
  const int64_t step_a = TA ? 2ll * BK * p.lda : 2 * BK, step_b = TB ? 2ll * BK * p.ldb : 2 * BK;
  const int m_left = (int)(p.M - m0 < BM ? p.M - m0 : BM), n_left = (int)(p.N - n0 < NCOLS ? p.N - n0 : NCOLS);
  {
    const T* A = static_cast<const T*>(p.A);
    const T* B = static_cast<const T*>(DUAL && ((wv * S::PER_B * 8) >> 5 & 1) ? p.B2 : p.B);  // a wave loads rows of one 32-row group
    static_assert(!DUAL || S::PER_B * 8 <= 32, "one matrix per wave");
    ba = reinterpret_cast<const char*>(TA ? A + k_begin * p.lda + m0 : A + m0 * p.lda + k_begin);
    bb = reinterpret_cast<const char*>(TB ? B + k_begin * p.ldb + n0 : B + n0 * p.ldb + k_begin);
#pragma unroll
    for (int j = 0; j < S::PER_A; ++j) {
      const int q = wv * S::PER_A + j;
      if constexpr (!TA) {
        const int row = q * 8 + (l >> 3), c = (l & 7) ^ small_swizzle<TA, true, BM>(row);
        const int r = row < m_left ? row : m_left - 1;  // rows past the edge repeat the last row: their results are not stored
        va[j] = (unsigned)((r * p.lda + c * 8) * 2);
      } else {
        const int k = (q * 64 + l) / A_CH, c = ((q * 64 + l) % A_CH) ^ small_swizzle<TA, true, BM>(k);
        va[j] = (unsigned)((k * p.lda + (c * 8 < m_left ? c * 8 : 0)) * 2);
      }
    }
#pragma unroll
    for (int j = 0; j < S::PER_B; ++j) {
      const int q = wv * S::PER_B + j;
      if constexpr (!TB) {
        const int row = q * 8 + (l >> 3), c = (l & 7) ^ small_swizzle<TB, false, BN>(row);
        int r = DUAL ? (row >> 6) * 32 + (row & 31) : row;
        if (r >= n_left) r = n_left - 1;
        vb[j] = (unsigned)((r * p.ldb + c * 8) * 2);
      } else {
        const int k = (q * 64 + l) / B_CH, c = ((q * 64 + l) % B_CH) ^ small_swizzle<TB, false, BN>(k);
        vb[j] = (unsigned)((k * p.ldb + (c * 8 < n_left ? c * 8 : 0)) * 2);
      }
    }
  }
  auto issue = [&](int t, unsigned stage_off) {
    const unsigned da = lds_base + stage_off + wv * S::PER_A * 1024, db = lds_base + stage_off + S::A_BYTES + wv * S::PER_B * 1024;
    if (k_tail != 0 && t == n_kt - 1) {  // partial K tile: chunks past the end of K are zeros
#pragma unroll
      for (int j = 0; j < S::PER_A; ++j) {
        const int q = wv * S::PER_A + j, row = q * 8 + (l >> 3);
        const int k = TA ? (q * 64 + l) / A_CH : 8 * ((l & 7) ^ small_swizzle<TA, true, BM>(row));
        pp_load_below(da + j * 1024, va[j], ba, k, k_tail);
        if (k >= k_tail) *reinterpret_cast<u32x4*>(smem_raw + (da - lds_base) + j * 1024 + l * 16) = u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int j = 0; j < S::PER_B; ++j) {
        const int q = wv * S::PER_B + j, row = q * 8 + (l >> 3);
        const int k = TB ? (q * 64 + l) / B_CH : 8 * ((l & 7) ^ small_swizzle<TB, false, BN>(row));
        pp_load_below(db + j * 1024, vb[j], bb, k, k_tail);
        if (k >= k_tail) *reinterpret_cast<u32x4*>(smem_raw + (db - lds_base) + j * 1024 + l * 16) = u32x4{0u, 0u, 0u, 0u};
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
#pragma unroll
      for (int j = 0; j < S::PER_A; ++j) pp_load(da + j * 1024, va[j], ba);
#pragma unroll
      for (int j = 0; j < S::PER_B; ++j) pp_load(db + j * 1024, vb[j], bb);
    }
    ba += step_a;
    bb += step_b;
  };
#pragma unroll
  for (int t = 0; t < NST - 1; ++t)
    if (t < n_kt) issue(t, t * S::STAGE);

  // ---- fragment addresses (stage 0)
  unsigned ra[TA ? NA : 2], rb[TB ? 2 * NGB : 2];
  if constexpr (!TA) {
    const int row = wm * S::WM + i16, f = small_swizzle<TA, true, BM>(row);
    ra[0] = row * 128 + ((g4 ^ f) << 4);
    ra[1] = row * 128 + (((4 + g4) ^ f) << 4);
  } else {
    const int k = 8 * g4 + (i16 >> 2), sw = small_swizzle<TA, true, BM>(k);
#pragma unroll
    for (int a = 0; a < NA; ++a) ra[a] = k * (BM * 2) + ((((wm * S::WM + a * 16) / 8 + ((i16 & 3) >> 1)) ^ sw) << 4) + (i16 & 1) * 8;
  }
  if constexpr (!TB) {
    const int row = wn * S::WN + 8 * (i16 >> 2) + (i16 & 3), f = small_swizzle<TB, false, BN>(row);
    rb[0] = S::A_BYTES + row * 128 + ((g4 ^ f) << 4);
    rb[1] = S::A_BYTES + row * 128 + (((4 + g4) ^ f) << 4);
  } else {
    const int k = 8 * g4 + (i16 >> 2), sw = small_swizzle<TB, false, BN>(k);
#pragma unroll
    for (int b = 0; b < 2 * NGB; ++b) rb[b] = S::A_BYTES + k * (BN * 2) + ((((wn * S::WN + b * 16) / 8 + ((i16 & 3) >> 1)) ^ sw) << 4) + (i16 & 1) * 8;
  }

  // ---- epilogue inputs of this lane: row l % 16 of each row block, columns 8 * (l / 16) .. of each 32-column group
  const bool to_ws = (EPI == MVIT_EPI_NONE) && p.split_k > 1;
  const bool vec = to_ws ? (p.N % 4 == 0) : p.vec_ok != 0;
  const bool interior = vec && m0 + BM <= p.M && n0 + NCOLS <= p.N;
  int64_t n_lane[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) n_lane[g] = n0 + (DUAL ? wn * 32 : wn * S::WN + g * 32) + (TB ? tr_first_column(g4) : 8 * g4);
  auto row_of = [&](int it) { return m0 + wm * S::WM + (it / NG) * 16 + i16; };
  constexpr int NLOAD = EPI == MVIT_EPI_SWIGLU_BWD ? 2 : 1;
  [[maybe_unused]] bf16x8 pre[HAS_IN ? ITEMS : 1][NLOAD];
  [[maybe_unused]] bf16x8 bias_g[HAS_BIAS ? NG : 1], bias_u;
  if (interior) {
    if constexpr (HAS_IN) {
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {
        const T* r = static_cast<const T*>(p.R) + row_of(it) * p.ldr + n_lane[it % NG];
        pre[it][0] = *reinterpret_cast<const bf16x8*>(r);
        if (NLOAD == 2) pre[it][NLOAD - 1] = *reinterpret_cast<const bf16x8*>(r + p.aux_off);
      }
    }
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int g = 0; g < NG; ++g) bias_g[g] = *reinterpret_cast<const bf16x8*>(static_cast<const T*>(p.bias) + n_lane[g]);
      if (DUAL) bias_u = *reinterpret_cast<const bf16x8*>(static_cast<const T*>(p.bias2) + n_lane[0]);
    }
  }

  constexpr bool INTERLEAVED = (NST >= 4 || S::WHOLE) && !TA;
  // sums of A's rows over k, see gemm_pingpong.hip: wave wn of a row group takes NRS row blocks, two MFMAs more each per K tile
  constexpr bool ROW_SUMS = TA && TB && EPI == MVIT_EPI_NONE;
  constexpr int NRS = NA / S::WGN;  // row blocks that a wave sums
  static_assert(!ROW_SUMS || (NA % S::WGN == 0 && !INTERLEAVED), "the waves of a row group share its row blocks");
  const bool do_rs = ROW_SUMS && p.row_sums != nullptr && tn == 0;
  [[maybe_unused]] f32x4 rs[ROW_SUMS ? NRS : 1];
#pragma unroll
  for (int i = 0; i < (ROW_SUMS ? NRS : 1); ++i) rs[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- main loop
  f32x4 acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned st = 0, st_in = (NST - 1) * S::STAGE;  // stage consumed, stage filled
  bf16x8 fa[2][NA], fb[2][NB];                    // fragments of the two halves of a K tile
  auto read_a = [&](const unsigned char* at, int ks, int a) {
    if constexpr (!TA) fa[ks][a] = *reinterpret_cast<const bf16x8*>(at + ra[ks] + a * 2048);
    else fa[ks][a] = pp_read_tr(at + ra[a] + ks * 32 * (BM * 2), 4 * (BM * 2));
  };
  auto read_b = [&](const unsigned char* at, int ks, int b) {
    if constexpr (!TB) fb[ks][b] = *reinterpret_cast<const bf16x8*>(at + rb[ks] + (b >> 1) * 4096 + (b & 1) * 512);
    else fb[ks][b] = pp_read_tr(at + rb[b] + ks * 32 * (BN * 2), 4 * (BN * 2));
  };
  auto multiply_row = [&](int ks, int a) {
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[ks][b], fa[ks][a], acc[a][b], 0, 0, 0);
  };
  auto landed = [&](int newer) {  // this wave's share of a K tile has landed once only the `newer` tiles requested after it are in flight
    wait_tiles<S::PER, NST - 2>(newer);
  };
  auto next_stage = [&](unsigned& stage) { stage = stage + S::STAGE == S::LDS ? 0 : stage + S::STAGE; };
  if constexpr (INTERLEAVED && S::WHOLE) {
    // The K tile of parity `par` in registers: its MFMAs row by row, between them the reads of the K tile after it (at `next`) and the loads
    // of the one NST ahead into the stage that this tile was read from.  The compiler keeps to this order.
    bf16x8 ga[2][2][NA], gb[2][2][NB];  // fragments: parity of the K tile, half, block
    auto read_next = [&](const unsigned char* at, int par, int r) {
      const int ks = r / (NA + NB), i = r % (NA + NB);
      if (i < NB) {
        if constexpr (!TB) gb[par][ks][i] = *reinterpret_cast<const bf16x8*>(at + rb[ks] + (i >> 1) * 4096 + (i & 1) * 512);
        else gb[par][ks][i] = pp_read_tr(at + rb[i] + ks * 32 * (BN * 2), 4 * (BN * 2));
      } else {
        if constexpr (!TA) ga[par][ks][i - NB] = *reinterpret_cast<const bf16x8*>(at + ra[ks] + (i - NB) * 2048);
        else ga[par][ks][i - NB] = pp_read_tr(at + ra[i - NB] + ks * 32 * (BM * 2), 4 * (BM * 2));
      }
    };
    auto step = [&](auto parity, auto with_loads, const unsigned char* next, unsigned stage_off) {
      constexpr int par = decltype(parity)::value, LOADS = decltype(with_loads)::value ? S::PER : 0, READS = 2 * (NA + NB), ROWS = 2 * NA;
#pragma unroll
      for (int a = 0; a < ROWS; ++a) {
#pragma unroll
        for (int r = a * READS / ROWS; r < (a + 1) * READS / ROWS; ++r) read_next(next, 1 - par, r);
#pragma unroll
        for (int j = a * LOADS / ROWS; j < (a + 1) * LOADS / ROWS; ++j) {
          if (j < S::PER_A) pp_load(lds_base + stage_off + (wv * S::PER_A + j) * 1024, va[j], ba);
          else pp_load(lds_base + stage_off + S::A_BYTES + (wv * S::PER_B + j - S::PER_A) * 1024, vb[j - S::PER_A], bb);
        }
        const int ks = a / NA, i = a % NA;
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gb[par][ks][b], ga[par][ks][i], acc[i][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto landed_after = [&](int newer) { wait_tiles<S::PER, NST - 2>(newer < 0 ? 0 : newer); };
    if (NST - 1 < n_kt) issue(NST - 1, st_in);  // the last stage is free as well
    wait_tiles<S::PER, NST - 1>(n_kt - 1);
    pp_barrier();
#pragma unroll
    for (int r = 0; r < 2 * (NA + NB); ++r) read_next(smem_raw, 0, r);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    landed_after(n_kt - 2);
    pp_barrier();
    // At the top of step t every wave has the fragments of K tile t, so its stage is free, and tile t + 1 has landed.  The last step's reads
    // past the end stay in the ring and are not used.
    int t = 0;
    auto advance = [&](auto parity) {  // tile t + NST exists and is a whole one
      const unsigned here = st;
      next_stage(st);
      step(parity, std::true_type{}, smem_raw + st, here);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      pp_wait_vm<(NST - 2) * S::PER>();
      pp_barrier();
      ba += step_a;
      bb += step_b;
      ++t;
    };
    auto finish = [&](auto parity) {
      const unsigned here = st;
      next_stage(st);
      if (t + NST < n_kt) issue(t + NST, here);
      step(parity, std::false_type{}, smem_raw + st, 0);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      landed_after(n_kt - 3 - t);
      pp_barrier();
      ++t;
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    for (const int whole = n_kt - NST - (k_tail != 0 ? 1 : 0); t + 1 < whole;) {
      advance(even);
      advance(odd);
    }
    while (t < n_kt) {
      finish(even);
      if (t < n_kt) finish(odd);
    }
  } else if constexpr (INTERLEAVED) {
    constexpr int FIRST = S::PER / 2;  // loads requested in the first half
    // half `ks` of a K tile: its MFMAs row by row, between them the reads of the half after it (at `next`) and loads into stage_off.
    // The compiler keeps to this order.
    auto half = [&](auto half_ks, auto with_loads, const unsigned char* next, unsigned stage_off) {
      constexpr int ks = decltype(half_ks)::value, LOADS = !decltype(with_loads)::value ? 0 : ks ? S::PER - FIRST : FIRST, READS = NA + NB;
#pragma unroll
      for (int a = 0; a < NA; ++a) {
#pragma unroll
        for (int i = a * LOADS / NA; i < (a + 1) * LOADS / NA; ++i) {
          const int j = ks * FIRST + i;
          if (j < S::PER_A) pp_load(lds_base + stage_off + (wv * S::PER_A + j) * 1024, va[j], ba);
          else pp_load(lds_base + stage_off + S::A_BYTES + (wv * S::PER_B + j - S::PER_A) * 1024, vb[j - S::PER_A], bb);
        }
#pragma unroll
        for (int r = a * READS / NA; r < (a + 1) * READS / NA; ++r) {
          if (r < NB) read_b(next, 1 - ks, r);
          else read_a(next, 1 - ks, r - NB);
        }
        multiply_row(ks, a);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    constexpr std::integral_constant<int, 0> first{};
    constexpr std::integral_constant<int, 1> second{};
    landed(n_kt - 1);
    pp_barrier();
#pragma unroll
    for (int b = 0; b < NB; ++b) read_b(smem_raw, 0, b);
#pragma unroll
    for (int a = 0; a < NA; ++a) read_a(smem_raw, 0, a);
    // The barrier between the halves of K tile t: every wave's share of tile t + 1 has landed, and every wave has read all of tile t,
    // whose stage tile t + NST overwrites from the next step on.  The last step's reads past the end stay in the ring and are not used.
    int t = 0;
    for (const int whole = n_kt - (NST - 1) - (k_tail != 0 ? 1 : 0); t < whole; ++t) {  // tile t + NST - 1 exists and is a whole one
      half(first, std::true_type{}, smem_raw + st, st_in);
      next_stage(st);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      pp_wait_vm<(NST - 3) * S::PER + FIRST>();
      pp_barrier();
      half(second, std::true_type{}, smem_raw + st, st_in);
      next_stage(st_in);
      ba += step_a;
      bb += step_b;
    }
    for (; t < n_kt; ++t) {
      if (t + NST - 1 < n_kt) issue(t + NST - 1, st_in);
      half(first, std::false_type{}, smem_raw + st, 0);
      next_stage(st);
      next_stage(st_in);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      landed(n_kt - 2 - t);
      pp_barrier();
      half(second, std::false_type{}, smem_raw + st, 0);
    }
  } else {
    auto loop = [&](auto with_row_sums) {
      for (int t = 0; t < n_kt; ++t) {
        landed(n_kt - 1 - t);
        pp_barrier();  // every wave's share of K tile t is in LDS; K tile t - 1 has been consumed
        if (t + NST - 1 < n_kt) issue(t + NST - 1, st_in);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
          for (int b = 0; b < NB; ++b) read_b(smem_raw + st, ks, b);
#pragma unroll
          for (int a = 0; a < NA; ++a) read_a(smem_raw + st, ks, a);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int a = 0; a < NA; ++a) multiply_row(ks, a);
        if constexpr (decltype(with_row_sums)::value) {
          const bf16_t one = (bf16_t)1.f;
          const bf16x8 ones = {one, one, one, one, one, one, one, one};
#pragma unroll
          for (int a = 0; a < NA; ++a)
            if (wn == a / NRS) {
#pragma unroll
              for (int ks = 0; ks < 2; ++ks) rs[a % NRS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, fa[ks][a], rs[a % NRS], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        next_stage(st);
        next_stage(st_in);
      }
    };
    if (ROW_SUMS && do_rs) loop(std::bool_constant<ROW_SUMS>{});
    else loop(std::false_type{});
  }

  // ---- epilogue
  constexpr bool CAN_CS = EPI == MVIT_EPI_SWIGLU_BWD;
  const bool do_cs = CAN_CS && p.colsum != nullptr;
  float cs[CAN_CS ? NG : 1][16];
#pragma unroll
  for (int g = 0; g < (CAN_CS ? NG : 1); ++g)
#pragma unroll
    for (int e = 0; e < 16; ++e) cs[g][e] = 0.f;
  // A lane's sums over two row blocks (32 rows) meet those of the 16 lanes that share its columns, parked in LDS in chunks of four, chunk
  // c of lane i in slot c ^ i: all banks.  A row of sums is 64 rows: 32 lanes' sums, added one after the other in the order of the
  // rows, so that it has the same bits whichever tile of this file made it (a tile of 128 rows makes two).
  constexpr int HALVES = BM / 64, PITCH = 2 * NCOLS;
  float* red = reinterpret_cast<float*>(smem_raw);
  auto park_sums = [&](int pair) {
    if constexpr (CAN_CS) {
      static_assert(S::WM % 32 == 0 && BM % 64 == 0 && BM / 2 * PITCH * 4 <= S::LDS, "pairs of row blocks, whose sums fit the operand stages");
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int chunk = ((h >> 1) * NCOLS + (int)(n_lane[g] - n0)) / 4 + (h & 1);
          *reinterpret_cast<f32x4*>(red + (wm * (S::WM / 2) + pair * 16 + i16) * PITCH + (chunk ^ i16) * 4) =
              f32x4{cs[g][4 * h], cs[g][4 * h + 1], cs[g][4 * h + 2], cs[g][4 * h + 3]};
          cs[g][4 * h] = cs[g][4 * h + 1] = cs[g][4 * h + 2] = cs[g][4 * h + 3] = 0.f;
        }
    }
  };
  if (do_cs) __syncthreads();  // the last K tile has been consumed
  float* ws = to_ws ? p.workspace + (int64_t)slice * p.M * p.N : nullptr;
  if constexpr (ROW_SUMS) {
#pragma unroll
    for (int i = 0; i < NRS; ++i) {
      const int64_t m = m0 + wm * S::WM + (wn * NRS + i) * 16 + i16;
      if (do_rs && g4 == 0 && m < p.M) {
        if (to_ws) p.row_ws[(int64_t)slice * p.M + m] = rs[i][0];
        else static_cast<TO*>(p.row_sums)[m] = from_f32<TO>(rs[i][0]);
      }
    }
  }
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int a = it / NG, g = it % NG;
    const int64_t m = row_of(it), n = n_lane[g];
    if (do_cs && g == 0 && a % 2 == 0 && a > 0) park_sums(a / 2 - 1);
    float v[8], u[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = acc[a][2 * g][e];
      v[4 + e] = acc[a][2 * g + 1][e];
      if (TB) tr_columns(v[e], v[4 + e]);
      if (DUAL) {
        u[e] = acc[a][NB - 2][e];
        u[4 + e] = acc[a][NB - 1][e];
      }
    }
    if (interior) {
      float hb[8], hb2[8];
      if (HAS_BIAS) unpack8<T>(bias_g[g], hb);
      if (HAS_BIAS && DUAL) unpack8<T>(bias_u, hb2);
      if (to_ws) store8(ws + m * p.N + n, v);
      else emit8_impl<T, TO, EPI, true, HAS_IN>(p, m, n, v, u, HAS_IN ? pre[it] : nullptr, cs[CAN_CS ? g : 0], do_cs, HAS_BIAS ? hb : nullptr, HAS_BIAS && DUAL ? hb2 : nullptr);
    } else {
      if (m >= p.M || n >= p.N) continue;
      if (to_ws) {
        float* w = ws + m * p.N + n;
        if (vec && n + 8 <= p.N) store8(w, v);
        else
          for (int e = 0; e < 8 && n + e < p.N; ++e) w[e] = v[e];
      } else {
        emit8<T, TO, EPI>(p, m, n, v, u, vec, cs[CAN_CS ? g : 0], do_cs);
      }
    }
  }
  if constexpr (CAN_CS) {
    if (do_cs) {
      park_sums(NA / 2 - 1);
      __syncthreads();
      for (int c = threadIdx.x; c < HALVES * PITCH; c += S::NTHREADS) {
        const int part = c / PITCH, cc = c % PITCH, half = cc / NCOLS, col = cc % NCOLS;
        float t = 0.f;
#pragma unroll
        for (int r = 0; r < 32; ++r) t += red[(part * 32 + r) * PITCH + (((cc >> 2) ^ (r & 15)) << 2) + (cc & 3)];
        if (n0 + col < p.N && m0 + part * 64 < p.M) p.colsum[((int64_t)tm * HALVES + part) * p.ldc + (half ? p.aux_off : 0) + n0 + col] = t;
      }
    }
  }
}

// A wave beside the others that reads two bytes of every 64 of B's part of its tile column, as fast as memory gives them: of the K tiles,
// tile row tm takes every tiles_m-th, so that together they bring all of it into the memory-side cache, where the main loops find it.  It passes no
// barrier, and the first barrier of the main loop waits until it has ended: the reading lies in front of the loops (beside the first loads of
// their rings), which is why it has to be short.
// For launches that have units to themselves: there a unit's requests in flight bound the main loop, the more the further away its
// operands are.  us without / with, weights from HBM, input gradients of 1280 columns, K = 6912, 3840, 3456 and 1280: 32 x 64, 256 rows 29.6, 17.8, 16.4, 8.0 / 25.0,
// 14.9, 13.9, 7.9; 64 x 64, 768 rows 35.7, 21.2, 19.5, 9.3 / 29.5, 17.7, 16.2, 8.6; 64 x 128, 1,600 rows 45.8, 27.3, 25.0, 11.8 / 38.6, 24.0, 22.1, 11.1;
// 128 x 128, 2,048 rows 60.4, 35.7, 32.6, 15.2 / 51.4, 30.9, 28.5, 14.5, 3,136 rows 58.4, 34.7, 31.2, 15.6 / 58.5, 34.8, 32.0, 15.9.  Where the weights are in the
// memory-side cache already (towers of some six blocks and fewer; a launch does not know) the reading is for nothing: K = 3456 / 1280 32 x 64 11.9, 6.6 / 13.2, 7.4, 64 x 64 14.4,
// 7.5 / 16.1, 8.4, 64 x 128 20.2, 10.0 / 22.4, 10.7.  Not on 192 x 128
// (4,096 rows 67.8, 40.2, 38.0, 17.5 / 70.7, 41.2, 38.8, 18.0) nor where two work-groups share a unit (1,024 rows on 64 x 64 43.3 / 46.1), nor for fewer than
// four tile rows, whose waves would have too much to read (encoding 64 patches 2.32 / 2.67 ms; 128 rows, four of 32 x 64, 30.5, 18.4, 16.9, 8.2 / 28.3, 16.9, 15.8, 8.2),
// nor on SwiGLU, which loses more than it gains (K = 1280, two of 3456 columns: 64 x 128, 200 rows 13.6 / 15.8, 256 14.7 / 15.8; 128 x 128, 448 rows
// 18.5 / 19.1, 512 18.7 / 18.0), nor on SwiGLU backward (K = 1280, 3456 columns: 64 x 64, 200 rows 9.7 / 10.5, 224 10.5 / 10.6, 256 11.0 / 10.8, with the weights in the caches
// 200 rows 9.1 / 10.2, 256 9.2 / 10.4; 64 x 128, 513 rows 14.8 / 16.3, 576 15.4 / 16.5; its kernel keeps the branch to the wave, without which it takes 10.1, 10.8, 11.4 / 15.1, 15.8), nor
// beside a second stream (ms per step without / with in the backward: 1,600 rows 14.14 / 13.81, 1,936 15.32 / 15.54, 2,600 18.83 / 18.91; checkpointed 1,600 16.55 / 16.65, 1,936 18.38 / 18.56).
template <bool TA, int EPI, typename S>
constexpr bool TOUCHES = !TA && S::BM < 192 && EPI != MVIT_EPI_SWIGLU;
template <bool TB, typename S>
__device__ __forceinline__ void touch_b(const GemmParams& p, const unsigned block) {
  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n), per_xcd = (tiles + 7) / 8, work = (block & 7) * per_xcd + (block >> 3);
  if ((block >> 3) >= per_xcd || work >= tiles) return;
  int tm, tn;
  tile_coords(p, (int)work, tm, tn);
  constexpr int STEP = 32, PER = S::BN * S::BK / STEP / 64, AT_ONCE = 16 / PER;  // elements; loads of a lane and K tile; K tiles at once
  const int64_t n0 = (int64_t)tn * S::BN;
  const int lane = threadIdx.x & 63, n_kt = (int)((p.K + S::BK - 1) / S::BK), n_last = (int)(p.N - n0 < S::BN ? p.N - n0 : S::BN) - 1;
  unsigned seen = 0;
  for (int t0 = tm; t0 < n_kt; t0 += p.tiles_m * AT_ONCE) {
    unsigned v[AT_ONCE][PER];
#pragma unroll
    for (int a = 0; a < AT_ONCE; ++a)
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int t = t0 + a * p.tiles_m, i = j * 64 + lane;  // past the end: the last K tile, column or k again
        const int64_t k = (int64_t)(t < n_kt ? t : n_kt - 1) * S::BK + (TB ? i / (S::BN / STEP) : i % (S::BK / STEP) * STEP), k_in = k < p.K ? k : p.K - 1;
        const int n = TB ? i % (S::BN / STEP) * STEP : i / (S::BK / STEP), n_in = n < n_last ? n : n_last;
        const bf16_t* B = static_cast<const bf16_t*>(p.B) + (TB ? n0 : n0 * p.ldb);
        v[a][j] = *reinterpret_cast<const unsigned short*>(B + (TB ? k_in * p.ldb + n_in : n_in * p.ldb + k_in));
      }
#pragma unroll
    for (int a = 0; a < AT_ONCE; ++a)
#pragma unroll
      for (int j = 0; j < PER; ++j) seen ^= v[a][j];
  }
  asm volatile("" : : "v"(seen));
}

// registers for two work-groups per compute unit; LDS holds two of the smaller rings, one of the deeper ones (Lone*)
template <typename TO, bool TA, bool TB, int EPI, typename S>
__global__ __launch_bounds__(S::NTHREADS + (TOUCHES<TA, EPI, S> ? 64 : 0), S::NW / 2) void gemm_small_kernel(const GemmParams p) {
  if constexpr (TOUCHES<TA, EPI, S>) {
    if (threadIdx.x >= S::NTHREADS) return touch_b<TB, S>(p, blockIdx.x);
  }
  gemm_small_tile<TO, TA, TB, EPI, S>(p, blockIdx.x);
}
// several independent products: each takes a range of work-groups, a multiple of eight so that it stays dealt to the XCDs
template <typename TO, bool TA, bool TB, int EPI, typename S>
__global__ __launch_bounds__(S::NTHREADS, S::NW / 2) void gemm_small_group_kernel(const GemmGroup g) {
  int i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.first_block[i + 1]) ++i;
  gemm_small_tile<TO, TA, TB, EPI, S>(g.p[i], blockIdx.x - g.first_block[i]);
}

using Small64 = SmallCfg<64, 64, 2, 2, 4>;       // 64 KiB of LDS
using Small64x128 = SmallCfg<64, 128, 2, 2, 3>;  // 72 KiB
using Small128 = SmallCfg<128, 128, 2, 2, 2>;    // 64 KiB
// one work-group per compute unit, which has work for one at most
using Lone32x64 = SmallCfg<32, 64, 2, 2, 5, true>;    // 60 KiB
using Lone64 = SmallCfg<64, 64, 2, 2, 4, true>;       // 64 KiB
using Lone64x128 = SmallCfg<64, 128, 2, 2, 4, true>;  // 96 KiB
using Lone128 = SmallCfg<128, 128, 2, 2, 4>;          // 128 KiB
using Lone192 = SmallCfg<192, 128, 2, 2, 4>;          // 160 KiB

template <typename S, typename P>
int launch_grid(void (*kern)(P), const P& p, unsigned grid, bool (&attr_set_on)[MVIT_MAX_DEVICES], hipStream_t stream, bool extra_wave = false) {
  const int dev = mvit_current_device("gemm");
  if (dev < 0) return MVIT_ERR_LAUNCH;
  if (!attr_set_on[dev] && S::LDS > 64 * 1024) {  // dynamic LDS above 64 KiB is opted into once per kernel and device
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    if (e != hipSuccess) return mvit_set_error(MVIT_ERR_LAUNCH, "gemm: hipFuncSetAttribute(%d B LDS): %s", S::LDS, hipGetErrorString(e));
    attr_set_on[dev] = true;
  }
  hipLaunchKernelGGL(kern, grid, S::NTHREADS + (extra_wave ? 64 : 0), S::LDS, stream, p);
  MVIT_CHECK_LAUNCH("gemm");
  return MVIT_OK;
}
inline unsigned grid_of(const GemmParams& p) { return (unsigned)((p.tiles_m * p.tiles_n * p.split_k + 7) / 8 * 8); }

template <typename TO, bool TA, bool TB, int EPI, typename S>
int launch_small(const GemmParams& p, bool ahead, hipStream_t stream) {
  static bool attr_set_on[MVIT_MAX_DEVICES] = {};
  return launch_grid<S>(gemm_small_kernel<TO, TA, TB, EPI, S>, p, grid_of(p), attr_set_on, stream, TOUCHES<TA, EPI, S> && ahead);
}
template <typename S>
int launch_group(GemmGroup& g, hipStream_t stream) {
  static bool attr_set_on[MVIT_MAX_DEVICES] = {};
  unsigned blocks = 0;
  for (int i = 0; i < g.n; ++i) {
    g.first_block[i] = blocks;
    blocks += grid_of(g.p[i]);
  }
  return launch_grid<S>(gemm_small_group_kernel<bf16_t, true, true, MVIT_EPI_NONE, S>, g, blocks, attr_set_on, stream);
}

template <typename S>
int dispatch_small(GemmTiledKind kind, const GemmParams& p, bool ahead, hipStream_t s) {
  switch (kind) {
    case NN_NONE: return launch_small<bf16_t, false, false, MVIT_EPI_NONE, S>(p, ahead, s);
    case NN_BIAS: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS, S>(p, ahead, s);
    case NN_BIAS_RES: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS_RES, S>(p, ahead, s);
    case NN_BIAS_GELU: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS_GELU, S>(p, ahead, s);
    case NN_SWIGLU:
      if constexpr (S::WN == 64) return launch_small<bf16_t, false, false, MVIT_EPI_SWIGLU, S>(p, ahead, s);
      break;
    case NT_NONE: return launch_small<bf16_t, false, true, MVIT_EPI_NONE, S>(p, ahead, s);
    case NT_GELU_BWD: return launch_small<bf16_t, false, true, MVIT_EPI_GELU_BWD, S>(p, ahead, s);
    case NT_SWIGLU_BWD: return launch_small<bf16_t, false, true, MVIT_EPI_SWIGLU_BWD, S>(p, ahead, s);
    case TT_NONE: return launch_small<bf16_t, true, true, MVIT_EPI_NONE, S>(p, ahead, s);
    case TT_NONE_F32: return launch_small<float, true, true, MVIT_EPI_NONE, S>(p, ahead, s);
    default: break;
  }
  return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: product kind %d has no %d x %d kernel", (int)kind, S::BM, S::BN);
}

// the tiles of which one work-group fills a compute unit: products with one operand or none behind the transposing LDS read
template <typename S>
int dispatch_lone(GemmTiledKind kind, const GemmParams& p, bool ahead, hipStream_t s) {
  switch (kind) {
    case NN_NONE: return launch_small<bf16_t, false, false, MVIT_EPI_NONE, S>(p, ahead, s);
    case NN_BIAS: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS, S>(p, ahead, s);
    case NN_BIAS_RES: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS_RES, S>(p, ahead, s);
    case NN_BIAS_GELU: return launch_small<bf16_t, false, false, MVIT_EPI_BIAS_GELU, S>(p, ahead, s);
    case NT_NONE: return launch_small<bf16_t, false, true, MVIT_EPI_NONE, S>(p, ahead, s);
    case NT_GELU_BWD: return launch_small<bf16_t, false, true, MVIT_EPI_GELU_BWD, S>(p, ahead, s);
    case NN_SWIGLU:
      if constexpr (S::BM == 128) return launch_small<bf16_t, false, false, MVIT_EPI_SWIGLU, S>(p, ahead, s);
      break;
    case NT_SWIGLU_BWD:
      if constexpr (S::BM == 64 && S::BN == 64) return launch_small<bf16_t, false, true, MVIT_EPI_SWIGLU_BWD, S>(p, ahead, s);
      break;
    default: break;
  }
  return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: product kind %d has no %d x %d kernel of one work-group per unit", (int)kind, S::BM, S::BN);
}

}  // namespace

int mvit_gemm_small(GemmTiledKind kind, int bm, int bn, bool lone, const GemmParams& p, int own_units, hipStream_t stream) {
  const bool ahead = gemm_reads_ahead(kind, bm, p.tiles_m, (int64_t)p.tiles_m * p.tiles_n, p.split_k, own_units);
  if (lone) {
    if (bm == 192) return dispatch_lone<Lone192>(kind, p, ahead, stream);
    if (bm == 128) return dispatch_lone<Lone128>(kind, p, ahead, stream);
    if (bm == 32) return dispatch_lone<Lone32x64>(kind, p, ahead, stream);
    return bn == 128 ? dispatch_lone<Lone64x128>(kind, p, ahead, stream) : dispatch_lone<Lone64>(kind, p, ahead, stream);
  }
  if (bm == 128) return dispatch_small<Small128>(kind, p, ahead, stream);
  if (bn == 128) return dispatch_small<Small64x128>(kind, p, ahead, stream);
  return dispatch_small<Small64>(kind, p, ahead, stream);
}
// weight gradients (both operands transposed, bf16 results), tiles_m / tiles_n set for bm x bn
int mvit_gemm_small_group(int bm, int bn, GemmGroup& g, hipStream_t stream) {
  if (bm == 128) return launch_group<Small128>(g, stream);
  if (bn == 128) return launch_group<Small64x128>(g, stream);
  return launch_group<Small64>(g, stream);
}
