// fp32 GEMM (the parity path) on v_mfma_f32_16x16x4_f32:  C[M,N] = epi( sum_k A[m,k] * B[n,k] ).
//
// What bounds it is the fp32 matrix rate (157 TFLOP/s, a sixteenth of bf16's) once enough compute units have work: a
// 64 x 64 tile per work-group of four waves (a K tile of 32 is 1,024 cycles of MFMA and 16 KiB of operands), or a 32 x 64 or 32 x 32
// tile where there are few of those (half_rows, quarters below).
// K tiles of 32 floats (128-byte rows) in a ring of four LDS stages filled by direct global -> LDS loads, two work-groups
// per compute unit.  MFMA (s, j) of a K tile contracts k = 16 s + 4 g + j over the lane groups g = 0..3, so one 16-byte read
// of a [row][k] operand feeds four of them; a [k][row] operand is read as two neighbouring rows (8 bytes) per k, and the two
// row blocks of a wave are its even and its odd rows.
// Loads, the LDS reads of the next half K tile and MFMAs alternate: one after the other, a wave's MFMAs waited for its requests
// and its reads (us: 512 rows K = 1280 x 3840 48.6 -> 44.6, input gradient K = 6912 137 -> 121, its weight gradient 92 -> 80; 2,048
// rows 340 -> 293, 337 -> 292, i.e. 123 TFLOP/s; 4-block step of 512 rows 4.00 -> 3.62 ms, of 2,048 11.8 -> 10.3).
// The products are computed transposed (B's fragment first), so a lane ends with eight consecutive columns of a row and
// stores them from registers (a 32 x 32 tile's lanes trade four for that).  All tiles add in the same order: a row's result does not depend on its batch.
#include "gemm_direct.h"

#include <type_traits>

namespace {

template <int BM_, int BN_, int WGM_, int WGN_>
struct F32Cfg {
  static constexpr int BM = BM_, BN = BN_, BK = 32, NST = 4, NTHREADS = 256, WGM = WGM_, WGN = WGN_, WM = BM / WGM, WN = BN / WGN;
  static constexpr int A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128, LDS = NST * STAGE;
  static constexpr int PER_A = BM / 32, PER_B = BN / 32, PER = PER_A + PER_B;  // 1 KiB loads per wave and K tile
};

// slot of chunk c (16 bytes) of row `major` ([row][k]: eight chunks) or k-row `major` ([k][row]: CHUNKS of them).  DEALT: rows as a
// fragment of two column blocks takes them
template <bool TR, bool DEALT, int CHUNKS>
__device__ __forceinline__ int f32_swizzle(int major) {
  if (TR) return ((major >> 2) & 1) * (CHUNKS / 2);
  return !DEALT ? (major >> 1) & 7 : ((major >> 1) & 1) | (((major >> 3) & 3) << 1);
}

template <bool TA, bool TB, int EPI, int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const GemmParams p) {
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  using S = F32Cfg<BM, BN, DUAL ? 4 : 2, DUAL ? 1 : 2>;
  constexpr int BK = S::BK, NST = S::NST, NA = S::WM / 16, NB = S::WN / 16, NG = DUAL || NB == 1 ? 1 : NB / 2, NCOLS = DUAL ? 32 : BN;
  constexpr bool DEALT = NB > 1;  // B's rows ([row][k]) are dealt to two column blocks
  static_assert((!TA || NA == 2) && (!TB || NB <= 2), "[k][row] operands are read as pairs of rows, or B's one by one");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n), total = tiles * (unsigned)p.split_k, per_xcd = (total + 7) / 8;
  const unsigned work = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per_xcd || work >= total) return;
  const unsigned slice = p.split_k > 1 ? work / tiles : 0;
  int tm, tn;
  tile_coords(p, (int)(work - slice * tiles), tm, tn);
  const int64_t m0 = (int64_t)tm * S::BM, n0 = (int64_t)tn * NCOLS;
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
  const char *pa[S::PER_A], *pb[S::PER_B];
  int ka[S::PER_A], kb[S::PER_B];  // first k of the lane's chunk inside a K tile
  const int64_t step_a = TA ? 4ll * BK * p.lda : 4 * BK, step_b = TB ? 4ll * BK * p.ldb : 4 * BK;
  const int m_left = (int)(p.M - m0 < S::BM ? p.M - m0 : S::BM), n_left = (int)(p.N - n0 < NCOLS ? p.N - n0 : NCOLS);
  auto place = [&](auto TR, auto DEALT_, auto CHUNKS, int q, const void* X, int64_t ld, int64_t row0, int left, int row_of_tile, const char*& ptr, int& k) {
    const float* x = static_cast<const float*>(X);
    if (!decltype(TR)::value) {
      const int c = (l & 7) ^ f32_swizzle<false, decltype(DEALT_)::value, 8>(q * 8 + (l >> 3));
      const int r = row_of_tile < left ? row_of_tile : left - 1;  // rows past the edge repeat the last row: their results are not stored
      k = c * 4;
      ptr = reinterpret_cast<const char*>(x + (row0 + r) * ld + k_begin + k);
    } else {
      constexpr int CH = decltype(CHUNKS)::value;
      k = q * (64 / CH) + l / CH;
      const int c = (l % CH) ^ f32_swizzle<true, false, CH>(k);
      ptr = reinterpret_cast<const char*>(x + (k_begin + k) * ld + row0 + (c * 4 < left ? c * 4 : 0));
    }
  };
#pragma unroll
  for (int j = 0; j < S::PER_A; ++j) {
    const int q = wv * S::PER_A + j;
    place(std::bool_constant<TA>{}, std::false_type{}, std::integral_constant<int, BM / 4>{}, q, p.A, p.lda, m0, m_left, q * 8 + (l >> 3), pa[j], ka[j]);
  }
#pragma unroll
  for (int j = 0; j < S::PER_B; ++j) {
    const int q = wv * S::PER_B + j, row = q * 8 + (l >> 3);
    // SWIGLU: tile rows 0-31 are gate rows, 32-63 up rows
    place(std::bool_constant<TB>{}, std::bool_constant<DEALT>{}, std::integral_constant<int, BN / 4>{}, q, DUAL && q >= 4 ? p.B2 : p.B, p.ldb, n0, n_left, DUAL ? row & 31 : row, pb[j], kb[j]);
  }
  auto issue = [&](int t, unsigned stage_off) {
    const unsigned da = lds_base + stage_off + wv * (S::PER_A * 1024), db = lds_base + stage_off + S::A_BYTES + wv * (S::PER_B * 1024);
    if (k_tail != 0 && t == n_kt - 1) {  // the partial K tile: chunks past the end of K are zeros
      auto load = [&](unsigned at, const char* ptr, int k) {
        pp_load_at_below(at, ptr, k, k_tail);
        if (k >= k_tail) *reinterpret_cast<u32x4*>(smem_raw + (at - lds_base) + l * 16) = u32x4{0u, 0u, 0u, 0u};
      };
#pragma unroll
      for (int j = 0; j < S::PER_A; ++j) load(da + j * 1024, pa[j], ka[j]);
#pragma unroll
      for (int j = 0; j < S::PER_B; ++j) load(db + j * 1024, pb[j], kb[j]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      return;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // A and B by turns
      if (j < S::PER_A) {
        pp_load_at(da + j * 1024, pa[j]);
        pa[j] += step_a;
      }
      if (j < S::PER_B) {
        pp_load_at(db + j * 1024, pb[j]);
        pb[j] += step_b;
      }
    }
  };
#pragma unroll
  for (int t = 0; t < NST - 1; ++t)
    if (t < n_kt) issue(t, t * S::STAGE);

  // ---- fragment addresses (stage 0)
  unsigned ra[2], rb[2];  // [row][k]: chunk 4 s + g of the lane's row; [k][row]: entry 0, k-row 4 g
  if constexpr (!TA) {
    const int row = wm * S::WM + i16, f = f32_swizzle<false, false, 8>(row);
    ra[0] = row * 128 + ((g4 ^ f) << 4);
    ra[1] = row * 128 + (((4 + g4) ^ f) << 4);
  } else {
    const int r = wm * S::WM + 2 * i16;
    ra[0] = ra[1] = 4 * g4 * 256 + (((r >> 2) ^ f32_swizzle<true, false, 16>(4 * g4)) << 4) + (r & 3) * 4;
  }
  if constexpr (!TB) {
    const int row = wn * S::WN + (DEALT ? 8 * (i16 >> 2) + (i16 & 3) : i16), f = f32_swizzle<false, DEALT, 8>(row);
    rb[0] = S::A_BYTES + row * 128 + ((g4 ^ f) << 4);
    rb[1] = S::A_BYTES + row * 128 + (((4 + g4) ^ f) << 4);
  } else {
    const int r = wn * S::WN + NB * i16;
    rb[0] = rb[1] = S::A_BYTES + 4 * g4 * (BN * 4) + (((r >> 2) ^ f32_swizzle<true, false, BN / 4>(4 * g4)) << 4) + (r & 3) * 4;
  }

  f32x4 acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned st = 0, st_in = (NST - 1) * S::STAGE;  // stage consumed, stage filled
  float fa[NA][8], fb[NB][8];                     // [block][4 s + j], s the half of the K tile
  constexpr int READS_A = TA ? 4 : NA, READS_B = TB ? 4 : NB, READS = READS_A + READS_B;
  auto read = [&](const unsigned char* at, int s, int r) {  // the r-th read of half s
    if (r < READS_A) {
      if constexpr (!TA) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(at + ra[s] + r * 2048);
#pragma unroll
        for (int j = 0; j < 4; ++j) fa[r < NA ? r : 0][4 * s + j] = v[j];
      } else {
        const f32x2 v = *reinterpret_cast<const f32x2*>(at + ra[0] + (16 * s + r) * 256);
        fa[0][4 * s + r] = v[0];
        fa[NA - 1][4 * s + r] = v[1];
      }
    } else {
      r -= READS_A;
      if constexpr (!TB) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(at + rb[s] + (r >> 1) * 4096 + (r & 1) * 512);
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[r < NB ? r : 0][4 * s + j] = v[j];
      } else if constexpr (NB == 2) {
        const f32x2 v = *reinterpret_cast<const f32x2*>(at + rb[0] + (16 * s + r) * (BN * 4));
        fb[0][4 * s + r] = v[0];
        fb[NB - 1][4 * s + r] = v[1];
      } else {
        fb[0][4 * s + r] = *reinterpret_cast<const float*>(at + rb[0] + (16 * s + r) * (BN * 4));
      }
    }
  };
  constexpr int FIRST = S::PER / 2;  // loads requested in the first half
  auto half = [&](auto half_s, auto with_loads, const unsigned char* next, unsigned stage_off) {
    constexpr int s = decltype(half_s)::value, LOADS = !decltype(with_loads)::value ? 0 : s ? S::PER - FIRST : FIRST;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int i = k * LOADS / 4; i < (k + 1) * LOADS / 4; ++i) {
        const int j = s * FIRST + i;
        if (j < S::PER_A) {
          pp_load_at(lds_base + stage_off + (wv * S::PER_A + j) * 1024, pa[j]);
          pa[j] += step_a;
        } else {
          pp_load_at(lds_base + stage_off + S::A_BYTES + (wv * S::PER_B + j - S::PER_A) * 1024, pb[j - S::PER_A]);
          pb[j - S::PER_A] += step_b;
        }
      }
#pragma unroll
      for (int r = k * READS / 4; r < (k + 1) * READS / 4; ++r) read(next, 1 - s, r);
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[b][4 * s + k], fa[a][4 * s + k], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto landed = [&](int newer) {  // this wave's share of a K tile has landed once only the `newer` tiles requested after it are in flight
    if (newer >= 2) pp_wait_vm<2 * S::PER>();
    else if (newer == 1) pp_wait_vm<S::PER>();
    else pp_wait_vm<0>();
  };
  auto next_stage = [&](unsigned& stage) { stage = stage + S::STAGE == S::LDS ? 0 : stage + S::STAGE; };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  landed(n_kt - 1);
  pp_barrier();
#pragma unroll
  for (int r = 0; r < READS; ++r) read(smem_raw, 0, r);
  // the barrier between the halves of K tile t: every wave's share of tile t + 1 has landed, and every wave has read all of tile t
  int t = 0;
  for (const int whole = n_kt - (NST - 1) - (k_tail != 0 ? 1 : 0); t < whole; ++t) {  // tile t + NST - 1 exists and is a whole one
    half(first, std::true_type{}, smem_raw + st, st_in);
    next_stage(st);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    pp_wait_vm<(NST - 3) * S::PER + FIRST>();
    pp_barrier();
    half(second, std::true_type{}, smem_raw + st, st_in);
    next_stage(st_in);
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

  // ---- epilogue: the lane holds columns 8 g .. 8 g + 7 of each 32-column group, one row per row block
  const bool to_ws = (EPI == MVIT_EPI_NONE) && p.split_k > 1;
  const bool vec = to_ws ? (p.N % 4 == 0) : p.vec_ok != 0;
  float* ws = to_ws ? p.workspace + (int64_t)slice * p.M * p.N : nullptr;
  float no_cs[16];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int64_t m = m0 + wm * S::WM + (TA ? 2 * i16 + a : a * 16 + i16), n = n0 + (DUAL ? 0 : wn * S::WN) + (NB == 1 ? 4 * g4 : g * 32 + 8 * g4);
      float v[8], u[8];
      if constexpr (NB == 1) {  // one block: every other group of 16 lanes takes its neighbour's four columns to its own
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = acc[a][0][r];
          v[4 + r] = __shfl_xor(v[r], 16);
        }
        if (g4 & 1) continue;
      }
      if (m >= p.M || n >= p.N) continue;
#pragma unroll
      for (int r = 0; r < (NB == 1 ? 0 : 4); ++r) {
        v[TB ? 2 * r : r] = acc[a][2 * g][r];
        v[TB ? 2 * r + 1 : 4 + r] = acc[a][NB == 1 ? 0 : 2 * g + 1][r];
        if (DUAL) {
          u[r] = acc[a][NB - 2][r];
          u[4 + r] = acc[a][NB - 1][r];
        }
      }
      if (to_ws) {
        float* w = ws + m * p.N + n;
        if (vec && n + 8 <= p.N) store8(w, v);
        else
          for (int e = 0; e < 8 && n + e < p.N; ++e) w[e] = v[e];
      } else {
        emit8<float, float, EPI>(p, m, n, v, u, vec, no_cs, false);
      }
    }
}

// 32-row tiles where they shorten the launch: while 64-row tiles leave a quarter of the compute units without one, and after that
// where halving saves part of the last round (us, 64 / 32 rows, input gradients: K = 1280 27 / 17 at 256 rows, 45 / 36 at 1,024,
// 45 / 49 at 1,536, 66 / 58 at 2,048; K = 6912 126 / 77 at 256 rows, 127 / 121 at 512).  Nearly a tile per unit stays whole: halves
// are hardly faster alone (256 rows x 3840: 28.5 / 27.6), and beside a second stream's products a step of 256 rows took 3.19 ms with
// them and 2.97 without.
inline bool half_rows(const GemmParams& p, int64_t units) {
  const int64_t tn = (p.N + 63) / 64 * p.split_k, tiles = (p.M + 63) / 64 * tn;
  const int64_t rounds = (tiles + units - 1) / units, half_rounds = ((p.M + 31) / 32 * tn + units - 1) / units;
  return tiles <= units * 3 / 4 || (rounds > 1 && rounds <= 3 && half_rounds < 2 * rounds);
}

// 32 x 32 tiles (a wave's share is one MFMA block) where every compute unit has at most one, or three where 32 x 64 tiles would be two
// to a unit: there the matrix pipes of a unit with two of those work 1.6 times as long as the average's.  At other counts halving saves
// no part of a round, or each tile's own steps cost more than it saves.  us, input gradients, 32 x 32 / 32 x 64 / 64 x 64 tiles by 32 x 32 tiles
// per unit, K = 6912: one 56 / 78 / 128 (3840 columns, 32 rows), two 86 / 80 / 129 (1280 columns, 256 rows), three 107 / 125 / 129 (512), four 130 / 126 /
// 130 (640), five 211 / 179 / 221 (896), seven 252 / 243 / 222 (1280); K = 1280: one 15.2 / 18.9 / 28.3, two 20.7 / 19.5 / 28.5, three 24.9 / 28.0 / 28.5,
// four 30.0 / 28.2 / 28.9, five 39.9 / 38.0 / 46.2, seven 48.4 / 50.4 / 46.2.  Of 168 products (1280 and 3840 columns, K = 1280, 3840 and 6912, 32 to 1,536
// rows, forward and input gradient) the tile taken is never more than 6 % behind the best, that at four per unit.  4-block step of 512 rows 3.62 ->
// 3.47 ms, of 64 (bound by the host) 2.21 -> 2.18.
inline bool quarters(const GemmParams& p, int64_t units) {
  const int64_t per_unit = ((p.M + 31) / 32 * ((p.N + 31) / 32) * p.split_k + units - 1) / units;
  return per_unit == 1 || per_unit == 3;
}

template <bool TA, bool TB, int EPI, int BM, int BN = 64>
int launch_f32_tiles(GemmParams p, hipStream_t stream) {
  constexpr int NCOLS = EPI == MVIT_EPI_SWIGLU ? 32 : BN;
  const int64_t tm = (p.M + BM - 1) / BM, tn = (p.N + NCOLS - 1) / NCOLS;
  MVIT_REQUIRE(tm * tn * p.split_k < (1ll << 30), "gemm: too many tiles");
  p.tiles_m = (int)tm; p.tiles_n = (int)tn;
  p.group_m = p.tiles_m;
  p.panel_w = tn <= 6 ? (int)tn : 4;
  hipLaunchKernelGGL((gemm_f32_kernel<TA, TB, EPI, BM, BN>), (p.tiles_m * p.tiles_n * p.split_k + 7) / 8 * 8, 256, (F32Cfg<BM, BN, 2, 2>::LDS), stream, p);
  MVIT_CHECK_LAUNCH("gemm");
  return MVIT_OK;
}

template <bool TA, bool TB, int EPI>
int launch_f32(const GemmParams& p, int n_cu, hipStream_t stream) {
  if constexpr (!TA && EPI != MVIT_EPI_SWIGLU) {
    if (quarters(p, n_cu)) return launch_f32_tiles<TA, TB, EPI, 32, 32>(p, stream);
    if (half_rows(p, n_cu)) return launch_f32_tiles<TA, TB, EPI, 32>(p, stream);
  }
  return launch_f32_tiles<TA, TB, EPI, 64>(p, stream);
}

}  // namespace

int mvit_gemm_f32(int ta, int tb, int epi, const GemmParams& p, int n_cu, hipStream_t s) {
  if (!ta && !tb) {
    switch (epi) {
      case MVIT_EPI_NONE: return launch_f32<false, false, MVIT_EPI_NONE>(p, n_cu, s);
      case MVIT_EPI_BIAS: return launch_f32<false, false, MVIT_EPI_BIAS>(p, n_cu, s);
      case MVIT_EPI_BIAS_RES: return launch_f32<false, false, MVIT_EPI_BIAS_RES>(p, n_cu, s);
      case MVIT_EPI_BIAS_GELU: return launch_f32<false, false, MVIT_EPI_BIAS_GELU>(p, n_cu, s);
      case MVIT_EPI_SWIGLU: return launch_f32<false, false, MVIT_EPI_SWIGLU>(p, n_cu, s);
      case MVIT_EPI_ACCUM: return launch_f32<false, false, MVIT_EPI_ACCUM>(p, n_cu, s);
      default: break;
    }
  } else if (!ta && tb) {
    switch (epi) {
      case MVIT_EPI_NONE: return launch_f32<false, true, MVIT_EPI_NONE>(p, n_cu, s);
      case MVIT_EPI_BIAS: return launch_f32<false, true, MVIT_EPI_BIAS>(p, n_cu, s);
      case MVIT_EPI_SWIGLU_BWD: return launch_f32<false, true, MVIT_EPI_SWIGLU_BWD>(p, n_cu, s);
      case MVIT_EPI_GELU_BWD: return launch_f32<false, true, MVIT_EPI_GELU_BWD>(p, n_cu, s);
      case MVIT_EPI_ACCUM: return launch_f32<false, true, MVIT_EPI_ACCUM>(p, n_cu, s);
      default: break;
    }
  } else if (ta && tb) {
    switch (epi) {
      case MVIT_EPI_NONE: return launch_f32<true, true, MVIT_EPI_NONE>(p, n_cu, s);
      case MVIT_EPI_BIAS: return launch_f32<true, true, MVIT_EPI_BIAS>(p, n_cu, s);
      case MVIT_EPI_ACCUM: return launch_f32<true, true, MVIT_EPI_ACCUM>(p, n_cu, s);
      default: break;
    }
  } else {
    return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: trans_a=1, trans_b=0 is not built");
  }
  return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: epilogue %d not built for trans_a=%d trans_b=%d", epi, ta, tb);
}
