// bf16 GEMM main loop in which the two waves of a SIMD take turns: while one feeds the matrix pipe, the other reads LDS
// and requests the operands to come.
//
// 256 x 256 output tile, eight waves: group wm = 0, 1 (four waves, one per SIMD) x wn = 0..3.  K tiles of 64 in two LDS
// stages of 64 KiB, each four half tiles of 16 KiB (rows 0-127 and 128-255 of A, two halves of B's columns).  A wave owns
// 64 rows of each A half and 32 columns of each B half; a K tile is four phases, one per (A half, B half), of 16
// v_mfma_f32_16x16x32_bf16 each.  A phase is: LDS reads for it, one half tile requested (two global -> LDS loads per
// wave), barrier, the MFMAs, barrier; group 1 runs one barrier behind group 0, so the matrix pipe of every SIMD always has
// a wave in its MFMA part.
//
// Half tiles are numbered n = 4 * K tile + {0: B half 0, 1: A half 0, 2: B half 1, 3: A half 1}.  Phase 4t + 0 reads
// B half 0 and A half 0 of K tile t, phase 4t + 1 B half 1, phase 4t + 2 A half 1 (B half 0 is still in registers for phase
// 4t + 3), i.e. half tile n is read in phase n - 1 or, B half 0, n.  Phase P requests n = P + 6 (six are requested before
// phase 0).  n overwrites n - 8, which was read at least two phases before n is requested, and by then both groups have
// passed a barrier behind those reads.  Before the barrier of phase P each wave waits until its own loads of n <= P + 2
// have landed: at most four half tiles (eight loads) may still be in flight, fewer at the end of K.
//
// The products are computed transposed (B's fragment is the MFMA's first operand) so that a lane ends up with eight consecutive
// columns of one row: by the way a row-major B's columns are dealt to the fragments, or, where the fragments come through the
// transposing read, by a lane exchange in the epilogue (tr_columns): results leave the registers as 16-byte vectors with no LDS
// staging and no barrier, and the next tile's first loads run under them.  K order and MFMA form are the same for every tile shape of
// this file, so a result does not depend on the shape that computed it.
//
// SwiGLU backward (two inputs and two outputs per element, column sums): us at 4,096 / 14,336 / 65,536 rows of 3456 columns 50 / 187 / 798,
// with K tiles of 32 and results staged in LDS 64 / 221 / 778; per 32-block step 14,336 rows 64.9 -> 64.5 ms, 16,384 96.2 -> 95.2, 25,524
// 111.4 -> 110.9.  What bounds it is the epilogue's memory traffic (stores left out: 652 us at 65,536 rows).
//
// LDS layouts (a direct load writes 1 KiB of contiguous LDS per instruction; the lanes choose which 16 bytes they fetch):
//   [row][k] operands: 128-byte rows of 8 chunks, chunk c of row r in slot c ^ f(r); f makes the 16 rows of a fragment read
//   fall on 16 different 16-byte slots of 256 bytes;
//   [k][row] operands: 256-byte k-rows of 16 chunks, read with the transposing ds_read_b64_tr_b16.
#include "gemm_direct.h"

namespace {

struct PpCfg {
  static constexpr int BM = 256, BN = 256, BK = 64, NTHREADS = 512;
  static constexpr int HALF = 16384, STAGE = 4 * HALF;      // A0 | A1 | B0 | B1
  static constexpr int BIAS_OFF = 2 * STAGE, BIAS_BYTES = 2 * 8 * 256;  // two tiles' worth, 256 bytes per wave
  static constexpr int SUMS_BYTES = 32768;  // SwiGLU backward, in place of the biases: 16 lanes' column sums of all 256 columns, gate and up
  static constexpr int lds(int epi) { return BIAS_OFF + (epi == MVIT_EPI_SWIGLU_BWD ? SUMS_BYTES : BIAS_BYTES); }
  static constexpr int MIN_K = 2 * BK + 1;  // at least three K tiles
};

template <typename TO, bool TA, bool TB, int EPI>
__global__ __launch_bounds__(PpCfg::NTHREADS, 2) void gemm_pp_kernel(const GemmParams p) {
  using T = bf16_t;
  constexpr int BM = PpCfg::BM, BK = PpCfg::BK, HALF = PpCfg::HALF, STAGE = PpCfg::STAGE;
  constexpr bool DUAL = (EPI == MVIT_EPI_SWIGLU);
  constexpr bool SW_BWD = EPI == MVIT_EPI_SWIGLU_BWD;
  constexpr bool HAS_IN = EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_GELU_BWD || SW_BWD;
  constexpr bool HAS_BIAS = EPI == MVIT_EPI_BIAS || EPI == MVIT_EPI_BIAS_RES || EPI == MVIT_EPI_BIAS_GELU || EPI == MVIT_EPI_SWIGLU;
  constexpr int NCOLS = DUAL ? 128 : 256;
  // sums of A's rows over k (the bias gradient of a weight-gradient product) from the fragments that are in registers anyway:
  // in the tiles of the first tile column the four waves of a group take one row block of each A half, 4 MFMAs with a vector
  // of ones beside 64.  In passes of their own the column sums of the gradients took 211 us and six launches per block of the
  // tower at 65,536 rows, 30 us and eight launches at 256 (forward + backward of the 32 blocks: 672 -> 666 ms and 15.4 -> 13.3).
  constexpr bool ROW_SUMS = TA && TB && EPI == MVIT_EPI_NONE;
  static_assert(!DUAL || !TB, "SWIGLU takes untransposed operands");
  // stores of an interior tile's epilogue that are issued after the next tile's first loads (memory instructions of a wave
  // complete in order, so a wait for those loads may leave this many more in flight)
  constexpr int STORES = DUAL ? 8 : (EPI == MVIT_EPI_BIAS_GELU ? 32 : (sizeof(TO) == 4 ? 32 : 16));
  constexpr int NIN = SW_BWD ? 2 : 1, DEPTH = SW_BWD ? 4 : 8;  // inputs of an item; items whose inputs are fetched ahead
  constexpr int TRAILING = HAS_IN ? DEPTH * NIN : STORES;  // an item stores as many vectors as it has inputs
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv >> 2, wn = wv & 3;
  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n);
  const unsigned total = tiles * (unsigned)p.split_k;
  const unsigned per_xcd = (total + 7) / 8;
  typedef __attribute__((address_space(3))) unsigned char lds_byte;
  const unsigned lds_base = (unsigned)(__UINTPTR_TYPE__)(lds_byte*)smem_raw;
  const unsigned lds0 = lds_base + wv * 2048;  // this wave's share of a half tile

  // ---- fragment addresses (stage 0, half 0)
  const int i16 = l & 15, g4 = l >> 4;
  // a transposing read takes 16 consecutive columns (32 bytes) of four k-rows per 16 lanes; this swizzle spreads the sixteen k-rows
  // of a wave's instruction over all 256 bytes of the banks
  auto tr_swizzle = [](int k) { return ((k & 3) << 1) | (((k >> 3) & 1) << 3); };
  unsigned ra[TA ? 4 : 2], rb[2];
  if constexpr (!TA) {
    const int row = wm * 64 + i16;
    ra[0] = row * 128 + ((g4 ^ ((i16 >> 1) & 7)) << 4);
    ra[1] = row * 128 + (((4 + g4) ^ ((i16 >> 1) & 7)) << 4);
  } else {
    const int k = 8 * g4 + (i16 >> 2), sw = tr_swizzle(k);
#pragma unroll
    for (int a = 0; a < 4; ++a) ra[a] = k * 256 + (((wm * 8 + a * 2 + ((i16 & 3) >> 1)) ^ sw) << 4) + (i16 & 1) * 8;
  }
  if constexpr (!TB) {
    const int row = wn * 32 + 8 * (i16 >> 2) + (i16 & 3), f = ((row >> 1) & 1) | (((row >> 3) & 3) << 1);
    rb[0] = 2 * HALF + row * 128 + ((g4 ^ f) << 4);
    rb[1] = 2 * HALF + row * 128 + (((4 + g4) ^ f) << 4);
  } else {
    const int k = 8 * g4 + (i16 >> 2), sw = tr_swizzle(k);
#pragma unroll
    for (int b = 0; b < 2; ++b) rb[b] = 2 * HALF + k * 256 + (((wn * 4 + b * 2 + ((i16 & 3) >> 1)) ^ sw) << 4) + (i16 & 1) * 8;
  }
  unsigned st = 0;  // byte offset of the stage being consumed
  auto read_a = [&](bf16x8 (&f)[4][2], int half) {
    const unsigned char* at = smem_raw + half * HALF;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if constexpr (!TA) f[a][ks] = *reinterpret_cast<const bf16x8*>(at + (ra[ks] + st) + a * 2048);
        else f[a][ks] = pp_read_tr(at + (ra[a] + st) + ks * 8192, 1024);
      }
  };
  auto read_b = [&](bf16x8 (&f)[2][2], int half) {
    const unsigned char* at = smem_raw + half * HALF;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if constexpr (!TB) f[b][ks] = *reinterpret_cast<const bf16x8*>(at + (rb[ks] + st) + b * 512);
        else f[b][ks] = pp_read_tr(at + (rb[b] + st) + ks * 8192, 1024);
      }
  };

  // ---- loader: two 16-byte chunks per lane and half tile
  unsigned va[2][2], vb[2][2];    // byte offsets of the lane's chunks from the half's base
  const char *ba[2], *bb[2];      // wave-uniform, advanced by one K tile per request
  const int64_t step_a = TA ? 2ll * BK * p.lda : 2 * BK, step_b = TB ? 2ll * BK * p.ldb : 2 * BK;
  int T_ = 0, n_kt = 0, k_tail = 0;
  int next_slice = 0;
  int64_t next_m0 = 0, next_n0 = 0;
  int bias_buf = 0;
  auto start_tile = [&](unsigned idx) -> bool {
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));  // recomputed per tile rather than held in registers across the main loop
    const unsigned work = (blockIdx.x & 7) * per_xcd + idx;
    if (idx >= per_xcd || work >= total) return false;
    const unsigned slice = p.split_k > 1 ? work / tiles : 0;
    int tm, tn;
    tile_coords(p, (int)(work - slice * tiles), tm, tn);
    next_slice = (int)slice;
    const int64_t k_begin = (int64_t)slice * p.k_chunk;
    const int64_t k_end = p.split_k > 1 ? (k_begin + p.k_chunk < p.K ? k_begin + p.k_chunk : p.K) : p.K;
    next_m0 = (int64_t)tm * BM;
    next_n0 = (int64_t)tn * NCOLS;
    const int klen = (int)(k_end - k_begin);
    T_ = (klen + BK - 1) / BK;
    k_tail = klen % BK;
    const T* A = static_cast<const T*>(p.A);
    const int m_left = (int)(p.M - next_m0 < BM ? p.M - next_m0 : BM), n_left = (int)(p.N - next_n0 < NCOLS ? p.N - next_n0 : NCOLS);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const T* B = static_cast<const T*>(DUAL && h ? p.B2 : p.B);
      ba[h] = reinterpret_cast<const char*>(TA ? A + k_begin * p.lda + next_m0 : A + next_m0 * p.lda + k_begin);
      bb[h] = reinterpret_cast<const char*>(TB ? B + k_begin * p.ldb + next_n0 : B + next_n0 * p.ldb + k_begin);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int q = wv * 2 + j;
        if constexpr (!TA) {
          const int row = q * 8 + (l >> 3), c = (l & 7) ^ ((row >> 1) & 7);
          int r = h * 128 + row;
          if (r >= m_left) r = m_left - 1;  // rows past the edge repeat the last row: they only feed results that are not stored
          va[h][j] = (unsigned)((r * p.lda + c * 8) * 2);
        } else {
          const int k = q * 4 + (l >> 4);
          int r = h * 128 + (((l & 15) ^ tr_swizzle(k)) << 3);
          if (r >= m_left) r = 0;
          va[h][j] = (unsigned)((k * p.lda + r) * 2);
        }
        if constexpr (!TB) {
          const int row = q * 8 + (l >> 3), c = (l & 7) ^ (((row >> 1) & 1) | (((row >> 3) & 3) << 1));
          int r = DUAL ? row : (row >> 5) * 64 + h * 32 + (row & 31);
          if (r >= n_left) r = n_left - 1;
          vb[h][j] = (unsigned)((r * p.ldb + c * 8) * 2);
        } else {
          const int k = q * 4 + (l >> 4);
          int r = h * 128 + (((l & 15) ^ tr_swizzle(k)) << 3);
          if (r >= n_left) r = 0;
          vb[h][j] = (unsigned)((k * p.ldb + r) * 2);
        }
      }
    }
    return true;
  };
  // X: 0 = B half 0, 1 = A half 0, 2 = B half 1, 3 = A half 1
  auto issue = [&](auto X, unsigned stage_off, bool tail) {
    constexpr int x = decltype(X)::value, h = x >> 1;
    constexpr bool is_a = (x & 1) != 0, tr = is_a ? TA : TB;
    const char*& base = is_a ? ba[h] : bb[h];
    const unsigned(&v)[2] = is_a ? va[h] : vb[h];
    const unsigned dst = lds0 + stage_off + (is_a ? 0 : 2 * HALF) + h * HALF;
    if (tail) {  // the last, partial K tile: chunks past the end of K are zeros
      int lane = l;
      asm volatile("" : "+v"(lane));  // not to be computed ahead of this rare path
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int q = wv * 2 + j, row = q * 8 + (lane >> 3);
        const int k = tr ? q * 4 + (lane >> 4) : 8 * ((lane & 7) ^ (is_a ? (row >> 1) & 7 : ((row >> 1) & 1) | (((row >> 3) & 3) << 1)));
        pp_load_below(dst + j * 1024, v[j], base, k, k_tail);
        if (k >= k_tail) *reinterpret_cast<u32x4*>(smem_raw + (dst - lds_base) + j * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    } else {
      pp_load(dst, v[0], base);
      pp_load(dst + 1024, v[1], base);
    }
    base += is_a ? step_a : step_b;
  };
  using X0 = std::integral_constant<int, 0>;
  using X1 = std::integral_constant<int, 1>;
  using X2 = std::integral_constant<int, 2>;
  using X3 = std::integral_constant<int, 3>;
  auto issue_first = [&]() {
    if constexpr (HAS_BIAS) {  // this wave's 2 x 32 bias values as dwords: lanes 0-15 half 0, lanes 16-31 half 1
      const int h = (l >> 4) & 1;
      int64_t n = next_n0 + (DUAL ? wn * 32 : (TB ? h * 128 + wn * 32 : wn * 64 + h * 32)) + 2 * (l & 15);
      if (n > p.N - 2) n = p.N - 2;
      const T* src = static_cast<const T*>(DUAL && h ? p.bias2 : p.bias);
      bias_buf ^= 1;
      pp_load_dword_at(lds_base + PpCfg::BIAS_OFF + bias_buf * 2048 + wv * 256, reinterpret_cast<const char*>(src + n));
    }
    issue(X0{}, 0, false);
    issue(X1{}, 0, false);
    issue(X2{}, 0, false);
    issue(X3{}, 0, false);
    issue(X0{}, STAGE, false);
    issue(X1{}, STAGE, false);
  };

  f32x4 acc[8][4];  // [row block of 16: 4 per A half][2 * B half + block of 16 columns]
  bf16x8 fa[4][2], fb[2][2][2];  // A half in use; both B halves
  auto mfma = [&](auto H, auto G, const bf16x8 (&b)[2][2], auto FIRST) {
    constexpr int h = decltype(H)::value, g = decltype(G)::value;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          f32x4& c = acc[h * 4 + a][g * 2 + n];
          const f32x4 c0 = (decltype(FIRST)::value && ks == 0) ? f32x4{0.f, 0.f, 0.f, 0.f} : c;
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[n][ks], fa[a][ks], c0, 0, 0, 0);
        }
    __builtin_amdgcn_s_setprio(0);
  };
  bool do_rs = false;  // this output tile also sums A's rows
  // (a loop of their own for these tiles: the branch inside the K loop cost the other tiles up to 2 %, 6912 x 1280 over 14,336 rows 260 -> 256 us,
  // and a step of 9,600 rows 49.2 -> 48.6 ms, of 25,524 114.3 -> 113.7)
  // row block wn of the group's four in each A half, one accumulator per half: every lane's element 0 is the sum of row l % 16.
  // The first operand is ones throughout, so a row's sum reads that row alone (zeros standing for "the other half's rows" would
  // carry its infinities and NaNs over: 0 x Inf)
  [[maybe_unused]] f32x4 rs[2];
  auto row_sums = [&](auto H, auto RS) {
    if constexpr (decltype(RS)::value) {
      unsigned o = 0x3f803f80u;
      asm volatile("" : "+v"(o));  // made where it is used rather than held in registers
      const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{o, o, o, o});
#pragma unroll
      for (int a = 0; a < 4; ++a)
        if (wn == a) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            f32x4& c = rs[decltype(H)::value];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, fa[a][ks], c, 0, 0, 0);
          }
        }
    }
  };
  // K tile t.  MODE 0: steady, 1: first of the output tile, 2: last but one, 3: last
  auto ktile = [&](auto MODE_, int t, auto RS) {
    constexpr int MODE = decltype(MODE_)::value;
    constexpr int W = MODE == 1 ? (8 + TRAILING < 63 ? 8 + TRAILING : 63) : 8;
    using F = std::integral_constant<bool, MODE == 1>;
    const bool tail1 = k_tail != 0 && t + 1 == n_kt - 1, tail2 = k_tail != 0 && t + 2 == n_kt - 1;
    const unsigned other = st ^ STAGE;
    // phase 0
    read_b(fb[0], 0);
    read_a(fa, 0);
    if constexpr (MODE != 3) issue(X2{}, other, tail1);
    pp_wait_vm<MODE == 3 ? 2 : W>();
    pp_barrier();
    mfma(X0{}, X0{}, fb[0], F{});
    pp_barrier();
    // phase 1
    read_b(fb[1], 1);
    if constexpr (MODE != 3) issue(X3{}, other, tail1);
    pp_wait_vm<MODE == 3 ? 0 : W>();
    pp_barrier();
    mfma(X0{}, X1{}, fb[1], F{});
    row_sums(X0{}, RS);
    pp_barrier();
    // phase 2
    read_a(fa, 1);
    if constexpr (MODE <= 1) issue(X0{}, st, tail2);
    if constexpr (MODE != 3) pp_wait_vm<MODE == 2 ? 6 : W>();
    pp_barrier();
    mfma(X1{}, X1{}, fb[1], F{});
    pp_barrier();
    // phase 3
    if constexpr (MODE <= 1) issue(X1{}, st, tail2);
    if constexpr (MODE != 3) pp_wait_vm<MODE == 2 ? 4 : W>();
    pp_barrier();
    mfma(X1{}, X0{}, fb[0], F{});
    row_sums(X1{}, RS);
    pp_barrier();
    st = other;
  };

  unsigned idx = blockIdx.x >> 3;
  if (!start_tile(idx)) return;
  issue_first();
  pp_wait_vm<0>();
  if (wm == 1) pp_barrier();  // group 1 runs one barrier behind
  pp_barrier();
  while (true) {
    const int64_t m0 = next_m0, n0 = next_n0;
    const int slice = next_slice, bias_now = bias_buf;
    n_kt = T_;
    st = 0;
    if constexpr (ROW_SUMS) {
      do_rs = p.row_sums != nullptr && n0 == 0;
      rs[0] = rs[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    pp_wait_vm<(8 + TRAILING < 63 ? 8 + TRAILING : 63)>();
    pp_barrier();  // group 1's loads have landed as well: it waited for them before the barrier that meets this one
    auto ktiles = [&](auto RS) {
      ktile(X1{}, 0, RS);
      for (int t = 1; t < n_kt - 2; ++t) ktile(X0{}, t, RS);
      ktile(X2{}, n_kt - 2, RS);
      ktile(X3{}, n_kt - 1, RS);
    };
    if (ROW_SUMS && do_rs) ktiles(std::integral_constant<bool, ROW_SUMS>{});
    else ktiles(std::false_type{});
    idx += gridDim.x >> 3;
    const bool have = start_tile(idx);
    if (have && !HAS_IN) issue_first();
    // Group 0 meets the end of group 1's MFMAs here, not behind its own epilogue, so that both groups' epilogues run side by side (SwiGLU
    // backward: after its first half, whose sums group 1 goes on from).  One behind the other -> now, us at 25,524 rows: SwiGLU 399 -> 397, its
    // backward 337 -> 333, 1280 x 1280 with residual 80.0 -> 77.4, input gradients within 1 %; the clock takes back most of what the units gain.
    // Steps 0.3 to 0.5 % shorter: 4,096 rows checkpointed, 14,336, 25,524 and 65,536 (paired passes, +- 0.1 %).
    if (!SW_BWD && wm == 0) pp_barrier();

    // ---- epilogue: row block a of 16, half g: lane owns row l % 16 and the eight columns 8 * (l / 16) ..
    const bool to_ws = (EPI == MVIT_EPI_NONE) && p.split_k > 1;
    const bool vec = to_ws ? (p.N % 4 == 0) : p.vec_ok != 0;
    const bool interior = vec && m0 + BM <= p.M && n0 + NCOLS <= p.N;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    const int i16 = lane & 15, g4 = lane >> 4;
    const int64_t m_lane = m0 + wm * 64 + i16;
    int64_t n_lane[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) n_lane[g] = TB ? n0 + g * 128 + wn * 32 + tr_first_column(g4) : n0 + (DUAL ? wn * 32 : wn * 64 + g * 32) + 8 * g4;
    float hb[2][8];
    if constexpr (HAS_BIAS) {
      const unsigned char* bl = smem_raw + PpCfg::BIAS_OFF + bias_now * 2048 + wv * 256;
#pragma unroll
      for (int g = 0; g < 2; ++g) load8(reinterpret_cast<const bf16_t*>(bl + g * 64 + g4 * 16), hb[g]);
    }
    // SW_BWD: column sums over the lane's rows, of the eight columns' gate and up halves.  They are added in the order of gemm_dl_kernel,
    // so that the sums of 256 rows have the same bits whichever kernel made them: lane l % 16 adds rows 32 a + {0, 16, 128, 144} for
    // a = 0 .. 3, i.e. group 1 goes on from group 0's sums, and the sums of the sixteen lanes are added one after the other.
    float no_cs[16];
    const bool do_cs = SW_BWD && p.colsum != nullptr;
    // A half of group 1's epilogue lies behind a barrier that group 0 arrives at after the same half of its own, so it finds group 0's sums
    // there.  Chunks of four sums, chunk c of lane i in slot c ^ i: stores of sixteen lanes, and loads of one chunk of each, fall on all banks.
    float* cs_lds = reinterpret_cast<float*>(smem_raw + PpCfg::BIAS_OFF) + wn * 2048;
    auto chunk_of = [&](int g, int h) { return reinterpret_cast<f32x4*>(cs_lds + g * 1024 + i16 * 64 + ((g4 * 4 + h) ^ i16) * 4); };
    auto begin_sums = [&](int g) {
      if constexpr (SW_BWD) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const f32x4 t = do_cs && wm == 1 ? *chunk_of(g, h) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) no_cs[4 * h + e] = t[e];
        }
      }
    };
    auto end_sums = [&](int g) {
      if constexpr (SW_BWD) {
#pragma unroll
        for (int h = 0; h < 4; ++h) *chunk_of(g, h) = f32x4{no_cs[4 * h], no_cs[4 * h + 1], no_cs[4 * h + 2], no_cs[4 * h + 3]};
        if (wm == 0) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // before this group's next barrier
        } else {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          float t = 0.f;
#pragma unroll
          for (int k = 0; k < 16; ++k) t += cs_lds[g * 1024 + k * 64 + (((lane >> 2) ^ k) << 2) + (lane & 3)];
          const int64_t n = n0 + g * 128 + wn * 32 + tr_first_column(g4) + (lane & 7);
          if (n < p.N) p.colsum[m0 / BM * p.ldc + (lane & 8 ? p.aux_off : 0) + n] = t;
        }
      }
    };
    float* ws = to_ws ? p.workspace + (int64_t)slice * p.M * p.N : nullptr;
    constexpr int NG = DUAL ? 1 : 2, ITEMS = 8 * NG;
    // item -> row block and column half: by rows, or all rows of a half first, in the order of their sums
    auto block_of = [](int it) { return SW_BWD ? (it & 1) | ((it & 2) << 1) | ((it & 4) >> 1) : it / NG; };
    auto half_of = [](int it) { return SW_BWD ? it >> 3 : it % NG; };
    auto row_of = [&](int it) { return m_lane + (block_of(it) >> 2) * 128 + (block_of(it) & 3) * 16; };
    auto values = [&](int it, float (&v)[8], float (&u)[8]) {
      const int a = block_of(it), g = half_of(it);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[a][2 * g][e];
        v[4 + e] = acc[a][2 * g + 1][e];
        if (TB) tr_columns(v[e], v[4 + e]);
        if (DUAL) {
          u[e] = acc[a][2][e];
          u[4 + e] = acc[a][3][e];
        }
      }
    };
    if constexpr (ROW_SUMS) {
      if (do_rs) {
        const int64_t m = m_lane + (g4 >> 1) * 128 + wn * 16;
        if ((g4 & 1) == 0 && m < p.M) {  // stores that the next tile's waits do not count only make them wait for more
          const float sum = g4 >> 1 ? rs[1][0] : rs[0][0];
          if (to_ws) p.row_ws[(int64_t)slice * p.M + m] = sum;
          else static_cast<TO*>(p.row_sums)[m] = from_f32<TO>(sum);
        }
      }
    }
    if (interior) {
      if constexpr (HAS_IN) {
        // the input was written a few launches ago and is often still in the memory-side cache: a plain load finds it there
        // (25,524 x 1280 x 1280 with residual: 98 us with non-temporal loads, 83 us with plain ones)
        bf16x8 pre[DEPTH][NIN];
        auto fetch = [&](int it, bf16x8 (&to)[NIN]) {
          const T* r = static_cast<const T*>(p.R) + row_of(it) * p.ldr + n_lane[half_of(it)];
          to[0] = *reinterpret_cast<const bf16x8*>(r);
          if constexpr (SW_BWD) to[1] = *reinterpret_cast<const bf16x8*>(r + p.aux_off);
        };
#pragma unroll
        for (int it = 0; it < DEPTH; ++it) fetch(it, pre[it]);
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
          if ((it & 7) == 0) begin_sums(it >> 3);
          float v[8], u[8];
          values(it, v, u);
          bf16x8 now[NIN];
#pragma unroll
          for (int i = 0; i < NIN; ++i) now[i] = pre[it % DEPTH][i];
          if (it + DEPTH < ITEMS) fetch(it + DEPTH, pre[it % DEPTH]);
          if (it == ITEMS - DEPTH && have) issue_first();  // behind the last of this tile's input loads
          emit8_impl<T, TO, EPI, true, true>(p, row_of(it), n_lane[half_of(it)], v, u, now, no_cs, do_cs, HAS_BIAS ? hb[half_of(it)] : nullptr, nullptr);
          if (do_cs && (it & 7) == 7) end_sums(it >> 3);
          __builtin_amdgcn_sched_barrier(0);
          if (SW_BWD && it == 7) pp_barrier();
        }
      } else {
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
          float v[8], u[8];
          values(it, v, u);
          if (to_ws) store8(ws + row_of(it) * p.N + n_lane[half_of(it)], v);
          else emit8_impl<T, TO, EPI, true, false>(p, row_of(it), n_lane[half_of(it)], v, u, nullptr, no_cs, false, HAS_BIAS ? hb[half_of(it)] : nullptr, HAS_BIAS && DUAL ? hb[1] : nullptr);
        }
      }
    } else {
      if (have && HAS_IN) issue_first();
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {
        if (do_cs && it == 8) end_sums(0);
        if (SW_BWD && it == 8) pp_barrier();
        if ((it & 7) == 0) begin_sums(it >> 3);
        float v[8], u[8];
        values(it, v, u);
        const int64_t m = row_of(it), n = n_lane[half_of(it)];
        if (m >= p.M || n >= p.N) continue;
        if (to_ws) {
          float* w = ws + m * p.N + n;
          if (vec && n + 8 <= p.N) store8(w, v);
          else
            for (int e = 0; e < 8 && n + e < p.N; ++e) w[e] = v[e];
        } else if (vec && n + 8 <= p.N) {
          emit8_impl<T, TO, EPI, true>(p, m, n, v, u, nullptr, no_cs, do_cs, HAS_BIAS ? hb[half_of(it)] : nullptr, HAS_BIAS && DUAL ? hb[1] : nullptr);
        } else {
          emit8<T, TO, EPI>(p, m, n, v, u, false, no_cs, do_cs);
        }
      }
      if (do_cs) end_sums(NG - 1);
      pp_wait_vm<0>();  // the count of this path's memory instructions is not known to the waits of the next tile
    }
    if (SW_BWD && wm == 0) pp_barrier();
    if (!have) break;
    if (wm == 1) {  // its share of the next tile's first half tiles, for group 0
      pp_wait_vm<(8 + TRAILING < 63 ? 8 + TRAILING : 63)>();
      pp_barrier();
    }
  }
}

}  // namespace

int mvit_gemm_pp(GemmTiledKind kind, const GemmParams& p, int n_cu, hipStream_t stream) {
  auto go = [&](auto kern, bool (&attr_set_on)[MVIT_MAX_DEVICES], int lds = PpCfg::lds(MVIT_EPI_NONE)) -> int {
    const int dev = mvit_current_device("gemm");
    if (dev < 0) return MVIT_ERR_LAUNCH;
    if (!attr_set_on[dev]) {  // dynamic LDS above 64 KiB is opted into once per kernel and device
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return mvit_set_error(MVIT_ERR_LAUNCH, "gemm: hipFuncSetAttribute(%d B LDS): %s", lds, hipGetErrorString(e));
      attr_set_on[dev] = true;
    }
    const int want = (p.tiles_m * p.tiles_n * p.split_k + 7) / 8 * 8;
    hipLaunchKernelGGL(kern, want < n_cu ? want : n_cu, PpCfg::NTHREADS, lds, stream, p);
    MVIT_CHECK_LAUNCH("gemm");
    return MVIT_OK;
  };
  static bool set[10][MVIT_MAX_DEVICES] = {};
  switch (kind) {
    case NN_NONE: return go(gemm_pp_kernel<bf16_t, false, false, MVIT_EPI_NONE>, set[0]);
    case NN_BIAS: return go(gemm_pp_kernel<bf16_t, false, false, MVIT_EPI_BIAS>, set[1]);
    case NN_BIAS_RES: return go(gemm_pp_kernel<bf16_t, false, false, MVIT_EPI_BIAS_RES>, set[2]);
    case NN_BIAS_GELU: return go(gemm_pp_kernel<bf16_t, false, false, MVIT_EPI_BIAS_GELU>, set[3]);
    case NN_SWIGLU: return go(gemm_pp_kernel<bf16_t, false, false, MVIT_EPI_SWIGLU>, set[4]);
    case NT_NONE: return go(gemm_pp_kernel<bf16_t, false, true, MVIT_EPI_NONE>, set[5]);
    case NT_GELU_BWD: return go(gemm_pp_kernel<bf16_t, false, true, MVIT_EPI_GELU_BWD>, set[6]);
    case NT_SWIGLU_BWD: return go(gemm_pp_kernel<bf16_t, false, true, MVIT_EPI_SWIGLU_BWD>, set[9], PpCfg::lds(MVIT_EPI_SWIGLU_BWD));
    case TT_NONE: return go(gemm_pp_kernel<bf16_t, true, true, MVIT_EPI_NONE>, set[7]);
    case TT_NONE_F32: return go(gemm_pp_kernel<float, true, true, MVIT_EPI_NONE>, set[8]);
    default: return mvit_set_error(MVIT_ERR_UNSUPPORTED, "gemm: product kind %d has no 256 x 256 ping-pong kernel", (int)kind);
  }
}
