// Decoded RGB frames (uint8) -> rows of pixel_values for gfx950: rescale, normalise and cut into 14x14x2 patches in
// the row order the vision tower expects, for a whole batch of images and videos in one launch.  HBM-bound: every
// output row is 1176 values (4704 bytes in fp32) made from 2 x 588 input bytes (588 for a still image, whose one
// frame fills both halves).  A work-group makes the four rows of a 2x2 merge block, one wave per row: it stages
// the block's 28x28 pixel square (28 lines of 84 bytes = 21 aligned dwords) in LDS with dword loads, a lane takes four
// pixels of it with all three channels (two pairs of dwords, twelve lookups in a table that holds the output type), and the output
// leaves as 16-byte (fp32) or 8-byte (bf16) stores.  The next square's loads travel meanwhile.  Bound by the writes to HBM.
// us, before (a lane took four values of one channel from single bytes, loads waited for) / now: four images of 896 x 896 bf16 15.3 / 14.4, 8 frames
// of 448 x 784 10.3 / 9.3, 3,584 x 3,584 bf16 43.3 / 41.9, fp32 93 - 102 / 87 - 91; grids of 1,024 / 2,048 / 4,096 work-groups 44.3 / 43.9 / 41.9 there.
//
// The arithmetic is that of the image processor the reference calls (transformers 4.57.0,
// Qwen2VLImageProcessor._preprocess: rescale in float64 rounded to float32, then (x - mean) / std in float32
// with an IEEE division), so fp32 results can be compared bit for bit with a numpy restatement.
#include "mvit_common.h"
#include <string.h>
#include <type_traits>

namespace {

constexpr int PATCH = 14, TPS = 2, ROW = MVIT_PIXEL_ROW;
constexpr int PLANE = PATCH * PATCH;   // 196 values of one (channel, frame) plane of a row
constexpr int QUADS = PLANE / 4;       // 49 groups of four consecutive values per plane

struct Norm {
  double rescale;
  float mean[3], std[3];
};

__device__ __forceinline__ int find_image(const mvit_image* t, int n, int64_t row) {
  int lo = 0, hi = n;  // invariant: t[lo].first_row <= row < t[hi].first_row
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (t[mid].first_row <= row) lo = mid;
    else hi = mid;
  }
  return lo;
}

template <typename T>
using quad_t = T __attribute__((ext_vector_type(4)));

constexpr int PATCHIFY_GROUPS = 4096;
constexpr int SQ = 2 * PATCH;          // a merge block is a square of 28 x 28 pixels
constexpr int SQ_LINE = SQ * 3;        // 84 bytes (21 dwords) per line of the square
constexpr int SQ_DWORDS = SQ * SQ_LINE / 4;  // 588

// The result for every byte value and channel, by the work-group (exact arithmetic, three divisions per thread)
template <typename TO>
__device__ __forceinline__ void make_lut(TO (&lut)[3][256], const Norm& nm) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float x = (float)((double)(int)threadIdx.x * nm.rescale);
    lut[c][threadIdx.x] = from_f32<TO>((x - nm.mean[c]) / nm.std[c]);
  }
}
// A wave makes one patch of the square, a lane four consecutive values of each plane: two pairs of pixels, six bytes each at even
// addresses, the second pair on the line below where the first ends one.
struct PatchLane {
  int q, pair0, pair1;
};
__device__ __forceinline__ PatchLane patch_lane() {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int q = lane < QUADS ? lane : 0, y = 4 * q / PATCH, x = 4 * q - y * PATCH;
  const int origin = (wave >> 1) * PATCH * SQ_LINE + (wave & 1) * PATCH * 3, pair0 = origin + y * SQ_LINE + x * 3;
  return {q, pair0, x + 2 < PATCH ? pair0 + 6 : origin + (y + 1) * SQ_LINE};
}
template <typename TO>
__device__ __forceinline__ void look_up(const uint32_t* square, const TO (&lut)[3][256], const PatchLane& pl, TO (&v)[3][4]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = h ? pl.pair1 : pl.pair0;
    const uint32_t *w = &square[at >> 2], w0 = w[0], w1 = w[1], lo = __builtin_amdgcn_alignbyte(w1, w0, at & 2), hi = w1 >> (8 * (at & 2));
    const uint32_t b[6] = {lo & 0xff, (lo >> 8) & 0xff, (lo >> 16) & 0xff, lo >> 24, hi & 0xff, (hi >> 8) & 0xff};
#pragma unroll
    for (int e = 0; e < 6; ++e) v[e % 3][2 * h + e / 3] = lut[e % 3][b[e]];
  }
}
template <typename TO>
__device__ __forceinline__ void store_patch(TO* row, int frame, const PatchLane& pl, const TO (&v)[3][4]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) *reinterpret_cast<quad_t<TO>*>(row + (c * TPS + frame) * PLANE + 4 * pl.q) = quad_t<TO>{v[c][0], v[c][1], v[c][2], v[c][3]};
}

// The image table travels as a kernel argument when it is short (no copy to the device in front of the launch).
constexpr int TABLE_ARG_IMAGES = 64;
struct TableArg {
  mvit_image im[TABLE_ARG_IMAGES + 1];
};
template <typename TO>
__device__ __forceinline__ void patchify_blocks(const mvit_image* images, int n_images, TO* __restrict__ out, int64_t total_rows, const Norm& nm) {
  // a byte has 256 values: the work-group computes the result for each of them and each channel once, and every element of its rows
  // is then a byte and a table lookup
  __shared__ TO lut[3][256];
  __shared__ __attribute__((aligned(16))) uint32_t square[TPS][SQ_DWORDS];  // the block's pixels, one copy per frame of the pair
  constexpr int LOADS = (TPS * SQ_DWORDS + 255) / 256;                       // dwords of the square per thread
  struct Block {
    const uint8_t* corner;  // of the square in the block's first frame; null: malformed entry, nothing is read or written
    int64_t line, second;   // bytes to the next line and to the second frame
    bool two;               // a still image's one frame fills both halves
  };
  // the same for the whole work-group: its four rows are one merge block
  auto locate = [&](int64_t row0) {
    const mvit_image im = images[find_image(images, n_images, row0)];
    const int gh = im.height / PATCH, gw = im.width / PATCH;
    const int per_t = gh * gw;
    const int64_t local = (row0 - im.first_row) & ~(int64_t)3;
    bool ok = im.frames > 0 && gh > 0 && gw > 0 && !((gh | gw) & 1);
    const int t = ok ? (int)(local / per_t) : 0, rem = ok ? (int)(local % per_t) : 0;
    ok = ok && t * TPS < im.frames;  // first_row entries that promise more rows than the frames give
    // rem = ((block row * (gw / 2) + block column) * 2 + row in block) * 2 + column in block
    const int blk = rem >> 2, hb = ok ? blk / (gw >> 1) : 0, wb = ok ? blk % (gw >> 1) : 0;
    const int64_t line = (int64_t)im.width * 3, frame_bytes = line * im.height;
    const int f0 = t * TPS, f1 = f0 + 1 < im.frames ? f0 + 1 : im.frames - 1;  // the last frame fills an odd count up
    return Block{ok ? im.pixels + f0 * frame_bytes + (int64_t)hb * SQ * line + wb * SQ_LINE : nullptr, line, frame_bytes, f1 != f0};
  };
  // width is a multiple of 28, so lines are a multiple of 84 bytes: with a 4-byte aligned frame buffer every line of the square is
  // 21 aligned dwords.  They are requested while the block before is worked on.
  auto in_dwords = [](const Block& b) { return (reinterpret_cast<uintptr_t>(b.corner) & 3u) == 0; };
  uint32_t held[LOADS];
  auto request = [&](const Block& b) {
    if (b.corner == nullptr || !in_dwords(b)) return;
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int i = k * 256 + threadIdx.x, fi = i / SQ_DWORDS, j = i % SQ_DWORDS, y = j / (SQ_LINE / 4), xw = j % (SQ_LINE / 4);
      if (i < (b.two ? TPS : 1) * SQ_DWORDS) held[k] = *reinterpret_cast<const uint32_t*>((fi ? b.corner + b.second : b.corner) + (unsigned)(y * (int)b.line + xw * 4));
    }
  };
  auto put = [&](const Block& b) {
    const int n = (b.two ? TPS : 1) * SQ_DWORDS;
    if (in_dwords(b)) {
#pragma unroll
      for (int k = 0; k < LOADS; ++k)
        if (k * 256 + (int)threadIdx.x < n) (&square[0][0])[k * 256 + threadIdx.x] = held[k];
    } else {
      uint8_t* sq8 = reinterpret_cast<uint8_t*>(&square[0][0]);
#pragma unroll 1
      for (int i = threadIdx.x; i < n * 4; i += 256) {
        const int fi = i / (SQ_DWORDS * 4), j = i % (SQ_DWORDS * 4), y = j / SQ_LINE, xb = j % SQ_LINE;
        sq8[i] = (fi ? b.corner + b.second : b.corner)[(unsigned)(y * (int)b.line + xb)];
      }
    }
  };

  // merge blocks blockIdx.x, blockIdx.x + gridDim.x, ...: the table is made once for all of them
  const int64_t stride = (int64_t)gridDim.x * 4;
  int64_t row0 = (int64_t)blockIdx.x * 4;
  if (row0 >= total_rows) return;
  Block now = locate(row0);
  request(now);
  make_lut<TO>(lut, nm);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const PatchLane pl = patch_lane();
  while (true) {
    __syncthreads();  // the previous block's pixels have been read
    if (now.corner != nullptr) put(now);
    __syncthreads();  // the table and the pixels are complete
    const int64_t next = row0 + stride;
    Block then{};
    if (next < total_rows) {
      then = locate(next);
      request(then);
    }
    if (now.corner != nullptr && lane < QUADS) {
      TO* dst = out + (row0 + wave) * ROW;
      TO v[3][4];
      look_up<TO>(&square[0][0], lut, pl, v);
      store_patch<TO>(dst, 0, pl, v);
      if (now.two) look_up<TO>(&square[1][0], lut, pl, v);
      store_patch<TO>(dst, 1, pl, v);
    }
    if (next >= total_rows) return;
    row0 = next;
    now = then;
  }
}
template <typename TO>
__global__ __launch_bounds__(256) void patchify_kernel(const mvit_image* __restrict__ images, int n_images, TO* __restrict__ out, int64_t total_rows, Norm nm) {
  patchify_blocks<TO>(images, n_images, out, total_rows, nm);
}
template <typename TO>
__global__ __launch_bounds__(256) void patchify_arg_kernel(const TableArg images, int n_images, TO* __restrict__ out, int64_t total_rows, Norm nm) {
  patchify_blocks<TO>(images.im, n_images, out, total_rows, nm);
}

}  // namespace
// A window as the kernels use it: first tap and tap count forced into the table's row (ksize entries) and into the
// input axis, so that a table that breaks the entry point's contract cannot make a kernel read outside its arrays.
struct TapWindow {
  int xmin, n;
};
__device__ __forceinline__ TapWindow tap_window(const int32_t* __restrict__ bounds, int64_t x, int ksize, int64_t in_len) {
  int xmin = bounds[2 * x], n = bounds[2 * x + 1];
  xmin = max(0, min(xmin, (int)in_len - 1));
  n = max(0, min(n, min(ksize, (int)in_len - xmin)));
  return {xmin, n};
}


// ------------------------------------------------------------------------------------------------
// One resampling pass along the middle axis of a uint8 array [outer][in_len][inner] -> [outer][out_len][inner], with
// Pillow's 8-bit arithmetic (libImaging/Resample.c, ImagingResampleHorizontal_8bpc / Vertical_8bpc): per output
// coordinate a window of `bounds[2*x + 1]` input coordinates starting at `bounds[2*x]`, 22-bit fixed-point weights
// kk[x * ksize + i], an accumulator that starts at one half, an arithmetic shift and a clamp to 0..255.
// inner is the contiguous dimension: pixels times channels for the vertical pass, 3 channels for the horizontal one.  The
// kernels for those two follow; resample_pass_kernel takes everything else.
constexpr int RESAMPLE_PRECISION_BITS = 22;
__device__ __forceinline__ unsigned clip8(int v) {
  v >>= RESAMPLE_PRECISION_BITS;
  // keeps the compiler from pairing shift and clamp into v_ashr_pk_u8_i32: it takes the upper half of that instruction's result
  // for zero, and the hardware leaves the old bits there
  asm("" : "+v"(v));
  return (unsigned)(v < 0 ? 0 : (v > 255 ? 255 : v));
}
// A thread makes four consecutive output bytes: of one output coordinate where inner is a multiple of four and the arrays are
// made of aligned words (WORDS), else of the flattened [out_len * inner] row, each byte with its own window.
template <bool WORDS>
__global__ __launch_bounds__(256) void resample_pass_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int64_t outer,
                                                            int64_t in_len, int64_t out_len, int64_t inner,
                                                            const int32_t* __restrict__ bounds, const int32_t* __restrict__ kk, int ksize) {
  const int64_t row_out = out_len * inner, row_in = in_len * inner, quads = (row_out + 3) / 4, total = outer * quads;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t o = i / quads, first = i % quads * 4;
    const uint8_t* s = src + o * row_in;
    uint8_t* d = dst + o * row_out + first;
    int64_t x = first / inner, c = first % inner;
    if constexpr (WORDS) {
      const TapWindow tw = tap_window(bounds, x, ksize, in_len);
      const int32_t* k = kk + x * ksize;
      int a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = 1 << (RESAMPLE_PRECISION_BITS - 1);
      for (int t = 0; t < tw.n; ++t) {
        const unsigned w = *reinterpret_cast<const unsigned*>(s + (int64_t)(tw.xmin + t) * inner + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] += (int)((w >> (8 * e)) & 0xffu) * k[t];
      }
      *reinterpret_cast<unsigned*>(d) = clip8(a[0]) | (clip8(a[1]) << 8) | (clip8(a[2]) << 16) | (clip8(a[3]) << 24);
    } else {
      const int n_bytes = row_out - first < 4 ? (int)(row_out - first) : 4;
      for (int e = 0; e < n_bytes; ++e) {
        const TapWindow tw = tap_window(bounds, x, ksize, in_len);
        const int32_t* k = kk + x * ksize;
        int a = 1 << (RESAMPLE_PRECISION_BITS - 1);
        for (int t = 0; t < tw.n; ++t) a += (int)s[(int64_t)(tw.xmin + t) * inner + c] * k[t];
        d[e] = (uint8_t)clip8(a);
        if (++c == inner) {
          c = 0;
          ++x;
        }
      }
    }
  }
}

// ---- several passes in one launch
constexpr int RESAMPLE_MAX_JOBS = 32;
struct ResampleJobs {
  int n, rows_per_wave;  // the latter of resample_narrow_lds_kernel and resample_matrix_kernel
  int first_block[RESAMPLE_MAX_JOBS];
  mvit_resample_job job[RESAMPLE_MAX_JOBS];
};
__device__ __forceinline__ int resample_job_of(const ResampleJobs& jobs, int block) {
  int j = 0;
  while (j + 1 < jobs.n && block >= jobs.first_block[j + 1]) ++j;
  return j;
}
// A weight that fits 24 bits is multiplied with one full-rate multiply-add (v_mad_i32_i24); the 22-bit weights of a
// resampling always do, tables of the caller's own need not.  The low 32 bits are the same either way.
__device__ __forceinline__ bool fits24(int k) { return k < (1 << 23) && k >= -(1 << 23); }
template <bool FAST>
__device__ __forceinline__ int tap(int acc, unsigned byte, int k) {
  return acc + (int)byte * (FAST ? (int)((unsigned)k << 8) >> 8 : k);  // the shifts tell the compiler that 24 bits suffice
}

// The pass for a short contiguous dimension (the horizontal pass: inner = channels).  A wave makes 64 consecutive output
// coordinates of RESAMPLE_ROWS rows: a thread holds 16 weights of its window in registers at a time and applies them to every
// row, whose 16 taps are INNER unaligned 16-byte loads (neighbouring windows overlap and are served by the L1), so there is no
// staging and no barrier.  Bound by the multiply-adds and by the L1; with full-width multiplies (16 cycles each) and single
// bytes from LDS the four photographs of 1080 x 1920 ... 2448 x 3264 took 300 us.
constexpr int RESAMPLE_ROWS = 8, RESAMPLE_TAPS = 16, RESAMPLE_MAX_CHANNELS = 4;
template <int INNER, bool FAST>
__device__ __forceinline__ void resample_narrow_rows(const uint8_t* p, int64_t row_in, int rows, const uint8_t* src_end, const int (&k)[RESAMPLE_TAPS],
                                                     int (&acc)[RESAMPLE_ROWS][INNER]) {
  typedef __attribute__((address_space(1))) const uint8_t* global_bytes;
#pragma unroll
  for (int r = 0; r < RESAMPLE_ROWS; ++r) {
    if (r >= rows) break;
    const uint8_t* q = p + r * row_in;
    unsigned w[4 * INNER];
    if (q + RESAMPLE_TAPS * INNER <= src_end) {
#pragma unroll
      for (int i = 0; i < INNER; ++i) __builtin_memcpy(w + 4 * i, (global_bytes)(uintptr_t)(q + 16 * i), 16);
    } else {  // the end of the array: only the bytes that belong to it
#pragma unroll
      for (int i = 0; i < 4 * INNER; ++i) {
        w[i] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (q + 4 * i + e < src_end) w[i] |= (unsigned)q[4 * i + e] << (8 * e);
      }
    }
#pragma unroll
    for (int t = 0; t < RESAMPLE_TAPS; ++t)
#pragma unroll
      for (int c = 0; c < INNER; ++c) acc[r][c] = tap<FAST>(acc[r][c], (w[(t * INNER + c) / 4] >> (8 * ((t * INNER + c) & 3))) & 0xffu, k[t]);
  }
}
template <int INNER>
__global__ __launch_bounds__(256) void resample_narrow_kernel(const ResampleJobs jobs) {
  const int j = resample_job_of(jobs, blockIdx.x);
  const mvit_resample_job& jb = jobs.job[j];
  const int block = blockIdx.x - jobs.first_block[j], lane = threadIdx.x & 63;
  const int in_len = (int)jb.in_len, out_len = (int)jb.out_len, ksize = jb.ksize;
  const int xblocks = (out_len + 63) / 64, xb = block % xblocks;
  const int64_t o0 = ((int64_t)(block / xblocks) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RESAMPLE_ROWS;
  if (o0 >= jb.outer) return;
  const int rows = jb.outer - o0 < RESAMPLE_ROWS ? (int)(jb.outer - o0) : RESAMPLE_ROWS;
  const bool mine = xb * 64 + lane < out_len;
  const int x = mine ? xb * 64 + lane : out_len - 1;
  const int64_t row_in = (int64_t)in_len * INNER, row_out = (int64_t)out_len * INNER;
  const uint8_t* src_end = jb.src + jb.outer * row_in;
  const TapWindow tw = tap_window(jb.bounds, x, ksize, in_len);
  int acc[RESAMPLE_ROWS][INNER];
#pragma unroll
  for (int r = 0; r < RESAMPLE_ROWS; ++r)
#pragma unroll
    for (int c = 0; c < INNER; ++c) acc[r][c] = 1 << (RESAMPLE_PRECISION_BITS - 1);
  for (int t0 = 0; t0 < ksize; t0 += RESAMPLE_TAPS) {
    if (!__any(t0 < tw.n)) break;
    int k[RESAMPLE_TAPS];
    bool narrow = true;
#pragma unroll
    for (int t = 0; t < RESAMPLE_TAPS; ++t) {
      k[t] = t0 + t < tw.n ? jb.kk[(int64_t)x * ksize + t0 + t] : 0;  // taps past the window have weight 0
      narrow = narrow && fits24(k[t]);
    }
    const uint8_t* p = jb.src + o0 * row_in + (int64_t)(tw.xmin + (t0 < tw.n ? t0 : 0)) * INNER;
    if (__all(narrow)) resample_narrow_rows<INNER, true>(p, row_in, rows, src_end, k, acc);
    else resample_narrow_rows<INNER, false>(p, row_in, rows, src_end, k, acc);
  }
  // four pixels of three channels leave as three words, each made by one lane from its own and its neighbour's bytes
  const bool words = INNER == 3 && out_len % 4 == 0 && (reinterpret_cast<uintptr_t>(jb.dst) & 3u) == 0;
#pragma unroll
  for (int r = 0; r < RESAMPLE_ROWS; ++r) {
    if (r >= rows) break;
    uint8_t* d = jb.dst + (o0 + r) * row_out;
    if (words) {
      const unsigned v = clip8(acc[r][0]) | (clip8(acc[r][INNER > 1 ? 1 : 0]) << 8) | (clip8(acc[r][INNER > 2 ? 2 : 0]) << 16);
      const unsigned next = __shfl_down(v, 1, 64);
      const int q = lane & 3;
      if (mine && q < 3) *reinterpret_cast<unsigned*>(d + (x - q) * 3 + 4 * q) = (v >> (8 * q)) | (next << (24 - 8 * q));
    } else if (mine) {
#pragma unroll
      for (int c = 0; c < INNER; ++c) d[(int64_t)x * INNER + c] = (uint8_t)clip8(acc[r][c]);
    }
  }
}

// The same pass where a wave's 64 windows span at most NARROW_SPAN bytes of a row (three channels shrunk up to fivefold) and have
// at most NARROW_TAPS taps.  Those bytes (the windows overlap) come in one coalesced 16-byte load per lane and row, through a
// piece of LDS of the wave's own, so there is no barrier; a thread then reads its window as aligned words and shifts it into
// place.  Windows loaded from memory, 16 unaligned bytes per lane, keep the address units busy (75 % of the time, one access per
// lane).  Four taps of a channel are one 8-bit dot product per digit: a weight is three signed digits of 8 bits, a pixel is taken
// less 128 (one exclusive or on the way into LDS), and 128 times the sum of the weights is added back.  Whole numbers modulo 2^32
// throughout, so the sums are those of plain multiply-adds.  us by the kernel above / this one: four photographs of 1,080 x 1,920 ...
// 2,448 x 3,264 to 0.8 million pixels each 42.6 / 28.1, 4,480 x 4,480 to 3,584 x 3,584 124 / 57, 480 x 640 to 0.2 million 11.0 / 8.7;
// what bounds it now is vector issue (a row of 64 outputs: 63 instructions at 8 taps, 99 at 16, and 18 to store it).
constexpr int NARROW_SPAN = 1024, NARROW_TAPS = 24, NARROW_BATCH = 2, NARROW_SLACK = NARROW_TAPS * RESAMPLE_MAX_CHANNELS + 16;  // a window's padding reads past its row
__device__ __forceinline__ bool fits_digits(int k) { return k <= 0x7f7f7f && k >= -0x808080; }
// bytes first, first + step, first + 2 step, first + 3 step of the consecutive words w
template <int STEP, int N>
__device__ __forceinline__ unsigned gather_bytes(const unsigned (&w)[N], int first) {
  if constexpr (STEP == 1) {
    return w[first / 4];
  } else {
    auto pair = [&](int i, int j) {  // bytes i and j in the lower half
      const int lo = i / 4, hi = j / 4;
      return __builtin_amdgcn_perm(w[hi], w[lo], 0x0c0c0000u | (unsigned)((j % 4 + 4) << 8) | (unsigned)(i % 4));
    };
    if (first / 4 + 1 >= (first + 2 * STEP) / 4 && STEP < 4) {  // the first three lie in two neighbouring words
      const int lo = first / 4, hi = (first + 3 * STEP) / 4, mid = (first + 2 * STEP) / 4;
      auto sel = [&](int b) { return (unsigned)(b / 4 == lo ? b % 4 : b % 4 + 4); };
      const unsigned three = __builtin_amdgcn_perm(w[mid], w[lo], sel(first) | sel(first + STEP) << 8 | sel(first + 2 * STEP) << 16 | 0x0c000000u);
      return __builtin_amdgcn_perm(w[hi], three, 0x00020100u | (unsigned)((first + 3 * STEP) % 4 + 4) << 24);
    }
    if ((first + STEP) / 4 + 1 >= (first + 3 * STEP) / 4 && STEP < 4) {  // the last three do
      const int lo = (first + STEP) / 4, hi = (first + 3 * STEP) / 4;
      auto sel = [&](int b) { return (unsigned)(b / 4 == lo ? b % 4 : b % 4 + 4); };
      const unsigned three = __builtin_amdgcn_perm(w[hi], w[lo], sel(first + STEP) << 8 | sel(first + 2 * STEP) << 16 | sel(first + 3 * STEP) << 24 | 0x0cu);
      return __builtin_amdgcn_perm(w[first / 4], three, 0x03020100u | (unsigned)(first % 4 + 4));
    }
    return __builtin_amdgcn_perm(pair(first + 2 * STEP, first + 3 * STEP), pair(first, first + STEP), 0x05040100u);
  }
}
// Output coordinate `x` of every staged row from GROUPS groups of four taps; at: byte offset of the window from the row's first
// staged byte; digit: the groups' digits of the lane's weights, 64 lanes apart, and behind them the sums of the weights
template <int INNER, int GROUPS, typename Emit>
__device__ __forceinline__ void resample_narrow_digits(const unsigned char* lds, int at, uintptr_t start, int64_t row_in, int rows,
                                                       const unsigned (*dig)[4][64], int lane, Emit emit) {
  unsigned digit[GROUPS][3], total = 0;
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
#pragma unroll
    for (int d = 0; d < 3; ++d) digit[g][d] = dig[g][d][lane];
    total += dig[g][3][lane];
  }
  total = total * 128 + (1u << (RESAMPLE_PRECISION_BITS - 1));
#pragma unroll 2
  for (int r = 0; r < rows; ++r) {
    const int b = r * NARROW_SPAN + at + (int)((start + r * row_in) & 15);
    const unsigned* q = reinterpret_cast<const unsigned*>(lds + (b & ~3));
    unsigned raw[GROUPS * INNER + 1], w[GROUPS * INNER];
#pragma unroll
    for (int i = 0; i <= GROUPS * INNER; ++i) raw[i] = q[i];
#pragma unroll
    for (int i = 0; i < GROUPS * INNER; ++i) w[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], b);
    unsigned out[INNER];
#pragma unroll
    for (int c = 0; c < INNER; ++c) {
      int sum[3] = {(int)total, 0, 0};
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        const unsigned four = gather_bytes<INNER>(w, g * 4 * INNER + c);
#pragma unroll
        for (int d = 0; d < 3; ++d) sum[d] = __builtin_amdgcn_sdot4((int)four, (int)digit[g][d], sum[d], false);
      }
      out[c] = clip8((int)((unsigned)sum[0] + ((unsigned)sum[1] << 8) + ((unsigned)sum[2] << 16)));
    }
    emit(r, out);
  }
}
template <int INNER>
__global__ __launch_bounds__(256, 5) void resample_narrow_lds_kernel(const ResampleJobs jobs) {
  const int j = resample_job_of(jobs, blockIdx.x);
  const mvit_resample_job& jb = jobs.job[j];
  const int block = blockIdx.x - jobs.first_block[j], lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int in_len = (int)jb.in_len, out_len = (int)jb.out_len, ksize = jb.ksize;
  const int xblocks = (out_len + 63) / 64, xb = block % xblocks;
  const bool mine = xb * 64 + lane < out_len;
  const int x = mine ? xb * 64 + lane : out_len - 1;
  const int64_t row_in = (int64_t)in_len * INNER, row_out = (int64_t)out_len * INNER;
  const int64_t o0 = ((int64_t)(block / xblocks) * 4 + wave) * jobs.rows_per_wave;
  const int rows = o0 >= jb.outer ? 0 : (jb.outer - o0 < jobs.rows_per_wave ? (int)(jb.outer - o0) : jobs.rows_per_wave);
  const int32_t* __restrict__ kk = jb.kk + (int64_t)x * ksize;
  const TapWindow tw = tap_window(jb.bounds, x, ksize, in_len);
  // the bytes of a row from the first output's window to the last one's; windows out of that order go tap by tap
  const int first = __builtin_amdgcn_readlane(tw.xmin, 0), last = __builtin_amdgcn_readlane(tw.xmin + tw.n, 63);
  const int span = (last - first) * INNER;
  bool fits = tw.xmin >= first && tw.xmin + tw.n <= last && tw.n <= NARROW_TAPS && span + 15 <= NARROW_SPAN;

  __shared__ __attribute__((aligned(16))) unsigned char staged[4][NARROW_BATCH * NARROW_SPAN + NARROW_SLACK];
  __shared__ unsigned dig[NARROW_TAPS / 4][4][64];
  unsigned char* lds = staged[wave];
  const uintptr_t start = reinterpret_cast<uintptr_t>(jb.src) + o0 * row_in + (int64_t)first * INNER;
  // aligned chunks; one that sticks out of the array is filled byte by byte
  const uintptr_t lo = reinterpret_cast<uintptr_t>(jb.src), hi = lo + jb.outer * row_in;
  u32x4 v[NARROW_BATCH];
  auto request = [&](int batch) {
#pragma unroll
    for (int r = 0; r < NARROW_BATCH; ++r) {
      v[r] = u32x4{0u, 0u, 0u, 0u};
      if (batch + r >= rows) continue;
      const uintptr_t from = start + (batch + r) * row_in, chunk = (from & ~(uintptr_t)15) + 16 * lane;
      typedef __attribute__((address_space(1))) const u32x4* global_words;
      if (chunk >= lo && chunk + 16 <= hi && chunk < from + span) v[r] = *(global_words)chunk;
    }
  };
  const bool in_lds = __all(fits);
  if (in_lds) request(0);
  // wave g makes the digits of tap group g (and g + 4) of the 64 outputs, for all four waves
  for (int g = wave; g < NARROW_TAPS / 4; g += 4) {
    unsigned d3[3] = {0u, 0u, 0u}, total = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      int k = 4 * g + t < tw.n ? kk[4 * g + t] : 0;  // taps past the window have weight 0
      fits = fits && fits_digits(k);
      total += (unsigned)k;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        d3[d] |= (unsigned)(k & 0xff) << (8 * t);
        k = (k + 128) >> 8;  // less the signed digit, by 256
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) dig[g][d][lane] = d3[d];
    dig[g][3][lane] = total;
  }
  const bool digits = __syncthreads_and(fits) != 0;

  // four pixels of three channels leave as three words, each made by one lane from its own and its neighbour's bytes
  const bool words = INNER == 3 && out_len % 4 == 0 && (reinterpret_cast<uintptr_t>(jb.dst) & 3u) == 0;
  auto emit = [&](uint8_t* d, const unsigned (&b)[INNER]) {  // d: output row
    if (words) {
      const unsigned p = b[0] | (b[INNER > 1 ? 1 : 0] << 8) | (b[INNER > 2 ? 2 : 0] << 16);
      const unsigned next = __builtin_amdgcn_mov_dpp((int)p, 0xf9, 0xf, 0xf, false);  // of the next lane of the four
      const int q = lane & 3;
      if (mine && q < 3) *reinterpret_cast<unsigned*>(d + (x - q) * 3 + 4 * q) = (p >> (8 * q)) | (next << (24 - 8 * q));
    } else if (mine) {
#pragma unroll
      for (int c = 0; c < INNER; ++c) d[(int64_t)x * INNER + c] = (uint8_t)b[c];
    }
  };
  uint8_t* out_row = jb.dst + o0 * row_out;
  if (!digits) {  // windows or weights that no resampling table has
    for (int r = 0; r < rows; ++r) {
      unsigned out[INNER];
#pragma unroll 1
      for (int c = 0; c < INNER; ++c) {
        const uint8_t* p = jb.src + (o0 + r) * row_in + (int64_t)tw.xmin * INNER + c;
        unsigned a = 1u << (RESAMPLE_PRECISION_BITS - 1);
        for (int t = 0; t < tw.n; ++t) a += (unsigned)p[t * INNER] * (unsigned)kk[t];
        out[c] = clip8((int)a);
      }
      emit(out_row + r * row_out, out);
    }
    return;
  }
  const int at = (tw.xmin - first) * INNER, groups = __any(tw.n > 16) ? 6 : __any(tw.n > 12) ? 4 : __any(tw.n > 8) ? 3 : __any(tw.n > 4) ? 2 : 1;
  for (int batch = 0; batch < rows; batch += NARROW_BATCH) {
    const int n = rows - batch < NARROW_BATCH ? rows - batch : NARROW_BATCH;
    const uintptr_t row0 = start + batch * row_in;
#pragma unroll
    for (int r = 0; r < NARROW_BATCH; ++r) *reinterpret_cast<u32x4*>(lds + r * NARROW_SPAN + 16 * lane) = v[r] ^ 0x80808080u;  // pixels less 128
    if ((row0 & ~(uintptr_t)15) < lo || ((row0 + (n - 1) * row_in) & ~(uintptr_t)15) + 1024 > hi) {
#pragma unroll 1
      for (int i = 0; i < n * 16; ++i) {
        const uintptr_t from = row0 + (i / 16) * row_in, chunk = (from & ~(uintptr_t)15) + 16 * lane, byte = chunk + i % 16;
        if ((chunk < lo || chunk + 16 > hi) && byte >= lo && byte < hi && byte < from + span)
          lds[(i / 16) * NARROW_SPAN + 16 * lane + i % 16] = *reinterpret_cast<const uint8_t*>(byte) ^ 0x80u;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    request(batch + NARROW_BATCH);  // past the wave's rows: nothing
    uint8_t* d0 = out_row + batch * row_out;
    auto put = [&](int r, const unsigned (&b)[INNER]) { emit(d0 + r * row_out, b); };
    switch (groups) {
      case 1: resample_narrow_digits<INNER, 1>(lds, at, row0, row_in, n, dig, lane, put); break;
      case 2: resample_narrow_digits<INNER, 2>(lds, at, row0, row_in, n, dig, lane, put); break;
      case 3: resample_narrow_digits<INNER, 3>(lds, at, row0, row_in, n, dig, lane, put); break;
      case 4: resample_narrow_digits<INNER, 4>(lds, at, row0, row_in, n, dig, lane, put); break;
      default: resample_narrow_digits<INNER, NARROW_TAPS / 4>(lds, at, row0, row_in, n, dig, lane, put); break;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// The same pass on the matrix cores, where a row's windows fit (on_mfma): a wave makes MATRIX_OUT output bytes of some rows, sixteen rows at
// a time.  Sixteen output bytes of sixteen rows are a product of a 16 x 64 (KB times) matrix of weights, as v_mfma_i32_16x16x64_i8 takes it,
// with the input bytes as they lie in the rows: a weight stands in the columns of its own channel's bytes, zeros elsewhere.  A weight is
// three signed digits of 8 bits and a pixel is taken less 128 (one exclusive or on the way into LDS); 128 times the sum of the weights is
// added back, itself a product with rows of -128.  Whole numbers modulo 2^32 throughout, so the sums are those of plain multiply-adds.
// A wave keeps the weights of its three tiles in registers for all rows; the rows come as aligned 16-byte loads, LPR lanes to a row, and
// are shifted on the way into the wave's own piece of LDS so that every row begins at the same alignment: no barrier.
// Rows of a work-group: as many as make one round of MATRIX_GROUPS, three to a compute unit (150 registers), because a wave's weights take as long
// to lay out as some fifty rows.  What bounds it: laying out the weights (6 us of 21), vector issue (145 instructions per sixteen rows) and stores
// of 16 bytes per row (4 us).  us by the kernel above / this one, to 0.8 million pixels: 800 x 1,333 10.5 / 9.2, 1,080 x 1,920 12.9 / 11.8, 1,800 x 2,400 15.6 / 12.8,
// 2,448 x 3,264 18.4 / 15.3, 2,700 x 3,600 17.9 / 15.6, these and 427 x 640 (below: made larger) together 25.9 / 20.2; 4,480 x 4,480 to 3,584 x 3,584 55 / 43; with 256 / 512 / 1,024
// work-groups 31.0 / 22.7 / 26.4 and 65.7 / 43.9 / 49.8.  Not taken: larger windows (three times 64 bytes: 3,000 x 4,000 20 / 36) and images made larger, whose
// four taps are little work for vector instructions (427 x 640 6.6 / 7.5, six of 240 x 320 12.7 / 14.2).
constexpr int MATRIX_OUT = 48, MATRIX_TILES = MATRIX_OUT / 16, MATRIX_ROWS = 16, MATRIX_BLOCKS = 2, MATRIX_GROUPS = 768;
// input bytes that sixteen output bytes' windows span at most, in units of 64, as bounds of any resampling between these lengths have them
__host__ __device__ inline int64_t matrix_blocks(const mvit_resample_job& j) { return (((5 * j.in_len + j.out_len - 1) / j.out_len + 1 + j.ksize) * 3 + 15 + 63) / 64; }
// v_perm selector that spreads a channel's taps, eight bytes, over word q of sixteen bytes of which its first is byte `skip`
template <int INNER>
constexpr unsigned tap_selector(int q, int skip) {
  unsigned sel = 0;
  for (int e = 0; e < 4; ++e) {
    const int n = 4 * q + e - skip;
    sel |= (unsigned)(n >= 0 && n % INNER == 0 ? (n / INNER) & 7 : 0x0c) << (8 * e);
  }
  return sel;
}
// Two values shifted right by the weights' fraction and clamped to a byte each, in the lower half; the upper half keeps old bits
__device__ __forceinline__ unsigned clip8_pair(int a, int b) {
  unsigned r;
  asm("v_ashr_pk_u8_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "n"(RESAMPLE_PRECISION_BITS));
  return r;
}
__global__ __launch_bounds__(256, 3) void resample_matrix_kernel(const ResampleJobs jobs) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(1))) const unsigned char* global_bytes;
  typedef __attribute__((address_space(1))) const u32x4* global_words;
  constexpr int INNER = 3, LPR = 16, PXS = MATRIX_OUT / INNER, ROWS_AT_ONCE = 64 / LPR, LOADS = MATRIX_ROWS / ROWS_AT_ONCE;
  constexpr int PITCH = LPR * 16 + 16;  // 16 bytes in front; sixteen rows fall on 16 different 16-byte slots of 256
  constexpr int TAPS = (16 + INNER - 1) / INNER, PAD = (TAPS + 3) & ~3;  // taps of one channel in sixteen bytes; zeros around a window's digits
  constexpr int DIG_DWORDS = (PAD + NARROW_TAPS + PAD) / 4;
  __shared__ __attribute__((aligned(16))) unsigned char staged_all[4][MATRIX_ROWS * PITCH + 64 * MATRIX_BLOCKS];
  __shared__ unsigned dig_all[4][3][PXS * DIG_DWORDS + 1];
  const int j = resample_job_of(jobs, blockIdx.x);
  const mvit_resample_job& jb = jobs.job[j];
  const int block = blockIdx.x - jobs.first_block[j], lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* const staged = staged_all[wave];
  unsigned(*const dig)[PXS * DIG_DWORDS + 1] = dig_all[wave];
  const int i16 = lane & 15, g4 = lane >> 4;
  const int in_len = (int)jb.in_len, out_len = (int)jb.out_len, ksize = jb.ksize;
  const int row_in = in_len * INNER, row_out = out_len * INNER;
  const int xblocks = (row_out + 4 * MATRIX_OUT - 1) / (4 * MATRIX_OUT), xb = (block % xblocks) * 4 + wave;
  const int64_t o0 = (int64_t)(block / xblocks) * jobs.rows_per_wave;
  const int rows = jb.outer - o0 < jobs.rows_per_wave ? (int)(jb.outer - o0) : jobs.rows_per_wave;
  const int px0 = xb * PXS, px1 = px0 + PXS < out_len ? px0 + PXS : out_len;
  if (px0 >= out_len) return;
  auto window = [&](int x) { return tap_window(jb.bounds, x, ksize, in_len); };
  // the bytes of a row from the first output's window to the last one's; windows out of that order go tap by tap
  const TapWindow head = window(px0), tail = window(px1 - 1);
  const int first = head.xmin, span = (tail.xmin + tail.n - first) * INNER;
  bool fits = span >= 0 && span + 15 <= LPR * 16;
  const uintptr_t start = reinterpret_cast<uintptr_t>(jb.src) + (uintptr_t)o0 * row_in + (unsigned)(first * INNER), start16 = start & ~(uintptr_t)15;
  const uintptr_t lo = reinterpret_cast<uintptr_t>(jb.src), hi = lo + jb.outer * row_in;
  const int below = lo > start16 ? (int)(lo - start16) : 0, end = hi - start16 < 0x7fffffff ? (int)(hi - start16) : 0x7fffffff;  // of the array, from start16

  // A lane's chunk of each of its rows, aligned.  Where a row's chunks may stick out of the array (its first and last rows), those that do are
  // filled byte by byte.
  const int chunk = (lane % LPR) * 16, lane_at = (int)(start & 15) + (lane / LPR) * row_in;
  const bool wanted = chunk < span + 15;
  auto inside = [&](int step) {  // all chunks of these sixteen rows, the same for the wave
    const int at = (int)(start & 15) + step * MATRIX_ROWS * row_in;
    return (at & ~15) >= below && at + (MATRIX_ROWS - 1) * row_in + LPR * 16 <= end && (step + 1) * MATRIX_ROWS <= rows;
  };
  u32x4 v[LOADS];
  auto request = [&](int step) {
    const int at0 = lane_at + step * MATRIX_ROWS * row_in;
    if (inside(step)) {
#pragma unroll
      for (int q = 0; q < LOADS; ++q)
        if (wanted) v[q] = *reinterpret_cast<global_words>((global_bytes)start16 + (unsigned)(((at0 + q * ROWS_AT_ONCE * row_in) & ~15) + chunk));
    } else {
#pragma unroll
      for (int q = 0; q < LOADS; ++q) {
        const int row = step * MATRIX_ROWS + q * ROWS_AT_ONCE + lane / LPR, at = at0 + q * ROWS_AT_ONCE * row_in, from = (at & ~15) + chunk;
        v[q] = u32x4{0u, 0u, 0u, 0u};
        if (row < rows && wanted) {
          if (from >= below && from + 16 <= end) {
            v[q] = *reinterpret_cast<global_words>((global_bytes)start16 + (unsigned)from);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll 1
              for (int e = 0; e < 4; ++e) {
                const int byte = from + 4 * i + e;
                if (byte >= below && byte < end) v[q][i] |= (unsigned)((global_bytes)start16)[(unsigned)byte] << (8 * e);
              }
          }
        }
      }
    }
  };
  unsigned char* const put_at = staged + (lane / LPR) * PITCH + 16 + chunk;
  auto put = [&](int step) {
    const int at0 = lane_at + step * MATRIX_ROWS * row_in;
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const unsigned at = (unsigned)(at0 + q * ROWS_AT_ONCE * row_in);
      unsigned w[5] = {v[q][0], v[q][1], v[q][2], v[q][3], 0u};
      w[4] = (unsigned)__builtin_amdgcn_update_dpp(0, (int)w[0], 0x101, 0xf, 0xf, true);  // of the next lane of the row's sixteen
      unsigned* to = reinterpret_cast<unsigned*>(put_at + q * ROWS_AT_ONCE * PITCH - (at & 12));
#pragma unroll
      for (int i = 0; i < 4; ++i) to[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], at) ^ 0x80808080u;  // pixels less 128
    }
  };
  if (fits) request(0);

  int base[MATRIX_TILES], xmin[MATRIX_TILES];  // first input byte of a tile's product; the lane's window
  const int k_blocks = matrix_blocks(jb);
  TapWindow tws[MATRIX_TILES];
#pragma unroll
  for (int tl = 0; tl < MATRIX_TILES; ++tl) {
    const int px = px0 + (tl * 16 + i16) / INNER;
    tws[tl] = window(px < out_len ? px : out_len - 1);
  }
  // ---- signed digits of every output's weights, four taps a word
  constexpr int DIG_LOOPS = (PXS * DIG_DWORDS + 63) / 64;
  int k[DIG_LOOPS][4];
#pragma unroll
  for (int l = 0; l < DIG_LOOPS; ++l) {
    const int i = l * 64 + lane, x = px0 + i / DIG_DWORDS, t0 = (i % DIG_DWORDS) * 4 - PAD;
    const bool weights = x < px1 && t0 >= 0 && t0 < NARROW_TAPS;
    const TapWindow tw = window(weights ? x : px0);
    const int32_t* __restrict__ kk = jb.kk + (int64_t)x * ksize;
    if (weights) fits = fits && tw.n <= NARROW_TAPS;
#pragma unroll
    for (int t = 0; t < 4; ++t) k[l][t] = weights && t0 + t < tw.n ? kk[t0 + t] : 0;  // taps past the window have weight 0
  }
#pragma unroll
  for (int l = 0; l < DIG_LOOPS; ++l) {
    const int i = l * 64 + lane;
    unsigned d[3] = {0u, 0u, 0u};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      int rest = k[l][t];
      fits = fits && fits_digits(rest);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        d[q] |= (unsigned)(rest & 0xff) << (8 * t);
        rest = (rest + 128) >> 8;  // less the signed digit, by 256
      }
    }
    if (i < PXS * DIG_DWORDS) {
#pragma unroll
      for (int q = 0; q < 3; ++q) dig[q][i] = d[q];
    }
  }
#pragma unroll
  for (int tl = 0; tl < MATRIX_TILES; ++tl) {
    const int tile_first = __builtin_amdgcn_readfirstlane(tws[tl].xmin), last = (tws[tl].xmin + tws[tl].n - first) * INNER;
    xmin[tl] = tws[tl].xmin;
    base[tl] = ((tile_first - first) * INNER) & ~15;
    fits = fits && tws[tl].xmin >= tile_first && tile_first >= first && last <= base[tl] + 64 * k_blocks && last <= span;
  }
  if (!__all(fits)) {  // windows or weights that no resampling table has
    const int px = px1 - px0;
    for (int i = lane; i < rows * px; i += 64) {
      const int r = i / px, x = px0 + i % px;
      const TapWindow tw = window(x);
      const int32_t* __restrict__ kk = jb.kk + (int64_t)x * ksize;
#pragma unroll 1
      for (int c = 0; c < INNER; ++c) {
        const uint8_t* p = jb.src + (o0 + r) * row_in + (int64_t)tw.xmin * INNER + c;
        unsigned a = 1u << (RESAMPLE_PRECISION_BITS - 1);
        for (int t = 0; t < tw.n; ++t) a += (unsigned)p[t * INNER] * (unsigned)kk[t];
        jb.dst[(o0 + r) * row_out + (int64_t)x * INNER + c] = (uint8_t)clip8((int)a);
      }
    }
    return;
  }
  auto in_order = [] {  // LDS operations of a wave are carried out in order; the compiler is to keep to it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  in_order();

  // ---- the lane's weights: output byte i16 of each tile, input bytes 16 * g4 .. + 15 of each 64
  i32x4 weight[MATRIX_TILES][MATRIX_BLOCKS][3];
#pragma unroll
  for (int tl = 0; tl < MATRIX_TILES; ++tl) {
    const int ob = tl * 16 + i16, x = ob / INNER, c = ob - x * INNER;
#pragma unroll
    for (int kb = 0; kb < MATRIX_BLOCKS; ++kb) {
      const int p0 = base[tl] + kb * 64 + g4 * 16, px = p0 / INNER, skip = (c + INNER - (p0 - px * INNER)) % INNER;  // the channel's first byte
      int t0 = px + (p0 - px * INNER > c ? 1 : 0) + first - xmin[tl];  // its tap
      t0 = max(-PAD, min(t0, NARROW_TAPS)) + PAD;
      unsigned sel[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sel[q] = tap_selector<INNER>(q, 0);
#pragma unroll
        for (int e = 1; e < INNER; ++e) sel[q] = skip == e ? tap_selector<INNER>(q, e) : sel[q];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const unsigned* at = &dig[i][x * DIG_DWORDS + (t0 >> 2)];
        constexpr int N = (TAPS + 3) / 4;
        unsigned raw[N + 1], taps[N];
#pragma unroll
        for (int q = 0; q <= N; ++q) raw[q] = at[q];
#pragma unroll
        for (int q = 0; q < N; ++q) taps[q] = __builtin_amdgcn_alignbyte(raw[q + 1], raw[q], (unsigned)t0);
#pragma unroll
        for (int q = 0; q < 4; ++q) weight[tl][kb][i][q] = (int)__builtin_amdgcn_perm(taps[1], taps[0], sel[q]);
      }
      __builtin_amdgcn_sched_barrier(0);  // one product's digits at a time: registers
    }
  }
  // a tile's sixteen output bytes of sixteen rows
  auto product = [&](int tl, const i32x4 (&b)[MATRIX_BLOCKS]) {
    i32x4 sum[3] = {};
#pragma unroll
    for (int kb = 0; kb < MATRIX_BLOCKS; ++kb)
      if (kb < k_blocks) {
#pragma unroll
        for (int i = 0; i < 3; ++i) sum[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(weight[tl][kb][i], b[kb], sum[i], 0, 0, 0);
      }
    i32x4 all;
#pragma unroll
    for (int e = 0; e < 4; ++e) all[e] = (int)((unsigned)sum[0][e] + ((unsigned)sum[1][e] << 8) + ((unsigned)sum[2][e] << 16));
    return all;
  };
  i32x4 offset[MATRIX_TILES];  // 128 times the sum of the weights, and one half
  {
    i32x4 b[MATRIX_BLOCKS];
#pragma unroll
    for (int kb = 0; kb < MATRIX_BLOCKS; ++kb) b[kb] = i32x4{(int)0x80808080u, (int)0x80808080u, (int)0x80808080u, (int)0x80808080u};
#pragma unroll
    for (int tl = 0; tl < MATRIX_TILES; ++tl) offset[tl] = (1 << (RESAMPLE_PRECISION_BITS - 1)) - product(tl, b);
  }
  const bool words = row_out % 4 == 0 && (reinterpret_cast<uintptr_t>(jb.dst) & 3u) == 0;
  const int steps = (rows + MATRIX_ROWS - 1) / MATRIX_ROWS, byte0 = 4 * g4, bytes = (px1 - px0) * INNER;
  // a lane ends up with four consecutive bytes of row i16
  uint8_t* d = jb.dst + o0 * row_out + (int64_t)px0 * INNER + ((int64_t)i16 * row_out + byte0);
  for (int s = 0; s < steps; ++s, d += (int64_t)MATRIX_ROWS * row_out) {
    put(s);
    request(s + 1);
    in_order();
    const bool mine = s * MATRIX_ROWS + i16 < rows;
    const unsigned char* at = staged + i16 * PITCH + 16 + 16 * g4;
#pragma unroll
    for (int tl = 0; tl < MATRIX_TILES; ++tl) {
      i32x4 b[MATRIX_BLOCKS];
#pragma unroll
      for (int kb = 0; kb < MATRIX_BLOCKS; ++kb)
        if (kb < k_blocks) b[kb] = *reinterpret_cast<const i32x4*>(at + base[tl] + kb * 64);
      const i32x4 sum = offset[tl] + product(tl, b);
      if (mine && byte0 + tl * 16 < bytes) {
        if (words) {
          *reinterpret_cast<unsigned*>(d + tl * 16) = __builtin_amdgcn_perm(clip8_pair(sum[2], sum[3]), clip8_pair(sum[0], sum[1]), 0x05040100u);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (byte0 + tl * 16 + e < bytes) d[tl * 16 + e] = (uint8_t)clip8(sum[e]);
        }
      }
    }
    in_order();
  }
}

// The pass for a long contiguous dimension of whole words (the vertical pass).  A wave makes 1 KiB of one output row: the window
// and its weights are the same for all of it (scalar loads), a lane makes 16 bytes from one 16-byte load per tap.  The four waves
// of a work-group make the same KiB of four consecutive rows, whose windows overlap and meet in the L1.  Bound by the byte
// extractions and multiply-adds (two instructions per byte and tap).  4,480 x 4,480 to 3,584 x 3,584 takes 137 us with the
// horizontal pass; one word per lane, a row per work-group and the weights read by each took 180, four bytes per lane of the
// flattened array 145.  A wave costs as much with few lanes as with 64: 480 rows to 168, 12 taps, 64 times, us of
// resample_pass_kernel<true> / this one: 336 bytes 11.5 by the first, 420: 16.3 / 13.4, 512: 17.7 / 13.4, 1,024: 32.7 / 16.0, 3,024: 87 / 40
constexpr int RESAMPLE_STRIP = 1024, RESAMPLE_WIDE_FROM = 400, RESAMPLE_FEW_ROWS = 4096;
template <bool FAST>
__device__ __forceinline__ void resample_wide_bytes(const uint8_t* p, int64_t inner, int n, const int32_t* __restrict__ k, unsigned (&out)[4]) {
  typedef __attribute__((address_space(1))) const uint8_t* global_bytes;
  int a[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) a[e] = 1 << (RESAMPLE_PRECISION_BITS - 1);
  auto taps = [&](auto COUNT, int t) {
    constexpr int N = decltype(COUNT)::value;
    unsigned w[N][4];
#pragma unroll
    for (int i = 0; i < N; ++i) __builtin_memcpy(w[i], (global_bytes)(uintptr_t)(p + (int64_t)(t + i) * inner), 16);
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) a[e] = tap<FAST>(a[e], (w[i][e >> 2] >> (8 * (e & 3))) & 0xffu, k[t + i]);
  };
  int t = 0;
  for (; t + 4 <= n; t += 4) taps(std::integral_constant<int, 4>{}, t);
  if (n & 2) {
    taps(std::integral_constant<int, 2>{}, t);
    t += 2;
  }
  if (n & 1) taps(std::integral_constant<int, 1>{}, t);
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = clip8(a[4 * e]) | (clip8(a[4 * e + 1]) << 8) | (clip8(a[4 * e + 2]) << 16) | (clip8(a[4 * e + 3]) << 24);
}
__global__ __launch_bounds__(256) void resample_wide_kernel(const ResampleJobs jobs) {
  const int j = resample_job_of(jobs, blockIdx.x);
  const mvit_resample_job& jb = jobs.job[j];
  const unsigned block = blockIdx.x - jobs.first_block[j];
  const unsigned strips = (unsigned)((jb.inner + RESAMPLE_STRIP - 1) / RESAMPLE_STRIP), groups = (unsigned)((jb.out_len + 3) / 4);
  const unsigned line = block / strips, o = line / groups;
  const int x = (int)(line % groups) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (x >= jb.out_len) return;
  const TapWindow tw = tap_window(jb.bounds, x, jb.ksize, jb.in_len);
  const int32_t* __restrict__ k = jb.kk + (int64_t)x * jb.ksize;
  bool narrow = true;
  for (int t = 0; t < tw.n; ++t) narrow = narrow && fits24(k[t]);
  int64_t at = (int64_t)(block % strips) * RESAMPLE_STRIP + (threadIdx.x & 63) * 16;
  if (at >= jb.inner) return;
  if (at > jb.inner - 16) at = jb.inner - 16;  // the last lane of a row ends with it and repeats bytes of its neighbour
  const uint8_t* p = jb.src + ((int64_t)o * jb.in_len + tw.xmin) * jb.inner + at;
  unsigned v[4];
  if (narrow) resample_wide_bytes<true>(p, jb.inner, tw.n, k, v);
  else resample_wide_bytes<false>(p, jb.inner, tw.n, k, v);
  __builtin_memcpy(jb.dst + ((int64_t)o * jb.out_len + x) * jb.inner + at, v, 16);
}

// The vertical pass and patchify in one: a work-group resamples the 28 x 28 square of its merge block into LDS, so the resized image is
// never written and one launch goes.  The rows that the square's windows span are staged as dwords, the weights beside them; a lane
// makes twelve bytes of a line (seven lanes a line, 196 of 256).  Rows or taps beyond what LDS is laid out for are the caller's to pass
// separately; windows that no resampling table has are read tap by tap.  The arithmetic is resample_wide_kernel's.
// Bound by vector issue (two instructions per byte and tap) beside patchify's writes, with eight work-groups to a unit to cover the loads.  us of the
// whole input side in bf16, vertical pass and patchify one after the other / this: to 0.8 million pixels 427 x 640 19.8 / 15.4, 1,080 x 1,920 26.7 / 23.0,
// 2,448 x 3,264 30.3 / 29.6, these and 800 x 1,333 together 47.2 / 44.5, eight of 240 x 320 58.5 / 45.5; 4,480 x 4,480 to 3,584 x 3,584 130 / 99
// (104 with six work-groups to a unit).
constexpr int FUSED_ROWS = 128, FUSED_TAPS = 32, FUSED_GROUPS = 2048;
struct ResizedTable {
  mvit_resized_image im[TABLE_ARG_IMAGES + 1];
};
template <typename TO>
__global__ __launch_bounds__(256, 8) void resize_patchify_kernel(const ResizedTable images, int n_images, TO* __restrict__ out, int64_t total_rows, Norm nm) {
  __shared__ TO lut[3][256];
  __shared__ __attribute__((aligned(16))) uint32_t square[SQ_DWORDS], staged[FUSED_ROWS * SQ_DWORDS / SQ];
  __shared__ int32_t weights[SQ * FUSED_TAPS];
  constexpr int LINE = SQ_LINE / 4, BYTES = 12, LANES = SQ_LINE / BYTES;  // dwords, bytes of a lane, lanes of a line
  make_lut<TO>(lut, nm);
  const PatchLane pl = patch_lane();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t row0 = (int64_t)blockIdx.x * 4; row0 < total_rows; row0 += (int64_t)gridDim.x * 4) {
    int lo = 0, hi = n_images;  // invariant: im[lo].first_row <= row0 < im[hi].first_row
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (images.im[mid].first_row <= row0) lo = mid;
      else hi = mid;
    }
    const mvit_resized_image& im = images.im[lo];
    const int gw = im.width / PATCH, blocks_across = gw >> 1;
    const int blk = (int)((row0 - im.first_row) >> 2), hb = blk / blocks_across, wb = blk % blocks_across;
    const int64_t line = (int64_t)im.width * 3;
    const uint8_t* corner = im.src + wb * SQ_LINE;
    const int y0 = hb * SQ, ksize = im.ksize;
    auto dword = [](const uint8_t* p) {
      uint32_t w;
      __builtin_memcpy(&w, p, 4);
      return w;
    };
    __syncthreads();  // the previous square has been read
    if (im.bounds == nullptr) {  // as high as it has to be
      for (int i = threadIdx.x; i < SQ_DWORDS; i += 256) square[i] = dword(corner + (y0 + i / LINE) * line + i % LINE * 4);
    } else {
      const TapWindow head = tap_window(im.bounds, y0, ksize, im.src_height), tail = tap_window(im.bounds, y0 + SQ - 1, ksize, im.src_height);
      const int first = head.xmin, rows = max(0, min(tail.xmin + tail.n - first, FUSED_ROWS));
      for (int i = threadIdx.x; i < rows * LINE; i += 256) staged[i] = dword(corner + (first + i / LINE) * line + i % LINE * 4);
      for (int i = threadIdx.x; i < SQ * ksize; i += 256) weights[i] = im.kk[(int64_t)y0 * ksize + i];
      __syncthreads();
      if ((int)threadIdx.x < SQ * LANES) {
        const int y = threadIdx.x / LANES, c = threadIdx.x % LANES;
        const TapWindow tw = tap_window(im.bounds, y0 + y, ksize, im.src_height);
        const int32_t* k = weights + y * ksize;
        const int from = tw.xmin - first;
        bool usual = from >= 0 && from + tw.n <= rows;
        for (int t = 0; t < tw.n; ++t) usual = usual && fits24(k[t]);
        int a[BYTES];
#pragma unroll
        for (int e = 0; e < BYTES; ++e) a[e] = 1 << (RESAMPLE_PRECISION_BITS - 1);
        if (usual) {
          const uint32_t* w = staged + from * LINE + c * 3;
#pragma unroll 1
          for (int t = 0; t < tw.n; ++t)
#pragma unroll
            for (int e = 0; e < BYTES; ++e) a[e] = tap<true>(a[e], (w[t * LINE + (e >> 2)] >> (8 * (e & 3))) & 0xffu, k[t]);
        } else {
          const uint8_t* p = corner + tw.xmin * line + c * BYTES;
#pragma unroll 1
          for (int t = 0; t < tw.n; ++t)
#pragma unroll
            for (int e = 0; e < BYTES; ++e) a[e] = tap<false>(a[e], p[t * line + e], k[t]);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
          square[y * LINE + c * 3 + i] = clip8(a[4 * i]) | (clip8(a[4 * i + 1]) << 8) | (clip8(a[4 * i + 2]) << 16) | (clip8(a[4 * i + 3]) << 24);
      }
    }
    __syncthreads();  // the square and the table are complete
    if (lane < QUADS) {
      TO* dst = out + (row0 + wave) * ROW;
      TO v[3][4];
      look_up<TO>(square, lut, pl, v);
      store_patch<TO>(dst, 0, pl, v);
      store_patch<TO>(dst, 1, pl, v);
    }
  }
}

extern "C" {

int mvit_patchify(const mvit_image* images, int n_images, int64_t total_rows, void* out, double rescale, float mean_r,
                  float mean_g, float mean_b, float std_r, float std_g, float std_b, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(images != nullptr && n_images > 0, "patchify: empty image table");
  MVIT_REQUIRE(total_rows >= 0 && total_rows % 4 == 0 && total_rows / 4 <= 0x7fffffffLL,
               "patchify: total_rows %lld must be a multiple of 4 (2x2 merge blocks) below 2^33", (long long)total_rows);
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "patchify: dtype %d", dtype);
  MVIT_REQUIRE(std_r != 0.f && std_g != 0.f && std_b != 0.f, "patchify: zero std");
  if (total_rows == 0) return MVIT_OK;
  MVIT_REQUIRE(out != nullptr && mvit_aligned16(out), "patchify: output must be a 16-byte aligned device pointer");
  Norm nm{rescale, {mean_r, mean_g, mean_b}, {std_r, std_g, std_b}};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)(total_rows / 4 < PATCHIFY_GROUPS ? total_rows / 4 : PATCHIFY_GROUPS);
  if (dtype == MVIT_BF16)
    hipLaunchKernelGGL((patchify_kernel<bf16_t>), dim3(grid), 256, 0, s, images, n_images, static_cast<bf16_t*>(out), total_rows, nm);
  else
    hipLaunchKernelGGL((patchify_kernel<float>), dim3(grid), 256, 0, s, images, n_images, static_cast<float*>(out), total_rows, nm);
  MVIT_CHECK_LAUNCH("patchify");
  return MVIT_OK;
}

int mvit_resize_patchify(const mvit_resized_image* images, int n_images, int64_t total_rows, void* out, double rescale, float mean_r,
                         float mean_g, float mean_b, float std_r, float std_g, float std_b, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(images != nullptr && n_images > 0, "resize_patchify: empty image table");
  if (n_images > TABLE_ARG_IMAGES) return mvit_set_error(MVIT_ERR_UNSUPPORTED, "resize_patchify: %d images; the table holds at most %d", n_images, TABLE_ARG_IMAGES);
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "resize_patchify: dtype %d", dtype);
  MVIT_REQUIRE(std_r != 0.f && std_g != 0.f && std_b != 0.f, "resize_patchify: zero std");
  int64_t rows = 0;
  for (int i = 0; i < n_images; ++i) {
    const mvit_resized_image& im = images[i];
    MVIT_REQUIRE(im.src && im.height > 0 && im.width > 0 && im.height % SQ == 0 && im.width % SQ == 0 && im.src_height > 0 && im.first_row == rows,
                 "resize_patchify: image %d, %d x %d from %d lines, first row %lld", i, im.height, im.width, im.src_height, (long long)im.first_row);
    MVIT_REQUIRE((im.bounds == nullptr) == (im.kk == nullptr) && (im.bounds ? im.ksize > 0 : im.src_height == im.height), "resize_patchify: image %d: tables", i);
    rows += (int64_t)(im.height / PATCH) * (im.width / PATCH);
    // lines that the windows of 28 output lines span at most, as any resampling between these heights has them
    if (im.bounds && (im.ksize > FUSED_TAPS || ((int64_t)SQ * im.src_height + im.height - 1) / im.height + 1 + im.ksize > FUSED_ROWS))
      return mvit_set_error(MVIT_ERR_UNSUPPORTED, "resize_patchify: image %d: %d lines from %d are passes of their own", i, im.height, im.src_height);
  }
  MVIT_REQUIRE(images[n_images].first_row == rows && total_rows == rows && rows / 4 <= 0x7fffffffLL, "resize_patchify: total_rows %lld", (long long)total_rows);
  MVIT_REQUIRE(out != nullptr && mvit_aligned16(out), "resize_patchify: output must be a 16-byte aligned device pointer");
  ResizedTable table;
  memset(&table, 0, sizeof(table));
  memcpy(table.im, images, sizeof(mvit_resized_image) * ((size_t)n_images + 1));
  Norm nm{rescale, {mean_r, mean_g, mean_b}, {std_r, std_g, std_b}};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)(rows / 4 < FUSED_GROUPS ? rows / 4 : FUSED_GROUPS);
  if (dtype == MVIT_BF16)
    hipLaunchKernelGGL((resize_patchify_kernel<bf16_t>), dim3(grid), 256, 0, s, table, n_images, static_cast<bf16_t*>(out), rows, nm);
  else
    hipLaunchKernelGGL((resize_patchify_kernel<float>), dim3(grid), 256, 0, s, table, n_images, static_cast<float*>(out), rows, nm);
  MVIT_CHECK_LAUNCH("resize_patchify");
  return MVIT_OK;
}

int mvit_patchify_host_table(const mvit_image* images, int n_images, int64_t total_rows, void* out, double rescale, float mean_r,
                             float mean_g, float mean_b, float std_r, float std_g, float std_b, int dtype, mvit_stream_t stream) {
  MVIT_REQUIRE(images != nullptr && n_images > 0, "patchify: empty image table");
  if (n_images > TABLE_ARG_IMAGES) return mvit_set_error(MVIT_ERR_UNSUPPORTED, "patchify: %d images; a host table holds at most %d", n_images, TABLE_ARG_IMAGES);
  MVIT_REQUIRE(total_rows >= 0 && total_rows % 4 == 0 && total_rows / 4 <= 0x7fffffffLL,
               "patchify: total_rows %lld must be a multiple of 4 (2x2 merge blocks) below 2^33", (long long)total_rows);
  MVIT_REQUIRE(dtype == MVIT_BF16 || dtype == MVIT_F32, "patchify: dtype %d", dtype);
  MVIT_REQUIRE(std_r != 0.f && std_g != 0.f && std_b != 0.f, "patchify: zero std");
  if (total_rows == 0) return MVIT_OK;
  MVIT_REQUIRE(out != nullptr && mvit_aligned16(out), "patchify: output must be a 16-byte aligned device pointer");
  TableArg table;
  memset(&table, 0, sizeof(table));
  memcpy(table.im, images, sizeof(mvit_image) * ((size_t)n_images + 1));
  Norm nm{rescale, {mean_r, mean_g, mean_b}, {std_r, std_g, std_b}};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)(total_rows / 4 < PATCHIFY_GROUPS ? total_rows / 4 : PATCHIFY_GROUPS);
  if (dtype == MVIT_BF16)
    hipLaunchKernelGGL((patchify_arg_kernel<bf16_t>), dim3(grid), 256, 0, s, table, n_images, static_cast<bf16_t*>(out), total_rows, nm);
  else
    hipLaunchKernelGGL((patchify_arg_kernel<float>), dim3(grid), 256, 0, s, table, n_images, static_cast<float*>(out), total_rows, nm);
  MVIT_CHECK_LAUNCH("patchify");
  return MVIT_OK;
}

int mvit_resample_u8_batch(const mvit_resample_job* list, int n_jobs, mvit_stream_t stream) {
  MVIT_REQUIRE(n_jobs >= 0 && (n_jobs == 0 || list), "resample_u8: null job list");
  for (int i = 0; i < n_jobs; ++i) {
    const mvit_resample_job& j = list[i];
    MVIT_REQUIRE(j.src && j.dst && j.bounds && j.kk, "resample_u8: null pointer");
    MVIT_REQUIRE(j.outer >= 0 && j.in_len > 0 && j.out_len > 0 && j.inner > 0 && j.ksize > 0, "resample_u8: bad sizes (outer=%lld in=%lld out=%lld inner=%lld ksize=%d)",
                 (long long)j.outer, (long long)j.in_len, (long long)j.out_len, (long long)j.inner, j.ksize);
    MVIT_REQUIRE(j.in_len < (1 << 24) && j.out_len < (1 << 24) && j.in_len * j.inner < (1ll << 40) && j.out_len * j.inner < (1ll << 40) && j.outer < (1ll << 40) / (j.in_len + j.out_len),
                 "resample_u8: axis too long");
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // Rows per wave of the short-row kernel: as many as keep 1,024 work-groups (four per compute unit) busy, up to 16, because the
  // weights' digits are made once per work-group.  us with 4 / 8 / 16 rows: 480 x 640 to 448 x 588-like sizes 11.5 / 13.2 / 16.6,
  // 2,448 x 3,264 and three smaller to 0.8 million pixels each 31.8 / 30.3 / 30.1, 4,480 x 4,480 to 3,584 x 3,584 69.5 / 59.6 / 56.2
  int rows_per_wave = 4;
  auto shared_rows = [&](int kind) -> int64_t { return kind == 5 ? 1 : kind == 10 ? rows_per_wave : kind > 5 ? 4 * rows_per_wave : 4 * RESAMPLE_ROWS; };  // of a work-group
  // work-groups for `outer` rows of the outermost axis
  auto groups = [&](int kind, const mvit_resample_job& j, int64_t outer) {
    if (kind == 5) return outer * ((j.out_len + 3) / 4) * ((j.inner + RESAMPLE_STRIP - 1) / RESAMPLE_STRIP);
    return (kind == 10 ? (j.out_len * 3 + 4 * MATRIX_OUT - 1) / (4 * MATRIX_OUT) : (j.out_len + 63) / 64) * ((outer + shared_rows(kind) - 1) / shared_rows(kind));
  };
  // jobs of one kind (wide words; 1 .. 4 bytes, with or without LDS) share launches; 0: everything else, a launch each.  Of short rows the
  // wide kernel only takes so few (about 5 us) that a launch of their own would cost as much
  auto words = [](const mvit_resample_job& j) { return j.inner % 4 == 0 && reinterpret_cast<uintptr_t>(j.src) % 4 == 0 && reinterpret_cast<uintptr_t>(j.dst) % 4 == 0; };
  // short rows through LDS (6 .. 9) where the windows of 64 outputs fit, as bounds of any resampling between these lengths do
  auto through_lds = [](const mvit_resample_job& j) {
    return j.ksize <= NARROW_TAPS && ((63 * j.in_len + j.out_len - 1) / j.out_len + j.ksize + 1) * j.inner + 15 <= NARROW_SPAN;
  };
  // three channels on the matrix cores (10), up to the windows that its registers hold the weights of, about 3.8-fold; rows made longer only go
  // along with others, because a launch of their own would cost more than the vector instructions save
  auto fits_matrix = [](const mvit_resample_job& j) {
    return j.inner == 3 && j.ksize <= NARROW_TAPS && matrix_blocks(j) <= MATRIX_BLOCKS && j.in_len < (1 << 18) && j.out_len < (1 << 28) &&
           (((MATRIX_OUT / 3 - 1) * j.in_len + j.out_len - 1) / j.out_len + 1 + j.ksize) * 3 + 15 <= 256;
  };
  bool matrix = false;
  for (int i = 0; i < n_jobs; ++i) matrix = matrix || (list[i].outer > 0 && list[i].out_len <= list[i].in_len && fits_matrix(list[i]));
  auto kind_of = [&](const mvit_resample_job& j) {
    if (matrix && fits_matrix(j)) return 10;
    if (j.inner <= RESAMPLE_MAX_CHANNELS) return (int)j.inner + (through_lds(j) ? 5 : 0);
    const bool wide = j.inner >= RESAMPLE_WIDE_FROM || (j.inner >= 16 && j.outer * j.out_len <= RESAMPLE_FEW_ROWS);
    return words(j) && wide && groups(5, j, 1) <= MVIT_MAX_GROUPS_256 ? 5 : 0;
  };
  for (int kind = 0; kind <= 10; ++kind) {
    if (kind > 5) {
      int64_t waves = 0;
      for (int i = 0; i < n_jobs; ++i)
        if (kind_of(list[i]) == kind) waves += (list[i].out_len + 63) / 64 * list[i].outer;
      rows_per_wave = waves >= 4 * 1024 * 16 ? 16 : waves >= 4 * 1024 * 8 ? 8 : 4;
    }
    if (kind == 10) {
      int64_t steps = 0;
      for (int i = 0; i < n_jobs; ++i)
        if (kind_of(list[i]) == kind) steps += (list[i].out_len * 3 + 4 * MATRIX_OUT - 1) / (4 * MATRIX_OUT) * ((list[i].outer + MATRIX_ROWS - 1) / MATRIX_ROWS);
      const int64_t each = (steps + MATRIX_GROUPS - 1) / MATRIX_GROUPS;
      rows_per_wave = MATRIX_ROWS * (int)(each < 1 ? 1 : each > 64 ? 64 : each);
    }
    ResampleJobs jobs;
    memset(&jobs, 0, sizeof(jobs));
    int64_t blocks = 0;
    auto flush = [&]() -> int {
      if (jobs.n == 0) return MVIT_OK;
      jobs.rows_per_wave = rows_per_wave;
      const dim3 grid((unsigned)blocks);
      switch (kind) {
        case 1: hipLaunchKernelGGL((resample_narrow_kernel<1>), grid, 256, 0, s, jobs); break;
        case 2: hipLaunchKernelGGL((resample_narrow_kernel<2>), grid, 256, 0, s, jobs); break;
        case 3: hipLaunchKernelGGL((resample_narrow_kernel<3>), grid, 256, 0, s, jobs); break;
        case 4: hipLaunchKernelGGL((resample_narrow_kernel<4>), grid, 256, 0, s, jobs); break;
        case 6: hipLaunchKernelGGL((resample_narrow_lds_kernel<1>), grid, 256, 0, s, jobs); break;
        case 7: hipLaunchKernelGGL((resample_narrow_lds_kernel<2>), grid, 256, 0, s, jobs); break;
        case 8: hipLaunchKernelGGL((resample_narrow_lds_kernel<3>), grid, 256, 0, s, jobs); break;
        case 9: hipLaunchKernelGGL((resample_narrow_lds_kernel<4>), grid, 256, 0, s, jobs); break;
        case 10: hipLaunchKernelGGL(resample_matrix_kernel, grid, 256, 0, s, jobs); break;
        default: hipLaunchKernelGGL(resample_wide_kernel, grid, 256, 0, s, jobs); break;
      }
      MVIT_CHECK_LAUNCH("resample_u8");
      jobs.n = 0;
      blocks = 0;
      return MVIT_OK;
    };
    for (int i = 0; i < n_jobs; ++i) {
      const mvit_resample_job& j = list[i];
      if (j.outer == 0 || kind_of(j) != kind) continue;
      if (kind == 0) {
        const int64_t total = j.outer * ((j.out_len * j.inner + 3) / 4), want = (total + 255) / 256;
        const dim3 grid((unsigned)(want < 65535 * 16 ? want : 65535 * 16));
        if (words(j)) hipLaunchKernelGGL((resample_pass_kernel<true>), grid, 256, 0, s, j.src, j.dst, j.outer, j.in_len, j.out_len, j.inner, j.bounds, j.kk, j.ksize);
        else hipLaunchKernelGGL((resample_pass_kernel<false>), grid, 256, 0, s, j.src, j.dst, j.outer, j.in_len, j.out_len, j.inner, j.bounds, j.kk, j.ksize);
        MVIT_CHECK_LAUNCH("resample_u8");
        continue;
      }
      // the grid of a launch is limited: what does not fit goes to the next one, a job of more work-groups in pieces of whole rows
      const int64_t unit = shared_rows(kind);
      for (int64_t o = 0; o < j.outer;) {
        const int64_t fit = (MVIT_MAX_GROUPS_256 - blocks) / groups(kind, j, 1) * unit;
        if (jobs.n == RESAMPLE_MAX_JOBS || fit == 0) {
          if (int rc = flush()) return rc;
          continue;
        }
        mvit_resample_job& piece = jobs.job[jobs.n];
        piece = j;
        piece.src = j.src + o * j.in_len * j.inner;
        piece.dst = j.dst + o * j.out_len * j.inner;
        piece.outer = j.outer - o < fit ? j.outer - o : fit;
        jobs.first_block[jobs.n++] = (int)blocks;
        blocks += groups(kind, j, piece.outer);
        o += piece.outer;
      }
    }
    if (int rc = flush()) return rc;
  }
  return MVIT_OK;
}

int mvit_resample_u8(const uint8_t* src, uint8_t* dst, int64_t outer, int64_t in_len, int64_t out_len, int64_t inner,
                     const int32_t* bounds, const int32_t* kk, int ksize, mvit_stream_t stream) {
  const mvit_resample_job job = {src, dst, bounds, kk, outer, in_len, out_len, inner, ksize, 0};
  return mvit_resample_u8_batch(&job, 1, stream);
}

}  // extern "C"
