// Launch parameters and segment scheduling shared by the attention kernels.
#pragma once
#include "mvit_common.h"

struct AttnParams {
  const void *q, *k, *v, *o, *d_o;
  void *out, *dq, *dk, *dv;
  float* lse;
  float* delta;
  const int32_t* cu;
  int64_t total;
  int nheads;
  int64_t q_stride, k_stride, v_stride, o_stride, do_stride, dq_stride, dk_stride, dv_stride;
  float scale;
  const void* q_scaled;  // wide backward: bf16(Q * scale * log2(e)), row stride qs_stride
  int64_t qs_stride;
  const float *nlse2, *ndelta;  // wide backward: - lse * log2(e) and - delta, [nheads, total]
  const int32_t* order;  // optional: the segment scheduled at grid position i is order[i] (null: i)
  int seg_major;         // 0: grid (x, segment, head); 1: grid (x, head, segment), all heads of a segment together
};

// fp32 parity kernels (attention_f32.hip)
int mvit_attn_f32(const AttnParams& p, int head_dim, int n_seg, int max_seqlen, bool bwd, hipStream_t stream);

namespace {

// Which segment and head this work-group serves.  Work per work-group grows with its segment's length, so
// callers list long segments first: the short ones then fill the tail of the launch.
//
// seg_major = 2 (short segments, grid (1, n_seg, heads) with n_seg * heads a multiple of 8): a head's slice of a
// token row is 160 bytes at head_dim 80, so the heads of one segment share their 128-byte lines.  Work-group ids
// are dealt round-robin to the 8 XCDs; id i therefore takes work item (i % 8) * (total / 8) + i / 8 of the
// head-fastest list, which puts all heads of a segment on one XCD at about the same time and lets its L2 serve
// the shared lines (the natural order reads them from memory once per head).
__device__ __forceinline__ void seg_and_head(const AttnParams& p, int& seg, int& h) {
  int pos = p.seg_major == 1 ? blockIdx.z : blockIdx.y;
  h = p.seg_major == 1 ? blockIdx.y : blockIdx.z;
  const int n_seg = p.seg_major == 1 ? gridDim.z : gridDim.y;
  if (p.seg_major == 2) {
    const int nh = gridDim.z, lin = blockIdx.y + n_seg * blockIdx.z;
    const int w = (lin & 7) * ((n_seg * nh) >> 3) + (lin >> 3);
    pos = w / nh;
    h = w % nh;
  }
  seg = pos;
  if (p.order) {
    const int listed = p.order[pos];
    if ((unsigned)listed < (unsigned)n_seg) seg = listed;  // an entry outside the list never becomes an address
  }
}

}  // namespace
