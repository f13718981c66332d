// One transformer block of the vision tower behind a single C call each way: the fixed launch sequence of the block's
// forward and of its backward (Qwen2_5_VLVisionBlock.forward, modeling_qwen2_5_vl.py:776-792, with _forward_standard
// :385-472 and the MLP :203-204, and their autograd), issued from here instead of one host-language call per kernel.
// Nothing is computed here: every step is one of the library's own entry points with the operands the caller laid out (or, for windows,
// one kernel in the place of rotation and attention that rounds where they do), so the results are those of the same sequence issued call by call.  No allocation, no synchronisation; the only
// streams and events used are the caller's.
#include <math.h>
#include <string.h>

#include "mvit_common.h"

namespace {

// work-groups (= partial rows) of the RMSNorm backward: four rows at a time each, up to 1,024 of them
inline int rms_partials(int64_t rows) { return (int)(rows < 1 ? 1 : (rows + 3) / 4 < 1024 ? (rows + 3) / 4 : 1024); }

// Whether the weight gradients go in one launch behind the input-gradient chain, and the column sums in another, instead of starting
// on the second stream as soon as their inputs are complete: seven launches and ten event calls fewer per block.  A host that issues
// slower than the GPU computes gains them, and so few rows leave the GPU little to overlap; where the GPU is the slower side its idle
// units are worth more.  So the line is one of work: the products of a block of 1280 columns (MLP 3420) of 1,280 rows, the reading and
// writing of the weights counted as 100 rows more.  ms per 32-block step of that width, second stream / one launch: 64 rows 12.7 / 9.3,
// 256 12.9 / 9.7, 1,024 13.2 / 11.6, 1,296 13.21 / 13.35, 1,600 14.6 / 14.9; per 8-block step, 1920 (MLP 5120): 512 rows (in) 3.61 / 3.34,
// 640 (out) 3.85 / 3.80, 768 3.93 / 4.03, 1,280 4.79 / 5.29; 2560 (6840): 128 (in) 3.70 / 3.63, 256 (out) 3.90 / 4.07, 1,024 6.14 / 6.91; 3840 (10240):
// 64 (out) 5.04 / 5.08, 512 8.42 / 9.10.  Narrower blocks stop at 1,280 rows too (not measured beyond).
constexpr int64_t GROUP_MAX_ROWS = 1280, GROUP_WEIGHT_ROWS = 100, GROUP_MAX_WORK = (GROUP_MAX_ROWS + GROUP_WEIGHT_ROWS) * 1280 * (4 * 1280 + 3 * 3420);
inline bool grouped_wgrads(const mvit_block_args* a) {
  return a->dtype == MVIT_BF16 && a->grad_dtype == MVIT_BF16 && a->S <= GROUP_MAX_ROWS &&
         (double)(a->S + GROUP_WEIGHT_ROWS) * a->C * (4. * a->C + 3. * a->I) <= (double)GROUP_MAX_WORK && a->split_k_down == 1 &&
         a->split_k_gate_up == 1 && a->split_k_proj == 1 && a->split_k_qkv == 1;
}

struct Bump {  // hands out 256-byte aligned pieces of the caller's workspace
  char* base;
  int64_t used, size;
  void* take(int64_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (bytes + 255) / 256 * 256;
    return p;
  }
};

inline int colsum_partials(int64_t rows) {
  const int64_t n = (rows + 15) / 16;
  return (int)(n < 1 ? 1 : (n > 64 ? 64 : n));
}

inline int64_t esize(int dtype) { return dtype == MVIT_BF16 ? 2 : 4; }

inline const char* at(const void* p, int64_t elems, int dtype) { return static_cast<const char*>(p) + elems * esize(dtype); }
inline char* at(void* p, int64_t elems, int dtype) { return static_cast<char*>(p) + elems * esize(dtype); }

mvit_gemm_args gemm_args(int dtype, int out_dtype) {
  mvit_gemm_args g;
  memset(&g, 0, sizeof(g));
  g.dtype = dtype;
  g.out_dtype = out_dtype;
  g.split_k = 1;
  return g;
}

// Layout of the backward's workspace; with base == nullptr only the size is computed.
struct BwdWorkspace {
  float *colsum, *swiglu_cols, *rms2, *rms1, *delta, *splitk;
  int colsum_rows, n_swiglu_cols;  // rows of dgu per row of swiglu_cols, and how many
  int64_t delta_elems, splitk_bytes, total;
};
BwdWorkspace plan_bwd_workspace(const mvit_block_args* a, void* base) {
  const int64_t S = a->S, C = a->C, I = a->I, Ipad = a->Ipad;
  Bump b{static_cast<char*>(base), 0, 0};
  BwdWorkspace w;
  w.colsum = static_cast<float*>(b.take(a->dtype == MVIT_BF16 ? 0 : 64 * (3 * C > 2 * Ipad ? 3 * C : 2 * Ipad) * 4));
  w.colsum_rows = mvit_gemm_swiglu_bwd_colsum_rows(S, Ipad, C);
  w.n_swiglu_cols = (int)((S + w.colsum_rows - 1) / w.colsum_rows);
  w.swiglu_cols = static_cast<float*>(b.take((int64_t)w.n_swiglu_cols * 2 * Ipad * 4));
  w.rms2 = static_cast<float*>(b.take((int64_t)rms_partials(S) * C * 4));
  w.rms1 = static_cast<float*>(b.take((int64_t)rms_partials(S) * C * 4));
  w.delta_elems = mvit_attn_bwd_delta_elems(a->max_seqlen, S, a->nheads, a->head_dim, a->dtype);
  w.delta = static_cast<float*>(b.take(w.delta_elems * 4));
  const int64_t sk[4] = {a->split_k_down * C * I, a->split_k_gate_up * 2 * Ipad * C, a->split_k_proj * C * C, a->split_k_qkv * 3 * C * C};
  w.splitk_bytes = 0;
  const int64_t rows[4] = {a->split_k_down * C, a->split_k_gate_up * 2 * Ipad, a->split_k_proj * C, a->split_k_qkv * 3 * C};  // bias gradients
  for (int i = 0; i < 4; ++i) {
    const int64_t n = sk[i] + rows[i];
    w.splitk_bytes = n * 4 > w.splitk_bytes ? n * 4 : w.splitk_bytes;
  }
  w.splitk = static_cast<float*>(b.take(w.splitk_bytes));
  w.total = b.used;
  return w;
}

int check_block(const char* who, const mvit_block_args* a) {
  MVIT_REQUIRE(a != nullptr, "%s: null arguments", who);
  MVIT_REQUIRE(a->dtype == MVIT_BF16 || a->dtype == MVIT_F32, "%s: dtype %d", who, a->dtype);
  MVIT_REQUIRE(a->S >= 0 && a->C > 0 && a->I > 0 && a->Ipad >= a->I && a->Ipad % 8 == 0 && a->nheads > 0 && a->head_dim > 0 &&
                   (int64_t)a->nheads * a->head_dim == a->C,
               "%s: bad sizes (S=%lld C=%d I=%d Ipad=%d heads=%d x %d)", who, (long long)a->S, a->C, a->I, a->Ipad, a->nheads, a->head_dim);
  MVIT_REQUIRE(a->norm1 && a->norm2 && a->wqkv && a->bqkv && a->wproj && a->bproj && a->wgu && a->bgu && a->wdown && a->bdown,
               "%s: null weight operand", who);
  MVIT_REQUIRE(a->cu && a->cos && a->sin && a->n_seg >= 0 && a->max_seqlen >= 0, "%s: attention geometry missing", who);
  MVIT_REQUIRE(a->x && a->n1 && a->rstd1 && a->qkv && a->o && a->lse && a->x1 && a->n2 && a->rstd2 && a->h, "%s: null activation buffer", who);
  return MVIT_OK;
}

}  // namespace

#define STEP(call)                \
  do {                            \
    if (int rc__ = (call)) return rc__; \
  } while (0)

extern "C" int mvit_block_fwd(const mvit_block_args* a, mvit_stream_t stream) {
  if (int rc = check_block("block_fwd", a)) return rc;
  if (a->S == 0) return MVIT_OK;
  const int dt = a->dtype;
  const int64_t S = a->S, C = a->C, Ipad = a->Ipad;
  const int H = a->nheads, hd = a->head_dim;

  STEP(mvit_rmsnorm_fwd(a->x, a->norm1, a->n1, a->rstd1, S, C, a->eps, dt, stream));
  {  // qkv = n1 . Wqkv^T + b
    mvit_gemm_args g = gemm_args(dt, dt);
    g.epilogue = MVIT_EPI_BIAS;
    g.M = S; g.N = 3 * C; g.K = C;
    g.A = a->n1; g.lda = C; g.B = a->wqkv; g.ldb = C; g.bias = a->bqkv; g.C = a->qkv; g.ldc = 3 * C;
    STEP(mvit_gemm(&g, stream));
  }
  // rotary embedding of q and k in place; the queries also take the softmax scale in base-2 units.  Windows: inside their attention
  const mvit_window_rope rotated{a->qkv, a->o, a->lse, a->cu, a->cos, a->sin, a->n_seg, H, S, a->q_lead_scale, a->attn_scale, a->gu != nullptr};
  const bool inside = !a->skip_attention && mvit_window_rope_takes(rotated, hd, a->max_seqlen, dt);
  if (inside) STEP(mvit_attn_fwd_window_rope(rotated, reinterpret_cast<hipStream_t>(stream)));
  else STEP(mvit_rope_scaled(a->qkv, a->cos, a->sin, S, 2 * H, hd, 3 * C, 0, H, a->q_lead_scale, dt, stream));
  if (!a->skip_attention && !inside)
    STEP(mvit_attn_fwd(a->qkv, at(a->qkv, C, dt), at(a->qkv, 2 * C, dt), a->o, a->lse, a->cu, a->seg_order, a->n_seg, a->max_seqlen, S, H, hd,
                       3 * C, 3 * C, 3 * C, C, a->attn_scale, dt, stream));
  {  // x1 = x + o . Wproj^T + b
    mvit_gemm_args g = gemm_args(dt, dt);
    g.epilogue = MVIT_EPI_BIAS_RES;
    g.M = S; g.N = C; g.K = C;
    g.A = a->o; g.lda = C; g.B = a->wproj; g.ldb = C; g.bias = a->bproj; g.C = a->x1; g.ldc = C; g.R = a->x; g.ldr = C;
    STEP(mvit_gemm(&g, stream));
  }
  STEP(mvit_rmsnorm_fwd(a->x1, a->norm2, a->n2, a->rstd2, S, C, a->eps, dt, stream));
  {  // h = silu(n2 . Wg^T + bg) * (n2 . Wu^T + bu); the pre-activations go to gu when the backward will want them
    mvit_gemm_args g = gemm_args(dt, dt);
    g.epilogue = MVIT_EPI_SWIGLU;
    g.M = S; g.N = Ipad; g.K = C;
    g.A = a->n2; g.lda = C; g.B = a->wgu; g.B2 = at(a->wgu, Ipad * C, dt); g.ldb = C;
    g.bias = a->bgu; g.bias2 = at(a->bgu, Ipad, dt);
    g.C = a->h; g.ldc = Ipad; g.aux = a->gu; g.ldaux = a->gu ? 2 * Ipad : 0; g.aux_off = Ipad;
    STEP(mvit_gemm(&g, stream));
  }
  if (a->x2) {  // x2 = x1 + h . Wdown^T + b
    mvit_gemm_args g = gemm_args(dt, dt);
    g.epilogue = MVIT_EPI_BIAS_RES;
    g.M = S; g.N = C; g.K = Ipad;
    g.A = a->h; g.lda = Ipad; g.B = a->wdown; g.ldb = Ipad; g.bias = a->bdown; g.C = a->x2; g.ldc = C; g.R = a->x1; g.ldr = C;
    STEP(mvit_gemm(&g, stream));
  }
  return MVIT_OK;
}

extern "C" int64_t mvit_block_bwd_workspace_bytes(const mvit_block_args* a) {
  if (a == nullptr) return 0;
  return plan_bwd_workspace(a, nullptr).total;
}

extern "C" int mvit_block_bwd_uses_side_stream(const mvit_block_args* a) { return a != nullptr && !grouped_wgrads(a); }

extern "C" int mvit_block_bwd(const mvit_block_args* a, mvit_stream_t stream) {
  if (int rc = check_block("block_bwd", a)) return rc;
  MVIT_REQUIRE(a->gu && a->dx2 && a->dx && a->dgu && a->dn && a->dx1 && a->dqkv, "block_bwd: null gradient buffer");
  MVIT_REQUIRE(a->g_norm1 && a->g_norm2 && a->g_wqkv && a->g_bqkv && a->g_wproj && a->g_bproj && a->g_wgu && a->g_bgu && a->g_wdown && a->g_bdown,
               "block_bwd: null parameter-gradient buffer");
  MVIT_REQUIRE(a->grad_dtype == MVIT_BF16 || a->grad_dtype == MVIT_F32, "block_bwd: grad_dtype %d", a->grad_dtype);
  MVIT_REQUIRE(a->split_k_down >= 1 && a->split_k_gate_up >= 1 && a->split_k_proj >= 1 && a->split_k_qkv >= 1, "block_bwd: split_k counts must be >= 1");
  const bool grouped = grouped_wgrads(a);
  const bool two = a->side_stream != nullptr && !grouped;
  if (a->side_stream != nullptr) MVIT_REQUIRE(a->events[0] && a->events[1] && a->events[2] && a->events[3] && a->events[4], "block_bwd: a second stream needs five events");
  if (a->S == 0) return MVIT_OK;
  const BwdWorkspace w = plan_bwd_workspace(a, a->workspace);
  MVIT_REQUIRE(a->workspace && mvit_aligned16(a->workspace) && a->workspace_bytes >= w.total, "block_bwd: the workspace holds %lld bytes, %lld are needed",
               (long long)a->workspace_bytes, (long long)w.total);
  const int dt = a->dtype, gdt = a->grad_dtype;
  const int64_t S = a->S, C = a->C, I = a->I, Ipad = a->Ipad;
  const int H = a->nheads, hd = a->head_dim;
  // windows: the inverse rotation of dq and dk is in their attention's backward
  const mvit_window_rope rotated{a->qkv, a->o, a->lse, a->cu, a->cos, a->sin, a->n_seg, H, S, a->q_lead_scale, a->attn_scale, true};
  const bool inside = mvit_window_rope_takes(rotated, hd, a->max_seqlen, dt) && mvit_aligned16(a->dqkv) && mvit_aligned16(a->dn);
  if (inside) {  // as mvit_attn_bwd asks of its outputs
    const struct { const void* ptr; int64_t cols; const char* name; } ins[] = {{a->qkv, 3 * C, "qkv"}, {a->o, C, "o"}, {a->dn, C, "d_o"}};
    for (const auto& r : ins) {
      const char *out = static_cast<const char*>(a->dqkv), *in = static_cast<const char*>(r.ptr);
      MVIT_REQUIRE(out + S * 3 * C * 2 <= in || in + S * r.cols * 2 <= out, "block_bwd: dqkv overlaps %s (outputs are written before all inputs have been read)", r.name);
    }
  }
  hipStream_t main_s = reinterpret_cast<hipStream_t>(stream), side_s = reinterpret_cast<hipStream_t>(a->side_stream);

  // Weight and bias gradients feed nothing else in the block: with a second stream they start there once their inputs
  // are complete on the main stream (event n) and are joined at the end; without one they run in line.
  auto fork = [&](int n) -> mvit_stream_t {
    if (!two) return stream;
    hipEvent_t ev = reinterpret_cast<hipEvent_t>(a->events[n]);
    if (hipEventRecord(ev, main_s) != hipSuccess || hipStreamWaitEvent(side_s, ev, 0) != hipSuccess) {
      mvit_set_error(MVIT_ERR_LAUNCH, "block_bwd: event %d: %s", n, hipGetErrorString(hipGetLastError()));
      return nullptr;
    }
    return a->side_stream;
  };
  auto bias_grad = [&](const void* dy, int64_t ld, int64_t cols, void* out, mvit_stream_t st) -> int {
    const int np = colsum_partials(S);
    STEP(mvit_colsum(dy, ld, S, cols, w.colsum, np, dt, st));
    return mvit_reduce_partials(w.colsum, np, cols, out, gdt, st);
  };
  // dW[M, N] = dY^T . X over the S rows and db[M], the column sums of dY: bf16 products sum them from the operand they read
  mvit_gemm_args later[4];
  int n_later = 0;
  auto weight_grad = [&](const void* dy, int64_t ldy, int64_t M, const void* x, int64_t ldx, int64_t N, void* out, void* bias, int split_k, mvit_stream_t st) -> int {
    if (bias && dt != MVIT_BF16) STEP(bias_grad(dy, ldy, M, bias, st));
    mvit_gemm_args g = gemm_args(dt, gdt);
    g.trans_a = 1; g.trans_b = 1; g.overlapped = two;
    g.M = M; g.N = N; g.K = S;
    g.A = dy; g.lda = ldy; g.B = x; g.ldb = ldx; g.C = out; g.ldc = N;
    if (split_k > 1) {
      g.split_k = split_k; g.workspace = w.splitk; g.workspace_bytes = (int64_t)split_k * M * (N + 1) * 4;
    }
    if (dt == MVIT_BF16) g.row_sums = bias;
    if (grouped) {
      later[n_later++] = g;
      return MVIT_OK;
    }
    return mvit_gemm(&g, st);
  };

  // ---- MLP: x2 = x1 + down(silu(g) * u)
  {
    mvit_stream_t st = fork(0);
    if (!st && two) return MVIT_ERR_LAUNCH;
    STEP(weight_grad(a->dx2, C, C, a->h, Ipad, I, a->g_wdown, a->g_bdown, a->split_k_down, st));
  }
  // dgu = (dx2 . Wdown) through the SwiGLU derivative.  In bf16 the per-tile column sums of dgu come back with it, from its fp32
  // values: the gate / up bias gradient
  const bool fused_cols = dt == MVIT_BF16;
  {
    mvit_gemm_args g = gemm_args(dt, dt);
    g.trans_b = 1; g.epilogue = MVIT_EPI_SWIGLU_BWD; g.overlapped = two;
    g.M = S; g.N = Ipad; g.K = C;
    g.A = a->dx2; g.lda = C; g.B = a->wdown; g.ldb = Ipad; g.C = a->dgu; g.ldc = 2 * Ipad; g.R = a->gu; g.ldr = 2 * Ipad; g.aux_off = Ipad;
    if (fused_cols) {
      g.workspace = w.swiglu_cols; g.workspace_bytes = (int64_t)w.n_swiglu_cols * 2 * Ipad * 4; g.colsum_rows = w.colsum_rows;
    }
    STEP(mvit_gemm(&g, stream));
  }
  {
    mvit_stream_t st = fork(1);
    if (!st && two) return MVIT_ERR_LAUNCH;
    if (fused_cols && !grouped) STEP(mvit_reduce_partials(w.swiglu_cols, w.n_swiglu_cols, 2 * Ipad, a->g_bgu, gdt, st));
    STEP(weight_grad(a->dgu, 2 * Ipad, 2 * Ipad, a->n2, C, C, a->g_wgu, fused_cols ? nullptr : a->g_bgu, a->split_k_gate_up, st));
  }
  {  // dn2 = dgu . Wgu
    mvit_gemm_args g = gemm_args(dt, dt);
    g.trans_b = 1; g.overlapped = two;
    g.M = S; g.N = C; g.K = 2 * Ipad;
    g.A = a->dgu; g.lda = 2 * Ipad; g.B = a->wgu; g.ldb = C; g.C = a->dn; g.ldc = C;
    STEP(mvit_gemm(&g, stream));
  }
  const int n_rms = rms_partials(S);
  STEP(mvit_rmsnorm_bwd(a->dn, a->x1, a->norm2, a->rstd2, a->dx2, a->dx1, w.rms2, n_rms, S, C, dt, stream));

  // ---- attention: x1 = x + proj(attn(rope(qkv(norm1(x)))))
  {
    mvit_stream_t st = fork(2);
    if (!st && two) return MVIT_ERR_LAUNCH;
    STEP(weight_grad(a->dx1, C, C, a->o, C, C, a->g_wproj, a->g_bproj, a->split_k_proj, st));
  }
  {  // d_o = dx1 . Wproj  (into the dn buffer, whose contents the norm backward above has consumed)
    mvit_gemm_args g = gemm_args(dt, dt);
    g.trans_b = 1; g.overlapped = two;
    g.M = S; g.N = C; g.K = C;
    g.A = a->dx1; g.lda = C; g.B = a->wproj; g.ldb = C; g.C = a->dn; g.ldc = C;
    STEP(mvit_gemm(&g, stream));
  }
  if (inside) STEP(mvit_attn_bwd_window_rope(rotated, a->dn, a->dqkv, w.delta, main_s));
  else STEP(mvit_attn_bwd(a->qkv, at(a->qkv, C, dt), at(a->qkv, 2 * C, dt), a->o, a->dn, a->lse, a->dqkv, at(a->dqkv, C, dt), at(a->dqkv, 2 * C, dt),
                     w.delta, w.delta_elems, a->cu, a->seg_order, a->n_seg, a->max_seqlen, S, H, hd, 3 * C, 3 * C, 3 * C, C, C, 3 * C, 3 * C, 3 * C,
                     a->attn_scale, dt, stream));
  if (!inside) STEP(mvit_rope_scaled(a->dqkv, a->cos, a->sin, S, 2 * H, hd, 3 * C, 1, H, a->q_lead_scale, dt, stream));
  {
    mvit_stream_t st = fork(3);
    if (!st && two) return MVIT_ERR_LAUNCH;
    STEP(weight_grad(a->dqkv, 3 * C, 3 * C, a->n1, C, C, a->g_wqkv, a->g_bqkv, a->split_k_qkv, st));
  }
  {  // dn1 = dqkv . Wqkv
    mvit_gemm_args g = gemm_args(dt, dt);
    g.trans_b = 1; g.overlapped = two;
    g.M = S; g.N = C; g.K = 3 * C;
    g.A = a->dqkv; g.lda = 3 * C; g.B = a->wqkv; g.ldb = C; g.C = a->dn; g.ldc = C;
    STEP(mvit_gemm(&g, stream));
  }
  STEP(mvit_rmsnorm_bwd(a->dn, a->x, a->norm1, a->rstd1, a->dx1, a->dx, w.rms1, n_rms, S, C, dt, stream));
  if (grouped) STEP(mvit_gemm_wgrad_group(later, n_later, main_s));
  const mvit_partials sums[3] = {{w.rms2, n_rms, C, a->g_norm2}, {w.rms1, n_rms, C, a->g_norm1}, {w.swiglu_cols, w.n_swiglu_cols, 2 * Ipad, a->g_bgu}};
  STEP(mvit_reduce_partials_group(sums, grouped ? 3 : 2, gdt, main_s));
  if (two) {  // the gradients are complete on the main stream when the call's work is
    hipEvent_t ev = reinterpret_cast<hipEvent_t>(a->events[4]);
    if (hipEventRecord(ev, side_s) != hipSuccess || hipStreamWaitEvent(main_s, ev, 0) != hipSuccess)
      return mvit_set_error(MVIT_ERR_LAUNCH, "block_bwd: joining the second stream: %s", hipGetErrorString(hipGetLastError()));
  }
  return MVIT_OK;
}
