// C entry points for the attention stages plus the library's error plumbing.  Argument checks live here so
// that a kernel is never launched on shapes its tiling does not cover.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <math.h>
#include <string.h>
#include <atomic>
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include "../../include/nsa_hip.h"

static thread_local char g_err[512] = "";

void nsa_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

// Tuning values that a caller may override through nsa_set_tuning (never read from the environment).
namespace {
struct Knob {
  const char* name;
  std::atomic<int> value;
  std::atomic<bool> is_set;
};
Knob g_knobs[] = {
    {"fwd_variant", {0}, {false}},      // forward tile kernel: staging / rows per wave variant
    {"dq_min_blocks", {0}, {false}},    // workgroups per CU of the dense dq kernel
    {"dkdv_key_blocks", {0}, {false}},  // 32-key blocks per wave of the dense dk/dv kernel
    {"topk_seg_blocks", {0}, {false}},  // selection blocks per segment of the block selector
    {"decode_waves", {0}, {false}},     // waves per workgroup of the one-launch decode kernel (0: from the batch; 4, 8)
    {"swa_dkdv_splits", {0}, {false}},  // query chunks per key tile of the window dk/dv kernel (0: from the sizes)
    {"slc_ds_mb", {0}, {false}},        // scratch for the dS of the selected branch, MB (0: dq and dk/dv computed apart)
    {"dense_ds_mb", {0}, {false}},      // scratch for the dS of the compressed branch, the window's, the keys' before it, MB each
    {"topk_two_pass", {0}, {false}},    // 0: the one-launch selector even when a workspace is given
};
Knob* find_knob(const char* name) {
  for (Knob& k : g_knobs)
    if (strcmp(k.name, name) == 0) return &k;
  return nullptr;
}
}  // namespace

int nsa_tuning_knob(const char* name, int default_value) {
  Knob* k = find_knob(name);
  return (k && k->is_set.load()) ? k->value.load() : default_value;
}

int nsa_check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    nsa_set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return NSA_ERR_LAUNCH;
  }
  return NSA_OK;
}

int nsa_device_cus() {
  static std::atomic<int> num_cus{0};
  int n = num_cus.load(std::memory_order_relaxed);
  if (n == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    n = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess &&
         prop.multiProcessorCount > 0) ? prop.multiProcessorCount : 256;
    num_cus.store(n, std::memory_order_relaxed);
  }
  return n;
}

static int check_heads(const char* who, int QH, int KH, int D, int VD) {
  NSA_REQUIRE(QH > 0 && KH > 0 && QH % KH == 0, NSA_ERR_BAD_ARG, "%s: q heads %d must be a multiple of kv heads %d",
              who, QH, KH);
  NSA_REQUIRE(D % 32 == 0 && VD % 32 == 0, NSA_ERR_BAD_ARG, "%s: head dims %d/%d must be multiples of 32", who, D, VD);
  return NSA_OK;
}
static int check_nsa_sizes(const char* who, int kernel_size, int stride, int block_size) {
  NSA_REQUIRE(stride > 0 && (stride & (stride - 1)) == 0, NSA_ERR_BAD_ARG, "%s: stride %d must be a power of 2", who,
              stride);
  NSA_REQUIRE(kernel_size % stride == 0 && kernel_size >= stride, NSA_ERR_BAD_ARG,
              "%s: kernel_size %d must be a multiple of stride %d", who, kernel_size, stride);
  if (block_size > 0) {
    NSA_REQUIRE(block_size >= kernel_size && block_size % stride == 0, NSA_ERR_BAD_ARG,
                "%s: block_size %d must be >= kernel_size %d and a multiple of stride %d", who, block_size,
                kernel_size, stride);
  }
  return NSA_OK;
}

extern "C" {

const char* nsa_last_error(void) { return g_err; }
int nsa_abi_version(void) { return 1; }

int nsa_set_tuning(const char* name, int value) {
  Knob* k = name ? find_knob(name) : nullptr;
  NSA_REQUIRE(k != nullptr, NSA_ERR_BAD_ARG, "set_tuning: unknown name '%s' (fwd_variant, dq_min_blocks, "
              "dkdv_key_blocks, topk_seg_blocks, swa_dkdv_splits, decode_waves, slc_ds_mb, dense_ds_mb, "
              "topk_two_pass)", name ? name : "(null)");
  k->value.store(value);
  k->is_set.store(true);
  return NSA_OK;
}
int nsa_reset_tuning(void) {
  for (Knob& k : g_knobs) k.is_set.store(false);
  return NSA_OK;
}

int nsa_cmp_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                     const void* cv, int64_t cv_sr, int64_t cv_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                     int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                     int QH, int KH, int D, int VD, int kernel_size, int stride, float sm_scale, void* stream) {
  int rc = check_heads("cmp_attn_fwd", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("cmp_attn_fwd", kernel_size, stride, 0);
  if (rc) return rc;
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)ck; p.k_sr = ck_sr; p.k_sh = ck_sh;
  p.v = (const bf16_t*)cv; p.v_sr = cv_sr; p.v_sh = cv_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.k_cu = y_cu;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.window = 0;
  return nsa_fwd_tile_launch(p, 0, false, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_swa_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                const void* v, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                int VD, int window, float sm_scale, void* stream) {
  int rc = check_heads("swa_fwd", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "swa_fwd: window %d must be >= 0", window);
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = 1; p.stride = 1; p.window = window;
  return nsa_fwd_tile_launch(p, 1, false, B, x_maxlen, D, VD, (hipStream_t)stream);
}

static int fill_swa_tail(NsaFwdTileParams& p, const char* who, void* slc_o, int64_t so_st, int64_t so_sh,
                         float* slc_lse, int64_t sl_st, int64_t sl_sh, int all_below, const void* cmp_o,
                         int64_t co_st, int64_t co_sh, const void* w, int64_t w_st, int64_t w_sh, void* out,
                         int64_t out_st, int64_t out_sh, int store_branches) {
  NSA_REQUIRE(all_below >= 0 && slc_o != nullptr, NSA_ERR_BAD_ARG,
              "%s: all_below %d must be >= 0 and the selected branch's output given", who, all_below);
  NSA_REQUIRE(out == nullptr || (cmp_o != nullptr && w != nullptr && p.o != nullptr), NSA_ERR_BAD_ARG,
              "%s: the combined output needs all branches and the gates", who);
  p.all_below = all_below; p.store_branches = store_branches;
  p.slc_o = (bf16_t*)slc_o; p.so_st = so_st; p.so_sh = so_sh;
  p.slc_lse = slc_lse; p.sl_st = sl_st; p.sl_sh = sl_sh;
  p.cmp_o = (const bf16_t*)cmp_o; p.co_st = co_st; p.co_sh = co_sh;
  p.w = (const bf16_t*)w; p.w_st = w_st; p.w_sh = w_sh;
  p.out = (bf16_t*)out; p.out_st = out_st; p.out_sh = out_sh;
  return NSA_OK;
}

int nsa_swa_fwd_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                     int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh, float* slc_lse,
                     int64_t sl_st, int64_t sl_sh, int all_below, const void* cmp_o, int64_t co_st, int64_t co_sh,
                     const void* w, int64_t w_st, int64_t w_sh, void* out, int64_t out_st, int64_t out_sh,
                     int store_branches, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD,
                     int window, float sm_scale, void* stream) {
  int rc = check_heads("swa_fwd_tail", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "swa_fwd_tail: window %d must be >= 0", window);
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = 1; p.stride = 1; p.window = window;
  rc = fill_swa_tail(p, "swa_fwd_tail", slc_o, so_st, so_sh, slc_lse, sl_st, sl_sh, all_below, cmp_o, co_st, co_sh, w,
                     w_st, w_sh, out, out_st, out_sh, store_branches);
  if (rc) return rc;
  return nsa_fwd_tile_launch(p, 2, false, B, x_maxlen, D, VD, (hipStream_t)stream);
}

// the compressed branch in the same launch
static void fill_cmp_branch(NsaFwdTileParams& p, const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cv, int64_t cv_sr,
                            int64_t cv_sh, void* cmp_o, float* cmp_lse, int64_t cl_st, int64_t cl_sh, int kernel_size, int stride) {
  p.ck = (const bf16_t*)ck; p.ck_sr = ck_sr; p.ck_sh = ck_sh;
  p.cv = (const bf16_t*)cv; p.cv_sr = cv_sr; p.cv_sh = cv_sh;
  p.cmp_o_out = (bf16_t*)cmp_o;
  p.cmp_lse = cmp_lse; p.cl_st = cl_st; p.cl_sh = cl_sh;
  p.kernel_size = kernel_size; p.stride = stride;
}

int nsa_fwd_short(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh, const void* v,
                  int64_t v_sr, int64_t v_sh, const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cv, int64_t cv_sr,
                  int64_t cv_sh, void* cmp_o, int64_t co_st, int64_t co_sh, float* cmp_lse, int64_t cl_st, int64_t cl_sh, void* o,
                  int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh,
                  float* slc_lse, int64_t sl_st, int64_t sl_sh, int all_below, const void* w, int64_t w_st, int64_t w_sh, void* out,
                  int64_t out_st, int64_t out_sh, int store_branches, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                  int QH, int KH, int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream) {
  int rc = check_heads("fwd_short", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("fwd_short", kernel_size, stride, 0);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "fwd_short: window %d must be >= 0", window);
  NSA_REQUIRE(x_maxlen <= all_below, NSA_ERR_BAD_ARG, "fwd_short: %d tokens are more than the %d that select everything", x_maxlen,
              all_below);
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.k_cu = y_cu;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.window = window;
  rc = fill_swa_tail(p, "fwd_short", slc_o, so_st, so_sh, slc_lse, sl_st, sl_sh, all_below, cmp_o, co_st, co_sh, w, w_st, w_sh, out,
                     out_st, out_sh, store_branches);
  if (rc) return rc;
  NSA_REQUIRE(cmp_o != nullptr, NSA_ERR_BAD_ARG, "fwd_short: the compressed branch's output is missing");
  fill_cmp_branch(p, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, cmp_o, cmp_lse, cl_st, cl_sh, kernel_size, stride);
  return nsa_fwd_tile_launch(p, 3, false, B, x_maxlen, D, VD, (hipStream_t)stream);
}

static int topk_select_impl(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                            const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                            int64_t tk_st, float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols,
                            const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                            int kernel_size, int stride, int block_size, int top_n, int num_init, int num_local,
                            int ignore_index, float sm_scale, int total_tokens, int t_begin, void* workspace,
                            int64_t workspace_bytes, void* stream) {
  int rc = check_heads("topk_select", QH, KH, D, 32);
  if (rc) return rc;
  rc = check_nsa_sizes("topk_select", kernel_size, stride, block_size);
  if (rc) return rc;
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "topk_select: top_n %d must be in [1,64]", top_n);
  NSA_REQUIRE(num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n, NSA_ERR_BAD_ARG,
              "topk_select: num_init %d + num_local %d must be <= top_n %d", num_init, num_local, top_n);
  NsaTopkParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.ck = (const bf16_t*)ck; p.ck_sr = ck_sr; p.ck_sh = ck_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.imp_out = imp_out; p.imp_sh = imp_sh; p.imp_st = imp_st; p.imp_cols = imp_cols;
  p.x_cu = x_cu; p.y_cu = y_cu;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.block_size = block_size;
  p.top_n = top_n; p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  p.nb_max = (x_maxlen + block_size - 1) / block_size;
  if (p.nb_max < 1) p.nb_max = 1;
  p.t_begin = t_begin;
  if (workspace != nullptr && nsa_tuning_knob("topk_two_pass", 1) != 0 && nsa_topk_two_pass_supported(p, D))
    return nsa_topk_two_pass_launch(p, false, B, x_maxlen, total_tokens, D, workspace, workspace_bytes,
                                    (hipStream_t)stream);
  return nsa_topk_launch(p, false, B, x_maxlen, D, (hipStream_t)stream);
}

int nsa_topk_select(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                    const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                    float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols, const int32_t* x_cu,
                    const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int kernel_size, int stride,
                    int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                    void* stream) {
  return topk_select_impl(q, q_st, q_sh, ck, ck_sr, ck_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, imp_out, imp_sh,
                          imp_st, imp_cols, x_cu, y_cu, B, x_maxlen, QH, KH, D, kernel_size, stride, block_size,
                          top_n, num_init, num_local, ignore_index, sm_scale, 0, 0, nullptr, 0, stream);
}

int64_t nsa_topk_workspace_bytes(int total_tokens, int max_blocks, int KH) {
  if (total_tokens <= 0 || max_blocks <= 0 || KH <= 0) return 0;
  return (int64_t)total_tokens * nsa_topk_two_pass_bytes_per_token(KH, max_blocks) + 512;
}

int nsa_topk_select_ws(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                       const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                       float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols, const int32_t* x_cu,
                       const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int kernel_size, int stride,
                       int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                       int total_tokens, void* workspace, int64_t workspace_bytes, void* stream) {
  return nsa_topk_select_ws_from(q, q_st, q_sh, ck, ck_sr, ck_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, imp_out,
                                 imp_sh, imp_st, imp_cols, x_cu, y_cu, B, x_maxlen, QH, KH, D, kernel_size, stride,
                                 block_size, top_n, num_init, num_local, ignore_index, sm_scale, total_tokens, 0,
                                 workspace, workspace_bytes, stream);
}

int nsa_topk_select_ws_from(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                            const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                            int64_t tk_st, float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols,
                            const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                            int kernel_size, int stride, int block_size, int top_n, int num_init, int num_local,
                            int ignore_index, float sm_scale, int total_tokens, int t_begin, void* workspace,
                            int64_t workspace_bytes, void* stream) {
  NSA_REQUIRE(total_tokens >= 0 && (workspace == nullptr || workspace_bytes > 0), NSA_ERR_BAD_ARG,
              "topk_select_ws: bad token count %d or workspace size %lld", total_tokens, (long long)workspace_bytes);
  return topk_select_impl(q, q_st, q_sh, ck, ck_sr, ck_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, imp_out, imp_sh,
                          imp_st, imp_cols, x_cu, y_cu, B, x_maxlen, QH, KH, D, kernel_size, stride, block_size,
                          top_n, num_init, num_local, ignore_index, sm_scale, total_tokens, t_begin, workspace,
                          workspace_bytes, stream);
}

static int check_positions(const char* who, int pos) {
  NSA_REQUIRE(pos >= 0, NSA_ERR_BAD_ARG, "%s: position %d must be >= 0", who, pos);
  return NSA_OK;
}

int nsa_slc_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st,
                     void* o, int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh,
                     const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD, int block_size,
                     int top_n, float sm_scale, void* stream) {
  return nsa_slc_attn_fwd_from(q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, topk, tk_sh, tk_st, o, o_st, o_sh, lse,
                               lse_st, lse_sh, x_cu, B, x_maxlen, QH, KH, D, VD, block_size, top_n, 0, sm_scale,
                               stream);
}

int nsa_slc_attn_fwd_from(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                          const void* v, int64_t v_sr, int64_t v_sh, const int32_t* topk, int64_t tk_sh,
                          int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st,
                          int64_t lse_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD,
                          int block_size, int top_n, int t_begin, float sm_scale, void* stream) {
  int rc = check_heads("slc_attn_fwd", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(block_size % 32 == 0 && block_size > 0, NSA_ERR_UNSUPPORTED,
              "slc_attn_fwd: block_size %d must be a multiple of 32", block_size);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "slc_attn_fwd: top_n %d must be in [1,64]", top_n);
  rc = check_positions("slc_attn_fwd", t_begin);
  if (rc) return rc;
  NsaSlcParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.x_cu = x_cu;
  p.G = QH / KH; p.KH = KH; p.top_n = top_n; p.block_size = block_size;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.t_begin = t_begin;
  return nsa_slc_fwd_launch(p, false, B, x_maxlen, D, VD, (hipStream_t)stream);
}

}  // extern "C"

// ------------------------------------------------------------------------------------------------ backward
namespace {
struct BwdCommon {
  const void* q; int64_t q_st, q_sh;
  const void* k; int64_t k_sr, k_sh;
  const void* v; int64_t v_sr, v_sh;
  const void* dO; int64_t do_st, do_sh;
  const float* lse; int64_t lse_st, lse_sh;
  const float* delta; int64_t delta_st, delta_sh;
};
NsaBwdTileParams make_bwd(const BwdCommon& c, int QH, int KH, float sm_scale) {
  NsaBwdTileParams p{};
  p.q = (const bf16_t*)c.q; p.q_st = c.q_st; p.q_sh = c.q_sh;
  p.k = (const bf16_t*)c.k; p.k_sr = c.k_sr; p.k_sh = c.k_sh;
  p.v = (const bf16_t*)c.v; p.v_sr = c.v_sr; p.v_sh = c.v_sh;
  p.dO = (const bf16_t*)c.dO; p.do_st = c.do_st; p.do_sh = c.do_sh;
  p.lse = c.lse; p.lse_st = c.lse_st; p.lse_sh = c.lse_sh;
  p.delta = c.delta; p.delta_st = c.delta_st; p.delta_sh = c.delta_sh;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E; p.sm_scale = sm_scale;
  p.kernel_size = 1; p.stride = 1; p.window = 0;
  return p;
}
}  // namespace

extern "C" {

static int cmp_bwd_dq_impl(const char* who, const BwdCommon& c, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode,
                           float* dq_partial, int64_t dqp_st, int64_t dqp_sh, const int32_t* x_cu,
                           const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                           int stride, float sm_scale, void* stream, int final_below = 0) {
  int rc = check_heads(who, QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes(who, kernel_size, stride, 0);
  if (rc) return rc;
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.dq_partial = dq_partial; p.dqp_st = dqp_st; p.dqp_sh = dqp_sh;
  p.x_cu = x_cu; p.k_cu = y_cu;
  p.kernel_size = kernel_size; p.stride = stride;
  p.all_below = final_below;
  return nsa_bwd_dq_tile_launch(p, 0, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_cmp_attn_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                        const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu,
                        const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                        int stride, float sm_scale, void* stream) {
  NSA_REQUIRE(dq_mode >= 0 && dq_mode <= 2, NSA_ERR_BAD_ARG, "cmp_attn_bwd_dq: dq_mode %d not in {0,1,2}", dq_mode);
  BwdCommon c{q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
              delta_st, delta_sh};
  return cmp_bwd_dq_impl("cmp_attn_bwd_dq", c, dq, dq_st, dq_sh, dq_mode, nullptr, 0, 0, x_cu, y_cu, B, x_maxlen, QH,
                         KH, D, VD, kernel_size, stride, sm_scale, stream);
}

int nsa_cmp_attn_bwd_dq_final(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                              int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                              int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                              const float* delta, int64_t delta_st, int64_t delta_sh, const float* dq_partial,
                              int64_t dqp_st, int64_t dqp_sh, void* dq, int64_t dq_st, int64_t dq_sh,
                              const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                              int VD, int kernel_size, int stride, float sm_scale, void* stream) {
  NSA_REQUIRE(dq_partial != nullptr && dq != nullptr, NSA_ERR_BAD_ARG, "cmp_attn_bwd_dq_final: null dq buffers");
  BwdCommon c{q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
              delta_st, delta_sh};
  return cmp_bwd_dq_impl("cmp_attn_bwd_dq_final", c, dq, dq_st, dq_sh, 3, const_cast<float*>(dq_partial), dqp_st, dqp_sh,
                         x_cu, y_cu, B, x_maxlen, QH, KH, D, VD, kernel_size, stride, sm_scale, stream);
}

int nsa_cmp_attn_bwd_dq_final_below(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                                    int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                                    int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                                    const float* delta, int64_t delta_st, int64_t delta_sh, float* dq_partial,
                                    int64_t dqp_st, int64_t dqp_sh, void* dq, int64_t dq_st, int64_t dq_sh, int final_below,
                                    const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                                    int VD, int kernel_size, int stride, float sm_scale, void* stream) {
  NSA_REQUIRE(dq_partial != nullptr && dq != nullptr, NSA_ERR_BAD_ARG, "cmp_attn_bwd_dq_final_below: null dq buffers");
  BwdCommon c{q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
              delta_st, delta_sh};
  return cmp_bwd_dq_impl("cmp_attn_bwd_dq_final_below", c, dq, dq_st, dq_sh, 4, dq_partial, dqp_st, dqp_sh, x_cu, y_cu, B,
                         x_maxlen, QH, KH, D, VD, kernel_size, stride, sm_scale, stream, final_below);
}

// Cost model of a dk/dv work item (128 keys x some query rows, 4 waves): fixed part (K / V fragments, epilogue, summing up)
// and time per 64-row tile, alone on a CU (tile_us) and as the CU's throughput with `per_cu` of them on it (cu_tile_us).
// Measured on MI355X; 8 / 16 / 32 / 64 heads per kv head with 64 or 128 channels: nsa_bwd_dkdv_dma.hip, the others on
// nsa_bwd_dkdv.hip.  192 / 128 channels run in the former but keep the latter's row (3.2 us per tile, where 2.65 are measured;
// the comparisons that the rules make hardly move).  us of the cut that the rules take and of the best one there, 32 q / 2 kv
// heads: compressed, 1200 tokens 41 / 41, 4K 67 / 67, 16K 595 / 567, 64K 7094 / 7094, 8 x 6K 763 / 762, 64 / 4 heads 16K 966 /
// 966; window, 1200 tokens 74 / 74, 4K 144 / 144, 16K 561 / 545, 64K 2033 / 1999, 8 x 6K 1813 / 1679, 64 / 4 heads 16K 1023 /
// 1015.
struct DkdvCost {
  double fixed_us, tile_us, cu_tile_us;
  int per_cu;
  int slots() const { return per_cu * nsa_device_cus(); }
  // one of `items` work items of `tiles` tiles, as many of them on a CU as there are
  double item(int64_t items, double tiles) const {
    const int64_t on_cu = (items + nsa_device_cus() - 1) / nsa_device_cus();
    const double shared = (on_cu < per_cu ? on_cu : per_cu) * cu_tile_us;
    return fixed_us + tiles * (shared > tile_us ? shared : tile_us);
  }
};
static DkdvCost dkdv_cost(int G, int D, int VD) {
  const bool dma = G == 8 || G == 16 || G == 32 || G == 64;
  if (dma && D == 128) return {14.0, 2.3, 2.03, 2};
  if (dma && D == 64) return {13.0, 1.45, 1.13, 3};
  if (D <= 64) return {12.0, 0.95, 0.95, 2};
  return {12.0, 2.55 * (D + VD) / 256.0, 2.55 * (D + VD) / 256.0, 1};
}

// Query tokens per work item of the compressed dk/dv kernel when the caller leaves the choice to the library.
static int cmp_dkdv_q_chunk(int q_chunk_tokens, int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                            int kernel_size, int stride, int lo = 0) {
  if (q_chunk_tokens <= 0) {
    // A work item is one (128-key tile, query chunk that sees it, kv head, sequence).  The launch takes as long as its
    // longest item when there are fewer items than workgroup slots, else about all the work over the slots plus a
    // quarter of an item for the last, partly empty round.  The chunk (a power of two in [32, 2048]) that minimises
    // this for the longest sequence (its queries from position lo on) is taken.  Fitted to sweeps of all chunks over one to
    // forty sequences of 600 to 64K tokens (chunk 64 / 128 / 256 / 512 / 2048, d = 128: 16 q / 1 kv heads, 4096 tokens 53 /
    // 86 / 157 / 304 / 1150 us; 64 / 4 heads, 16K tokens 701 / 587 / 610 / 726 / 1166 us, 64K 10.3 / 9.3 / 8.6 / 8.1 / 8.8
    // ms).
    const int G = QH / KH;
    const DkdvCost c = dkdv_cost(G, D, VD);
    double best = 0.0;
    for (int chunk = 32; chunk <= 2048; chunk *= 2) {
      const int64_t nch = (x_maxlen - lo + chunk - 1) / chunk;
      int64_t items = 0;
      double rows = 0.0;
      for (int64_t kt = 0; kt * 128 < y_maxlen; kt++) {
        const int64_t at = (int64_t)stride * kt * 128 + kernel_size - 1, first = at > lo ? at - lo : 0;
        if (first >= x_maxlen - lo) break;
        items += nch - first / chunk;
        rows += (double)(x_maxlen - lo - first) * G;
      }
      items *= (int64_t)B * KH;
      rows *= (double)B * KH;
      const int n = chunk < x_maxlen - lo ? chunk : x_maxlen - lo;
      const double item = c.item(items, (double)n * G / 64.0);
      const double all = items * c.fixed_us / c.slots() + rows / 64.0 * c.cu_tile_us / nsa_device_cus() + 0.25 * item;
      const double cost = items <= c.slots() || all < item ? item : all;
      if (q_chunk_tokens <= 0 || cost < best) { best = cost; q_chunk_tokens = chunk; }
    }
  }
  return q_chunk_tokens;
}

static int cmp_attn_bwd_dkdv_impl(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                                  int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                                  int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                                  const float* delta, int64_t delta_st, int64_t delta_sh, float* dck, int64_t dck_sr,
                                  int64_t dck_sh, float* dcv, int64_t dcv_sr, int64_t dcv_sh, const int32_t* x_cu,
                                  const int32_t* y_cu, int B, int x_maxlen, int y_maxlen, int QH, int KH, int D,
                                  int VD, int kernel_size, int stride, int q_chunk_tokens, float sm_scale,
                                  bool deterministic, void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = check_heads("cmp_attn_bwd_dkdv", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("cmp_attn_bwd_dkdv", kernel_size, stride, 0);
  if (rc) return rc;
  q_chunk_tokens = cmp_dkdv_q_chunk(q_chunk_tokens, B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride);
  BwdCommon c{q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
              delta_st, delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dck; p.dk_sr = dck_sr; p.dk_sh = dck_sh;
  p.dv = dcv; p.dv_sr = dcv_sr; p.dv_sh = dcv_sh;
  p.dkv_mode = 3;
  p.x_cu = x_cu; p.k_cu = y_cu;
  p.kernel_size = kernel_size; p.stride = stride;
  p.q_chunk_tokens = q_chunk_tokens;
  if (!deterministic) return nsa_bwd_dkdv_launch(p, 0, B, x_maxlen, y_maxlen, D, VD, 0, (hipStream_t)stream);
  if (B <= 0 || y_maxlen <= 0) return NSA_OK;
  // every work item stores into its own slot, then one pass sums the slots of a key in ascending chunk order
  const int64_t slots = nsa_bwd_dkdv_cmp_slots(B, KH, x_maxlen, y_maxlen, D, q_chunk_tokens, kernel_size, stride, 0, 0,
                                               B);
  const int64_t kw = nsa_bwd_dkdv_slot_keys(0, 0, D);
  const int64_t dk_bytes = (slots * kw * D * 4 + 255) & ~(int64_t)255;
  const int64_t need = dk_bytes + slots * kw * VD * 4;
  NSA_REQUIRE(workspace != nullptr && workspace_bytes >= need, NSA_ERR_WORKSPACE,
              "cmp_attn_bwd_dkdv_det: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
              (long long)need);
  p.dkv_mode = 4;
  p.part_dk = (float*)workspace;
  p.part_dv = (float*)((char*)workspace + dk_bytes);
  rc = nsa_bwd_dkdv_launch(p, 0, B, x_maxlen, y_maxlen, D, VD, 0, (hipStream_t)stream);
  if (rc) return rc;
  return nsa_dkdv_reduce_cmp_launch(p, false, B, x_maxlen, y_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_cmp_attn_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                          const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st,
                          int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                          int64_t delta_st, int64_t delta_sh, float* dck, int64_t dck_sr, int64_t dck_sh,
                          float* dcv, int64_t dcv_sr, int64_t dcv_sh, const int32_t* x_cu, const int32_t* y_cu,
                          int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                          int stride, int q_chunk_tokens, float sm_scale, void* stream) {
  return cmp_attn_bwd_dkdv_impl(q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st,
                                lse_sh, delta, delta_st, delta_sh, dck, dck_sr, dck_sh, dcv, dcv_sr, dcv_sh, x_cu,
                                y_cu, B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, q_chunk_tokens,
                                sm_scale, false, nullptr, 0, stream);
}

int64_t nsa_cmp_attn_bwd_dkdv_det_bytes(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                                        int kernel_size, int stride, int q_chunk_tokens) {
  if (B <= 0 || x_maxlen <= 0 || y_maxlen <= 0 || KH <= 0 || QH <= 0 || stride <= 0) return 0;
  q_chunk_tokens = cmp_dkdv_q_chunk(q_chunk_tokens, B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride);
  const int64_t slots = nsa_bwd_dkdv_cmp_slots(B, KH, x_maxlen, y_maxlen, D, q_chunk_tokens, kernel_size, stride, 0, 0,
                                               B);
  const int64_t kw = nsa_bwd_dkdv_slot_keys(0, 0, D);
  return ((slots * kw * D * 4 + 255) & ~(int64_t)255) + slots * kw * VD * 4;
}

int nsa_cmp_attn_bwd_dkdv_det(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                              int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                              int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                              const float* delta, int64_t delta_st, int64_t delta_sh, float* dck, int64_t dck_sr,
                              int64_t dck_sh, float* dcv, int64_t dcv_sr, int64_t dcv_sh, const int32_t* x_cu,
                              const int32_t* y_cu, int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                              int kernel_size, int stride, int q_chunk_tokens, float sm_scale, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  return cmp_attn_bwd_dkdv_impl(q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st,
                                lse_sh, delta, delta_st, delta_sh, dck, dck_sr, dck_sh, dcv, dcv_sr, dcv_sh, x_cu,
                                y_cu, B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, q_chunk_tokens,
                                sm_scale, true, workspace, workspace_bytes, stream);
}



int nsa_slc_bwd_chunk_tokens(int T, int KH, int top_n) {
  // List chunk (tokens per work item of the selected-attention dk/dv pass; T: the tokens of one call, a range of the batch
  // where the dS is stored).  An item of 256 tokens alone takes 110 us at 128 channels (16 q-heads per kv head), so a batch that
  // has fewer of them than the 512 workgroups the GPU holds (two per CU at 128 channels) takes that long whatever its size: it
  // is cut finer, down to 64.  Longer items than 256 only add imbalance; shorter ones than the GPU needs add K / V loads and
  // fp32 atomics.  us of the kernel that stores dS at 32 / 64 / 128 / 256 / 512 / 1024 tokens, the rule's marked: 16 q / 1 kv
  // heads of 128, 2K tokens 86 / *59 / 70 / 114 / 212 / 409, 4K 162 / 122 / *103 / 120 / 210 / 408, 8K 302 / 240 / 244 / *265 /
  // 274 / 411, 16K 548 / 469 / 438 / *468 / 574 / 508; 64 / 4 heads, 4K 512 / 407 / 379 / *381 / 475 / 505, 16K 2207 / 1755 /
  // 1624 / *1619 / 1603 / 1713, 8 x 6K 7108 / 5634 / 5226 / *5228 / 5395 / 5836, 64K 9276 / 7355 / 6759 / *6530 / 6617 / 6773;
  // 32 / 2 heads of 192 (one workgroup per CU), 4K 524 / 424 / 353 / *319 / 529 / 567, 16K 2204 / 1640 / 1427 / *1377 / 1431 /
  // 1450; 16 / 2 heads of 64, 2K 65 / 51 / *38 / 55 / 75 / 140, 16K 431 / 300 / 271 / *264 / 279 / 300, 40 samples of up to
  // 1.2K 321 / 216 / 181 / *191 / 225 / 253.
  const int64_t want = (int64_t)KH * T * top_n / 512;
  int c = 64;
  while (c < 256 && c * 2 <= want) c *= 2;
  return c;
}

int nsa_swa_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                   const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                   const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                   int64_t delta_sh, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu,
                   int B, int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream) {
  int rc = check_heads("swa_bwd_dq", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(dq_mode >= 0 && dq_mode <= 2, NSA_ERR_BAD_ARG, "swa_bwd_dq: dq_mode %d not in {0,1,2}", dq_mode);
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.window = window;
  return nsa_bwd_dq_tile_launch(p, 1, B, x_maxlen, D, VD, (hipStream_t)stream);
}

static int swa_bwd_dq_tail_impl(int dq_mode, const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh, const float* slc_lse,
                        int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                        int all_below, float* dq, int64_t dq_st, int64_t dq_sh, const int32_t* x_cu, int B,
                        int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream) {
  int rc = check_heads("swa_bwd_dq_tail", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0 && all_below >= 0, NSA_ERR_BAD_ARG, "swa_bwd_dq_tail: window %d and all_below %d must be >= 0",
              window, all_below);
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.window = window;
  p.all_below = all_below;
  p.dO2 = (const bf16_t*)slc_dO; p.do2_st = sdo_st; p.do2_sh = sdo_sh;
  p.lse2 = slc_lse; p.lse2_st = sl_st; p.lse2_sh = sl_sh;
  p.delta2 = slc_delta; p.delta2_st = sd_st; p.delta2_sh = sd_sh;
  return nsa_bwd_dq_tile_launch(p, 2, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_bwd_dq_dense(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh, const void* v, int64_t v_sr,
                     int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                     const float* delta, int64_t delta_st, int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh,
                     const float* slc_lse, int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                     int all_below, const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh,
                     const void* cmp_dO, int64_t cdo_st, int64_t cdo_sh, const float* cmp_lse, int64_t cl_st, int64_t cl_sh,
                     const float* cmp_delta, int64_t cd_st, int64_t cd_sh, void* dq, int64_t dq_st, int64_t dq_sh, float* dq_partial,
                     int64_t dqp_st, int64_t dqp_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH,
                     int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream) {
  int rc = check_heads("bwd_dq_dense", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("bwd_dq_dense", kernel_size, stride, 0);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0 && all_below >= 0, NSA_ERR_BAD_ARG, "bwd_dq_dense: window %d and all_below %d must be >= 0", window,
              all_below);
  NSA_REQUIRE(dq != nullptr && (dq_partial != nullptr || x_maxlen <= all_below), NSA_ERR_BAD_ARG, "bwd_dq_dense: null dq buffers");
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh;
  p.dq_partial = dq_partial; p.dqp_st = dqp_st; p.dqp_sh = dqp_sh;
  p.x_cu = x_cu; p.k_cu = x_cu; p.c_cu = y_cu;
  p.kernel_size = kernel_size; p.stride = stride; p.window = window;
  p.all_below = all_below;
  p.dO2 = (const bf16_t*)slc_dO; p.do2_st = sdo_st; p.do2_sh = sdo_sh;
  p.lse2 = slc_lse; p.lse2_st = sl_st; p.lse2_sh = sl_sh;
  p.delta2 = slc_delta; p.delta2_st = sd_st; p.delta2_sh = sd_sh;
  p.ck = (const bf16_t*)ck; p.ck_sr = ck_sr; p.ck_sh = ck_sh;
  p.cv = (const bf16_t*)cv; p.cv_sr = cv_sr; p.cv_sh = cv_sh;
  p.dO3 = (const bf16_t*)cmp_dO; p.do3_st = cdo_st; p.do3_sh = cdo_sh;
  p.lse3 = cmp_lse; p.lse3_st = cl_st; p.lse3_sh = cl_sh;
  p.delta3 = cmp_delta; p.delta3_st = cd_st; p.delta3_sh = cd_sh;
  return nsa_bwd_dq_tile_launch(p, 3, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_swa_bwd_dq_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh, const float* slc_lse,
                        int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                        int all_below, float* dq, int64_t dq_st, int64_t dq_sh, const int32_t* x_cu, int B,
                        int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream) {
  return swa_bwd_dq_tail_impl(2, q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
                              delta_sh, slc_dO, sdo_st, sdo_sh, slc_lse, sl_st, sl_sh, slc_delta, sd_st, sd_sh, all_below, dq,
                              dq_st, dq_sh, x_cu, B, x_maxlen, QH, KH, D, VD, window, sm_scale, stream);
}

int nsa_swa_bwd_dq_tail_store(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                              const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                              const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                              int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh, const float* slc_lse,
                              int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                              int all_below, float* dq, int64_t dq_st, int64_t dq_sh, const int32_t* x_cu, int B,
                              int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream) {
  return swa_bwd_dq_tail_impl(1, q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
                              delta_sh, slc_dO, sdo_st, sdo_sh, slc_lse, sl_st, sl_sh, slc_delta, sd_st, sd_sh, all_below, dq,
                              dq_st, dq_sh, x_cu, B, x_maxlen, QH, KH, D, VD, window, sm_scale, stream);
}

// bytes of the partial dk / dv of the window branch with `splits` query chunks per key tile; dk_bytes: those of dk
static int64_t swa_dkdv_slot_bytes(int splits, int B, int x_maxlen, int KH, int D, int VD, int64_t* dk_bytes) {
  const int64_t kw = nsa_bwd_dkdv_slot_keys(1, 0, D);
  const int64_t rows = (x_maxlen + kw - 1) / kw * B * KH * splits * kw;
  *dk_bytes = (rows * D * 4 + 255) & ~(int64_t)255;
  return *dk_bytes + rows * VD * 4;
}

// Query chunks per key tile of the window branch's dk/dv; at most max_bytes of partial results.  tokens: of the batch, where the
// caller knows.
static int swa_dkdv_splits(int B, int x_maxlen, int QH, int KH, int D, int VD, int window, int64_t max_bytes,
                           int tokens = 0) {
  if (B <= 0 || x_maxlen <= 0 || QH <= 0 || KH <= 0) return 1;
  const int knob = nsa_tuning_knob("swa_dkdv_splits", 0);
  if (knob > 0) return knob > 16 ? 16 : knob;
  // A key tile's queries are cut while the rounds of workgroups times the time of one keeps falling (by a tenth at
  // least: every cut adds a pass over partial results).  1 / 2 / 4 / 8 / 16 chunks, their sum included, d = 128: one
  // sequence of 4096 tokens, 16 q / 1 kv heads 365 / 196 / 110 / 70 / 63 us, 64 q / 4 kv heads 389 / 224 / 167 / 206 /
  // 256 us; 8192 tokens, 64 q / 4 kv heads 422 / 333 / 370 / 397 / 486 us.
  const DkdvCost c = dkdv_cost(QH / KH, D, VD);
  int64_t wgs = (int64_t)((x_maxlen + 127) / 128) * B * KH;
  if (tokens > 0 && ((int64_t)tokens / 128 + B) * KH < wgs) wgs = ((int64_t)tokens / 128 + B) * KH;
  const double tiles = (128.0 + (window < x_maxlen ? window : x_maxlen)) * (QH / KH) / 64.0;
  int best = 1;
  double best_cost = 0.0;
  int64_t dk_bytes;
  for (int s = 1; s <= 16; s *= 2) {
    if (s > 1 && swa_dkdv_slot_bytes(s, B, x_maxlen, KH, D, VD, &dk_bytes) > max_bytes) break;
    const double cost = (double)((wgs * s + c.slots() - 1) / c.slots()) * c.item(wgs * s, tiles / s);
    if (s == 1 || cost < 0.9 * best_cost) { best = s; best_cost = cost; }
  }
  return best;
}

// (the batches that gain from cuts have few key tiles: 64 MB is 512 work items of 128 keys and 128 channels)
static const int64_t SWA_SLOTS_LIMIT = (int64_t)64 << 20;

int64_t nsa_swa_bwd_dkdv_ws_bytes(int B, int x_maxlen, int QH, int KH, int D, int VD, int window) {
  const int splits = swa_dkdv_splits(B, x_maxlen, QH, KH, D, VD, window, SWA_SLOTS_LIMIT);
  int64_t dk_bytes;
  return splits > 1 ? swa_dkdv_slot_bytes(splits, B, x_maxlen, KH, D, VD, &dk_bytes) : 0;
}

int nsa_swa_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                     const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                     int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                     int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                     int VD, int window, float sm_scale, void* stream) {
  return nsa_swa_bwd_dkdv_ws(q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
                             delta_st, delta_sh, dk, dk_sr, dk_sh, dv, dv_sr, dv_sh, dkv_is_f32, x_cu, B, x_maxlen, QH,
                             KH, D, VD, window, sm_scale, nullptr, 0, stream);
}

int nsa_swa_bwd_dkdv_ws(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                        int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                        int D, int VD, int window, float sm_scale, void* workspace, int64_t workspace_bytes,
                        void* stream) {
  int rc = check_heads("swa_bwd_dkdv", QH, KH, D, VD);
  if (rc) return rc;
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = dkv_is_f32 ? 1 : 0;
  p.grid_chunks = workspace != nullptr ? swa_dkdv_splits(B, x_maxlen, QH, KH, D, VD, window, SWA_SLOTS_LIMIT) : 1;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.window = window;
  if (p.grid_chunks == 1) return nsa_bwd_dkdv_launch(p, 1, B, x_maxlen, x_maxlen, D, VD, 0, (hipStream_t)stream);
  int64_t dk_bytes;
  const int64_t need = swa_dkdv_slot_bytes(p.grid_chunks, B, x_maxlen, KH, D, VD, &dk_bytes);
  NSA_REQUIRE(workspace_bytes >= need, NSA_ERR_WORKSPACE, "swa_bwd_dkdv: workspace of %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)need);
  p.dkv_mode = 4;
  p.part_dk = (float*)workspace;
  p.part_dv = (float*)((char*)workspace + dk_bytes);
  rc = nsa_bwd_dkdv_launch(p, 1, B, x_maxlen, x_maxlen, D, VD, 0, (hipStream_t)stream);
  if (rc) return rc;
  return nsa_dkdv_reduce_swa_launch(p, dkv_is_f32 != 0, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_slc_attn_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st, void* dq,
                        int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu, int B, int x_maxlen, int QH,
                        int KH, int D, int VD, int block_size, int top_n, float sm_scale, void* stream) {
  return nsa_slc_attn_bwd_dq_from(q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh,
                                  delta, delta_st, delta_sh, topk, tk_sh, tk_st, dq, dq_st, dq_sh, dq_mode, x_cu, B,
                                  x_maxlen, QH, KH, D, VD, block_size, top_n, 0, sm_scale, stream);
}

int nsa_slc_attn_bwd_dq_from(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st, void* dq,
                        int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu, int B, int x_maxlen, int QH,
                        int KH, int D, int VD, int block_size, int top_n, int t_begin,
                        float sm_scale, void* stream) {
  int rc = check_heads("slc_attn_bwd_dq", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(block_size % 32 == 0 && block_size > 0, NSA_ERR_UNSUPPORTED,
              "slc_attn_bwd_dq: block_size %d must be a multiple of 32", block_size);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "slc_attn_bwd_dq: top_n %d must be in [1,64]", top_n);
  NSA_REQUIRE(dq_mode >= 0 && dq_mode <= 2, NSA_ERR_BAD_ARG, "slc_attn_bwd_dq: dq_mode %d not in {0,1,2}", dq_mode);
  rc = check_positions("slc_attn_bwd_dq", t_begin);
  if (rc) return rc;
  NsaSlcBwdDqParams p{};
  p.t_begin = t_begin;
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v; p.v_sr = v_sr; p.v_sh = v_sh;
  p.dO = (const bf16_t*)dO; p.do_st = do_st; p.do_sh = do_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.delta = delta; p.delta_st = delta_st; p.delta_sh = delta_sh;
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.x_cu = x_cu;
  p.G = QH / KH; p.KH = KH; p.top_n = top_n; p.block_size = block_size;
  p.scale_log2 = sm_scale * NSA_LOG2E; p.sm_scale = sm_scale;
  return nsa_slc_bwd_dq_launch(p, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_slc_attn_bwd_dkdv_before_window(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr,
                                        int64_t k_sh, const void* v, int64_t v_sr, int64_t v_sh, const void* dO,
                                        int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st,
                                        int64_t lse_sh, const float* delta, int64_t delta_st, int64_t delta_sh,
                                        float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                                        int64_t dv_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                                        int D, int VD, int window, int all_below, int ordered, float sm_scale,
                                        void* stream) {
  int rc = check_heads("slc_attn_bwd_dkdv_before_window", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0 && all_below >= 0, NSA_ERR_BAD_ARG,
              "slc_attn_bwd_dkdv_before_window: window %d and all_below %d must be >= 0", window, all_below);
  const int len = (x_maxlen < all_below ? x_maxlen : all_below) - window - 1;  // positions that are some query's keys
  if (len <= 0) return NSA_OK;
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = 3;
  // one workgroup per key tile adds exactly once to every element: no order to vary
  p.grid_chunks = ordered ? 1 : swa_dkdv_splits(B, len, QH, KH, D, VD, len, INT64_MAX);
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.min_dist = window + 1; p.window = all_below; p.t_end = all_below;
  return nsa_bwd_dkdv_launch(p, 1, B, x_maxlen, x_maxlen, D, VD, 0, (hipStream_t)stream);
}

static int slc_attn_bwd_dkdv_impl(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                          const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st,
                          int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                          int64_t delta_st, int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh, float* dv,
                          int64_t dv_sr, int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu,
                          const int32_t* blk_seq, const int32_t* csr_off, const int32_t* csr_tok,
                          const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B,
                          int QH, int KH, int D, int VD, int block_size, float sm_scale, bool deterministic,
                          void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = check_heads("slc_attn_bwd_dkdv", QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(block_size % 32 == 0 && block_size > 0, NSA_ERR_UNSUPPORTED,
              "slc_attn_bwd_dkdv: block_size %d must be a multiple of 32", block_size);
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = 3;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.csr_off = csr_off; p.csr_tok = csr_tok; p.item_off = item_off; p.blk_seq = blk_seq; p.kblk_cu = kblk_cu;
  p.nblk_total = nblk_total; p.chunk_tokens = chunk_tokens; p.block_size = block_size;
  p.csr_sh = nblk_total + 1;
  if (!deterministic) return nsa_bwd_dkdv_launch(p, 2, B, 0, 0, D, VD, n_items_bound, (hipStream_t)stream);
  if (n_items_bound <= 0) return NSA_OK;
  const int64_t slots = nsa_bwd_dkdv_slc_slots(KH, n_items_bound, block_size);
  const int64_t kw = nsa_bwd_dkdv_slot_keys(2, block_size, D);
  const int64_t dk_bytes = (slots * kw * D * 4 + 255) & ~(int64_t)255;
  const int64_t need = dk_bytes + slots * kw * VD * 4;
  NSA_REQUIRE(workspace != nullptr && workspace_bytes >= need, NSA_ERR_WORKSPACE,
              "slc_attn_bwd_dkdv_det: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
              (long long)need);
  p.dkv_mode = 4;
  p.part_dk = (float*)workspace;
  p.part_dv = (float*)((char*)workspace + dk_bytes);
  rc = nsa_bwd_dkdv_launch(p, 2, B, 0, 0, D, VD, n_items_bound, (hipStream_t)stream);
  if (rc) return rc;
  return nsa_dkdv_reduce_slc_launch(p, n_items_bound, D, VD, (hipStream_t)stream);
}

int nsa_slc_attn_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                          const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st,
                          int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                          int64_t delta_st, int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh, float* dv,
                          int64_t dv_sr, int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu,
                          const int32_t* blk_seq, const int32_t* csr_off, const int32_t* csr_tok,
                          const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B,
                          int QH, int KH, int D, int VD, int block_size, float sm_scale, void* stream) {
  return slc_attn_bwd_dkdv_impl(q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh,
                                delta, delta_st, delta_sh, dk, dk_sr, dk_sh, dv, dv_sr, dv_sh, x_cu, kblk_cu, blk_seq,
                                csr_off, csr_tok, item_off, nblk_total, chunk_tokens, n_items_bound, B, QH, KH, D, VD,
                                block_size, sm_scale, false, nullptr, 0, stream);
}

int64_t nsa_slc_attn_bwd_dkdv_det_bytes(int n_items_bound, int KH, int D, int VD, int block_size) {
  if (n_items_bound <= 0 || KH <= 0 || block_size <= 0) return 0;
  const int64_t slots = nsa_bwd_dkdv_slc_slots(KH, n_items_bound, block_size);
  const int64_t kw = nsa_bwd_dkdv_slot_keys(2, block_size, D);
  return ((slots * kw * D * 4 + 255) & ~(int64_t)255) + slots * kw * VD * 4;
}

int nsa_slc_attn_bwd_dkdv_det(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                              const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st,
                              int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                              int64_t delta_st, int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh,
                              float* dv, int64_t dv_sr, int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu,
                              const int32_t* blk_seq, const int32_t* csr_off, const int32_t* csr_tok,
                              const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B,
                              int QH, int KH, int D, int VD, int block_size, float sm_scale, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  return slc_attn_bwd_dkdv_impl(q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh,
                                delta, delta_st, delta_sh, dk, dk_sr, dk_sh, dv, dv_sr, dv_sh, x_cu, kblk_cu, blk_seq,
                                csr_off, csr_tok, item_off, nblk_total, chunk_tokens, n_items_bound, B, QH, KH, D, VD,
                                block_size, sm_scale, true, workspace, workspace_bytes, stream);
}

// dK / dV and dQ of the selected branch in one go: the dK/dV kernel leaves the dS of every (token, block) behind, and dQ = dS K
// gathers half of what the kernel gathers that computes S and dP again.  Both kernels alone on the GPU, 64 heads of 128: 64K
// tokens dQ 10.3 -> 5.55, dK/dV 6.4 -> 6.7 ms, 8 x 6K tokens 5.2 -> 2.93 and 3.84 -> 4.01 ms.
// The dS of a token takes 32 KB per kv head (16 q-heads, 16 blocks of 64 keys), and 2 GB of it in flight do: longer batches
// are cut into ranges of tokens (64K tokens, whole step with 1 / 2 / 4 / 8.6 GB: 55.5 / 55.3 / 55.7 / 56.3 ms; 32K tokens 20.5
// / 20.6 / 20.5 / 20.5 ms).  The ranges do not grow with the batch, so a block's list per range gets shorter: index, dK/dV and
// dQ with dq recomputed / with 1 / 2 / 4 / 8 GB, ms, 64 heads: 128K tokens 38.7 / 28.8 / 27.6 / 28.3 / 28.5, 256K 86.4 / 66.5 /
// 61.0 / 60.9 / 62.1, 512K 184 / 172 / 147 / 144 / 144.  Shapes of which 2 GB do not hold 512 tokens (8 kv heads of 16 q-heads
// with 64 blocks of 512 keys: 4 GB) compute dq and dk/dv apart: the lists of such ranges would be a few tokens long.
// No rule on the number of tokens: a query's dq is to be the same bits whatever follows it in the batch.  Steps with dq
// recomputed / from the dS, us: 16 heads of 128, 16K tokens 2315 / 2277; 64 heads, 4K 1730 / 1744, 8K 3980 / 3863; 32 heads of
// 192, 4K 1340 / 1402, 16K 6660 / 6630; 16 heads of 64 in 2 groups, 16K 1632 / 1642, 48K 6448 / 6105.
static bool slc_bwd_ds_takes(int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, int block_size,
                             int top_n, float sm_scale) {
  if (KH <= 0 || QH % KH != 0 || block_size <= 0 || block_size % 32 != 0 || block_size > 2048) return false;
  if (top_n < 1 || top_n > 64 || k_sr < 0 || k_sr >= (1 << 27)) return false;
  NsaBwdTileParams p{};
  p.G = QH / KH; p.q_sh = q_sh; p.do_sh = do_sh; p.scale_log2 = sm_scale * NSA_LOG2E;
  return nsa_bwd_dkdv_dma_takes(p, D, VD);
}

int nsa_slc_bwd_ds_tokens(int T, int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, int block_size,
                          int top_n, float sm_scale) {
  if (T <= 0 || !slc_bwd_ds_takes(q_sh, do_sh, k_sr, QH, KH, D, VD, block_size, top_n, sm_scale)) return 0;
  const int64_t budget = (int64_t)nsa_tuning_knob("slc_ds_mb", 2048) << 20;
  const int64_t per_token = nsa_slc_ds_entry_elems(QH / KH, block_size) * 2 * top_n * KH;
  if (budget <= 0) return 0;
  const int64_t fit = budget / per_token;
  if (fit < 512) return 0;
  if (fit >= T) return T;
  const int64_t ranges = (T + fit - 1) / fit;
  return (int)((T + ranges - 1) / ranges);
}

int64_t nsa_slc_bwd_ds_bytes(int ntok, int QH, int KH, int block_size, int top_n) {
  if (ntok <= 0) return 0;
  const int G = QH / KH;
  // per kv head one more entry, for the dS of rows that stand for nothing
  return KH * ((int64_t)ntok * top_n + 1) * nsa_slc_ds_entry_elems(G, block_size) * 2;
}

static int slc_ds_check(const char* who, int QH, int KH, int D, int VD, int block_size, int top_n, int tok0, int ntok, int B,
                        const void* ds, int64_t ds_bytes, bool takes) {
  int rc = check_heads(who, QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(tok0 >= 0 && ntok >= 0 && B >= 1, NSA_ERR_BAD_ARG, "%s: tokens %d + %d of %d sequences", who, tok0, ntok, B);
  NSA_REQUIRE(takes, NSA_ERR_UNSUPPORTED, "%s: these shapes take slc_attn_bwd_dq and slc_attn_bwd_dkdv", who);
  const int64_t need = nsa_slc_bwd_ds_bytes(ntok, QH, KH, block_size, top_n);
  NSA_REQUIRE(ntok == 0 || (ds != nullptr && ds_bytes >= need), NSA_ERR_WORKSPACE, "%s: dS buffer of %lld bytes, %lld needed", who,
              (long long)ds_bytes, (long long)need);
  return NSA_OK;
}

int nsa_slc_attn_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                             const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                             const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                             int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                             int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu, const int32_t* blk_seq,
                             const int32_t* csr_off, const int32_t* csr_tok, const uint8_t* csr_slot,
                             const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B, int QH,
                             int KH, int D, int VD, int block_size, int top_n, int tok0, int ntok, float sm_scale, void* ds,
                             int64_t ds_bytes, void* stream) {
  int rc = slc_ds_check("slc_attn_bwd_dkdv_ds", QH, KH, D, VD, block_size, top_n, tok0, ntok, B, ds, ds_bytes,
                        slc_bwd_ds_takes(q_sh, do_sh, k_sr, QH, KH, D, VD, block_size, top_n, sm_scale));
  if (rc) return rc;
  if (ntok == 0 || n_items_bound <= 0) return NSA_OK;
  NSA_REQUIRE(csr_slot != nullptr, NSA_ERR_BAD_ARG, "slc_attn_bwd_dkdv_ds: csr_slot, the place of every entry's dS, is null");
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = 3;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.csr_off = csr_off; p.csr_tok = csr_tok; p.item_off = item_off; p.blk_seq = blk_seq; p.kblk_cu = kblk_cu;
  p.nblk_total = nblk_total; p.chunk_tokens = chunk_tokens; p.block_size = block_size;
  p.csr_sh = nblk_total + 1;
  p.ds = (bf16_t*)ds; p.csr_slot = csr_slot;
  p.ds_sh = ((int64_t)ntok * top_n + 1) * nsa_slc_ds_entry_elems(p.G, block_size);
  p.ds_tok0 = tok0; p.ds_ntok = ntok; p.top_n = top_n;
  p.ds_dump = ntok * top_n * (p.G > 16 ? p.G / 16 : 1);
  NSA_REQUIRE(nsa_bwd_dkdv_dma_takes(p, D, VD), NSA_ERR_UNSUPPORTED,
              "slc_attn_bwd_dkdv_ds: chunk_tokens %d exceeds what a work item's kernel holds", chunk_tokens);
  return nsa_bwd_dkdv_launch(p, 2, B, 0, 0, D, VD, n_items_bound, (hipStream_t)stream);
}

int nsa_slc_attn_bwd_dq_ds(const void* k, int64_t k_sr, int64_t k_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st,
                           void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const float* dq_partial, int64_t dqp_st,
                           int64_t dqp_sh, const int32_t* x_cu, int B, int QH, int KH, int D, int VD, int block_size,
                           int top_n, int t_begin, int tok0, int ntok, float sm_scale, const void* ds, int64_t ds_bytes,
                           void* stream) {
  int rc = slc_ds_check("slc_attn_bwd_dq_ds", QH, KH, D, VD, block_size, top_n, tok0, ntok, B, ds, ds_bytes,
                        slc_bwd_ds_takes(0, 0, k_sr, QH, KH, D, VD, block_size, top_n, sm_scale));
  if (rc) return rc;
  NSA_REQUIRE(dq_mode >= 0 && dq_mode <= 3 && (dq_mode != 3 || dq_partial != nullptr), NSA_ERR_BAD_ARG,
              "slc_attn_bwd_dq_ds: dq_mode %d not in {0,1,2,3}, or 3 without dq_partial", dq_mode);
  rc = check_positions("slc_attn_bwd_dq_ds", t_begin);
  if (rc) return rc;
  NsaSlcDqDsParams p{};
  p.k = (const bf16_t*)k; p.k_sr = k_sr; p.k_sh = k_sh;
  p.G = QH / KH;
  p.ds = (const bf16_t*)ds; p.ds_sh = ((int64_t)ntok * top_n + 1) * nsa_slc_ds_entry_elems(p.G, block_size);
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.dq_partial = dq_partial; p.dqp_st = dqp_st; p.dqp_sh = dqp_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.x_cu = x_cu;
  p.B = B; p.KH = KH; p.top_n = top_n; p.block_size = block_size;
  p.t_begin = t_begin; p.tok0 = tok0; p.ntok = ntok;
  p.sm_scale = sm_scale;
  return nsa_slc_dq_ds_launch(p, D, (hipStream_t)stream);
}

// ---- dQ of the range-keyed branches from stored dS.  A 64-row tile's dS takes 4 KB per 32 keys that it sees.
// What it is worth: whole step with dq recomputed / from the dS, us: 64 heads of 128, 64K tokens 53.2 / 50.7 ms, 8 x 6K 20500 /
// 19060, 16K 8200 / 7760; 32 heads of 192, 16K 6500 / 5800, 20 samples of up to 2K 4700 / 4320; 16 heads of 128, 4K 850 / 711,
// 16K 2212 / 2115, 30 samples of up to 1.5K 1364 / 1201.  Not with 64 channels, whose dS is as large for half of the products:
// 16 heads in 2 groups, 16K 1602 / 1699, 48K 5810 / 6207.
namespace {
struct DsLayout {
  int tiles, seq_tiles, pitch;
  int64_t sh, bytes;  // elements per kv head, bytes in all
};
// 68 KB behind the last tile that nobody reads
DsLayout ds_layout(int64_t tiles, int seq_tiles, int pitch, int KH) {
  DsLayout l;
  l.tiles = (int)tiles; l.seq_tiles = seq_tiles; l.pitch = pitch;
  l.sh = tiles * pitch * 2048;
  l.bytes = (l.sh * KH + 68 * 512) * 2;
  return l;
}
int64_t ds_all_tiles(int T, int B, int G) { return (int64_t)T * G / 64 + B + 1; }
// compressed branch, the tokens tok0 .. tok1 - 1 (tok1 = 0: all).  Several sequences: any of them may be the longest.
DsLayout ds_layout_cmp(int T, int B, int x_maxlen, int G, int KH, int kernel_size, int stride, int tok0, int tok1) {
  const int end = B == 1 && tok1 > 0 && ((tok1 + 127) & ~127) < x_maxlen ? (tok1 + 127) & ~127 : x_maxlen;
  const int keys = end >= kernel_size ? (end - kernel_size) / stride + 1 : 0;
  int64_t tiles = ds_all_tiles(T, B, G);
  if (tok1 > 0) {
    const int64_t n = (int64_t)(tok1 - tok0 + 127) * G / 64 + B + 2;
    if (n < tiles) tiles = n;
  }
  return ds_layout(tiles, 0, keys > 0 ? (keys + 31) / 32 : 1, KH);
}
// window, and the keys before it of the queries below all_below: ranges of up to `ring` tokens (0: all in one).  The keys of a
// range leave dS for the tokens up to reach behind them, so the tiles of a range and of those are kept.
int64_t ds_ring_tiles(int T, int B, int G, int ring, int64_t reach) {
  const int64_t all = ds_all_tiles(T, B, G);
  if (ring <= 0) return all;
  const int64_t n = (ring + 127 + 128 + reach + 8) * G / 64 + B + 2;
  return n < all ? n : all;
}
DsLayout ds_layout_win(int T, int B, int x_maxlen, int G, int KH, int window, int ring) {
  const int w = window < x_maxlen ? window : x_maxlen;
  int pitch = (w + 64 / G - 1) / 32 + 2;
  if (pitch > (x_maxlen + 31) / 32) pitch = (x_maxlen + 31) / 32;
  return ds_layout(ds_ring_tiles(T, B, G, ring, w), 0, pitch > 0 ? pitch : 1, KH);
}
// pitch 0: no query has such keys
DsLayout ds_layout_far(int T, int B, int x_maxlen, int G, int KH, int window, int all_below, int ring) {
  const int end = all_below < x_maxlen ? all_below : x_maxlen;
  if ((int64_t)end - 1 - window - 1 < 0) return DsLayout{0, 0, 0, 0, 0};
  const int pitch = (end - 1 - window - 1) / 32 + 1;
  const int seq_tiles = (int)(((int64_t)end * G + 63) / 64);
  const int64_t tiles = ds_ring_tiles(T, B, G, ring, end);
  if ((int64_t)seq_tiles * B < tiles) return ds_layout((int64_t)seq_tiles * B, seq_tiles, pitch, KH);
  return ds_layout(tiles, 0, pitch, KH);
}
void set_ds(NsaBwdTileParams& p, const DsLayout& l, void* ds, int tok0, int tok1) {
  p.ds = (bf16_t*)ds; p.ds_sh = l.sh;
  p.ds_tiles = l.tiles; p.ds_seq_tiles = l.seq_tiles; p.ds_pitch = l.pitch;
  p.tok0 = tok0; p.tok1 = tok1;
}
NsaDsOperand ds_operand(const DsLayout& l, const void* k, int64_t k_sr, int64_t k_sh, const void* ds) {
  return NsaDsOperand{(const bf16_t*)k, k_sr, k_sh, (const bf16_t*)ds, l.sh, l.tiles, l.seq_tiles, l.pitch};
}
int check_ds(const char* who, int QH, int KH, int D, int VD, int T, int B, int x_maxlen, int tok0, int tok1, const void* ds,
             int64_t ds_bytes, int64_t need, bool takes) {
  int rc = check_heads(who, QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(T >= 0 && B >= 0 && x_maxlen >= 0 && x_maxlen <= T && tok0 >= 0 && tok1 >= 0 && (tok1 == 0 || tok0 < tok1),
              NSA_ERR_BAD_ARG, "%s: tokens %d to %d of %d in %d sequences", who, tok0, tok1, T, B);
  NSA_REQUIRE(takes, NSA_ERR_UNSUPPORTED, "%s: these shapes have no stored dS", who);
  NSA_REQUIRE(ds != nullptr && ds_bytes >= need, NSA_ERR_WORKSPACE, "%s: dS buffer of %lld bytes, %lld needed", who,
              (long long)ds_bytes, (long long)need);
  return NSA_OK;
}
bool bwd_ds_takes(int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, float sm_scale) {
  if (D < 128 || KH <= 0 || QH % KH != 0 || k_sr < 0 || k_sr >= (1 << 26)) return false;
  if (nsa_tuning_knob("dkdv_key_blocks", 1) == 2) return false;
  NsaBwdTileParams p{};
  p.G = QH / KH; p.q_sh = q_sh; p.do_sh = do_sh; p.scale_log2 = sm_scale * NSA_LOG2E;
  return nsa_bwd_dkdv_dma_takes(p, D, VD);
}
}  // namespace

int nsa_bwd_ds_takes(int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, float sm_scale) {
  return bwd_ds_takes(q_sh, do_sh, k_sr, QH, KH, D, VD, sm_scale);
}

int64_t nsa_cmp_attn_bwd_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int tok0,
                                  int tok1) {
  if (T <= 0 || B <= 0 || KH <= 0 || QH < KH || stride <= 0) return 0;
  return ds_layout_cmp(T, B, x_maxlen, QH / KH, KH, kernel_size, stride, tok0, tok1).bytes;
}
int64_t nsa_swa_bwd_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int window, int ring) {
  if (T <= 0 || B <= 0 || KH <= 0 || QH < KH) return 0;
  return ds_layout_win(T, B, x_maxlen, QH / KH, KH, window, ring).bytes;
}
int64_t nsa_slc_bwd_before_window_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int window, int all_below, int ring) {
  if (T <= 0 || B <= 0 || KH <= 0 || QH < KH) return 0;
  return ds_layout_far(T, B, x_maxlen, QH / KH, KH, window, all_below, ring).bytes;
}

// End of the range of tokens that begins at tok0: `budget` bytes for each branch's dS (stride 0: without the compressed branch,
// window -1: without the window, all_below 0: without the keys before it), but never fewer tokens than `least`, and no shorter
// rest; *fit: whether that holds the budget.
static int ds_range_end(int tok0, int T, int B, int x_maxlen, int G, int KH, int kernel_size, int stride, int window,
                        int all_below, int64_t budget, int least, bool* fit) {
  auto fits = [&](int tok1) {
    if (stride > 0 && ds_layout_cmp(T, B, x_maxlen, G, KH, kernel_size, stride, tok0, tok1).bytes > budget) return false;
    if (window < 0) return true;
    return ds_layout_win(T, B, x_maxlen, G, KH, window, tok1 - tok0).bytes <= budget &&
           ds_layout_far(T, B, x_maxlen, G, KH, window, all_below, tok1 - tok0).bytes <= budget;
  };
  *fit = true;
  if (fits(T)) return T;
  int lo = tok0 + least;
  *fit = lo < T && fits(lo);
  if (lo >= T) return T;
  int hi = T;  // fits(lo) or lo is the least; !fits(hi)
  while (hi - lo > 128) {
    const int mid = lo + (((hi - lo) / 2 + 127) & ~127);
    if (mid >= hi) break;
    if (fits(mid)) lo = mid; else hi = mid;
  }
  if (T - lo >= least) return lo;
  if (!*fit) return T;
  const int half = ((T - tok0) / 2 + 127) & ~127;
  return T - tok0 - half >= least ? tok0 + half : lo;
}
// 4 GB.  Whole step with 2 / 4 / 8 / 40 GB, 64 heads of 128, ms: 64K tokens 52.7 / 52.2 / 51.8 / 52.2, 8 x 6K 19.9 / 19.2 / 19.2 /
// 19.2.
static int64_t ds_budget() { return (int64_t)nsa_tuning_knob("dense_ds_mb", 4096) << 20; }
// Tokens of a range that give the dQ kernel 512 workgroups of 256 rows, and, where the budget does not hold those, the fewest: an
// eighth.  Backward of one sequence, 64 / 4 heads of 128, ms, dq recomputed / from stored dS with ranges of the budget at its end
// (tokens) / with the former whatever they take: 256K 321 / 284 (1.9K) / 282, 512K 1147 / 1001 (0.9K) / 950, 768K 2521 / 2258
// (0.5K), 1M 4406 / 4257 (256).
static int ds_least(int QH) { return (131072 / QH + 127) & ~127; }
static int ds_short(int QH) { return (16384 / QH + 127) & ~127; }

int nsa_bwd_ds_range_end(int tok0, int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int window,
                         int all_below) {
  if (T <= 0 || B <= 0 || KH <= 0 || QH < KH || tok0 < 0 || tok0 >= T) return T;
  const int G = QH / KH, longest = 1 << 24;
  const int64_t budget = ds_budget();
  // What decides whether dq comes from stored dS is not the number of tokens: a query's dq is to be the same bits whatever follows
  // it in the batch.  So where top_n * block_size is too far beyond the window for one sequence of so many tokens, there is none
  // for a shorter one either.  (Two exceptions: sequences past a million tokens, and windows of many thousand keys, which act as
  // the longest sequence's where that is shorter.)
  if (window >= 0 && ds_layout_far(longest, 1, longest, G, KH, window, all_below, 0).bytes > budget) return -1;
  bool fit;
  int end = ds_range_end(tok0, T, B, x_maxlen, G, KH, kernel_size, stride, window, all_below, budget, ds_least(QH), &fit);
  if (!fit) end = ds_range_end(tok0, T, B, x_maxlen, G, KH, kernel_size, stride, window, all_below, budget, ds_short(QH), &fit);
  return fit ? end : -1;
}

int nsa_bwd_ds_next(int tok0, int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int window) {
  if (T <= 0 || B <= 0 || KH <= 0 || QH < KH || stride <= 0 || tok0 >= T) return T;
  bool fit;
  const int end = ds_range_end(tok0, T, B, x_maxlen, QH / KH, KH, kernel_size, stride, window, 0, ds_budget(), ds_least(QH), &fit);
  return T - end < ds_least(QH) ? T : end;
}

// query tokens per work item of a range's launch (one sequence: of its share; of several, one may have any share)
static int cmp_ds_q_chunk(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD, int kernel_size, int stride,
                          int tok0, int tok1) {
  int lo, hi;
  nsa_local_range(tok0, tok1, 0, x_maxlen, lo, hi);
  if (B > 1) { lo = 0; hi = x_maxlen; }
  return cmp_dkdv_q_chunk(0, B, hi, y_maxlen, QH, KH, D, VD, kernel_size, stride, lo);
}

int64_t nsa_cmp_attn_bwd_dkdv_ds_items(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                                       int stride, int q_chunk_tokens, int tok0, int tok1) {
  if (B <= 0 || x_maxlen <= 0 || y_maxlen <= 0 || KH <= 0 || QH < KH || stride <= 0) return 0;
  if (q_chunk_tokens <= 0)
    q_chunk_tokens = cmp_ds_q_chunk(B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, tok0, tok1);
  return nsa_bwd_dkdv_cmp_slots(1, 1, x_maxlen, y_maxlen, D, q_chunk_tokens, kernel_size, stride, tok0, tok1, B);
}

int64_t nsa_cmp_attn_bwd_dkdv_ds_slot_bytes(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                                            int kernel_size, int stride, int tok0, int tok1) {
  const int64_t slots = B * (int64_t)KH *
                        nsa_cmp_attn_bwd_dkdv_ds_items(B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, 0, tok0, tok1);
  const int64_t kw = nsa_bwd_dkdv_slot_keys(0, 0, D);
  return ((slots * kw * D * 4 + 255) & ~(int64_t)255) + slots * kw * VD * 4;
}

int nsa_cmp_attn_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                             const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st, int64_t do_sh,
                             const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                             int64_t delta_sh, float* dck, int64_t dck_sr, int64_t dck_sh, float* dcv, int64_t dcv_sr,
                             int64_t dcv_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int y_maxlen,
                             int QH, int KH, int D, int VD, int kernel_size, int stride, float sm_scale, int T, int tok0,
                             int tok1, void* ds, int64_t ds_bytes, void* workspace, int64_t workspace_bytes, int add,
                             void* stream) {
  const DsLayout l = KH > 0 && QH >= KH && stride > 0
                         ? ds_layout_cmp(T, B, x_maxlen, QH / KH, KH, kernel_size, stride, tok0, tok1) : DsLayout{};
  int rc = check_ds("cmp_attn_bwd_dkdv_ds", QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, ds, ds_bytes, l.bytes,
                    bwd_ds_takes(q_sh, do_sh, ck_sr, QH, KH, D, VD, sm_scale));
  if (rc) return rc;
  rc = check_nsa_sizes("cmp_attn_bwd_dkdv_ds", kernel_size, stride, 0);
  if (rc) return rc;
  if (B <= 0 || x_maxlen <= 0 || y_maxlen <= 0) return NSA_OK;
  BwdCommon c{q, q_st, q_sh, ck, ck_sr, ck_sh, cv, cv_sr, cv_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta,
              delta_st, delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dck; p.dk_sr = dck_sr; p.dk_sh = dck_sh;
  p.dv = dcv; p.dv_sr = dcv_sr; p.dv_sh = dcv_sh;
  p.dkv_mode = 3;
  p.x_cu = x_cu; p.k_cu = y_cu;
  p.kernel_size = kernel_size; p.stride = stride;
  set_ds(p, l, ds, tok0, tok1);
  p.q_chunk_tokens = cmp_ds_q_chunk(B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, tok0, tok1);
  if (workspace == nullptr) return nsa_bwd_dkdv_launch(p, 0, B, x_maxlen, y_maxlen, D, VD, 0, (hipStream_t)stream);
  const int64_t need = nsa_cmp_attn_bwd_dkdv_ds_slot_bytes(B, x_maxlen, y_maxlen, QH, KH, D, VD, kernel_size, stride, tok0, tok1);
  NSA_REQUIRE(workspace_bytes >= need, NSA_ERR_WORKSPACE, "cmp_attn_bwd_dkdv_ds: workspace of %lld bytes, %lld needed",
              (long long)workspace_bytes, (long long)need);
  const int64_t slots = nsa_bwd_dkdv_cmp_slots(B, KH, x_maxlen, y_maxlen, D, p.q_chunk_tokens, kernel_size, stride, tok0, tok1, B);
  p.dkv_mode = 4;
  p.part_dk = (float*)workspace;
  p.part_dv = (float*)((char*)workspace + ((slots * nsa_bwd_dkdv_slot_keys(0, 0, D) * D * 4 + 255) & ~(int64_t)255));
  rc = nsa_bwd_dkdv_launch(p, 0, B, x_maxlen, y_maxlen, D, VD, 0, (hipStream_t)stream);
  if (rc) return rc;
  return nsa_dkdv_reduce_cmp_launch(p, add != 0, B, x_maxlen, y_maxlen, D, VD, (hipStream_t)stream);
}

// Slots are numbered by the longest sequence: a ragged batch takes memory for all of them and writes few, so the limit is wider
// than that of batches that fill theirs.
static const int64_t SWA_DS_SLOTS_LIMIT = (int64_t)512 << 20;

// length of the longest share of a sequence
static int ds_share(int x_maxlen, int tok0, int tok1) {
  return tok1 > 0 && tok1 - tok0 + 127 < x_maxlen ? tok1 - tok0 + 127 : x_maxlen;
}

static int swa_ds_splits(int T, int B, int x_maxlen, int QH, int KH, int D, int VD, int window, int tok0, int tok1) {
  return swa_dkdv_splits(B, ds_share(x_maxlen, tok0, tok1), QH, KH, D, VD, window, SWA_DS_SLOTS_LIMIT,
                         tok1 > 0 ? tok1 - tok0 : T);
}

int64_t nsa_swa_bwd_dkdv_ds_ws_bytes(int T, int B, int x_maxlen, int QH, int KH, int D, int VD, int window, int tok0,
                                     int tok1) {
  const int splits = swa_ds_splits(T, B, x_maxlen, QH, KH, D, VD, window, tok0, tok1);
  int64_t dk_bytes;
  return splits > 1 ? swa_dkdv_slot_bytes(splits, B, ds_share(x_maxlen, tok0, tok1), KH, D, VD, &dk_bytes) : 0;
}

int nsa_swa_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                        int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                        int VD, int window, float sm_scale, int T, int ring, int tok0, int tok1, void* ds,
                        int64_t ds_bytes, void* workspace, int64_t workspace_bytes, void* stream) {
  const DsLayout l = KH > 0 && QH >= KH ? ds_layout_win(T, B, x_maxlen, QH / KH, KH, window, ring) : DsLayout{};
  int rc = check_ds("swa_bwd_dkdv_ds", QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, ds, ds_bytes, l.bytes,
                    bwd_ds_takes(q_sh, do_sh, k_sr, QH, KH, D, VD, sm_scale));
  if (rc) return rc;
  NSA_REQUIRE(window >= 0 && (ring == 0 ? tok1 == 0 : tok1 > 0 && tok1 - tok0 <= ring), NSA_ERR_BAD_ARG,
              "swa_bwd_dkdv_ds: window %d, tokens %d to %d in ranges of up to %d", window, tok0, tok1, ring);
  if (B <= 0 || x_maxlen <= 0) return NSA_OK;
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = dkv_is_f32 ? 1 : 0;
  const int share = ds_share(x_maxlen, tok0, tok1);
  p.grid_chunks = workspace != nullptr ? swa_ds_splits(T, B, x_maxlen, QH, KH, D, VD, window, tok0, tok1) : 1;
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.window = window;
  set_ds(p, l, ds, tok0, tok1);
  if (p.grid_chunks > 1) {
    int64_t dk_bytes;
    const int64_t need = swa_dkdv_slot_bytes(p.grid_chunks, B, share, KH, D, VD, &dk_bytes);
    NSA_REQUIRE(workspace_bytes >= need, NSA_ERR_WORKSPACE, "swa_bwd_dkdv_ds: workspace of %lld bytes, %lld needed",
                (long long)workspace_bytes, (long long)need);
    p.dkv_mode = 4;
    p.part_dk = (float*)workspace;
    p.part_dv = (float*)((char*)workspace + dk_bytes);
  }
  rc = nsa_bwd_dkdv_launch(p, 1, B, x_maxlen, x_maxlen, D, VD, 0, (hipStream_t)stream);
  if (rc || p.grid_chunks == 1) return rc;
  return nsa_dkdv_reduce_swa_launch(p, dkv_is_f32 != 0, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_slc_attn_bwd_dkdv_before_window_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr,
                                           int64_t k_sh, const void* v, int64_t v_sr, int64_t v_sh, const void* dO,
                                           int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st,
                                           int64_t lse_sh, const float* delta, int64_t delta_st, int64_t delta_sh,
                                           float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                                           int64_t dv_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                                           int D, int VD, int window, int all_below, float sm_scale, int T, int ring,
                                           int tok0, int tok1, void* ds, int64_t ds_bytes, void* stream) {
  const DsLayout l = KH > 0 && QH >= KH ? ds_layout_far(T, B, x_maxlen, QH / KH, KH, window, all_below, ring) : DsLayout{};
  NSA_REQUIRE(window >= 0 && all_below >= 0 && all_below % 8 == 0 && (ring == 0 ? tok1 == 0 : tok1 > 0 && tok1 - tok0 <= ring),
              NSA_ERR_BAD_ARG, "slc_attn_bwd_dkdv_before_window_ds: window %d, all_below %d, tokens %d to %d in ranges of up to %d",
              window, all_below, tok0, tok1, ring);
  if (l.pitch == 0) return NSA_OK;  // no query has keys before its window
  int rc = check_ds("slc_attn_bwd_dkdv_before_window_ds", QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, ds, ds_bytes, l.bytes,
                    bwd_ds_takes(q_sh, do_sh, k_sr, QH, KH, D, VD, sm_scale));
  if (rc) return rc;
  const int len = (x_maxlen < all_below ? x_maxlen : all_below) - window - 1;  // positions that are some query's keys
  BwdCommon c{q, q_st, q_sh, k, k_sr, k_sh, v, v_sr, v_sh, dO, do_st, do_sh, lse, lse_st, lse_sh, delta, delta_st,
              delta_sh};
  NsaBwdTileParams p = make_bwd(c, QH, KH, sm_scale);
  p.dk = dk; p.dk_sr = dk_sr; p.dk_sh = dk_sh;
  p.dv = dv; p.dv_sr = dv_sr; p.dv_sh = dv_sh;
  p.dkv_mode = 3;
  p.grid_chunks = swa_dkdv_splits(B, len, QH, KH, D, VD, len, INT64_MAX);
  p.x_cu = x_cu; p.k_cu = x_cu;
  p.min_dist = window + 1; p.window = all_below; p.t_end = all_below;
  set_ds(p, l, ds, tok0, tok1);
  return nsa_bwd_dkdv_launch(p, 1, B, x_maxlen, x_maxlen, D, VD, 0, (hipStream_t)stream);
}

int nsa_attn_bwd_dq_ds(const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cmp_ds, int64_t cmp_ds_bytes, const void* k,
                       int64_t k_sr, int64_t k_sh, const void* swa_ds, int64_t swa_ds_bytes, const void* far_ds,
                       int64_t far_ds_bytes, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, float* dq_partial,
                       int64_t dqp_st, int64_t dqp_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH,
                       int KH, int D, int VD, int kernel_size, int stride, int window, int all_below, float sm_scale, int T,
                       int ring, int tok0, int tok1, void* stream) {
  const char* const who = "attn_bwd_dq_ds";
  int rc = check_heads(who, QH, KH, D, VD);
  if (rc) return rc;
  NSA_REQUIRE(cmp_ds != nullptr || swa_ds != nullptr, NSA_ERR_BAD_ARG, "%s: no branch's dS", who);
  NSA_REQUIRE(dq_mode >= 0 && dq_mode <= 3 && (dq_mode != 3 || dq_partial != nullptr) && window >= 0 && all_below % 8 == 0,
              NSA_ERR_BAD_ARG, "%s: dq_mode %d, window %d, all_below %d", who, dq_mode, window, all_below);
  const int G = QH / KH;
  NsaDqDsParams p{};
  if (cmp_ds != nullptr) {
    rc = check_nsa_sizes(who, kernel_size, stride, 0);
    if (rc) return rc;
    const DsLayout l = ds_layout_cmp(T, B, x_maxlen, G, KH, kernel_size, stride, tok0, tok1);
    rc = check_ds(who, QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, cmp_ds, cmp_ds_bytes, l.bytes,
                  bwd_ds_takes(0, 0, ck_sr, QH, KH, D, VD, sm_scale));
    if (rc) return rc;
    p.cmp = ds_operand(l, ck, ck_sr, ck_sh, cmp_ds);
  }
  if (swa_ds != nullptr) {
    const DsLayout l = ds_layout_win(T, B, x_maxlen, G, KH, window, ring);
    rc = check_ds(who, QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, swa_ds, swa_ds_bytes, l.bytes,
                  bwd_ds_takes(0, 0, k_sr, QH, KH, D, VD, sm_scale));
    if (rc) return rc;
    p.win = ds_operand(l, k, k_sr, k_sh, swa_ds);
    const DsLayout f = ds_layout_far(T, B, x_maxlen, G, KH, window, all_below, ring);
    if (far_ds != nullptr && f.pitch > 0) {
      rc = check_ds(who, QH, KH, D, VD, T, B, x_maxlen, tok0, tok1, far_ds, far_ds_bytes, f.bytes, true);
      if (rc) return rc;
      p.far = ds_operand(f, k, k_sr, k_sh, far_ds);
    }
  }
  p.dq = dq; p.dq_st = dq_st; p.dq_sh = dq_sh; p.dq_mode = dq_mode;
  p.dq_partial = dq_partial; p.dqp_st = dqp_st; p.dqp_sh = dqp_sh;
  p.x_cu = x_cu; p.y_cu = y_cu;
  p.G = G; p.KH = KH;
  p.kernel_size = kernel_size; p.stride = stride; p.window = window; p.all_below = all_below;
  p.tok0 = tok0; p.tok1 = tok1;
  p.sm_scale = sm_scale;
  return nsa_bwd_dq_ds_launch(p, B, x_maxlen, D, (hipStream_t)stream);
}

}  // extern "C"

// ------------------------------------------------------------------------------------------------ paged KV
namespace {
int check_page(const char* who, int page_size) {
  NSA_REQUIRE(page_size > 0 && page_size % 64 == 0, NSA_ERR_BAD_ARG, "%s: page_size %d must be a multiple of 64", who,
              page_size);
  return NSA_OK;
}
}  // namespace

extern "C" {

int nsa_paged_cmp_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st,
                           int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh, const int32_t* x_cu,
                           const int32_t* context_lens, const int32_t* cmp_block_tables, int table_stride,
                           int page_size, int B, int x_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                           int stride, float sm_scale, void* stream) {
  int rc = check_heads("paged_cmp_attn_fwd", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("paged_cmp_attn_fwd", kernel_size, stride, 0);
  if (rc) return rc;
  rc = check_page("paged_cmp_attn_fwd", page_size);
  if (rc) return rc;
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.ctx_lens = context_lens;
  p.table = cmp_block_tables; p.table_stride = table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.window = 0;
  return nsa_fwd_tile_launch(p, 0, true, B, x_maxlen, D, VD, (hipStream_t)stream);
}

static NsaFwdTileParams paged_window_params(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                                            int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, void* o,
                                            int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh,
                                            const int32_t* x_cu, const int32_t* context_lens,
                                            const int32_t* block_tables, int table_stride, int page_size, int QH,
                                            int KH, int window, float sm_scale) {
  NsaFwdTileParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.x_cu = x_cu; p.ctx_lens = context_lens;
  p.table = block_tables; p.table_stride = table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = 1; p.stride = 1; p.window = window;
  return p;
}

int nsa_paged_swa_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                      const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh,
                      float* lse, int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                      const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen, int QH,
                      int KH, int D, int VD, int window, float sm_scale, void* stream) {
  int rc = check_heads("paged_swa_fwd", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_page("paged_swa_fwd", page_size);
  if (rc) return rc;
  return nsa_fwd_tile_launch(paged_window_params(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, o, o_st, o_sh,
                                                 lse, lse_st, lse_sh, x_cu, context_lens, block_tables, table_stride,
                                                 page_size, QH, KH, window, sm_scale),
                             1, true, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_paged_swa_fwd_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                           const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh,
                           float* lse, int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh,
                           float* slc_lse, int64_t sl_st, int64_t sl_sh, int all_below, const void* cmp_o,
                           int64_t co_st, int64_t co_sh, const void* w, int64_t w_st, int64_t w_sh, void* out,
                           int64_t out_st, int64_t out_sh, int store_branches, const int32_t* x_cu,
                           const int32_t* context_lens, const int32_t* block_tables, int table_stride, int page_size,
                           int B, int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale,
                           void* stream) {
  int rc = check_heads("paged_swa_fwd_tail", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_page("paged_swa_fwd_tail", page_size);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "paged_swa_fwd_tail: window %d must be >= 0", window);
  NsaFwdTileParams p = paged_window_params(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, o, o_st, o_sh, lse,
                                           lse_st, lse_sh, x_cu, context_lens, block_tables, table_stride, page_size,
                                           QH, KH, window, sm_scale);
  rc = fill_swa_tail(p, "paged_swa_fwd_tail", slc_o, so_st, so_sh, slc_lse, sl_st, sl_sh, all_below, cmp_o, co_st,
                     co_sh, w, w_st, w_sh, out, out_st, out_sh, store_branches);
  if (rc) return rc;
  return nsa_fwd_tile_launch(p, 2, true, B, x_maxlen, D, VD, (hipStream_t)stream);
}

int nsa_paged_fwd_short(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                        const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh, void* o,
                        int64_t o_st, int64_t o_sh, void* slc_o, int64_t so_st, int64_t so_sh, int all_below, const void* w,
                        int64_t w_st, int64_t w_sh, void* out, int64_t out_st, int64_t out_sh, const int32_t* x_cu,
                        const int32_t* context_lens, const int32_t* block_tables, int table_stride,
                        const int32_t* cmp_block_tables, int cmp_table_stride, int page_size, int B, int x_maxlen, int QH, int KH,
                        int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream) {
  int rc = check_heads("paged_fwd_short", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("paged_fwd_short", kernel_size, stride, 0);
  if (rc) return rc;
  rc = check_page("paged_fwd_short", page_size);
  if (rc) return rc;
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "paged_fwd_short: window %d must be >= 0", window);
  NsaFwdTileParams p = paged_window_params(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, o, o_st, o_sh, nullptr, 0, 0,
                                           x_cu, context_lens, block_tables, table_stride, page_size, QH, KH, window, sm_scale);
  rc = fill_swa_tail(p, "paged_fwd_short", slc_o, so_st, so_sh, nullptr, 0, 0, all_below, cmp_o, co_st, co_sh, w, w_st, w_sh, out,
                     out_st, out_sh, 0);
  if (rc) return rc;
  NSA_REQUIRE(cmp_o != nullptr && out != nullptr, NSA_ERR_BAD_ARG, "paged_fwd_short: an output is missing");
  fill_cmp_branch(p, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, cmp_o, nullptr, 0, 0, kernel_size, stride);
  p.c_table = cmp_block_tables; p.c_table_stride = cmp_table_stride;
  return nsa_fwd_tile_launch(p, 3, true, B, x_maxlen, D, VD, (hipStream_t)stream);
}

static int paged_topk_select_impl(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                          int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                          int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                          const int32_t* cmp_block_tables, int table_stride, int page_size, int B, int x_maxlen,
                          int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size, int stride,
                          int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                          int total_tokens, int t_begin, void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = check_heads("paged_topk_select", QH, KH, D, 32);
  if (rc) return rc;
  rc = check_nsa_sizes("paged_topk_select", kernel_size, stride, block_size);
  if (rc) return rc;
  rc = check_page("paged_topk_select", page_size);
  if (rc) return rc;
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "paged_topk_select: top_n %d must be in [1,64]", top_n);
  NSA_REQUIRE(num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n, NSA_ERR_BAD_ARG,
              "paged_topk_select: num_init %d + num_local %d must be <= top_n %d", num_init, num_local, top_n);
  NSA_REQUIRE(fixed_num_slc_blocks >= 1, NSA_ERR_BAD_ARG, "paged_topk_select: fixed_num_slc_blocks must be >= 1");
  NsaTopkParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.ck = (const bf16_t*)k_cache; p.ck_sr = k_sr; p.ck_sh = k_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.x_cu = x_cu; p.ctx_lens = context_lens;
  p.table = cmp_block_tables; p.table_stride = table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.block_size = block_size;
  p.top_n = top_n; p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  p.nb_max = fixed_num_slc_blocks;
  p.t_begin = t_begin;
  if (workspace != nullptr && nsa_tuning_knob("topk_two_pass", 1) != 0 && nsa_topk_two_pass_supported(p, D))
    return nsa_topk_two_pass_launch(p, true, B, x_maxlen, total_tokens, D, workspace, workspace_bytes,
                                    (hipStream_t)stream);
  return nsa_topk_launch(p, true, B, x_maxlen, D, (hipStream_t)stream);
}

int nsa_paged_topk_select(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                          int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                          int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                          const int32_t* cmp_block_tables, int table_stride, int page_size, int B, int x_maxlen,
                          int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size, int stride,
                          int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                          void* stream) {
  return paged_topk_select_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, x_cu,
                                context_lens, cmp_block_tables, table_stride, page_size, B, x_maxlen,
                                fixed_num_slc_blocks, QH, KH, D, kernel_size, stride, block_size, top_n, num_init,
                                num_local, ignore_index, sm_scale, 0, 0, nullptr, 0, stream);
}

int nsa_paged_topk_select_ws(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                             int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                             int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                             const int32_t* cmp_block_tables, int table_stride, int page_size, int B, int x_maxlen,
                             int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size, int stride,
                             int block_size, int top_n, int num_init, int num_local, int ignore_index,
                             float sm_scale, int total_tokens, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  return nsa_paged_topk_select_ws_from(q, q_st, q_sh, k_cache, k_sr, k_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st,
                                       x_cu, context_lens, cmp_block_tables, table_stride, page_size, B, x_maxlen,
                                       fixed_num_slc_blocks, QH, KH, D, kernel_size, stride, block_size, top_n,
                                       num_init, num_local, ignore_index, sm_scale, total_tokens, 0, workspace,
                                       workspace_bytes, stream);
}

int nsa_paged_topk_select_ws_from(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                                  int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                                  int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                                  const int32_t* cmp_block_tables, int table_stride, int page_size, int B,
                                  int x_maxlen, int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size,
                                  int stride, int block_size, int top_n, int num_init, int num_local,
                                  int ignore_index, float sm_scale, int total_tokens, int t_begin, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
  NSA_REQUIRE(total_tokens >= 0 && (workspace == nullptr || workspace_bytes > 0), NSA_ERR_BAD_ARG,
              "paged_topk_select_ws: bad token count %d or workspace size %lld", total_tokens,
              (long long)workspace_bytes);
  return paged_topk_select_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, x_cu,
                                context_lens, cmp_block_tables, table_stride, page_size, B, x_maxlen,
                                fixed_num_slc_blocks, QH, KH, D, kernel_size, stride, block_size, top_n, num_init,
                                num_local, ignore_index, sm_scale, total_tokens, t_begin, workspace, workspace_bytes,
                                stream);
}

int nsa_paged_slc_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const int32_t* topk,
                           int64_t tk_sh, int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse,
                           int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                           const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen,
                           int QH, int KH, int D, int VD, int block_size, int top_n, float sm_scale, void* stream) {
  return nsa_paged_slc_attn_fwd_from(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, topk, tk_sh, tk_st, o,
                                     o_st, o_sh, lse, lse_st, lse_sh, x_cu, context_lens, block_tables, table_stride,
                                     page_size, B, x_maxlen, QH, KH, D, VD, block_size, top_n, 0, sm_scale, stream);
}

int nsa_paged_slc_attn_fwd_from(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const int32_t* topk,
                           int64_t tk_sh, int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse,
                           int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                           const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen,
                           int QH, int KH, int D, int VD, int block_size, int top_n, int t_begin,
                           float sm_scale, void* stream) {
  int rc = check_heads("paged_slc_attn_fwd", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_page("paged_slc_attn_fwd", page_size);
  if (rc) return rc;
  NSA_REQUIRE(block_size % 32 == 0 && block_size > 0, NSA_ERR_UNSUPPORTED,
              "paged_slc_attn_fwd: block_size %d must be a multiple of 32", block_size);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "paged_slc_attn_fwd: top_n %d must be in [1,64]", top_n);
  rc = check_positions("paged_slc_attn_fwd", t_begin);
  if (rc) return rc;
  NsaSlcParams p{};
  p.t_begin = t_begin;
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.o = (bf16_t*)o; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.x_cu = x_cu; p.ctx_lens = context_lens;
  p.table = block_tables; p.table_stride = table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH; p.top_n = top_n; p.block_size = block_size;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  return nsa_slc_fwd_launch(p, true, B, x_maxlen, D, VD, (hipStream_t)stream);
}

}  // extern "C"

// ------------------------------------------------------------------------------------------------ fused decode
extern "C" {

int nsa_decode_cmp_topk(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                        const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh,
                        float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                        const int32_t* context_lens, const int32_t* cmp_block_tables, int cmp_table_stride,
                        int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                        int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n,
                        int num_init, int num_local, int ignore_index, float sm_scale, void* stream) {
  int rc = check_heads("decode_cmp_topk", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("decode_cmp_topk", kernel_size, stride, block_size);
  if (rc) return rc;
  rc = check_page("decode_cmp_topk", page_size);
  if (rc) return rc;
  NSA_REQUIRE(QH / KH <= 16, NSA_ERR_UNSUPPORTED, "decode_cmp_topk: at most 16 q-heads per kv head (got %d)", QH / KH);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64 && num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n,
              NSA_ERR_BAD_ARG, "decode_cmp_topk: bad top_n/num_init/num_local %d/%d/%d", top_n, num_init, num_local);
  NSA_REQUIRE(fixed_y_maxlen >= 1 && fixed_num_slc_blocks >= 1, NSA_ERR_BAD_ARG,
              "decode_cmp_topk: fixed_y_maxlen and fixed_num_slc_blocks must be positive");
  NsaDecodeParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.cmp_o = (bf16_t*)cmp_o; p.co_st = co_st; p.co_sh = co_sh;
  p.lse_out = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.ctx_lens = context_lens;
  p.cmp_table = cmp_block_tables; p.cmp_table_stride = cmp_table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.block_size = block_size;
  p.top_n = top_n; p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks;
  return nsa_decode_cmp_topk_launch(p, B, D, VD, (hipStream_t)stream);
}

int nsa_decode_cmp_split(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                         const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh,
                         float* lse, int64_t lse_st, int64_t lse_sh, float* pg, float* sp_m, float* sp_l, float* sp_o,
                         int nsplit, const int32_t* context_lens, const int32_t* cmp_block_tables,
                         int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD,
                         int fixed_y_maxlen, int kernel_size, int stride, float sm_scale, void* stream) {
  int rc = check_heads("decode_cmp_split", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("decode_cmp_split", kernel_size, stride, 0);
  if (rc) return rc;
  rc = check_page("decode_cmp_split", page_size);
  if (rc) return rc;
  NSA_REQUIRE(QH / KH <= 16, NSA_ERR_UNSUPPORTED, "decode_cmp_split: at most 16 q-heads per kv head (got %d)", QH / KH);
  NSA_REQUIRE(nsplit >= 1 && nsplit <= 64, NSA_ERR_BAD_ARG, "decode_cmp_split: nsplit %d must be in [1,64]", nsplit);
  NSA_REQUIRE(fixed_y_maxlen >= 1 && fixed_y_maxlen <= 32768, NSA_ERR_BAD_ARG,
              "decode_cmp_split: fixed_y_maxlen %d must be in [1,32768]", fixed_y_maxlen);
  NsaDecodeParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.cmp_o = (bf16_t*)cmp_o; p.co_st = co_st; p.co_sh = co_sh;
  p.lse_out = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.pg = pg; p.sp_m = sp_m; p.sp_l = sp_l; p.sp_o = sp_o;
  p.ctx_lens = context_lens;
  p.cmp_table = cmp_block_tables; p.cmp_table_stride = cmp_table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride;
  p.y_cap = fixed_y_maxlen;
  return nsa_decode_cmp_split_launch(p, B, nsplit, D, VD, (hipStream_t)stream);
}

static void fill_decode_split(NsaDecodeParams& p, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride) {
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks; p.table_stride = table_stride;
}

int nsa_decode_split_fits(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride) {
  NsaDecodeParams p{};
  fill_decode_split(p, fixed_y_maxlen, fixed_num_slc_blocks, table_stride);
  return nsa_decode_split_lds_bytes(p, D, VD) > 0 ? 1 : 0;
}

int nsa_decode_split_lds_total(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride) {
  NsaDecodeParams p{};
  fill_decode_split(p, fixed_y_maxlen, fixed_num_slc_blocks, table_stride);
  const int dyn = nsa_decode_split_lds_bytes(p, D, VD);
  return dyn > 0 ? dyn + nsa_decode_split_static_lds_bytes() : 0;
}

int nsa_decode_two_launch_lds(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride,
                              int page_size, int parts) {
  if (fixed_y_maxlen < 1 || fixed_num_slc_blocks < 1 || table_stride < 1 || page_size < 1) return 0;
  NsaDecodeParams p{};
  fill_decode_split(p, fixed_y_maxlen, fixed_num_slc_blocks, table_stride);
  p.page_size = page_size;
  return nsa_decode_two_launch_lds_bytes(p, D, VD, parts != 0);
}

int nsa_decode_split_window_parts(int window, int fixed_y_maxlen, int nsplit) {
  // as many as give a wave of the window no more units than a wave of the compressed branch has
  if (window < 0 || window > 65536 || nsplit <= 0) return 0;
  const int units = window / 32 + 2;
  const int cmp = (fixed_y_maxlen / 32 + 4 * nsplit - 1) / (4 * nsplit);
  const int n = (units + 4 * (cmp > 2 ? cmp : 2) - 1) / (4 * (cmp > 2 ? cmp : 2));
  return n < 4 ? n : 4;
}

static int decode_split_impl(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, int slc_nsplit, float* sp2_ml,
                     float* sp2_o, void* cmp_tmp, int win_parts, float* win_ml, float* win_o, void* stream,
                     const void* new_k = nullptr, int64_t nk_st = 0, int64_t nk_sh = 0, const void* new_v = nullptr,
                     int64_t nv_st = 0, int64_t nv_sh = 0, const int32_t* slot_mapping = nullptr) {
  int rc = check_heads("decode_split", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("decode_split", kernel_size, stride, block_size);
  if (rc) return rc;
  rc = check_page("decode_split", page_size);
  if (rc) return rc;
  NSA_REQUIRE(QH / KH <= 16, NSA_ERR_UNSUPPORTED, "decode_split: at most 16 q-heads per kv head (got %d)", QH / KH);
  NSA_REQUIRE(nsplit >= 1 && nsplit <= 64, NSA_ERR_BAD_ARG, "decode_split: nsplit %d must be in [1,64]", nsplit);
  NSA_REQUIRE(block_size % 32 == 0, NSA_ERR_UNSUPPORTED, "decode_split: block_size %d must be a multiple of 32",
              block_size);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64 && num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n,
              NSA_ERR_BAD_ARG, "decode_split: bad top_n %d / num_init %d / num_local %d", top_n, num_init, num_local);
  NSA_REQUIRE(fixed_y_maxlen >= 1 && fixed_num_slc_blocks >= 1, NSA_ERR_BAD_ARG,
              "decode_split: fixed_y_maxlen %d and fixed_num_slc_blocks %d must be positive", fixed_y_maxlen,
              fixed_num_slc_blocks);
  NSA_REQUIRE(out && w && sp_m && sp_l && sp_o && sp_keep_p && sp_keep_m, NSA_ERR_BAD_ARG,
              "decode_split: out, w and the five scratch buffers are required");
  NSA_REQUIRE(slc_nsplit >= 1 && slc_nsplit <= 16, NSA_ERR_BAD_ARG, "decode_split: slc_nsplit %d must be in [1,16]",
              slc_nsplit);
  NSA_REQUIRE(slc_nsplit == 1 || (sp2_ml && sp2_o && cmp_tmp), NSA_ERR_BAD_ARG,
              "decode_split: slc_nsplit > 1 needs the three buffers of the window / selected parts");
  NSA_REQUIRE(win_parts >= 0 && win_parts <= 4 && (win_parts == 0 || (win_ml && win_o)), NSA_ERR_BAD_ARG,
              "decode_split: win_parts %d must be in [0,4], with its two buffers", win_parts);
  NSA_REQUIRE(win_parts == 0 || (window >= 0 && window <= 65536), NSA_ERR_BAD_ARG,
              "decode_split: window %d must be in [0,65536] to be attended in parts", window);
  NSA_REQUIRE((new_k == nullptr) == (new_v == nullptr) && (new_k == nullptr) == (slot_mapping == nullptr) &&
                  (new_k == nullptr || win_parts > 0),
              NSA_ERR_BAD_ARG, "decode_split: new_k, new_v and slot_mapping must be given together, and with win_parts > 0");
  NsaDecodeParams p{};
  p.new_k = (const bf16_t*)new_k; p.nk_st = nk_st; p.nk_sh = nk_sh;
  p.new_v = (const bf16_t*)new_v; p.nv_st = nv_st; p.nv_sh = nv_sh;
  p.raw_slots = slot_mapping;
  p.win_parts = win_parts; p.win_m = win_ml; p.win_o = win_o;
  p.win_l = win_ml ? win_ml + (int64_t)B * KH * win_parts * 16 : nullptr;
  p.slc_nsplit = slc_nsplit; p.sp2_ml = sp2_ml; p.sp2_o = sp2_o; p.cmp_tmp = (bf16_t*)cmp_tmp;
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.w = (const bf16_t*)w; p.w_st = w_st; p.w_sh = w_sh;
  p.out = (bf16_t*)out; p.o_st = o_st; p.o_sh = o_sh;
  p.cmp_o = (bf16_t*)cmp_o; p.slc_o = (bf16_t*)slc_o; p.swa_o = (bf16_t*)swa_o; p.co_st = co_st; p.co_sh = co_sh;
  p.lse_out = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.sp_m = sp_m; p.sp_l = sp_l; p.sp_o = sp_o;
  p.sp_keep_p = sp_keep_p; p.sp_keep_m = sp_keep_m; p.nsplit = nsplit;
  p.ctx_lens = context_lens;
  p.cmp_slots = cmp_slot_mapping;
  p.table = block_tables;
  p.cmp_table = cmp_block_tables; p.cmp_table_stride = cmp_table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.block_size = block_size; p.window = window; p.top_n = top_n;
  p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  fill_decode_split(p, fixed_y_maxlen, fixed_num_slc_blocks, table_stride);
  return nsa_decode_split_launch(p, B, D, VD, (hipStream_t)stream);
}

int nsa_decode_split(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, void* stream) {
  return decode_split_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, w, w_st, w_sh, out, o_st, o_sh, cmp_o, slc_o,
                           swa_o, co_st, co_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, sp_m, sp_l, sp_o, sp_keep_p,
                           sp_keep_m, nsplit, cmp_slot_mapping, context_lens, block_tables, table_stride,
                           cmp_block_tables, cmp_table_stride, page_size, B, QH, KH, D, VD, fixed_y_maxlen,
                           fixed_num_slc_blocks, kernel_size, stride, block_size, top_n, num_init, num_local,
                           ignore_index, window, sm_scale, 1, nullptr, nullptr, nullptr, 0, nullptr, nullptr, stream);
}

int nsa_decode_split_window(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, int win_parts,
                     float* win_ml, float* win_o, void* stream) {
  return decode_split_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, w, w_st, w_sh, out, o_st, o_sh, cmp_o, slc_o,
                           swa_o, co_st, co_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, sp_m, sp_l, sp_o, sp_keep_p,
                           sp_keep_m, nsplit, cmp_slot_mapping, context_lens, block_tables, table_stride,
                           cmp_block_tables, cmp_table_stride, page_size, B, QH, KH, D, VD, fixed_y_maxlen,
                           fixed_num_slc_blocks, kernel_size, stride, block_size, top_n, num_init, num_local,
                           ignore_index, window, sm_scale, 1, nullptr, nullptr, nullptr, win_parts, win_ml, win_o, stream);
}

int nsa_decode_split_window_store(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, int win_parts,
                     float* win_ml, float* win_o, const void* new_k, int64_t nk_st, int64_t nk_sh, const void* new_v,
                     int64_t nv_st, int64_t nv_sh, const int32_t* slot_mapping, void* stream) {
  return decode_split_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, w, w_st, w_sh, out, o_st, o_sh, cmp_o, slc_o,
                           swa_o, co_st, co_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, sp_m, sp_l, sp_o, sp_keep_p,
                           sp_keep_m, nsplit, cmp_slot_mapping, context_lens, block_tables, table_stride,
                           cmp_block_tables, cmp_table_stride, page_size, B, QH, KH, D, VD, fixed_y_maxlen,
                           fixed_num_slc_blocks, kernel_size, stride, block_size, top_n, num_init, num_local,
                           ignore_index, window, sm_scale, 1, nullptr, nullptr, nullptr, win_parts, win_ml, win_o, stream,
                           new_k, nk_st, nk_sh, new_v, nv_st, nv_sh, slot_mapping);
}

int nsa_decode_split_parts(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, int slc_nsplit, float* sp2_ml,
                     float* sp2_o, void* cmp_tmp, void* stream) {
  return decode_split_impl(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, w, w_st, w_sh, out, o_st, o_sh, cmp_o, slc_o,
                           swa_o, co_st, co_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st, sp_m, sp_l, sp_o, sp_keep_p,
                           sp_keep_m, nsplit, cmp_slot_mapping, context_lens, block_tables, table_stride,
                           cmp_block_tables, cmp_table_stride, page_size, B, QH, KH, D, VD, fixed_y_maxlen,
                           fixed_num_slc_blocks, kernel_size, stride, block_size, top_n, num_init, num_local,
                           ignore_index, window, sm_scale, slc_nsplit, sp2_ml, sp2_o, cmp_tmp, 0, nullptr,
                           nullptr, stream);
}

int nsa_decode_slc_swa_combine(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                               int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w,
                               int64_t w_st, int64_t w_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                               const float* pg, int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size,
                               int stride, int num_init, int num_local, int ignore_index, const void* cmp_o,
                               void* slc_o, void* swa_o, int64_t co_st, int64_t co_sh, void* out, int64_t o_st,
                               int64_t o_sh, const int32_t* context_lens, const int32_t* block_tables,
                               int table_stride, int page_size, int B, int QH, int KH, int D, int VD, int block_size,
                               int top_n, int window, float sm_scale, void* stream) {
  int rc = check_heads("decode_slc_swa_combine", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_page("decode_slc_swa_combine", page_size);
  if (rc) return rc;
  NSA_REQUIRE(QH / KH <= 16, NSA_ERR_UNSUPPORTED, "decode_slc_swa_combine: at most 16 q-heads per kv head (got %d)",
              QH / KH);
  NSA_REQUIRE(block_size % 32 == 0 && block_size > 0, NSA_ERR_UNSUPPORTED,
              "decode_slc_swa_combine: block_size %d must be a multiple of 32", block_size);
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "decode_slc_swa_combine: top_n %d must be in [1,64]", top_n);
  NSA_REQUIRE(out == nullptr || (w != nullptr && cmp_o != nullptr), NSA_ERR_BAD_ARG,
              "decode_slc_swa_combine: the combined output needs the gates and the compressed-branch output");
  if (pg != nullptr) {
    rc = check_nsa_sizes("decode_slc_swa_combine", kernel_size, stride, block_size);
    if (rc) return rc;
    NSA_REQUIRE(num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n, NSA_ERR_BAD_ARG,
                "decode_slc_swa_combine: num_init %d + num_local %d must be <= top_n %d", num_init, num_local, top_n);
    NSA_REQUIRE(fixed_num_slc_blocks >= 1 && fixed_num_slc_blocks <= 8192 && fixed_y_maxlen >= 1, NSA_ERR_BAD_ARG,
                "decode_slc_swa_combine: fixed_num_slc_blocks %d must be in [1,8192]", fixed_num_slc_blocks);
  }
  NsaDecodeParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.w = (const bf16_t*)w; p.w_st = w_st; p.w_sh = w_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.pg = const_cast<float*>(pg);
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks;
  p.kernel_size = kernel_size; p.stride = stride;
  p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  p.cmp_o = (bf16_t*)const_cast<void*>(cmp_o); p.slc_o = (bf16_t*)slc_o; p.swa_o = (bf16_t*)swa_o;
  p.co_st = co_st; p.co_sh = co_sh;
  p.out = (bf16_t*)out; p.o_st = o_st; p.o_sh = o_sh;
  p.ctx_lens = context_lens;
  p.table = block_tables; p.table_stride = table_stride; p.page_size = page_size;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.block_size = block_size; p.window = window; p.top_n = top_n;
  return nsa_decode_slc_swa_launch(p, B, D, VD, (hipStream_t)stream);
}

int nsa_decode_fused_fits(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride,
                          int page_size) {
  if (fixed_y_maxlen < 1 || fixed_num_slc_blocks < 1 || table_stride < 1 || page_size < 1) return 0;
  NsaDecodeParams p{};
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks; p.table_stride = table_stride; p.page_size = page_size;
  return nsa_decode_fused_lds_bytes(p, D, VD) > 0 ? 1 : 0;
}

int64_t nsa_decode_fused_scratch_bytes(int B, int KH, int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks,
                                       int table_stride, int page_size) {
  if (B <= 0 || KH <= 0 || fixed_y_maxlen < 1 || fixed_num_slc_blocks < 1 || table_stride < 1 || page_size < 1) return 0;
  NsaDecodeParams p{};
  p.KH = KH;
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks; p.table_stride = table_stride; p.page_size = page_size;
  return nsa_decode_fused_scratch(p, B, D, VD);
}

int nsa_decode_fused(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, const int32_t* context_lens, const int32_t* block_tables, int table_stride,
                     const int32_t* cmp_block_tables, int cmp_table_stride,
                     const int32_t* cmp_slot_mapping, const void* new_k, int64_t nk_st, int64_t nk_sh,
                     const void* new_v, int64_t nv_st, int64_t nv_sh, const int32_t* slot_mapping, int page_size, int B, int QH, int KH,
                     int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size, int stride,
                     int block_size, int top_n, int num_init, int num_local, int ignore_index, int window,
                     float sm_scale, void* stream) {
  return nsa_decode_fused_ws(q, q_st, q_sh, k_cache, k_sr, k_sh, v_cache, v_sr, v_sh, w, w_st, w_sh, out, o_st, o_sh,
                             cmp_o, slc_o, swa_o, co_st, co_sh, lse, lse_st, lse_sh, topk, tk_sh, tk_st,
                             context_lens, block_tables, table_stride, cmp_block_tables, cmp_table_stride,
                             cmp_slot_mapping, new_k, nk_st, nk_sh, new_v, nv_st, nv_sh, slot_mapping, page_size, B,
                             QH, KH, D, VD, fixed_y_maxlen, fixed_num_slc_blocks, kernel_size, stride, block_size,
                             top_n, num_init, num_local, ignore_index, window, sm_scale, nullptr, 0, stream);
}

int nsa_decode_fused_ws(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, const int32_t* context_lens, const int32_t* block_tables, int table_stride,
                     const int32_t* cmp_block_tables, int cmp_table_stride,
                     const int32_t* cmp_slot_mapping, const void* new_k, int64_t nk_st, int64_t nk_sh,
                     const void* new_v, int64_t nv_st, int64_t nv_sh, const int32_t* slot_mapping, int page_size, int B, int QH, int KH,
                     int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size, int stride,
                     int block_size, int top_n, int num_init, int num_local, int ignore_index, int window,
                     float sm_scale, void* scratch, int64_t scratch_bytes, void* stream) {
  int rc = check_heads("decode_fused", QH, KH, D, VD);
  if (rc) return rc;
  rc = check_nsa_sizes("decode_fused", kernel_size, stride, block_size);
  if (rc) return rc;
  rc = check_page("decode_fused", page_size);
  if (rc) return rc;
  NSA_REQUIRE(QH / KH <= 16, NSA_ERR_UNSUPPORTED, "decode_fused: at most 16 q-heads per kv head (got %d)", QH / KH);
  NSA_REQUIRE(block_size % 32 == 0, NSA_ERR_UNSUPPORTED, "decode_fused: block_size %d must be a multiple of 32",
              block_size);
  NSA_REQUIRE(o_st % 4 == 0 && o_sh % 4 == 0 && co_st % 4 == 0 && co_sh % 4 == 0, NSA_ERR_BAD_ARG,
              "decode_fused: output strides must be multiples of 4 elements (8-byte stores)");
  NSA_REQUIRE(top_n >= 1 && top_n <= 64 && num_init >= 0 && num_local >= 0 && num_init + num_local <= top_n,
              NSA_ERR_BAD_ARG, "decode_fused: bad top_n/num_init/num_local %d/%d/%d", top_n, num_init, num_local);
  NSA_REQUIRE(fixed_y_maxlen >= 1 && fixed_num_slc_blocks >= 1 && table_stride >= 1 && cmp_table_stride >= 1,
              NSA_ERR_BAD_ARG, "decode_fused: fixed_y_maxlen, fixed_num_slc_blocks and the table widths must be positive");
  NSA_REQUIRE(out != nullptr && w != nullptr, NSA_ERR_BAD_ARG, "decode_fused: out and w are required");
  NSA_REQUIRE(window >= 0, NSA_ERR_BAD_ARG, "decode_fused: window %d must be >= 0", window);
  NsaDecodeParams p{};
  p.q = (const bf16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.k = (const bf16_t*)k_cache; p.k_sr = k_sr; p.k_sh = k_sh;
  p.v = (const bf16_t*)v_cache; p.v_sr = v_sr; p.v_sh = v_sh;
  p.w = (const bf16_t*)w; p.w_st = w_st; p.w_sh = w_sh;
  p.out = (bf16_t*)out; p.o_st = o_st; p.o_sh = o_sh;
  p.cmp_o = (bf16_t*)cmp_o; p.slc_o = (bf16_t*)slc_o; p.swa_o = (bf16_t*)swa_o; p.co_st = co_st; p.co_sh = co_sh;
  p.lse_out = lse; p.lse_st = lse_st; p.lse_sh = lse_sh;
  p.topk = topk; p.tk_sh = tk_sh; p.tk_st = tk_st;
  p.ctx_lens = context_lens;
  p.table = block_tables; p.table_stride = table_stride;
  p.cmp_table = cmp_block_tables; p.cmp_table_stride = cmp_table_stride; p.page_size = page_size;
  p.cmp_slots = cmp_slot_mapping;
  NSA_REQUIRE((new_k == nullptr) == (new_v == nullptr) && (new_k == nullptr) == (slot_mapping == nullptr),
              NSA_ERR_BAD_ARG, "decode_fused: new_k, new_v and slot_mapping must be given together");
  p.new_k = (const bf16_t*)new_k; p.nk_st = nk_st; p.nk_sh = nk_sh;
  p.new_v = (const bf16_t*)new_v; p.nv_st = nv_st; p.nv_sh = nv_sh;
  p.raw_slots = slot_mapping;
  p.G = QH / KH; p.KH = KH;
  p.scale_log2 = sm_scale * NSA_LOG2E;
  p.kernel_size = kernel_size; p.stride = stride; p.block_size = block_size; p.window = window;
  p.top_n = top_n; p.num_init = num_init; p.num_local = num_local; p.ignore_index = ignore_index;
  p.y_cap = fixed_y_maxlen; p.nb_cap = fixed_num_slc_blocks;
  const int64_t need = nsa_decode_fused_scratch(p, B, D, VD);
  if (scratch != nullptr && need > 0) {
    NSA_REQUIRE(scratch_bytes >= need, NSA_ERR_WORKSPACE, "decode_fused: scratch of %lld bytes, %lld needed",
                (long long)scratch_bytes, (long long)need);
    p.sp_keep_p = scratch;
  }
  return nsa_decode_fused_launch(p, B, D, VD, (hipStream_t)stream);
}

}  // extern "C"
