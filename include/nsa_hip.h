/* C ABI of libnsa_hip.so: MI355X (gfx950) kernels for the Native-Sparse-Attention hot path.
 *
 * Conventions
 *   - every pointer is a DEVICE pointer unless stated otherwise; tensors are bf16 unless stated otherwise;
 *   - strides are in ELEMENTS; "_st" = token/row stride, "_sh" = head stride; the channel dim is contiguous;
 *   - packed variable-length batches: x_cu [B+1] int32 token offsets, y_cu [B+1] int32 compressed-row offsets
 *     (y_len = max((L-kernel)/stride+1, 0) per sequence);
 *   - `stream` is a hipStream_t passed as void*; kernels are enqueued, never synchronised;
 *   - return value: 0 = ok, otherwise an error code; nsa_last_error() gives the message (thread local);
 *   - log-sum-exp outputs are in log2 units (m + log2(l)), as upstream stores them.
 * Citations name the upstream (mdy666/Scalable-Flash-Native-Sparse-Attention) interface each entry replaces.
 */
#ifndef NSA_HIP_H
#define NSA_HIP_H
#include <stdint.h>
#ifdef __cplusplus
extern "C" {
#endif

const char* nsa_last_error(void);
int nsa_abi_version(void);
/* Overrides one of the library's launch heuristics for this process (experiments and tests; nothing is read from
 * the environment): name (host string) = "fwd_variant", "dq_min_blocks", "dkdv_key_blocks" or "topk_seg_blocks"
 * (selection blocks per segment of the block selector: -1 = from the LDS budget, 0 = never segment).
 * nsa_reset_tuning restores every default.  No upstream counterpart. */
int nsa_set_tuning(const char* name, int value);
int nsa_reset_tuning(void);

/* flash_nsa/ops/compress_kv.py:335-366 mean_pooling_fwd */
int nsa_mean_pool_fwd(const void* x, int64_t x_st, int64_t x_sh, void* y, int64_t y_st, int64_t y_sh,
                      const int32_t* x_cu, const int32_t* y_cu, int B, int y_maxlen, int H, int D, int kernel_size,
                      int stride, void* stream);
/* flash_nsa/ops/compress_kv.py:368-399 mean_pooling_bwd; dx fp32 (optionally accumulated into) or bf16 */
int nsa_mean_pool_bwd(const void* dy, int64_t dy_st, int64_t dy_sh, void* dx, int64_t dx_st, int64_t dx_sh,
                      int dx_is_f32, int accumulate, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                      int H, int D, int kernel_size, int stride, void* stream);
/* flash_nsa/ops/compress_kv.py:126-170 construct_block_fwd; y contiguous [y_len,H,kernel,D] */
int nsa_construct_block_fwd(const void* x, int64_t x_st, int64_t x_sh, void* y, const int32_t* x_cu,
                            const int32_t* y_cu, int B, int y_maxlen, int H, int D, int kernel_size, int stride,
                            void* stream);
/* flash_nsa/ops/compress_kv.py:172-218 construct_block_bwd */
int nsa_construct_block_bwd(const void* dblock, void* dx, int64_t dx_st, int64_t dx_sh, int dx_is_f32,
                            int accumulate, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int H,
                            int D, int kernel_size, int stride, void* stream);
/* flash_nsa/ops/act.py:175-208 sigmoid_mul_fwd/bwd (act 0) and :60-100 swiglu_fwd/bwd (act 1);
 * x [N,2d] = gate|up, y [N,d], dx [N,2d] = dgate|dup (dx may alias x) */
int nsa_glu_fwd(const void* x, void* y, int64_t N, int d, int act, void* stream);
int nsa_glu_bwd(const void* x, const void* dy, void* dx, int64_t N, int d, int act, void* stream);

/* Learned compression without the windows in memory (flash_nsa/modules/megatron_level_nsa.py:46-86: construct_block, the
 * product with the weight and the activation).  w [N, kernel*D] with row stride w_st and contiguous columns; hidden [y_len,H,N]
 * contiguous = windows w^T in bf16; act -1: no activation, N = D; 0 / 1 as nsa_glu_fwd, N = 2D, out [y_len,H,D] = its activation, hidden
 * may be null. */
int nsa_compress_linear_fwd(const void* x, int64_t x_st, int64_t x_sh, const void* w, int64_t w_st, void* hidden, void* out,
                            const int32_t* x_cu, const int32_t* y_cu, int B, int y_maxlen, int H, int D, int kernel_size,
                            int stride, int N, int act, void* stream);
/* Its gradient with respect to x, from that of hidden: added to the fp32 dx, or, with dst, dst = bf16(dx + it) for every token
 * (dx is then only read; null: zeros). */
int nsa_compress_linear_bwd_dx(const void* dhidden, const void* w, int64_t w_st, void* dx, int64_t dx_st, int64_t dx_sh, void* dst,
                               int64_t dst_st, int64_t dst_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                               int H, int D, int kernel_size, int stride, int N, void* stream);
/* Its gradient with respect to w, summed in a fixed order: dw [N, kernel*D] contiguous, bf16 (stored) or fp32 (added to).
 * y_len = y_cu[B] > 0. */
int64_t nsa_compress_linear_bwd_dw_ws_bytes(int64_t y_len, int H, int D, int kernel_size, int N);
int nsa_compress_linear_bwd_dw(const void* dhidden, const void* x, int64_t x_st, int64_t x_sh, void* dw, int dw_is_f32,
                               const int32_t* x_cu, const int32_t* y_cu, int B, int64_t y_len, int H, int D, int kernel_size,
                               int stride, int N, void* ws, int64_t ws_bytes, void* stream);

/* dhidden [rows, N] (bf16) from the fp32 dy [rows, D], which is rounded to bf16 first; act as above (-1: dhidden = bf16(dy)). */
int nsa_compress_act_bwd(const void* hidden, const void* dy, void* dhidden, int64_t rows, int D, int act, void* stream);
/* nsa_mean_pool_bwd from the fp32 dy [y_len,H,D] (contiguous, rounded to bf16 first): dst = bf16(dx + it), dx fp32. */
int nsa_mean_pool_bwd_sum(const void* dy, const void* dx, int64_t dx_st, int64_t dx_sh, void* dst, int64_t dst_st, int64_t dst_sh,
                          const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int H, int D, int kernel_size, int stride,
                          void* stream);

/* flash_nsa/ops/combine.py:114-144 combine_fwd */
int nsa_combine_fwd(const void* a, const void* b, const void* c, int64_t i_st, int64_t i_sh, const void* w,
                    int64_t w_st, int64_t w_sh, void* o, int64_t o_st, int64_t o_sh, int64_t T, int H, int D,
                    void* stream);
/* flash_nsa/ops/combine.py:146-177 combine_bwd; da/db/dc contiguous [T,H,D], dw [T,H,3];
 * delta3 (optional, fp32 [3,T,H]) receives rowsum(x_k * dx_k) for the three branches */
int nsa_combine_bwd(const void* a, const void* b, const void* c, int64_t i_st, int64_t i_sh, const void* w,
                    int64_t w_st, int64_t w_sh, const void* dy, int64_t dy_st, int64_t dy_sh, void* da, void* db,
                    void* dc, void* dw, float* delta3, int64_t T, int H, int D, void* stream);
/* the same for kernels of the branches b = selected and c = window that read dy itself: da and delta3[0] as above;
 * delta3[k] = rowsum(x_k * dy) and lse2 [2,T,H] = lse_k - log2 sigmoid(w_k) (lse_k: the branch's log-sum-exp, any strides)
 * take the place of these branches' delta and lse.  For the tokens at positions below all_below, which select every
 * block they can see, c's values also carry b's gradient over the window's keys */
int nsa_combine_bwd_gates(const void* a, const void* b, const void* c, int64_t i_st, int64_t i_sh, const void* w,
                          int64_t w_st, int64_t w_sh, const void* dy, int64_t dy_st, int64_t dy_sh, const float* lse_b,
                          int64_t lb_st, int64_t lb_sh, const float* lse_c, int64_t lc_st, int64_t lc_sh, void* da,
                          void* dw, float* delta3, float* lse2, const int32_t* x_cu, int B, int all_below, int64_t T,
                          int H, int D, void* stream);
/* flash_nsa/ops/compress_attn.py:160-184 _bwd_preprocess: delta[T,H] fp32 = rowsum(o*do) */
int nsa_delta(const void* o, int64_t o_st, int64_t o_sh, const void* dO, int64_t d_st, int64_t d_sh, float* delta,
              int64_t T, int H, int D, void* stream);

/* flash_nsa/ops/compress_attn.py:531-592 cmp_attn_fwd; lse addressed tok*lse_st + head*lse_sh */
int nsa_cmp_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                     const void* cv, int64_t cv_sr, int64_t cv_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                     int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                     int QH, int KH, int D, int VD, int kernel_size, int stride, float sm_scale, void* stream);
/* flash_nsa/ops/sliding_window_attention.py:42-95 swa_fwd (FlashAttention varlen, window=(W,-1), causal) */
int nsa_swa_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                const void* v, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                int VD, int window, float sm_scale, void* stream);
/* nsa_swa_fwd, and in the same launch
 *   - the selected branch of the queries at positions below all_below, which select every block they can see: the window
 *     branch continued over the keys before the window -> slc_o / slc_lse (may be null) of those queries;
 *   - with `out`: the gated sum of the three branches (nsa_combine_fwd), the selected branch of the other queries read
 *     from slc_o.  store_branches 0: o and slc_o are then scratch that may or may not be written.
 * Without `out`, o may be null: x_maxlen = all_below then finishes the selected branch of those queries alone. */
int nsa_swa_fwd_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh, float* lse,
                     int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh, float* slc_lse,
                     int64_t sl_st, int64_t sl_sh, int all_below, const void* cmp_o, int64_t co_st, int64_t co_sh,
                     const void* w, int64_t w_st, int64_t w_sh, void* out, int64_t out_st, int64_t out_sh,
                     int store_branches, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD,
                     int window, float sm_scale, void* stream);
/* nsa_cmp_attn_fwd and nsa_swa_fwd_tail in one launch, for batches whose queries all select every block they can see: x_maxlen <=
 * all_below. */
int nsa_fwd_short(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh, const void* v,
                  int64_t v_sr, int64_t v_sh, const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cv, int64_t cv_sr,
                  int64_t cv_sh, void* cmp_o, int64_t co_st, int64_t co_sh, float* cmp_lse, int64_t cl_st, int64_t cl_sh, void* o,
                  int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh,
                  float* slc_lse, int64_t sl_st, int64_t sl_sh, int all_below, const void* w, int64_t w_st, int64_t w_sh, void* out,
                  int64_t out_st, int64_t out_sh, int store_branches, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                  int QH, int KH, int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream);
/* flash_nsa/ops/topk.py:630-775 slc_topk_indices; topk int32 addressed kh*tk_sh + tok*tk_st + slot;
 * imp_out optional fp32 block scores [KH, T, imp_cols] */
int nsa_topk_select(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                    const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                    float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols, const int32_t* x_cu,
                    const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int kernel_size, int stride,
                    int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                    void* stream);
/* The same selection in two launches, the fp32 block scores between them in `workspace` (upstream keeps them in its
 * slc_probs tensor between its two kernels, flash_nsa/ops/topk.py:226-425, 498-560): scoring then runs at twice the
 * occupancy of the one-launch kernel, which keeps the scores of its tokens in LDS.  total_tokens = tokens of the packed
 * batch (x_cu[B]).  nsa_topk_workspace_bytes(total_tokens, max_blocks, KH), max_blocks = selection blocks of the
 * longest sequence, is what one pass over all tokens needs; a smaller workspace makes the call work in chunks of as
 * many tokens as it holds (identical results).  workspace NULL, or a shape the two launches do not take (more than 16
 * q-heads per kv head, more than 2048 selection blocks, block sizes that are not 1..64 strides in powers of two):
 * the one-launch kernel runs, as in nsa_topk_select.  The workspace is scratch: nothing is kept between calls. */
int64_t nsa_topk_workspace_bytes(int total_tokens, int max_blocks, int KH);
int nsa_topk_select_ws(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                       const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                       float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols, const int32_t* x_cu,
                       const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int kernel_size, int stride,
                       int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                       int total_tokens, void* workspace, int64_t workspace_bytes, void* stream);
/* nsa_topk_select_ws without the selection of the queries at positions below t_begin: where the two launches run, their
 * topk rows are not written */
int nsa_topk_select_ws_from(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                            const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                            int64_t tk_st, float* imp_out, int64_t imp_sh, int64_t imp_st, int imp_cols,
                            const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                            int kernel_size, int stride, int block_size, int top_n, int num_init, int num_local,
                            int ignore_index, float sm_scale, int total_tokens, int t_begin, void* workspace,
                            int64_t workspace_bytes, void* stream);
/* flash_nsa/ops/select_attn.py:439-507 slc_attn_fwd */
int nsa_slc_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st,
                     void* o, int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh,
                     const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD, int block_size,
                     int top_n, float sm_scale, void* stream);
/* the same for the queries at positions >= t_begin only, as nsa_slc_attn_bwd_dq_from, nsa_paged_slc_attn_fwd_from and
 * nsa_build_inverse_index_from: the queries below top_n * block_size select every block they can see, and
 * nsa_swa_fwd_tail / nsa_swa_bwd_dq_tail / nsa_combine_bwd_gates finish their selected branch with the window's */
int nsa_slc_attn_fwd_from(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                          const void* v, int64_t v_sr, int64_t v_sh, const int32_t* topk, int64_t tk_sh,
                          int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st,
                          int64_t lse_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D, int VD,
                          int block_size, int top_n, int t_begin, float sm_scale, void* stream);

/* ---- backward ----
 * dq_mode: 0 = store bf16, 1 = store fp32, 2 = add into an existing fp32 buffer (single writer per element).
 * delta = rowsum(o * do) of the branch, fp32; lse as produced by the matching forward. */

/* flash_nsa/ops/compress_attn.py:701-736 (_cmp_dq_kernel launch) */
int nsa_cmp_attn_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                        const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu,
                        const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                        int stride, float sm_scale, void* stream);
/* Same kernel as nsa_cmp_attn_bwd_dq, as the LAST branch of the fused backward
 * (flash_nsa/modules/megatron_level_nsa.py:129-159 accumulates the three branches' dq and returns it in q's dtype):
 * dq [T,QH,D] bf16 = this branch's dq + dq_partial (fp32, the sum of the other branches), which saves the fp32
 * read-modify-write and the separate cast pass. */
int nsa_cmp_attn_bwd_dq_final(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                              int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                              int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                              const float* delta, int64_t delta_st, int64_t delta_sh, const float* dq_partial,
                              int64_t dqp_st, int64_t dqp_sh, void* dq, int64_t dq_st, int64_t dq_sh,
                              const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                              int VD, int kernel_size, int stride, float sm_scale, void* stream);
/* the same where the selected branch's dq is still to be added: dq of the positions below final_below, and this branch's dq
 * added into dq_partial for the others */
int nsa_cmp_attn_bwd_dq_final_below(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                                    int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                                    int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                                    const float* delta, int64_t delta_st, int64_t delta_sh, float* dq_partial,
                                    int64_t dqp_st, int64_t dqp_sh, void* dq, int64_t dq_st, int64_t dq_sh, int final_below,
                                    const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH, int D,
                                    int VD, int kernel_size, int stride, float sm_scale, void* stream);
/* flash_nsa/ops/compress_attn.py:650-690 (_cmp_dkdv_kernel launch, dkdv_repeat=False): fp32 atomic adds into
 * dck/dcv [y_len,KH,*], which the caller zero-fills; queries are cut into chunks of q_chunk_tokens
 * (<= 0: chosen from the sizes so that short batches still fill the GPU) */
int nsa_cmp_attn_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                          const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st,
                          int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                          int64_t delta_st, int64_t delta_sh, float* dck, int64_t dck_sr, int64_t dck_sh,
                          float* dcv, int64_t dcv_sr, int64_t dcv_sh, const int32_t* x_cu, const int32_t* y_cu,
                          int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                          int stride, int q_chunk_tokens, float sm_scale, void* stream);
/* The same with a summation order that does not depend on the run (upstream's dkdv_repeat=True: per-head buffers and a
 * final sum, flash_nsa/ops/compress_attn.py:594-598,691-693; here the q-heads of a group are summed inside the matrix
 * accumulators and what remains to be ordered are the query chunks): every work item stores its fp32 partial result
 * in its own slot of `workspace` (nsa_cmp_attn_bwd_dkdv_det_bytes(...) bytes, same sizes and q_chunk_tokens as the
 * call), a second launch sums the slots of a key in ascending chunk order and stores dck / dcv (no zero-fill needed
 * for the keys it writes; keys no query sees keep what the buffers held). */
int64_t nsa_cmp_attn_bwd_dkdv_det_bytes(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                                        int kernel_size, int stride, int q_chunk_tokens);
int nsa_cmp_attn_bwd_dkdv_det(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr,
                              int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO,
                              int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                              const float* delta, int64_t delta_st, int64_t delta_sh, float* dck, int64_t dck_sr,
                              int64_t dck_sh, float* dcv, int64_t dcv_sr, int64_t dcv_sh, const int32_t* x_cu,
                              const int32_t* y_cu, int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                              int kernel_size, int stride, int q_chunk_tokens, float sm_scale, void* workspace,
                              int64_t workspace_bytes, void* stream);
/* flash_nsa/ops/sliding_window_attention.py:98-157 swa_bwd (FlashAttention varlen backward) */
int nsa_swa_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                   const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                   const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                   int64_t delta_sh, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu,
                   int B, int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream);
/* dq of the compressed branch, the window and, for the queries at positions below all_below, the keys before it, in one: those
 * queries' dq goes to dq in bf16, that of the others to the fp32 dq_partial (may be null if x_maxlen <= all_below).  The gradients,
 * log-sum-exps and deltas of window, selected and compressed branch as nsa_swa_bwd_dq_tail and nsa_cmp_attn_bwd_dq take them. */
int nsa_bwd_dq_dense(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh, const void* v, int64_t v_sr,
                     int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh,
                     const float* delta, int64_t delta_st, int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh,
                     const float* slc_lse, int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                     int all_below, const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cv, int64_t cv_sr, int64_t cv_sh,
                     const void* cmp_dO, int64_t cdo_st, int64_t cdo_sh, const float* cmp_lse, int64_t cl_st, int64_t cl_sh,
                     const float* cmp_delta, int64_t cd_st, int64_t cd_sh, void* dq, int64_t dq_st, int64_t dq_sh, float* dq_partial,
                     int64_t dqp_st, int64_t dqp_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH, int KH,
                     int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream);
/* nsa_swa_bwd_dq with dq_mode 2 (add into fp32) for gradients from nsa_combine_bwd_gates: the queries at positions below
 * all_below also take the selected branch's keys before their window, and their dq is stored instead of added */
int nsa_swa_bwd_dq_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh, const float* slc_lse,
                        int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                        int all_below, float* dq, int64_t dq_st, int64_t dq_sh, const int32_t* x_cu, int B,
                        int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream);
/* the same where this branch is the first to write dq: stores for every query */
int nsa_swa_bwd_dq_tail_store(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                              const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                              const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                              int64_t delta_sh, const void* slc_dO, int64_t sdo_st, int64_t sdo_sh, const float* slc_lse,
                              int64_t sl_st, int64_t sl_sh, const float* slc_delta, int64_t sd_st, int64_t sd_sh,
                              int all_below, float* dq, int64_t dq_st, int64_t dq_sh, const int32_t* x_cu, int B,
                              int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale, void* stream);
/* same upstream site; dk/dv are stored (every key row has exactly one writer), bf16 or fp32 */
int nsa_swa_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                     const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                     const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                     int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                     int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                     int VD, int window, float sm_scale, void* stream);
/* the same with a workspace (16-byte aligned, contents undefined) of nsa_swa_bwd_dkdv_ws_bytes(...): where that is not 0,
 * the queries of a key tile are cut into chunks, so that a batch of few key tiles fills the GPU; every chunk stores its
 * partial result in the workspace and a second launch adds them in a fixed order: no run differs from another */
int64_t nsa_swa_bwd_dkdv_ws_bytes(int B, int x_maxlen, int QH, int KH, int D, int VD, int window);
int nsa_swa_bwd_dkdv_ws(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                        int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                        int D, int VD, int window, float sm_scale, void* workspace, int64_t workspace_bytes,
                        void* stream);
/* flash_nsa/ops/select_attn.py:650-695 (_dq_kernel launch) */
int nsa_slc_attn_bwd_dq(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st, void* dq,
                        int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu, int B, int x_maxlen, int QH,
                        int KH, int D, int VD, int block_size, int top_n, float sm_scale, void* stream);
int nsa_slc_attn_bwd_dq_from(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st, void* dq,
                        int64_t dq_st, int64_t dq_sh, int dq_mode, const int32_t* x_cu, int B, int x_maxlen, int QH,
                        int KH, int D, int VD, int block_size, int top_n, int t_begin,
                        float sm_scale, void* stream);
/* dk/dv of the selected branch of the queries at positions below all_below over the keys before their window, added into
 * the caller's fp32 buffers (the keys of the window are in the window branch's gradient: nsa_combine_bwd_gates).  ordered:
 * the summation order does not change between runs */
int nsa_slc_attn_bwd_dkdv_before_window(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr,
                                        int64_t k_sh, const void* v, int64_t v_sr, int64_t v_sh, const void* dO,
                                        int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st,
                                        int64_t lse_sh, const float* delta, int64_t delta_st, int64_t delta_sh,
                                        float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                                        int64_t dv_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                                        int D, int VD, int window, int all_below, int ordered, float sm_scale,
                                        void* stream);
/* flash_nsa/ops/topk.py:889-945 get_bind_from_find: inverse of the selection as a CSR.
 *   csr_off  [KH][nblk_total+1] absolute start of each (kv head, global block) list inside csr_tok
 *   csr_tok  [KH*T*top_n]       query tokens (index local to their sequence), ascending within a list
 *   item_off [KH][nblk_total+1] prefix count of list chunks of chunk_tokens tokens (work items of the dk/dv pass)
 *   workspace: int32 scratch of nsa_inverse_index_workspace_elems(T,KH,nblk_total) elements
 * nsa_slc_bwd_chunk_tokens: the chunk_tokens this library suggests for a batch of T tokens (256, less when that
 * would leave the dk/dv pass too few work items); any positive value is valid as long as the
 * builder and nsa_slc_attn_bwd_dkdv get the same one */
int64_t nsa_inverse_index_workspace_elems(int T, int KH, int nblk_total);
int nsa_slc_bwd_chunk_tokens(int T, int KH, int top_n);
int nsa_build_inverse_index(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                            const int32_t* kblk_cu, int B, int T, int KH, int nblk_total, int block_size,
                            int chunk_tokens, int32_t* csr_off, int32_t* csr_tok, int32_t* item_off,
                            int32_t* workspace, int64_t workspace_elems, void* stream);
/* the same over the queries at positions >= t_begin only */
int nsa_build_inverse_index_from(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                                 const int32_t* kblk_cu, int B, int T, int KH, int nblk_total, int block_size,
                                 int chunk_tokens, int t_begin, int32_t* csr_off, int32_t* csr_tok, int32_t* item_off,
                                 int32_t* workspace, int64_t workspace_elems, void* stream);
/* the same over the tokens tok0 .. tok0 + T - 1 of the batch (csr_tok [KH*T*top_n]); csr_slot (or NULL) [KH*T*top_n]: the
 * position in the token's selection that an entry of csr_tok stands for */
int nsa_build_inverse_index_slots(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                                  const int32_t* kblk_cu, int B, int tok0, int T, int KH, int nblk_total,
                                  int block_size, int chunk_tokens, int t_begin, int32_t* csr_off, int32_t* csr_tok,
                                  uint8_t* csr_slot, int32_t* item_off, int32_t* workspace, int64_t workspace_elems,
                                  void* stream);
/* flash_nsa/ops/select_attn.py:593-637 (_dkdv_kernel launch): fp32 atomic adds into dk/dv [T,KH,*];
 * blk_seq [nblk_total] = sequence of each global block; n_items_bound >= max over kv heads of item_off[kh][nblk_total] */
int nsa_slc_attn_bwd_dkdv(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                          const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st,
                          int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                          int64_t delta_st, int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh, float* dv,
                          int64_t dv_sr, int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu,
                          const int32_t* blk_seq, const int32_t* csr_off, const int32_t* csr_tok,
                          const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B,
                          int QH, int KH, int D, int VD, int block_size, float sm_scale, void* stream);
/* nsa_slc_attn_bwd_dkdv and nsa_slc_attn_bwd_dq_from for the tokens tok0 .. tok0 + ntok - 1 of the batch (with the index that
 * nsa_build_inverse_index_slots makes of them): the dk/dv pass leaves its dS in `ds` (nsa_slc_bwd_ds_bytes(ntok, ...) bytes),
 * from which the dq pass has dq = dS k.  dq_mode 3: bf16 store of the result added to the fp32 dq_partial.
 * nsa_slc_bwd_ds_tokens: tokens per call for a batch of T tokens, T where one call does; 0: shapes, strides or a scale that
 * take the other entry points, or shapes of which the scratch's limit (2 GB) does not hold 512 tokens. */
int nsa_slc_bwd_ds_tokens(int T, int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, int block_size,
                          int top_n, float sm_scale);
int64_t nsa_slc_bwd_ds_bytes(int ntok, int QH, int KH, int block_size, int top_n);
int nsa_slc_attn_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                             const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                             const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                             int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                             int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu, const int32_t* blk_seq,
                             const int32_t* csr_off, const int32_t* csr_tok, const uint8_t* csr_slot,
                             const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B, int QH,
                             int KH, int D, int VD, int block_size, int top_n, int tok0, int ntok, float sm_scale, void* ds,
                             int64_t ds_bytes, void* stream);
int nsa_slc_attn_bwd_dq_ds(const void* k, int64_t k_sr, int64_t k_sh, const int32_t* topk, int64_t tk_sh, int64_t tk_st,
                           void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, const float* dq_partial, int64_t dqp_st,
                           int64_t dqp_sh, const int32_t* x_cu, int B, int QH, int KH, int D, int VD, int block_size,
                           int top_n, int t_begin, int tok0, int ntok, float sm_scale, const void* ds, int64_t ds_bytes,
                           void* stream);
/* The same with a run-independent summation order (upstream's dkdv_repeat=True, flash_nsa/ops/select_attn.py:528-531,
 * 639-641): every work item (a chunk of a block's token list) stores its partial result in its own slot of
 * `workspace` (nsa_slc_attn_bwd_dkdv_det_bytes(...) bytes), a second launch adds the slots of a block to dk / dv in
 * ascending chunk order, one thread per element. */
int64_t nsa_slc_attn_bwd_dkdv_det_bytes(int n_items_bound, int KH, int D, int VD, int block_size);
int nsa_slc_attn_bwd_dkdv_det(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                              const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st,
                              int64_t do_sh, const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta,
                              int64_t delta_st, int64_t delta_sh, float* dk, int64_t dk_sr, int64_t dk_sh,
                              float* dv, int64_t dv_sr, int64_t dv_sh, const int32_t* x_cu, const int32_t* kblk_cu,
                              const int32_t* blk_seq, const int32_t* csr_off, const int32_t* csr_tok,
                              const int32_t* item_off, int nblk_total, int chunk_tokens, int n_items_bound, int B,
                              int QH, int KH, int D, int VD, int block_size, float sm_scale, void* workspace,
                              int64_t workspace_bytes, void* stream);
/* dQ of the range-keyed branches from the dS that their dk / dv kernels leave behind (8, 16, 32 or 64 q-heads per kv head with
 * head dims 128/128 or 192/128): the dk / dv kernel of a branch also stores dS, bf16, in tiles of 64 rows, and one
 * launch forms dQ = dS K of the compressed branch, the window and the keys before the window (of the queries below all_below)
 * together.  The batch (T rows) is processed in ranges of tokens [tok0, tok1) in ascending order (tok1 = 0: all of it in one;
 * otherwise the range of 128-position groups of a sequence whose first token it holds), so that the scratch stays bounded:
 * nsa_bwd_ds_range_end gives the end of the range that begins at tok0 (T: the last one), in which no branch takes more than
 * 4 GB (stride 0: without the compressed branch, window -1: without the window), or -1 where a range of 16384 / QH tokens would
 * (sequences past a million tokens; past a window of many thousand keys) or all_below tokens of one sequence would: dq is then
 * to be computed apart.  nsa_bwd_ds_next: the same ranges of the compressed branch and the window alone, at
 * least as long as fills the GPU, whatever they take.
 * nsa_bwd_ds_takes: 1 where these shapes, strides and scale have this path.  nsa_*_ds_bytes: scratch of a branch; `ring` is
 * the length of the longest range (0: one range).  The window's scratch holds what the next range needs: the same buffer is
 * passed for all ranges, and a range's dk / dv kernels run after the dq launch of the range before. */
int nsa_bwd_ds_takes(int64_t q_sh, int64_t do_sh, int64_t k_sr, int QH, int KH, int D, int VD, float sm_scale);
int nsa_bwd_ds_range_end(int tok0, int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int window,
                         int all_below);
int nsa_bwd_ds_next(int tok0, int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int window);
int64_t nsa_cmp_attn_bwd_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int kernel_size, int stride, int tok0,
                                  int tok1);
int64_t nsa_swa_bwd_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int window, int ring);
int64_t nsa_slc_bwd_before_window_ds_bytes(int T, int B, int x_maxlen, int QH, int KH, int window, int all_below, int ring);
/* nsa_cmp_attn_bwd_dkdv that stores dS.  Without workspace dck / dcv are added into with fp32 atomics; with
 * nsa_cmp_attn_bwd_dkdv_ds_slot_bytes(...) bytes of it the work items' sums are added in a fixed order and stored (add: added
 * to what the ranges before have left).  nsa_cmp_attn_bwd_dkdv_ds_items: work items of the launch per sequence and kv head,
 * with q_chunk_tokens query tokens in one (0: as many as the launch takes); one slot each. */
int64_t nsa_cmp_attn_bwd_dkdv_ds_items(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                                       int stride, int q_chunk_tokens, int tok0, int tok1);
int64_t nsa_cmp_attn_bwd_dkdv_ds_slot_bytes(int B, int x_maxlen, int y_maxlen, int QH, int KH, int D, int VD,
                                            int kernel_size, int stride, int tok0, int tok1);
int nsa_cmp_attn_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* ck, int64_t ck_sr, int64_t ck_sh,
                             const void* cv, int64_t cv_sr, int64_t cv_sh, const void* dO, int64_t do_st, int64_t do_sh,
                             const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                             int64_t delta_sh, float* dck, int64_t dck_sr, int64_t dck_sh, float* dcv, int64_t dcv_sr,
                             int64_t dcv_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int y_maxlen,
                             int QH, int KH, int D, int VD, int kernel_size, int stride, float sm_scale, int T, int tok0,
                             int tok1, void* ds, int64_t ds_bytes, void* workspace, int64_t workspace_bytes, int add,
                             void* stream);
/* nsa_swa_bwd_dkdv_ws and nsa_slc_attn_bwd_dkdv_before_window that store dS: keys of the range, every key once. */
int64_t nsa_swa_bwd_dkdv_ds_ws_bytes(int T, int B, int x_maxlen, int QH, int KH, int D, int VD, int window, int tok0,
                                     int tok1);
int nsa_swa_bwd_dkdv_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr, int64_t k_sh,
                        const void* v, int64_t v_sr, int64_t v_sh, const void* dO, int64_t do_st, int64_t do_sh,
                        const float* lse, int64_t lse_st, int64_t lse_sh, const float* delta, int64_t delta_st,
                        int64_t delta_sh, void* dk, int64_t dk_sr, int64_t dk_sh, void* dv, int64_t dv_sr,
                        int64_t dv_sh, int dkv_is_f32, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH, int D,
                        int VD, int window, float sm_scale, int T, int ring, int tok0, int tok1, void* ds,
                        int64_t ds_bytes, void* workspace, int64_t workspace_bytes, void* stream);
int nsa_slc_attn_bwd_dkdv_before_window_ds(const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sr,
                                           int64_t k_sh, const void* v, int64_t v_sr, int64_t v_sh, const void* dO,
                                           int64_t do_st, int64_t do_sh, const float* lse, int64_t lse_st,
                                           int64_t lse_sh, const float* delta, int64_t delta_st, int64_t delta_sh,
                                           float* dk, int64_t dk_sr, int64_t dk_sh, float* dv, int64_t dv_sr,
                                           int64_t dv_sh, const int32_t* x_cu, int B, int x_maxlen, int QH, int KH,
                                           int D, int VD, int window, int all_below, float sm_scale, int T, int ring,
                                           int tok0, int tok1, void* ds, int64_t ds_bytes, void* stream);
/* dq of the tokens of a range from what the calls above have stored (a null dS leaves the branch out).  dq_mode 0: bf16, 1:
 * fp32, 2: added into fp32, 3: bf16 to dq at positions below all_below, fp32 to dq_partial for the others. */
int nsa_attn_bwd_dq_ds(const void* ck, int64_t ck_sr, int64_t ck_sh, const void* cmp_ds, int64_t cmp_ds_bytes, const void* k,
                       int64_t k_sr, int64_t k_sh, const void* swa_ds, int64_t swa_ds_bytes, const void* far_ds,
                       int64_t far_ds_bytes, void* dq, int64_t dq_st, int64_t dq_sh, int dq_mode, float* dq_partial,
                       int64_t dqp_st, int64_t dqp_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int QH,
                       int KH, int D, int VD, int kernel_size, int stride, int window, int all_below, float sm_scale, int T,
                       int ring, int tok0, int tok1, void* stream);

/* ---- paged KV (inference).  Caches are [num_pages, page_size, KH, D]; *_sr is the stride of a flat row
 * (page*page_size + offset), *_sh the head stride.  Request b's raw token n lives at flat row
 * block_tables[b][n/page]*page + n%page; its compressed row i at cmp_block_tables[b][i/page]*page + i%page of the
 * SAME pool.  x_cu counts only the new query tokens; query n of request b sits at absolute position
 * n + context_lens[b] - x_len[b].  page_size must be a multiple of 64. */

/* flash_nsa/inference/compress_attn.py:486-538 cmp_attn_prefill (and, with one query per request, :540-667 decode) */
int nsa_paged_cmp_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st,
                           int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh, const int32_t* x_cu,
                           const int32_t* context_lens, const int32_t* cmp_block_tables, int table_stride,
                           int page_size, int B, int x_maxlen, int QH, int KH, int D, int VD, int kernel_size,
                           int stride, float sm_scale, void* stream);
/* flash_nsa/inference/__init__.py:125-155 (FlashAttention with page table and window) */
int nsa_paged_swa_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                      const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh,
                      float* lse, int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                      const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen, int QH,
                      int KH, int D, int VD, int window, float sm_scale, void* stream);
int nsa_paged_swa_fwd_tail(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                           const void* v_cache, int64_t v_sr, int64_t v_sh, void* o, int64_t o_st, int64_t o_sh,
                           float* lse, int64_t lse_st, int64_t lse_sh, void* slc_o, int64_t so_st, int64_t so_sh,
                           float* slc_lse, int64_t sl_st, int64_t sl_sh, int all_below, const void* cmp_o,
                           int64_t co_st, int64_t co_sh, const void* w, int64_t w_st, int64_t w_sh, void* out,
                           int64_t out_st, int64_t out_sh, int store_branches, const int32_t* x_cu,
                           const int32_t* context_lens, const int32_t* block_tables, int table_stride, int page_size,
                           int B, int x_maxlen, int QH, int KH, int D, int VD, int window, float sm_scale,
                           void* stream);
/* nsa_paged_cmp_attn_fwd and nsa_paged_swa_fwd_tail (gated sum alone) in one launch, for requests whose contexts are no longer than
 * all_below; cmp_o, o and slc_o are scratch. */
int nsa_paged_fwd_short(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                        const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh, void* o,
                        int64_t o_st, int64_t o_sh, void* slc_o, int64_t so_st, int64_t so_sh, int all_below, const void* w,
                        int64_t w_st, int64_t w_sh, void* out, int64_t out_st, int64_t out_sh, const int32_t* x_cu,
                        const int32_t* context_lens, const int32_t* block_tables, int table_stride,
                        const int32_t* cmp_block_tables, int cmp_table_stride, int page_size, int B, int x_maxlen, int QH, int KH,
                        int D, int VD, int kernel_size, int stride, int window, float sm_scale, void* stream);
/* flash_nsa/inference/topk.py:184-298 topk_prefill / :495-623 topk_decode (causality is masked per row here) */
int nsa_paged_topk_select(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                          int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                          int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                          const int32_t* cmp_block_tables, int table_stride, int page_size, int B, int x_maxlen,
                          int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size, int stride,
                          int block_size, int top_n, int num_init, int num_local, int ignore_index, float sm_scale,
                          void* stream);
/* nsa_paged_topk_select in two launches with a workspace, as nsa_topk_select_ws (max_blocks = fixed_num_slc_blocks) */
int nsa_paged_topk_select_ws(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                             int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                             int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                             const int32_t* cmp_block_tables, int table_stride, int page_size, int B, int x_maxlen,
                             int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size, int stride,
                             int block_size, int top_n, int num_init, int num_local, int ignore_index,
                             float sm_scale, int total_tokens, void* workspace, int64_t workspace_bytes,
                             void* stream);
int nsa_paged_topk_select_ws_from(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                                  int64_t k_sh, const float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                                  int64_t tk_sh, int64_t tk_st, const int32_t* x_cu, const int32_t* context_lens,
                                  const int32_t* cmp_block_tables, int table_stride, int page_size, int B,
                                  int x_maxlen, int fixed_num_slc_blocks, int QH, int KH, int D, int kernel_size,
                                  int stride, int block_size, int top_n, int num_init, int num_local,
                                  int ignore_index, float sm_scale, int total_tokens, int t_begin, void* workspace,
                                  int64_t workspace_bytes, void* stream);
/* flash_nsa/inference/select_attn.py:103-166 slc_attn_prefill */
int nsa_paged_slc_attn_fwd(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const int32_t* topk,
                           int64_t tk_sh, int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse,
                           int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                           const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen,
                           int QH, int KH, int D, int VD, int block_size, int top_n, float sm_scale, void* stream);
int nsa_paged_slc_attn_fwd_from(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const int32_t* topk,
                           int64_t tk_sh, int64_t tk_st, void* o, int64_t o_st, int64_t o_sh, float* lse,
                           int64_t lse_st, int64_t lse_sh, const int32_t* x_cu, const int32_t* context_lens,
                           const int32_t* block_tables, int table_stride, int page_size, int B, int x_maxlen,
                           int QH, int KH, int D, int VD, int block_size, int top_n, int t_begin,
                           float sm_scale, void* stream);

/* flash_nsa/inference/compress_kv.py:191-220 mean_pooling_prefill (in-pool write at flat row slot) */
int nsa_paged_pool_prefill(void* cache, int64_t c_sr, int64_t c_sh, const int32_t* y_cu, const int32_t* block_tables,
                           int table_stride, const int32_t* cmp_slot_mapping, int B, int y_maxlen, int page_size,
                           int H, int D, int kernel_size, int stride, void* stream);
/* flash_nsa/inference/compress_kv.py:253-287 kv_mean_pooling_decode */
int nsa_paged_pool_decode(void* k_cache, int64_t k_sr, int64_t k_sh, int Dk, void* v_cache, int64_t v_sr,
                          int64_t v_sh, int Dv, const int32_t* context_lens, const int32_t* block_tables,
                          int table_stride, const int32_t* cmp_slot_mapping, int B, int page_size, int H,
                          int kernel_size, int stride, void* stream);

/* ---- the layer around the core ----
 * flash_nsa/ops/rope.py:13-232 fused_apply_rope: rotate-half RoPE of q [B,N,QH,D] and k [B,N,KH,D] (element strides
 * per batch / token / head, last dim contiguous) with cos / sin [B,N,D] (bf16, or fp32 when cos_is_fp32; a batch
 * stride of 0 broadcasts one table); qe / ke may alias q / k (in place).  backward != 0 applies the inverse
 * rotation to incoming gradients. */
int nsa_rope(const void* q, int64_t q_sb, int64_t q_sn, int64_t q_sh, const void* k, int64_t k_sb, int64_t k_sn,
             int64_t k_sh, void* qe, int64_t qe_sb, int64_t qe_sn, int64_t qe_sh, void* ke, int64_t ke_sb,
             int64_t ke_sn, int64_t ke_sh, const void* cos, const void* sin, int64_t c_sb, int64_t c_sn,
             int cos_is_fp32, int B, int N, int QH, int KH, int D, int backward, void* stream);

/* ---- KV-cache writer (the caller side of the paged entry points) ----
 * nano-vllm/nanovllm/layers/attention.py:123-153 store_kvcache: row n of key / value (k_row_elems = KH*D contiguous
 * elements, row stride k_st) is copied to flat pool row slot_mapping[n] of k_cache / v_cache (row stride kc_sr);
 * negative slots are skipped. */
int nsa_store_kvcache(const void* key, int64_t k_st, const void* value, int64_t v_st, void* k_cache, int64_t kc_sr,
                      void* v_cache, int64_t vc_sr, const int32_t* slot_mapping, int N, int k_row_elems,
                      int v_row_elems, void* stream);
/* One launch for a prefill chunk: store_kvcache of the chunk's new tokens (key / value [t,KH,D] packed by x_cu,
 * slot_mapping [t]) + mean pooling of the compressed rows listed in cmp_slot_mapping (as nsa_paged_pool_prefill,
 * flash_nsa/inference/compress_kv.py:191-220, for K and V).  Source rows of a pooled window are taken from the
 * chunk when they are new (position >= context_lens[b] - new tokens of b) and from the pool otherwise. */
int nsa_paged_store_pool_prefill(const void* key, int64_t k_st, int64_t k_sh, int Dk, const void* value, int64_t v_st,
                                 int64_t v_sh, int Dv, void* k_cache, int64_t kc_sr, int64_t kc_sh, void* v_cache,
                                 int64_t vc_sr, int64_t vc_sh, const int32_t* x_cu, const int32_t* context_lens,
                                 const int32_t* slot_mapping, const int32_t* y_cu, const int32_t* cmp_slot_mapping,
                                 const int32_t* block_tables, int table_stride, int B, int x_maxlen, int y_maxlen,
                                 int page_size, int H, int kernel_size, int stride, void* stream);

/* ---- fused decode step (one query token per request; q [B,QH,D], at most 16 q-heads per kv head) ----
 * Replaces flash_nsa/inference/compress_attn.py:540-667 (cmp_attn_decode) + inference/topk.py:495-623 (topk_decode):
 * compressed attention (cmp_o [B,QH,VD], optional lse addressed b*lse_st + head*lse_sh) and the top-n selection
 * topk[kh*tk_sh + b*tk_st + slot]; call after nsa_paged_pool_decode. */
int nsa_decode_cmp_topk(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                        const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh,
                        float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                        const int32_t* context_lens, const int32_t* cmp_block_tables, int cmp_table_stride,
                        int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                        int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n,
                        int num_init, int num_local, int ignore_index, float sm_scale, void* stream);
/* Split variant of the compressed branch for batches whose context lengths differ widely (two launches, grid
 * B x KH x nsplit): partial attention per key-interleaved split, then merge (cmp_o, lse) + head-summed probabilities
 * pg [B,KH,fixed_y_maxlen] fp32 of every compressed key.  Scratch (fp32): sp_m, sp_l [B,KH,nsplit,16],
 * sp_o [B,KH,nsplit,16,VD].  The selection itself then runs in the prologue of nsa_decode_slc_swa_combine. */
int nsa_decode_cmp_split(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                         const void* v_cache, int64_t v_sr, int64_t v_sh, void* cmp_o, int64_t co_st, int64_t co_sh,
                         float* lse, int64_t lse_st, int64_t lse_sh, float* pg, float* sp_m, float* sp_l, float* sp_o,
                         int nsplit, const int32_t* context_lens, const int32_t* cmp_block_tables,
                         int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD,
                         int fixed_y_maxlen, int kernel_size, int stride, float sm_scale, void* stream);
/* The decode step of flash_nsa/inference/__init__.py:207-257 for small batches of long contexts, in two launches:
 * (1) the compressed branch cut into nsplit key-interleaved parts per (request, kv head) -- partial (m, l, o) and the
 * un-normalised fp16 probabilities of every compressed key go to scratch; (2) per (request, kv head): merge of the
 * parts, block scores, selection, selected-block + window attention, gated combine.  cmp_slot_mapping [B] (-1: no
 * compressed row completes at this step) makes launch (1) pool the newest compressed row, as nsa_paged_pool_decode
 * would; null: the row must be in the pool already.  Scratch, all caller-allocated, contents undefined:
 *   sp_m, sp_l [B,KH,nsplit,16] fp32; sp_o [B,KH,nsplit,16,VD] fp32;
 *   sp_keep_p [B,KH,Y/32,16,32] fp16 and sp_keep_m [B,KH,Y/32,16] fp32 with Y = fixed_y_maxlen rounded up to 32.
 * cmp_o / slc_o / swa_o / lse / topk are optional outputs (null: not written).
 * nsa_decode_split_fits: 1 when fixed_y_maxlen / fixed_num_slc_blocks / the raw table width fit the LDS of (2). */
int nsa_decode_split_fits(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride);
/* LDS bytes of launch (2), dynamic + statically declared, for these capacities; 0 when they do not fit 160 KB */
int nsa_decode_split_lds_total(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride);
/* LDS bytes of the larger launch of nsa_decode_cmp_topk (parts != 0: nsa_decode_cmp_split) + nsa_decode_slc_swa_combine at
 * these capacities; 0: over the limit, the launches would be refused */
int nsa_decode_two_launch_lds(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride,
                              int page_size, int parts);
int nsa_decode_split(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr, int64_t k_sh,
                     const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st, int64_t w_sh,
                     void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o, int64_t co_st,
                     int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk, int64_t tk_sh,
                     int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p, float* sp_keep_m,
                     int nsplit, const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                     const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                     int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD, int fixed_y_maxlen,
                     int fixed_num_slc_blocks, int kernel_size, int stride, int block_size, int top_n, int num_init,
                     int num_local, int ignore_index, int window, float sm_scale, void* stream);
/* nsa_decode_split with the window attended in launch (1), by win_parts (0..4; 0 = nsa_decode_split) workgroups per
 * (request, kv head); launch (2) attends the blocks that are selected whatever their score next to the selection instead.
 * Extra scratch (caller-allocated, contents undefined): win_ml [2,B,KH,win_parts,16] fp32, win_o
 * [B,KH,win_parts,16,VD] fp32.  nsa_decode_split_window_parts: the number of parts this library suggests. */
int nsa_decode_split_window_parts(int window, int fixed_y_maxlen, int nsplit);
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
                     float* win_ml, float* win_o, void* stream);
/* the same (win_parts > 0), launch (1) also writing the newest token's K / V new_k / new_v [B,KH,*] to the flat pool rows
 * slot_mapping [B] (-1: none), as nsa_decode_fused does */
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
                     int64_t nv_st, int64_t nv_sh, const int32_t* slot_mapping, void* stream);
/* nsa_decode_split with launch (2) cut as well: upstream's slc_num_splits (flash_nsa/inference/__init__.py:195-196,
 * inference/select_attn.py:329-331,492-498 -- the selected blocks of one token dealt over several programs, merged
 * through fp32 partials).  Here slc_nsplit workgroups per (request, kv head) share the window units and the selected
 * blocks (every one of them repeats the merge of the compressed parts and the selection), and a third launch merges
 * their partial results and applies the gates.  Worth it only when B x KH workgroups leave most of the GPU idle.
 * slc_nsplit in [1,16]; 1 = nsa_decode_split.  Extra scratch (caller-allocated, contents undefined):
 *   sp2_ml [B,KH,slc_nsplit,2,2,16] fp32, sp2_o [B,KH,slc_nsplit,2,16,VD] fp32, cmp_tmp [B,QH,VD] bf16 addressed with
 *   co_st / co_sh. */
int nsa_decode_split_parts(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                           int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w, int64_t w_st,
                           int64_t w_sh, void* out, int64_t o_st, int64_t o_sh, void* cmp_o, void* slc_o, void* swa_o,
                           int64_t co_st, int64_t co_sh, float* lse, int64_t lse_st, int64_t lse_sh, int32_t* topk,
                           int64_t tk_sh, int64_t tk_st, float* sp_m, float* sp_l, float* sp_o, void* sp_keep_p,
                           float* sp_keep_m, int nsplit, const int32_t* cmp_slot_mapping,
                           const int32_t* context_lens, const int32_t* block_tables, int table_stride,
                           const int32_t* cmp_block_tables, int cmp_table_stride, int page_size, int B, int QH,
                           int KH, int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size,
                           int stride, int block_size, int top_n, int num_init, int num_local, int ignore_index,
                           int window, float sm_scale, int slc_nsplit, float* sp2_ml, float* sp2_o, void* cmp_tmp,
                           void* stream);
/* nsa_decode_split without any allocation.  No counterpart upstream: it is for callers that cannot allocate device
 * memory around the call (code under graph capture, tight serving loops, harnesses that forbid hipMalloc).  The
 * arguments are those of nsa_decode_split minus the five scratch buffers, which are carved out of one file-scope
 * device array of nsa_decode_split_static_capacity() bytes (32 MiB, held by every GPU the library runs on until the
 * process ends).  nsa_decode_split_static_bytes gives the bytes a call needs (e.g. 22.1 MB for 16 requests x 4 kv
 * heads x 8 parts at fixed_y_maxlen 8192); a call that needs more is refused with NSA_ERR_UNSUPPORTED.  All calls on
 * one GPU share the array: calls that overlap there (other streams or threads) race.  Neither this entry point nor
 * anything below it calls hipMalloc / hipFree. */
int64_t nsa_decode_split_static_capacity(void);
int64_t nsa_decode_split_static_bytes(int B, int KH, int VD, int nsplit, int fixed_y_maxlen);
int nsa_decode_split_static(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                            int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w,
                            int64_t w_st, int64_t w_sh, void* out, int64_t o_st, int64_t o_sh, void* cmp_o,
                            void* slc_o, void* swa_o, int64_t co_st, int64_t co_sh, float* lse, int64_t lse_st,
                            int64_t lse_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st, int nsplit,
                            const int32_t* cmp_slot_mapping, const int32_t* context_lens,
                            const int32_t* block_tables, int table_stride, const int32_t* cmp_block_tables,
                            int cmp_table_stride, int page_size, int B, int QH, int KH, int D, int VD,
                            int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size, int stride,
                            int block_size, int top_n, int num_init, int num_local, int ignore_index, int window,
                            float sm_scale, void* stream);
/* Replaces flash_nsa/inference/select_attn.py:655-787 (fused_slc_swa_attn_decode) + inference/combine.py:104-127
 * (combine_decode): selected-block and window attention; slc_o / swa_o (optional, same strides as cmp_o) receive the
 * branch outputs; out (optional) = cmp_o*sig(w0) + slc_o*sig(w1) + swa_o*sig(w2).
 * pg == NULL: topk is an input.  pg != NULL (from nsa_decode_cmp_split): the block scores are folded from pg and
 * the selection (inference/topk.py:433-493) runs in the kernel's prologue; topk is then an output. */
int nsa_decode_slc_swa_combine(const void* q, int64_t q_st, int64_t q_sh, const void* k_cache, int64_t k_sr,
                               int64_t k_sh, const void* v_cache, int64_t v_sr, int64_t v_sh, const void* w,
                               int64_t w_st, int64_t w_sh, int32_t* topk, int64_t tk_sh, int64_t tk_st,
                               const float* pg, int fixed_y_maxlen, int fixed_num_slc_blocks, int kernel_size,
                               int stride, int num_init, int num_local, int ignore_index, const void* cmp_o,
                               void* slc_o, void* swa_o, int64_t co_st, int64_t co_sh, void* out, int64_t o_st,
                               int64_t o_sh, const int32_t* context_lens, const int32_t* block_tables,
                               int table_stride, int page_size, int B, int QH, int KH, int D, int VD, int block_size,
                               int top_n, int window, float sm_scale, void* stream);

/* The whole decode step in ONE launch (one workgroup per request and kv head):
 * replaces flash_nsa/inference/__init__.py:207-257 (cmp_attn_decode, topk_decode, fused_slc_swa_attn_decode,
 * combine_decode).  out [B,QH,VD] is required; cmp_o / slc_o / swa_o (shared strides co_st, co_sh), lse and topk
 * are optional outputs (NULL to skip).  cmp_slot_mapping [B] (optional): when given, the kernel also pools the
 * compressed K and V row that the newest token completes (flat pool row, -1: none), i.e. it includes
 * nsa_paged_pool_decode (flash_nsa/inference/compress_kv.py:253-287) and the step is a single launch.
 * new_k / new_v [B,KH,D] / [B,KH,VD] + slot_mapping [B] (optional, all three or none): the newest token's K and V
 * rows are first written to flat pool row slot_mapping[b] (-1: skip), i.e. the kernel also includes
 * store_kvcache (nano-vllm/nanovllm/layers/attention.py:123-153).
 * Needs fixed_y_maxlen / fixed_num_slc_blocks / table_stride small enough for
 * 160 KB of LDS (nsa_decode_fused_fits returns 1; e.g. contexts up to 32K tokens at kernel 32 / stride 16);
 * otherwise use nsa_decode_cmp_topk + nsa_decode_slc_swa_combine. */
int nsa_decode_fused_fits(int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks, int table_stride,
                          int page_size);
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
                     float sm_scale, void* stream);
/* the same with scratch memory (16-byte aligned, nothing is kept in it between calls) of
 * nsa_decode_fused_scratch_bytes(...): where that is not 0, large batches run two workgroups per CU instead of one and
 * keep the probabilities that LDS does not hold in the scratch; with 192 q/k channels the scratch is required */
int64_t nsa_decode_fused_scratch_bytes(int B, int KH, int D, int VD, int fixed_y_maxlen, int fixed_num_slc_blocks,
                                       int table_stride, int page_size);
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
                     float sm_scale, void* scratch, int64_t scratch_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif
