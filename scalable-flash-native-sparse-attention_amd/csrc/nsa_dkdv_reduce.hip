// Deterministic dK / dV: the dk/dv kernels store every workgroup's fp32 partial result in its own slot instead of
// adding it with atomics, and the kernels here sum the slots of a key in a fixed (ascending work-item) order.
// Upstream's counterpart is dkdv_repeat=True: per-q-head buffers followed by a sum over the heads
// (flash_nsa/ops/compress_attn.py:594-598,691-693, flash_nsa/ops/select_attn.py:528-531,639-641); here the q-heads of
// a group are already summed inside the MFMA accumulators, and what is left to order are the query chunks.
#include "nsa_common.h"
#include "nsa_api_internal.h"

namespace {

// compressed branch: grid (key tiles x pieces of 256 sums, B, KH), one thread per four channels of a key.  The work
// items of a key tile are consecutive in the dk/dv kernel's grid.x (key-tile major), one per query chunk that sees the
// tile.  The sum is a chain of loads from slots that lie KH * KW rows apart: eight are in flight at once, and a tile is
// spread over many workgroups, since short batches have few tiles and many chunks (one sequence of 4096 tokens, 16 q /
// 1 kv heads, 64 chunks: 650 us with a workgroup per tile, 5 us so).
template <int KW>
__global__ __launch_bounds__(256) void cmp_dkdv_reduce_kernel(NsaBwdTileParams p, int D, int VD, int grid_x_items,
                                                              int pieces, bool add) {
  const int ktile = blockIdx.x / pieces, b = blockIdx.y, kh = blockIdx.z;
  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  const int kbase = p.k_cu[b];
  const int nkeys = p.k_cu[b + 1] - kbase;
  const int key0 = ktile * KW;
  const int n4k = D / 4, n4v = VD / 4;
  const int per_key = n4k + n4v;
  const int e = (blockIdx.x - ktile * pieces) * 256 + threadIdx.x;
  const int kl = e / per_key, c4 = e - kl * per_key;
  if (kl >= min(KW, nkeys - key0)) return;
  // the enumeration of bwd_dkdv_kernel MODE_CMP
  int lo, hi;
  nsa_local_range(p.tok0, p.tok1, x0, xl, lo, hi);
  const int nch = cdiv_i(max(hi - lo, 0), p.q_chunk_tokens);
  int start = 0;
  for (int kt = 0; kt < ktile; kt++)
    start += nch - min(nch, max(p.stride * kt * KW + p.kernel_size - 1 - lo, 0) / p.q_chunk_tokens);
  // chunk fc holds the tile's first visible row, if the launch's share of the sequence holds one
  const int seen = p.stride * key0 + p.kernel_size - 1;
  const int fc = seen < hi ? max(seen - lo, 0) / p.q_chunk_tokens : nch;
  if (add && fc >= nch) return;
  const bool is_v = c4 >= n4k;
  const int d = (is_v ? c4 - n4k : c4) * 4;
  const int W = is_v ? VD : D;
  const int64_t slot0 = ((int64_t)b * grid_x_items + start) * p.KH + kh;
  const float* src = (is_v ? p.part_dv : p.part_dk) + (slot0 * KW + kl) * W + d;
  const int64_t step = (int64_t)p.KH * KW * W;
  const int n = nch - fc;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int ch = 0;
  for (; ch + 8 <= n; ch += 8) {
    f32x4 x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = *reinterpret_cast<const f32x4*>(src + (ch + u) * step);
#pragma unroll
    for (int u = 0; u < 8; u++) acc += x[u];
  }
  for (; ch < n; ch++) acc += *reinterpret_cast<const f32x4*>(src + ch * step);
  float* dst = is_v ? (float*)p.dv + ((int64_t)kbase + key0 + kl) * p.dv_sr + (int64_t)kh * p.dv_sh + d
                    : (float*)p.dk + ((int64_t)kbase + key0 + kl) * p.dk_sr + (int64_t)kh * p.dk_sh + d;
  if (add) acc += *reinterpret_cast<const f32x4*>(dst);
  *reinterpret_cast<f32x4*>(dst) = acc;
}

// window branch: grid (key tiles x pieces of 256 sums, B, KH), one thread per four channels of a key, all (at most 16)
// chunks of the tile's queries in flight at once.  Chunks behind the tile's last query have written nothing.
template <bool F32>
__global__ __launch_bounds__(256) void swa_dkdv_reduce_kernel(NsaBwdTileParams p, int KW, int D, int VD, int pieces) {
  const int ktile = blockIdx.x / pieces, b = blockIdx.y, kh = blockIdx.z;
  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  int lo, hi;
  nsa_local_range(p.tok0, p.tok1, x0, xl, lo, hi);
  const int key0 = lo + ktile * KW;
  const int n4k = D / 4, n4v = VD / 4;
  const int per_key = n4k + n4v;
  const int e = (blockIdx.x - ktile * pieces) * 256 + threadIdx.x;
  const int kl = e / per_key, c4 = e - kl * per_key;
  if (kl >= min(KW, hi - key0)) return;
  const int rows = min(xl - key0, KW + p.window);
  const int n = min(p.grid_chunks, cdiv_i(rows, p.q_chunk_tokens));
  const bool is_v = c4 >= n4k;
  const int d = (is_v ? c4 - n4k : c4) * 4;
  const int W = is_v ? VD : D;
  const int64_t slot0 = ((int64_t)b * (gridDim.x / pieces) + ktile) * p.grid_chunks * p.KH + kh;
  const float* src = (is_v ? p.part_dv : p.part_dk) + (slot0 * KW + kl) * W + d;
  const int64_t step = (int64_t)p.KH * KW * W;
  constexpr int MAX = 16;
  f32x4 x[MAX], acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < MAX; u++)
    if (u < n) x[u] = *reinterpret_cast<const f32x4*>(src + u * step);
#pragma unroll
  for (int u = 0; u < MAX; u++)
    if (u < n) acc += x[u];
  const int64_t at = is_v ? ((int64_t)x0 + key0 + kl) * p.dv_sr + (int64_t)kh * p.dv_sh + d
                          : ((int64_t)x0 + key0 + kl) * p.dk_sr + (int64_t)kh * p.dk_sh + d;
  void* const dst = is_v ? p.dv : p.dk;
  if (F32) *reinterpret_cast<f32x4*>((float*)dst + at) = acc;
  else *reinterpret_cast<bf16x4*>((bf16_t*)dst + at) = pack4(acc[0], acc[1], acc[2], acc[3]);
}

// selected branch: grid (selection blocks, sub-blocks, KH).  The work items of a block are the chunks of its token
// list, consecutive in the dk/dv kernel's grid.x; their sum is added to what dk / dv already hold (the window
// branch's result), one thread per element.
template <int KW>
__global__ __launch_bounds__(256) void slc_dkdv_reduce_kernel(NsaBwdTileParams p, int D, int VD, int grid_x_items,
                                                              int grid_y) {
  const int jb = blockIdx.x, sy = blockIdx.y, kh = blockIdx.z;
  const int32_t* ioff = p.item_off + (int64_t)kh * (p.nblk_total + 1);
  const int w0 = ioff[jb], w1 = ioff[jb + 1];
  if (w0 >= w1) return;
  const int b = p.blk_seq[jb];
  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  const int key0 = (jb - p.kblk_cu[b]) * p.block_size + sy * KW;
  const int nkeys = min(xl, (key0 / p.block_size + 1) * p.block_size);
  if (key0 >= nkeys) return;
  const int n4k = D / 4, n4v = VD / 4;
  const int per_key = n4k + n4v;
  const int nk_here = min(KW, nkeys - key0);
  for (int e = threadIdx.x; e < nk_here * per_key; e += 256) {
    const int kl = e / per_key, c4 = e - kl * per_key;
    const bool is_v = c4 >= n4k;
    const int d = (is_v ? c4 - n4k : c4) * 4;
    const int W = is_v ? VD : D;
    const float* part = is_v ? p.part_dv : p.part_dk;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int w = w0; w < w1; w++) {
      const int64_t slot = ((int64_t)kh * grid_x_items + w) * grid_y + sy;
      const f32x4 x = *reinterpret_cast<const f32x4*>(part + (slot * KW + kl) * W + d);
      acc[0] += x[0]; acc[1] += x[1]; acc[2] += x[2]; acc[3] += x[3];
    }
    float* dst = is_v ? (float*)p.dv + ((int64_t)x0 + key0 + kl) * p.dv_sr + (int64_t)kh * p.dv_sh + d
                      : (float*)p.dk + ((int64_t)x0 + key0 + kl) * p.dk_sr + (int64_t)kh * p.dk_sh + d;
    f32x4 cur = *reinterpret_cast<f32x4*>(dst);
    cur[0] += acc[0]; cur[1] += acc[1]; cur[2] += acc[2]; cur[3] += acc[3];
    *reinterpret_cast<f32x4*>(dst) = cur;
  }
}

}  // namespace

int nsa_dkdv_reduce_cmp_launch(const NsaBwdTileParams& p, bool add, int B, int max_q_len, int max_k_len, int D, int VD,
                               hipStream_t stream) {
  if (B <= 0 || max_k_len <= 0) return NSA_OK;
  const int KW = nsa_bwd_dkdv_slot_keys(0, 0, D);
  const int grid_x_items = (int)nsa_bwd_dkdv_cmp_slots(1, 1, max_q_len, max_k_len, D, p.q_chunk_tokens, p.kernel_size,
                                                       p.stride, p.tok0, p.tok1, B);
  if (grid_x_items <= 0 && add) return NSA_OK;
  const int pieces = cdiv_i(KW * (D + VD) / 4, 256);
  dim3 grid(cdiv_i(max_k_len, KW) * pieces, B, p.KH);
  if (KW == 128) cmp_dkdv_reduce_kernel<128><<<grid, 256, 0, stream>>>(p, D, VD, grid_x_items, pieces, add);
  else cmp_dkdv_reduce_kernel<256><<<grid, 256, 0, stream>>>(p, D, VD, grid_x_items, pieces, add);
  return nsa_check_launch("cmp_dkdv_reduce_kernel");
}

int nsa_dkdv_reduce_swa_launch(const NsaBwdTileParams& p0, bool to_f32, int B, int x_maxlen, int D, int VD,
                               hipStream_t stream) {
  if (B <= 0 || x_maxlen <= 0) return NSA_OK;
  NsaBwdTileParams p = p0;
  const int KW = nsa_bwd_dkdv_slot_keys(1, 0, D);
  // as the dk/dv launch cuts them
  p.window = min(p.window, x_maxlen);
  p.q_chunk_tokens = nsa_swa_dkdv_q_chunk(p, KW);
  const int pieces = cdiv_i(KW * (D + VD) / 4, 256);
  const int len = p.tok1 > 0 ? min(x_maxlen, p.tok1 - p.tok0 + 127) : x_maxlen;
  dim3 grid(cdiv_i(len, KW) * pieces, B, p.KH);
  if (to_f32) swa_dkdv_reduce_kernel<true><<<grid, 256, 0, stream>>>(p, KW, D, VD, pieces);
  else swa_dkdv_reduce_kernel<false><<<grid, 256, 0, stream>>>(p, KW, D, VD, pieces);
  return nsa_check_launch("swa_dkdv_reduce_kernel");
}

int nsa_dkdv_reduce_slc_launch(const NsaBwdTileParams& p, int n_items_bound, int D, int VD, hipStream_t stream) {
  if (n_items_bound <= 0 || p.nblk_total <= 0) return NSA_OK;
  const int KW = nsa_bwd_dkdv_slot_keys(2, p.block_size, D);
  const int grid_y = p.block_size <= 64 ? 1 : cdiv_i(p.block_size, 128);
  dim3 grid(p.nblk_total, grid_y, p.KH);
  if (KW == 64) slc_dkdv_reduce_kernel<64><<<grid, 256, 0, stream>>>(p, D, VD, n_items_bound, grid_y);
  else slc_dkdv_reduce_kernel<128><<<grid, 256, 0, stream>>>(p, D, VD, n_items_bound, grid_y);
  return nsa_check_launch("slc_dkdv_reduce_kernel");
}
