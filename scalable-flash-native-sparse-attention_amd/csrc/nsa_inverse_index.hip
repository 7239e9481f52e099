// Inverse of the top-n selection: for every (kv head, selection block) the ascending list of query tokens that
// selected the block, as a CSR (offsets + token ids), plus the prefix of fixed-size list chunks that the dK/dV
// kernel uses as its work items.  Built by a deterministic counting sort: per-token-chunk histograms,
// a scan over chunks and blocks, then an in-order fill, so no sort and no dense (block x token) scratch.
// All three are bound by round trips to memory and LDS, not by bytes, and stand on the critical path in front of the
// selected dK/dV kernel.  us for count + scan + fill, with one search per entry, a scan and a fill that wait for every
// element -> as below: one sequence of 4K tokens, 1 kv head 79 -> 24, 40 of up to 1.2K, 2 kv heads 101 -> 31, 8 x 6K,
// 4 kv heads 149 -> 58, 64K 171 -> 82.  Four threads per token, and sequences found at one look, fill alone: 40 of up to 1.2K
// 14 -> 8, 4K 14 to 29 -> 10, 16K 19 -> 12 (a chunk's workgroup is often alone on its CU: one wave per SIMD before); 64 sequences a look also
// where there are more (two binary searches before): 1000 sequences of 60, 4 kv heads, 61 -> 55, 8 kv heads 84 -> 72.  Reading 32
// chunk counts at a time in the scan takes 109 registers a thread, and the launch then waits for the kernels beside it: 8 x 6K
// 34 -> 217.
// Upstream: flash_nsa/ops/topk.py:782-945 (get_bind_from_find, dense scatter + per-row sort).
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include "../../include/nsa_hip.h"

namespace {

// Tokens per counting chunk: short chunks give the serial in-order fill more parallelism, long ones keep the
// [KH][chunks][blocks] histogram workspace small for very long batches.
__host__ __device__ inline int counting_chunk(int T) { return T <= 131072 ? 256 : 1024; }

__device__ __forceinline__ int find_seq(const int32_t* x_cu, int B, int tok) {
  int lo = 0, hi = B;  // last b with x_cu[b] <= tok
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (x_cu[mid] <= tok) lo = mid; else hi = mid;
  }
  return lo;
}

// The same for a token that is the same in all lanes: 64 sequences, or parts of their list, at a look
__device__ __forceinline__ int find_seq_uniform(const int32_t* x_cu, int B, int tok) {
  const int lane = lane_id();
  int lo = 0;
  for (int n = B; n > 1;) {
    const int step = (n + 63) >> 6, i = lane * step;
    const bool from = x_cu[lo + min(i, n - 1)] <= tok && lane > 0 && i < n;
    const int k = (int)__builtin_popcountll(__builtin_amdgcn_ballot_w64(from));
    lo += k * step;
    n = min(step, n - k * step);
  }
  return lo;
}

// A query token of the sequences b0 .. b1: where its sequence's blocks begin, how many there are and how many slots of its selection
// count.  (One search per token; one per entry was most of the counting kernel.)
struct TokenRow {
  const int32_t* slots;
  int n, kb, nb, nvalid;
};
__device__ __forceinline__ TokenRow token_row(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n,
                                              const int32_t* x_cu, const int32_t* kblk_cu, int b0, int b1, int tok, int t1,
                                              int kh, int block_size, int t_begin) {
  TokenRow r{topk, 0, 0, 0, 0};
  if (tok >= t1) return r;
  const int b = b0 + find_seq(x_cu + b0, b1 - b0 + 1, tok);
  if (tok >= x_cu[b + 1]) return r;  // behind the last sequence
  r.slots = topk + (int64_t)kh * tk_sh + (int64_t)tok * tk_st;
  r.n = tok - x_cu[b];
  r.kb = kblk_cu[b];
  r.nb = kblk_cu[b + 1] - r.kb;
  r.nvalid = r.n >= t_begin ? min(top_n, r.n / block_size + 1) : 0;
  return r;
}
// fn(global block, slot) for the blocks that the token selected, slots ROW part .. ROW part + ROW - 1 of every 16: PARTS threads share
// a token; the ids are fetched ROW at a time, so that they share one round trip to memory
template <int PARTS, class Fn>
__device__ __forceinline__ void for_each_block(const TokenRow& r, int part, Fn fn) {
  constexpr int ROW = 16 / PARTS;
  for (int s0 = part * ROW; s0 < r.nvalid; s0 += 16) {
    int j[ROW];
#pragma unroll
    for (int s = 0; s < ROW; s++) j[s] = s0 + s < r.nvalid ? r.slots[s0 + s] : -1;
#pragma unroll
    for (int s = 0; s < ROW; s++)
      if (j[s] >= 0 && j[s] < r.nb) fn(r.kb + j[s], s0 + s);
  }
}

// grid (nchunks, KH), dynamic LDS nblk ints
template <int PARTS>
__global__ __launch_bounds__(256 * PARTS) void csr_count_kernel(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n,
                                                        const int32_t* x_cu, const int32_t* kblk_cu, int B, int tok0,
                                                        int T, int nblk, int block_size, int t_begin,
                                                        int32_t* chunk_cnt) {
  constexpr int NT = 256 * PARTS;
  extern __shared__ int hist[];
  const int chunk = blockIdx.x, kh = blockIdx.y;
  const int part = threadIdx.x >> 8;
  for (int i = threadIdx.x; i < nblk; i += NT) hist[i] = 0;
  __syncthreads();
  const int CT = counting_chunk(T);
  const int t0 = tok0 + chunk * CT;
  const int t1 = min(tok0 + T, t0 + CT);
  const int b0 = find_seq_uniform(x_cu, B, t0), b1 = find_seq_uniform(x_cu, B, t1 - 1);
  for (int tb = t0; tb < t1; tb += 256) {
    const TokenRow r = token_row(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, b0, b1, tb + (threadIdx.x & 255), t1, kh, block_size,
                                 t_begin);
    for_each_block<PARTS>(r, part, [&](int jb, int) { atomicAdd(&hist[jb], 1); });
  }
  __syncthreads();
  int32_t* dst = chunk_cnt + ((int64_t)kh * gridDim.x + chunk) * nblk;
  for (int i = threadIdx.x; i < nblk; i += NT) dst[i] = hist[i];
}

// grid (KH), 1024 threads: chunk counts -> chunk bases (in place), list offsets, work-item offsets
__global__ __launch_bounds__(1024) void csr_scan_kernel(int32_t* chunk_cnt, int nchunks, int nblk, int64_t list_cap,
                                                        int chunk_tokens, int32_t* csr_off, int32_t* item_off) {
  __shared__ int part_a[1024];
  __shared__ int part_b[1024];
  const int kh = blockIdx.x;
  const int tid = threadIdx.x;
  int32_t* cnt = chunk_cnt + (int64_t)kh * nchunks * nblk;
  const int per = (nblk + 1023) / 1024;
  const int j0 = tid * per, j1 = min(nblk, j0 + per);
  int sum_a = 0, sum_b = 0;
  for (int j = j0; j < j1; j++) {
    // counts are read SCAN at a time: reading and replacing them one by one is a chain of round trips to memory
    constexpr int SCAN = 16;
    int base = 0;
    for (int c0 = 0; c0 < nchunks; c0 += SCAN) {
      int v[SCAN];
#pragma unroll
      for (int u = 0; u < SCAN; u++) v[u] = c0 + u < nchunks ? cnt[(int64_t)(c0 + u) * nblk + j] : 0;
#pragma unroll
      for (int u = 0; u < SCAN; u++) {
        if (c0 + u < nchunks) cnt[(int64_t)(c0 + u) * nblk + j] = base;
        base += v[u];
      }
    }
    // totals are parked in the output arrays and replaced by their prefixes below
    csr_off[(int64_t)kh * (nblk + 1) + j] = base;
    sum_a += base;
    sum_b += (base + chunk_tokens - 1) / chunk_tokens;
  }
  // exclusive scan of the per-thread sums (Hillis-Steele over the 1024 threads)
  part_a[tid] = sum_a;
  part_b[tid] = sum_b;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const int a = tid >= d ? part_a[tid - d] : 0, bb = tid >= d ? part_b[tid - d] : 0;
    __syncthreads();
    part_a[tid] += a;
    part_b[tid] += bb;
    __syncthreads();
  }
  part_a[tid] -= sum_a;
  part_b[tid] -= sum_b;
  int ra = part_a[tid] + (int)((int64_t)kh * list_cap), rb = part_b[tid];
  for (int j = j0; j < j1; j++) {
    int total = csr_off[(int64_t)kh * (nblk + 1) + j];
    csr_off[(int64_t)kh * (nblk + 1) + j] = ra;
    item_off[(int64_t)kh * (nblk + 1) + j] = rb;
    ra += total;
    rb += (total + chunk_tokens - 1) / chunk_tokens;
  }
  if (j0 < j1 && j1 == nblk) {  // the owner of the last block also writes the end markers
    csr_off[(int64_t)kh * (nblk + 1) + nblk] = ra;
    item_off[(int64_t)kh * (nblk + 1) + nblk] = rb;
  }
}

// grid (nchunks, KH): in-order fill.  The position of a token in a block's list is the number of earlier
// tokens that selected the block.  256 tokens at a time set their bit in the block's 256-bit mask, so the count is that
// of the bits below the token's own and no token waits for another (a wave that walked the tokens one by one took as
// long as 256 dependent LDS updates, whatever the size of the batch).  LDS holds the masks of FILL_BLOCKS blocks; more
// blocks than that are taken in several rounds.
constexpr int FILL_BLOCKS = 1024, FILL_WORDS = 256 / 32;
template <int PARTS>
__global__ __launch_bounds__(256 * PARTS) void csr_fill_kernel(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n,
                                                       const int32_t* x_cu, const int32_t* kblk_cu, int B, int tok0,
                                                       int T, int nblk, int block_size, int t_begin,
                                                       const int32_t* chunk_base, const int32_t* csr_off,
                                                       int32_t* csr_tok, uint8_t* csr_slot) {
  constexpr int NT = 256 * PARTS;
  __shared__ int cursor[FILL_BLOCKS];
  __shared__ __attribute__((aligned(16))) uint32_t mask[FILL_BLOCKS * FILL_WORDS];
  const int chunk = blockIdx.x, kh = blockIdx.y;
  const int tid = threadIdx.x, part = tid >> 8, row = tid & 255;
  const int CT = counting_chunk(T);
  const int t0 = tok0 + chunk * CT;
  const int t1 = min(tok0 + T, t0 + CT);
  if (t0 >= t1) return;
  const int32_t* base = chunk_base + ((int64_t)kh * gridDim.x + chunk) * nblk;
  const int32_t* off = csr_off + (int64_t)kh * (nblk + 1);
  // the blocks of this chunk's sequences
  const int b0 = find_seq_uniform(x_cu, B, t0), b1 = find_seq_uniform(x_cu, B, t1 - 1);
  const int blk_lo = kblk_cu[b0];
  const int blk_hi = kblk_cu[b1 + 1];
  const int word = row >> 5;
  const uint32_t bit = 1u << (row & 31);
  for (int r0 = blk_lo; r0 < blk_hi; r0 += FILL_BLOCKS) {
    const int nr = min(FILL_BLOCKS, blk_hi - r0);
    for (int i = tid; i < nr; i += NT) cursor[i] = base[r0 + i] + off[r0 + i];
    for (int tb = t0; tb < t1; tb += 256) {
      for (int i = tid; i < nr * FILL_WORDS; i += NT) mask[i] = 0;
      __syncthreads();
      const TokenRow r = token_row(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, b0, b1, tb + row, t1, kh, block_size,
                                   t_begin);
      for_each_block<PARTS>(r, part, [&](int jb, int) {
        if ((unsigned)(jb - r0) < (unsigned)nr) atomicOr(&mask[(jb - r0) * FILL_WORDS + word], bit);
      });
      __syncthreads();
      for_each_block<PARTS>(r, part, [&](int jb, int slot) {
        if ((unsigned)(jb - r0) >= (unsigned)nr) return;
        const uint32_t* m = &mask[(jb - r0) * FILL_WORDS];
        int pos = cursor[jb - r0];
#pragma unroll
        for (int w = 0; w < FILL_WORDS; w++) pos += __popc(w < word ? m[w] : w == word ? m[w] & (bit - 1) : 0u);
        csr_tok[pos] = r.n;
        if (csr_slot != nullptr) csr_slot[pos] = (uint8_t)slot;
      });
      __syncthreads();
      if (tb + 256 < t1) {
        for (int i = tid; i < nr; i += NT) {
          int add = 0;
#pragma unroll
          for (int w = 0; w < FILL_WORDS; w++) add += __popc(mask[i * FILL_WORDS + w]);
          cursor[i] += add;
        }
        __syncthreads();
      }
    }
  }
}

}  // namespace

extern "C" {

int64_t nsa_inverse_index_workspace_elems(int T, int KH, int nblk_total) {
  const int CT = counting_chunk(T);
  int64_t nchunks = (T + CT - 1) / CT;
  return (int64_t)KH * nchunks * nblk_total;
}

int nsa_build_inverse_index(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                            const int32_t* kblk_cu, int B, int T, int KH, int nblk_total, int block_size,
                            int chunk_tokens, int32_t* csr_off, int32_t* csr_tok, int32_t* item_off,
                            int32_t* workspace, int64_t workspace_elems, void* stream) {
  return nsa_build_inverse_index_from(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, B, T, KH, nblk_total, block_size,
                                      chunk_tokens, 0, csr_off, csr_tok, item_off, workspace, workspace_elems, stream);
}

int nsa_build_inverse_index_from(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                                 const int32_t* kblk_cu, int B, int T, int KH, int nblk_total, int block_size,
                                 int chunk_tokens, int t_begin, int32_t* csr_off, int32_t* csr_tok, int32_t* item_off,
                                 int32_t* workspace, int64_t workspace_elems, void* stream) {
  return nsa_build_inverse_index_slots(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, B, 0, T, KH, nblk_total, block_size,
                                       chunk_tokens, t_begin, csr_off, csr_tok, nullptr, item_off, workspace,
                                       workspace_elems, stream);
}

int nsa_build_inverse_index_slots(const int32_t* topk, int64_t tk_sh, int64_t tk_st, int top_n, const int32_t* x_cu,
                                  const int32_t* kblk_cu, int B, int tok0, int T, int KH, int nblk_total,
                                  int block_size, int chunk_tokens, int t_begin, int32_t* csr_off, int32_t* csr_tok,
                                  uint8_t* csr_slot, int32_t* item_off, int32_t* workspace, int64_t workspace_elems,
                                  void* stream) {
  if (T <= 0 || B <= 0 || nblk_total <= 0) return NSA_OK;
  NSA_REQUIRE(top_n >= 1 && top_n <= 64, NSA_ERR_BAD_ARG, "build_inverse_index: top_n %d must be in [1,64]", top_n);
  NSA_REQUIRE(chunk_tokens >= 1, NSA_ERR_BAD_ARG, "build_inverse_index: chunk_tokens must be positive");
  NSA_REQUIRE(nblk_total * 4 <= 64 * 1024, NSA_ERR_UNSUPPORTED,
              "build_inverse_index: %d selection blocks exceed the LDS histogram (16384)", nblk_total);
  NSA_REQUIRE((int64_t)KH * T * top_n < 0x7fffffffLL, NSA_ERR_UNSUPPORTED,
              "build_inverse_index: KH*T*top_n exceeds int32 positions");
  NSA_REQUIRE(workspace_elems >= nsa_inverse_index_workspace_elems(T, KH, nblk_total), NSA_ERR_WORKSPACE,
              "build_inverse_index: workspace of %lld ints is too small", (long long)workspace_elems);
  hipStream_t s = (hipStream_t)stream;
  const int CT = counting_chunk(T);
  int nchunks = (T + CT - 1) / CT;
  size_t lds = (size_t)nblk_total * sizeof(int);
  dim3 grid(nchunks, KH);
  // Four threads per token: workgroups of 1024, of which a CU holds two, so more than that pay only where a token has many slots to look at
  // (blocks per sequence on average; 16 slots are one thread's read).  One thread / four, us, count + scan + fill, by workgroups: 16K tokens
  // of 1 kv head (64) 27 / 22, 40 x 1200 of 2 (376) 43 / 39, 64K of 2 (512) 61 / 56, 200 x 300 of 2 (470) 45.3 / 45.7; of 4: 8 x 6K, top_n 16
  // (752) 56.2 / 55.8, 8 37 / 42, 32 147 / 138, 64 153 / 145, 200 x 300 (940) 51 / 57, 40 x 3000 (1876) 278 / 279, top_n 32 847 / 828; of 8: 200
  // x 300 (1880) 60 / 75.  (64K of 1, top_n 64, 256 workgroups: 91 / 97.)
  const int seq_blocks = nblk_total / B;
  const bool few = (int64_t)nchunks * KH <= 2 * nsa_device_cus() || (top_n < seq_blocks ? top_n : seq_blocks) > 16;
  auto count = [&](auto kernel, int threads) {
    kernel<<<grid, threads, lds, s>>>(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, B, tok0, T, nblk_total, block_size, t_begin, workspace);
  };
  if (few) count(csr_count_kernel<4>, 1024);
  else count(csr_count_kernel<1>, 256);
  int rc = nsa_check_launch("csr_count_kernel");
  if (rc) return rc;
  csr_scan_kernel<<<KH, 1024, 0, s>>>(workspace, nchunks, nblk_total, (int64_t)T * top_n, chunk_tokens, csr_off,
                                      item_off);
  rc = nsa_check_launch("csr_scan_kernel");
  if (rc) return rc;
  auto fill = [&](auto kernel, int threads) {
    kernel<<<grid, threads, 0, s>>>(topk, tk_sh, tk_st, top_n, x_cu, kblk_cu, B, tok0, T, nblk_total, block_size, t_begin, workspace, csr_off,
                                    csr_tok, csr_slot);
  };
  if (few) fill(csr_fill_kernel<4>, 1024);
  else fill(csr_fill_kernel<1>, 256);
  return nsa_check_launch("csr_fill_kernel");
}

}  // extern "C"
