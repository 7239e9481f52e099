// Selected-block attention forward: one wave per (query token, kv head); the MFMA M dimension is the group of
// (up to 16) q-heads that share the kv head, N is 16 keys, v_mfma_f32_16x16x32_bf16.
// Upstream: flash_nsa/ops/select_attn.py:21-108 (training), flash_nsa/inference/select_attn.py:21-100 (paged).
//
// The keys of the selected blocks are processed in units of 32.  The K and V rows of a unit are fetched as whole
// coalesced rows (16 lanes x 16 bytes per row) into registers one unit ahead, pass through a wave-private LDS
// region, and are read back as MFMA fragments (K row-major, V through ds_read_b64_tr_b16, which delivers the
// key-contraction slices).  Keys are gathered by the per-token block list topk[kh, t, 0 .. min(top_n, t/block+1)).
//
// What bounds it is the gather: 512 KB of rows per token and kv head, from L2 while the keys of the sequences in flight
// fit there, else from the memory-side cache (13.5 TB/s of requests at 64K tokens).  Two units in flight per wave and
// separate K and V regions bought nothing over one, and took the registers and the LDS of a second workgroup per CU at
// 192 channels: 32 heads, 16K tokens 1726 -> 1080 us; 64 heads of 128, 8 x 6K tokens 4207 -> 3920 us.
#include "nsa_common.h"
#include "nsa_api_internal.h"

namespace {

// waves per SIMD the register budget is cut for; at 256 channels two waves with 30 spilled registers beat one without
// (1039 against 1165 us for 16 heads, 16K tokens)
constexpr int slc_waves(int d) { return d <= 64 ? 4 : d <= 128 ? 3 : 2; }

template <int D, int VD, bool PAGED>
__global__ __launch_bounds__(256, slc_waves(D)) void slc_fwd_kernel(NsaSlcParams p) {
  // Work unit = 32 keys (half of a 64-key tile).  One set of registers holds the rows of the next unit: its K rows are
  // requested when this unit's have gone to LDS, its V rows when this unit's have, which is when the scores are known
  // and the K rows in LDS are no longer needed: K and V take turns in one LDS region.
  constexpr int UK = 32;                      // keys per unit
  constexpr int KC = D / 32;                  // K fragments per 16-key tile
  constexpr int VJ = (UK * (VD / 8)) / 64;    // 16-byte V loads per lane and unit
  constexpr int KJ = (UK * (D / 8)) / 64;     // 16-byte K loads per lane and unit
  constexpr int KLD = D + NSA_LDS_PAD, VLD = VD + NSA_LDS_PAD;
  constexpr int LD = KLD > VLD ? KLD : VLD;
  constexpr int KP = D / 8, VP = VD / 8;                                             // 16-byte pieces per row
  constexpr int KPAT = 64 % KP == 0 ? 1 : 3, VPAT = 64 % VP == 0 ? 1 : 3;            // 192 channels: 3 * 64 = 8 * 24
  static_assert((KPAT * 64) % KP == 0 && (VPAT * 64) % VP == 0, "");
  __shared__ __attribute__((aligned(16))) bf16_t rows_all[4 * UK * LD];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  bf16_t* const rows = rows_all + wave * UK * LD;
  const int l16 = lane & 15;
  const int kq = lane >> 4;
  const int b = blockIdx.y;
  const int n_hc = (p.G + 15) / 16;
  const int kh = blockIdx.z / n_hc;
  const int hc = blockIdx.z - kh * n_hc;

  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  const int ctx = PAGED ? p.ctx_lens[b] : xl;
  const int n = (p.t_begin > 0 ? max(p.t_begin - (ctx - xl), 0) : 0) + blockIdx.x * 4 + wave;
  if (n >= xl) return;
  const int t = n + (ctx - xl);
  const int64_t tok = x0 + n;
  const int32_t* table = PAGED ? p.table + (int64_t)b * p.table_stride : nullptr;
  const int Bs = p.block_size;
  const int nvalid = t >= 0 ? min(p.top_n, t / Bs + 1) : 0;  // t < 0: padded request, output row = 0
  const int upb = Bs / UK;                    // units per selection block
  const int nu = nvalid * upb;
  const int key_last = min(ctx - 1, t);       // last key this token may attend

  int g = hc * 16 + l16;
  const bool head_ok = g < p.G;
  if (!head_ok) g = p.G - 1;
  const int head = kh * p.G + g;

  bf16x8 qf[KC];
  {
    const bf16_t* qp = p.q + tok * p.q_st + (int64_t)head * p.q_sh + kq * 8;
#pragma unroll
    for (int kc = 0; kc < KC; kc++) qf[kc] = ld_global_b128(qp + kc * 32);
  }
  int my_blk = 0;
  if (lane < nvalid) my_blk = p.topk[(int64_t)kh * p.tk_sh + tok * p.tk_st + lane];
  my_blk = sort_blocks(my_blk, nvalid, lane);

  f32x4 oacc[VD / 16];
#pragma unroll
  for (int dt = 0; dt < VD / 16; dt++) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = NSA_NEG_INF, l_run = 0.f;
  const float sc = p.scale_log2;

  // first key of the next unit with something to attend, at or behind unit u, -1: none left; wave-uniform.  Units that
  // start past the last attendable key (second half of the current block) and ignore values (negative ids) are skipped.
  auto next_unit = [&](int& u) {
    for (; u < nu; u++) {
      const int slot = u / upb;
      const int blk = __builtin_amdgcn_readlane(my_blk, slot);
      const int key0 = blk * Bs + (u - slot * upb) * UK;
      if (blk >= 0 && key0 <= key_last) {
        u++;
        return key0;
      }
    }
    return -1;
  };
  // K and V rows are fetched as whole 16-byte-per-lane coalesced rows (every cache line is requested once and used
  // completely) and go through wave-private LDS; the MFMA fragments are read from there.
  // A unit's rows are fetched 64 pieces of 16 bytes at a time; after KPAT (VPAT) instructions the pieces fall on the same
  // columns again, so the lane part of the addresses is KPAT + VPAT 32-bit offsets and the rest is wave-uniform.
  uint32_t koff[KPAT], voff[VPAT];
#pragma unroll
  for (int j = 0; j < KPAT; j++) {
    int pc = lane + j * 64;
    koff[j] = (uint32_t)(pc / KP) * (uint32_t)(p.k_sr * 2) + (pc % KP) * 16;
  }
#pragma unroll
  for (int j = 0; j < VPAT; j++) {
    int pc = lane + j * 64;
    voff[j] = (uint32_t)(pc / VP) * (uint32_t)(p.v_sr * 2) + (pc % VP) * 16;
  }
  bf16x8 kr[KJ], vr[VJ];
  auto flat_row = [&](int key0) -> int64_t {  // flat row of the unit's first key (a unit never straddles a page)
    if (PAGED) return (int64_t)__builtin_amdgcn_readfirstlane(table[key0 / p.page_size]) * p.page_size + (key0 % p.page_size);
    return (int64_t)x0 + key0;
  };
  // the unit holding the causal boundary: rows past it are replaced by the boundary row (masked later)
  auto issue_k = [&](int key0) {
    const bf16_t* kb = p.k + flat_row(key0) * p.k_sr + (int64_t)kh * p.k_sh;
    const int kmax = key_last - key0;  // >= 0
    if (kmax >= UK - 1) {
#pragma unroll
      for (int j = 0; j < KJ; j++)
        kr[j] = ld_global_b128((const bf16_t*)((const char*)(kb + (j / KPAT) * (KPAT * 64 / KP) * p.k_sr) + koff[j % KPAT]));
    } else {
#pragma unroll
      for (int j = 0; j < KJ; j++) {
        int pc = lane + j * 64;
        kr[j] = ld_global_b128(kb + (int64_t)min(pc / KP, kmax) * p.k_sr + (pc % KP) * 8);
      }
    }
  };
  auto issue_v = [&](int key0) {
    const bf16_t* vb = p.v + flat_row(key0) * p.v_sr + (int64_t)kh * p.v_sh;
    const int kmax = key_last - key0;  // >= 0
    if (kmax >= UK - 1) {
#pragma unroll
      for (int j = 0; j < VJ; j++)
        vr[j] = ld_global_b128((const bf16_t*)((const char*)(vb + (j / VPAT) * (VPAT * 64 / VP) * p.v_sr) + voff[j % VPAT]));
    } else {
#pragma unroll
      for (int j = 0; j < VJ; j++) {
        int pc = lane + j * 64;
        vr[j] = ld_global_b128(vb + (int64_t)min(pc / VP, kmax) * p.v_sr + (pc % VP) * 8);
      }
    }
  };
  auto lds_order = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  int u = 0;
  int key0 = next_unit(u);
  if (key0 >= 0) { issue_k(key0); issue_v(key0); }
  while (key0 >= 0) {
    const int key_next = next_unit(u);
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&rows[(pc / KP) * KLD + (pc % KP) * 8]) = kr[j];
    }
    lds_order();
    if (key_next >= 0) issue_k(key_next);
    f32x4 sacc[2];
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      sacc[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* kp = &rows[(jt * 16 + l16) * KLD + kq * 8];
#pragma unroll
      for (int kc = 0; kc < KC; kc++) sacc[jt] = mfma16(*reinterpret_cast<const bf16x8*>(kp + kc * 32), qf[kc], sacc[jt]);
    }
    const int kmax = key_last - key0;  // last usable key offset inside this unit
    if (kmax < UK - 1) {               // wave-uniform: only the unit holding the causal boundary is masked
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          int ko = jt * 16 + kq * 4 + i;
          if (ko > kmax) sacc[jt][i] = NSA_NEG_INF;
        }
    }
    float tmax = fmaxf(fmaxf(fmaxf(sacc[0][0], sacc[0][1]), fmaxf(sacc[0][2], sacc[0][3])),
                       fmaxf(fmaxf(sacc[1][0], sacc[1][1]), fmaxf(sacc[1][2], sacc[1][3])));
    tmax = xrow_max(tmax);
    tmax = xhalf_max(tmax);
    const float m_old = m_run;
    const float m_new = fmaxf(m_old, tmax);
    const float m_safe = (m_new == NSA_NEG_INF) ? 0.f : m_new;
    const float msc = m_safe * sc;
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float pv = fast_exp2(__builtin_fmaf(sacc[jt][i], sc, -msc));
        sacc[jt][i] = pv;
        psum += pv;
      }
    if (__builtin_amdgcn_ballot_w64(m_new != m_old) != 0) {
      const float alpha = fast_exp2((m_old - m_safe) * sc);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < VD / 16; dt++) oacc[dt] *= alpha;
    }
    l_run += psum;
    lds_order();
#pragma unroll
    for (int j = 0; j < VJ; j++) {
      int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&rows[(pc / VP) * VLD + (pc % VP) * 8]) = vr[j];
    }
    lds_order();
    if (key_next >= 0) issue_v(key_next);
    // O^T += V^T P^T over the 32 keys of the unit
    bf16x8 pf = pack8(sacc[0][0], sacc[0][1], sacc[0][2], sacc[0][3], sacc[1][0], sacc[1][1], sacc[1][2], sacc[1][3]);
    const int kb0 = kq * 4 + (l16 >> 2);
    const int kb1 = kb0 + 16;
#pragma unroll
    for (int dt = 0; dt < VD / 16; dt++) {
      const int col = dt * 16 + 4 * (l16 & 3);
      bf16x4 v0 = lds_read_tr(&rows[kb0 * VLD + col]);
      bf16x4 v1 = lds_read_tr(&rows[kb1 * VLD + col]);
      oacc[dt] = mfma16(cat4(v0, v1), pf, oacc[dt]);
    }
    lds_order();
    key0 = key_next;
  }

  float l_tot = xrow_sum(l_run);
  l_tot = xhalf_sum(l_tot);
  if (!head_ok) return;
  float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  bf16_t* op = p.o + tok * p.o_st + (int64_t)head * p.o_sh + kq * 4;
#pragma unroll
  for (int dt = 0; dt < VD / 16; dt++) {
    bf16x4 w = pack4(oacc[dt][0] * inv, oacc[dt][1] * inv, oacc[dt][2] * inv, oacc[dt][3] * inv);
    *reinterpret_cast<bf16x4*>(op + dt * 16) = w;
  }
  if (kq == 0 && p.lse != nullptr) {
    p.lse[tok * p.lse_st + (int64_t)head * p.lse_sh] = l_tot > 0.f ? m_run * sc + fast_log2(l_tot) : 0.f;
  }
}

template <int D, int VD, bool PAGED>
int launch_slc(const NsaSlcParams& p, int B, int max_q_len, hipStream_t stream) {
  if (!PAGED) max_q_len -= p.t_begin;
  if (B <= 0 || max_q_len <= 0) return NSA_OK;
  dim3 grid(cdiv_i(max_q_len, 4), B, p.KH * ((p.G + 15) / 16));
  slc_fwd_kernel<D, VD, PAGED><<<grid, 256, 0, stream>>>(p);
  return nsa_check_launch("slc_fwd_kernel");
}

template <bool PAGED>
int dispatch_slc(const NsaSlcParams& p, int B, int max_q_len, int D, int VD, hipStream_t stream) {
  if (D == 128 && VD == 128) return launch_slc<128, 128, PAGED>(p, B, max_q_len, stream);
  if (D == 64 && VD == 64) return launch_slc<64, 64, PAGED>(p, B, max_q_len, stream);
  if (D == 192 && VD == 128) return launch_slc<192, 128, PAGED>(p, B, max_q_len, stream);
  if (D == 256 && VD == 256) return launch_slc<256, 256, PAGED>(p, B, max_q_len, stream);
  if (D == 32 && VD == 32) return launch_slc<32, 32, PAGED>(p, B, max_q_len, stream);
  nsa_set_error("selected attention forward: unsupported head dims D=%d VD=%d", D, VD);
  return NSA_ERR_UNSUPPORTED;
}

}  // namespace

int nsa_slc_fwd_launch(const NsaSlcParams& p, bool paged, int B, int max_q_len, int D, int VD, hipStream_t stream) {
  return paged ? dispatch_slc<true>(p, B, max_q_len, D, VD, stream)
               : dispatch_slc<false>(p, B, max_q_len, D, VD, stream);
}
