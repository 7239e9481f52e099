// dQ of selected-block attention: one wave per (query token, kv head), 16 q-heads as the MFMA N dimension.
//   S^T = K Q^T,  P^T = exp2(S^T*c - lse),  dP^T = V dO^T,  dS^T = P^T o (dP^T - delta),  dQ^T += K^T dS^T
// K and V rows are fetched coalesced and pass through a wave-private LDS region in turn: V for dP, then K, which is read
// both as row fragments and, transposed, through ds_read_b64_tr_b16.  V fragments straight from memory (16 rows x 64
// bytes per load) cost the CU's vector memory pipeline four times the cycles of whole rows, and two units in flight per
// wave the registers of other waves: 64 heads of 128, 8 x 6K tokens 7.07 -> 4.92 ms, 64K tokens 11.6 -> 10.5 ms;
// 32 heads of 192 / 128, 16K tokens 5.68 -> 1.29 ms (142 registers had been spilled).
// Upstream: flash_nsa/ops/select_attn.py:336-437 (_dq_kernel).
#include "nsa_common.h"
#include "nsa_api_internal.h"

namespace {

// waves per SIMD the register budget is cut for: three at 128 channels spill 15 registers (11.8 against 10.5 ms for 64
// heads, 64K tokens), two at 256 channels 104 (2.19 against 1.42 ms for 16 heads, 16K tokens)
constexpr int slc_dq_waves(int d) { return d <= 64 ? 4 : d <= 192 ? 2 : 1; }

template <int D, int VD>
__global__ __launch_bounds__(256, slc_dq_waves(D)) void slc_dq_kernel(NsaSlcBwdDqParams p) {
  // Work unit = 32 keys.  One set of registers holds the rows of the next unit, requested when this unit's have gone to
  // the wave-private LDS region that the V rows (for dP) and the K rows (for S and dQ) share in turn.
  constexpr int UK = 32;
  constexpr int KLD = D + NSA_LDS_PAD, VLD = VD + NSA_LDS_PAD;
  constexpr int LD = KLD > VLD ? KLD : VLD;
  constexpr int KC = D / 32, VC = VD / 32;
  constexpr int KJ = (UK * (D / 8)) / 64, VJ = (UK * (VD / 8)) / 64;
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
  const int n = p.t_begin + blockIdx.x * 4 + wave;
  if (n >= xl) return;
  const int t = n;
  const int64_t tok = x0 + n;
  const int Bs = p.block_size;
  const int nvalid = min(p.top_n, t / Bs + 1);
  const int upb = Bs / UK;
  const int nu = nvalid * upb;
  const int key_last = min(xl - 1, t);

  int g = hc * 16 + l16;
  const bool head_ok = g < p.G;
  if (!head_ok) g = p.G - 1;
  const int head = kh * p.G + g;

  bf16x8 qf[KC], dof[VC];
  {
    const bf16_t* qp = p.q + tok * p.q_st + (int64_t)head * p.q_sh + kq * 8;
#pragma unroll
    for (int kc = 0; kc < KC; kc++) qf[kc] = ld_global_b128(qp + kc * 32);
    const bf16_t* dp = p.dO + tok * p.do_st + (int64_t)head * p.do_sh + kq * 8;
#pragma unroll
    for (int kc = 0; kc < VC; kc++) dof[kc] = ld_global_b128(dp + kc * 32);
  }
  const float lse = p.lse[tok * p.lse_st + (int64_t)head * p.lse_sh];
  const float delta = p.delta[tok * p.delta_st + (int64_t)head * p.delta_sh];
  int my_blk = 0;
  if (lane < nvalid) my_blk = p.topk[(int64_t)kh * p.tk_sh + tok * p.tk_st + lane];
  my_blk = sort_blocks(my_blk, nvalid, lane);

  f32x4 dqacc[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; dt++) dqacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
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
  // the unit holding the causal boundary: rows past it are replaced by the boundary row (masked later)
  auto issue_k = [&](int key0) {
    const bf16_t* kb = p.k + ((int64_t)x0 + key0) * p.k_sr + (int64_t)kh * p.k_sh;
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
    const bf16_t* vb = p.v + ((int64_t)x0 + key0) * p.v_sr + (int64_t)kh * p.v_sh;
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
  if (key0 >= 0) { issue_v(key0); issue_k(key0); }
  while (key0 >= 0) {
    const int key_next = next_unit(u);
#pragma unroll
    for (int j = 0; j < VJ; j++) {
      int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&rows[(pc / VP) * VLD + (pc % VP) * 8]) = vr[j];
    }
    lds_order();
    if (key_next >= 0) issue_v(key_next);
    f32x4 sacc[2], pacc[2];
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      pacc[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* vp = &rows[(jt * 16 + l16) * VLD + kq * 8];
#pragma unroll
      for (int kc = 0; kc < VC; kc++)
        pacc[jt] = mfma16(*reinterpret_cast<const bf16x8*>(vp + kc * 32), dof[kc], pacc[jt]);
    }
    lds_order();
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&rows[(pc / KP) * KLD + (pc % KP) * 8]) = kr[j];
    }
    lds_order();
    if (key_next >= 0) issue_k(key_next);
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      sacc[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* kp = &rows[(jt * 16 + l16) * KLD + kq * 8];
#pragma unroll
      for (int kc = 0; kc < KC; kc++)
        sacc[jt] = mfma16(*reinterpret_cast<const bf16x8*>(kp + kc * 32), qf[kc], sacc[jt]);
    }
    const int kmax = key_last - key0;
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
      for (int i = 0; i < 4; i++) sacc[jt][i] = fast_exp2(__builtin_fmaf(sacc[jt][i], sc, -lse));
    if (kmax < UK - 1) {  // wave-uniform
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (jt * 16 + kq * 4 + i > kmax) sacc[jt][i] = 0.f;
    }
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
      for (int i = 0; i < 4; i++) sacc[jt][i] *= (pacc[jt][i] - delta);
    bf16x8 df = pack8(sacc[0][0], sacc[0][1], sacc[0][2], sacc[0][3], sacc[1][0], sacc[1][1], sacc[1][2], sacc[1][3]);
    const int kb0 = kq * 4 + (l16 >> 2);
    const int kb1 = kb0 + 16;
#pragma unroll
    for (int dt = 0; dt < D / 16; dt++) {
      const int col = dt * 16 + 4 * (l16 & 3);
      bf16x4 a0 = lds_read_tr(&rows[kb0 * KLD + col]);
      bf16x4 a1 = lds_read_tr(&rows[kb1 * KLD + col]);
      dqacc[dt] = mfma16(cat4(a0, a1), df, dqacc[dt]);
    }
    lds_order();
    key0 = key_next;
  }

  if (!head_ok) return;
  const float osc = p.sm_scale;
  const int64_t off = tok * p.dq_st + (int64_t)head * p.dq_sh + kq * 4;
#pragma unroll
  for (int dt = 0; dt < D / 16; dt++) {
    f32x4 val = dqacc[dt] * osc;
    if (p.dq_mode == 0) {
      *reinterpret_cast<bf16x4*>((bf16_t*)p.dq + off + dt * 16) = pack4(val[0], val[1], val[2], val[3]);
    } else {
      float* dst = (float*)p.dq + off + dt * 16;
      if (p.dq_mode == 2) val += *reinterpret_cast<f32x4*>(dst);
      *reinterpret_cast<f32x4*>(dst) = val;
    }
  }
}

}  // namespace

int nsa_slc_bwd_dq_launch(const NsaSlcBwdDqParams& p, int B, int max_q_len, int D, int VD, hipStream_t stream) {
  max_q_len -= p.t_begin;
  if (B <= 0 || max_q_len <= 0) return NSA_OK;
  dim3 grid(cdiv_i(max_q_len, 4), B, p.KH * ((p.G + 15) / 16));
  if (D == 128 && VD == 128) slc_dq_kernel<128, 128><<<grid, 256, 0, stream>>>(p);
  else if (D == 64 && VD == 64) slc_dq_kernel<64, 64><<<grid, 256, 0, stream>>>(p);
  else if (D == 192 && VD == 128) slc_dq_kernel<192, 128><<<grid, 256, 0, stream>>>(p);
  else if (D == 256 && VD == 256) slc_dq_kernel<256, 256><<<grid, 256, 0, stream>>>(p);
  else if (D == 32 && VD == 32) slc_dq_kernel<32, 32><<<grid, 256, 0, stream>>>(p);
  else {
    nsa_set_error("selected attention dq: unsupported head dims D=%d VD=%d", D, VD);
    return NSA_ERR_UNSUPPORTED;
  }
  return nsa_check_launch("slc_dq_kernel");
}
