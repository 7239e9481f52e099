// dQ of the compressed and the window branch from the dS that their dK/dV kernels stored (nsa_bwd_dkdv_dma.hip): dQ = dS K over
// the branches' keys, 64 rows (token, q-head) per wave, the sum of both branches in the same accumulators.
//
// Layout of the stored dS, per branch and kv head: tiles of 64 rows (64 / G tokens of one sequence), in a tile the units of 32
// keys that its tokens see (counted from the branch's first key, for the window from the unit that holds the first key that the
// tile's first token sees), in a unit four blobs of 16 rows, 1 KB each, as the dK/dV kernel's lanes hold them: lane l = key
// l % 32 and the rows (l / 32) * 4 .. +3, then 8 + (l / 32) * 4 .. +3.
//
// What bounds it: reading the dS, 4 KB per wave and unit, once and in order; K passes through LDS for the four waves together.
// Three units are in LDS, two of them in flight, two workgroups on a CU (three named arrays, so that the compiler's waits for
// one do not cover the loads of the others).  The two kernels that compute S and dP again and this one, us, 64 heads of 128: 64K
// tokens 7180 + 2450 and 4930 (22 GB of dS read, 2.1 GB of dQ written: 4.9 TB/s), 8 x 6K tokens 1390 + 1710 and 1235; storing
// the dS adds 1.2 and 1.0 ms to the 8.9 and 2.8 of the dK/dV kernels at 64K tokens.
//
// LDS layout of K: row r holds its 16-byte chunk c at c ^ 4 (r & 3) (64 or 192 channels: c ^ 4 ((r >> 1) & 1)); of a blob: the
// chunk of lane l at l ^ 4 (l / 32).  Both spread the transposed reads (4 keys x 32 or 64 bytes) over all banks.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include <utility>

namespace {

typedef __attribute__((address_space(1))) const void* nsa_gptr_t;
typedef __attribute__((address_space(3))) void* nsa_lptr_t;

// (by value: a conditional expression of two variables is one of their addresses, which puts them into scratch memory)
template <class T>
NSA_DEVICE T pick(bool c, T x, T y) { return c ? x : y; }

template <int D>
__global__ __launch_bounds__(256, 2) void bwd_dq_ds_kernel(NsaDqDsParams p) {
  constexpr int P = D / 8;             // 16-byte chunks per row of K
  constexpr int KJ = 32 * P / 256;     // K loads per thread and unit
  constexpr int KEL = 32 * D;          // elements of a unit's K rows
  constexpr int STAGE = KEL + 4 * 2048;
  constexpr int NST = D <= 128 ? 3 : 2;  // units in LDS
  constexpr int NL = KJ + 4;             // loads of a wave per unit
  __shared__ __attribute__((aligned(1024))) bf16_t stage_a[STAGE];
  __shared__ __attribute__((aligned(1024))) bf16_t stage_b[STAGE];
  __shared__ __attribute__((aligned(1024))) bf16_t stage_c[NST == 3 ? STAGE : 8];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y, kh = blockIdx.z;
  const int G = p.G, gshift = __builtin_ctz(G), tshift = 6 - gshift;
  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  int lo, hi;
  nsa_local_range(p.tok0, p.tok1, x0, xl, lo, hi);
  const int tile_wg = (lo >> tshift) + blockIdx.x * 4;
  const int tile_end = (hi + (1 << tshift) - 1) >> tshift;
  if (tile_wg >= tile_end) return;
  const bool active = tile_wg + wave < tile_end;
  const int tile = min(tile_wg + wave, tile_end - 1);
  // tokens of the workgroup, of the wave
  const int t0_wg = tile_wg << tshift, t1_wg = min((tile_wg + 4) << tshift, hi) - 1;
  const int t0 = tile << tshift, t1 = min((tile + 1) << tshift, hi) - 1;

  // ---- the units of the three segments: compressed keys, window, keys before the window (of the queries whose selected branch
  // the window branch continues).  `w_*`: those of the wave among the workgroup's
  const int x0_tiles = x0 >> tshift;
  int n_seg0 = 0, n_seg1 = 0, n_seg2 = 0;
  int w_n0 = 0, w_lo1 = 0, w_n1 = 0, w_n2 = 0, lo1 = 0;
  int last0 = 0, last2 = 0;  // last key that the workgroup sees
  const bf16_t *k0 = nullptr, *k1 = nullptr, *d0 = nullptr, *d1 = nullptr, *d2 = nullptr;
  if (p.cmp.ds != nullptr) {
    const int kb = p.y_cu[b], nk = p.y_cu[b + 1] - kb;
    auto seen = [&](int t) {
      return t >= p.kernel_size - 1 ? min(__builtin_amdgcn_readfirstlane((t - p.kernel_size + 1) / p.stride) + 1, nk) : 0;
    };
    last0 = seen(t1_wg) - 1;
    n_seg0 = (last0 + 32) >> 5;
    w_n0 = (seen(t1) + 31) >> 5;
    k0 = p.cmp.k + (int64_t)kb * p.cmp.k_sr + (int64_t)kh * p.cmp.k_sh;
    d0 = p.cmp.ds + (int64_t)kh * p.cmp.ds_sh +
         (int64_t)nsa_ds_tile(p.cmp.tiles, p.cmp.seq_tiles, x0_tiles, b, tile) * p.cmp.pitch * 2048;
  }
  if (p.win.ds != nullptr) {
    k1 = p.win.k + (int64_t)x0 * p.win.k_sr + (int64_t)kh * p.win.k_sh;
    lo1 = max(0, t0_wg - p.window) >> 5;
    n_seg1 = (t1_wg >> 5) - lo1 + 1;
    w_lo1 = max(0, t0 - p.window) >> 5;
    w_n1 = (t1 >> 5) - w_lo1 + 1;
    d1 = p.win.ds + (int64_t)kh * p.win.ds_sh +
         (int64_t)nsa_ds_tile(p.win.tiles, p.win.seq_tiles, x0_tiles, b, tile) * p.win.pitch * 2048;
    if (p.far.ds != nullptr && t0_wg < p.all_below) {
      last2 = min(t1_wg, p.all_below - 1) - p.window - 1;
      n_seg2 = last2 >= 0 ? (last2 >> 5) + 1 : 0;
      const int w_last = min(t1, p.all_below - 1) - p.window - 1;
      w_n2 = t0 < p.all_below && w_last >= 0 ? (w_last >> 5) + 1 : 0;
      d2 = p.far.ds + (int64_t)kh * p.far.ds_sh +
           (int64_t)nsa_ds_tile(p.far.tiles, p.far.seq_tiles, x0_tiles, b, w_n2 > 0 ? tile : tile_wg) * p.far.pitch * 2048;
    }
  }
  const int n_units = n_seg0 + n_seg1 + n_seg2;

  f32x16 acc[2][D / 32];
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[rb][dt][i] = 0.f;

  auto swz = [](int r) { return D == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2; };
  // this lane's piece of every K load: row, byte offset of the chunk that its place holds
  int krow[KJ];
  uint32_t kcol[KJ];
#pragma unroll
  for (int j = 0; j < KJ; j++) {
    const int pc = (j * 4 + wave) * 64 + lane;
    krow[j] = pc / P;
    kcol[j] = (uint32_t)((pc % P) ^ swz(krow[j])) * 16;
  }
  const uint32_t dcol = (uint32_t)(lane ^ ((lane >> 5) << 2)) * 16;

  // Loads of unit i (behind the last one: of that once more, so that the waits can count).  Units that the workgroup sees and
  // this wave does not: the dS of one that it sees, or of any written one, which nobody reads.
  auto issue = [&](int i, bf16_t* buf) {
    i = min(i, n_units - 1);
    const bool s0 = i < n_seg0, s1 = i < n_seg0 + n_seg1;
    const int j = i - pick(s0, 0, pick(s1, n_seg0, n_seg0 + n_seg1));
    const int unit = j + (!s0 && s1 ? lo1 : 0);
    const int last = pick(s0, last0, pick(s1, t1_wg, last2)) - unit * 32;
    const int64_t k_sr = pick(s0, p.cmp.k_sr, p.win.k_sr);
    const bf16_t* const kb = pick(s0, k0, k1) + (int64_t)unit * 32 * k_sr;
    const uint32_t row_bytes = (uint32_t)k_sr * 2;
#pragma unroll
    for (int l = 0; l < KJ; l++) {
      const char* at = reinterpret_cast<const char*>(kb);
      uint32_t off = (uint32_t)min(krow[l], last) * row_bytes + kcol[l];
      asm volatile("" : "+s"(at), "+v"(off));  // (scalar base + 32-bit lane offset)
      __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + off), (nsa_lptr_t)(buf + (l * 4 + wave) * 512), 16, 0, 0);
    }
    const int wu = min(max(unit - pick(!s0 && s1, w_lo1, 0), 0), max(pick(s0, w_n0, pick(s1, w_n1, w_n2)) - 1, 0));
    const char* const at = reinterpret_cast<const char*>(pick(s0, d0, pick(s1, d1, d2)) + (int64_t)wu * 2048);
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const char* am = at + m * 1024;
      uint32_t off = dcol;
      asm volatile("" : "+s"(am), "+v"(off));
      __builtin_amdgcn_global_load_lds((nsa_gptr_t)(am + off), (nsa_lptr_t)(buf + KEL + wave * 2048 + m * 512), 16, 0, 0);
    }
  };

  // ---- fragment addresses (bytes)
  const int i16 = lane & 15, g16 = lane >> 4, hl = lane >> 5;
  // K transposed: row hl * 8 + i16 / 4 (+ 4, + 16 ks), channels dt * 32 + (g16 & 1) * 16 + 4 (i16 & 3)
  const int kr = hl * 8 + (i16 >> 2);
  const int ka0 = kr * D * 2 + ((g16 & 1) * 2 + ((i16 & 3) >> 1)) * 16 + (i16 & 1) * 8, ksw = swz(kr) * 16;
  auto k_at = [&](int dt) {
    if (D <= 128) return (ka0 + ksw) ^ (dt << 6);              // (a row is a power of two)
    return ka0 + (dt & 1 ? -ksw : ksw) + dt * 64;              // one bit of swizzle
  };
  // dS: keys as K's rows, rows (g16 & 1) * 16 + 4 (i16 & 3) of 32
  const int pp = i16 & 1;
  const int da0 = KEL * 2 + wave * 4096 + (g16 & 1) * 1024 + ((pp * 32 + kr) ^ (pp << 2)) * 16 + ((i16 & 3) >> 1) * 8;
  const int da1 = da0 ^ 64;

  // one unit: `cur` holds it (its loads are in flight), `nxt` receives the one NST - 1 further
  auto step = [&](const bf16_t* cur, bf16_t* nxt, int i) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70 + (NST - 2) * NL);  // vmcnt: the loads of the units behind this one
    __builtin_amdgcn_s_barrier();  // everybody's K rows are there; nobody reads `nxt` any more
    asm volatile("" ::: "memory");
    issue(i + NST - 1, nxt);
    const bool s0 = i < n_seg0, s1 = i < n_seg0 + n_seg1;
    const int at = i - pick(s0, 0, pick(s1, n_seg0 - lo1 + w_lo1, n_seg0 + n_seg1));
    const bool mine = (unsigned)at < (unsigned)pick(s0, w_n0, pick(s1, w_n1, w_n2));
    if (mine && active) {
      const char* const base = reinterpret_cast<const char*>(cur);
      auto tr = [&](int at) { return lds_read_tr(reinterpret_cast<const bf16_t*>(base + at)); };
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        bf16x8 df[2];
#pragma unroll
        for (int rb = 0; rb < 2; rb++) df[rb] = cat4(tr(da0 + rb * 2048 + ks * 256), tr(da1 + rb * 2048 + ks * 256));
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++) {
          const int ka = k_at(dt) + ks * 16 * D * 2;
          const bf16x8 kf = cat4(tr(ka), tr(ka + 4 * D * 2));
          acc[0][dt] = mfma32(kf, df[0], acc[0][dt]);
          acc[1][dt] = mfma32(kf, df[1], acc[1][dt]);
        }
      }
    }
    // the reads have to have been answered before anybody loads over them
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  };

  if (n_units > 0) {
    issue(0, stage_a);
    if (NST == 3) issue(1, stage_b);
    // (whole turns through the buffers, with steps behind the last unit that add nothing: where the loop can end behind every
    // step, the compiler waits for all loads in its first one)
    for (int i = 0; i < n_units;) {
      if constexpr (NST == 3) {
        step(stage_a, stage_c, i++);
        step(stage_b, stage_a, i++);
        step(stage_c, stage_b, i++);
      } else {
        step(stage_a, stage_b, i++);
        step(stage_b, stage_a, i++);
      }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // nothing lands in LDS behind the workgroup's end
    asm volatile("" ::: "memory");
  }

  if (!active) return;
  const float osc = p.sm_scale;
  const int l32 = lane & 31;
#pragma unroll
  for (int rb = 0; rb < 2; rb++) {
    const int r = rb * 32 + l32;
    const int t = t0 + (r >> gshift);
    if (t > t1) continue;
    const int64_t tok = x0 + t;
    const int head = kh * G + (r & (G - 1));
    // mode 3: q's dtype below all_below, the fp32 buffer for the others
    const bool to_final = p.dq_mode == 0 || (p.dq_mode == 3 && t < p.all_below);
    float* const f = p.dq_mode == 3 ? p.dq_partial + tok * p.dqp_st + (int64_t)head * p.dqp_sh
                                    : (float*)p.dq + tok * p.dq_st + (int64_t)head * p.dq_sh;
    bf16_t* const h = (bf16_t*)p.dq + tok * p.dq_st + (int64_t)head * p.dq_sh;
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        const int d = dt * 32 + i4 * 8 + hl * 4;
        f32x4 val = {acc[rb][dt][i4 * 4 + 0] * osc, acc[rb][dt][i4 * 4 + 1] * osc, acc[rb][dt][i4 * 4 + 2] * osc,
                     acc[rb][dt][i4 * 4 + 3] * osc};
        if (to_final) {
          *reinterpret_cast<bf16x4*>(h + d) = pack4(val[0], val[1], val[2], val[3]);
        } else {
          if (p.dq_mode == 2) val += *reinterpret_cast<const f32x4*>(f + d);
          *reinterpret_cast<f32x4*>(f + d) = val;
        }
      }
  }
}

template <int D>
int launch(const NsaDqDsParams& p, dim3 grid, hipStream_t stream) {
  bwd_dq_ds_kernel<D><<<grid, 256, 0, stream>>>(p);
  return nsa_check_launch("bwd_dq_ds_kernel");
}

}  // namespace

int nsa_bwd_dq_ds_launch(const NsaDqDsParams& p, int B, int max_q_len, int D, hipStream_t stream) {
  if (B <= 0 || max_q_len <= 0) return NSA_OK;
  int len = max_q_len;  // longest share of a sequence
  if (p.tok1 > 0) len = min(len, p.tok1 - p.tok0 + 127);
  const int tile = 64 / p.G;
  const dim3 grid(cdiv_i(cdiv_i(len, tile), 4), B, p.KH);
  if (D == 128) return launch<128>(p, grid, stream);
  if (D == 192) return launch<192>(p, grid, stream);
  nsa_set_error("attention dq from stored dS: unsupported head dim D=%d", D);
  return NSA_ERR_UNSUPPORTED;
}
