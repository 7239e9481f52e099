// Dense-tile flash forward for the two branches whose key set is a contiguous range per query:
//   MODE_CMP: compressed attention, key i visible to absolute query position t iff t >= stride*i + kernel-1
//             (upstream flash_nsa/ops/compress_attn.py:17-153; paged: flash_nsa/inference/compress_attn.py:19-149)
//   MODE_SWA: causal sliding window, keys max(0,t-W) <= j <= t
//             (upstream flash_nsa/ops/sliding_window_attention.py:26-95, which calls FlashAttention)
//
// Work decomposition: a "row" is one (query token, q-head) pair of one kv-head group, rows ordered
// token-major / head-minor so that the G heads sharing K/V sit next to each other.  A workgroup of 4 waves
// owns 4*32*RS consecutive rows; every lane owns RS rows (lane l and l+32 share a row and split its keys), so
// the online-softmax statistics are per-lane scalars.  Key tiles of 64 rows are staged in LDS (row-major) and
// shared by the 4 waves.  S^T = K Q^T and O^T = V^T P^T are computed with v_mfma_f32_32x32x16_bf16; the V^T
// operand comes from ds_read_b64_tr_b16 so V never needs an explicit transpose.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include <type_traits>

namespace {

constexpr int MODE_CMP = 0;
constexpr int MODE_SWA = 1;
constexpr int MODE_TAIL = 2;  // MODE_SWA, and what can be finished in the same launch (below)
constexpr int MODE_ALL = 3;   // MODE_TAIL behind the compressed branch of the same queries (all of them below all_below)

typedef __attribute__((address_space(1))) const void* nsa_gptr_t;
typedef __attribute__((address_space(3))) void* nsa_lptr_t;

// position swizzle of the 16-byte chunks of row r in an unpadded LDS tile with CP chunks per row: chunk c sits at
// position c ^ swz(r), which spreads the rows that a fragment read touches over all banks
template <int CP>
NSA_DEVICE constexpr int swz(int r) { return CP % 16 == 0 ? (r & 15) : ((r >> 1) & 7); }
// the same for the V tile, whose transposed reads fetch 32 bytes (two chunks) from each of four consecutive rows
// per group of 16 lanes: the swizzle moves whole chunk pairs, so that the rows of a group (and of the wave's other
// groups) land in different 32-byte bank slots (measured: 108 bytes/clk/CU against 61 with swz above)
template <int CP>
NSA_DEVICE constexpr int swzv(int r) { return CP % 16 == 0 ? ((r & 7) << 1) : (((r >> 1) & 3) << 1); }

// a wave-uniform address in scalar registers (one that divisions went into is uniform and in vector registers)
NSA_DEVICE const char* scalar_ptr(const void* x) {
  const uint64_t v = reinterpret_cast<uint64_t>(x);
  const uint32_t l = __builtin_amdgcn_readfirstlane((uint32_t)v), h = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const char*>(((uint64_t)h << 32) | l);
}

// The widest row stride of ASYNC: a lane's offset inside a period of its loads (up to 32 rows, 64 of 32 channels) has 32 bits.
constexpr int64_t async_row_stride(int D, int VD) { return D >= 64 && VD >= 64 ? 1 << 26 : 1 << 25; }

// ASYNC: the K/V tiles go from global memory straight into LDS (global_load_lds, 16 bytes per lane, no staging
// registers, no ds_write); the tiles are then unpadded and swizzled instead of padded.
template <int D, int VD, int MODE, bool PAGED, int RS, int MINB, bool ASYNC>
__global__ __launch_bounds__(256, MINB) void fwd_tile_kernel(NsaFwdTileParams p) {
  static_assert(RS == 1 || RS == 2, "one or two 32-row sets per wave");
  constexpr int ROWS_W = 32 * RS;
  constexpr int ROWS_WG = 4 * ROWS_W;
  constexpr int KT = 64;
  constexpr int KLD = ASYNC ? D : D + NSA_LDS_PAD;
  constexpr int VLD = ASYNC ? VD : VD + NSA_LDS_PAD;
  // two K/V tile buffers: the tile after the one being computed is stored while the other waves may still read the
  // current one, so a tile costs one barrier
  __shared__ __attribute__((aligned(16))) bf16_t Ks2[2][KT * KLD];
  __shared__ __attribute__((aligned(16))) bf16_t Vs2[2][KT * VLD];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hl = lane >> 5;
  const int g16 = lane >> 4, i16 = lane & 15;
  // (sequences and heads take turns on the XCDs, whose workgroups come round robin)
  const int seq_head = (blockIdx.x + blockIdx.y) % gridDim.x;
  const int b = p.last_first ? seq_head / p.KH : blockIdx.y;
  const int kh = p.last_first ? seq_head % p.KH : blockIdx.z;
  const int G = p.G;

  const int x0 = p.x_cu[b];
  const int xl = p.x_cu[b + 1] - x0;
  const int ctx = PAGED ? p.ctx_lens[b] : xl;
  const int qoff = ctx - xl;
  const int rows_total = xl * G;
  const int r0 = (p.last_first ? gridDim.y - 1 - blockIdx.y : blockIdx.x) * ROWS_WG;
  if (r0 >= rows_total) return;
  constexpr bool TAIL = MODE == MODE_TAIL || MODE == MODE_ALL;
  constexpr bool HAS_CMP = MODE == MODE_CMP || MODE == MODE_ALL;
  int nkeys, kbase = 0;
  if (HAS_CMP) {
    nkeys = ctx >= p.kernel_size ? (ctx - p.kernel_size) / p.stride + 1 : 0;
    if (!PAGED) kbase = p.k_cu[b];
  } else {
    nkeys = ctx;
    if (!PAGED) kbase = x0;
  }
  // where the keys lie: MODE_ALL starts with the compressed rows
  bool in_cmp = HAS_CMP;
  const bf16_t *ksrc = MODE == MODE_ALL ? p.ck : p.k, *vsrc = MODE == MODE_ALL ? p.cv : p.v;
  int64_t k_sr = MODE == MODE_ALL ? p.ck_sr : p.k_sr, v_sr = MODE == MODE_ALL ? p.cv_sr : p.v_sr;
  int64_t k_sh = MODE == MODE_ALL ? p.ck_sh : p.k_sh, v_sh = MODE == MODE_ALL ? p.cv_sh : p.v_sh;
  const int32_t* table = !PAGED ? nullptr : MODE == MODE_ALL ? p.c_table + (int64_t)b * p.c_table_stride : p.table + (int64_t)b * p.table_stride;

  // ---- per-lane rows ----
  int t_row[RS];
  bool valid[RS];
  int64_t tok[RS];
  int head[RS];
  int key_hi[RS];  // the last compressed key that the row sees
  bf16x8 qf[RS][D / 16];
#pragma unroll
  for (int rs = 0; rs < RS; rs++) {
    int r = r0 + wave * ROWS_W + rs * 32 + l32;
    valid[rs] = r < rows_total;
    int rr = valid[rs] ? r : rows_total - 1;
    int n = rr / G;
    int g = rr - n * G;
    t_row[rs] = n + qoff;
    if (HAS_CMP) key_hi[rs] = t_row[rs] >= p.kernel_size - 1 ? min((t_row[rs] - p.kernel_size + 1) / p.stride, nkeys - 1) : -1;
    tok[rs] = x0 + n;
    head[rs] = kh * G + g;
    const bf16_t* qp = p.q + tok[rs] * p.q_st + (int64_t)head[rs] * p.q_sh + hl * 8;
#pragma unroll
    for (int kc = 0; kc < D / 16; kc++) qf[rs][kc] = ld_global_b128(qp + kc * 16);
  }
  // wave-uniform position range (scalar registers)
  const int rw_lo = r0 + wave * ROWS_W;
  const int rw_hi = min(rw_lo + ROWS_W - 1, rows_total - 1);
  const bool wave_active = rw_lo < rows_total;
  const int tw_lo = (wave_active ? rw_lo / G : 0) + qoff;
  const int tw_hi = (wave_active ? rw_hi / G : 0) + qoff;
  const int t_lo = r0 / G + qoff;
  const int t_hi = min(r0 + ROWS_WG - 1, rows_total - 1) / G + qoff;

  int key_begin, key_end;
  if (HAS_CMP) {
    key_begin = 0;
    key_end = t_hi >= p.kernel_size - 1 ? min((t_hi - p.kernel_size + 1) / p.stride + 1, nkeys) : 0;
  }
  if (MODE != MODE_CMP && MODE != MODE_ALL) {
    key_begin = (max(0, t_lo - p.window) / KT) * KT;
    key_end = min(t_hi + 1, nkeys);
  }

  // window: keys t + klo .. t + khi; before the window: keys .. t + khi, of queries at positions below t_end
  int klo = -p.window, khi = 0, t_end = 0x7fffffff;

  f32x16 oacc[RS][VD / 32];
  float m_run[RS], l_run[RS];
  auto reset = [&]() {
#pragma unroll
    for (int rs = 0; rs < RS; rs++) {
      m_run[rs] = NSA_NEG_INF;
      l_run[rs] = 0.f;
#pragma unroll
      for (int dt = 0; dt < VD / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[rs][dt][i] = 0.f;
    }
  };
  reset();
  const float sc = p.scale_log2;

  // software pipeline: the next tile's global loads are in flight while the current tile is computed.
  // Rows past the end of the key range are replaced by the last valid row; their scores are masked, so the
  // duplicated data never contributes.
  constexpr int KP = D / 8, VP = VD / 8;
  constexpr int KJ = (KT * KP) / 256, VJ = (KT * VP) / 256;
  bf16x8 kreg[KJ], vreg[VJ];
  auto gload = [&](int kt) {
    int64_t page_row0 = 0;
    if (PAGED) {
      int pg = table[kt / p.page_size];
      page_row0 = (int64_t)pg * p.page_size + (kt % p.page_size);
    }
    const int last = key_end - 1 - kt;  // >= 0
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      int pc = tid + j * 256;
      int kr = min(pc / KP, last), dp = pc % KP;
      int64_t row = PAGED ? page_row0 + kr : (int64_t)kbase + kt + kr;
      kreg[j] = ld_global_b128(ksrc + row * k_sr + (int64_t)kh * k_sh + dp * 8);
    }
#pragma unroll
    for (int j = 0; j < VJ; j++) {
      int pc = tid + j * 256;
      int kr = min(pc / VP, last), dp = pc % VP;
      int64_t row = PAGED ? page_row0 + kr : (int64_t)kbase + kt + kr;
      vreg[j] = ld_global_b128(vsrc + row * v_sr + (int64_t)kh * v_sh + dp * 8);
    }
  };

  // one 64-key tile for one row set
  // Fragment addresses.  Padded tiles: row * stride + column, the compiler folds everything but the lane part into
  // immediates.  Swizzled tiles with a power-of-two row size: byte address = lane part XOR (index << 5 or 6) +
  // compile-time row offset, with the lane parts computed once (kx, vxa, vxb), so a read costs at most one v_xor.
  // (192 channels: a row of three 128-byte pieces, the swizzle stays inside a piece)
  constexpr bool XORED = (D == 64 || D == 128 || D == 192) && (VD == 64 || VD == 128);
  int kx = 0, vxa = 0, vxb = 0;
  if constexpr (ASYNC && XORED) {
    const int s0 = swz<D / 8>(l32);
    kx = (l32 * D * 2 + ((hl ^ (s0 & 1)) << 4)) ^ ((s0 >> 1) << 5);
    const int sl = hl * 4 + (i16 >> 2);                 // row of the fragment inside its group of 16 rows
    const int cl = (g16 & 1) * 2 + ((i16 & 3) >> 1);    // chunk inside its group of 4 chunks
    const int sa = swzv<VD / 8>(sl), sb = swzv<VD / 8>(sl + 8);
    vxa = (sl * VD * 2 + ((cl ^ (sa & 3)) << 4) + (i16 & 1) * 8) ^ ((sa >> 2) << 6);
    vxb = ((sl + 8) * VD * 2 + ((cl ^ (sb & 3)) << 4) + (i16 & 1) * 8) ^ ((sb >> 2) << 6);
  }
  // K fragment: rows l32 + 32*half, chunk 2*kc + hl
  auto kfrag = [&](const bf16_t* Ks, int half, int kc) -> bf16x8 {
    if constexpr (ASYNC && XORED && D == 192)
      return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(Ks) + half * 32 * D * 2 + (kc >> 2) * 128 +
                                              (kx ^ ((kc & 3) << 5)));
    else if constexpr (ASYNC && XORED)
      return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(Ks) + half * 32 * D * 2 + (kx ^ (kc << 5)));
    else if constexpr (ASYNC)
      return *reinterpret_cast<const bf16x8*>(
          Ks + ((l32 + 32 * half) * (D / 8) + ((2 * kc + hl) ^ swz<D / 8>(l32))) * 8);
    else
      return *reinterpret_cast<const bf16x8*>(Ks + (l32 + 32 * half) * KLD + (2 * kc + hl) * 8);
  };
  // transposed V fragment piece: row kb + (i16 >> 2) (kb a multiple of 16, plus 8 for the second piece), columns
  // dt*32 + (g16&1)*16 + 4*(i16&3) ..
  auto vfrag = [&](const bf16_t* Vs, int kb16, int second, int dt) -> bf16x4 {
    if constexpr (ASYNC && XORED) {
      const int x = (second ? vxb : vxa) ^ (dt << 6);
      return lds_read_tr(reinterpret_cast<const bf16_t*>(reinterpret_cast<const char*>(Vs) + kb16 * VD * 2 + x));
    } else {
      const int row = kb16 + second * 8 + hl * 4 + (i16 >> 2);
      const int col = dt * 32 + (g16 & 1) * 16 + 4 * (i16 & 3);
      if constexpr (ASYNC) return lds_read_tr(Vs + (row * (VD / 8) + ((col >> 3) ^ swzv<VD / 8>(row))) * 8 + (col & 7));
      else return lds_read_tr(Vs + row * VLD + col);
    }
  };
  auto process = [&](bool mask_hi, bool mask_lo, auto rs_tag, int kt, const bf16_t* Ks, const bf16_t* Vs) {
    constexpr int rs = decltype(rs_tag)::value;
    // ---- S^T = K Q^T : two 32-key sub tiles, interleaved accumulators ----
    f32x16 sacc[2];
#pragma unroll
    for (int i = 0; i < 16; i++) { sacc[0][i] = 0.f; sacc[1][i] = 0.f; }
#pragma unroll
    for (int kc = 0; kc < D / 16; kc++) {
      bf16x8 k0 = kfrag(Ks, 0, kc);
      bf16x8 k1 = kfrag(Ks, 1, kc);
      sacc[0] = mfma32(k0, qf[rs][kc], sacc[0]);
      sacc[1] = mfma32(k1, qf[rs][kc], sacc[1]);
    }
    // ---- mask, online softmax (running max in raw score units; scale folded into the exp2 fma) ----
    // Wave-uniform: only tiles that straddle a visibility boundary pay for its mask, which compares the key's place in the tile
    // (a constant) with the row's bound: two instructions per score.  (Three terms per score in one test: four and two scalar
    // ones, 64 more of a wave's 250 vector instructions per tile; short sequences mask two to four of their 2 to 12 tiles.)
    if (mask_hi) {
      asm volatile("");  // keeps it a branch: if-converted, every tile would pay
      const int bound = (HAS_CMP && in_cmp ? key_hi[rs] : TAIL && t_row[rs] >= t_end ? -0x40000000 : t_row[rs] + khi) -
                        kt - hl * 4;
#pragma unroll
      for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          sacc[nt][i] = nt * 32 + (i >> 2) * 8 + (i & 3) <= bound ? sacc[nt][i] : NSA_NEG_INF;
    }
    if (MODE != MODE_CMP && mask_lo) {
      asm volatile("");
      const int bound = t_row[rs] + klo - kt - hl * 4;
#pragma unroll
      for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          sacc[nt][i] = nt * 32 + (i >> 2) * 8 + (i & 3) >= bound ? sacc[nt][i] : NSA_NEG_INF;
    }
    float tmax = NSA_NEG_INF;
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
      for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, sacc[nt][i]);
    tmax = xhalf_max(tmax);
    const float m_old = m_run[rs];
    const float m_new = fmaxf(m_old, tmax);
    const float m_safe = (m_new == NSA_NEG_INF) ? 0.f : m_new;
    const float msc = m_safe * sc;
    m_run[rs] = m_new;
    float psum = 0.f;
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        float pv = fast_exp2(__builtin_fmaf(sacc[nt][i], sc, -msc));
        sacc[nt][i] = pv;
        psum += pv;
      }
    if (__builtin_amdgcn_ballot_w64(m_new != m_old) != 0) {  // rescale only when some row's max moved
      const float alpha = fast_exp2((m_old - m_safe) * sc);
      l_run[rs] *= alpha;
#pragma unroll
      for (int dt = 0; dt < VD / 32; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[rs][dt][i] *= alpha;
    }
    l_run[rs] += psum;

    // ---- O^T += V^T P^T ----
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int nt = c >> 1, ch = c & 1;
      bf16x8 pf = pack8(sacc[nt][ch * 8 + 0], sacc[nt][ch * 8 + 1], sacc[nt][ch * 8 + 2], sacc[nt][ch * 8 + 3],
                        sacc[nt][ch * 8 + 4], sacc[nt][ch * 8 + 5], sacc[nt][ch * 8 + 6], sacc[nt][ch * 8 + 7]);
      const int kb16 = nt * 32 + ch * 16;  // the lane's rows: kb16 + hl*4 + (i16>>2) and 8 further
#pragma unroll
      for (int dt = 0; dt < VD / 32; dt++) {
        bf16x4 v0 = vfrag(Vs, kb16, 0, dt);
        bf16x4 v1 = vfrag(Vs, kb16, 1, dt);
        oacc[rs][dt] = mfma32(cat4(v0, v1), pf, oacc[rs][dt]);
      }
    }
  };

  auto stage = [&](int buf) {
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      int pc = tid + j * 256;
      *reinterpret_cast<bf16x8*>(&Ks2[buf][(pc / KP) * KLD + (pc % KP) * 8]) = kreg[j];
    }
#pragma unroll
    for (int j = 0; j < VJ; j++) {
      int pc = tid + j * 256;
      *reinterpret_cast<bf16x8*>(&Vs2[buf][(pc / VP) * VLD + (pc % VP) * 8]) = vreg[j];
    }
  };
  // ASYNC staging: lane L of a wave's j-th load fills LDS piece j*256 + wave*64 + L (row = piece / chunks per row,
  // position = piece % chunks per row), i.e. it fetches the chunk that the swizzle puts at that position
  // Per-lane byte offsets of its pieces from the first row of a tile (the same for every full tile): after KPAT / VPAT loads
  // columns and swizzle repeat, KROWS / VROWS rows further.
  constexpr int KPAT = 256 % KP == 0 ? 1 : 3, VPAT = 256 % VP == 0 ? 1 : 3;
  constexpr int KROWS = KPAT * 256 / KP, VROWS = VPAT * 256 / VP;
  static_assert(!ASYNC || (KROWS % 16 == 0 && VROWS % 16 == 0 && KJ % KPAT == 0 && VJ % VPAT == 0), "period of the swizzles");
  static_assert(!ASYNC || ((KROWS > VROWS ? KROWS : VROWS) - 1) * async_row_stride(D, VD) * 2 + 512 < (int64_t)1 << 32, "a lane's offset");
  uint32_t goffk[KPAT], goffv[VPAT];
  auto set_offsets = [&]() {
    if constexpr (ASYNC) {
#pragma unroll
      for (int j = 0; j < KPAT; j++) {
        const int pc = tid + j * 256, row = pc / KP;
        goffk[j] = (uint32_t)((row * k_sr + ((pc % KP) ^ swz<KP>(row)) * 8) * 2);
      }
#pragma unroll
      for (int j = 0; j < VPAT; j++) {
        const int pc = tid + j * 256, row = pc / VP;
        goffv[j] = (uint32_t)((row * v_sr + ((pc % VP) ^ swzv<VP>(row)) * 8) * 2);
      }
    }
  };
  set_offsets();
  auto stage_async = [&](int kt, int buf) {
    int64_t row0;
    if (PAGED) row0 = (int64_t)table[kt / p.page_size] * p.page_size + (kt % p.page_size);
    else row0 = (int64_t)kbase + kt;
    const int last = key_end - 1 - kt;  // >= 0; rows past it repeat it (masked)
    const char* kb = scalar_ptr(ksrc + row0 * k_sr + (int64_t)kh * k_sh);
    const char* vb = scalar_ptr(vsrc + row0 * v_sr + (int64_t)kh * v_sh);
    if (last >= KT - 1) {  // wave-uniform
#pragma unroll
      for (int j = 0; j < KJ; j++) {
        const char* at = kb + (int64_t)(j / KPAT) * KROWS * k_sr * 2;
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + goffk[j % KPAT]), (nsa_lptr_t)&Ks2[buf][(j * 256 + wave * 64) * 8], 16, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < VJ; j++) {
        const char* at = vb + (int64_t)(j / VPAT) * VROWS * v_sr * 2;
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + goffv[j % VPAT]), (nsa_lptr_t)&Vs2[buf][(j * 256 + wave * 64) * 8], 16, 0, 0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < KJ; j++) {
        const int pc = tid + j * 256;
        const int row = pc / KP, c = (pc % KP) ^ swz<KP>(row);
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(kb + ((int64_t)min(row, last) * k_sr + c * 8) * 2),
                                         (nsa_lptr_t)&Ks2[buf][(j * 256 + wave * 64) * 8], 16, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < VJ; j++) {
        const int pc = tid + j * 256;
        const int row = pc / VP, c = (pc % VP) ^ swzv<VP>(row);
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(vb + ((int64_t)min(row, last) * v_sr + c * 8) * 2),
                                         (nsa_lptr_t)&Vs2[buf][(j * 256 + wave * 64) * 8], 16, 0, 0);
      }
    }
  };
  auto run_keys = [&]() {
    if (key_begin < key_end) {
      if constexpr (ASYNC) {
        stage_async(key_begin, 0);
      } else {
        gload(key_begin);
        stage(0);
        if (key_begin + KT < key_end) gload(key_begin + KT);
      }
    }
    int buf = 0;
    for (int kt = key_begin; kt < key_end; kt += KT, buf ^= 1) {
      if constexpr (ASYNC) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of tile kt have landed
      __syncthreads();  // tile kt is visible; nobody reads the other buffer (tile kt - KT) any more
      if (kt + KT < key_end) {
        if constexpr (ASYNC) {
          stage_async(kt + KT, buf ^ 1);
        } else {
          stage(buf ^ 1);
          if (kt + 2 * KT < key_end) gload(kt + 2 * KT);
        }
      }
      if (!wave_active) continue;

      // wave-uniform visibility classification of this tile
      bool any_vis, mask_hi, mask_lo = false;
      if (HAS_CMP && in_cmp) {
        any_vis = tw_hi >= p.stride * kt + p.kernel_size - 1;
        mask_hi = tw_lo < p.stride * (kt + KT - 1) + p.kernel_size - 1 || kt + KT > nkeys;
      } else {
        any_vis = (kt <= tw_hi + khi) && (kt + KT - 1 >= tw_lo + klo);
        mask_hi = kt + KT - 1 > tw_lo + khi || (TAIL && tw_hi >= t_end);
        mask_lo = kt < tw_hi + klo;
      }
      if (!any_vis) continue;
      process(mask_hi, mask_lo, std::integral_constant<int, 0>{}, kt, Ks2[buf], Vs2[buf]);
      if constexpr (RS > 1) process(mask_hi, mask_lo, std::integral_constant<int, RS - 1>{}, kt, Ks2[buf], Vs2[buf]);
    }
  };

  // Epilogue.  A lane holds 4-channel pieces of one row; stored (or combined with other tensors) as they lie, every
  // instruction would touch 32 rows.  The rows pass through LDS instead (bf16, wave-private, 16-byte chunks swizzled by
  // row) and are handled as whole rows, 16 bytes per lane.
  constexpr int NC = VD / 8;                     // chunks per row
  constexpr int RPI = 64 / NC;                   // rows per instruction
  static_assert(32 * VD * 4 <= 2 * KT * KLD, "the K tiles hold the rows of the four waves");
  bf16_t* const rows = &Ks2[0][0] + wave * 32 * VD;
  auto chunk_at = [&](int row, int c) { return rows + row * VD + ((c ^ (row & (NC - 1))) * 8); };
  // (token, head) of a row of the wave, from the lane that holds it; token -1: none
  auto row_id = [&](auto rs_tag, int r) {
    constexpr int rs = decltype(rs_tag)::value;
    return make_int2(__shfl(valid[rs] ? t_row[rs] - qoff : -1, r, 64), __shfl(head[rs], r, 64));
  };
  auto rows_to_lds = [&](auto rs_tag, float inv) {
    constexpr int rs = decltype(rs_tag)::value;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int dt = 0; dt < VD / 32; dt++)
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++)
        *reinterpret_cast<bf16x4*>(chunk_at(l32, dt * 4 + i4) + hl * 4) =
            pack4(oacc[rs][dt][i4 * 4 + 0] * inv, oacc[rs][dt][i4 * 4 + 1] * inv, oacc[rs][dt][i4 * 4 + 2] * inv,
                  oacc[rs][dt][i4 * 4 + 3] * inv);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // the branch output and log-sum-exp of the keys so far, of the queries at positions below `below`
  auto emit = [&](bf16_t* o, int64_t o_st, int64_t o_sh, float* lse, int64_t lse_st, int64_t lse_sh, int below) {
    auto one = [&](auto rs_tag) {
      constexpr int rs = decltype(rs_tag)::value;
      const float l_tot = xhalf_sum(l_run[rs]);
      rows_to_lds(rs_tag, l_tot > 0.f ? 1.f / l_tot : 0.f);
      const int c = lane % NC;
#pragma unroll
      for (int r = lane / NC; r < 32; r += RPI) {
        const int2 th = row_id(rs_tag, r);
        if (th.x < 0 || th.x + qoff >= below) continue;
        *reinterpret_cast<bf16x8*>(o + ((int64_t)x0 + th.x) * o_st + (int64_t)th.y * o_sh + c * 8) =
            *reinterpret_cast<const bf16x8*>(chunk_at(r, c));
      }
      if (hl == 0 && lse != nullptr && valid[rs] && t_row[rs] < below)
        lse[tok[rs] * lse_st + (int64_t)head[rs] * lse_sh] = l_tot > 0.f ? m_run[rs] * sc + fast_log2(l_tot) : 0.f;
    };
    one(std::integral_constant<int, 0>{});
    if constexpr (RS > 1) one(std::integral_constant<int, RS - 1>{});
  };
  constexpr int ALL = 0x7fffffff;
  run_keys();
  __syncthreads();  // the tile buffers are free
  if constexpr (MODE == MODE_ALL) {
    // Sequences whose queries all select everything have few compressed keys (63 at 1024 tokens: one tile), and nothing waits for
    // their log-sum-exps: the branch needs no launch of its own, and the same queries are read once.  Calls in two launches / in
    // one, us, 64 / 4 heads of 128: 3 prompts of 60 to 700 tokens 64.5 / 61, 2 of 300 to 900 69 / 65, 6 of 60 to 1000 125 / 119, 12
    // 252 / 237; forward of 1000 tokens 68 / 66, 16 / 1 heads, 3 of 100 to 400 65 / 47; 16 / 2 heads of 64, 40 of up to 1000 117 / 98,
    // 8 prompts 62 / 50.
    emit(p.cmp_o_out, p.co_st, p.co_sh, p.cmp_lse, p.cl_st, p.cl_sh, ALL);
    __syncthreads();
    reset();
    in_cmp = false;
    ksrc = p.k; vsrc = p.v; k_sr = p.k_sr; v_sr = p.v_sr; k_sh = p.k_sh; v_sh = p.v_sh;
    if (PAGED) table = p.table + (int64_t)b * p.table_stride;
    else kbase = x0;
    nkeys = ctx;
    set_offsets();
    key_begin = (max(0, t_lo - p.window) / KT) * KT;
    key_end = min(t_hi + 1, nkeys);
    run_keys();
    __syncthreads();
  }
  if constexpr (!TAIL) {
    emit(p.o, p.o_st, p.o_sh, p.lse, p.lse_st, p.lse_sh, ALL);
  } else {
    static_assert(RS == 1, "");
    // Queries at positions below all_below select every block they can see: their selected branch is the window branch
    // continued over the keys before the window (nothing at all up to position `window`), instead of a second pass
    // over all of their keys.  40 samples of up to 1.2K tokens, 16 heads of 64: selected kernel 278 -> 39 us, window
    // kernel 69 -> 92 us; 8 x 6K tokens, 64 heads of 128: 4477 -> 3947 us, and with the gated sum at its end
    // (one read of the branch outputs less) 1774 -> 1674 us.
    const int far_end = min(t_hi, p.all_below - 1) - p.window;  // keys before some query's window
    const bool far = far_end > 0 && t_lo < p.all_below;         // workgroup-uniform
    const bool store = p.store_branches || p.out == nullptr;
    if ((store || far) && p.o != nullptr) emit(p.o, p.o_st, p.o_sh, p.lse, p.lse_st, p.lse_sh, ALL);
    if (far) {
      __syncthreads();  // the rows in the tile buffers have been stored
      key_begin = 0;
      key_end = far_end;
      klo = -0x40000000;
      khi = -p.window - 1;
      t_end = p.all_below;
      run_keys();
      __syncthreads();
    }
    if (store && t_lo < p.all_below) emit(p.slc_o, p.so_st, p.so_sh, p.slc_lse, p.sl_st, p.sl_sh, p.all_below);
    if (p.out != nullptr) {
      // Gated sum.  What this launch holds in fp32 enters it unrounded: the selected branch of the queries that select
      // everything, the window branch of all but those of them that have keys before the window (read back as stored).
      // The two branches of the former share the bf16 roundings of P, which the gather of their blocks would make anew,
      // so their errors add up instead of averaging out; with the branch rows rounded as well the sum is further off than
      // the gated sum of separate launches (relative to 64 bits, 128 channels, up to 1024 tokens: 2.23e-3 separately,
      // 2.45e-3 from rounded rows, 2.0e-3 so).  The rows pass through LDS in two halves of their channels, which costs 2 to
      // 4 % of the launch against rounded rows in one pass (8 x 6K tokens, 64 heads of 128 1685 -> 1750 us, 16 x 2K paged
      // rows 1120 -> 1168 us, three short prompts 56 -> 57 us).
      constexpr int HC = NC / 2;                 // chunks of 8 channels per half row
      constexpr int HRPI = 64 / HC;              // rows per instruction
      float* const half = reinterpret_cast<float*>(rows);
      auto half_at = [&](int row, int c) { return half + row * (VD / 2) + ((c ^ (row & (HC - 1))) * 8); };
      const float l_tot = xhalf_sum(l_run[0]);
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
      auto lds_order = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      };
      // The gates of a row are computed by the lane that holds it, and everything else that a lane adds is requested before the
      // first row comes out of LDS: one round trip instead of one per row and half.  Calls before / with this, us: 16 x 2K paged
      // rows 5447 / 5370, 8 x 6K tokens 6060 / 5980, three short prompts 76.9 / 73.3; the same bits.
      float gate[3] = {0.f, 0.f, 0.f};
      if (valid[0]) {
        const bf16_t* wp = p.w + tok[0] * p.w_st + (int64_t)head[0] * p.w_sh;
#pragma unroll
        for (int e = 0; e < 3; e++) gate[e] = 1.f / (1.f + __expf(-(float)wp[e]));
      }
      constexpr int NR = 32 / HRPI;              // rows of a lane
      const int cl = lane % HC;
      int2 th[NR];
      bf16x8 vc[NR][2], vx[NR][2];               // compressed branch; selected or window branch where it is not in registers
#pragma unroll
      for (int k = 0; k < NR; k++) {
        th[k] = row_id(std::integral_constant<int, 0>{}, lane / HC + k * HRPI);
        const int64_t tk = (int64_t)x0 + max(th[k].x, 0), hd = th[k].y;
        const bf16_t* const cp = p.cmp_o + tk * p.co_st + hd * p.co_sh + cl * 8;
        const bool all_of_it = th[k].x + qoff < p.all_below;
        const bf16_t* const xp = all_of_it ? p.o + tk * p.o_st + hd * p.o_sh + cl * 8
                                           : p.slc_o + tk * p.so_st + hd * p.so_sh + cl * 8;
        const bool stored = th[k].x >= 0 && (!all_of_it || th[k].x + qoff > p.window);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          vc[k][h] = th[k].x >= 0 ? ld_global_b128(cp + h * HC * 8) : zero_bf16x8();
          vx[k][h] = stored ? ld_global_b128(xp + h * HC * 8) : zero_bf16x8();
        }
      }
#pragma unroll
      for (int h = 0; h < 2; h++) {
        lds_order();
#pragma unroll
        for (int c8 = h * HC; c8 < (h + 1) * HC; c8++) {
          const int dt = c8 / 4, i = (c8 % 4) * 4;
          *reinterpret_cast<f32x4*>(half_at(l32, c8 - h * HC) + hl * 4) =
              f32x4{oacc[0][dt][i] * inv, oacc[0][dt][i + 1] * inv, oacc[0][dt][i + 2] * inv, oacc[0][dt][i + 3] * inv};
        }
        lds_order();
#pragma unroll
        for (int k = 0; k < NR; k++) {
          const int r = lane / HC + k * HRPI;
          const float s0 = __shfl(gate[0], r, 64), s1 = __shfl(gate[1], r, 64), s2 = __shfl(gate[2], r, 64);
          if (th[k].x < 0) continue;
          const bool all_of_it = th[k].x + qoff < p.all_below, from_o = all_of_it && th[k].x + qoff > p.window;
          const f32x4 x0v = *reinterpret_cast<const f32x4*>(half_at(r, cl));
          const f32x4 x1v = *reinterpret_cast<const f32x4*>(half_at(r, cl) + 4);
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float own = e < 4 ? x0v[e] : x1v[e - 4], other = (float)vx[k][h][e];
            x[e] = (float)vc[k][h][e] * s0 + (all_of_it ? own : other) * s1 + (from_o ? other : own) * s2;
          }
          *reinterpret_cast<bf16x8*>(p.out + ((int64_t)x0 + th[k].x) * p.out_st + (int64_t)th[k].y * p.out_sh + (h * HC + cl) * 8) =
              pack8(x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
        }
      }
    }
  }
}

template <int D, int VD, int MODE, bool PAGED>
int launch_fwd_tile(const NsaFwdTileParams& p0, int B, int max_q_len, hipStream_t stream) {
  if (B <= 0 || max_q_len <= 0) return NSA_OK;
  NsaFwdTileParams p = p0;
  // Queries that select everything see 1 to 24 tiles of keys, the last rows of a short prompt the most: in a launch of few
  // rounds of workgroups the last rows of all sequences and heads go first, so that the longest workgroups start together, on a
  // CU each, and the short ones fill up.  (Last rows first within each sequence and head: the first rows of the second head met
  // those of the first on the same CUs while other CUs had one workgroup.)  Whole calls, that / so, us, 64 / 4 heads of 128: 3
  // prompts of 60 to 700 tokens 79 / 65, 2 of 300 to 900 78 / 68, 6 of 60 to 1000 134 / 125, 16 x 128 to 256 behind up to 256 107 /
  // 105.  Forwards, rows in their order / so, us, by workgroups per CU: sequences of at most all_below (1024) tokens, 64 / 4 heads of
  // 128: 1000 tokens (2.0) 65 / 57, 8 x 600 (9.4) 148 / 145; 32 / 8 heads: 20 x 1000 (20.0) 524 / 419; 16 / 2 of 64: 20 x 1000 (9.8)
  // 122 / 112, 60 x 1000 (29.5) 324 / 322; 16 / 4 of 256: 20 x 1000 (10.0) 929 / 642; of up to twice as many: 64 / 4 of 128: 1500 (2.9)
  // 151 / 139, 2000 (3.9) 209 / 201; 16 / 1: 4 x 2000 (3.9) 208 / 200, 16 x 1100 (8.6) 246 / 235; 16 / 2 of 64: 24 x 100 to 1940 (22.9) 297 /
  // 287, 40 x 17 to 1187 (23.4) 176 / 164.  Not so, there in one round, which has no order to speak of: 16 / 1 of 128: 1500 (0.7) 97 /
  // 99, 2000 (1.0) 100 / 103; not longer sequences, whose longest rows are the first: 3000 (1.5) 119 / 125, 6000 (2.9) 213 / 220, 4 x
  // 1500 to 3000 (5.9) 256 / 261, 32 / 2 of 192: 3000 (2.9) 217 / 228 (64 / 4 heads of 128 alone gain 1 %); not launches of more
  // workgroups, where neighbours' keys stay in L2 with rows in their order: 64 / 4 of 128: 16 x 1100 (34.5) 844 / 866, 20 x 1000 (39.1)
  // 756 / 781, paged 8 x 500 to 2000 (31.3) 703 / 715, with 192 and 256 channels, of whose rows L2 holds fewer, from half as many on: 32 / 2
  // of 192: 8 x 600 (4.7) 100 / 90, 4 x 2000 (7.8) 425 / 418, 16 x 1100 (17.2) 517 / 533, 20 x 1000 (19.5) 442 / 460; 16 / 4 of 256: 24 x
  // 100 to 2000 (23.6) 4376 / 4428.  The compressed branch gains nothing (1500 tokens 205 / 203, 4 x 300 to 1500 156 / 160).
  const int64_t wgs = (int64_t)cdiv_i(max_q_len * p.G, 128) * B * p.KH;
  const int cus = nsa_device_cus();
  const bool all = max_q_len <= p.all_below;
  p.last_first = MODE >= MODE_TAIL && max_q_len / 2 <= p.all_below && wgs <= (D >= 192 ? 16 : all ? 32 : 24) * cus && (all || wgs > cus);
  const int tiles = cdiv_i(max_q_len * p.G, 128);
  const dim3 grid = p.last_first ? dim3(B * p.KH, tiles) : dim3(tiles, B, p.KH);
  // 0 (default): direct-to-LDS staging for the compressed branch with power-of-two head dims (4.5 % faster there; the window
  // branch, with its short key loops, is level with register staging) and for 192 channels everywhere: two of its unpadded
  // tile buffers fill half of a CU's LDS, two padded ones more than that, which leaves one workgroup on a CU.  32 heads of 192,
  // 16K tokens, register staging / so, us: staged forward 1921 / 1640, fused 1925 / 1587, training step 5830 / 5495; 8 x 2K paged
  // queries behind up to 8K 1352 / 1118.  1..4 force one variant for experiments.
  const int variant = nsa_tuning_knob("fwd_variant", 0);
  constexpr bool pow2 = (D == 64 || D == 128) && (VD == 64 || VD == 128);
  auto fits = [](int64_t stride) { return stride >= 0 && stride <= async_row_stride(D, VD); };
  const bool narrow = fits(p.k_sr) && fits(p.v_sr) && (MODE != MODE_ALL || (fits(p.ck_sr) && fits(p.cv_sr)));
  const bool async = narrow && (variant == 4 || (variant == 0 && ((MODE == MODE_CMP && pow2) || D == 192)));
  if constexpr (D > 192 || VD > 128) {
    // head dims of 256: the output accumulators alone take 128 registers, one workgroup per CU
    fwd_tile_kernel<D, VD, MODE, PAGED, 1, 1, false><<<grid, 256, 0, stream>>>(p);
    return nsa_check_launch("fwd_tile_kernel");
  } else if constexpr (MODE >= MODE_TAIL) {
    if constexpr (D == 192) {
      if (variant != 1 && narrow) {
        fwd_tile_kernel<D, VD, MODE, PAGED, 1, 2, true><<<grid, 256, 0, stream>>>(p);
        return nsa_check_launch("fwd_tile_kernel");
      }
    }
    fwd_tile_kernel<D, VD, MODE, PAGED, 1, 2, false><<<grid, 256, 0, stream>>>(p);
  } else if (variant == 2) {
    fwd_tile_kernel<D, VD, MODE, PAGED, 2, 1, false><<<dim3(cdiv_i(max_q_len * p.G, 256), B, p.KH), 256, 0, stream>>>(p);
  } else if (variant == 3) {
    fwd_tile_kernel<D, VD, MODE, PAGED, 1, 1, false><<<grid, 256, 0, stream>>>(p);
  } else if (async) {
    fwd_tile_kernel<D, VD, MODE, PAGED, 1, 2, true><<<grid, 256, 0, stream>>>(p);
  } else {
    fwd_tile_kernel<D, VD, MODE, PAGED, 1, 2, false><<<grid, 256, 0, stream>>>(p);
  }
  return nsa_check_launch("fwd_tile_kernel");
}

template <int MODE, bool PAGED>
int dispatch_fwd_tile(const NsaFwdTileParams& p, int B, int max_q_len, int D, int VD, hipStream_t stream) {
  if (D == 128 && VD == 128) return launch_fwd_tile<128, 128, MODE, PAGED>(p, B, max_q_len, stream);
  if (D == 64 && VD == 64) return launch_fwd_tile<64, 64, MODE, PAGED>(p, B, max_q_len, stream);
  if (D == 192 && VD == 128) return launch_fwd_tile<192, 128, MODE, PAGED>(p, B, max_q_len, stream);
  if constexpr (MODE != MODE_ALL) {
    if (D == 256 && VD == 256) return launch_fwd_tile<256, 256, MODE, PAGED>(p, B, max_q_len, stream);
  }
  if (D == 32 && VD == 32) return launch_fwd_tile<32, 32, MODE, PAGED>(p, B, max_q_len, stream);
  nsa_set_error("attention forward: unsupported head dims D=%d VD=%d (built: 128/128, 64/64, 192/128, 256/256, 32/32)", D, VD);
  return NSA_ERR_UNSUPPORTED;
}

}  // namespace

int nsa_fwd_tile_launch(const NsaFwdTileParams& p, int mode, bool paged, int B, int max_q_len, int D, int VD,
                        hipStream_t stream) {
  if (mode == MODE_CMP) {
    return paged ? dispatch_fwd_tile<MODE_CMP, true>(p, B, max_q_len, D, VD, stream)
                 : dispatch_fwd_tile<MODE_CMP, false>(p, B, max_q_len, D, VD, stream);
  }
  if (mode == MODE_ALL && D == 256) {
    // The branches' pointers do not fit beside 256 channels' accumulators: in one launch 96 to 116 bytes a lane are spilled.  16 / 4 heads,
    // one launch / two, us: 1000 tokens 102 / 96, paged 32 x 1 to 32 behind up to 600 80 / 75, 64 x 100 to 1000 1095 / 1075.
    NsaFwdTileParams c = p;
    c.k = p.ck; c.k_sr = p.ck_sr; c.k_sh = p.ck_sh;
    c.v = p.cv; c.v_sr = p.cv_sr; c.v_sh = p.cv_sh;
    c.table = p.c_table; c.table_stride = p.c_table_stride;
    c.o = p.cmp_o_out; c.o_st = p.co_st; c.o_sh = p.co_sh;
    c.lse = p.cmp_lse; c.lse_st = p.cl_st; c.lse_sh = p.cl_sh;
    const int rc = nsa_fwd_tile_launch(c, MODE_CMP, paged, B, max_q_len, D, VD, stream);
    return rc != NSA_OK ? rc : nsa_fwd_tile_launch(p, MODE_TAIL, paged, B, max_q_len, D, VD, stream);
  }
  if (mode == MODE_ALL) {
    return paged ? dispatch_fwd_tile<MODE_ALL, true>(p, B, max_q_len, D, VD, stream)
                 : dispatch_fwd_tile<MODE_ALL, false>(p, B, max_q_len, D, VD, stream);
  }
  if (mode == MODE_TAIL) {
    return paged ? dispatch_fwd_tile<MODE_TAIL, true>(p, B, max_q_len, D, VD, stream)
                 : dispatch_fwd_tile<MODE_TAIL, false>(p, B, max_q_len, D, VD, stream);
  }
  return paged ? dispatch_fwd_tile<MODE_SWA, true>(p, B, max_q_len, D, VD, stream)
               : dispatch_fwd_tile<MODE_SWA, false>(p, B, max_q_len, D, VD, stream);
}
