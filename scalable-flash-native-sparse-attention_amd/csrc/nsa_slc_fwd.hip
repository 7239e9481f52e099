// Selected-block attention forward: one wave per (query token, kv head); the MFMA M dimension is the group of
// (up to 16) q-heads that share the kv head, N is 16 keys, v_mfma_f32_16x16x32_bf16.
// Upstream: flash_nsa/ops/select_attn.py:21-108 (training), flash_nsa/inference/select_attn.py:21-100 (paged).
//
// The keys of the selected blocks are processed in units of 32.  The K and V rows of a unit are fetched as whole
// coalesced rows (16 lanes x 16 bytes per row) into registers one unit ahead, pass through a wave-private LDS
// region (V: see below), and are read back as MFMA fragments (K row-major, V through ds_read_b64_tr_b16, which delivers the
// key-contraction slices).  Keys are gathered by the per-token block list topk[kh, t, 0 .. min(top_n, t/block+1)).
//
// What bounds it is the gather: 512 KB of rows per token and kv head, from L2 while the keys of the sequences in flight
// fit there (64 heads of 128, 8 x 6K tokens: the CU's address unit is busy 96 % of the cycles, LDS 32 %), else from the
// memory-side cache (64K tokens: 15.3 TB/s of requests, 6.4 of them past L2).  Two units in flight per wave and separate K and V
// regions bought nothing over one, and took the registers and the LDS of a second workgroup per CU at 192 channels: 32 heads,
// 16K tokens 1726 -> 1080 us; 64 heads of 128, 8 x 6K tokens 4207 -> 3920 us.  The rows lie unpadded and swizzled in LDS
// (UnitRows::place): padded by 48 bytes, a quarter of the cycles in which LDS worked were bank conflicts, and the padded offsets
// took registers (14 spilled at 128 channels).  Whole calls, padded / so, us: 64 heads of 128, 64K tokens 18930 / 18590, 16 x 2K
// paged queries 5290 / 5170, 16 heads, 4K tokens 185 / 182.
// With 128 v channels the V rows of all but long sequences do not pass through LDS at all: an instruction fetches the rows whose
// scores its lanes hold, so the transposition stays inside a lane (UnitColumns128).  LDS moves 16 KB per unit instead of 32 (a
// quarter of them transposed reads, the slowest).  This kernel, us, through LDS / so: 64 heads of 128, 8 x 6K tokens 3830 / 3180
// (26 TB/s of requests), 16 x 2K paged queries behind up to 16K 2941 / 2761, one sequence of 4K tokens, 16 heads 105 / 85; 32 heads of
// 192, 16K tokens 964 / 869.  Outputs are the same bits.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include "nsa_units.h"
#include <type_traits>

namespace {

// waves per SIMD the register budget is cut for; at 256 channels two waves with 30 spilled registers beat one without
// (1039 against 1165 us for 16 heads, 16K tokens)
constexpr int slc_waves(int d) { return d <= 64 ? 4 : d <= 128 ? 3 : 2; }

// The probabilities are 31/16 of their value relative to the running maximum (the row sum takes the factor out again).  The
// window branch attends many of the same keys, often behind the same maximum: relative to that alone both branches would
// round P to the same bf16 values, and their errors would add up in the gated sum instead of averaging out.  31/16 keeps
// the largest probabilities where bf16 is finest relative to them, and the maximum's own exact.  Gated sum of separately
// launched branches, relative to 64 bits (16 heads of 128, factor 1 / 31/16): 2.385e-3 / 2.276e-3 at 900 to 1700 tokens,
// 2.449e-3 / 2.434e-3 for tokens 1024 to 4096; the selected branch alone 2.206e-3 / 2.209e-3 there.  Times as before.
constexpr float SLC_P_LOG2 = 0.95419631f;  // log2(31/16)

template <int D, int VD, bool PAGED>
__global__ __launch_bounds__(256, slc_waves(D)) void slc_fwd_kernel(NsaSlcParams p) {
  // Work unit = 32 keys (half of a 64-key tile).  One set of registers holds the rows of the next unit: its K rows are
  // requested when this unit's have gone to LDS, its V rows when this unit's have, which is when the scores are known
  // and the K rows in LDS are no longer needed: K and V take turns in one LDS region.
  constexpr int UK = 32;                      // keys per unit
  constexpr int KC = D / 32;                  // K fragments per 16-key tile
  constexpr bool SWZ = D >= 64 && VD >= 64;    // unpadded rows, chunks swizzled
  constexpr int KLD = SWZ ? D : D + NSA_LDS_PAD, VLD = SWZ ? VD : VD + NSA_LDS_PAD;
  constexpr int LD = KLD > VLD ? KLD : VLD;
  __shared__ __attribute__((aligned(1024))) bf16_t rows_all[4 * UK * LD];
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
  const int nu = nvalid * (Bs / UK);
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
  // Where a head's K and V do not fit the 4 MB of an XCD's L2, the waves that run at the same time should be at the same part
  // of the sequence, whenever they started: `sweep` queries run at once, one starts whenever another ends, so query t starts
  // its way through the blocks at the part of them that the others have reached by then, (t / sweep) mod 1.  Every wave still
  // goes once round, in an order that depends on its position (and, paged, on the launch: walk_together) alone.  64 heads of
  // 128, 64K tokens 10.03 -> 8.97 ms; 32 heads of 192, 16K tokens 1078 -> 1000 us; below that length 1 % slower.
  if (p.sweep > 0 && t > (4 << 20) / ((D + VD) * 2))
    my_blk = rotate_blocks(my_blk, nvalid, lane, (int)((int64_t)(t % p.sweep) * (t / Bs + 1) / p.sweep));

  auto attend = [&](auto vreg_tag) {
    constexpr bool VREG = decltype(vreg_tag)::value;  // V is transposed in registers
    f32x4 oacc[VD / 16];
#pragma unroll
    for (int dt = 0; dt < VD / 16; dt++) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = NSA_NEG_INF, l_run = 0.f;
    const float sc = p.scale_log2;

    // K and V rows are fetched as whole 16-byte-per-lane coalesced rows (every cache line is requested once and used
    // completely) and go through wave-private LDS; the MFMA fragments are read from there.
    using KRows = UnitRows<D>;
    using VRows = std::conditional_t<VREG, UnitColumns128, UnitRows<VD>>;
    uint32_t koff[KRows::PAT], voff[VRows::PAT];
#pragma unroll
    for (int j = 0; j < KRows::PAT; j++) koff[j] = KRows::offset(j, lane, p.k_sr);
#pragma unroll
    for (int j = 0; j < VRows::PAT; j++) voff[j] = VRows::offset(j, lane, p.v_sr);
    KRows kr;
    VRows vr;
    // place in LDS of the lane's piece of instruction j
    int kput[KRows::SPAT], vput[UnitRows<VD>::SPAT];
    if (SWZ) {
#pragma unroll
      for (int j = 0; j < KRows::SPAT; j++) kput[j] = KRows::place(j, lane);
#pragma unroll
      for (int j = 0; j < UnitRows<VD>::SPAT; j++) vput[j] = UnitRows<VD>::place(j, lane);
    }
    const int ksw = KRows::swz(l16), vsw = UnitRows<VD>::swz(kq * 4 + (l16 >> 2));
    UnitList ul;
    // flat row of the first key of unit i (a unit never straddles a page)
    auto flat_row = [&](int i) -> int64_t {
      if (PAGED) return (int64_t)__builtin_amdgcn_readlane(ul.page, i) * p.page_size + __builtin_amdgcn_readlane(ul.off, i);
      return (int64_t)x0 + __builtin_amdgcn_readlane(ul.key0, i);
    };
    // how the rows of a unit are requested: not at all, the unit is known to be full, or with the rows past the causal boundary
    // replaced by the boundary row (masked later) and any stride
    enum { NONE, FULL, ANY };
    auto issue_k = [&](auto how, int i) {
      if constexpr (decltype(how)::value == NONE) return;
      const bf16_t* kb = p.k + flat_row(i) * p.k_sr + (int64_t)kh * p.k_sh;
      if constexpr (decltype(how)::value == FULL) kr.load(kb, p.k_sr, koff);
      else kr.load_clamped(kb, p.k_sr, min(key_last - __builtin_amdgcn_readlane(ul.key0, i), UK - 1));
    };
    auto issue_v = [&](auto how, int i) {
      if constexpr (decltype(how)::value == NONE) return;
      const bf16_t* vb = p.v + flat_row(i) * p.v_sr + (int64_t)kh * p.v_sh;
      if constexpr (decltype(how)::value == FULL) vr.load(vb, p.v_sr, voff);
      else vr.load_clamped(vb, p.v_sr, min(key_last - __builtin_amdgcn_readlane(ul.key0, i), UK - 1));
    };
    auto lds_order = [&]() {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // Unit i, the rows of unit i + 1 being requested meanwhile.  How is fixed per copy of the code: with a branch around the
    // requests the compiler cannot tell this unit's V rows from them and waits for both.  With the unit list in lanes: 64 heads
    // of 128, 8 x 6K tokens 3.85 -> 3.60 ms, paged, 16 x 2K queries behind up to 16K 3.11 -> 3.06 ms; 16 heads, one sequence of
    // 4K tokens 113 -> 109 us; 32 heads of 192, 16K tokens 1072 -> 1043 us.
    auto unit = [&](auto how_next, int i) {
      const int key0 = __builtin_amdgcn_readlane(ul.key0, i);
      if (SWZ) kr.to_lds_swz(rows, kput);
      else kr.to_lds(rows, KLD, lane);
      lds_order();
      issue_k(how_next, i + 1);
      f32x4 sacc[2];
#pragma unroll
      for (int jt = 0; jt < 2; jt++) {
        sacc[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
          const int at = SWZ ? KRows::col(kc * 4, kq ^ (ksw & 3), ksw & ~3) * 8 : kc * 32 + kq * 8;
          sacc[jt] = mfma16(*reinterpret_cast<const bf16x8*>(&rows[(jt * 16 + l16) * KLD + at]), qf[kc], sacc[jt]);
        }
      }
      const int kmax = key_last - key0;  // last usable key offset inside this unit
      if (decltype(how_next)::value != FULL && kmax < UK - 1) {  // wave-uniform: the unit holding the causal boundary
#pragma unroll
        for (int jt = 0; jt < 2; jt++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            int ko = jt * 16 + (lane_id() >> 4) * 4 + i;
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
      const float msc = __builtin_fmaf(m_safe, sc, -SLC_P_LOG2);
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
      // O^T += V^T P^T over the 32 keys of the unit
      const bf16x8 pf = pack8(sacc[0][0], sacc[0][1], sacc[0][2], sacc[0][3], sacc[1][0], sacc[1][1], sacc[1][2], sacc[1][3]);
      if constexpr (VREG) {
        vr.multiply(oacc, pf, std::make_integer_sequence<int, 8>{});
        issue_v(how_next, i + 1);
      } else {
        lds_order();
        if (SWZ) vr.to_lds_swz(rows, vput);
        else vr.to_lds(rows, VLD, lane);
        lds_order();
        issue_v(how_next, i + 1);
        const int kb0 = kq * 4 + (l16 >> 2);
        const int kb1 = kb0 + 16;
#pragma unroll
        for (int dt = 0; dt < VD / 16; dt++) {
          const int col = SWZ ? UnitRows<VD>::col(dt * 2, (l16 & 3) >> 1, vsw) * 8 + (l16 & 1) * 4 : dt * 16 + 4 * (l16 & 3);
          bf16x4 v0 = lds_read_tr(&rows[kb0 * VLD + col]);
          bf16x4 v1 = lds_read_tr(&rows[kb1 * VLD + col]);
          oacc[dt] = mfma16(cat4(v0, v1), pf, oacc[dt]);
        }
      }
      lds_order();
    };
    for (int base = 0; base < nu; base += 64) {
      ul = unit_list<PAGED>(my_blk, nvalid, base, Bs, key_last, table, p.page_size, lane, [](int, int, int) { return 0; });
      if (ul.n == 0) continue;
      const int n_full = p.k_sr < KRows::NARROW && p.v_sr < VRows::NARROW ? ul.n_full : 0;
      int i = 0;
      issue_k(std::integral_constant<int, ANY>{}, 0);
      issue_v(std::integral_constant<int, ANY>{}, 0);
      for (; i + 1 < n_full; i++) unit(std::integral_constant<int, FULL>{}, i);
      for (; i + 1 < ul.n; i++) unit(std::integral_constant<int, ANY>{}, i);
      unit(std::integral_constant<int, NONE>{}, i);
    }

    float l_tot = xrow_sum(l_run);
    l_tot = xhalf_sum(l_tot);
    if (!head_ok) return;
    float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    bf16_t* const op = p.o + tok * p.o_st + (int64_t)head * p.o_sh;
    if constexpr (VREG) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        *reinterpret_cast<bf16x8*>(op + (kq * 4 + i) * 8) =
            pack8(oacc[0][i] * inv, oacc[1][i] * inv, oacc[2][i] * inv, oacc[3][i] * inv, oacc[4][i] * inv, oacc[5][i] * inv,
                  oacc[6][i] * inv, oacc[7][i] * inv);
    } else {
#pragma unroll
      for (int dt = 0; dt < VD / 16; dt++)
        *reinterpret_cast<bf16x4*>(op + kq * 4 + dt * 16) =
            pack4(oacc[dt][0] * inv, oacc[dt][1] * inv, oacc[dt][2] * inv, oacc[dt][3] * inv);
    }
    if (kq == 0 && p.lse != nullptr) {
      p.lse[tok * p.lse_st + (int64_t)head * p.lse_sh] = l_tot > 0.f ? __builtin_fmaf(m_run, sc, -SLC_P_LOG2) + fast_log2(l_tot) : 0.f;
    }
  };
  if constexpr (VD == 128) {
    if (t < p.reg_below) {  // wave-uniform
      attend(std::true_type{});
      return;
    }
  }
  attend(std::false_type{});
}

// Paged: queries far behind their sequence's start are in flight from the launch's first moment on.  The first `sweep` of them
// start together, and so do the next ones, when those end: all are at the same part of the sequence anyhow, until the waves
// have drifted apart, and orders that expect starts spread over a wave's time (above) only spread them.  The wider the head,
// the longer a wave and the later that is.  Chunks shorter than a sweep share it with other sequences and stay close anyhow.
// Prefill calls without / with the rotation, us, contexts of 8K to 16K before the chunk:
//   64 / 4 heads of 128 (sweep 3072): 16 x 256 1144 / 1207, 16 x 1024 3157 / 3646, 16 x 1536 4949 / 5009, 16 x 2048 6351 / 6178,
//     16 x 2560 7971 / 7606, 8 x 2048 3267 / 3238, 4 x 2048 1691 / 1713, 1 x 2048 416 / 449, 5 x 2560 2438 / 2361, 1 x 4096 928 /
//     909, 4 x 8192 7442 / 6625, 16 / 1 heads: 16 x 2048 1523 / 1556, 4 x 4096 917 / 903, 1 x 8192 494 / 483
//   32 / 2 heads of 192 (2048): 16 x 1024 2386 / 2783, 4 x 2048 1285 / 1407, 8 x 2048 2443 / 2623, 2 x 4096 1333 / 1460, 4 x 4096
//     2634 / 2770, 1 x 8192 1464 / 1545, 4 x 8192 6067 / 5827, 1 x 32K from the start 5566 / 5264
//   16 / 2 heads of 64 (4096): 16 x 1024 849 / 926, 16 x 2048 1550 / 1549, 8 x 3072 1262 / 1232, 4 x 3072 646 / 645, 1 x 4096
//     260 / 261, 2 x 3.5K to 5K 540 / 524, 2 x 8192 917 / 865
bool walk_together(int D, int chunk, int64_t queries, int sweep) {
  if (D <= 128 && chunk * 3 >= sweep * 4) return true;
  return chunk * 3 >= sweep * 2 && queries / sweep >= (D <= 64 ? 4 : D <= 128 ? 12 : 24);
}

template <int D, int VD, bool PAGED>
int launch_slc(const NsaSlcParams& p, int B, int max_q_len, hipStream_t stream) {
  if (!PAGED) max_q_len -= p.t_begin;
  if (B <= 0 || max_q_len <= 0) return NSA_OK;
  dim3 grid(cdiv_i(max_q_len, 4), B, p.KH * ((p.G + 15) / 16));
  NsaSlcParams p2 = p;
  const int sweep = nsa_device_cus() * slc_waves(D) * 4;
  const bool together = !PAGED || walk_together(D, max_q_len, (int64_t)max_q_len * grid.y * grid.z, sweep);
  p2.sweep = together ? sweep : 0;
  // V in registers while the sequence fits the L2 of an XCD about one and a half times: LDS is what the gather waits for there.
  // Beyond, memory is, and waves that wait for LDS in turn keep more together: 64K tokens with V in registers everywhere have 11 %
  // more L2 misses.  Calls with V in registers below 0 / 6 / infinitely many MB of K and V per head, us, 64 / 4 heads of 128: one
  // sequence of 8K tokens 1072 / 1012 / 1003, 16K 2489 / 2395 / 2354, 24K 4159 / 4074 / 4136, 32K 6168 / 6060 / 6604, 64K 18988 /
  // 18979 / 19789; paged, 16 x 2K queries behind 2K 4425 / 4295 / 4264, behind 12K 6625 / 6687 / 6998.  64 channels gain nothing (4K
  // to 8K tokens the same to 0.3 %, 16K 550 -> 567).
  // 192 channels, with half of the waves in flight: the line is at 10 MB unpaged.  This launch, us, 32 / 2 heads, 6 / 8 / 10 MB:
  // 12K tokens 544 / 537 / 537, 16K 785 / 774 / 753, 24K 1328 / 1314 / 1313, 48K 4083 / 4075 / 4099, 3 x 16K 2353 / 2294 / 2250; 10 /
  // 12 / 16 MB: 16K 757 / 753 / 758, 24K 1288 / 1295 / 1303, 32K 2033 / 2047 / 2084, 48K 4028 / 4029 / 4096.  64 / 4 heads, 6 / 8 / 10:
  // 16K 1566 / 1543 / 1515, 32K 4026 / 3995 / 3996, 2 x 24K 5381 / 5263 / 5180; 10 / 12 / 16: 24K 2621 / 2648 / 2666, 32K 4004 / 4058 /
  // 4112, 48K 8200 / 8230 / 8310.  Paged, whole calls, 0 / 6 / 10 MB / all, 8 x 2K queries behind 12K 1945 / 1947 / 1971 / 1966, behind
  // 16K 2235 / 2235 / 2234 / 2432.
  p2.reg_below = ((D > 128 && !PAGED ? 10 : 6) << 20) / ((D + VD) * 2);
  slc_fwd_kernel<D, VD, PAGED><<<grid, 256, 0, stream>>>(p2);
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
