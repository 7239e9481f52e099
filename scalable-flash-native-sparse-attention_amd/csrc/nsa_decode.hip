// Paged-KV decode (one query token per request): two fused kernels after the pooling of the newest compressed row.
//   decode_cmp_topk_kernel      compressed attention (o, lse) + block importance + top-n selection
//   decode_slc_swa_kernel       selected-block attention + sliding-window attention + gated combine with the
//                               compressed-branch output -> final o
// Upstream runs this step as 7 launches (flash_nsa/inference/__init__.py:207-257: cmp_attn_decode stage1/2,
// topk_decode probs/select, fused_slc_swa_attn_decode stage1/2, combine_decode).
//
// One workgroup of 8 waves per (request, kv head); the G <= 16 q-heads of the group are the MFMA N dimension
// (v_mfma_f32_16x16x32_bf16, S^T = K Q^T so that softmax statistics are per-lane).  The key range is cut in units
// of 32 keys dealt round-robin to the waves; every wave runs an online softmax over its units with the K
// fragments and V rows of the next unit in flight (register double buffering), and the partial (m, l, o) of the
// waves are merged through LDS.  The step is HBM-bound: every K/V row is read once per pass straight from the
// pool through the block tables.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include <algorithm>
#include <type_traits>
#include "nsa_select.h"
#include "nsa_units.h"

namespace {

constexpr int DEC_WAVES = 8;
// static LDS of decode_slc_swa_kernel (statistics and weights of up to 64 parts of the compressed branch); the host
// adds it to the dynamic size when it decides whether a launch fits the 160 KB of a CU
constexpr size_t SLC_SWA_STATIC_LDS = (3 * 16 + 64 * 16) * sizeof(float);
constexpr int UK = 32;  // keys per unit
constexpr int SEL_INTS = 192;  // LDS words of a selecting wave: 64 selected blocks + candidate list (64 scores, 64 indices)

// Sum of K raw rows from position st on, in row order in fp32: one 16-byte piece (col: its column in the pool).  The row
// at position `given` is not read but taken from given_row (the lane has just stored it).  It stands in front of
// everything else that the workgroup does and is a chain of round trips and of a lone wave's instructions, so the page is
// divided out once (a window of at most a page touches two) and 16 rows are fetched at a time.  One-launch step at which
// every request completes a compressed row, 64 q / 4 kv heads, us, row by row -> so: 16 x 4K 47.5 -> 36.5, 64 x 4K 63 -> 51,
// 512 x 4K 398 -> 329; 64 ragged requests, four of which complete one, 78.8 -> 73.5.
NSA_DEVICE void sum_rows(float (&a)[8], const bf16_t* col, int64_t c_sr, const int32_t* tab, int page, int st, int K,
                         int given, bf16x8 given_row) {
#pragma unroll
  for (int e = 0; e < 8; e++) a[e] = 0.f;
  if (K > page) {
    for (int n = st; n < st + K; n++) {
      bf16x8 x = given_row;
      if (n != given) x = ld_global_b128(col + ((int64_t)tab[n / page] * page + (n % page)) * c_sr);
#pragma unroll
      for (int e = 0; e < 8; e++) a[e] += (float)x[e];
    }
    return;
  }
  const int p0 = st / page, off = st - p0 * page;
  const int64_t row0 = (int64_t)tab[p0] * page + off;
  const int64_t row1 = off + K > page ? (int64_t)tab[p0 + 1] * page + off - page : row0;
  const int skip = given - st;  // < K; negative: none
  constexpr int RB = 16;
  for (int r0 = 0; r0 < K; r0 += RB) {
    bf16x8 x[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) {
      int k = min(r0 + r, K - 1);
      if (k == skip) k = max(k - 1, 0);
      x[r] = ld_global_b128(col + ((off + k < page ? row0 : row1) + k) * c_sr);
    }
#pragma unroll
    for (int r = 0; r < RB; r++)
      if (r0 + r < K) {
        if (r0 + r == skip) x[r] = given_row;
#pragma unroll
        for (int e = 0; e < 8; e++) a[e] += (float)x[r][e];
      }
  }
}

// One wave's flash-attention state over units of 32 keys for the 16 heads of a kv group.
// K and V rows of a unit are fetched as whole rows (16 lanes x 16 bytes per row: every cache line is requested once
// and used completely), held in registers while the previous unit is computed, and pass through one wave-private
// LDS slot: first the K rows (read back as MFMA A fragments), then the V rows (read back transposed; VREG: these do not).
// The un-normalised probabilities exp2((s - m_unit) * c) of every unit can be kept (in LDS, or spilled to scratch
// memory, or both), together with the m_unit they refer to, so that the importance pass needs no second pass over the
// keys: as fp16, or, with 192 channels, as fp32.
// TWO_DEEP: two sets of K / V registers, the next unit is loaded while one is computed.  Otherwise one set, whose K and
// V halves are loaded again as soon as their rows have gone to LDS: half the registers (192 channels do not fit two sets
// into 256), the loads in flight for most of a unit instead of all of it.
// STREAMS: a unit's m_unit is the running maximum of its stream, the units of the wave a fixed step apart; the wave
// walks that many streams in turn.  With two of them (units dealt to four waves instead of eight) the kept values are
// those of the eight-wave kernel.
// KEEP: where kept probabilities go.
constexpr int KEEP_LDS = 0, KEEP_MEM = 1, KEEP_BOTH = 2;
template <int D, int VD, int KEEP = KEEP_LDS, int STREAMS = 1, bool TWO_DEEP = (D <= 128)>
struct UnitFlash {
  using keep_t = std::conditional_t<(D <= 128), _Float16, float>;
  typedef keep_t keep4 __attribute__((ext_vector_type(4)));
  static constexpr int KC = D / 32;
  static constexpr int KJ = (UK * (D / 8)) / 64;
  static constexpr int VJ = (UK * (VD / 8)) / 64;
  // 128 v channels: V is transposed in the lanes' registers (UnitColumns128), the slot takes K alone, and a unit is a shorter
  // chain.  Calls through the slot / so, us: one request of 32K tokens 31.7 / 30.1, 8 of up to 16K with 192 channels 39.7 / 38.9, 64 of
  // 4K to 32K 73.9 / 73.2, 16 of 128K 106.8 / 106.5.  Not with four waves and two workgroups on a CU, which wait for memory: 512 of
  // 4K 330.2 / 331.0.
  static constexpr bool VREG = VD == 128 && STREAMS == 1;
  typedef UnitColumns128 Cols;
  // row of the unit and first channel that V register j of a lane holds
  static NSA_DEVICE int v_row(int j, int lane) { return VREG ? Cols::row(j) + (lane >> 4) * 4 : (lane + j * 64) / (VD / 8); }
  static NSA_DEVICE int v_chunk(int j, int lane) { return VREG ? lane & 15 : (lane + j * 64) % (VD / 8); }
  static constexpr int KLD = D + NSA_LDS_PAD;
  static constexpr int VLD = VD + NSA_LDS_PAD;
  static constexpr int SLOT = UK * (KLD > VLD ? KLD : VLD);  // bf16 elements of a wave's staging slot
  // row stride (floats) of a published partial output [16 heads][OLD]: with VD floats the 16 rows that one
  // 16-byte store instruction writes would all start in the same LDS bank (a 16-way conflict); 4 more floats
  // spread them over all 64 banks
  static constexpr int OLD = VD + 4;
  bf16x8 qf[KC];
  f32x4 oacc[VD / 16];
  float m_run, l_run;
  float sc;
  int l16, kq, lane;
  bf16_t* Ss;          // wave-private staging slot
  keep_t* keep_p;      // LDS [16][keep_ld], the units that start below key keep_lds_end
  keep_t* spill_p;     // memory [units][16][UK] (whole units contiguous), the other units
  float* keep_m;       // [units][16]
  int keep_ld, keep_lds_end;
  int keep_end;        // probabilities of the units that start below this key are kept
  float m_even, m_odd;  // STREAMS 2: running maxima of the stream of the next unit, of the other one

  NSA_DEVICE void init(const bf16_t* qrow, float scale_log2, int lane_, bf16_t* slot) {
    lane = lane_;
    l16 = lane & 15;
    kq = lane >> 4;
    sc = scale_log2;
    Ss = slot;
    keep_p = spill_p = nullptr;
    keep_m = nullptr;
    keep_ld = keep_lds_end = 0;
    keep_end = 0;
    m_even = m_odd = NSA_NEG_INF;
#pragma unroll
    for (int kc = 0; kc < KC; kc++) qf[kc] = ld_global_b128(qrow + kq * 8 + kc * 32);
#pragma unroll
    for (int dt = 0; dt < VD / 16; dt++) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run = NSA_NEG_INF;
    l_run = 0.f;
  }
  // start another branch with the same q fragments
  NSA_DEVICE void reset() {
#pragma unroll
    for (int dt = 0; dt < VD / 16; dt++) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run = NSA_NEG_INF;
    l_run = 0.f;
    keep_end = 0;
  }
  // loads of the unit starting at key0 (wave-uniform); keys outside [klo, khi] are replaced by a clamped key
  // (masked later).  A unit spans at most two pages: the page of its first usable key is looked up once.
  template <bool K = true, bool V = true>
  NSA_DEVICE void issue(int key0, int klo, int khi, const int* tab_s, int page, const bf16_t* kbase, int64_t k_sr,
                        const bf16_t* vbase, int64_t v_sr, bf16x8 (&kf)[KJ], bf16x8 (&vr)[VJ]) {
    const int ks = __builtin_amdgcn_readfirstlane(max(klo, min(key0, khi)));
    const int pi = ks / page;
    const int rem0 = ks - pi * page;
    // (a row of 192 channels is 24 sixteen-byte pieces: three groups of 64 lanes are eight whole rows, so three
    // per-lane offsets that never change)
    constexpr int KP = D / 8, VP = VD / 8;
    constexpr int KG = 64 % KP == 0 ? 1 : KP / 8, VG = 64 % VP == 0 ? 1 : VP / 8;  // groups of 64 lanes per period
    constexpr int KR = 64 * KG / KP, VR = 64 * VG / VP;                            // rows of a period
    static_assert(64 * KG % KP == 0 && 64 * VG % VP == 0 && KJ % KG == 0 && VJ % VG == 0, "");
    {
      // A unit that lies inside [klo, khi] and inside one page (nearly all of them) is UK consecutive pool rows:
      // one wave-uniform row address per group of 64 lanes' rows, and a per-lane byte offset that never changes.
      const int k0 = __builtin_amdgcn_readfirstlane(key0);
      // (the lanes' row offsets inside a period, up to 12 rows with VREG, are 32 bits wide)
      constexpr int64_t V_NARROW = VREG ? Cols::NARROW : 1 << 28;
      if (k0 >= klo && k0 + UK - 1 <= khi && rem0 + UK <= page && k_sr > 0 && v_sr > 0 && k_sr < (1 << 28) &&
          v_sr < V_NARROW) {
        const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane(tab_s[pi]) * page + rem0;
        const char* kp = reinterpret_cast<const char*>(kbase + row0 * k_sr);
        const char* vp = reinterpret_cast<const char*>(vbase + row0 * v_sr);
        uint32_t koff[KG], voff[VG];
#pragma unroll
        for (int g = 0; g < KG; g++)
          koff[g] = (uint32_t)((lane + g * 64) / KP) * (uint32_t)k_sr * 2u + (uint32_t)((lane + g * 64) % KP) * 16u;
#pragma unroll
        for (int g = 0; g < VG; g++)
          voff[g] = (uint32_t)v_row(g, lane) * (uint32_t)v_sr * 2u + (uint32_t)v_chunk(g, lane) * 16u;
#pragma unroll
        for (int j = 0; j < (K ? KJ : 0); j++)
          kf[j] = *reinterpret_cast<const bf16x8*>(kp + (int64_t)(j / KG * KR) * k_sr * 2 + koff[j % KG]);
#pragma unroll
        for (int j = 0; j < (V ? VJ : 0); j++)
          vr[j] = *reinterpret_cast<const bf16x8*>(vp + (int64_t)(VREG ? Cols::row(j) : j / VG * VR) * v_sr * 2 + voff[j % VG]);
        return;
      }
    }
    const int64_t base0 = (int64_t)tab_s[pi] * page;
    const int64_t base1 = (rem0 + UK > page && (int64_t)(pi + 1) * page <= khi) ? (int64_t)tab_s[pi + 1] * page - page : base0;
#pragma unroll
    for (int j = 0; j < (K ? KJ : 0); j++) {
      int pc = lane + j * 64;
      int r = rem0 + max(klo, min(key0 + pc / (D / 8), khi)) - ks;
      int64_t row = (r >= page ? base1 : base0) + r;
      kf[j] = ld_global_b128(kbase + row * k_sr + (pc % (D / 8)) * 8);
    }
#pragma unroll
    for (int j = 0; j < (V ? VJ : 0); j++) {
      int r = rem0 + max(klo, min(key0 + v_row(j, lane), khi)) - ks;
      int64_t row = (r >= page ? base1 : base0) + r;
      vr[j] = ld_global_b128(vbase + row * v_sr + v_chunk(j, lane) * 8);
    }
  }
  // next_k / next_v run as soon as the K / V registers have gone to LDS (they may load the next unit into them)
  // PATCH: row patch_row, that of key khi, is not (or not yet) in the pool, its K pieces are in `patch` of the lanes from 0 on,
  // its V pieces in those of the lanes from 32 on.  issue() has read the pool's row of khi also for every key clamped to it:
  // those V rows are zeroed, since what a slot held before it was first written may be infinite or NaN, which a probability
  // of 0 does not remove (a masked key's scores are replaced, whatever its K row holds).
  template <bool PATCH, class NextK, class NextV>
  NSA_DEVICE void compute(int key0, int klo, int khi, bf16x8 (&kf)[KJ], bf16x8 (&vr)[VJ], NextK next_k, NextV next_v,
                          int patch_row = 0, bf16x8 patch = bf16x8{}) {
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&Ss[(pc / (D / 8)) * KLD + (pc % (D / 8)) * 8]) = kf[j];
    }
    if (PATCH && lane < D / 8) *reinterpret_cast<bf16x8*>(&Ss[patch_row * KLD + lane * 8]) = patch;
    next_k();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    f32x4 sacc[2];
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      sacc[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* kp = &Ss[(jt * 16 + l16) * KLD + kq * 8];
#pragma unroll
      for (int kc = 0; kc < KC; kc++)
        sacc[jt] = mfma16(*reinterpret_cast<const bf16x8*>(kp + kc * 32), qf[kc], sacc[jt]);
    }
    // the K fragments are consumed (LDS operations of a wave complete in order): the slot now takes the V rows
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (PATCH) {
#pragma unroll
      for (int j = 0; j < VJ; j++)
        if (key0 + v_row(j, lane) >= khi || klo >= khi) vr[j] = zero_bf16x8();
      if constexpr (VREG) {
        const u32x4 x = __builtin_bit_cast(u32x4, patch);
        u32x4 mine;
#pragma unroll
        for (int e = 0; e < 4; e++) mine[e] = __shfl(x[e], 32 + l16, 64);
#pragma unroll
        for (int j = 0; j < VJ; j++)
          if (v_row(j, lane) == patch_row) vr[j] = __builtin_bit_cast(bf16x8, mine);
      }
    }
    if constexpr (!VREG) {
#pragma unroll
      for (int j = 0; j < VJ; j++) {
        int pc = lane + j * 64;
        *reinterpret_cast<bf16x8*>(&Ss[(pc / (VD / 8)) * VLD + (pc % (VD / 8)) * 8]) = vr[j];
      }
      if (PATCH && lane >= 32 && lane < 32 + VD / 8)
        *reinterpret_cast<bf16x8*>(&Ss[patch_row * VLD + (lane - 32) * 8]) = patch;
      next_v();
    }
    if (key0 < klo || key0 + UK - 1 > khi) {  // wave-uniform: only boundary units are masked
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          int key = key0 + jt * 16 + kq * 4 + i;
          if (key < klo || key > khi) sacc[jt][i] = NSA_NEG_INF;
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
    auto keep = [&](const f32x4 (&x)[2], float m_unit) {
#pragma unroll
      for (int jt = 0; jt < 2; jt++) {
        const keep4 hv = {(keep_t)x[jt][0], (keep_t)x[jt][1], (keep_t)x[jt][2], (keep_t)x[jt][3]};
        if (KEEP == KEEP_LDS || (KEEP == KEEP_BOTH && key0 < keep_lds_end))
          *reinterpret_cast<keep4*>(&keep_p[l16 * keep_ld + key0 + jt * 16 + kq * 4]) = hv;
        else
          *reinterpret_cast<keep4*>(&spill_p[(key0 / UK) * (16 * UK) + l16 * UK + jt * 16 + kq * 4]) = hv;
      }
      if (kq == 0) keep_m[(key0 / UK) * 16 + l16] = m_unit;
    };
    if (STREAMS == 2 && key0 < keep_end) {  // relative to the stream's maximum
      const float ms = fmaxf(m_even, tmax);
      m_even = m_odd;
      m_odd = ms;
      const float m_unit = ms == NSA_NEG_INF ? 0.f : ms, ksc = m_unit * sc;
      f32x4 x[2];
#pragma unroll
      for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int i = 0; i < 4; i++) x[jt][i] = fast_exp2(__builtin_fmaf(sacc[jt][i], sc, -ksc));
      keep(x, m_unit);
    }
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float pv = fast_exp2(__builtin_fmaf(sacc[jt][i], sc, -msc));
        sacc[jt][i] = pv;
        psum += pv;
      }
    if (STREAMS == 1 && key0 < keep_end) keep(sacc, m_safe);
    if (__builtin_amdgcn_ballot_w64(m_new != m_old) != 0) {
      const float alpha = fast_exp2((m_old - m_safe) * sc);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < VD / 16; dt++) oacc[dt] *= alpha;
    }
    l_run += psum;
    bf16x8 pf = pack8(sacc[0][0], sacc[0][1], sacc[0][2], sacc[0][3], sacc[1][0], sacc[1][1], sacc[1][2], sacc[1][3]);
    if constexpr (VREG) {
      Cols cols;
#pragma unroll
      for (int j = 0; j < VJ; j++) cols.r[j] = vr[j];
      cols.multiply(oacc, pf, std::make_integer_sequence<int, 8>{});
      next_v();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int kb0 = kq * 4 + (l16 >> 2);
      const int kb1 = kb0 + 16;
#pragma unroll
      for (int dt = 0; dt < VD / 16; dt++) {
        const int col = dt * 16 + 4 * (l16 & 3);
        bf16x4 v0 = lds_read_tr(&Ss[kb0 * VLD + col]);
        bf16x4 v1 = lds_read_tr(&Ss[kb1 * VLD + col]);
        oacc[dt] = mfma16(cat4(v0, v1), pf, oacc[dt]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // Loads of the first unit of the next run(), issued early (before a serial section of the kernel that does not
  // touch the staging slot) so that their latency is hidden behind it; the next run() must be called with the same
  // arguments.
  bf16x8 pre_k[KJ], pre_v[VJ];
  int pre_key;
  template <class KeyFn>
  NSA_DEVICE void prefetch(int first, int nu, int klo, int khi, KeyFn key0_of, const int* tab_s, int page,
                           const bf16_t* kbase, int64_t k_sr, const bf16_t* vbase, int64_t v_sr) {
    if (first < nu) { pre_key = key0_of(first); issue(pre_key, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, pre_k, pre_v); }
  }
  // pipelined loop over units u = first, first+step, ... < nu ; key0_of(u) gives the unit's first key
  // USE_PRE: the first unit was fetched by prefetch() with the same arguments.  Only the call that consumes the
  // prefetched registers is instantiated with it, so that they are dead everywhere else.
  template <bool USE_PRE = false, class KeyFn>
  NSA_DEVICE void run(int first, int step, int nu, int klo, int khi, KeyFn key0_of, const int* tab_s, int page,
                      const bf16_t* kbase, int64_t k_sr, const bf16_t* vbase, int64_t v_sr) {
    if constexpr (!TWO_DEEP) {
      static_assert(!USE_PRE, "");
      bf16x8 kf[KJ], vr[VJ];
      if (first >= nu) return;
      int key = key0_of(first);
      issue(key, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kf, vr);
      for (int u = first; u < nu; u += step) {
        const bool more = u + step < nu;
        const int nxt = more ? key0_of(u + step) : 0;
        compute<false>(
            key, klo, khi, kf, vr,
            [&]() { if (more) issue<true, false>(nxt, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kf, vr); },
            [&]() { if (more) issue<false, true>(nxt, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kf, vr); });
        key = nxt;
      }
      return;
    } else {
    auto none = []() {};
    bf16x8 kfA[KJ], kfB[KJ], vrA[VJ], vrB[VJ];
    int keyA = 0, keyB = 0;
    if (USE_PRE) {
      keyA = pre_key;
#pragma unroll
      for (int j = 0; j < KJ; j++) kfA[j] = pre_k[j];
#pragma unroll
      for (int j = 0; j < VJ; j++) vrA[j] = pre_v[j];
    } else if (first < nu) {
      keyA = key0_of(first);
      issue(keyA, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kfA, vrA);
    }
    for (int u = first; u < nu; u += 2 * step) {
      const bool hasB = u + step < nu;
      if (hasB) { keyB = key0_of(u + step); issue(keyB, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kfB, vrB); }
      compute<false>(keyA, klo, khi, kfA, vrA, none, none);
      if (hasB) {
        if (u + 2 * step < nu) {
          keyA = key0_of(u + 2 * step);
          issue(keyA, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kfA, vrA);
        }
        compute<false>(keyB, klo, khi, kfB, vrB, none, none);
      }
    }
    }
  }
  // One unit, one row of which row_of() returns: called when the unit's rows have been requested (attend: the row belongs to
  // the unit).  Apart from run(): inside its loop the exchange of a row costs every unit (16 x 128K 106.4 -> 108.6 us).
  template <class RowFn>
  NSA_DEVICE void run_patched(bool attend, int key, int klo, int khi, const int* tab_s, int page, const bf16_t* kbase,
                              int64_t k_sr, const bf16_t* vbase, int64_t v_sr, int patch_row, RowFn row_of) {
    bf16x8 kf[KJ], vr[VJ];
    if (attend) issue(key, klo, khi, tab_s, page, kbase, k_sr, vbase, v_sr, kf, vr);
    const bf16x8 patch = row_of();
    auto none = []() {};
    if (attend) compute<true>(key, klo, khi, kf, vr, none, none, patch_row, patch);
  }
  // wave partial -> LDS slot: m (raw units), l, o[16 heads][VD]
  NSA_DEVICE void publish(float* pm, float* pl, float* po) {
    float l_tot = xrow_sum(l_run);
    l_tot = xhalf_sum(l_tot);
    if (kq == 0) { pm[l16] = m_run; pl[l16] = l_tot; }
    if constexpr (VREG) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          *reinterpret_cast<f32x4*>(&po[l16 * OLD + (kq * 4 + i) * 8 + h * 4]) =
              f32x4{oacc[h * 4][i], oacc[h * 4 + 1][i], oacc[h * 4 + 2][i], oacc[h * 4 + 3][i]};
    } else {
#pragma unroll
      for (int dt = 0; dt < VD / 16; dt++)
        *reinterpret_cast<f32x4*>(&po[l16 * OLD + dt * 16 + kq * 4]) = oacc[dt];
    }
  }
};

// Merge of n wave partials (m in raw score units, l, un-normalised o) in two steps, so that the exponentials are
// evaluated once per (part, head) and not once per output channel:
//   merge_weights: one thread per head turns the l of every part into its normalised weight
//                  exp2((m_part - m) * c) / l_total, in place, and returns lse2 (0 when nothing was visible);
//   merge_value:   after a barrier, o[head][d] = sum over parts of weight * o_part.
NSA_DEVICE float merge_weights(const float* pm, float* pl, int nparts, int part_stride_ml, int head, float sc) {
  float m = NSA_NEG_INF;
  for (int w = 0; w < nparts; w++) m = fmaxf(m, pm[w * part_stride_ml + head]);
  if (m == NSA_NEG_INF) {
    for (int w = 0; w < nparts; w++) pl[w * part_stride_ml + head] = 0.f;
    return 0.f;
  }
  float l = 0.f;
  for (int w = 0; w < nparts; w++) {
    const float mw = pm[w * part_stride_ml + head];
    const float a = (mw == NSA_NEG_INF) ? 0.f : fast_exp2((mw - m) * sc);
    l += a * pl[w * part_stride_ml + head];
    pl[w * part_stride_ml + head] = a;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  for (int w = 0; w < nparts; w++) pl[w * part_stride_ml + head] *= inv;
  return l > 0.f ? m * sc + fast_log2(l) : 0.f;
}
NSA_DEVICE float merge_value(const float* wgt, const float* po, int nparts, int part_stride_ml, int part_stride_o,
                             int head, int d, int row_ld) {
  float o = 0.f;
  for (int w = 0; w < nparts; w++) o += wgt[w * part_stride_ml + head] * po[w * part_stride_o + head * row_ld + d];
  return o;
}

// four consecutive channels at once (16-byte LDS reads; same summation order over the parts as merge_value)
NSA_DEVICE f32x4 merge_value4(const float* wgt, const float* po, int nparts, int part_stride_ml, int part_stride_o,
                              int head, int d, int row_ld) {
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int w = 0; w < nparts; w++) {
    const float a = wgt[w * part_stride_ml + head];
    const f32x4 x = *reinterpret_cast<const f32x4*>(&po[w * part_stride_o + head * row_ld + d]);
    o[0] += a * x[0]; o[1] += a * x[1]; o[2] += a * x[2]; o[3] += a * x[3];
  }
  return o;
}
// The same merge without the shared weights: every thread evaluates the weights of its own head in registers
// (the same operations in the same order as merge_weights, so the results are bit-identical) -- 2 * NP broadcast
// LDS reads and NP exponentials per thread buy one barrier and a serial 16-thread step less.
template <int NP>
NSA_DEVICE float merge_weights_local(const float* pm, const float* pl, int part_stride_ml, int head, float sc,
                                     float (&wgt)[NP]) {
  float mw[NP];
  float m = NSA_NEG_INF;
#pragma unroll
  for (int w = 0; w < NP; w++) { mw[w] = pm[w * part_stride_ml + head]; m = fmaxf(m, mw[w]); }
  if (m == NSA_NEG_INF) {
#pragma unroll
    for (int w = 0; w < NP; w++) wgt[w] = 0.f;
    return 0.f;
  }
  float l = 0.f;
#pragma unroll
  for (int w = 0; w < NP; w++) {
    const float a = (mw[w] == NSA_NEG_INF) ? 0.f : fast_exp2((mw[w] - m) * sc);
    l += a * pl[w * part_stride_ml + head];
    wgt[w] = a;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int w = 0; w < NP; w++) wgt[w] *= inv;
  return l > 0.f ? m * sc + fast_log2(l) : 0.f;
}
template <int NP>
NSA_DEVICE f32x4 merge_value4_local(const float (&wgt)[NP], const float* po, int part_stride_o, int head, int d, int row_ld) {
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NP; w++) {
    const float a = wgt[w];
    const f32x4 x = *reinterpret_cast<const f32x4*>(&po[w * part_stride_o + head * row_ld + d]);
    o[0] += a * x[0]; o[1] += a * x[1]; o[2] += a * x[2]; o[3] += a * x[3];
  }
  return o;
}
NSA_DEVICE f32x4 round_bf16x4(f32x4 x) {
  return f32x4{(float)(bf16_t)x[0], (float)(bf16_t)x[1], (float)(bf16_t)x[2], (float)(bf16_t)x[3]};
}

// head-summed probabilities of the compressed keys -> scores of the selection blocks (ascending key order per
// block); all threads of the workgroup
NSA_DEVICE void fold_block_scores(const float* pg, float* imp, int y, int nb, int nb_cap, const NsaDecodeParams& p,
                                  int tid, int nthreads) {
  // stride is a power of two and divides kernel_size and block_size: block j covers the compressed keys
  // j*Bs/St - Kz/St + 1 + r, r = 0 .. (Bs+Kz-St)/St - 1, with overlap area (in positions) / St as the weight
  const int Bs = p.block_size, Kz = p.kernel_size, St = p.stride;
  const int bps = Bs / St, kps = Kz / St;
  const int nloops = bps + kps - 1;
  const float inv_st = 1.f / (float)St;
  for (int j = tid; j < nb_cap; j += nthreads) {
    float acc = 0.f;
    if (j < nb) {
      const int i0 = j * bps - kps + 1;
      int cs = St - Kz;
      for (int r = 0; r < nloops; r++, cs += St) {
        const int i = i0 + r;
        if (i >= 0 && i < y) {
          const int area = min(cs + Kz, Bs) - max(cs, 0);
          acc += pg[i] * ((float)area * inv_st);
        }
      }
    }
    imp[j] = acc;
  }
}

// more than 2048 blocks: the same selection with the scores rescanned in LDS every round (taken scores are
// overwritten with -1)
NSA_DEVICE int select_blocks_lds(float* imp, int t, int nb_cap, const NsaDecodeParams& p, int lane) {
  const int nk = t >= 0 ? t / p.block_size : -1;
  int result = p.ignore_index;
  if (lane == 0) {
    for (int s = 0; s < p.num_init; s++)
      if (s < nb_cap) imp[s] = -1.f;
    for (int i = 0; i < p.num_local; i++)
      if (nk - i >= 0 && nk - i < nb_cap) imp[nk - i] = -1.f;
  }
  if (lane < p.num_init) {
    if (lane <= nk) result = lane;
  } else if (lane < p.num_init + p.num_local) {
    if (lane <= nk) result = nk - (lane - p.num_init);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int nsel = min(p.top_n, nk + 1);
  const int jmax = min(nk, nb_cap - 1);
  for (int slot = p.num_init + p.num_local; slot < nsel; slot++) {
    float best = -2.f;
    int bj = 0x7fffffff;
    for (int j = lane; j <= jmax; j += 64) {
      float v = imp[j];
      if (v > best) { best = v; bj = j; }
    }
    bj = wave_argmax_lowest(best, bj, bj != 0x7fffffff);
    if (lane == slot) result = bj;
    if (lane == 0 && bj <= jmax) imp[bj] = -1.f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  return result;
}

// cand_v / cand_i: 64 floats (16-byte aligned) + 64 ints of LDS private to the selecting wave
template <bool SHORT_CODE>
NSA_DEVICE int select_blocks_wave(float* imp, int t, int nb_cap, const NsaDecodeParams& p, int lane, float* cand_v,
                                  int* cand_i) {
  if (nb_cap <= 512) return select_blocks_short_list<SHORT_CODE, 8>(imp, t, nb_cap, p, lane, cand_v, cand_i);
  if (nb_cap <= 1024) return select_blocks_short_list<SHORT_CODE, 16>(imp, t, nb_cap, p, lane, cand_v, cand_i);
  if (nb_cap <= 2048) return select_blocks_short_list<SHORT_CODE, 32>(imp, t, nb_cap, p, lane, cand_v, cand_i);
  return select_blocks_lds(imp, t, nb_cap, p, lane);
}

template <int D, int VD, bool KEEP>
__global__ __launch_bounds__(DEC_WAVES * 64) void decode_cmp_topk_kernel(NsaDecodeParams p) {
  using UF = UnitFlash<D, VD>;
  constexpr int NW = DEC_WAVES;
  // dynamic LDS: [staging slot per wave (reused for the wave's partial o, then for pg)] [m][l][lse] [imp] [table]
  //              KEEP: [un-normalised p, fp16 [16][keep_ld]] [m of every unit [units][16]]
  //              else: [pg]
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_raw[];
  constexpr int SLOT = UF::SLOT;
  static_assert(SLOT * 2 >= 16 * UF::OLD * 4, "a wave's slot must hold its partial output");
  bf16_t* Vs_all = reinterpret_cast<bf16_t*>(dyn_raw);
  float* part_m = reinterpret_cast<float*>(dyn_raw + (size_t)NW * SLOT * 2);
  float* part_l = part_m + NW * 16;
  float* lse_s = part_l + NW * 16;
  float* imp = lse_s + 16;
  int* tab_s = reinterpret_cast<int*>(imp + p.nb_cap);  // the request's compressed-row page table
  const int ntab = (p.y_cap + p.page_size - 1) / p.page_size;
  const int n_units_cap = (p.y_cap + UK - 1) / UK;
  const int keep_ld = n_units_cap * UK + 8;  // +8 halves: the 16 head rows start in different banks
  float* after_tab = reinterpret_cast<float*>(tab_s + ((ntab + 3) & ~3));
  float* keep_m = after_tab;                                               // KEEP
  using keep_t = typename UF::keep_t;
  keep_t* keep_p = reinterpret_cast<keep_t*>(keep_m + n_units_cap * 16);  // KEEP
  float* pg = KEEP ? reinterpret_cast<float*>(dyn_raw) : after_tab;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, kh = blockIdx.y;
  const int G = p.G;
  const int L = p.ctx_lens[b];
  const int t = L - 1;
  const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
  const int nb = min(L > 0 ? (L - 1) / p.block_size + 1 : 0, p.nb_cap);
  const int32_t* ctab = p.cmp_table + (int64_t)b * p.cmp_table_stride;
  const int page = p.page_size;
  // page-table entries go to LDS first: a table lookup in global memory in front of every gather would serialise
  // the pipelined K/V loads behind it (memory operations of a wave retire in order)
  for (int i = tid; i < (y + page - 1) / page; i += NW * 64) tab_s[i] = ctab[i];
  __syncthreads();
  const bf16_t* kbase = p.k + (int64_t)kh * p.k_sh;
  const bf16_t* vbase = p.v + (int64_t)kh * p.v_sh;
  const int l16 = lane & 15, kq = lane >> 4;
  const int g = min(l16, G - 1);
  const int head = kh * G + g;

  UF uf;
  uf.init(p.q + (int64_t)b * p.q_st + (int64_t)head * p.q_sh, p.scale_log2, lane, Vs_all + wave * SLOT);
  if (KEEP) {
    uf.keep_p = keep_p;
    uf.keep_m = keep_m;
    uf.keep_ld = keep_ld;
    uf.keep_end = uf.keep_lds_end = y;
  }
  const int nu = (y + UK - 1) / UK;

  // ---- phase A: compressed attention, units dealt round-robin to the waves ----
  uf.run(wave, NW, nu, 0, y - 1, [&](int u) { return u * UK; }, tab_s, page, kbase, p.k_sr, vbase, p.v_sr);
  uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(Vs_all + wave * SLOT));
  __syncthreads();
  if (tid < 16) {
    const float lse2 = merge_weights(part_m, part_l, NW, 16, tid, p.scale_log2);
    lse_s[tid] = tid < G ? lse2 : 0.f;
    if (tid < G && p.lse_out) p.lse_out[(int64_t)b * p.lse_st + (kh * G + tid) * p.lse_sh] = lse2;
  }
  __syncthreads();
  for (int idx = tid; idx < G * VD; idx += NW * 64) {
    int h = idx / VD, d = idx - h * VD;
    float o = merge_value(part_l, reinterpret_cast<const float*>(Vs_all), NW, 16, SLOT / 2, h, d, UF::OLD);
    p.cmp_o[(int64_t)b * p.co_st + (int64_t)(kh * G + h) * p.co_sh + d] = (bf16_t)o;
  }
  __syncthreads();

  // ---- phase B: p = exp2(s*c - lse) summed over the heads of the group, per compressed key ----
  if (KEEP) {
    // p = kept exp2((s - m_unit)*c) * exp2(m_unit*c - lse): turn the m table into these factors, then one thread per key
    for (int i = tid; i < nu * 16; i += NW * 64) {
      int h = i & 15;
      keep_m[i] = h < G ? fast_exp2(__builtin_fmaf(keep_m[i], p.scale_log2, -lse_s[h])) : 0.f;
    }
    __syncthreads();
    for (int key = tid; key < y; key += NW * 64) {
      const float* fac = keep_m + (key / UK) * 16;
      float acc = 0.f;
#pragma unroll
      for (int h = 0; h < 16; h++) acc += (float)keep_p[h * keep_ld + key] * fac[h];
      pg[key] = acc;
    }
  } else {
    // second pass over the compressed keys: S[head][key] = Q K^T, lane holds key = l16, heads kq*4 .. +3
    auto row_of = [&](int key) -> int64_t { return (int64_t)tab_s[key / page] * page + (key % page); };
    float lse4[4];
#pragma unroll
    for (int i = 0; i < 4; i++) lse4[i] = lse_s[kq * 4 + i];
    bf16x8 kf[2][UF::KC];
    for (int u = wave; u < nu; u += NW) {
      const int key0 = u * UK;
#pragma unroll
      for (int jt = 0; jt < 2; jt++) {
        int key = min(key0 + jt * 16 + l16, y - 1);
        const bf16_t* kp = kbase + row_of(key) * p.k_sr + kq * 8;
#pragma unroll
        for (int kc = 0; kc < UF::KC; kc++) kf[jt][kc] = ld_global_b128(kp + kc * 32);
      }
#pragma unroll
      for (int jt = 0; jt < 2; jt++) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < UF::KC; kc++) s = mfma16(uf.qf[kc], kf[jt][kc], s);
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (kq * 4 + i < G) acc += fast_exp2(__builtin_fmaf(s[i], p.scale_log2, -lse4[i]));
        acc = xrow_sum(acc);
        acc = xhalf_sum(acc);
        int key = key0 + jt * 16 + l16;
        if (kq == 0 && key < y) pg[key] = acc;
      }
    }
  }
  __syncthreads();
  fold_block_scores(pg, imp, y, nb, p.nb_cap, p, tid, NW * 64);
  __syncthreads();
  if (wave != 0) return;
  // the waves' partial statistics are consumed: their space is the selector's candidate list
  const int result = select_blocks_wave<false>(imp, t, p.nb_cap, p, lane, part_m, reinterpret_cast<int*>(part_l));
  if (lane < p.top_n) p.topk[(int64_t)kh * p.tk_sh + (int64_t)b * p.tk_st + lane] = result;
}

// ---- split variant of the compressed branch: requests are cut in NSPLIT key-interleaved parts so that long
// contexts do not leave most CUs idle; partial (m, l, o) go through a small fp32 scratch in global memory.
constexpr int SPLIT_WAVES = 4;
// scratch of the caller: float-aligned
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// grid (B, KH, nsplit + win_parts): compressed attention over the units u = s*4 + wave (mod 4*nsplit); the last win_parts
// parts of a pair attend the window in the same way, which needs nothing from the block selection and so stays out of
// the second launch (0 / 1 / 2 / 3 / 4 parts, both launches: 1 x 32K 38.2 / 39.3 / 37.5 / 36.8 / 37.0 us, 16 x 128K
// 99.9 / 98.0 / 97.7 / 97.8 / 99.9).  Two workgroups per CU, or the window's would wait for a CU.
// STORE: the caller passes the newest token's row.  (A kernel of its own: the launch is short, and the code that it does not
// need costs the others 0.6 us.)
template <int D, int VD, bool STORE>
__global__ __launch_bounds__(SPLIT_WAVES * 64, 2) void decode_cmp_partial_kernel(NsaDecodeParams p) {
  using UF = UnitFlash<D, VD, KEEP_MEM>;
  constexpr int NW = SPLIT_WAVES;
  constexpr int SLOT = UF::SLOT;
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_raw[];
  bf16_t* Vs_all = reinterpret_cast<bf16_t*>(dyn_raw);
  float* part_m = reinterpret_cast<float*>(dyn_raw + (size_t)NW * SLOT * 2);
  float* part_l = part_m + NW * 16;
  int* tab_s = reinterpret_cast<int*>(part_l + NW * 16);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, kh = blockIdx.y, sp = blockIdx.z;
  const int nsplit = gridDim.z - p.win_parts;
  const bool in_window = sp >= nsplit;  // workgroup-uniform
  const int G = p.G;
  const int L = p.ctx_lens[b];
  const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
  const int32_t* ctab = p.cmp_table + (int64_t)b * p.cmp_table_stride;
  const int page = p.page_size;
  const int t = L - 1;
  const int klo = in_window ? max(0, t - p.window) : 0;
  const int khi = in_window ? t : y - 1;
  const int page0 = klo / page;  // tab_s: pages of the keys klo .. khi
  if (in_window) ctab = p.table + (int64_t)b * p.table_stride;
  for (int i = page0 + tid; i <= (khi < 0 ? -1 : khi / page); i += NW * 64) tab_s[i - page0] = ctab[i];
  // The newest token's row (upstream store_kvcache) is written by the wave that owns the window's
  // last unit, which attends it from its registers; nobody else reads it in this launch (8 requests with 192 channels, 42.6
  // us with a launch of its own in front, 39.5 so).  in_place: the block table has the caller's slot for it, else the
  // table's row is what is attended.
  const int new_slot = STORE ? p.raw_slots[b] : -1;
  const bool newest_in_place =
      STORE && new_slot >= 0 && t >= 0 && (int64_t)p.table[(int64_t)b * p.table_stride + t / page] * page + t % page == new_slot;
  // The compressed row that the newest token completes (mean of the last kernel_size raw rows, fp32 sums in row
  // order like nsa_paged_pool_decode; flash_nsa/inference/compress_kv.py:253-287 upstream) is written by the part
  // that attends it -- the one whose waves own the last unit -- wave 0 for K and wave 1 for V, one 16-byte piece per
  // lane.  Only this workgroup reads it back in this launch, so a workgroup-scope release and the barrier suffice.
  {
    const int cmp_slot = p.cmp_slots != nullptr ? p.cmp_slots[b] : -1;
    const int last_unit = y > 0 ? (y - 1) / UK : 0;
    if (cmp_slot >= 0 && L >= p.kernel_size && sp == (last_unit % (NW * nsplit)) / NW && wave < 2) {
      bf16_t* cache = const_cast<bf16_t*>(wave == 0 ? p.k : p.v);
      const int64_t c_sr = wave == 0 ? p.k_sr : p.v_sr, c_sh = wave == 0 ? p.k_sh : p.v_sh;
      if (lane < (wave == 0 ? D : VD) / 8) {
        const int32_t* tab = p.table + (int64_t)b * p.table_stride;
        const int st = ((L - p.kernel_size) / p.stride) * p.stride;
        float a[8];
        bf16x8 newest = zero_bf16x8();
        if (newest_in_place)
          newest = ld_global_b128((wave == 0 ? p.new_k + (int64_t)b * p.nk_st + (int64_t)kh * p.nk_sh
                                             : p.new_v + (int64_t)b * p.nv_st + (int64_t)kh * p.nv_sh) + lane * 8);
        sum_rows(a, cache + (int64_t)kh * c_sh + lane * 8, c_sr, tab, page, st, p.kernel_size, newest_in_place ? t : -1, newest);
        const float inv = 1.f / (float)p.kernel_size;
        *reinterpret_cast<bf16x8*>(cache + (int64_t)cmp_slot * c_sr + (int64_t)kh * c_sh + lane * 8) =
            pack8(a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv, a[4] * inv, a[5] * inv, a[6] * inv, a[7] * inv);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    }
  }
  __syncthreads();
  const bf16_t* kbase = p.k + (int64_t)kh * p.k_sh;
  const bf16_t* vbase = p.v + (int64_t)kh * p.v_sh;
  const int l16 = lane & 15;
  const int head = kh * G + min(l16, G - 1);

  UF uf;
  uf.init(p.q + (int64_t)b * p.q_st + (int64_t)head * p.q_sh, p.scale_log2, lane, Vs_all + wave * SLOT);
  if (p.sp_keep_p != nullptr && !in_window) {  // spill the un-normalised probabilities of every unit for the final kernel
    const int nuc = (p.y_cap + UK - 1) / UK;
    // unit-major: a wave writes the 1 KB of a unit as whole cache lines
    uf.spill_p = (typename UF::keep_t*)p.sp_keep_p + ((int64_t)b * p.KH + kh) * 16 * nuc * UK;
    uf.keep_m = p.sp_keep_m + ((int64_t)b * p.KH + kh) * nuc * 16;
    uf.keep_end = y;
  }
  const int k0 = (klo / UK) * UK;
  const int nu = khi < 0 ? 0 : (khi - k0) / UK + 1;
  const int first = in_window ? (sp - nsplit) * NW + wave : sp * NW + wave;
  const int key_base = page0 * page;  // keys are counted from the first page in tab_s (a multiple of UK)
  auto key0_of = [&](int u) { return k0 - key_base + u * UK; };
  const int step = NW * (in_window ? p.win_parts : nsplit);
  const int last = max(nu - 1, 0);
  const bool new_here = STORE && in_window && new_slot >= 0 && first == last % step;
  uf.run(first, step, new_here && newest_in_place ? last : nu, klo - key_base, khi - key_base, key0_of, tab_s, page, kbase,
         p.k_sr, vbase, p.v_sr);
  if (new_here)
    uf.run_patched(newest_in_place, key0_of(last), klo - key_base, khi - key_base, tab_s, page, kbase, p.k_sr, vbase, p.v_sr,
                   khi - key_base - key0_of(last), [&]() {  // K in the lanes from 0 on, V in the lanes from 32 on
                     const bool of_v = lane >= 32;
                     const int c = (lane & 31) * 8;
                     bf16x8 row = zero_bf16x8();
                     if (c < (of_v ? VD : D)) {
                       row = ld_global_b128((of_v ? p.new_v + (int64_t)b * p.nv_st + (int64_t)kh * p.nv_sh
                                                  : p.new_k + (int64_t)b * p.nk_st + (int64_t)kh * p.nk_sh) + c);
                       bf16_t* const cache = const_cast<bf16_t*>(of_v ? p.v : p.k) + (int64_t)kh * (of_v ? p.v_sh : p.k_sh);
                       *reinterpret_cast<bf16x8*>(cache + (int64_t)new_slot * (of_v ? p.v_sr : p.k_sr) + c) = row;
                     }
                     return row;
                   });
  uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(Vs_all + wave * SLOT));
  __syncthreads();
  // merge the 4 waves; store the part's un-normalised partial
  const int64_t pair = (int64_t)b * p.KH + kh;
  const int64_t base = (in_window ? pair * p.win_parts + (sp - nsplit) : pair * nsplit + sp) * 16;
  float* const m_dst = (in_window ? p.win_m : p.sp_m) + base;
  float* const l_dst = (in_window ? p.win_l : p.sp_l) + base;
  float* const o_dst = (in_window ? p.win_o : p.sp_o) + base * VD;
  const float* po = reinterpret_cast<const float*>(Vs_all);
  for (int idx = tid * 4; idx < 16 * VD; idx += NW * 64 * 4) {
    const int h = idx / VD, d = idx - h * VD;
    float m = NSA_NEG_INF;
    for (int w = 0; w < NW; w++) m = fmaxf(m, part_m[w * 16 + h]);
    float l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (m != NSA_NEG_INF) {
      for (int w = 0; w < NW; w++) {
        const float mw = part_m[w * 16 + h];
        const float a = (mw == NSA_NEG_INF) ? 0.f : fast_exp2((mw - m) * p.scale_log2);
        l += a * part_l[w * 16 + h];
        o += a * *reinterpret_cast<const f32x4*>(&po[w * (SLOT / 2) + h * UF::OLD + d]);
      }
    }
    *reinterpret_cast<f32x4u*>(o_dst + idx) = o;
    if (d == 0) { m_dst[h] = m; l_dst[h] = l; }
  }
}

// grid (B, KH, nsplit): merge the splits (lse; split 0 also writes cmp_o), then the head-summed probabilities of
// this split's compressed keys -> pg [B, KH, y_cap] fp32
template <int D, int VD>
__global__ __launch_bounds__(SPLIT_WAVES * 64) void decode_importance_kernel(NsaDecodeParams p) {
  constexpr int NW = SPLIT_WAVES;
  constexpr int KC = D / 32;
  __shared__ float lse_s[16];
  __shared__ float m_s[16], l_s[16];
  extern __shared__ int tab_dyn[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, kh = blockIdx.y, sp = blockIdx.z;
  const int nsplit = gridDim.z;
  const int G = p.G;
  const int L = p.ctx_lens[b];
  const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
  const int32_t* ctab = p.cmp_table + (int64_t)b * p.cmp_table_stride;
  const int page = p.page_size;
  for (int i = tid; i < (y + page - 1) / page; i += NW * 64) tab_dyn[i] = ctab[i];
  const int64_t base = ((int64_t)b * p.KH + kh) * nsplit * 16;
  if (tid < 16) {
    float m = NSA_NEG_INF;
    for (int s2 = 0; s2 < nsplit; s2++) m = fmaxf(m, p.sp_m[base + s2 * 16 + tid]);
    float l = 0.f;
    if (m != NSA_NEG_INF)
      for (int s2 = 0; s2 < nsplit; s2++) {
        float ms = p.sp_m[base + s2 * 16 + tid];
        if (ms != NSA_NEG_INF) l += fast_exp2((ms - m) * p.scale_log2) * p.sp_l[base + s2 * 16 + tid];
      }
    m_s[tid] = m;
    l_s[tid] = l;
    float lse2 = (m != NSA_NEG_INF && l > 0.f) ? m * p.scale_log2 + fast_log2(l) : 0.f;
    lse_s[tid] = lse2;
    if (sp == 0 && tid < G && p.lse_out) p.lse_out[(int64_t)b * p.lse_st + (kh * G + tid) * p.lse_sh] = lse2;
  }
  __syncthreads();
  if (sp == 0) {
    for (int idx = tid; idx < G * VD; idx += NW * 64) {
      int h = idx / VD, d = idx - h * VD;
      float m = m_s[h], l = l_s[h], o = 0.f;
      if (m != NSA_NEG_INF && l > 0.f) {
        for (int s2 = 0; s2 < nsplit; s2++) {
          float ms = p.sp_m[base + s2 * 16 + h];
          if (ms != NSA_NEG_INF) o += fast_exp2((ms - m) * p.scale_log2) * p.sp_o[(base + s2 * 16 + h) * VD + d];
        }
        o /= l;
      }
      p.cmp_o[(int64_t)b * p.co_st + (int64_t)(kh * G + h) * p.co_sh + d] = (bf16_t)o;
    }
  }
  // S[head][key] = Q K^T : lane holds key = l16, heads kq*4 .. +3
  auto row_of = [&](int key) -> int64_t { return (int64_t)tab_dyn[key / page] * page + (key % page); };
  const bf16_t* kbase = p.k + (int64_t)kh * p.k_sh;
  const int l16 = lane & 15, kq = lane >> 4;
  const int head = kh * G + min(l16, G - 1);
  bf16x8 qf[KC];
  {
    const bf16_t* qp = p.q + (int64_t)b * p.q_st + (int64_t)head * p.q_sh + kq * 8;
#pragma unroll
    for (int kc = 0; kc < KC; kc++) qf[kc] = ld_global_b128(qp + kc * 32);
  }
  float lse4[4];
#pragma unroll
  for (int i = 0; i < 4; i++) lse4[i] = lse_s[kq * 4 + i];
  float* pg = p.pg + ((int64_t)b * p.KH + kh) * p.y_cap;
  const int nu = (y + UK - 1) / UK;
  const int step = NW * nsplit;
  bf16x8 kfA[2][KC], kfB[2][KC];
  auto issue = [&](int u, bf16x8 (&kf)[2][KC]) {
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      int key = min(u * UK + jt * 16 + l16, y - 1);
      const bf16_t* kp = kbase + row_of(key) * p.k_sr + kq * 8;
#pragma unroll
      for (int kc = 0; kc < KC; kc++) kf[jt][kc] = ld_global_b128(kp + kc * 32);
    }
  };
  auto compute = [&](int u, bf16x8 (&kf)[2][KC]) {
#pragma unroll
    for (int jt = 0; jt < 2; jt++) {
      f32x4 sv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; kc++) sv = mfma16(qf[kc], kf[jt][kc], sv);
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (kq * 4 + i < G) acc += fast_exp2(__builtin_fmaf(sv[i], p.scale_log2, -lse4[i]));
      acc = xrow_sum(acc);
      acc = xhalf_sum(acc);
      int key = u * UK + jt * 16 + l16;
      if (kq == 0 && key < y) pg[key] = acc;
    }
  };
  const int first = sp * NW + wave;
  if (first < nu) issue(first, kfA);
  for (int u = first; u < nu; u += 2 * step) {
    const bool hasB = u + step < nu;
    if (hasB) issue(u + step, kfB);
    compute(u, kfA);
    if (hasB) {
      if (u + 2 * step < nu) issue(u + 2 * step, kfA);
      compute(u + step, kfB);
    }
  }
}

template <int D, int VD>
__global__ __launch_bounds__(DEC_WAVES * 64) void decode_slc_swa_kernel(NsaDecodeParams p) {
  using UF = UnitFlash<D, VD>;
  constexpr int NW = DEC_WAVES;
  constexpr int NT = NW * 64;
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_raw[];
  constexpr int SLOT = UF::SLOT;
  static_assert(SLOT * 2 >= 16 * UF::OLD * 4, "a wave's slot must hold its partial output");
  bf16_t* Vs_all = reinterpret_cast<bf16_t*>(dyn_raw);
  float* part_m = reinterpret_cast<float*>(dyn_raw + (size_t)NW * SLOT * 2);
  float* part_l = part_m + NW * 16;
  int* blk_s = reinterpret_cast<int*>(part_l + NW * 16);
  float* cand_v = reinterpret_cast<float*>(blk_s + 64);  // the selector's candidate list (64 scores + 64 indices)
  int* cand_i = blk_s + 128;
  int* tab_s = blk_s + SEL_INTS;  // the request's raw page table

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, kh = blockIdx.y;
  // the window and selected units of a (request, kv head) may be cut into gridDim.z parts (every part repeats the
  // prologue and the selection, which all of them need, and writes partial results for a merging launch)
  const int part = blockIdx.z, nparts = gridDim.z;
  const int G = p.G;
  const int L = p.ctx_lens[b];
  const int t = L - 1;
  const int32_t* tab = p.table + (int64_t)b * p.table_stride;
  const int page = p.page_size;
  for (int i = tid; i < (L + page - 1) / page; i += NT) tab_s[i] = tab[i];
  const bf16_t* kbase = p.k + (int64_t)kh * p.k_sh;
  const bf16_t* vbase = p.v + (int64_t)kh * p.v_sh;
  const int l16 = lane & 15;
  const int g = min(l16, G - 1);
  const int head = kh * G + g;
  const int Bs = p.block_size;
  const int nvalid = t >= 0 ? min(p.top_n, t / Bs + 1) : 0;
  const int nb = min(L > 0 ? (L - 1) / Bs + 1 : 0, p.nb_cap);
  __shared__ float sp_lse_s[16], sp_m_s[16], sp_l_s[16];
  __shared__ float sp_w_s[64 * 16];  // weights of the parts of the compressed branch (nsplit <= 64)
  static_assert(sizeof(sp_lse_s) + sizeof(sp_m_s) + sizeof(sp_l_s) + sizeof(sp_w_s) == SLC_SWA_STATIC_LDS,
                "the host-side LDS budget must count this kernel's static arrays");
  constexpr int OPT = 16 * VD / NT;  // output values per thread
  static_assert((16 * VD) % NT == 0, "output values must divide over the threads");
  // output values of a thread: OPT consecutive channels of one head
  typedef float fvec __attribute__((ext_vector_type(OPT)));
  typedef float fvecu __attribute__((ext_vector_type(OPT), aligned(4)));
  typedef bf16_t bvecu __attribute__((ext_vector_type(OPT), aligned(2)));
  const int oi = tid * OPT;
  const int oh = oi / VD, od = oi - oh * VD;
  const int hq = kh * G + oh;
  bf16_t gate_raw[3] = {};           // requested long before the merge that uses them
  if (p.out && oh < G) {
    const bf16_t* wp = p.w + (int64_t)b * p.w_st + (int64_t)hq * p.w_sh;
#pragma unroll
    for (int i = 0; i < 3; i++) gate_raw[i] = wp[i];
  }
  const int W = p.win_parts;         // > 0: the first launch has attended the window
  fvec ocmp_pre, o_swa_pre;          // merged outputs of the compressed branch (split path) and of the window
#pragma unroll
  for (int r = 0; r < OPT; r++) ocmp_pre[r] = o_swa_pre[r] = 0.f;
  float* imp = nullptr;              // block scores, when the selection runs here
  const bool select_here = p.sp_keep_p != nullptr || p.pg != nullptr;
  if (p.sp_keep_p != nullptr) {
    // Prologue of the two-launch split path: merge the statistics of the parts of the compressed branch, turn the
    // spilled fp16 probabilities into head-summed probabilities (over the not-yet-used staging slots) and fold them
    // into block scores.  The same arithmetic as the one-launch kernel.
    typedef typename UF::keep4 h4;
    const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
    const int nuc = (p.y_cap + UK - 1) / UK, keep_ld = nuc * UK;
    const int nsplit = p.nsplit;
    float* pgs = reinterpret_cast<float*>(Vs_all);
    imp = reinterpret_cast<float*>(tab_s + ((p.table_stride + 3) & ~3));
    float* fac = imp + ((p.nb_cap + 3) & ~3);
    const int64_t sp_base = ((int64_t)b * p.KH + kh) * nsplit * 16;
    const typename UF::keep_t* keep_p = (const typename UF::keep_t*)p.sp_keep_p + ((int64_t)b * p.KH + kh) * 16 * keep_ld;
    const float* keep_m = p.sp_keep_m + ((int64_t)b * p.KH + kh) * nuc * 16;
    // Everything that comes from the first launch is requested here, in one round trip to memory: statistics, outputs of
    // the parts, maxima and the first probabilities (the rest of the prologue is a chain of short steps with barriers).
    // Us of this launch, with a round trip per step and the window attended next to the selection -> so: one request of
    // 32K tokens 28.9 -> 22.4, 16 of 128K 45.4 -> 36.0, 8 of up to 16K with 192 channels 29.8 -> 23.4; 1-2 us of it come
    // from the window, the rest from the loads.
    constexpr int PRE = 8, KM = 2, WMAX = 4;
    float* st_m = fac;
    float* st_l = fac + 64 * 16;
    for (int i = tid; i < nsplit * 16; i += NT) { st_m[i] = p.sp_m[sp_base + i]; st_l[i] = p.sp_l[sp_base + i]; }
    const int64_t w_base = ((int64_t)b * p.KH + kh) * W * 16;
    if (tid < W * 16) { part_m[tid] = p.win_m[w_base + tid]; part_l[tid] = p.win_l[w_base + tid]; }
    auto part_out = [&](const float* o, int64_t base16, int s2) {
      return (fvec)*reinterpret_cast<const fvecu*>(o + (base16 + s2 * 16 + oh) * VD + od);
    };
    fvec po[PRE], wo[WMAX];
#pragma unroll
    for (int s2 = 0; s2 < PRE; s2++) po[s2] = part_out(p.sp_o, sp_base, min(s2, nsplit - 1));
    if (W > 0) {
#pragma unroll
      for (int s2 = 0; s2 < WMAX; s2++) wo[s2] = part_out(p.win_o, w_base, min(s2, W - 1));
    }
    const int nu = (y + UK - 1) / UK;
    float km[KM];
#pragma unroll
    for (int r = 0; r < KM; r++) km[r] = tid + r * NT < nu * 16 ? keep_m[tid + r * NT] : 0.f;
    h4 v[16];
    auto fetch_probs = [&](int k4) {
#pragma unroll
      for (int h = 0; h < 16; h++)
        v[h] = *reinterpret_cast<const h4*>(keep_p + (k4 / UK) * (16 * UK) + h * UK + (k4 % UK));
    };
    if (tid * 4 < y) fetch_probs(tid * 4);
    __syncthreads();
    if (tid < 16) {  // one thread per head
      float m = NSA_NEG_INF;
      for (int s2 = 0; s2 < nsplit; s2++) m = fmaxf(m, st_m[s2 * 16 + tid]);
      float l = 0.f;
      for (int s2 = 0; s2 < nsplit; s2++) {
        const float ms = st_m[s2 * 16 + tid];
        const float a = (ms == NSA_NEG_INF) ? 0.f : fast_exp2((ms - m) * p.scale_log2);
        sp_w_s[s2 * 16 + tid] = a;
        l += a * st_l[s2 * 16 + tid];
      }
      const float inv = l > 0.f ? 1.f / l : 0.f;
      for (int s2 = 0; s2 < nsplit; s2++) sp_w_s[s2 * 16 + tid] *= inv;
      const float lse2 = (m != NSA_NEG_INF && l > 0.f) ? m * p.scale_log2 + fast_log2(l) : 0.f;
      sp_lse_s[tid] = lse2;
      if (tid < G && p.lse_out) p.lse_out[(int64_t)b * p.lse_st + (kh * G + tid) * p.lse_sh] = lse2;
    } else if (wave == 1 && lane < 16 && W > 0) {
      merge_weights(part_m, part_l, W, 16, lane, p.scale_log2);
    }
    __syncthreads();
    for (int s0 = 0; s0 < nsplit; s0 += PRE) {
      if (s0 > 0) {
#pragma unroll
        for (int s2 = 0; s2 < PRE; s2++) po[s2] = part_out(p.sp_o, sp_base, min(s0 + s2, nsplit - 1));
      }
#pragma unroll
      for (int s2 = 0; s2 < PRE; s2++)
        if (s0 + s2 < nsplit) ocmp_pre += sp_w_s[(s0 + s2) * 16 + oh] * po[s2];
    }
    if (W > 0) {
#pragma unroll
      for (int s2 = 0; s2 < WMAX; s2++)
        if (s2 < W) o_swa_pre += part_l[s2 * 16 + oh] * wo[s2];
    }
#pragma unroll
    for (int r = 0; r < KM; r++) {
      const int i = tid + r * NT, h = i & 15;
      if (i < nu * 16) fac[i] = h < G ? fast_exp2(__builtin_fmaf(km[r], p.scale_log2, -sp_lse_s[h])) : 0.f;
    }
    for (int i = tid + KM * NT; i < nu * 16; i += NT) {
      const int h = i & 15;
      fac[i] = h < G ? fast_exp2(__builtin_fmaf(keep_m[i], p.scale_log2, -sp_lse_s[h])) : 0.f;
    }
    __syncthreads();
    for (int k4 = tid * 4; k4 < y; k4 += NT * 4) {
      const float* f = fac + (k4 / UK) * 16;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 16; h++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] += (float)v[h][e] * f[h];
      if (k4 + NT * 4 < y) fetch_probs(k4 + NT * 4);
      *reinterpret_cast<f32x4*>(pgs + k4) = acc;
    }
    __syncthreads();
    fold_block_scores(pgs, imp, y, nb, nb, p, tid, NT);
  } else if (p.pg != nullptr) {
    // fold the head-summed probabilities of the compressed keys (computed by the importance kernel) into block
    // scores; they live behind the page table, the staging slots belong to the window waves
    imp = reinterpret_cast<float*>(tab_s + ((p.table_stride + 3) & ~3));
    const float* pg = p.pg + ((int64_t)b * p.KH + kh) * p.y_cap;
    const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
    fold_block_scores(pg, imp, y, nb, nb, p, tid, NT);
  } else if (tid < 64) {
    blk_s[tid] = tid < nvalid ? max(p.topk[(int64_t)kh * p.tk_sh + (int64_t)b * p.tk_st + tid], 0) : 0;
  }
  __syncthreads();

  // ---- window attention, or, when the first launch has done it, the blocks that are selected whatever their score (they
  // open the selected branch); when the selection runs here, wave 0 selects meanwhile ----
  const int upb = Bs / UK;
  const int n_forced = W > 0 ? min(p.num_init + p.num_local, nvalid) : 0;
  UF uf;
  uf.init(p.q + (int64_t)b * p.q_st + (int64_t)head * p.q_sh, p.scale_log2, lane, Vs_all + wave * SLOT);
  const int w_first = select_here ? 1 : 0;
  if (wave < w_first) {
    const int result = select_blocks_wave<false>(imp, t, nb, p, lane, cand_v, cand_i);
    blk_s[lane] = lane < nvalid ? max(result, 0) : 0;
    if (p.topk && part == 0 && lane < p.top_n) p.topk[(int64_t)kh * p.tk_sh + (int64_t)b * p.tk_st + lane] = result;
  } else {
    if (t >= 0) {
      const int klo = W > 0 ? 0 : max(0, t - p.window);
      const int k0 = (klo / UK) * UK;
      const int nu = W > 0 ? n_forced * upb : (t - k0) / UK + 1;
      uf.run(part * (NW - w_first) + wave - w_first, nparts * (NW - w_first), nu, klo, t,
             [&](int u) {
               if (W == 0) return k0 + u * UK;
               const int slot = u / upb;
               return (slot < p.num_init ? slot : t / Bs - (slot - p.num_init)) * Bs + (u - slot * upb) * UK;
             },
             tab_s, page, kbase, p.k_sr, vbase, p.v_sr);
    }
    if (W == 0) uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(Vs_all + wave * SLOT));
  }
  __syncthreads();
  const float* part_o = reinterpret_cast<const float*>(Vs_all);
  // parts: the un-normalised (m, l, o) of this part's waves, one thread per output value (same arithmetic as the
  // partial kernel of the compressed branch)
  auto spill_part = [&](int branch, int w0, int nw) {
    const int64_t base = ((((int64_t)b * p.KH + kh) * nparts + part) * 2 + branch);
    for (int idx = tid; idx < 16 * VD; idx += NT) {
      const int h = idx / VD, d = idx - h * VD;
      float m = NSA_NEG_INF;
      for (int w = w0; w < w0 + nw; w++) m = fmaxf(m, part_m[w * 16 + h]);
      float l = 0.f, o = 0.f;
      if (m != NSA_NEG_INF) {
        for (int w = w0; w < w0 + nw; w++) {
          const float mw = part_m[w * 16 + h];
          const float a = (mw == NSA_NEG_INF) ? 0.f : fast_exp2((mw - m) * p.scale_log2);
          l += a * part_l[w * 16 + h];
          o += a * part_o[w * (SLOT / 2) + h * UF::OLD + d];
        }
      }
      p.sp2_o[(base * 16 + h) * VD + d] = o;
      if (d == 0) { p.sp2_ml[(base * 2 + 0) * 16 + h] = m; p.sp2_ml[(base * 2 + 1) * 16 + h] = l; }
    }
  };
  if (nparts > 1) {
    spill_part(1, w_first, NW - w_first);
    __syncthreads();  // the slots are staging space again
    uf.reset();
    if (t >= 0) {
      uf.run(part * NW + wave, nparts * NW, nvalid * upb, 0, t,
             [&](int u) { int slot = u / upb; return blk_s[slot] * Bs + (u - slot * upb) * UK; }, tab_s, page, kbase,
             p.k_sr, vbase, p.v_sr);
    }
    uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(Vs_all + wave * SLOT));
    __syncthreads();
    spill_part(0, 0, NW);
    if (part == 0 && p.sp_keep_p != nullptr && oh < G) {  // the compressed branch's output, merged in the prologue
      bvecu c;
#pragma unroll
      for (int r = 0; r < OPT; r++) c[r] = (bf16_t)ocmp_pre[r];
      *reinterpret_cast<bvecu*>(p.cmp_tmp + (int64_t)b * p.co_st + (int64_t)(kh * G + oh) * p.co_sh + od) = c;
    }
    return;
  }
  // the weighted sum of the partial outputs of waves w0 .. w0 + NP - 1
  auto merged = [&](auto np, int w0) {
    constexpr int NP = decltype(np)::value;
    float wgt[NP];
    merge_weights_local<NP>(part_m + w0 * 16, part_l + w0 * 16, 16, oh, p.scale_log2, wgt);
    fvec o;
#pragma unroll
    for (int r = 0; r < OPT; r++) o[r] = 0.f;
#pragma unroll
    for (int w = 0; w < NP; w++)
      o += wgt[w] * *reinterpret_cast<const fvec*>(&part_o[(w0 + w) * (SLOT / 2) + oh * UF::OLD + od]);
    return o;
  };
  if (W == 0) {
    if (w_first) o_swa_pre = merged(std::integral_constant<int, NW - 1>{}, 1);
    else o_swa_pre = merged(std::integral_constant<int, NW>{}, 0);
    __syncthreads();  // the slots are staging space again
    uf.reset();
  }

  // ---- selected blocks (behind the forced ones), all waves; the last wave and wave 0 have had fewest units so far ----
  if (t >= 0) {
    uf.run(W > 0 ? (wave + 1) % NW : wave, NW, (nvalid - n_forced) * upb, 0, t,
           [&](int u) { const int slot = u / upb; return blk_s[n_forced + slot] * Bs + (u - slot * upb) * UK; }, tab_s, page,
           kbase, p.k_sr, vbase, p.v_sr);
  }
  float gate[3];
#pragma unroll
  for (int i = 0; i < 3; i++) gate[i] = 1.f / (1.f + __expf(-(float)gate_raw[i]));
  uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(Vs_all + wave * SLOT));
  __syncthreads();
  if (oh >= G) return;
  const fvec o_slc = merged(std::integral_constant<int, NW>{}, 0);
  const int64_t co = (int64_t)b * p.co_st + (int64_t)hq * p.co_sh + od;
  // branch outputs are rounded to bf16 before the gated sum, as the three-kernel path stores them
  bvecu slc, swa, cmp;
#pragma unroll
  for (int r = 0; r < OPT; r++) { slc[r] = (bf16_t)o_slc[r]; swa[r] = (bf16_t)o_swa_pre[r]; }
  if (p.slc_o) *reinterpret_cast<bvecu*>(p.slc_o + co) = slc;
  if (p.swa_o) *reinterpret_cast<bvecu*>(p.swa_o + co) = swa;
  if (p.sp_keep_p != nullptr) {  // merged in the prologue
#pragma unroll
    for (int r = 0; r < OPT; r++) cmp[r] = (bf16_t)ocmp_pre[r];
    if (p.cmp_o) *reinterpret_cast<bvecu*>(p.cmp_o + co) = cmp;
  } else if (p.out) {
    cmp = *reinterpret_cast<const bvecu*>(p.cmp_o + co);
  }
  if (p.out) {
    bvecu o;
#pragma unroll
    for (int r = 0; r < OPT; r++)
      o[r] = (bf16_t)((float)cmp[r] * gate[0] + (float)slc[r] * gate[1] + (float)swa[r] * gate[2]);
    *reinterpret_cast<bvecu*>(p.out + (int64_t)b * p.o_st + (int64_t)hq * p.o_sh + od) = o;
  }
}

// grid (B, KH): merges the parts written by decode_slc_swa_kernel when it ran with several parts per (request, kv
// head) and applies the gates -> final output (and the branch outputs on request)
template <int VD>
__global__ __launch_bounds__(256) void decode_split_final_kernel(NsaDecodeParams p) {
  const int b = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x;
  const int G = p.G, S = p.slc_nsplit;
  for (int idx = tid; idx < G * (VD / 4); idx += 256) {
    const int h = idx / (VD / 4), d = (idx - h * (VD / 4)) * 4;
    const int hq = kh * G + h;
    f32x4 res[2];
#pragma unroll
    for (int br = 0; br < 2; br++) {
      const int64_t base0 = (((int64_t)b * p.KH + kh) * S) * 2 + br;
      float m = NSA_NEG_INF;
      for (int s2 = 0; s2 < S; s2++) m = fmaxf(m, p.sp2_ml[((base0 + s2 * 2) * 2 + 0) * 16 + h]);
      float l = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      if (m != NSA_NEG_INF) {
        for (int s2 = 0; s2 < S; s2++) {
          const int64_t base = base0 + s2 * 2;
          const float ms = p.sp2_ml[(base * 2 + 0) * 16 + h];
          const float a = (ms == NSA_NEG_INF) ? 0.f : fast_exp2((ms - m) * p.scale_log2);
          l += a * p.sp2_ml[(base * 2 + 1) * 16 + h];
          const f32x4 x = *reinterpret_cast<const f32x4*>(p.sp2_o + (base * 16 + h) * VD + d);
          o[0] += a * x[0]; o[1] += a * x[1]; o[2] += a * x[2]; o[3] += a * x[3];
        }
      }
      const float inv = l > 0.f ? 1.f / l : 0.f;
      // branch outputs are rounded to bf16 before the gated sum, as the other decode paths store them
      res[br] = round_bf16x4(f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
    }
    const int64_t co = (int64_t)b * p.co_st + (int64_t)hq * p.co_sh + d;
    if (p.slc_o) *reinterpret_cast<bf16x4*>(p.slc_o + co) = pack4(res[0][0], res[0][1], res[0][2], res[0][3]);
    if (p.swa_o) *reinterpret_cast<bf16x4*>(p.swa_o + co) = pack4(res[1][0], res[1][1], res[1][2], res[1][3]);
    const bf16x4 c4 = *reinterpret_cast<const bf16x4*>(p.cmp_tmp + co);
    if (p.cmp_o) *reinterpret_cast<bf16x4*>(p.cmp_o + co) = c4;
    const bf16_t* wp = p.w + (int64_t)b * p.w_st + (int64_t)hq * p.w_sh;
    const float s0 = 1.f / (1.f + __expf(-(float)wp[0]));
    const float s1 = 1.f / (1.f + __expf(-(float)wp[1]));
    const float s2g = 1.f / (1.f + __expf(-(float)wp[2]));
    *reinterpret_cast<bf16x4*>(p.out + (int64_t)b * p.o_st + (int64_t)hq * p.o_sh + d) =
        pack4((float)c4[0] * s0 + res[0][0] * s1 + res[1][0] * s2g, (float)c4[1] * s0 + res[0][1] * s1 + res[1][1] * s2g,
              (float)c4[2] * s0 + res[0][2] * s1 + res[1][2] * s2g, (float)c4[3] * s0 + res[0][3] * s1 + res[1][3] * s2g);
  }
}

// ---- the whole decode step of one (request, kv head) in one workgroup ------------------------------------------
// compressed attention -> block scores -> [wave 0: selection | waves 1..7: window attention] -> selected-block
// attention -> gated combine.  Nothing but the final output (and, on request, topk / the branch outputs) goes
// back to global memory; the compressed-branch output stays in registers, the window partials in the LDS region
// that held the fp16 probabilities.
template <int D, int VD, int NW>
__global__ __launch_bounds__(NW * 64, 2) void decode_fused_kernel(NsaDecodeParams p, int keep_units) {
  using UF = UnitFlash<D, VD, (D > 128) ? KEEP_MEM : (NW == DEC_WAVES ? KEEP_LDS : KEEP_BOTH),
                       (D > 128) ? 1 : DEC_WAVES / NW, NW == DEC_WAVES>;
  constexpr int SLOT = UF::SLOT;
  constexpr int NTHREADS = NW * 64;
  constexpr int NV4 = 16 * VD / 4;                             // groups of four merged output values
  constexpr int OPT4 = (NV4 + NTHREADS - 1) / NTHREADS;        // groups per thread
  static_assert(SLOT * 2 >= 16 * UF::OLD * 4, "a wave's slot must hold its partial output");
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_raw[];
  bf16_t* slots = reinterpret_cast<bf16_t*>(dyn_raw);
  float* part_m = reinterpret_cast<float*>(dyn_raw + (size_t)NW * SLOT * 2);
  float* part_l = part_m + NW * 16;
  float* swa_m = part_l + NW * 16;
  float* swa_l = swa_m + NW * 16;
  float* lse_s = swa_l + NW * 16;
  float* imp = lse_s + 16;
  int* blk_s = reinterpret_cast<int*>(imp + ((p.nb_cap + 3) & ~3));
  float* cand_v = reinterpret_cast<float*>(blk_s + 64);  // the selector's candidate list (64 scores + 64 indices)
  int* cand_i = blk_s + 128;
  int* ctab_s = blk_s + SEL_INTS;
  const int ntab_c = (p.y_cap + p.page_size - 1) / p.page_size;
  int* tab_s = ctab_s + ((ntab_c + 3) & ~3);
  const int keep_ld = keep_units * UK + 8;
  const int n_units_cap = (p.y_cap + UK - 1) / UK;
  using keep_t = typename UF::keep_t;
  float* keep_m = reinterpret_cast<float*>(tab_s + ((p.table_stride + 3) & ~3));
  keep_t* keep_p = reinterpret_cast<keep_t*>(keep_m + n_units_cap * 16);
  float* swa_o = reinterpret_cast<float*>(keep_p);  // [NW-1][16][VD], after the probabilities are consumed
  float* pg = reinterpret_cast<float*>(dyn_raw);    // over the staging slots, between the phases

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, kh = blockIdx.y;
  const int G = p.G;
  const int L = p.ctx_lens[b];
  const int t = L - 1;
  const int y = L >= p.kernel_size ? min((L - p.kernel_size) / p.stride + 1, p.y_cap) : 0;
  const int Bs = p.block_size;
  const int nb = min(L > 0 ? (L - 1) / Bs + 1 : 0, p.nb_cap);
  const int page = p.page_size;
  {
    const int32_t* ctab = p.cmp_table + (int64_t)b * p.cmp_table_stride;
    const int32_t* tab = p.table + (int64_t)b * p.table_stride;
    // whole table rows (their widths are the capacity, the entries past a request's pages are never used), so that
    // these loads do not wait for the context length and both round trips overlap
    const int nc = min(ntab_c, p.cmp_table_stride), nr = p.table_stride;
    for (int i = tid; i < nc + nr; i += NTHREADS) {
      if (i < nc) ctab_s[i] = ctab[i];
      else tab_s[i - nc] = tab[i - nc];
    }
  }
  // Cache maintenance of this (request, kv head), wave 0 for K and wave 1 for V, one 16-byte piece per lane:
  //  * the newest token's row goes to its pool row (upstream store_kvcache,
  //    nano-vllm/nanovllm/layers/attention.py:123-153), when the caller passes it;
  //  * the compressed row that the newest token completes = mean of the last kernel_size raw rows, summed in
  //    row order in fp32 like nsa_paged_pool_decode (flash_nsa/inference/compress_kv.py:253-287 upstream).
  // Both are written to the pool and read back by the attention phases of this workgroup after a fence and a
  // barrier.  The compressed phase only needs the pooled row, so when nothing is pooled at this step the store
  // runs after the first barrier and its fence is covered by the barriers that separate the phases.
  const int raw_slot = (p.raw_slots != nullptr && L > 0) ? p.raw_slots[b] : -1;
  const int cmp_slot = p.cmp_slots != nullptr ? p.cmp_slots[b] : -1;
  const bool pool_now = cmp_slot >= 0 && L >= p.kernel_size;
  auto maintain = [&]() {
    bf16_t* cache = const_cast<bf16_t*>(wave == 0 ? p.k : p.v);
    const int64_t c_sr = wave == 0 ? p.k_sr : p.v_sr, c_sh = wave == 0 ? p.k_sh : p.v_sh;
    const int C = (wave == 0 ? D : VD) / 8;
    if (lane < C) {
      bf16x8 newest = zero_bf16x8();
      if (raw_slot >= 0) {
        const bf16_t* src = wave == 0 ? p.new_k + (int64_t)b * p.nk_st + (int64_t)kh * p.nk_sh
                                      : p.new_v + (int64_t)b * p.nv_st + (int64_t)kh * p.nv_sh;
        newest = ld_global_b128(src + lane * 8);
        *reinterpret_cast<bf16x8*>(cache + (int64_t)raw_slot * c_sr + (int64_t)kh * c_sh + lane * 8) = newest;
      }
      if (pool_now) {
        const int32_t* tab = p.table + (int64_t)b * p.table_stride;
        const int st = ((L - p.kernel_size) / p.stride) * p.stride;
        float a[8];
        sum_rows(a, cache + (int64_t)kh * c_sh + lane * 8, c_sr, tab, page, st, p.kernel_size,
                 raw_slot >= 0 ? L - 1 : -1, newest);
        const float inv = 1.f / (float)p.kernel_size;
        *reinterpret_cast<bf16x8*>(cache + (int64_t)cmp_slot * c_sr + (int64_t)kh * c_sh + lane * 8) =
            pack8(a[0] * inv, a[1] * inv, a[2] * inv, a[3] * inv, a[4] * inv, a[5] * inv, a[6] * inv, a[7] * inv);
      }
    }
    // the rows are read back only by waves of this workgroup (same CU, same vector L1): a workgroup-scope release
    // is enough, and much cheaper than a device-scope fence, which writes back the L2 slice of the XCD
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  };
  if (pool_now && wave < 2) maintain();
  __syncthreads();
  if (!pool_now && raw_slot >= 0 && wave < 2) maintain();
  const bf16_t* kbase = p.k + (int64_t)kh * p.k_sh;
  const bf16_t* vbase = p.v + (int64_t)kh * p.v_sh;
  const int l16 = lane & 15;
  const int head = kh * G + min(l16, G - 1);

  UF uf;
  uf.init(p.q + (int64_t)b * p.q_st + (int64_t)head * p.q_sh, p.scale_log2, lane, slots + wave * SLOT);
  uf.keep_p = keep_p;
  uf.keep_m = keep_m;
  uf.keep_ld = keep_ld;
  const int y_keep = min(y, keep_units * UK);  // keys whose probabilities stay in LDS; the others go to scratch memory
  const keep_t* spill = (const keep_t*)p.sp_keep_p + ((int64_t)b * p.KH + kh) * 16 * n_units_cap * UK;
  uf.spill_p = const_cast<keep_t*>(spill);
  uf.keep_lds_end = y_keep;
  uf.keep_end = y;
  const int nu = (y + UK - 1) / UK;

  // ---- compressed attention, units dealt round-robin to the waves ----
  uf.run(wave, NW, nu, 0, y - 1, [&](int u) { return u * UK; }, ctab_s, page, kbase, p.k_sr, vbase, p.v_sr);
  uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(slots + wave * SLOT));
  // the window branch does not depend on anything computed here: the waves that will run it fetch their first
  // unit now, behind the merge of the compressed branch, the block scores and the selection
  const int swa_klo = max(0, t - p.window);
  const int swa_k0 = (swa_klo / UK) * UK;
  const int swa_nu = t >= 0 ? (t - swa_k0) / UK + 1 : 0;
  auto swa_key = [&](int u) { return swa_k0 + u * UK; };
  // (with two workgroups per CU the other one hides that latency, and the prefetched unit's registers would spill)
  constexpr bool PREFETCH_SWA = NW == DEC_WAVES;
  // When the newest token's row was stored by waves 0 / 1 after the first barrier (nothing pooled at this step),
  // only the next barrier orders that store before other waves' reads of the row, and the window's last unit holds
  // it: the prefetch then waits for the barrier (workgroup-uniform condition).
  const bool stored_late = !pool_now && raw_slot >= 0;
  if (PREFETCH_SWA && !stored_late && wave != 0 && t >= 0)
    uf.prefetch(wave - 1, swa_nu, swa_klo, t, swa_key, tab_s, page, kbase, p.k_sr, vbase, p.v_sr);
  __syncthreads();
  if (PREFETCH_SWA && stored_late && wave != 0 && t >= 0)
    uf.prefetch(wave - 1, swa_nu, swa_klo, t, swa_key, tab_s, page, kbase, p.k_sr, vbase, p.v_sr);
  // every thread merges four consecutive channels of one head (16-byte LDS reads, 8-byte stores) with weights it
  // evaluates itself; the thread that holds channel 0 of a head also publishes the head's lse
  f32x4 o_cmp[OPT4];
#pragma unroll
  for (int r = 0; r < OPT4; r++) {
    const int idx = tid + r * NTHREADS;
    const int h = min(idx / (VD / 4), 15), d = (idx % (VD / 4)) * 4;
    float wgt[NW];
    const float lse2 = merge_weights_local<NW>(part_m, part_l, 16, h, p.scale_log2, wgt);
    if (idx < NV4 && d == 0) {
      lse_s[h] = h < G ? lse2 : 0.f;
      if (h < G && p.lse_out) p.lse_out[(int64_t)b * p.lse_st + (kh * G + h) * p.lse_sh] = lse2;
    }
    // the staged path stores the branch output as bf16 before the gated sum
    o_cmp[r] = round_bf16x4(merge_value4_local<NW>(wgt, reinterpret_cast<const float*>(slots), SLOT / 2, h, d, UF::OLD));
    if (idx < NV4 && h < G && p.cmp_o)
      *reinterpret_cast<bf16x4*>(p.cmp_o + (int64_t)b * p.co_st + (int64_t)(kh * G + h) * p.co_sh + d) =
          pack4(o_cmp[r][0], o_cmp[r][1], o_cmp[r][2], o_cmp[r][3]);
  }
  __syncthreads();
  // ---- probabilities p = kept exp2((s - m_unit)*c) * exp2(m_unit*c - lse), summed over the heads; a thread takes
  // four consecutive keys (one unit, so one set of 16 per-head factors) ----
  for (int key = tid * 4; key < y; key += NTHREADS * 4) {
    const float* um = keep_m + (key / UK) * 16;
    typename UF::keep4 kp[16];
    if (NW == DEC_WAVES || (D <= 128 && key < y_keep)) {
#pragma unroll
      for (int h = 0; h < 16; h++) kp[h] = *reinterpret_cast<const typename UF::keep4*>(&keep_p[h * keep_ld + key]);
    } else {
      const keep_t* up = spill + (int64_t)(key / UK) * (16 * UK) + (key % UK);
#pragma unroll
      for (int h = 0; h < 16; h++) kp[h] = *reinterpret_cast<const typename UF::keep4*>(up + h * UK);
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 16; h++) {
      const float fac = h < G ? fast_exp2(__builtin_fmaf(um[h], p.scale_log2, -lse_s[h])) : 0.f;
      acc[0] += (float)kp[h][0] * fac; acc[1] += (float)kp[h][1] * fac;
      acc[2] += (float)kp[h][2] * fac; acc[3] += (float)kp[h][3] * fac;
    }
    *reinterpret_cast<f32x4*>(&pg[key]) = acc;
  }
  __syncthreads();
  fold_block_scores(pg, imp, y, nb, p.nb_cap, p, tid, NTHREADS);
  __syncthreads();

  // ---- wave 0 selects the blocks while the other waves run the window ----
  const int nvalid = t >= 0 ? min(p.top_n, t / Bs + 1) : 0;
  uf.reset();
  if (wave == 0) {
    const int result = select_blocks_wave<true>(imp, t, p.nb_cap, p, lane, cand_v, cand_i);
    blk_s[lane] = lane < nvalid ? max(result, 0) : 0;
    if (p.topk && lane < p.top_n) p.topk[(int64_t)kh * p.tk_sh + (int64_t)b * p.tk_st + lane] = result;
  } else {
    if (t >= 0)
      uf.template run<PREFETCH_SWA>(wave - 1, NW - 1, swa_nu, swa_klo, t, swa_key, tab_s, page, kbase, p.k_sr, vbase,
                                    p.v_sr);
    uf.publish(swa_m + wave * 16, swa_l + wave * 16, swa_o + (wave - 1) * 16 * UF::OLD);
  }
  __syncthreads();

  // ---- selected blocks, all waves ----
  uf.reset();
  if (t >= 0) {
    const int upb = Bs / UK;
    uf.run(wave, NW, nvalid * upb, 0, t,
           [&](int u) { int slot = u / upb; return blk_s[slot] * Bs + (u - slot * upb) * UK; }, tab_s, page, kbase,
           p.k_sr, vbase, p.v_sr);
  }
  uf.publish(part_m + wave * 16, part_l + wave * 16, reinterpret_cast<float*>(slots + wave * SLOT));
  __syncthreads();
#pragma unroll
  for (int r = 0; r < OPT4; r++) {
    const int idx = tid + r * NTHREADS;
    const int h = idx / (VD / 4), d = (idx % (VD / 4)) * 4;
    if (idx >= NV4 || h >= G) continue;
    const int hq = kh * G + h;
    float w_slc[NW], w_swa[NW - 1];
    merge_weights_local<NW>(part_m, part_l, 16, h, p.scale_log2, w_slc);
    merge_weights_local<NW - 1>(swa_m + 16, swa_l + 16, 16, h, p.scale_log2, w_swa);
    const f32x4 o_slc =
        round_bf16x4(merge_value4_local<NW>(w_slc, reinterpret_cast<const float*>(slots), SLOT / 2, h, d, UF::OLD));
    const f32x4 o_swa = round_bf16x4(merge_value4_local<NW - 1>(w_swa, swa_o, 16 * UF::OLD, h, d, UF::OLD));
    const int64_t co = (int64_t)b * p.co_st + (int64_t)hq * p.co_sh + d;
    if (p.slc_o) *reinterpret_cast<bf16x4*>(p.slc_o + co) = pack4(o_slc[0], o_slc[1], o_slc[2], o_slc[3]);
    if (p.swa_o) *reinterpret_cast<bf16x4*>(p.swa_o + co) = pack4(o_swa[0], o_swa[1], o_swa[2], o_swa[3]);
    const bf16_t* wp = p.w + (int64_t)b * p.w_st + (int64_t)hq * p.w_sh;
    const float s0 = 1.f / (1.f + __expf(-(float)wp[0]));
    const float s1 = 1.f / (1.f + __expf(-(float)wp[1]));
    const float s2 = 1.f / (1.f + __expf(-(float)wp[2]));
    *reinterpret_cast<bf16x4*>(p.out + (int64_t)b * p.o_st + (int64_t)hq * p.o_sh + d) =
        pack4(o_cmp[r][0] * s0 + o_slc[0] * s1 + o_swa[0] * s2, o_cmp[r][1] * s0 + o_slc[1] * s1 + o_swa[1] * s2,
              o_cmp[r][2] * s0 + o_slc[2] * s1 + o_swa[2] * s2, o_cmp[r][3] * s0 + o_slc[3] * s1 + o_swa[3] * s2);
  }
}

}  // namespace

template <class K, class... Args>
static int launch_dyn(K kern, dim3 grid, int waves, size_t dyn, hipStream_t stream, const char* name,
                      size_t static_lds, Args... args) {
  if (dyn + static_lds > 160 * 1024) {
    nsa_set_error("%s: %zu bytes of LDS needed (fixed_y_maxlen / fixed_num_slc_blocks too large)", name,
                  dyn + static_lds);
    return NSA_ERR_UNSUPPORTED;
  }
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
  if (e != hipSuccess) {
    nsa_set_error("%s: hipFuncSetAttribute(%zu) failed: %s", name, dyn, hipGetErrorString(e));
    return NSA_ERR_LAUNCH;
  }
  kern<<<grid, waves * 64, dyn, stream>>>(args...);
  return nsa_check_launch(name);
}

template <int D, int VD>
static size_t slot_bytes(int waves = DEC_WAVES) { return (size_t)waves * UnitFlash<D, VD>::SLOT * 2; }

// LDS of the fused compressed-attention + selection kernel; `keep` adds the fp16 probabilities of every compressed
// key and the per-unit maxima (no second pass over the keys) and drops the separate pg array
static size_t cmp_topk_lds(size_t slots, size_t keep_size, const NsaDecodeParams& p, bool keep) {
  const size_t ntab = (size_t)(p.y_cap + p.page_size - 1) / p.page_size;
  const size_t units = (size_t)(p.y_cap + UK - 1) / UK;
  size_t n = slots + (size_t)(2 * DEC_WAVES * 16 + 16 + p.nb_cap + ((ntab + 3) & ~(size_t)3)) * sizeof(float);
  if (keep) n += units * 16 * sizeof(float) + 16 * (units * UK + 8) * keep_size;
  else n += (size_t)p.y_cap * sizeof(float);
  return n;
}

template <int D, int VD>
static int launch_cmp_topk(const NsaDecodeParams& p, dim3 grid, hipStream_t stream) {
  const size_t keep_bytes = cmp_topk_lds(slot_bytes<D, VD>(), sizeof(typename UnitFlash<D, VD>::keep_t), p, true);
  if (keep_bytes <= 160 * 1024)
    return launch_dyn(decode_cmp_topk_kernel<D, VD, true>, grid, DEC_WAVES, keep_bytes, stream, "decode_cmp_topk_kernel",
                      0, p);
  return launch_dyn(decode_cmp_topk_kernel<D, VD, false>, grid, DEC_WAVES, cmp_topk_lds(slot_bytes<D, VD>(), 0, p, false),
                    stream, "decode_cmp_topk_kernel", 0, p);
}

static int bad_decode_dims(int D, int VD) {
  nsa_set_error("decode: unsupported head dims D=%d VD=%d (built: 128/128, 64/64, 192/128)", D, VD);
  return NSA_ERR_UNSUPPORTED;
}

int nsa_decode_cmp_topk_launch(const NsaDecodeParams& p, int B, int D, int VD, hipStream_t stream) {
  if (B <= 0) return NSA_OK;
  dim3 grid(B, p.KH);
  if (D == 128 && VD == 128) return launch_cmp_topk<128, 128>(p, grid, stream);
  if (D == 64 && VD == 64) return launch_cmp_topk<64, 64>(p, grid, stream);
  if (D == 192 && VD == 128) return launch_cmp_topk<192, 128>(p, grid, stream);
  return bad_decode_dims(D, VD);
}

// dynamic LDS of the selected + window launch behind the staging slots; scores: it selects the blocks as well
static size_t slc_swa_lds(const NsaDecodeParams& p, bool scores) {
  return (size_t)(2 * DEC_WAVES * 16 + SEL_INTS + ((p.table_stride + 3) & ~3) + (scores ? (p.nb_cap + 3) & ~3 : 0)) *
         sizeof(float);
}

template <int D, int VD>
static int launch_slc_swa(const NsaDecodeParams& p, dim3 grid, size_t dyn, hipStream_t stream) {
  return launch_dyn(decode_slc_swa_kernel<D, VD>, grid, DEC_WAVES, dyn, stream, "decode_slc_swa_kernel",
                    SLC_SWA_STATIC_LDS, p);
}

int nsa_decode_slc_swa_launch(const NsaDecodeParams& p, int B, int D, int VD, hipStream_t stream) {
  if (B <= 0) return NSA_OK;
  dim3 grid(B, p.KH);
  const size_t extra = slc_swa_lds(p, p.pg != nullptr);
  if (D == 128 && VD == 128) return launch_slc_swa<128, 128>(p, grid, slot_bytes<128, 128>() + extra, stream);
  if (D == 64 && VD == 64) return launch_slc_swa<64, 64>(p, grid, slot_bytes<64, 64>() + extra, stream);
  if (D == 192 && VD == 128) return launch_slc_swa<192, 128>(p, grid, slot_bytes<192, 128>() + extra, stream);
  return bad_decode_dims(D, VD);
}

template <int D, int VD>
static size_t cmp_partial_lds(const NsaDecodeParams& p) {
  const int ntab = std::max((p.y_cap + p.page_size - 1) / p.page_size,
                            p.win_parts > 0 ? p.window / p.page_size + 2 : 0);
  return slot_bytes<D, VD>(SPLIT_WAVES) + (size_t)(2 * SPLIT_WAVES * 16 + ntab) * 4;
}

template <int D, int VD>
static int launch_cmp_partial(const NsaDecodeParams& p, dim3 grid, hipStream_t stream) {
  return launch_dyn(p.raw_slots != nullptr ? decode_cmp_partial_kernel<D, VD, true> : decode_cmp_partial_kernel<D, VD, false>,
                    grid, SPLIT_WAVES, cmp_partial_lds<D, VD>(p), stream, "decode_cmp_partial_kernel", 0, p);
}

template <int D, int VD>
static int launch_cmp_split(const NsaDecodeParams& p, dim3 grid, hipStream_t stream) {
  const int rc = launch_cmp_partial<D, VD>(p, grid, stream);
  if (rc) return rc;
  const size_t ntab = (size_t)(p.y_cap + p.page_size - 1) / p.page_size;
  decode_importance_kernel<D, VD><<<grid, SPLIT_WAVES * 64, ntab * 4, stream>>>(p);
  return nsa_check_launch("decode_importance_kernel");
}

int nsa_decode_cmp_split_launch(const NsaDecodeParams& p, int B, int nsplit, int D, int VD, hipStream_t stream) {
  if (B <= 0) return NSA_OK;
  dim3 grid(B, p.KH, nsplit);
  if (D == 128 && VD == 128) return launch_cmp_split<128, 128>(p, grid, stream);
  if (D == 64 && VD == 64) return launch_cmp_split<64, 64>(p, grid, stream);
  if (D == 192 && VD == 128) return launch_cmp_split<192, 128>(p, grid, stream);
  return bad_decode_dims(D, VD);
}

// LDS of the larger of the fused launches: compressed attention + selection (parts: the cut compressed branch, which also
// has a launch with the page table alone and leaves the selection to the next), then selected + window.  0: over the limit
template <int D, int VD>
static size_t two_launch_lds(const NsaDecodeParams& p, bool parts) {
  const size_t first = parts ? cmp_partial_lds<D, VD>(p) : cmp_topk_lds(slot_bytes<D, VD>(), 0, p, false);
  const size_t second = slot_bytes<D, VD>() + slc_swa_lds(p, parts) + SLC_SWA_STATIC_LDS;
  if (parts && (size_t)(p.y_cap + p.page_size - 1) / p.page_size * 4 > 64 * 1024) return 0;
  const size_t n = std::max(first, second);
  return n <= 160 * 1024 ? n : 0;
}

int nsa_decode_two_launch_lds_bytes(const NsaDecodeParams& p, int D, int VD, bool parts) {
  if (D == 128 && VD == 128) return (int)two_launch_lds<128, 128>(p, parts);
  if (D == 64 && VD == 64) return (int)two_launch_lds<64, 64>(p, parts);
  if (D == 192 && VD == 128) return (int)two_launch_lds<192, 128>(p, parts);
  return 0;
}

// ---- two-launch split path: partial kernel with the probability spill, then the final kernel ----
template <int D, int VD>
static size_t split_final_lds(const NsaDecodeParams& p) {
  const size_t slots = slot_bytes<D, VD>();
  if ((size_t)((p.y_cap + UK - 1) / UK) * UK * 4 > slots) return 0;  // head-summed probabilities overlay the slots
  const size_t nuc = (size_t)(p.y_cap + UK - 1) / UK;
  const size_t fac = std::max<size_t>(nuc * 16, 2 * 64 * 16);  // factors, or the parts' (m, l)
  const size_t total = slots + (size_t)(2 * DEC_WAVES * 16 + SEL_INTS + ((p.table_stride + 3) & ~3)) * 4 +
                       (((p.nb_cap + 3) & ~3) + fac) * 4;
  return total + SLC_SWA_STATIC_LDS <= 160 * 1024 ? total : 0;
}

int nsa_decode_split_lds_bytes(const NsaDecodeParams& p, int D, int VD) {
  if (D == 128 && VD == 128) return (int)split_final_lds<128, 128>(p);
  if (D == 64 && VD == 64) return (int)split_final_lds<64, 64>(p);
  if (D == 192 && VD == 128) return (int)split_final_lds<192, 128>(p);
  return 0;
}

int nsa_decode_split_static_lds_bytes() { return (int)SLC_SWA_STATIC_LDS; }

template <int D, int VD>
static int launch_split(const NsaDecodeParams& p, int B, size_t lds2, hipStream_t stream) {
  const int S = p.slc_nsplit > 1 ? p.slc_nsplit : 1;
  int rc = launch_cmp_partial<D, VD>(p, dim3(B, p.KH, p.nsplit + p.win_parts), stream);
  if (rc) return rc;
  rc = launch_slc_swa<D, VD>(p, dim3(B, p.KH, S), lds2, stream);
  if (rc || S == 1) return rc;
  decode_split_final_kernel<VD><<<dim3(B, p.KH), 256, 0, stream>>>(p);
  return nsa_check_launch("decode_split_final_kernel");
}

int nsa_decode_split_launch(const NsaDecodeParams& p, int B, int D, int VD, hipStream_t stream) {
  if (B <= 0) return NSA_OK;
  const int lds2 = nsa_decode_split_lds_bytes(p, D, VD);
  if (lds2 == 0) {
    nsa_set_error("decode_split: head dims %d/%d or fixed_y_maxlen %d / fixed_num_slc_blocks %d / table width %d do "
                  "not fit the final kernel's LDS", D, VD, p.y_cap, p.nb_cap, p.table_stride);
    return NSA_ERR_UNSUPPORTED;
  }
  if (D == 128) return launch_split<128, 128>(p, B, (size_t)lds2, stream);
  if (D == 64) return launch_split<64, 64>(p, B, (size_t)lds2, stream);
  return launch_split<192, 128>(p, B, (size_t)lds2, stream);
}

// LDS of the one-launch decode kernel with `waves` waves that keeps the probabilities of keep_units units
template <int D, int VD>
static size_t fused_lds(const NsaDecodeParams& p, int waves, size_t keep_units) {
  const size_t ntab_c = (size_t)(p.y_cap + p.page_size - 1) / p.page_size;
  const size_t units = (size_t)(p.y_cap + UK - 1) / UK;
  size_t region = 16 * (keep_units * UK + 8) * sizeof(typename UnitFlash<D, VD>::keep_t);
  const size_t swa_part = (size_t)(waves - 1) * 16 * UnitFlash<D, VD>::OLD * sizeof(float);
  if (region < swa_part) region = swa_part;
  region = (region + 15) & ~(size_t)15;
  return slot_bytes<D, VD>(waves) +
         (size_t)(4 * waves * 16 + 16 + (((size_t)p.nb_cap + 3) & ~(size_t)3) + SEL_INTS + ((ntab_c + 3) & ~(size_t)3) +
                  (((size_t)p.table_stride + 3) & ~(size_t)3) + units * 16) * sizeof(float) + region;
}

// Shape of a one-launch decode: waves per workgroup and units whose probabilities stay in LDS (those of the others are
// spilled to scratch memory, if the caller gives it); lds 0: it does not fit (the caller then takes a path with more
// launches).
//   * One workgroup of 8 waves per CU, all probabilities in LDS, while the (request, kv head) pairs fill the CUs less
//     than twice: the waves share a request's units, so more of them shorten the longest request.
//   * From there on two workgroups of 4 waves per CU, so that the serial sections of one (merges, block scores,
//     selection) run beside the loads of the other; their 80 KB hold the probabilities of about 1000 keys (contexts of
//     16K tokens).  64 q / 4 kv heads, d = 128, one / two workgroups: 512 x 4K 505 / 400 us (1.9 GB: 4.7 TB/s, what a
//     copy reaches), 256 x 8K 287 / 231, 128 x 16K 173 / 146, 128 x 4K-32K 171 / 155; with one pair per CU two lose:
//     64 x 4K-32K 78 / 83, 64 x 32K 118 / 126.  With one set of K / V registers per wave (two sets spill: 423 us).
//   * 192 channels: four waves, fp32 probabilities in scratch memory.
struct FusedShape {
  int waves, keep_units;
  size_t lds;
  bool spills;
};
template <int D, int VD>
static FusedShape fused_shape(const NsaDecodeParams& p, int pairs, bool may_spill) {
  const int units = (p.y_cap + UK - 1) / UK;
  auto pg_fits = [&](int waves) { return (size_t)p.y_cap * sizeof(float) <= slot_bytes<D, VD>(waves); };
  if (D > 128) {
    const size_t lds = fused_lds<D, VD>(p, 4, 0);
    return pg_fits(4) && lds <= 160 * 1024 ? FusedShape{4, 0, lds, true} : FusedShape{0, 0, 0, false};
  }
  const size_t lds8 = fused_lds<D, VD>(p, DEC_WAVES, units);
  const FusedShape one = pg_fits(DEC_WAVES) && lds8 <= 160 * 1024 ? FusedShape{DEC_WAVES, units, lds8, false}
                                                                  : FusedShape{0, 0, 0, false};
  const int forced = nsa_tuning_knob("decode_waves", 0);
  const bool many = forced ? forced == 4 : pairs >= 2 * nsa_device_cus();
  if (one.lds == 0 || !many || !pg_fits(4)) return one;
  // (64 channels: three workgroups per CU, what their registers allow)
  constexpr size_t budget = 160 * 1024 / (D <= 64 ? 3 : 2);
  int keep = units;
  while (keep > 0 && fused_lds<D, VD>(p, 4, keep) > budget) keep--;
  const size_t lds = fused_lds<D, VD>(p, 4, keep);
  return lds <= budget && (keep == units || may_spill) ? FusedShape{4, keep, lds, keep < units} : one;
}

static FusedShape fused_shape_of(const NsaDecodeParams& p, int pairs, bool may_spill, int D, int VD) {
  if (D == 128 && VD == 128) return fused_shape<128, 128>(p, pairs, may_spill);
  if (D == 64 && VD == 64) return fused_shape<64, 64>(p, pairs, may_spill);
  if (D == 192 && VD == 128) return fused_shape<192, 128>(p, pairs, may_spill);
  return {0, 0, 0, false};
}

int nsa_decode_fused_lds_bytes(const NsaDecodeParams& p, int D, int VD) {
  return (int)fused_shape_of(p, 1, true, D, VD).lds;
}

int64_t nsa_decode_fused_scratch(const NsaDecodeParams& p, int B, int D, int VD) {
  if (!fused_shape_of(p, B * p.KH, true, D, VD).spills) return 0;
  return (int64_t)B * p.KH * 16 * ((p.y_cap + UK - 1) / UK * UK) * (D <= 128 ? 2 : 4);
}

template <int D, int VD>
static int launch_fused(const NsaDecodeParams& p, const FusedShape& s, dim3 grid, hipStream_t stream) {
  if constexpr (D <= 128) {
    if (s.waves == DEC_WAVES)
      return launch_dyn(decode_fused_kernel<D, VD, DEC_WAVES>, grid, DEC_WAVES, s.lds, stream, "decode_fused_kernel", 0,
                        p, s.keep_units);
  }
  return launch_dyn(decode_fused_kernel<D, VD, 4>, grid, 4, s.lds, stream, "decode_fused_kernel", 0, p, s.keep_units);
}

int nsa_decode_fused_launch(const NsaDecodeParams& p, int B, int D, int VD, hipStream_t stream) {
  if (B <= 0) return NSA_OK;
  const FusedShape s = fused_shape_of(p, B * p.KH, p.sp_keep_p != nullptr, D, VD);
  if (s.spills && p.sp_keep_p == nullptr) {
    nsa_set_error("decode_fused: head dims %d/%d need scratch memory", D, VD);
    return NSA_ERR_WORKSPACE;
  }
  if (s.lds == 0) {
    nsa_set_error("decode_fused: head dims %d/%d or fixed_y_maxlen %d / fixed_num_slc_blocks %d / table width %d do "
                  "not fit the one-launch kernel (160 KB of LDS); use the two-launch path", D, VD, p.y_cap, p.nb_cap,
                  p.table_stride);
    return NSA_ERR_UNSUPPORTED;
  }
  const dim3 grid(B, p.KH);
  if (D == 128) return launch_fused<128, 128>(p, s, grid, stream);
  if (D == 64) return launch_fused<64, 64>(p, s, grid, stream);
  return launch_fused<192, 128>(p, s, grid, stream);
}
