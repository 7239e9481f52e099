// dK / dV of the three attention branches for 8, 16, 32 or 64 q-heads per kv head and head dims that are multiples of 64:
// the arithmetic and the work items of nsa_bwd_dkdv.hip (which keeps the other shapes) in a kernel that fits two waves on a
// SIMD.  Alone on the GPU, us before and now: compressed branch, 64 heads of 128, 64K tokens 10989 -> 8552 (1.03 PFLOP/s of
// executed products), window 3668 -> 2513; 8 x 6K tokens 1389 -> 890 and 3231 -> 2224, selected 4582 -> 4367 with the dS
// stored beside it; 32 heads of 192 / 128 (one wave per SIMD), 16K tokens, selected 4574 -> 1535.
//
// What bounds it: LDS reads and matrix instructions about equally (each of the four operands is read once per matrix
// instruction of 32 cycles and SIMD, 4 KB per CU, which LDS delivers in 32 cycles; compressed branch at 64K tokens: LDS busy
// 53 % of the cycles, matrix cores 60 %, at the 1.64 GHz that the power limit leaves), then instruction issue.  So nothing is
// computed per lane that is uniform, and the order of reads, matrix instructions and softmax arithmetic is fixed (below).
//
// A wave keeps the K and V fragments of 32 keys and their dK / dV accumulators in registers (192 of 256 at 128 channels);
// 64 query rows at a time pass through LDS.  What makes the rest fit:
//  * The rows go from global memory straight into LDS (global_load_lds), two tiles in turn, one barrier per tile.  Eight
//    rows are the heads of one token (8 divides the group size), so a load's address is a scalar base plus a per-lane
//    offset that never changes.
//  * Position, visibility and the place of the stored dS belong to eight rows as well: scalars, taken from one register
//    whose lane i holds the token of row group i / 8.
//  * -lse / c and -delta are what the accumulators of S = Q K^T and dP = dO V^T start from, so the probability is
//    exp2(c S) and dS = P o dP without registers for either.
// Two tile buffers are two named arrays: with one indexed array the compiler waits for the loads in flight before every read
// of the other half.
//
// LDS layout of a tile: rows in groups of eight, 64 channels at a time, as 1 KB blocks of 8 rows x 128 bytes (what one load
// instruction of a wave writes); the 16-byte chunk c of row r sits at position c ^ (r & 7) ^ ((r >> 3) & 1), which spreads
// both the row fragments (32 rows x 16 bytes) and the transposed ones (8 rows x 64 bytes) over all banks.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include <utility>

namespace {

constexpr int MODE_CMP = 0;
constexpr int MODE_SWA = 1;
constexpr int MODE_SLC = 2;

typedef __attribute__((address_space(1))) const void* nsa_gptr_t;
typedef __attribute__((address_space(3))) void* nsa_lptr_t;

// keys per workgroup: four waves of 32 keys; selection blocks of up to 64 keys: two of them, each in two waves that take
// half of the rows and add up their results at the end
template <int MODE, bool NARROW>
constexpr int key_waves() { return MODE == MODE_SLC && NARROW ? 2 : 4; }

// fn(integral_constant 0 .. N - 1): the matrix instruction stream of a tile is longer than what a loop is unrolled to
template <class Fn, int... I>
NSA_DEVICE void for_constants(Fn fn, std::integer_sequence<int, I...>) { (fn(std::integral_constant<int, I>{}), ...); }
template <int N, class Fn>
NSA_DEVICE void static_for(Fn fn) { for_constants(fn, std::make_integer_sequence<int, N>{}); }

// x ^ X, computed where it is asked for
template <int X>
NSA_DEVICE int xored(int x) {
  int r = x;
  if constexpr (X != 0) asm volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(X), "v"(x));
  return r;
}
// s_waitcnt immediates: vmcnt(0) (+ n: vmcnt(n), n < 16), lgkmcnt(0)
constexpr int WAIT_LOADS = 0x0f70, WAIT_LDS = 0xc07f;

constexpr int DMA_LIST = 1024;  // tokens of a work item that the kernel holds in LDS

constexpr int dma_waves(int d) { return d <= 128 ? 2 : 1; }

// DSH > 0: the dS is also stored, for the dQ of the same rows.  MODE_SLC: that of every (token, block), in blobs of DSH heads
// (nsa_slc_bwd_dq_ds.hip); else that of every 64 rows and 32 keys, in four blobs of 16 rows (nsa_bwd_dq_ds.hip).  No path through
// the tile loop leaves the stores out (rows without an entry, and waves that see nothing, store to a place that nobody reads):
// where one did, the compiler waited for all of them and not just for the next tile's loads.
template <int D, int VD, int MODE, bool NARROW, int DSH>
__global__ __launch_bounds__(256, dma_waves(D)) void bwd_dkdv_dma_kernel(NsaBwdTileParams p) {
  constexpr bool DS = DSH > 0;
  constexpr int NW = 4;
  constexpr int NK = key_waves<MODE, NARROW>();  // key groups
  constexpr int RG = NW / NK;                    // row groups
  constexpr int KW = NK * 32;
  constexpr int RT = 64;
  constexpr int MT = RT / 32 / RG;               // 32-row steps of a wave per tile
  constexpr int QS = D / 64, OS = VD / 64;       // 1 KB blocks per eight rows
  constexpr int BLK = 512;                       // elements of a block
  constexpr int GS = (QS + OS) * BLK;            // eight rows: the Q blocks, then the dO blocks
  constexpr int TILE = (RT / 8) * GS;
  // Behind a tile's rows their statistics: -lse / c, -delta.  (In arrays of their own: the compiler takes a read of an array
  // that no load goes to for one that may meet any of them, and waits for those in flight.)
  constexpr int STAT = TILE * 2;                 // byte offset
  __shared__ __attribute__((aligned(1024))) bf16_t tile_a[TILE + 4 * RT];
  __shared__ __attribute__((aligned(1024))) bf16_t tile_b[TILE + 4 * RT];
  __shared__ int tok_s[MODE == MODE_SLC ? DMA_LIST : 1];           // the work item's tokens and, for the stored dS, slots
  __shared__ uint8_t slot_s[DS ? DMA_LIST : 1];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave % NK, rg = wave / NK;
  const int l32 = lane & 31;
  const int hl = lane >> 5;
  const int kh = blockIdx.z;
  const int G = p.G;
  const int gshift = __builtin_ctz(G);

  // ---- work item: the keys and the tokens n_begin .. n_end - 1 (MODE_SLC: positions in the list)
  int b, key0, n_begin, n_end;
  const int32_t* list = nullptr;
  const uint8_t* slots = nullptr;
  if (MODE == MODE_SLC) {
    const int32_t* ioff = p.item_off + kh * p.csr_sh;
    const int w = blockIdx.x;
    if (w >= ioff[p.nblk_total]) return;
    int lo = 0, hi = p.nblk_total;  // last jb with ioff[jb] <= w
    while (hi - lo > 1) {
      int mid = (lo + hi) >> 1;
      if (ioff[mid] <= w) lo = mid; else hi = mid;
    }
    const int jb = lo;
    b = p.blk_seq[jb];
    key0 = (jb - p.kblk_cu[b]) * p.block_size + blockIdx.y * KW;
    const int s0 = p.csr_off[kh * p.csr_sh + jb];
    const int s1 = p.csr_off[kh * p.csr_sh + jb + 1];
    const int a = s0 + (w - ioff[jb]) * p.chunk_tokens;
    list = p.csr_tok + a;
    if (DS) slots = p.csr_slot + a;
    n_begin = 0;
    n_end = min(s1 - a, p.chunk_tokens);
  } else {
    b = blockIdx.y;
  }
  const int x0 = p.x_cu[b];
  int xl = p.x_cu[b + 1] - x0;
  const int tshift = 6 - gshift;  // log2 of the tokens of a 64-row tile
  // stored dS of the range-keyed branches: tiles of 64 rows from the first of a sequence on
  constexpr bool TILE_DS = DS && MODE != MODE_SLC;
  int lo = 0, hi = xl;  // the launch's share of the sequence
  if (TILE_DS) nsa_local_range(p.tok0, p.tok1, x0, xl, lo, hi);
  if (MODE == MODE_SWA && p.t_end > 0) xl = min(xl, p.t_end);
  int nkeys, kbase;
  if (MODE == MODE_CMP) {
    kbase = p.k_cu[b];
    nkeys = p.k_cu[b + 1] - kbase;
    // only the (key tile, query chunk) pairs that have visible rows, key-tile major, as nsa_bwd_dkdv.hip numbers them
    const int nch = cdiv_i(max(hi - lo, 0), p.q_chunk_tokens);
    int rem = blockIdx.x, ktile = 0, ch = -1;
    for (; ktile * KW < nkeys; ktile++) {
      const int fc = min(nch, max(p.stride * ktile * KW + p.kernel_size - 1 - lo, 0) / p.q_chunk_tokens);
      const int cnt = nch - fc;
      if (rem < cnt) { ch = fc + rem; break; }
      rem -= cnt;
    }
    if (ch < 0) return;
    key0 = ktile * KW;
    n_begin = max(lo + ch * p.q_chunk_tokens, p.stride * key0 + p.kernel_size - 1);
    n_end = min(lo + (ch + 1) * p.q_chunk_tokens, hi);
    if (n_begin >= n_end) return;
    if (TILE_DS) n_begin &= -(1 << tshift);  // (chunks and ranges begin with a tile)
  } else {
    kbase = x0;
    nkeys = xl;
    if (MODE == MODE_SLC) nkeys = min(xl, (key0 / p.block_size + 1) * p.block_size);
    if (MODE == MODE_SWA) {
      const int ktile = blockIdx.x / p.grid_chunks;
      key0 = lo + ktile * KW;
      if (key0 >= min(nkeys, hi)) return;
      n_begin = key0 + (TILE_DS ? p.min_dist & -(1 << tshift) : p.min_dist) +
                (blockIdx.x - ktile * p.grid_chunks) * p.q_chunk_tokens;
      n_end = min(min(xl, key0 + KW + p.window), n_begin + p.q_chunk_tokens);
    } else if (key0 >= nkeys) {
      return;
    }
  }
  if (n_begin >= n_end) return;

  if (MODE == MODE_SLC) {
    for (int i = threadIdx.x; i < n_end; i += 256) {
      tok_s[i] = list[i];
      if (DS) slot_s[i] = slots[i];
    }
    __syncthreads();
  }

  // ---- this wave's keys: K and V fragments as B operands
  const int kw0 = key0 + kg * 32;
  const bool wave_has_keys = kw0 < nkeys;
  bf16x8 kf[D / 16], vf[VD / 16];
  {
    const int kr = min(kw0 + l32, nkeys - 1);
    const bf16_t* kp = p.k + ((int64_t)kbase + kr) * p.k_sr + (int64_t)kh * p.k_sh + hl * 8;
#pragma unroll
    for (int kc = 0; kc < D / 16; kc++) kf[kc] = ld_global_b128(kp + kc * 16);
    const bf16_t* vp = p.v + ((int64_t)kbase + kr) * p.v_sr + (int64_t)kh * p.v_sh + hl * 8;
#pragma unroll
    for (int kc = 0; kc < VD / 16; kc++) vf[kc] = ld_global_b128(vp + kc * 16);
  }
  const float sc = p.scale_log2;

  // ---- staging: wave w moves the row groups w and w + 4 of every tile
  const int n_step = RT >> gshift;  // tokens per tile
  const int n_last = n_end - 1;
  // number (of the token, or of the list entry) that row group grp of the tile starting at n0 belongs to
  auto nth = [&](int n0, int grp) { return min(n0 + ((grp * 8) >> gshift), n_last); };
  // MODE_SLC: lane i holds the token of row group i / 8
  auto tokens_of = [&](int n0) { return MODE == MODE_SLC ? tok_s[nth(n0, lane_id() >> 3)] : 0; };
  auto position = [&](int tv, int n0, int grp) { return MODE == MODE_SLC ? __builtin_amdgcn_readlane(tv, grp * 8) : nth(n0, grp); };
  auto stage = [&](int tv, int n0, bf16_t* buf) {
    // byte offsets of this lane's piece (the chunk that its position holds) from the first of eight rows
    const int ln = lane_id(), r8 = ln >> 3;
    const uint32_t cpos = (uint32_t)((ln & 7) ^ r8 ^ (wave & 1)) * 16;
    const uint32_t qoff = (uint32_t)r8 * (uint32_t)(p.q_sh * 2) + cpos, ooff = (uint32_t)r8 * (uint32_t)(p.do_sh * 2) + cpos;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int grp = wave + h * 4;
      const int64_t tok = x0 + position(tv, n0, grp);
      const int head = kh * G + ((grp * 8) & (G - 1));
      const char* qb = reinterpret_cast<const char*>(p.q + tok * p.q_st + (int64_t)head * p.q_sh);
      const char* ob = reinterpret_cast<const char*>(p.dO + tok * p.do_st + (int64_t)head * p.do_sh);
      // (the statements without instructions: scalar base + 32-bit lane offset, not a 64-bit address per lane)
#pragma unroll
      for (int s = 0; s < QS + OS; s++) {
        const char* at = s < QS ? qb + s * 128 : ob + (s - QS) * 128;
        uint32_t off = s < QS ? qoff : ooff;
        asm volatile("" : "+s"(at), "+v"(off));
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + off), (nsa_lptr_t)(buf + grp * GS + s * BLK), 16, 0, 0);
      }
    }
  };
  // waves 0, 2: log-sum-exp of row `lane`, waves 1, 3: delta (0 and 1 store theirs)
  const float* const sptr = (wave & 1) ? p.delta : p.lse;
  const int64_t s_st = (wave & 1) ? p.delta_st : p.lse_st, s_sh = (wave & 1) ? p.delta_sh : p.lse_sh;
  const float s_mul = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (wave & 1) ? -1.f : -1.f / sc)));
  auto stat_of = [&](int tv, int n0) {
    const int ln = lane_id();
    const int64_t tok = x0 + (MODE == MODE_SLC ? tv : nth(n0, ln >> 3));
    return sptr[tok * s_st + (int64_t)(kh * G + (ln & (G - 1))) * s_sh];
  };

  // ---- fragment addresses: byte offsets of the lane parts; the rest are compile-time offsets and one XOR
  const int i16 = lane & 15, g16 = lane >> 4;
  // row fragments: row l32 of a 32-row step, chunk pair j: fa0 ^ (j << 5)
  const int fa0 = (rg * MT * 4 + (l32 >> 3)) * GS * 2 + (l32 & 7) * 128 + (hl ^ (l32 & 7) ^ ((l32 >> 3) & 1)) * 16;
  // transposed fragments: row r = hl * 4 + i16 / 4 of eight rows, 32-channel half j of a block: ta0 ^ (j << 6); of the
  // following eight rows: ta0 ^ (j << 6) ^ 16, one group further
  const int tr_row = hl * 4 + (i16 >> 2);
  const int ta0 = rg * MT * 4 * GS * 2 + tr_row * 128 + (((g16 & 1) * 2 + ((i16 & 3) >> 1)) ^ tr_row) * 16 + (i16 & 1) * 8;

  float st_reg;
  // stored dS: tile number of the work item's first tile, place for what nobody reads
  int64_t ds_head = 0, ds_dump = 0;
  int ds_tile = 0;
  if (TILE_DS) {
    ds_head = (int64_t)kh * p.ds_sh;
    ds_dump = (int64_t)p.KH * p.ds_sh + ((blockIdx.x & 15) * 4 + wave) * 512;  // (and three blobs more)
    ds_tile = nsa_ds_tile(p.ds_tiles, p.ds_seq_tiles, x0 >> tshift, b, n_begin >> tshift);
  }

  f32x16 dkacc[D / 32], dvacc[VD / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dkacc[dt][i] = 0.f;
#pragma unroll
  for (int dt = 0; dt < VD / 32; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dvacc[dt][i] = 0.f;
  // one tile: `cur` holds it (its loads are in flight), `nxt` receives the next one
  auto step = [&](bf16_t* cur, bf16_t* nxt, int n0) {
    const int tv = tokens_of(n0), tvn = tokens_of(n0 + n_step);
    // lane i: place of the dS of row group i / 8 (rows without a token of the list, waves without keys: an entry nobody reads)
    int ds_ent = 0;
    if (MODE == MODE_SLC && DS) {
      const int grp = lane_id() >> 3, n = n0 + ((grp * 8) >> gshift);
      const int tok = x0 + tv - p.ds_tok0;
      const int e = (tok * p.top_n + slot_s[min(n, n_last)]) * (G > 16 ? G >> 4 : 1) + (((grp * 8) & (G - 1)) >> 4);
      ds_ent = wave_has_keys && n < n_end && (unsigned)tok < (unsigned)p.ds_ntok ? e : p.ds_dump;
    }
    // The loads of this tile are this wave's oldest; younger are the previous tile's dS stores (two per 32 rows).
    // (The builtin, not inline assembly: the compiler has to know that they have landed.)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT_LOADS + (DSH == 8 ? MT * 4 : DS ? MT * 2 : 0));
    asm volatile("" ::: "memory");
    if (wave < 2) reinterpret_cast<float*>(cur + TILE)[wave * RT + lane_id()] = st_reg * s_mul;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT_LDS);
    __builtin_amdgcn_s_barrier();  // everybody's rows of this tile are there; nobody reads the other buffer any more
    asm volatile("" ::: "memory");
    // (behind the last tile the last tokens are loaded once more: no branch around loads that the waits have to count)
    stage(tvn, n0 + n_step, nxt);
    st_reg = stat_of(tvn, n0 + n_step);

    const int n_in = min(n_step, n_end - n0);  // tokens of the tile
    const int t_min = position(tv, n0, 0);
    const int t_max = position(tv, n0, 7);
    bool any_vis, full_vis;
    if (MODE == MODE_CMP) {
      any_vis = t_max >= p.stride * kw0 + p.kernel_size - 1;
      full_vis = n_in == n_step && t_min >= p.stride * (kw0 + 31) + p.kernel_size - 1 && kw0 + 31 < nkeys;
    } else if (MODE == MODE_SWA) {
      any_vis = kw0 <= t_max - p.min_dist && kw0 + 31 >= t_min - p.window;
      full_vis = n_in == n_step && kw0 + 31 <= t_min - p.min_dist && kw0 >= t_max - p.window && kw0 + 31 < nkeys;
    } else {
      any_vis = kw0 <= t_max;
      full_vis = n_in == n_step && kw0 + 31 <= t_min && kw0 + 31 < nkeys;
    }
    const bool seen = any_vis && wave_has_keys;
    if (!DS && !seen) return;
    bf16_t* ds_out = nullptr;
    if (TILE_DS) {
      int tile = ds_tile + ((n0 - n_begin) >> tshift);
      if (tile >= p.ds_tiles) tile -= p.ds_tiles;
      const int unit = (kw0 >> 5) - (MODE == MODE_SWA ? max(0, n0 - p.window) >> 5 : 0);
      ds_out = p.ds + (seen ? ds_head + ((int64_t)tile * p.ds_pitch + unit) * 2048 : ds_dump);
    }

    // The A operands of a step's matrix instructions, in the order in which they are used: Q rows (S), dO rows (dP),
    // dO transposed (dV), Q transposed (dK).  They are read PF operands ahead, and the softmax arithmetic is placed between
    // the matrix instructions that do not wait for it; sched_barrier keeps the compiler from collecting either.
    constexpr int F_DP = D / 16, F_DV = F_DP + VD / 16, F_DK = F_DV + VD / 16, NF = F_DK + D / 16;
    constexpr int PF = MODE == MODE_SLC && D > 64 ? 1 : 2;
    const char* const base = reinterpret_cast<const char*>(cur);
    bf16x8 ring[PF + 1];
    // Operands whose addresses share an XOR follow each other, and the XOR is redone for every such run: held in registers
    // for all of them, they would push fragments out.
    int ax = 0, ay = 0;
    auto order_kc = [](int i, int n) constexpr { return n == 4 ? i : (i % (n / 4)) * 4 + i / (n / 4); };  // 0 4 1 5 2 6 3 7
    auto order_dt = [](int i, int n) constexpr { return (i % (n / 2)) * 2 + i / (n / 2); };          // 0 2 1 3
    auto load = [&](auto at_tag) -> bf16x8 {
      constexpr int mt = decltype(at_tag)::value / NF, f = decltype(at_tag)::value % NF;
      if constexpr (f < F_DV) {
        constexpr int nk = f < F_DP ? D / 16 : VD / 16, i = f < F_DP ? f : f - F_DP, kc = order_kc(i, nk);
        if constexpr (i % (nk / 4) == 0) {
          ax = xored<(kc % 4) << 5>(fa0);
        }
        return *reinterpret_cast<const bf16x8*>(base + (ax + (mt * 4 * GS * 2 + ((f < F_DP ? 0 : QS) + kc / 4) * BLK * 2)));
      } else {
        constexpr bool of_q = f >= F_DK;
        constexpr int n = f - (of_q ? F_DK : F_DV), nd = of_q ? D / 32 : VD / 32, c = n / nd, dt = order_dt(n % nd, nd);
        if constexpr (n % (nd / 2) == 0) {
          ax = xored<(dt % 2) << 6>(ta0);
          ay = xored<((dt % 2) << 6) + 16>(ta0);
        }
        constexpr int at = (mt * 4 + c * 2) * GS * 2 + ((of_q ? 0 : QS) + dt / 2) * BLK * 2;
        return cat4(lds_read_tr(reinterpret_cast<const bf16_t*>(base + (ax + at))),
                    lds_read_tr(reinterpret_cast<const bf16_t*>(base + (ay + at + GS * 2))));
      }
    };
    f32x16 s, pd;
    bf16x8 pf, df[2];
    auto init = [&](f32x16& acc, int which, int mt) {
      const int sa0 = rg * MT * 128 + (lane_id() >> 5) * 16;
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(base + (sa0 + STAT + (which * RT + mt * 32 + i4 * 8) * 4));
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i4 * 4 + i] = v[i];
      }
    };
    auto half8 = [&](const f32x16& x, int c) {
      return pack8(x[c * 8 + 0], x[c * 8 + 1], x[c * 8 + 2], x[c * 8 + 3], x[c * 8 + 4], x[c * 8 + 5], x[c * 8 + 6], x[c * 8 + 7]);
    };
    init(s, 0, 0);
    static_for<PF>([&](auto ft) { ring[decltype(ft)::value] = load(ft); });
    static_for<MT * NF>([&](auto ft) {
        constexpr int ff = decltype(ft)::value, mt = ff / NF, f = ff % NF;
        if constexpr (ff + PF < MT * NF) ring[(ff + PF) % (PF + 1)] = load(std::integral_constant<int, ff + PF>{});
        const bf16x8 a = ring[ff % (PF + 1)];
        if constexpr (f < F_DP) {                           // S
          s = mfma32(a, kf[order_kc(f, F_DP)], s);
          if (f == F_DP / 2) init(pd, 1, mt);
        } else if constexpr (f < F_DV) {                    // dP, and P from S
          constexpr int kc = f - F_DP, n = F_DV - F_DP;
          pd = mfma32(a, vf[order_kc(kc, n)], pd);
#pragma unroll
          for (int i = 0; i < 16; i++)
            if (i * (n - 1) / 16 + 1 == kc) s[i] = fast_exp2(s[i] * sc);
          if (f == F_DV - 1 && !full_vis) {  // wave-uniform: only tiles that straddle a visibility boundary pay for the mask
            asm volatile("");  // keeps it a branch
            // a key is visible from the positions lo .. hi
            const int my_key = kw0 + (lane_id() & 31);
            int lo = MODE == MODE_CMP ? p.stride * my_key + p.kernel_size - 1 : MODE == MODE_SWA ? my_key + p.min_dist : my_key;
            if (my_key >= nkeys) lo = 0x7fffffff;
            const int hi = MODE == MODE_SWA ? my_key + p.window : 0;
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
              const int grp = (rg * MT + mt) * 4 + i4;
              const int t = n0 + ((grp * 8) >> gshift) < n_end ? position(tv, n0, grp) : -0x40000000;  // scalar
              const bool vis = t >= lo && (MODE != MODE_SWA || t <= hi);
#pragma unroll
              for (int i = 0; i < 4; i++) {
                s[i4 * 4 + i] = vis ? s[i4 * 4 + i] : 0.f;
                // (dQ sums over all keys of a unit: what a query may not see must not reach it through 0 * inf either)
                if (DS) pd[i4 * 4 + i] = vis ? pd[i4 * 4 + i] : 0.f;
              }
            }
          }
        } else if constexpr (f < F_DK) {                    // dV, and dS from P and dP
          constexpr int nd = VD / 32;
          constexpr int c = (f - F_DV) / nd, dt = (f - F_DV) % nd;
          if (dt == 0) pf = half8(s, c);
          dvacc[order_dt(dt, nd)] = mfma32(a, pf, dvacc[order_dt(dt, nd)]);
#pragma unroll
          for (int i = 0; i < 8; i++)
            if (i * nd / 8 == dt) pd[c * 8 + i] *= s[c * 8 + i];
          if (dt == nd - 1) df[c] = half8(pd, c);
        } else {                                            // dK
          constexpr int nd = D / 32;
          constexpr int c = (f - F_DK) / nd, dt = (f - F_DK) % nd;
          dkacc[order_dt(dt, nd)] = mfma32(a, df[c], dkacc[order_dt(dt, nd)]);
          if (dt == 0 && c == 1 && mt + 1 < MT) init(s, 0, mt + 1);
          if (TILE_DS && dt == 0) {
            __builtin_nontemporal_store(__builtin_bit_cast(u32x4, df[c]), reinterpret_cast<u32x4*>(ds_out + ((mt * 2 + c) * 512 + lane_id() * 8)));
          } else if (DS && dt == 0) {
            const int upb = p.block_size >> 5, unit = min((int)blockIdx.y * NK + kg, upb - 1);  // 32-key units of the block
            auto entry = [&](int grp) { return (int64_t)__builtin_amdgcn_readlane(ds_ent, grp * 8) * upb + unit; };
            const int grp = (rg * MT + mt) * 4 + c * 2;
            bf16_t* const out = p.ds + kh * p.ds_sh;
            if (DSH == 8) {
              *reinterpret_cast<bf16x4*>(out + entry(grp) * 256 + lane * 4) = __builtin_shufflevector(df[c], df[c], 0, 1, 2, 3);
              *reinterpret_cast<bf16x4*>(out + entry(grp + 1) * 256 + lane * 4) =
                  __builtin_shufflevector(df[c], df[c], 4, 5, 6, 7);
            } else {
              *reinterpret_cast<bf16x8*>(out + entry(grp) * 512 + lane * 8) = df[c];
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
    });
  };

  {
    const int tv = tokens_of(n_begin);
    stage(tv, n_begin, tile_a);
    st_reg = stat_of(tv, n_begin);
  }
  int n0 = n_begin;
  // TILE_DS: tiles of which a wave sees nothing, two at a time: it only helps with the rows.  (Not a branch inside a step: the
  // compiler then spills half of the accumulators.)
  int n_stop = n_end;
  auto skim = [&](bf16_t* cur, bf16_t* nxt) {
    const int tvn = tokens_of(n0 + n_step);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT_LOADS);
    asm volatile("" ::: "memory");
    if (wave < 2) reinterpret_cast<float*>(cur + TILE)[wave * RT + lane_id()] = st_reg * s_mul;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT_LDS);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    stage(tvn, n0 + n_step, nxt);
    st_reg = stat_of(tvn, n0 + n_step);
    n0 += n_step;
  };
  if constexpr (TILE_DS) {
    int n_first = MODE == MODE_CMP ? p.stride * kw0 + p.kernel_size - 1 : kw0 + p.min_dist;
    if (!wave_has_keys) n_first = n_end;
    if (MODE == MODE_SWA) n_stop = min(n_end, kw0 + 32 + p.window);
    while (n0 + 2 * n_step <= n_first && n0 + 2 * n_step < n_end) {
      skim(tile_a, tile_b);
      skim(tile_b, tile_a);
    }
  }
  if (DS) __builtin_amdgcn_s_waitcnt(WAIT_LOADS);  // no stores behind the first tile's loads yet
  for (;;) {
    step(tile_a, tile_b, n0);
    n0 += n_step;
    if (n0 >= n_end) break;
    step(tile_b, tile_a, n0);
    n0 += n_step;
    if (n0 >= n_stop) break;
  }
  if constexpr (TILE_DS) {
    while (n0 < n_end) {
      skim(tile_a, tile_b);
      if (n0 >= n_end) break;
      skim(tile_b, tile_a);
    }
  }

  // ---- epilogue: the tile buffers are free once the loads behind the last tile have landed
  __syncthreads();
  const float osc = p.sm_scale;
  const int le = lane_id(), l32e = le & 31, hle = le >> 5;
  // Accumulators hold one key per lane; they leave through LDS, C channels of the wave's 32 keys at a time, as row pieces.
  constexpr int HALF_BYTES = TILE * 2;  // two waves per tile buffer
  constexpr int C = 2 * 32 * 68 * 4 <= HALF_BYTES ? 64 : 32, ELD = C + 4;
  static_assert(2 * 32 * ELD * 4 <= HALF_BYTES, "a tile buffer holds the strips of two waves");
  char* const mine = reinterpret_cast<char*>((wave & 1) ? tile_b : tile_a);
  float* const strip = reinterpret_cast<float*>(mine + (wave >> 1) * (HALF_BYTES / 2));
  auto lds_order = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto emit = [&](auto& acc, auto width_tag, void* base, int64_t off, int64_t row_stride, float scale, int n_keys) {
    constexpr int W = decltype(width_tag)::value;
#pragma unroll
    for (int c0 = 0; c0 < W; c0 += C) {
#pragma unroll
      for (int q4 = 0; q4 < C / 8; q4++) {
        const int dt = (c0 + q4 * 8) / 32, i0 = (q4 % 4) * 4;
        *reinterpret_cast<f32x4*>(&strip[l32e * ELD + q4 * 8 + hle * 4]) =
            f32x4{acc[dt][i0] * scale, acc[dt][i0 + 1] * scale, acc[dt][i0 + 2] * scale, acc[dt][i0 + 3] * scale};
      }
      lds_order();
      if (p.dkv_mode == 3) {
        constexpr int RPI = 64 / C;  // rows per instruction
        const int r0 = le / C, col = le % C;
#pragma unroll
        for (int r = 0; r < 32; r += RPI)
          if (r + r0 < n_keys)
            unsafeAtomicAdd((float*)base + off + (int64_t)(r + r0) * row_stride + c0 + col, strip[(r + r0) * ELD + col]);
      } else {
        constexpr int LPR = C / 4;  // lanes per row, four channels each
        const int r0 = le / LPR, col = (le % LPR) * 4;
#pragma unroll
        for (int r = 0; r < 32; r += 64 / LPR) {
          if (r + r0 >= n_keys) continue;
          const f32x4 val = *reinterpret_cast<const f32x4*>(&strip[(r + r0) * ELD + col]);
          const int64_t at = off + (int64_t)(r + r0) * row_stride + c0 + col;
          if (p.dkv_mode == 0) *reinterpret_cast<bf16x4*>((bf16_t*)base + at) = pack4(val[0], val[1], val[2], val[3]);
          else *reinterpret_cast<f32x4*>((float*)base + at) = val;
        }
      }
      lds_order();
    }
  };
  // Row groups: wave (kg, 0) adds up and stores dK, wave (kg, 1) dV.  What they hand to each other lies in LDS as the lanes
  // hold it.
  if constexpr (RG == 2) {
    char* const boxes = reinterpret_cast<char*>(kg ? tile_b : tile_a);
    f32x4* const box_v = reinterpret_cast<f32x4*>(boxes) + le;
    f32x4* const box_k = reinterpret_cast<f32x4*>(boxes + VD * 128) + le;
    static_assert((D + VD) * 128 <= TILE * 2, "a tile buffer holds the halves that two waves hand over");
    auto give = [&](auto& acc, f32x4* box, auto n_tag) {
#pragma unroll
      for (int n = 0; n < decltype(n_tag)::value * 4; n++)
        box[n * 64] = f32x4{acc[n / 4][n % 4 * 4], acc[n / 4][n % 4 * 4 + 1], acc[n / 4][n % 4 * 4 + 2], acc[n / 4][n % 4 * 4 + 3]};
    };
    auto take = [&](auto& acc, const f32x4* box, auto n_tag) {
#pragma unroll
      for (int n = 0; n < decltype(n_tag)::value * 4; n++) {
        const f32x4 v = box[n * 64];
#pragma unroll
        for (int i = 0; i < 4; i++) acc[n / 4][n % 4 * 4 + i] += v[i];
      }
    };
    if (rg == 0) give(dvacc, box_v, std::integral_constant<int, VD / 32>{});
    else give(dkacc, box_k, std::integral_constant<int, D / 32>{});
    __syncthreads();
    if (rg == 0) take(dkacc, box_k, std::integral_constant<int, D / 32>{});
    else take(dvacc, box_v, std::integral_constant<int, VD / 32>{});
    __syncthreads();
  }
  if (!wave_has_keys) return;
  const int n_keys = min(32, nkeys - kw0);
  // dkv_mode 4: the workgroup's own slot of the partial buffers (summed in a fixed order by a second kernel)
  const int64_t slot = MODE == MODE_SLC ? ((int64_t)kh * gridDim.x + blockIdx.x) * gridDim.y + blockIdx.y
                                        : ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * p.KH + kh;
  const int64_t part_row = slot * KW + kg * 32, row = (int64_t)kbase + kw0;
  if (RG == 1 || rg == 0) {
    if (p.dkv_mode == 4) emit(dkacc, std::integral_constant<int, D>{}, p.part_dk, part_row * D, D, osc, n_keys);
    else emit(dkacc, std::integral_constant<int, D>{}, p.dk, row * p.dk_sr + (int64_t)kh * p.dk_sh, p.dk_sr, osc, n_keys);
  }
  if (RG == 1 || rg == 1) {
    if (p.dkv_mode == 4) emit(dvacc, std::integral_constant<int, VD>{}, p.part_dv, part_row * VD, VD, 1.f, n_keys);
    else emit(dvacc, std::integral_constant<int, VD>{}, p.dv, row * p.dv_sr + (int64_t)kh * p.dv_sh, p.dv_sr, 1.f, n_keys);
  }
}

template <int D, int VD>
int launch(const NsaBwdTileParams& p, int mode, dim3 grid, hipStream_t stream) {
  constexpr int TILE_DSH = D >= 128 ? 16 : 0;  // (64 channels: dq is faster without)
  if (mode == MODE_CMP) {
    if (TILE_DSH == 0 || p.ds == nullptr) bwd_dkdv_dma_kernel<D, VD, MODE_CMP, false, 0><<<grid, 256, 0, stream>>>(p);
    else bwd_dkdv_dma_kernel<D, VD, MODE_CMP, false, TILE_DSH><<<grid, 256, 0, stream>>>(p);
  } else if (mode == MODE_SWA) {
    if (TILE_DSH == 0 || p.ds == nullptr) bwd_dkdv_dma_kernel<D, VD, MODE_SWA, false, 0><<<grid, 256, 0, stream>>>(p);
    else bwd_dkdv_dma_kernel<D, VD, MODE_SWA, false, TILE_DSH><<<grid, 256, 0, stream>>>(p);
  }
  else if (p.block_size <= 64) {
    if (p.ds == nullptr) bwd_dkdv_dma_kernel<D, VD, MODE_SLC, true, 0><<<grid, 256, 0, stream>>>(p);
    else if (p.G == 8) bwd_dkdv_dma_kernel<D, VD, MODE_SLC, true, 8><<<grid, 256, 0, stream>>>(p);
    else bwd_dkdv_dma_kernel<D, VD, MODE_SLC, true, 16><<<grid, 256, 0, stream>>>(p);
  } else {
    if (p.ds == nullptr) bwd_dkdv_dma_kernel<D, VD, MODE_SLC, false, 0><<<grid, 256, 0, stream>>>(p);
    else if (p.G == 8) bwd_dkdv_dma_kernel<D, VD, MODE_SLC, false, 8><<<grid, 256, 0, stream>>>(p);
    else bwd_dkdv_dma_kernel<D, VD, MODE_SLC, false, 16><<<grid, 256, 0, stream>>>(p);
  }
  return nsa_check_launch("bwd_dkdv_dma_kernel");
}

}  // namespace

bool nsa_bwd_dkdv_dma_takes(const NsaBwdTileParams& p, int D, int VD) {
  if (p.G != 8 && p.G != 16 && p.G != 32 && p.G != 64) return false;
  // the lanes' offsets inside eight rows are 32 bits wide
  if (p.q_sh < 0 || p.do_sh < 0 || p.q_sh > (1 << 28) || p.do_sh > (1 << 28)) return false;
  // (the log-sum-exps are divided by the scale)
  if (!(p.scale_log2 > 1e-12f && p.scale_log2 < 1e12f)) return false;
  if (p.csr_tok != nullptr && p.chunk_tokens > DMA_LIST) return false;
  return (D == 128 && VD == 128) || (D == 64 && VD == 64) || (D == 192 && VD == 128);
}

int nsa_bwd_dkdv_dma_launch(const NsaBwdTileParams& p, int mode, dim3 grid, int D, int VD, hipStream_t stream) {
  if (D == 192) return launch<192, 128>(p, mode, grid, stream);
  return D == 128 ? launch<128, 128>(p, mode, grid, stream) : launch<64, 64>(p, mode, grid, stream);
}
