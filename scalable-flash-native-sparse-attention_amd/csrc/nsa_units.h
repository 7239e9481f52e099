// The 32-key units that a query token's selected blocks consist of, as a list in the lanes of a wave.
#pragma once
#include <utility>
#include "nsa_common.h"

// Lane i of a wave holds unit i of a list of `n` (lanes from n on: leftovers).  Made for 64 units at a time by all lanes in
// parallel: a loop over them then reads its next unit with one readlane per number instead of finding it step by step (slot
// and part of the block by division, skipped units, page lookup).  The unit that holds the causal boundary comes last: the
// query's own block is among the first selected, and all others can be loaded and scored without looking at the boundary.
struct UnitList {
  int n;
  int n_full;     // how many of them end at or before key_last: the first ones
  int key0;       // first key, position inside the sequence
  int page, off;  // paged: page id and row inside the page; else unused
  int aux;        // caller's number of the unit (unit_list's aux_of)
};

// Units base .. base + 63 of the blocks blk[0 .. nvalid-1] (lane s: block of position s, negative: ignored), block_size /
// 32 of them per block, without those that start behind key_last.  aux_of(position, part of the block, lanes' blk).
template <bool PAGED, class Aux>
NSA_DEVICE UnitList unit_list(int blk, int nvalid, int base, int block_size, int key_last, const int32_t* table, int page_size,
                              int lane, Aux aux_of) {
  const int upb = block_size / 32;
  const int u = base + lane;
  const int pos = upb == 2 ? u >> 1 : u / upb, part = u - pos * upb;
  const int b = __shfl(blk, min(pos, 63), 64);
  const int key0 = b * block_size + part * 32;
  const bool ok = pos < nvalid && b >= 0 && key0 <= key_last;
  const bool full = ok && key0 + 31 <= key_last;
  const uint64_t mask = __builtin_amdgcn_ballot_w64(ok), mask_full = __builtin_amdgcn_ballot_w64(full);
  UnitList l;
  l.n = __popcll(mask);
  l.n_full = __popcll(mask_full);
  const uint64_t below = (1ull << lane) - 1;
  const int before = __popcll(mask & below), before_full = __popcll(mask_full & below);
  // (the ones that are no units behind them, so that every lane is written)
  const int dest = (full ? before_full : ok ? l.n_full + before - before_full : l.n + lane - before) * 4;
  l.key0 = __builtin_amdgcn_ds_permute(dest, key0);
  l.aux = __builtin_amdgcn_ds_permute(dest, aux_of(pos, part, b));
  l.page = l.off = 0;
  if (PAGED && lane < l.n) {
    const int pg = l.key0 / page_size;
    l.page = table[pg];
    l.off = l.key0 - pg * page_size;
  }
  return l;
}

// Rows of one unit as 16-byte pieces of a wave, N instructions of 64 pieces with P pieces per row: after PAT instructions
// the pieces fall on the same columns again.
template <int CHANNELS>
struct UnitRows {
  static constexpr int P = CHANNELS / 8;
  static constexpr int N = 32 * P / 64;
  static constexpr int PAT = 64 % P == 0 ? 1 : 3;  // 192 channels: 3 * 64 = 8 * 24
  static_assert((PAT * 64) % P == 0, "");
  bf16x8 r[N];

  // byte offset of this lane's piece of instruction j (j < PAT) from the unit's first row
  static NSA_DEVICE uint32_t offset(int j, int lane, int64_t row_stride) {
    const int pc = lane + j * 64;
    return (uint32_t)(pc / P) * (uint32_t)(row_stride * 2) + (pc % P) * 16;
  }
  // all 32 rows: scalar base + 32-bit lane offsets (row strides below NARROW elements)
  static constexpr int64_t NARROW = 1 << 27;
  NSA_DEVICE void load(const bf16_t* first, int64_t row_stride, const uint32_t (&off)[PAT]) {
#pragma unroll
    for (int j = 0; j < N; j++) {
      const char* at = reinterpret_cast<const char*>(first + (j / PAT) * (PAT * 64 / P) * row_stride);
      uint32_t o = off[j % PAT];
      asm volatile("" : "+s"(at), "+v"(o));  // (the compiler would widen the offset outside of the loop and add 64 bits per lane)
      r[j] = *(const __attribute__((address_space(1))) bf16x8*)((const __attribute__((address_space(1))) char*)at + o);
    }
  }
  // rows past row `last` replaced by it; any stride
  NSA_DEVICE void load_clamped(const bf16_t* first, int64_t row_stride, int last) {
    const int lane = lane_id();  // (nothing of this rarely taken path is to be held in registers)
#pragma unroll
    for (int j = 0; j < N; j++) {
      const int pc = lane + j * 64;
      r[j] = ld_global_b128(first + (int64_t)min(pc / P, last) * row_stride + (pc % P) * 8);
    }
  }
  // Rows in LDS without padding: row r holds its 16-byte chunk c at c ^ swz(r), which spreads row fragments (16 rows x 64 bytes)
  // and transposed ones (16 rows x 32 bytes) over all banks.  swz: even, below 16 (rows of whole bank rounds) or 8.
  static constexpr bool WIDE = CHANNELS % 128 == 0;
  static constexpr int SPAT = 64 % P == 0 ? (64 / P < 8 ? (WIDE ? 8 * P / 64 : 2) : 1) : 3;  // instructions after which it repeats
  static NSA_DEVICE int swz(int r) { return WIDE ? (r & 7) << 1 : ((r >> 1) & 3) << 1; }
  static NSA_DEVICE int place(int j, int lane) {
    const int pc = lane + j * 64, r = pc / P;
    return r * CHANNELS + ((pc % P) ^ swz(r)) * 8;
  }
  // chunk c0 + c (c0 a constant multiple of what the swizzle's remaining bits sw count in), swizzled
  static NSA_DEVICE int col(int c0, int c, int sw) {
    constexpr int M = WIDE ? 16 : 8;
    return c0 / M * M + (((c0 % M) ^ sw) + c);
  }
  NSA_DEVICE void to_lds_swz(bf16_t* rows, const int (&put)[SPAT]) const {
#pragma unroll
    for (int j = 0; j < N; j++)
      *reinterpret_cast<bf16x8*>(&rows[put[j % SPAT] + j / SPAT * (SPAT * 64 / P) * CHANNELS]) = r[j];
  }
  NSA_DEVICE void to_lds(bf16_t* rows, int ld, int lane) const {
#pragma unroll
    for (int j = 0; j < N; j++) {
      const int pc = lane + j * 64;
      *reinterpret_cast<bf16x8*>(&rows[(pc / P) * ld + (pc % P) * 8]) = r[j];
    }
  }
};

// Rows of one unit as the operand whose contraction index is the row (V^T of O^T = V^T P^T): transposed in the lanes' own
// registers instead of through LDS.  Lane (kq, l16) holds of every row that it loads the channels 8 l16 .. 8 l16 + 7: of the rows
// jt * 16 + kq * 4 + i (jt < 2, i < 4), whose scores it holds (result rows of v_mfma_f32_16x16x32).  The operand of channel e of
// all pieces is element e of the lane's own eight rows, four v_perm_b32; the matrix instruction with it yields the channels
// 8 c + e, so lane (kq, head) ends up with the pieces c = kq * 4 + i, eight neighbouring channels each.
struct UnitColumns128 {
  static constexpr int N = 8, PAT = 1;
  static constexpr int64_t NARROW = UnitRows<128>::NARROW;
  static_assert(12 * NARROW * 2 + 256 <= (int64_t)1 << 32, "a lane's offset: up to twelve rows and a piece");
  bf16x8 r[N];

  static constexpr int row(int j) { return (j >> 2) * 16 + (j & 3); }  // of the lanes with kq 0
  static NSA_DEVICE uint32_t offset(int, int lane, int64_t row_stride) {
    return (uint32_t)((lane >> 4) * 4) * (uint32_t)(row_stride * 2) + (lane & 15) * 16;
  }
  // all 32 rows (row strides below NARROW elements)
  NSA_DEVICE void load(const bf16_t* first, int64_t row_stride, const uint32_t (&off)[PAT]) {
#pragma unroll
    for (int j = 0; j < N; j++) {
      const char* at = reinterpret_cast<const char*>(first + row(j) * row_stride);
      uint32_t o = off[0];
      asm volatile("" : "+s"(at), "+v"(o));  // (scalar base + 32-bit lane offset, as in UnitRows)
      r[j] = *(const __attribute__((address_space(1))) bf16x8*)((const __attribute__((address_space(1))) char*)at + o);
    }
  }
  // rows past row `last` replaced by it; any stride
  NSA_DEVICE void load_clamped(const bf16_t* first, int64_t row_stride, int last) {
    const int lane = lane_id();
#pragma unroll
    for (int j = 0; j < N; j++)
      r[j] = ld_global_b128(first + (int64_t)min(row(j) + (lane >> 4) * 4, last) * row_stride + (lane & 15) * 8);
  }
  template <int E>
  NSA_DEVICE bf16x8 operand() const {
    u32x4 x;
#pragma unroll
    for (int m = 0; m < 4; m++)
      x[m] = __builtin_amdgcn_perm(__builtin_bit_cast(u32x4, r[2 * m + 1])[E / 2], __builtin_bit_cast(u32x4, r[2 * m])[E / 2],
                                   E % 2 ? 0x07060302u : 0x05040100u);
    return __builtin_bit_cast(bf16x8, x);
  }
  // acc[e] += operand e times b
  template <int... E>
  NSA_DEVICE void multiply(f32x4 (&acc)[N], bf16x8 b, std::integer_sequence<int, E...>) const {
    ((acc[E] = mfma16(operand<E>(), b, acc[E])), ...);
  }
};
