// Block selection of one token by one wave, with the candidates in registers; shared by the decode kernels and the
// two-pass block selector of the training / prefill path.
#pragma once
#include <type_traits>
#include "nsa_common.h"

// one wave: forced initial and local blocks, then repeated arg-max over imp[0 .. min(t/block, nb_cap-1)] (lowest
// index on ties).  Returns the block of slot `lane`.
// The candidates of a lane (blocks lane, lane+64, ...) are read once into NV registers; after every round only the
// winner's lane rescans its registers, so a round costs one wave reduction instead of a dependent chain of LDS reads.
template <int NV, class P>
NSA_DEVICE int select_blocks_regs(const float* imp, int t, int nb_cap, const P& p, int lane) {
  static_assert(NV % 8 == 0, "candidates per lane come in groups of 8");
  constexpr int NG = NV / 8;
  const int nk = t >= 0 ? t / p.block_size : -1;
  int result = p.ignore_index;
  if (lane < p.num_init) {
    if (lane <= nk) result = lane;
  } else if (lane < p.num_init + p.num_local) {
    if (lane <= nk) result = nk - (lane - p.num_init);
  }
  const int nsel = min(p.top_n, nk + 1);
  const int jmax = min(nk, nb_cap - 1);
  float v[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const int j = lane + 64 * k;
    float x = j <= jmax ? imp[min(j, nb_cap - 1)] : -3.f;
    if (j <= jmax && (j < p.num_init || j > nk - p.num_local)) x = -1.f;  // forced blocks: behind every real score
    v[k] = x;
  }
  // best candidate of every group of 8 registers; a round only rescans the group the winner came from (the group
  // number is wave-uniform, so that is one uniform branch)
  float gbest[NG];
  int gidx[NG];
  auto rescan = [&](auto g_tag) {
    constexpr int g = decltype(g_tag)::value;
    float bs = -2.f;
    int bi = 0x7fffffff;
#pragma unroll
    for (int k = g * 8; k < g * 8 + 8; k++)
      if (v[k] > bs) { bs = v[k]; bi = lane + 64 * k; }
    gbest[g] = bs;
    gidx[g] = bi;
  };
  auto for_group = [&](int g, auto&& fn) {
    if constexpr (NG == 1) { fn(std::integral_constant<int, 0>{}); }
    else if constexpr (NG == 2) { if (g == 0) fn(std::integral_constant<int, 0>{}); else fn(std::integral_constant<int, 1>{}); }
    else {
      static_assert(NG == 4, "8, 16 or 32 candidates per lane");
      if (g == 0) fn(std::integral_constant<int, 0>{});
      else if (g == 1) fn(std::integral_constant<int, 1>{});
      else if (g == 2) fn(std::integral_constant<int, 2>{});
      else fn(std::integral_constant<int, 3>{});
    }
  };
#pragma unroll
  for (int g = 0; g < NG; g++) for_group(g, rescan);
  for (int slot = p.num_init + p.num_local; slot < nsel; slot++) {
    float best = -2.f;
    int bj = 0x7fffffff;
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (gbest[g] > best) { best = gbest[g]; bj = gidx[g]; }
    const int w = wave_argmax_lowest(best, bj, bj != 0x7fffffff);
    if (lane == slot) result = w;
    if (w > jmax) continue;  // wave-uniform: no candidate left
    const bool mine = (w & 63) == lane;
    const int kk = w >> 6;
    for_group(kk >> 3, [&](auto g_tag) {  // take the winner out of its group, then rescan that group only
      constexpr int g = decltype(g_tag)::value;
#pragma unroll
      for (int k = g * 8; k < g * 8 + 8; k++)
        if (mine && k == kk) v[k] = -1.f;
      rescan(g_tag);
    });
  }
  return result;
}


// wave-wide maximum of a float on the DPP crossbar, the same value in every lane
NSA_DEVICE float wave_fmax_uniform(float x) {
  float m = x;
  m = dpp_fmax_step<0x111, 0xf>(m);  // row_shr:1
  m = dpp_fmax_step<0x112, 0xf>(m);  // row_shr:2
  m = dpp_fmax_step<0x114, 0xf>(m);  // row_shr:4
  m = dpp_fmax_step<0x118, 0xf>(m);  // row_shr:8
  m = dpp_fmax_step<0x142, 0xa>(m);  // row_bcast:15
  m = dpp_fmax_step<0x143, 0xc>(m);  // row_bcast:31 -> lane 63 holds the wave maximum
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 63));
}

// A theta that at least `rounds` lanes' m reach, -1 where fewer hold a score (scores are not negative): their bits order as
// integers do.  Halved between the wave's maximum and 2^-16 of it (or 0, if too few reach that) until at most SLACK lanes more
// than `rounds` reach theta: every lower bound of the rounds-th largest score selects the same, only the list gets longer.
template <bool SHORT_CODE>
NSA_DEVICE float lane_bound(float m, int rounds) {
  if constexpr (SHORT_CODE) {  // the largest such m: every lane compares its own with all others
    int above = 0;
#pragma unroll 8
    for (int j = 0; j < 64; j++)
      above += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), j)) > m;
    return fmaxf(-wave_fmax_uniform(above < rounds ? -m : -__builtin_inff()), -1.f);
  }
  constexpr int SLACK = 3;
  const int key = __builtin_bit_cast(int, m);
  auto reach = [&](int at) { return (int)__builtin_popcountll(__builtin_amdgcn_ballot_w64(key >= at)); };
  const int top = max(__builtin_bit_cast(int, wave_fmax_uniform(m)), 0);
  int lo = max(top - (16 << 23), 0), n = reach(lo);
  if (n < rounds) {
    lo = 0;
    n = reach(0);
    if (n < rounds) return -1.f;
  }
  int width = top - lo;  // (the maximum itself: fewer than `rounds` above it)
  while (n > rounds + SLACK && width > 0) {
    const int half = (width + 1) >> 1, at = reach(lo + half);
    if (at >= rounds) {
      lo += half;
      width -= half;
      n = at;
    } else {
      width = half - 1;
    }
  }
  return __builtin_bit_cast(float, lo);
}

// Makes the loads of all N values precede the first use of one (else the compiler puts each behind the condition under which it is
// used, and one round trip after another is waited for)
template <int N>
NSA_DEVICE void load_together(float (&v)[N]) {
  static_assert(N == 2 || N % 4 == 0, "");
  if constexpr (N == 2) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]));
  } else if constexpr (N == 4) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
  } else {
#pragma unroll
    for (int k = 0; k < N; k += 8)
      asm volatile("" : "+v"(v[k]), "+v"(v[k + 1]), "+v"(v[k + 2]), "+v"(v[k + 3]), "+v"(v[k + 4]), "+v"(v[k + 5]), "+v"(v[k + 6]),
                        "+v"(v[k + 7]));
  }
}

// The same selection as select_blocks_regs over a short list instead of the NV registers of every lane: a lower bound of the R-th
// largest of the 64 lane maxima is one of the R-th largest score (R = number of scored slots), so only the scores at or
// above it can be selected; they are compacted (ballot + prefix count) into a wave-private list of at most 64 entries in LDS
// (cand_v, 16-byte aligned, / cand_i), one per lane, in ascending order of the block.  The picks and their order are those of
// select_blocks_regs (descending score, lowest index on ties); rows with more than 64 scores at the bound (many equal values)
// take that function.
// Places come from counting: every entry is compared with all others, which are independent instructions.  (Repeated wave-wide
// maxima are a dependent chain of about 200 ns per round, twice R of them: one request of 32K tokens, 512 blocks, the selection
// 5.5 -> 2.7 us; 16 of 128K, 2048 blocks, 8.0 -> 5.1.)
// SHORT_CODE: bound and places with one broadcast per lane and entry, and scores loaded as they are used: for the one-launch decode
// kernel, where more code costs batches that wait for memory and not for this (512 requests of 4K tokens 327.8 us; 330.8 with the
// other form, which gains the split kernel's 16 of 128K 1 %, 8 of 2K to 8K with 16 / 2 heads of 64 25.6 -> 24.8 us, and a wave per
// row of the training and prefill path 460 -> 175 vector instructions).
template <bool SHORT_CODE, int NV, class P>
NSA_DEVICE int select_blocks_short_list(const float* imp, int t, int nb_cap, const P& p, int lane, float* cand_v,
                                        int* cand_i) {
  const int nk = t >= 0 ? t / p.block_size : -1;
  const int forced = p.num_init + p.num_local;
  const int nsel = min(p.top_n, nk + 1);
  const int rounds = nsel - forced;
  int result = p.ignore_index;
  if (lane < p.num_init) {
    if (lane <= nk) result = lane;
  } else if (lane < forced) {
    if (lane <= nk) result = nk - (lane - p.num_init);
  }
  if (rounds <= 0) return result;
  const int jmax = min(nk, nb_cap - 1);
  float v[NV];
  float m = -3.f;
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = !SHORT_CODE || lane + 64 * k <= jmax ? imp[min(lane + 64 * k, jmax)] : -3.f;
  if constexpr (!SHORT_CODE) load_together(v);
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const int j = lane + 64 * k;
    float x = j < p.num_init || j > nk - p.num_local ? -1.f : v[k];  // forced blocks: behind every real score
    v[k] = x = j <= jmax ? x : -3.f;
    m = fmaxf(m, x);
  }
  const float theta = lane_bound<SHORT_CODE>(m, rounds);
  if (!SHORT_CODE) cand_v[lane] = -3.f;  // (behind the last entry)
  // compaction of the scores >= theta, register by register (ascending block number within a register)
  int base = 0;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const uint64_t mask = __builtin_amdgcn_ballot_w64(v[k] >= theta);
    const int pos = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)base));
    if (v[k] >= theta && pos < 64) { cand_v[pos] = v[k]; cand_i[pos] = lane + 64 * k; }
    base += __builtin_popcountll(mask);
  }
  if (base > 64) return select_blocks_regs<(NV < 8 ? 8 : NV)>(imp, t, nb_cap, p, lane);  // wave-uniform
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const float cv = !SHORT_CODE || lane < base ? cand_v[lane] : -3.f;
  const int ci = !SHORT_CODE || lane < base ? cand_i[lane] : 0;
  int place = 0;  // scores ahead of this lane's: greater ones, and equal ones of lower blocks
  auto store = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < base && place < rounds) cand_i[place] = ci;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  bool equal = SHORT_CODE || base > 32;
  if (!equal) {
    // the two halves of the wave compare the same 32 entries with 16 each, read as they lie instead of broadcast lane by lane
    const float mine = cand_v[lane & 31];
    const f32x4* others = reinterpret_cast<const f32x4*>(cand_v + (lane >> 5) * 16);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f32x4 o = others[i];
#pragma unroll
      for (int e = 0; e < 4; e++) place += o[e] > mine;
    }
    const auto both = __builtin_amdgcn_permlane32_swap((uint32_t)place, (uint32_t)place, false, false);
    place = (int)(both[0] + both[1]);
    store();
    // equal scores have taken the same place: only one of them finds itself there
    const bool lost = lane < base && place < rounds && cand_i[min(place, 63)] != ci;
    equal = __builtin_amdgcn_ballot_w64(lost) != 0;
  }
  if (equal) {
    place = 0;
#pragma unroll 4
    for (int j = 0; j < base; j++) {
      const float other = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cv), j));
      place += other > cv || (other == cv && j < lane);
    }
    store();
  }
  if (lane >= forced && lane < nsel) result = lane - forced < base ? cand_i[lane - forced] : 0x7fffffff;
  return result;
}
