// dQ of selected-block attention from the dS that the dK/dV kernel stored (nsa_bwd_dkdv_dma.hip): dQ = dS K, one wave per
// (query token, kv head, up to 16 q-heads), dQ^T += K^T dS^T over the 32-key units of the token's blocks.
//
// Layout of the stored dS: an entry per (token, position in the token's selection, 16-head chunk), in it a blob of 512 bf16
// (256 for 8 heads per kv head) per 32-key unit of the block, as the dK/dV kernel's lanes hold it: lane l = key l % 32 and
// the heads (l / 32) * 4 .. +3, then 8 + (l / 32) * 4 .. +3.
//
// What bounds it: the gather of the K rows, which is half of what the kernel that recomputes S and dP gathers
// (nsa_slc_bwd_dq.hip), beside the dS read once in order.  Nothing of a unit passes through registers on its way to LDS: each wave
// keeps two units in flight into a region of its own (global_load_lds), K as transposed fragments from there.  The two
// regions are two named arrays, so that the compiler's waits for one do not cover the loads of the other.
//
// LDS layout of K: row r holds its 16-byte chunk c at c ^ 2 (r & 7) (rows of 64 or 192 channels: c ^ 2 ((r >> 1) & 3)), which
// spreads the transposed reads (16 rows x 32 bytes) over all banks; the loads fetch the chunk that their place holds.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include "nsa_units.h"

namespace {

typedef __attribute__((address_space(1))) const void* nsa_gptr_t;
typedef __attribute__((address_space(3))) void* nsa_lptr_t;

// waves per workgroup: as many units in flight as LDS holds (18 KB per wave at 128 channels, 26 KB at 192)
constexpr int dq_ds_waves(int d) { return d <= 128 ? 4 : 2; }

template <int D, int DSH, bool STREAM>
__global__ __launch_bounds__(dq_ds_waves(D) * 64) void slc_dq_ds_kernel(NsaSlcDqDsParams p) {
  constexpr int NW = dq_ds_waves(D);
  constexpr int UK = 32;
  constexpr int P = D / 8;                 // 16-byte chunks per row
  constexpr int KJ = UK * P / 64;          // loads per unit
  constexpr int PAT = 64 % P == 0 ? (64 / P < 8 ? 2 : 1) : 3;  // loads after which columns and swizzle repeat
  constexpr int KEL = UK * D, UNIT = KEL + 512;
  constexpr bool WIDE = D % 128 == 0;      // rows of whole bank rounds
  __shared__ __attribute__((aligned(1024))) bf16_t unit_a[NW * UNIT];
  __shared__ __attribute__((aligned(1024))) bf16_t unit_b[NW * UNIT];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  const int n_hc = p.G > 16 ? p.G >> 4 : 1;
  const int kh = blockIdx.y / n_hc, hc = blockIdx.y - kh * n_hc;

  const int i_tok = blockIdx.x * NW + wave;
  if (i_tok >= p.ntok) return;
  const int tok = p.tok0 + i_tok;
  int b = 0;
  for (int hi = p.B; hi - b > 1;) {  // last sequence that starts at or before tok
    const int mid = (b + hi) >> 1;
    if (p.x_cu[mid] <= tok) b = mid; else hi = mid;
  }
  const int x0 = p.x_cu[b];
  const int t = tok - x0;
  if (t < p.t_begin || tok >= p.x_cu[b + 1]) return;  // (rows behind the last sequence are left alone)
  const int Bs = p.block_size, upb = Bs / UK;
  const int nvalid = min(p.top_n, t / Bs + 1);
  const int nu = nvalid * upb;

  // blocks in ascending order, each with its position in the selection (at most 64); ids that no key up to t belongs to
  // are no blocks
  int mine = -1;
  if (lane < nvalid) {
    const int blk = p.topk[(int64_t)kh * p.tk_sh + (int64_t)tok * p.tk_st + lane];
    mine = (unsigned)blk > (unsigned)(t / Bs) ? -1 : blk * 64 + lane;
  }
  mine = sort_blocks(mine, nvalid, lane);

  auto swz = [](int r) { return WIDE ? (r & 7) << 1 : ((r >> 1) & 3) << 1; };
  // byte offset of this lane's piece of load j from the unit's first row
  uint32_t koff[PAT];
#pragma unroll
  for (int j = 0; j < PAT; j++) {
    const int pc = lane + j * 64, r = pc / P;
    koff[j] = (uint32_t)r * (uint32_t)(p.k_sr * 2) + (uint32_t)((pc % P) ^ swz(r)) * 16;
  }
  UnitList ul;
  const bf16_t* const kbase = p.k + (int64_t)x0 * p.k_sr + (int64_t)kh * p.k_sh;
  const bf16_t* const dbase = p.ds + kh * p.ds_sh + ((int64_t)i_tok * p.top_n * n_hc + hc) * upb * (DSH * 32);
  auto issue = [&](auto full_tag, int i, bf16_t* buf) {
    constexpr bool FULL = decltype(full_tag)::value;
    const int key0 = __builtin_amdgcn_readlane(ul.key0, i);
    const int aux = __builtin_amdgcn_readlane(ul.aux, i);  // position * 64 + part
    const bf16_t* const kb = kbase + (int64_t)key0 * p.k_sr;
#pragma unroll
    for (int j = 0; j < KJ; j++) {
      if (FULL) {
        const char* at = reinterpret_cast<const char*>(kb + (int64_t)(j / PAT) * (PAT * 64 / P) * p.k_sr);
        uint32_t off = koff[j % PAT];
        asm volatile("" : "+s"(at), "+v"(off));  // (scalar base + 32-bit lane offset)
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + off), (nsa_lptr_t)(buf + j * 512), 16, 0, 0);
      } else {  // rows past the causal boundary replaced by the boundary row: their dS is 0, they must be finite if it is
        const int pc = lane_id() + j * 64, r = pc / P;
        const bf16_t* at = kb + (int64_t)min(r, t - key0) * p.k_sr + ((pc % P) ^ swz(r)) * 8;
        __builtin_amdgcn_global_load_lds((nsa_gptr_t)at, (nsa_lptr_t)(buf + j * 512), 16, 0, 0);
      }
    }
    const char* at = reinterpret_cast<const char*>(dbase + ((int64_t)(aux >> 6) * n_hc * upb + (aux & 63)) * (DSH * 32));
    uint32_t off = DSH == 8 ? (lane & 31) * 16 : lane * 16;  // (8 heads: the blob twice)
    asm volatile("" : "+s"(at), "+v"(off));
    __builtin_amdgcn_global_load_lds((nsa_gptr_t)(at + off), (nsa_lptr_t)(buf + KEL), 16, 0, STREAM ? 2 : 0);  // (2: non-temporal)
  };

  f32x4 dqacc[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; dt++) dqacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // transposed fragments: this lane points at 4 channels of row kq * 4 + l16 / 4 (and of the row 16 further)
  const int r0 = kq * 4 + (l16 >> 2);
  const int ka = r0 * D + ((l16 & 3) >> 1) * 8 + (l16 & 1) * 4;
  const int ksw = swz(r0);  // (row + 16 has the same)
  const int da = DSH == 8 ? ((l16 & 1) * 32 + r0) * 4 : ((l16 & 1) * 32 + r0) * 8 + ((l16 & 3) >> 1) * 4;

  // `younger`: loads in flight that are younger than the unit's
  auto consume = [&](auto younger, const bf16_t* buf) {
    constexpr int N = decltype(younger)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70 + N);  // vmcnt(N)
    asm volatile("" ::: "memory");
    const bf16x8 df = cat4(lds_read_tr(buf + KEL + da), lds_read_tr(buf + KEL + da + 16 * (DSH == 8 ? 4 : 8)));
#pragma unroll
    for (int dt = 0; dt < D / 16; dt++) {
      // chunk 2 dt (+ 1) of the row, swizzled: the XOR meets the bits above the lowest of the chunk's number
      const int col = WIDE ? ((dt * 2) ^ ksw) * 8 : (dt / 4) * 64 + (((dt % 4) * 2) ^ ksw) * 8;
      dqacc[dt] = mfma16(cat4(lds_read_tr(buf + ka + col), lds_read_tr(buf + ka + col + 16 * D)), df, dqacc[dt]);
    }
    // the region is loaded again next: its reads have to have been answered
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  };
  constexpr int NL = KJ + 1;
  static_assert(NL <= 15, "the wait's immediate");
  typedef std::integral_constant<bool, true> FullT;
  typedef std::integral_constant<bool, false> AnyT;
  bf16_t* const a = unit_a + wave * UNIT;
  bf16_t* const c = unit_b + wave * UNIT;
  for (int base = 0; base < nu; base += 64) {
    ul = unit_list<false>(mine >> 6, nvalid, base, Bs, t, nullptr, 1, lane, [&](int pos, int part, int) {
      return (__shfl(mine, min(pos, 63), 64) & 63) * 64 + part;
    });
    if (ul.n == 0) continue;
    const int n = ul.n, n_full = ul.n_full;
    // units 0 .. n_full - 1 without a look at the boundary; the loads of unit i + 2 follow the use of unit i
    int i = 0;
    issue(AnyT{}, 0, a);
    issue(AnyT{}, min(1, n - 1), c);  // (without a branch: behind one, the compiler's waits would be for everything)
    for (; i + 3 < n_full; i += 2) {
      consume(std::integral_constant<int, NL>{}, a);
      issue(FullT{}, i + 2, a);
      consume(std::integral_constant<int, NL>{}, c);
      issue(FullT{}, i + 3, c);
    }
    for (; i < n; i += 2) {
      if (i + 1 < n) consume(std::integral_constant<int, NL>{}, a);
      else consume(std::integral_constant<int, 0>{}, a);
      if (i + 2 < n) issue(AnyT{}, i + 2, a);
      if (i + 1 >= n) break;
      if (i + 2 < n) consume(std::integral_constant<int, NL>{}, c);
      else consume(std::integral_constant<int, 0>{}, c);
      if (i + 3 < n) issue(AnyT{}, i + 3, c);
    }
  }

  if (DSH == 8 && l16 >= 8) return;
  const int head = kh * p.G + hc * 16 + l16;
  const int64_t off = (int64_t)tok * p.dq_st + (int64_t)head * p.dq_sh + kq * 4;
  f32x4 part[D / 16];
  if (p.dq_mode == 3) {
    const float* pp = p.dq_partial + (int64_t)tok * p.dqp_st + (int64_t)head * p.dqp_sh + kq * 4;
#pragma unroll
    for (int dt = 0; dt < D / 16; dt++) part[dt] = *reinterpret_cast<const f32x4*>(pp + dt * 16);
  }
#pragma unroll
  for (int dt = 0; dt < D / 16; dt++) {
    f32x4 val = dqacc[dt] * p.sm_scale;
    if (p.dq_mode == 0) {
      *reinterpret_cast<bf16x4*>((bf16_t*)p.dq + off + dt * 16) = pack4(val[0], val[1], val[2], val[3]);
    } else if (p.dq_mode == 3) {
      val += part[dt];
      *reinterpret_cast<bf16x4*>((bf16_t*)p.dq + off + dt * 16) = pack4(val[0], val[1], val[2], val[3]);
    } else {
      float* dst = (float*)p.dq + off + dt * 16;
      if (p.dq_mode == 2) val += *reinterpret_cast<f32x4*>(dst);
      *reinterpret_cast<f32x4*>(dst) = val;
    }
  }
}

template <int D>
int launch(const NsaSlcDqDsParams& p, hipStream_t stream) {
  const dim3 grid(cdiv_i(p.ntok, dq_ds_waves(D)), p.KH * (p.G > 16 ? p.G / 16 : 1));
  // The dS is read once: where it is more than the 256 MB that the memory-side cache holds, so that all of it comes from memory
  // anyhow, it is not to push K rows out of L2.  This kernel, us, kept / so: 64 heads of 128, 64K tokens 5500 / 5320, 8 x 6K tokens
  // 2972 / 2947, 16 heads of 64, 16K tokens (0.5 GB) 348 / 324, 32 heads of 192, 16K tokens 860 / 850; 16 heads of 128, 4K tokens
  // (0.13 GB) 51.3 / 53.9.
  auto run = [&](auto stream_tag) {
    constexpr bool S = decltype(stream_tag)::value;
    if (p.G == 8) slc_dq_ds_kernel<D, 8, S><<<grid, dq_ds_waves(D) * 64, 0, stream>>>(p);
    else slc_dq_ds_kernel<D, 16, S><<<grid, dq_ds_waves(D) * 64, 0, stream>>>(p);
  };
  if (p.ds_sh * p.KH * 2 > (int64_t)256 << 20) run(std::true_type{});
  else run(std::false_type{});
  return nsa_check_launch("slc_dq_ds_kernel");
}

}  // namespace

int64_t nsa_slc_ds_entry_elems(int G, int block_size) {
  return G == 8 ? (int64_t)block_size / 32 * 256 : (int64_t)block_size / 32 * 512 * (G / 16);
}

int nsa_slc_dq_ds_launch(const NsaSlcDqDsParams& p, int D, hipStream_t stream) {
  if (p.ntok <= 0) return NSA_OK;
  if (D == 128) return launch<128>(p, stream);
  if (D == 64) return launch<64>(p, stream);
  if (D == 192) return launch<192>(p, stream);
  nsa_set_error("selected attention dq from stored dS: unsupported head dim D=%d", D);
  return NSA_ERR_UNSUPPORTED;
}
