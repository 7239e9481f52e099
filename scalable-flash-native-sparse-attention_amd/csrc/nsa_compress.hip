// Learned compression of K and V: hidden = windows W^T, its activation, and their gradients, without the windows in memory.
// Upstream materialises the windows (flash_nsa/ops/compress_kv.py:126-218) and calls GEMMs on them
// (flash_nsa/modules/megatron_level_nsa.py:46-86, flash_nsa/modules/hf_level_nsa.py:17-52).  Here window i of a sequence, kernel
// rows of D channels every `stride` rows, is read where it lies in x: element j * D + d of it is x[stride * i + j][d].
// A row of these products is a (compressed row, kv head) pair, row-major in that order.
//
// What bounds them at long batches is round trips to L2: every tile reads the weight (forward, dx) or the windows (dW) again, and the waves
// wait 30 % (forward), 58 % (dx) and 69 % (dW) of their cycles, with the matrix cores busy 18, 17 and 10 % and LDS 38, 34 and 18 % (64K
// tokens, 4 heads of 128, gated).  At short batches it is the launches: a library product costs the host 33 us, and the windows took two more
// launches and two passes over them.
#include "nsa_common.h"
#include "nsa_api_internal.h"
#include "../../include/nsa_hip.h"

namespace {

struct CompressParams {
  const bf16_t* x; int64_t x_st, x_sh;   // [tokens, H, D]
  const bf16_t* w; int64_t w_st;         // [N, kernel * D]
  bf16_t* hidden;                        // [y_len, H, N]: products (act >= 0: may be null); backward: their gradient
  bf16_t* out;                           // act >= 0: [y_len, H, D]
  float* dx; int64_t dx_st, dx_sh;       // backward: fp32 [tokens, H, D], added to (null: zeros)
  bf16_t* dst; int64_t dst_st, dst_sh;   //           takes the sum in bf16 (null: dx does)
  const int32_t* x_cu; const int32_t* y_cu;
  int B, H, D, K, S, N, act;
};

NSA_DEVICE float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }

// Forward.  A workgroup: 32 * RS rows by GB * 32 channels (GLU: of the gate and of the value), its eight waves an eighth of the
// contraction each.  Pieces of 64 bytes of 16 rows per instruction (fragments straight from memory, 16 bytes of 32 rows each, take
// the address unit four times as long: 1200 tokens, 1 head of 128 45 us instead of 12), through a wave-private LDS slot, AHEAD
// chunks of 32 elements on their way.  grid (row tiles, B, D / 32 / GB)
template <int GB, bool GLU, int RS, int AHEAD>
__global__ __launch_bounds__(512, 2) void compress_linear_kernel(CompressParams p) {
  constexpr int NW = 8;
  constexpr int NA = GLU ? 2 * GB : GB;      // 32-column blocks
  constexpr int HLD = NA * 32 + 8;
  constexpr int LDC = 40;                    // a chunk's row in LDS: 32 elements and a pad that spreads 8 rows over all banks
  constexpr int SLOT = (NA + RS) * 32 * LDC;
  constexpr int REDS = NW * 32 * 36 * 2;     // (elements of 2 bytes)
  __shared__ __attribute__((aligned(16))) bf16_t stage[NW * SLOT > REDS ? NW * SLOT : REDS];
  __shared__ __attribute__((aligned(16))) bf16_t hid[32 * RS * HLD];
  float (*const red)[32][36] = reinterpret_cast<float (*)[32][36]>(stage);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hl = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y, group = blockIdx.z;
  const int x0 = p.x_cu[b], y0 = p.y_cu[b];
  const int rows = (p.y_cu[b + 1] - y0) * p.H;
  const int r0 = blockIdx.x * 32 * RS;
  if (r0 >= rows) return;
  const int D = p.D;
  // instruction u fetches a chunk of rows 16 u .. 16 u + 15: of the weight, then of x
  const bf16_t* xp[RS * 2];
#pragma unroll
  for (int u = 0; u < RS * 2; u++) {
    const int m = min(r0 + u * 16 + (lane >> 2), rows - 1), i = m / p.H, h = m - i * p.H;
    xp[u] = p.x + (int64_t)(x0 + (int64_t)p.S * i) * p.x_st + (int64_t)h * p.x_sh + (lane & 3) * 8;
  }
  const bf16_t* const w0 = p.w + (int64_t)(group * GB * 32) * p.w_st;
  const int64_t wl = (int64_t)(lane >> 2) * p.w_st + (lane & 3) * 8;
  const int chunks = p.K * D / 32;
  const int s0 = wave * chunks / NW, s1 = (wave + 1) * chunks / NW;
  f32x16 acc[RS][NA];
#pragma unroll
  for (int rs = 0; rs < RS; rs++)
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[rs][a][i] = 0.f;
  bf16_t* const slot = stage + wave * SLOT;
  bf16_t* const put = slot + (lane >> 2) * LDC + (lane & 3) * 8;
  const bf16_t* const get = slot + l32 * LDC + hl * 8;
  bf16x8 reg[AHEAD][(NA + RS) * 2];
  int j = s0 * 32 / D, d = s0 * 32 - j * D;  // of the next chunk to be fetched
  auto fetch = [&](bf16x8 (&r)[(NA + RS) * 2], int s) {
    if (s >= s1) return;
    const int64_t xo = (int64_t)j * p.x_st + d;
#pragma unroll
    for (int u = 0; u < NA * 2; u++) {
      const bf16_t* const at = w0 + (int64_t)((u >> 1 < GB ? 0 : D) + (u >> 1) % GB * 32 + (u & 1) * 16) * p.w_st + s * 32;
      r[u] = ld_global_b128(at + wl);
    }
#pragma unroll
    for (int u = 0; u < RS * 2; u++) r[NA * 2 + u] = ld_global_b128(xp[u] + xo);
    d += 32;
    if (d == D) { d = 0; j++; }
  };
  auto lds_order = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto chunk = [&](bf16x8 (&r)[(NA + RS) * 2], int s) {
    if (s >= s1) return;
#pragma unroll
    for (int u = 0; u < (NA + RS) * 2; u++) *reinterpret_cast<bf16x8*>(put + u * 16 * LDC) = r[u];
    lds_order();
    fetch(r, s + AHEAD);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      bf16x8 xf[RS];
#pragma unroll
      for (int rs = 0; rs < RS; rs++) xf[rs] = *reinterpret_cast<const bf16x8*>(get + (NA + rs) * 32 * LDC + ks * 16);
#pragma unroll
      for (int a = 0; a < NA; a++) {
        const bf16x8 wf = *reinterpret_cast<const bf16x8*>(get + a * 32 * LDC + ks * 16);
#pragma unroll
        for (int rs = 0; rs < RS; rs++) acc[rs][a] = mfma32(wf, xf[rs], acc[rs][a]);
      }
    }
    lds_order();
  };
#pragma unroll
  for (int k = 0; k < AHEAD; k++) fetch(reg[k], s0 + k);
  for (int s = s0; s < s1; s += AHEAD) {
#pragma unroll
    for (int k = 0; k < AHEAD; k++) chunk(reg[k], s + k);
  }
  __syncthreads();
  // The waves' sums, in wave order, rounded: a lane holds four neighbouring columns of its row.
#pragma unroll
  for (int rs = 0; rs < RS; rs++)
#pragma unroll
    for (int a = 0; a < NA; a++) {
#pragma unroll
      for (int i4 = 0; i4 < 4; i4++)
        *reinterpret_cast<f32x4*>(&red[wave][l32][i4 * 8 + hl * 4]) =
            f32x4{acc[rs][a][i4 * 4], acc[rs][a][i4 * 4 + 1], acc[rs][a][i4 * 4 + 2], acc[rs][a][i4 * 4 + 3]};
      __syncthreads();
      if (tid < 256) {
        const int rr = tid >> 3, rc = (tid & 7) * 4;
        f32x4 sum = *reinterpret_cast<const f32x4*>(&red[0][rr][rc]);
#pragma unroll
        for (int w = 1; w < NW; w++) sum += *reinterpret_cast<const f32x4*>(&red[w][rr][rc]);
        *reinterpret_cast<bf16x4*>(&hid[(rs * 32 + rr) * HLD + a * 32 + rc]) = pack4(sum[0], sum[1], sum[2], sum[3]);
      }
      __syncthreads();
    }
  const int64_t row0 = (int64_t)y0 * p.H + r0;
  if (p.hidden != nullptr)
    for (int e = tid; e < 32 * RS * NA * 4; e += NW * 64) {
      const int r = e / (NA * 4), c = e - r * (NA * 4), a = c >> 2;
      if (r0 + r >= rows) break;
      *reinterpret_cast<bf16x8*>(p.hidden + (row0 + r) * p.N + (a < GB ? 0 : D) + (group * GB + a % GB) * 32 + (c & 3) * 8) =
          *reinterpret_cast<const bf16x8*>(&hid[r * HLD + c * 8]);
    }
  if constexpr (GLU) {
    for (int e = tid; e < 32 * RS * GB * 4; e += NW * 64) {
      const int r = e / (GB * 4), c = e - r * (GB * 4);
      if (r0 + r >= rows) break;
      const bf16x8 g = *reinterpret_cast<const bf16x8*>(&hid[r * HLD + c * 8]);
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(&hid[r * HLD + GB * 32 + c * 8]);
      float o[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const float gf = (float)g[k], sg = sigmoidf_(gf);
        o[k] = (p.act == 0 ? sg : sg * gf) * (float)v[k];
      }
      *reinterpret_cast<bf16x8*>(p.out + (row0 + r) * D + group * GB * 32 + c * 8) =
          pack8(o[0], o[1], o[2], o[3], o[4], o[5], o[6], o[7]);
    }
  }
}

// dx.  Token stride * c + jj, jj < stride, lies in the windows c, c - 1, .. c - kernel / stride + 1, in that of c - r at place
// jj + r * stride: the gradients of a chunk of `stride` tokens are one row of a product whose contraction runs over r and the
// columns of the gradient of `hidden`.  A workgroup: 128 (chunk, head) rows by 128 of the stride * D columns, the weight tile (its
// rows are the contraction index) in LDS, read transposed.  It moves the fp32 gradient in and the bf16 one out, 201 MB at 64K tokens, 4
// heads of 128, in 87 us (library product, sum over the windows and conversion: 67 + 61 + 43); stored from the accumulators as they
// lie 158.  grid (row tiles, column tiles, B)
__global__ __launch_bounds__(256, 2) void compress_linear_dx_kernel(CompressParams p) {
  constexpr int LDW = 128 + NSA_LDS_PAD, LDG = 40, LDO = 36;
  __shared__ __attribute__((aligned(16))) bf16_t wt[2][32 * LDW];
  __shared__ __attribute__((aligned(16))) float own[4][32 * LDO];  // a wave's rows: gradients of a step, then its results
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hl = lane >> 5, g16 = lane >> 4, i16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.z;
  const int x0 = p.x_cu[b], xl = p.x_cu[b + 1] - x0, y0 = p.y_cu[b], yl = p.y_cu[b + 1] - y0;
  const int D = p.D, N = p.N, SD = p.S * D;
  const int rows = (xl + p.S - 1) / p.S * p.H;
  const int r0 = blockIdx.x * 128, c0 = blockIdx.y * 128;
  if (r0 >= rows) return;
  const int per = N / 32, steps = yl > 0 ? p.K / p.S * per : 0;
  f32x16 acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[dt][i] = 0.f;
  // gradients: instruction u fetches 64 bytes of the wave's rows 16 u .. 16 u + 15
  int gc[2], gh[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int m = r0 + wave * 32 + u * 16 + (lane >> 2);
    gc[u] = m < rows ? m / p.H : -1;
    gh[u] = m - gc[u] * p.H;
  }
  bf16_t* const gs = reinterpret_cast<bf16_t*>(own[wave]);
  bf16x8 wreg[2], greg[2];
  auto fetch = [&](int s) {
    const int r = s / per, n0 = (s - r * per) * 32;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int row = (tid >> 4) + u * 16, col = c0 + (tid & 15) * 8;
      wreg[u] = col < SD ? ld_global_b128(p.w + (int64_t)(n0 + row) * p.w_st + (int64_t)r * SD + col) : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int i = gc[u] - r;
      const bool ok = i >= 0 && i < yl;
      greg[u] = ok ? ld_global_b128(p.hidden + ((int64_t)(y0 + i) * p.H + gh[u]) * N + n0 + (lane & 3) * 8) : zero_bf16x8();
    }
  };
  if (steps > 0) fetch(0);
  for (int s = 0; s < steps; s++) {
    bf16_t* const t = wt[s & 1];
#pragma unroll
    for (int u = 0; u < 2; u++) *reinterpret_cast<bf16x8*>(&t[((tid >> 4) + u * 16) * LDW + (tid & 15) * 8]) = wreg[u];
#pragma unroll
    for (int u = 0; u < 2; u++) *reinterpret_cast<bf16x8*>(&gs[(u * 16 + (lane >> 2)) * LDG + (lane & 3) * 8]) = greg[u];
    __syncthreads();  // (the tile of step s - 1 is not written before every wave has come to the next barrier)
    if (s + 1 < steps) fetch(s + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const bf16x8 g = *reinterpret_cast<const bf16x8*>(&gs[l32 * LDG + ks * 16 + hl * 8]);
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        const bf16_t* at = &t[(ks * 16 + hl * 8 + (i16 >> 2)) * LDW + dt * 32 + (g16 & 1) * 16 + 4 * (i16 & 3)];
        acc[dt] = mfma32(cat4(lds_read_tr(at), lds_read_tr(at + 4 * LDW)), g, acc[dt]);
      }
    }
  }
  // The results leave as whole pieces of 128 bytes: 8 lanes a row, through the wave's part of LDS.
  auto lds_order = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  float* const os = own[wave];
  int oc[4], oh[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int m = r0 + wave * 32 + k * 8 + (lane >> 3);
    oc[k] = m < rows ? m / p.H : -1;
    oh[k] = m - oc[k] * p.H;
  }
#pragma unroll
  for (int dt = 0; dt < 4; dt++) {
    const int col = c0 + dt * 32, jj = col / D, ch = col - jj * D + (lane & 7) * 4;
    if (col >= SD) break;  // workgroup-uniform
    f32x4 old[4];
    int64_t tok[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int n = oc[k] * p.S + jj;
      tok[k] = oc[k] >= 0 && n < xl ? x0 + n : -1;
      old[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (tok[k] >= 0 && p.dx != nullptr) old[k] = *reinterpret_cast<const f32x4*>(p.dx + tok[k] * p.dx_st + (int64_t)oh[k] * p.dx_sh + ch);
    }
    lds_order();
#pragma unroll
    for (int i4 = 0; i4 < 4; i4++)
      *reinterpret_cast<f32x4*>(&os[l32 * LDO + i4 * 8 + hl * 4]) =
          f32x4{acc[dt][i4 * 4], acc[dt][i4 * 4 + 1], acc[dt][i4 * 4 + 2], acc[dt][i4 * 4 + 3]};
    lds_order();
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const f32x4 val = old[k] + *reinterpret_cast<const f32x4*>(&os[(k * 8 + (lane >> 3)) * LDO + (lane & 7) * 4]);
      if (tok[k] < 0) continue;
      if (p.dst != nullptr)
        *reinterpret_cast<bf16x4*>(p.dst + tok[k] * p.dst_st + (int64_t)oh[k] * p.dst_sh + ch) = pack4(val[0], val[1], val[2], val[3]);
      else
        *reinterpret_cast<f32x4*>(p.dx + tok[k] * p.dx_st + (int64_t)oh[k] * p.dx_sh + ch) = val;
    }
  }
}

// dW, 64K tokens, 4 heads of 128, N 256: 131 us, of which the waves wait 69 % for the next step's rows (library product 152); 40 samples of
// up to 1.2K, 2 heads of 64, both weights 35 + 12 for the sums (72: 32 workgroups).
// dW = (gradient of hidden)^T windows, cut along the contraction into gridDim.z parts whose sums go to slots.  A workgroup: NT * 32
// rows of dW by 128 columns, both tiles (their rows are the contraction index) in LDS, read transposed.
// grid (N / 32 / NT, ceil(kernel * D / 128), parts)
template <int NT>
__global__ __launch_bounds__(256, 2) void compress_linear_dw_kernel(CompressParams p, float* slots) {
  constexpr int LDG = NT * 32 + NSA_LDS_PAD, LDX = 128 + NSA_LDS_PAD;
  constexpr int GP = NT * 4;                          // pieces of a gradient row
  constexpr int GU = (32 * GP + 255) / 256;
  __shared__ __attribute__((aligned(16))) bf16_t gt[2][32 * LDG];
  __shared__ __attribute__((aligned(16))) bf16_t xt[2][32 * LDX];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hl = lane >> 5, g16 = lane >> 4, i16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H, D = p.D, KD = p.K * D;
  const int n0 = blockIdx.x * NT * 32, c0 = blockIdx.y * 128;
  const int64_t rows = (int64_t)p.y_cu[p.B] * H;
  const int steps = (int)((rows + 31) / 32);
  const int s0 = (int)((int64_t)blockIdx.z * steps / gridDim.z), s1 = (int)((int64_t)(blockIdx.z + 1) * steps / gridDim.z);
  f32x16 acc[NT];
#pragma unroll
  for (int a = 0; a < NT; a++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[a][i] = 0.f;
  // the thread's columns of the windows, and the sequences of its two rows, which only go on
  const int col = c0 + (tid & 15) * 8, j = col / D, ch = col - j * D;
  int seq[2] = {0, 0};
  {
    const int64_t y = min((int64_t)s0 * 32, rows - 1) / H;
    int lo = 0, hi = p.B - 1;                         // the last sequence that starts at or before y
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (p.y_cu[mid] <= y) lo = mid;
      else hi = mid - 1;
    }
    seq[0] = seq[1] = lo;
  }
  bf16x8 greg[GU], xreg[2];
  auto fetch = [&](int s) {
#pragma unroll
    for (int u = 0; u < GU; u++) {
      const int pc = tid + u * 256, row = pc / GP;
      const int64_t m = (int64_t)s * 32 + row;
      greg[u] = row < 32 && m < rows ? ld_global_b128(p.hidden + m * p.N + n0 + (pc - row * GP) * 8) : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int64_t m = (int64_t)s * 32 + (tid >> 4) + u * 16;
      xreg[u] = zero_bf16x8();
      if (m < rows && col < KD) {
        const int y = (int)(m / H), h = (int)(m - (int64_t)y * H);
        while (y >= p.y_cu[seq[u] + 1]) seq[u]++;
        xreg[u] = ld_global_b128(p.x + (p.x_cu[seq[u]] + (int64_t)p.S * (y - p.y_cu[seq[u]]) + j) * p.x_st + (int64_t)h * p.x_sh + ch);
      }
    }
  };
  if (s0 < s1) fetch(s0);
  for (int s = s0; s < s1; s++) {
    bf16_t *const g = gt[s & 1], *const x = xt[s & 1];
#pragma unroll
    for (int u = 0; u < GU; u++) {
      const int pc = tid + u * 256, row = pc / GP;
      if (row < 32) *reinterpret_cast<bf16x8*>(&g[row * LDG + (pc - row * GP) * 8]) = greg[u];
    }
#pragma unroll
    for (int u = 0; u < 2; u++) *reinterpret_cast<bf16x8*>(&x[((tid >> 4) + u * 16) * LDX + (tid & 15) * 8]) = xreg[u];
    __syncthreads();
    if (s + 1 < s1) fetch(s + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const int row = ks * 16 + hl * 8 + (i16 >> 2), cl = (g16 & 1) * 16 + 4 * (i16 & 3);
      const bf16_t* xa = &x[row * LDX + wave * 32 + cl];
      const bf16x8 xv = cat4(lds_read_tr(xa), lds_read_tr(xa + 4 * LDX));
#pragma unroll
      for (int a = 0; a < NT; a++) {
        const bf16_t* ga = &g[row * LDG + a * 32 + cl];
        acc[a] = mfma32(cat4(lds_read_tr(ga), lds_read_tr(ga + 4 * LDG)), xv, acc[a]);
      }
    }
  }
  const int oc = c0 + wave * 32 + l32;
  if (oc >= KD) return;
  float* const o = slots + ((int64_t)blockIdx.z * p.N + n0) * KD + oc;
#pragma unroll
  for (int a = 0; a < NT; a++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[(int64_t)(a * 32 + (i >> 2) * 8 + hl * 4 + (i & 3)) * KD] = acc[a][i];
}

// The parts' sums, in order: rounded into dw, or added to an fp32 buffer.
__global__ void compress_dw_reduce_kernel(const float* slots, int parts, int64_t n4, bf16_t* dw, float* dw32) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n4) return;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  // READ parts in flight: one by one they are a chain of round trips to memory (two launches of 40 samples of up to 1.2K tokens 18.4 -> 11.5 us)
  constexpr int READ = 8;
  int k = 0;
  for (; k + READ <= parts; k += READ) {
    f32x4 v[READ];
#pragma unroll
    for (int u = 0; u < READ; u++) v[u] = *reinterpret_cast<const f32x4*>(slots + ((k + u) * n4 + i) * 4);
#pragma unroll
    for (int u = 0; u < READ; u++) sum += v[u];
  }
  for (; k < parts; k++) sum += *reinterpret_cast<const f32x4*>(slots + (k * n4 + i) * 4);
  if (dw != nullptr) *reinterpret_cast<bf16x4*>(dw + i * 4) = pack4(sum[0], sum[1], sum[2], sum[3]);
  else *reinterpret_cast<f32x4*>(dw32 + i * 4) += sum;
}

// The gradient of hidden from that of the compressed rows (fp32, rounded to bf16 first): ACT -1 the rounding alone.
template <int ACT>
__global__ void compress_act_bwd_kernel(const bf16_t* x, const float* dy, bf16_t* dx, int64_t n8, int d) {
  const int64_t e = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (e >= n8 * 8) return;
  const f32x4 lo = *reinterpret_cast<const f32x4*>(dy + e), hi = *reinterpret_cast<const f32x4*>(dy + e + 4);
  const bf16x8 g8 = pack8(lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]);
  if constexpr (ACT < 0) {
    *reinterpret_cast<bf16x8*>(dx + e) = g8;
  } else {
    const int64_t row = e / d, c = e - row * d;
    const bf16x8 g = ld_global_b128(x + row * 2 * d + c), v = ld_global_b128(x + row * 2 * d + d + c);
    float dg[8], dv[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float gf = (float)g[k], vf = (float)v[k], d0 = (float)g8[k], s = sigmoidf_(gf);
      if (ACT == 0) {
        dv[k] = d0 * s;
        dg[k] = d0 * vf * s * (1.f - s);
      } else {
        dv[k] = d0 * s * gf;
        dg[k] = d0 * vf * (s + gf * s * (1.f - s));
      }
    }
    *reinterpret_cast<bf16x8*>(dx + row * 2 * d + c) = pack8(dg[0], dg[1], dg[2], dg[3], dg[4], dg[5], dg[6], dg[7]);
    *reinterpret_cast<bf16x8*>(dx + row * 2 * d + d + c) = pack8(dv[0], dv[1], dv[2], dv[3], dv[4], dv[5], dv[6], dv[7]);
  }
}

// Mean pooling: dst = bf16(dx + gradient), that of the compressed rows in fp32, rounded to bf16 first.  One thread per 8 channels
// of a (token, head); grid (ceil(x_maxlen * H * D / 8 / 256), B).
__global__ void mean_pool_bwd_sum_kernel(const float* dy, const float* dx, int64_t dx_st, int64_t dx_sh, bf16_t* dst, int64_t dst_st,
                                         int64_t dst_sh, const int32_t* x_cu, const int32_t* y_cu, int H, int D, int K, int S) {
  const int b = blockIdx.y, x0 = x_cu[b], y0 = y_cu[b], xl = x_cu[b + 1] - x0, yl = y_cu[b + 1] - y0, C = D / 8;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)xl * H * C) return;
  const int c = idx % C, h = (idx / C) % H, n = idx / ((int64_t)C * H);
  const int i_lo = n < K ? 0 : (n - K) / S + 1, i_hi = min(n / S, yl - 1);
  float a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = i_lo; i <= i_hi; i++) {
    const float* g = dy + ((int64_t)(y0 + i) * H + h) * D + c * 8;
    const f32x4 lo = *reinterpret_cast<const f32x4*>(g), hi = *reinterpret_cast<const f32x4*>(g + 4);
#pragma unroll
    for (int e = 0; e < 8; e++) a[e] += (float)(bf16_t)(e < 4 ? lo[e] : hi[e - 4]);
  }
  const float inv = 1.f / (float)K;
  const float* at = dx + (int64_t)(x0 + n) * dx_st + (int64_t)h * dx_sh + c * 8;
  const f32x4 lo = *reinterpret_cast<const f32x4*>(at), hi = *reinterpret_cast<const f32x4*>(at + 4);
  *reinterpret_cast<bf16x8*>(dst + (int64_t)(x0 + n) * dst_st + (int64_t)h * dst_sh + c * 8) =
      pack8(lo[0] + a[0] * inv, lo[1] + a[1] * inv, lo[2] + a[2] * inv, lo[3] + a[3] * inv, hi[0] + a[4] * inv, hi[1] + a[5] * inv,
            hi[2] + a[6] * inv, hi[3] + a[7] * inv);
}

int check(const char* who, int H, int D, int K, int S, int N, int act) {
  NSA_REQUIRE(H > 0 && D >= 32 && D % 32 == 0 && S > 0 && K > 0 && K % S == 0, NSA_ERR_BAD_ARG,
              "%s: head dim %d must be a multiple of 32, the window %d one of the stride %d", who, D, K, S);
  NSA_REQUIRE(act >= -1 && act <= 1 && N == (act < 0 ? D : 2 * D), NSA_ERR_BAD_ARG,
              "%s: act must be -1 (linear), 0 (sigmoid-mul) or 1 (swiglu) and the width %d fit it", who, N);
  return NSA_OK;
}

// Parts of the contraction of dW: about two workgroups per CU, each of at least four steps of 32 rows, in slots of at most 64 MB.
int dw_parts(int64_t rows, int KD, int N) {
  const int nt = N % 128 == 0 ? 4 : N % 64 == 0 ? 2 : 1;
  const int64_t tiles = (int64_t)(N / 32 / nt) * cdiv_i(KD, 128);
  int64_t parts = (2 * nsa_device_cus() + tiles - 1) / tiles;
  const int64_t most = (rows + 127) / 128, room = ((int64_t)64 << 20) / ((int64_t)N * KD * 4);
  parts = parts < most ? parts : most;
  parts = parts < room ? parts : room;
  return parts > 1 ? (int)parts : 1;
}

template <int GB, bool GLU, int RS, int AHEAD>
void launch_fwd(const CompressParams& p, int y_maxlen, hipStream_t s) {
  const int64_t rows = (int64_t)y_maxlen * p.H;
  compress_linear_kernel<GB, GLU, RS, AHEAD><<<dim3((unsigned)((rows + 32 * RS - 1) / (32 * RS)), p.B, p.D / 32 / GB), 512, 0, s>>>(p);
}
// All forms sum a product in the same order, so a row's bits do not depend on the batch it is in.  Few rows: 32 by 32 channels per
// workgroup, so that as much of the GPU as there is reads the weight; more of both where that still gives the GPU one round of
// workgroups, of which the larger forms fit a CU once (their stages take 82 to 140 KB of LDS): 64 by 32 up to half as many workgroups
// as CUs, 64 by 64 beyond, which reads the weight and the windows least often.  This launch without the hidden rows, us, 32 rows by 32
// channels / 64 by 32 / 64 by 64 (windows + library product), by rows (workgroups of the first form): gated, 128 channels: 2000 (252)
// 18.5 / 18.7 / 25.8 (40), 3000 (376) 30.6 / 24.2 / 30.0 (40), 4100 (516) 44.0 / 40.3 / 30.9 (50), 6000 (752) 47.4 / 54.3 / 35.6 (54), 24000
// 172 / 148 / 111 (146); 64 channels: 6000 (376) 17.1 / 13.9 / 17.5, 8200 (514) 22.6 / 24.5 / 19.9 (40), 12000 (750) 25.8 / 27.9 / 21.0; linear:
// 128 channels 3000 21.3 / 18.3 / 18.7 (33), 6000 32.6 / 43.5 / 24.8 (41); 192: 2000 (378) 31.6 / 21.1 / 23.7 (35), 3000 (564) 47.4 / 51.4 /
// 30.6 (51); 256: 2000 (504) 50.9 / 29.5 / 31.6 (40), 3000 (752) 71.0 / 71.8 / 39.3 (50).
template <bool GLU>
void dispatch_fwd(const CompressParams& p, int y_maxlen, hipStream_t s) {
  const int64_t blocks = p.D / 32, wgs = ((int64_t)y_maxlen * p.H + 31) / 32 * p.B * blocks;
  const int cus = nsa_device_cus();
  if (wgs <= cus) launch_fwd<1, GLU, 1, 2>(p, y_maxlen, s);
  else if (wgs <= 2 * cus || blocks % 2 != 0) launch_fwd<1, GLU, 2, 2>(p, y_maxlen, s);
  else launch_fwd<2, GLU, 2, 1>(p, y_maxlen, s);
}

}  // namespace

extern "C" {

int nsa_compress_linear_fwd(const void* x, int64_t x_st, int64_t x_sh, const void* w, int64_t w_st, void* hidden, void* out,
                            const int32_t* x_cu, const int32_t* y_cu, int B, int y_maxlen, int H, int D, int kernel_size,
                            int stride, int N, int act, void* stream) {
  const int rc = check("compress_linear_fwd", H, D, kernel_size, stride, N, act);
  if (rc != NSA_OK) return rc;
  if (B <= 0 || y_maxlen <= 0) return NSA_OK;  // (no compressed row: the outputs are empty and may be null)
  NSA_REQUIRE(act < 0 ? hidden != nullptr : out != nullptr, NSA_ERR_BAD_ARG, "compress_linear_fwd: no output given");
  NSA_REQUIRE(x != nullptr && w != nullptr, NSA_ERR_BAD_ARG, "compress_linear_fwd: x or the weight is null");
  CompressParams p = {};
  p.x = (const bf16_t*)x; p.x_st = x_st; p.x_sh = x_sh; p.w = (const bf16_t*)w; p.w_st = w_st;
  p.hidden = (bf16_t*)hidden; p.out = (bf16_t*)out; p.x_cu = x_cu; p.y_cu = y_cu;
  p.B = B; p.H = H; p.D = D; p.K = kernel_size; p.S = stride; p.N = N; p.act = act;
  hipStream_t s = (hipStream_t)stream;
  if (act >= 0) dispatch_fwd<true>(p, y_maxlen, s);
  else dispatch_fwd<false>(p, y_maxlen, s);
  return nsa_check_launch("compress_linear_fwd");
}

int nsa_compress_linear_bwd_dx(const void* dhidden, const void* w, int64_t w_st, void* dx, int64_t dx_st, int64_t dx_sh, void* dst,
                               int64_t dst_st, int64_t dst_sh, const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen,
                               int H, int D, int kernel_size, int stride, int N, void* stream) {
  const int rc = check("compress_linear_bwd_dx", H, D, kernel_size, stride, N, N == D ? -1 : 0);
  if (rc != NSA_OK) return rc;
  NSA_REQUIRE(dx != nullptr || dst != nullptr, NSA_ERR_BAD_ARG, "compress_linear_bwd_dx: no output given");
  if (B <= 0 || x_maxlen <= 0) return NSA_OK;
  // (the gradient of no compressed row is not read and may be null)
  NSA_REQUIRE(w != nullptr && (dhidden != nullptr || x_maxlen < kernel_size), NSA_ERR_BAD_ARG,
              "compress_linear_bwd_dx: the weight or the gradient is null");
  CompressParams p = {};
  p.hidden = (bf16_t*)dhidden; p.w = (const bf16_t*)w; p.w_st = w_st;
  p.dx = (float*)dx; p.dx_st = dx_st; p.dx_sh = dx_sh; p.dst = (bf16_t*)dst; p.dst_st = dst_st; p.dst_sh = dst_sh;
  p.x_cu = x_cu; p.y_cu = y_cu; p.B = B; p.H = H; p.D = D; p.K = kernel_size; p.S = stride; p.N = N;
  const int64_t rows = (int64_t)cdiv_i(x_maxlen, stride) * H;
  compress_linear_dx_kernel<<<dim3((unsigned)((rows + 127) / 128), cdiv_i(stride * D, 128), B), 256, 0, (hipStream_t)stream>>>(p);
  return nsa_check_launch("compress_linear_bwd_dx");
}

int64_t nsa_compress_linear_bwd_dw_ws_bytes(int64_t y_len, int H, int D, int kernel_size, int N) {
  return (int64_t)dw_parts(y_len * H, kernel_size * D, N) * N * kernel_size * D * 4;
}

int nsa_compress_linear_bwd_dw(const void* dhidden, const void* x, int64_t x_st, int64_t x_sh, void* dw, int dw_is_f32,
                               const int32_t* x_cu, const int32_t* y_cu, int B, int64_t y_len, int H, int D, int kernel_size,
                               int stride, int N, void* ws, int64_t ws_bytes, void* stream) {
  const int rc = check("compress_linear_bwd_dw", H, D, kernel_size, stride, N, N == D ? -1 : 0);
  if (rc != NSA_OK) return rc;
  NSA_REQUIRE(B > 0 && y_len > 0, NSA_ERR_BAD_ARG, "compress_linear_bwd_dw: no compressed rows");
  NSA_REQUIRE(dhidden != nullptr && x != nullptr && dw != nullptr && ws != nullptr, NSA_ERR_BAD_ARG,
              "compress_linear_bwd_dw: an operand or the workspace is null");
  NSA_REQUIRE(ws_bytes >= nsa_compress_linear_bwd_dw_ws_bytes(y_len, H, D, kernel_size, N), NSA_ERR_WORKSPACE,
              "compress_linear_bwd_dw: workspace of %lld bytes is too small", (long long)ws_bytes);
  CompressParams p = {};
  p.hidden = (bf16_t*)dhidden; p.x = (const bf16_t*)x; p.x_st = x_st; p.x_sh = x_sh;
  p.x_cu = x_cu; p.y_cu = y_cu; p.B = B; p.H = H; p.D = D; p.K = kernel_size; p.S = stride; p.N = N;
  const int KD = kernel_size * D, parts = dw_parts(y_len * H, KD, N);
  hipStream_t s = (hipStream_t)stream;
  const int cols = cdiv_i(KD, 128);
  if (N % 128 == 0) compress_linear_dw_kernel<4><<<dim3(N / 128, cols, parts), 256, 0, s>>>(p, (float*)ws);
  else if (N % 64 == 0) compress_linear_dw_kernel<2><<<dim3(N / 64, cols, parts), 256, 0, s>>>(p, (float*)ws);
  else compress_linear_dw_kernel<1><<<dim3(N / 32, cols, parts), 256, 0, s>>>(p, (float*)ws);
  int rc2 = nsa_check_launch("compress_linear_bwd_dw");
  if (rc2 != NSA_OK) return rc2;
  const int64_t n4 = (int64_t)N * KD / 4;
  compress_dw_reduce_kernel<<<(unsigned)((n4 + 255) / 256), 256, 0, s>>>((const float*)ws, parts, n4, dw_is_f32 ? nullptr : (bf16_t*)dw,
                                                                      dw_is_f32 ? (float*)dw : nullptr);
  return nsa_check_launch("compress_linear_bwd_dw");
}

int nsa_compress_act_bwd(const void* hidden, const void* dy, void* dhidden, int64_t rows, int D, int act, void* stream) {
  NSA_REQUIRE(D % 8 == 0 && D > 0 && act >= -1 && act <= 1, NSA_ERR_BAD_ARG, "compress_act_bwd: head dim %d, act %d", D, act);
  if (rows <= 0) return NSA_OK;
  NSA_REQUIRE(dy != nullptr && dhidden != nullptr && (act < 0 || hidden != nullptr), NSA_ERR_BAD_ARG, "compress_act_bwd: an operand is null");
  const int64_t n8 = rows * (D / 8);
  const unsigned g = (unsigned)((n8 + 255) / 256);
  hipStream_t s = (hipStream_t)stream;
  if (act < 0) compress_act_bwd_kernel<-1><<<g, 256, 0, s>>>(nullptr, (const float*)dy, (bf16_t*)dhidden, n8, D);
  else if (act == 0) compress_act_bwd_kernel<0><<<g, 256, 0, s>>>((const bf16_t*)hidden, (const float*)dy, (bf16_t*)dhidden, n8, D);
  else compress_act_bwd_kernel<1><<<g, 256, 0, s>>>((const bf16_t*)hidden, (const float*)dy, (bf16_t*)dhidden, n8, D);
  return nsa_check_launch("compress_act_bwd");
}

int nsa_mean_pool_bwd_sum(const void* dy, const void* dx, int64_t dx_st, int64_t dx_sh, void* dst, int64_t dst_st, int64_t dst_sh,
                          const int32_t* x_cu, const int32_t* y_cu, int B, int x_maxlen, int H, int D, int kernel_size, int stride,
                          void* stream) {
  NSA_REQUIRE(D % 8 == 0 && D > 0, NSA_ERR_BAD_ARG, "mean_pool_bwd_sum: head dim %d must be a multiple of 8", D);
  if (B <= 0 || x_maxlen <= 0) return NSA_OK;
  NSA_REQUIRE(dx != nullptr && dst != nullptr && (dy != nullptr || x_maxlen < kernel_size), NSA_ERR_BAD_ARG,
              "mean_pool_bwd_sum: an operand is null");
  const dim3 grid((unsigned)(((int64_t)x_maxlen * H * (D / 8) + 255) / 256), B);
  mean_pool_bwd_sum_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const float*)dy, (const float*)dx, dx_st, dx_sh, (bf16_t*)dst,
                                                                  dst_st, dst_sh, x_cu, y_cu, H, D, kernel_size, stride);
  return nsa_check_launch("mean_pool_bwd_sum");
}

}  // extern "C"
