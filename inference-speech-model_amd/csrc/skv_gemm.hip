// Projections of many rows (prompts, encoder frames) on the matrix cores, y = act(x W^T + b) (+ residual), 16-bit.
//
// What bounds them here: 128 to a few thousand rows leave one or two tiles per compute unit, so a tile's own chain
// decides: 1020 clocks for a 128 x 128 x 64 step with one workgroup on its unit (products 512, LDS 530, the 32 KB through
// L1 at the 31-50 bytes a clock that its 32 KB of lines in flight allow). Hence 128 x 128 and smaller tiles with
// 32 x 32 x 16 products, rows two steps ahead in registers (one step: 1500 x 1280 x 5120 64 us, two: 39), LDS rows
// swizzled instead of padded (padded: 260 of 1050 LDS clocks a step were conflicts), and LDS operations placed between
// products. What the library's GEMM cannot do is in the epilogue: GELU on the fp32 sums, and K and V written by head (and
// a residual add, for callers of the C interface: the models' adds share the LayerNorm's launch).
// Measured (us, bf16, against the library's GEMM and the launches it needs): q/k/v 1500 x 3840 x 1280 with K and V by head
// 24 / 32, 512 x 1152 x 384 5.4 / 14.6, 12000 x 2304 x 768 59 / 93; with GELU 1500 x 5120 x 1280 32 / 34,
// 512 x 2048 x 512 7.3 / 12.1, 130 x 5120 x 1280 10.3 / 14.5.
// Tried: the XCDs' tiles as other blocks of rows and columns (within 3 %, but 40 % worse when a unit gets two);
// workgroups starting at different k (no change); 192 x 128 tiles for every shape (38 against 26 us at 1500 x 5120).
#include <hip/hip_runtime.h>

#include "skv_common.h"
#include "skv_device.h"
#include "speech_kv.h"

using namespace skv;

namespace {

constexpr int kBk = 128;              // bytes of a row per step: 64 elements
constexpr int kLdsRow = kBk;          // chunk c of row r stands at c ^ (r / 2 mod 8): reads and writes both free of conflicts
constexpr int kWavesM = 2, kWavesN = 2, kThreads = 64 * kWavesM * kWavesN;

struct GemmParams {
  const char* x;
  const char* w;
  uint32_t ldx, ldw, x_bytes, w_bytes;  // bytes
  uint32_t m, n, kbytes;
  uint32_t tiles_m, tiles_n;    // output tiles
  uint32_t am, cm, cn, per_xcd;  // XCDs side by side along m; a block of cm x cn tiles = per_xcd each
  const char* bias;             // [n] or NULL
  const char* res;              // [m, n] at ldr (elements) or NULL
  char* y;                      // [m, n] at ldy (elements)
  int64_t ldy, ldr;
  int32_t act;
  // Columns from hd on go to k_out, from 2 hd on to v_out, as [m / t, hd / 64, t, 64] (hd 0: all to y).
  uint32_t hd, t;
  char* k_out;
  char* v_out;
};

// The four rows 8 e + 4 (lane / 32) .. + 3 of a 32 x 32 product's column lane % 32.
__device__ __forceinline__ f32x4 quad(const f32x16& c, int e) {
  return f32x4{c[4 * e], c[4 * e + 1], c[4 * e + 2], c[4 * e + 3]};
}

// v[e] += the eight elements at p (16-byte aligned).
template <int DT>
__device__ __forceinline__ void add16(float* v, const char* p) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) v[2 * i] += lo16<DT>(w[i]), v[2 * i + 1] += hi16<DT>(w[i]);
}

// 64 MI x 64 NI outputs per workgroup, 32 MI x 32 NI per wave.
template <int DT, int MI, int NI>
__global__ __launch_bounds__(kThreads, 2) void gemm_kernel(GemmParams p) {
  constexpr int MT = 2 * MI, NT = 2 * NI;  // 32-row loads of x and w per step and workgroup
  constexpr int kRowsX = 32 * MT, kRowsW = 32 * NT, kBuf = (kRowsX + kRowsW) * kLdsRow;
  constexpr int kOutRow = 64 * NT + 16, kOut = 4 * 16 * MT * kOutRow;
  __shared__ __attribute__((aligned(16))) char s_mem[2 * kBuf > kOut ? 2 * kBuf : kOut];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int g = lane >> 5, r = lane & 31;
  // Consecutive workgroups go round the XCDs; each takes a block of cm x cn tiles (down the rows first).
  const uint32_t xcd = blockIdx.x & 7u;
  const uint32_t slot = blockIdx.x >> 3;
  const uint32_t in_n = slot / p.cm, tm = (xcd % p.am) * p.cm + (slot - in_n * p.cm), tn = (xcd / p.am) * p.cn + in_n;
  if (tm >= p.tiles_m || tn >= p.tiles_n) return;
  const uint32_t m0 = tm * kRowsX, n0 = tn * kRowsW;
  const int steps = (int)((p.kbytes + kBk - 1) / kBk);
  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.x), (short)0, (int)p.x_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t wres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.w), (short)0, (int)p.w_bytes, kBufWord3);
  // Wave w loads rows 8 (w + 4 i) .. + 7 of the tile's x and w rows; rows past the end are out of range: zeros.
  const uint32_t nat_row = lane >> 3, nat_col = (lane & 7) * 16;
  const uint32_t lrow = 8 * wave + nat_row;
  uint32_t xoff[MT], woff[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xoff[i] = m0 + lrow + 32 * i < p.m ? (m0 + lrow + 32 * i) * p.ldx + nat_col : kBufOutOfRange;
#pragma unroll
  for (int i = 0; i < NT; ++i) woff[i] = n0 + lrow + 32 * i < p.n ? (n0 + lrow + 32 * i) * p.ldw + nat_col : kBufOutOfRange;

  uint4 xr[2][MT], wr[2][NT];
  auto issue = [&](int step, int s) __attribute__((always_inline)) {
    const uint32_t k = (uint32_t)step * kBk;
    const uint32_t past = k + nat_col < p.kbytes ? 0u : kBufOutOfRange;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xres, (xoff[i] + k) | past, 0, 0);
      xr[s][i] = make_uint4(v.x, v.y, v.z, v.w);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(wres, (woff[i] + k) | past, 0, 0);
      wr[s][i] = make_uint4(v.x, v.y, v.z, v.w);
    }
  };
  auto stage = [&](int s, int buf) __attribute__((always_inline)) {
    char* d = s_mem + buf * kBuf + lrow * kLdsRow + (nat_col ^ (((lrow >> 1) & 7) * 16));
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<uint4*>(d + 32 * i * kLdsRow) = xr[s][i];
#pragma unroll
    for (int i = 0; i < NT; ++i) *reinterpret_cast<uint4*>(d + (kRowsX + 32 * i) * kLdsRow) = wr[s][i];
  };
  const int wm = wave & 1, wn = wave >> 1;
  // Products of 32 x 32 x 16: lane (g, r) holds 8 elements of row r; a 128-byte row is four of them.
  const int xbase = (32 * MI * wm + r) * kLdsRow, wbase = (kRowsX + 32 * NI * wn + r) * kLdsRow;
  const int rcol = 16 * (g ^ ((r >> 1) & 7));
  uint4 fx[2][2][MI], fw[2][2][NI];
  auto read = [&](int buf, int h) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const char* b = s_mem + buf * kBuf + (rcol ^ (64 * h + 32 * q));
#pragma unroll
      for (int i = 0; i < NI; ++i) fw[h][q][i] = *reinterpret_cast<const uint4*>(b + wbase + 32 * i * kLdsRow);
#pragma unroll
      for (int i = 0; i < MI; ++i) fx[h][q][i] = *reinterpret_cast<const uint4*>(b + xbase + 32 * i * kLdsRow);
    }
  };
  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  auto mma = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = mfma_32x32x16<DT>(fw[h][q][j], fx[h][q][i], acc[i][j]);
  };
  // Step t: LDS buffer t & 1 holds its rows, registers hold those of t + 1 and, in flight, t + 2. One barrier a
  // step: past it the next rows are in LDS and this step's buffer has been read. Each half's LDS traffic goes
  // between its products, one operation each.
  auto step = [&](int t, int s) __attribute__((always_inline)) {
    read(s, 1);
    mma(0);
    stage(s ^ 1, s ^ 1);
#pragma unroll
    for (int i = 0; i < MT + NT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      if (i < 2 * MI * NI) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // product
    }
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(s ^ 1, 0);
    issue(t + 3, s ^ 1);
    mma(1);
#pragma unroll
    for (int i = 0; i < MT + NT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);  // memory read
      if (i < 2 * MI * NI) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  issue(0, 0);
  issue(1, 1);
  stage(0, 0);
  issue(2, 0);
  lds_barrier();
  read(0, 0);
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    step(t, 0);
    step(t + 1, 1);
  }
  if (t < steps) step(t, 0);

  const uint32_t wm0 = m0 + 32 * MI * wm, wn0 = n0 + 32 * NI * wn;
  // The fp32 sums through the wave's LDS rows; bias, activation and residual on whole 16-byte output vectors, in a
  // loop (unrolled, its code alone costs more than its work).
  lds_barrier();
  char* out = s_mem + wave * (16 * MT * kOutRow);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<f32x4*>(out + (32 * i + r) * kOutRow + 128 * j + 32 * e + 16 * g) = quad(acc[i][j], e);
  __builtin_amdgcn_wave_barrier();
  constexpr int kVecs = 2 * NT;
#pragma unroll 1
  for (int o = 0; o < MT * NT / 2; ++o) {
    const uint32_t i = o * 64 + lane, lr = i / kVecs, c = i - lr * kVecs;
    const uint32_t row = wm0 + lr, col = wn0 + 8 * c;
    if (row >= p.m || col >= p.n) continue;
    float v[8];
    *reinterpret_cast<f32x4*>(v) = *reinterpret_cast<const f32x4*>(out + lr * kOutRow + 32 * c);
    *reinterpret_cast<f32x4*>(v + 4) = *reinterpret_cast<const f32x4*>(out + lr * kOutRow + 32 * c + 16);
    if (p.bias) add16<DT>(v, p.bias + 2 * col);
    if (p.act) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = gelu<DT>(v[e]);
    }
    if (p.res) add16<DT>(v, p.res + 2 * ((int64_t)row * p.ldr + col));
    char* d;
    if (p.hd == 0 || col < p.hd) {
      d = p.y + 2 * ((int64_t)row * p.ldy + col);
    } else {
      const uint32_t kv = col >= 2 * p.hd, hc = col - (kv + 1) * p.hd;
      const uint32_t b = row / p.t, tt = row - b * p.t;
      d = (kv ? p.v_out : p.k_out) + 2 * ((((int64_t)b * (p.hd / 64) + hc / 64) * p.t + tt) * 64 + (hc & 63));
    }
    *reinterpret_cast<uint4*>(d) =
        make_uint4(pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3]), pack2<DT>(v[4], v[5]), pack2<DT>(v[6], v[7]));
  }
}

// Tiles in units of 64 x 64, and their measured time for one step of 64 elements (us) with a workgroup per compute unit.
struct Tile { int mi, ni; float step; };
constexpr Tile kTiles[] = {{1, 1, 0.256f}, {1, 2, 0.328f}, {2, 1, 0.334f}, {2, 2, 0.435f}, {2, 3, 0.585f}, {3, 2, 0.58f}};

// The tile with the least estimated time, and that time (us). A unit's workgroups share it, so the steps and epilogues of
// all of them add up (up to 128 x 128 two are resident; the largest tiles' run one after the other); past two rounds
// the last one is half empty on average. Estimate / measured (bf16): 1500 x 5120 x 1280 128 x 128 26.4 / 26.5, 192 x 128
// 41.4 / 38.1; 512 x 1280 x 1280 64 x 64 9.1 / 9.1; 1500 x 3840 x 1280 192 x 128 20.7 / 21.9, 128 x 128 26.5 / 23.8; with
// GELU 3000 x 4096 x 1024 192 x 128 44.6 / 44.7 (the library and its GELU launch 38.4).
int pick_tile(uint32_t m, uint32_t n, int steps, bool act, float* us) {
  int best = 0;
  float best_cost = 1e30f;
  const int64_t cus = compute_units();
  for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); ++i) {
    const Tile& t = kTiles[i];
    const int64_t tiles = cdiv(m, 64 * t.mi) * cdiv(n, 64 * t.ni);
    const float rounds = tiles > 2 * cus ? (float)tiles / (float)cus + 0.5f : (float)cdiv(tiles, cus);
    const float area = (float)(t.mi * t.ni);
    const float cost = rounds * ((float)steps * t.step + (act ? 1.37f : 0.72f) * area) + (area > 4.f ? 4.8f * rounds : 3.3f);
    if (cost < best_cost) best = i, best_cost = cost;
  }
  *us = best_cost;
  return best;
}

// The library's GEMM and a GELU launch after it (us). Estimate / measured (bf16): 512 x 5120 x 1280 20.4 / 21.5, 1500 35.6 /
// 34.0, 3000 58.7 / 55; 1024 x 4096 x 1024 22.6 / 22.3; 1500 x 3072 x 768 20.8 / 23.2.
float library_gelu_us(float m, float n, float k) { return 12.5f + 2.35e-9f * m * n * k; }

// The blocks of tiles that the XCDs take: the shape that reads the fewest rows (each XCD reads its own from memory), of
// those that leave no unit with more tiles than an even spread would.
void place(GemmParams& p, const Tile& t) {
  const int64_t cus = cdiv(compute_units(), 8);  // of one XCD
  const int64_t even = cdiv(cdiv((int64_t)p.tiles_m * p.tiles_n, 8), cus);
  int64_t best = -1;
  for (uint32_t am = 1; am <= 8; am *= 2) {
    const int64_t cm = cdiv(p.tiles_m, am), cn = cdiv(p.tiles_n, 8 / am);
    const int64_t rows = cm * t.mi + cn * t.ni;
    const bool fits = cdiv(cm * cn, cus) <= even;
    if (best < 0 || (fits && rows < best)) {
      p.am = am, p.cm = (uint32_t)cm, p.cn = (uint32_t)cn, p.per_xcd = (uint32_t)(cm * cn);
      best = fits ? rows : (int64_t)1 << 60;
    }
  }
}

template <int DT>
void launch_gemm(const GemmParams& p, int tile, hipStream_t st) {
  const dim3 grid(8 * p.per_xcd);
  switch (tile) {
    case 0: hipLaunchKernelGGL((gemm_kernel<DT, 1, 1>), grid, dim3(kThreads), 0, st, p); break;
    case 1: hipLaunchKernelGGL((gemm_kernel<DT, 1, 2>), grid, dim3(kThreads), 0, st, p); break;
    case 2: hipLaunchKernelGGL((gemm_kernel<DT, 2, 1>), grid, dim3(kThreads), 0, st, p); break;
    case 3: hipLaunchKernelGGL((gemm_kernel<DT, 2, 2>), grid, dim3(kThreads), 0, st, p); break;
    case 4: hipLaunchKernelGGL((gemm_kernel<DT, 2, 3>), grid, dim3(kThreads), 0, st, p); break;
    default: hipLaunchKernelGGL((gemm_kernel<DT, 3, 2>), grid, dim3(kThreads), 0, st, p); break;
  }
}

}  // namespace

int skv_rows_linear(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, int32_t act,
                    const void* res, int64_t ldr, void* y, int64_t ldy, void* k_out, void* v_out, int32_t hd,
                    int32_t tokens, int32_t m, int32_t n, int32_t k, int32_t dtype, void* stream) {
  const char* who = "skv_rows_linear";
  const int eb = elt_bytes(dtype);
  if (eb == 0) return fail(SKV_EDTYPE, "%s: unknown dtype %d", who, dtype);
  const int64_t ny = hd > 0 ? hd : n;
  if (m < 0 || n <= 0 || k <= 0 || ldx < k || ldw < k || ldy < ny || (res && ldr < n) || hd < 0 ||
      (act != 0 && act != SKV_ACT_GELU))
    return fail(SKV_EINVAL, "%s: bad sizes m=%d n=%d k=%d ldx=%lld ldw=%lld ldy=%lld ldr=%lld hd=%d act=%d", who, m, n, k,
                (long long)ldx, (long long)ldw, (long long)ldy, (long long)ldr, hd, act);
  if (hd > 0 && (n != 3 * (int64_t)hd || hd % 64 || tokens <= 0 || m % tokens || res))
    return fail(SKV_EINVAL, "%s: q/k/v columns need n = 3 hd, hd a multiple of 64 and m of tokens, no residual", who);
  if (m == 0) return SKV_OK;
  if (!x || !w || !y || (hd > 0 && (!k_out || !v_out))) return fail(SKV_EINVAL, "%s: null pointer argument", who);
  const int64_t kb = (int64_t)k * eb;
  const int64_t xb = (int64_t)(m - 1) * ldx * eb + kb, wb = (int64_t)(n - 1) * ldw * eb + kb;
  if (eb != 2 || n % 8 || kb % 16 || ldx % 8 || ldw % 8 || ldy % 8 || (res && ldr % 8) || xb > 0x7fffffff ||
      wb > 0x7fffffff || !aligned16(x) || !aligned16(w) || !aligned16(y) || !aligned16(bias) ||
      !aligned16(res) || (hd > 0 && (!aligned16(k_out) || !aligned16(v_out))))
    return fail(SKV_EUNSUPPORTED, "%s: m=%d n=%d k=%d dtype=%d or a layout that is not whole 16-byte vectors", who, m, n, k,
                dtype);
  // Past about 1.5 x 2^35 products the library's larger tiles win (q/k/v of 12000 x 3840 x 1280: 162 us against 152 with
  // the two copies, 12000 x 3072 x 1024: 110 against 141).
  if ((int64_t)m * n * k > (int64_t)3 << 34)
    return fail(SKV_EUNSUPPORTED, "%s: m=%d n=%d k=%d is a large GEMM", who, m, n, k);
  GemmParams p{};
  p.x = (const char*)x, p.w = (const char*)w;
  p.ldx = m > 1 ? (uint32_t)(ldx * eb) : (uint32_t)kb, p.ldw = n > 1 ? (uint32_t)(ldw * eb) : (uint32_t)kb;
  p.x_bytes = (uint32_t)xb, p.w_bytes = (uint32_t)wb;
  p.m = (uint32_t)m, p.n = (uint32_t)n, p.kbytes = (uint32_t)kb;
  float us = 0.f;
  const int tile = pick_tile(p.m, p.n, (int)cdiv(kb, kBk), act != 0, &us);
  // own / library measured (us, bf16, GELU): 130 x 5120 x 1280 10.1 / 14.4, 512 x 2048 x 512 7.4 / 12.1, 1500 x 5120 x 1280
  // 30.1 / 31.9, 1608 x 4096 x 1024 25.2 / 27.9; the library: 3000 x 4096 x 1024 44.7 / 38.4, 1608 x 5120 x 1280 38.7 / 34.2,
  // 3000 x 5120 x 1280 59.7 / 48.3. The library's line is that of one version: with another both ways stay right, and the
  // crossover may lie elsewhere.
  if (act && us > 1.05f * library_gelu_us((float)m, (float)n, (float)k))
    return fail(SKV_EUNSUPPORTED, "%s: m=%d n=%d k=%d fills the units badly", who, m, n, k);
  p.tiles_m = (uint32_t)cdiv(m, 64 * kTiles[tile].mi);
  p.tiles_n = (uint32_t)cdiv(n, 64 * kTiles[tile].ni);
  place(p, kTiles[tile]);
  p.bias = (const char*)bias, p.res = (const char*)res, p.y = (char*)y;
  p.ldy = ldy, p.ldr = ldr, p.act = act;
  p.hd = (uint32_t)hd, p.t = (uint32_t)tokens, p.k_out = (char*)k_out, p.v_out = (char*)v_out;
  if (dtype == SKV_BF16)
    launch_gemm<SKV_BF16>(p, tile, (hipStream_t)stream);
  else
    launch_gemm<SKV_F16>(p, tile, (hipStream_t)stream);
  return check_launch(who);
}
