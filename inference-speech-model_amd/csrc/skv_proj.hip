// Decode-batch projections on the matrix cores, y = act(x W^T + b), and the residual
// add + LayerNorm between them.
//
// What bounds them: few rows (the decode batch), so the products are nothing and W is read
// once; a launch is its ~1.8 us floor, one trip to HBM for W (~0.6 us, loaded), and the bytes each
// compute unit takes through its L1 (W and, many times over the chip, x: ~35-45 B/clk). Hence:
//   * one workgroup per compute unit or fewer, with the smallest tile that allows it: the
//     bytes a unit loads are (tile rows + tile columns) * k;
//   * the waves split k, so all of a workgroup's loads (R 128-byte chunks per row and wave)
//     are in flight at once, before the first product; nothing is issued past the row;
//   * loads read whole 128-byte lines (8 lanes per row) and reach the operand layout
//     through the wave's own padded LDS rows: in operand order every 16 lanes would touch 16 lines;
//   * rows past 6 KiB (a large MLP's second product) are split over workgroups too; the fp32 partials
//     are summed by the residual add + LayerNorm that follows, which costs no launch of its own.
// Workgroups with the same weight tile sit on one XCD (block x is the tile modulo 8), so each XCD's L2 reads
// its weights from memory once.
// Measured (graph-timed, bf16, weights from HBM), against hipBLASLt: 64 rows, n x k 3840 x 1280 5.9 / 9.3 us,
// 1280 x 1280 4.7 / 8.8, 5120 x 1280 7.7 / 9.7, 1280 x 5120 7.2 / 17.0, 768 x 768 2.7 / 7.1, 256 x 256 2.0 / 6.5.
// Tried: one chunk in flight per wave (1280 x 1280 5.2 us); two or three in a ring whose loads ran past the row's
// end (5.4, 5.6: an out-of-range load still takes its L1 cycles); k = 1280 split over three
// workgroups (3.5 us alone, but the sum in the next launch takes the gain back: 7.45 / 7.46 us for the pair).
#include <hip/hip_runtime.h>

#include "skv_common.h"
#include "skv_device.h"
#include "speech_kv.h"

using namespace skv;

namespace {

constexpr int kChunkBytes = 128;              // bytes of one row that a step stages (8 lanes x 16 bytes)
constexpr int kStageRow = kChunkBytes + 16;   // LDS row of a staged chunk, padded: operand reads hit all banks once

struct ProjEpilogue {
  const void* bias;  // [n] or NULL
  char* y;           // [m, n] at row stride ldy
  float* part;       // split: fp32 partials [splits][m][n]; else NULL
  int64_t ldy;       // elements
  int32_t act;       // 1: GELU (erf)
  const char* res;   // [m, n] added to the fp32 result, at row stride ldr; or NULL
  int64_t ldr;
  float2* stats;     // [m, n / 16]: sum and squared deviations of each 16 stored elements; or NULL
};

// LayerNorm of the x rows before the product (gamma NULL: none).
struct ProjNorm {
  const void* gamma;  // [k]
  const void* beta;
  const float2* stats;  // [m, k / 16] as ProjEpilogue::stats of the projection that stored x
  float eps, inv_k;
};

// One 16 x 16 product step over a 128-byte chunk of 16 weight rows and 16 rows of x, both in LDS
// rows of kStageRow bytes; lane (g, r) of the operands is row r. The contraction index an element
// stands for only has to agree between the two operands.
template <int DT>
__device__ __forceinline__ f32x4 chunk_mfma(const uint4& a0, const uint4& a1, const uint4& b0, const uint4& b1, f32x4 c) {
  if constexpr (DT == SKV_F32) {
    const float af[8] = {__uint_as_float(a0.x), __uint_as_float(a0.y), __uint_as_float(a0.z), __uint_as_float(a0.w),
                         __uint_as_float(a1.x), __uint_as_float(a1.y), __uint_as_float(a1.z), __uint_as_float(a1.w)};
    const float bf[8] = {__uint_as_float(b0.x), __uint_as_float(b0.y), __uint_as_float(b0.z), __uint_as_float(b0.w),
                         __uint_as_float(b1.x), __uint_as_float(b1.y), __uint_as_float(b1.z), __uint_as_float(b1.w)};
#pragma unroll
    for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], bf[e], c, 0, 0, 0);
    return c;
  } else {
    c = mfma_16x16x32<DT>(a0, b0, c);
    return mfma_16x16x32<DT>(a1, b1, c);
  }
}

__device__ __forceinline__ uint4 load_cached(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// The elements of a 16-byte vector of x, normalised and rounded to the dtype: (x - mean) * rstd * gamma + beta.
// st: mean and rstd, for 16-bit rows -mean * rstd and rstd (one operation less; with the subtraction first 64 x 1280 x 1280
// takes 6.1 us instead of 5.9). The rounding this adds is no larger than the mean's own in fp32: over identity weights the
// error against float64 is that of the LayerNorm launch to 0.1 %, for a mean of 8 to 475 times the spread (fp16, mean 400:
// 2.080e-4 / 2.078e-4, torch in fp32 2.081e-4; mean 64 2.075e-4 in all three).
template <int DT>
__device__ __forceinline__ uint4 norm16(const uint4& x, const uint4& gamma, const uint4& beta, float2 st) {
  const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, gw[4] = {gamma.x, gamma.y, gamma.z, gamma.w};
  const uint32_t bw[4] = {beta.x, beta.y, beta.z, beta.w};
  uint32_t r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == SKV_F32) {
      r[i] = __float_as_uint(
          fmaf((__uint_as_float(xw[i]) - st.x) * st.y, __uint_as_float(gw[i]), __uint_as_float(bw[i])));
    } else {
      r[i] = pack2<DT>(fmaf(fmaf(lo16<DT>(xw[i]), st.y, st.x), lo16<DT>(gw[i]), lo16<DT>(bw[i])),
                       fmaf(fmaf(hi16<DT>(xw[i]), st.y, st.x), hi16<DT>(gw[i]), hi16<DT>(bw[i])));
    }
  }
  return make_uint4(r[0], r[1], r[2], r[3]);
}

// Four elements as loaded, and their fp32 values.
template <int DT> struct Quad { uint2 v; };
template <> struct Quad<SKV_F32> { f32x4 v; };
template <int DT>
__device__ __forceinline__ Quad<DT> load_raw(const char* p, int64_t elt) {
  return *reinterpret_cast<const Quad<DT>*>(p + elt * (DT == SKV_F32 ? 4 : 2));
}
template <int DT>
__device__ __forceinline__ f32x4 widen(const Quad<DT>& q) {
  if constexpr (DT == SKV_F32) {
    return q.v;
  } else {
    return f32x4{lo16<DT>(q.v.x), hi16<DT>(q.v.x), lo16<DT>(q.v.y), hi16<DT>(q.v.y)};
  }
}
template <int DT>
__device__ __forceinline__ f32x4 load_quad(const char* p, int64_t elt) {
  return widen<DT>(load_raw<DT>(p, elt));
}
template <int DT>
__device__ __forceinline__ void store_quad(char* p, int64_t elt, const f32x4& v) {
  if constexpr (DT == SKV_F32) {
    *reinterpret_cast<f32x4*>(p + elt * 4) = v;
  } else {
    *reinterpret_cast<uint2*>(p + elt * 2) = make_uint2(pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3]));
  }
}
// The value as it reads back from the tensor type.
template <int DT>
__device__ __forceinline__ f32x4 round_quad(const f32x4& v) {
  if constexpr (DT == SKV_F32) {
    return v;
  } else {
    const uint32_t a = pack2<DT>(v[0], v[1]), b = pack2<DT>(v[2], v[3]);
    return f32x4{lo16<DT>(a), hi16<DT>(a), lo16<DT>(b), hi16<DT>(b)};
  }
}

// Sum of N values in each of LANES adjacent lanes, value i of lane l standing at index l + i * LANES of the row: over the
// indices equal modulo 32 in order, then a tree over the 32 sums, so the bits do not depend on LANES.
template <int LANES, int N>
__device__ __forceinline__ float sum_mod32(const float* v) {
  constexpr int kClasses = 32 / LANES;
  static_assert(N % kClasses == 0, "whole rounds of 32 indices");
  float s[kClasses];
#pragma unroll
  for (int c = 0; c < kClasses; ++c) s[c] = v[c];
#pragma unroll
  for (int i = kClasses; i < N; ++i) s[i % kClasses] += v[i];
#pragma unroll
  for (int h = kClasses / 2; h > 0; h /= 2)
#pragma unroll
    for (int c = 0; c < h; ++c) s[c] += s[c + h];
  float x = s[0];
  if constexpr (LANES >= 32) x += xor_lane<16>(x);
  if constexpr (LANES >= 16) x += xor_lane<8>(x);
  if constexpr (LANES >= 8) x += xor_lane<4>(x);
  x += xor_lane<2>(x);
  return x + xor_lane<1>(x);
}

// A workgroup of WAVES waves owns 16 MI rows x 16 NI columns of y over split_chunks chunks of k.
// Grid: (weight tile mod 8, row tile, weight tile / 8 * splits + split).
//
// NORM: x is the LayerNorm of the given rows. The projection that stored them left the sum and the squared deviations
// of every 16 elements, so a workgroup has its rows' mean and variance from k / 16 pairs a row (one load ahead of the
// x loads) and normalises in registers on the way to LDS; a launch of its own costs 2.0 (k = 256) to 2.7 us (1280).
template <int DT, int MI, int NI, int WAVES, int R, bool NORM>
__global__ __launch_bounds__(64 * WAVES) void proj_kernel(
    const char* __restrict__ x, const char* __restrict__ w, uint32_t ldx, uint32_t ldw, uint32_t x_bytes,
    uint32_t w_bytes, uint32_t m, uint32_t n, uint32_t kbytes, uint32_t split_chunks, uint32_t splits, ProjNorm q,
    ProjEpilogue p) {
  constexpr int kRows = 16 * (MI + NI);
  constexpr int kStage = WAVES * kRows * kStageRow;
  constexpr int kTiles = MI * NI;
  constexpr int kReduce = WAVES * kTiles * 64 * 16;
  __shared__ __attribute__((aligned(16))) char s_mem[kStage > kReduce ? kStage : kReduce];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int g = lane >> 4, r = lane & 15;
  uint32_t grp = blockIdx.z, split = 0;
  if (splits > 1) {
    grp = blockIdx.z / splits;
    split = blockIdx.z - grp * splits;
  }
  const uint32_t n0 = (grp * 8u + blockIdx.x) * (16 * NI), m0 = blockIdx.y * (16 * MI);
  if (n0 >= n) return;
  const uint32_t k_begin = split * split_chunks * kChunkBytes;
  const uint32_t k_end = min(kbytes, k_begin + split_chunks * kChunkBytes);
  const __amdgpu_buffer_rsrc_t wres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w), (short)0, (int)w_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t xres =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(x), (short)0, (int)x_bytes, kBufWord3);
  // Byte offsets of the wave's loads (8 rows each); a row past the end is out of range and reads zeros.
  const uint32_t nat_row = lane >> 3, nat_col = (lane & 7) * 16;
  uint32_t woff[2 * NI], xoff[2 * MI];
#pragma unroll
  for (int j = 0; j < 2 * NI; ++j) {
    const uint32_t row = n0 + 8 * j + nat_row;
    woff[j] = row < n ? row * ldw + nat_col : kBufOutOfRange;
  }
#pragma unroll
  for (int j = 0; j < 2 * MI; ++j) {
    const uint32_t row = m0 + 8 * j + nat_row;
    xoff[j] = row < m ? row * ldx + nat_col : kBufOutOfRange;
  }
  char* stage = s_mem + wave * (kRows * kStageRow);
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // NORM: 16 MI / WAVES rows of statistics per wave, kNormLanes lanes each.
  constexpr int kElt = DT == SKV_F32 ? 4 : 2;
  constexpr int kNormRows = 16 * MI / WAVES, kNormLanes = 64 / kNormRows;
  constexpr int kNormLoads = (WAVES * R * (kChunkBytes / (16 * kElt)) + 31) / 32 * (32 / kNormLanes);
  __shared__ float2 s_norm[NORM ? 16 * MI : 1];
  [[maybe_unused]] const uint32_t groups = kbytes / (16 * kElt);
  [[maybe_unused]] const uint32_t srow = wave * kNormRows + lane / kNormLanes, sl = lane % kNormLanes;
  float2 st[NORM ? kNormLoads : 1];
  __amdgpu_buffer_rsrc_t gres, bres;
  if constexpr (NORM) {
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float2*>(q.stats), (short)0, (int)(m * groups * 8u), kBufWord3);
    gres = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q.gamma), (short)0, (int)kbytes, kBufWord3);
    bres = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q.beta), (short)0, (int)kbytes, kBufWord3);
    const uint32_t row = m0 + srow;
    const uint32_t base = row < m ? row * groups * 8u : kBufOutOfRange;
#pragma unroll
    for (int i = 0; i < kNormLoads; ++i) {
      const uint32_t c = sl + i * kNormLanes;
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(sres, (base + c * 8u) | (c < groups ? 0u : kBufOutOfRange),
                                                          0, 0);
      st[i] = make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    }
  }
  // The epilogue's operands (thread's outputs: 4 columns of one row per trip), loaded ahead of the rows.
  constexpr int kOut = (kTiles + WAVES - 1) / WAVES;
  Quad<DT> bias[kOut] = {}, res[kOut] = {};
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    const int tile = o * WAVES + wave;
    const uint32_t mrow = m0 + 16 * (tile / NI) + r, ncol = n0 + 16 * (tile % NI) + 4 * g;
    if (tile < kTiles && ncol < n) {
      if (p.bias) bias[o] = load_raw<DT>(static_cast<const char*>(p.bias), ncol);
      if (p.res && mrow < m) res[o] = load_raw<DT>(p.res, (int64_t)mrow * p.ldr + ncol);
    }
  }
  uint4 wr[R][2 * NI], xr[R][2 * MI];
  uint4 gr[NORM ? R : 1], br[NORM ? R : 1];
  float2 rowst[2 * MI];
  auto issue = [&](uint32_t k0, int s) __attribute__((always_inline)) {
    const uint32_t past = k0 + nat_col < k_end ? 0u : kBufOutOfRange;
#pragma unroll
    for (int j = 0; j < 2 * NI; ++j) wr[s][j] = load_cached(wres, (woff[j] + k0) | past);
#pragma unroll
    for (int j = 0; j < 2 * MI; ++j) xr[s][j] = load_cached(xres, (xoff[j] + k0) | past);
    if constexpr (NORM) {
      gr[s] = load_cached(gres, (k0 + nat_col) | past);
      br[s] = load_cached(bres, (k0 + nat_col) | past);
    }
  };
  auto compute = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2 * NI; ++j)
      *reinterpret_cast<uint4*>(stage + (8 * j + nat_row) * kStageRow + nat_col) = wr[s][j];
#pragma unroll
    for (int j = 0; j < 2 * MI; ++j) {
      uint4 v = xr[s][j];
      if constexpr (NORM) v = norm16<DT>(v, gr[s], br[s], rowst[j]);
      *reinterpret_cast<uint4*>(stage + (16 * NI + 8 * j + nat_row) * kStageRow + nat_col) = v;
    }
    __builtin_amdgcn_wave_barrier();
    uint4 a[NI][2];
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const char* row = stage + (16 * j + r) * kStageRow + 16 * g;
      a[j][0] = *reinterpret_cast<const uint4*>(row);
      a[j][1] = *reinterpret_cast<const uint4*>(row + 64);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const char* row = stage + (16 * (NI + i) + r) * kStageRow + 16 * g;
      const uint4 b0 = *reinterpret_cast<const uint4*>(row);
      const uint4 b1 = *reinterpret_cast<const uint4*>(row + 64);
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = chunk_mfma<DT>(a[j][0], a[j][1], b0, b1, acc[i][j]);
    }
    __builtin_amdgcn_wave_barrier();
  };
  // The wave's chunks are wave, wave + WAVES, ... of the split, R at most. All their loads are in flight
  // before the first product; the last one, which only some waves have, first, so that every wait
  // counts a fixed number of younger loads.
  const uint32_t k0 = k_begin + wave * kChunkBytes;
  constexpr uint32_t kRound = WAVES * kChunkBytes;
  const bool last = k0 + (R - 1) * kRound < k_end;
  if (last) issue(k0 + (R - 1) * kRound, R - 1);
#pragma unroll
  for (int s = 0; s < R - 1; ++s) issue(k0 + s * kRound, s);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORM) {
    float v[kNormLoads];
#pragma unroll
    for (int i = 0; i < kNormLoads; ++i) v[i] = st[i].x;  // pairs past the row read zeros
    const float mean = sum_mod32<kNormLanes, kNormLoads>(v) * q.inv_k;
#pragma unroll
    for (int i = 0; i < kNormLoads; ++i) {
      const float d = fmaf(-16.f, mean, st[i].x);  // 16 (group mean - row mean)
      v[i] = sl + i * kNormLanes < groups ? fmaf(d * 0.0625f, d, st[i].y) : 0.f;
    }
    const float rstd = rsqrtf(sum_mod32<kNormLanes, kNormLoads>(v) * q.inv_k + q.eps);
    if (sl == 0) s_norm[srow] = make_float2(DT == SKV_F32 ? mean : -mean * rstd, rstd);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 2 * MI; ++j) rowst[j] = s_norm[8 * j + nat_row];
  }
  if (last) compute(R - 1);
#pragma unroll
  for (int s = 0; s < R - 1; ++s) compute(s);
  // Sum the waves' partial tiles through LDS.
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(s_mem);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) red[(wave * kTiles + i * NI + j) * 64 + lane] = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    const int tile = o * WAVES + wave, t = tile * 64 + lane;
    if (tile >= kTiles) break;
    f32x4 v = red[t];
#pragma unroll
    for (int wv = 1; wv < WAVES; ++wv) v += red[wv * kTiles * 64 + t];
    const uint32_t mrow = m0 + 16 * (tile / NI) + r;
    const uint32_t ncol = n0 + 16 * (tile % NI) + 4 * g;
    const bool in = mrow < m && ncol < n;
    if (p.part) {
      if (in) *reinterpret_cast<f32x4*>(p.part + ((int64_t)split * m + mrow) * n + ncol) = v;
      continue;
    }
    v += widen<DT>(bias[o]);
    if (p.act) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu<DT>(v[e]);
    }
    v += widen<DT>(res[o]);
    v = round_quad<DT>(v);
    if (in) store_quad<DT>(p.y, (int64_t)mrow * p.ldy + ncol, v);
    if (p.stats) {  // n is a multiple of 16; the four lanes of a row's 16 elements, every lane active
      float s16 = (v[0] + v[1]) + (v[2] + v[3]);
      s16 += xor_lane<16>(s16);
      s16 += xor_lane<32>(s16);
      const f32x4 d = v - s16 * 0.0625f;
      float q16 = fmaf(d[0], d[0], d[1] * d[1]) + fmaf(d[2], d[2], d[3] * d[3]);
      q16 += xor_lane<16>(q16);
      q16 += xor_lane<32>(q16);
      if (in && g == 0) p.stats[(int64_t)mrow * (n / 16) + ncol / 16] = make_float2(s16, q16);
    }
  }
}

// ---------------------------------------------------------------------------
// Residual add + LayerNorm, optionally summing a split projection's partials:
//   y   = sum_s part[s] + bias   (fp32, splits in order), or the given tensor
//   sum = x + y rounded to the tensor type
//   norm = LayerNorm(sum) * gamma + beta, fp32 statistics in two passes over registers
// One workgroup per row, 4 elements per thread: for few rows a launch is its floor, one round of loads and two
// reductions, so the elements per lane decide (64 x 1280 fp32 3.1 us, one wave per row 3.8). Many rows and short ones take
// add_norm_rows_kernel.
// ---------------------------------------------------------------------------
constexpr int kMaxNormVecs = 512;  // 16-byte vectors of a row

struct AddNormParams {
  const char* x;       // NULL: the sum is y
  const char* y;       // NULL: no tensor to add
  const float* part;   // NULL: no partials
  const char* bias;    // with partials; NULL: none
  const char* gamma;   // NULL: the sum alone
  const char* beta;
  char* sum;           // NULL: not stored
  char* norm;
  int64_t ldx, ldy, lds, ldn;  // elements
  int64_t part_stride;         // floats between partials
  int32_t quads, splits;
  float eps, inv_n;
};

// Sum over the workgroup; every thread gets the same bits. `slot` holds one float per wave.
__device__ __forceinline__ float block_sum(float v, float* slot, int waves) {
  v = group_sum<64>(v);
  if (waves == 1) return v;
  if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = slot[0];
  for (int w = 1; w < waves; ++w) t += slot[w];
  return t;
}

template <int DT>
__global__ __launch_bounds__(1024) void add_norm_kernel(AddNormParams p) {
  __shared__ float s_red[2][16];
  const int c = threadIdx.x;
  const int waves = blockDim.x >> 6;
  const int64_t row = blockIdx.x;
  const bool in = c < p.quads;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f}, gm = v, bt = v;
  if (in) {
    if (p.gamma) {
      gm = load_quad<DT>(p.gamma, 4 * c);
      bt = load_quad<DT>(p.beta, 4 * c);
    }
    f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.x) x = load_quad<DT>(p.x, row * p.ldx + 4 * c);
    if (p.part) {
      const float* part = p.part + (row * p.quads + c) * 4;
      v = *reinterpret_cast<const f32x4*>(part);
      for (int s = 1; s < p.splits; ++s) v += *reinterpret_cast<const f32x4*>(part + s * p.part_stride);
      if (p.bias) v += load_quad<DT>(p.bias, 4 * c);
    } else if (p.y) {
      v = load_quad<DT>(p.y, row * p.ldy + 4 * c);
    }
    v = p.x ? round_quad<DT>(x + v) : round_quad<DT>(v);
    if (p.sum) store_quad<DT>(p.sum, row * p.lds + 4 * c, v);
  }
  if (!p.gamma) return;
  const float mean = block_sum((v[0] + v[1]) + (v[2] + v[3]), s_red[0], waves) * p.inv_n;
  const f32x4 d = v - mean;
  float q = in ? fmaf(d[0], d[0], d[1] * d[1]) + fmaf(d[2], d[2], d[3] * d[3]) : 0.f;
  const float rstd = rsqrtf(block_sum(q, s_red[1], waves) * p.inv_n + p.eps);
  if (in) store_quad<DT>(p.norm, row * p.ldn + 4 * c, d * rstd * gm + bt);
}

// The same without partials, one wave per row (4 rows per workgroup, VPL 16-byte vectors per lane). Many rows are bound by
// memory, and there its wide accesses and the want of a barrier count: 12000 x 1280 bf16 22.3 us (5.5 TB/s; one
// workgroup per row 37.4), without the add 12.3 (22.9), fp16 22.4 (38.0).
template <int DT, int VPL>
__global__ __launch_bounds__(256) void add_norm_rows_kernel(AddNormParams p, int32_t rows) {
  constexpr int EPL = Elt<DT>::EPL;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // uniform over the wave
  const int vecs = p.quads * 4 / EPL;
  const uint4* x = reinterpret_cast<const uint4*>(p.x) + row * (p.ldx / EPL);
  uint4 raw[VPL], gv[VPL], bv[VPL];
  // Every load up front (x, y, gamma, beta): one memory round trip per row.
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int c = lane + 64 * j;
    raw[j] = gv[j] = bv[j] = make_uint4(0u, 0u, 0u, 0u);
    if (c < vecs) {
      raw[j] = x[c];
      gv[j] = reinterpret_cast<const uint4*>(p.gamma)[c];
      bv[j] = reinterpret_cast<const uint4*>(p.beta)[c];
    }
  }
  auto pack = [](const float* f) __attribute__((always_inline)) {
    if constexpr (DT == SKV_BF16) {  // fp16: the packed form is the slower one here (64 x 1280 3.9 us against 3.4)
      return make_uint4(pack2<DT>(f[0], f[1]), pack2<DT>(f[2], f[3]), pack2<DT>(f[4], f[5]), pack2<DT>(f[6], f[7]));
    } else {
      return pack16<DT>(f);
    }
  };
  if (p.y) {
    const uint4* y = reinterpret_cast<const uint4*>(p.y) + row * (p.ldy / EPL);
    uint4 ry[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      ry[j] = make_uint4(0u, 0u, 0u, 0u);
      if (lane + 64 * j < vecs) ry[j] = y[lane + 64 * j];
    }
    uint4* sum = reinterpret_cast<uint4*>(p.sum) + (p.sum ? row * (p.lds / EPL) : 0);
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      float a[EPL], b[EPL];
      unpack16<DT>(raw[j], a);
      unpack16<DT>(ry[j], b);
#pragma unroll
      for (int e = 0; e < EPL; ++e) a[e] += b[e];
      raw[j] = pack(a);  // rounded to the tensor type, like the stored sum
      if (p.sum && lane + 64 * j < vecs) sum[lane + 64 * j] = raw[j];
    }
  }
  float v[VPL][EPL], s = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    unpack16<DT>(raw[j], v[j]);
#pragma unroll
    for (int e = 0; e < EPL; ++e) s += v[j][e];
  }
  const float mean = group_sum<64>(s) * p.inv_n;
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      v[j][e] -= mean;
      if (lane + 64 * j < vecs) q = fmaf(v[j][e], v[j][e], q);
    }
  }
  const float rstd = rsqrtf(group_sum<64>(q) * p.inv_n + p.eps);
  uint4* norm = reinterpret_cast<uint4*>(p.norm) + row * (p.ldn / EPL);
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    if (lane + 64 * j >= vecs) continue;
    float g[EPL], b[EPL];
    unpack16<DT>(gv[j], g);
    unpack16<DT>(bv[j], b);
#pragma unroll
    for (int e = 0; e < EPL; ++e) g[e] = v[j][e] * rstd * g[e] + b[e];
    norm[lane + 64 * j] = pack(g);
  }
}

// One wave per row but for long rows (past 2 KiB) of a decode batch or a short prompt, where the elements per lane decide.
// Wave / workgroup per row (us, with the add): bf16 64 x 1024 3.0 / 3.1, 64 x 1280 3.5 / 3.3, 256 x 2048 4.1 / 4.0,
// 512 x 1280 4.0 / 4.1, 800 x 2048 5.4 / 5.9, 3000 x 1280 7.9 / 9.9; fp32 64 x 512 2.8 / 2.7, 64 x 1280 3.8 / 3.1,
// 800 x 1280 5.6 / 5.3, 1500 x 1280 7.6 / 7.9, without the add 3000 x 1280 7.3 / 8.2.
bool norm_by_waves(int rows, int vecs, int32_t dtype) { return vecs <= 128 || rows >= (dtype == SKV_F32 ? 1024 : 512); }

template <int DT>
void launch_add_norm_rows(const AddNormParams& p, int rows, int vecs, hipStream_t s) {
  const dim3 grid((uint32_t)cdiv(rows, 4)), block(256);
  switch (cdiv(vecs, 64)) {
    case 1: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 1>), grid, block, 0, s, p, rows); break;
    case 2: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 2>), grid, block, 0, s, p, rows); break;
    case 3: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 3>), grid, block, 0, s, p, rows); break;
    case 4: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 4>), grid, block, 0, s, p, rows); break;
    case 5: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 5>), grid, block, 0, s, p, rows); break;
    default: hipLaunchKernelGGL((add_norm_rows_kernel<DT, 8>), grid, block, 0, s, p, rows); break;
  }
}

void launch_add_norm(const AddNormParams& p, int rows, int32_t dtype, hipStream_t s) {
  const int vecs = p.quads / (dtype == SKV_F32 ? 1 : 2);
  if (!p.part && norm_by_waves(rows, vecs, dtype)) {
    switch (dtype) {
      case SKV_F32: launch_add_norm_rows<SKV_F32>(p, rows, vecs, s); break;
      case SKV_F16: launch_add_norm_rows<SKV_F16>(p, rows, vecs, s); break;
      default: launch_add_norm_rows<SKV_BF16>(p, rows, vecs, s); break;
    }
    return;
  }
  const dim3 grid((uint32_t)rows), block((uint32_t)cdiv(p.quads, 64) * 64);
  switch (dtype) {
    case SKV_F32: hipLaunchKernelGGL((add_norm_kernel<SKV_F32>), grid, block, 0, s, p); break;
    case SKV_F16: hipLaunchKernelGGL((add_norm_kernel<SKV_F16>), grid, block, 0, s, p); break;
    default: hipLaunchKernelGGL((add_norm_kernel<SKV_BF16>), grid, block, 0, s, p); break;
  }
}

// Largest batch: a decode batch of up to 128 rows always (at k = 1280, n = 1280 / 3840 / 5120 bf16: 64 rows 4.7 /
// 5.9 / 7.7 us against 8.8 / 9.3 / 9.7 through hipBLASLt, 128 rows 5.5 / 7.6 / 11.5 against 8.3 / 14.6 / 14.8), and
// up to 512 rows (a prompt batch) while m * n stays under the library's crossover: 16-bit 2^20 (512 x 1280 10.6
// against 13.1 us, 512 x 2304 10.4 / 10.4, 384 x 3840 18.5 / 14.8), fp32 2^18 (160 x 1536 4.9 / 7.4, 256 x 1536
// 7.5 / 7.3). A split contraction stays at 128 (k = 5120, n = 1280: 128 rows 9.6 / 15.4, 160 rows 15.6 / 15.2).
constexpr int kDecodeRows = 128;
constexpr int kMaxRows = 512;
constexpr int kMinChunks = 4;             // 512-byte rows: a chunk for each wave
constexpr uint32_t kMaxChunks = 32;       // 4 KiB rows: 8 waves x 4, and every tile's registers
// Rows of up to 6 KiB stay in one workgroup too (8 waves x 6, tiles of at most 32 x 32), so that the residual goes into
// the epilogue and the launch that sums partials (2.3-2.9 us) falls away: 768 x 3072 bf16, 64 rows, with the residual
// 5.0 us; a 12-layer step of that shape 1099 -> 1089 us, a 384-wide fp32 layer 42.1 -> 41.4 (with norm16's fma).
constexpr uint32_t kMaxSplitChunks = 48;

struct ProjShape {
  uint32_t m, n, kbytes, chunks, splits, split_chunks;
  int mi, ni, waves, rounds;
  bool one_each;  // at most one workgroup per compute unit
};

int proj_splits(int64_t chunks) { return chunks <= kMaxSplitChunks ? 1 : (int)cdiv(chunks, kMaxChunks); }

// The contraction's split over workgroups, waves and rounds depends on k and the dtype alone, so a row's
// bits do not depend on the batch it is in.
void pick_shape(ProjShape& p, int32_t m, int32_t n, int32_t kbytes) {
  p.m = (uint32_t)m, p.n = (uint32_t)n, p.kbytes = (uint32_t)kbytes;
  p.chunks = (uint32_t)cdiv(kbytes, kChunkBytes);
  p.splits = (uint32_t)proj_splits(p.chunks);
  p.split_chunks = (uint32_t)cdiv(p.chunks, p.splits);
  p.waves = p.split_chunks <= 12 ? 4 : 8;
  p.rounds = (int)cdiv(p.split_chunks, p.waves);
  // The smallest tile that leaves at most one workgroup per compute unit: fewer idle units than a larger
  // one, and a second workgroup on some units costs a whole round (64 rows, k = 1280: n = 1280 32 x 16 4.6 us, 16 x 16
  // (320 workgroups) 4.9; n = 3840 32 x 32 5.8, 32 x 16 6.9, 64 x 32 7.3; n = 5120 64 x 32 7.5, 32 x 32 8.7).
  // Past 64 x 32 tiles for every unit, 32 x 32 again: two resident per unit (128 rows, n = 5120: 11.2 against 13.1).
  const int tiles[4][2] = {{1, 1}, {2, 1}, {2, 2}, {4, 2}};
  const int64_t cus = compute_units();
  p.mi = p.ni = 2;
  p.one_each = false;
  for (const auto& t : tiles) {
    if (t[0] > 1 && 8 * t[0] >= m) continue;  // half the tile's rows would be empty
    if (t[0] > 2 && p.split_chunks > kMaxChunks) continue;
    if (cdiv(m, 16 * t[0]) * cdiv(n, 16 * t[1]) * p.splits <= cus) {
      p.mi = t[0], p.ni = t[1];
      p.one_each = true;
      break;
    }
  }
}

template <int DT, int MI, int NI, bool NORM>
void launch_tile(const ProjShape& s, const char* x, const char* w, uint32_t ldx, uint32_t ldw, uint32_t xb,
                 uint32_t wb, const ProjNorm& q, const ProjEpilogue& e, hipStream_t st) {
  const dim3 grid(8, (uint32_t)cdiv(s.m, 16 * MI), (uint32_t)(cdiv(s.n, 8 * 16 * NI) * s.splits));
#define SKV_PROJ(W, R)                                                                                            \
  hipLaunchKernelGGL((proj_kernel<DT, MI, NI, W, R, NORM>), grid, dim3(64 * W), 0, st, x, w, ldx, ldw, xb, wb, s.m, \
                     s.n, s.kbytes, s.split_chunks, s.splits, q, e)
  switch (s.waves * 4 + s.rounds) {
    case 17: SKV_PROJ(4, 1); break;
    case 18: SKV_PROJ(4, 2); break;
    case 19: SKV_PROJ(4, 3); break;
    case 34: SKV_PROJ(8, 2); break;
    case 35: SKV_PROJ(8, 3); break;
    case 36: SKV_PROJ(8, 4); break;
    default:
      if constexpr (MI <= 2 && !NORM) {
        if (s.rounds == 5)
          SKV_PROJ(8, 5);
        else
          SKV_PROJ(8, 6);
      }
  }
#undef SKV_PROJ
}

template <int DT, bool NORM>
void launch_proj(const ProjShape& s, const char* x, const char* w, uint32_t ldx, uint32_t ldw, uint32_t xb,
                 uint32_t wb, const ProjNorm& q, const ProjEpilogue& e, hipStream_t st) {
  switch (s.mi * 4 + s.ni) {
    case 5: launch_tile<DT, 1, 1, NORM>(s, x, w, ldx, ldw, xb, wb, q, e, st); break;
    case 9: launch_tile<DT, 2, 1, NORM>(s, x, w, ldx, ldw, xb, wb, q, e, st); break;
    case 10: launch_tile<DT, 2, 2, NORM>(s, x, w, ldx, ldw, xb, wb, q, e, st); break;
    default:
      if constexpr (!NORM) launch_tile<DT, 4, 2, NORM>(s, x, w, ldx, ldw, xb, wb, q, e, st);
  }
}

// Checks shared by the two projection entry points; fills the shape and the byte ranges.
int prepare_proj(const char* who, ProjShape& s, const void* x, int64_t ldx, const void* w, int64_t ldw, int32_t m,
                 int32_t n, int32_t k, int32_t dtype, uint32_t& xb, uint32_t& wb) {
  const int eb = elt_bytes(dtype);
  if (eb == 0) return fail(SKV_EDTYPE, "%s: unknown dtype %d", who, dtype);
  if (m < 0 || n <= 0 || k <= 0 || ldx < k || ldw < k)
    return fail(SKV_EINVAL, "%s: bad sizes m=%d n=%d k=%d ldx=%lld ldw=%lld", who, m, n, k, (long long)ldx,
                (long long)ldw);
  const int64_t kb = (int64_t)k * eb;
  const int64_t xr = m > 0 ? (int64_t)(m - 1) * ldx * eb + kb : kb, wr = (int64_t)(n - 1) * ldw * eb + kb;
  const int64_t chunks = cdiv(kb, kChunkBytes);
  const bool batch_ok = m <= kDecodeRows || (m <= kMaxRows && chunks <= kMaxChunks &&
                                             (int64_t)m * n <= (int64_t)1 << (eb == 4 ? 18 : 20));
  if (!batch_ok || n % 4 || kb % 16 || kb < kMinChunks * kChunkBytes || ldx * eb % 16 || ldw * eb % 16 ||
      xr > 0x7fffffff || wr > 0x7fffffff || kb > (int64_t)kMaxSplitChunks * kChunkBytes * 64)
    return fail(SKV_EUNSUPPORTED, "%s: m=%d n=%d k=%d ldx=%lld ldw=%lld dtype=%d is not a decode projection", who, m, n,
                k, (long long)ldx, (long long)ldw, dtype);
  xb = (uint32_t)xr, wb = (uint32_t)wr;
  pick_shape(s, m, n, (int32_t)kb);
  return SKV_OK;
}

int run_proj(const char* who, const ProjShape& s, const void* x, int64_t ldx, const void* w, int64_t ldw, int32_t dtype,
             uint32_t xb, uint32_t wb, const ProjNorm& q, const ProjEpilogue& e, hipStream_t st) {
  const uint32_t eb = (uint32_t)elt_bytes(dtype);
  const uint32_t lx = s.m > 1 ? (uint32_t)ldx * eb : s.kbytes, lw = s.n > 1 ? (uint32_t)ldw * eb : s.kbytes;
  const char *xp = (const char*)x, *wp = (const char*)w;
#define SKV_PROJ_DT(DT)                                                \
  if (q.gamma)                                                         \
    launch_proj<DT, true>(s, xp, wp, lx, lw, xb, wb, q, e, st);        \
  else                                                                 \
    launch_proj<DT, false>(s, xp, wp, lx, lw, xb, wb, q, e, st);
  switch (dtype) {
    case SKV_F32: SKV_PROJ_DT(SKV_F32) break;
    case SKV_F16: SKV_PROJ_DT(SKV_F16) break;
    default: SKV_PROJ_DT(SKV_BF16) break;
  }
#undef SKV_PROJ_DT
  return check_launch(who);
}

}  // namespace

int32_t skv_decode_linear_splits(int32_t k, int32_t dtype) {
  const int eb = elt_bytes(dtype);
  return eb == 0 || k <= 0 ? 0 : proj_splits(cdiv((int64_t)k * eb, kChunkBytes));
}

int skv_decode_linear(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, int32_t act, void* y,
                      int64_t ldy, int32_t m, int32_t n, int32_t k, int32_t dtype, void* stream) {
  return skv_decode_linear_fused(x, ldx, nullptr, nullptr, nullptr, 0.f, w, ldw, bias, act, nullptr, 0, y, ldy, nullptr,
                                 m, n, k, dtype, stream);
}

int skv_decode_linear_fused(const void* x, int64_t ldx, const float* x_stats, const void* gamma, const void* beta,
                            float eps, const void* w, int64_t ldw, const void* bias, int32_t act, const void* res,
                            int64_t ldr, void* y, int64_t ldy, float* y_stats, int32_t m, int32_t n, int32_t k,
                            int32_t dtype, void* stream) {
  const char* who = "skv_decode_linear";
  ProjShape s;
  uint32_t xb = 0, wb = 0;
  const int rc = prepare_proj(who, s, x, ldx, w, ldw, m, n, k, dtype, xb, wb);
  if (rc != SKV_OK) return rc;
  if (ldy < n || (res && ldr < n) || (act != 0 && act != SKV_ACT_GELU))
    return fail(SKV_EINVAL, "%s: bad ldy=%lld, ldr=%lld (n=%d) or act=%d", who, (long long)ldy, (long long)ldr, n, act);
  if (s.splits > 1 || ldy % 4 || (res && ldr % 4))
    return fail(SKV_EUNSUPPORTED, "%s: k=%d (dtype %d) is split over %u workgroups; ldy=%lld ldr=%lld", who, k, dtype,
                s.splits, (long long)ldy, (long long)ldr);
  const bool norm = x_stats || gamma || beta;
  if (norm && !(eps >= 0.f)) return fail(SKV_EINVAL, "%s: eps must be >= 0", who);
  // Every workgroup normalises its rows again, so that pays where a unit has one workgroup of at most 32 rows (us, a
  // LayerNorm launch and the plain projection / normalising; bf16): k = 1280, 64 rows, n = 3840 2.9 + 5.6 / 7.5, 1280
  // 2.9 + 4.1 / 5.8; 128 rows, n = 1280 3.0 + 5.0 / 6.6; k = 768, 64 rows, n = 2304 2.6 + 4.2 / 5.6; k = 256 2.2 + 2.3 /
  // 2.8. With 64-row tiles or more workgroups than units it does not: 64 rows, n = 5120 2.9 + 7.8 / 11.0, 128 rows
  // 3.0 + 11.0 / 18.6.
  const bool norm_ok = k % 16 == 0 && m <= kDecodeRows && s.one_each && s.mi <= 2 && s.chunks <= kMaxChunks;
  if ((norm && !norm_ok) || (y_stats && n % 16))
    return fail(SKV_EUNSUPPORTED, "%s: m=%d n=%d k=%d with row statistics", who, m, n, k);
  if (m == 0) return SKV_OK;
  if (!x || !w || !y || (norm && (!x_stats || !gamma || !beta)))
    return fail(SKV_EINVAL, "%s: null pointer argument", who);
  const uintptr_t quad = 4 * (uintptr_t)elt_bytes(dtype) - 1;
  if (!aligned16(x) || !aligned16(w) || ((uintptr_t)y & quad) || ((uintptr_t)res & quad) || ((uintptr_t)bias & quad) ||
      !aligned16(gamma) ||
      !aligned16(beta) || ((uintptr_t)x_stats & 7) || ((uintptr_t)y_stats & 7))
    return fail(SKV_EUNSUPPORTED, "%s: x, w, gamma and beta must be 16-byte aligned, y, res and bias to four elements",
                who);
  const ProjNorm q{gamma, beta, (const float2*)x_stats, eps, 1.f / (float)k};
  const ProjEpilogue e{bias, (char*)y, nullptr, ldy, act, (const char*)res, ldr, (float2*)y_stats};
  return run_proj(who, s, x, ldx, w, ldw, dtype, xb, wb, q, e, (hipStream_t)stream);
}

int skv_decode_linear_partials(const void* x, int64_t ldx, const void* w, int64_t ldw, float* part, int64_t part_floats,
                               int32_t m, int32_t n, int32_t k, int32_t dtype, void* stream) {
  ProjShape s;
  uint32_t xb = 0, wb = 0;
  const int rc = prepare_proj("skv_decode_linear_partials", s, x, ldx, w, ldw, m, n, k, dtype, xb, wb);
  if (rc != SKV_OK) return rc;
  if (m == 0) return SKV_OK;
  if (!x || !w || !part) return fail(SKV_EINVAL, "skv_decode_linear_partials: null pointer argument");
  if (!aligned16(x) || !aligned16(w) || !aligned16(part))
    return fail(SKV_EUNSUPPORTED, "skv_decode_linear_partials: x, w and part must be 16-byte aligned");
  if (part_floats < (int64_t)s.splits * m * n)
    return fail(SKV_EWORKSPACE, "skv_decode_linear_partials: part needs %lld floats, got %lld",
                (long long)s.splits * m * n, (long long)part_floats);
  const ProjEpilogue e{nullptr, nullptr, part, 0, 0, nullptr, 0, nullptr};
  return run_proj("skv_decode_linear_partials", s, x, ldx, w, ldw, dtype, xb, wb, ProjNorm{}, e, (hipStream_t)stream);
}

int skv_add_layernorm(const void* x, int64_t ldx, const void* y, int64_t ldy, const void* gamma, const void* beta,
                      float eps, void* sum, int64_t lds, void* norm, int64_t ldn, int32_t rows, int32_t hidden,
                      int32_t dtype, void* stream) {
  const int eb = elt_bytes(dtype);
  if (eb == 0) return fail(SKV_EDTYPE, "skv_add_layernorm: unknown dtype %d", dtype);
  const int epl = 16 / eb;
  if (rows < 0 || hidden <= 0 || hidden % epl || hidden > kMaxNormVecs * epl)
    return fail(SKV_EINVAL, "skv_add_layernorm: hidden %d must be a multiple of %d and at most %d (rows=%d)", hidden,
                epl, kMaxNormVecs * epl, rows);
  if (rows == 0) return SKV_OK;
  if (!x || !gamma || !beta || !norm) return fail(SKV_EINVAL, "skv_add_layernorm: null pointer argument");
  if (!aligned16(x) || !aligned16(gamma) || !aligned16(beta) || !aligned16(norm) || (y && !aligned16(y)) ||
      (sum && !aligned16(sum)) || ldx % epl || ldy % epl || lds % epl || ldn % epl)
    return fail(SKV_EALIGN, "skv_add_layernorm: rows must be 16-byte aligned");
  if (!(eps >= 0.f)) return fail(SKV_EINVAL, "skv_add_layernorm: eps must be >= 0");
  AddNormParams p{};
  p.x = (const char*)x;
  p.y = (const char*)y;
  p.gamma = (const char*)gamma;
  p.beta = (const char*)beta;
  p.sum = y ? (char*)sum : nullptr;
  p.norm = (char*)norm;
  p.ldx = ldx;
  p.ldy = ldy;
  p.lds = lds;
  p.ldn = ldn;
  p.quads = hidden / 4;
  p.eps = eps;
  p.inv_n = 1.f / (float)hidden;
  launch_add_norm(p, rows, dtype, (hipStream_t)stream);
  return check_launch("skv_add_layernorm");
}

int skv_reduce_add_layernorm(const float* part, int32_t splits, const void* bias, const void* x, int64_t ldx,
                             const void* gamma, const void* beta, float eps, void* sum, int64_t lds, void* norm,
                             int64_t ldn, int32_t rows, int32_t hidden, int32_t dtype, void* stream) {
  const int eb = elt_bytes(dtype);
  if (eb == 0) return fail(SKV_EDTYPE, "skv_reduce_add_layernorm: unknown dtype %d", dtype);
  const int epl = 16 / eb;
  if (rows < 0 || splits <= 0 || hidden <= 0 || hidden % epl || hidden > kMaxNormVecs * epl)
    return fail(SKV_EINVAL, "skv_reduce_add_layernorm: bad sizes rows=%d splits=%d hidden=%d (a multiple of %d, at most %d)",
                rows, splits, hidden, epl, kMaxNormVecs * epl);
  if (rows == 0) return SKV_OK;
  if (!part || !sum || (gamma == nullptr) != (norm == nullptr) || (gamma == nullptr) != (beta == nullptr))
    return fail(SKV_EINVAL, "skv_reduce_add_layernorm: null pointer argument");
  if (!aligned16(part) || !aligned16(sum) || (bias && !aligned16(bias)) || (x && !aligned16(x)) || lds % epl ||
      (x && ldx % epl) || (norm && (!aligned16(norm) || !aligned16(gamma) || !aligned16(beta) || ldn % epl)))
    return fail(SKV_EALIGN, "skv_reduce_add_layernorm: rows must be 16-byte aligned");
  if (!(eps >= 0.f)) return fail(SKV_EINVAL, "skv_reduce_add_layernorm: eps must be >= 0");
  AddNormParams p{};
  p.x = (const char*)x;
  p.part = part;
  p.bias = (const char*)bias;
  p.gamma = (const char*)gamma;
  p.beta = (const char*)beta;
  p.sum = (char*)sum;
  p.norm = (char*)norm;
  p.ldx = ldx;
  p.lds = lds;
  p.ldn = ldn;
  p.part_stride = (int64_t)rows * hidden;
  p.quads = hidden / 4;
  p.splits = splits;
  p.eps = eps;
  p.inv_n = 1.f / (float)hidden;
  launch_add_norm(p, rows, dtype, (hipStream_t)stream);
  return check_launch("skv_reduce_add_layernorm");
}
