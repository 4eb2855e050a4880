// quantize.hip -- the step before the layer: bf16 hidden states -> e4m3 rows
// with one fp32 scale per 128-column block, stored transposed ([56, T]), i.e.
// exactly the `hidden_states` / `hidden_states_scale` pair the layer consumes
// (layout: moe.py:32-33; the reference repository holds no quantiser, so the
// convention is the DeepSeek-V3 one this build's generator also uses):
//   scale = absmax(block) / 448          (1 for an all-zero block)
//   q     = e4m3(x / scale), round to nearest even, saturating to +-448
// NaN elements do not enter the absmax and encode as NaN.
//
// Design (gfx950): HBM-bound (reads 2 B and writes 1 B per element), so the
// arithmetic per element has to stay under the memory time.  Up to T = 2048
// one workgroup per token row, wave p quantising pass p (7 waves per row, so
// that enough loads are in flight at small T).  From T = 5120 half a row per
// wave with nontemporal loads (quantize_hidden_stream_kernel).  Between, one wave
// per token row, four rows per workgroup (T/4 workgroups: 1024 at T = 4096).  A
// wave issues all 14 row loads (16 B per lane each) before any arithmetic, so
// a token has its whole 14 KB row in flight at once; each of the 7 passes
// then covers 1024 columns = 8 scale blocks, 8 lanes per block and 16
// contiguous elements per lane.  A block's absmax is an 8-lane DPP max of
// bf16 magnitudes (compared as integers); the scales go through LDS so that
// each transposed scale row is written as 4 contiguous tokens.
//
// Fast path (every pass whose blocks all have 2^-96 <= absmax < inf or
// absmax = 0, and no NaN): with s = absmax / 448 and r = 1 / s (both
// correctly rounded),
//   q = x * r;  q' = fma(fma(-s, q, x), r, q);  code = e4m3_rne(|q'|) | sign(x)
// and the rounding to e4m3 is v_cvt_pk_fp8_f32.  Both steps were checked
// exhaustively against the correctly rounded x / s followed by the software
// RNE conversion below: q' gives the same e4m3 code for every bf16 pair
// |x| <= absmax in that range (about 1.07e9 pairs), and the hardware
// conversion equals the software one for every fp32 with |y| < 464 (|q'| is
// at most 448 * (1 + 2^-22)).  Passes with a NaN, an infinity or a tiny
// absmax in any of the wave's blocks take the exact path (IEEE division and
// the software conversion) instead; that branch is wave-uniform.
#include "kernels.hpp"

namespace moe {
namespace {

constexpr int kQTokens = 4;   // tokens (waves) per workgroup
constexpr int kQThreads = kQTokens * kWave;
constexpr int kQLaneCols = 16;                 // elements per lane per pass
constexpr int kQPass = kWave * kQLaneCols;     // 1024 columns per wave pass
constexpr int kQPasses = kH / kQPass;          // 7
constexpr int kQLanesPerBlk = kBlk / kQLaneCols;  // 8
constexpr uint32_t kQTinyBf16 = 0x0F80u;       // bf16 bits of 2^-96

// fp32 -> OCP e4m3fn, round to nearest even, saturating finite values and
// infinities to +-448; NaN -> 0x7F (sign kept).  Branch-free:
//   normal range (|x| >= 2^-6): adding 2^19 - 1 + (bit 20) to the magnitude's
//     bits rounds its 23-bit mantissa to 3 bits, nearest even, with the carry
//     running into the exponent; the code is then (bits >> 20) - (120 << 3)
//     (exponent rebias 127 -> 7), clamped to 0x7E (448);
//   subnormal range: the code is |x| / 2^-9 rounded to nearest even (0..8,
//     8 being the smallest normal, 0x08).
__device__ __forceinline__ uint32_t f32_to_e4m3_satfinite(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t sign = (u >> 24) & 0x80u;
  const uint32_t a = u & 0x7FFFFFFFu;
  const uint32_t normal = min(((a + 0x7FFFFu + ((a >> 20) & 1u)) >> 20) - 960u, 0x7Eu);
  const uint32_t sub = (uint32_t)rintf(__uint_as_float(a) * 512.0f);
  uint32_t code = a < 0x3C800000u ? sub : normal;
  code = a > 0x7F800000u ? 0x7Fu : code;
  return sign | code;
}

__device__ __forceinline__ float bf16_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __uint_as_float(u & 0xFFFF0000u); }

// Largest bf16 magnitude (as bits, 0..0x7FFF) of one lane's 2N elements; NaN
// patterns (> 0x7F80) order above every number, so a NaN shows as > 0x7F80.
template <int N>
__device__ __forceinline__ uint32_t lane_absmax_bits(const uint32_t (&e)[N]) {
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    lo = max(lo, e[i] & 0x7FFFu);
    hi = max(hi, (e[i] >> 16) & 0x7FFFu);
  }
  return max(lo, hi);
}

// The same with NaN elements left out (the exact path's absmax).
template <int N>
__device__ __forceinline__ uint32_t lane_absmax_bits_nonnan(const uint32_t (&e)[N]) {
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uint32_t lo = e[i] & 0x7FFFu, hi = (e[i] >> 16) & 0x7FFFu;
    m = max(m, lo > 0x7F80u ? 0u : lo);
    m = max(m, hi > 0x7F80u ? 0u : hi);
  }
  return m;
}

// Maximum over the lanes of a scale block (8 lanes of 16 elements or 16 lanes
// of 8), in every lane of it.
template <int LANES>
__device__ __forceinline__ uint32_t block_max_u32(uint32_t k) {
  static_assert(LANES == 8 || LANES == 16, "DPP rows");
  if (LANES == 16) return row16_max_u32(k);
  k = max(k, dpp_u32<kDppQuad1032, 0xF>(k));
  k = max(k, dpp_u32<kDppQuad2301, 0xF>(k));
  return max(k, dpp_u32<kDppRowHalfMirror, 0xF>(k));
}

// Four elements (signs from the inputs) -> four e4m3 bytes, fast path.
__device__ __forceinline__ uint32_t fast_pack4(float x0, float x1, float x2, float x3, float s, float r) {
  const float x[4] = {x0, x1, x2, x3};
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float q = x[i] * r;
    const float q2 = fmaf(fmaf(-s, q, x[i]), r, q);
    y[i] = __uint_as_float((__float_as_uint(q2) & 0x7FFFFFFFu) | (__float_as_uint(x[i]) & 0x80000000u));
  }
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], lo, true);
}

// The same, exact path: IEEE division and the software conversion.
__device__ __forceinline__ uint32_t exact_pack4(float x0, float x1, float x2, float x3, float s) {
  return f32_to_e4m3_satfinite(x0 / s) | (f32_to_e4m3_satfinite(x1 / s) << 8) |
         (f32_to_e4m3_satfinite(x2 / s) << 16) | (f32_to_e4m3_satfinite(x3 / s) << 24);
}

// One pass of a wave: 2N elements per lane, kBlk / 2N lanes per scale block;
// the e4m3 codes and this lane's block scale (wave-uniform fast/exact branch).
template <int N>
__device__ __forceinline__ void quantize_pass(const uint32_t (&e)[N], uint32_t (&out)[N / 2], float& s) {
  constexpr int kLanes = kBlk / (2 * N);
  const uint32_t m = block_max_u32<kLanes>(lane_absmax_bits(e));
  const bool odd = m > 0x7F7Fu || (m != 0u && m < kQTinyBf16);
  if (__ballot(odd) == 0) {
    const float amax = __uint_as_float(m << 16);
    s = amax > 0.0f ? amax / 448.0f : 1.0f;
    const float r = 1.0f / s;
#pragma unroll
    for (int i = 0; i < N / 2; ++i)
      out[i] = fast_pack4(bf16_lo(e[2 * i]), bf16_hi(e[2 * i]), bf16_lo(e[2 * i + 1]), bf16_hi(e[2 * i + 1]), s, r);
  } else {
    const float amax = __uint_as_float(block_max_u32<kLanes>(lane_absmax_bits_nonnan(e)) << 16);
    s = amax > 0.0f ? amax / 448.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < N / 2; ++i)
      out[i] = exact_pack4(bf16_lo(e[2 * i]), bf16_hi(e[2 * i]), bf16_lo(e[2 * i + 1]), bf16_hi(e[2 * i + 1]), s);
  }
}

// 16 elements of one lane (two 16-byte loads), 8 lanes per scale block.
__device__ __forceinline__ void quantize_pass16(const uint4& a, const uint4& b, uint4& out, float& s) {
  const uint32_t e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t o[4];
  quantize_pass(e, o, s);
  out = uint4{o[0], o[1], o[2], o[3]};
}

__global__ void __launch_bounds__(kQThreads)
quantize_hidden_kernel(const uint16_t* __restrict__ x, int T, uint8_t* __restrict__ q,
                       float* __restrict__ scale) {
  __shared__ float sc[kNHBlk][kQTokens];
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int t = blockIdx.x * kQTokens + w;
  if (t < T) {
    const uint16_t* row = x + (size_t)t * kH + lane * kQLaneCols;
    uint8_t* qrow = q + (size_t)t * kH + lane * kQLaneCols;
    // the whole row (14 x 16 B per lane) is in flight before any arithmetic
    uint4 raw[2 * kQPasses];
#pragma unroll
    for (int c = 0; c < kQPasses; ++c) {
      raw[2 * c] = *(const uint4*)(row + c * kQPass);
      raw[2 * c + 1] = *(const uint4*)(row + c * kQPass + 8);
    }
#pragma unroll
    for (int c = 0; c < kQPasses; ++c) {
      uint4 out;
      float s;
      quantize_pass16(raw[2 * c], raw[2 * c + 1], out, s);
      *(uint4*)(qrow + c * kQPass) = out;
      if ((lane & (kQLanesPerBlk - 1)) == 0) sc[c * (kQPass / kBlk) + lane / kQLanesPerBlk][w] = s;
    }
  }
  __syncthreads();
  // scale[b][t0 .. t0+kQTokens-1]: contiguous floats per block row
  const int t0 = blockIdx.x * kQTokens;
  for (int i = threadIdx.x; i < kNHBlk * kQTokens; i += kQThreads) {
    const int b = i / kQTokens, k = i % kQTokens;
    if (t0 + k < T) scale[(size_t)b * T + t0 + k] = sc[b][k];
  }
}

// Small T (latency-bound with one wave per row): one workgroup per token
// row, wave p quantises pass p (columns 1024p ..) and writes its 8 block
// scales directly.  Same arithmetic as above, so the same bits.
constexpr int kQSmallMaxTokens = 2048;

__global__ void __launch_bounds__(kQPasses * kWave)
quantize_hidden_rows_kernel(const uint16_t* __restrict__ x, int T, uint8_t* __restrict__ q,
                            float* __restrict__ scale) {
  const int t = blockIdx.x;
  const int c = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const uint16_t* src = x + (size_t)t * kH + c * kQPass + lane * kQLaneCols;
  const uint4 a = *(const uint4*)src, b = *(const uint4*)(src + 8);
  uint4 out;
  float s;
  quantize_pass16(a, b, out, s);
  *(uint4*)(q + (size_t)t * kH + c * kQPass + lane * kQLaneCols) = out;
  if ((lane & (kQLanesPerBlk - 1)) == 0) scale[(size_t)(c * (kQPass / kBlk) + lane / kQLanesPerBlk) * T + t] = s;
}

// Large T: one wave per half token row, 7 passes of 512 columns.  A lane takes 8
// elements a pass (16 lanes per scale block), so each load instruction covers
// 1 KB of contiguous bytes (16 elements per lane would touch every line
// twice), and the rows, read once, are loaded nontemporally.  Same arithmetic,
// same bits.  It fetches what the rows hold (T = 8192 117.6 of 117.4 MB).  us, one
// wave per row with temporal loads -> this, where rows and outputs of the last
// calls push each other out of the caches: T = 14107 58.5 -> 53.6, 10000 42.5 ->
// 37.7 (5.8 TB/s), 8192 36.1 -> 31.5, 7000 30.9 -> 27.5, 5632 25.4 -> 23.5, 5120
// 22.2 -> 22.0; below it the nontemporal loads lose (4096 17.4 -> 18.4).  Rows
// that the step before has just written, into an output that every call
// reuses, are partly in the caches, where nontemporal loads gain less or lose:
// 5120 22.6 -> 25.2, 7000 29.4 -> 31.0, 8192 33.5 -> 34.6, 10000 40.4 -> 41.0,
// 14107 60.0 -> 55.6 (one kernel timed as both sides there differs by 2 %).  This
// layout with temporal loads keeps the old kernel's times in both (8192 38.2 and
// 33.3).  Nontemporal stores gained another 0-4 % but would send the layer's
// input past the caches.
constexpr int kQStreamMinTokens = 5120;
constexpr int kQHalf = kH / 2;                     // columns per wave
constexpr int kQStreamPass = kWave * 8;            // 512 columns
constexpr int kQStreamPasses = kQHalf / kQStreamPass;  // 7
static_assert(kQStreamPasses * kQStreamPass == kQHalf && 16 * 8 == kBlk, "whole passes, 16 lanes per scale block");

__global__ void __launch_bounds__(kWave)
quantize_hidden_stream_kernel(const uint16_t* __restrict__ x, int T, uint8_t* __restrict__ q,
                              float* __restrict__ scale) {
  const int t = blockIdx.x >> 1, c0 = (blockIdx.x & 1) * kQHalf;
  const int lane = threadIdx.x;
  const uint16_t* src = x + (size_t)t * kH + c0 + lane * 8;
  uint8_t* dst = q + (size_t)t * kH + c0 + lane * 8;
  v4i raw[kQStreamPasses];
#pragma unroll
  for (int c = 0; c < kQStreamPasses; ++c) raw[c] = __builtin_nontemporal_load((const v4i*)(src + c * kQStreamPass));
#pragma unroll
  for (int c = 0; c < kQStreamPasses; ++c) {
    const uint32_t e[4] = {(uint32_t)raw[c][0], (uint32_t)raw[c][1], (uint32_t)raw[c][2], (uint32_t)raw[c][3]};
    uint32_t out[2];
    float s;
    quantize_pass(e, out, s);
    *(uint2*)(dst + c * kQStreamPass) = uint2{out[0], out[1]};
    if ((lane & 15) == 0) scale[(size_t)((c0 + c * kQStreamPass) / kBlk + (lane >> 4)) * T + t] = s;
  }
}

}  // namespace

hipError_t launch_quantize_hidden(const uint16_t* x, int T, uint8_t* q, float* scale, hipStream_t stream) {
  if (T <= kQSmallMaxTokens) {
    hipLaunchKernelGGL(quantize_hidden_rows_kernel, dim3(T), dim3(kQPasses * kWave), 0, stream, x, T, q, scale);
    return hipGetLastError();
  }
  if (T >= kQStreamMinTokens) {
    hipLaunchKernelGGL(quantize_hidden_stream_kernel, dim3(2 * T), dim3(kWave), 0, stream, x, T, q, scale);
    return hipGetLastError();
  }
  const int blocks = (T + kQTokens - 1) / kQTokens;
  hipLaunchKernelGGL(quantize_hidden_kernel, dim3(blocks), dim3(kQThreads), 0, stream, x, T, q, scale);
  return hipGetLastError();
}

}  // namespace moe
