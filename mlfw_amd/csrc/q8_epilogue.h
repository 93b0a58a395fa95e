// q8_epilogue.h -- what the GEMM kernels share: the epilogue of one output
// element, the LDS chunk swizzle and the workgroup -> tile order.
#pragma once

#include "q8_device.h"
#include "q8_internal.h"

namespace q8 {

// ------------------------------------------------------------------ epilogue
// y = fround(acc * sv) for an f32 scale sv.  When acc is exactly an f32
// (|acc| <= 2^24) the f32 multiply rounds the exact product once, which is
// what Math.fround((+acc) * sv) does in f64 (a binary32 product of two
// binary32 values is exact in binary64); otherwise the f64 form is used.
__device__ __forceinline__ float mul_acc_f32scale(int acc, float sv) {
  if ((unsigned)(acc + (1 << 24)) <= (2u << 24)) return (float)acc * sv;
  return (float)((double)acc * (double)sv);
}

__device__ __forceinline__ float epi_finish(float y, int64_t n, const GemmEpi& e) {
  if (e.bias) y = y + e.bias[n];   // binary32 add == Math.fround(f64 add) for f32 operands
  if (e.act == 1) y = relu_js(y);
  else if (e.act == 2) y = silu_js(y);
  return y;
}

__device__ __forceinline__ float epi_value(int acc, int64_t m, int64_t n, const GemmEpi& e) {
  float y;
  if (e.mode == 0) {
    y = (float)((double)acc * e.s_out);
  } else {
    const float sv = (float)(e.sA[m * e.sA_stride] * e.sB[n * e.sB_stride]);
    y = mul_acc_f32scale(acc, sv);
  }
  return epi_finish(y, n, e);
}

// The compiled `quantize` (quant_math.ts:16-27) of an epilogue value with the
// next layer's static scale: q = (min(max(Math.round(fround(y / s)), -128), 127) | 0).
__device__ __forceinline__ int requant(float y, const GemmEpi& e) {
  return e.q_fast ? quant_sym_fast(y, e.rq32, e.s_q) : quant_exact(y, e.s_q, 0.0, -128, 127);
}

// Final store of one output element of the GEMV / generic kernels.
__device__ __forceinline__ void store_out(void* out, int64_t idx, int acc, int64_t m, int64_t n,
                                          const GemmEpi& e) {
  if (e.col_blk > 0) idx = (n / e.col_blk) * e.blk_stride + m * e.ld_out + n % e.col_blk;
  if (e.out_i32) static_cast<int32_t*>(out)[idx] = acc;
  else if (e.out_q8) static_cast<int8_t*>(out)[idx] = (int8_t)requant(epi_value(acc, m, n, e), e);
  else static_cast<float*>(out)[idx] = epi_value(acc, m, n, e);
}

// ------------------------------------------------------------------ tiles
// Chunk position of logical 16-byte chunk c of LDS row r (128-byte rows): c ^ swz(r).
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// Workgroup id -> (tile row, tile col).  Dispatch places consecutive ids on
// consecutive XCDs (id % 8); the remap gives each XCD a contiguous run of
// the grouped tile order below.
__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int G = tiles_m * tiles_n;
  const int xcd = bid & 7, k = bid >> 3;
  const int per = G >> 3, rem = G & 7;
  const int id = xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
  constexpr int GROUP = 4;
  const int group = id / (GROUP * tiles_n);
  const int first = group * GROUP;
  const int gm = min(tiles_m - first, GROUP);
  const int in = id - group * GROUP * tiles_n;
  tm = first + in % gm;
  tn = in / gm;
}

// ------------------------------------------------------------------ conv frames
// Implicit conv B operand (GemmEpi::ConvB): frame offset of tap t relative
// to tap 0, in positions.
__device__ __forceinline__ uint32_t convb_tap(const GemmEpi::ConvB& c, uint32_t t) {
  const uint32_t k2 = t % c.K2, r = t / c.K2, k1 = r % c.K1, k0 = r / c.K1;
  return (k0 * c.dl0 * c.E1 + k1 * c.dl1) * c.E2 + k2 * c.dl2;
}
// frame byte offset of GEMM column n's contraction byte 0 (tap 0, channel 0)
__device__ __forceinline__ uint32_t convb_row(const GemmEpi::ConvB& c, uint32_t n) {
  const uint32_t y = n / c.Pn, p = n - y * c.Pn;
  const uint32_t o2 = p % c.P2, q = p / c.P2, o1 = q % c.P1, o0 = q / c.P1;
  return (y * c.Ep + (o0 * c.st0 * c.E1 + o1 * c.st1) * c.E2 + o2 * c.st2) * c.Cg;
}
}  // namespace q8
