// q8_gemm_tile.h -- what the register-staged (q8_gemm_any.hip) and the
// deep-ring (q8_gemm_ring.hip) GEMM kernels share: the multiplication of one
// LDS stage and the epilogue over K groups.
#pragma once

#include <type_traits>

#include "q8_device.h"
#include "q8_epilogue.h"
#include "q8_internal.h"

namespace q8 {

constexpr int AK = 128;   // K bytes per LDS stage

// One 128-byte stage: the wave's (32 TM) x (32 TN) sub-tile at (wm, wn).
template <class C>
__device__ __forceinline__ void mfma_stage(const int8_t* st, int wm, int wn, int lane, v16i (&acc)[C::TM][C::TN]) {
  const int r32 = lane & 31, kh = lane >> 5;
  // small sub-tiles read the whole stage's fragments before the first MFMA
  // (one LDS latency per stage, not four); larger ones a 32-byte step at a time
  constexpr int KB = C::TM * C::TN <= 2 ? 4 : 1;
#pragma unroll
  for (int k0 = 0; k0 < 4; k0 += KB) {
    v4i fa[KB][C::TM], fb[KB][C::TN];
#pragma unroll
    for (int q = 0; q < KB; ++q) {
#pragma unroll
      for (int i = 0; i < C::TM; ++i) {
        const int row = wm + 32 * i + r32;
        fa[q][i] = *reinterpret_cast<const v4i*>(st + row * AK + 16 * ((2 * (k0 + q) + kh) ^ swz(row)));
      }
#pragma unroll
      for (int j = 0; j < C::TN; ++j) {
        const int row = wn + 32 * j + r32;
        fb[q][j] = *reinterpret_cast<const v4i*>(st + C::A_BYTES + row * AK + 16 * ((2 * (k0 + q) + kh) ^ swz(row)));
      }
    }
    if constexpr (KB > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < KB; ++q)
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[q][i], fb[q][j], acc[i][j], 0, 0, 0);
  }
}

// The tile's results (every stage buffer free, a barrier passed): KG groups'
// partial sums in acc, group grp's buffers at lds + grp * C::RING.
template <class C, int KG, bool ZP>
__device__ __forceinline__ void tile_epilogue(v16i (&acc)[C::TM][C::TN], int8_t* lds, const double* s_rows,
                                             const int* sum_a, const int* sum_b, int wave, int grp, int lane,
                                             int m0, int n0, int wm, int wn, int M, int N, int64_t o_base,
                                             const GemmEpi& e, const AffineDot& z, const AnyPlan& p,
                                             void* __restrict__ out) {
  const int r32 = lane & 31, kh = lane >> 5;
  int8_t* const ring = lds + grp * C::RING;
  // Epilogue: a 32-row strip of the wave's sub-tile at a time through its
  // own LDS region (the stages are no longer read), then a rolled loop, one
  // epilogue's code, over V = 4 columns per lane stored as one 16-byte (int8
  // out: 4-byte) quad where every quad is aligned and inside, else over
  // single columns, the lanes of a row taking consecutive ones.
  constexpr int PITCH = C::WN + 8;
  static_assert(C::WAVES * 32 * PITCH * 4 <= C::RING, "strips fit in the stage buffers");
  // group g's strip of sub-tile `wave`; with KG groups each stores 32 / KG of
  // the strip's rows, adding the groups' sums
  int* strip = reinterpret_cast<int*>(ring) + wave * 32 * PITCH;
  const int* strip0 = reinterpret_cast<const int*>(KG > 1 ? lds : ring) + wave * 32 * PITCH;
  const bool fp = !e.out_i32;
  auto strips = [&](auto vc) {
    constexpr int V = decltype(vc)::value;
    constexpr int LPR = C::WN / V;                     // lanes per strip row
    constexpr int RPI = 64 / LPR;                      // strip rows per pass
    constexpr int NIT = 32 / RPI / KG;
    static_assert(NIT >= 1, "every group has rows to store");
    const int col = V * (lane % LPR), qrow = lane / LPR;
    const int n = n0 + wn + col;
    const bool live = n < N;
    double sbn[V];
    float bn[V];
    uint32_t zc[V];
#pragma unroll
    for (int c = 0; c < V; ++c) {
      const int nc = live ? n + c : N - 1;
      sbn[c] = fp && e.mode == 1 ? e.sB[(int64_t)nc * e.sB_stride] : 0.0;
      bn[c] = e.bias ? e.bias[nc] : 0.0f;
      zc[c] = 0u;
      if constexpr (ZP) zc[c] = (uint32_t)z.cA * (uint32_t)sum_b[wn + col + c] + z.kcc;
    }
    int64_t at0 = o_base + n, ld = N;       // where column n's elements go
    if (e.col_blk > 0) {                    // n and the block size fit 31 bits
      const unsigned blk = (unsigned)n / (unsigned)e.col_blk;
      at0 = o_base + blk * e.blk_stride + (unsigned)n - blk * (unsigned)e.col_blk;
      ld = e.ld_out;
    }
    auto strip_out = [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if constexpr (KG > 1 && i > 0) __syncthreads();   // the previous strip's sums have been read
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) strip[((r >> 2) * 8 + kh * 4 + (r & 3)) * PITCH + 32 * j + r32] = acc[i][j][r];
      if constexpr (KG > 1) __syncthreads();
#pragma unroll 1
      for (int it = 0; it < NIT; ++it) {
        const int srow = (grp * NIT + it) * RPI + qrow, trow = wm + 32 * i + srow, m = m0 + trow;
        uint32_t a[V];
#pragma unroll
        for (int c = 0; c < V; ++c) a[c] = 0u;
#pragma unroll
        for (int g = 0; g < KG; ++g) {
          const int* s = strip0 + g * (C::RING / 4) + srow * PITCH + col;
          if constexpr (V == 4) {
            const v4i q = *reinterpret_cast<const v4i*>(s);
#pragma unroll
            for (int c = 0; c < V; ++c) a[c] += (uint32_t)q[c];
          } else {
            a[0] += (uint32_t)s[0];
          }
        }
        if constexpr (ZP) {
#pragma unroll
          for (int c = 0; c < V; ++c) a[c] += zc[c] + (uint32_t)z.cB * (uint32_t)sum_a[trow];
        }
        if (m >= M || !live) continue;
        const int64_t at = (int64_t)m * ld + at0;
        int w[V];
#pragma unroll
        for (int c = 0; c < V; ++c) w[c] = (int)a[c];
        if (fp) {
          const double sr = s_rows[trow];
          float y[V];
#pragma unroll
          for (int c = 0; c < V; ++c) {
            y[c] = e.mode == 0 ? (float)((double)w[c] * e.s_out) : mul_acc_f32scale(w[c], (float)(sr * sbn[c]));
            if (e.bias) y[c] = y[c] + bn[c];
          }
          if (e.act == 1) {
#pragma unroll
            for (int c = 0; c < V; ++c) y[c] = relu_js(y[c]);
          } else if (e.act == 2) {
#pragma unroll
            for (int c = 0; c < V; ++c) y[c] = silu_js(y[c]);
          }
          if (e.out_q8) {
            int8_t* o = static_cast<int8_t*>(out) + at;
#pragma unroll
            for (int c = 0; c < V; ++c) w[c] = requant(y[c], e);
            if constexpr (V == 4) *reinterpret_cast<int*>(o) = pack4(w[0], w[1], w[2], w[3]);
            else *o = (int8_t)w[0];
            continue;
          }
#pragma unroll
          for (int c = 0; c < V; ++c) w[c] = __float_as_int(y[c]);
        }
        int* o = static_cast<int*>(out) + at;
        if constexpr (V == 4) __builtin_nontemporal_store(v4i{w[0], w[1], w[2], w[3]}, reinterpret_cast<v4i*>(o));
        else *o = w[0];
      }
    };
    strip_out(std::integral_constant<int, 0>{});
    if constexpr (C::TM > 1) strip_out(std::integral_constant<int, 1>{});
    static_assert(C::TM <= 2, "strip_out calls cover TM <= 2");
  };
  // quads: N, and with column blocks every block's start and pitch, multiples
  // of 4 elements from an aligned base
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 && (p.o_step & 3) == 0 &&
                   (e.col_blk == 0 || ((e.col_blk | e.blk_stride | e.ld_out) & 3) == 0);
  if (vec) strips(std::integral_constant<int, 4>{});
  else strips(std::integral_constant<int, 1>{});
}

}  // namespace q8
