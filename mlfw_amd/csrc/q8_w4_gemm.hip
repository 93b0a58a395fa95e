// q8_w4_gemm.hip -- the W4A8 linear (q8_w4.hip defines it) for prompts and
// larger decode batches: a tiled GEMM over 4-bit per-group weights.
//
// The GEMV walks the weights once per 16 tokens; from a few dozen tokens on
// that is most of its time.  Here a workgroup (4 waves, 2 x 2) computes BM
// tokens x BN weight rows and reads each weight once per BM tokens.
//
// What bounds it: the definition adds the groups' sums in order in f64,
//   S = acc_0 * sw_0 + acc_1 * sw_1 + ...,
// three f64 instructions per output and group (convert, multiply, add; none
// may be fused), about 1.5 times the MFMA time at groups of 128.  So the rest
// is kept off the VALU:
//   * the conversion is one subtraction: the MFMA accumulator starts at 2^31
//     (mod 2^32), so its bits are the low word of a double whose high word is
//     a constant, 2^48 + (v + 2^31) / 16 for an accumulator v = 16 acc, and
//     subtracting 2^48 + 2^27 leaves acc exactly;
//   * v = 16 acc because nibbles are used where they lie: a byte masked to
//     its high nibble is 16 q as a signed int8, and shifted left by 4 its low
//     nibble is too.  A 16-byte chunk of 32 codes gives two operand fragments
//     (even and odd codes) for 12 instructions;
//   * activations are split into the same even / odd order once per tile, on
//     their way through registers into LDS;
//   * weights and scales pass through LDS too, in 128-byte row segments: read
//     straight into the MFMA layout (64 bytes of each of 16 rows per load, a
//     scale per lane and group) those loads were most of the kernel's time
//     (512 tokens, 4096 x 22016 and 11008 x 4096: 303 us; without the scale
//     loads 223, without either 176).
// A step is 128 codes of K: two 16x16x64 MFMAs per 16 x 16 block.  Groups of
// 64 or 32 share a step: their MFMAs see the other groups' chunks of the
// activations as zeros.  Groups of several steps keep accumulating.
#include <algorithm>
#include <type_traits>

#include "q8_device.h"
#include "q8_epilogue.h"
#include "q8_internal.h"

namespace q8 {

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// 32 activation codes into their even- and odd-indexed halves.
__device__ __forceinline__ void split_even_odd(v4i lo, v4i hi, v4i& ev, v4i& od) {
  const uint32_t w[8] = {(uint32_t)lo.x, (uint32_t)lo.y, (uint32_t)lo.z, (uint32_t)lo.w,
                         (uint32_t)hi.x, (uint32_t)hi.y, (uint32_t)hi.z, (uint32_t)hi.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {   // v_perm: bytes 0-3 of the second operand, 4-7 of the first
    ev[i] = (int)__builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], 0x06040200u);
    od[i] = (int)__builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], 0x07050301u);
  }
}

// GPSX groups per step (1, 2, 4); 0: a group is `spg` >= 2 steps.
template <int BM, int BN, int GPSX>
__global__ __launch_bounds__(256, 2)
void k_gemm_w4(const int8_t* __restrict__ xq, const double* __restrict__ sx, int sx_stride,
               const uint8_t* __restrict__ wq4, const double* __restrict__ sw, int M, int N, int K, int spg, int G,
               int tiles_m, int tiles_n, const float* __restrict__ bias, int act, float* __restrict__ y) {
  constexpr int TM = BM / 32, TN = BN / 32;            // 16 x 16 blocks per wave
  constexpr bool LONG = GPSX == 0;
  constexpr int GPS = LONG ? 1 : GPSX;
  constexpr int GW = 16, GP = GW + 1;                  // scale window: groups, row pitch in doubles
  // a stage is two steps: 256 codes
  __shared__ __align__(1024) int8_t xs[2][BM * 256];   // chunk c (32 codes) even / odd at slots 2c, 2c + 1
  __shared__ __align__(1024) int8_t ws[2][BN * 128];
  __shared__ double ss[2][BN * GP];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  int tm, tn;
  tile_of((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int steps = (K + 127) / 128, stages = (K + 255) / 256;

  // activations: thread t stages chunk t % 8 of tokens t / 8, + 32, ...
  constexpr int XR = BM / 32;
  const __amdgpu_buffer_rsrc_t rx = rsrc_of(xq, (uint32_t)M * (uint32_t)K);
  const int xc = tid & 7;
  v4i xr[XR][2];
  // weights: thread t stages 16 bytes (chunk t % 8 of a stage) of rows t / 8, + 32, ...
  constexpr int WR = BN / 32;
  const int half = K / 2;
  const int rows_w = min(BN, N - n0);
  const __amdgpu_buffer_rsrc_t rw = rsrc_of(wq4 + (int64_t)n0 * half, (uint32_t)rows_w * (uint32_t)half);
  v4i wr[WR];
  constexpr uint32_t PAST = 0x80000000u;               // past every buffer's end: reads zero
  auto load_stage = [&](int p) {
#pragma unroll
    for (int u = 0; u < XR; ++u) {
      const int t = (tid >> 3) + 32 * u, k = 256 * p + 32 * xc;
      const uint32_t off = m0 + t < M && k < K ? (uint32_t)(m0 + t) * (uint32_t)K + (uint32_t)k : PAST;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        xr[u][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rx, off + 16u * h, 0, 0));
    }
#pragma unroll
    for (int u = 0; u < WR; ++u) {
      const int r = (tid >> 3) + 32 * u, k = 128 * p + 16 * xc;
      const uint32_t off = r < rows_w && k < half ? (uint32_t)r * (uint32_t)half + (uint32_t)k : PAST;
      wr[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0));
    }
  };
  auto put_stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < XR; ++u) {
      const int t = (tid >> 3) + 32 * u;
      v4i ev, od;
      split_even_odd(xr[u][0], xr[u][1], ev, od);
      int8_t* row = &xs[buf][t * 256];
      *reinterpret_cast<v4i*>(row + 16 * ((2 * xc) ^ (t & 15))) = ev;
      *reinterpret_cast<v4i*>(row + 16 * ((2 * xc + 1) ^ (t & 15))) = od;
    }
#pragma unroll
    for (int u = 0; u < WR; ++u) {
      const int r = (tid >> 3) + 32 * u;
      *reinterpret_cast<v4i*>(&ws[buf][r * 128 + 16 * (xc ^ swz(r))]) = wr[u];
    }
  };
  // scales: a window of 16 groups of every row, 16 lanes per row
  constexpr int SR = BN / 16;
  double sr_[SR];
  auto load_scales = [&](int win) {
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int r = (tid >> 4) + 16 * u;
      sr_[u] = sw[(int64_t)min(n0 + r, N - 1) * G + min(GW * win + (tid & 15), G - 1)];
    }
  };
  auto put_scales = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SR; ++u) ss[buf][((tid >> 4) + 16 * u) * GP + (tid & 15)] = sr_[u];
  };

  // S starts at -0.0: -0.0 + t is t for every t, the definition's first term
  double S[TM][TN][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][j][r] = -0.0;
  const v4i zero_acc = {(int)0x80000000, (int)0x80000000, (int)0x80000000, (int)0x80000000};
  v4i run[TM][TN];                                     // groups of several steps only
  if constexpr (LONG) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) run[i][j] = zero_acc;
  }

  auto compute = [&](int s, int buf) {
    const int h = s & 1;
    v4i xe[TM], xo[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = wm + 16 * i + r16;
      const int8_t* p = &xs[buf][row * 256];
      xe[i] = *reinterpret_cast<const v4i*>(p + 16 * ((8 * h + 2 * g4) ^ r16));
      xo[i] = *reinterpret_cast<const v4i*>(p + 16 * ((8 * h + 2 * g4 + 1) ^ r16));
    }
    const bool last = !LONG || (s + 1) % spg == 0;     // uniform: a group ends with this step
    const int g0 = LONG ? s / spg : GPS * s;           // uniform
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int wrow = wn + 16 * j + r16;
      const v4i w = *reinterpret_cast<const v4i*>(&ws[buf][wrow * 128 + 16 * ((4 * h + g4) ^ swz(wrow))]);
      double sc[GPS];
#pragma unroll
      for (int u = 0; u < GPS; ++u) sc[u] = ss[(g0 / GW) & 1][wrow * GP + (g0 + u) % GW];
      v4i we, wo;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        we[c] = (int)(((uint32_t)w[c] << 4) & 0xF0F0F0F0u);
        wo[c] = (int)((uint32_t)w[c] & 0xF0F0F0F0u);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int u = 0; u < GPS; ++u) {
          v4i a;
          if constexpr (GPS == 1) {
            a = __builtin_amdgcn_mfma_i32_16x16x64_i8(xe[i], we, LONG ? run[i][j] : zero_acc, 0, 0, 0);
            a = __builtin_amdgcn_mfma_i32_16x16x64_i8(xo[i], wo, a, 0, 0, 0);
            if constexpr (LONG) {
              run[i][j] = last ? zero_acc : a;
              if (!last) continue;
            }
          } else {
            // group u of the step: chunks 4 u / GPS ... of the activations, zeros elsewhere
            const bool mine = g4 / (4 / GPS) == u;
            const v4i z = {0, 0, 0, 0};
            const v4i e = mine ? xe[i] : z, o = mine ? xo[i] : z;
            a = __builtin_amdgcn_mfma_i32_16x16x64_i8(e, we, zero_acc, 0, 0, 0);
            a = __builtin_amdgcn_mfma_i32_16x16x64_i8(o, wo, a, 0, 0, 0);
            if (g0 + u >= G) continue;                 // uniform: groups past K
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            // 2^48 + (16 acc + 2^31) / 16, less 2^48 + 2^27: acc, exactly
            const double d = __hiloint2double(0x42F00000, a[r]) - (0x1p48 + 0x1p27);
            S[i][j][r] = S[i][j][r] + d * sc[u];
          }
        }
      }
    }
  };

  // Stage p's buffer is p % 2: while it is multiplied the next stage's loads
  // land in registers, and go into the other buffer once this stage's reads
  // have started; window w's scales likewise, a window ahead.
  const int spw = LONG ? GW * spg : GW / GPS;          // steps per scale window, even
  load_stage(0);
  load_scales(0);
  put_stage(0);
  put_scales(0);
  __syncthreads();
  for (int p = 0; p < stages; ++p) {
    const int s = 2 * p, buf = p & 1;
    const bool more = p + 1 < stages, win = s % spw == 0 && s + spw < steps;   // uniform
    if (more) load_stage(p + 1);
    if (win) load_scales(s / spw + 1);
    compute(s, buf);
    if (s + 1 < steps) compute(s + 1, buf);
    // buffers (p + 1) % 2: stage p - 1 and window s / spw - 1 were last read
    // before the barrier that ended stage p - 1
    if (more) put_stage(buf ^ 1);
    if (win) put_scales((s / spw + 1) & 1);
    __syncthreads();
  }

  // y = act(fround(S * sx[m]) + bias[n]): lane (r16, g4) holds column r16 and rows 4 g4 + r of each block
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    double sr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm + 16 * i + 4 * g4 + r;
      sr[r] = sx[(int64_t)min(m, M - 1) * sx_stride];
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + 16 * j + r16;
      const float b = bias && n < N ? bias[n] : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * g4 + r;
        float v = (float)(S[i][j][r] * sr[r]);
        if (bias) v = v + b;
        if (act == 1) v = relu_js(v);
        else if (act == 2) v = silu_js(v);
        if (m < M && n < N) y[(int64_t)m * N + n] = v;
      }
    }
  }
}

template <int BM, int BN>
hipError_t launch_tile(const int8_t* xq, const double* sx, int sx_stride, const uint8_t* wq4, const double* sw, int M,
                       int N, int K, int group, const float* bias, int act, float* y, hipStream_t st) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN, G = K / group;
  const dim3 grid((unsigned)(tm * tn)), block(256);
  note_route("w4", BM, BN);
#define Q8_W4G(GPS, spg)                                                                                            \
  hipLaunchKernelGGL((k_gemm_w4<BM, BN, GPS>), grid, block, 0, st, xq, sx, sx_stride, wq4, sw, M, N, K, spg, G, tm, \
                     tn, bias, act, y)
  if (group == 32) Q8_W4G(4, 1);
  else if (group == 64) Q8_W4G(2, 1);
  else if (group == 128) Q8_W4G(1, 1);
  else Q8_W4G(0, group / 128);
#undef Q8_W4G
  return hipGetLastError();
}

}  // namespace

// Tile and estimated time (us).  A step of one tile costs `step` by tile and
// group size; with more than a tile per CU the steps of resident workgroups
// overlap until about T tiles are in flight.  Fitted to every tile on M in
// 17..512 x five [N, K] x groups of 32 and 128 (22016 x 4096, group 128:
// M = 64 32.0 / 27.4 / 30.8 us on 32 x 32, 32 x 64, 64 x 64; M = 512 189 / 163
// / 149; 4096 x 11008: M = 64 27.7 / 37.0 / 50.0, M = 512 96 / 87 / 72).
static int w4_tile(int64_t M, int64_t N, int64_t K, int64_t group, double* us) {
  static const double step[3][3] = {{0.28, 0.40, 0.55}, {0.38, 0.58, 0.85}, {0.55, 0.88, 1.48}};   // groups >= 128, 64, 32
  const double T[3] = {400.0, 360.0, 300.0};
  const int bm[3] = {32, 32, 64}, bn[3] = {32, 64, 64};
  const double cus = cu_count() > 0 ? cu_count() : 256, steps = (double)((K + 127) / 128);
  const int gi = group == 32 ? 2 : group == 64 ? 1 : 0;
  int best = 0;
  for (int c = 0; c < 3; ++c) {
    const double tiles = (double)(((M + bm[c] - 1) / bm[c]) * ((N + bn[c] - 1) / bn[c]));
    const double rounds = tiles <= cus ? 1.0 : std::max(1.5, tiles / (T[c] * cus / 256.0));
    const double t = 2.6 + steps * step[gi][c] * rounds;
    if (c == 0 || t < *us) {
      *us = t;
      best = c;
    }
  }
  return best;
}

// Groups of 32 or 64, or multiples of 128 up to 65536 (16 q x summed over a
// group stays below 2^31); K then is a multiple of 32, so is every offset of
// 16; activations within 31-bit offsets.  And where the estimate is below
// the GEMV's, about 4 us and 8e13 multiply-adds a second (5e13 and 2.6e13
// with groups of 64 and 32): from some 20 tokens on wide layers (17 x 22016 x
// 4096: 32.4 -> 19.1 us), from 128 on small ones (1280 x 3456: 10.4 both).
// Both estimates miss by some 5%, which goes to the GEMV: over 533 shapes, M 17
// to 1024, cold weights and warm, 20 of 1000 timings are then slower than the
// GEMV's by more than 3% (without it 33), and the mean is better.
bool gemm_w4_ok(const int8_t* xq, const uint8_t* wq4, int64_t M, int64_t N, int64_t K, int64_t group) {
  const bool g = group == 32 || group == 64 || (group % 128 == 0 && group <= 65536);
  if (!g || M <= 16 || K < 32 || K % 32 != 0 || M * K >= ((int64_t)1 << 31) ||
      ((reinterpret_cast<uintptr_t>(xq) | reinterpret_cast<uintptr_t>(wq4)) & 15) != 0)
    return false;
  double us = 0.0;
  (void)w4_tile(M, N, K, group, &us);
  const double rate = group == 32 ? 2.6e7 : group == 64 ? 5e7 : 8e7;   // per us
  return 1.05 * us < 4.0 + (double)M * (double)N * (double)K / rate;
}

hipError_t launch_gemm_w4(const int8_t* xq, const double* sx, int sx_stride, const uint8_t* wq4, const double* sw,
                          int64_t M, int64_t N, int64_t K, int64_t group, const float* bias, int act, float* y,
                          hipStream_t st) {
  const int m = (int)M, n = (int)N, k = (int)K, g = (int)group;
  double us = 0.0;
  switch (w4_tile(M, N, K, group, &us)) {
    case 0: return launch_tile<32, 32>(xq, sx, sx_stride, wq4, sw, m, n, k, g, bias, act, y, st);
    case 1: return launch_tile<32, 64>(xq, sx, sx_stride, wq4, sw, m, n, k, g, bias, act, y, st);
    default: return launch_tile<64, 64>(xq, sx, sx_stride, wq4, sw, m, n, k, g, bias, act, y, st);
  }
}

}  // namespace q8
