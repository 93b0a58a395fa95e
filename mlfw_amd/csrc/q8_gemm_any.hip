// q8_gemm_any.hip -- the int8 MFMA GEMM for operands the direct-to-LDS GEMM
// (q8_gemm.hip) cannot copy: any K (not only multiples of 16), any alignment,
// and the affine quantized_dot (ui8 operands and zero points in the same
// launch).
//
// What bounds it: the copies.  buffer_load ... lds moves 16-byte chunks at
// 16-byte aligned addresses, so a row pitch that is not a multiple of 16 has
// no such form.  Here a lane loads its 16-byte chunk of a row into registers
// (an unaligned global_load_dwordx4), and writes it to the same swizzled LDS
// layout with ds_write_b128; the loads of the stage after next are in flight
// while a stage is multiplied.  The contraction's tail never reads past the
// row: a chunk that would cross the row's end is loaded 16 bytes before the
// end and shifted down, zeros coming in.  Passing through registers costs
// VGPRs and LDS write cycles that the direct copies do not pay, so operands
// those can take stay with them (launch_gemm).
//
// The affine form uses the pass through registers: a ui8 operand's bytes are
// flipped by 0x80 there (a - 128), and v_dot4 against ones adds up the row
// sums that the zero-point correction needs, so quantized_dot with zero
// points reads each operand once and writes its result once -- as separate
// passes the flips, row sums and correction were up to four more launches.
//
// Measured (MI355X, whole calls, before: one thread per output with byte
// loads): quantized_dot 788 x 1000 x 1500 with ui8 activations 4350 -> 12.9
// us (the host's share of the call; 9.1 replayed from a graph); dynamic linear
// 42 x 3777 x 7986 5400 -> 57 us, 1183 x 3917 x 3001 59300 -> 72 us.
#include <type_traits>

#include "q8_device.h"
#include "q8_epilogue.h"
#include "q8_gemm_tile.h"
#include "q8_internal.h"

namespace q8 {

namespace {

template <int BM, int BN, int KG>
struct AnyCfg {
  static constexpr int WM = BM / 2, WN = BN / 2;        // per-wave sub-tile, waves 2 x 2
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int A_BYTES = BM * AK;
  static constexpr int STAGE = (BM + BN) * AK;
  static constexpr int RING = 2 * STAGE;                // a group's stages
  static constexpr int WAVES = 4;                       // per group
  static constexpr int LDS = KG * RING + 8 * BM + 4 * (BM + BN);   // + row scales, row and column sums
  static constexpr int CA = BM / 32, CB = BN / 32;      // 16-byte chunks per lane and stage
  static_assert(TM >= 1 && TN >= 1 && BM % 64 == 0 && BN % 64 == 0, "tile shape");
};

// v's 16 bytes moved down by sh bytes (sh >= 0), zeros coming in at the top.
__device__ __forceinline__ v4i shift_down(v4i v, int sh) {
  if (sh >= 16) return v4i{0, 0, 0, 0};
  const int dw = sh >> 2;
  v4i t = (dw & 1) ? v4i{v.y, v.z, v.w, 0} : v;
  t = (dw & 2) ? v4i{t.z, t.w, 0, 0} : t;
  const uint32_t b = (uint32_t)(sh & 3);
  return v4i{(int)__builtin_amdgcn_alignbyte((uint32_t)t.y, (uint32_t)t.x, b),
             (int)__builtin_amdgcn_alignbyte((uint32_t)t.z, (uint32_t)t.y, b),
             (int)__builtin_amdgcn_alignbyte((uint32_t)t.w, (uint32_t)t.z, b),
             (int)__builtin_amdgcn_alignbyte(0u, (uint32_t)t.w, b)};
}

__device__ __forceinline__ int sum16(v4i v, int s) {
  s = __builtin_amdgcn_sdot4(v.x, 0x01010101, s, false);
  s = __builtin_amdgcn_sdot4(v.y, 0x01010101, s, false);
  s = __builtin_amdgcn_sdot4(v.z, 0x01010101, s, false);
  return __builtin_amdgcn_sdot4(v.w, 0x01010101, s, false);
}

// The offset of every 16-byte chunk of a conv's contraction from its column's
// frame position.
__device__ __forceinline__ void fill_taps(int* taps, const GemmEpi& e, const AnyPlan& p, int K, int tid, int threads) {
  for (int i = tid; i < (K >> 4); i += threads) {
    const uint32_t t = 16u * (uint32_t)i / (uint32_t)p.conv_cg;
    taps[i] = (int)(convb_tap(e.cb, t) * e.cb.Cg + (16u * (uint32_t)i - t * (uint32_t)p.conv_cg));
  }
}

// out = epilogue(A [M, K] . B [N, K]^T).  ZP: operands flipped by z.xa / z.xb
// (0 or 0x80808080) and the int32 result corrected by
// cB * rowsum(a') + cA * rowsum(b') + K * cA * cB (q8_zp.hip states why).
//
// KG groups of 4 waves share a tile and take every KG-th K stage, each with
// a ring of its own; their partial sums meet in LDS (int32 addition does not
// depend on the order).  A stage costs its load latency whatever the tile, so
// with a workgroup per CU or less a quarter of the stages in sequence is
// close to a quarter of the time.
//
// CONV: B is a channel-last conv frame (GemmEpi::ConvB); a 16-byte chunk of
// the contraction lies in one kernel position, and a table in LDS holds every
// chunk's offset from its column's frame position.
template <int BM, int BN, int KG, bool ZP, bool CONV>
__global__ __launch_bounds__(256 * KG, KG == 4 ? 4 : 2)
void k_qgemm_any(const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M, int N, int K,
                 int tiles_m, int tiles_n, GemmEpi e, AffineDot z, AnyPlan p, void* __restrict__ out) {
  using C = AnyCfg<BM, BN, KG>;
  extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
  double* s_rows = reinterpret_cast<double*>(lds + KG * C::RING);
  int* sum_a = reinterpret_cast<int*>(s_rows + BM);
  int* sum_b = sum_a + BM;
  int* taps = sum_b + BN;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wv & 3, grp = wv >> 2;
  int8_t* const ring = lds + grp * C::RING;
  int tm, tn;
  tile_of((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int rows_a = min(BM, M - m0), rows_b = min(BN, N - n0);
  if (tid < BM)
    s_rows[tid] = e.mode == 1 && !e.out_i32 && tid < rows_a ? e.sA[(int64_t)(m0 + tid) * e.sA_stride] : 0.0;
  if (ZP && tid < BM + BN) sum_a[tid] = 0;
  A += blockIdx.y * p.a_step;
  B += blockIdx.y * p.b_step;
  const int64_t o_base = blockIdx.y * p.o_step;
  if constexpr (CONV) {
    fill_taps(taps, e, p, K, tid, 256 * KG);
    __syncthreads();
  }

  // Copy plan, as k_qgemm's: wave w fills tile rows [w * BM / 4, ...) of A
  // and its share of B, 8 lanes per row.  A row past the edge repeats the
  // last one: its results are never stored.
  const int rl = lane >> 3, c16 = 16 * (lane & 7);
  const int8_t* pa[C::CA];
  const int8_t* pb[C::CB];
  int la[C::CA], lb[C::CB];        // LDS byte offsets within a stage
#pragma unroll
  for (int j = 0; j < C::CA; ++j) {
    const int row = wave * (BM / 4) + 8 * j + rl;
    pa[j] = A + (m0 + min(row, rows_a - 1)) * p.lda;
    la[j] = row * AK + 16 * ((lane & 7) ^ swz(row));
  }
#pragma unroll
  for (int j = 0; j < C::CB; ++j) {
    const int row = wave * (BN / 4) + 8 * j + rl;
    const int n = n0 + min(row, rows_b - 1);
    pb[j] = B + (CONV ? (int64_t)convb_row(e.cb, (uint32_t)n) : n * p.ldb);
    lb[j] = (BM + row) * AK + 16 * ((lane & 7) ^ swz(row));
  }
  const int KT = (K + AK - 1) / AK;
  const int xa = ZP ? z.xa : 0, xb = ZP ? z.xb : 0;
  int sa[C::CA], sb[C::CB];
#pragma unroll
  for (int j = 0; j < C::CA; ++j) sa[j] = 0;
#pragma unroll
  for (int j = 0; j < C::CB; ++j) sb[j] = 0;
  v4i ra[C::CA], rb[C::CB];
  auto load = [&](int kt) {
    const int kc = kt * AK + c16;
    if (CONV || K >= 16) {
      const int kk = min(kc, K - 16);
      const int kb = CONV ? taps[kk >> 4] : kk;
#pragma unroll
      for (int j = 0; j < C::CA; ++j) ra[j] = load16_any(pa[j] + kk);
#pragma unroll
      for (int j = 0; j < C::CB; ++j) rb[j] = load16_any(pb[j] + kb);
    } else {                       // a row shorter than a chunk: byte by byte
      auto bytes = [&](const int8_t* q, int x) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll 1
        for (int k = 0; k < K; ++k) {
          const uint32_t b = (uint32_t)(uint8_t)(q[k] ^ (int8_t)x) << (8 * (k & 3));
          w[0] |= k < 4 ? b : 0u;
          w[1] |= k >= 4 && k < 8 ? b : 0u;
          w[2] |= k >= 8 && k < 12 ? b : 0u;
          w[3] |= k >= 12 ? b : 0u;
        }
        return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]} ^ x;   // undone by put's flip: zeros past K
      };
#pragma unroll
      for (int j = 0; j < C::CA; ++j) ra[j] = bytes(pa[j], xa);
#pragma unroll
      for (int j = 0; j < C::CB; ++j) rb[j] = bytes(pb[j], xb);
    }
  };
  // the loaded stage kt into its buffer
  auto put = [&](int kt) {
    int8_t* st = ring + (kt / KG & 1) * C::STAGE;
    if constexpr (ZP) {
#pragma unroll
      for (int j = 0; j < C::CA; ++j) ra[j] ^= xa;
#pragma unroll
      for (int j = 0; j < C::CB; ++j) rb[j] ^= xb;
    }
    if (kt == KT - 1) {            // uniform: only the last stage has a tail to shift
      // how far below its place load() took the chunk
      const int kc = kt * AK + c16, sh = CONV || K >= 16 ? kc - min(kc, K - 16) : c16;
#pragma unroll
      for (int j = 0; j < C::CA; ++j) ra[j] = shift_down(ra[j], sh);
#pragma unroll
      for (int j = 0; j < C::CB; ++j) rb[j] = shift_down(rb[j], sh);
    }
#pragma unroll
    for (int j = 0; j < C::CA; ++j) *reinterpret_cast<v4i*>(st + la[j]) = ra[j];
#pragma unroll
    for (int j = 0; j < C::CB; ++j) *reinterpret_cast<v4i*>(st + lb[j]) = rb[j];
    if constexpr (ZP) {
#pragma unroll
      for (int j = 0; j < C::CA; ++j) sa[j] = sum16(ra[j], sa[j]);
#pragma unroll
      for (int j = 0; j < C::CB; ++j) sb[j] = sum16(rb[j], sb[j]);
    }
  };

  const int wm = (wave >> 1) * C::WM, wn = (wave & 1) * C::WN;
  v16i acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  if (grp < KT) {
    load(grp);
    put(grp);
    if (grp + KG < KT) load(grp + KG);
  }
  __syncthreads();
  for (int k0 = 0; k0 < KT; k0 += KG) {      // every group runs every iteration: the barriers are the workgroup's
    const int kt = k0 + grp;
    const int8_t* st = ring + (kt / KG & 1) * C::STAGE;
    // the next stage goes into the other buffer, whose last reads ended
    // before the barrier that closed the previous iteration; then the loads
    // of the one after it, which have this stage's MFMAs to land (a second
    // register set, two stages in flight, measured no faster)
    if (kt + KG < KT) {
      put(kt + KG);
      if (kt + 2 * KG < KT) load(kt + 2 * KG);
    }
    if (kt < KT) mfma_stage<C>(st, wm, wn, lane, acc);
    __syncthreads();
  }

  if constexpr (ZP) {
    // row sums: the 8 lanes of a row (and the K groups) hold its parts
#pragma unroll
    for (int j = 0; j < C::CA; ++j) {
      int s = sa[j];
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += __shfl_xor(s, 4, 64);
      if ((lane & 7) == 0) atomicAdd(&sum_a[wave * (BM / 4) + 8 * j + rl], s);
    }
#pragma unroll
    for (int j = 0; j < C::CB; ++j) {
      int s = sb[j];
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += __shfl_xor(s, 4, 64);
      if ((lane & 7) == 0) atomicAdd(&sum_b[wave * (BN / 4) + 8 * j + rl], s);
    }
    __syncthreads();
  }

  tile_epilogue<C, KG, ZP>(acc, lds, s_rows, sum_a, sum_b, wave, grp, lane, m0, n0, wm, wn, M, N, o_base, e, z, p, out);
}

// The same product with the K range split over the 8 waves of a workgroup,
// for up to one 32 x 32 tile per CU: each wave computes the whole tile over
// its own 128-byte slices of K, its operands loaded straight into the MFMA
// layout (16x16x64: lane l holds 16 bytes of row l % 16, chunk l / 16), two
// 64-byte steps in flight.  No LDS staging and no barrier until the partial
// tiles meet in LDS: with so few tiles the time is one workgroup's load
// latencies, and a staged stage costs a barrier on top of its own.  (17 x 4096
// x 4096: 16.5 us in four K groups of 64 x 64 tiles, 11.1 here; 512 x 49 x
// 4608, a 7 x 7 x 512 conv of one image: 15.6 and 8.1 us.  Larger tiles of
// this form lose: 64 x 11008 x 4096 takes 25 us with 64 x 64, 21 staged.)
constexpr int WKT = 2, WKW = 8, WKB = 16 * WKT;       // 16-row blocks, waves, tile edge
constexpr int WK_PITCH = WKB + 4;
constexpr int ANY_SPLIT_K = 5120;
constexpr int WK_LDS = WKT * WKW * 16 * WK_PITCH * 4 + 8 * WKB + 8 * WKB;
template <bool SPLIT, bool ZP, bool CONV>
__global__ __launch_bounds__(64 * WKW, 2)
void k_qgemm_wk(const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M, int N, int K,
                int tiles_m, int tiles_n, GemmEpi e, AffineDot z, AnyPlan p, void* __restrict__ out) {
  extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
  int* red = reinterpret_cast<int*>(lds);                 // [strip][wave][16][WK_PITCH]
  double* s_rows = reinterpret_cast<double*>(red + WKT * WKW * 16 * WK_PITCH);
  int* sum_a = reinterpret_cast<int*>(s_rows + WKB);
  int* sum_b = sum_a + WKB;
  int* taps = sum_b + WKB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  int tm, tn;
  tile_of((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * WKB, n0 = tn * WKB;
  if (tid < WKB)
    s_rows[tid] = e.mode == 1 && !e.out_i32 && m0 + tid < M ? e.sA[(int64_t)(m0 + tid) * e.sA_stride] : 0.0;
  if (ZP && tid < 2 * WKB) sum_a[tid] = 0;
  A += blockIdx.y * p.a_step;
  B += blockIdx.y * p.b_step;
  const int64_t o_base = blockIdx.y * p.o_step;
  if constexpr (CONV) fill_taps(taps, e, p, K, tid, 64 * WKW);
  if (CONV || ZP) __syncthreads();
  const int xa = ZP ? z.xa : 0, xb = ZP ? z.xb : 0;
  // rows past the edge repeat the last one: their results are never stored
  const int8_t* pa[WKT];
  const int8_t* pb[WKT];
#pragma unroll
  for (int i = 0; i < WKT; ++i) {
    pa[i] = A + (int64_t)min(m0 + 16 * i + r16, M - 1) * p.lda;
    const int n = min(n0 + 16 * i + r16, N - 1);
    pb[i] = B + (CONV ? (int64_t)convb_row(e.cb, (uint32_t)n) : n * p.ldb);
  }
  int sa[WKT], sb[WKT];
  v4i acc[WKT][WKT];
#pragma unroll
  for (int i = 0; i < WKT; ++i) {
    sa[i] = sb[i] = 0;
#pragma unroll
    for (int j = 0; j < WKT; ++j) acc[i][j] = v4i{0, 0, 0, 0};
  }
  struct Frag {
    v4i a[WKT], b[WKT];
  };
  // 64-byte step s of the contraction: steps 2 c and 2 c + 1 are slice c,
  // wave w takes slices w, w + 8, ...  K >= 16.
  const int KS = (K + 63) / 64;
  auto load = [&](int s, Frag& f) {
    const int kk = min(64 * s + 16 * g, K - 16);
    const int kb = CONV ? taps[kk >> 4] : kk;
#pragma unroll
    for (int i = 0; i < WKT; ++i) {
      f.a[i] = load16_any(pa[i] + kk);
      f.b[i] = load16_any(pb[i] + kb);
    }
  };
  auto mul = [&](int s, Frag& f) {
    if constexpr (ZP) {
#pragma unroll
      for (int i = 0; i < WKT; ++i) {
        f.a[i] ^= xa;
        f.b[i] ^= xb;
      }
    }
    if (s == KS - 1) {                                   // uniform: the tail moves down, zeros come in
      const int kc = 64 * s + 16 * g, sh = kc - min(kc, K - 16);
#pragma unroll
      for (int i = 0; i < WKT; ++i) {
        f.a[i] = shift_down(f.a[i], sh);
        f.b[i] = shift_down(f.b[i], sh);
      }
    }
#pragma unroll
    for (int i = 0; i < WKT; ++i)
#pragma unroll
      for (int j = 0; j < WKT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
    if constexpr (ZP) {
#pragma unroll
      for (int i = 0; i < WKT; ++i) {
        sa[i] = sum16(f.a[i], sa[i]);
        sb[i] = sum16(f.b[i], sb[i]);
      }
    }
  };
  // SPLIT: split blockIdx.z of gridDim.z, whose waves take every 8 * splits-th
  // slice (a form of its own: 3% on products of a few microseconds)
  Frag f0, f1;
  const int zs = SPLIT ? (int)blockIdx.z : 0, stride = 2 * WKW * (SPLIT ? (int)gridDim.z : 1);
  int s = 2 * (wave + WKW * zs);
  if (s < KS) load(s, f0);
  while (s < KS) {
    const bool two = s + 1 < KS;
    if (two) load(s + 1, f1);
    mul(s, f0);
    const int nx = s + stride;
    if (nx < KS) load(nx, f0);
    if (two) mul(s + 1, f1);
    s = nx;
  }
  if constexpr (ZP) {
    // lanes of one row differ in g
#pragma unroll
    for (int i = 0; i < WKT; ++i) {
      int va = sa[i], vb = sb[i];
      va += __shfl_xor(va, 16, 64);
      va += __shfl_xor(va, 32, 64);
      vb += __shfl_xor(vb, 16, 64);
      vb += __shfl_xor(vb, 32, 64);
      if (g == 0) {
        atomicAdd(&sum_a[16 * i + r16], va);
        atomicAdd(&sum_b[16 * i + r16], vb);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < WKT; ++i)
#pragma unroll
    for (int j = 0; j < WKT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((i * WKW + wave) * 16 + 4 * g + r) * WK_PITCH + 16 * j + r16] = acc[i][j][r];
  __syncthreads();
  // two outputs per thread, consecutive columns over the lanes
#pragma unroll
  for (int t = tid; t < WKB * WKB; t += 64 * WKW) {
    const int row = t / WKB, col = t % WKB, m = m0 + row, n = n0 + col;
    uint32_t a = 0u;
#pragma unroll
    for (int w = 0; w < WKW; ++w) a += (uint32_t)red[((row / 16 * WKW + w) * 16 + row % 16) * WK_PITCH + col];
    if constexpr (ZP) a += (zs == 0 ? z.kcc : 0u) + (uint32_t)z.cA * (uint32_t)sum_b[col] + (uint32_t)z.cB * (uint32_t)sum_a[row];
    if constexpr (SPLIT) {
      p.part[(((int64_t)zs * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (WKB * WKB) + t] = (int32_t)a;
      continue;
    }
    if (m >= M || n >= N) continue;
    int64_t at = o_base + (int64_t)m * N + n;
    if (e.col_blk > 0) {
      const unsigned blk = (unsigned)n / (unsigned)e.col_blk;
      at = o_base + blk * e.blk_stride + (int64_t)m * e.ld_out + (unsigned)n - blk * (unsigned)e.col_blk;
    }
    if (e.out_i32) {
      static_cast<int32_t*>(out)[at] = (int32_t)a;
    } else {
      float y = e.mode == 0 ? (float)((double)(int32_t)a * e.s_out)
                            : mul_acc_f32scale((int32_t)a, (float)(s_rows[row] * e.sB[(int64_t)n * e.sB_stride]));
      y = epi_finish(y, n, e);
      if (e.out_q8) static_cast<int8_t*>(out)[at] = (int8_t)requant(y, e);
      else static_cast<float*>(out)[at] = y;
    }
  }
}

// The splits' partial sums of a 32 x 32 tile, stored as k_qgemm_wk does.
__global__ __launch_bounds__(256) void k_wk_finish(int M, int N, int tiles_m, int tiles_n, GemmEpi e, AnyPlan p,
                                                   void* __restrict__ out) {
  int tm, tn;
  tile_of((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t step = (int64_t)gridDim.y * gridDim.x * (WKB * WKB);
  const int32_t* part = p.part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (WKB * WKB);
  void* o = static_cast<char*>(out) + blockIdx.y * p.o_step * (e.out_q8 ? 1 : 4);
  for (int t = threadIdx.x; t < WKB * WKB; t += 256) {
    const int m = tm * WKB + t / WKB, n = tn * WKB + t % WKB;
    uint32_t a = 0u;
    for (int s = 0; s < p.splits; s += 4) {
#pragma unroll
      for (int q = 0; q < 4; ++q) a += s + q < p.splits ? (uint32_t)part[(s + q) * step + t] : 0u;
    }
    if (m < M && n < N) store_out(o, (int64_t)m * N + n, (int)a, m, n, e);
  }
}

// One thread per output with byte loads: short rows are a launch and a few
// load latencies either way, and this kernel's few instructions arrive sooner
// than the tiled kernel's (any_tiny has the line).  Affine operands term by
// term: (a' + cA)(b' + cB) summed over k is the corrected sum.
template <bool ZP>
__global__ __launch_bounds__(256) void k_qgemm_tiny(const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M,
                                                    int N, int K, GemmEpi e, AffineDot z, void* __restrict__ out) {
  const int64_t idx = blockIdx.x * 256LL + threadIdx.x;
  if (idx >= (int64_t)M * N) return;
  const int64_t m = idx / N, n = idx % N;
  uint32_t s = 0;
  for (int k = 0; k < K; ++k) {
    if constexpr (ZP) {
      const int a = (int8_t)(A[m * K + k] ^ (int8_t)z.xa), b = (int8_t)(B[n * K + k] ^ (int8_t)z.xb);
      s += ((uint32_t)a + (uint32_t)z.cA) * ((uint32_t)b + (uint32_t)z.cB);
    } else {
      s += (uint32_t)((int)A[m * K + k] * (int)B[n * K + k]);
    }
  }
  store_out(out, idx, (int)s, m, n, e);
}

// Whether one thread per output serves an M x N product over rows of K bytes
// sooner than tiles.  A thread's chain is about 0.15 us a byte, the launch
// 1.2e6 multiply-adds (0.75e6 over longer rows) and 4.2e5 outputs a us; a tile
// is worth 5 ns where it is full, 3.5 with few rows and 6.6 with few columns (a
// lane's loads and stores then go one row each), and rows shorter than 16
// bytes are loaded byte by byte.  us, thread per output / tiles: 500000 x 3 x 3 8.9 / 64.8, 100000 x 1 x
// 33 8.2 / 17.1, 60000 x 10 x 15 12.9 / 20.0 and x 17 14.1 / 11.3, 300 x 300 x
// 15 5.6 / 13.4, 64 x 8192 x 15 9.7 / 13.4 and x 17 10.5 / 7.5, 4096 x 4096 x
// 3 59 / 33.  Up to 2^16 outputs a symmetric product over rows of less
// than 64 bytes stays here throughout (355 x 10 x 33, the last layer of a
// small MLP: 2 us less than a tile).
bool any_tiny(int64_t M, int64_t N, int64_t K, int64_t t64, bool affine) {
  const double mn = (double)M * (double)N, k = (double)K, t = (double)t64;
  if (mn <= 65536.0 && K < 64 && !affine) return true;
  if (K > 256 || mn >= 0x1p32 - 256) return false;
  const double chain = 3.0 + 0.15 * k, rate = mn * k / (K < 16 ? 1.2e6 : 0.75e6);
  const double thread = (chain > 5.5 ? chain : 5.5) > rate ? (chain > 5.5 ? chain : 5.5) : rate;
  const double tiles = K < 16 ? 7.0 + 0.4 * k + t * (0.0066 + 0.0006 * k)
                              : 5.6 + t * (N < 64 ? 0.0066 : M < 64 ? 0.0035 : 0.0052);
  return thread + mn / 4.2e5 < tiles;
}

#define Q8_ANY_LAUNCH(KERN, ...)                                                                                   \
  do {                                                                                                             \
    if (p.conv_cg) {                                                                                               \
      if (z) hipLaunchKernelGGL((KERN<__VA_ARGS__ true, true>), grid, block, lds, st, A, B, M, N, K, tm, tn, e, zz, p, out); \
      else hipLaunchKernelGGL((KERN<__VA_ARGS__ false, true>), grid, block, lds, st, A, B, M, N, K, tm, tn, e, zz, p, out);  \
    } else {                                                                                                       \
      if (z) hipLaunchKernelGGL((KERN<__VA_ARGS__ true, false>), grid, block, lds, st, A, B, M, N, K, tm, tn, e, zz, p, out); \
      else hipLaunchKernelGGL((KERN<__VA_ARGS__ false, false>), grid, block, lds, st, A, B, M, N, K, tm, tn, e, zz, p, out);  \
    }                                                                                                              \
  } while (0)

template <int BM, int BN, int KG>
hipError_t launch_any_tile(const int8_t* A, const int8_t* B, int M, int N, int K, const GemmEpi& e,
                           const AffineDot* z, const AnyPlan& p, void* out, hipStream_t st) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  const dim3 grid((unsigned)(tm * tn), (unsigned)p.groups), block(256 * KG);
  const unsigned lds = AnyCfg<BM, BN, KG>::LDS + (p.conv_cg ? (unsigned)K / 4 : 0u);
  note_route(p.conv_cg ? "any conv" : "any", BM, BN, KG);
  const AffineDot zz = z ? *z : AffineDot{};
  Q8_ANY_LAUNCH(k_qgemm_any, BM, BN, KG, );
  return hipGetLastError();
}

hipError_t launch_wk(const int8_t* A, const int8_t* B, int M, int N, int K, const GemmEpi& e,
                     const AffineDot* z, const AnyPlan& p, void* out, hipStream_t st) {
  const int tm = (M + WKB - 1) / WKB, tn = (N + WKB - 1) / WKB;
  const dim3 grid((unsigned)(tm * tn), (unsigned)p.groups, (unsigned)p.splits), block(64 * WKW);
  const unsigned lds = WK_LDS + (p.conv_cg ? (unsigned)K / 4 : 0u);
  note_route(p.conv_cg ? "any conv" : "any", WKB, WKB, WKW);
  const AffineDot zz = z ? *z : AffineDot{};
  if (p.splits == 1) {
    Q8_ANY_LAUNCH(k_qgemm_wk, false, );
    return hipGetLastError();
  }
  Q8_ANY_LAUNCH(k_qgemm_wk, true, );
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  note_route("any conv split", WKB, WKB, p.splits);
  hipLaunchKernelGGL(k_wk_finish, dim3((unsigned)(tm * tn), (unsigned)p.groups), dim3(256), 0, st, M, N, tm, tn, e, p, out);
  return hipGetLastError();
}
#undef Q8_ANY_LAUNCH

}  // namespace

// With fewer tiles than CUs and a long K, the time is what one CU can load
// (2, 4, 6 and 8 steps in flight take the same): the K of the tiles is spread
// over up to 8 workgroups each, at least 8 slices of 128 bytes to one, whose
// sums cost a second launch.  Whole convs of one image, us, unsplit / split: 512
// x 7 x 7 -> 16, 7 x 7 (2 tiles, K 25088) 42.3 / 17.8; 256 x 13 x 13 -> 3, 7 x 7
// (6, 12544) 21.8 / 15.1; 1024 x 14 x 14 -> 10, 3 x 3 (7, 9216) 19.2 / 15.5; 256
// x 28 x 28 -> 3, 5 x 5 (25, 6400) 14.8 / 14.3; 512 x 7 x 7 -> 512, 3 x 3 (32,
// 4608) 15.5 / 13.7, but 192 x 13 x 13 -> 64, 5 x 5 (12, 4800) 12.8 / 13.9 and 256
// x 14 x 14 -> 256, 3 x 3 (56, 2304) 11.9 / 13.7.
int any_splits(int64_t M, int64_t N, int64_t K, int64_t groups) {
  const int64_t cus = cu_count() > 0 ? cu_count() : 256, t32 = groups * ((M + 31) / 32) * ((N + 31) / 32);
  if (K < ANY_SPLIT_K || 2 * t32 > cus) return 1;
  int64_t s = cus / t32;
  s = s < 8 ? s : 8;
  s = s < K / 1024 ? s : K / 1024;
  return (int)s;
}
size_t any_part_bytes(int64_t M, int64_t N, int64_t groups, int splits) {
  return splits > 1 ? (size_t)splits * (size_t)groups * (size_t)((M + 31) / 32) * (size_t)((N + 31) / 32) * WKB * WKB * 4 : 0;
}

hipError_t launch_gemm_any(const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t K,
                           const GemmEpi& e, const AffineDot* z, const AnyPlan& p, void* out, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  if (p.conv_cg && (p.conv_cg % 16 != 0 || K % 16 != 0 || K <= 0 || K > ANY_CONV_MAX_K)) return hipErrorInvalidValue;
  const int64_t cus = cu_count() > 0 ? cu_count() : 256;
  const int64_t t128 = p.groups * ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t t64 = p.groups * ((M + 63) / 64) * ((N + 63) / 64);
  // a launch has fewer than 2^32 threads: 2^24 - 1 tiles of 256, or as many
  // outputs of a thread each (one row by 2^30 columns); and the tiles count K
  // in 31 bits, stages past its end included
  const bool plain = !p.conv_cg && p.groups == 1 && p.lda == K && p.ldb == K;
  const bool wide = t64 >= ((int64_t)1 << 24) || K > INT32_MAX - 4096;
  if (p.groups > 65535 || (wide && !(plain && (double)M * (double)N < 0x1p32 - 256))) return hipErrorInvalidValue;
  const int m = (int)M, n = (int)N, k = (int)K;
  if (plain && (wide || any_tiny(M, N, K, t64, z != nullptr))) {
    note_route("tiny");
    const dim3 grid((unsigned)((M * N + 255) / 256));
    if (z) hipLaunchKernelGGL(k_qgemm_tiny<true>, grid, dim3(256), 0, st, A, B, m, n, k, e, *z, out);
    else hipLaunchKernelGGL(k_qgemm_tiny<false>, grid, dim3(256), 0, st, A, B, m, n, k, e, AffineDot{}, out);
    return hipGetLastError();
  }
  // Up to one 64 x 64 tile per CU: four K groups each (512 x 7 x 7 conv, 200
  // tiles of 36 stages: 35 us with one group, 26 with two, 22 with four); up
  // to two per CU: two (392 tiles, 18 stages: 25 / 21 / 25 us).  Above that
  // the tiles fill the chip, and 128 x 128 halves the bytes per operation
  // (4096 x 4096 x 1001: 43 us, 64 x 64 60 us) where the product has the
  // rows for it and stages enough to cover its longer fill (1183 x 3917 x
  // 319, three stages: 22 against 19 us), in two K groups while a CU gets at
  // most one (2048 x 2048 x 8192: 76 -> 60 us).
  const int KT = (k + AK - 1) / AK;
  const bool big = M > 64 && N > 64 && KT >= 6;
  const int64_t t32 = p.groups * ((M + 31) / 32) * ((N + 31) / 32);
  if (p.splits > 1 && (t32 > cus || K < 16 || p.part == nullptr)) return hipErrorInvalidValue;
  if (t32 <= cus && K >= 16) return launch_wk(A, B, m, n, k, e, z, p, out, st);
  if (KT > 2) {
    if (t64 <= cus) return launch_any_tile<64, 64, 4>(A, B, m, n, k, e, z, p, out, st);
    if (t64 <= 2 * cus) return launch_any_tile<64, 64, 2>(A, B, m, n, k, e, z, p, out, st);
  }
  if (big && t128 > cus) return launch_any_tile<128, 128, 1>(A, B, m, n, k, e, z, p, out, st);
  if (big && 2 * t128 > cus) return launch_any_tile<128, 128, 2>(A, B, m, n, k, e, z, p, out, st);
  return launch_any_tile<64, 64, 1>(A, B, m, n, k, e, z, p, out, st);
}

hipError_t setup_any_attributes() {
  hipError_t err = hipSuccess;
  auto set = [&](const void* k, int bytes) {
    if (err == hipSuccess) err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  };
#define Q8_SET_ANY(BM, BN, KG)                                                                          \
  set(reinterpret_cast<const void*>(k_qgemm_any<BM, BN, KG, false, false>), AnyCfg<BM, BN, KG>::LDS);   \
  set(reinterpret_cast<const void*>(k_qgemm_any<BM, BN, KG, true, false>), AnyCfg<BM, BN, KG>::LDS);    \
  set(reinterpret_cast<const void*>(k_qgemm_any<BM, BN, KG, false, true>), AnyCfg<BM, BN, KG>::LDS + ANY_CONV_MAX_K / 4); \
  set(reinterpret_cast<const void*>(k_qgemm_any<BM, BN, KG, true, true>), AnyCfg<BM, BN, KG>::LDS + ANY_CONV_MAX_K / 4);
  Q8_SET_ANY(128, 128, 1)
  Q8_SET_ANY(128, 128, 2)
  Q8_SET_ANY(64, 64, 1)
  Q8_SET_ANY(64, 64, 2)
  Q8_SET_ANY(64, 64, 4)
#undef Q8_SET_ANY
#define Q8_SET_WK(SPLIT)                                                                     \
  set(reinterpret_cast<const void*>(k_qgemm_wk<SPLIT, false, false>), WK_LDS);                   \
  set(reinterpret_cast<const void*>(k_qgemm_wk<SPLIT, true, false>), WK_LDS);                    \
  set(reinterpret_cast<const void*>(k_qgemm_wk<SPLIT, false, true>), WK_LDS + ANY_CONV_MAX_K / 4); \
  set(reinterpret_cast<const void*>(k_qgemm_wk<SPLIT, true, true>), WK_LDS + ANY_CONV_MAX_K / 4);
  Q8_SET_WK(false)
  Q8_SET_WK(true)
#undef Q8_SET_WK
  return err;
}

}  // namespace q8
