// q8_gemm_ring.hip -- the int8 MFMA GEMM for a few dozen to a few hundred
// tokens: no more tiles than the chip has CUs, so a workgroup has its CU to
// itself and nothing but its own copies in flight to hide load latency.
//
// What bounds k_qgemm there: its two-stage ring keeps one stage in flight per
// workgroup, and a 64 x 64 tile walks K / 128 stages one after another at a
// memory latency each (64 x 11008 x 4096: 172 tiles, 32 stages, 19.3 us for
// the 45 MB of weights that a streaming read takes 8 us for).  Here the CU's
// whole LDS is the ring: KG groups of waves take every KG-th stage, each with
// NB stages (direct-to-LDS copies, in the swizzled layout of k_qgemm), NB - 1
// of them in flight, and the groups' partial sums meet in LDS (tile_epilogue;
// int32 addition does not depend on the order).  One barrier per stage of
// each group, shared by all.
#include "q8_device.h"
#include "q8_epilogue.h"
#include "q8_gemm_tile.h"
#include "q8_internal.h"

namespace q8 {

namespace {

template <int BM, int BN, int GM, int GN, int KG, int NB>
struct RingCfg {
  static constexpr int WAVES = GM * GN;                 // per group
  static constexpr int WM = BM / GM, WN = BN / GN;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int A_BYTES = BM * AK;
  static constexpr int STAGE = (BM + BN) * AK;
  static constexpr int RING = NB * STAGE;
  static constexpr int LDS = KG * RING + 8 * BM;        // + row scales
  static constexpr int NA = BM / 8 / WAVES, NBC = BN / 8 / WAVES, NV = NA + NBC;   // 8-row copies per wave and stage
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && TM >= 1 && TN >= 1 && LDS <= 160 * 1024, "tile");
};

constexpr uint32_t PAST = 0x80000000u;                  // past every buffer's num_records: reads zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc8(const int8_t* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base), (short)0, (int)bytes, 0x00020000);
}

// 16 bytes per lane from buffer offset voff to LDS dst + 16 * lane.
__device__ __forceinline__ void copy_lds(__amdgpu_buffer_rsrc_t r, int8_t* dst, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, 0, 0, 0);
}

// All but this wave's N most recent copies have landed (loads complete in
// order) and its LDS reads have returned, then all waves meet.  One asm
// statement: the compiler's own wait for the reads may come later.
template <int N>
__device__ __forceinline__ void wait_stage() {
  static_assert(N >= 0 && N <= 63, "vmcnt immediate");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int BM, int BN, int GM, int GN, int KG, int NB>
__global__ __launch_bounds__(64 * GM * GN * KG, 1)
void k_qgemm_ring(const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M, int N, int K,
                  int tiles_m, int tiles_n, GemmEpi e, void* __restrict__ out) {
  using C = RingCfg<BM, BN, GM, GN, KG, NB>;
  extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
  double* s_rows = reinterpret_cast<double*>(lds + KG * C::RING);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wv % C::WAVES, grp = wv / C::WAVES;
  int8_t* const ring = lds + grp * C::RING;
  int tm, tn;
  tile_of((int)blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int rows_a = min(BM, M - m0), rows_b = min(BN, N - n0);
  double sr = 0.0;
  if (tid < BM && tid < rows_a && e.mode == 1 && !e.out_i32) sr = e.sA[(int64_t)(m0 + tid) * e.sA_stride];

  // Copy plan: a wave fills its share of the stage's rows, 8 rows x 128 B per
  // instruction; lane l lands in row 8 j + l / 8 at chunk l % 8 and fetches
  // logical chunk (l % 8) ^ swz(row).  Rows past the edge and chunks past K
  // read past the buffer's end: zeros, without memory traffic.
  const int8_t* Ab = A + (int64_t)m0 * K;
  const int8_t* Bb = B + (int64_t)n0 * K;
  uint32_t offa[C::NA], offb[C::NBC];
  int kca[C::NA], kcb[C::NBC];
#pragma unroll
  for (int j = 0; j < C::NA; ++j) {
    const int row = (wave * C::NA + j) * 8 + (lane >> 3);
    kca[j] = 16 * ((lane & 7) ^ swz(row));
    offa[j] = row < rows_a ? (uint32_t)(row * K + kca[j]) : PAST;
  }
#pragma unroll
  for (int j = 0; j < C::NBC; ++j) {
    const int row = (wave * C::NBC + j) * 8 + (lane >> 3);
    kcb[j] = 16 * ((lane & 7) ^ swz(row));
    offb[j] = row < rows_b ? (uint32_t)(row * K + kcb[j]) : PAST;
  }
  const uint32_t bytes_a = (uint32_t)rows_a * (uint32_t)K, bytes_b = (uint32_t)rows_b * (uint32_t)K;
  const int KT = (K + AK - 1) / AK;
  // Tiles start at different stages: in step, they would all read one 128-byte
  // column of rows a power of two apart.  (17 x 22016 x 4096: 30.4 -> 27.2 us;
  // up to 3% elsewhere.)
  const int rot = (int)((unsigned)(5 * tn) % (unsigned)KT);
  auto issue = [&](int i, int buf) {
    const int kt = grp + i * KG;
    const bool live = kt < KT;                          // past the end: zeros into a stage nobody adds to
    const int kr = kt + rot;
    const int kb = live ? (kr >= KT ? kr - KT : kr) * AK : 0;
    const bool tail = kb + AK > K;
    const __amdgpu_buffer_rsrc_t ra = rsrc8(Ab + kb, live ? bytes_a - (uint32_t)kb : 0u);
    const __amdgpu_buffer_rsrc_t rb = rsrc8(Bb + kb, live ? bytes_b - (uint32_t)kb : 0u);
    int8_t* st = ring + buf * C::STAGE;
#pragma unroll
    for (int j = 0; j < C::NA; ++j)
      copy_lds(ra, st + (wave * C::NA + j) * 8 * AK, tail && kb + kca[j] >= K ? PAST : offa[j]);
#pragma unroll
    for (int j = 0; j < C::NBC; ++j)
      copy_lds(rb, st + C::A_BYTES + (wave * C::NBC + j) * 8 * AK, tail && kb + kcb[j] >= K ? PAST : offb[j]);
  };

  const int wm = (wave / GN) * C::WM, wn = (wave % GN) * C::WN;
  v16i acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

#pragma unroll
  for (int i = 0; i < NB - 1; ++i) issue(i, i);
  if (tid < BM) s_rows[tid] = sr;
  const int NI = (KT + KG - 1) / KG;                    // every group runs as many: the barriers are the workgroup's
  int buf = 0;
  for (int i = 0; i < NI; ++i) {
    wait_stage<(NB - 2) * C::NV>();       // stage i is there, the stage before it no longer read
    issue(i + NB - 1, buf == 0 ? NB - 1 : buf - 1);
    mfma_stage<C>(ring + buf * C::STAGE, wm, wn, lane, acc);
    buf = buf + 1 == NB ? 0 : buf + 1;
  }
  // the zero-filling copies past the end have landed before the epilogue
  // reuses the ring
  wait_stage<0>();
  tile_epilogue<C, KG, false>(acc, lds, s_rows, nullptr, nullptr, wave, grp, lane, m0, n0, wm, wn, M, N, 0, e,
                              AffineDot{}, AnyPlan{}, out);
}

template <int BM, int BN, int GM, int GN, int KG, int NB>
hipError_t launch_ring_tile(const int8_t* A, const int8_t* B, int M, int N, int K, const GemmEpi& e, void* out,
                            hipStream_t st) {
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  note_route("ring", BM, BN, KG);
  hipLaunchKernelGGL((k_qgemm_ring<BM, BN, GM, GN, KG, NB>), dim3((unsigned)(tm * tn)), dim3(64 * GM * GN * KG),
                     (unsigned)(RingCfg<BM, BN, GM, GN, KG, NB>::LDS), st, A, B, M, N, K, tm, tn, e, out);
  return hipGetLastError();
}

}  // namespace

#define Q8_RING_TILES(X) \
  X(32, 32, 1, 1, 4, 4)    \
  X(64, 32, 2, 1, 4, 3)    \
  X(32, 64, 1, 2, 4, 3)    \
  X(64, 64, 2, 2, 2, 4)    \
  X(128, 64, 2, 2, 2, 3)   \
  X(64, 128, 2, 2, 2, 3)   \
  X(128, 128, 2, 2, 1, 4)

// The smallest tile that leaves every tile a CU of its own (a second round
// costs a workgroup's whole time again, while more and smaller tiles spread
// the weights' load over more CUs), -1 where none does, and from the tile's
// `stages` on: filling the ring and adding up the groups cost the same however
// short K is, and the larger the tile the more MFMAs k_qgemm hides its copies
// behind.  Time against k_qgemm with the weights in the MALL / in HBM, median
// over 1 to 51 products of M 17..2048, N 64..32000 at K = 128 x stages:
//   32 x 32     3: 1.00 / 1.01    4: 0.92 / 0.91    8: 0.72 / 0.72   32: 0.36 / 0.35
//   64 x 32     4: 0.95 / 0.95    6: 0.89 / 0.88    8: 0.78 / 0.77   32: 0.47 / 0.40
//   32 x 64     3: 0.99 / 0.97    4: 0.90 / 0.90    8: 0.79 / 0.68   32: 0.54 / 0.46
//   64 x 64     6: 0.99 / 0.98    8: 0.93 / 0.92   16: 0.76 / 0.67   32: 0.64 / 0.52
//   128 x 64   12: 1.04 / 0.92   16: 0.98 / 0.80   20: 0.92 / 0.83   32: 0.85 / 0.66
//   64 x 128   12: 1.03 / 0.89   16: 0.98 / 0.87   20: 0.97 / 0.86   32: 0.77 / 0.78
//   128 x 128  16: 1.38 / 1.14   32: 1.16 / 0.92   48: 1.03 / 0.86   86: 0.89 / 0.78
// (64 x 32 waits for 6: weights still in L2 take 1.07 at 4.)  One row of 128 x
// 128 tiles, 90 MB of weights and more, is bound by their load sooner: 128 x
// 32000, 32 stages, 0.86 / 0.83.
int gemm_ring_tile(int64_t M, int64_t N, int64_t K) {
  static const struct { int bm, bn, stages; } tiles[] = {{32, 32, 4},   {64, 32, 6},    {32, 64, 4},  {64, 64, 8},
                                                         {128, 64, 20}, {64, 128, 16}, {128, 128, 48}};
  const int64_t cus = cu_count() > 0 ? cu_count() : 256, KT = (K + AK - 1) / AK;
  for (int t = 0; t < 7; ++t) {
    if ((t == 2 && M > 32) || (t == 4 && M <= 64)) continue;   // rows of padding
    if (((M + tiles[t].bm - 1) / tiles[t].bm) * ((N + tiles[t].bn - 1) / tiles[t].bn) > cus) continue;
    return KT >= (t == 6 && M <= 128 ? 32 : tiles[t].stages) ? t : -1;
  }
  return -1;
}

hipError_t launch_gemm_ring(const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t K,
                            const GemmEpi& e, int tile, void* out, hipStream_t st) {
  int t = 0;
#define Q8_RING_CASE(...) if (tile == t++) return launch_ring_tile<__VA_ARGS__>(A, B, (int)M, (int)N, (int)K, e, out, st);
  Q8_RING_TILES(Q8_RING_CASE)
#undef Q8_RING_CASE
  return hipErrorInvalidValue;
}

hipError_t setup_ring_attributes() {
  hipError_t err = hipSuccess;
#define Q8_RING_SET(...)                                                                              \
  if (err == hipSuccess)                                                                              \
    err = hipFuncSetAttribute(reinterpret_cast<const void*>(k_qgemm_ring<__VA_ARGS__>),               \
                              hipFuncAttributeMaxDynamicSharedMemorySize, RingCfg<__VA_ARGS__>::LDS);
  Q8_RING_TILES(Q8_RING_SET)
#undef Q8_RING_SET
  return err;
}

}  // namespace q8
