// q8_conv.hip -- quantized_conv for gfx950 (CDNA4).
//
// The reference op (src/compiler/ir/graph/ops/quantization.ts:156-190,
// lowered by rules/quantization.ts:44-62 through buildConvNest,
// src/compiler/passes/lowering/lowering_registry.ts:335-449) is an exact
// int32 convolution of int8 operands in NC(spatial) / OI(spatial) layout,
// with strides, [lo, hi] padding, dilation and groups; a tap whose input
// coordinate lies in the padding adds 0.
//
// Paths, all exact:
//   * GEMM form for contractions of 64 or more (Kc = Cg * prod(K)), and for
//     large products over shorter ones:
//     out[n, g*Og : (g+1)*Og, :] = W_g [Og, Kc] x (receptive fields)^T -- the
//     weight is the A operand, so the [Og, P] result is already the
//     NC(spatial) output block and the dequant epilogue is fused as in
//     q8_gemm.  Images go in batches: one GEMM computes [Og, nb * P], its
//     epilogue storing column n * P + p of the product at image n, position
//     p (column-blocked output), and the groups are a second grid dimension,
//     so a grouped conv is two launches, not two per group (two per group
//     where each group's product fills the chip by itself).  The receptive
//     fields come one of two ways:
//       - channels per group a multiple of 16: the input is transposed to a
//         padded channel-last frame and the contraction is taken tap-major
//         (k = tap * Cg + c, the weight permuted to match, in the same launch
//         as the frame where it was not prepacked): each 16 bytes of a
//         column are 16 channels of one frame position, which the GEMM reads
//         where they lie.  Integer addition does not depend on the order of
//         the taps, so the sums are the same;
//       - otherwise a matrix (im2col) by a byte gather in the OI(spatial)
//         order (ic-major, then kernel positions).
//     Zero points and ui8 operands run the same paths: bytes are flipped on
//     the way (u - 128), padding holds the input's zero point, and the GEMM
//     corrects its sums with the operands' row sums (q8_zp.hip states the
//     identity).  28 x 28 x 128 at batch 32 with ui8 input: 2700 us one
//     thread per output, 21.4 us here.
//   * a direct kernel (one thread per output element) for other short
//     contractions -- depthwise and other small-group convolutions -- for an
//     input zero point outside its type, and for calls whose workspace is so
//     small that the GEMM's passes do not fit or pay.
// conv_plan decides the route, the images and groups of a pass and every byte
// of the workspace that is written.
// Spatial ranks 1..3 share the code: unused trailing dimensions have size 1,
// stride 1, no padding and dilation 1.
#include "q8_device.h"
#include "q8_internal.h"

namespace q8 {

// im2col tile: I2C_TP output positions x I2C_TK contraction bytes of one
// image (contraction index k: ic-major, then kernel positions in row-major
// order -- the OI(spatial) weight's own order), zero past Kc.  Gather: the
// lanes of a wave take consecutive positions and one run of 32 contraction
// indices per wave, so each byte load of a wave reads neighbouring input
// bytes (with stride 1, consecutive bytes of a row); the tile is transposed
// through LDS so that the stores are 128-byte row segments of the matrix.
// Affine operands: ui8 bytes are flipped (`flip` = 0x80), and a tap in the
// padding holds `fill`, the input's zero point as an int8 code, so that its
// (x - zp) is 0; both 0 in the symmetric scheme.
constexpr int I2C_TP = 64, I2C_TK = 128, I2C_PITCH = I2C_TK + 16;

template <bool AFFINE>
__global__ __launch_bounds__(256) void k_im2col(const int8_t* __restrict__ x, ConvGeom G,
                                                int64_t n0, int64_t g, uint32_t flip, uint32_t fill,
                                                int8_t* __restrict__ col) {
  __shared__ __align__(16) uint32_t tile[I2C_TP * I2C_PITCH / 4];
  // blockIdx.y: image n0 + y of a batch, written at matrix rows y * P ..
  // blockIdx.z: group g + z, a matrix of its own
  const int64_t n = n0 + blockIdx.y;
  g += blockIdx.z;
  col += ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * G.Pn * G.Kc16;
  const int tk = (G.Kc16 + I2C_TK - 1) / I2C_TK;
  const int64_t pt = blockIdx.x / tk;
  const int k0 = (int)(blockIdx.x - pt * tk) * I2C_TK;
  const int64_t p0 = pt * I2C_TP;
  const int pl = threadIdx.x & 63;
  const int kq = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the wave's 32 indices
  const int64_t p = p0 + pl;
  uint32_t w[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  int k = k0 + 32 * kq;
  if (p < G.Pn && k < G.Kc) {
    // output coordinates of p and the input coordinates of tap (0, 0, 0)
    const int o2 = (int)(p % G.P[2]);
    const int64_t t = p / G.P[2];
    const int o1 = (int)(t % G.P[1]);
    const int o0 = (int)(t / G.P[1]);
    const int b0 = (int)(o0 * G.st[0] - G.lo[0]);
    const int b1 = (int)(o1 * G.st[1] - G.lo[1]);
    const int b2 = (int)(o2 * G.st[2] - G.lo[2]);
    // contraction coordinates of the first byte, advanced with carries
    int ic = k / G.Kn;
    int r = k - ic * G.Kn;
    int k2 = r % G.K[2];
    r /= G.K[2];
    int k1 = r % G.K[1];
    int k0i = r / G.K[1];
    const int8_t* xg = x + (n * G.C + g * G.Cg) * G.Sn;
    // The contraction coordinates are the wave's own (uniform), advanced
    // with branch-free carries; a lane whose tap falls in the padding (or
    // past Kc) loads the plane's first byte and keeps 0.  The loop body is
    // one basic block, so its 32 loads issue back to back.
    uint32_t v[32];
#pragma unroll
    for (int b = 0; b < 32; ++b) {
      const int s0 = b0 + k0i * (int)G.dl[0];
      const int s1 = b1 + k1 * (int)G.dl[1];
      const int s2 = b2 + k2 * (int)G.dl[2];
      const bool kin = k + b < G.Kc;                       // uniform
      const bool in = kin && (unsigned)s0 < (unsigned)G.S[0] && (unsigned)s1 < (unsigned)G.S[1] &&
                      (unsigned)s2 < (unsigned)G.S[2];
      // offset in the plane, computed unconditionally (unsigned: no overflow
      // for a tap outside the image) and selected, so that no branch forms
      const uint32_t sp = ((uint32_t)s0 * (uint32_t)G.S[1] + (uint32_t)s1) * (uint32_t)G.S[2] + (uint32_t)s2;
      const int8_t* plane = xg + (int64_t)(kin ? ic : 0) * G.Sn;
      const uint32_t raw = (uint8_t)plane[in ? sp : 0u];   // in bounds either way
      v[b] = AFFINE ? (in ? raw ^ flip : (kin ? fill : 0u)) : (in ? raw : 0u);
      ++k2;
      const bool c2 = k2 == G.K[2];
      k2 = c2 ? 0 : k2;
      k1 += c2;
      const bool c1 = k1 == G.K[1];
      k1 = c1 ? 0 : k1;
      k0i += c1;
      const bool c0 = k0i == G.K[0];
      k0i = c0 ? 0 : k0i;
      ic += c0;
    }
#pragma unroll
    for (int b = 0; b < 32; ++b) w[b >> 2] |= v[b] << (8 * (b & 3));
  }
  uint32_t* trow = tile + (pl * I2C_PITCH + 32 * kq) / 4;
  reinterpret_cast<v4i*>(trow)[0] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
  reinterpret_cast<v4i*>(trow)[1] = v4i{(int)w[4], (int)w[5], (int)w[6], (int)w[7]};
  __syncthreads();
  // store: 8 lanes per 128-byte row segment, 32 rows per pass
  const int ch = threadIdx.x & 7;
#pragma unroll
  for (int pass = 0; pass < I2C_TP / 32; ++pass) {
    const int row = pass * 32 + (threadIdx.x >> 3);
    const int64_t prow = p0 + row;
    const int kk = k0 + 16 * ch;
    if (prow < G.Pn && kk < G.Kc16)
      *reinterpret_cast<v4i*>(col + prow * G.Kc16 + kk) =
          *reinterpret_cast<const v4i*>(tile + (row * I2C_PITCH + 16 * ch) / 4);
  }
}

// Launch grid of k_im2col for nb images: x = position tiles * contraction
// tiles, y = nb.  False if it does not fit a launch.
static bool im2col_grid(const ConvGeom& G, int64_t nb, dim3* grid) {
  const int64_t tiles = ((G.Pn + I2C_TP - 1) / I2C_TP) * ((G.Kc16 + I2C_TK - 1) / I2C_TK);
  if (tiles * 256 >= ((int64_t)1 << 32) || nb > 65535) return false;
  *grid = dim3((unsigned)tiles, (unsigned)nb);
  return true;
}

// Weight rows [O, Kc] -> [O, Kc16] with zero padding.
__global__ __launch_bounds__(256) void k_pad_rows(const int8_t* __restrict__ w, int64_t O, int64_t Kc,
                                                  int64_t Kc16, int8_t* __restrict__ wp) {
  const int64_t i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= O * Kc16) return;
  const int64_t o = i / Kc16, k = i - o * Kc16;
  wp[i] = k < Kc ? w[o * Kc + k] : (int8_t)0;
}

// ---------------------------------------------------------------- channel-last path
// For Cg a multiple of 16 the contraction is taken tap-major, k = t * Cg + c
// (t: kernel position in row-major order, c: input channel of the group):
// the same products summed in another order, and int32 wrap-around addition
// does not depend on the order.  The input goes once to a padded
// channel-last frame xp[y][e][c], e over E0 x E1 x E2 with
// E_i = (P_i - 1) * st_i + (K_i - 1) * dl_i + 1 (input coordinate e_i - lo_i),
// so that the receptive field of output p at tap t is the Cg contiguous
// bytes xp[y][e(p) + off(t)][:] and the GEMM reads them as they lie.
struct ConvFrame {
  int E[3];
  int64_t Ep;   // E0 * E1 * E2
};

// The frame of nb images and Cb channels from channel c0 on:
// xp[y][e][c] = x[n0 + y][c0 + c][e - lo], `fill` outside the image, bytes
// flipped by `flip` (see k_im2col).  A workgroup transposes 64 frame
// positions x 64 channels through LDS: in the gather each thread takes one
// position and 16 channels, the lanes of a wave consecutive positions, so
// each byte load of a wave reads neighbouring bytes of one channel plane; in
// the store the lanes take consecutive 16-byte chunks of the frame rows.
constexpr int FR_PITCH = 64 + 16;   // LDS row: 64 channel bytes + pad
struct FrameJob {
  int64_t n0;
  int c0, Cb;
  uint32_t flip, fill;
};
template <bool AFFINE>
__device__ __forceinline__ void frame_tile(const int8_t* __restrict__ x, const ConvGeom& G, const ConvFrame& F,
                                           const FrameJob& J, uint32_t* tile, int64_t y, int eb, int ct,
                                           int8_t* __restrict__ xp) {
  const int el = (int)(threadIdx.x & 63), e = eb + el, Ep = (int)F.Ep;
  const int cs = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the wave's 16-channel slice
  bool in = false;
  uint32_t sp = 0u;
  if (e < Ep) {
    const int q = e / F.E[2], e2 = e - q * F.E[2];
    const int e0 = q / F.E[1], e1 = q - e0 * F.E[1];
    const int s0 = e0 - (int)G.lo[0], s1 = e1 - (int)G.lo[1], s2 = e2 - (int)G.lo[2];
    in = (unsigned)s0 < (unsigned)G.S[0] && (unsigned)s1 < (unsigned)G.S[1] &&
         (unsigned)s2 < (unsigned)G.S[2];
    // a position in the padding (or past the frame) reads the plane's
    // first byte and keeps the fill
    sp = in ? ((uint32_t)s0 * (uint32_t)G.S[1] + (uint32_t)s1) * (uint32_t)G.S[2] + (uint32_t)s2 : 0u;
  }
  const int c = ct + 16 * cs;
  uint32_t w4[4] = {0u, 0u, 0u, 0u};
  if (c < J.Cb) {
    const int8_t* sc = x + ((J.n0 + y) * G.C + J.c0 + c) * G.Sn + sp;
    uint32_t v[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) v[b] = (uint8_t)sc[(int64_t)b * G.Sn];
#pragma unroll
    for (int b = 0; b < 16; ++b) w4[b >> 2] |= (AFFINE ? (in ? v[b] ^ J.flip : J.fill) : (in ? v[b] : 0u)) << (8 * (b & 3));
  }
  reinterpret_cast<v4i*>(tile + (el * FR_PITCH + 16 * cs) / 4)[0] =
      v4i{(int)w4[0], (int)w4[1], (int)w4[2], (int)w4[3]};
  __syncthreads();
  // store: chunk ch of row r; 4 chunks per row of this channel tile
  const int cw = J.Cb - ct < 64 ? (J.Cb - ct) >> 4 : 4;   // chunks in this tile
  for (int i = threadIdx.x; i < 64 * cw; i += 256) {
    const int r = i / cw, ch = i - r * cw;
    if (eb + r < Ep)
      *reinterpret_cast<v4i*>(xp + (y * F.Ep + eb + r) * J.Cb + ct + 16 * ch) =
          *reinterpret_cast<const v4i*>(tile + (r * FR_PITCH + 16 * ch) / 4);
  }
}

// wt[o][t * Cg + c] = w[o][c * Kn + t]: the OI(spatial) weight with its
// contraction in tap-major order.  A slice is 16 channels of one output
// channel o (slice s = o * (Cg / 16) + c / 16); its 16 * Kn weight bytes are
// contiguous, and so are those of consecutive slices.  A workgroup stages
// `ns` consecutive slices in LDS with 16-byte loads, then writes their
// ns * Kn 16-byte chunks wt[o][t * Cg + c0 .. + 16], tap-major so that
// neighbouring lanes write neighbouring chunks.  ns * Kn <= WT_CHUNKS.
constexpr int WT_CHUNKS = 1024;
__device__ __forceinline__ void weight_taps(const int8_t* __restrict__ w, int64_t nslices, int Cg, int Kn,
                                            int ns, int64_t blk, uint8_t* buf, int8_t* __restrict__ wt) {
  const int64_t Kc = (int64_t)Cg * Kn;
  const int slices = Cg >> 4;
  const int64_t s0 = blk * ns;
  const int n = (int)(nslices - s0 < ns ? nslices - s0 : ns);      // slices of this workgroup
  const int8_t* src = w + s0 * 16 * Kn;                            // any byte address
  for (int i = threadIdx.x; i < n * Kn; i += 256) reinterpret_cast<v4i*>(buf)[i] = load16_any(src + 16 * (int64_t)i);
  __syncthreads();
  for (int i = threadIdx.x; i < n * Kn; i += 256) {
    const int t = i / n, sl = i - t * n;
    uint32_t w4[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 0; b < 16; ++b) w4[b >> 2] |= (uint32_t)buf[(sl * 16 + b) * Kn + t] << (8 * (b & 3));
    const int64_t s = s0 + sl;
    const int64_t o = s / slices;
    const int c0 = (int)(s - o * slices) * 16;
    *reinterpret_cast<v4i*>(wt + o * Kc + (int64_t)t * Cg + c0) =
        v4i{(int)w4[0], (int)w4[1], (int)w4[2], (int)w4[3]};
  }
}

__global__ __launch_bounds__(256) void k_conv_weight_taps(const int8_t* __restrict__ w, int64_t nslices,
                                                          int Cg, int Kn, int ns,
                                                          int8_t* __restrict__ wt) {
  __shared__ __align__(16) uint8_t buf[16 * WT_CHUNKS];
  weight_taps(w, nslices, Cg, Kn, ns, blockIdx.x, buf, wt);
}

// The frame of a batch and, for a weight that was not prepacked, its
// tap-major form in one launch: the first nb * etiles * ctiles workgroups
// transpose the frame, the rest the weight.  The two do not depend on each
// other and each alone is a launch's fixed cost.
template <bool AFFINE>
__global__ __launch_bounds__(256) void k_conv_prep(const int8_t* __restrict__ x, ConvGeom G, ConvFrame F,
                                                   FrameJob J, int64_t nb, int etiles, int8_t* __restrict__ xp,
                                                   const int8_t* __restrict__ w, int64_t nslices, int ns,
                                                   int8_t* __restrict__ wt) {
  __shared__ __align__(16) uint8_t buf[16 * WT_CHUNKS];
  const int64_t nfr = nb * etiles * ((J.Cb + 63) / 64), id = blockIdx.x;
  if (id >= nfr) {   // uniform
    weight_taps(w, nslices, G.Cg, G.Kn, ns, id - nfr, buf, wt);
    return;
  }
  const unsigned q = (unsigned)id / (unsigned)etiles, ct = q / (unsigned)nb;
  frame_tile<AFFINE>(x, G, F, J, reinterpret_cast<uint32_t*>(buf), q - ct * (unsigned)nb,
                     64 * (int)((unsigned)id - q * (unsigned)etiles), 64 * (int)ct, xp);
}
template <bool AFFINE>
__global__ __launch_bounds__(256) void k_conv_to_frame(const int8_t* __restrict__ x, ConvGeom G, ConvFrame F,
                                                       FrameJob J, int8_t* __restrict__ xp) {
  __shared__ __align__(16) uint32_t tile[64 * FR_PITCH / 4];
  frame_tile<AFFINE>(x, G, F, J, tile, blockIdx.y, 64 * (int)blockIdx.x, 64 * (int)blockIdx.z, xp);
}

// Direct form: one thread per output element, taps in the reference's
// order (ic, then kernel positions), int32 wrap-around sum of
// (x - zpx) * (w - zpw) over the taps inside the image (a padded tap adds
// 0), operands read as i8 or ui8.
__global__ __launch_bounds__(256) void k_conv_direct(const int8_t* __restrict__ x,
                                                     const int8_t* __restrict__ w, ConvGeom G,
                                                     GemmEpi e, void* __restrict__ out) {
  const int64_t idx = blockIdx.x * 256LL + threadIdx.x;
  const int64_t total = G.N * G.O * G.Pn;
  if (idx >= total) return;
  const int64_t p = idx % G.Pn;
  const int64_t no = idx / G.Pn;
  const int64_t o = no % G.O, n = no / G.O;
  const int64_t g = o / G.Og;
  const int o2 = (int)(p % G.P[2]);
  const int64_t t = p / G.P[2];
  const int o1 = (int)(t % G.P[1]);
  const int o0 = (int)(t / G.P[1]);
  const int8_t* xg = x + (n * G.C + g * G.Cg) * G.Sn;
  const int8_t* wo = w + o * (int64_t)G.Kc;
  uint32_t acc = 0;
  for (int ic = 0; ic < G.Cg; ++ic) {
    const int8_t* xc = xg + (int64_t)ic * G.Sn;
    const int8_t* wc = wo + (int64_t)ic * G.Kn;
    for (int k0 = 0; k0 < G.K[0]; ++k0) {
      const int64_t s0 = (int64_t)o0 * G.st[0] + (int64_t)k0 * G.dl[0] - G.lo[0];
      if (s0 < 0 || s0 >= G.S[0]) continue;
      for (int k1 = 0; k1 < G.K[1]; ++k1) {
        const int64_t s1 = (int64_t)o1 * G.st[1] + (int64_t)k1 * G.dl[1] - G.lo[1];
        if (s1 < 0 || s1 >= G.S[1]) continue;
        for (int k2 = 0; k2 < G.K[2]; ++k2) {
          const int64_t s2 = (int64_t)o2 * G.st[2] + (int64_t)k2 * G.dl[2] - G.lo[2];
          if (s2 < 0 || s2 >= G.S[2]) continue;
          const int64_t xi = (s0 * G.S[1] + s1) * G.S[2] + s2;
          const int64_t wi = (k0 * G.K[1] + k1) * G.K[2] + k2;
          const int xv = G.x_u8 ? (int)reinterpret_cast<const uint8_t*>(xc)[xi] : (int)xc[xi];
          const int wv = G.w_u8 ? (int)reinterpret_cast<const uint8_t*>(wc)[wi] : (int)wc[wi];
          acc += (uint32_t)((xv - G.zpx) * (wv - G.zpw));
        }
      }
    }
  }
  if (e.out_i32) static_cast<int32_t*>(out)[idx] = (int32_t)acc;
  else static_cast<float*>(out)[idx] = (float)((double)(int32_t)acc * e.s_out);
}

// k_im2col computes input coordinates and offsets within one channel plane
// in 32 bits: every coordinate lies in [-lo, (P - 1) * st + (K - 1) * dl].
static bool conv_gemm_fits(const ConvGeom& G) {
  if (G.Sn >= ((int64_t)1 << 31)) return false;
  for (int i = 0; i < 3; ++i)
    if ((int64_t)(G.P[i] - 1) * G.st[i] + (int64_t)(G.K[i] - 1) * G.dl[i] >= ((int64_t)1 << 31)) return false;
  return true;
}
bool conv_uses_gemm(const ConvGeom& G) { return G.Kc >= 64 && conv_gemm_fits(G); }

// Short contractions (Cg * prod(K) < 64) that the GEMM still serves better
// than one thread per output: from 2^24 multiply-adds on (the direct kernel
// does about 1.2e12 a second: 32 x 3 x 112 x 112 -> 32, 3 x 3, takes 299 us
// direct and 72 us as im2col + GEMM; 8 x 3 x 56 x 56 -> 32 26 and 12 us)
// with at least 8 output channels per group in a 64-row tile.
static bool conv_short_gemm(const ConvGeom& G) {
  return G.Kc < 64 && G.Og >= 8 && conv_gemm_fits(G) &&
         (double)G.N * (double)G.O * (double)G.Pn * (double)G.Kc >= 0x1p24;
}

// The input zero point as an int8 code, zpx - 128 for ui8 operands: what a
// tap in the padding holds.  Zero points outside the type's range have none.
static int64_t conv_fill(const ConvGeom& G) { return (int64_t)G.zpx - (G.x_u8 ? 128 : 0); }

bool conv_affine(const ConvGeom& G) { return G.zpx != 0 || G.zpw != 0 || G.x_u8 || G.w_u8; }

constexpr size_t CONV_BATCH_BYTES = (size_t)128 << 20;   // workspace per batch of images
static size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

// The channel-last path: Cg a multiple of 16, at most WT_CHUNKS kernel
// positions, frame and matrix offsets of one image within 31 bits.
static bool conv_frame_of(const ConvGeom& G, ConvFrame* F) {
  if (G.Cg % 16 != 0 || G.Kn > WT_CHUNKS) return false;
  int64_t ep = 1;
  for (int i = 0; i < 3; ++i) {
    const int64_t E = (int64_t)(G.P[i] - 1) * G.st[i] + (int64_t)(G.K[i] - 1) * G.dl[i] + 1;
    if (E > ((int64_t)1 << 31) / ep) return false;
    F->E[i] = (int)E;
    ep *= E;
  }
  F->Ep = ep;
  return ep * G.Cg < ((int64_t)1 << 31) && G.Pn * G.Kc < ((int64_t)1 << 31);
}

static bool conv_pointwise(const ConvGeom& G) {
  return G.Kn == 1 && G.st[0] == 1 && G.st[1] == 1 && G.st[2] == 1;
}

// The frame path: the GEMM reads the frame itself.
static bool conv_frame_path(const ConvGeom& G, ConvFrame* F) {
  return conv_frame_of(G, F) && G.Kc <= ANY_CONV_MAX_K;
}
static size_t conv_wt_bytes(const ConvGeom& G) {   // 1 x 1: the weight as given
  return G.Kn == 1 ? 0 : round256((size_t)G.O * (size_t)G.Kc);
}

// Symmetric int8 with more than two tiles per CU: weight rows padded to the
// matrix's pitch for the direct-to-LDS GEMM (32 x 3 x 112 x 112, 7 x 7 at
// stride 2: 48.4 us against 53.5 with the weight at its own pitch).
static bool conv_im2col_many(const ConvGeom& G) {
  const int64_t t64 = ((G.Og + 63) / 64) * ((G.N * G.Pn + 63) / 64);
  return !conv_affine(G) && G.groups == 1 && t64 > 2 * (cu_count() > 0 ? cu_count() : 256) &&
         (int64_t)G.Kc16 * 256 < ((int64_t)1 << 31);
}

// Groups one after another, each through the direct-to-LDS GEMM, where a
// group's product alone fills the chip with 128 x 128 tiles.  That GEMM's lead
// over the one launch for all groups grows with the contraction, and the frame
// and GEMM launches of every group and the all-groups launch's fuller rounds
// count against it with every group more: up to one group per 288 of Kc.  Time
// by group against all at once, 3 x 3, 392 to 784 tiles a group: 256 channels a
// group 0.80-0.87 in two groups, 0.85-0.95 in four, 0.91-1.01 in eight, 1.04-1.08
// in sixteen; 128 channels 0.83-0.92, 0.95-1.00, 0.99-1.11; 64 channels 0.89-1.02
// in two, 0.98-1.13 in three.  Outputs that leave 128-row tiles a quarter empty
// (192: 0.97-1.01 in two groups, 1.04-1.12 in three), fewer tiles than CUs (32 x
// 256 x 28 x 28 -> 256 in two groups: 39 against 33 us) and 1 x 1 kernels
// (0.92-1.08 in two groups, 1.03-1.27 in three) stay with the one launch.
static bool conv_by_group(const ConvGeom& G) {
  if (G.groups == 1 || conv_affine(G) || conv_pointwise(G) || G.Cg % 64 != 0 || G.Kc > 16384 || G.Og < 128) return false;
  const int64_t cus = cu_count() > 0 ? cu_count() : 256, rows = (G.Og + 127) / 128;
  return G.groups * 288 <= G.Kc && G.Og * 8 >= rows * 128 * 7 && rows * ((G.N * G.Pn + 127) / 128) >= cus;
}

// Workspace bytes of one image and group, and of the weight rows beside them.
struct ConvUnit {
  size_t unit, wt;
};
static ConvUnit conv_unit(const ConvGeom& G) {
  ConvFrame F;
  if (conv_frame_path(G, &F)) return {(size_t)F.Ep * (size_t)G.Cg, conv_wt_bytes(G)};
  return {(size_t)G.Pn * (size_t)G.Kc16, conv_im2col_many(G) && G.Kc16 != G.Kc ? (size_t)G.O * (size_t)G.Kc16 : 0};
}

// The least workspace a symmetric int8 conv is accepted with: one image of
// one group at a time (where its first bytes are skipped for alignment and
// that no longer fits, the direct kernel runs).
size_t conv_workspace_need(const ConvGeom& G) {
  if (!conv_uses_gemm(G)) return 0;
  const ConvUnit u = conv_unit(G);
  ConvFrame F;
  return u.unit + (conv_frame_path(G, &F) ? u.wt : 0);
}

// What q8_quantized_conv_workspace asks for: as many groups, and images of
// all groups, as fit CONV_BATCH_BYTES, and room to start at a 16-byte
// boundary.
size_t conv_workspace_bytes(const ConvGeom& G) {
  if (!conv_uses_gemm(G) && !conv_short_gemm(G)) return 0;
  const ConvUnit u = conv_unit(G);
  size_t n = CONV_BATCH_BYTES / u.unit;
  const size_t groups = (size_t)G.groups, images = n / groups;
  n = images > 0 ? groups * (images < (size_t)G.N ? images : (size_t)(G.N > 0 ? G.N : 1)) : n > 0 ? n : 1;
  // (a batch of fewer images than this or of part of the groups splits K no
  // further: a split is for fewer tiles than CUs)
  const int64_t nb = images > 0 ? (int64_t)(n / groups) : 1, gc = images > 0 ? G.groups : (int64_t)n;
  return round256(n * u.unit + 15) + round256(u.wt) + any_part_bytes(G.Og, nb * G.Pn, gc, any_splits(G.Og, nb * G.Pn, G.Kc, gc));
}

// Images and groups of one pass over `unit` workspace bytes each, with the
// weight rows' wt before or after them: as many as fit `avail` and the launch
// limits.  False where not even one does.
static bool conv_batch(const ConvGeom& G, size_t unit, size_t wt, size_t avail, ConvPlan* p, bool by_group = false) {
  if (avail < wt || avail - wt < unit) return false;
  const int64_t units = (int64_t)((avail - wt) / unit);
  const int64_t fit = (((int64_t)1 << 31) - 1) / (int64_t)unit;           // one pass's offsets in 31 bits
  int64_t gc = units < G.groups ? units : G.groups;
  gc = gc < fit ? gc : fit;
  gc = gc < 65535 ? gc : 65535;
  gc = gc < 1 || by_group ? 1 : gc;
  int64_t nb = gc == G.groups || by_group ? units / gc : 1;
  nb = nb > G.N ? G.N : nb;
  nb = nb > 65535 ? 65535 : nb;                                           // grid.y of the per-image launches
  const int64_t cap = ((int64_t)1 << 31) / G.Pn - 1;                      // GEMM N = nb * P in an int
  nb = nb > cap ? cap : nb;
  nb = nb > fit / gc ? fit / gc : nb;
  p->gc = (int)gc;
  p->nb = nb < 1 ? 1 : nb;
  p->wt = wt;
  p->bytes = p->skip + wt + (size_t)p->nb * (size_t)gc * unit;
  return true;
}

ConvPlan conv_plan(const ConvGeom& G, const void* ws, size_t ws_bytes, bool prepacked) {
  ConvPlan p;
  if (ws == nullptr || G.N * G.O * G.Pn == 0 || !(conv_uses_gemm(G) || conv_short_gemm(G))) return p;
  if (conv_fill(G) < -128 || conv_fill(G) > 127) return p;
  p.skip = (16 - (reinterpret_cast<uintptr_t>(ws) & 15)) & 15;
  const size_t avail = ws_bytes > p.skip ? ws_bytes - p.skip : 0;
  ConvFrame F;
  const size_t mat = (size_t)G.Pn * (size_t)G.Kc16;
  if (conv_frame_path(G, &F) && conv_batch(G, (size_t)F.Ep * (size_t)G.Cg, prepacked ? 0 : conv_wt_bytes(G), avail, &p,
                                          conv_by_group(G))) {
    p.route = ConvPlan::FRAME;
    // the frame launch: 64 x 64 tiles of positions and channels in 2^23
    // workgroups, the channel tiles in grid.z
    const int64_t wide = (int64_t)64 * 65535 / G.Cg;
    if (p.gc > wide) p.gc = (int)wide, p.nb = 1;
    const int64_t tiles = ((F.Ep + 63) / 64) * (((int64_t)p.gc * G.Cg + 63) / 64);
    const int64_t cap = ((int64_t)1 << 23) / tiles;
    if (p.nb > cap) p.nb = cap;
    p.bytes = p.skip + p.wt + (size_t)p.nb * (size_t)p.gc * (size_t)F.Ep * (size_t)G.Cg;
  } else if ((conv_im2col_many(G) && G.Kc16 != G.Kc && conv_batch(G, mat, (size_t)G.O * (size_t)G.Kc16, avail, &p)) ||
           conv_batch(G, mat, 0, avail, &p))
    p.route = ConvPlan::IM2COL;
  if (p.route == ConvPlan::DIRECT) return p;
  // few tiles over a long contraction: partial sums of a K split behind the rest
  const int splits = any_splits(G.Og, p.nb * G.Pn, G.Kc, p.gc);
  const size_t part = any_part_bytes(G.Og, p.nb * G.Pn, p.gc, splits);
  if (splits > 1 && p.bytes + part <= ws_bytes) {
    p.splits = splits;
    p.part = p.bytes;
    p.bytes += part;
  }
  // A workspace that holds a part of the batch: a pass is two launches, about
  // 8 us, and the direct kernel does about 1.2e12 multiply-adds a second.
  const double passes = (double)((G.N + p.nb - 1) / p.nb) * (double)((G.groups + p.gc - 1) / p.gc);
  const double macs = (double)G.N * (double)G.O * (double)G.Pn * (double)G.Kc;
  return passes > 1.0 && 8.0 * passes > macs / 1.2e6 ? ConvPlan{} : p;
}

// The affine correction of the conv's GEMM (A: weights, B: input).
static AffineDot conv_zp(const ConvGeom& G) {
  AffineDot z{};
  z.xa = G.w_u8 ? (int)0x80808080u : 0;
  z.cA = (G.w_u8 ? 128 : 0) - G.zpw;
  z.cB = (int32_t)-conv_fill(G);
  z.kcc = (uint32_t)G.Kc * (uint32_t)z.cA * (uint32_t)z.cB;
  return z;
}

static hipError_t launch_conv_channel_last(const int8_t* x, const int8_t* w, const int8_t* w_taps,
                                           const ConvGeom& G, const ConvFrame& F, const GemmEpi& e,
                                           const ConvPlan& cb, int8_t* workspace, int32_t* part, void* out,
                                           hipStream_t st) {
  int8_t* wt_ws = workspace;
  int8_t* xp = wt_ws + cb.wt;
  // a 1 x 1 kernel's weight is its own tap-major form; a prepacked one
  // (q8_conv_weight_taps) is used as given
  const int8_t* wt = G.Kn == 1 ? w : w_taps ? w_taps : wt_ws;
  const bool affine = conv_affine(G);
  const AffineDot z = conv_zp(G);
  const AffineDot* zp = z.xa || z.cA || z.cB ? &z : nullptr;
  const int64_t nsl = G.O * (G.Cg >> 4);                   // weight slices
  const int wns = G.Kn >= 256 ? WT_CHUNKS / G.Kn : 256 / G.Kn;   // slices per workgroup
  bool weight_todo = G.Kn > 1 && !w_taps;
  const int etiles = (int)((F.Ep + 63) / 64);
  const size_t osz = e.out_i32 ? sizeof(int32_t) : sizeof(float);
  for (int64_t n0 = 0; n0 < G.N; n0 += cb.nb) {
    const int64_t nb = G.N - n0 < cb.nb ? G.N - n0 : cb.nb;
    for (int64_t g = 0; g < G.groups; g += cb.gc) {
      const int gc = (int)(G.groups - g < cb.gc ? G.groups - g : cb.gc);
      const int Cb = gc * G.Cg;
      const FrameJob J{n0, (int)(g * G.Cg), Cb, G.x_u8 ? 0x80u : 0u, (uint32_t)conv_fill(G) & 0xffu};
      const int64_t nfr = nb * etiles * ((Cb + 63) / 64), nw = weight_todo ? (nsl + wns - 1) / wns : 0;
      if (nfr + nw >= ((int64_t)1 << 24) || (Cb + 63) / 64 > 65535) return hipErrorInvalidValue;
      if (weight_todo) {
        const dim3 grid((unsigned)(nfr + nw));
        if (affine) hipLaunchKernelGGL(k_conv_prep<true>, grid, dim3(256), 0, st, x, G, F, J, nb, etiles, xp, w, nsl, wns, wt_ws);
        else hipLaunchKernelGGL(k_conv_prep<false>, grid, dim3(256), 0, st, x, G, F, J, nb, etiles, xp, w, nsl, wns, wt_ws);
      } else {
        const dim3 grid((unsigned)etiles, (unsigned)nb, (unsigned)((Cb + 63) / 64));
        if (affine) hipLaunchKernelGGL(k_conv_to_frame<true>, grid, dim3(256), 0, st, x, G, F, J, xp);
        else hipLaunchKernelGGL(k_conv_to_frame<false>, grid, dim3(256), 0, st, x, G, F, J, xp);
      }
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
      weight_todo = false;
      GemmEpi eb = e;
      eb.col_blk = G.Pn;
      eb.blk_stride = G.O * G.Pn;
      eb.ld_out = G.Pn;
      GemmEpi::ConvB& c = eb.cb;
      c.Pn = (uint32_t)G.Pn;
      c.P1 = (uint32_t)G.P[1];
      c.P2 = (uint32_t)G.P[2];
      c.st0 = (uint32_t)G.st[0];
      c.st1 = (uint32_t)G.st[1];
      c.st2 = (uint32_t)G.st[2];
      c.E1 = (uint32_t)F.E[1];
      c.E2 = (uint32_t)F.E[2];
      c.Ep = (uint32_t)F.Ep;
      c.Cg = (uint32_t)Cb;
      c.K1 = (uint32_t)G.K[1];
      c.K2 = (uint32_t)G.K[2];
      c.Kn = (uint32_t)G.Kn;
      c.dl0 = (uint32_t)G.dl[0];
      c.dl1 = (uint32_t)G.dl[1];
      c.dl2 = (uint32_t)G.dl[2];
      c.frame_bytes = (uint32_t)(nb * F.Ep * Cb);
      const int8_t* A = wt + g * G.Og * G.Kc;
      void* o = static_cast<char*>(out) + (size_t)((n0 * G.O + g * G.Og) * G.Pn) * osz;
      // With more than one 64 x 64 tile per CU the direct-to-LDS GEMM's
      // cheaper copies win (56 x 56 x 64: 24.3 against 25.7 us; 1 x 1 14 x
      // 14 x 1024 -> 256: 16.6 against 18.9); with fewer, K groups do (7 x 7 x
      // 512: 25.1, split over K in two launches, against 21.6 us).  A 1 x 1
      // conv needs no more than a 32 x 32 tile per CU: its rows are short (16 x
      // 256 x 28 x 28 -> 64, 196 64 x 64 tiles: 9.3 against 11.5; 8 x 64 x 14 x
      // 14 -> 64, 98 of 32 x 32: 8.6 against 7.7).
      const int64_t cus = cu_count() > 0 ? cu_count() : 256;
      const int64_t t32 = ((G.Og + 31) / 32) * ((nb * G.Pn + 31) / 32), t64 = ((G.Og + 63) / 64) * ((nb * G.Pn + 63) / 64);
      const bool aligned = !affine && cb.gc == 1;
      if (aligned && t64 > cus && !conv_pointwise(G) && G.Cg % 64 == 0 && G.Kc <= 16384) {
        err = launch_gemm_conv(A, xp, G.Og, nb * G.Pn, G.Kc, eb, o, st);
      } else if (aligned && t32 > cus && conv_pointwise(G) && (reinterpret_cast<uintptr_t>(A) & 15) == 0) {
        err = launch_gemm(A, xp, G.Og, nb * G.Pn, G.Kc, eb, o, st);
      } else {
        AnyPlan p;
        p.lda = G.Kc;
        p.ldb = 0;
        p.groups = gc;
        p.a_step = (int64_t)G.Og * G.Kc;
        p.b_step = G.Cg;
        p.o_step = (int64_t)G.Og * G.Pn;
        p.conv_cg = G.Cg;
        p.splits = cb.splits;
        p.part = part;
        err = launch_gemm_any(A, xp, G.Og, nb * G.Pn, G.Kc, eb, zp, p, o, st);
      }
      if (err != hipSuccess) return err;
    }
  }
  return hipSuccess;
}

// Receptive fields as a matrix (k_im2col), every group of a batch of images
// at once; the GEMM takes the weight rows at their own pitch.
static hipError_t launch_conv_im2col(const int8_t* x, const int8_t* w, const ConvGeom& G, const GemmEpi& e,
                                     const ConvPlan& cb, int8_t* col, int32_t* part, void* out, hipStream_t st) {
  const bool many = conv_im2col_many(G);
  const int8_t* wmat = w;
  if (cb.wt) {
    int8_t* wp = col + (size_t)cb.nb * (size_t)G.Pn * (size_t)G.Kc16;   // Kc16 % 16 == 0: stays aligned
    const int64_t n = G.O * G.Kc16;
    hipLaunchKernelGGL(k_pad_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w, G.O, (int64_t)G.Kc,
                       (int64_t)G.Kc16, wp);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    wmat = wp;
  }
  const AffineDot z = conv_zp(G);
  const AffineDot* zp = z.xa || z.cA || z.cB ? &z : nullptr;
  const size_t osz = e.out_i32 ? sizeof(int32_t) : sizeof(float);
  GemmEpi eb = e;
  eb.col_blk = G.Pn;
  eb.blk_stride = G.O * G.Pn;
  eb.ld_out = G.Pn;
  for (int64_t n0 = 0; n0 < G.N; n0 += cb.nb) {
    const int64_t nb = G.N - n0 < cb.nb ? G.N - n0 : cb.nb;
    for (int64_t g = 0; g < G.groups; g += cb.gc) {
      const int gc = (int)(G.groups - g < cb.gc ? G.groups - g : cb.gc);
      dim3 grid;
      if (!im2col_grid(G, nb, &grid)) return hipErrorInvalidValue;
      grid.z = (unsigned)gc;
      const uint32_t flip = G.x_u8 ? 0x80u : 0u, fill = (uint32_t)conv_fill(G) & 0xffu;
      if (conv_affine(G)) hipLaunchKernelGGL(k_im2col<true>, grid, dim3(256), 0, st, x, G, n0, g, flip, fill, col);
      else hipLaunchKernelGGL(k_im2col<false>, grid, dim3(256), 0, st, x, G, n0, g, flip, fill, col);
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
      void* o = static_cast<char*>(out) + (size_t)((n0 * G.O + g * G.Og) * G.Pn) * osz;
      if (many && (cb.wt || G.Kc16 == G.Kc) && (reinterpret_cast<uintptr_t>(wmat) & 15) == 0) {
        err = launch_gemm(wmat, col, G.Og, nb * G.Pn, G.Kc16, eb, o, st);
        if (err != hipSuccess) return err;
        continue;
      }
      AnyPlan p;
      p.lda = G.Kc;
      p.ldb = G.Kc16;
      p.groups = gc;
      p.a_step = (int64_t)G.Og * G.Kc;
      p.b_step = nb * G.Pn * G.Kc16;
      p.o_step = (int64_t)G.Og * G.Pn;
      p.splits = cb.splits;
      p.part = part;
      err = launch_gemm_any(w + g * G.Og * G.Kc, col, G.Og, nb * G.Pn, G.Kc, eb, zp, p, o, st);
      if (err != hipSuccess) return err;
    }
  }
  return hipSuccess;
}

bool conv_taps_used(const ConvGeom& G) { return G.Cg % 16 == 0 && G.Kn > 1 && G.Kn <= WT_CHUNKS; }

hipError_t launch_conv_weight_taps(const int8_t* w, const ConvGeom& G, int8_t* w_taps, hipStream_t st) {
  if (!conv_taps_used(G) || G.O == 0) return hipErrorInvalidValue;
  const int64_t nsl = G.O * (G.Cg >> 4);
  const int wns = G.Kn >= 256 ? WT_CHUNKS / G.Kn : 256 / G.Kn;
  const int64_t wblk = (nsl + wns - 1) / wns;
  if (wblk >= ((int64_t)1 << 24)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_conv_weight_taps, dim3((unsigned)wblk), dim3(256), 0, st, w, nsl, G.Cg, G.Kn, wns, w_taps);
  return hipGetLastError();
}

hipError_t launch_conv(const int8_t* x, const int8_t* w, const int8_t* w_taps, const ConvGeom& G,
                       const GemmEpi& e, const ConvPlan& p, void* workspace, void* out, hipStream_t st) {
  if (G.N * G.O * G.Pn == 0) return hipSuccess;
  if (p.route == ConvPlan::DIRECT) {
    const int64_t total = G.N * G.O * G.Pn;
    note_route("conv direct");
    hipLaunchKernelGGL(k_conv_direct, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, x,
                       w, G, e, out);
    return hipGetLastError();
  }
  int8_t* ws = static_cast<int8_t*>(workspace) + p.skip;
  int32_t* part = reinterpret_cast<int32_t*>(static_cast<int8_t*>(workspace) + p.part);
  if (p.route == ConvPlan::IM2COL) return launch_conv_im2col(x, w, G, e, p, ws, part, out, st);
  ConvFrame F;
  if (!conv_frame_path(G, &F)) return hipErrorInvalidValue;
  return launch_conv_channel_last(x, w, w_taps, G, F, e, p, ws, part, out, st);
}

}  // namespace q8
