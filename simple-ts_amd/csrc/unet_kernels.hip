// Kernels of the warm-start U-Net (gfx950): BF16 activations and weights,
// FP32 accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).
//
// Tensors are NHWC with channels fastest; a pixel index p runs over
// (n, j, i) with i fastest.  Every BF16 value is stored as its 16 raw bits.
//
// 3x3 convolution = implicit GEMM  Y[p][co] = sum_k A[p][k] * Wt[co][k],
// k = tap * Cx + ci (Cx = channel stride of the input, a multiple of 8, so
// the 8 consecutive k of one MFMA lane are 8 channels of one tap: one 16-byte
// load), Kp = k range rounded up to 32 with zero weights.  A 16x16x32 MFMA
// takes from lane l = r + 16 g the A row r (pixel) and the B column r (output
// channel), both at k = 8g..8g+7, and leaves D rows 4g..4g+3 of column r.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "unet_launch.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

struct alignas(16) U16x8 {
  u16 v[8];
};

struct alignas(8) U16x4 {
  u16 v[4];
};

__device__ __forceinline__ u16 f2bf(float f) {  // round to nearest even
  unsigned b = __float_as_uint(f);
  b += 0x7FFFu + ((b >> 16) & 1u);
  return (u16)(b >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((unsigned)h << 16); }

__device__ __forceinline__ bf16x8 load8(const u16 *p) {
  const U16x8 q = *reinterpret_cast<const U16x8 *>(p);
  return __builtin_bit_cast(bf16x8, q);
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, U16x8{}); }

// Outputs of a convolution, channels co .. co + 3 (of a multiple of 4) of the
// pixel at offset `at` of Y: bias, ReLU, the given ReLU's mask, rounding.
__device__ __forceinline__ void conv_out(const ConvArgs &a, size_t at, int co, const floatx4 &acc) {
  floatx4 bias = {0.f, 0.f, 0.f, 0.f};
  if (a.bias) bias = *reinterpret_cast<const floatx4 *>(a.bias + co);
  U16x4 act, out;
  if (a.act) act = *reinterpret_cast<const U16x4 *>(a.act + at);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    float v = acc[q] + bias[q];
    if (a.relu) v = fmaxf(v, 0.f);
    out.v[q] = a.act && !(bf2f(act.v[q]) > 0.f) ? (u16)0 : f2bf(v);
  }
  *reinterpret_cast<U16x4 *>(a.Y + at) = out;
}

// ---------------------------------------------------------------------------
// Convolution (forward, and backward-data with flipped weights) of any channel
// stride.  Block: 4 waves stacked along the pixels; a wave computes TM x TN
// tiles of 16 pixels x 16 channels: pixels [p0, p0 + 16 TM) x channels
// [c0, c0 + 16 TN), p0 = (4 blockIdx.x + w) * 16 TM, c0 = 16 TN blockIdx.y.
// Per 32-wide k chunk a lane loads TM + TN 16-byte fragments for TM * TN
// MFMAs, those of the next chunk while they run (a fragment outside the image
// from a.zero: no branch around a load); every output sums its k chunks in the
// same order for any TM, TN.  D rows = channels: a lane stores 4 of a pixel.
// ---------------------------------------------------------------------------
template <int TM, int TN>
__global__ void __launch_bounds__(256) k_conv(ConvArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int npix = a.N * a.H * a.W;
  const int p0 = (blockIdx.x * 4 + wave) * (16 * TM), c0 = blockIdx.y * (16 * TN);
  if (p0 >= npix) return;
  const int rad = a.ks / 2, taps = a.ks * a.ks;
  int pn[TM], pj[TM], pi[TM];
  bool pv[TM];
#pragma unroll
  for (int s = 0; s < TM; s++) {
    const int p = p0 + 16 * s + r;
    pv[s] = p < npix;
    const int q = pv[s] ? p : 0;
    pi[s] = q % a.W;
    const int t = q / a.W;
    pj[s] = t % a.H;
    pn[s] = t / a.H;
  }
  floatx4 acc[TM][TN];
#pragma unroll
  for (int x = 0; x < TM; x++)
#pragma unroll
    for (int y = 0; y < TN; y++) acc[x][y] = floatx4{0.f, 0.f, 0.f, 0.f};
  const u16 *zero = (const u16 *)a.zero;
  auto fetch = [&](int kc, bf16x8 (&A)[TM], bf16x8 (&B)[TN]) {
    const int k = kc + 8 * g;
    const int t = k / a.Cx, ci = k - t * a.Cx;
    const int dy = t / a.ks - rad, dx = t % a.ks - rad;
    // the tensor of channel ci: full size, or (u = 1) the half-size one
    const int u = a.X2 && ci < a.Cb ? 1 : 0, Cs = !a.X2 ? a.Cx : u ? a.Cb : a.Cx - a.Cb;
    const u16 *X = (a.X2 && !u ? a.X2 - a.Cb : a.X) + ci;
#pragma unroll
    for (int s = 0; s < TM; s++) {
      const int jj = pj[s] + dy, ii = pi[s] + dx;
      const u16 *at = X + ((size_t)(pn[s] * (a.H >> u) + (jj >> u)) * (a.W >> u) + (ii >> u)) * Cs;
      A[s] = load8(t < taps && pv[s] && jj >= 0 && jj < a.H && ii >= 0 && ii < a.W ? at : zero);
    }
#pragma unroll
    for (int s = 0; s < TN; s++) {
      const int co = c0 + 16 * s + r;
      const u16 *at = a.Wt + (size_t)co * a.Kp + k;
      B[s] = load8(co < a.Cout && kc < a.Kp ? at : zero);
    }
  };
  auto mul = [&](const bf16x8 (&A)[TM], const bf16x8 (&B)[TN]) {
#pragma unroll
    for (int x = 0; x < TM; x++)
#pragma unroll
      for (int y = 0; y < TN; y++) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[y], A[x], acc[x][y], 0, 0, 0);
  };
  bf16x8 A0[TM], B0[TN], A1[TM], B1[TN];
  fetch(0, A0, B0);
  for (int kc = 0; kc < a.Kp; kc += 64) {  // (beyond the end: zeros)
    fetch(kc + 32, A1, B1);
    mul(A0, B0);
    fetch(kc + 64, A0, B0);
    if (kc + 32 < a.Kp) mul(A1, B1);
  }
#pragma unroll
  for (int y = 0; y < TN; y++) {
    const int co = c0 + 16 * y + 4 * g;
    if (co >= a.Cout) continue;
#pragma unroll
    for (int x = 0; x < TM; x++) {
      const int p = p0 + 16 * x + r;
      if (p < npix) conv_out(a, (size_t)p * a.Cout + co, co, acc[x][y]);
    }
  }
}

// ---------------------------------------------------------------------------
// 3x3 convolution with its operands staged in LDS (input channel strides
// that are multiples of 32).  Four waves, WP along the rows x WC along the
// channels, compute a tile of R WP rows x 16 C pixels of one image for 16 TN WC
// output channels; a wave R rows x 16 C pixels x 16 TN channels.  Per chunk of
// 32 input channels the workgroup stages the input tile with a one-pixel halo
// (zeros outside the image) and the chunk's weights of all 9 taps, AHEAD chunks
// ahead in registers and NBUF of them in LDS.  A wave keeps the weights of the
// 9 taps in registers and walks the rows of the input tile: a row is the lower
// neighbour of one output row, the middle one of the next and the upper one of
// the third, so it is read from LDS 3 times (once per dx), not 9, and every
// output's sum still runs over the chunks, then the taps in order.
//
// Large images are bound by LDS reads and the chunks' loads in about equal parts
// (1920 x 384: 32 -> 32 channels 35 us, 94 MB; 96 -> 32 59 us, 34 us of MFMAs at
// the rate of a large product); small ones by the chain of a chunk (512 x 128: 6 ..
// 17 us per layer): the tile shrinks until there is a workgroup per CU, and two
// chunks are in flight.  With loads behind branches at the image's edge, which are
// waited for one by one, and every input fragment read once per tap: 61, 90 and 24 us.
// ---------------------------------------------------------------------------
constexpr int CONV_CI = 32;

// LDS slot of 16-byte vector g (of 4) of the pixel or output channel at
// position c: a pixel's 4 vectors are rotated by c / 2, so that the 8 lanes
// reading vector g of 8 consecutive positions in one LDS access hit 8
// different groups of 4 banks (unrotated, the 64-byte stride between
// positions puts them on 2 groups: 4-way conflicts).
__device__ __forceinline__ int conv_slot(int c, int g) { return (g + (c >> 1)) & 3; }

// Reads of one tensor from a workgroup-uniform address on, by byte offsets;
// those not below 2^31 - 16 give zeros, without a branch around the load
// (which would have to be waited for at the branch's end).
constexpr unsigned BUF_NONE = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_from(const u16 *p) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0x7ffffff0, 0x00027000);
}
__device__ __forceinline__ u32x4 buf_load(__amdgpu_buffer_rsrc_t b, unsigned off, unsigned uniform) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, (int)off, (int)uniform, 0));
}

template <int WP, int WC, int R, int C, int TN, int NBUF, int AHEAD, bool CAT>
__global__ void __launch_bounds__(256, NBUF == 1 ? 2 : 1) k_conv_lds(ConvArgs a) {
  static_assert(WP * WC == 4 && AHEAD % NBUF == 0, "four waves");
  constexpr int PH = R * WP, PW = 16 * C, CO = 16 * TN * WC, NV = CONV_CI / 8;
  constexpr int NA = (PH + 2) * (PW + 2) * NV, NB = 9 * CO * NV;  // 16-byte vectors of a chunk
  constexpr int RA = (NA + 255) / 256, RB = (NB + 255) / 256;    // per thread
  __shared__ u32x4 As[NBUF][256 * RA], Bs[NBUF][256 * RB];        // (the rest of the last ones: not read)
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 15, g = lane >> 4, wp = wave % WP, wc = wave / WP;
  const int tiles_x = (a.W + PW - 1) / PW, tiles_y = (a.H + PH - 1) / PH;
  const int bx = blockIdx.x, n = bx / (tiles_x * tiles_y), ty = (bx / tiles_x) % tiles_y, tx = bx % tiles_x;
  const int i0 = tx * PW, j0 = ty * PH, c0 = blockIdx.y * CO;
  floatx4 acc[R][C][TN];
#pragma unroll
  for (int o = 0; o < R; o++)
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
      for (int y = 0; y < TN; y++) acc[o][c][y] = floatx4{0.f, 0.f, 0.f, 0.f};
  // Offsets of the thread's vectors from the row above the tile (of the half-size
  // image: from its row); the channel is a uniform offset.
  const int jb = max(j0 - 1, 0), Cs = CAT ? a.Cx - a.Cb : a.Cx, H2 = a.H / 2, W2 = a.W / 2;
  const __amdgpu_buffer_rsrc_t bufX = buf_from((CAT ? a.X2 : a.X) + ((size_t)n * a.H + jb) * a.W * Cs);
  const __amdgpu_buffer_rsrc_t bufU = buf_from(CAT ? a.X + ((size_t)n * H2 + jb / 2) * W2 * a.Cb : a.X);
  const __amdgpu_buffer_rsrc_t bufW = buf_from(a.Wt + (size_t)c0 * a.Kp);
  unsigned oa[RA], ob[RB];
  auto offsets = [&](bool up) {
#pragma unroll
    for (int k = 0; k < RA; k++) {
      const int e = t + 256 * k, pos = e / NV, col = pos % (PW + 2), v = (e % NV - (col >> 1)) & 3;
      const int ii = i0 + col - 1, jj = j0 + pos / (PW + 2) - 1;
      const unsigned px = up ? (unsigned)((jj / 2 - jb / 2) * W2 + ii / 2) * a.Cb : (unsigned)((jj - jb) * a.W + ii) * Cs;
      oa[k] = e < NA && ii >= 0 && ii < a.W && jj >= 0 && jj < a.H ? 2 * (px + 8 * v) : BUF_NONE;
    }
  };
#pragma unroll
  for (int k = 0; k < RB; k++) {
    const int e = t + 256 * k, pos = e / NV, col = pos % CO, tap = pos / CO, v = (e % NV - (col >> 1)) & 3;
    ob[k] = e < NB && c0 + col < a.Cout ? 2 * (unsigned)(col * a.Kp + tap * a.Cx + 8 * v) : BUF_NONE;
  }
  offsets(CAT);
  u32x4 qa[AHEAD][RA], qb[AHEAD][RB];
  int cf = 0;  // the next chunk to fetch
  auto fetch = [&](u32x4 (&x)[RA], u32x4 (&w)[RB]) {
    if (CAT && cf == a.Cb) offsets(false);
    const bool up = CAT && cf < a.Cb;
    const __amdgpu_buffer_rsrc_t b = up ? bufU : bufX;
    const unsigned ch = 2 * (unsigned)(CAT && !up ? cf - a.Cb : cf);
#pragma unroll
    for (int k = 0; k < RA; k++) x[k] = buf_load(b, oa[k], ch);
#pragma unroll
    for (int k = 0; k < RB; k++) w[k] = buf_load(bufW, ob[k], 2 * (unsigned)cf);
    cf = min(cf + CONV_CI, a.Cx - CONV_CI);  // (at the end the last chunk again, not used)
  };
#pragma unroll
  for (int k = 0; k < AHEAD; k++) fetch(qa[k], qb[k]);
  for (int ci0 = 0; ci0 < a.Cx; ci0 += CONV_CI * AHEAD) {
#pragma unroll
    for (int h = 0; h < AHEAD; h++) {
      if (AHEAD > 1 && ci0 + CONV_CI * h >= a.Cx) break;
      const int buf = h % NBUF;
      if (NBUF == 1) __syncthreads();  // the last chunk has been read
#pragma unroll
      for (int k = 0; k < RA; k++) As[buf][t + 256 * k] = qa[h][k];
#pragma unroll
      for (int k = 0; k < RB; k++) Bs[buf][t + 256 * k] = qb[h][k];
      __syncthreads();
      fetch(qa[h], qb[h]);  // in flight while this chunk's MFMAs run
      bf16x8 B[9][TN];
#pragma unroll
      for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int y = 0; y < TN; y++) {
          const int col = 16 * (TN * wc + y) + r;
          B[tap][y] = __builtin_bit_cast(bf16x8, Bs[buf][(tap * CO + col) * NV + conv_slot(col, g)]);
        }
#pragma unroll
      for (int y = 0; y < R + 2; y++)  // input row R wp + y of the tile
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
#pragma unroll
          for (int c = 0; c < C; c++) {
            const int col = 16 * c + r + dx;
            const bf16x8 A = __builtin_bit_cast(
                bf16x8, As[buf][((R * wp + y) * (PW + 2) + col) * NV + conv_slot(col, g)]);
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
              const int o = y - dy;
              if (o < 0 || o >= R) continue;
#pragma unroll
              for (int q = 0; q < TN; q++)
                acc[o][c][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[3 * dy + dx][q], A, acc[o][c][q], 0, 0, 0);
            }
          }
    }
  }
  // D rows = channels 4 g .. 4 g + 3 of 16, column = pixel r of 16
#pragma unroll
  for (int y = 0; y < TN; y++) {
    const int co = c0 + 16 * (TN * wc + y) + 4 * g;
    if (co >= a.Cout) continue;
#pragma unroll
    for (int o = 0; o < R; o++) {
      const int j = j0 + R * wp + o;
      if (j >= a.H) continue;
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int i = i0 + 16 * c + r;
        if (i < a.W) conv_out(a, ((size_t)(n * a.H + j) * a.W + i) * a.Cout + co, co, acc[o][c][y]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 3x3 convolution of few input channels (stride 8 CV, CV <= 3: the network's
// first layer), whose 32-wide k chunks take several taps each.  A workgroup
// computes PH rows x 64 pixels for 16 TN channels from the tile and its halo in
// LDS; a lane's place in it for each chunk (its tap's shift and channel vector)
// and the weights of all chunks stay in registers.  Same k order as k_conv, which
// spends its time on addresses here: 1920 x 384, 9 .. 16 -> 32 channels 47 -> 26
// us, 8 x 512 x 128, 8 -> 32 27 -> 16 us.
// ---------------------------------------------------------------------------
constexpr int FEW_PW = 64;

template <int CV, int TN, int PH>
__global__ void __launch_bounds__(256) k_conv_few(ConvArgs a) {
  constexpr int NS = (72 * CV + 31) / 32;  // chunks
  constexpr int NA = (PH + 2) * (FEW_PW + 2) * CV, RA = (NA + 255) / 256;
  __shared__ u32x4 As[256 * RA + 1];  // the last one: zeros
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, r = lane & 15, g = lane >> 4;
  const int tiles_x = (a.W + FEW_PW - 1) / FEW_PW, tiles_y = (a.H + PH - 1) / PH;
  const int bx = blockIdx.x, n = bx / (tiles_x * tiles_y), ty = (bx / tiles_x) % tiles_y, tx = bx % tiles_x;
  const int i0 = tx * FEW_PW, j0 = ty * PH, c0 = blockIdx.y * (16 * TN);
  const u16 *zero = (const u16 *)a.zero;
#pragma unroll
  for (int k = 0; k < RA; k++) {
    const int e = t + 256 * k, pos = e / CV, v = e % CV;
    const int ii = i0 + pos % (FEW_PW + 2) - 1, jj = j0 + pos / (FEW_PW + 2) - 1;
    const u16 *at = a.X + (((size_t)n * a.H + jj) * a.W + ii) * (8 * CV) + 8 * v;
    As[e] = *reinterpret_cast<const u32x4 *>(ii >= 0 && ii < a.W && jj >= 0 && jj < a.H ? at : zero);
  }
  if (t == 0) As[256 * RA] = u32x4{0u, 0u, 0u, 0u};
  bf16x8 B[NS][TN];
  int off[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int v = 4 * s + g, tap = v / CV;  // the lane's 16-byte vector of k
    off[s] = tap < 9 ? ((tap / 3) * (FEW_PW + 2) + tap % 3) * CV + v % CV : -1;
#pragma unroll
    for (int y = 0; y < TN; y++) {
      const int co = c0 + 16 * y + r;
      const u16 *at = a.Wt + (size_t)co * a.Kp + 8 * v;
      B[s][y] = load8(co < a.Cout ? at : zero);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PH; q++) {  // 4 tiles of 16 pixels per row, one of each per wave
    const int px = 16 * wave + r, i = i0 + px, j = j0 + q;
    floatx4 acc[TN];
#pragma unroll
    for (int y = 0; y < TN; y++) acc[y] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const int at = off[s] < 0 ? 256 * RA : (q * (FEW_PW + 2) + px) * CV + off[s];
      const bf16x8 A = __builtin_bit_cast(bf16x8, As[at]);
#pragma unroll
      for (int y = 0; y < TN; y++) acc[y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B[s][y], A, acc[y], 0, 0, 0);
    }
    if (j >= a.H || i >= a.W) continue;
#pragma unroll
    for (int y = 0; y < TN; y++) {
      const int co = c0 + 16 * y + 4 * g;
      if (co < a.Cout) conv_out(a, (((size_t)n * a.H + j) * a.W + i) * a.Cout + co, co, acc[y]);
    }
  }
}

// ---------------------------------------------------------------------------
// Weight gradient of a 3x3 convolution, dW[t][ci][co] = sum_p X[p + off(t)][ci] *
// dZ[p][co]: a GEMM with M = co, N = ci for each of the 9 taps, reduced over
// pixels.
//
// A workgroup takes one run of WG_RUN consecutive pixels for 16 WCI input
// channels x 16 MT WCO output channels x 9 taps; a wave owns 16 x 16 MT of them
// for five or four of the taps.  Per step of 64 pixels (8 groups of 8, each
// within an image row; 32 pixels with 4 waves) a wave stages one group: dZ and
// the 3 x 10 pixels of X that the taps read, as they lie in memory, in one of two
// LDS buffers, the loads of the next AHEAD steps in flight in registers: one
// barrier per step.  Both operands need 8 consecutive pixels of one channel per
// lane: ds_read_b64_tr_b16 reads them transposed (lane i of 16 gets channel i of
// 4 pixels), and a tap's shift is then only another pixel address.  The workgroup
// leaves its sums in its own slot of `part` (laid out as the gradient is);
// k_sum_parts adds the slots in their order: no atomics, and the same gradients on
// every run.
//
// The bound is the chain of a step (LDS write, barrier, transposed reads, MFMA):
// a layer with one workgroup per CU takes 27 us whatever its size.  At 8 x 512 x
// 128, base 32: 455 us per training step for the 14 convolutions, biases
// included; with one wave per 16 x 16 of one tap, channel-strided 2-byte loads and
// atomics 3,484 us, and 2,958 for the biases in kernels of their own.  Loads
// under an exec mask had to be waited for at each branch's end (73 us per layer);
// the bias summed by a wave of the tile's own added 13 us to each layer: it has
// workgroups of its own, behind the others (between them they left every second
// chiplet without a tile: 40 us).  Pixel strides of 96 and 160 bytes put 4 pixels x 32
// bytes on distinct banks.
// ---------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// Channels c0 .. c0 + 15 (lane i = channel i) of 8 pixels of a row, as MFMA
// operand: base = LDS address of channel c0 + 4 (lane & 3) of pixel (lane & 15)
// / 4 of them.
__device__ __forceinline__ bf16x8 load_tr(const unsigned char *base, int stride) {
  typedef __attribute__((address_space(3))) s16x4 *Lp;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lp)(base));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lp)(base + 4 * stride));
  return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

constexpr int WG_RUN = 2048, WG_BIAS = 1024;  // pixels per slot of the weights and of the bias

template <int WCI, int WCO, int MT, int AHEAD, bool CAT>
__global__ void __launch_bounds__(128 * WCI * WCO, MT == 4 ? 2 : 4) k_wgrad(WgradArgs a, int run0, int runs) {
  constexpr int NW = 2 * WCI * WCO, CI = 16 * WCI, CO = 16 * MT * WCO;
  static_assert((NW == 4 || NW == 8) && CI <= 64 && CO <= 64, "tile");
  constexpr int SX = CI == 64 ? 160 : 96, SZ = CO == 64 ? 160 : 96;  // bytes per pixel
  constexpr int VX = CI / 8, VZ = CO / 8;                            // 16-byte vectors per pixel
  // A step takes NW groups, one staged by each wave: vectors per lane, and the
  // pixels that the lanes then write (those past 30 and 8 are not read: no branch
  // around a store to LDS either).
  constexpr int STEP = 8 * NW, RX = 32 * VX / 64, NX = 32, NZ = 64 / VZ;
  static_assert(AHEAD % 2 == 0 && VX >= 2, "buffers, vectors");
  __shared__ alignas(16) unsigned char Xs[2][NW][NX * SX], Zs[2][NW][NZ * SZ];
  const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int wci = wave % WCI, wco = wave / WCI % WCO, wt = wave / (WCI * WCO);
  const int ci0 = blockIdx.x * CI, co0 = blockIdx.y * CO, H = a.H, W = a.W;
  const int npix = a.N * H * W;
  // workgroups behind those of the runs: the biases' (not between them: a launch's
  // workgroups go to the chiplets in turn, and every other one would be theirs)
  const bool biased = (int)blockIdx.z >= runs;
  const int run = run0 + (biased ? ((int)blockIdx.z - runs) * (int)gridDim.x + (int)blockIdx.x : (int)blockIdx.z);
  const int pbeg = run * WG_RUN, pend = min(npix, pbeg + WG_RUN);
  if (biased) {  // a lane takes a channel of one of the run's two halves
    if (run >= run0 + runs) return;
    const int co = co0 + (int)threadIdx.x % CO, p0 = pbeg + (int)threadIdx.x / CO * WG_BIAS;
    const int p1 = min(npix, p0 + WG_BIAS);
    if ((int)threadIdx.x >= WG_RUN / WG_BIAS * CO || co >= a.Cout || p0 >= p1) return;
    const u16 *z = a.dZ + (size_t)p0 * a.Cout + co;
    const int C = a.Cout;
    float s = 0.f;
    int p = 0;
    const int n = p1 - p0;  // a multiple of 8
    if (n >= 32) {          // two batches of pixels, one in flight (at the end the last one again)
      u16 v0[32], v1[32];
      auto load = [&](u16 (&d)[32], int at) {
        const u16 *q0 = z + (size_t)min(at, n - 32) * C;
#pragma unroll
        for (int q = 0; q < 32; q++) d[q] = *q0, q0 += C;
      };
      auto add = [&](const u16 (&d)[32]) {
#pragma unroll
        for (int q = 0; q < 32; q++) s += bf2f(d[q]);
      };
      load(v0, 0);
      for (; p + 64 <= n; p += 64) {
        load(v1, p + 32);
        add(v0);
        load(v0, p + 64);
        add(v1);
      }
      if (p + 32 <= n) add(v0), p += 32;
    }
    for (; p < n; p += 8) {
      float d[8];
#pragma unroll
      for (int q = 0; q < 8; q++) d[q] = bf2f(z[(size_t)(p + q) * C]);
#pragma unroll
      for (int q = 0; q < 8; q++) s += d[q];
    }
    a.bpart[(size_t)(p0 / WG_BIAS) * a.Cout + co] = s;
    return;
  }
  floatx4 acc[5][MT];  // taps 5 wt ..
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int q = 0; q < 5; q++) acc[q][m] = floatx4{0.f, 0.f, 0.f, 0.f};
  u32x4 qx[AHEAD][RX], qz[AHEAD];
  // first pixel (fp), column, row and image of the wave's group in the next
  // step to fetch
  int fp = pbeg + 8 * wave, fi = fp % W, fn = fp / W / H, fj = fp / W - fn * H;
  // Per vector: its address, and where it lies outside the image: bit 0 / 1 in
  // the first / last row's group, 2 / 3 in the first / last column's, 4 past the
  // run's end, 5 always.  A vector outside is loaded from a.zero: no branch around
  // a load, which would have to be waited for at the branch's end.
  // bu: in the half-size image, less the group's first pixel's address and for an
  // even row (in an odd one the rows above and below are one row further down).
  typedef unsigned long long U64;
  U64 bx[RX], bu[CAT ? RX : 1];
  int ox[RX];
  bool up[RX];
  const int Cs = CAT ? a.Cx - a.Cb : a.Cx;
#pragma unroll
  for (int k = 0; k < RX; k++) {
    const int e = lane + 64 * k, px = e / VX, ci = ci0 + 8 * (e % VX);
    const int dy = px / 10 - 1, dx = px % 10 - 1;
    up[k] = CAT && ci < a.Cb;
    bx[k] = (U64)(CAT ? a.X2 : a.X) + 2ll * ((fp + (long long)dy * W + dx) * Cs + (CAT ? ci - a.Cb : ci));
    if (CAT) bu[k] = (U64)a.X + 2ll * (((long long)(dy >> 1) * (W / 2) + (dx >> 1)) * a.Cb + ci);
    ox[k] = (dy < 0) | (dy > 0) << 1 | (dx < 0) << 2 | (dx > 7) << 3 | 16 | (e >= 30 * VX || ci >= a.Cx) << 5;
  }
  const int zpx = lane / VZ, zco = co0 + 8 * (lane % VZ);
  U64 bz = (U64)a.dZ + 2ll * (((long long)fp + zpx) * a.Cout + zco);
  const int oz = 16 | (zpx >= 8 || zco >= a.Cout) << 5;
  typedef const __attribute__((address_space(1))) u32x4 *Gp;
  auto fetch = [&](u32x4 (&x)[RX], u32x4 &z) {
    const int i = fi, j = fj;
    const int out = (j == 0 ? 1 : 0) + (j == H - 1 ? 2 : 0) + (i == 0 ? 4 : 0) + (i + 8 == W ? 8 : 0) +
                    (fp >= pend ? 16 : 0) + 32;
    const U64 su = CAT ? 2ull * ((U64)(fn * (H / 2) + j / 2) * (U64)(W / 2) + (U64)(i / 2)) * (U64)a.Cb : 0;
    const U64 su1 = CAT && (j & 1) ? su + 2ull * (U64)(W / 2) * (U64)a.Cb : su;
#pragma unroll
    for (int k = 0; k < RX; k++) {
      U64 at = bx[k];
      if (CAT) {
        const U64 half = bu[k] + (ox[k] & 3 ? su1 : su);
        at = up[k] ? half : at;
      }
      x[k] = *(Gp)(ox[k] & out ? (U64)a.zero : at);
      bx[k] += 2ull * STEP * (U64)Cs;
    }
    z = *(Gp)(oz & out ? (U64)a.zero : bz);
    bz += 2ull * STEP * (U64)a.Cout;
    fp += STEP;
    for (fi += STEP; fi >= W; fi -= W)
      if (++fj == H) fj = 0, fn++;
  };
#pragma unroll
  for (int k = 0; k < AHEAD; k++) fetch(qx[k], qz[k]);
  for (int p0 = pbeg; p0 < pend; p0 += STEP * AHEAD) {  // (zeros past the end)
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
      const int buf = k & 1;  // its readers are past the last barrier
#pragma unroll
      for (int v = 0; v < RX; v++) {
        const int e = lane + 64 * v;
        *reinterpret_cast<u32x4 *>(&Xs[buf][wave][(e / VX) * SX + 16 * (e % VX)]) = qx[k][v];
      }
      *reinterpret_cast<u32x4 *>(&Zs[buf][wave][zpx * SZ + 16 * (lane % VZ)]) = qz[k];
      __syncthreads();
      fetch(qx[k], qz[k]);
#pragma unroll
      for (int h = 0; h < NW; h += 4) {
        const int x = r >> 2;
        const unsigned char *zb = &Zs[buf][h + g][x * SZ + 2 * (16 * MT * wco + 4 * (r & 3))];
        const unsigned char *xb = &Xs[buf][h + g][(11 + x) * SX + 2 * (16 * wci + 4 * (r & 3))];
        bf16x8 A[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) A[m] = load_tr(zb + 32 * m, SZ);
        auto tap = [&](int t, floatx4 (&d)[MT]) {
          const bf16x8 B = load_tr(xb + ((t / 3 - 1) * 10 + t % 3 - 1) * SX, SX);
#pragma unroll
          for (int m = 0; m < MT; m++) d[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[m], B, d[m], 0, 0, 0);
        };
        if (wt == 0) {
#pragma unroll
          for (int q = 0; q < 5; q++) tap(q, acc[q]);
        } else {
#pragma unroll
          for (int q = 0; q < 4; q++) tap(5 + q, acc[q]);
        }
      }
    }
  }
  // D rows = co (4 g + q of the tile), column = ci
  float *out = a.part + (size_t)blockIdx.z * (9 * a.Cin) * a.Cout;
  const int ci = ci0 + 16 * wci + r;
  if (ci >= a.Cin) return;
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int co = co0 + 16 * (MT * wco + m) + 4 * g;
    if (co >= a.Cout) continue;
#pragma unroll
    for (int q = 0; q < 5; q++)
      if (5 * wt + q < 9) *reinterpret_cast<floatx4 *>(out + ((size_t)(5 * wt + q) * a.Cin + ci) * a.Cout + co) = acc[q][m];
  }
}

// Sums of slots of FP32 partial sums, one slot after the other in FP32: out[e] =
// sum of part[q * P + e], q < S, onto out's own value unless `first`; P a multiple
// of 4.  The order is the one in which runs that start together end: a last run
// of at most three quarters of the others' length first (`ragged`: its slot is the
// last), then from the first one on.  Another order gives other last bits (1e-7 of
// a gradient's norm), and an Adam step shows them.  FP32 parameters that differ after
// one step from those of sums by atomics, in order of arrival: at 5 x 72 x 192 samples
// and base 32 1,540 of 1.9 million (8,800 with the short run last; two runs of the
// atomics 1,400), at 8 x 512 x 128 3,900 (3,800).
//
// Many slots: a workgroup takes 256 consecutive e; wave y has slots SUM_SLOTS y ..
// of SUM_WAVES * SUM_SLOTS at a time in registers, all loads in flight, and the
// waves add theirs in turn.
constexpr int SUM_WAVES = 8, SUM_SLOTS = 16;

// The q-th slot of the sum's order.
__device__ __forceinline__ int slot_at(int q, int S, bool ragged) { return !ragged ? q : q == 0 ? S - 1 : q - 1; }

__device__ __forceinline__ void sum_turns(const float *part, int S, size_t P, bool first, bool ragged, float *out,
                                          int group) {
  __shared__ floatx4 run[64];
  const int x = threadIdx.x & 63, y = threadIdx.x >> 6;
  const size_t e = 4 * ((size_t)group * 64 + x);
  const bool in = e < P;
  if (y == 0) run[x] = in && !first ? *reinterpret_cast<const floatx4 *>(out + e) : (floatx4)0.f;
  for (int q0 = 0; q0 < S; q0 += SUM_WAVES * SUM_SLOTS) {
    floatx4 v[SUM_SLOTS];
#pragma unroll
    for (int k = 0; k < SUM_SLOTS; k++)
      v[k] = *reinterpret_cast<const floatx4 *>(
          part + (size_t)slot_at(min(q0 + SUM_SLOTS * y + k, S - 1), S, ragged) * P + (in ? e : 0));
    for (int w = 0; w < SUM_WAVES; w++) {
      __syncthreads();
      if (w != y) continue;
      floatx4 s = run[x];
#pragma unroll
      for (int k = 0; k < SUM_SLOTS; k++)
        if (q0 + SUM_SLOTS * y + k < S) s += v[k];
      run[x] = s;
    }
  }
  __syncthreads();
  if (y == 0 && in) *reinterpret_cast<floatx4 *>(out + e) = run[x];
}

// Few slots: a thread takes 4 consecutive e, 8 slots' loads at a time.
__device__ __forceinline__ void sum_each(const float *part, int S, size_t P, bool first, bool ragged, float *out,
                                         int group) {
  const size_t e = 4 * ((size_t)group * (64 * SUM_WAVES) + threadIdx.x);
  if (e >= P) return;
  floatx4 s = first ? (floatx4)0.f : *reinterpret_cast<const floatx4 *>(out + e);
  for (int q0 = 0; q0 < S; q0 += 8) {
    floatx4 v[8];
#pragma unroll
    for (int k = 0; k < 8; k++)
      v[k] = *reinterpret_cast<const floatx4 *>(part + (size_t)slot_at(min(q0 + k, S - 1), S, ragged) * P + e);
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (q0 + k < S) s += v[k];
  }
  *reinterpret_cast<floatx4 *>(out + e) = s;
}

// The weights' slots (each: by sum_each) and, by the workgroups past the first
// `groups`, the bias's (rpart[rS][rP]).
struct SumArgs {
  const float *part;
  int S;
  size_t P;
  bool each, first, ragged;
  float *out;
  int groups;
  const float *rpart;
  int rS, rP;
  bool rragged;
  float *rout;
};
__global__ void __launch_bounds__(64 * SUM_WAVES) k_sum_parts(SumArgs a) {
  const int q = (int)blockIdx.x - a.groups;
  if (q >= 0) sum_turns(a.rpart, a.rS, a.rP, true, a.rragged, a.rout, q);
  else if (a.each) sum_each(a.part, a.S, a.P, a.first, a.ragged, a.out, blockIdx.x);
  else sum_turns(a.part, a.S, a.P, a.first, a.ragged, a.out, blockIdx.x);
}

// out[e] = sum of part[q * P + e], q < S, for few e, in FP64 (as good as exact):
// one wave per e, lane l adds slots l, l + 64, .., then the lanes in a fixed tree.
__global__ void __launch_bounds__(256) k_sum_rows(const float *part, int S, int P, float *out) {
  const int e = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (e >= P) return;
  double v = 0.0;
#pragma unroll 8
  for (int q = lane; q < S; q += 64) v += (double)part[(size_t)q * P + e];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) out[e] = (float)v;
}

// ---------------------------------------------------------------------------
// Element-wise and layout kernels
// ---------------------------------------------------------------------------
// Channel counts are multiples of 8: a thread moves 8 channels (16 bytes) of
// one output pixel.
__device__ __forceinline__ void load8f(const u16 *p, float (&v)[8]) {
  const U16x8 q = *reinterpret_cast<const U16x8 *>(p);
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = bf2f(q.v[k]);
}

// Sum of the 2x2 children (row pitch W) of output pixel (n, j, i), channels
// c .. c + 7 of a tensor of stride C: (00 + 01) + (10 + 11).
__device__ __forceinline__ void sum4(const u16 *X, int H, int W, int C, int n, int j, int i, int c, float (&s)[8]) {
  const size_t b = ((size_t)(n * H + 2 * j) * W + 2 * i) * C + c;
  float x[4][8];
  load8f(X + b, x[0]);
  load8f(X + b + C, x[1]);
  load8f(X + b + (size_t)W * C, x[2]);
  load8f(X + b + (size_t)W * C + C, x[3]);
#pragma unroll
  for (int k = 0; k < 8; k++) s[k] = (x[0][k] + x[1][k]) + (x[2][k] + x[3][k]);
}

// 2x2 average pool: X [N][H][W][C] -> Y [N][H/2][W/2][C]
__global__ void __launch_bounds__(256) k_pool(const u16 *X, int N, int H, int W, int C, u16 *Y) {
  const int V = C / 8, h = H / 2, w = W / 2;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)N * h * w * V) return;
  const int v = (int)(e % V), p = (int)(e / V), i = p % w, j = (p / w) % h, n = p / (w * h);
  float s[8];
  sum4(X, H, W, C, n, j, i, 8 * v, s);
  U16x8 o;
#pragma unroll
  for (int k = 0; k < 8; k++) o.v[k] = f2bf(s[k] * 0.25f);
  *reinterpret_cast<U16x8 *>(Y + 8 * e) = o;
}

// Backward of nearest-up on channels [0, Cu) of D [N][H][W][Cd], through the
// ReLU of the upsampled tensor Act: O [N][H/2][W/2][Cu] = round(sum of the 4
// children) where Act > 0, else 0
__global__ void __launch_bounds__(256) k_up_back(const u16 *D, int Cd, int Cu, const u16 *Act, int N, int H, int W,
                                                 u16 *O) {
  const int V = Cu / 8, h = H / 2, w = W / 2;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)N * h * w * V) return;
  const int v = (int)(e % V), p = (int)(e / V), i = p % w, j = (p / w) % h, n = p / (w * h);
  float s[8], m[8];
  sum4(D, H, W, Cd, n, j, i, 8 * v, s);
  load8f(Act + 8 * e, m);
  U16x8 o;
#pragma unroll
  for (int k = 0; k < 8; k++) o.v[k] = m[k] > 0.f ? f2bf(s[k]) : (u16)0;
  *reinterpret_cast<U16x8 *>(O + 8 * e) = o;
}

// Backward of the pool plus the skip branch, through the ReLU of the pooled
// tensor Act: O [N][H][W][C] = round(round(P[parent] / 4) + Skip[p][off + c])
// where Act > 0, else 0, with Skip of stride Cs.
__global__ void __launch_bounds__(256) k_pool_back_add(const u16 *P, const u16 *Skip, int Cs, int off, const u16 *Act,
                                                       int N, int H, int W, int C, u16 *O) {
  const int V = C / 8;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)N * H * W * V) return;
  const int v = (int)(e % V), p = (int)(e / V), i = p % W, j = (p / W) % H, n = p / (W * H);
  float q[8], s[8], m[8];
  load8f(P + ((size_t)(n * (H / 2) + j / 2) * (W / 2) + i / 2) * C + 8 * v, q);
  load8f(Skip + (size_t)p * Cs + off + 8 * v, s);
  load8f(Act + 8 * e, m);
  U16x8 o;
#pragma unroll
  for (int k = 0; k < 8; k++) o.v[k] = m[k] > 0.f ? f2bf(bf2f(f2bf(q[k] * 0.25f)) + s[k]) : (u16)0;
  *reinterpret_cast<U16x8 *>(O + 8 * e) = o;
}

// Head (1x1 conv, linear): Y[p][o] = sum_c X[p][c] * Wb[c][o] + b[o], FP32 out.
// Co <= CO <= HEAD_MAX_CO; the sums are kept in registers.  The weights (C x Co
// <= HEAD_MAX_W) are read from LDS, CO at a time, the pixel's channels 32 at a
// time (16-byte loads, C is a multiple of 8).
constexpr int HEAD_MAX_CO = 8, HEAD_MAX_W = 1024;
template <int CO>
__global__ void __launch_bounds__(256) k_head(const u16 *X, int C, const u16 *Wb, const float *b, int Co, int npix,
                                              float *Y) {
  __shared__ alignas(16) float Ws[CO * HEAD_MAX_W];  // [C][CO]
  for (int e = threadIdx.x; e < C * CO; e += blockDim.x)
    Ws[e] = e % CO < Co ? bf2f(Wb[e / CO * Co + e % CO]) : 0.f;
  __syncthreads();
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  float s[CO];
#pragma unroll
  for (int o = 0; o < CO; o++) s[o] = 0.f;
  for (int c0 = 0; c0 < C; c0 += 32) {
    U16x8 x[4];
#pragma unroll
    for (int v = 0; v < 4; v++)
      x[v] = *reinterpret_cast<const U16x8 *>(X + (size_t)p * C + min(c0 + 8 * v, C - 8));
#pragma unroll
    for (int v = 0; v < 4; v++) {
      if (c0 + 8 * v >= C) break;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const float xv = bf2f(x[v].v[q]);
#pragma unroll
        for (int o = 0; o < CO; o++) s[o] += xv * Ws[(c0 + 8 * v + q) * CO + o];
      }
    }
  }
#pragma unroll
  for (int o = 0; o < CO; o++)
    if (o < Co) Y[(size_t)p * Co + o] = s[o] + b[o];
}

// Head backward, through the ReLU of its input: dX[p][c] = round(sum_o
// dY[p][o] Wb[c][o]) where X > 0, else 0; and per workgroup of 256 pixels one
// slot of partial sums of dW[c][o] = sum_p dY[p][o] X[p][c] and (behind them)
// db[o] = sum_p dY[p][o].  A workgroup's sum is the pairwise tree over its
// threads (t + 128, t + 64, .. t + 1); the products of 8 channels at a time meet
// in LDS and the 4 waves share the sums, 4 at once: the levels 32 and 16 put two
// sums into one register each, the rest are moves within 16 lanes.  8 x 512 x 128,
// 32 -> 2: 40 us (64 MB of X and dX: 10 us); 759 us with a tree through LDS and
// barriers per sum and atomics.
template <int CO>
__global__ void __launch_bounds__(256) k_head_back(const float *dY, const u16 *X, int C, const u16 *Wb, int Co,
                                                   int npix, u16 *dX, float *part) {
  __shared__ float Ws[HEAD_MAX_W], red[8 * CO][256];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, p = (int)blockIdx.x * 256 + t;
  const bool ok = p < npix;
  for (int e = t; e < C * Co; e += 256) Ws[e] = bf2f(Wb[e]);
  float dy[CO];
#pragma unroll
  for (int o = 0; o < CO; o++) dy[o] = ok && o < Co ? dY[(size_t)p * Co + o] : 0.f;
  float *out = part + (size_t)blockIdx.x * (C + 1) * Co;
  // sums of rows q, q + 1, .. q + 3: in lanes 0, 32, 16, 48
  auto trees = [&](int q) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
      v[k] = (red[q + k][lane] + red[q + k][lane + 128]) + (red[q + k][lane + 64] + red[q + k][lane + 192]);
    auto swap = [](float &x, float &y, auto f) {
      const auto z = f(__float_as_uint(x), __float_as_uint(y));
      x = __uint_as_float(z[0]), y = __uint_as_float(z[1]);
    };
    auto p32 = [](unsigned x, unsigned y) { return __builtin_amdgcn_permlane32_swap(x, y, false, false); };
    auto p16 = [](unsigned x, unsigned y) { return __builtin_amdgcn_permlane16_swap(x, y, false, false); };
    swap(v[0], v[1], p32);
    swap(v[2], v[3], p32);
    v[0] += v[1], v[2] += v[3];
    swap(v[0], v[2], p16);
    float t = v[0] + v[2];
    t += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(t), 0x128, 0xf, 0xf, true));  // row_ror:8
    t += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(t), 0x124, 0xf, 0xf, true));
    t += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(t), 0x122, 0xf, 0xf, true));
    t += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(t), 0x121, 0xf, 0xf, true));
    return t;
  };
  const int mine = (lane >> 4 & 1) * 2 + (lane >> 5);  // the row of this lane's 16
  for (int c0 = 0; c0 < C; c0 += 8) {
    __syncthreads();  // Ws; the last channels' sums have been read
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ok) load8f(X + (size_t)p * C + c0, x);
    U16x8 d;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      float s = 0.f;
#pragma unroll
      for (int o = 0; o < CO; o++) {
        red[k * CO + o][t] = dy[o] * x[k];
        if (o < Co) s += dy[o] * Ws[(c0 + k) * Co + o];
      }
      d.v[k] = x[k] > 0.f ? f2bf(s) : (u16)0;
    }
    if (ok) *reinterpret_cast<U16x8 *>(dX + (size_t)p * C + c0) = d;
    __syncthreads();
#pragma unroll
    for (int q = 4 * wave; q < 8 * CO; q += 16) {
      const float v = trees(q);
      const int k = (q + mine) / CO, o = (q + mine) % CO;
      if ((lane & 15) == 0 && o < Co) out[(size_t)(c0 + k) * Co + o] = v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int o = 0; o < CO; o++) red[o][t] = dy[o];
  __syncthreads();
  if (4 * wave < CO) {
    const float v = trees(4 * wave);  // (rows past CO: not kept)
    if ((lane & 15) == 0 && 4 * wave + mine < Co) out[(size_t)C * Co + 4 * wave + mine] = v;
  }
}

// Masked MSE: dY = (Y - T) * m / count; loss += sum((Y - T)^2 m) / (2 count)
__global__ void __launch_bounds__(256) k_mse(const float *Y, const float *T, const uint8_t *M, int Co, int npix,
                                             float inv_count, float *dY, double *loss) {
  double s = 0.0;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < npix; p += gridDim.x * blockDim.x) {
    const float m = M[p] ? 1.f : 0.f;
    for (int o = 0; o < Co; o++) {
      const float e = (Y[(size_t)p * Co + o] - T[(size_t)p * Co + o]) * m;
      dY[(size_t)p * Co + o] = e * inv_count;
      s += (double)e * (double)e;
    }
  }
  __shared__ double red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0] * 0.5 * (double)inv_count);
}

// Adam on FP32 master parameters.
__global__ void k_adam(float *P, const float *G, float *m, float *v, size_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float g = G[e];
  const float mm = b1 * m[e] + (1.f - b1) * g;
  const float vv = b2 * v[e] + (1.f - b2) * g * g;
  m[e] = mm;
  v[e] = vv;
  const float mh = mm / c1, vh = vv / c2;
  P[e] -= lr * mh / (sqrtf(vh) + eps);
}

// Weight layouts from the FP32 master W[t][ci][co]:
//   Wt[co][t*Cx + ci]       forward (zero for ci >= Cin and k >= taps*Cx)
//   Wb[ci][t'*Co + co] = W[taps-1-t'][ci][co]   backward data (flipped taps)
//   Wh[ci][co]              1x1 head
// All convolutions of the network in one launch: workgroup b works on the
// convolution c with first[c] <= b < first[c + 1].
__global__ void __launch_bounds__(256) k_pack(PackArgs a) {
  int c = 0;
  while (c + 1 < a.n && (int)blockIdx.x >= a.first[c + 1]) c++;
  const PackConv &L = a.c[c];
  const size_t e = (size_t)((int)blockIdx.x - a.first[c]) * 256 + threadIdx.x;
  const float *W = a.P + L.w_off;
  const size_t nf = (size_t)L.Cout * L.Kp;
  if (e < nf) {  // forward layout (head: W as it is, Kp = Cin)
    if (L.taps == 1) {
      L.Wt[e] = f2bf(W[e]);
      return;
    }
    const int co = (int)(e / L.Kp), k = (int)(e % L.Kp), t = k / L.Cx, ci = k - t * L.Cx;
    L.Wt[e] = (t < L.taps && ci < L.Cin) ? f2bf(W[((size_t)t * L.Cin + ci) * L.Cout + co]) : (u16)0;
    return;
  }
  const size_t q = e - nf;  // backward-data layout
  if (!L.Wb || q >= (size_t)L.Cin * L.Kpb) return;
  const int ci = (int)(q / L.Kpb), k = (int)(q % L.Kpb), t = k / L.Cout, co = k - t * L.Cout;
  L.Wb[q] = (t < L.taps) ? f2bf(W[((size_t)(L.taps - 1 - t) * L.Cin + ci) * L.Cout + co]) : (u16)0;
}

// FP32 NHWC [n][C] -> BF16 with channel stride Cx (zero padding channels).
__global__ void k_to_bf16(const float *X, int C, int Cx, size_t npix, u16 *Y) {
  const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  for (int c0 = 0; c0 < Cx; c0 += 8) {  // Cx is a multiple of 8: 16-byte stores
    U16x8 o;
#pragma unroll
    for (int q = 0; q < 8; q++) o.v[q] = (c0 + q < C) ? f2bf(X[p * C + c0 + q]) : (u16)0;
    *reinterpret_cast<U16x8 *>(Y + p * Cx + c0) = o;
  }
}

// Solver state -> network input [H][W][Cx] (H = Ny rows j, W = Nx columns i):
// (u/u_ref, v/u_ref, p/p_ref - 1, T - 1, fluid mask), zero padding channels.
__global__ void k_pack_state(const double *u, const double *v, const double *p, const double *T, const uint8_t *m,
                             int npix, int Cx, double inv_u, double inv_p, u16 *X) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  u16 *o = X + (size_t)q * Cx;
  o[0] = f2bf((float)(u[q] * inv_u));
  o[1] = f2bf((float)(v[q] * inv_u));
  o[2] = f2bf((float)(p[q] * inv_p - 1.0));
  o[3] = f2bf((float)(T[q] - 1.0));
  o[4] = m[q] ? f2bf(1.f) : (u16)0;
  for (int c = 5; c < Cx; c++) o[c] = 0;
}

// Training target (dp / (p_ref dp_scale), dT / dT_scale) and mask.
__global__ void k_pack_target(const double *p, const double *p_pr, const double *T, const double *T_pr,
                              const uint8_t *m, int npix, double sp, double sT, float *Tg, uint8_t *M) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  Tg[2 * (size_t)q] = (float)((p[q] - p_pr[q]) * sp);
  Tg[2 * (size_t)q + 1] = (float)((T[q] - T_pr[q]) * sT);
  M[q] = m[q];
}

// Predicted guess: p' = p + y0 * (p_ref dp_scale), T' = T + y1 * dT_scale on
// the cells loop 3 updates (fluid cells of the p/T box [x0,x1) x [y0,y1)),
// copies elsewhere: fixed-value cells keep their boundary values.
__global__ void k_apply_pred(const float *Y, const double *p, const double *T, const uint8_t *m, int Nx, int npix,
                             int x0, int x1, int y0, int y1, double sp, double sT, double *pw, double *Tw) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  const int i = q % Nx, j = q / Nx;
  const bool upd = m[q] && i >= x0 && i < x1 && j >= y0 && j < y1;
  pw[q] = upd ? p[q] + (double)Y[2 * (size_t)q] * sp : p[q];
  Tw[q] = upd ? T[q] + (double)Y[2 * (size_t)q + 1] * sT : T[q];
}

// Corrector input [H][W][Cx]: the state x^n of the step (u/u_ref, v/u_ref,
// p/p_ref - 1, T - 1), the predicted start's change x_e - x^n in the same
// units divided by `step`, the fluid mask; zero padding channels.
__global__ void k_pack_corr_in(CorrFields xn, CorrFields xe, const uint8_t *m, int npix, int Cx, double inv_u,
                               double inv_p, double inv_step, u16 *X) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  u16 *o = X + (size_t)q * Cx;
  const double sc[4] = {inv_u, inv_u, inv_p, 1.0};
  o[0] = f2bf((float)(xn.f[0][q] * inv_u));
  o[1] = f2bf((float)(xn.f[1][q] * inv_u));
  o[2] = f2bf((float)(xn.f[2][q] * inv_p - 1.0));
  o[3] = f2bf((float)(xn.f[3][q] - 1.0));
#pragma unroll
  for (int c = 0; c < 4; c++) o[4 + c] = f2bf((float)((xe.f[c][q] - xn.f[c][q]) * sc[c] * inv_step));
  o[8] = m[q] ? f2bf(1.f) : (u16)0;
  for (int c = 9; c < Cx; c++) o[c] = 0;
}

// Corrector target: the converged step x^(n+1) minus the predicted start
// x_e, normalised as the input and divided by `corr`; mask = fluid cells.
__global__ void k_pack_corr_target(CorrFields x1, CorrFields xe, const uint8_t *m, int npix, double inv_u,
                                   double inv_p, double inv_corr, float *Tg, uint8_t *M) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  const double sc[4] = {inv_u, inv_u, inv_p, 1.0};
#pragma unroll
  for (int c = 0; c < 4; c++) Tg[4 * (size_t)q + c] = (float)((x1.f[c][q] - xe.f[c][q]) * sc[c] * inv_corr);
  M[q] = m[q];
}

// Corrected start x = x_e + y * scale on the cells loop 2 updates (u: fluid
// faces of the u box, v: of the v box, p and T: fluid cells of the p/T
// box); every other cell keeps x_e.  A value that is not finite, or a p or T
// that is not positive, keeps x_e.
__global__ void k_apply_corr(const float *Y, CorrFields xe, const uint8_t *m, CorrBoxes bx, int npix, double su,
                             double sp, double sT, CorrOut out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= npix) return;
  const int Nx = bx.Nx, i = q % Nx, j = q / Nx;
  const int iw = i > 0 ? q - 1 : (bx.px ? q + Nx - 1 : q), js = j > 0 ? q - Nx : q;
  const bool c = m[q];
  const bool upd[4] = {c && m[iw] && i >= bx.u[0] && i < bx.u[1] && j >= bx.u[2] && j < bx.u[3],
                       c && m[js] && i >= bx.v[0] && i < bx.v[1] && j >= bx.v[2] && j < bx.v[3],
                       c && i >= bx.o[0] && i < bx.o[1] && j >= bx.o[2] && j < bx.o[3],
                       c && i >= bx.o[0] && i < bx.o[1] && j >= bx.o[2] && j < bx.o[3]};
  const double sc[4] = {su, su, sp, sT};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const double e = xe.f[k][q];
    double x = upd[k] ? e + (double)Y[4 * (size_t)q + k] * sc[k] : e;
    if (!isfinite(x) || (k >= 2 && !(x > 0.0))) x = e;
    out.f[k][q] = x;
  }
}

// Gathers dataset samples into a batch.
__global__ void k_gather(const u16 *Xs, const float *Ts, const uint8_t *Ms, const int *slots, int n, int npix, int Cx,
                         int Co, u16 *X, float *Tg, uint8_t *M) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)n * npix) return;
  const int b = (int)(e / npix), q = (int)(e % npix);
  const size_t src = (size_t)slots[b] * npix + q;
  for (int c = 0; c < Cx; c += 8)  // Cx is a multiple of 8
    *reinterpret_cast<U16x8 *>(X + e * Cx + c) = *reinterpret_cast<const U16x8 *>(Xs + src * Cx + c);
  for (int c = 0; c < Co; c++) Tg[e * Co + c] = Ts[src * Co + c];
  M[e] = Ms[src];
}

}  // namespace

// ---------------------------------------------------------------------------
// Launch wrappers
// ---------------------------------------------------------------------------
static inline unsigned nblk(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

// The largest tile of a class that gives a workgroup per CU.  64 channels: 4 rows
// x 32 pixels (8 rows: 52 -> 57 us for 384 -> 128 at 480 x 96, 30 -> 31 for 64 -> 64
// at 960 x 192), else 4 or 2 rows x 16 pixels with two chunks in flight (64 -> 64
// at 256 x 64: 7.0 us, with 4 x 32 8.9, with 2 x 16 10; 256 -> 256 at 64 x 16: 9.9,
// with 4 x 16 11, with 4 x 32 16).  32 channels: 8 rows x 32 pixels where that gives
// two workgroups per CU (16 rows: 35 -> 41 us for 32 -> 32 at 1920 x 384), else 8 x
// 16 (512 x 128: 7.1 -> 6.1 us).
constexpr unsigned CONV_FULL = 256;

template <int WP, int WC, int R, int C, int TN>
static dim3 conv_grid(const ConvArgs &a) {
  return dim3((unsigned)a.N * nblk(a.H, R * WP) * nblk(a.W, 16 * C), nblk(a.Cout, 16 * TN * WC));
}
template <int WP, int WC, int R, int C, int TN>
static unsigned conv_groups(const ConvArgs &a) {
  const dim3 g = conv_grid<WP, WC, R, C, TN>(a);
  return g.x * g.y;
}
template <int WP, int WC, int R, int C, int TN, int NBUF, int AHEAD>
static void launch_conv(const ConvArgs &a, hipStream_t s) {
  const dim3 g = conv_grid<WP, WC, R, C, TN>(a);
  if (a.X2) hipLaunchKernelGGL((k_conv_lds<WP, WC, R, C, TN, NBUF, AHEAD, true>), g, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((k_conv_lds<WP, WC, R, C, TN, NBUF, AHEAD, false>), g, dim3(256), 0, s, a);
}

hipError_t unet_conv(const ConvArgs &a, hipStream_t s) {
  if (a.Cout % 4) return hipErrorInvalidValue;
  const size_t npix = (size_t)a.N * a.H * a.W;
  // (offsets within a tile's rows are 32 bits)
  const bool far = (size_t)20 * a.W * a.Cx >= ((size_t)1 << 30) || (size_t)64 * a.Kp >= ((size_t)1 << 30);
  if (a.ks == 3 && a.Cx % CONV_CI == 0 && (!a.X2 || a.Cb % CONV_CI == 0) && !far) {
    if (a.Cout % 64 == 0) {
      if (conv_groups<2, 2, 2, 2, 2>(a) >= CONV_FULL) launch_conv<2, 2, 2, 2, 2, 1, 1>(a, s);
      else if (conv_groups<1, 4, 4, 1, 1>(a) >= CONV_FULL) launch_conv<1, 4, 4, 1, 1, 2, 2>(a, s);
      else launch_conv<1, 4, 2, 1, 1, 2, 2>(a, s);
    } else {
      if (conv_groups<4, 1, 2, 2, 2>(a) > 2 * CONV_FULL) launch_conv<4, 1, 2, 2, 2, 1, 1>(a, s);
      else launch_conv<4, 1, 2, 1, 2, 1, 1>(a, s);
    }
    return hipGetLastError();
  }
  if (a.ks == 3 && a.Cx <= 24 && !a.X2) {
    auto launch = [&](auto ph) {
      constexpr int PH = decltype(ph)::value;
      const dim3 g((unsigned)a.N * nblk(a.H, PH) * nblk(a.W, FEW_PW), nblk(a.Cout, 32));
      if (a.Cx == 8) hipLaunchKernelGGL((k_conv_few<1, 2, PH>), g, dim3(256), 0, s, a);
      else if (a.Cx == 16) hipLaunchKernelGGL((k_conv_few<2, 2, PH>), g, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((k_conv_few<3, 2, PH>), g, dim3(256), 0, s, a);
    };
    // 8 rows where that gives two workgroups per CU (2 rows: 34 us instead of 26 at
    // 1920 x 384, but 6.6 instead of 11 at 512 x 128)
    if ((unsigned)a.N * nblk(a.H, 8) * nblk(a.W, FEW_PW) * nblk(a.Cout, 32) >= 2 * CONV_FULL)
      launch(std::integral_constant<int, 8>());
    else launch(std::integral_constant<int, 2>());
    return hipGetLastError();
  }
  // 4 pixel tiles per wave; 4 channel tiles where there are 64+ channels
  if (a.Cout >= 64)
    hipLaunchKernelGGL((k_conv<4, 4>), dim3(nblk(npix, 256), nblk(a.Cout, 64)), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_conv<4, 2>), dim3(nblk(npix, 256), nblk(a.Cout, 32)), dim3(256), 0, s, a);
  return hipGetLastError();
}
// Tiles of the weight gradient: the widest (64 x 64 channels; it reads least from
// LDS per MFMA) that leaves 128 workgroups, else 32 x 64, else 32 x 32 (16 x 32
// for a narrow input): a workgroup takes as long however few there are (64 -> 64
// channels, 131,072 pixels: 64 workgroups of 64 x 64 44 us, 128 of 32 x 64 28, 256 of
// 32 x 32, that read the pixels twice as often, 48).
constexpr long WGRAD_FULL = 128;
constexpr int SUM_EACH = 32;
static bool short_last(int npix, int run) { return npix % run != 0 && 4 * (npix % run) <= 3 * run; }

hipError_t unet_wgrad(const WgradArgs &a, float *dW, float *db, hipStream_t s) {
  if (a.W % 8 || a.Cx % 8 || a.Cout % 8 || (a.X2 && a.Cb % 8)) return hipErrorInvalidValue;
  const int npix = a.N * a.H * a.W, S = (int)nblk(npix, WG_RUN);
  auto groups = [&](int CI, int CO) { return (long)nblk(a.Cx, CI) * nblk(a.Cout, CO) * S; };
  const int CI = a.Cx <= 16 && !a.X2 ? 16 : a.Cx % 64 == 0 && a.Cout % 64 == 0 && groups(64, 64) >= WGRAD_FULL ? 64 : 32;
  const int CO = CI == 64 || (CI == 32 && a.Cout % 64 == 0 && groups(32, 64) >= WGRAD_FULL) ? 64 : 32;
  // as many slots at a time as the workspace holds
  const size_t P = (size_t)9 * a.Cin * a.Cout;
  const int most = (int)std::min<size_t>(std::max<size_t>(1, UNET_PART_FLOATS / P), 32767);
  for (int q = 0; q < S; q += most) {
    const int n = std::min(most, S - q);
    const bool each = n <= SUM_EACH;
    const int nsum = (int)nblk(P, each ? 256 * SUM_WAVES : 256);
    const bool last = q + n == S;
    const unsigned X = nblk(a.Cx, CI);
    const dim3 gr(X, nblk(a.Cout, CO), n + (n + X - 1) / X);  // + the biases
    if (CI == 64 && a.X2) hipLaunchKernelGGL((k_wgrad<4, 1, 4, 2, true>), gr, dim3(512), 0, s, a, q, n);
    else if (CI == 64) hipLaunchKernelGGL((k_wgrad<4, 1, 4, 2, false>), gr, dim3(512), 0, s, a, q, n);
    else if (CO == 64 && a.X2) hipLaunchKernelGGL((k_wgrad<2, 2, 2, 2, true>), gr, dim3(512), 0, s, a, q, n);
    else if (CO == 64) hipLaunchKernelGGL((k_wgrad<2, 2, 2, 2, false>), gr, dim3(512), 0, s, a, q, n);
    else if (a.X2) hipLaunchKernelGGL((k_wgrad<2, 2, 1, 2, true>), gr, dim3(512), 0, s, a, q, n);
    else if (CI == 32) hipLaunchKernelGGL((k_wgrad<2, 2, 1, 2, false>), gr, dim3(512), 0, s, a, q, n);
    else hipLaunchKernelGGL((k_wgrad<1, 2, 1, 4, false>), gr, dim3(256), 0, s, a, q, n);
    const SumArgs b{a.part, n, P, each, q == 0, last && short_last(npix, WG_RUN), dW, nsum,
                    a.bpart, (int)nblk(npix, WG_BIAS), a.Cout, short_last(npix, WG_BIAS), db};
    hipLaunchKernelGGL(k_sum_parts, dim3(nsum + (last ? nblk(a.Cout, 256) : 0)), dim3(64 * SUM_WAVES), 0, s, b);
  }
  return hipGetLastError();
}
hipError_t unet_pool(const uint16_t *X, int N, int H, int W, int C, uint16_t *Y, hipStream_t s) {
  hipLaunchKernelGGL(k_pool, dim3(nblk((size_t)N * (H / 2) * (W / 2) * (C / 8), 256)), dim3(256), 0, s, X, N, H, W, C,
                     Y);
  return hipGetLastError();
}
hipError_t unet_up_back(const uint16_t *D, int Cd, int Cu, const uint16_t *Act, int N, int H, int W, uint16_t *O,
                        hipStream_t s) {
  hipLaunchKernelGGL(k_up_back, dim3(nblk((size_t)N * (H / 2) * (W / 2) * (Cu / 8), 256)), dim3(256), 0, s, D, Cd, Cu,
                     Act, N, H, W, O);
  return hipGetLastError();
}
hipError_t unet_pool_back_add(const uint16_t *P, const uint16_t *Skip, int Cs, int off, const uint16_t *Act, int N,
                              int H, int W, int C, uint16_t *O, hipStream_t s) {
  hipLaunchKernelGGL(k_pool_back_add, dim3(nblk((size_t)N * H * W * (C / 8), 256)), dim3(256), 0, s, P, Skip, Cs, off,
                     Act, N, H, W, C, O);
  return hipGetLastError();
}
hipError_t unet_head(const uint16_t *X, int C, const uint16_t *Wh, const float *b, int Co, int npix, float *Y,
                     hipStream_t s) {
  if (Co > HEAD_MAX_CO || C * Co > HEAD_MAX_W) return hipErrorInvalidValue;
  if (Co <= 2) hipLaunchKernelGGL(k_head<2>, dim3(nblk(npix, 256)), dim3(256), 0, s, X, C, Wh, b, Co, npix, Y);
  else if (Co <= 4) hipLaunchKernelGGL(k_head<4>, dim3(nblk(npix, 256)), dim3(256), 0, s, X, C, Wh, b, Co, npix, Y);
  else hipLaunchKernelGGL(k_head<8>, dim3(nblk(npix, 256)), dim3(256), 0, s, X, C, Wh, b, Co, npix, Y);
  return hipGetLastError();
}
hipError_t unet_head_back(const float *dY, const uint16_t *X, int C, const uint16_t *Wh, int Co, int npix,
                          uint16_t *dX, float *part, float *grads, hipStream_t s) {
  if (Co > HEAD_MAX_CO || C * Co > HEAD_MAX_W || C % 8) return hipErrorInvalidValue;
  const int groups = (int)nblk(npix, 256);
  if (Co <= 2) hipLaunchKernelGGL(k_head_back<2>, dim3(groups), dim3(256), 0, s, dY, X, C, Wh, Co, npix, dX, part);
  else if (Co <= 4) hipLaunchKernelGGL(k_head_back<4>, dim3(groups), dim3(256), 0, s, dY, X, C, Wh, Co, npix, dX, part);
  else hipLaunchKernelGGL(k_head_back<8>, dim3(groups), dim3(256), 0, s, dY, X, C, Wh, Co, npix, dX, part);
  hipLaunchKernelGGL(k_sum_rows, dim3(nblk((size_t)(C + 1) * Co, 4)), dim3(256), 0, s, part, groups, (C + 1) * Co,
                     grads);
  return hipGetLastError();
}
hipError_t unet_mse(const float *Y, const float *T, const uint8_t *M, int Co, int npix, float inv_count, float *dY,
                    double *loss, hipStream_t s) {
  // a workgroup per CU (one atomic each: with a thread per pixel the 2,048
  // atomics on one word took 29 us at 8 x 512 x 128)
  hipLaunchKernelGGL(k_mse, dim3(std::min(256u, nblk(npix, 256))), dim3(256), 0, s, Y, T, M, Co, npix, inv_count, dY, loss);
  return hipGetLastError();
}
hipError_t unet_adam(float *P, const float *G, float *m, float *v, size_t n, float lr, float b1, float b2, float eps,
                     float c1, float c2, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, dim3(nblk(n, 256)), dim3(256), 0, s, P, G, m, v, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}
hipError_t unet_pack(PackArgs a, hipStream_t s) {
  int blocks = 0;
  for (int c = 0; c < a.n; c++) {
    a.first[c] = blocks;
    const PackConv &L = a.c[c];
    blocks += (int)nblk((size_t)L.Cout * L.Kp + (L.Wb ? (size_t)L.Cin * L.Kpb : 0), 256);
  }
  a.first[a.n] = blocks;
  hipLaunchKernelGGL(k_pack, dim3(blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t unet_to_bf16(const float *X, int C, int Cx, size_t npix, uint16_t *Y, hipStream_t s) {
  hipLaunchKernelGGL(k_to_bf16, dim3(nblk(npix, 256)), dim3(256), 0, s, X, C, Cx, npix, Y);
  return hipGetLastError();
}
hipError_t unet_pack_state(const double *u, const double *v, const double *p, const double *T, const uint8_t *m,
                           int npix, int Cx, double inv_u, double inv_p, uint16_t *X, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_state, dim3(nblk(npix, 256)), dim3(256), 0, s, u, v, p, T, m, npix, Cx, inv_u, inv_p, X);
  return hipGetLastError();
}
hipError_t unet_pack_target(const double *p, const double *p_pr, const double *T, const double *T_pr,
                            const uint8_t *m, int npix, double sp, double sT, float *Tg, uint8_t *M, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_target, dim3(nblk(npix, 256)), dim3(256), 0, s, p, p_pr, T, T_pr, m, npix, sp, sT, Tg, M);
  return hipGetLastError();
}
hipError_t unet_apply_pred(const float *Y, const double *p, const double *T, const uint8_t *m, int Nx, int npix,
                           const int box[4], double sp, double sT, double *pw, double *Tw, hipStream_t s) {
  hipLaunchKernelGGL(k_apply_pred, dim3(nblk(npix, 256)), dim3(256), 0, s, Y, p, T, m, Nx, npix, box[0], box[1],
                     box[2], box[3], sp, sT, pw, Tw);
  return hipGetLastError();
}
hipError_t unet_pack_corr_in(const CorrFields &xn, const CorrFields &xe, const uint8_t *m, int npix, int Cx,
                            double inv_u, double inv_p, double inv_step, uint16_t *X, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_corr_in, dim3(nblk(npix, 256)), dim3(256), 0, s, xn, xe, m, npix, Cx, inv_u, inv_p,
                     inv_step, X);
  return hipGetLastError();
}
hipError_t unet_pack_corr_target(const CorrFields &x1, const CorrFields &xe, const uint8_t *m, int npix, double inv_u,
                                 double inv_p, double inv_corr, float *Tg, uint8_t *M, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_corr_target, dim3(nblk(npix, 256)), dim3(256), 0, s, x1, xe, m, npix, inv_u, inv_p,
                     inv_corr, Tg, M);
  return hipGetLastError();
}
hipError_t unet_apply_corr(const float *Y, const CorrFields &xe, const uint8_t *m, const CorrBoxes &bx, int npix,
                           double su, double sp, double sT, const CorrOut &out, hipStream_t s) {
  hipLaunchKernelGGL(k_apply_corr, dim3(nblk(npix, 256)), dim3(256), 0, s, Y, xe, m, bx, npix, su, sp, sT, out);
  return hipGetLastError();
}
hipError_t unet_gather(const uint16_t *Xs, const float *Ts, const uint8_t *Ms, const int *slots, int n, int npix,
                       int Cx, int Co, uint16_t *X, float *Tg, uint8_t *M, hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3(nblk((size_t)n * npix, 256)), dim3(256), 0, s, Xs, Ts, Ms, slots, n, npix, Cx, Co,
                     X, Tg, M);
  return hipGetLastError();
}
