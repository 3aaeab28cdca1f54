// Layers of the warm-start U-Net (include/gvm_nn.h): convolutions with
// optional ReLU, 2x2 average pooling, nearest 2x upsampling into a channel
// block, channel copies, the MSE loss and Adam, forward and backward.
//
// Convolutions run on the FP32 MFMA units (forward, input gradient, and weight
// gradient in pixel ranges whose partials are summed in FP64 in a fixed order);
// bias gradients and the loss are FP64 fixed-order reductions, so training is
// reproducible bit for bit.  Layouts are NCHW.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "gvm_internal.h"
#include "gvm_nn.h"
#include "gvm_nn_pixels.h"

namespace gvm {
namespace {

constexpr int kT = 256;

int nblocks(long n) { return (int)std::max(1L, std::min<long>((n + kT - 1) / kT, 1L << 20)); }

// A weight as float: FP32 storage, or BF16 (the upper half of an FP32).
__device__ __forceinline__ float wload(const float* w, long i) { return w[i]; }
__device__ __forceinline__ float wload(const unsigned short* w, long i) {
  return __uint_as_float((unsigned int)w[i] << 16);
}

// ---------------------------------------------------------------------------
// Convolutions on the FP32 MFMA units (v_mfma_f32_32x32x2_f32: FP32 products,
// FP32 accumulation).  tap (ky, kx) shifts a pixel by (ky - K/2, kx - K/2), zero
// outside the image; g is the output gradient masked by the ReLU of the forward
// output.
//
//   forward      out[co][q]   = sum_{ci,tap} w[co][ci][tap] in[ci][q + tap]
//   input grad   din[ci][q]   = sum_{co,tap} w[co][ci][tap] g[co][q - tap]
//   weight grad  dw[co][ci][tap] = sum_q g[co][q] in[ci][q + tap]
//
// The instruction takes 64 cycles for a 32 x 32 block and two values of K, so a
// kernel that keeps its index arithmetic out of the loop runs at its rate (154
// TFLOP/s measured): pixels are tiled in the image's plane, a tile with its halo
// is staged in LDS once per chunk of channels and read at nine shifts, and the
// addresses of a thread's loads are computed once per block.  Weights are read
// along memory (lanes a row apart read 64 lines per load: 326 against 235 us for 512
// channels at 32 x 32 x 4) and no load sits in a branch of its own.  Forward and
// input gradient run at 90-110 TFLOP/s.  (An im2col loop that formed every
// element's coordinates as it loaded it ran at 26.)
// ---------------------------------------------------------------------------
typedef float f32x16_t __attribute__((ext_vector_type(16)));
enum { CONV_FWD = 0, CONV_BWD_DATA = 1 };

template <class WT>
struct ConvArgs {
  const float* in;    // forward: [B][Ci][H][W]; input grad: dout [B][Co][H][W]
  const float* mask;  // input grad: the forward output (ReLU mask), or NULL
  const WT* w;        // [Co][Ci][K][K]
  const float* bias;  // [Co] (forward)
  float* dst;         // [B][M][H][W]
  int B, M, C;        // output and input channels of this product
  int H, W, relu;
  int tiles_x, tiles_y;
};

// One block of 4 waves: MT output channels x a TH x TW tile of pixels; input
// channels in chunks of CK, the next chunk's values loaded into registers while
// this one is multiplied.  K runs over (channel, tap), tap fastest, two values
// per MFMA: the products and their order are an im2col GEMM's, so the sums do
// not depend on the tiling.  LDS: the tile's planes, and the weights [K][MT].
// The two halves of a wave read K values 2 s and 2 s + 1, whose places in the
// planes differ by a step that repeats every two channels: a lane keeps those
// addresses, and the rest of a read's address is an immediate.
template <int MODE, int KS, int MT, int TH, int TW, int CK, class WT>
__global__ __launch_bounds__(256) void conv_tile_kernel(ConvArgs<WT> a) {
  constexpr int KK = KS * KS, P = KS / 2, PH = TH + KS - 1, PW = TW + KS - 1;
  // a row's pitch in LDS: 32 pixels in rows of 8 on 32 banks
  constexpr int PP = TW == 8 ? 24 : PW;
  constexpr int PLANE = PH * PP, MTP = MT + 4;
  constexpr int NBT = TH * TW / 32, WN = NBT < 4 ? NBT : 4, WM = 4 / WN;
  constexpr int NB = NBT / WN, MB = MT / 32 / WM;
  static_assert(NB * WN == NBT && MB * WM * 32 == MT, "four waves share the tile");
  constexpr int NI = (CK * PH * PW + 255) / 256;   // input values per thread
  // weights: forward, 8 threads take a row (an output channel), whose chunk lies
  // together in memory; input grad, MT threads a channel, whose rows do
  constexpr int CP = 256 / MT, NW = CK / CP, KR = CK * KK / 8;
  static_assert(NW * CP == CK && KR * 8 == CK * KK, "whole channels and rows");
  __shared__ float li[CK * PLANE];
  __shared__ float lw[KK * CK * MTP];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 31, lh = lane >> 5;
  const int wn = wave % WN, wm = wave / WN;
  const int HW = a.H * a.W;
  const int tile = blockIdx.x, m0 = blockIdx.y * MT;
  const int tx = tile % a.tiles_x, ty = tile / a.tiles_x % a.tiles_y, b = tile / a.tiles_x / a.tiles_y;
  const int x0 = tx * TW, y0 = ty * TH;
  // this thread's input values: offset within a plane (-1: zero), plane, LDS place
  int off[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int e = t + 256 * j, r = e % (PH * PW);
    const int y = y0 + r / PW - P, x = x0 + r % PW - P;
    off[j] = e < CK * PH * PW && y >= 0 && y < a.H && x >= 0 && x < a.W ? y * a.W + x : -1;
  }
  const long in0 = (long)b * a.C * HW;
  const int wr = MODE == CONV_FWD ? t & 7 : t % MT, wq = MODE == CONV_FWD ? t >> 3 : t / MT;
  float ri[NI], rm[NI], rw[NW * KK];
  // Addresses out of range read element 0 and become zero when they are stored:
  // no branch keeps the loads of a chunk apart.
  auto load = [&](int c0, int j) {  // the j-th of a thread's NI + NW * KK values
    if (j < NI) {
      const int c = c0 + (t + 256 * j) / (PH * PW);
      const long i = off[j] >= 0 && c < a.C ? in0 + (long)c * HW + off[j] : 0;
      ri[j] = a.in[i];
      if (MODE == CONV_BWD_DATA && a.mask) rm[j] = a.mask[i];
    } else if (MODE == CONV_FWD) {  // w[m][c][tap]
      const int q = (j - NI) / KR, k = (j - NI) % KR, m = m0 + wq + 32 * q;
      const bool ok = m < a.M && wr + 8 * k < (a.C - c0) * KK;
      rw[j - NI] = wload(a.w, ok ? ((long)m * a.C + c0) * KK + wr + 8 * k : 0);
    } else {  // w[c][m][tap]
      const int q = (j - NI) / KK, k = (j - NI) % KK, c = c0 + wq + q * CP;
      const bool ok = c < a.C && wr + MT * k < (a.M - m0) * KK;
      rw[j - NI] = wload(a.w, ok ? ((long)c * a.M + m0) * KK + wr + MT * k : 0);
    }
  };
  auto store = [&](int c0) {
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int e = t + 256 * j;
      const bool ok = off[j] >= 0 && c0 + e / (PH * PW) < a.C &&
                      (MODE == CONV_FWD || !a.mask || rm[j] > 0.0f);
      if (e < CK * PH * PW)
        li[e / (PH * PW) * PLANE + e % (PH * PW) / PW * PP + e % PW] = ok ? ri[j] : 0.0f;
    }
    if constexpr (MODE == CONV_FWD) {
      const int left = (a.C - c0) * KK;
#pragma unroll
      for (int q = 0; q < MT / 32; q++)
#pragma unroll
        for (int k = 0; k < KR; k++)
          lw[(wr + 8 * k) * MTP + wq + 32 * q] =
              m0 + wq + 32 * q < a.M && wr + 8 * k < left ? rw[q * KR + k] : 0.0f;
    } else {
      const int left = (a.M - m0) * KK;
#pragma unroll
      for (int q = 0; q < NW; q++)
#pragma unroll
        for (int k = 0; k < KK; k++) {
          const int r = wr + MT * k;
          lw[((wq + q * CP) * KK + r % KK) * MTP + r / KK] =
              c0 + wq + q * CP < a.C && r < left ? rw[q * KK + k] : 0.0f;
        }
    }
  };
  f32x16_t acc[MB][NB];
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[m][n][e] = 0.0f;
  // places of the K values of two channels, less those of the pixel block:
  // tap (ky, kx) reads the pixel shifted by +tap (forward) or -tap (input grad)
  const float* pb[KK];
  {
    const int p = wn * NB * 32 + lr;
#pragma unroll
    for (int j = 0; j < KK; j++) {
      int place[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = 2 * j + h, c = k / KK, tap = MODE == CONV_FWD ? k % KK : KK - 1 - k % KK;
        place[h] = c * PLANE + tap / KS * PP + tap % KS;
      }
      pb[j] = li + p / TW * PP + p % TW + (lh ? place[1] : place[0]);
    }
  }
  constexpr int NSTEP = TW == 32 ? PP : 32 / TW * PP;  // from a pixel block to the next
  const float* pa = lw + lh * MTP + wm * MB * 32 + lr;
  constexpr int STEPS = CK / 2 * KK, NL = NI + NW * KK, LS = (NL + STEPS - 1) / STEPS;
#pragma unroll
  for (int j = 0; j < NL; j++) load(0, j);
  for (int c0 = 0; c0 < a.C; c0 += CK) {
    __syncthreads();  // the chunk before has been read
    store(c0);
    __syncthreads();
    // the operands of a step are read, and the next chunk's values loaded, while
    // the step before is multiplied (left to itself the compiler reads operands
    // right before their use and waits); past the end all loads read element 0
    float va[2][MB], vb[2][NB];
    auto read = [&](int i, int at) {
      const int c = i / KK, j = i % KK;
#pragma unroll
      for (int m = 0; m < MB; m++) va[at][m] = pa[(2 * KK * c + 2 * j) * MTP + m * 32];
#pragma unroll
      for (int n = 0; n < NB; n++) vb[at][n] = pb[j][2 * c * PLANE + n * NSTEP];
    };
    read(0, 0);
#pragma unroll
    for (int i = 0; i < STEPS; i++) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < MB; m++)
#pragma unroll
        for (int n = 0; n < NB; n++) {
          acc[m][n] =
              __builtin_amdgcn_mfma_f32_32x32x2f32(va[i & 1][m], vb[i & 1][n], acc[m][n], 0, 0, 0);
          if (m + n == 0) {
            if (i + 1 < STEPS) read(i + 1, (i + 1) & 1);
#pragma unroll
            for (int j = 0; j < LS; j++)
              if (i * LS + j < NL) load(c0 + CK, i * LS + j);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
    }
  }
  // 32 x 32 accumulator layout: lane l, register e -> row 8 (e / 4) + 4 (l / 32)
  // + e % 4, column l % 32
#pragma unroll
  for (int n = 0; n < NB; n++) {
    const int p = (wn * NB + n) * 32 + lr, y = y0 + p / TW, x = x0 + p % TW;
    if (y >= a.H || x >= a.W) continue;
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int co = m0 + (wm * MB + m) * 32 + 8 * (e >> 2) + 4 * lh + (e & 3);
        if (co >= a.M) continue;
        float v = acc[m][n][e];
        if constexpr (MODE == CONV_FWD) {
          v = v + a.bias[co];
          if (a.relu) v = fmaxf(v, 0.0f);
        }
        a.dst[((long)b * a.M + co) * HW + y * a.W + x] = v;
      }
  }
}

// The same product for shapes whose tiles would be mostly padding: an im2col GEMM
// of 64 outputs x 64 consecutive pixels (of any rows and images) per block, each wave
// a 32 x 32 block of it.  K advances in chunks of 16 that are staged k-major, every
// value's coordinates formed as it is loaded (26 TFLOP/s; a tile kernel's 90-110 need
// tiles that are full).  K's order is the tile kernel's, so are the bits.
template <int MODE, int KS, class WT>
__global__ __launch_bounds__(256) void conv_im2col_kernel(ConvArgs<WT> a) {
  constexpr int KK = KS * KS, P = KS / 2, CK = 16, T = 64;
  __shared__ float As[CK][T + 4];
  __shared__ float Bs[CK][T + 4];
  const int HW = a.H * a.W, npix = a.B * HW, Kd = a.C * KK;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  auto weight = [&](int m, int k) {
    if (m >= a.M || k >= Kd) return 0.0f;
    if constexpr (MODE == CONV_FWD) return wload(a.w, (long)m * Kd + k);  // w[m][c][tap]
    const int c = k / KK, tap = k - c * KK;  // w[c][m][tap]
    return wload(a.w, ((long)c * a.M + m) * KK + tap);
  };
  auto value = [&](int k, int q) {
    if (k >= Kd || q >= npix) return 0.0f;
    const int c = k / KK, tap = k - c * KK, b = q / HW, p = q - b * HW;
    const int dy = tap / KS - P, dx = tap % KS - P;
    const int y = p / a.W + (MODE == CONV_FWD ? dy : -dy);
    const int x = p % a.W + (MODE == CONV_FWD ? dx : -dx);
    if (y < 0 || y >= a.H || x < 0 || x >= a.W) return 0.0f;
    const long i = ((long)b * a.C + c) * HW + (long)y * a.W + x;
    if (MODE == CONV_BWD_DATA && a.mask && !(a.mask[i] > 0.0f)) return 0.0f;
    return a.in[i];
  };
  float ra[4], rb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int e = t + 256 * j;
      ra[j] = weight(m0 + e / CK, k0 + e % CK);
      rb[j] = value(k0 + e / T, n0 + e % T);
    }
  };
  f32x16_t acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.0f;
  load(0);
  for (int k0 = 0; k0 < Kd; k0 += CK) {
    __syncthreads();  // the chunk before has been read
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int e = t + 256 * j;
      As[e % CK][e / CK] = ra[j];
      Bs[e / T][e % T] = rb[j];
    }
    __syncthreads();
    if (k0 + CK < Kd) load(k0 + CK);
#pragma unroll
    for (int s = 0; s < CK / 2; s++)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[2 * s + lh][wm + lr], Bs[2 * s + lh][wn + lr],
                                                 acc, 0, 0, 0);
  }
  const int n = n0 + wn + lr;
  if (n >= npix) return;
  const int b = n / HW, p = n - b * HW;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int co = m0 + wm + 8 * (e >> 2) + 4 * lh + (e & 3);
    if (co >= a.M) continue;
    float v = acc[e];
    if constexpr (MODE == CONV_FWD) {
      v = v + a.bias[co];
      if (a.relu) v = fmaxf(v, 0.0f);
    }
    a.dst[((long)b * a.M + co) * HW + p] = v;
  }
}

// ---- weight gradient ----
constexpr int kWgradPixels = 8192;  // pixels of an FP32 partial

struct WgradArgs {
  const float* in;    // [B][Ci][H][W]
  const float* out;   // forward output (ReLU mask), or NULL
  const float* dout;  // [B][Co][H][W]
  float* part;        // [range][Co][Ci][K][K]
  double* bpart;      // [range][Co]
  int B, Ci, Co, H, W;
  unsigned int rw;    // about 2^32 / W
  int step_b, step_p; // kWgradChunk pixels as whole images and pixels of the next
};

// A wave owns one tap's 32 output x 32 input channels over a range of 8192 pixels
// (a FP32 partial; FP64 after that): K = pixels in their linear order (b, y, x), A =
// g[co][q], B = in[ci][q + tap].  That is an im2col GEMM's order, so the bits do not
// depend on how taps and channels are spread over waves; one tap per wave makes more
// waves of every layer of a network (9 x 128 for 2^20 pixels of 32 x 32 channels, and
// for each level down) than the chip has matrix units.  A block's waves share the row
// ky = blockIdx.x % KS of taps: for them the input is one linear run of pixels, (ky -
// K/2) W away and one to either side, staged without regard to the image's edges; a
// wave clears the operands of pixels whose tap lies outside with a mask of the
// chunk's 128 pixels.
// KS waves multiply and eight load: address arithmetic between the MFMAs of three
// waves took four times their time (2^20 pixels of 32 x 32 channels: 595 us, with
// three loaders 490, with eight 326; the MFMAs alone 125).  A wave's sum is one chain
// of dependent MFMAs, which take 50 ns each: 205 us is the least for a range.  LDS is double buffered, one barrier per chunk;
// values are loaded two chunks ahead.  Odd pitches keep 32 channels on 32 banks.  The
// loaders of the first taps also sum the bias gradient's partials (FP64).
constexpr int kWgradLoaders = 8;

// I: a byte offset into the tensors, 32 bits where they are below 4 GiB (one
// addition per load instead of three).
template <int KS, class I>
__global__ __launch_bounds__(64 * (KS + kWgradLoaders)) void conv_wgrad_kernel(WgradArgs a) {
  constexpr int KK = KS * KS, P = KS / 2, NL = kWgradLoaders, NCH = 32 / NL;
  constexpr int GP = kWgradChunk + 1, IP = (kWgradChunk + KS - 1) | 1;
  __shared__ float lg[2][32 * GP];
  __shared__ float li[2][32 * IP];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int HW = a.H * a.W, npix = a.B * HW;
  const int ky = blockIdx.x % KS, ci0 = blockIdx.x / KS * 32, co0 = blockIdx.y * 32;
  const int kbeg = blockIdx.z * kWgradPixels, kend = min(npix, kbeg + kWgradPixels);
  const int chunks = (kend - kbeg + kWgradChunk - 1) / kWgradChunk;
  // this lane's pixels of the chunk
  PixelPos gp[2];
#pragma unroll
  for (int h = 0; h < 2; h++) gp[h].start(kbeg + lane + 64 * h, HW);
  if (wave >= KS) {
    // ---- loaders: channels w, w + NL, ... of both operands ----
    const int w = wave - KS, te = w * 64 + lane;
    // the staged run starts P before the chunk; its last KS - 1 values by thread
    PixelPos ip[2], tail;
#pragma unroll
    for (int h = 0; h < 2; h++) ip[h].start(kbeg + lane + 64 * h - P, HW);
    tail.start(kbeg + kWgradChunk - P + te % 2, HW);
    float rg[2][NCH], rm[2][NCH], ri[2][NCH], re = 0.0f;
    bool og[2];
    double bs[NCH];
#pragma unroll
    for (int j = 0; j < NCH; j++) bs[j] = 0.0;
    // how many of this wave's channels exist; a pixel out of range reads as that of
    // element 0, a channel out of range as the last one, and both become zero when
    // they are stored
    const int ng = max(0, (a.Co - co0 - w + NL - 1) / NL);
    const int ni = max(0, (a.Ci - ci0 - w + NL - 1) / NL);
    const I plane = (I)HW * 4u, step = plane * NL, gi = plane * a.Co, ii = plane * a.Ci;
    const I g0 = plane * (co0 + (ng ? w : 0)), i0 = plane * (ci0 + (ni ? w : 0));
    const float* mask = a.out ? a.out : a.dout;
    const int tc = te / 2;
    const bool end = KS > 1 && te < 64, ot = end && ci0 + tc < a.Ci;
    const I t0 = plane * (ci0 + (ot ? tc : 0));
    auto at = [](const float* p, I k) { return *(const float*)((const char*)p + k); };
    auto load = [&]() {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        og[h] = gp[h].q < kend;
        I k = og[h] ? gi * gp[h].b + (I)gp[h].p * 4u + g0 : 0;
#pragma unroll
        for (int j = 0; j < NCH; j++) {
          rg[h][j] = at(a.dout, k);
          rm[h][j] = at(mask, k);
          k += j + 1 < ng ? step : 0;
        }
      }
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int p = ip[h].shifted((ky - P) * a.W, HW, npix);
        I k = p >= 0 ? ii * ip[h].b + (I)p * 4u + i0 : 0;
#pragma unroll
        for (int j = 0; j < NCH; j++) {
          ri[h][j] = at(a.in, k);
          k += j + 1 < ni ? step : 0;
        }
      }
      if (end) {
        const int p = tail.shifted((ky - P) * a.W, HW, npix);
        re = at(a.in, p >= 0 ? ii * tail.b + (I)p * 4u + t0 : 0);
        tail.next(HW, a.step_b, a.step_p);
      }
#pragma unroll
      for (int h = 0; h < 2; h++) {
        gp[h].next(HW, a.step_b, a.step_p);
        ip[h].next(HW, a.step_b, a.step_p);
      }
    };
    const bool all = !a.out;
    auto store = [&](int buf) {
      float* dg = &lg[buf][w * GP + lane];
      float* di = &li[buf][w * IP + lane];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < NCH; j++) {
          rg[h][j] = og[h] && j < ng && (all || rm[h][j] > 0.0f) ? rg[h][j] : 0.0f;
          dg[j * NL * GP + 64 * h] = rg[h][j];
          di[j * NL * IP + 64 * h] = j < ni ? ri[h][j] : 0.0f;
        }
      if (end) li[buf][tc * IP + kWgradChunk + te % 2] = ot ? re : 0.0f;
      if (blockIdx.x == 0)
#pragma unroll
        for (int j = 0; j < NCH; j++) bs[j] += (double)rg[0][j] + (double)rg[1][j];
    };
    load();
    store(0);
    load();
    __syncthreads();
    for (int k = 1; k <= chunks; k++) {
      if (k < chunks) {
        store(k & 1);
        load();
      }
      __syncthreads();
    }
    if (blockIdx.x == 0) {
#pragma unroll
      for (int j = 0; j < NCH; j++) {
        const int c = w + j * NL;
        double v = bs[j];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
        if (lane == 0 && co0 + c < a.Co)
          a.bpart[(long)blockIdx.z * a.Co + co0 + c] = v;
      }
    }
    return;
  }
  // ---- the waves that multiply ----
  const int lr = lane & 31, lh = lane >> 5;
  const int kx = wave;
  f32x16_t acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.0f;
  __syncthreads();
  for (int k = 0; k < chunks; k++) {
    // the chunk's pixels whose tap lies inside, as this half wave's bits
    unsigned int bits[4];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      int y = (int)__umulhi((unsigned int)gp[h].p, a.rw), x = gp[h].p - y * a.W;
      if (x < 0) {
        y--;
        x += a.W;
      } else if (x >= a.W) {
        y++;
        x -= a.W;
      }
      x += kx - P;
      y += ky - P;
      const unsigned long long m =
          __ballot(gp[h].q < kend && x >= 0 && x < a.W && y >= 0 && y < a.H) >> lh;
      bits[2 * h] = (unsigned int)m;
      bits[2 * h + 1] = (unsigned int)(m >> 32);
      gp[h].next(HW, a.step_b, a.step_p);
    }
    const float* pa = &lg[k & 1][lr * GP + lh];
    const float* pb = &li[k & 1][lr * IP + kx + lh];
    // operands four steps ahead
    constexpr int STEPS = kWgradChunk / 2, AHEAD = 4;
    float va[AHEAD], vb[AHEAD];
#pragma unroll
    for (int s = 0; s < AHEAD; s++) {
      va[s] = pa[2 * s];
      vb[s] = pb[2 * s];
    }
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      // all ones where the pixel's bit is set
      const int on = __builtin_amdgcn_sbfe((int)bits[s / 16], 2 * s % 32, 1);
      const float x = __int_as_float(__float_as_int(vb[s % AHEAD]) & on);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(va[s % AHEAD], x, acc, 0, 0, 0);
      if (s + AHEAD < STEPS) {
        va[s % AHEAD] = pa[2 * (s + AHEAD)];
        vb[s % AHEAD] = pb[2 * (s + AHEAD)];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  }
  float* dst = a.part + (long)blockIdx.z * a.Co * a.Ci * KK;
  const int ci = ci0 + lr;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int co = co0 + 8 * (e >> 2) + 4 * lh + (e & 3);
    if (co < a.Co && ci < a.Ci) dst[((long)co * a.Ci + ci) * KK + ky * KS + kx] = acc[e];
  }
}

// At most NP pixels, 16 or 32 (the deepest levels of a network on a small image,
// layers of one pixel): the kernel above would stage mostly padding for few MFMAs (us, it
// / this one: 512 x 512 channels of 4 x 4 pixels 27 / 6.6, of 5 x 4 27.1 / 9.6, 200,000 x
// 8 of one pixel 124 / 11.8).  A block forms 64 outputs x 64 (input channel, tap) pairs, K =
// the pixels, all of them staged at once; the sums are complete, and have the kernel's
// order.
template <int KS, int NP>
__global__ __launch_bounds__(256) void conv_wgrad_few_kernel(WgradArgs a, float* __restrict__ dw,
                                                             float* __restrict__ dbias) {
  constexpr int KK = KS * KS, P = KS / 2, T = 64;
  __shared__ float As[NP][T + 4];
  __shared__ float Bs[NP][T + 4];
  const int HW = a.H * a.W, npix = a.B * HW, N = a.Ci * KK;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
#pragma unroll
  for (int j = 0; j < NP * T / 256; j++) {
    const int e = t + 256 * j, q = e % NP, m = m0 + e / NP, n = n0 + e / NP;
    const int b = q / HW, p = q - b * HW;
    float g = 0.0f, v = 0.0f;
    if (q < npix && m < a.Co) {
      const long i = ((long)b * a.Co + m) * HW + p;
      g = !a.out || a.out[i] > 0.0f ? a.dout[i] : 0.0f;
    }
    if (q < npix && n < N) {
      const int c = n / KK, tap = n - c * KK;
      const int y = p / a.W + tap / KS - P, x = p % a.W + tap % KS - P;
      if (y >= 0 && y < a.H && x >= 0 && x < a.W)
        v = a.in[((long)b * a.Ci + c) * HW + y * a.W + x];
    }
    As[q][e / NP] = g;
    Bs[q][e / NP] = v;
  }
  __syncthreads();
  f32x16_t acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.0f;
#pragma unroll
  for (int s = 0; s < NP / 2; s++)
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[2 * s + lh][wm + lr], Bs[2 * s + lh][wn + lr],
                                               acc, 0, 0, 0);
  const int n = n0 + wn + lr;
#pragma unroll
  for (int e = 0; e < 16; e++) {
    const int m = m0 + wm + 8 * (e >> 2) + 4 * lh + (e & 3);
    if (m < a.Co && n < N) dw[(long)m * N + n] = acc[e];
  }
  if (blockIdx.x == 0 && t < T && m0 + t < a.Co) {
    double s[NP];
#pragma unroll
    for (int q = 0; q < NP; q++) s[q] = (double)As[q][t];
#pragma unroll
    for (int h = NP / 2; h > 0; h >>= 1)
#pragma unroll
      for (int q = 0; q < h; q++) s[q] += s[q + h];
    dbias[m0 + t] = (float)s[0];
  }
}

// dw = the FP64 sum of the weight-grad partials, dbias that of the bias partials,
// in the ranges' order.
__global__ __launch_bounds__(kT) void wgrad_reduce_kernel(const float* __restrict__ part, int npart,
                                                          long n, float* __restrict__ dw,
                                                          const double* __restrict__ bpart, int Co,
                                                          float* __restrict__ dbias) {
  for (long i = blockIdx.x * (long)kT + threadIdx.x; i < n + Co; i += (long)gridDim.x * kT) {
    double s = 0.0;
    if (i < n) {
      int r = 0;
      for (; r + 16 <= npart; r += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = part[(long)(r + u) * n + i];
#pragma unroll
        for (int u = 0; u < 16; u++) s += (double)v[u];
      }
      for (; r < npart; r++) s += (double)part[(long)r * n + i];
      dw[i] = (float)s;
    } else {
      for (int r = 0; r < npart; r++) s += bpart[(long)r * Co + (i - n)];
      dbias[i - n] = (float)s;
    }
  }
}

// Pooling, upsampling and channel copies move memory and nothing else.  A block
// takes part of one plane (blockIdx.y: the planes, a grid-stride loop), so that an
// index is split once, in 32 bits, and a thread moves V values with a wide access.
// (One value per thread and three 64-bit divisions: upsampling to 1024 x 1024 x 32
// took 129 us, 1.3 TB/s.)  Planes of fewer units than a block has threads are taken
// `group` at a time: one by one, 65,536 planes of 4 x 4 took 30 us, most threads idle.
template <class I, class F>
__device__ __forceinline__ void for_planes(long planes, int group, I n, F f) {
  if (group == 1) {
    for (long p = blockIdx.y; p < planes; p += gridDim.y)
      for (I o = blockIdx.x * (I)kT + threadIdx.x; o < n; o += (I)gridDim.x * kT) f(p, o);
    return;
  }
  // group * n <= kT: one pass of the block
  const int q = threadIdx.x / (int)n, o = threadIdx.x - q * (int)n;
  if (q >= group) return;
  for (long p = (long)blockIdx.y * group + q; p < planes; p += (long)gridDim.y * group) f(p, (I)o);
}

template <int V>
struct Vec;
template <>
struct Vec<1> {
  typedef float type;
};
template <>
struct Vec<2> {
  typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct Vec<4> {
  typedef float type __attribute__((ext_vector_type(4)));
};

// V pixels of two rows of `in` averaged by pairs: V / 2 pixels (V = 2: one).
template <int V, class I>
__global__ __launch_bounds__(kT) void pool_fwd_kernel(const float* __restrict__ in,
                                                      float* __restrict__ out, long nbc, int group,
                                                      I H, I W) {
  typedef typename Vec<V>::type vin;
  typedef typename Vec<V / 2>::type vout;
  const I h = H / 2, w = W / 2, wv = W / V;
  for_planes(nbc, group, h * wv, [&](long c, I o) {
    const I y = o / wv, x = o - y * wv;
    const float* s = in + c * ((long)H * W) + (long)(2 * y) * W + x * V;
    vin r[2];
    // V = 2: W is even, but a row may start at any 4 bytes
    __builtin_memcpy(&r[0], V == 4 ? __builtin_assume_aligned(s, 16) : s, sizeof(vin));
    __builtin_memcpy(&r[1], V == 4 ? __builtin_assume_aligned(s + W, 16) : s + W, sizeof(vin));
    vout v;
    if constexpr (V == 4) {
      v[0] = 0.25f * ((r[0][0] + r[0][1]) + (r[1][0] + r[1][1]));
      v[1] = 0.25f * ((r[0][2] + r[0][3]) + (r[1][2] + r[1][3]));
    } else {
      v = 0.25f * ((r[0][0] + r[0][1]) + (r[1][0] + r[1][1]));
    }
    *(vout*)(out + c * ((long)h * w) + (long)y * w + x * (V / 2)) = v;
  });
}

// out[b][c0 + c][Y][X] = scale in[b][c][Y/2][X/2]: V / 2 pixels to V pixels of two
// rows (up_fwd: scale 1; pool_bwd: 1/4, C == Cd)
template <int V, class I>
__global__ __launch_bounds__(kT) void up_kernel(const float* __restrict__ in,
                                                float* __restrict__ out, int B, int C, int Cd,
                                                int c0, int group, I H, I W, float scale) {
  typedef typename Vec<V / 2>::type vin;
  typedef typename Vec<V>::type vout;
  const I W2 = 2 * W, wv = W2 / V;
  for_planes((long)B * C, group, H * wv, [&](long p, I o) {
    const long b = p / C, c = p - b * C;
    const I y = o / wv, x = o - y * wv;
    const vin r = scale * *(const vin*)(in + p * ((long)H * W) + (long)y * W + x * (V / 2));
    vout v;
    if constexpr (V == 4)
      v = vout{r[0], r[0], r[1], r[1]};
    else
      v = vout{r, r};
    float* d = out + (b * Cd + c0 + c) * (4 * (long)H * W) + (long)(2 * y) * W2 + x * V;
    __builtin_memcpy(V == 4 ? __builtin_assume_aligned(d, 16) : d, &v, sizeof(vout));
    __builtin_memcpy(V == 4 ? __builtin_assume_aligned(d + W2, 16) : d + W2, &v, sizeof(vout));
  });
}

// din[b][c][y][x] = sum of the four dout[b][c0 + c][2y + dy][2x + dx]
template <int V, class I>
__global__ __launch_bounds__(kT) void up_bwd_kernel(const float* __restrict__ dout,
                                                    float* __restrict__ din, int B, int C, int Cd,
                                                    int c0, int group, I H, I W) {
  typedef typename Vec<V>::type vin;
  typedef typename Vec<V / 2>::type vout;
  const I W2 = 2 * W, wv = W2 / V;
  for_planes((long)B * C, group, H * wv, [&](long p, I o) {
    const long b = p / C, c = p - b * C;
    const I y = o / wv, x = o - y * wv;
    const float* s = dout + (b * Cd + c0 + c) * (4 * (long)H * W) + (long)(2 * y) * W2 + x * V;
    vin r[2];
    __builtin_memcpy(&r[0], V == 4 ? __builtin_assume_aligned(s, 16) : s, sizeof(vin));
    __builtin_memcpy(&r[1], V == 4 ? __builtin_assume_aligned(s + W2, 16) : s + W2, sizeof(vin));
    vout v;
    if constexpr (V == 4) {
      v[0] = (r[0][0] + r[0][1]) + (r[1][0] + r[1][1]);
      v[1] = (r[0][2] + r[0][3]) + (r[1][2] + r[1][3]);
    } else {
      v = (r[0][0] + r[0][1]) + (r[1][0] + r[1][1]);
    }
    *(vout*)(din + p * ((long)H * W) + (long)y * W + x * (V / 2)) = v;
  });
}

template <int V, class I>
__global__ __launch_bounds__(kT) void copy_channels_kernel(const float* __restrict__ src,
                                                           float* __restrict__ dst, int B, int C,
                                                           int Cs, int s0, int Cd, int d0,
                                                           int group, I HW) {
  typedef typename Vec<V>::type vec;
  for_planes((long)B * C, group, (I)(HW / V), [&](long p, I o) {
    const long b = p / C, c = p - b * C;
    ((vec*)(dst + (b * Cd + d0 + c) * (long)HW))[o] =
        ((const vec*)(src + (b * Cs + s0 + c) * (long)HW))[o];
  });
}

__global__ __launch_bounds__(kT) void add_kernel(const float* __restrict__ src,
                                                 float* __restrict__ dst, long n) {
  for (long o = blockIdx.x * (long)kT + threadIdx.x; o < n; o += (long)gridDim.x * kT)
    dst[o] += src[o];
}

constexpr int kMseBlocks = 1024;

__global__ __launch_bounds__(kT) void mse_kernel(const float* __restrict__ y,
                                                 const float* __restrict__ t,
                                                 float* __restrict__ dy, long n,
                                                 double* __restrict__ part) {
  __shared__ double red[kT];
  const float inv = 2.0f / (float)n;
  double acc = 0.0;
  for (long o = blockIdx.x * (long)kT + threadIdx.x; o < n; o += (long)gridDim.x * kT) {
    const float d = y[o] - t[o];
    dy[o] = inv * d;
    acc += (double)d * (double)d;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int h = kT / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kT) void mse_finish_kernel(const double* __restrict__ part, int nb,
                                                        long n, double* __restrict__ value) {
  __shared__ double red[kT];
  double acc = 0.0;
  for (int i = threadIdx.x; i < nb; i += kT) acc += part[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int h = kT / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *value = red[0] / (double)n;
}

__global__ __launch_bounds__(kT) void adam_kernel(float* __restrict__ p,
                                                  const float* __restrict__ g,
                                                  float* __restrict__ m, float* __restrict__ v,
                                                  long n, float lr, float b1, float b2,
                                                  float eps, float c1, float c2) {
  for (long o = blockIdx.x * (long)kT + threadIdx.x; o < n; o += (long)gridDim.x * kT) {
    const float gi = g[o];
    const float mi = b1 * m[o] + (1.0f - b1) * gi;
    const float vi = b2 * v[o] + (1.0f - b2) * gi * gi;
    m[o] = mi;
    v[o] = vi;
    p[o] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// Round to BF16, nearest even (finite values).
__global__ __launch_bounds__(kT) void to_bf16_kernel(const float* __restrict__ src,
                                                     unsigned short* __restrict__ dst, long n) {
  for (long o = blockIdx.x * (long)kT + threadIdx.x; o < n; o += (long)gridDim.x * kT) {
    const unsigned int u = __float_as_uint(src[o]);
    dst[o] = (unsigned short)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
  }
}

gvm_status launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return GVM_ERR_HIP;
  }
  return GVM_OK;
}

bool dims_ok(long a, long b, long c, long d, long e) {
  return a > 0 && b > 0 && c > 0 && d > 0 && e > 0 && a * b * c * d * e < (1L << 40);
}

}  // namespace
}  // namespace gvm

using namespace gvm;

namespace {

bool aligned(const void* p, size_t n) { return (uintptr_t)p % n == 0; }

// Planes of n units that a block takes at a time.
int plane_group(long n) { return (int)std::max(1L, kT / n); }

// Blocks for n units of each of `planes` planes.
dim3 plane_grid(long n, long planes) {
  const int group = plane_group(n);
  return dim3((unsigned)std::max(1L, std::min(65535L, (n + kT - 1) / kT)),
              (unsigned)std::min(65535L, (planes + group - 1) / group));
}

// The variant of a plane kernel: four values a thread where rows and pointers allow
// it, else two (upsampled pixels come in pairs); indices of 32 bits where a plane
// has no more than 2^30 values.
template <class F>
void plane_launch(long plane, bool wide, F f) {
  if (plane > (1L << 30))
    f(std::integral_constant<int, 2>(), 0L);
  else if (wide)
    f(std::integral_constant<int, 4>(), 0);
  else
    f(std::integral_constant<int, 2>(), 0);
}

// A launch of 2^32 threads or more wraps around without an error.
constexpr long kMaxBlocks = (1L << 32) / 256 - 1;

template <int MODE, int KS, int MT, int TH, int TW, int CK, class WT>
gvm_status launch_tile(gvm_ctx* ctx, ConvArgs<WT> a) {
  a.tiles_x = (a.W + TW - 1) / TW;
  a.tiles_y = (a.H + TH - 1) / TH;
  const long tiles = (long)a.tiles_x * a.tiles_y * a.B;
  GVM_REQUIRE(tiles <= kMaxBlocks, "gvm_nn_conv: too large and narrow an image");
  const dim3 grid((unsigned)tiles, (unsigned)((a.M + MT - 1) / MT));
  hipLaunchKernelGGL((conv_tile_kernel<MODE, KS, MT, TH, TW, CK, WT>), grid, dim3(256), 0,
                     ctx->stream, a);
  return GVM_OK;
}

// What a launch would take, in microseconds: a start, a chain of chunks, and the chip's
// share of every block's chunks (fits to 1,280 shapes of 1 to 128 channels and 1 to
// 1024 x 1024 pixels; within 15 % for two shapes of three).
struct ConvCost {
  double start, chain, block, extra;
  double us(long blocks, long chunks) const {
    return start + chain * chunks + block * blocks * (chunks + extra);
  }
};

// 3 x 3: the tile is 8 x 32 pixels and 64 channels (32 where there are no more) when
// that gives every CU two blocks, else 8 x 8 pixels and 64 channels.  The wide tile
// reads each weight for four times the pixels: layers of 19 GFLOP take 170-183 us with
// it (64 channels at 256 x 256 x 4) and 207-220 with the narrow one (256 channels at 64 x
// 64 x 4, 512 at 32 x 32 x 4), where it would have 256 and 128 blocks for 256 CUs.
// Images much smaller or narrower than a tile leave it mostly empty, and one input
// channel leaves a chunk of eight so: there the im2col kernel is the faster one (us, tiles /
// im2col: 128 channels, 2,048 images of 4 x 4: 1283 / 175; 64 channels, 4 images of 4096 x
// 1: 347 / 43; 1 to 64 channels at 1024 x 1024: 176 / 113; but 16 channels at 1024 x
// 1024: 112 / 314).
// 1 x 1: the tile kernel has nothing to share between taps.  It is ahead with full
// tiles for every CU, 32 output channels or fewer and 16 input channels or more (16 to
// 16 channels at 1024 x 1024: 76 / 81 us, 64 to 1: 94 / 119), and behind elsewhere (64 to
// 64 channels at 1024 x 1024: 213 / 194, 1 to 16: 76 / 60, 32 to 16 at 64 x 64: 8.7 / 5.7,
// 65,536 images of one pixel: 2263 / 21).  More outputs than 32 on 8 x 8 tiles of which
// no CU gets a second are a shorter chain (64 to 128 channels, 32 images of 7 x 7: 7.3 / 9.2).
template <int MODE, int KS, class WT>
gvm_status conv_launch_part(gvm_ctx* ctx, const ConvArgs<WT>& a) {
  auto blocks = [&](long th, long tw, long mt) {
    return (a.W + tw - 1) / tw * ((a.H + th - 1) / th) * a.B * ((a.M + mt - 1) / mt);
  };
  const long npix = (long)a.B * a.H * a.W;
  const dim3 cols((unsigned)((npix + 63) / 64), (unsigned)((a.M + 63) / 64));
  const long tiles = blocks(8, 32, 32);
  const bool fits = (long)cols.x <= kMaxBlocks;
  auto im2col = [&]() {
    hipLaunchKernelGGL((conv_im2col_kernel<MODE, KS, WT>), cols, dim3(256), 0, ctx->stream, a);
    return GVM_OK;
  };
  if constexpr (KS == 1) {
    const bool full = tiles >= ctx->cu_count && 2 * 256 * tiles <= 3 * npix;
    if (a.M > 32 && a.C >= 16 && blocks(8, 8, 64) <= ctx->cu_count)
      return launch_tile<MODE, 1, 64, 8, 8, 32, WT>(ctx, a);
    else if (fits && (a.M > 32 || a.C < 16 || !full))
      return im2col();
    else
      return launch_tile<MODE, 1, 32, 8, 32, 32, WT>(ctx, a);
  } else {
    const long wide = blocks(8, 32, 64), chunks = (a.C + 7) / 8, two_each = 2L * ctx->cu_count;
    const double tile_us = a.M <= 32     ? ConvCost{5.2, 2.6, 0.0069, 0.75}.us(tiles, chunks)
                           : wide >= two_each ? ConvCost{5.0, 0.15, 0.018, 1.1}.us(wide, chunks)
                                         : ConvCost{4.8, 1.75, 0.0036, 1.4}.us(blocks(8, 8, 64), chunks);
    const double im2col_us = ConvCost{3.6, 1.0, 0.00143, 2.7}.us(
        (long)cols.x * cols.y, ((long)a.C * 9 + 15) / 16);
    if (fits && (a.C == 1 || im2col_us < tile_us))
      return im2col();
    else if (a.M <= 32)
      return launch_tile<MODE, 3, 32, 8, 32, 8, WT>(ctx, a);
    else if (wide >= two_each)
      return launch_tile<MODE, 3, 64, 8, 32, 8, WT>(ctx, a);
    else
      return launch_tile<MODE, 3, 64, 8, 8, 8, WT>(ctx, a);
  }
}

// At most 2^29 pixels of whole images at a time: every kernel chosen above then has
// room for them in one launch.
template <int MODE, int KS, class WT>
gvm_status conv_launch(gvm_ctx* ctx, ConvArgs<WT> a) {
  const long hw = (long)a.H * a.W, B = a.B, per = std::max(1L, (1L << 29) / hw);
  for (long b = 0; b < B; b += per) {
    a.B = (int)std::min(per, B - b);
    const gvm_status st = conv_launch_part<MODE, KS>(ctx, a);
    if (st) return st;
    a.in += a.B * a.C * hw;
    if (a.mask) a.mask += a.B * a.C * hw;
    a.dst += a.B * a.M * hw;
  }
  return GVM_OK;
}

template <class WT>
gvm_status conv_fwd_launch(gvm_ctx* ctx, const float* in, const WT* w, const float* bias,
                           float* out, int B, int Ci, int Co, int H, int W, int K, int relu) {
  GVM_REQUIRE(ctx && in && w && bias && out, "gvm_nn_conv_fwd: null argument");
  GVM_REQUIRE(K == 1 || K == 3, "gvm_nn_conv_fwd: K must be 1 or 3");
  GVM_REQUIRE(dims_ok(B, Ci, Co, H, W), "gvm_nn_conv_fwd: bad sizes");
  GVM_REQUIRE((long)B * H * W < (1L << 31) && (long)Ci * K * K < (1L << 24) &&
                  (long)Co * K * K < (1L << 24),
              "gvm_nn_conv_fwd: sizes beyond the kernels' 32-bit indices");
  const ConvArgs<WT> a{in, nullptr, w, bias, out, B, Co, Ci, H, W, relu, 0, 0};
  const gvm_status st = K == 3 ? conv_launch<CONV_FWD, 3>(ctx, a) : conv_launch<CONV_FWD, 1>(ctx, a);
  return st ? st : launched("gvm_nn_conv_fwd");
}

template <int KS>
void launch_wgrad(gvm_ctx* ctx, const WgradArgs& a, int ranges) {
  const dim3 grid((unsigned)((a.Ci + 31) / 32 * KS), (unsigned)((a.Co + 31) / 32), (unsigned)ranges);
  const dim3 block(64 * (KS + kWgradLoaders));
  if ((long)a.B * std::max(a.Ci, a.Co) * a.H * a.W < (1L << 30))
    hipLaunchKernelGGL((conv_wgrad_kernel<KS, unsigned int>), grid, block, 0, ctx->stream, a);
  else
    hipLaunchKernelGGL((conv_wgrad_kernel<KS, unsigned long>), grid, block, 0, ctx->stream, a);
}

template <int KS>
void launch_wgrad_few(gvm_ctx* ctx, const WgradArgs& a, float* dw, float* dbias) {
  const dim3 grid((unsigned)((a.Ci * KS * KS + 63) / 64), (unsigned)((a.Co + 63) / 64));
  if (a.B * a.H * a.W <= 16)
    hipLaunchKernelGGL((conv_wgrad_few_kernel<KS, 16>), grid, dim3(256), 0, ctx->stream, a, dw,
                       dbias);
  else
    hipLaunchKernelGGL((conv_wgrad_few_kernel<KS, 32>), grid, dim3(256), 0, ctx->stream, a, dw,
                       dbias);
}

template <class WT>
gvm_status conv_bwd_launch(gvm_ctx* ctx, const float* in, const WT* w, const float* out,
                           const float* dout, float* din, float* dw, float* dbias, int B, int Ci,
                           int Co, int H, int W, int K, int relu) {
  GVM_REQUIRE(ctx && in && w && dout && dw && dbias, "gvm_nn_conv_bwd: null argument");
  GVM_REQUIRE(!relu || out, "gvm_nn_conv_bwd: the ReLU mask needs the forward output");
  GVM_REQUIRE(K == 1 || K == 3, "gvm_nn_conv_bwd: K must be 1 or 3");
  GVM_REQUIRE(dims_ok(B, Ci, Co, H, W), "gvm_nn_conv_bwd: bad sizes");
  GVM_REQUIRE((long)Co * Ci < (1L << 31), "gvm_nn_conv_bwd: too many channel pairs");
  GVM_REQUIRE((long)B * H * W < (1L << 31) && (long)Ci * K * K < (1L << 24) &&
                  (long)Co * K * K < (1L << 24),
              "gvm_nn_conv_bwd: sizes beyond the kernels' 32-bit indices");
  // (the end of the last range, and two chunks past it, are 32-bit indices too)
  GVM_REQUIRE((long)B * H * W <= (1L << 31) - kWgradPixels,
              "gvm_nn_conv_bwd: pixels beyond the weight gradient's 32-bit indices");
  const float* mask = relu ? out : nullptr;
  if (din) {
    const ConvArgs<WT> a{dout, mask, w, nullptr, din, B, Ci, Co, H, W, 0, 0, 0};
    const gvm_status st =
        K == 3 ? conv_launch<CONV_BWD_DATA, 3>(ctx, a) : conv_launch<CONV_BWD_DATA, 1>(ctx, a);
    if (st) return st;
  }
  if ((long)B * H * W <= 32) {
    const WgradArgs a{in, mask, dout, nullptr, nullptr, B, Ci, Co, H, W, 0, 0, 0};
    if (K == 3)
      launch_wgrad_few<3>(ctx, a, dw, dbias);
    else
      launch_wgrad_few<1>(ctx, a, dw, dbias);
    return launched("gvm_nn_conv_bwd");
  }
  // weight and bias gradients: partials in the context's network workspace (the
  // bias's first, in FP64), then their FP64 sums
  const int ranges = (int)(((long)B * H * W + kWgradPixels - 1) / kWgradPixels);
  const long nw = (long)Co * Ci * K * K;
  const size_t bias_elems = 2 * (size_t)ranges * Co;
  const size_t need = bias_elems + (size_t)ranges * nw;
  if (need > ctx->nn_part_elems) {
    GVM_REQUIRE(!ctx->capturing, "gvm_nn_conv_bwd: the workspace would grow under capture");
    GVM_HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (ctx->nn_part) GVM_HIP_TRY(hipFree(ctx->nn_part));
    ctx->nn_part = nullptr;
    ctx->nn_part_elems = 0;
    GVM_HIP_TRY(hipMalloc((void**)&ctx->nn_part, sizeof(float) * need));
    ctx->nn_part_elems = need;
  }
  const WgradArgs a{in, mask, dout, ctx->nn_part + bias_elems, (double*)ctx->nn_part, B, Ci, Co, H,
                    W,  (unsigned int)std::min(0xffffffffUL, ((1UL << 32) + W - 1) / W),
                    kWgradChunk / (H * W), kWgradChunk % (H * W)};
  if (K == 3)
    launch_wgrad<3>(ctx, a, ranges);
  else
    launch_wgrad<1>(ctx, a, ranges);
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(nblocks(nw + Co)), dim3(kT), 0,
                     ctx->stream, a.part, ranges, nw, dw, a.bpart, Co, dbias);
  return launched("gvm_nn_conv_bwd");
}

}  // namespace

extern "C" gvm_status gvm_nn_conv_fwd(gvm_ctx* ctx, const float* in, const float* w,
                                      const float* bias, float* out, int B, int Ci, int Co, int H,
                                      int W, int K, int relu) {
  return conv_fwd_launch(ctx, in, w, bias, out, B, Ci, Co, H, W, K, relu);
}

extern "C" gvm_status gvm_nn_conv_fwd_bf16(gvm_ctx* ctx, const float* in,
                                           const unsigned short* w, const float* bias, float* out,
                                           int B, int Ci, int Co, int H, int W, int K, int relu) {
  return conv_fwd_launch(ctx, in, w, bias, out, B, Ci, Co, H, W, K, relu);
}

extern "C" gvm_status gvm_nn_conv_bwd(gvm_ctx* ctx, const float* in, const float* w,
                                      const float* out, const float* dout, float* din, float* dw,
                                      float* dbias, int B, int Ci, int Co, int H, int W, int K,
                                      int relu) {
  return conv_bwd_launch(ctx, in, w, out, dout, din, dw, dbias, B, Ci, Co, H, W, K, relu);
}

extern "C" gvm_status gvm_nn_conv_bwd_bf16(gvm_ctx* ctx, const float* in,
                                           const unsigned short* w, const float* out,
                                           const float* dout, float* din, float* dw, float* dbias,
                                           int B, int Ci, int Co, int H, int W, int K, int relu) {
  return conv_bwd_launch(ctx, in, w, out, dout, din, dw, dbias, B, Ci, Co, H, W, K, relu);
}

extern "C" gvm_status gvm_nn_to_bf16(gvm_ctx* ctx, const float* src, unsigned short* dst, long n) {
  GVM_REQUIRE(ctx && src && dst && n > 0, "gvm_nn_to_bf16: bad argument");
  hipLaunchKernelGGL(to_bf16_kernel, dim3(nblocks(n)), dim3(kT), 0, ctx->stream, src, dst, n);
  return launched("gvm_nn_to_bf16");
}

extern "C" gvm_status gvm_nn_pool_fwd(gvm_ctx* ctx, const float* in, float* out, int B, int C,
                                      int H, int W) {
  GVM_REQUIRE(ctx && in && out, "gvm_nn_pool_fwd: null argument");
  GVM_REQUIRE(dims_ok(B, C, H, W, 1) && H % 2 == 0 && W % 2 == 0, "gvm_nn_pool_fwd: bad sizes");
  plane_launch(H * (long)W, W % 4 == 0 && aligned(in, 16) && aligned(out, 8), [&](auto v, auto i) {
    constexpr int V = v.value;
    typedef decltype(i) I;
    const long n = (long)H / 2 * (W / V);
    hipLaunchKernelGGL((pool_fwd_kernel<V, I>), plane_grid(n, (long)B * C), dim3(kT), 0,
                       ctx->stream, in, out, (long)B * C, plane_group(n), (I)H, (I)W);
  });
  return launched("gvm_nn_pool_fwd");
}

extern "C" gvm_status gvm_nn_pool_bwd(gvm_ctx* ctx, const float* dout, float* din, int B, int C,
                                      int H, int W) {
  GVM_REQUIRE(ctx && dout && din, "gvm_nn_pool_bwd: null argument");
  GVM_REQUIRE(dims_ok(B, C, H, W, 1) && H % 2 == 0 && W % 2 == 0, "gvm_nn_pool_bwd: bad sizes");
  plane_launch(H * (long)W, W % 4 == 0 && aligned(dout, 8) && aligned(din, 16),
               [&](auto v, auto i) {
                 constexpr int V = v.value;
                 typedef decltype(i) I;
                 const long n = (long)H / 2 * (W / V);
                 hipLaunchKernelGGL((up_kernel<V, I>), plane_grid(n, (long)B * C), dim3(kT), 0,
                                    ctx->stream, dout, din, B, C, C, 0, plane_group(n),
                                    (I)(H / 2), (I)(W / 2), 0.25f);
               });
  return launched("gvm_nn_pool_bwd");
}

extern "C" gvm_status gvm_nn_up_fwd(gvm_ctx* ctx, const float* in, float* out, int B, int C, int Cd,
                                    int c0, int H, int W) {
  GVM_REQUIRE(ctx && in && out, "gvm_nn_up_fwd: null argument");
  GVM_REQUIRE(dims_ok(B, C, H, W, 1) && c0 >= 0 && c0 + C <= Cd, "gvm_nn_up_fwd: bad sizes");
  plane_launch(4 * (long)H * W, W % 2 == 0 && aligned(in, 8) && aligned(out, 16),
               [&](auto v, auto i) {
                 constexpr int V = v.value;
                 typedef decltype(i) I;
                 const long n = (long)H * (2L * W / V);
                 hipLaunchKernelGGL((up_kernel<V, I>), plane_grid(n, (long)B * C), dim3(kT), 0,
                                    ctx->stream, in, out, B, C, Cd, c0, plane_group(n), (I)H, (I)W,
                                    1.0f);
               });
  return launched("gvm_nn_up_fwd");
}

extern "C" gvm_status gvm_nn_up_bwd(gvm_ctx* ctx, const float* dout, float* din, int B, int C,
                                    int Cd, int c0, int H, int W) {
  GVM_REQUIRE(ctx && dout && din, "gvm_nn_up_bwd: null argument");
  GVM_REQUIRE(dims_ok(B, C, H, W, 1) && c0 >= 0 && c0 + C <= Cd, "gvm_nn_up_bwd: bad sizes");
  plane_launch(4 * (long)H * W, W % 2 == 0 && aligned(dout, 16) && aligned(din, 8),
               [&](auto v, auto i) {
                 constexpr int V = v.value;
                 typedef decltype(i) I;
                 const long n = (long)H * (2L * W / V);
                 hipLaunchKernelGGL((up_bwd_kernel<V, I>), plane_grid(n, (long)B * C), dim3(kT), 0,
                                    ctx->stream, dout, din, B, C, Cd, c0, plane_group(n), (I)H,
                                    (I)W);
               });
  return launched("gvm_nn_up_bwd");
}

extern "C" gvm_status gvm_nn_copy_channels(gvm_ctx* ctx, const float* src, float* dst, int B, int C,
                                           int Cs, int s0, int Cd, int d0, int HW) {
  GVM_REQUIRE(ctx && src && dst, "gvm_nn_copy_channels: null argument");
  GVM_REQUIRE(dims_ok(B, C, HW, 1, 1) && s0 >= 0 && s0 + C <= Cs && d0 >= 0 && d0 + C <= Cd,
              "gvm_nn_copy_channels: bad sizes");
  const bool wide = HW % 4 == 0 && aligned(src, 16) && aligned(dst, 16);
  const dim3 grid = plane_grid(wide ? HW / 4 : HW, (long)B * C);
  const int group = plane_group(wide ? HW / 4 : HW);
  if (wide)
    hipLaunchKernelGGL((copy_channels_kernel<4, int>), grid, dim3(kT), 0, ctx->stream, src, dst, B,
                       C, Cs, s0, Cd, d0, group, HW);
  else
    hipLaunchKernelGGL((copy_channels_kernel<1, long>), grid, dim3(kT), 0, ctx->stream, src, dst, B,
                       C, Cs, s0, Cd, d0, group, (long)HW);
  return launched("gvm_nn_copy_channels");
}

extern "C" gvm_status gvm_nn_add(gvm_ctx* ctx, const float* src, float* dst, long n) {
  GVM_REQUIRE(ctx && src && dst && n > 0, "gvm_nn_add: bad argument");
  hipLaunchKernelGGL(add_kernel, dim3(nblocks(n)), dim3(kT), 0, ctx->stream, src, dst, n);
  return launched("gvm_nn_add");
}

extern "C" gvm_status gvm_nn_mse(gvm_ctx* ctx, const float* y, const float* t, float* dy, long n,
                                 int slot) {
  GVM_REQUIRE(ctx && y && t && dy && n > 0, "gvm_nn_mse: bad argument");
  GVM_REQUIRE(slot >= 0 && slot < kValueSlots, "gvm_nn_mse: value slot out of range");
  // block partials in the last reduction slot of the context
  double* part = ctx->partials + (long)(kMaxSlots - 1) * kReduceBlocks;
  const int nb = std::min(kMseBlocks, nblocks(n));
  hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(kT), 0, ctx->stream, y, t, dy, n, part);
  hipLaunchKernelGGL(mse_finish_kernel, dim3(1), dim3(kT), 0, ctx->stream, part, nb, n,
                     ctx->dvalues + slot);
  return launched("gvm_nn_mse");
}

extern "C" gvm_status gvm_nn_adam(gvm_ctx* ctx, float* p, const float* g, float* m, float* v,
                                  long n, float lr, float beta1, float beta2, float eps, int t) {
  GVM_REQUIRE(ctx && p && g && m && v && n > 0 && t >= 1, "gvm_nn_adam: bad argument");
  const float c1 = 1.0f - std::pow(beta1, (float)t);
  const float c2 = 1.0f - std::pow(beta2, (float)t);
  hipLaunchKernelGGL(adam_kernel, dim3(nblocks(n)), dim3(kT), 0, ctx->stream, p, g, m, v, n, lr,
                     beta1, beta2, eps, c1, c2);
  return launched("gvm_nn_adam");
}
