// Stockham FFTs in LDS (e^{+2 pi i}, unnormalised), shared by the forward
// model's image-to-grid transform and the adjoint's grid-to-image transform.
#pragma once

#include <hip/hip_runtime.h>

namespace gvm {

// ---------------------------------------------------------------------------
// Stockham FFT in LDS
// ---------------------------------------------------------------------------
// Complex product, each operation rounded (no multiply-add contraction), so
// the transform's rounding does not depend on how the compiler schedules the
// unrolled stages of a given batching.
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
#pragma clang fp contract(off)
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// One Stockham stage (radix R, current sub-transform length NS) over B
// transforms of length N held in LDS.  COLS selects the LDS layout:
//   rows: element (t, p) at t * N + p;  cols: element (t, p) at p * B + t.
// All reads of the stage complete (barrier) before any write, so the stage
// runs in place in one buffer.
// Radix-4 butterfly in place: b_m = sum_r a_r e^{+2 pi i r m / 4}.
__device__ __forceinline__ void bfly4(float2& a0, float2& a1, float2& a2, float2& a3) {
#pragma clang fp contract(off)
  const float2 s02 = make_float2(a0.x + a2.x, a0.y + a2.y);
  const float2 d02 = make_float2(a0.x - a2.x, a0.y - a2.y);
  const float2 s13 = make_float2(a1.x + a3.x, a1.y + a3.y);
  const float2 d13 = make_float2(a1.x - a3.x, a1.y - a3.y);
  a0 = make_float2(s02.x + s13.x, s02.y + s13.y);
  a2 = make_float2(s02.x - s13.x, s02.y - s13.y);
  // i * d13 = (-d13.y, d13.x)
  a1 = make_float2(d02.x - d13.y, d02.y + d13.x);
  a3 = make_float2(d02.x + d13.y, d02.y - d13.x);
}

// One Stockham stage (radix R = 2, 4 or 8, current sub-transform length NS)
// over B transforms of length N held in LDS.  A thread takes butterflies
// q = threadIdx.x + b T while q < B N / R.
template <int N, int B, bool COLS, int R, int NS, int T>
__device__ __forceinline__ void stockham_stage(float2* lds, const float2* __restrict__ tw) {
#pragma clang fp contract(off)
  constexpr int NB = B * N / R;          // butterflies in this stage
  constexpr int BPT = (NB + T - 1) / T;  // per thread (the last round may be partial)
  constexpr int STRIDE = N / R;
  float2 v[BPT][R];
  int base_t[BPT], out_j[BPT];
#pragma unroll
  for (int b = 0; b < BPT; b++) {
    const int q = threadIdx.x + b * T;
    if (NB % T != 0 && q >= NB) break;
    const int t = COLS ? (q % B) : (q / STRIDE);
    const int j = COLS ? (q / B) : (q % STRIDE);
    const int k = j % NS;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int p = j + r * STRIDE;
      v[b][r] = COLS ? lds[p * B + t] : lds[t * N + p];
    }
    if (NS > 1) {
#pragma unroll
      for (int r = 1; r < R; r++) {
        const int e = r * k * (N / (NS * R));
        v[b][r] = cmul(v[b][r], tw[e]);
      }
    }
    if constexpr (R == 8) {
      // b_m = sum_r a_r e^{+2 pi i r m / 8}: radix-4 over the even and the
      // odd inputs, then b_m = E_m + W^m O_m, b_{m+4} = E_m - W^m O_m with
      // W = e^{+2 pi i / 8}
      float2 e0 = v[b][0], e1 = v[b][2], e2 = v[b][4], e3 = v[b][6];
      float2 o0 = v[b][1], o1 = v[b][3], o2 = v[b][5], o3 = v[b][7];
      bfly4(e0, e1, e2, e3);
      bfly4(o0, o1, o2, o3);
      constexpr float h = 0.70710678118654752f;  // sqrt(1/2)
      const float2 w1 = make_float2(h * (o1.x - o1.y), h * (o1.x + o1.y));     // W o1
      const float2 w2 = make_float2(-o2.y, o2.x);                              // i o2
      const float2 w3 = make_float2(-h * (o3.x + o3.y), h * (o3.x - o3.y));    // W^3 o3
      v[b][0] = make_float2(e0.x + o0.x, e0.y + o0.y);
      v[b][4] = make_float2(e0.x - o0.x, e0.y - o0.y);
      v[b][1] = make_float2(e1.x + w1.x, e1.y + w1.y);
      v[b][5] = make_float2(e1.x - w1.x, e1.y - w1.y);
      v[b][2] = make_float2(e2.x + w2.x, e2.y + w2.y);
      v[b][6] = make_float2(e2.x - w2.x, e2.y - w2.y);
      v[b][3] = make_float2(e3.x + w3.x, e3.y + w3.y);
      v[b][7] = make_float2(e3.x - w3.x, e3.y - w3.y);
    } else if constexpr (R == 4) {
      bfly4(v[b][0], v[b][1], v[b][2], v[b][3]);
    } else {
      const float2 a0 = v[b][0], a1 = v[b][1];
      v[b][0] = make_float2(a0.x + a1.x, a0.y + a1.y);
      v[b][1] = make_float2(a0.x - a1.x, a0.y - a1.y);
    }
    base_t[b] = t;
    out_j[b] = (j / NS) * NS * R + k;
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < BPT; b++) {
    if (NB % T != 0 && threadIdx.x + b * T >= NB) break;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int p = out_j[b] + r * NS;
      if (COLS)
        lds[p * B + base_t[b]] = v[b][r];
      else
        lds[base_t[b] * N + p] = v[b][r];
    }
  }
  __syncthreads();
}

template <int N>
constexpr int log2_of() {
  int l = 0;
  int n = N;
  while (n > 1) {
    n >>= 1;
    l++;
  }
  return l;
}

// Radix of the stage that starts at sub-transform length NS: radix-8 stages
// first, then radix-4 (two when log2 N = 1 mod 3, one when 2 mod 3).
template <int N, int NS>
constexpr int stage_radix() {
  constexpr int left = log2_of<N>() - log2_of<NS>();  // log2 of what remains
  if (left % 3 == 0) return 8;
  if (left % 3 == 1) return left >= 4 ? (left == 4 ? 4 : 8) : 2;
  return left == 2 ? 4 : 8;
}

template <int N, int B, bool COLS, int NS, int T>
__device__ __forceinline__ void fft_stages(float2* lds, const float2* __restrict__ tw) {
  if constexpr (NS < N) {
    constexpr int R = stage_radix<N, NS>();
    stockham_stage<N, B, COLS, R, NS, T>(lds, tw);
    fft_stages<N, B, COLS, NS * R, T>(lds, tw);
  }
}

// N-point transforms (e^{+2 pi i}, unnormalised) of the B sequences in LDS:
// N = 8^a 4^b with b <= 2 (2 for N = 2), e.g. 1024 = 8 8 4 4.
template <int N, int B, bool COLS, int T>
__device__ __forceinline__ void fft_lds(float2* lds, const float2* __restrict__ tw) {
  fft_stages<N, B, COLS, 1, T>(lds, tw);
}

}  // namespace gvm
