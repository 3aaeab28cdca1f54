// DChi2 adjoint by gridding and FFT on gfx950.
//
// The adjoint's sums G(i,j) = Re sum_v c_v e^{i phi_v(i,j)}, c_v = w_v
// conj(Vr_v), phi = 2 pi (x_j u_v + y_i v_v + (z_ij - 1) w_v)
// (src/functions.cu:3698-3791) are a non-uniform discrete Fourier transform.
// Here it is evaluated as one: every visibility is spread onto a uv grid
// oversampled twice with a narrow kernel, the grid is transformed with FFTs
// and the image is divided by the kernel's transform (the method of Dutt and
// Rokhlin, SIAM J. Sci. Comput. 14 (1993) 1368; a kernel exp(-polynomial) in the
// manner of the "exponential of semicircle" of Barnett, Magland and af
// Klinteberg, SIAM J. Sci. Comput. 41 (2019) C479).  The work falls from 4 N^2 Nvis flop (the GEMM of
// gvm_adjoint.hip) to about 81 K grid updates per visibility and K FFTs of
// (2N)^2; all arithmetic is FP32 or better, and the approximation (9 taps at
// twice oversampling, 2.3e-8) is under FP32 rounding.
//
// w term.  With t = w / W in [-1, 1] and zeta = 2 pi W (z - 1), the
// Jacobi-Anger expansion e^{i zeta t} = J_0(zeta) + 2 sum_k i^k J_k(zeta)
// T_k(t) turns the w phase into K planes: plane k grids i^k c T_k(t) and is
// weighted by J_k(zeta) per pixel.  K is the smallest count whose truncation
// 2 (|zeta|/2)^K / K! over the pixels on the mask is below kPlaneTol.  (The
// pixel coordinate is the exact z - 1, not the per-axis split of the GEMM.)
//
// Real output.  Only Re is wanted, so a visibility with u beyond the grid's
// Nyquist column is folded to the conjugate point, only columns X = 0 .. N of
// the 2N x 2N grid exist, and the second transform is complex-to-real.
//
// Steps of one evaluation:
//  1. spread_kernel   one wave per work item (at most `chunk` visibilities of
//                     one 8 x 8 tile of the grid, sorted at set-up): the
//                     item's 16 x 16 subgrid of every plane as a product on
//                     the FP32 MFMA units, sum_v ky_v(row) [kx_v(col) c_v T_k];
//  2. merge_kernel    subgrids of tiles with several items, summed in FP64;
//  3. cols_kernel     gathers the (up to four) subgrids that overlap each grid
//                     cell and transforms the columns (2N points);
//  4. rows_kernel     per image row: complex-to-real transforms of the K
//                     planes, their combination, the kernel correction,
//                     -fg PB, the chain rule (the GEMM form's epilogue).
// Every sum has a fixed order, so results are reproducible bit for bit.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "gvm_fft.h"
#include "gvm_internal.h"

namespace gvm {

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr double kPi = 3.14159265358979323846;
constexpr int kTaps = 9;                 // kernel width in cells of the 2N grid
constexpr double kPlaneTol = 5e-8;       // truncation of the w expansion
constexpr int kMaxPlanes = 32;
constexpr int kMaxTerms = 40;            // of a plane weight's series (32 planes need 31)
constexpr int kPlaneGroup = 8;           // planes one spread launch accumulates
constexpr int kSub = 512;                // floats of a 16 x 16 complex subgrid
constexpr long kGroupRows = 1L << 27;    // rows sorted together at set-up
constexpr size_t kBatchBytes = 512u << 20;  // workspace one batch of slices aims at

// The spreading kernel: 2^-P(v), v = (d / 4.5)^2, 0 beyond 4.5 cells.  P's
// coefficients minimise the aliased part of the kernel's transform over the
// pixels kept (least squares over |offset| <= N / 2 and the first six images
// of the band): 2.3e-8 rms, 3.9e-8 at most, where the exponential of semicircle
// of the same width (beta 20.7) has 1.3e-8 and 5.0e-8 but takes a square root
// and a reciprocal more per value.
constexpr float kInvHalf = (float)(2.0 / kTaps);
constexpr double kLog2e = 1.44269504088896340736;
constexpr float kP1 = (float)(10.596313090281376 * kLog2e);
constexpr float kP2 = (float)(2.670875389609385 * kLog2e);
constexpr float kP3 = (float)(1.278424264908622 * kLog2e);
constexpr float kP4 = (float)(0.7525254439992803 * kLog2e);
constexpr float kP5 = (float)(0.31046272601257235 * kLog2e);
constexpr float kP6 = (float)(0.4732201062869989 * kLog2e);
__device__ __forceinline__ float spread_value(float d) {
  const float u = d * kInvHalf, v = u * u;
  float p = fmaf(v, kP6, kP5);
  p = fmaf(v, p, kP4);
  p = fmaf(v, p, kP3);
  p = fmaf(v, p, kP2);
  p = fmaf(v, p, kP1);
  const float e = __builtin_amdgcn_exp2f(-(v * p));
  return v <= 1.0f ? e : 0.0f;
}

int blocks_for(long n) { return (int)std::max(1L, std::min<long>((n + 255) / 256, 8192)); }

// ---------------------------------------------------------------------------
// set-up: visibilities of a group of slices sorted by (slice, tile)
// ---------------------------------------------------------------------------

// Position of a visibility on the oversampled half grid.
struct GridPos {
  int bx, by;     // nearest cell, bx in [0, N], by in [0, 2N)
  double dx, dy;  // offset from it, in [-1/2, 1/2]
  bool conj;      // folded: the conjugate point
};

__device__ __forceinline__ GridPos grid_pos(float4 p, int N) {
  // turns per pixel, exact (gvm_add_visibilities splits them into two floats)
  const double a = (double)p.x + (double)p.y;
  double b = (double)p.z + (double)p.w;
  const double L = 2.0 * N;
  GridPos g;
  const double X = (a - floor(a)) * L;
  double bx = rint(X);
  g.dx = X - bx;
  g.conj = bx > (double)N;
  if (g.conj) {
    bx = L - bx;
    g.dx = -g.dx;
    b = -b;
  }
  const double Y = (b - floor(b)) * L;
  const double by = rint(Y);
  g.dy = Y - by;
  g.bx = (int)bx;
  g.by = (int)by & (2 * N - 1);
  return g;
}

// max |w| over rows with a weight, as float bits; an infinite or NaN w counts
// with any weight (it makes the sums NaN) and is larger than any number
__global__ __launch_bounds__(256) void wmax_kernel(const SliceDev* __restrict__ tab,
                                                   unsigned int* __restrict__ out) {
  const SliceDev& sd = tab[blockIdx.y];
  unsigned int m = 0u;
  for (long v = blockIdx.x * 256L + threadIdx.x; v < sd.nvis; v += (long)gridDim.x * 256) {
    const unsigned int b = __float_as_uint(ldg(sd.wcoord + v)) & 0x7fffffffu;
    if (ldg(sd.weight + v) != 0.0f || b >= 0x7f800000u) m = max(m, b);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned int)__shfl_xor((int)m, o, 64));
  if ((threadIdx.x & 63) == 0 && m) atomicMax(out, m);
}

// keys of the rows of slice s0 + blockIdx.y; off[] are the slices' first rows
// within the group
__global__ __launch_bounds__(256) void plan_keys_kernel(const SliceDev* __restrict__ tab, int s0,
                                                        const unsigned int* __restrict__ off, int N,
                                                        unsigned int* __restrict__ keys,
                                                        unsigned int* __restrict__ ids) {
  const SliceDev& sd = tab[s0 + blockIdx.y];
  const unsigned int ntiles = (unsigned int)(N / 8 + 1) * (N / 4);
  const unsigned int o = off[blockIdx.y];
  for (long v = blockIdx.x * 256L + threadIdx.x; v < sd.nvis; v += (long)gridDim.x * 256) {
    const GridPos g = grid_pos(ldg(sd.phs + v), N);
    keys[o + v] = blockIdx.y * ntiles + (unsigned int)(g.bx >> 3) * (N / 4) + (g.by >> 3);
    ids[o + v] = o + (unsigned int)v;
  }
}

// Sorted records: (dx, dy, w, weight) and (row of its slice, cell within the
// tile and fold), and the phase-centre rotation when the image is not centred
// on it.
__global__ __launch_bounds__(256) void plan_records_kernel(
    const SliceDev* __restrict__ tab, int s0, const unsigned int* __restrict__ off, int N, long n,
    const unsigned int* __restrict__ keys, const unsigned int* __restrict__ ids,
    int shift_x, int shift_y, float4* __restrict__ rec, uint2* __restrict__ meta,
    float2* __restrict__ rot) {
  const unsigned int ntiles = (unsigned int)(N / 8 + 1) * (N / 4);
  for (long p = blockIdx.x * 256L + threadIdx.x; p < n; p += (long)gridDim.x * 256) {
    const unsigned int s = keys[p] / ntiles;
    const SliceDev& sd = tab[s0 + s];
    const unsigned int v = ids[p] - off[s];
    const float4 ph = ldg(sd.phs + v);
    const GridPos g = grid_pos(ph, N);
    const float w = ldg(sd.wcoord + v);
    rec[p] = make_float4((float)g.dx, (float)g.dy, g.conj ? -w : w, ldg(sd.weight + v));
    meta[p] = make_uint2(v, (unsigned int)(g.bx & 7) | (g.by & 7) << 3 | (g.conj ? 64u : 0u));
    if (rot) {
      double r = ((double)ph.x + (double)ph.y) * shift_x + ((double)ph.z + (double)ph.w) * shift_y;
      r -= rint(r);
      double sn, cs;
      sincospi(2.0 * r, &sn, &cs);
      rot[p] = make_float2((float)cs, (float)sn);
    }
  }
}

// start[k] = the first sorted row with key >= k, k in [0, nkeys]
__global__ __launch_bounds__(256) void tile_starts_kernel(const unsigned int* __restrict__ keys,
                                                          long n, long nkeys,
                                                          unsigned int* __restrict__ start) {
  for (long k = blockIdx.x * 256L + threadIdx.x; k <= nkeys; k += (long)gridDim.x * 256) {
    long lo = 0, hi = n;
    while (lo < hi) {
      const long m = (lo + hi) >> 1;
      if ((long)keys[m] < k)
        lo = m + 1;
      else
        hi = m;
    }
    start[k] = (unsigned int)lo;
  }
}

// items per tile, and whether it has several (0 past the last tile)
__global__ __launch_bounds__(256) void item_counts_kernel(const unsigned int* __restrict__ start,
                                                          long nkeys, int chunk,
                                                          unsigned int* __restrict__ cnt,
                                                          unsigned int* __restrict__ several) {
  for (long k = blockIdx.x * 256L + threadIdx.x; k <= nkeys; k += (long)gridDim.x * 256) {
    const unsigned int c =
        k < nkeys ? (start[k + 1] - start[k] + (unsigned int)chunk - 1) / (unsigned int)chunk : 0u;
    cnt[k] = c;
    several[k] = c > 1 ? 1u : 0u;
  }
}

// Items of tile k at [islot[k], islot[k + 1]): (first row, rows, slice, .); .w of
// item i of a slice is the item to take i-th: those of half a chunk or
// more first, so that short ones fill the launch's end (which of two comes first
// does not matter).  full[], rest[]: how many of a slice have been placed.  islot[k]
// becomes tile_slot[k] (-1 for a tile without rows); merge mslot[k]
// is tile k's when it has several items.
__global__ __launch_bounds__(256) void items_kernel(const unsigned int* __restrict__ start,
                                                    const unsigned int* __restrict__ islot,
                                                    const unsigned int* __restrict__ mslot,
                                                    long nkeys, int chunk, long row0,
                                                    unsigned int ntiles, int s0,
                                                    unsigned int item0, unsigned int merge0,
                                                    unsigned int* __restrict__ full,
                                                    unsigned int* __restrict__ rest,
                                                    long4* __restrict__ items,
                                                    int2* __restrict__ merges,
                                                    int* __restrict__ tile_slot) {
  for (long k = blockIdx.x * 256L + threadIdx.x; k < nkeys; k += (long)gridDim.x * 256) {
    const unsigned int a = islot[k], e = islot[k + 1];
    tile_slot[k] = e > a ? (int)a : -1;
    if (e > a + 1) merges[mslot[k] - merge0] = make_int2((int)a, (int)(e - a));
    const long first = start[k], last = start[k + 1];
    for (unsigned int i = a; i < e; i++) {
      const long b = first + (long)(i - a) * chunk;
      long4 it;
      it.x = row0 + b;
      it.y = min((long)chunk, last - b);
      const unsigned int s = (unsigned int)(k / ntiles);
      it.z = s0 + (long)s;
      long4* o = items + (i - item0);
      o->x = it.x;
      o->y = it.y;
      o->z = it.z;
      const unsigned int at = it.y >= chunk / 2 ? islot[(long)s * ntiles] + atomicAdd(full + s, 1u)
                                                : islot[(long)(s + 1) * ntiles] - 1 - atomicAdd(rest + s, 1u);
      items[at - item0].w = (long)i;
    }
  }
}

// the slices' first items and merges
__global__ void pick_kernel(const unsigned int* __restrict__ islot,
                            const unsigned int* __restrict__ mslot, unsigned int ntiles, int nsl,
                            uint2* __restrict__ out) {
  for (int s = threadIdx.x; s <= nsl; s += blockDim.x)
    out[s] = make_uint2(islot[(long)s * ntiles], mslot[(long)s * ntiles]);
}

// ---------------------------------------------------------------------------
// 1. spreading
// ---------------------------------------------------------------------------
// One wave per item.  64 rows at a time: each lane loads one row, forms c
// (scaled as the GEMM form scales it, by a power of two undone at the end) and
// leaves it in LDS; then four rows per step, lane l evaluates the kernel of
// row l / 16 at grid row and column l % 16, and the planes' products go to
// v_mfma_f32_16x16x4_f32 (A: ky, B: kx c T_k; real and imaginary parts).
// Per step and wave 2 NP MFMAs of 32 cycles against about 50 VALU instructions,
// which take as long at NP = 4: the next step's operands are formed between this
// step's MFMAs (in turn: 128 us for 1.76 M visibilities, so: 117; the MFMAs alone
// would take 46).  A block is one wave (four held a CU until the longest was done).
template <int NP>
__global__ __launch_bounds__(64) void spread_kernel(
    const long4* __restrict__ items, long slot0, const float4* __restrict__ rec,
    const uint2* __restrict__ meta, const float2* __restrict__ rot,
    const SliceDev* __restrict__ tab, const unsigned int* __restrict__ cmaxs, double inv_w, int k0,
    int nplanes, float* __restrict__ part) {
  __shared__ float4 sa[64];  // (dx, dy, c)
  __shared__ float2 sb[64];  // the row's cell within the subgrid
  __shared__ float st[64][(NP + 3) / 4 * 4];  // T_k0 .. of each row
  const int lane = threadIdx.x, item = (int)(items[blockIdx.x].w - slot0);
  const long4 it = items[item];
  const float2* __restrict__ vr = tab[it.z].vr;
  const float scale = ldexpf(1.0f, p_scale_exponent(__uint_as_float(cmaxs[it.z])));
  const float q = (float)(lane & 15);
  // 64 rows accumulate in the MFMAs, the item's (at most eight) sums of 64 in a
  // second FP32 sum: one long FP32 sum would round more than the whole
  // transform does
  f32x4_t tre[NP], tim[NP];
#pragma unroll
  for (int k = 0; k < NP; k++) tre[k] = tim[k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // the next 64 rows are loaded (their residuals too: a dependent gather)
  // while these are spread
  const int rows = (int)it.y;
  auto load_row = [&](int i, float4* r, uint2* m) {
    const long p = it.x + min(i, rows - 1);
    *r = rec[p];
    *m = meta[p];
  };
  float4 r, rn;
  uint2 m, mn;
  load_row(lane, &r, &m);
  float2 v = ldg(vr + m.x);
  load_row(64 + lane, &rn, &mn);
  for (int b = 0; b < rows; b += 64) {
    const int cnt = min(64, rows - b);
    f32x4_t re[NP], im[NP];
#pragma unroll
    for (int k = 0; k < NP; k++) re[k] = im[k] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    float2 c = make_float2(4.f, 4.f);
    double t = 0.0;
    if (lane < cnt) {
      float cr = r.w * v.x, ci = -(r.w * v.y);
      if (rot) {
        const float2 e = rot[it.x + b + lane];
        const float x = cr * e.x - ci * e.y;
        ci = cr * e.y + ci * e.x;
        cr = x;
      }
      if (m.y & 64u) ci = -ci;
      a = make_float4(r.x, r.y, cr * scale, ci * scale);
      c = make_float2((float)(4 + (m.y & 7u)), (float)(4 + ((m.y >> 3) & 7u)));
      t = fmin(1.0, fmax(-1.0, (double)r.z * inv_w));  // rows without weight may lie beyond W
    }
    if (b + 64 < rows) {
      r = rn;
      m = mn;
      v = ldg(vr + m.x);
      load_row(b + 128 + lane, &rn, &mn);
    }
    __builtin_amdgcn_wave_barrier();
    sa[lane] = a;
    sb[lane] = c;
    double ta = 1.0, tb = t;
    for (int k = 0; k < k0; k++) {
      const double tn = 2.0 * t * tb - ta;
      ta = tb;
      tb = tn;
    }
#pragma unroll
    for (int k = 0; k < NP; k++) {
      st[lane][k] = (float)ta;
      const double tn = 2.0 * t * tb - ta;
      ta = tb;
      tb = tn;
    }
    __builtin_amdgcn_wave_barrier();
    // eight rows per turn: while four are multiplied the operands of the next four
    // are formed, from LDS values read a step before that (rows past cnt are zero)
    float4 va;
    float2 vb;
    float vt[NP], ky[2], br[2][NP], bi[2][NP];
    auto fetch = [&](int s) {
      const int j = (s & 63) + (lane >> 4);
      va = sa[j];
      vb = sb[j];
#pragma unroll
      for (int k = 0; k < NP; k++) vt[k] = st[j][k];
    };
    auto operands = [&](int h) {
      const float kx = spread_value((q - vb.x) - va.x);
      ky[h] = spread_value((q - vb.y) - va.y);
      const float ux = kx * va.z, ui = kx * va.w;
#pragma unroll
      for (int k = 0; k < NP; k++) {
        // even planes grid c T_k, odd ones -i c T_k
        br[h][k] = (k & 1) ? ui * vt[k] : ux * vt[k];
        bi[h][k] = (k & 1) ? -(ux * vt[k]) : ui * vt[k];
      }
    };
    auto multiply = [&](int h) {
#pragma unroll
      for (int k = 0; k < NP; k++) {
        re[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(ky[h], br[h][k], re[k], 0, 0, 0);
        im[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(ky[h], bi[h][k], im[k], 0, 0, 0);
      }
    };
    fetch(0);
    operands(0);
    fetch(4);
    for (int s = 0; s < cnt; s += 8) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        __builtin_amdgcn_sched_barrier(0);
        multiply(h);
        operands(1 - h);
        fetch(s + 4 * h + 8);
#pragma unroll
        for (int k = 0; k < 2 * NP; k++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);            // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, 40 / (2 * NP) + 2, 0);  // VALU
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // LDS reads
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int k = 0; k < NP; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        tre[k][e] += re[k][e];
        tim[k][e] += im[k][e];
      }
  }
  // subgrid layout: [plane][column half][16 rows][8 columns] complex
  const int col = lane & 15, row = 4 * (lane >> 4);
#pragma unroll
  for (int k = 0; k < NP; k++) {
    if (k0 + k >= nplanes) break;
    float2* o = (float2*)(part + ((long)item * nplanes + k0 + k) * kSub) + (col >> 3) * 128 +
                (col & 7);
#pragma unroll
    for (int e = 0; e < 4; e++) o[(row + e) * 8] = make_float2(tre[k][e], tim[k][e]);
  }
}

// 2. The items of a tile with several, summed into its first one, in item
// order, in FP64.
__global__ __launch_bounds__(256) void merge_kernel(const int2* __restrict__ merges, int slot0,
                                                    int nplanes, float* __restrict__ part) {
  const int2 mg = merges[blockIdx.x];  // (first item, items)
  const int cnt = mg.y;
  const long stride = (long)nplanes * kSub;
  float* p = part + (long)(mg.x - slot0) * stride + blockIdx.y * 256 + threadIdx.x;
  double s = 0.0;
  int i = 0;
  for (; i + 16 <= cnt; i += 16) {
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = p[(long)(i + u) * stride];
#pragma unroll
    for (int u = 0; u < 16; u++) s += (double)v[u];
  }
  for (; i < cnt; i++) s += (double)p[(long)i * stride];
  *p = (float)s;
}

// ---------------------------------------------------------------------------
// 3. columns
// ---------------------------------------------------------------------------
// Tile column X_t covers columns 8 X_t - 4 .. 8 X_t + 11, so grid column X
// lies in the left half of tile column (X + 4) / 8 and in the right half of
// the one before; likewise tile rows and Y, which wraps at 2N.  A cell is the
// sum of up to four subgrids.

// Four of the columns beyond an end of the half grid (X < 0 or X > N), folded:
// minus the conjugate cell (mx, -Y).  ss: the slots of tile columns txb and txb - 1,
// which hold these cells too.
template <int N>
__device__ __forceinline__ float2 folded_cell(const float2* __restrict__ part,
                                              const int (*ss)[N / 4], int txb, int nplanes,
                                              int plane, int mx, int Y) {
  const int nty = N / 4, tx = (mx + 4) >> 3;
  const int My = -Y & (2 * N - 1);
  const int ty = ((My + 4) >> 3) & (nty - 1), c = (mx + 4) & 7, r = (My + 4) & 7;
  float2 s = make_float2(0.f, 0.f);
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int tc = tx - (u >> 1);
    if (tc < 0 || tc > N / 8 || tc > txb || tc < txb - 1) continue;
    const int i = ss[txb - tc][(ty - (u & 1)) & (nty - 1)];
    if (i < 0) continue;
    const float2 v = part[((long)i * nplanes + plane) * (kSub / 2) + (u >> 1) * 128 +
                          (r + (u & 1) * 8) * 8 + c];
    s.x += v.x;
    s.y -= v.y;
  }
  return s;
}

// H[slice][plane][image row][X], X in [0, N], rows of `pitch` values: BC
// columns (a divisor of four, so they share their two tile columns) of one
// plane per block.  The tiles' slots are staged in LDS and two columns are
// loaded at a time, so that a thread keeps sixteen loads in flight: a gather
// through slots in memory waited twice per cell and took 97 us at 1024^2, staged
// 45, and 42 since blocks without rows leave at the edges too.
template <int N, int BC, int T>
__global__ __launch_bounds__(T) void grid_cols_kernel(const float2* __restrict__ part,
                                                      const int* __restrict__ tile_slot, int slot0,
                                                      int nplanes, const float2* __restrict__ tw,
                                                      int pitch, float2* __restrict__ Hbuf) {
  constexpr int L = 2 * N, NTY = N / 4, CP = BC / 2;
  __shared__ float2 lds[BC * L];
  __shared__ int ss[2][NTY];
  // consecutive column blocks, which write the same lines of H, on one XCD; column
  // N by itself (33 blocks on every XCD for 257 would take a third round)
  constexpr int PER = N / BC / 8;
  const int X0 = blockIdx.x < N / BC ? ((blockIdx.x % 8) * PER + blockIdx.x / 8) * BC : N;
  const int plane = blockIdx.y, sl = blockIdx.z;
  const int* slot = tile_slot + (long)sl * (N / 8 + 1) * NTY;
  const int tx = (X0 + 4) >> 3;
  // a block without any row's subgrid needs no transform
  // (cells beyond either end of the half grid lie in the same two tile columns)
  int any = 0;
  for (int y = threadIdx.x; y < 2 * NTY; y += T) {
    const int h = y / NTY, t = tx - h;
    const int s = t >= 0 && t <= N / 8 ? slot[t * NTY + y % NTY] : -1;
    // (the smallest valid index where there is none: loaded, not used)
    ss[h][y % NTY] = s < 0 ? -1 : s - slot0;
    any |= s >= 0;
  }
  any = __syncthreads_or(any);
  float2* H = Hbuf + ((long)sl * nplanes + plane) * (long)N * pitch;
  if (any) {
    const float4* p4 = (const float4*)part;
    const long per_item = (long)nplanes * (kSub / 4), at_plane = (long)plane * (kSub / 4);
    const int c0 = (X0 + 4) & 7;
    constexpr int U = 4, IT = CP * L / T;
    static_assert(IT * T == CP * L && IT % U == 0, "whole rounds");
    for (int i0 = 0; i0 < IT; i0 += U) {
      float4 v[U][4];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int idx = threadIdx.x + (i0 + u) * T;
        const int t = idx % CP, Y = idx / CP;
        const int ty = ((Y + 4) >> 3) & (NTY - 1), r = (Y + 4) & 7;
        const int c = (c0 >> 1) + t;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int s = ss[q >> 1][(ty - (q & 1)) & (NTY - 1)];
          v[u][q] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (s >= 0)
            v[u][q] = p4[s * per_item + at_plane + (q >> 1) * 64 + (r + (q & 1) * 8) * 4 + c];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int idx = threadIdx.x + (i0 + u) * T;
        float4 s;
        s.x = (v[u][0].x + v[u][1].x) + (v[u][2].x + v[u][3].x);
        s.y = (v[u][0].y + v[u][1].y) + (v[u][2].y + v[u][3].y);
        s.z = (v[u][0].z + v[u][1].z) + (v[u][2].z + v[u][3].z);
        s.w = (v[u][0].w + v[u][1].w) + (v[u][2].w + v[u][3].w);
        ((float4*)lds)[idx] = s;
      }
    }
    __syncthreads();
    // cells beyond either end are the conjugates of cells inside
    if (X0 <= 4 || X0 + BC - 1 >= N - 4) {
      for (int idx = threadIdx.x; idx < BC * L; idx += T) {
        const int X = X0 + idx % BC, Y = idx / BC;
        const int mx = X >= 1 && X <= 4 ? -X : X >= N - 4 && X < N ? L - X : 0;
        if (mx == 0) continue;
        const float2 m = folded_cell<N>(part, ss, tx, nplanes, plane, mx, Y);
        lds[idx].x += m.x;
        lds[idx].y += m.y;
      }
      __syncthreads();
    }
    fft_lds<L, BC, true, T>(lds, tw);
  }
  // image row i is frequency row i - N / 2 (mod 2N)
  for (int idx = threadIdx.x; idx < CP * N; idx += T) {
    const int t = idx % CP, i = idx / CP, X = X0 + 2 * t;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (any) v = ((const float4*)lds)[((i - N / 2) & (L - 1)) * CP + t];
    if (X <= N) *(float4*)(H + (long)i * pitch + X) = v;  // (column N + 1 is padding)
  }
}

// ---------------------------------------------------------------------------
// 4. rows
// ---------------------------------------------------------------------------
struct RowsArgs {
  const float2* H;
  int pitch, nplanes, terms;
  const float2* tw;   // e^{2 pi i k / N}
  const float2* tw2;  // e^{2 pi i k / 2N}
  const double* corr; // 1 / the kernel's transform per axis offset
  const double* wcoef;
  const SliceDev* tab;
  int s0, nsl;        // slices [s0, s0 + nsl); H holds these
  const unsigned int* cmaxs;
  const float* noise;
  float noise_cut, fg_scale, threshold;
  const float* gcf;
  int normalize, flag_opt;
  int set;            // images of a result to be written whole, 0 to add to it
  double wz;          // 2 pi W
  double dx, dy;      // radians per pixel
  int x0, y0;         // phase centre
  const float* I;
  float* result;
  float* each;        // per-slice d, or none (one slice: straight to result)
};

// One slice's contribution d at pixel k to the running gradient r: the chain
// rule of DChi2_total_I_nu_0 / DChi2_total_alpha (src/functions.cu:4000-4024,
// 3968-3998), in float.
__device__ __forceinline__ float chain_rule(float r, float d, float nudiv, float i0, float alpha,
                                            const RowsArgs& a) {
  const float dI = powf(nudiv, alpha);
  if ((a.flag_opt & 1) == 0) return r + d * dI;
  if (i0 > a.threshold) return r + d * (i0 * dI * a.fg_scale * logf(nudiv));
  return r;
}

// One block per image row; B planes are transformed together.  The transform
// of 2N real values from N + 1 complex ones runs as one complex transform of N
// points (even outputs in the real part, odd ones in the imaginary part), whose
// inputs X and N - X need the same two values.  A plane's weight at a pixel is
// zeta^k times a power series in zeta^2; the series' coefficients are read from
// LDS, once for all of a thread's pixels (from memory, per pixel, they were two
// thirds of the kernel's loads: 310 us at 2048^2 with 6 planes, now 185).
template <int N, int B, int T>
__global__ __launch_bounds__(T, 4) void grid_rows_kernel(RowsArgs a) {
  __shared__ float2 lds[B * N];
  __shared__ double sc[B * kMaxTerms];
  constexpr int PP = (N / 2 + T - 1) / T;  // column pairs per thread
  const int i = blockIdx.x;
  const long n = (long)N * N;
  const float* noise = a.noise + (long)i * N;
  bool on[PP][2];
  bool some = false;
#pragma unroll
  for (int u = 0; u < PP; u++) {
    const int cp = threadIdx.x + u * T;
#pragma unroll
    for (int e = 0; e < 2; e++) {
      on[u][e] = cp < N / 2 && noise[2 * cp + e] < a.noise_cut;
      some |= on[u][e];
    }
  }
  some = __syncthreads_or(some);
  if (a.set && !a.each)  // zero outside the mask, and the other images
    for (int m = 0; m < a.set; m++) {
#pragma unroll
      for (int u = 0; u < PP; u++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int cp = threadIdx.x + u * T;
          if (cp < N / 2 && (m != (a.flag_opt & 1) || !on[u][e]))
            a.result[m * n + (long)i * N + 2 * cp + e] = 0.0f;
        }
    }
  if (!some) return;
  double zeta[PP][2];
#pragma unroll
  for (int u = 0; u < PP; u++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int j = 2 * ((int)threadIdx.x + u * T) + e;
      const double x = (j - a.x0) * a.dx, y = (i - a.y0) * a.dy;
      const double r2 = x * x + y * y;
      zeta[u][e] = a.wz * (-r2 / (1.0 + sqrt(fmax(0.0, 1.0 - r2))));
    }
  const int s = blockIdx.y;
  double g[PP][2], zk[PP][2], z2[PP][2];
#pragma unroll
  for (int u = 0; u < PP; u++) {
    g[u][0] = g[u][1] = 0.0;
    zk[u][0] = zk[u][1] = 1.0;  // zeta^k
    z2[u][0] = zeta[u][0] * zeta[u][0];
    z2[u][1] = zeta[u][1] * zeta[u][1];
  }
  for (int k0 = 0; k0 < a.nplanes; k0 += B) {
    __syncthreads();  // the previous group's outputs have been read
#pragma unroll
    for (int b = 0; b < B; b++) {
      const int k = k0 + b;
      const float2* h = a.H + (((long)s * a.nplanes + min(k, a.nplanes - 1)) * N + i) * a.pitch;
#pragma unroll
      for (int u = 0; u < PP; u++) {
        const int X = threadIdx.x + u * T;
        if (X >= N / 2) break;
        float2 f = h[X], m = h[N - X];
        float2 z, y;  // inputs X and N - X; for X = 0: inputs 0 and N / 2
        if (X == 0) {
          const float2 c = h[N / 2];
          z = make_float2(f.x + m.x, f.x - m.x);
          y = make_float2(c.x, -c.y);
        } else {
          f = make_float2(0.5f * f.x, 0.5f * f.y);
          m = make_float2(0.5f * m.x, -0.5f * m.y);
          const float2 d = cmul(make_float2(f.x - m.x, f.y - m.y), a.tw2[X]);
          const float2 e = make_float2(f.x + m.x, f.y + m.y);
          z = make_float2(e.x - d.y, e.y + d.x);
          y = make_float2(e.x + d.y, d.x - e.y);
        }
        const bool in = k < a.nplanes;
        lds[b * N + X] = in ? z : make_float2(0.f, 0.f);
        lds[b * N + (X ? N - X : N / 2)] = in ? y : make_float2(0.f, 0.f);
      }
    }
    for (int c = threadIdx.x; c < B * a.terms; c += T)
      sc[c] = k0 * a.terms + c < a.nplanes * a.terms ? a.wcoef[k0 * a.terms + c] : 0.0;
    __syncthreads();
    fft_lds<N, B, false, T>(lds, a.tw);
    for (int b = 0; b < B && k0 + b < a.nplanes; b++) {
      const double* c = sc + b * a.terms;
      double w[PP][2];
#pragma unroll
      for (int u = 0; u < PP; u++) w[u][0] = w[u][1] = c[a.terms - 1];
      for (int m = a.terms - 2; m >= 0; m--) {
        const double cm = c[m];
#pragma unroll
        for (int u = 0; u < PP; u++)
#pragma unroll
          for (int e = 0; e < 2; e++) w[u][e] = fma(w[u][e], z2[u][e], cm);
      }
#pragma unroll
      for (int u = 0; u < PP; u++) {
        const int cp = threadIdx.x + u * T;
        const float2 z = lds[b * N + ((cp - N / 4) & (N - 1))];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          g[u][e] += (double)(e ? z.y : z.x) * zk[u][e] * w[u][e];
          zk[u][e] *= zeta[u][e];
        }
      }
    }
  }
  const SliceDev& sd = a.tab[a.s0 + s];
  const double inv_scale = ldexp(1.0, -p_scale_exponent(__uint_as_float(a.cmaxs[a.s0 + s])));
  const double inv_nvis = a.normalize ? 1.0 / (double)sd.nvis : 1.0;
  float* out = a.each ? a.each + (long)s * n : a.result + (a.flag_opt & 1) * n;
#pragma unroll
  for (int u = 0; u < PP; u++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      if (!on[u][e]) continue;
      const int j = 2 * ((int)threadIdx.x + u * T) + e;
      const long k = (long)i * N + j;
      const double gv = g[u][e] * (a.corr[i] * a.corr[j]);
      float sc = a.fg_scale * sd.pb[k];
      if (a.gcf) sc = sc * a.gcf[k];
      const float d = (float)(-(gv * inv_scale) * (double)sc * inv_nvis);
      out[k] = a.each ? d : chain_rule(a.set ? 0.0f : out[k], d, sd.nudiv, a.I[k], a.I[n + k], a);
    }
}

// Several slices: their d's into the result, one slice after the other as
// the reference's per-channel launches do (src/functions.cu:4456-4558).
__global__ __launch_bounds__(256) void chain_kernel(RowsArgs a, int N) {
  const long n = (long)N * N;
  for (long k = blockIdx.x * 256L + threadIdx.x; k < n; k += (long)gridDim.x * 256) {
    const bool on = a.noise[k] < a.noise_cut;
    for (int m = 0; m < a.set; m++)
      if (!on || m != (a.flag_opt & 1)) a.result[m * n + k] = 0.0f;
    if (!on) continue;
    const float i0 = a.I[k], alpha = a.I[n + k];
    float* out = a.result + (a.flag_opt & 1) * n + k;
    float r = a.set ? 0.0f : *out;
    for (int s = 0; s < a.nsl; s++)
      r = chain_rule(r, a.each[(long)s * n + k], a.tab[a.s0 + s].nudiv, i0, alpha, a);
    *out = r;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// 1 / integral of the kernel times cos(2 pi x d / 2N), for pixel offsets from
// the image centre: Gauss-Legendre over the (even) kernel's half width, with
// the constants as the device evaluates them.
std::vector<double> kernel_correction(int N) {
  constexpr int Q = 64;
  double x[Q], w[Q];
  for (int q = 0; q < Q; q++) {
    double t = std::cos(kPi * (q + 0.75) / (Q + 0.5)), d = 1.0;
    for (int it = 0; it < 100; it++) {
      double p0 = 1.0, p1 = t;
      for (int k = 2; k <= Q; k++) {
        const double p2 = ((2 * k - 1) * t * p1 - (k - 1) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      d = Q * (t * p1 - p0) / (t * t - 1.0);
      const double s = p1 / d;
      t -= s;
      if (std::fabs(s) < 1e-15) break;
    }
    x[q] = t;
    w[q] = 2.0 / ((1.0 - t * t) * d * d);
  }
  const double half = 0.5 * kTaps;
  double pos[Q], val[Q];
  for (int q = 0; q < Q; q++) {
    pos[q] = 0.5 * half * (x[q] + 1.0);
    const double u = pos[q] * (double)kInvHalf, v = u * u;
    const double p =
        v * (kP1 + v * (kP2 + v * (kP3 + v * (kP4 + v * (kP5 + v * (double)kP6)))));
    val[q] = half * w[q] * std::exp2(-p);
  }
  // cos(o t) by the recurrence in o
  double c0[Q], c1[Q], t2[Q];
  for (int q = 0; q < Q; q++) {
    c0[q] = 1.0;
    c1[q] = std::cos(kPi * pos[q] / N);
    t2[q] = 2.0 * c1[q];
  }
  std::vector<double> c(N);
  for (int o = 0; o <= N / 2; o++) {
    double s = 0.0;
    for (int q = 0; q < Q; q++) {
      s += val[q] * c0[q];
      const double next = t2[q] * c1[q] - c0[q];
      c0[q] = c1[q];
      c1[q] = next;
    }
    if (o < N / 2) c[N / 2 + o] = 1.0 / s;
    c[N / 2 - o] = 1.0 / s;
  }
  return c;
}

template <typename T>
bool device_array(T** p, size_t count) {
  *p = nullptr;
  if (hipMalloc((void**)p, sizeof(T) * std::max<size_t>(count, 1)) == hipSuccess) return true;
  (void)hipGetLastError();
  *p = nullptr;
  return false;
}

int row_pitch(int N) { return N + 8; }

}  // namespace

void release_grid_plan(GridPlan& g) {
  (void)hipFree(g.tables);
  (void)hipFree(g.lists);
  (void)hipFree(g.ws);
  g.tables = g.lists = g.ws = nullptr;
  g.bytes = 0;
  g.built = g.usable = false;
}

void free_grid_plan(GridPlan& g) {
  release_grid_plan(g);
  g = GridPlan{};
}

// W and the planes it needs.  *ok = false when they are too many, or there is an
// infinite or NaN w; the GEMM form then takes the call.
gvm_status probe_grid_plan(gvm_ctx* ctx, bool* ok) {
  *ok = false;
  GridPlan& g = ctx->gplan;
  if (g.probed) {
    *ok = g.applies;
    return GVM_OK;
  }
  hipStream_t st = ctx->stream;
  GVM_HIP_TRY(hipStreamSynchronize(st));
  free_grid_plan(g);
  const int nsl = (int)ctx->slices.size();
  const unsigned int zero = 0u;
  long vmax = 0;
  for (const Slice& s : ctx->slices) vmax = std::max(vmax, s.nvis);
  unsigned int wbits = 0;
  {
    Scratch sc(ctx);
    sc.add(sizeof(unsigned int));
    if (sc.reserve("adjoint plan")) return GVM_OK;
    unsigned int* wmax = sc.take<unsigned int>(1);
    GVM_HIP_TRY(hipMemcpyAsync(wmax, &zero, sizeof zero, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(wmax_kernel, dim3((unsigned)std::min<long>(256, (vmax + 255) / 256), nsl),
                       dim3(256), 0, st, ctx->slice_tab, wmax);
    GVM_CHECK_LAUNCH();
    GVM_HIP_TRY(hipMemcpyAsync(&wbits, wmax, sizeof wbits, hipMemcpyDeviceToHost, st));
    GVM_HIP_TRY(hipStreamSynchronize(st));
    sc.idle();
  }
  g.probed = true;
  if (wbits >= 0x7f800000u) return GVM_OK;  // an infinite or NaN w
  float W;
  static_assert(sizeof W == sizeof wbits, "float bits");
  __builtin_memcpy(&W, &wbits, sizeof W);
  const double zmax = 2.0 * kPi * (double)W * ctx->mask_fmax;
  int K = 1;
  for (double e = zmax; e > kPlaneTol; e *= 0.5 * zmax / K) {  // 2 (zmax / 2)^K / K!
    K++;
    if (K > kMaxPlanes) return GVM_OK;
  }
  g.planes = K;
  g.wz = 2.0 * kPi * (double)W;
  // terms of the J_k series until they fall below 1e-11 of the first
  g.terms = 2;
  for (double t = 0.25 * zmax * zmax; t > 1e-11; g.terms++)
    t *= 0.25 * zmax * zmax / ((double)g.terms * g.terms);
  if (g.terms > kMaxTerms) return GVM_OK;
  g.inv_w = W > 0.0f ? 1.0 / (double)W : 0.0;
  g.applies = *ok = true;
  return GVM_OK;
}

// Sorts every slice's visibilities by tile and lays out the work items and
// the workspace, for the planes of probe_grid_plan.  *ok = false (and GVM_OK) when there
// is not enough memory; the GEMM form then takes the call.
// (Scratch from the context's set-up workspace and a few allocations for what the plan
// keeps: one for every array, and as many hipFree's, took more of a small observation's
// first pass than the sort.)
gvm_status build_grid_plan(gvm_ctx* ctx, bool* ok) {
  *ok = false;
  GridPlan& g = ctx->gplan;
  if (g.built) {
    *ok = g.usable;
    return GVM_OK;
  }
  g.built = true;
  const int N = ctx->g.N, nsl = (int)ctx->slices.size(), K = g.planes;
  const unsigned int ntiles = (unsigned int)(N / 8 + 1) * (N / 4);
  hipStream_t st = ctx->stream;
  auto give_up = [&]() {
    release_grid_plan(g);
    g.built = true;
    return GVM_OK;
  };
  long vmax = 0, total = 0;
  for (const Slice& s : ctx->slices) {
    vmax = std::max(vmax, s.nvis);
    total += s.nvis;
  }

  // items of at most `chunk` rows: long enough to amortise a subgrid's
  // stores, short enough that a small observation fills the chip
  g.chunk = (int)std::min(512L, std::max(64L, (total / 4096 + 63) / 64 * 64));
  const int shift_x = N / 2 - (int)ctx->g.x0_phs, shift_y = N / 2 - (int)ctx->g.y0_phs;
  const bool shifted = shift_x != 0 || shift_y != 0;
  std::vector<float2> tw2(2 * (size_t)N);
  for (int k = 0; k < 2 * N; k++) {
    const double t = (double)k / (2 * N);
    tw2[k] = make_float2((float)std::cos(2.0 * kPi * t), (float)std::sin(2.0 * kPi * t));
  }
  const std::vector<double> corr = kernel_correction(N);
  // J_0, then 2 (+-) J_k (the planes hold c T_k for even k, -i c T_k for odd):
  // J_k(zeta) = zeta^k / (2^k k!) sum_m (-1)^m (zeta / 2)^2m k! / (m! (m + k)!)
  std::vector<double> wc((size_t)K * g.terms);
  double lead = 1.0;
  for (int k = 0; k < K; k++) {
    if (k > 0) lead *= 0.5 / k;
    const int odd = (k & 1) ? ((k + 1) >> 1) & 1 : (k >> 1) & 1;
    double c = k == 0 ? 1.0 : odd ? -2.0 * lead : 2.0 * lead;
    for (int m = 0; m < g.terms; m++) {
      wc[(size_t)k * g.terms + m] = c;
      c *= -0.25 / ((m + 1.0) * (m + 1.0 + k));
    }
  }
  // one allocation for the tables and the rows; the tables first, in one upload
  auto place = [](size_t& at, size_t bytes) {
    const size_t p = at;
    at += Scratch::round(bytes);
    return p;
  };
  size_t at = 0;
  const size_t p_tw2 = place(at, sizeof(float2) * tw2.size());
  const size_t p_corr = place(at, sizeof(double) * corr.size());
  const size_t p_wcoef = place(at, sizeof(double) * wc.size());
  std::vector<char> up(at);
  std::memcpy(up.data() + p_tw2, tw2.data(), sizeof(float2) * tw2.size());
  std::memcpy(up.data() + p_corr, corr.data(), sizeof(double) * corr.size());
  std::memcpy(up.data() + p_wcoef, wc.data(), sizeof(double) * wc.size());
  const size_t p_slot = place(at, sizeof(int) * (size_t)nsl * ntiles);
  const size_t p_rec = place(at, sizeof(float4) * (size_t)total);
  const size_t p_meta = place(at, sizeof(uint2) * (size_t)total);
  const size_t p_rot = place(at, shifted ? sizeof(float2) * (size_t)total : 0);
  if (!device_array(&g.tables, at)) return give_up();
  g.bytes = at;
  GVM_HIP_TRY(hipMemcpy(g.tables, up.data(), up.size(), hipMemcpyHostToDevice));
  g.tw2 = (float2*)(g.tables + p_tw2);
  g.corr = (double*)(g.tables + p_corr);
  g.wcoef = (double*)(g.tables + p_wcoef);
  g.tile_slot = (int*)(g.tables + p_slot);
  g.rec = (float4*)(g.tables + p_rec);
  g.meta = (uint2*)(g.tables + p_meta);
  g.rot = shifted ? (float2*)(g.tables + p_rot) : nullptr;

  std::vector<char*> parts;  // a group's items, then its merges
  std::vector<std::pair<long, long>> counts;
  struct PartsFree {
    std::vector<char*>& v;
    ~PartsFree() {
      for (char* p : v) (void)hipFree(p);
    }
  } parts_free{parts};
  g.slice_slot.assign(nsl + 1, 0);
  g.slice_merge.assign(nsl + 1, 0);
  long row0 = 0, nitems = 0, nmerges = 0;
  for (int s0 = 0; s0 < nsl;) {
    int s1 = s0;
    long n = 0;
    while (s1 < nsl && (s1 == s0 || n + ctx->slices[s1].nvis <= kGroupRows) &&
           (unsigned long)(s1 - s0 + 1) * ntiles < 0x7fffffffUL)
      n += ctx->slices[s1++].nvis;
    const int ns = s1 - s0;
    const long nkeys = (long)ns * ntiles;
    std::vector<unsigned int> off(ns);
    unsigned int first = 0;
    for (int s = 0; s < ns; s++) {
      off[s] = first;
      first += (unsigned int)ctx->slices[s0 + s].nvis;
    }
    int bits = 1;
    while (bits < 32 && (nkeys >> bits) != 0) bits++;
    size_t bytes = 0, scan_bytes = 0;
    {
      rocprim::double_buffer<unsigned int> none(nullptr, nullptr);
      GVM_HIP_TRY(rocprim::radix_sort_pairs(nullptr, bytes, none, none, (size_t)n, 0u,
                                            (unsigned)bits, st));
      unsigned int* u = nullptr;
      GVM_HIP_TRY(rocprim::exclusive_scan(nullptr, scan_bytes, u, u, 0u, (size_t)nkeys + 1,
                                          rocprim::plus<unsigned int>(), st));
    }
    const size_t tmp_bytes = std::max(bytes, scan_bytes);
    Scratch sc(ctx);
    const size_t rows_b = sizeof(unsigned int) * (size_t)n, keys_b = sizeof(unsigned int) * (nkeys + 1);
    for (size_t b : {rows_b, rows_b, rows_b, rows_b, keys_b, keys_b, keys_b, keys_b, keys_b,
                     sizeof(unsigned int) * ns, sizeof(unsigned int) * 2 * ns,
                     sizeof(uint2) * (ns + 1), tmp_bytes})
      sc.add(b);
    if (sc.reserve("adjoint plan")) return give_up();
    struct {
      unsigned int *k0, *k1, *v0, *v1, *start, *cnt, *islot, *several, *mslot, *off, *placed;
      uint2* pick;
      char* tmp;
    } gs;
    for (unsigned int** p : {&gs.k0, &gs.k1, &gs.v0, &gs.v1}) *p = sc.take<unsigned int>(n);
    for (unsigned int** p : {&gs.start, &gs.cnt, &gs.islot, &gs.several, &gs.mslot})
      *p = sc.take<unsigned int>(nkeys + 1);
    gs.off = sc.take<unsigned int>(ns);
    gs.placed = sc.take<unsigned int>(2 * ns);
    gs.pick = sc.take<uint2>(ns + 1);
    gs.tmp = sc.take<char>(tmp_bytes);
    GVM_HIP_TRY(hipMemcpyAsync(gs.off, off.data(), sizeof(unsigned int) * ns,
                               hipMemcpyHostToDevice, st));
    GVM_HIP_TRY(hipMemsetAsync(gs.placed, 0, sizeof(unsigned int) * 2 * ns, st));
    hipLaunchKernelGGL(plan_keys_kernel, dim3((unsigned)std::min<long>(1024, (vmax + 255) / 256), ns),
                       dim3(256), 0, st, ctx->slice_tab, s0, gs.off, N, gs.k0, gs.v0);
    GVM_CHECK_LAUNCH();
    rocprim::double_buffer<unsigned int> kb(gs.k0, gs.k1), vb(gs.v0, gs.v1);
    GVM_HIP_TRY(rocprim::radix_sort_pairs(gs.tmp, bytes, kb, vb, (size_t)n, 0u, (unsigned)bits, st));
    hipLaunchKernelGGL(plan_records_kernel, dim3(blocks_for(n)), dim3(256), 0, st, ctx->slice_tab,
                       s0, gs.off, N, n, kb.current(), vb.current(), shift_x, shift_y,
                       g.rec + row0, g.meta + row0, shifted ? g.rot + row0 : nullptr);
    GVM_CHECK_LAUNCH();
    hipLaunchKernelGGL(tile_starts_kernel, dim3(blocks_for(nkeys + 1)), dim3(256), 0, st,
                       kb.current(), n, nkeys, gs.start);
    GVM_CHECK_LAUNCH();
    hipLaunchKernelGGL(item_counts_kernel, dim3(blocks_for(nkeys + 1)), dim3(256), 0, st, gs.start,
                       nkeys, g.chunk, gs.cnt, gs.several);
    GVM_CHECK_LAUNCH();
    GVM_HIP_TRY(rocprim::exclusive_scan(gs.tmp, scan_bytes, gs.cnt, gs.islot, (unsigned int)nitems,
                                        (size_t)nkeys + 1, rocprim::plus<unsigned int>(), st));
    GVM_HIP_TRY(rocprim::exclusive_scan(gs.tmp, scan_bytes, gs.several, gs.mslot,
                                        (unsigned int)nmerges, (size_t)nkeys + 1,
                                        rocprim::plus<unsigned int>(), st));
    hipLaunchKernelGGL(pick_kernel, dim3(1), dim3(256), 0, st, gs.islot, gs.mslot, ntiles, ns,
                       gs.pick);
    GVM_CHECK_LAUNCH();
    std::vector<uint2> pick(ns + 1);
    GVM_HIP_TRY(hipMemcpyAsync(pick.data(), gs.pick, sizeof(uint2) * (ns + 1),
                               hipMemcpyDeviceToHost, st));
    GVM_HIP_TRY(hipStreamSynchronize(st));
    for (int s = 0; s <= ns; s++) {
      g.slice_slot[s0 + s] = (long)pick[s].x;
      g.slice_merge[s0 + s] = (long)pick[s].y;
    }
    const long ni = (long)pick[ns].x - nitems, nm = (long)pick[ns].y - nmerges;
    char* part = nullptr;
    if (!device_array(&part, sizeof(long4) * (size_t)ni + sizeof(int2) * (size_t)nm)) return give_up();
    parts.push_back(part);
    counts.push_back({ni, nm});
    long4* items = (long4*)part;
    int2* merges = (int2*)(items + ni);
    hipLaunchKernelGGL(items_kernel, dim3(blocks_for(nkeys)), dim3(256), 0, st, gs.start, gs.islot,
                       gs.mslot, nkeys, g.chunk, row0, ntiles, s0, (unsigned int)nitems,
                       (unsigned int)nmerges, gs.placed, gs.placed + ns, items, merges,
                       g.tile_slot + (long)s0 * ntiles);
    GVM_CHECK_LAUNCH();
    GVM_HIP_TRY(hipStreamSynchronize(st));  // the group's scratch is freed
    sc.idle();
    nitems += ni;
    nmerges += nm;
    if (nitems > 0x7fffffffL) return give_up();
    row0 += n;
    s0 = s1;
  }
  if (parts.size() == 1) {
    g.lists = parts[0];
    parts.clear();
  } else {
    if (!device_array(&g.lists, sizeof(long4) * (size_t)nitems + sizeof(int2) * (size_t)nmerges))
      return give_up();
    char* o = g.lists;
    char* om = g.lists + sizeof(long4) * (size_t)nitems;
    for (size_t k = 0; k < parts.size(); k++) {
      const size_t bi = sizeof(long4) * counts[k].first, bm = sizeof(int2) * counts[k].second;
      GVM_HIP_TRY(hipMemcpyAsync(o, parts[k], bi, hipMemcpyDeviceToDevice, st));
      GVM_HIP_TRY(hipMemcpyAsync(om, parts[k] + bi, bm, hipMemcpyDeviceToDevice, st));
      o += bi;
      om += bm;
    }
    GVM_HIP_TRY(hipStreamSynchronize(st));
  }
  g.bytes += sizeof(long4) * (size_t)nitems + sizeof(int2) * (size_t)nmerges;
  g.items = (long4*)g.lists;
  g.merges = (int2*)(g.items + nitems);

  // batches of slices that share the workspace
  const size_t per_item = sizeof(float) * kSub * (size_t)K;
  const size_t per_slice = sizeof(float2) * (size_t)K * N * row_pitch(N);
  size_t free_b = 0, total_b = 0;
  GVM_HIP_TRY(hipMemGetInfo(&free_b, &total_b));
  const size_t budget = std::min<size_t>(32UL << 30, free_b / 2);
  g.batch0.clear();
  size_t need_part = 0, need_slices = 0;
  for (int s = 0; s < nsl;) {
    g.batch0.push_back(s);
    size_t b = 0;
    int e = s;
    while (e < nsl) {
      const size_t add = per_item * (size_t)(g.slice_slot[e + 1] - g.slice_slot[e]) + per_slice;
      if (e > s && b + add > kBatchBytes) break;
      b += add;
      e++;
    }
    // subgrids; after them, with several slices, their N x N images
    need_part = std::max({need_part, per_item * (size_t)(g.slice_slot[e] - g.slice_slot[s]),
                          sizeof(float) * (size_t)N * N * (size_t)(e - s > 1 ? e - s : 0)});
    need_slices = std::max(need_slices, (size_t)(e - s));
    s = e;
  }
  g.batch0.push_back(nsl);
  g.part_bytes = (need_part + 255) / 256 * 256;
  const size_t bytes = g.part_bytes + per_slice * need_slices;
  if (bytes > budget) return give_up();
  if (!device_array((char**)&g.ws, bytes)) return give_up();
  g.bytes += bytes;
  g.usable = true;
  *ok = true;
  return GVM_OK;
}

namespace {

template <int NP>
void launch_spread(gvm_ctx* ctx, long slot0, int nitems, int k0, float* part) {
  const GridPlan& g = ctx->gplan;
  hipLaunchKernelGGL((spread_kernel<NP>), dim3(nitems), dim3(64), 0, ctx->stream,
                     g.items + slot0, slot0, g.rec, g.meta, g.rot, ctx->slice_tab, ctx->cmax,
                     g.inv_w, k0, g.planes, part);
}

template <int N>
void launch_cols(gvm_ctx* ctx, int s0, int ns, const float* part, float2* H) {
  // four columns per block (64 KB of LDS at 2N = 2048, two blocks per CU), two
  // where four would need 256 KB
  constexpr int BC = N <= 2048 ? 4 : 2;
  constexpr int T = N <= 128 ? 64 : N >= 2048 ? 1024 : N / 2;
  const GridPlan& g = ctx->gplan;
  const int nb = (N + BC) / BC;  // columns 0 .. N
  hipLaunchKernelGGL((grid_cols_kernel<N, BC, T>), dim3(nb, g.planes, ns), dim3(T), 0,
                     ctx->stream, (const float2*)part,
                     g.tile_slot + (long)s0 * (N / 8 + 1) * (N / 4), (int)g.slice_slot[s0],
                     g.planes, g.tw2, row_pitch(N), H);
}

template <int N, int B>
void launch_rows(gvm_ctx* ctx, const RowsArgs& a) {
  constexpr int T = N / 4 < 64 ? 64 : N / 4;
  hipLaunchKernelGGL((grid_rows_kernel<N, B, T>), dim3(N, a.nsl), dim3(T), 0, ctx->stream, a);
}

template <int N>
gvm_status run_batch(gvm_ctx* ctx, int s0, int s1, const float* I, float* result, int flag_opt,
                     int normalize, bool set) {
  const GridPlan& g = ctx->gplan;
  const int K = g.planes;
  const long slot0 = g.slice_slot[s0];
  const int nitems = (int)(g.slice_slot[s1] - slot0);
  float* part = (float*)g.ws;
  float2* H = (float2*)(g.ws + g.part_bytes);
  for (int k0 = 0; k0 < K; k0 += kPlaneGroup) {
    const int np = std::min(kPlaneGroup, K - k0);
    switch (np) {
      case 1: launch_spread<1>(ctx, slot0, nitems, k0, part); break;
      case 2: launch_spread<2>(ctx, slot0, nitems, k0, part); break;
      case 3: launch_spread<3>(ctx, slot0, nitems, k0, part); break;
      case 4: launch_spread<4>(ctx, slot0, nitems, k0, part); break;
      case 5: launch_spread<5>(ctx, slot0, nitems, k0, part); break;
      case 6: launch_spread<6>(ctx, slot0, nitems, k0, part); break;
      case 7: launch_spread<7>(ctx, slot0, nitems, k0, part); break;
      default: launch_spread<8>(ctx, slot0, nitems, k0, part); break;
    }
    GVM_CHECK_LAUNCH();
  }
  const int nmerges = (int)(g.slice_merge[s1] - g.slice_merge[s0]);
  if (nmerges > 0) {
    hipLaunchKernelGGL(merge_kernel, dim3(nmerges, K * kSub / 256), dim3(256), 0, ctx->stream,
                       g.merges + g.slice_merge[s0], (int)slot0, K, part);
    GVM_CHECK_LAUNCH();
  }
  launch_cols<N>(ctx, s0, s1 - s0, part, H);
  GVM_CHECK_LAUNCH();
  RowsArgs a{};
  a.H = H;
  a.pitch = row_pitch(N);
  a.nplanes = K;
  a.terms = g.terms;
  a.tw = ctx->twiddle;
  a.tw2 = g.tw2;
  a.corr = g.corr;
  a.wcoef = g.wcoef;
  a.tab = ctx->slice_tab;
  a.s0 = s0;
  a.nsl = s1 - s0;
  a.cmaxs = ctx->cmax;
  a.noise = ctx->noise;
  a.noise_cut = ctx->g.noise_cut;
  a.fg_scale = ctx->g.fg_scale;
  a.threshold = ctx->g.threshold;
  a.gcf = ctx->gcf;
  a.normalize = normalize;
  a.flag_opt = flag_opt;
  a.set = set ? ctx->g.image_count : 0;
  a.wz = g.wz;
  a.dx = ctx->g.deltax * kPi / 180.0;
  a.dy = ctx->g.deltay * kPi / 180.0;
  a.x0 = (int)ctx->g.x0_phs;
  a.y0 = (int)ctx->g.y0_phs;
  a.I = I;
  a.result = result;
  // the subgrids have been read when the rows run: their memory takes the
  // slices' d's
  a.each = a.nsl > 1 ? part : nullptr;
  // planes per transform: as few groups of at most four as K needs
  const int groups = (K + 3) / 4, B = (K + groups - 1) / groups;
  if (B <= 2)
    launch_rows<N, 2>(ctx, a);
  else if (B == 3)
    launch_rows<N, 3>(ctx, a);
  else
    launch_rows<N, 4>(ctx, a);
  GVM_CHECK_LAUNCH();
  if (a.each) {
    hipLaunchKernelGGL(chain_kernel, dim3(blocks_for((long)N * N)), dim3(256), 0, ctx->stream, a, N);
    GVM_CHECK_LAUNCH();
  }
  return GVM_OK;
}

}  // namespace

gvm_status adjoint_grid(gvm_ctx* ctx, const float* I, float* result, int flag_opt, int normalize,
                        bool set) {
  const GridPlan& g = ctx->gplan;
  for (size_t b = 0; b + 1 < g.batch0.size(); b++) {
    const int s0 = g.batch0[b], s1 = g.batch0[b + 1];
    gvm_status st = GVM_ERR_ARG;
    switch (ctx->g.N) {
      case 64: st = run_batch<64>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 128: st = run_batch<128>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 256: st = run_batch<256>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 512: st = run_batch<512>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 1024: st = run_batch<1024>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 2048: st = run_batch<2048>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
      case 4096: st = run_batch<4096>(ctx, s0, s1, I, result, flag_opt, normalize, set && b == 0); break;
    }
    if (st) return st;
  }
  return GVM_OK;
}

}  // namespace gvm
