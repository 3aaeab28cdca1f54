// Gridded-visibility mode on the device: convolutional gridding of the rows
// of one slice (do_gridding, src/functions.cu:1339-1653), the weighting
// schemes (src/naturalweightingscheme.cu, src/uniformweightingscheme.cu,
// src/briggsweightingscheme.cu, src/radialweightingscheme.cu) and the
// gridding correction image (apply_GCF, src/functions.cu:2468-2476).
//
// Both the gridder and the weighting schemes accumulate per-cell sums in
// float.  The reference adds rows to a cell one at a time in row order (with
// one OpenMP thread), so a parallel float sum would not reproduce its
// rounding.  Here rows are sorted by where they fall (a stable radix sort keeps
// their order) and each cell's owner adds its rows in sequence.  The result is
// the reference's single-thread sum, bit for bit, and does not depend on
// scheduling.
//
// Gridder: rows are sorted by 8 x 8 tile of cells, once for every tile that
// their taps reach (at most four tiles for kernels up to 9 x 9), and a block
// owns a tile.  Sorting every (row, tap) pair instead, 173 M
// pairs for 1.76 M rows and 7 x 7 taps, took 12 ms and 5 GB of scratch memory
// allocated and freed on each call, 107 - 137 ms in all; it is kept for single taps and
// for few rows on a large grid, where it is the faster one (use_entries).
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "gvm_internal.h"

namespace gvm {
namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr double kRad = kPi / 180.0;
constexpr int kThreads = 256;
constexpr int kSumBlocks = 1024;

int blocks_for(long n) {
  return (int)std::max(1L, std::min<long>((n + kThreads - 1) / kThreads, 65536));
}

// Number of bits a radix sort needs for keys in [0, sentinel].
int key_bits(uint32_t sentinel) {
  int b = 1;
  while (b < 32 && (sentinel >> b) != 0) b++;
  return b;
}

// Stable sort of up to `cap` (key, id) pairs.
struct PairSort {
  uint32_t *k[2] = {}, *v[2] = {};
  char* tmp = nullptr;
  size_t cap = 0, tmp_bytes = 0;
  rocprim::double_buffer<uint32_t> kb, vb;

  // room for a sort of n pairs (call it for every n that will be sorted)
  gvm_status size(size_t n, int bits, const char* what) {
    rocprim::double_buffer<uint32_t> a((uint32_t*)nullptr, (uint32_t*)nullptr), b = a;
    size_t bytes = 0;
    if (rocprim::radix_sort_pairs(nullptr, bytes, a, b, n, 0u, (unsigned)bits) != hipSuccess) {
      set_error(std::string(what) + ": radix sort sizing failed");
      return GVM_ERR_HIP;
    }
    cap = std::max(cap, n);
    tmp_bytes = std::max(tmp_bytes, bytes);
    return GVM_OK;
  }
  void add(Scratch& sc) const {
    for (int i = 0; i < 4; i++) sc.add(sizeof(uint32_t) * cap);
    sc.add(tmp_bytes);
  }
  void take(Scratch& sc) {
    for (int i = 0; i < 2; i++) {
      k[i] = sc.take<uint32_t>(cap);
      v[i] = sc.take<uint32_t>(cap);
    }
    tmp = sc.take<char>(tmp_bytes);
  }
  // sorts k[0] / v[0]; keys() / ids() are the sorted arrays
  gvm_status sort(size_t n, int bits, const char* what) {
    kb = rocprim::double_buffer<uint32_t>(k[0], k[1]);
    vb = rocprim::double_buffer<uint32_t>(v[0], v[1]);
    size_t bytes = tmp_bytes;
    if (rocprim::radix_sort_pairs(tmp, bytes, kb, vb, n, 0u, (unsigned)bits) != hipSuccess) {
      set_error(std::string(what) + ": radix sort failed");
      return GVM_ERR_HIP;
    }
    return GVM_OK;
  }
  const uint32_t* keys() { return kb.current(); }
  const uint32_t* ids() { return vb.current(); }
};

// ---- convolutional gridding -----------------------------------------------

constexpr int kGTile = 8;           // edge of a tile of cells
constexpr int kLdsTaps = 1024;      // taps staged in LDS; larger kernels read memory

struct GridGeom {
  double deltau, deltav;  // 1 / (M dx), 1 / (N dy), radians (dx < 0: deltau < 0)
  double cj, ck;          // floor(N / 2), floor(M / 2)
  double lambda;          // float wavelength of the slice, promoted
  int M, N;
  int kn;                 // kernel columns
  int supx, supy;         // supports
  int wx, wy;             // columns and rows of taps a row of data reaches
  int tx, ty;             // tiles they can span
  int ntx, nty;           // tiles of the grid
};

// A record of every row and its Hermitian twin (row z >= nvis is the twin of
// z - nvis): w, w Vo.x, w Vo.y and the first cell reached (16 bits each); and one
// (tile, row) entry per tile that the row's taps can span, in row order: the
// tile's index, or ntx nty for none.
// (do_gridding, src/functions.cu:1424-1480)
__global__ __launch_bounds__(kThreads) void grid_keys_kernel(const double* __restrict__ uvw,
                                                             const float* __restrict__ weight,
                                                             const float2* __restrict__ vo,
                                                             long nvis, GridGeom g,
                                                             float4* __restrict__ rec,
                                                             uint32_t* __restrict__ keys,
                                                             uint32_t* __restrict__ ids) {
#pragma clang fp contract(off)
  const int T = g.tx * g.ty;
  for (long vi = blockIdx.x * (long)blockDim.x + threadIdx.x; vi < nvis;
       vi += (long)gridDim.x * blockDim.x) {
    for (int twin = 0; twin < 2; twin++) {
      double u = uvw[3 * vi], v = uvw[3 * vi + 1];
      if (twin) {
        u = -u;
        v = -v;
      }
      u = u / g.lambda;  // metres_to_lambda (src/MSFITSIO.cu:41-45)
      v = v / g.lambda;
      const double jf = u / g.deltau + g.cj + 0.5;
      const double kf = v / g.deltav + g.ck + 0.5;
      const long z = vi + (twin ? nvis : 0);
      int j = 0, k = 0;
      const bool ok = fabs(jf) < 1073741824.0 && fabs(kf) < 1073741824.0;
      if (ok) {
        j = (int)jf - g.supx;  // C truncation, as int(j_fp); the first cell reached
        k = (int)kf - g.supy;
      }
      // (a row that reaches a tile starts within 255 cells of the grid)
      const float w = weight[vi];
      const float2 d = vo[vi];
      const int jc = min(max(j, -32768), 32767), kc = min(max(k, -32768), 32767);
      rec[z] = make_float4(w, w * d.x, w * (twin ? -d.y : d.y),
                           __int_as_float((jc & 0xffff) | kc << 16));
      const int ca = j >> 3, cb = (j + g.wx - 1) >> 3, ra = k >> 3, rb = (k + g.wy - 1) >> 3;
      for (int t = 0; t < T; t++) {
        const int c = ca + t % g.tx, r = ra + t / g.tx;
        const bool in = ok && c <= cb && r <= rb && c >= 0 && r >= 0 && c < g.ntx && r < g.nty;
        keys[z * T + t] = (uint32_t)(in ? r * g.ntx + c : g.ntx * g.nty);
        ids[z * T + t] = (uint32_t)z;
      }
    }
  }
}

// start[k] = the first sorted entry with key >= k, k in [0, nkeys]
__global__ __launch_bounds__(kThreads) void tile_first_kernel(const uint32_t* __restrict__ keys,
                                                              long n, int nkeys,
                                                              uint32_t* __restrict__ start) {
  for (int k = blockIdx.x * kThreads + threadIdx.x; k <= nkeys; k += gridDim.x * kThreads) {
    long lo = 0, hi = n;
    while (lo < hi) {
      const long m = (lo + hi) >> 1;
      if (keys[m] < (uint32_t)k)
        lo = m + 1;
      else
        hi = m;
    }
    start[k] = (uint32_t)lo;
  }
}

// One block per tile, one wave per quadrant (4 x 4 cells), 16 lanes for each of
// the four float sums of do_gridding: a lane adds one sum of one cell over the
// rows in order; then the normalisation (src/functions.cu:1424-1559).  256 rows
// at a time are staged in LDS; each wave keeps, in order, those that reach its
// quadrant (half of a tile's for 7 x 7 taps) and every lane goes through them.
// 1.6 ms for 1.76 M rows and 7 x 7 taps on 1024^2, set by the fullest tiles' chains
// (29,000 rows).  Before: one wave per tile, a lane per cell with its four sums,
// 3.9 ms; a branch per row instead of the selection, 2.8 ms; each wave gathering
// the rows' values itself, 2.2 ms.
typedef short short2_t __attribute__((ext_vector_type(2)));
typedef short short8_t __attribute__((ext_vector_type(8)));

// A cell's value and weight from its sums (src/functions.cu:1527-1559)
__device__ __forceinline__ void cell_value(float ws, float aux, float re, float im, float2* vo,
                                           float* w) {
#pragma clang fp contract(off)
  *w = 0.f;
  *vo = make_float2(0.f, 0.f);
  if (aux != 0.0f && ws != 0.0f) {
    *w = ws * ws / aux;
    *vo = make_float2(re / ws, im / ws);
  }
}

template <bool LDS_TAPS>
__global__ __launch_bounds__(kThreads) void grid_tiles_kernel(
    const uint32_t* __restrict__ ids, const uint32_t* __restrict__ start, GridGeom g,
    const float* __restrict__ taps, const float4* __restrict__ rec, float2* __restrict__ cell_vo,
    float* __restrict__ cell_w) {
#pragma clang fp contract(off)
  __shared__ float lt[2][LDS_TAPS ? kLdsTaps : 1];  // k and k^2
  __shared__ float4 stage[kThreads];                // the block's next rows
  __shared__ __align__(16) float val[4][4][68];     // w, w, w Vo.x, w Vo.y of each row
  __shared__ __align__(16) short2_t rel[4][68];     // the first cell it reaches
  if constexpr (LDS_TAPS) {
    for (int t = threadIdx.x; t < g.wx * g.wy; t += kThreads) {
      const float k = taps[g.kn * (t / g.wx) + t % g.wx];
      lt[0][t] = k;
      lt[1][t] = k * k;
    }
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sum = lane >> 4;
  const int tile = blockIdx.x;
  // the quadrant's first cell, and this lane's
  const int c0 = tile % g.ntx * kGTile + (wave & 1) * 4, r0 = tile / g.ntx * kGTile + (wave >> 1) * 4;
  const short2_t cell = {(short)(lane & 3), (short)((lane >> 2) & 3)};
  const short2_t size = {(short)g.wx, (short)g.wy}, origin = {(short)c0, (short)r0};
  const float* tap = lt[sum == 1 ? 1 : 0];
  const long s = start[tile], e = start[tile + 1];
  float acc = 0.f;
  // a record is a gather behind its id: ids are loaded two rounds ahead,
  // records one, so that a round waits for neither
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
  uint32_t z = 0;
  auto fetch = [&](long p) {
    if (p < e) r = rec[z];
    z = p + kThreads < e ? ids[p + kThreads] : 0;
  };
  if (s + threadIdx.x < e) z = ids[s + threadIdx.x];
  fetch(s + threadIdx.x);
  for (long c = s; c < e; c += kThreads) {
    __syncthreads();  // the round before has been read (and the taps are there)
    stage[threadIdx.x] = r;
    __syncthreads();
    fetch(c + kThreads + threadIdx.x);
    const int rows = (int)min((long)kThreads, e - c);
    for (int o = 0; o < rows; o += 64) {
      const float4 q0 = stage[o + lane];
      const short2_t first = __builtin_bit_cast(short2_t, q0.w) - origin;
      const bool in = o + lane < rows && first.x < 4 && first.y < 4 && first.x + g.wx > 0 &&
                      first.y + g.wy > 0;
      const unsigned long long m = __ballot(in);
      const int cnt = __popcll(m), at = __popcll(m & ((1ull << lane) - 1));
      __builtin_amdgcn_wave_barrier();
      if (in) {
        val[wave][0][at] = val[wave][1][at] = q0.x;
        val[wave][2][at] = q0.y;
        val[wave][3][at] = q0.z;
        rel[wave][at] = first;
      }
      // rounds of four rows: the last is filled with rows that reach nothing
      if (lane < 4) rel[wave][cnt + lane] = short2_t{16384, 16384};
      __builtin_amdgcn_wave_barrier();
      for (int j = 0; j < cnt; j += 4) {
        const short8_t r4 = *(const short8_t*)&rel[wave][j];
        const float4 q4 = *(const float4*)&val[wave][sum][j];
        const float q[4] = {q4.x, q4.y, q4.z, q4.w};
        // every load first, then the sums in row order by selection: a branch per
        // row waited for two dependent LDS reads each time (2.8 ms)
        bool hit[4];
        float k[4];
  #pragma unroll
        for (int u = 0; u < 4; u++) {
          const short2_t d = cell - short2_t{r4[2 * u], r4[2 * u + 1]};
          const short2_t past = d - size;
          // 0 <= d < size in both: d not negative, d - size negative
          const unsigned int out = __builtin_bit_cast(unsigned int, d) |
                                   ~__builtin_bit_cast(unsigned int, past);
          hit[u] = (out & 0x80008000u) == 0u;
          const unsigned int pitch = LDS_TAPS ? (unsigned int)g.wx : (unsigned int)g.kn;
          unsigned int at = __umul24((unsigned int)(unsigned short)d.y, pitch) +
                            (unsigned int)(unsigned short)d.x;
          at = hit[u] ? at : 0u;
          if constexpr (LDS_TAPS) {
            k[u] = tap[at];
          } else {
            k[u] = taps[at];
            if (sum == 1) k[u] = k[u] * k[u];
          }
        }
  #pragma unroll
        for (int u = 0; u < 4; u++) {
          const float t = acc + q[u] * k[u];
          acc = hit[u] ? t : acc;
        }
      }
    }
  }
  // lane l < 16 takes its cell's four sums
  const float ws = acc, aux = __shfl(acc, (lane & 15) + 16, 64), re = __shfl(acc, (lane & 15) + 32, 64),
              im = __shfl(acc, (lane & 15) + 48, 64);
  if (lane >= 16) return;
  const int cx = c0 + cell.x, cy = r0 + cell.y;
  cell_value(ws, aux, re, im, cell_vo + (long)g.N * cy + cx, cell_w + (long)g.N * cy + cx);
}

// The same sums from (row, tap) entries sorted by cell, for single taps and for few rows
// on a large grid: nothing here goes over the grid's cells or a tile's rows.  Entry
// e is tap e % taps of row e / taps (rows and twins as above); a stable sort keeps a
// cell's entries in row order.
__global__ __launch_bounds__(kThreads) void entry_keys_kernel(const double* __restrict__ uvw,
                                                              long nvis, GridGeom g,
                                                              uint32_t* __restrict__ keys,
                                                              uint32_t* __restrict__ ids) {
#pragma clang fp contract(off)
  const uint32_t taps = (uint32_t)(g.wx * g.wy), n = (uint32_t)(2 * nvis) * taps;
  for (uint32_t e = blockIdx.x * kThreads + threadIdx.x; e < n; e += gridDim.x * kThreads) {
    const uint32_t z = e / taps, t = e - z * taps;
    const bool twin = z >= nvis;
    const long vi = twin ? z - nvis : z;
    double u = uvw[3 * vi], v = uvw[3 * vi + 1];
    if (twin) {
      u = -u;
      v = -v;
    }
    u = u / g.lambda;
    v = v / g.lambda;
    const double jf = u / g.deltau + g.cj + 0.5;
    const double kf = v / g.deltav + g.ck + 0.5;
    uint32_t key = (uint32_t)((long)g.M * g.N);
    if (fabs(jf) < 1073741824.0 && fabs(kf) < 1073741824.0) {
      const int j = (int)jf - g.supx + (int)(t % (uint32_t)g.wx);
      const int k = (int)kf - g.supy + (int)(t / (uint32_t)g.wx);
      if (k >= 0 && k < g.M && j >= 0 && j < g.N) key = (uint32_t)((long)g.N * k + j);
    }
    keys[e] = key;
    ids[e] = e;
  }
}

// The cell that starts at sorted entry p: its value and weight at index p, weight 0 where
// none starts.  64 entries' products at a time are formed by a wave's lanes and left in
// LDS; lanes 0 to 3 add one sum each, four entries a read: 16 ns an entry (one lane
// adding all four sums: 26).  A thread adds a short run itself.
__global__ __launch_bounds__(kThreads) void entry_cells_kernel(
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ ids, long n, long nvis,
    GridGeom g, const float* __restrict__ taps, const float* __restrict__ weight,
    const float2* __restrict__ vo, float2* __restrict__ cell_vo, float* __restrict__ cell_w) {
#pragma clang fp contract(off)
  constexpr int kShort = 16;
  __shared__ __align__(16) float prod[kThreads / 64][4][64 + 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t off = (uint32_t)((long)g.M * g.N), nt = (uint32_t)(g.wx * g.wy);
  auto products = [&](uint32_t id, float* q) {
    const uint32_t z = id / nt, t = id - z * nt;
    const long vi = z >= nvis ? z - nvis : z;
    const float w = weight[vi];
    float2 v = vo[vi];
    if (z >= nvis) v.y = -v.y;
    const float k = taps[g.kn * (t / (uint32_t)g.wx) + t % (uint32_t)g.wx];
    q[0] = w * k;
    q[1] = w * (k * k);
    q[2] = w * v.x * k;
    q[3] = w * v.y * k;
  };
  for (long i0 = (long)blockIdx.x * kThreads + threadIdx.x - lane; i0 < n;
       i0 += (long)gridDim.x * kThreads) {
    const long i = i0 + lane;
    const uint32_t key = i < n ? keys[i] : off;
    const bool head = key != off && (i == 0 || keys[i - 1] != key);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    bool more = head;
    if (head) {
      uint32_t id[kShort];
      int cnt = 1;
#pragma unroll
      for (int u = 0; u < kShort; u++) {
        const long p = min(i + u, n - 1);
        id[u] = ids[p];
        cnt = u == cnt && i + u < n && keys[p] == key ? u + 1 : cnt;
      }
      more = cnt == kShort;
#pragma unroll
      for (int u = 0; u < kShort; u += 4) {
        if (u >= cnt) break;
        float q[4][4];
#pragma unroll
        for (int h = 0; h < 4; h++) products(id[u + h], q[h]);  // (past the run's end: not added)
#pragma unroll
        for (int h = 0; h < 4; h++)
#pragma unroll
          for (int c = 0; c < 4; c++) s[c] = u + h < cnt ? s[c] + q[h][c] : s[c];
      }
    }
    for (unsigned long long m = __ballot(more); m; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      const uint32_t lk = (uint32_t)__builtin_amdgcn_readlane((int)key, l);
      // sum c continues in lane c
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float from = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[c]), l));
        t = lane == c ? from : t;
      }
      // products are a gather behind their ids: a round's are formed while the round
      // before is added, its ids read a round before that
      long p = i0 + l + kShort + lane;
      auto entry = [&](long p, uint32_t* id) {
        *id = ids[min(p, n - 1)];
        return __popcll(__ballot(p < n && keys[min(p, n - 1)] == lk));  // a run is contiguous
      };
      uint32_t id, id1;
      float q[4];
      int cnt = entry(p, &id), cnt1 = entry(p + 64, &id1);
      products(id, q);  // (of other runs' entries, too: not added)
      while (cnt > 0) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < 4; c++) prod[wave][c][lane] = q[c];
        __builtin_amdgcn_wave_barrier();
        p += 64;
        uint32_t id2;
        const int cnt2 = entry(p + 64, &id2);
        if (cnt1 > 0) products(id1, q);
        const float* mine = prod[wave][lane & 3];
        if (cnt == 64) {
#pragma unroll
          for (int j = 0; j < 64; j += 4) {
            const float4 v = *(const float4*)(mine + j);
            t = t + v.x;
            t = t + v.y;
            t = t + v.z;
            t = t + v.w;
          }
        } else {
          for (int j = 0; j < cnt; j++) t = t + mine[j];
        }
        if (cnt < 64) break;
        cnt = cnt1;
        cnt1 = cnt2;
        id1 = id2;
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), c));
        if (lane == l) s[c] = sum;
      }
    }
    if (i >= n) continue;
    cell_w[i] = 0.f;
    if (head) cell_value(s[0], s[1], s[2], s[3], cell_vo + i, cell_w + i);
  }
}

struct IsKept {
  __device__ __host__ int operator()(float w) const { return w > 0.0f ? 1 : 0; }
};

// Kept cells (weight > 0) to rows at the cell centre, in row-major cell order
// (src/functions.cu:1527-1539, 1587-1607): uvw in metres, w = 0.
// keys: the cells' indices (sorted entries), or none (every cell in turn).
__global__ __launch_bounds__(kThreads) void grid_emit_kernel(
    const int* __restrict__ pos, GridGeom g, const uint32_t* __restrict__ keys, long n,
    const float2* __restrict__ cell_vo, const float* __restrict__ cell_w, long capacity,
    double* __restrict__ uvw_out, float2* __restrict__ vo_out, float* __restrict__ w_out) {
#pragma clang fp contract(off)
  for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < n;
       r += (long)gridDim.x * blockDim.x) {
    const float w = cell_w[r];
    if (!(w > 0.0f)) continue;
    const long o = pos[r];
    if (o >= capacity) continue;
    const long cell = keys ? (long)keys[r] : r;
    const int gj = (int)(cell % g.N), gk = (int)(cell / g.N);
    const double ul = ((double)gj - g.cj) * g.deltau;
    const double vl = ((double)gk - g.ck) * g.deltav;
    uvw_out[3 * o] = ul * g.lambda;
    uvw_out[3 * o + 1] = vl * g.lambda;
    uvw_out[3 * o + 2] = 0.0;
    vo_out[o] = cell_vo[r];
    w_out[o] = w;
  }
}

// Single taps are summed by entry: as many entries as rows, no chain but a cell's own (us,
// entries / tiles: 300,000 rows on 64 x 64 243 / 589, all in one cell 4,850 / 11,800; the
// 1.76 M rows of the 1024 x 1024 workload 2,760 / 2,970 with the copy of their cells to the
// host; but 1.7 M rows spread evenly over 1024 x 1024 371 / 298).  Else by the estimated time in
// microseconds.  Entries: their sort and sums.  Tiles: passes over the cells, the sort, and
// the chain of the rows that reach a tile (0.06 for each of an even share: the fullest
// tiles, whose 40 ns a row decide, have more).  1.7 M rows on 64 x 64 with 3 x 3 taps take
// 1,840 / 4,410, 100 rows on 4096 x 4096 with 7 x 7 taps 104 / 268; but 10,000 rows on 64 x
// 64 with 7 x 7 taps 276 / 189, 1.7 M on 512 x 512 with 3 x 3 taps 2,050 / 661.  At most 2^26
// entries (2.4 GB of scratch).
bool use_entries(const GridGeom& g, long nvis) {
  const double rows = 2.0 * nvis, cells = (double)g.M * g.N, taps = (double)g.wx * g.wy;
  const double reached = (1.0 + (g.wx - 1) / 8.0) * (1.0 + (g.wy - 1) / 8.0);
  const double share = rows * reached / ((double)g.ntx * g.nty);
  const double entry_us = 25.0 + 8.5e-5 * rows * taps;
  const double tile_us = 1.1e-5 * cells + 6e-5 * rows * g.tx * g.ty + 0.06 * share;
  return rows * taps <= 67108864.0 && (taps == 1.0 || entry_us < tile_us);
}

// ---- weighting schemes -----------------------------------------------------

struct WeightGeom {
  double absdu, absdv;  // |deltau|, |deltav|
  double cx, cy;        // int(floor(N / 2)), int(floor(M / 2))
  double lambda;
  int M, N;
  uint32_t off;
};

struct TaperCoef {
  float amplitude, a, b, c;
  double u0, v0;
  int on;
};

// Cell of one row for the weighting schemes: wavelengths, rows with u < 0
// mirrored, cells of |deltau| x |deltav| (src/uniformweightingscheme.cu:35-51).
__device__ inline uint32_t weight_cell(double u, double v, const WeightGeom& g) {
#pragma clang fp contract(off)
  const double xf = u / g.absdu + g.cx + 0.5;
  const double yf = v / g.absdv + g.cy + 0.5;
  if (!(fabs(xf) < 1073741824.0 && fabs(yf) < 1073741824.0)) return g.off;
  const int x = (int)xf, y = (int)yf;
  if (x >= 0 && y >= 0 && x < g.N && y < g.M) return (uint32_t)((long)g.N * y + x);
  return g.off;
}

__device__ inline void mirrored_lambda(const double* uvw, long z, double lambda, double* u,
                                       double* v) {
#pragma clang fp contract(off)
  *u = uvw[3 * z] / lambda;
  *v = uvw[3 * z + 1] / lambda;
  if (*u < 0.0) {
    *u = -*u;
    *v = -*v;
  }
}

__global__ __launch_bounds__(kThreads) void weight_keys_kernel(const double* __restrict__ uvw,
                                                               long nvis, WeightGeom g,
                                                               uint32_t* __restrict__ keys,
                                                               uint32_t* __restrict__ ids) {
  for (long z = blockIdx.x * (long)blockDim.x + threadIdx.x; z < nvis;
       z += (long)gridDim.x * blockDim.x) {
    double u, v;
    mirrored_lambda(uvw, z, g.lambda, &u, &v);
    keys[z] = weight_cell(u, v, g);
    ids[z] = (uint32_t)z;
  }
}

// sorted[p] = weight[ids[p]]
__global__ __launch_bounds__(kThreads) void weight_gather_kernel(const uint32_t* __restrict__ ids,
                                                                 const float* __restrict__ weight,
                                                                 long n,
                                                                 float* __restrict__ sorted) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    sorted[i] = weight[ids[i]];
}

// Per cell: grid[cell] = (cumulative ? grid[cell] : 0) + the cell's weights
// added in row order.  The weights are gathered into sorted order first; a
// thread adds a short run of rows itself, a long one is added by its wave, 64
// rows a load: one dependent gather per added row took 463 us for 1.76 M rows,
// one thread's batches of eight 218 us, set by the fullest cell.
__global__ __launch_bounds__(kThreads) void weight_cells_kernel(
    const uint32_t* __restrict__ keys, const float* __restrict__ sorted, long n, uint32_t off,
    int cumulative, float* __restrict__ grid) {
#pragma clang fp contract(off)
  constexpr int kShort = 16;
  const int lane = threadIdx.x & 63;
  const long step = (long)gridDim.x * blockDim.x;
  for (long i0 = blockIdx.x * (long)blockDim.x + threadIdx.x - lane; i0 < n; i0 += step) {
    const long i = i0 + lane;
    const uint32_t key = i < n ? keys[i] : off;
    const bool head = key != off && (i == 0 || keys[i - 1] != key);
    float s = 0.0f;
    bool more = false;
    if (head) {
      s = cumulative ? grid[key] : 0.0f;
      uint32_t k[kShort];
      float w[kShort];
#pragma unroll
      for (int u = 0; u < kShort; u++) {
        const long q = min(i + u, n - 1);
        k[u] = i + u < n ? keys[q] : off;
        w[u] = sorted[q];
      }
      more = true;
#pragma unroll
      for (int u = 0; u < kShort; u++) {
        more = more && k[u] == key;
        if (more) s = s + w[u];
      }
      if (!more) grid[key] = s;
    }
    for (unsigned long long m = __ballot(more); m; m &= m - 1) {
      const int l = __builtin_ctzll(m);
      const uint32_t lk = (uint32_t)__builtin_amdgcn_readlane((int)key, l);
      float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), l));
      long p = i0 + l + kShort;
      auto at = [&](long q, float* w) {
        const bool ok = q < n && keys[min(q, n - 1)] == lk;
        *w = sorted[min(q, n - 1)];
        return __popcll(__ballot(ok));  // a run is contiguous
      };
      float w, wn;
      int cnt = at(p + lane, &w);
      while (cnt > 0) {
        const int next = at(p + 64 + lane, &wn);
        for (int j = 0; j < cnt; j++)
          t = t + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j));
        p += 64;
        cnt = cnt < 64 ? 0 : next;
        w = wn;
      }
      if (lane == 0) grid[lk] = t;
    }
  }
}

// Block partial sums (FP64) of sum_k w_k, or of G^2 over the columns
// n >= N/2 of every row (src/briggsweightingscheme.cu:47-53, 96-101).
__global__ __launch_bounds__(kThreads) void weight_sum_kernel(const float* __restrict__ x,
                                                              long n, double* __restrict__ part) {
  __shared__ double red[kThreads];
  double s = 0.0;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    s += (double)x[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = kThreads / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kThreads) void grid_sq_sum_kernel(const float* __restrict__ grid,
                                                               int M, int N,
                                                               double* __restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double red[kThreads];
  const int half = N - N / 2;
  const long n = (long)M * half;
  double s = 0.0;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x) {
    const float gv = grid[(i / half) * N + N / 2 + (i % half)];
    s += (double)(gv * gv);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = kThreads / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// UVTaper::getValue (include/classes/uvtaper.cuh:101-114) with a, b, c
// computed on the host in float.
__device__ inline float taper_value(double u, double v, const TaperCoef& t) {
#pragma clang fp contract(off)
  const double x = u - t.u0, y = v - t.v0;
  const double e = -(double)t.a * x * x - (double)t.b * x * y - (double)t.c * y * y;
  return (float)((double)t.amplitude * exp(e));
}

// The per-row weight update of each scheme (second loops of
// src/uniformweightingscheme.cu:66-90, src/briggsweightingscheme.cu:151-175;
// src/naturalweightingscheme.cu:23-44; src/radialweightingscheme.cu:20-39).
__global__ __launch_bounds__(kThreads) void weight_apply_kernel(
    int scheme, const double* __restrict__ uvw, long nvis, WeightGeom g,
    const float* __restrict__ grid, float f2, TaperCoef taper, float* __restrict__ weight) {
#pragma clang fp contract(off)
  for (long z = blockIdx.x * (long)blockDim.x + threadIdx.x; z < nvis;
       z += (long)gridDim.x * blockDim.x) {
    float w = weight[z];
    double u, v;
    if (scheme == GVM_WEIGHTING_RADIAL) {
      u = uvw[3 * z] / g.lambda;
      v = uvw[3 * z + 1] / g.lambda;
      const float fu = (float)u, fv = (float)v;
      w = w * sqrtf(fu * fu + fv * fv);  // distance(u, v, 0, 0), src/MSFITSIO.cu:47-51
    } else {
      mirrored_lambda(uvw, z, g.lambda, &u, &v);
      if (scheme == GVM_WEIGHTING_UNIFORM || scheme == GVM_WEIGHTING_BRIGGS) {
        const uint32_t cell = weight_cell(u, v, g);
        if (cell == g.off)
          w = 0.0f;
        else if (scheme == GVM_WEIGHTING_UNIFORM)
          w = w / grid[cell];
        else
          w = (float)((double)w / (1.0 + (double)(grid[cell] * f2)));
      }
    }
    if (taper.on) w = w * taper_value(u, v, taper);
    weight[z] = w;
  }
}

gvm_status launch_ok(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return GVM_ERR_HIP;
  }
  return GVM_OK;
}

}  // namespace
}  // namespace gvm

using namespace gvm;

extern "C" gvm_status gvm_grid_visibilities_dev(gvm_ctx* ctx, const gvm_ckernel* kernel,
                                                float freq, long nvis, const double* uvw_m_dev,
                                                const float* vo_dev, const float* weight_dev,
                                                double* uvw_out_dev, float* vo_out_dev,
                                                float* weight_out_dev, long capacity,
                                                long* nout) {
  static const char* what = "gvm_grid_visibilities_dev";
  GVM_REQUIRE(ctx && kernel && kernel->taps && uvw_m_dev && vo_dev && weight_dev && uvw_out_dev &&
                  vo_out_dev && weight_out_dev && nout,
              "gvm_grid_visibilities_dev: null argument");
  GVM_REQUIRE(freq > 0.f, "gvm_grid_visibilities_dev: frequency must be positive");
  GVM_REQUIRE(kernel->m >= 1 && kernel->n >= 1 && kernel->m <= 255 && kernel->n <= 255 &&
                  kernel->support_x >= 0 && kernel->support_y >= 0 &&
                  kernel->support_x <= 127 && kernel->support_y <= 127,
              "gvm_grid_visibilities_dev: kernel size out of range");
  GVM_REQUIRE(capacity >= 0, "gvm_grid_visibilities_dev: negative capacity");
  const gvm_geometry& geo = ctx->g;
  GridGeom g;
  g.M = geo.M;
  g.N = geo.N;
  const double dxr = geo.deltax * kRad, dyr = geo.deltay * kRad;
  g.deltau = 1.0 / (geo.M * dxr);
  g.deltav = 1.0 / (geo.N * dyr);
  g.cj = std::floor(geo.N / 2.0);
  g.ck = std::floor(geo.M / 2.0);
  g.lambda = (double)(2.99792458E8f / freq);
  g.kn = kernel->n;
  g.supx = kernel->support_x;
  g.supy = kernel->support_y;
  const int nx = 2 * g.supx + 1, ny = 2 * g.supy + 1;
  g.wx = std::min(nx, kernel->n);
  g.wy = std::min(ny, kernel->m);
  g.tx = (g.wx + kGTile - 2) / kGTile + 1;
  g.ty = (g.wy + kGTile - 2) / kGTile + 1;
  g.ntx = geo.N / kGTile;
  g.nty = geo.M / kGTile;
  *nout = 0;
  GVM_REQUIRE(nvis >= 0 && nvis <= (((1L << 31) - 1) / (2L * nx * ny)),
              "gvm_grid_visibilities_dev: rows x taps exceed 2^31 entries");
  if (nvis == 0) return GVM_OK;
  const long cells = (long)geo.M * geo.N, entries = 2 * nvis * g.wx * g.wy;
  const bool by_entry = use_entries(g, nvis);
  const long n = by_entry ? entries : 2 * nvis * g.tx * g.ty;
  const long slots = by_entry ? entries : cells;  // where a cell's sums may be
  const int ntiles = g.ntx * g.nty, bits = key_bits((uint32_t)(by_entry ? cells : ntiles));
  GVM_HIP_TRY(hipSetDevice(ctx->device));

  gvm_status st;
  Scratch sc(ctx);
  PairSort ps;
  if ((st = ps.size((size_t)n, bits, what))) return st;
  ps.add(sc);
  size_t scan_bytes = 0;
  const auto kept = [](const float* w) { return rocprim::make_transform_iterator(w, IsKept()); };
  GVM_HIP_TRY(rocprim::exclusive_scan(nullptr, scan_bytes, kept(nullptr), (int*)nullptr, 0,
                                      (size_t)slots, rocprim::plus<int>()));
  const size_t ntaps = (size_t)kernel->m * kernel->n;
  sc.add(sizeof(float) * ntaps);
  if (!by_entry) {
    sc.add(sizeof(float4) * 2 * nvis);
    sc.add(sizeof(uint32_t) * (ntiles + 1));
  }
  sc.add(scan_bytes);
  sc.add(sizeof(int) * slots);
  sc.add(sizeof(float2) * slots);
  sc.add(sizeof(float) * slots);
  if ((st = sc.reserve(what))) return st;
  ps.take(sc);
  float* taps_d = sc.take<float>(ntaps);
  float4* rec = by_entry ? nullptr : sc.take<float4>(2 * nvis);
  uint32_t* start = by_entry ? nullptr : sc.take<uint32_t>(ntiles + 1);
  char* stmp = sc.take<char>(scan_bytes);
  int* pos = sc.take<int>(slots);
  float2* cvo = sc.take<float2>(slots);
  float* cw = sc.take<float>(slots);
  GVM_HIP_TRY(hipMemcpy(taps_d, kernel->taps, sizeof(float) * ntaps, hipMemcpyHostToDevice));
  const float2* vo = reinterpret_cast<const float2*>(vo_dev);
  if (by_entry) {
    hipLaunchKernelGGL(entry_keys_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, nullptr,
                       uvw_m_dev, nvis, g, ps.k[0], ps.v[0]);
    if ((st = launch_ok(what)) || (st = ps.sort((size_t)n, bits, what))) return st;
    hipLaunchKernelGGL(entry_cells_kernel, dim3(blocks_for(n)), dim3(kThreads), 0, nullptr,
                       ps.keys(), ps.ids(), n, nvis, g, taps_d, weight_dev, vo, cvo, cw);
    if ((st = launch_ok(what))) return st;
  } else {
    hipLaunchKernelGGL(grid_keys_kernel, dim3(blocks_for(nvis)), dim3(kThreads), 0, nullptr,
                       uvw_m_dev, weight_dev, vo, nvis, g, rec, ps.k[0], ps.v[0]);
    if ((st = launch_ok(what)) || (st = ps.sort((size_t)n, bits, what))) return st;
    hipLaunchKernelGGL(tile_first_kernel, dim3(blocks_for(ntiles + 1)), dim3(kThreads), 0, nullptr,
                       ps.keys(), n, ntiles, start);
    if ((st = launch_ok(what))) return st;
    const dim3 tiles(ntiles);
    if (g.wx * g.wy <= kLdsTaps)
      hipLaunchKernelGGL((grid_tiles_kernel<true>), tiles, dim3(kThreads), 0, nullptr, ps.ids(),
                         start, g, taps_d, rec, cvo, cw);
    else
      hipLaunchKernelGGL((grid_tiles_kernel<false>), tiles, dim3(kThreads), 0, nullptr, ps.ids(),
                         start, g, taps_d, rec, cvo, cw);
    if ((st = launch_ok(what))) return st;
  }
  // output row of each kept cell
  GVM_HIP_TRY(rocprim::exclusive_scan(stmp, scan_bytes, kept(cw), pos, 0, (size_t)slots,
                                      rocprim::plus<int>()));
  int last = 0;
  float last_w = 0.f;
  GVM_HIP_TRY(hipMemcpy(&last, pos + slots - 1, sizeof(int), hipMemcpyDeviceToHost));
  GVM_HIP_TRY(hipMemcpy(&last_w, cw + slots - 1, sizeof(float), hipMemcpyDeviceToHost));
  const long count = (long)last + IsKept()(last_w);
  if (count > capacity) {
    set_error("gvm_grid_visibilities_dev: " + std::to_string(count) +
              " gridded rows exceed the output capacity " + std::to_string(capacity));
    return GVM_ERR_ARG;
  }
  hipLaunchKernelGGL(grid_emit_kernel, dim3(blocks_for(slots)), dim3(kThreads), 0, nullptr, pos, g,
                     by_entry ? ps.keys() : nullptr, slots, cvo, cw, capacity, uvw_out_dev,
                     reinterpret_cast<float2*>(vo_out_dev), weight_out_dev);
  if ((st = launch_ok(what))) return st;
  GVM_HIP_TRY(hipDeviceSynchronize());
  sc.idle();
  *nout = count;
  return GVM_OK;
}

extern "C" gvm_status gvm_add_visibilities_gridded_dev(gvm_ctx* ctx, const gvm_ckernel* kernel,
                                                       float freq, long nvis,
                                                       const double* uvw_m_dev,
                                                       const float* vo_dev,
                                                       const float* weight_dev, long* ngridded,
                                                       int* slice_out) {
  static const char* what = "gvm_add_visibilities_gridded_dev";
  GVM_REQUIRE(ctx, "gvm_add_visibilities_gridded_dev: null context");
  GVM_HIP_TRY(hipSetDevice(ctx->device));
  const size_t cap = (size_t)ctx->g.M * ctx->g.N;
  // the gridded rows: uvw, Vo, weight (the gridder's scratch is the context's)
  struct Rows {
    char* p = nullptr;
    ~Rows() { (void)hipFree(p); }
  } rows;
  if (hipMalloc((void**)&rows.p, cap * (3 * sizeof(double) + 3 * sizeof(float))) != hipSuccess) {
    (void)hipGetLastError();
    rows.p = nullptr;
    set_error(std::string(what) + ": out of device memory");
    return GVM_ERR_OOM;
  }
  double* u = (double*)rows.p;
  float *v = (float*)(u + 3 * cap), *w = v + 2 * cap;
  long count = 0;
  gvm_status st = gvm_grid_visibilities_dev(ctx, kernel, freq, nvis, uvw_m_dev, vo_dev, weight_dev,
                                            u, v, w, (long)cap, &count);
  if (st) return st;
  GVM_REQUIRE(count > 0, "gvm_add_visibilities_gridded_dev: no visibility falls on the grid");
  if (ngridded) *ngridded = count;
  return gvm_add_visibilities_dev(ctx, freq, count, u, v, w, slice_out);
}

extern "C" gvm_status gvm_set_gcf(gvm_ctx* ctx, const float* gcf_host) {
  GVM_REQUIRE(ctx, "gvm_set_gcf: null context");
  GVM_REQUIRE(!ctx->capturing, "gvm_set_gcf: capturing");
  GVM_HIP_TRY(hipSetDevice(ctx->device));
  GVM_HIP_TRY(hipStreamSynchronize(ctx->stream));
  ctx->epoch++;
  if (!gcf_host) {
    if (ctx->gcf) (void)hipFree(ctx->gcf);
    ctx->gcf = nullptr;
    return GVM_OK;
  }
  const size_t n = (size_t)ctx->g.M * ctx->g.N;
  if (!ctx->gcf) GVM_HIP_TRY(hipMalloc((void**)&ctx->gcf, sizeof(float) * n));
  GVM_HIP_TRY(hipMemcpy(ctx->gcf, gcf_host, sizeof(float) * n, hipMemcpyHostToDevice));
  return GVM_OK;
}

extern "C" gvm_status gvm_weighting_apply_dev(gvm_ctx* ctx, int scheme, float robust,
                                              const gvm_uvtaper* taper, int nsl,
                                              const float* freq, const long* nvis,
                                              const double* const* uvw_m_dev,
                                              float* const* weight_dev) {
  static const char* what = "gvm_weighting_apply_dev";
  GVM_REQUIRE(ctx && (nsl == 0 || (freq && nvis && uvw_m_dev && weight_dev)),
              "gvm_weighting_apply_dev: null argument");
  GVM_REQUIRE(scheme >= GVM_WEIGHTING_NATURAL && scheme <= GVM_WEIGHTING_RADIAL,
              "gvm_weighting_apply_dev: unknown weighting scheme");
  // BriggsWeightingScheme::setRobustParam (src/briggsweightingscheme.cu:13-21)
  GVM_REQUIRE(scheme != GVM_WEIGHTING_BRIGGS || (robust >= -2.0f && robust <= 2.0f),
              "gvm_weighting_apply_dev: robust parameter must be in [-2, 2]");
  GVM_HIP_TRY(hipSetDevice(ctx->device));
  const gvm_geometry& geo = ctx->g;
  const double dxr = geo.deltax * kRad, dyr = geo.deltay * kRad;
  WeightGeom g;
  g.absdu = std::fabs(1.0 / (geo.M * dxr));
  g.absdv = std::fabs(1.0 / (geo.N * dyr));
  g.cx = (double)(int)std::floor((double)(geo.N / 2));
  g.cy = (double)(int)std::floor((double)(geo.M / 2));
  g.M = geo.M;
  g.N = geo.N;
  g.off = (uint32_t)((long)geo.M * geo.N);
  TaperCoef tc{};
  if (taper) {
    // the float coefficients of UVTaper::getValue
    const float cb = std::cos(taper->bpa), sb = std::sin(taper->bpa);
    const float s2 = std::sin(2.0f * taper->bpa);
    const float smaj2 = 2.0f * taper->sigma_maj * taper->sigma_maj;
    const float smin2 = 2.0f * taper->sigma_min * taper->sigma_min;
    tc.a = (cb * cb) / smaj2 + (sb * sb) / smin2;
    tc.b = s2 / smaj2 - s2 / smin2;
    tc.c = (sb * sb) / smaj2 + (cb * cb) / smin2;
    tc.amplitude = taper->amplitude;
    tc.u0 = taper->u_0;
    tc.v0 = taper->v_0;
    tc.on = 1;
  }
  long nmax = 0;
  for (int s = 0; s < nsl; s++) {
    GVM_REQUIRE(nvis[s] >= 0 && nvis[s] < (1L << 31) && freq[s] > 0.f &&
                    (nvis[s] == 0 || (uvw_m_dev[s] && weight_dev[s])),
                "gvm_weighting_apply_dev: bad slice");
    nmax = std::max(nmax, nvis[s]);
  }
  if (nsl == 0 || nmax == 0) return GVM_OK;
  const bool gridded = scheme == GVM_WEIGHTING_UNIFORM || scheme == GVM_WEIGHTING_BRIGGS;
  const int bits = key_bits(g.off);
  gvm_status st;
  const size_t cells = (size_t)geo.M * geo.N, gbytes = sizeof(float) * cells;
  Scratch sc(ctx);
  PairSort ps;
  float *grid = nullptr, *sorted = nullptr;
  double* part = nullptr;  // per slice: kSumBlocks partials of sum w, then of sum G^2
  if (gridded) {
    for (int s = 0; s < nsl; s++)
      if (nvis[s] > 0 && (st = ps.size((size_t)nvis[s], bits, what))) return st;
    ps.add(sc);
    sc.add(gbytes);
    sc.add(sizeof(float) * nmax);
    if (scheme == GVM_WEIGHTING_BRIGGS) sc.add(sizeof(double) * 2 * kSumBlocks * nsl);
    if ((st = sc.reserve(what))) return st;
    ps.take(sc);
    grid = sc.take<float>(cells);
    sorted = sc.take<float>(nmax);
    if (scheme == GVM_WEIGHTING_BRIGGS) part = sc.take<double>(2 * (size_t)kSumBlocks * nsl);
  }
  // the cell sums of slice s (added to the grid's when cumulative)
  auto cell_sums = [&](int s, int cumulative) -> gvm_status {
    g.lambda = (double)(2.99792458E8f / freq[s]);
    hipLaunchKernelGGL(weight_keys_kernel, dim3(blocks_for(nvis[s])), dim3(kThreads), 0, nullptr,
                       uvw_m_dev[s], nvis[s], g, ps.k[0], ps.v[0]);
    gvm_status r;
    if ((r = launch_ok(what)) || (r = ps.sort((size_t)nvis[s], bits, what))) return r;
    hipLaunchKernelGGL(weight_gather_kernel, dim3(blocks_for(nvis[s])), dim3(kThreads), 0, nullptr,
                       ps.ids(), weight_dev[s], nvis[s], sorted);
    hipLaunchKernelGGL(weight_cells_kernel, dim3(blocks_for(nvis[s])), dim3(kThreads), 0, nullptr,
                       ps.keys(), sorted, nvis[s], g.off, cumulative, grid);
    return launch_ok(what);
  };

  float f2 = 0.0f;
  if (scheme == GVM_WEIGHTING_BRIGGS) {
    // Pass 1 (src/briggsweightingscheme.cu:44-105): the sum of the weights,
    // and per slice the sum of G^2 over the right half of a grid that is not
    // cleared between slices (the reference clears it only after the pass).
    GVM_HIP_TRY(hipMemsetAsync(grid, 0, gbytes, nullptr));
    const int nbg = std::min(kSumBlocks, blocks_for((long)geo.M * (geo.N - geo.N / 2)));
    for (int s = 0; s < nsl; s++) {
      if (nvis[s] == 0) continue;
      double* p = part + 2 * (size_t)kSumBlocks * s;
      hipLaunchKernelGGL(weight_sum_kernel, dim3(std::min(kSumBlocks, blocks_for(nvis[s]))),
                         dim3(kThreads), 0, nullptr, weight_dev[s], nvis[s], p);
      if ((st = launch_ok(what)) || (st = cell_sums(s, 1))) return st;
      hipLaunchKernelGGL(grid_sq_sum_kernel, dim3(nbg), dim3(kThreads), 0, nullptr, grid, geo.M,
                         geo.N, p + kSumBlocks);
      if ((st = launch_ok(what))) return st;
    }
    // the FP64 sums of the block partials, in block order, slice after slice
    std::vector<double> h(2 * (size_t)kSumBlocks * nsl);
    GVM_HIP_TRY(hipMemcpy(h.data(), part, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
    double sum_w = 0.0, sum_g2 = 0.0;
    for (int s = 0; s < nsl; s++) {
      if (nvis[s] == 0) continue;
      const double* p = h.data() + 2 * (size_t)kSumBlocks * s;
      double a = 0.0, b = 0.0;
      for (int k = 0; k < std::min(kSumBlocks, blocks_for(nvis[s])); k++) a += p[k];
      for (int k = 0; k < nbg; k++) b += p[kSumBlocks + k];
      sum_w += a;
      sum_g2 += b;
    }
    GVM_REQUIRE(sum_w != 0.0, "gvm_weighting_apply_dev: the sum of the weights is zero");
    const float average_weights = (float)sum_g2 / (float)sum_w;
    const float f = 5.0f * std::pow(10.0f, -robust);
    f2 = f * f / average_weights;
  }

  // Pass 2: per slice, the slice's own weight grid, then the row update.  (With
  // one slice Briggs' first pass has left that grid.)
  for (int s = 0; s < nsl; s++) {
    if (nvis[s] == 0) continue;
    g.lambda = (double)(2.99792458E8f / freq[s]);
    if (gridded && !(scheme == GVM_WEIGHTING_BRIGGS && nsl == 1)) {
      GVM_HIP_TRY(hipMemsetAsync(grid, 0, gbytes, nullptr));
      if ((st = cell_sums(s, 0))) return st;
    }
    hipLaunchKernelGGL(weight_apply_kernel, dim3(blocks_for(nvis[s])), dim3(kThreads), 0, nullptr,
                       scheme, uvw_m_dev[s], nvis[s], g, grid, f2, tc, weight_dev[s]);
    if ((st = launch_ok(what))) return st;
  }
  GVM_HIP_TRY(hipDeviceSynchronize());
  sc.idle();
  return GVM_OK;
}
