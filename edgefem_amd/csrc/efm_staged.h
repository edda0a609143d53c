// q = A p with the columns that a tile of rows reads staged in LDS.
//
// A row-by-row SpMV looks every entry's column up through the address unit: 16 entries per row,
// two 16-byte values each for two right-hand sides, and at 1.6 M rows and 25 M entries these
// lookups, not the matrix's bytes, set its time (reading 8 instead of 16 bytes per value
// changed 135 us to 138).  kTile consecutive rows read about 3.4 kTile distinct columns
// (a 49 x 25 x 193-node guide; 256 rows: 4.1, 64 rows: 4.4), so a block loads those into LDS
// once and its rows gather them there by 16-bit local indices.
//
// Matrix storage, per tile: rows sorted by length (ties in row order), one row per thread, the
// entries of a wavefront's 64 rows step-major in pairs: the real parts of two entries are one
// 16-byte load per lane and their indices one 4-byte load, every load of a wavefront is
// contiguous, and the padding (to the wavefront's longest row, in pairs) is 9 % of the entries.
// Imaginary parts have an array of the same shape, read by the tiles that have any.
// A block has the first pairs of its rows on the way while it waits for the staged columns.
//
// Two right-hand sides, us per launch, entries looked up one by one against this: 173 k rows 15,
// 10; 378 k 37, 24; 1.59 M, real values 135, 86; 1.59 M with an absorbing slab in half the tiles
// 135, 111.  Measured worse: all pairs of a row loaded ahead (100), eight or one instead of four
// (97, 97), the loads before the staged columns' (87 and 20 % at 378 k), values through the caches
// (107), streamed stores of q (116), 256 rows per tile (90; 1,024: 85, at one block per CU).
#pragma once

#include "efm_internal.h"

#include <type_traits>

namespace efm_staged {

using namespace efm;

constexpr int kTile = 512;                // rows of a tile, threads of a block
constexpr int kWavesT = kTile / 64;
constexpr int kPre = 2;                   // pairs of a row loaded at a time, two groups ahead
constexpr int kMostRhs = 2;
constexpr int kRedBytes = kWavesT * kMostRhs * 16;
constexpr int kMaxLds = 80 * 1024 - kRedBytes;  // staged columns: with the sums' LDS, two blocks per CU
constexpr int kMaxWords = 16384;          // words of the window of columns of a tile
constexpr int kMaxLen = 255;              // entries of a row

// Rows of every tile by decreasing length: srow[tile kTile + t] = local row (0xFFFF: none), pairs
// of every wavefront, first and last column of the tile.  One block per tile.
__global__ void __launch_bounds__(kTile)
    k_order(int n, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
            uint16_t *__restrict__ srow, int32_t *__restrict__ pairs, int2 *__restrict__ window,
            int *__restrict__ bad) {
  __shared__ int len[kTile], lo, hi;
  const int t = threadIdx.x, r0 = blockIdx.x * kTile, row = r0 + t;
  const int32_t k0 = row < n ? row_ptr[row] : 0, k1 = row < n ? row_ptr[row + 1] : 0;
  len[t] = row < n ? k1 - k0 : -1;
  if (t == 0) {
    lo = r0;
    hi = min(n, r0 + kTile) - 1;
  }
  srow[r0 + t] = 0xFFFF;
  __syncthreads();
  int mn = n, mx = -1;
  for (int32_t k = k0; k < k1; ++k) {
    mn = min(mn, col[k]);
    mx = max(mx, col[k]);
  }
  atomicMin(&lo, mn);
  atomicMax(&hi, mx);
  if (len[t] > kMaxLen)
    *bad = 1;
  // rank of this row: longer rows, and rows of the same length before it
  int rank = 0;
  for (int j = 0; j < kTile; ++j)
    rank += len[j] > len[t] || (len[j] == len[t] && j < t);
  __syncthreads();
  if (row < n)
    srow[r0 + rank] = (uint16_t)t;
  if (rank % 64 == 0)  // the longest row of its wavefront
    pairs[blockIdx.x * kWavesT + rank / 64] = (max(len[t], 0) + 1) / 2;
  if (t == 0)
    window[blockIdx.x] = make_int2(lo, hi);
}

// Distinct columns of every tile (its rows included), ascending, nu of them (-1: more than cap);
// local indices of the entries (pairs, padding 0) and of the rows.  One block per tile; dynamic
// LDS 2 * words uint32, words = of the widest window.
__global__ void __launch_bounds__(kTile)
    k_index(int n, int words, int cap, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
            const uint16_t *__restrict__ srow, const int2 *__restrict__ steps, const int2 *__restrict__ window,
            int32_t *__restrict__ ucol, int32_t *__restrict__ nu, uint16_t *__restrict__ sown,
            uint32_t *__restrict__ sidx) {
  extern __shared__ uint32_t sm[];
  __shared__ uint32_t wsum[kTile];
  uint32_t *bits = sm, *pre = sm + words;
  const int t = threadIdx.x, r0 = blockIdx.x * kTile;
  const int base = window[blockIdx.x].x & ~31, nw = (window[blockIdx.x].y - base) / 32 + 1;
  const int32_t e0 = row_ptr[r0], e1 = row_ptr[min(n, r0 + kTile)];
  for (int w = t; w < nw; w += kTile)
    bits[w] = 0;
  __syncthreads();
  for (int32_t k = e0 + t; k < e1; k += kTile) {
    const int c = col[k] - base;
    atomicOr(&bits[c >> 5], 1u << (c & 31));
  }
  if (r0 + t < n)
    atomicOr(&bits[(r0 + t - base) >> 5], 1u << ((r0 + t - base) & 31));
  __syncthreads();
  const int per = (nw + kTile - 1) / kTile, w0 = min(nw, t * per), w1 = min(nw, w0 + per);
  uint32_t s = 0;
  for (int w = w0; w < w1; ++w) {
    pre[w] = s;
    s += __popc(bits[w]);
  }
  wsum[t] = s;
  __syncthreads();
  for (int off = 1; off < kTile; off <<= 1) {
    const uint32_t v = t >= off ? wsum[t - off] : 0;
    __syncthreads();
    wsum[t] += v;
    __syncthreads();
  }
  const bool fits = wsum[kTile - 1] <= (uint32_t)cap;
  if (t == 0)
    nu[blockIdx.x] = fits ? (int)wsum[kTile - 1] : -1;
  if (!fits)
    return;
  const uint32_t first = wsum[t] - s;
  int32_t *out = ucol + (int64_t)blockIdx.x * cap;
  for (int w = w0; w < w1; ++w) {
    pre[w] += first;
    uint32_t b = bits[w], at = pre[w];
    while (b) {
      out[at++] = base + w * 32 + __ffs(b) - 1;
      b &= b - 1;
    }
  }
  __syncthreads();
  auto rank = [&](int c) { return pre[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1)); };
  const int lr = srow[r0 + t];
  const bool in = lr != 0xFFFF;
  const int row = r0 + (in ? lr : 0);
  const int32_t k0 = row_ptr[row], k1 = in ? row_ptr[row + 1] : k0;
  sown[r0 + t] = (uint16_t)rank(row - base);
  const int2 stp = steps[blockIdx.x * kWavesT + t / 64];
  for (int j = 0; j < stp.y; ++j) {
    const int32_t k = k0 + 2 * j;
    uint32_t v = 0;
    if (k < k1)
      v = rank(col[k] - base);
    if (k + 1 < k1)
      v |= rank(col[k + 1] - base) << 16;
    sidx[((int64_t)stp.x + j) * 64 + t % 64] = v;
  }
}

// Real and imaginary parts of the installed values in the layout of k_index; iflag[tile] = 1
// where an imaginary part is not zero.  One block per tile.
__global__ void __launch_bounds__(kTile)
    k_values(int n, const int32_t *__restrict__ row_ptr, const double2 *__restrict__ val,
             const uint16_t *__restrict__ srow, const int2 *__restrict__ steps, double2 *__restrict__ sre,
             double2 *__restrict__ sim, int *__restrict__ iflag) {
  const int t = threadIdx.x, r0 = blockIdx.x * kTile;
  const int lr = srow[r0 + t];
  const int32_t k0 = lr != 0xFFFF ? row_ptr[r0 + lr] : 0, k1 = lr != 0xFFFF ? row_ptr[r0 + lr + 1] : 0;
  const int2 stp = steps[blockIdx.x * kWavesT + t / 64];
  int any = 0;
  for (int j = 0; j < stp.y; ++j) {
    const int32_t k = k0 + 2 * j;
    const double2 a = k < k1 ? val[k] : make_double2(0, 0), b = k + 1 < k1 ? val[k + 1] : make_double2(0, 0);
    const int64_t at = ((int64_t)stp.x + j) * 64 + t % 64;
    sre[at] = make_double2(a.x, b.x);
    if (sim)
      sim[at] = make_double2(a.y, b.y);
    any |= a.y != 0.0 || b.y != 0.0;
  }
  any = __syncthreads_or(any);
  if (t == 0)
    iflag[blockIdx.x] = any;
}

// q = A p, partials p^T q.  One block per tile, the tiles of an XCD consecutive; dynamic LDS of
// the largest tile's columns.
template <int R, typename State>
__global__ void __launch_bounds__(kTile) __attribute__((amdgpu_waves_per_eu(6, 8)))
    k_staged(int n, int ntiles, int xcd_span, int cap, const int2 *__restrict__ steps,
           const uint16_t *__restrict__ srow, const uint16_t *__restrict__ sown, const int32_t *__restrict__ ucol,
           const int32_t *__restrict__ nu, const uint32_t *__restrict__ sidx, const double2 *__restrict__ sre,
           const double2 *__restrict__ sim, const int *__restrict__ iflag, const double2 *__restrict__ p,
           double2 *__restrict__ q, double2 *__restrict__ partial, const State *__restrict__ st) {
  extern __shared__ double2 xs[];
  __shared__ double2 red[kWavesT][R];
  static_assert(R <= kMostRhs && sizeof(red) <= kRedBytes, "two blocks per CU");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lb = blockIdx.x >> 3, tile = (blockIdx.x & 7) * xcd_span + lb;
  double2 pq[R];
#pragma unroll
  for (int s = 0; s < R; ++s)
    pq[s] = make_double2(0, 0);
  if (lb < xcd_span && tile < ntiles) {
    const int r0 = tile * kTile;
    const int2 stp = steps[tile * kWavesT + wave];
    const bool cplx = iflag[tile] != 0;
    const int lr = srow[r0 + t], own = sown[r0 + t] * R;
    const int64_t at = (int64_t)stp.x * 64 + lane;
    const int m = nu[tile] * R;
    const int32_t *uc = ucol + (int64_t)tile * cap;
    for (int i0 = t; i0 < m; i0 += 4 * kTile) {
      int g[4];
      double2 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = min(i0 + k * kTile, m - 1);
        g[k] = uc[i / R] * R + i % R;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = p[g[k]];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i0 + k * kTile < m)
          xs[i0 + k * kTile] = v[k];
    }
    double2 acc[R];
#pragma unroll
    for (int s = 0; s < R; ++s)
      acc[s] = make_double2(0, 0);
    auto rows = [&](auto with_im) {
      constexpr bool C = decltype(with_im)::value;
      // two groups of kPre pairs are on their way; past the wavefront's last pair the first one
      // is read again, and not used
      double2 a[2][kPre], b[2][C ? kPre : 1];
      uint32_t c[2][kPre];
      auto load = [&](int h, int j0) {
#pragma unroll
        for (int j = 0; j < kPre; ++j) {
          const int64_t i = at + (j0 + j < stp.y ? j0 + j : 0) * 64;
          a[h][j] = ld_stream(sre + i);
          if (C)
            b[h][j] = ld_stream(sim + i);
          c[h][j] = __builtin_nontemporal_load(sidx + i);
        }
      };
      load(0, 0);
      load(1, kPre);
      __syncthreads();
      for (int j0 = 0; j0 < stp.y; j0 += 2 * kPre)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int jh = j0 + h * kPre;
          if (jh >= stp.y)
            break;
#pragma unroll
          for (int j = 0; j < kPre; ++j) {
            if (jh + j >= stp.y)
              continue;
            const int c0 = (int)(c[h][j] & 0xFFFFu) * R, c1 = (int)(c[h][j] >> 16) * R;
            const double2 re = a[h][j], im = C ? b[h][j] : make_double2(0, 0);
#pragma unroll
            for (int s = 0; s < R; ++s) {
              const double2 x0 = xs[c0 + s], x1 = xs[c1 + s];
              if (C) {
                acc[s] = cfma(make_double2(re.x, im.x), x0, acc[s]);
                acc[s] = cfma(make_double2(re.y, im.y), x1, acc[s]);
              } else {
                acc[s].x = fma(re.x, x0.x, acc[s].x);
                acc[s].y = fma(re.x, x0.y, acc[s].y);
                acc[s].x = fma(re.y, x1.x, acc[s].x);
                acc[s].y = fma(re.y, x1.y, acc[s].y);
              }
            }
          }
          if (jh + 2 * kPre < stp.y)
            load(h, jh + 2 * kPre);
        }
    };
    if (cplx)
      rows(std::true_type{});
    else
      rows(std::false_type{});
    if (lr != 0xFFFF) {
#pragma unroll
      for (int s = 0; s < R; ++s) {
        if (st[s].active == 0)
          continue;
        q[(int64_t)(r0 + lr) * R + s] = acc[s];
        pq[s] = cmul(xs[own + s], acc[s]);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < R; ++s) {
    group_sum<64>(pq[s]);
    if (lane == 0)
      red[wave][s] = pq[s];
  }
  __syncthreads();
  if (t < R) {
    double2 sum = red[0][t];
    for (int w = 1; w < kWavesT; ++w)
      sum = cadd(sum, red[w][t]);
    partial[(int64_t)blockIdx.x * R + t] = sum;
  }
}

} // namespace efm_staged
