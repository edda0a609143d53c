// COCG in one persistent kernel, for systems whose matrix fits in the register files.
//
// On systems of up to about 10^5 rows every kernel of an iteration is a chain of a few
// memory round trips behind a launch: 4-8 us each, five per iteration, whatever the size.
// Here one launch runs all iterations.  us per iteration with two right-hand sides, the best
// variant in launches against this kernel: 780 rows 22.1, 11.7; 4.3 k 23.5, 13.1; 31 k 27.5, 18.0;
// 103 k 37.4, 32.9; 130 k 40.8, 37.7.  31 k rows, one right-hand side 20.7, 14.1; three 33.8, 26.3;
// four 41.2, 36.1; two with two low-rank terms 35.1, 29.9 (103 k: 51.5, 49.6).  Of the 18 us (123
// blocks) about two thirds are the two grid sums and a sixth the third barrier: what is left is
// waiting, not work.
// Block b owns rpb consecutive rows: their z, r, p live in registers of their element's
// thread, their matrix entries in registers of their row's lanes (kRL lanes per row, kJ
// entries each; longer rows read the rest from memory), so an iteration moves only what
// blocks exchange: z, p, q, r, the nodal y and the partial sums.  p = z + beta p is formed
// wherever it is gathered (z and the previous p are exchanged), which costs no wait of its own.
//
// Exchange.  The L2 caches of the XCDs are not coherent with each other for ordinary
// accesses.  Exchanged values are stored and loaded with the device-coherent cache policy
// (sc1: past the XCD's L2), a block waits for its stores before it tells the others, and
// nothing else that another block reads is written, so no cache is written back or
// invalidated (with agent-scope fences by one thread per block a barrier of 64 blocks took
// 2.6-3.3 us instead of 1.3).
//
// Barrier.  Eight arrival counters on cache lines of their own; the first wave adds one to
// its block's counter and polls all eight at once (1.3 us with 64 blocks, 1.6 with 256; one
// counter for all: 1.9 and 4.1).  A sum over the grid is a barrier after the blocks' partial
// sums are stored: every block adds all of them in the same order and advances the same
// scalars, so the control flow is the same in every block and the result does not depend on
// timing.  (Publishing data and arrival in one word, 32 bits of data and a tag each, saves a
// round trip with few blocks, 13.4 against 14.5 us per iteration with 4, and loses with many:
// every block polls 12 words of every other, 22 against 19 us with 123.)
//
// A block needs a CU to itself at most, and a launch has no more blocks than CUs.  Launches of
// several threads on streams of their own could each get a part of the CUs and wait for
// the rest, so a launch is admitted (Gate) while the blocks in flight on its device fit
// on every XCD: block b of a launch runs on XCD b % 8.
//
// Every wait ends: after Args::polls polls a block gives up, sets the error flag and leaves,
// and so do the others; the caller then solves with one launch per step.  The launch is
// cooperative, so all blocks are resident.  kRowsMin rows per block: 64 and 128 measured no
// better at any size, as every block adds to the grid sums.
//
// The columns a block reads are loaded once per iteration into LDS (the block's distinct
// columns, k_persist_cols) and gathered from there by 16-bit local indices.
#pragma once

#include "efm_internal.h"

#include <condition_variable>
#include <mutex>
#include <type_traits>

namespace efm_persist {

using namespace efm;

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kRL = 4;                     // lanes per row
constexpr int kGroups = kThreads / kRL;    // rows per round
constexpr int kJ = 6;                      // entries of a row per lane in registers
constexpr int kCounters = 8;
constexpr int kCounterStride = 32;         // uint32 per 128-byte line
constexpr int kPolls = 1 << 21;            // of one wait at most, by default: a second or two
constexpr int kStage = 4;                  // staged columns per thread with their index in registers
constexpr int kNodeLanes = 8;
constexpr int kMaxLds = 150 * 1024;        // staged columns and LDS rows of a block
constexpr int kKR = 2;                     // rows per lane group in registers
constexpr int kRowsMin = 256;              // rows per block at least (fewer only add blocks to each grid sum)
// Entries of the longest row, and of a row on average, at most.  Entries past a lane group's
// registers are a serial walk through memory, which the other blocks wait for at the next sum.
// us per iteration with one right-hand side, launches per step against this: 31 k rows of 16 with
// one of 256 17, 14, of 512 20, 21, of 1,000 24, 32; 31 k rows of 91 on average (118 at most) 27,
// 24, of 150 (186) 27, 36.
constexpr int kMaxRow = 256, kMaxMean = 96;
constexpr int kMaxLr = 4;                  // low-rank terms times right-hand sides
constexpr int kMaxD = 16;                  // doubles of a grid sum

struct Args {
  int n, N, nb, rpb, npb;                  // rows, nodes, blocks, rows and nodes per block
  int nsm;                                 // most distinct columns of a block
  int polls;                               // of one wait at most
  const int32_t *row_ptr;
  const uint16_t *lidx, *rloc;             // local index of every entry's column, of every row
  const int32_t *ucol, *nu;                // distinct columns of block b at row_ptr[r0] + r0
  const double2 *val, *dinv;
  const int2 *en;                          // edge end nodes (-1: none)
  const int32_t *n2e_ptr, *n2e;
  const int8_t *gsign;
  const double2 *dninv;
  double2 *x, *r, *z, *p, *p2, *q, *y;     // p2: the other copy of p
  double *part;                            // three regions of [nb][kMaxD] partial sums
  unsigned *cnt;
  int *err;
  int lr_P;                                // low-rank terms
  const int8_t *lr_port;                   // term of every row (-1: none)
  const double2 *lr_w, *lr_coef;
};

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t Rsrc;

// Device-coherent 16-byte accesses, element index i (range-checked by the descriptor).
__device__ inline Rsrc rsrc(const void *p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (unsigned)bytes, 0x00027000);
}
constexpr int kSc1 = 16;
__device__ inline double2 ldc(Rsrc r, int i) {
  const v4u v = __builtin_amdgcn_raw_buffer_load_b128(r, i * 16, 0, kSc1);
  double2 d;
  __builtin_memcpy(&d, &v, 16);
  return d;
}
__device__ inline void stc(Rsrc r, int i, double2 d) {
  v4u v;
  __builtin_memcpy(&v, &d, 16);
  __builtin_amdgcn_raw_buffer_store_b128(v, r, i * 16, 0, kSc1);
}
// every vector memory operation of this wave has completed
__device__ inline void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Launches in flight on a device of this process, each from its launch until its stream has ended
// it.  The first to wait is the next to enter, so small launches do not pass a large one by.
class Gate {
  struct Device {
    std::mutex turn, lock;
    std::condition_variable left;
    int used = 0;  // blocks per XCD
  };
  static Device &of(int dev) {
    static Device d[64];
    return d[dev & 63];
  }
  Device &d;
  const int mine;

public:
  Gate(int dev, int blocks, int ncu) : d(of(dev)), mine((blocks + 7) / 8) {
    std::lock_guard<std::mutex> t(d.turn);
    std::unique_lock<std::mutex> l(d.lock);
    d.left.wait(l, [&] { return d.used == 0 || d.used + mine <= ncu / 8; });
    d.used += mine;
  }
  ~Gate() {
    std::lock_guard<std::mutex> l(d.lock);
    d.used -= mine;
    d.left.notify_all();
  }
  Gate(const Gate &) = delete;
  Gate &operator=(const Gate &) = delete;
};

// The scalars that a solve in separate launches keeps in memory (one system per lane).
struct Scal {
  double2 rho, alpha, beta;
  double bnorm2, rnorm2;
  int active, iters, breakdown;
};

// Distinct columns of every block's rows (and the rows themselves), ascending, and the local
// index of every entry: a bitmap of all columns in LDS, ranks by prefix sums of its words.
// longest: entries of the block's longest row.
// One block of kThreads per row block; dynamic LDS 2 * words uint32.
__global__ void __launch_bounds__(kThreads)
    k_persist_cols(int n, int rpb, const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col,
                   uint16_t *__restrict__ lidx, uint16_t *__restrict__ rloc, int32_t *__restrict__ ucol,
                   int32_t *__restrict__ nu, int32_t *__restrict__ longest) {
  extern __shared__ uint32_t sm[];
  const int words = (n + 31) / 32;
  uint32_t *bits = sm, *pre = sm + words;
  __shared__ uint32_t wsum[kThreads];
  __shared__ int mx;
  const int r0 = blockIdx.x * rpb, r1 = min(n, r0 + rpb);
  const int32_t k0 = row_ptr[r0], k1 = row_ptr[r1];
  for (int w = threadIdx.x; w < words; w += kThreads)
    bits[w] = 0;
  if (threadIdx.x == 0)
    mx = 0;
  __syncthreads();
  for (int32_t k = k0 + threadIdx.x; k < k1; k += kThreads) {
    const int32_t c = col[k];
    atomicOr(&bits[c >> 5], 1u << (c & 31));
  }
  for (int r = r0 + threadIdx.x; r < r1; r += kThreads) {
    atomicOr(&bits[r >> 5], 1u << (r & 31));
    atomicMax(&mx, row_ptr[r + 1] - row_ptr[r]);
  }
  __syncthreads();
  const int per = (words + kThreads - 1) / kThreads;
  const int w0 = min(words, (int)threadIdx.x * per), w1 = min(words, w0 + per);
  uint32_t s = 0;
  for (int w = w0; w < w1; ++w) {
    pre[w] = s;
    s += __popc(bits[w]);
  }
  wsum[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < kThreads; off <<= 1) {
    const uint32_t v = (int)threadIdx.x >= off ? wsum[threadIdx.x - off] : 0;
    __syncthreads();
    wsum[threadIdx.x] += v;
    __syncthreads();
  }
  const uint32_t base = wsum[threadIdx.x] - s;
  int32_t *out = ucol + (int64_t)k0 + r0;
  for (int w = w0; w < w1; ++w) {
    pre[w] += base;
    uint32_t b = bits[w], at = pre[w];
    while (b) {
      out[at++] = w * 32 + __ffs(b) - 1;
      b &= b - 1;
    }
  }
  if (threadIdx.x == 0) {
    nu[blockIdx.x] = (int32_t)wsum[kThreads - 1];
    longest[blockIdx.x] = mx;
  }
  __syncthreads();
  auto rank = [&](int32_t c) {
    return (uint16_t)(pre[c >> 5] + __popc(bits[c >> 5] & ((1u << (c & 31)) - 1)));
  };
  for (int32_t k = k0 + threadIdx.x; k < k1; k += kThreads)
    lidx[k] = rank(col[k]);
  for (int r = r0 + threadIdx.x; r < r1; r += kThreads)
    rloc[r] = rank(r);
}

__global__ void k_persist_lr_rows(int n, int64_t m, int64_t len, const int32_t *__restrict__ idx,
                                  const double2 *__restrict__ wv, int8_t *__restrict__ port,
                                  double2 *__restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m)
    return;
  const int32_t r = idx[i];
  if (r < 0 || r >= n)
    return;
  port[r] = (int8_t)(i / len);
  w[r] = wv[i];
}

template <int R> struct Shared {
  double2 alpha[R], beta[R];
  double2 t[kMaxLr];
  double wsum[kWaves][kMaxD];
  double tot[kMaxD];
  int act[R];
  int nact, err;
};

// Rows of a block at most, and its elements (row, system) per thread.  MORE: the matrix rows past
// kKR * kGroups of a block live in LDS (values and local indices) behind the staged columns.
constexpr int max_rows(bool more) { return (more ? 2 : 1) * kKR * kGroups; }
template <int R, bool MORE> constexpr int elems() { return (max_rows(MORE) * R + kThreads - 1) / kThreads; }

// R right-hand sides; AUX: with the nodal part of the preconditioner; LR: with low-rank
// terms.  nsm: staged columns of the largest block.  Starts from z, p, x, r and the state in memory, runs at most
// max_launch iterations, leaves the same there.
template <int R, bool AUX, bool MORE, bool LR, typename State, typename Ctl>
__global__ void __launch_bounds__(kThreads)
    k_cocg_persist(const Args a, State *__restrict__ st, Ctl *__restrict__ ctl, int max_launch, double tol2,
                   int max_it) {
  constexpr int KE = elems<R, MORE>(), KR = kKR;
  // doubles of the grid sums: p^T q; r^T z, |r|^2 and the terms' w^H z; w^H z and w^H p
  constexpr int DB = 2 * R, DD = 3 * R + (LR ? 2 * kMaxLr : 0), DL = 4 * kMaxLr;
  static_assert(DD <= kMaxD && DL <= kMaxD, "words of a record");
  extern __shared__ double2 lds_p[];
  __shared__ Shared<R> sh;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int blk = blockIdx.x;
  const int r0 = blk * a.rpb, r1 = min(a.n, r0 + a.rpb);
  const int nel = (r1 - r0) * R;
  const size_t vb = (size_t)a.n * R * 16;
  const Rsrc rz = rsrc(a.z, vb), rq = rsrc(a.q, vb), rr = rsrc(a.r, vb);
  const Rsrc ry = rsrc(a.y, AUX ? (size_t)a.N * R * 16 : 16);
  const Rsrc rpart = rsrc(a.part, (size_t)3 * a.nb * kMaxD * 8);
  unsigned epoch = 0;

  // ---- registers for the whole launch -------------------------------------------------
  double2 z[KE], rv[KE], pv[KE];
  int2 en[KE];
#pragma unroll
  for (int k = 0; k < KE; ++k) {
    const int e = tid + k * kThreads;
    const bool in = e < nel;
    const int i = r0 * R + (in ? e : 0), row = i / R;
    z[k] = a.z[i];
    rv[k] = a.r[i];
    pv[k] = a.p[i];
    en[k] = AUX ? a.en[row] : make_int2(-1, -1);
  }
  const int g = tid / kRL, l = tid % kRL;
  double2 av[KR][kJ];
  unsigned ai[KR][kJ / 2];      // two 16-bit local indices each
  int32_t kmore[KR], kend[KR];  // entries past the registers
  int own[KR];
#pragma unroll
  for (int h = 0; h < KR; ++h) {
    const int row = r0 + g + h * kGroups;
    const bool in = row < r1;
    const int rc = in ? row : r0;
    const int32_t kb = a.row_ptr[rc], ke = in ? a.row_ptr[rc + 1] : kb;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      const int32_t k = kb + l + j * kRL;
      const bool on = k < ke;
      av[h][j] = on ? a.val[k] : make_double2(0, 0);
      const unsigned c = on ? a.lidx[k] : 0;
      ai[h][j / 2] = (j & 1) ? ai[h][j / 2] | (c << 16) : c;
    }
    kmore[h] = kb + l + kJ * kRL;
    kend[h] = ke;
    own[h] = a.rloc[rc] * R;
  }
  // rows past the registers: values and local indices in LDS
  double2 *lds_v = lds_p + a.nsm * R;
  const int32_t km0 = MORE ? a.row_ptr[min(r1, r0 + KR * kGroups)] : 0;
  const int nmv = MORE ? a.row_ptr[r1] - km0 : 0;
  uint16_t *lds_i = reinterpret_cast<uint16_t *>(lds_v + nmv);
  if (MORE)
    for (int i = tid; i < nmv; i += kThreads) {
      lds_v[i] = a.val[km0 + i];
      lds_i[i] = a.lidx[km0 + i];
    }
  const int nst = a.nu[blk] * R;  // staged elements
  const int32_t *uc = a.ucol + (int64_t)a.row_ptr[r0] + r0;
  int sidx[kStage];
#pragma unroll
  for (int k = 0; k < kStage; ++k) {
    const int i = tid + k * kThreads;
    sidx[k] = i < nst ? uc[i / R] * R + i % R : 0;
  }
  // nodes of this block: the first round's incidence in registers
  const int m0 = AUX ? min(a.N, blk * a.npb) : 0, m1 = AUX ? min(a.N, m0 + a.npb) : 0;
  const int nlane = tid % kNodeLanes, ngrp = tid / kNodeLanes;
  int ne[2] = {0, 0}, ng[2] = {0, 0};
  int32_t nmore = 0, nend = 0;
  if (AUX && m0 + ngrp < m1) {
    const int nd = m0 + ngrp;
    const int32_t b = a.n2e_ptr[nd];
    nend = a.n2e_ptr[nd + 1];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int32_t k = b + nlane + j * kNodeLanes;
      if (k < nend) {
        ne[j] = a.n2e[k];
        ng[j] = a.gsign[k];
      }
    }
    nmore = b + nlane + 2 * kNodeLanes;
  }
  // scalars: system s in lane s of the first wave
  Scal sc{};
  if (wave == 0 && lane < R) {
    const State S = st[lane];
    sc.rho = S.rho;
    sc.alpha = S.alpha;
    sc.beta = S.beta;
    sc.bnorm2 = S.bnorm2;
    sc.rnorm2 = S.rnorm2;
    sc.active = S.active;
    sc.iters = S.iters;
    sc.breakdown = S.breakdown;
  }
  auto publish = [&]() {  // first wave
    if (lane < R) {
      sh.alpha[lane] = sc.alpha;
      sh.beta[lane] = sc.beta;
      sh.act[lane] = sc.active;
    }
    const int na = __popcll(__ballot(lane < R && sc.active != 0));
    if (lane == 0)
      sh.nact = na;
  };
  if (tid == 0)
    sh.err = 0;
  if (wave == 0)
    publish();
  __syncthreads();

  // First wave: arrive at the grid's barrier and wait for all blocks.
  auto arrive = [&]() {
    ++epoch;
    if (lane == 0)
      __hip_atomic_fetch_add(a.cnt + (blk % kCounters) * kCounterStride, 1u, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    const int c = lane < kCounters ? lane : 0;
    const unsigned want = epoch * (unsigned)((a.nb - c + kCounters - 1) / kCounters);
    int k = 0;
    for (; k < a.polls; ++k) {
      const unsigned v =
          __hip_atomic_load(a.cnt + c * kCounterStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__all((int)(v - want) >= 0))
        break;
    }
    if (k >= a.polls && lane == 0)
      sh.err = 1;
  };
  auto wave_sum = [&](double &v) {
#pragma unroll
    for (int off = 32; off >= 4; off >>= 1)
      v += __shfl_xor(v, off, 64);
    v += dpp_quad<0x4E>(v);
    v += dpp_quad<0xB1>(v);
  };
  // Sum v over the grid through partial region `reg`.  The return is a barrier of the grid for
  // the exchanged stores; the totals are in sh.tot for the first wave, which the caller's next
  // __syncthreads holds the others for.
  auto reduce = [&](auto &v, int reg) {
    constexpr int D = sizeof(v) / sizeof(v[0]), DP = (D + 1) / 2;
    static_assert(D <= kMaxD, "partial sums");
#pragma unroll
    for (int i = 0; i < D; ++i)
      wave_sum(v[i]);
    if (lane == 0)
#pragma unroll
      for (int i = 0; i < D; ++i)
        sh.wsum[wave][i] = v[i];
    __syncthreads();
    const int base = reg * a.nb * (kMaxD / 2);
    if (tid < DP) {
      double2 t = make_double2(0, 0);
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        t.x += sh.wsum[w][2 * tid];
        if (2 * tid + 1 < D)
          t.y += sh.wsum[w][2 * tid + 1];
      }
      stc(rpart, base + blk * DP + tid, t);
    }
    wait_stores();
    __syncthreads();
    if (wave == 0)
      arrive();
    __syncthreads();  // every block has arrived: what they exchanged may be read
    if (wave == 0) {
      double2 t[DP];
#pragma unroll
      for (int i = 0; i < DP; ++i)
        t[i] = make_double2(0, 0);
      for (int b = lane; b < a.nb; b += 64)
#pragma unroll
        for (int i = 0; i < DP; ++i)
          t[i] = cadd(t[i], ldc(rpart, base + b * DP + i));
#pragma unroll
      for (int i = 0; i < DP; ++i) {
        wave_sum(t[i].x);
        wave_sum(t[i].y);
        if (lane == 0) {
          sh.tot[2 * i] = t[i].x;
          if (2 * i + 1 < D)
            sh.tot[2 * i + 1] = t[i].y;
        }
      }
    }
  };
  auto total = [&](int i) { return sh.tot[i]; };
  auto barrier = [&]() {
    wait_stores();
    __syncthreads();
    if (wave == 0)
      arrive();
    __syncthreads();
  };
  // the low-rank terms' w^H u of this thread's elements, added to d[at + 2 i], d[at + 2 i + 1]
  auto lr_dot = [&](auto &d, auto at, const double2(&u)[KE]) {
#pragma unroll
    for (int k = 0; k < KE; ++k) {
      const int e = tid + k * kThreads, s = e % R, row = r0 + e / R;
      const int port = e < nel ? (int)a.lr_port[row] : -1;
      if (port < 0)
        continue;
      const double2 c = cmul(cconj(a.lr_w[row]), u[k]);
#pragma unroll
      for (int i = 0; i < kMaxLr; ++i)
        if (i == port * R + s) {
          d[at.value + 2 * i] += c.x;
          d[at.value + 2 * i + 1] += c.y;
        }
    }
  };
  // t = w^H p per term and system in lanes < kMaxLr of the first wave, by the recurrence of p
  double2 tz = make_double2(0, 0), tp = make_double2(0, 0);
  if (LR) {
    double d[DL];
#pragma unroll
    for (int i = 0; i < DL; ++i)
      d[i] = 0.0;
    lr_dot(d, std::integral_constant<int, 0>{}, z);
    lr_dot(d, std::integral_constant<int, 2 * kMaxLr>{}, pv);
    reduce(d, 2);
    __syncthreads();
    if (wave == 0 && lane < kMaxLr) {
      tz = make_double2(total(2 * lane), total(2 * lane + 1));
      tp = make_double2(total(2 * (kMaxLr + lane)), total(2 * (kMaxLr + lane) + 1));
    }
  }

  // z and the previous p of the staged columns, loaded while beta is formed
  double2 tzv[kStage], tpv[kStage];
  auto stage_loads = [&](const Rsrc &rpo) {
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
      tzv[k] = ldc(rz, sidx[k]);
      tpv[k] = ldc(rpo, sidx[k]);
    }
  };
  stage_loads(rsrc(a.p, vb));
  for (int it = 0; it < max_launch && sh.nact > 0 && !sh.err; ++it) {
    const Rsrc rpo = rsrc((it & 1) ? a.p2 : a.p, vb), rpn = rsrc((it & 1) ? a.p : a.p2, vb);
    // ---- p = z + beta p: the block's columns into LDS, its own elements exchanged ---------
    {
#pragma unroll
      for (int k = 0; k < KE; ++k) {
        const int e = tid + k * kThreads, s = e % R;
        if (e < nel && sh.act[s]) {
          pv[k] = cfma(sh.beta[s], pv[k], z[k]);
          stc(rpn, r0 * R + e, pv[k]);
        }
      }
      if (LR && wave == 0 && lane < kMaxLr) {
        const int s = lane % R;
        if (sh.act[s])
          tp = cfma(sh.beta[s], tp, tz);
        sh.t[lane] = lane / R < a.lr_P ? cmul(a.lr_coef[lane / R], tp) : make_double2(0, 0);
      }
#pragma unroll
      for (int k = 0; k < kStage; ++k) {
        const int i = tid + k * kThreads;
        if (i < nst)
          lds_p[i] = cfma(sh.beta[i % R], tpv[k], tzv[k]);
      }
      for (int i = tid + kStage * kThreads; i < nst; i += kThreads) {
        const int c = uc[i / R] * R + i % R;
        lds_p[i] = cfma(sh.beta[i % R], ldc(rpo, c), ldc(rz, c));
      }
    }
    __syncthreads();
    // ---- q = A p, partials p^T q ----------------------------------------------------------
    double pq[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
      pq[i] = 0.0;
    // the row's sum over its lanes, the terms, q and p^T q
    auto finish = [&](int row, int own_s, double2(&acc)[R]) {
#pragma unroll
      for (int s = 0; s < R; ++s)
        group_sum<kRL>(acc[s]);
      if (l == 0 && row < r1) {
        const int port = LR ? (int)a.lr_port[row] : -1;
        const double2 w = LR && port >= 0 ? a.lr_w[row] : make_double2(0, 0);
#pragma unroll
        for (int s = 0; s < R; ++s) {
          if (!sh.act[s])
            continue;
          if (LR && port >= 0)
            acc[s] = cfma(w, sh.t[port * R + s], acc[s]);
          stc(rq, row * R + s, acc[s]);
          const double2 c = cmul(lds_p[own_s + s], acc[s]);
          pq[2 * s] += c.x;
          pq[2 * s + 1] += c.y;
        }
      }
    };
#pragma unroll
    for (int h = 0; h < KR; ++h) {
      double2 acc[R];
#pragma unroll
      for (int s = 0; s < R; ++s)
        acc[s] = make_double2(0, 0);
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const int c = (int)((j & 1) ? ai[h][j / 2] >> 16 : ai[h][j / 2] & 0xFFFFu) * R;
#pragma unroll
        for (int s = 0; s < R; ++s)
          acc[s] = cfma(av[h][j], lds_p[c + s], acc[s]);
      }
      for (int32_t k = kmore[h]; k < kend[h]; k += kRL) {
        const double2 v = a.val[k];
        const int c = a.lidx[k] * R;
#pragma unroll
        for (int s = 0; s < R; ++s)
          acc[s] = cfma(v, lds_p[c + s], acc[s]);
      }
      finish(r0 + g + h * kGroups, own[h], acc);
    }
    if (MORE)
      for (int row0 = r0 + KR * kGroups; row0 < r1; row0 += kGroups) {
        const int row = row0 + g, rc = min(row, r1 - 1);
        const int kb = a.row_ptr[rc] - km0 + l, ke = row < r1 ? a.row_ptr[rc + 1] - km0 : 0;
        double2 acc[R];
#pragma unroll
        for (int s = 0; s < R; ++s)
          acc[s] = make_double2(0, 0);
        for (int k = kb; k < ke; k += kRL) {
          const double2 v = lds_v[k];
          const int c = lds_i[k] * R;
#pragma unroll
          for (int s = 0; s < R; ++s)
            acc[s] = cfma(v, lds_p[c + s], acc[s]);
        }
        finish(row, a.rloc[rc] * R, acc);
      }
    reduce(pq, 0);
    if (wave == 0) {
      if (lane < R && sc.active) {
        const double2 t = make_double2(total(2 * lane), total(2 * lane + 1));
        if (t.x == 0.0 && t.y == 0.0) {
          sc.breakdown = 1;
          sc.alpha = make_double2(0, 0);
        } else {
          sc.alpha = cdiv(sc.rho, t);
        }
      }
      publish();
    }
    // the loads below do not depend on alpha: they are on their way while it is formed
    double2 qv[KE];
#pragma unroll
    for (int k = 0; k < KE; ++k) {
      const int e = tid + k * kThreads;
      qv[k] = ldc(rq, r0 * R + (e < nel ? e : 0));
    }
    // ---- y = Dn^{-1} G^T (r - alpha q) ----------------------------------------------------
    if (AUX) {
      double2 fr[2][R], fq[2][R];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int s = 0; s < R; ++s) {
          fr[j][s] = ldc(rr, ne[j] * R + s);
          fq[j][s] = ldc(rq, ne[j] * R + s);
        }
      __syncthreads();
      for (int nd = m0 + ngrp; nd < m1; nd += kThreads / kNodeLanes) {
        double2 acc[R];
#pragma unroll
        for (int s = 0; s < R; ++s)
          acc[s] = make_double2(0, 0);
        const bool first = nd == m0 + ngrp;
        if (first)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int s = 0; s < R; ++s) {
              const double2 d = csub(fr[j][s], cmul(sh.alpha[s], fq[j][s]));
              acc[s].x += (double)ng[j] * d.x;
              acc[s].y += (double)ng[j] * d.y;
            }
        int32_t k = first ? nmore : a.n2e_ptr[nd] + nlane;
        const int32_t ke = first ? nend : a.n2e_ptr[nd + 1];
        for (; k < ke; k += kNodeLanes) {
          const int e = a.n2e[k];
          const double sg = (double)a.gsign[k];
#pragma unroll
          for (int s = 0; s < R; ++s) {
            const double2 d = csub(ldc(rr, e * R + s), cmul(sh.alpha[s], ldc(rq, e * R + s)));
            acc[s].x += sg * d.x;
            acc[s].y += sg * d.y;
          }
        }
        const double2 di = a.dninv[nd];
#pragma unroll
        for (int s = 0; s < R; ++s)
          group_sum<kNodeLanes>(acc[s]);
        if (nlane == 0)
#pragma unroll
          for (int s = 0; s < R; ++s)
            if (sh.act[s])
              stc(ry, nd * R + s, cmul(di, acc[s]));
      }
      barrier();
    } else {
      __syncthreads();
    }
    if (sh.err)
      break;
    // ---- x += alpha p, r -= alpha q, z = D^{-1} r + G y; partials r^T z, |r|^2 --------------
    double sd[DD];
#pragma unroll
    for (int i = 0; i < DD; ++i)
      sd[i] = 0.0;
    double2 ya[KE], yb[KE], xv[KE], dv[KE];
#pragma unroll
    for (int k = 0; k < KE; ++k) {
      const int e = tid + k * kThreads, s = e % R, i = r0 * R + (e < nel ? e : 0);
      const bool hn = en[k].x >= 0;
      if (AUX) {
        ya[k] = ldc(ry, (hn ? en[k].x : 0) * R + s);
        yb[k] = ldc(ry, (hn ? en[k].y : 0) * R + s);
      }
      xv[k] = a.x[i];
      dv[k] = a.dinv[i / R];
    }
#pragma unroll
    for (int k = 0; k < KE; ++k) {
      const int e = tid + k * kThreads, s = e % R;
      if (e >= nel || !sh.act[s])
        continue;
      const double2 al = sh.alpha[s];
      a.x[r0 * R + e] = cfma(al, pv[k], xv[k]);
      rv[k] = csub(rv[k], cmul(al, qv[k]));
      double2 zv = cmul(dv[k], rv[k]);
      if (AUX && en[k].x >= 0)
        zv = cadd(zv, csub(yb[k], ya[k]));
      z[k] = zv;
      stc(rz, r0 * R + e, zv);
      if (AUX)
        stc(rr, r0 * R + e, rv[k]);
      const double2 c = cmul(rv[k], zv);
      const double n2 = cabs2(rv[k]);
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (i == s) {
          sd[2 * i] += c.x;
          sd[2 * i + 1] += c.y;
          sd[2 * R + i] += n2;
        }
    }
    if (LR)
      lr_dot(sd, std::integral_constant<int, 3 * R>{}, z);
    reduce(sd, 1);
    stage_loads(rpn);
    if (wave == 0) {
      if (lane < R && sc.active) {
        const double2 c = make_double2(total(2 * lane), total(2 * lane + 1));
        const double n2 = total(2 * R + lane);
        sc.iters += 1;
        sc.rnorm2 = n2;
        if (n2 <= tol2 * sc.bnorm2 || sc.breakdown || (sc.rho.x == 0.0 && sc.rho.y == 0.0) || sc.iters >= max_it) {
          sc.active = 0;
        } else {
          sc.beta = cdiv(c, sc.rho);
          sc.rho = c;
        }
      }
      if (LR && lane < kMaxLr)
        tz = make_double2(total(3 * R + 2 * lane), total(3 * R + 2 * lane + 1));
      publish();
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < KE; ++k) {
    const int e = tid + k * kThreads, i = r0 * R + e;
    if (e < nel) {
      a.r[i] = rv[k];
      a.z[i] = z[k];
      a.p[i] = pv[k];
    }
  }
  if (sh.err && tid == 0)
    atomicOr(a.err, 1);
  if (blk == 0 && wave == 0) {
    if (lane < R) {
      State &S = st[lane];
      S.rho = sc.rho;
      S.alpha = sc.alpha;
      S.beta = sc.beta;
      S.rnorm2 = sc.rnorm2;
      S.active = sc.active;
      S.iters = sc.iters;
      S.breakdown = sc.breakdown;
    }
    if (lane == 0)
      ctl->n_active = sh.nact;
  }
}

} // namespace efm_persist
