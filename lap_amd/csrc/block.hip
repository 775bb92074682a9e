// block.hip -- Jacobi PCG for k right-hand sides sharing every SpMM
// (lap_pcg_block), and the SpMM itself (lap_csr_matmat).
//
// The k columns run k independent CG recurrences (cg.c:5-140 each, with
// line_jacobi) whose SpMVs are fused into one SpMM Q = A P: the CSR matrix
// is read once per iteration for all k columns (12 B per nonzero amortised
// over k).  Block vectors are row-interleaved (n x k, element (i, j) at
// i*k + j), so a row of P is one contiguous 8k-byte run and a CSR column
// index addresses a whole run.
//
// SpMM: one column per lane; a wave holds G = 64/k row groups of k lanes and
// takes kRW consecutive rows (a chunk) at a time, whose row pointers, column
// indices and values it loads into LDS while it works on the chunk before: the
// gathers of P then wait for nothing but P.  (Loading index, value and P one
// after the other left 2/3 of the time to the index's latency.)  A gather past
// a row's end reads +0.0 by the buffer's bounds check, which saves the compares
// and selects of 8 nonzeros per row.  Each group takes RU rows per step
// and issues the gathers of EU nonzeros of each before summing them; the sums
// themselves run in CSR order, one per column, which is the reference's
// simple_csr_matvec sum (simple_blas.c:24-44) bit for bit whatever RU is.  RU
// (1, 2, 4) is picked per (matrix, k) by timing the candidates once.  A chunk
// with too many nonzeros for its LDS reads them from memory as it goes (add_far).
//
// Workgroups are dealt to the 8 XCDs in turn, each with an L2 of its own, so
// the chunks are handed out such that a row's neighbours are mostly worked on
// by the same XCD (spmm_shape).
//
// Measured at 96^3, k = 32: 418 -> 200 us, the whole iteration 785 -> 505.  It
// moves 347 MB in and 228 out of memory (the least is 300 and 226), and 1.4 GB
// from the L2s to the CUs: 6 of the 8 rows of P that a row reads are not in the
// CU's L1, and that is what bounds it now (RU, 2 to 8 workgroups per CU and
// fewer instructions change little).
//
// Per-column scalars (rho, alpha, beta, tolrel, flags) live in a device
// control block.  One iteration is five launches, graph-replayed:
//   spmm    Q = A P, per-workgroup per-column partials of P.Q
//   alpha   a workgroup per column: alpha_j = rho_j / (p.q)_j
//   update  R -= alpha Q; partials of R.W (W = d_r R) and R.R
//   conv    a workgroup per column: convergence test (cg.c:106-123), beta
//   dir     X += alpha P for the columns live in this iteration, then
//           P = beta P + d_r R for the columns still live
// Moving x += alpha p from `update` into `dir` reads P once per iteration
// instead of twice; the x of a column that stops is still updated in the
// iteration it stops, as in cg.c.  A stopped column keeps its x, iteration
// count and residual, as a single-RHS solve does.
#include <algorithm>
#include <climits>
#include <cmath>

#include "boxed.hpp"
#include "cls.hpp"
#include "lap_core.hpp"

namespace lap {

namespace {

constexpr int kMaxK = 64;         // columns per block solve

struct BlkCtl {
  double rho[kMaxK], alpha[kMaxK], beta[kMaxK], tolrel[kMaxK], res0[kMaxK], res[kMaxK];
  int done[kMaxK];  // column stopped (converged / maxit / non-finite)
  int xup[kMaxK];   // column was live in the last finished iteration
  int flag[kMaxK], iters[kMaxK];
  int maxit, all_done;  // all_done: every column has stopped
  int left, pad;        // columns that have not
};

// ---------------------------------------------------------------- SpMM

// The rows a wave works on at a time, and the nonzeros of them it has room for
// (a lane's loads of each).  ONE: a row per lane group instead of 16 rows or
// more.  16 rows in a row are one wave's serial work where they are long or hubs,
// and few waves' where there are few.  Gain of k = 32 and 64 over a kernel
// without chunks, 16 rows and ONE: power-law graph of 100,000 nodes (rows of up to
// 10,676 entries) 0.96 / 0.32 and 3.7 / 3.0; 10,000 rows of 17 entries 1.11 / 0.89
// and 1.16 / 0.98, 2000 of 101 0.76 / 0.46 and 1.58 / 1.32; but the 96^3 grid 2.17
// / 1.39 and 1.24 / 0.82, 200,000 rows of 17 1.79 / 1.24 and 1.39 / 0.96.  So ONE
// for up to one chunk of 16 rows per SIMD and for rows of more than the LDS of a
// chunk; with k < 16, whose groups are more, it is not needed.
constexpr int kOneK = 16, kOneRows = 16 * 1024, kOneLong = 256;
template <int K, bool ONE>
struct Chunk {
  static constexpr int G = 64 / K;
  static constexpr int kRW = ONE || G > 16 ? G : 16;
  static constexpr int kEPL = G > 16 ? 8 : 4;
  static constexpr int kCap = kEPL * 64;
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Q = A P for K columns.  MODE 0: plain (lap_csr_matmat); 1: partials of
// P.Q per column; 2: Q = -(A P - B) (initial residual) with partials of
// Q.Q.  Partials: part[col * gridDim.x + blockIdx.x].
// FAR: P has 4 GB or more, beyond the 32-bit offsets of a buffer load.
template <int BS, int K, int RU, int EU, int MODE, bool FAR, bool ONE>
__global__ __launch_bounds__(BS) void k_spmm(int n, const int *__restrict__ ia,
                                             const int *__restrict__ ja,
                                             const double *__restrict__ a,
                                             const double *__restrict__ P, double *__restrict__ Q,
                                             const double *__restrict__ Bm, double *part,
                                             const BlkCtl *ctl, int group) {
  if (MODE == 1 && ctl->all_done) return;
  using C = Chunk<K, ONE>;
  constexpr int G = C::G, RW = C::kRW, EPL = C::kEPL, NW = BS / 64;
  static_assert(RW % (G * RU) == 0 && RW <= 64, "whole steps per chunk");
  // a nonzero: its value and the byte offset (FAR: the number) of its row of P;
  // the last one stands for none
  struct __align__(16) Nz {
    double v;
    unsigned at, pad;
  };
  __shared__ Nz s_nz[NW][C::kCap + 1];
  __shared__ int s_ptr[NW][RW + 1];
  __shared__ double lds[K * NW];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int g = lane / K, c = lane % K;
  Nz *const nz = s_nz[wave];
  int *const ptr = s_ptr[wave];
  constexpr unsigned kRowBytes = FAR ? 1 : K * 8, kNone = 0xffffffffu;
  if (lane == 0) nz[C::kCap] = Nz{0.0, kNone, 0};
  const __amdgpu_buffer_rsrc_t pb = fl_buffer(P, FAR ? 0 : (unsigned)((size_t)n * K * 8));
  // P at a nonzero's row; +0.0 where there is none, which with the value 0
  // leaves a sum as it is (it started at +0.0, so it is never -0.0)
  auto gather = [&](unsigned at) {
    if constexpr (FAR) return at != kNone ? P[(size_t)at * K + c] : 0.0;
    // (no row at kNone: the load's bounds check gives 0)
    const fl_u2 u = __builtin_amdgcn_raw_buffer_load_b64(pb, at | (unsigned)(c * 8), 0, 0);
    return fl_f64(u.x, u.y);
  };
  const int nblk = (n - 1) / (RW * NW) + 1;

  // a chunk's row pointers (lane l: rows l and l + 1), then its entries
  struct Ptr {
    int row0, p0, p1;
  };
  struct Ent {
    int row0, p0, e0, cnt;
    int j[EPL];
    double v[EPL];
  };
  auto ask_ptr = [&](int blk) {
    Ptr p;
    p.row0 = blk < nblk ? (blk * NW + wave) * RW : n;
    p.p0 = p.p1 = 0;
    if (lane < RW) {
      p.p0 = ia[p.row0 + min(lane, n - p.row0)];
      p.p1 = ia[p.row0 + min(lane + 1, n - p.row0)];
    }
    return p;
  };
  auto ask_ent = [&](const Ptr &p) {
    Ent e;
    e.row0 = p.row0;
    e.e0 = __builtin_amdgcn_readfirstlane(p.p0);
    e.cnt = __builtin_amdgcn_readlane(p.p1, RW - 1) - e.e0;
    e.p0 = p.p0 - e.e0;
    if (e.cnt <= C::kCap) {
#pragma unroll
      for (int u = 0; u < EPL; ++u) {
        const int i = u * 64 + lane;
        e.j[u] = i < e.cnt ? ja[e.e0 + i] : 0;
        e.v[u] = i < e.cnt ? a[e.e0 + i] : 0.0;
      }
    }
    return e;
  };
  double acc = 0.0;
  // the rows of a chunk; sum(e0, e1, s): the sums s of the group's rows, row j's
  // nonzeros being e0[j] to e1[j] of the chunk's
  auto rows = [&](int row0, auto sum) {
    for (int base = 0; base < RW && base < n - row0; base += G * RU) {
      int e0[RU], e1[RU];
      double s[RU], own[RU];
#pragma unroll
      for (int j = 0; j < RU; ++j) {
        const int r = base + j * G + g;
        e0[j] = ptr[r];
        e1[j] = ptr[r + 1];
        s[j] = 0.0;
        if (MODE == 1) own[j] = r < n - row0 ? P[(size_t)(row0 + r) * K + c] : 0.0;
      }
      sum(e0, e1, s);
#pragma unroll
      for (int j = 0; j < RU; ++j) {
        const int row = row0 + base + j * G + g;
        if (row < n) {
          const size_t o = (size_t)row * K + c;
          if (MODE == 2) {
            const double r = -(s[j] - Bm[o]);  // r = A x; r += -1*b; r *= -1
            Q[o] = r;
            acc += r * r;
          } else {
            st_nt(Q + o, s[j]);
            if (MODE == 1) acc += own[j] * s[j];
          }
        }
      }
    }
  };
  // entry(e, end): a nonzero, or none from end on; no row has more than most
  auto add = [&](const int(&e0)[RU], const int(&e1)[RU], int most, double(&s)[RU], auto entry) {
    for (int off = 0; off < most; off += EU) {
      bool any = false;
#pragma unroll
      for (int j = 0; j < RU; ++j) any |= e0[j] + off < e1[j];
      if (!any) break;
      double av[RU][EU], v[RU][EU];
      unsigned at[RU][EU];
#pragma unroll
      for (int j = 0; j < RU; ++j)
#pragma unroll
        for (int t = 0; t < EU; ++t) {
          const Nz x = entry(e0[j] + off + t, e1[j]);
          av[j][t] = x.v;
          at[j][t] = x.at;
        }
#pragma unroll
      for (int j = 0; j < RU; ++j)
#pragma unroll
        for (int t = 0; t < EU; ++t) v[j][t] = gather(at[j][t]);
#pragma unroll
      for (int j = 0; j < RU; ++j)
#pragma unroll
        for (int t = 0; t < EU; ++t) s[j] += av[j][t] * v[j][t];
    }
  };
  // a chunk with more nonzeros than its LDS holds: every lane reads its row's
  // entries, EU of each of its rows at a time (the index is
  // clamped: with a return past the row's end the loads wait for each other), or
  // with 1 or 2 groups, whose lanes would all read the same few, the group's
  // lanes read a window of each row together, the next one while this one is
  // added.  us per call at 50,000 rows of 101 entries, k = 8, 32 and 64: 92, 262
  // and 239 entry by entry, 73, 119 and 213 so
  constexpr int WIN = C::kCap / (G * RU), WL = WIN >= K ? WIN / K : 1;
  auto add_far = [&](int eb, const int(&e0)[RU], const int(&e1)[RU], double(&s)[RU]) {
    if constexpr (K < 32) {
      add(e0, e1, INT_MAX, s, [&](int i, int end) {
        const int q = eb + (i < end ? i : 0);
        const double v = a[q];
        const unsigned at = (unsigned)ja[q] * kRowBytes;
        return Nz{i < end ? v : 0.0, i < end ? at : kNone, 0};
      });
    } else {
      int longest = 0;
#pragma unroll
      for (int j = 0; j < RU; ++j) longest = max(longest, e1[j] - e0[j]);
      for (int off = K; off < 64; off <<= 1) longest = max(longest, __shfl_xor(longest, off));
      longest = __builtin_amdgcn_readfirstlane(longest);
      Nz win[RU][WL];
      auto ask = [&](int w) {
#pragma unroll
        for (int j = 0; j < RU; ++j)
#pragma unroll
          for (int u = 0; u < WL; ++u) {
            const int i = e0[j] + w + u * K + c;
            const bool in = i < e1[j];
            const double v = a[eb + (in ? i : 0)];
            const unsigned at = (unsigned)ja[eb + (in ? i : 0)] * kRowBytes;
            win[j][u] = Nz{in ? v : 0.0, in ? at : kNone, 0};
          }
      };
      ask(0);
      for (int w = 0; w < longest; w += WIN) {
        wave_sync();  // (the last window's reads are done)
#pragma unroll
        for (int j = 0; j < RU; ++j)
#pragma unroll
          for (int u = 0; u < WL; ++u) nz[(j * G + g) * WIN + u * K + c] = win[j][u];
        wave_sync();
        ask(w + WIN);
        int w0[RU], w1[RU];
#pragma unroll
        for (int j = 0; j < RU; ++j) {
          w0[j] = (j * G + g) * WIN;
          w1[j] = w0[j] + min(WIN, e1[j] - e0[j] - w);
        }
        add(w0, w1, WIN, s, [&](int i, int end) { return nz[i < end ? i : C::kCap]; });
      }
    }
  };

  const int first = cls_block(blockIdx.x, group), step = (int)gridDim.x;
  Ptr p = ask_ptr(first);
  Ent e = ask_ent(p);
  p = ask_ptr(first + step);
  for (int blk = first; blk < nblk; blk += step) {
    const int row0 = e.row0, cnt = e.cnt, eb = e.e0;
    wave_sync();  // (the last chunk's reads are done)
    if (lane < RW) ptr[lane] = e.p0;
    if (lane == 0) ptr[RW] = cnt;
    if (cnt <= C::kCap) {
#pragma unroll
      for (int u = 0; u < EPL; ++u) {
        nz[u * 64 + lane] = Nz{e.v[u], (unsigned)e.j[u] * kRowBytes, 0};
      }
    }
    wave_sync();
    e = ask_ent(p);
    p = ask_ptr(blk + 2 * step);
    if (cnt <= C::kCap)
      rows(row0, [&](auto &e0, auto &e1, auto &s) {
        add(e0, e1, INT_MAX, s, [&](int i, int end) { return nz[i < end ? i : C::kCap]; });
      });
    else
      rows(row0, [&](auto &e0, auto &e1, auto &s) { add_far(eb, e0, e1, s); });
  }
  if (MODE == 0) return;
  // fixed-order reduction: butterfly over the row groups of a wave, then
  // over the waves of the workgroup
  for (int off = K; off < 64; off <<= 1) acc += __shfl_xor(acc, off);
  if (g == 0) lds[c * NW + wave] = acc;
  __syncthreads();
  for (int cc = threadIdx.x; cc < K; cc += BS) {
    double t = 0.0;
    for (int w = 0; w < NW; ++w) t += lds[cc * NW + w];
    part[(size_t)cc * gridDim.x + blockIdx.x] = t;
  }
}

// --------------------------------------------------- column reductions
// A workgroup per column (blockIdx.x): its partial sums lie together.

// column `j` stops; the last one ends the solve
__device__ __forceinline__ void stop_column(BlkCtl *ctl, int j) {
  ctl->done[j] = 1;
  if (atomicSub(&ctl->left, 1) == 1) ctl->all_done = 1;
}

// start: ||r0||, tolrel and the stop state of the column
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_res0(const double *part, int nparts, double tol,
                                                 BlkCtl *ctl, double *hist) {
  __shared__ double red[BS / kWave];
  const int j = blockIdx.x;
  const double sum = sum_partials<BS>(part + (size_t)j * nparts, nparts, 1, red);
  if (threadIdx.x != 0) return;
  const double r0 = sqrt(sum);
  const bool stop = !isfinite(r0) || r0 == 0.0;  // r0 == 0: x0 solves column j
  ctl->res0[j] = r0;
  ctl->res[j] = r0;
  ctl->tolrel[j] = tol * r0;
  ctl->flag[j] = isfinite(r0) ? 0 : 2;
  if (hist) hist[j] = r0;
  if (stop) stop_column(ctl, j);
}

// W = d_r R; P = W; per-workgroup partials of R.W
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_start(int n, int k, int lk,
                                                  const double *__restrict__ R,
                                                  const double *__restrict__ d_r,
                                                  double *__restrict__ P, double *part) {
  __shared__ double lds[BS];
  const size_t total = (size_t)n * k, stride = (size_t)gridDim.x * BS;
  double acc = 0.0;  // this thread's column is threadIdx.x % k (k | BS)
  for (size_t o = (size_t)blockIdx.x * BS + threadIdx.x; o < total; o += stride) {
    const double ri = R[o];
    const double wi = d_r[o >> lk] * ri;  // line_jacobi: w = d_r .* r
    P[o] = wi;                            // first iteration: p = w
    acc += ri * wi;
  }
  lds[threadIdx.x] = acc;
  __syncthreads();
  for (int col = threadIdx.x; col < k; col += BS) {
    double s = 0.0;
    for (int t = col; t < BS; t += k) s += lds[t];
    part[(size_t)col * gridDim.x + blockIdx.x] = s;
  }
}

// rho_j from the R.W partials
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_rho(const double *part, int nparts, BlkCtl *ctl) {
  __shared__ double red[BS / kWave];
  const int j = blockIdx.x;
  const double sum = sum_partials<BS>(part + (size_t)j * nparts, nparts, 1, red);
  if (threadIdx.x == 0) ctl->rho[j] = sum;
}

// alpha_j = rho_j / (p.q)_j
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_alpha(const double *part, int nparts, BlkCtl *ctl) {
  __shared__ double red[BS / kWave];
  const int j = blockIdx.x;
  if (ctl->done[j]) return;
  const double sum = sum_partials<BS>(part + (size_t)j * nparts, nparts, 1, red);
  if (threadIdx.x == 0) ctl->alpha[j] = ctl->rho[j] / sum;
}

// R -= alpha Q for the live columns; per-workgroup partials of R.W and R.R
// (part[j * gridDim.x + b] and part[(k + j) * gridDim.x + b])
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_update(int n, int k, int lk, double *__restrict__ R,
                                                   const double *__restrict__ Q,
                                                   const double *__restrict__ d_r,
                                                   const BlkCtl *ctl, double *part) {
  if (ctl->all_done) return;
  __shared__ double lds[2 * BS];
  const int col = (int)threadIdx.x & (k - 1);
  const double nalpha = -1.0 * ctl->alpha[col];
  const size_t total = (size_t)n * k, stride = (size_t)gridDim.x * BS;
  double rz = 0.0, rr = 0.0;
  if (!ctl->done[col]) {
    for (size_t o = (size_t)blockIdx.x * BS + threadIdx.x; o < total; o += stride) {
      // R and Q streamed once: non-temporal (d_r, shared by a row's k
      // columns, stays cached)
      const double ri = ld_nt(R + o) + nalpha * ld_nt(Q + o);  // r += -alpha*q
      st_nt(R + o, ri);
      rz += ri * (d_r[o >> lk] * ri);
      rr += ri * ri;
    }
  }
  lds[threadIdx.x] = rz;
  lds[BS + threadIdx.x] = rr;
  __syncthreads();
  for (int cc = threadIdx.x; cc < k; cc += BS) {
    double s1 = 0.0, s2 = 0.0;
    for (int t = cc; t < BS; t += k) {
      s1 += lds[t];
      s2 += lds[BS + t];
    }
    part[(size_t)cc * gridDim.x + blockIdx.x] = s1;
    part[(size_t)(k + cc) * gridDim.x + blockIdx.x] = s2;
  }
}

// convergence test of the column (cg.c:106-123) and beta; hist[it*k + j]
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_conv(const double *part, int nparts, double *hist,
                                                 BlkCtl *ctl) {
  __shared__ double red[BS / kWave];
  const int j = blockIdx.x, k = gridDim.x;
  if (ctl->done[j]) {  // its x has had its last update
    if (threadIdx.x == 0) ctl->xup[j] = 0;
    return;
  }
  const double rz = sum_partials<BS>(part + (size_t)j * nparts, nparts, 1, red);
  const double rr = sum_partials<BS>(part + (size_t)(k + j) * nparts, nparts, 1, red);
  if (threadIdx.x != 0) return;
  const int it = ctl->iters[j] + 1;
  const double res = sqrt(rr);
  ctl->xup[j] = 1;
  ctl->res[j] = res;
  ctl->iters[j] = it;
  if (hist) hist[(size_t)it * k + j] = res;
  int flag = -1;
  if (!isfinite(res))
    flag = 2;
  else if (res < ctl->tolrel[j])
    flag = 0;
  else if (it > ctl->maxit)
    flag = 1;
  if (flag >= 0) {
    ctl->flag[j] = flag;
    stop_column(ctl, j);
  } else {
    ctl->beta[j] = rz / ctl->rho[j];
    ctl->rho[j] = rz;
  }
}

// X += alpha P (columns live in this iteration); P = beta P + d_r R
// (columns still live).  Four elements' loads in flight per thread: 177 us for
// 1.13 GB at 96^3, k = 32 (one: 208).
constexpr int kVU = 4;
template <int BS>
__global__ __launch_bounds__(BS) void k_blk_dir(int n, int k, int lk, double *__restrict__ X,
                                                const double *__restrict__ R,
                                                const double *__restrict__ d_r,
                                                double *__restrict__ P, const BlkCtl *ctl) {
  const int col = (int)threadIdx.x & (k - 1);
  const bool xup = ctl->xup[col], live = !ctl->done[col];
  if (!xup && !live) return;
  const double alpha = ctl->alpha[col], beta = ctl->beta[col];
  const size_t total = (size_t)n * k, stride = (size_t)gridDim.x * BS;
  for (size_t o0 = (size_t)blockIdx.x * BS + threadIdx.x; o0 < total; o0 += kVU * stride) {
    double p[kVU], x[kVU], r[kVU], d[kVU];
#pragma unroll
    for (int u = 0; u < kVU; ++u) {
      const size_t o = o0 + u * stride;
      if (o >= total) continue;
      p[u] = ld_nt(P + o);
      x[u] = xup ? ld_nt(X + o) : 0.0;
      r[u] = live ? ld_nt(R + o) : 0.0;
      d[u] = live ? d_r[o >> lk] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kVU; ++u) {
      const size_t o = o0 + u * stride;
      if (o >= total) continue;
      if (xup) st_nt(X + o, x[u] + alpha * p[u]);             // x += alpha*p
      if (live) st_nt(P + o, p[u] * beta + d[u] * r[u]);  // p = beta p + w
    }
  }
}

// col - row of the first kSampleLen entries of row t n / kBlock, kNoEntry past its end
constexpr int kSampleLen = 32, kNoEntry = INT_MIN;
__global__ __launch_bounds__(kBlock) void k_spmm_sample(int n, const int *__restrict__ ia,
                                                        const int *__restrict__ ja,
                                                        int *__restrict__ out) {
  const int t = threadIdx.x, row = (int)((long long)t * n / kBlock);
  const int e0 = ia[row], len = ia[row + 1] - e0;
  for (int j = 0; j < kSampleLen; ++j)
    out[t * kSampleLen + j] = j < len ? ja[e0 + j] - row : kNoEntry;
}

// The workgroups of an SpMM and how they are dealt to the XCDs (cls_block).
struct SpmmShape {
  unsigned grid;
  int group;
  bool one;
};

using SpmmFn = void (*)(SpmmShape, int, const int *, const int *, const double *, const double *,
                        double *, const double *, double *, const BlkCtl *, int);

template <int K, int RU0, bool ONE>
void spmm_launch(SpmmShape g, int n, const int *ia, const int *ja, const double *a,
                 const double *P, double *Q, const double *Bm, double *part, const BlkCtl *ctl,
                 int mode) {
  constexpr int kMost = Chunk<K, ONE>::kRW / Chunk<K, ONE>::G;  // rows per group in a chunk
  constexpr int RU = RU0 < kMost ? RU0 : kMost, EU = ONE ? 16 : RU == 4 ? 4 : 8;
  auto pick = [&](auto far) {
    constexpr bool F = decltype(far)::value;
    return mode == 2   ? k_spmm<kBlock, K, RU, EU, 2, F, ONE>
           : mode == 1 ? k_spmm<kBlock, K, RU, EU, 1, F, ONE>
                       : k_spmm<kBlock, K, RU, EU, 0, F, ONE>;
  };
  const bool far = (size_t)n * K * 8 > 0xfffffff0u;
  auto *f = far ? pick(std::true_type{}) : pick(std::false_type{});
  f<<<g.grid, kBlock, 0, stream()>>>(n, ia, ja, a, P, Q, Bm, part, ctl, g.group);
}

template <int K>
SpmmFn spmm_for_k(int ru, bool one) {
  if constexpr (K >= kOneK)
    if (one) return spmm_launch<K, 1, true>;
  switch (ru) {
    case 1: return spmm_launch<K, 1, false>;
    case 2: return spmm_launch<K, 2, false>;
    default: return spmm_launch<K, 4, false>;
  }
}

SpmmFn spmm_for(int k, int ru, bool one) {
  switch (k) {
    case 1: return spmm_for_k<1>(ru, one);
    case 2: return spmm_for_k<2>(ru, one);
    case 4: return spmm_for_k<4>(ru, one);
    case 8: return spmm_for_k<8>(ru, one);
    case 16: return spmm_for_k<16>(ru, one);
    case 32: return spmm_for_k<32>(ru, one);
    case 64: return spmm_for_k<64>(ru, one);
    default: return nullptr;
  }
}

// 1, 2, 4: rows per lane group at a time; 8, 16 (k = 64) as 4
bool tile_ok(int k, int ru) {
  return ru == 1 || ru == 2 || ru == 4 || (k == 64 && (ru == 8 || ru == 16));
}

int log2i(int k) {
  int l = 0;
  while ((1 << l) < k) ++l;
  return l;
}

// (ia, ja, a, n, k, mode) -> chosen tile
std::map<std::tuple<const void *, const void *, const void *, int, int, int>, int> g_tile;

// spmm_wg_per_cu workgroups per CU, dealt to the XCDs by a sample of the column
// offsets, taken once per plan (a matrix without locality has no better group
// than 1, nor has one of too few row blocks for two).
SpmmShape spmm_shape(const SpmvPlan &A, const int *ia, const int *ja, int k) {
  const int per_cu = std::max(1, std::min(16, options().spmm_wg_per_cu));
  const int grid = std::max(8, per_cu * device_cus());
  const bool one = k >= kOneK && (A.n <= kOneRows || A.max_row > kOneLong);
  const int rows = (one ? 64 / k : std::max(64 / k, 16)) * (kBlock / kWave);
  const long nblk = ((long)A.n + rows - 1) / rows;
  const auto known = A.spmm_shapes.find({rows, grid});
  if (known != A.spmm_shapes.end()) return {known->second.first, known->second.second, one};
  std::vector<int> offsets;
  if (nblk >= 2 * 64) {
    const DevBufPtr d = dev_try(sizeof(int) * kBlock * kSampleLen);
    if (!d) return {(unsigned)grid, 1, one};
    k_spmm_sample<<<1, kBlock, 0, stream()>>>(A.n, ia, ja, d->as<int>());
    for (int o : dev_download(d->as<int>(), (size_t)kBlock * kSampleLen))
      if (o != kNoEntry) offsets.push_back(o);
  }
  const auto best = xcd_grid(offsets, rows, nblk, grid);
  A.spmm_shapes[{rows, grid}] = best;
  return {best.first, best.second, one};
}

unsigned vec_grid(size_t elems) {
  return (unsigned)std::max<size_t>(
      1, std::min<size_t>(1024, (elems + 4 * kBlock - 1) / (4 * kBlock)));
}

// Times every rows-per-group choice on Y = A X (three runs each, after a
// warm-up).
int pick_tile(SpmmShape g, int n, const int *ia, const int *ja, const double *a, int k,
              const double *X, double *Y, int mode = 0, double *part = nullptr, const BlkCtl *ctl = nullptr) {
  auto key = std::make_tuple((const void *)ia, (const void *)ja, (const void *)a, n, k, mode);
  if (g.one) return 1;  // (the tile says nothing)
  auto it = g_tile.find(key);
  if (it != g_tile.end()) return it->second;
  int best_ru = 0;
  float best = 1e30f;
  hipEvent_t e0, e1;
  if (!LAP_HIP(hipEventCreate(&e0))) return 0;
  if (!LAP_HIP(hipEventCreate(&e1))) {
    (void)hipEventDestroy(e0);
    return 0;
  }
  for (int ru = 1; ru <= 4; ru *= 2) {
    SpmmFn fn = spmm_for(k, ru, g.one);
    fn(g, n, ia, ja, a, X, Y, nullptr, part, ctl, mode);
    LAP_HIP(hipEventRecord(e0, stream()));
    for (int r = 0; r < 3; ++r) fn(g, n, ia, ja, a, X, Y, nullptr, part, ctl, mode);
    LAP_HIP(hipEventRecord(e1, stream()));
    LAP_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    LAP_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (ms < best) {
      best = ms;
      best_ru = ru;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (best_ru) g_tile[key] = best_ru;
  return best_ru;
}

bool block_args(const char *fn, int n, int nnz, const int *ia, const int *ja, const double *a,
                int k, int tile) {
  if (n <= 0 || nnz < 0 || k <= 0 || k > kMaxK || (k & (k - 1))) {
    set_error(LAP_ERR_ARG,
              "%s: need n > 0, nnz >= 0 and k a power of two in [1, %d] (n=%d k=%d)", fn,
              kMaxK, n, k);
    return false;
  }
  if (tile && !tile_ok(k, tile)) {
    set_error(LAP_ERR_ARG, "%s: tile must be 1, 2 or 4 (or 8, 16 with k = 64), not %d", fn, tile);
    return false;
  }
  return check_device(fn, {{ia, "ia", sizeof(int) * ((size_t)n + 1)},
                           {ja, "ja", sizeof(int) * (size_t)nnz},
                           {a, "a", sizeof(double) * (size_t)nnz}});
}

}  // namespace

void release_block_plans() { g_tile.clear(); }
void forget_block_plans(const void *p) {
  for (auto it = g_tile.begin(); it != g_tile.end();) {
    if (std::get<0>(it->first) == p || std::get<1>(it->first) == p ||
        std::get<2>(it->first) == p)
      it = g_tile.erase(it);
    else
      ++it;
  }
}

}  // namespace lap

using namespace lap;

extern "C" int lap_csr_matmat(int n, int nnz, const int *ia, const int *ja, const double *a, int k,
                              const double *X, double *Y, int tile) {
  if (!block_args("csr_matmat", n, nnz, ia, ja, a, k, tile)) return lap_last_status();
  const size_t nk = sizeof(double) * (size_t)n * (size_t)k;
  if (!check_device("csr_matmat", {{X, "X", nk}, {Y, "Y", nk}})) return lap_last_status();
  const SpmvPlan *A = spmv_plan(n, nnz, ia, ja);  // validates ia / ja
  if (!A) return lap_last_status();
  const SpmmShape g = spmm_shape(*A, ia, ja, k);
  if (!tile) tile = pick_tile(g, n, ia, ja, a, k, X, Y);
  if (!tile) return LAP_ERR_HIP;
  spmm_for(k, tile, g.one)(g, n, ia, ja, a, X, Y, nullptr, nullptr, nullptr, 0);
  if (!LAP_HIP(hipGetLastError())) return LAP_ERR_HIP;
  sync();
  return LAP_OK;
}

extern "C" int lap_pcg_block(int n, int nnz, const int *ia, const int *ja, const double *a,
                             const double *d_r, int k, double *X, const double *Bm, double tol,
                             int maxit, int tile, double *h_hist, int *iters, int *flags,
                             double *res0, double *res, double *gpu_ms) {
  if (!block_args("pcg_block", n, nnz, ia, ja, a, k, tile)) return lap_last_status();
  if (maxit < 0) {
    set_error(LAP_ERR_ARG, "pcg_block: maxit %d < 0", maxit);
    return LAP_ERR_ARG;
  }
  const size_t nk = sizeof(double) * (size_t)n * (size_t)k;
  if (!check_device("pcg_block", {{d_r, "d_r", sizeof(double) * (size_t)n},
                                  {X, "X", nk},
                                  {Bm, "B", nk}}))
    return lap_last_status();
  const SpmvPlan *A = spmv_plan(n, nnz, ia, ja);  // validates ia / ja
  if (!A) return lap_last_status();
  double *R = scratch_vec("blk_r", (size_t)n * k), *P = scratch_vec("blk_p", (size_t)n * k),
         *Q = scratch_vec("blk_q", (size_t)n * k);
  BlkCtl *ctl =
      reinterpret_cast<BlkCtl *>(scratch_vec("blk_ctl", sizeof(BlkCtl) / sizeof(double) + 1));
  const SpmmShape g = spmm_shape(*A, ia, ja, k);
  const unsigned gv = vec_grid((size_t)n * k);
  double *part = scratch_vec("blk_part", (size_t)2 * kMaxK * std::max(g.grid, gv));
  const size_t hist_len = ((size_t)maxit + 2) * (size_t)k;
  if (h_hist && hist_len > (size_t)INT_MAX) {
    set_error(LAP_ERR_ARG, "pcg_block: history of (maxit+2)*k entries is too long");
    return LAP_ERR_ARG;
  }
  double *hist = h_hist ? scratch_vec("blk_hist", hist_len) : nullptr;
  if (!R || !P || !Q || !ctl || !part || (h_hist && !hist)) return lap_last_status();
  // rows past a column's own stop stay 0
  if (hist) launch_fill((int)hist_len, 0.0, hist);
  BlkCtl h{};
  h.maxit = maxit;
  h.left = k;
  LAP_HIP(hipMemcpyAsync(ctl, &h, sizeof h, hipMemcpyHostToDevice, stream()));
  // timed in the solve's own mode (q = A p with the p.q epilogue)
  if (!tile) tile = pick_tile(g, n, ia, ja, a, k, Bm, Q, 1, part, ctl);
  if (!tile) return LAP_ERR_HIP;
  SpmmFn spmm = spmm_for(k, tile, g.one);
  const int lk = log2i(k);

  hipEvent_t ev0, ev1;
  if (!LAP_HIP(hipEventCreate(&ev0))) return LAP_ERR_HIP;
  if (!LAP_HIP(hipEventCreate(&ev1))) {
    (void)hipEventDestroy(ev0);
    return LAP_ERR_HIP;
  }
  LAP_HIP(hipEventRecord(ev0, stream()));
  spmm(g, n, ia, ja, a, X, R, Bm, part, ctl, 2);
  k_blk_res0<kBlock><<<k, kBlock, 0, stream()>>>(part, (int)g.grid, tol, ctl, hist);
  k_blk_start<kBlock><<<gv, kBlock, 0, stream()>>>(n, k, lk, R, d_r, P, part);
  k_blk_rho<kBlock><<<k, kBlock, 0, stream()>>>(part, (int)gv, ctl);
  auto iteration = [&]() {
    spmm(g, n, ia, ja, a, P, Q, nullptr, part, ctl, 1);
    k_blk_alpha<kBlock><<<k, kBlock, 0, stream()>>>(part, (int)g.grid, ctl);
    k_blk_update<kBlock><<<gv, kBlock, 0, stream()>>>(n, k, lk, R, Q, d_r, ctl, part);
    k_blk_conv<kBlock><<<k, kBlock, 0, stream()>>>(part, (int)gv, hist, ctl);
    k_blk_dir<kBlock><<<gv, kBlock, 0, stream()>>>(n, k, lk, X, R, d_r, P, ctl);
  };
  // iter <= maxit + 1 for every column, so G * max_batches iterations
  // always reach all_done
  const int G = std::max(1, (int)std::min<long>(options().graph_iters, (long)maxit + 2));
  const long max_batches = ((long)maxit + 1) / G + 3;
  int status = LAP_OK;
  hipGraphExec_t gexec = nullptr;
  if (options().use_graph) {
    hipGraph_t graph = nullptr;
    bool ok = LAP_HIP(hipStreamBeginCapture(stream(), hipStreamCaptureModeThreadLocal));
    if (ok) {
      for (int s = 0; s < G; ++s) iteration();
      ok = LAP_HIP(hipStreamEndCapture(stream(), &graph));
    }
    if (ok) ok = LAP_HIP(hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0));
    if (graph) (void)hipGraphDestroy(graph);
    if (!ok) status = LAP_ERR_HIP;
  }
  int *flag_h = pinned_flags();
  if (!flag_h) status = LAP_ERR_HIP;
  if (status == LAP_OK) {
    bool finished = false;
    for (long b = 0; b < max_batches && !finished; ++b) {
      if (gexec) {
        if (!LAP_HIP(hipGraphLaunch(gexec, stream()))) break;
      } else {
        for (int s = 0; s < G; ++s) iteration();
      }
      LAP_HIP(hipMemcpyAsync(flag_h, &ctl->all_done, sizeof(int), hipMemcpyDeviceToHost,
                             stream()));
      sync();
      finished = flag_h[0] != 0;
    }
    if (!finished) {
      set_error(LAP_ERR_NUMERIC, "pcg_block: stop flags never set");
      status = LAP_ERR_NUMERIC;
    }
  }
  LAP_HIP(hipEventRecord(ev1, stream()));
  sync();
  float ms = 0.f;
  LAP_HIP(hipEventElapsedTime(&ms, ev0, ev1));
  (void)hipEventDestroy(ev0);
  (void)hipEventDestroy(ev1);
  if (gexec) (void)hipGraphExecDestroy(gexec);
  if (gpu_ms) *gpu_ms = ms;
  LAP_HIP(hipMemcpy(&h, ctl, sizeof h, hipMemcpyDeviceToHost));
  int last = 0;
  for (int j = 0; j < k; ++j) {
    last = std::max(last, h.iters[j]);
    if (iters) iters[j] = h.iters[j];
    if (flags) flags[j] = h.flag[j];
    if (res0) res0[j] = h.res0[j];
    if (res) res[j] = h.res[j];
  }
  if (h_hist && hist)
    LAP_HIP(hipMemcpy(h_hist, hist, sizeof(double) * ((size_t)last + 1) * k,
                      hipMemcpyDeviceToHost));
  if (status == LAP_OK && lap_last_status() == LAP_ERR_HIP) status = LAP_ERR_HIP;
  return status;
}
