// resident.hip -- Jacobi PCG of small and medium systems as one launch, the
// whole system on the chip.
//
// Why: three launches per iteration cost 12 us whatever the system's size
// (n = 16,384: 13.5 us per iteration for 0.7 MB of traffic), and a system of
// up to a few hundred thousand rows fits the registers and LDS of the 256
// CUs: 2^17 rows of 11 entries are 15 MB of matrix against 128 MiB of
// registers.
//
// How: a workgroup of 1024 (or 512) threads owns a contiguous range of rows, R per
// thread, for the whole solve.  A thread keeps its rows' values, column slots,
// x, r, p and 1/diag in registers; the LDS holds the p of the workgroup's rows
// and of the other rows they refer to (its halo).  What crosses between
// workgroups per iteration:
//   1. p.q, one partial sum per workgroup, read by all of them;
//   2. r.w and r.r likewise, and w = d_r r of the rows others refer to: the
//      owner of a halo entry keeps p = beta p + w itself, from the same
//      operands, so p is never sent.
// They travel as tagged words (boxed.hpp), two trips through memory per
// iteration and no barrier between workgroups.  A place is written again only
// after every reader has taken the value it held: the writer is then past a
// sum to which each reader contributed after reading.
//
// Arithmetic: the recurrence of k_jac_update_nx / k_jac_px (pcg.hip), each row
// summed in CSR order and each vector entry updated by the same operations;
// the three dot products are summed in another fixed order (rows of a thread,
// lanes of a wave, waves, workgroups).
//
// Several systems (lap_pcg_batched's lockstep mode) run in one launch, each by a
// team of consecutive workgroups of its own, the largest first: as teams end,
// the next ones take their CUs.  A team waits for its own workgroups only, and
// workgroups start in order, so the first team still running always has all of
// its workgroups.  A team is at most one workgroup per CU.
//
// Nothing keeps other work off the GPU: another process' or stream's kernel can
// hold CUs that a team's last workgroups wait for, and two one-launch solves of
// two processes can each hold what the other waits for.  So waits are bounded
// (option resident_polls); one that runs out ends every workgroup, x is put back
// and the solve goes by launches, which need no two workgroups at once.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "boxed.hpp"
#include "lap_core.hpp"

namespace lap {

namespace {

constexpr int kResThreads = 1024;
constexpr int kResHalo = 8192;     // halo entries of a workgroup at most
constexpr int kResMaxWg = 256;     // workgroups at most (partials: one per thread of 4 waves)
// Rows per workgroup at least: fewer workgroups have fewer partial sums to
// exchange, until the LDS reads of a thread's rows take longer than that
// saves.  us per iteration with 512 / 1024 / 2048 rows: 128^2 4.66 / 4.44 /
// 3.89, 512^2 9.05 / 9.08 / 6.86, 40^3 7.15 / 6.66 / 6.70, 64^3 9.4 / 9.4 /
// 11.1, 97 x 90 x 31 8.7 / 8.7 / 10.6: 2048 for rows of up to 5 entries.
constexpr int kResRows = 1024, kResRowsShort = 2048, kResShort = 5;
// Rows of a system at most (the analysis' bitmap in LDS); of more than 8 entries,
// which have a row per thread, 2^18 (256 workgroups of 1024).
constexpr int kResMaxN = 1 << 19;
constexpr int kResMaxRows = 1 << 26;  // rows of all systems at most (box_w stays below 2^31 bytes)
// Workgroups of a batch at most (their halo lists take up to 32 KB each: 1 GB).
constexpr int kResMaxWgs = 1 << 15;
// Iterations of a system per launch.  A team that has only some of its workgroups
// running waits for the CUs of systems ahead of it, and that wait counts against
// resident_polls too: a launch of 8192 iterations holds a CU for at most 0.13 s
// (15.7 us per iteration at 64 x 64 x 128), whatever maxit is, where a wait runs
// out after 1 to 2 s (2^23 looks).
constexpr int kResIters = 8192;
// Every workgroup of a team reads every sum, through whichever XCD it is on and
// past the caches: with many workgroups the few lines that hold the boxes are
// what they wait for.  So a sum is sent in 8 copies and an XCD reads its own: us
// per iteration with 1 and 8 copies, 128^2 (8 workgroups) 4.1 and 4.1, 256^2 5.2
// and 4.4, 512^2 7.1 and 5.6, 40^3 6.6 and 5.7, 64^3 9.1 and 8.5, 97 x 90 x 31 8.2
// and 7.5, a geometric graph of 150k nodes 8.2 and 7.4; the batch of 160 grids
// 5.6 and 5.0 ms.
constexpr int kResCopies = 8;
constexpr int kResSkew = 256;  // places between the copies

struct ResState {
  double rho, tolrel, res0, res;
  int iter, flag;  // flag: -1 not finished
};
enum { kResWait = 1, kResStale = 2 };
struct ResShared {
  int error;     // kResWait: a wait ran out; kResStale: the plan is of other columns
  unsigned tag;  // highest tag used
  // (both stay from solve to solve; cleared with the boxes after an error)
};
// A workgroup: its first row and row count, its team's first workgroup and
// workgroup count, its system and that system's rows.
struct ResWg {
  int base, rows, team, size, sys, s0, s1, pad;
};

struct ResArgs {
  int nhmax;
  const ResWg *wg;
  const int *ia;
  const double *a;
  const unsigned short *lcol;
  const int *hcnt, *hcol;
  const unsigned char *sent;
  const double *d_r, *b;
  double *x, *r, *p;
  double tol;
  int maxit, resume, iters;
  unsigned tag0, polls;
  double *hist;  // of a single system (may be null)
  void *box_a, *box_b, *box_w;
  int n, stride;  // stride: places from a copy of the sums' boxes to the next
  ResState *st;  // per system
  ResShared *sh;
};

// Sum over the wave's first 16 (W16) or all 64 lanes, valid in the last of
// them; fixed order.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + fl_f64((unsigned)lo, (unsigned)hi);
}
__device__ __forceinline__ double row_sum_dpp(double v) {  // lane 15 of each row of 16
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  return dpp_add<0x118, 0xf>(v);
}
__device__ __forceinline__ double wave_sum_dpp(double v) {  // lane 63
  v = row_sum_dpp(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  return dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const long long b = __double_as_longlong(v);
  return fl_f64((unsigned)__builtin_amdgcn_readlane((int)b, l),
                (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l));
}

// The launch.  R rows per thread, rows of at most L entries, T threads.  512
// threads add up as 1024 do, each what two of those would (the even and the odd
// rows of its R), so x does not depend on T: two such workgroups share a CU and
// one's waits are the other's time, but one by itself has its rows' work on half
// the lanes.
template <int R, int L, int T>
__global__ __launch_bounds__(T, 4) void k_resident(ResArgs g) {
  constexpr int V = kResThreads / T, W = T / kWave, C = L % 4 ? L : 4;  // waves; entries in flight
  extern __shared__ double ps[];  // own rows, halo, a zero; the halo's rows
  __shared__ double red[2][V * W], tot[2][4], one[2];
  __shared__ int dead;
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int w = blockIdx.x;
  const ResWg wg = g.wg[w];
  const int base = wg.base, rows = wg.rows, team = wg.team, size = wg.size;
  ResState *const st = g.st + wg.sys;
  if (g.resume && st->flag >= 0) return;  // its system has ended (the whole team's)
  const int nh = g.hcnt[w];
  double *const halo = ps + R * T;
  const int zero = R * T + g.nhmax;
  int *const hcol = reinterpret_cast<int *>(ps + zero + 1);  // the halo's rows
  const __amdgpu_buffer_rsrc_t box_a = fl_buffer(g.box_a, kResCopies * g.stride * 16);
  const __amdgpu_buffer_rsrc_t box_b = fl_buffer(g.box_b, kResCopies * g.stride * 32);
  // the team's boxes in the copy that this workgroup reads
  const size_t at = (size_t)((w & (kResCopies - 1)) * g.stride + team) * 16;
  const __amdgpu_buffer_rsrc_t mine_a = fl_buffer(static_cast<char *>(g.box_a) + at, size * 16);
  const __amdgpu_buffer_rsrc_t mine_b = fl_buffer(static_cast<char *>(g.box_b) + 2 * at, size * 32);
  const __amdgpu_buffer_rsrc_t box_w = fl_buffer(g.box_w, g.n * 16);
  if (t == 0) {
    dead = g.sh->error;  // (k_res_prep's, or a wait's that ran out already)
    ps[zero] = 0.0;
  }
  for (int h = t; h < nh; h += T) hcol[h] = g.hcol[(size_t)w * g.nhmax + h];
  __syncthreads();
  if (dead) return;  // (it changes behind the next barrier only)
  // the thread's rows
  double val[R][L], x[R], r[R], p[R], d[R];
  unsigned slot[R][(L + 1) / 2];
  bool have[R], sent[R];
  int longest[R];  // of the wave's rows
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int l = t + k * T, row = base + l;
    have[k] = l < rows;
    const int e0 = have[k] ? g.ia[row] : 0, len = have[k] ? g.ia[row + 1] - e0 : 0;
#pragma unroll
    for (int j = 0; j < L; ++j) {
      val[k][j] = j < len ? g.a[e0 + j] : 0.0;
      const unsigned s = j < len ? g.lcol[e0 + j] : (unsigned)zero;
      if (j & 1)
        slot[k][j / 2] |= s << 16;
      else
        slot[k][j / 2] = s;
    }
    d[k] = have[k] ? g.d_r[row] : 0.0;
    x[k] = have[k] ? g.x[row] : 0.0;
    r[k] = p[k] = 0.0;
    sent[k] = have[k] && g.sent[row];
    int m = len;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    longest[k] = __builtin_amdgcn_readfirstlane(m);
  }
  auto row_sums = [&](double(&s)[R]) {  // CSR order; padding adds 0 * 0
#pragma unroll
    for (int k = 0; k < R; ++k) {
      s[k] = 0.0;
#pragma unroll
      for (int j = 0; j < L; j += C) {
        if (j >= longest[k]) break;
        double v[C];
#pragma unroll
        for (int i = 0; i < C; ++i)
          v[i] = ps[(i & 1) ? slot[k][(j + i) / 2] >> 16 : slot[k][(j + i) / 2] & 0xffffu];
#pragma unroll
        for (int i = 0; i < C; ++i) s[k] += val[k][j + i] * v[i];
      }
    }
  };
  // One wait of this wave (every lane that still misses something): false
  // once it has to be given up.
  auto again = [&](unsigned &spins) {
    if (++spins > g.polls ||
        ((spins & 63u) == 0 && __hip_atomic_load(&g.sh->error, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))) {
      if (lane == 0) {
        dead = 1;
        __hip_atomic_fetch_max(&g.sh->error, (int)kResWait, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
      }
      return false;
    }
    return true;
  };
  // Sums of v over the team (N = 1: box_a, 2: box_b), to every thread;
  // `between` runs while they are on their way.
  auto all_sums = [&](auto &sum, auto &v, unsigned tag, auto &&between) {
    constexpr int N = sizeof(sum) / sizeof(sum[0]);
    const __amdgpu_buffer_rsrc_t box = N == 1 ? box_a : box_b;
    const __amdgpu_buffer_rsrc_t mine = N == 1 ? mine_a : mine_b;
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const double s = wave_sum_dpp(v[j][i]);
        if (lane == kWave - 1) red[i][j * W + wave] = s;
      }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double s = row_sum_dpp(lane < V * W ? red[i][lane] : 0.0);
        const double u = readlane_f64(s, V * W - 1);
        if (size == 1)
          one[i] = u;
        else if (lane < kResCopies)
          fl_put(box, (lane * g.stride + w) * N + i, tag, u);
      }
    }
    between();
    if (wave < 4 && size > 1) {
      double got[N];
      if (wave * kWave < size) {
        FlBoxed<double> f[N];
        unsigned spins = 0;
        for (;;) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < N; ++i) f[i].load(mine, t * N + i);
#pragma unroll
          for (int i = 0; i < N; ++i) ok = ok && f[i].is(tag);
          fl_fence();
          if (__builtin_amdgcn_ballot_w64(!ok && t < size) == 0) break;
          if (!again(spins)) break;
        }
#pragma unroll
        for (int i = 0; i < N; ++i) got[i] = t < size ? f[i].value() : 0.0;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) got[i] = 0.0;
      }
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double s = wave_sum_dpp(got[i]);
        if (lane == kWave - 1) tot[i][wave] = s;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i)
      sum[i] = size > 1 ? ((tot[i][0] + tot[i][1]) + tot[i][2]) + tot[i][3] : one[i];
  };
  // halo entries: p = w (first) or beta p + w, w as its owner sent it.  The
  // first entry of each thread is asked for ahead (halo_ask).
  FlBoxed<double> ahead;
  auto halo_ask = [&] { ahead.load(box_w, t < nh ? hcol[t] : 0); };
  auto halo_update = [&](unsigned tag, bool first, double beta) {
    for (int h0 = wave * kWave; h0 < nh; h0 += T) {
      const int h = h0 + lane;
      const int c = h < nh ? hcol[h] : 0;
      FlBoxed<double> f;
      if (h0 < T)
        f = ahead;
      else
        f.load(box_w, c);
      unsigned spins = 0;
      while (__builtin_amdgcn_ballot_w64(h < nh && !f.is(tag)) != 0) {
        if (!again(spins)) break;
        f.load(box_w, c);
        fl_fence();
      }
      if (h < nh) halo[h] = first ? f.value() : halo[h] * beta + f.value();
    }
  };
  auto own_update = [&]() {
#pragma unroll
    for (int k = 0; k < R; ++k) ps[t + k * T] = p[k];
  };
  auto nothing = [] {};

  double rho, tolrel, res0, res;
  int it, flag = -1;
  unsigned tag = g.tag0;
  if (g.resume) {
    rho = st->rho;
    tolrel = st->tolrel;
    res0 = st->res0;
    res = st->res;
    it = st->iter;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int row = base + t + k * T;
      r[k] = have[k] ? g.r[row] : 0.0;
      p[k] = have[k] ? g.p[row] : 0.0;
    }
    for (int h = t; h < nh; h += T) halo[h] = g.p[hcol[h]];
    own_update();
    __syncthreads();
  } else {
    // r = -(A x - b) (cg.c:48-55), w = d_r r, p = w
#pragma unroll
    for (int k = 0; k < R; ++k) ps[t + k * T] = x[k];
    for (int h = t; h < nh; h += T) halo[h] = g.x[hcol[h]];
    __syncthreads();
    double s[R], v[V][2] = {}, sum[2];
    row_sums(s);
    ++tag;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int row = base + t + k * T;
      r[k] = have[k] ? -(s[k] - g.b[row]) : 0.0;
      p[k] = d[k] * r[k];
      if (sent[k]) fl_put(box_w, row, tag, p[k]);
      v[k % V][0] += r[k] * p[k];
      v[k % V][1] += r[k] * r[k];
    }
    all_sums(sum, v, tag, halo_ask);
    rho = sum[0];
    res0 = res = sqrt(sum[1]);
    tolrel = g.tol * res0;
    it = 0;
    if (g.hist && w == 0 && t == 0) g.hist[0] = res0;
    if (!isfinite(res0)) flag = 2;
    if (res0 == 0.0) flag = 0;  // x0 solves the system
    flag = __builtin_amdgcn_readfirstlane(flag);
    if (flag < 0) {
      own_update();
      halo_update(tag, true, 0.0);
    }
    __syncthreads();
  }
  const long long stop = (long long)it + g.iters;
  while (flag < 0 && it < stop && !__builtin_amdgcn_readfirstlane(dead)) {
    ++it;
    // q = A p, p.q, alpha
    double q[R], v1[V][1] = {}, pq[1];
    row_sums(q);
#pragma unroll
    for (int k = 0; k < R; ++k) v1[k % V][0] += p[k] * q[k];
    all_sums(pq, v1, ++tag, nothing);
    const double alpha = rho / pq[0], nalpha = -1.0 * alpha;
    // r -= alpha q, w = d_r r, r.w, r.r; x += alpha p on the way
    double v[V][2] = {}, sum[2];
    ++tag;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      r[k] = r[k] + nalpha * q[k];
      const double wk = d[k] * r[k];
      if (sent[k]) fl_put(box_w, base + t + k * T, tag, wk);
      v[k % V][0] += r[k] * wk;
      v[k % V][1] += r[k] * r[k];
    }
    all_sums(sum, v, tag, [&] {
#pragma unroll
      for (int k = 0; k < R; ++k) x[k] += alpha * p[k];
      halo_ask();
    });
    // convergence test (cg.c:106-123) and beta
    res = sqrt(sum[1]);
    if (g.hist && w == 0 && t == 0) g.hist[it] = res;
    if (!isfinite(res)) flag = 2;
    else if (res < tolrel) flag = 0;
    else if (it > g.maxit) flag = 1;
    flag = __builtin_amdgcn_readfirstlane(flag);
    if (flag >= 0) break;
    const double beta = sum[0] / rho;
    rho = sum[0];
#pragma unroll
    for (int k = 0; k < R; ++k) p[k] = p[k] * beta + d[k] * r[k];
    own_update();
    halo_update(tag, false, beta);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int row = base + t + k * T;
    if (!have[k]) continue;
    g.x[row] = x[k];
    if (flag < 0) {
      g.r[row] = r[k];
      g.p[row] = p[k];
    }
  }
  if (w == team && t == 0) {
    *st = ResState{rho, tolrel, res0, res, it, flag};
    atomicMax(&g.sh->tag, tag);
  }
}

// Before a solve: keeps x in x0 for one that ends in an error, clears the systems'
// states, and compares every nonzero's slot with ja, from whose columns it was
// made at the first solve: where ja has been rewritten since, the solve does not
// begin (kResStale) and the host makes a new plan.  A workgroup per one of the
// solve's; longest: entries of a row that the solve has room for.
__global__ __launch_bounds__(kResThreads) void k_res_prep(
    const ResWg *__restrict__ wgs, int own, int longest, int nhmax, const int *__restrict__ ia,
    const int *__restrict__ ja, const unsigned short *__restrict__ lcol,
    const int *__restrict__ hcnt, const int *__restrict__ hcol, const double *__restrict__ x,
    double *__restrict__ x0, int nsys, ResState *st, ResShared *sh) {
  const int w = blockIdx.x, t = threadIdx.x;
  const ResWg wg = wgs[w];
  const int nh = hcnt[w], *const halo = hcol + (size_t)w * nhmax;
  bool stale = false;
  for (int l = t; l < wg.rows; l += kResThreads) {
    x0[wg.base + l] = x[wg.base + l];
    stale |= ia[wg.base + l + 1] - ia[wg.base + l] > longest;
  }
  const int e1 = ia[wg.base + wg.rows];
  for (int e = ia[wg.base] + t; e < e1; e += kResThreads) {
    const int c = ja[e], s = lcol[e], h = s - own;
    stale |= h < 0 ? s >= wg.rows || wg.base + s != c : h >= nh || halo[h] != c;
  }
  if (stale) atomicMax(&sh->error, (int)kResStale);
  for (int s = w * kResThreads + t; s < nsys; s += (int)gridDim.x * kResThreads) st[s] = ResState{};
}

// The analysis: workgroup w lists the rows outside its own that its rows refer
// to (ascending), marks them as sent, and gives every nonzero its slot: own
// rows first, then the halo.  Without FILL only cnt[w], the halo's length (more
// than kResHalo also for a column outside the system); with FILL the rest, once
// the longest halo, nhmax, is known.  Dynamic LDS: a bitmap of the system's rows
// and the rank of each of its words.
template <bool FILL>
__global__ __launch_bounds__(kResThreads) void k_res_plan(const ResWg *__restrict__ wgs, int own,
                                                          int nhmax,
                                                          const int *__restrict__ ia,
                                                          const int *__restrict__ ja,
                                                          int *__restrict__ cnt,
                                                          int *__restrict__ hcol,
                                                          unsigned char *__restrict__ sent,
                                                          unsigned short *__restrict__ lcol) {
  extern __shared__ unsigned bits[];
  __shared__ int scan[kResThreads];
  __shared__ int bad;
  const int w = blockIdx.x, t = threadIdx.x;
  const ResWg wg = wgs[w];
  const int words = (wg.s1 - wg.s0 + 31) / 32;
  unsigned short *rank = reinterpret_cast<unsigned short *>(bits + words);
  const int base = wg.base, end = wg.base + wg.rows;
  const int e0 = ia[base], e1 = ia[end];
  if (t == 0) bad = 0;
  for (int i = t; i < words; i += kResThreads) bits[i] = 0;
  __syncthreads();
  for (int e = e0 + t; e < e1; e += kResThreads) {
    const int c = ja[e], i = c - wg.s0;
    if (c < wg.s0 || c >= wg.s1)
      bad = 1;
    else if (c < base || c >= end)
      atomicOr(&bits[i >> 5], 1u << (i & 31));
  }
  __syncthreads();
  // ranks of the words: each thread a run of them
  const int per = (words + kResThreads - 1) / kResThreads;
  const int i0 = min(words, t * per), i1 = min(words, i0 + per);
  int c = 0;
  for (int i = i0; i < i1; ++i) c += __popc(bits[i]);
  scan[t] = c;
  __syncthreads();
  for (int o = 1; o < kResThreads; o <<= 1) {
    const int v = t >= o ? scan[t - o] : 0;
    __syncthreads();
    scan[t] += v;
    __syncthreads();
  }
  const int total = scan[kResThreads - 1];
  if (!FILL && t == 0) cnt[w] = bad ? kResHalo + 1 : total;
  if (!FILL || bad || total > nhmax) return;
  int at = scan[t] - c;
  for (int i = i0; i < i1; ++i) {
    rank[i] = (unsigned short)at;
    for (unsigned m = bits[i]; m; m &= m - 1) {
      const int col = wg.s0 + i * 32 + __ffs((int)m) - 1;
      hcol[(size_t)w * nhmax + at++] = col;
      sent[col] = 1;
    }
  }
  __syncthreads();
  for (int e = e0 + t; e < e1; e += kResThreads) {
    const int col = ja[e], i = col - wg.s0;
    lcol[e] = (unsigned short)(col >= base && col < end
                                   ? col - base
                                   : own + rank[i >> 5] +
                                         __popc(bits[i >> 5] & ((1u << (i & 31)) - 1u)));
  }
}

__global__ void k_res_zero(long long n, unsigned *p) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = 0;
}

using ResKernel = void (*)(ResArgs);
struct ResShape {
  int r, l, threads;
  ResKernel fn;
};
// A thread's registers hold R (2.5 L + 8) words beside the work of a row: 128
// registers per thread at 1024 threads allow these.
const ResShape kShapes[] = {{4, 5, 512, k_resident<4, 5, 512>},
                            {1, 8, 1024, k_resident<1, 8, 1024>},
                            {2, 8, 1024, k_resident<2, 8, 1024>},
                            {1, 16, 1024, k_resident<1, 16, 1024>},
                            {1, 24, 1024, k_resident<1, 24, 1024>},
                            {1, 32, 1024, k_resident<1, 32, 1024>}};

}  // namespace

struct ResPlan {
  bool ok = false;
  std::vector<int> off;
  int nsys = 0, nwg = 0, stride = 0, nhmax = 0, lds = 0, threads = 0, own = 0, longest = 0;
  ResKernel fn = nullptr;
  DevBufPtr wg, hcnt, hcol, sent, lcol, boxes, state, shared;
  size_t box_words = 0;
  unsigned tag = 0;
};

// The plan; not ok where the systems do not fit, null where there is no memory
// for it now (the next solve looks again).  Nothing here is an error of the
// solve, which can go by launches.
static std::shared_ptr<ResPlan> res_plan_build(const SpmvPlan &A, const int *ia, const int *ja,
                                               const std::vector<int> &off) {
  auto P = std::make_shared<ResPlan>();
  P->off = off;
  const int n = A.n, cus = std::min(device_cus(), kResMaxWg), ns = (int)off.size() - 1;
  int big = 0;
  for (int s = 0; s < ns; ++s) big = std::max(big, off[(size_t)s + 1] - off[(size_t)s]);
  if (big < 1 || big > kResMaxN || n > kResMaxRows || A.max_row > 32) return P;
  const ResShape *s = nullptr;
  const int least = A.max_row <= kResShort ? kResRowsShort : kResRows;
  auto rows_per = [&](int rows) {
    return std::max(least, ((rows + cus - 1) / cus + kWave - 1) / kWave * kWave);
  };
  long wgs_all = 0;  // workgroups
  for (int q = 0; q < ns; ++q) {
    const int rows = off[(size_t)q + 1] - off[(size_t)q];
    wgs_all += rows ? (rows + rows_per(rows) - 1) / rows_per(rows) : 0;
  }
  if (wgs_all > kResMaxWgs) return P;
  // Two workgroups per CU where there are half as many again as CUs.  With 1024
  // and 512 threads, ms: 160 grids of up to 150^2 (600 workgroups) 7.9 and 5.6, 60
  // of up to 400^2 132 and 89, 2000 of up to 20^2 1.3 and 1.0, but 300 of up to
  // 60^2 (340 workgroups) 1.57 and 1.79.  One system gains little (512^2 7.1 and
  // 7.0 us per iteration, 128^2 4.0 and 4.2).
  const bool half = A.max_row <= kResShort && 2 * wgs_all > 3 * cus;
  for (const ResShape &c : kShapes) {
    if (A.max_row > c.l || half != (c.threads < kResThreads)) continue;
    if (rows_per(big) <= c.r * c.threads) {
      s = &c;
      break;
    }
  }
  if (!s) return P;
  // teams, the largest system first
  std::vector<int> ord((size_t)ns);
  std::iota(ord.begin(), ord.end(), 0);
  std::stable_sort(ord.begin(), ord.end(), [&](int u, int v) {
    return off[(size_t)u + 1] - off[(size_t)u] > off[(size_t)v + 1] - off[(size_t)v];
  });
  std::vector<ResWg> wgs;
  for (int q : ord) {
    const int s0 = off[(size_t)q], s1 = off[(size_t)q + 1], rows = s1 - s0;
    if (!rows) continue;
    // as few workgroups as hold the rows, of about equal size
    const int k = (rows + rows_per(rows) - 1) / rows_per(rows), team = (int)wgs.size();
    const int nr = std::min(rows_per(rows), ((rows + k - 1) / k + kWave - 1) / kWave * kWave);
    const int size = (rows + nr - 1) / nr;
    for (int i = 0; i < size; ++i)
      wgs.push_back(ResWg{s0 + i * nr, std::min(nr, rows - i * nr), team, size, q, s0, s1, 0});
  }
  P->nsys = ns;
  P->nwg = (int)wgs.size();
  P->fn = s->fn;
  P->threads = s->threads;
  P->own = s->r * s->threads;
  P->longest = s->l;
  P->stride = (P->nwg + 15) / 16 * 16 + kResSkew;
  P->box_words = 4 * ((size_t)n + 3 * (size_t)kResCopies * P->stride);
  auto lds = [&](int halo) {
    return (int)sizeof(double) * (s->r * s->threads + halo + 1) + 4 * halo;
  };
  // the limit belongs to the kernel, which other plans of the shape launch too:
  // the same for all of them
  if (!hip_try(hipFuncSetAttribute(reinterpret_cast<const void *>(P->fn),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds(kResHalo))))
    return P;
  const int words = (big + 31) / 32;
  const int plan_lds = words * 4 + (words + 1) / 2 * 4;
  for (auto *k : {k_res_plan<false>, k_res_plan<true>})
    if (!hip_try(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, plan_lds)))
      return P;
  // the halos' lengths first: a plan that does not fit keeps no memory, one that
  // does what its halos need
  const size_t wgs_bytes = sizeof(ResWg) * wgs.size();
  DevBufPtr wg = dev_try(wgs_bytes), hcnt = dev_try(sizeof(int) * wgs.size());
  if (!wg || !hcnt) return nullptr;
  std::vector<int> cnt(wgs.size());
  auto plan = [&](auto *k, int *hcol, unsigned char *sent, unsigned short *lcol) {
    k<<<P->nwg, kResThreads, plan_lds, stream()>>>(wg->as<ResWg>(), s->r * s->threads, P->nhmax,
                                                   ia, ja, hcnt->as<int>(), hcol, sent, lcol);
  };
  if (!hip_try(hipMemcpyAsync(wg->p, wgs.data(), wgs_bytes, hipMemcpyHostToDevice, stream())))
    return nullptr;
  plan(k_res_plan<false>, nullptr, nullptr, nullptr);
  if (!hip_try(hipMemcpyAsync(cnt.data(), hcnt->p, sizeof(int) * cnt.size(), hipMemcpyDeviceToHost,
                              stream())) ||
      !hip_try(hipStreamSynchronize(stream())))
    return nullptr;
  P->nhmax = *std::max_element(cnt.begin(), cnt.end());
  if (P->nhmax > kResHalo) return P;
  const size_t lists = sizeof(int) * (size_t)P->nwg * P->nhmax;
  size_t avail = 0, all = 0;
  const size_t need = sizeof(unsigned) * P->box_words + lists +
                      sizeof(unsigned short) * (size_t)A.nnz + (size_t)n + ((size_t)64 << 20);
  if (!hip_try(hipMemGetInfo(&avail, &all)) || avail < need) return nullptr;
  P->wg = wg;
  P->hcnt = hcnt;
  P->hcol = dev_try(lists);
  P->sent = dev_try(((size_t)n + 3) / 4 * 4);
  P->lcol = dev_try(sizeof(unsigned short) * (size_t)A.nnz);
  P->state = dev_try(sizeof(ResState) * (size_t)ns);
  P->shared = dev_try(sizeof(ResShared));
  P->boxes = dev_try(sizeof(unsigned) * P->box_words);
  for (const DevBufPtr &b : {P->hcol, P->sent, P->lcol, P->state, P->shared, P->boxes})
    if (!b) return nullptr;
  k_res_zero<<<256, kBlock, 0, stream()>>>(((long long)n + 3) / 4, P->sent->as<unsigned>());
  k_res_zero<<<256, kBlock, 0, stream()>>>((long long)P->box_words, P->boxes->as<unsigned>());
  k_res_zero<<<1, kWave, 0, stream()>>>((long long)(sizeof(ResShared) / 4),
                                        P->shared->as<unsigned>());
  plan(k_res_plan<true>, P->hcol->as<int>(), P->sent->as<unsigned char>(),
       P->lcol->as<unsigned short>());
  P->lds = lds(P->nhmax);
  P->ok = true;
  return P;
}

// Solves by the plan.  kResDone, or x is as it was: kResWait: a wait ran out (or
// the launch was refused), kResStale: the plan is of other columns than ja's, kResError: an error was
// recorded.
enum { kResDone = 0, kResError = -1 };
static int res_run(ResPlan &P, int n, const int *ia, const int *ja, const double *a,
                   const double *d_r, double *x, const double *b, double tol, int maxit,
                   double *hist, double *r, double *p, double *x0, ResOut *out) {
  char *box = P.boxes->as<char>();
  ResArgs g{};
  g.n = n;
  g.stride = P.stride;
  g.wg = P.wg->as<ResWg>();
  g.nhmax = P.nhmax;
  g.ia = ia;
  g.a = a;
  g.lcol = P.lcol->as<unsigned short>();
  g.hcnt = P.hcnt->as<int>();
  g.hcol = P.hcol->as<int>();
  g.sent = P.sent->as<unsigned char>();
  g.d_r = d_r;
  g.b = b;
  g.x = x;
  g.r = r;
  g.p = p;
  g.tol = tol;
  g.maxit = maxit;
  g.polls = (unsigned)options().resident_polls;
  g.iters = kResIters;
  g.hist = hist;
  g.box_a = box;
  g.box_b = box + 16 * (size_t)kResCopies * P.stride;
  g.box_w = box + 48 * (size_t)kResCopies * P.stride;
  g.st = P.state->as<ResState>();
  g.sh = P.shared->as<ResShared>();
  std::vector<ResState> h((size_t)P.nsys);
  auto clear_boxes = [&] {
    k_res_zero<<<256, kBlock, 0, stream()>>>((long long)P.box_words, P.boxes->as<unsigned>());
    k_res_zero<<<1, kWave, 0, stream()>>>((long long)(sizeof(ResShared) / 4),
                                          P.shared->as<unsigned>());
    P.tag = 0;
  };
  k_res_prep<<<P.nwg, kResThreads, 0, stream()>>>(g.wg, P.own, P.longest, P.nhmax, ia, ja, g.lcol,
                                                  g.hcnt, g.hcol, x, x0, P.nsys, g.st, g.sh);
  auto restore = [&] {
    return LAP_HIP(hipMemcpyAsync(x, x0, sizeof(double) * (size_t)n, hipMemcpyDeviceToDevice,
                                  stream())) &&
           LAP_HIP(hipStreamSynchronize(stream()));
  };
  // iter <= maxit + 1, so this many launches always finish
  for (long k = 0; k <= ((long)maxit + 1) / kResIters + 1; ++k) {
    if (P.tag > 0xf0000000u) clear_boxes();  // tags only grow
    g.resume = k > 0;
    g.tag0 = P.tag;
    // (this launch's own status: hipGetLastError would also give what an earlier
    // call of the program left)
    void *args[] = {&g};
    ResShared sh{};
    if (!hip_try(hipLaunchKernel(reinterpret_cast<const void *>(P.fn), dim3((unsigned)P.nwg),
                                 dim3((unsigned)P.threads), args, (size_t)P.lds, stream()))) {
      clear_boxes();
      return restore() ? kResWait : kResError;
    }
    if (!LAP_HIP(hipMemcpyAsync(h.data(), g.st, sizeof(ResState) * h.size(),
                                hipMemcpyDeviceToHost, stream())) ||
        !LAP_HIP(hipMemcpyAsync(&sh, g.sh, sizeof sh, hipMemcpyDeviceToHost, stream())) ||
        !LAP_HIP(hipStreamSynchronize(stream())))
      return kResError;
    if (sh.error) {
      clear_boxes();  // start over with unused tags next time
      return restore() ? sh.error : kResError;
    }
    P.tag = sh.tag;
    if (std::all_of(h.begin(), h.end(), [](const ResState &s) { return s.flag >= 0; })) break;
  }
  for (int s = 0; s < P.nsys; ++s)
    out[s] = ResOut{h[(size_t)s].iter, h[(size_t)s].flag < 0 ? 2 : h[(size_t)s].flag,
                    h[(size_t)s].res0, h[(size_t)s].res};
  return kResDone;
}

int pcg_resident(const SpmvPlan &A, std::shared_ptr<ResPlan> &plan, const std::vector<int> &off,
                 const int *ia, const int *ja, const double *a, const double *d_r, double *x,
                 const double *b, double tol, int maxit, double *hist, double *r, double *p,
                 double *x0, ResOut *out, float *ms) {
  if (!options().resident_polls) return 0;
  int st = kResStale;
  for (int tries = 0; tries < 2 && st == kResStale; ++tries) {
    if (tries || !plan || plan->off != off) plan = res_plan_build(A, ia, ja, off);
    if (!plan || !plan->ok) return 0;
    hipEvent_t e0, e1;
    if (!LAP_HIP(hipEventCreate(&e0))) return -1;
    if (!LAP_HIP(hipEventCreate(&e1))) {
      (void)hipEventDestroy(e0);
      return -1;
    }
    LAP_HIP(hipEventRecord(e0, stream()));
    st = res_run(*plan, A.n, ia, ja, a, d_r, x, b, tol, maxit, hist, r, p, x0, out);
    LAP_HIP(hipEventRecord(e1, stream()));
    LAP_HIP(hipEventSynchronize(e1));
    LAP_HIP(hipEventElapsedTime(ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
  return st == kResDone ? 1 : st == kResError ? -1 : 0;
}

}  // namespace lap
