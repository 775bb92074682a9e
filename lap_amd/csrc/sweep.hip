// sweep.hip -- one launch per sweep of the SpMV-only preconditioners
// it_jacobi (it_jacobi.c:4-32), GS_it (GS.c:45-92) and GS_it2 (GS.c:95-159).
//
// The reference runs every sweep as two or three SpMVs plus copies, axpys
// and an element-wise product, each a pass over n-vectors.  Every sweep is
// one of two forms, and each is one kernel here:
//
//   single  y_i = base_i - sum_T a_ij x_j      (sum in CSR order, starting
//           from base_i: csr_matvec with alpha = -1, beta = 1 on a copy of
//           base), then stored as y_i, y_i * d_r_i, or both, or added into
//           w (w_i + y_i * d_r_i);
//   pair    y_i = (base_i - (sum_U a_ij x_j + sum_L a_ij x_j)) * d_r_i
//           (two SpMVs from zero, their sum, the difference, the scaling).
//
// Both use the row-block SpMV body: nonzeros are read coalesced into LDS
// products, then one lane per row sums its products in CSR order, so every
// value equals the unfused sequence bit for bit (rows longer than the LDS
// tile use the same workgroup tree as the plain SpMV).  A pair sweep walks
// row blocks of L and U together (PairPlan: at most kSpmvTile nonzeros of
// L and U per block).
#include <algorithm>

#include "cls.hpp"
#include "lap_core.hpp"
#include "spmv_core.hpp"

namespace lap {

namespace {

// single-form store modes
enum SweepStore : int {
  kStoreScaled = 0,  // out = y * d_r
  kStorePlain = 1,   // out = y
  kStoreBoth = 2,    // out = y, out2 = y * d_r
  kStoreAccum = 3,   // out2 = (first ? 0 : out2) + y * d_r
};

template <int MODE>
struct SweepEpi {
  const double *base, *d_r;
  double *out, *out2;
  int first;
  __device__ double init(int row) const { return base[row]; }
  __device__ void store(int row, double v) const {
    if constexpr (MODE == kStoreScaled) {
      out[row] = v * d_r[row];
    } else if constexpr (MODE == kStorePlain) {
      out[row] = v;
    } else if constexpr (MODE == kStoreBoth) {
      out[row] = v;
      out2[row] = v * d_r[row];
    } else {
      const double s = v * d_r[row];
      out2[row] = (first ? 0.0 : out2[row]) + s;
    }
  }
};

template <int BS, int TILE, int MODE>
__global__ __launch_bounds__(BS) void k_sweep_one(int nblk, const int *__restrict__ rowblk,
                                                  const int *__restrict__ ia,
                                                  const int *__restrict__ ja,
                                                  const double *__restrict__ a,
                                                  const double *__restrict__ x,
                                                  const double *base, const double *d_r,
                                                  double *out, double *out2, int first, int xcd,
                                                  const int *done) {
  if (done && *done) return;
  __shared__ double prod[TILE];
  __shared__ double red[BS / kWave];
  SweepEpi<MODE> epi{base, d_r, out, out2, first};
  spmv_walk<BS, TILE>(block_walk(nblk, xcd), rowblk, ia, ja, a, x, -1.0, prod, red, epi);
}

// Sum of a[e] * x[ja[e]] over [e0, e1) from 0.0, as the plain SpMV sums one
// row: in CSR order through LDS when it fits the tile, else the workgroup
// tree of spmv_long_row.  All threads call it; the result is returned to
// all of them.
template <int BS, int TILE>
__device__ double row_sum_any(int e0, int e1, const int *__restrict__ ja,
                              const double *__restrict__ a, const double *__restrict__ x,
                              double *prod, double *red) {
  const int cnt = e1 - e0;
  double r;
  if (cnt > TILE) {
    double s = 0.0;
    for (int e = e0 + (int)threadIdx.x; e < e1; e += BS) s += (1.0 * a[e]) * x[ja[e]];
    const double t = block_sum<BS>(s, red);
    if (threadIdx.x == 0) red[0] = 0.0 + t;
  } else {
    for (int k = threadIdx.x; k < cnt; k += BS) prod[k] = (1.0 * a[e0 + k]) * x[ja[e0 + k]];
    __syncthreads();
    if (threadIdx.x == 0) {
      red[0] = lds_seq_sum(0.0, prod, 0, cnt);
    }
  }
  __syncthreads();
  r = red[0];
  __syncthreads();
  return r;
}

template <int BS, int TILE>
__global__ __launch_bounds__(BS) void k_sweep_pair(
    int nblk, const int *__restrict__ rowblk, const int *__restrict__ lia,
    const int *__restrict__ lja, const double *__restrict__ la, const int *__restrict__ uia,
    const int *__restrict__ uja, const double *__restrict__ ua, const double *__restrict__ x,
    const double *base, const double *d_r, double *out, int xcd, const int *done) {
  if (done && *done) return;
  __shared__ double prod[TILE];
  __shared__ double red[BS / kWave];
  const BlockWalk w = block_walk(nblk, xcd);
  for (int s = w.begin; s < w.end; s += w.step) {
    const int b = w.block(s);
    if (b >= nblk) continue;
    const int r0 = rowblk[b], r1 = rowblk[b + 1];
    const int l0 = lia[r0], l1 = lia[r1], u0 = uia[r0], u1 = uia[r1];
    const int cl = l1 - l0, cu = u1 - u0;
    if (cl + cu > TILE) {  // a row of its own (the plan guarantees r1 == r0 + 1)
      const double sl = row_sum_any<BS, TILE>(l0, l1, lja, la, x, prod, red);
      const double su = row_sum_any<BS, TILE>(u0, u1, uja, ua, x, prod, red);
      if (threadIdx.x == 0) out[r0] = (base[r0] - (su + sl)) * d_r[r0];
      continue;
    }
#pragma unroll 4
    for (int k = threadIdx.x; k < cl; k += BS) prod[k] = (1.0 * la[l0 + k]) * x[lja[l0 + k]];
#pragma unroll 4
    for (int k = threadIdx.x; k < cu; k += BS)
      prod[cl + k] = (1.0 * ua[u0 + k]) * x[uja[u0 + k]];
    __syncthreads();
    for (int row = r0 + (int)threadIdx.x; row < r1; row += BS) {
      const int a0 = lia[row] - l0, a1 = lia[row + 1] - l0;
      const double sl = lds_seq_sum(0.0, prod, a0, a1);
      const int c0 = uia[row] - u0 + cl, c1 = uia[row + 1] - u0 + cl;
      const double su = lds_seq_sum(0.0, prod, c0, c1);
      out[row] = (base[row] - (su + sl)) * d_r[row];
    }
    __syncthreads();
  }
}

// The same sweeps over row classes (cls.hpp): a byte per row for the matrix and
// d_r, a lane per row, the sums in the same order, so every value is the CSR
// sweep's bit for bit.  Bound by memory latency, so a workgroup has K row
// blocks in flight; the blocks are dealt to the XCDs so that a row's neighbours
// are mostly read through one L2.
//
// Measured at 121 x 93 x 140 (1.6M rows): the single sweep 21 -> 13 us (38 MB:
// 3 TB/s with the launch), without d_r 19 -> 10, the pair 32 -> 14.  Taken from
// the second batch of a large solve's iterations on, as in lap_pcg; matrices
// with many distinct rows and small systems keep the CSR sweeps.
struct ClsArg {
  const unsigned char *cls;
  int ncls;
  const int *off;
  const double *val;
  const int *len;
};
enum { kStorePair = 4 };  // out = (base - (U x + L x)) * d_r: B is U, A is L

template <int BS, int W, int MODE>
__global__ __launch_bounds__(BS, 8) void k_sweep_cls(int n, ClsArg A, ClsArg B,
                                                     const double *__restrict__ d,
                                                     const double *__restrict__ x,
                                                     const double *base, double *out,
                                                     double *out2, int first, int group,
                                                     const int *done) {
  if (done && *done) return;
  constexpr bool kPair = MODE == kStorePair;
  constexpr int K = W <= 4 ? (kPair ? 2 : 4) : W <= 8 && !kPair ? 2 : 1;
  extern __shared__ double sweep_mem[];
  ClsLds<W> ta;
  ClsLds<W> tb;
  double *const dt = sweep_mem;  // d_r of each class of A
  char *const at = reinterpret_cast<char *>(sweep_mem + (A.ncls + 1) / 2 * 2);
  for (int i = threadIdx.x; i < A.ncls; i += BS) dt[i] = d[i];
  const int t = threadIdx.x, nblk = (n - 1) / BS + 1;
  int ca[K], cb[K];
  auto ask = [&](int blk, int &a, int &b) {
    const long long row = (long long)blk * BS + t;
    a = row < n ? A.cls[row] : 0;
    b = kPair && row < n ? B.cls[row] : 0;
  };
  const int me = cls_block(blockIdx.x, group), step = gridDim.x;
#pragma unroll
  for (int u = 0; u < K; ++u) ask(me + u * step, ca[u], cb[u]);
  if (kPair) tb.init(at + A.ncls * ClsLds<W>::kRec, B.ncls, B.off, B.val, B.len);
  ta.init(at, A.ncls, A.off, A.val, A.len);
  for (int blk = me; blk < nblk; blk += K * step) {
    double xa[K][W], xb[K][kPair ? W : 1], bv[K], ov[K];
    int na[K], nb[K];
#pragma unroll
    for (int u = 0; u < K; ++u) ask(blk + (K + u) * step, na[u], nb[u]);
#pragma unroll
    for (int u = 0; u < K; ++u) {
      const long long row = (long long)(blk + u * step) * BS + t;
      if (row >= n) continue;
      ta.load(ca[u], x + row, xa[u]);
      if constexpr (kPair) tb.load(cb[u], x + row, xb[u]);
      bv[u] = base[row];
      if (MODE == kStoreAccum) ov[u] = first ? 0.0 : out2[row];
    }
#pragma unroll
    for (int u = 0; u < K; ++u) {
      const long long row = (long long)(blk + u * step) * BS + t;
      if (row < n) {
        const double dr = dt[ca[u]];
        if constexpr (kPair) {
          const double sl = ta.sum(ca[u], xa[u]), su = tb.sum(cb[u], xb[u]);
          out[row] = (bv[u] - (su + sl)) * dr;
        } else {
          const double v = ta.sum_from(bv[u], -1.0, ca[u], xa[u]);
          if constexpr (MODE == kStoreScaled) {
            out[row] = v * dr;
          } else if constexpr (MODE == kStorePlain) {
            out[row] = v;
          } else if constexpr (MODE == kStoreBoth) {
            out[row] = v;
            out2[row] = v * dr;
          } else {
            const double s = v * dr;
            out2[row] = ov[u] + s;
          }
        }
      }
      ca[u] = na[u];
      cb[u] = nb[u];
    }
  }
}

ClsArg cls_arg(const ClsMat &m) { return ClsArg{m.cls, m.ncls, m.off, m.val, m.len}; }

template <int W>
int sweep_lds(const ClsMat &A, const ClsMat &B) {
  return (A.ncls + 1) / 2 * 16 + (A.ncls + B.ncls) * ClsLds<W>::kRec;
}

template <int W, int MODE>
void sweep_cls_go(const SweepCls &s, const ClsMat &A, const ClsMat &B, const double *x,
                  const double *base, double *out, double *out2, bool first, const int *done) {
  k_sweep_cls<kBlock, W, MODE><<<s.grid, kBlock, sweep_lds<W>(A, B), stream()>>>(
      s.n, cls_arg(A), cls_arg(B), A.d, x, base, out, out2, first ? 1 : 0, s.group, done);
}

template <int W>
void sweep_cls_mode(const SweepCls &s, const ClsMat &A, const ClsMat &B, const double *x,
                    const double *base, double *out, double *out2, int mode, bool first,
                    const int *done) {
  switch (mode) {
    case kStoreScaled:
      return sweep_cls_go<W, kStoreScaled>(s, A, B, x, base, out, out2, first, done);
    case kStorePlain:
      return sweep_cls_go<W, kStorePlain>(s, A, B, x, base, out, out2, first, done);
    case kStoreBoth:
      return sweep_cls_go<W, kStoreBoth>(s, A, B, x, base, out, out2, first, done);
    case kStoreAccum:
      return sweep_cls_go<W, kStoreAccum>(s, A, B, x, base, out, out2, first, done);
    case kStorePair:
      if constexpr (W <= kClsPair)
        return sweep_cls_go<W, kStorePair>(s, A, B, x, base, out, out2, first, done);
    default:
      return;
  }
}

void sweep_cls(const SweepCls &s, const ClsMat &A, const ClsMat &B, const double *x,
               const double *base, double *out, double *out2, int mode, bool first,
               const int *done) {
  auto *f = A.width == 4 ? sweep_cls_mode<4> : A.width == 8 ? sweep_cls_mode<8> : sweep_cls_mode<16>;
  f(s, A, B, x, base, out, out2, mode, first, done);
}

using PairKey = std::tuple<const int *, const int *, int, int, int, int>;
std::map<PairKey, std::unique_ptr<PairPlan>> g_pair;

}  // namespace

const PairPlan *pair_plan(int n, int nl, const int *lia, int nu, const int *uia) {
  const int R = options().spmv_rows;
  PairKey key{lia, uia, n, nl, nu, R};
  auto it = g_pair.find(key);
  if (it != g_pair.end()) return it->second.get();
  const std::vector<int> hl = dev_download(lia, (size_t)n + 1), hu = dev_download(uia, (size_t)n + 1);
  std::vector<int> starts{0};
  int r = 0;
  while (r < n) {
    const int len = (hl[r + 1] - hl[r]) + (hu[r + 1] - hu[r]);
    if (len > kSpmvTile) {
      starts.push_back(++r);
      continue;
    }
    int r1 = r + 1;
    while (r1 < n && r1 - r < R &&
           (hl[r1 + 1] - hl[r]) + (hu[r1 + 1] - hu[r]) <= kSpmvTile)
      ++r1;
    starts.push_back(r1);
    r = r1;
  }
  auto plan = std::make_unique<PairPlan>();
  plan->n = n;
  plan->nblocks = (int)starts.size() - 1;
  plan->rowblk = dev_upload(starts);
  PairPlan *raw = plan.get();
  g_pair[key] = std::move(plan);
  return raw;
}

void forget_pair_plans(const void *p) {
  for (auto it = g_pair.begin(); it != g_pair.end();) {
    if (std::get<0>(it->first) == p || std::get<1>(it->first) == p)
      it = g_pair.erase(it);
    else
      ++it;
  }
}
void release_pair_plans() { g_pair.clear(); }

SweepCls sweep_encode(const SpmvPlan &L, const int *lia, const int *lja, const double *la,
                      const SpmvPlan &U, const int *uia, const int *uja, const double *ua,
                      const SpmvPlan *A, const int *ia, const int *ja, const double *a,
                      const double *d_r, bool pairs) {
  SweepCls s, none;
  const int longest = std::max(L.max_row, U.max_row);
  const int width = longest <= 4 ? 4 : (longest + 7) / 8 * 8;
  // Tables 16 wide: a pair would read 32 values of x for a row that has 15 of them
  // at most, so pairs keep the CSR arrays.  us per iteration with classes and
  // CSR pairs at 3 million rows of a ring (wide because its ends wrap round), 11,
  // 13 and 15 entries a row: it_jacobi 295, 303, 312 and 231, 256, 286; GS_it2 (one
  // pair an iteration) 497, 506, 514 and 436, 470, 498.
  if (pairs && width > kClsPair) return none;
  s.n = L.n;
  s.L = cls_encode("L", L.n, L.nnz, lia, lja, la, d_r, L.max_row, width);
  if (!s.L.cls) return none;
  s.U = cls_encode("U", U.n, U.nnz, uia, uja, ua, d_r, U.max_row, width);
  if (!s.U.cls) return none;
  if (A) {
    s.A = cls_encode("S", A->n, A->nnz, ia, ja, a, d_r, A->max_row);
    if (!s.A.cls) return none;
  }
  // (the pair's two tables: 64 KB of LDS at most)
  if ((width == 4   ? sweep_lds<4>(s.L, s.U)
       : width == 8 ? sweep_lds<8>(s.L, s.U)
                    : sweep_lds<16>(s.L, s.U)) > 65536)
    return none;
  std::vector<int> offs = s.L.offsets;
  offs.insert(offs.end(), s.U.offsets.begin(), s.U.offsets.end());
  const auto g = xcd_grid(offs, kBlock, ((long)s.n - 1) / kBlock + 1, 8 * device_cus());
  s.grid = g.first;
  s.group = g.second;
  return s;
}

void sweep_one_launch(const SweepCls &s, const ClsMat &A, const double *x, const double *base,
                      double *out, double *out2, int mode, bool first, const int *done) {
  sweep_cls(s, A, ClsMat(), x, base, out, out2, mode, first, done);
}

void sweep_pair_launch(const SweepCls &s, const double *x, const double *base, double *out,
                       const int *done) {
  sweep_cls(s, s.L, s.U, x, base, out, nullptr, kStorePair, false, done);
}

void sweep_one_launch(const SpmvPlan &p, const int *ia, const int *ja, const double *a,
                      const double *x, const double *base, const double *d_r, double *out,
                      double *out2, int mode, bool first, const int *done) {
  if (p.nblocks == 0) return;
  const unsigned g = spmv_grid(p);
  const int xcd = options().spmv_walk;
  const int *rb = p.rowblk->as<int>();
#define LAP_SWEEP_CASE(M)                                                                   \
  case M:                                                                                   \
    k_sweep_one<kBlock, kSpmvTile, M><<<g, kBlock, 0, stream()>>>(                          \
        p.nblocks, rb, ia, ja, a, x, base, d_r, out, out2, first ? 1 : 0, xcd, done);        \
    break;
  switch (mode) {
    LAP_SWEEP_CASE(kStoreScaled)
    LAP_SWEEP_CASE(kStorePlain)
    LAP_SWEEP_CASE(kStoreBoth)
    LAP_SWEEP_CASE(kStoreAccum)
    default:
      break;
  }
#undef LAP_SWEEP_CASE
}

void sweep_pair_launch(const PairPlan &p, const int *lia, const int *lja, const double *la,
                       const int *uia, const int *uja, const double *ua, const double *x,
                       const double *base, const double *d_r, double *out, const int *done) {
  if (p.nblocks == 0) return;
  const unsigned g = (unsigned)std::max(1, std::min(p.nblocks, 8 * device_cus()));
  k_sweep_pair<kBlock, kSpmvTile><<<g, kBlock, 0, stream()>>>(
      p.nblocks, p.rowblk->as<int>(), lia, lja, la, uia, uja, ua, x, base, d_r, out,
      options().spmv_walk, done);
}

}  // namespace lap
