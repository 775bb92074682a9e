// convert.hip -- matrix set-up on the device: COO -> CSR (lap_coo_to_csr),
// A = L + D + U with or without the diagonal in both triangles
// (lap_csr_split) and the graph Laplacian of an adjacency matrix
// (lap_adjacency_laplacian).
//
// COO -> CSR follows coo_to_csr (io_utils.c:141-235): rows are counted,
// every entry (and, for a symmetric matrix, its mirror) is put into its row,
// and each row is sorted by column.  Atomics hand out the places in a row, so
// the order inside it is arbitrary; what is put there (into ja, for the time) is the entry's fill sequence, the position the reference's serial
// fill gives it (2*i for COO entry i, 2*i+1 for its mirror), and rows are
// sorted by the key (column << 32 | fill sequence).  Keys are unique, so the
// sorted rows do not depend on timing and equal a stable sort of the
// reference's fill, which is the reference's result (glibc's qsort is a merge
// sort, and for distinct columns the order is unique anyway).  Rows are sorted
// by length class:
//   <= 32 entries      in LDS, a lane per entry: its place is the number of
//                      smaller keys in its row;
//   <= 4096 entries    one workgroup per row, bitonic sort in LDS;
//   longer             one workgroup per row: 4096-entry runs sorted in LDS,
//                      then merged pairwise (merge path) through global
//                      scratch.
//
// Bound by atomics and by scattered writes.  Files list their entries by row or
// by column, so neighbouring lanes mostly count for the same row: a run of
// them takes one atomic.  One 4-byte word per CSR entry is scattered (the
// column and value are gathered through it by the sort), by workgroups that
// give each XCD one stretch of the file, so that the words of a line meet in
// one L2.  150 x 160 x 170 (16.2M symmetric entries by row, 28.4M in CSR), the
// size query and the conversion: 5.0 -> 0.8 ms (count 530 -> 78 us, twice;
// placing 1590 -> 98; sorting 1160 -> 215, where its 450 MB take 92; scratch of
// 16 bytes per CSR entry allocated before).  The same entries by column 4.7 ->
// 1.2 ms; in random order, where each takes an atomic and a line of its own, 7.9
// -> 5.7.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/lap_io.h"
#include "lap_core.hpp"

namespace lap {
namespace {

constexpr int kShortRow = 32;
constexpr int kLdsSort = 4096;  // entries per LDS sort (32 KiB of keys)

// --------------------------------------------------------------- scans
constexpr int kScanPer = 4;
constexpr int kScanTile = kBlock * kScanPer;

// Exclusive scan of one value per thread over the workgroup; *total gets
// the workgroup's sum.
__device__ long long block_exscan(long long v, long long *lds, long long *total) {
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  long long x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const long long y = __shfl_up(x, o, kWave);
    if (lane >= o) x += y;
  }
  if (lane == kWave - 1) lds[w] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    long long s = 0;
    for (int i = 0; i < kBlock / kWave; ++i) {
      const long long t = lds[i];
      lds[i] = s;
      s += t;
    }
    lds[kBlock / kWave] = s;
  }
  __syncthreads();
  const long long r = x - v + lds[w];
  *total = lds[kBlock / kWave];
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(kBlock) k_tile_sums(const int *in, long long n, long long *sums) {
  __shared__ long long lds[kBlock / kWave + 1];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) s += in[base + k];
  long long total;
  block_exscan(s, lds, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// One workgroup: exclusive scan of sums[0..nb) in place; sums[nb] = total.
__global__ void __launch_bounds__(kBlock) k_scan_sums(long long *sums, int nb) {
  __shared__ long long lds[kBlock / kWave + 1];
  long long carry = 0;
  for (int b0 = 0; b0 < nb; b0 += kBlock) {
    const int i = b0 + (int)threadIdx.x;
    const long long v = i < nb ? sums[i] : 0;
    long long total;
    const long long r = block_exscan(v, lds, &total);
    if (i < nb) sums[i] = carry + r;
    carry += total;
  }
  if (threadIdx.x == 0) sums[nb] = carry;
}

// out[i] = sum of in[0..i) for i <= n (out has n + 1 entries).
__global__ void __launch_bounds__(kBlock) k_scan_tiles(const int *in, long long n,
                                                       const long long *sums, int nb, int *out) {
  __shared__ long long lds[kBlock / kWave + 1];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  int v[kScanPer];
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    v[k] = base + k < n ? in[base + k] : 0;
    s += v[k];
  }
  long long total;
  long long r = block_exscan(s, lds, &total) + sums[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    if (base + k < n) out[base + k] = (int)r;
    r += v[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = (int)sums[nb];
}

}  // namespace

// out[0..n] = exclusive scan of in[0..n); returns the total (or -1 after a
// HIP error).  ws needs scan_ws_bytes(n).
size_t scan_ws_bytes(long long n) {
  return sizeof(long long) * (size_t)((n + kScanTile - 1) / kScanTile + 2);
}
long long scan_exclusive(const int *in, long long n, int *out, long long *ws) {
  const int nb = (int)std::max<long long>(1, (n + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_tile_sums, dim3(nb), dim3(kBlock), 0, stream(), in, n, ws);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kBlock), 0, stream(), ws, nb);
  hipLaunchKernelGGL(k_scan_tiles, dim3(nb), dim3(kBlock), 0, stream(), in, n, ws, nb, out);
  long long total = -1;
  if (!LAP_HIP(hipMemcpyAsync(&total, ws + nb, sizeof total, hipMemcpyDeviceToHost, stream())))
    return -1;
  sync();
  return total;
}

namespace {

__global__ void k_fill_int(long long n, int v, int *dst) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    dst[i] = v;
}

// ---------------------------------------------------------- COO -> CSR
// Counts this lane's entry for row r (active lanes) and returns its place among
// the row's: neighbouring lanes of one row take one atomic together.
__device__ __forceinline__ int count_run(int *cnt, int r, bool active) {
  const int lane = threadIdx.x & (kWave - 1);
  const unsigned long long on = __builtin_amdgcn_ballot_w64(active);
  const int before = __shfl_up(r, 1, kWave);
  const bool head = active && (lane == 0 || !((on >> (lane - 1)) & 1) || before != r);
  const unsigned long long heads = __builtin_amdgcn_ballot_w64(head);
  // the lanes up to this one that start a run; the first lane past this run
  const unsigned long long upto = ~0ull >> (kWave - 1 - lane);
  const int first = active ? kWave - 1 - __builtin_clzll(heads & upto) : lane;
  const unsigned long long past = (heads | ~on) & ~upto;
  int base = 0;
  if (head) base = atomicAdd(&cnt[r], (past ? __builtin_ctzll(past) : kWave) - lane);
  return __shfl(base, first, kWave) + (lane - first);
}

__global__ void __launch_bounds__(kBlock) k_coo_count(long long nnz, int n, int m,
                                                      const int *__restrict__ rows,
                                                      const int *__restrict__ cols, int sym,
                                                      int *cnt, int *err) {
  // (whole waves stay together)
  for (long long i0 = (long long)blockIdx.x * kBlock; i0 < nnz;
       i0 += (long long)gridDim.x * kBlock) {
    const long long i = i0 + threadIdx.x;
    const bool live = i < nnz;
    const int r = live ? rows[i] : 0, c = live ? cols[i] : 0;
    const bool ok = live && r >= 0 && r < n && c >= 0 && c < m;
    if (live && !ok) atomicOr(err, 1);
    count_run(cnt, r, ok);
    if (sym) count_run(cnt, c, ok && r != c);
  }
}

// fill: ia[0..n) at the start
__global__ void __launch_bounds__(kBlock) k_coo_place(long long nnz, const int *__restrict__ rows,
                                                      const int *__restrict__ cols, int sym,
                                                      int *fill, unsigned *__restrict__ seq) {
  // XCD x (workgroups x, x + 8, ..) takes the x-th eighth of the entries
  const long long tiles = (nnz + kBlock - 1) / kBlock, per = (tiles + 7) / 8;
  const long long t0 = (blockIdx.x & 7) * per, t1 = min(tiles, t0 + per);
  for (long long t = t0 + (blockIdx.x >> 3); t < t1; t += gridDim.x >> 3) {
    const long long i = t * kBlock + threadIdx.x;
    const bool live = i < nnz;
    const int r = live ? rows[i] : 0, c = live ? cols[i] : 0;
    const int a = count_run(fill, r, live);
    if (live) seq[a] = (unsigned)(2 * i);
    if (!sym) continue;
    const int b = count_run(fill, c, live && r != c);
    if (live && r != c) seq[b] = (unsigned)(2 * i) + 1u;
  }
}

// What an entry's fill sequence stands for.
struct CooSrc {
  const int *rows, *cols;
  const double *vals;
  __device__ __forceinline__ unsigned long long key(unsigned q) const {
    const int c = (q & 1) ? rows[q >> 1] : cols[q >> 1];
    return ((unsigned long long)(unsigned)c << 32) | q;
  }
  __device__ __forceinline__ double val(unsigned q) const { return vals[q >> 1]; }
};

// Lists rows longer than kShortRow: medium (<= kLdsSort) and long rows,
// long rows with a scratch offset.  cnt: [0] medium, [1] long; off: scratch
// entries handed out so far.
__global__ void k_row_classes(int n, const int *ia, int *med, int *lng, long long *lng_off,
                              int *cnt, unsigned long long *off) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int len = ia[i + 1] - ia[i];
    if (len <= kShortRow) continue;
    if (len <= kLdsSort) {
      med[atomicAdd(&cnt[0], 1)] = i;
    } else {
      const int k = atomicAdd(&cnt[1], 1);
      lng[k] = i;
      lng_off[k] = (long long)atomicAdd(off, (unsigned long long)len);
    }
  }
}

__device__ __forceinline__ int col_of(unsigned long long k) { return (int)(k >> 32); }

// Rows of at most kShortRow entries, kSortRows of them by a workgroup, up to
// kSortCap entries in LDS; counts the longer rows (ctr as k_row_classes).  seq
// may be ja: a row's words are read before its columns are written.
constexpr int kSortRows = 128, kSortCap = 2048;
__global__ void __launch_bounds__(kBlock) k_sort_short(int n, const int *__restrict__ ia,
                                                       const unsigned *seq, CooSrc src, int *ja,
                                                       double *__restrict__ a, int *ctr,
                                                       unsigned long long *off) {
  constexpr int kPer = kSortCap / kBlock;
  __shared__ unsigned long long key[kSortCap];
  __shared__ __align__(16) unsigned char rowof[kSortCap];
  __shared__ int st[kSortRows + 1];
  const int tid = threadIdx.x;
  for (long long r0 = (long long)blockIdx.x * kSortRows; r0 < n;
       r0 += (long long)gridDim.x * kSortRows) {
    const int nr = (int)min((long long)kSortRows, n - r0);
    __syncthreads();  // (the last rows' keys are read)
    for (int t = tid; t <= nr; t += kBlock) st[t] = ia[r0 + t];
    __syncthreads();
    const int e0 = st[0], cnt = st[nr] - e0;
    if (tid < nr) {
      const int len = st[tid + 1] - st[tid];
      if (len > kLdsSort) {
        atomicAdd(&ctr[1], 1);
        atomicAdd(off, (unsigned long long)len);
      } else if (len > kShortRow) {
        atomicAdd(&ctr[0], 1);
      }
    }
    if (cnt <= kSortCap) {
      unsigned q[kPer];
      unsigned long long k[kPer];
      double v[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u) q[u] = u * kBlock + tid < cnt ? seq[e0 + u * kBlock + tid] : 0;
#pragma unroll
      for (int u = 0; u < kPer; ++u)
        if (u * kBlock + tid < cnt) {
          k[u] = src.key(q[u]);
          v[u] = src.val(q[u]);
        }
      for (int t = tid * 16; t < cnt; t += kBlock * 16)
        *reinterpret_cast<uint4 *>(rowof + t) = uint4{~0u, ~0u, ~0u, ~0u};
      __syncthreads();
      if (tid < nr) {
        const int s = st[tid] - e0, len = st[tid + 1] - e0 - s;
        if (len <= kShortRow)
          for (int j = 0; j < len; ++j) rowof[s + j] = (unsigned char)tid;
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u)
        if (u * kBlock + tid < cnt) key[u * kBlock + tid] = k[u];
      __syncthreads();
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        if (u * kBlock + tid >= cnt) continue;
        const int row = rowof[u * kBlock + tid];
        if (row == 255) continue;  // of a longer row
        const int s = st[row] - e0, len = st[row + 1] - e0 - s;
        int rank = 0;
        for (int j = 0; j < len; ++j) rank += key[s + j] < k[u];
        ja[e0 + s + rank] = col_of(k[u]);
        a[e0 + s + rank] = v[u];
      }
      continue;
    }
    // many entries, or long rows among them: a wave per short row
    for (int row = threadIdx.x / kWave; row < nr; row += kBlock / kWave) {
      const int s = st[row], len = st[row + 1] - s, lane = threadIdx.x & (kWave - 1);
      if (len > kShortRow) continue;
      const unsigned long long k = lane < len ? src.key(seq[s + lane]) : ~0ull;
      int rank = 0;
      for (int j = 0; j < len; ++j) rank += __shfl(k, j, kWave) < k;
      if (lane < len) {
        ja[s + rank] = col_of(k);
        a[s + rank] = src.val((unsigned)k);
      }
    }
  }
}

// Sorts k[0..P) ascending (P a power of two <= kLdsSort), all threads of the
// workgroup.
__device__ void lds_bitonic(unsigned long long *k, int P) {
  for (int w = 2; w <= P; w <<= 1)
    for (int j = w >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < P; i += kBlock) {
        const int l = i ^ j;
        if (l > i) {
          const unsigned long long x = k[i], y = k[l];
          const bool up = (i & w) == 0;
          if ((x > y) == up) {
            k[i] = y;
            k[l] = x;
          }
        }
      }
      __syncthreads();
    }
}

// Loads the keys of seq[s..s+len) (len <= kLdsSort) into LDS padded to a
// power of two and sorts them.
__device__ void lds_load_sort(const unsigned *seq, const CooSrc &src, long long s, int len,
                              unsigned long long *k) {
  int P = 1;
  while (P < len) P <<= 1;
  for (int t = threadIdx.x; t < P; t += kBlock) k[t] = t < len ? src.key(seq[s + t]) : ~0ull;
  __syncthreads();
  lds_bitonic(k, P);
}

__global__ void __launch_bounds__(kBlock) k_sort_medium(const int *rowlist, const int *ia,
                                                        const unsigned *seq, CooSrc src, int *ja,
                                                        double *a) {
  __shared__ unsigned long long k[kLdsSort];
  const int row = rowlist[blockIdx.x];
  const int s = ia[row], len = ia[row + 1] - s;
  lds_load_sort(seq, src, s, len, k);
  for (int t = threadIdx.x; t < len; t += kBlock) {
    ja[s + t] = col_of(k[t]);
    a[s + t] = src.val((unsigned)k[t]);
  }
}

// Number of entries of run A among the first d outputs of merge(A, B)
// (keys unique).
__device__ int merge_split(const unsigned long long *A, int la, const unsigned long long *B,
                           int lb, int d) {
  int lo = d > lb ? d - lb : 0, hi = d < la ? d : la;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (A[mid] < B[d - 1 - mid])
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

__global__ void __launch_bounds__(kBlock) k_sort_long(const int *rowlist, const long long *rowoff,
                                                      const int *ia, const unsigned *seq,
                                                      CooSrc src, unsigned long long *k0,
                                                      unsigned long long *k1, int *ja,
                                                      double *a) {
  __shared__ unsigned long long k[kLdsSort];
  const int row = rowlist[blockIdx.x];
  const long long s = ia[row];
  const int len = ia[row + 1] - (int)s;
  const long long o = rowoff[blockIdx.x];
  unsigned long long *kb[2] = {k0 + o, k1 + o};
  // runs of kLdsSort sorted in LDS
  for (int c0 = 0; c0 < len; c0 += kLdsSort) {
    const int cl = min(kLdsSort, len - c0);
    lds_load_sort(seq, src, s + c0, cl, k);
    for (int t = threadIdx.x; t < cl; t += kBlock) kb[0][c0 + t] = k[t];
    __syncthreads();
  }
  // pairwise merges; each thread produces a contiguous slice of every merge
  int cur = 0;
  for (int w = kLdsSort; w < len; w <<= 1) {
    for (int lo = 0; lo < len; lo += 2 * w) {
      const int la = min(w, len - lo), lb = max(0, min(w, len - lo - w));
      const unsigned long long *A = kb[cur] + lo, *B = A + la;
      unsigned long long *O = kb[cur ^ 1] + lo;
      const int m = la + lb;
      const int d0 = (int)((long long)m * threadIdx.x / kBlock);
      const int d1 = (int)((long long)m * (threadIdx.x + 1) / kBlock);
      int x = merge_split(A, la, B, lb, d0), y = d0 - x;
      for (int d = d0; d < d1; ++d) {
        const bool takeA = y >= lb || (x < la && A[x] < B[y]);
        O[d] = takeA ? A[x++] : B[y++];
      }
    }
    __syncthreads();
    cur ^= 1;
  }
  for (int t = threadIdx.x; t < len; t += kBlock) {
    ja[s + t] = col_of(kb[cur][t]);
    a[s + t] = src.val((unsigned)kb[cur][t]);
  }
}

// ---------------------------------------------------------------- split
__global__ void k_split_count(int n, const int *ia, const int *ja, int aug, int *cl, int *cu) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    int l = 0, u = 0;
    for (int e = ia[i]; e < ia[i + 1]; ++e) {
      const int c = ja[e];
      l += c < i;
      u += c > i;
    }
    cl[i] = l + aug;
    cu[i] = u + aug;
  }
}

__global__ void k_split_fill(int n, const int *ia, const int *ja, const double *a, int aug,
                             const int *lia, int *lja, double *la, const int *uia, int *uja,
                             double *ua, double *d) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    int pl = lia[i], pu = uia[i] + aug;
    double dv = 0.0;
    for (int e = ia[i]; e < ia[i + 1]; ++e) {
      const int c = ja[e];
      if (c < i) {
        lja[pl] = c;
        la[pl++] = a[e];
      } else if (c > i) {
        uja[pu] = c;
        ua[pu++] = a[e];
      } else {
        dv = a[e];
      }
    }
    if (aug) {
      lja[pl] = i;
      la[pl] = dv;
      uja[uia[i]] = i;
      ua[uia[i]] = dv;
    }
    if (d) d[i] = dv;
  }
}

// ------------------------------------------------- adjacency Laplacian
__global__ void k_adj_degree(int n, const int *ia, const double *a, int *deg) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    int dd = -1;
    for (int e = ia[i]; e < ia[i + 1]; ++e) dd = (int)((double)dd + a[e]);
    deg[i] = dd;
  }
}

__global__ void k_adj_values(int n, const int *ia, const int *ja, double *a, const int *deg,
                             int weighted) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double dsq = weighted ? 1.0 / sqrt((double)deg[i]) : 0.0;
    for (int e = ia[i]; e < ia[i + 1]; ++e) {
      const int c = ja[e];
      if (c == i)
        a[e] = weighted ? 1.0 : (double)deg[i];
      else
        a[e] = weighted ? (-1.0 * a[e]) * dsq * (1.0 / sqrt((double)deg[c])) : -1.0 * a[e];
    }
  }
}

unsigned rows_grid(long long n) { return grid_for((size_t)std::max<long long>(n, 1), 1, kBlock, 65536); }

bool overlap(const void *p, size_t pb, const void *q, size_t qb) {
  return (const char *)p < (const char *)q + qb && (const char *)q < (const char *)p + pb;
}

}  // namespace
}  // namespace lap

using namespace lap;

extern "C" {

int lap_coo_to_csr(int n, int m, int nnz, const int *rows, const int *cols, const double *vals,
                   int symmetric, int cap, int *ia, int *ja, double *a, int *nnz_csr) {
  if (n < 1 || m < 1 || nnz < 0 || cap < 0 || !nnz_csr || (symmetric && n != m)) {
    set_error(LAP_ERR_ARG, "coo_to_csr: bad sizes (n %d, m %d, nnz %d, cap %d)", n, m, nnz, cap);
    return LAP_ERR_ARG;
  }
  if (!check_device("coo_to_csr", {{rows, "rows", 4 * (size_t)nnz},
                                   {cols, "cols", 4 * (size_t)nnz},
                                   {vals, "vals", 8 * (size_t)nnz},
                                   {ia, "ia", 4 * ((size_t)n + 1)}}))
    return LAP_ERR_ARG;
  DevBuf cnt(4 * ((size_t)n + 1) + 16), ws(scan_ws_bytes(n) + 16);
  int *c = cnt.as<int>();
  if (!cnt.p || !ws.p) return lap_last_status();
  hipLaunchKernelGGL(k_fill_int, dim3(rows_grid(n + 1)), dim3(kBlock), 0, stream(),
                     (long long)n + 1, 0, c);
  if (nnz)
    hipLaunchKernelGGL(k_coo_count, dim3(rows_grid(nnz)), dim3(kBlock), 0, stream(),
                       (long long)nnz, n, m, rows, cols, symmetric, c, c + n);
  int err = 0;
  LAP_HIP(hipMemcpyAsync(&err, c + n, sizeof err, hipMemcpyDeviceToHost, stream()));
  sync();
  if (err) {
    set_error(LAP_ERR_STRUCT, "coo_to_csr: an entry lies outside %d x %d", n, m);
    return LAP_ERR_STRUCT;
  }
  const long long total = scan_exclusive(c, n, ia, ws.as<long long>());
  if (total < 0) return LAP_ERR_HIP;
  if (total > 0x7fffffffll) {
    set_error(LAP_ERR_STRUCT, "coo_to_csr: %lld CSR entries exceed int32", total);
    return LAP_ERR_STRUCT;
  }
  *nnz_csr = (int)total;
  if (total > cap) {
    if (cap == 0) return LAP_OK;  // size query
    set_error(LAP_ERR_ARG, "coo_to_csr: %lld CSR entries, capacity %d", total, cap);
    return LAP_ERR_ARG;
  }
  if (total == 0) return LAP_OK;
  if (!check_device("coo_to_csr", {{ja, "ja", 4 * (size_t)total}, {a, "a", 8 * (size_t)total}}))
    return LAP_ERR_ARG;
  DevBuf ctr(32);
  if (!ctr.p) return lap_last_status();
  // the entries are read until the last row is sorted, while ja and a are
  // written: inputs that share memory with them are copied first
  DevBufPtr held[3];
  auto apart = [&](const void *in, size_t bytes, DevBufPtr &copy) {
    if (!overlap(in, bytes, ja, 4 * (size_t)total) && !overlap(in, bytes, a, 8 * (size_t)total))
      return in;
    copy = dev_alloc(bytes);
    if (copy->p)
      LAP_HIP(hipMemcpyAsync(copy->p, in, bytes, hipMemcpyDeviceToDevice, stream()));
    return (const void *)copy->p;
  };
  rows = static_cast<const int *>(apart(rows, 4 * (size_t)nnz, held[0]));
  cols = static_cast<const int *>(apart(cols, 4 * (size_t)nnz, held[1]));
  vals = static_cast<const double *>(apart(vals, 8 * (size_t)nnz, held[2]));
  if (!rows || !cols || !vals) return lap_last_status();
  unsigned *seq = reinterpret_cast<unsigned *>(ja);  // until the rows are sorted
  const CooSrc src{rows, cols, vals};
  LAP_HIP(hipMemcpyAsync(c, ia, 4 * (size_t)n, hipMemcpyDeviceToDevice, stream()));
  hipLaunchKernelGGL(k_coo_place, dim3((rows_grid(nnz) + 7) / 8 * 8), dim3(kBlock), 0, stream(),
                     (long long)nnz, rows, cols, symmetric, c, seq);
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(kBlock), 0, stream(), 8ll, 0, ctr.as<int>());
  hipLaunchKernelGGL(k_sort_short, dim3(rows_grid(((long long)n + kSortRows - 1) / kSortRows * kBlock)),
                     dim3(kBlock), 0, stream(), n, ia, seq, src, ja, a, ctr.as<int>(),
                     (unsigned long long *)(ctr.as<int>() + 2));
  int h[4] = {0, 0, 0, 0};
  LAP_HIP(hipMemcpyAsync(h, ctr.p, sizeof h, hipMemcpyDeviceToHost, stream()));
  sync();
  unsigned long long long_total;
  memcpy(&long_total, h + 2, sizeof long_total);
  if (h[0] || h[1]) {
    DevBuf med(4 * (size_t)h[0] + 16), lng(4 * (size_t)h[1] + 16), lng_off(8 * (size_t)h[1] + 16);
    if (!med.p || !lng.p || !lng_off.p) return lap_last_status();
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(kBlock), 0, stream(), 8ll, 0, ctr.as<int>());
    hipLaunchKernelGGL(k_row_classes, dim3(rows_grid(n)), dim3(kBlock), 0, stream(), n, ia,
                       med.as<int>(), lng.as<int>(), lng_off.as<long long>(), ctr.as<int>(),
                       (unsigned long long *)(ctr.as<int>() + 2));
    if (h[0])
      hipLaunchKernelGGL(k_sort_medium, dim3(h[0]), dim3(kBlock), 0, stream(), med.as<int>(), ia,
                         seq, src, ja, a);
    if (h[1]) {
      DevBuf k0(8 * long_total), k1(8 * long_total);
      if (!k0.p || !k1.p) return lap_last_status();
      hipLaunchKernelGGL(k_sort_long, dim3(h[1]), dim3(kBlock), 0, stream(), lng.as<int>(),
                         lng_off.as<long long>(), ia, seq, src, k0.as<unsigned long long>(),
                         k1.as<unsigned long long>(), ja, a);
      sync();
    }
    sync();
  }
  sync();
  forget_plans(ia);
  forget_plans(ja);
  forget_plans(a);
  return lap_last_status();
}

int lap_csr_split(int n, const int *ia, const int *ja, const double *a, int augmented, int cap_l,
                  int *lia, int *lja, double *la, int cap_u, int *uia, int *uja, double *ua,
                  double *d, int *nnz_l, int *nnz_u) {
  if (n < 1 || cap_l < 0 || cap_u < 0 || !nnz_l || !nnz_u || (augmented != 0 && augmented != 1)) {
    set_error(LAP_ERR_ARG, "csr_split: bad arguments");
    return LAP_ERR_ARG;
  }
  if (!check_device("csr_split", {{ia, "ia", 4 * ((size_t)n + 1)},
                                  {lia, "lia", 4 * ((size_t)n + 1)},
                                  {uia, "uia", 4 * ((size_t)n + 1)}}))
    return LAP_ERR_ARG;
  const int nnz = dev_download(ia + n, 1)[0];
  if (!check_device("csr_split", {{ja, "ja", 4 * (size_t)nnz}, {a, "a", 8 * (size_t)nnz}}))
    return LAP_ERR_ARG;
  if (d && !check_device("csr_split", {{d, "d", 8 * (size_t)n}})) return LAP_ERR_ARG;
  if (!spmv_plan(n, nnz, ia, ja)) return lap_last_status();  // validates ia / ja
  DevBuf cl(4 * (size_t)n + 16), cu(4 * (size_t)n + 16), ws(scan_ws_bytes(n) + 16);
  hipLaunchKernelGGL(k_split_count, dim3(rows_grid(n)), dim3(kBlock), 0, stream(), n, ia, ja,
                     augmented, cl.as<int>(), cu.as<int>());
  const long long tl = scan_exclusive(cl.as<int>(), n, lia, ws.as<long long>());
  const long long tu = scan_exclusive(cu.as<int>(), n, uia, ws.as<long long>());
  if (tl < 0 || tu < 0) return LAP_ERR_HIP;
  *nnz_l = (int)tl;
  *nnz_u = (int)tu;
  if (cap_l == 0 && cap_u == 0) return LAP_OK;  // size query
  if (tl > cap_l || tu > cap_u) {
    set_error(LAP_ERR_ARG, "csr_split: needs %lld / %lld entries, capacities %d / %d", tl, tu,
              cap_l, cap_u);
    return LAP_ERR_ARG;
  }
  if (!check_device("csr_split", {{lja, "lja", 4 * (size_t)tl},
                                  {la, "la", 8 * (size_t)tl},
                                  {uja, "uja", 4 * (size_t)tu},
                                  {ua, "ua", 8 * (size_t)tu}}))
    return LAP_ERR_ARG;
  hipLaunchKernelGGL(k_split_fill, dim3(rows_grid(n)), dim3(kBlock), 0, stream(), n, ia, ja, a,
                     augmented, lia, lja, la, uia, uja, ua, d);
  sync();
  for (const void *p : {(const void *)lia, (const void *)lja, (const void *)la,
                        (const void *)uia, (const void *)uja, (const void *)ua})
    forget_plans(p);
  return lap_last_status();
}

int lap_adjacency_laplacian(int n, const int *ia, const int *ja, double *a, int weighted,
                            int *deg) {
  if (n < 1 || (weighted != 0 && weighted != 1)) {
    set_error(LAP_ERR_ARG, "adjacency_laplacian: bad arguments");
    return LAP_ERR_ARG;
  }
  if (!check_device("adjacency_laplacian", {{ia, "ia", 4 * ((size_t)n + 1)}})) return LAP_ERR_ARG;
  const int nnz = dev_download(ia + n, 1)[0];
  if (!check_device("adjacency_laplacian",
                    {{ja, "ja", 4 * (size_t)nnz}, {a, "a", 8 * (size_t)nnz}}))
    return LAP_ERR_ARG;
  if (deg && !check_device("adjacency_laplacian", {{deg, "deg", 4 * (size_t)n}}))
    return LAP_ERR_ARG;
  if (!spmv_plan(n, nnz, ia, ja)) return lap_last_status();  // validates ia / ja
  DevBuf own(deg ? 16 : 4 * (size_t)n + 16);
  int *dd = deg ? deg : own.as<int>();
  hipLaunchKernelGGL(k_adj_degree, dim3(rows_grid(n)), dim3(kBlock), 0, stream(), n, ia, a, dd);
  hipLaunchKernelGGL(k_adj_values, dim3(rows_grid(n)), dim3(kBlock), 0, stream(), n, ia, ja, a,
                     dd, weighted);
  sync();
  forget_plans(a);
  return lap_last_status();
}

}  // extern "C"
