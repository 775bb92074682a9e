// cls.hip -- encoding a matrix as row classes (cls.hpp).
//
// Once per solve (the values may change between solves at the same address),
// two passes over the matrix and two synchronisations:
//   1. every workgroup hashes its rows and collects the distinct hashes in an
//      LDS set, merged into a global one with one row of each; more than
//      kClsMax hashes, or a row of more than kClsRow entries, raise the
//      overflow flag, which every workgroup looks at as it goes;
//   2. the host sorts the hashes and one workgroup writes the table from the
//      rows found;
//   3. every row finds its hash and is compared with the class entry by entry:
//      a difference (two rows of one hash) raises the same flag.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <string>

#include "cls.hpp"

namespace lap {

namespace {

constexpr int kClsSlots = 1024;  // global hash set
constexpr int kClsLds = 512;     // per workgroup
constexpr unsigned long long kClsEmpty = ~0ull;

struct ClsState {
  int count, over;      // distinct hashes, overflow / mismatch
};

__device__ __forceinline__ unsigned long long cls_mix(unsigned long long h, unsigned long long k) {
  h = (h ^ k) * 0x9E3779B97F4A7C15ull;
  return h ^ (h >> 29);
}

// the row's hash; kClsEmpty when it is too long
__device__ __forceinline__ unsigned long long cls_hash(int row, const int *__restrict__ ia,
                                                       const int *__restrict__ ja,
                                                       const double *__restrict__ a,
                                                       const double *__restrict__ d_r) {
  const int e0 = ia[row], e1 = ia[row + 1];
  if (e1 - e0 > kClsRow) return kClsEmpty;
  unsigned long long h = (unsigned long long)(e1 - e0) + 1;
  for (int e = e0; e < e1; ++e) {
    h = cls_mix(h, (unsigned)(ja[e] - row));
    h = cls_mix(h, (unsigned long long)__double_as_longlong(a[e]));
  }
  if (d_r) h = cls_mix(h, (unsigned long long)__double_as_longlong(d_r[row]));
  return h == kClsEmpty ? 0 : h;
}

__global__ __launch_bounds__(kBlock) void k_cls_clear(unsigned long long *keys, int *rep,
                                                      ClsState *st) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < kClsSlots; i += gridDim.x * kBlock) {
    keys[i] = kClsEmpty;
    rep[i] = 0x7fffffff;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *st = ClsState{};
}

__global__ __launch_bounds__(kBlock) void k_cls_collect(int n, const int *__restrict__ ia,
                                                        const int *__restrict__ ja,
                                                        const double *__restrict__ a,
                                                        const double *__restrict__ d_r,
                                                        unsigned long long *keys, int *rep,
                                                        ClsState *st) {
  __shared__ unsigned long long set[kClsLds];
  __shared__ int first[kClsLds];
  __shared__ int count, over;
  for (int i = threadIdx.x; i < kClsLds; i += kBlock) set[i] = kClsEmpty;
  if (threadIdx.x == 0) count = over = 0;
  __syncthreads();
  for (int row = blockIdx.x * kBlock + threadIdx.x; row < n; row += gridDim.x * kBlock) {
    const unsigned long long k = cls_hash(row, ia, ja, a, d_r);
    if (k == kClsEmpty) over = 1;
    if (over || __hip_atomic_load(&st->over, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      over = 1;
      break;
    }
    unsigned h = (unsigned)(k >> 40) & (kClsLds - 1);
    for (int probe = 0; probe < kClsLds; ++probe, h = (h + 1) & (kClsLds - 1)) {
      const unsigned long long cur = set[h];
      if (cur == k) break;
      if (cur == kClsEmpty) {
        const unsigned long long prev = atomicCAS(&set[h], kClsEmpty, k);
        if (prev == kClsEmpty) {
          first[h] = row;
          if (atomicAdd(&count, 1) >= kClsMax) over = 1;
          break;
        }
        if (prev == k) break;
      }
    }
  }
  __syncthreads();
  if (over) {
    if (threadIdx.x == 0) atomicOr(&st->over, 1);
    return;
  }
  for (int i = threadIdx.x; i < kClsLds; i += kBlock) {
    const unsigned long long k = set[i];
    if (k == kClsEmpty) continue;
    unsigned h = (unsigned)(k >> 32) & (kClsSlots - 1);
    for (int probe = 0; probe < kClsSlots; ++probe, h = (h + 1) & (kClsSlots - 1)) {
      const unsigned long long prev = atomicCAS(&keys[h], kClsEmpty, k);
      if (prev == kClsEmpty && atomicAdd(&st->count, 1) >= kClsMax) atomicOr(&st->over, 1);
      if (prev == kClsEmpty || prev == k) {
        atomicMin(&rep[h], first[i]);
        break;
      }
    }
  }
}

// one workgroup: *out = 1 when kClsProbe rows, evenly spread, have too many
// hashes already
constexpr int kClsProbe = 1024;
__global__ __launch_bounds__(kClsProbe) void k_cls_probe(int n, const int *__restrict__ ia,
                                                         const int *__restrict__ ja,
                                                         const double *__restrict__ a,
                                                         const double *__restrict__ d_r,
                                                         int *out) {
  __shared__ unsigned long long set[2 * kClsProbe];
  __shared__ int count;
  const int t = threadIdx.x;
  set[t] = set[t + kClsProbe] = kClsEmpty;
  if (t == 0) count = 0;
  __syncthreads();
  const unsigned long long k = cls_hash((int)((long long)t * n / kClsProbe), ia, ja, a, d_r);
  unsigned h = (unsigned)(k >> 40) & (2 * kClsProbe - 1);
  for (int probe = 0; probe < 2 * kClsProbe; ++probe, h = (h + 1) & (2 * kClsProbe - 1)) {
    const unsigned long long prev = atomicCAS(&set[h], kClsEmpty, k);
    if (prev == kClsEmpty) atomicAdd(&count, 1);
    if (prev == kClsEmpty || prev == k) break;
  }
  __syncthreads();
  if (t == 0) *out = count > kClsMax;
}

// one workgroup, a thread per class: the table from the class's row
__global__ __launch_bounds__(kBlock) void k_cls_table(int ncls, int width,
                                                      const int *__restrict__ rep,
                                                      const int *__restrict__ ia,
                                                      const int *__restrict__ ja,
                                                      const double *__restrict__ a,
                                                      const double *__restrict__ d_r,
                                                      int *__restrict__ off,
                                                      int *__restrict__ lens,
                                                      double *__restrict__ val,
                                                      double *__restrict__ d) {
  const int c = threadIdx.x;
  if (c >= ncls) return;
  const int row = rep[c], e0 = ia[row], len = ia[row + 1] - e0;
  for (int j = 0; j < width; ++j) {
    off[c * width + j] = j < len ? ja[e0 + j] - row : 0;
    val[c * width + j] = j < len ? a[e0 + j] : 0.0;
  }
  lens[c] = len;
  d[c] = d_r ? d_r[row] : 0.0;
}

__global__ __launch_bounds__(kBlock) void k_cls_assign(
    int n, const int *__restrict__ ia, const int *__restrict__ ja, const double *__restrict__ a,
    const double *__restrict__ d_r, int ncls, const unsigned long long *__restrict__ sorted,
    const int *__restrict__ rep, unsigned char *__restrict__ cls, ClsState *st) {
  __shared__ unsigned long long key[kClsMax];
  __shared__ int reps[kClsMax];
  for (int i = threadIdx.x; i < ncls; i += kBlock) {
    key[i] = sorted[i];
    reps[i] = rep[i];
  }
  __syncthreads();
  for (long long r0 = (long long)blockIdx.x * kBlock; r0 < n; r0 += (long long)gridDim.x * kBlock) {
    if (r0 + threadIdx.x >= n) break;
    const int row = (int)(r0 + threadIdx.x);
    const unsigned long long k = cls_hash(row, ia, ja, a, d_r);
    int lo = 0, hi = ncls - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (key[mid] < k)
        lo = mid + 1;
      else
        hi = mid;
    }
    const int q = reps[lo];
    const int e0 = ia[row], e1 = ia[row + 1], q0 = ia[q];
    bool same = key[lo] == k && ia[q + 1] - q0 == e1 - e0 &&
                (!d_r || __double_as_longlong(d_r[row]) == __double_as_longlong(d_r[q]));
    for (int j = 0; same && j < e1 - e0; ++j)
      same = ja[e0 + j] - row == ja[q0 + j] - q &&
             __double_as_longlong(a[e0 + j]) == __double_as_longlong(a[q0 + j]);
    if (!same) atomicOr(&st->over, 1);
    cls[row] = (unsigned char)lo;
  }
}

// one workgroup, a thread per class: cls_inner's table, from the entries in
// k_mx_values's order
__global__ __launch_bounds__(kBlock) void k_cls_inner(int ncls, int width, int width_o,
                                                      const int *__restrict__ off,
                                                      const double *__restrict__ val,
                                                      const int *__restrict__ len,
                                                      int *__restrict__ off_o,
                                                      double *__restrict__ val_o,
                                                      int *__restrict__ len_o) {
  const int c = threadIdx.x;
  if (c >= ncls) return;
  double d = 0.0, comp = 0.0;
  int m = 1;
  for (int j = 0; j < len[c]; ++j) {
    const double v = val[c * width + j];
    if (off[c * width + j] == 0) {
      d += v;
      continue;
    }
    const float f = (float)v;
    comp += v - (double)f;
    off_o[c * width_o + m] = off[c * width + j];
    val_o[c * width_o + m] = (double)f;
    ++m;
  }
  off_o[c * width_o] = 0;
  val_o[c * width_o] = d + comp;
  len_o[c] = m;
  for (; m < width_o; ++m) {
    off_o[c * width_o + m] = 0;
    val_o[c * width_o + m] = 0.0;
  }
}

}  // namespace

ClsMat cls_inner(const ClsMat &A, int max_row) {
  ClsMat m = A;
  m.width = (max_row + 8) / 8 * 8;
  double *val = scratch_try("cls_inner_val", (size_t)kClsMax * kClsRow);
  int *off = reinterpret_cast<int *>(
      scratch_try("cls_inner_off", kClsMax * (kClsRow + 1) / 2 + 1));
  if (!A.cls || m.width > kClsRow || !val || !off) return ClsMat();
  m.off = off;
  m.val = val;
  m.len = off + kClsMax * kClsRow;
  k_cls_inner<<<1, kBlock, 0, stream()>>>(A.ncls, A.width, m.width, A.off, A.val, A.len, off, val,
                                          off + kClsMax * kClsRow);
  return m;
}

double xcd_cost(const std::vector<int> &offsets, int rows, int group) {
  double cost = 0.0;
  for (int o : offsets) {
    const double d = std::fmod(std::abs((double)o) / rows, 8.0 * group);
    cost += std::min(1.0, std::min(d, 8.0 * group - d) / group);
  }
  return cost;
}

std::pair<unsigned, int> xcd_grid(const std::vector<int> &offsets, int rows, long nblk, int most) {
  std::pair<unsigned, int> best{(unsigned)most, 1};
  double least = 1e30;
  for (int g = 1; g * 8 <= most && (g == 1 || (long)g * 64 <= nblk); ++g) {
    const int used = most / (8 * g) * (8 * g);
    if (used < 0.9 * most) continue;
    const double cost = xcd_cost(offsets, rows, g);
    if (cost < 0.97 * least) {
      least = cost;
      best = {(unsigned)used, g};
    }
  }
  return best;
}

int cls_group(const std::vector<int> &offsets, int rows, unsigned grid) {
  int best = 1;
  double least = 1e30;
  for (int g = 1; g <= 256 && grid % (8u * (unsigned)g) == 0; g *= 2) {
    const double cost = xcd_cost(offsets, rows, g);
    if (cost < least - 1e-9) {
      least = cost;
      best = g;
    }
  }
  return best;
}

bool cls_probe(int n, int nnz, const int *ia, const int *ja, const double *a, const double *d_r,
               int max_row, int *host) {
  if (n < 1 || nnz < 1 || max_row > kClsRow) return false;
  int *out = reinterpret_cast<int *>(scratch_try("cls_probe", 1));
  if (!out) return false;
  k_cls_probe<<<1, kClsProbe, 0, stream()>>>(n, ia, ja, a, d_r, out);
  return LAP_HIP(hipMemcpyAsync(host, out, sizeof(int), hipMemcpyDeviceToHost, stream()));
}

ClsMat cls_encode(const char *tag, int n, int nnz, const int *ia, const int *ja, const double *a,
                  const double *d_r, int max_row, int least) {
  ClsMat m;
  if (n < 1 || nnz < 1 || max_row > kClsRow || lap_last_status() == LAP_ERR_HIP) return m;
  // what the host reads after the first pass and writes before the second, in
  // one copy each
  struct Table {
    ClsState st;
    int reps[kClsMax + 1];
    unsigned long long sorted[kClsMax];
    unsigned long long key[kClsSlots];
    int rep[kClsSlots];
  };
  static DevBufPtr table;
  static Table *h = nullptr;
  if (!table) table = dev_try(sizeof(Table));
  if (!h && !hip_try(hipHostMalloc((void **)&h, sizeof(Table), hipHostMallocDefault))) h = nullptr;
  if (!table || !h) return m;
  Table *t = table->as<Table>();
  k_cls_clear<<<4, kBlock, 0, stream()>>>(t->key, t->rep, &t->st);
  k_cls_collect<<<grid_for((size_t)n, 4, kBlock, 2048), kBlock, 0, stream()>>>(
      n, ia, ja, a, d_r, t->key, t->rep, &t->st);
  LAP_HIP(hipMemcpyAsync(h, t, sizeof(Table), hipMemcpyDeviceToHost, stream()));
  sync();
  if (lap_last_status() == LAP_ERR_HIP || h->st.over || h->st.count < 1 || h->st.count > kClsMax)
    return m;
  std::vector<std::pair<unsigned long long, int>> found;
  for (int i = 0; i < kClsSlots; ++i)
    if (h->key[i] != kClsEmpty) found.emplace_back(h->key[i], h->rep[i]);
  std::sort(found.begin(), found.end());
  const int nc = (int)found.size();
  if (nc > kClsMax) return m;
  for (int i = 0; i < nc; ++i) {
    h->sorted[i] = found[i].first;
    h->reps[i] = found[i].second;
  }
  const std::string name = std::string("cls_") + tag;
  const int width = max_row <= least ? least : (max_row + 7) / 8 * 8;
  // without the memory for a byte per row the solve keeps its matrix
  size_t avail = 0, all = 0;
  if (!hip_try(hipMemGetInfo(&avail, &all)) || avail < (size_t)n + ((size_t)4 << 20)) return m;
  unsigned char *cls =
      reinterpret_cast<unsigned char *>(scratch_try(name.c_str(), ((size_t)n + 7) / 8));
  double *val = scratch_try((name + "_val").c_str(), (size_t)kClsMax * kClsRow);
  int *off = reinterpret_cast<int *>(
      scratch_try((name + "_off").c_str(), kClsMax * (kClsRow + 1) / 2 + 1));
  int *len = off + kClsMax * kClsRow;
  double *d = scratch_try((name + "_d").c_str(), kClsMax + 1);
  if (!cls || !val || !off || !d) return m;
  LAP_HIP(hipMemcpyAsync(t, h, offsetof(Table, key), hipMemcpyHostToDevice, stream()));
  k_cls_table<<<1, kBlock, 0, stream()>>>(nc, width, t->reps, ia, ja, a, d_r, off, len, val, d);
  k_cls_assign<<<grid_for((size_t)n, 4, kBlock, 4096), kBlock, 0, stream()>>>(
      n, ia, ja, a, d_r, nc, t->sorted, t->reps, cls, &t->st);
  LAP_HIP(hipMemcpyAsync(&h->st, &t->st, sizeof h->st, hipMemcpyDeviceToHost, stream()));
  m.offsets.resize((size_t)nc * width);
  LAP_HIP(hipMemcpyAsync(m.offsets.data(), off, 4 * m.offsets.size(), hipMemcpyDeviceToHost,
                         stream()));
  sync();
  std::sort(m.offsets.begin(), m.offsets.end());
  m.offsets.erase(std::unique(m.offsets.begin(), m.offsets.end()), m.offsets.end());
  if (lap_last_status() == LAP_ERR_HIP || h->st.over) return m;
  m.cls = cls;
  m.off = off;
  m.val = val;
  m.len = len;
  m.d = d;
  m.ncls = nc;
  m.width = width;
  return m;
}

}  // namespace lap
