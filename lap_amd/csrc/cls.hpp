// cls.hpp -- row classes: a matrix stored as one byte per row.
//
// The Laplacian of a regular grid with few distinct weights has few distinct
// rows, where a row is its column offsets (col - row), its values and, for the
// Jacobi solve, its entry of 1/diag: the 256^3 grid has 27.  One byte per row
// and a small table then hold the whole matrix: 17 MB instead of 1.47 GB.  The
// table holds the very doubles of the matrix in CSR order, so every product
// and sum is the CSR one bit for bit.
//
// Measured, Jacobi PCG at 256^3, per iteration: SpMV 352 -> 120 us (440 MB to
// and from memory, 3.7 TB/s; 286 MB is the least), the r update 86 -> 72 and
// the x and p updates 124 -> 100 us (5.8 and 6.9 TB/s): 574 -> 309 us.  With
// the offsets and values in scalar registers, a class of the wave at a time,
// the SpMV took 150 us; without the order of cls_block 4 us more, and it read
// 573 MB instead of 306.
#pragma once

#include "lap_core.hpp"

namespace lap {

constexpr int kClsMax = 255;   // classes
constexpr int kClsRow = 16;    // entries of a row at most
constexpr int kClsPair = 8;    // width of the triangles' tables at most for sweeps of both

// Systems of fewer rows keep the CSR arrays: their matrix is in the Infinity
// Cache and an iteration is mostly launches (at 10^6 rows of 7 entries an
// iteration of Jacobi PCG takes 45 us with the CSR arrays and 35 with classes).
constexpr int kClsMinRows = 1 << 19;

// A row-class matrix on the device; cls == nullptr: the matrix has too many
// distinct rows (or none was asked for).  Class c's entries are off / val
// [c * width .. + width), padded with offset 0 (the row itself) and value +0.0.
struct ClsMat {
  const unsigned char *cls = nullptr;
  const int *off = nullptr;
  const double *val = nullptr;
  const int *len = nullptr;   // entries of each class
  const double *d = nullptr;  // 1/diag of each class (where d_r was given)
  int ncls = 0, width = 0;
  std::vector<int> offsets;  // the distinct column offsets, ascending
};

// The first row block of workgroup `wg` of a persistent grid that walks its row
// blocks with stride `grid`: blocks are dealt to the 8 XCDs in turn, and this
// gives XCD k the k-th run of `group` blocks of every 8 * group.  With the
// group an eighth of a grid plane, a row's neighbours in its plane and in the
// planes beside it are nearly all read through the same L2.  Which blocks a
// workgroup walks, and so its partial sums, does not change.  (grid: a multiple
// of 8 * group, or group 1.)
__host__ __device__ __forceinline__ int cls_block(int wg, int group) {
  const int x = wg & 7, s = wg >> 3;
  return s / group * (8 * group) + x * group + s % group;
}
// How many of the column offsets lead to a row block of another XCD, for row
// blocks of `rows` rows.
double xcd_cost(const std::vector<int> &offsets, int rows, int group);
// A grid of at most `most` workgroups (and at least 0.9 of it) for row blocks
// of `rows` rows, and its group: the one with the least cost, at most a 64th of
// the nblk row blocks, so that no XCD is left without work.
std::pair<unsigned, int> xcd_grid(const std::vector<int> &offsets, int rows, long nblk, int most);
// The group for row blocks of `rows` rows and a grid of `grid` workgroups: the
// power of two with the fewest lines of x read by several XCDs, by the
// matrix's column offsets.
int cls_group(const std::vector<int> &offsets, int rows, unsigned grid);

// Sends off a look at 1024 rows: *host (pinned) becomes 1 when they have too
// many classes already, as a matrix of random weights has.  About 10 us on the
// stream, where finding out in cls_encode takes 0.15 ms with the waits.  false:
// the matrix cannot be encoded.
bool cls_probe(int n, int nnz, const int *ia, const int *ja, const double *a, const double *d_r,
               int max_row, int *host);

// The table's width is `least` (4, 8 or 16), or 8 or 16 where rows are longer.
// Encodes the matrix (tag: names the buffers that hold the result until the
// next encoding with the same tag).  d_r may be null.  Two passes over the
// matrix; a matrix with too many distinct rows is noticed within a few
// thousand rows.
ClsMat cls_encode(const char *tag, int n, int nnz, const int *ia, const int *ja, const double *a,
                  const double *d_r, int max_row, int least = 8);

// The triangles (and A, for GS_it) of the sweep preconditioners as row classes
// with d_r, and the grid of their sweeps; n == 0: not encoded.  pairs: the sweeps
// will all be of L and U together.
struct SweepCls {
  int n = 0, group = 1;
  unsigned grid = 1;
  ClsMat L, U, A;
};
SweepCls sweep_encode(const SpmvPlan &L, const int *lia, const int *lja, const double *la,
                      const SpmvPlan &U, const int *uia, const int *uja, const double *ua,
                      const SpmvPlan *A, const int *ia, const int *ja, const double *a,
                      const double *d_r, bool pairs);
// The sweeps over classes (A: one of s's matrices).
void sweep_one_launch(const SweepCls &s, const ClsMat &A, const double *x, const double *base,
                      double *out, double *out2, int mode, bool first, const int *done);
void sweep_pair_launch(const SweepCls &s, const double *x, const double *base, double *out,
                       const int *done);

// The mixed solver's inner operator of the same rows: per class first the
// diagonal (with what rounding took from the row's off-diagonals), then the
// off-diagonals rounded to FP32, in CSR order.  Wide enough for
// max_row + 1 entries; cls == nullptr where that is too many.
ClsMat cls_inner(const ClsMat &A, int max_row);

// The table in LDS, a record per class: W values, W offsets, the number of
// entries, and 12 bytes so that the records of different classes start in
// different banks.
template <int W>
struct ClsLds {
  static constexpr int kRec = W * 12 + 16;
  char *t;
  // (every thread of the workgroup; ends in a barrier)
  __device__ __forceinline__ void init(char *lds, int ncls, const int *off, const double *val,
                                       const int *len) {
    t = lds;
    for (int i = threadIdx.x; i < ncls * W; i += blockDim.x) {
      const int c = i / W, j = i % W;
      reinterpret_cast<double *>(t + c * kRec)[j] = val[i];
      reinterpret_cast<int *>(t + c * kRec + W * 8)[j] = off[i];
      if (j == 0) reinterpret_cast<int *>(t + c * kRec + W * 12)[0] = len[c];
    }
    __syncthreads();
  }
  // x at the entries of a row of class c, xr = x + row
  template <class XT>
  __device__ __forceinline__ void load(int c, const XT *__restrict__ xr, XT (&xv)[W]) const {
    const int *o = reinterpret_cast<const int *>(t + c * kRec + W * 8);
#pragma unroll
    for (int i = 0; i < W; ++i) xv[i] = xr[o[i]];
  }
  // sum_j a_rj x_j in CSR order (the padding is left out: 0 * inf is not 0)
  template <class XT>
  __device__ __forceinline__ double sum(int c, const XT (&xv)[W]) const {
    return sum_from(0.0, 1.0, c, xv);
  }
  // s + sum_j (alpha a_rj) x_j, term by term
  template <class XT>
  __device__ __forceinline__ double sum_from(double s, double alpha, int c,
                                             const XT (&xv)[W]) const {
    const double *v = reinterpret_cast<const double *>(t + c * kRec);
    const int len = reinterpret_cast<const int *>(t + c * kRec + W * 12)[0];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const double e = s + (alpha * v[i]) * (double)xv[i];
      s = i < len ? e : s;
    }
    return s;
  }
  // the same for cls_inner's tables: the sum starts with the diagonal's product
  template <class XT>
  __device__ __forceinline__ double sum_inner(int c, const XT (&xv)[W]) const {
    const double *v = reinterpret_cast<const double *>(t + c * kRec);
    const int len = reinterpret_cast<const int *>(t + c * kRec + W * 12)[0];
    double s = v[0] * (double)xv[0];
#pragma unroll
    for (int i = 1; i < W; ++i) {
      const double e = s + (1.0 * v[i]) * (double)xv[i];
      s = i < len ? e : s;
    }
    return s;
  }
};

// 1/diag of row i: from the vector, or (row classes) one byte and a table in
// LDS, 7 of 8 bytes (FP32: 3 of 4) less to read
template <class T>
struct JacD {
  const T *d_r;
  __device__ __forceinline__ void init() {}
  __device__ __forceinline__ T at(size_t i) const { return ld_nt(d_r + i); }
};
template <class T>
struct JacDCls {
  const unsigned char *cls;
  const double *d;
  int ncls;
  T *lds;
  __device__ __forceinline__ void init() {
    __shared__ T t[kClsMax + 1];
    lds = t;
    for (int i = threadIdx.x; i < ncls; i += blockDim.x) t[i] = (T)d[i];
    __syncthreads();
  }
  __device__ __forceinline__ T at(size_t i) const { return lds[ld_nt(cls + i)]; }
};

}  // namespace lap
