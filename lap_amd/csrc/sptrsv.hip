// sptrsv.hip -- sparse triangular solves (hip_lower/upper_triangular_solve,
// initialize_and_analyze_L_and_U_solve).
//
// Level scheduling: the analysis assigns each row the length of its longest
// dependency chain (level) and sorts rows by level; a solve runs the levels
// in order, one launch per level, one lane per row (a workgroup per row for
// rows of more than kTriLongRow entries).  Each row's off-diagonal terms are
// subtracted in CSR order and the sum divided by the pivot, so every row is
// computed with exactly the reference's sequential arithmetic
// (simple_blas.c:46-85) and the result equals the sequential solve bitwise.
//
// Chunked mode (option sptrsv_mode 3, the default): one launch per solve over
// chunks of rows that are all resident, values between chunks passed as
// tagged words through memory (k_tri_flow).  Same row arithmetic as the level
// launches: bitwise identical.  Triangles whose rows do not fit a record keep
// the level launches (option sptrsv_mode 0 forces them everywhere), and so do those
// that are faster that way (tri_choose).  Measured
// against the level launches and against one workgroup of 256-row steps per
// chunk with progress counters, which it replaced, per IC0 / GS_std PCG
// iteration (us): 128^3 434 / 480 against 1840 / 2100; 256^3 2100 / 2690
// against 4460 / 4970; level launches at 256^3 7780 / 8310.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <thread>

#include "boxed.hpp"
#include "cls.hpp"
#include "lap_core.hpp"

namespace lap {

namespace {

// desc[t] = {row, first nonzero, end, pivot}: one load gives the row, its
// range and the position of its last diagonal entry (-1: none) (the row
// pointers are not read in the solve).
//
// One launch per level.  The level's short rows (the first `cnt` records)
// take one lane each; each of its `nlong` long rows (the records after them)
// takes a workgroup of its own: the workgroup forms the row's products a
// chunk at a time into LDS (two buffers: waves 1.. form the next chunk while
// lane 0 subtracts the current one in CSR order; the pivot's slot holds
// +0.0, and x - (+0.0) == x bit for bit), so a long row gets exactly the
// lane path's arithmetic while its loads proceed in parallel.  AT/VT
// (value/vector type) = double/double: the FP64 solve; float/float: FP32
// values and vectors with FP64 products and sums (the mixed-precision inner
// solve).
constexpr int kTriChunk = 2048;
constexpr int kTriFill = 12;  // products per thread per fill batch (2048 / 192 <= 12)

__device__ __forceinline__ double sf_load(const double *p) {
  const unsigned long long v = __hip_atomic_load(
      reinterpret_cast<const unsigned long long *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __longlong_as_double((long long)v);
}
__device__ __forceinline__ float sf_load(const float *p) {
  const unsigned v = __hip_atomic_load(reinterpret_cast<const unsigned *>(p), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return __uint_as_float(v);
}
__device__ __forceinline__ void sf_store(double *p, double v) {
  __hip_atomic_store(reinterpret_cast<unsigned long long *>(p),
                     (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sf_store(float *p, float v) {
  __hip_atomic_store(reinterpret_cast<unsigned *>(p), __float_as_uint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// s - p[0] - p[1] - ... - p[m - 1], one term at a time in that order (the
// sequential loop's result bit for bit).  p is LDS, 16-byte aligned, with at
// least 12 readable elements past m (their values are never used).  Batches
// of 12 terms alternate between two register sets and the next batch's loads
// are issued before the current batch's subtractions, so the dependent chain
// pays the FP64 add latency (~6.5 cycles) per term rather than an LDS round
// trip per batch; at most 12 LDS loads are in flight (the counter holds 15).
__device__ __forceinline__ double lds_seq_sub_ahead(double s, const double *p, int m) {
  constexpr int H = 6;  // 16-byte loads per batch
  const double2 *q = reinterpret_cast<const double2 *>(p);
  const int full = m / (2 * H);
  double2 v[H], w[H];
#pragma unroll
  for (int j = 0; j < H; ++j) v[j] = q[j];
  int b = 0;
  // (the scheduling barriers keep the compiler from gathering both batches'
  // loads in one place, which would expose a round trip again)
  for (; b + 2 <= full; b += 2) {
#pragma unroll
    for (int j = 0; j < H; ++j) w[j] = q[(b + 1) * H + j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s -= v[j].x;
      s -= v[j].y;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < H; ++j) v[j] = q[(b + 2) * H + j];  // ends <= m + 11
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s -= w[j].x;
      s -= w[j].y;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (b < full) {
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s -= v[j].x;
      s -= v[j].y;
    }
    ++b;
  }
  for (int k = b * 2 * H; k < m; ++k) s -= p[k];
  return s;
}

// TREE (option sptrsv_long 1): a long row's products are summed in a fixed
// tree order instead -- deterministic, no serial chain, but not the
// sequential order (tolerance parity, not bitwise).  The row is split into
// segments of kTriSeg entries, one workgroup each (the launch's long-row
// workgroups index segd: {level position, segment, segments of the row, the
// row's slot}); each forms its segment's sum as a workgroup tree, and a row
// of several segments is finished by the workgroup that arrives last on the
// row's ticket: it adds the segments' sums in segment order (so the result
// does not depend on which one that is) and resets the ticket for the next
// solve.  Partial sums and the ticket are agent-scope, ordered by fences.
template <class AT, class VT, bool TREE = false>
__global__ __launch_bounds__(kBlock) void k_tri_level(
    int cnt, int nlong, const int4 *__restrict__ desc, const int *__restrict__ ja,
    const AT *__restrict__ a, const double *__restrict__ diag, const VT *x, VT *y,
    const int *__restrict__ done, const int4 *__restrict__ segd, double *part, int *tick) {
  if (done && *done) return;
  const int gshort = (cnt + kBlock - 1) / kBlock;
  if ((int)blockIdx.x < gshort) {
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= cnt) return;
    const int4 d = desc[t];
    const int row = d.x;
    double acc = (double)x[row];
    double piv = 0.0;
    bool in_row = false;
    const int e1 = d.z;
    for (int e = d.y; e < e1; ++e) {
      const int c = ja[e];
      if (c == row) {
        piv = (double)a[e];
        in_row = true;
        continue;
      }
      acc -= (double)a[e] * (double)y[c];
    }
    // diag is only passed (and only read) for matrices without in-row pivots
    if (!in_row && diag) piv = diag[row];
    y[row] = (VT)(acc / piv);
    return;
  }
  const int lr = (int)blockIdx.x - gshort;
  if (lr >= nlong) return;
  if (TREE) {
    __shared__ double red[kBlock / kWave];
    __shared__ int last;
    const int4 sd = segd[lr];
    const int4 d = desc[sd.x];
    const int row = d.x;
    const int e0 = d.y + sd.y * kTriSeg, e1 = min(d.z, e0 + kTriSeg);
    constexpr int B = kTriSeg / kBlock;
    int c[B];
    AT av[B];
    VT yv[B];
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int e = e0 + (int)threadIdx.x + j * kBlock;
      c[j] = e < e1 ? ja[e] : row;
      av[j] = e < e1 ? a[e] : AT(0);
    }
#pragma unroll
    for (int j = 0; j < B; ++j) yv[j] = c[j] != row ? y[c[j]] : VT(0);
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (c[j] != row) s += (double)av[j] * (double)yv[j];
    const double t = block_sum<kBlock>(s, red);  // valid in thread 0
    auto finish = [&](double sum) {
      const double piv = d.w >= 0 ? (double)a[d.w] : diag ? diag[row] : 0.0;
      y[row] = (VT)(((double)x[row] - sum) / piv);
    };
    if (sd.z == 1) {
      if (threadIdx.x == 0) finish(t);
      return;
    }
    if (threadIdx.x == 0) {
      sf_store(part + sd.w + sd.y, t);
      __threadfence();
      last = atomicAdd(tick + sd.w, 1) == sd.z - 1;
    }
    __syncthreads();
    if (threadIdx.x != 0 || !last) return;
    __threadfence();
    double sum = 0.0;
    for (int j = 0; j < sd.z; ++j) sum += sf_load(part + sd.w + j);
    __hip_atomic_store(tick + sd.w, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    finish(sum);
    return;
  }
  __shared__ __align__(16) double prod[2][kTriChunk + 16];  // + lds_seq_sub_ahead's read-ahead
  __shared__ int dpos;
  const int4 d = desc[cnt + lr];
  const int row = d.x;
  const int nch = (d.z - d.y + kTriChunk - 1) / kTriChunk;
  if (threadIdx.x == 0) dpos = -1;
  __syncthreads();
  double acc = (double)x[row];
  // threads t0 .. t0 + nt - 1 form chunk ch's products, all of a thread's
  // loads for the chunk issued together (one batch of kTriFill)
  auto fill = [&](int ch, int t0, int nt) {
    const int base = d.y + ch * kTriChunk;
    const int m = min(kTriChunk, d.z - base);
    double *buf = prod[ch & 1];
    for (int k0 = (int)threadIdx.x - t0; k0 < m; k0 += kTriFill * nt) {
      int c[kTriFill];
      AT av[kTriFill];
      VT yv[kTriFill];
#pragma unroll
      for (int j = 0; j < kTriFill; ++j) {
        const int k = k0 + j * nt;
        c[j] = k < m ? ja[base + k] : row;
        av[j] = k < m ? a[base + k] : AT(0);
      }
#pragma unroll
      for (int j = 0; j < kTriFill; ++j) yv[j] = c[j] != row ? y[c[j]] : VT(0);
#pragma unroll
      for (int j = 0; j < kTriFill; ++j) {
        const int k = k0 + j * nt;
        if (k >= m) continue;
        if (c[j] == row) {
          buf[k] = 0.0;
          atomicMax(&dpos, base + k);  // the last pivot entry, as the lane path keeps
        } else {
          buf[k] = (double)av[j] * (double)yv[j];
        }
      }
    }
  };
  fill(0, 0, kBlock);
  // chunk ch is subtracted by lane 0 while waves 1.. form chunk ch + 1
  for (int ch = 0; ch < nch; ++ch) {
    __syncthreads();  // chunk ch formed, chunk ch - 1 consumed
    if (threadIdx.x < kWave) {
      if (threadIdx.x == 0)
        acc = lds_seq_sub_ahead(acc, prod[ch & 1], min(kTriChunk, d.z - d.y - ch * kTriChunk));
    } else if (ch + 1 < nch) {
      fill(ch + 1, kWave, kBlock - kWave);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double piv = 0.0;
    if (dpos >= 0)
      piv = (double)a[dpos];
    else if (diag)
      piv = diag[row];
    y[row] = (VT)(acc / piv);
  }
}

// Packed rows: lane t loads its row's w columns and values together (one
// dependent stage less than through desc), then the y of earlier levels.
// Same subtraction order and pivot as k_tri_level: bitwise identical.
template <int W>
__global__ __launch_bounds__(kBlock) void k_ell_pack(int n, const int4 *__restrict__ desc,
                                                     const int *__restrict__ ja,
                                                     const double *__restrict__ a,
                                                     int *__restrict__ eja,
                                                     double *__restrict__ ea) {
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < n; t += gridDim.x * kBlock) {
    const int4 d = desc[t];
    const int cnt = d.z - d.y;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      eja[(size_t)t * W + k] = k < cnt ? ja[d.y + k] : -1;
      ea[(size_t)t * W + k] = k < cnt ? a[d.y + k] : 0.0;
    }
  }
}

template <int W>
__global__ __launch_bounds__(kBlock) void k_tri_level_ell(
    int cnt, const int *__restrict__ rows, const int *__restrict__ eja,
    const double *__restrict__ ea, const double *__restrict__ diag, const double *x, double *y,
    const int *__restrict__ done) {
  if (done && *done) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= cnt) return;
  const int row = rows[t];
  int c[W];
  double v[W];
#pragma unroll
  for (int k = 0; k < W; k += 4) {
    const int4 q = *reinterpret_cast<const int4 *>(eja + (size_t)t * W + k);
    c[k] = q.x;
    c[k + 1] = q.y;
    c[k + 2] = q.z;
    c[k + 3] = q.w;
  }
#pragma unroll
  for (int k = 0; k < W; k += 2) {
    const double2 q = *reinterpret_cast<const double2 *>(ea + (size_t)t * W + k);
    v[k] = q.x;
    v[k + 1] = q.y;
  }
  double acc = x[row];
  double piv = 0.0;
  bool in_row = false;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    if (c[k] < 0) break;
    if (c[k] == row) {
      piv = v[k];
      in_row = true;
      continue;
    }
    acc -= v[k] * y[c[k]];
  }
  if (!in_row && diag) piv = diag[row];
  y[row] = acc / piv;
}

// ---------------------------------------------------------- chunked mode
constexpr int kFlRing = 16;       // steps of results kept in LDS
constexpr int kFlHalo = 512;      // values from other chunks kept in LDS (>= 256 = one step's)
constexpr int kFlGroup = 4;       // steps per unrolled group (chunks are padded to it)
constexpr int kFlTeam = 2;        // chunks per workgroup
constexpr int kFlPerCu = 2;       // workgroups per CU at most
constexpr int kFlAhead = 4;       // windows of the export list read ahead
constexpr int kFlMaxSteps = 1 << 18;  // of a chunk: its records stay below 2^31 bytes
// LDS entries per chunk: ring, halo buffer, a zero
constexpr int kFlLds = kFlRing * kWave + kFlHalo + 8;
constexpr int kFlZero = kFlLds - 8;
constexpr unsigned kFlSpins = 1u << 22;  // polls of one wait before the solve fails

// The schedule's records, one block per step of kWave rows, each field
// stored for the 64 rows together so that every load of the compute wave is
// contiguous (bytes, l = lane):
//   [0, 1024)     int4: the LDS byte offsets of the row's four dependencies in
//                 CSR order, 16 bits each (.x, .y; padding: a zero entry,
//                 value 0), the step's word for lane l (.z, see FlLane) and
//                 the base of the row's range test (.w, see fl_out)
//   then W = 4 off-diagonal values per row (FP64: two double2 planes, FP32:
//   one float4 plane), then double2 {pivot, 1/pivot}.
template <class AT>
struct FlRec;
template <>
struct FlRec<double> {
  static constexpr int bytes = kWave * 64;
  fl_u4 c, v0, v1, pv;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int lane16, int off) {
    c = __builtin_amdgcn_raw_buffer_load_b128(b, lane16, off, 0);
    v0 = __builtin_amdgcn_raw_buffer_load_b128(b, lane16 + 1024, off, 0);
    v1 = __builtin_amdgcn_raw_buffer_load_b128(b, lane16 + 2048, off, 0);
    pv = __builtin_amdgcn_raw_buffer_load_b128(b, lane16 + 3072, off, 0);
  }
  __device__ __forceinline__ double val(int j) const {
    return j == 0   ? fl_f64(v0.x, v0.y)
           : j == 1 ? fl_f64(v0.z, v0.w)
           : j == 2 ? fl_f64(v1.x, v1.y)
                    : fl_f64(v1.z, v1.w);
  }
};
template <>
struct FlRec<float> {
  static constexpr int bytes = kWave * 48;
  fl_u4 c, v, pv;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int lane16, int off) {
    c = __builtin_amdgcn_raw_buffer_load_b128(b, lane16, off, 0);
    v = __builtin_amdgcn_raw_buffer_load_b128(b, lane16 + 1024, off, 0);
    pv = __builtin_amdgcn_raw_buffer_load_b128(b, lane16 + 2048, off, 0);
  }
  __device__ __forceinline__ double val(int j) const {
    return (double)__uint_as_float(j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w);
  }
};
__device__ __forceinline__ void fl_load_x(__amdgpu_buffer_rsrc_t b, int lane, int step, double *x) {
  const fl_u2 u = __builtin_amdgcn_raw_buffer_load_b64(b, lane * 8, step * (kWave * 8), 0);
  *x = fl_f64(u.x, u.y);
}
__device__ __forceinline__ void fl_load_x(__amdgpu_buffer_rsrc_t b, int lane, int step, float *x) {
  *x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, lane * 4, step * (kWave * 4), 0));
}
// Whether x lies outside [2^-400, 2^400): inside it (and with the pivot in
// it) the refined division below neither overflows nor loses bits to
// underflow in any step.  `base` is kFlBase, or kFlNever where the pivot is
// outside, which makes every x fail.
constexpr unsigned kFlBase = 623u << 20, kFlSpan = 800u << 20, kFlNever = 0x80000000u;
__device__ __forceinline__ bool fl_out(double x, unsigned base) {
  const unsigned h = (unsigned)((unsigned long long)__double_as_longlong(x) >> 32) & 0x7fffffffu;
  return h - base >= kFlSpan;
}

// a / b correctly rounded, from y = 1/b correctly rounded: two residual
// corrections of a*y by fused multiply-adds.  The first leaves the quotient
// within one unit in the last place, and Markstein's theorem (P. W.
// Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", IBM J. Res. Dev. 34, 1990) makes the second's result the
// rounded quotient, so the bits are the divide instruction sequence's at less
// than half its dependent latency (five operations).  a and b not fl_out.
__device__ __forceinline__ double fl_div(double a, double b, double y) {
  double q = a * y;
  q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// (Values between workgroups: boxed.hpp.  A chunk's inbox is one box per use,
// the tag is the solve's number.  LDS operations of a wave execute in issue
// order, so between them fl_fence, which binds only the compiler, is enough.)

// LDS progress words of a chunk, each written by one wave.
struct FlProg {
  int hready;        // halo: values in LDS so far
  int xdone, ydone;  // export / store: steps whose results they no longer need
  int failed;        // 0, or -1
  int cdone, hcons;  // compute: steps finished, halo values consumed
};
__device__ __forceinline__ int fl_ld(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void fl_st(int *p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// What a step waits for, one word per lane of the compute wave: lane l of the
// step's record holds the least value that the progress word of lane l must
// have, and the wave keeps the words as last seen in one register, so the
// test is one comparison, and one LDS read when it fails.  Lanes 0 and 7 of
// the record are also what the wave publishes when the step is done.
enum FlLane {
  FL_HALO = 0,   // hready >= halo values the step uses (published to hcons)
  FL_SIB = 1,    // cdone of the workgroup's other chunk
  FL_X = 2,      // xdone and ydone: the step's ring entries are free
  FL_Y = 3,
  FL_FAILED = 4, // failed >= 0
  FL_DONE = 5,   // nothing to wait for (published to cdone)
};

// Two chunks per workgroup, four waves per chunk.  A chunk runs its rows
// level by level in steps of at most 64 rows; each of its waves has one job
// and they hand over through LDS words, with no barrier and no wait on global
// memory between a step and the next:
//   wave 0, compute: a row per lane; dependencies come from the LDS rings (the
//     last kFlRing steps of each chunk of the workgroup) or from the chunk's
//     LDS halo buffer, the result goes into its own ring.  Records and
//     right-hand sides are loaded kFlGroup steps ahead into registers.
//   wave 1, halo: takes the values other workgroups put into this chunk's
//     inbox, in the order the steps use them, into the halo buffer.  It never
//     waits for a later value while an earlier one is there, so a chunk's
//     progress depends only on values it needs next.
//   wave 2, export: puts results other workgroups use into their inboxes.
//   wave 3, store: writes results over the right-hand sides they came from
//     (schedule order, contiguous).  Scattered to their rows from here they
//     cost 64 write requests a step, which held up the CU's loads;
//     k_fl_spread does it afterwards with the whole chip.
// What bounds it: the chain of levels.  A step costs the LDS round trip of
// the previous step's results, four dependent subtractions and the division,
// 0.16 us.  Crossing into another workgroup costs a trip through memory, about
// 3 us, but only once per boundary on the longest path: a chunk runs behind
// its neighbours by that much and then at their pace.  Two chunks per
// workgroup save a third of the boundaries; four saved half, but a CU reads
// records at no more than about 57 GB/s, which four chunks' steps exceed.
// (Before: a workgroup took a step of 256 rows between two barriers, loaded
// its neighbours' values inside the step and published a counter after it:
// about 2.2 us per level.)  Every wait is bounded; one that runs out raises
// state[1] and ends the workgroup, and the others follow.
// AT: the values' type, VT: the vectors' (FP32 values and vectors are
// summed in FP64 and the result rounded once, as the FP32 level launches do).
template <class AT, class VT>
__global__ __launch_bounds__(4 * kFlTeam * kWave, 4) void k_tri_flow(
    const int *__restrict__ cstep, const char *__restrict__ rec, VT *xc, const int *__restrict__ hbase,
    const int *__restrict__ ebase, const int2 *__restrict__ exps, void *inbox, int inbox_bytes,
    const unsigned *epoch, int *state, const int *__restrict__ done) {
  if (done && *done) return;
  __shared__ VT all[kFlTeam * kFlLds];  // per chunk: ring, halo buffer, a zero
  __shared__ FlProg progs[kFlTeam];
  __shared__ int free_word, spare[kFlTeam * kWave];
  // a workgroup's waves are dealt to the CU's four SIMDs in turn: each chunk's
  // jobs are rotated by one against the last's, so that every SIMD gets one
  // compute wave
  const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x / (4 * kWave));
  const int wave = (__builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave) - team) & 3;
  const int lane = threadIdx.x & (kWave - 1);
  const int c = blockIdx.x * kFlTeam + team;
  const int k0 = __builtin_amdgcn_readfirstlane(cstep[c]);
  const int ns = __builtin_amdgcn_readfirstlane(cstep[c + 1]) - k0;  // a multiple of kFlGroup
  const unsigned tag = (unsigned)__builtin_amdgcn_readfirstlane((int)*epoch);
  VT *vals = all + team * kFlLds;
  FlProg &prog = progs[team];
  if (threadIdx.x < kFlTeam) {
    progs[threadIdx.x] = FlProg{0, 0, 0, 0, 0, 0};
    all[threadIdx.x * kFlLds + kFlZero] = VT(0);
  }
  if (threadIdx.x == 0) free_word = 0x7fffffff;
  __syncthreads();
  auto fail = [&]() {
    if (lane < kFlTeam) fl_st(&progs[lane].failed, -1);
    if (lane == 0)
      __hip_atomic_store(&state[1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  VT *const xk = xc + (size_t)k0 * kWave;
  const __amdgpu_buffer_rsrc_t box = fl_buffer(inbox, inbox_bytes);
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);
    const __amdgpu_buffer_rsrc_t rb =
        fl_buffer(rec + (size_t)k0 * FlRec<AT>::bytes, (ns + kFlGroup) * FlRec<AT>::bytes);
    const __amdgpu_buffer_rsrc_t xb =
        fl_buffer(xk, (ns + kFlGroup) * kWave * (int)sizeof(VT));
    // this lane's progress word (see FlLane) and where it publishes
    const int *word = lane == FL_HALO     ? &prog.hready
                      : lane == FL_SIB    ? &progs[team ^ 1].cdone
                      : lane == FL_X      ? &prog.xdone
                      : lane == FL_Y      ? &prog.ydone
                      : lane == FL_FAILED ? &prog.failed
                                          : &free_word;
    int *const out = lane == FL_HALO   ? &prog.hcons
                     : lane == FL_DONE ? &prog.cdone
                                       : &spare[team * kWave + lane];
    FlRec<AT> R[kFlGroup];
    VT X[kFlGroup];
#pragma unroll
    for (int j = 0; j < kFlGroup; ++j) {
      R[j].load(rb, lane * 16, j * FlRec<AT>::bytes);
      fl_load_x(xb, lane, j, &X[j]);
    }
    // every load complete here, so that the waits inside the loop (which count
    // loads in flight) follow the loop's own order and leave the other steps'
    // loads in flight
#pragma unroll
    for (int j = 0; j < kFlGroup; ++j) {
      asm volatile("" ::"v"(R[j].c), "v"(R[j].pv), "v"(X[j]));
#pragma unroll
      for (int d = 0; d < 4; ++d) asm volatile("" ::"v"(R[j].val(d)));
    }
    int seen = lane < FL_DONE ? 0 : 0x7fffffff;  // the lane's progress word, as last seen
    // (a failed wait ends the loop with its group: leaving it inside would
    // merge the steps' load counts and make every wait a full one)
    int dead = 0;
    for (int k = 0; k < ns && !dead; k += kFlGroup) {
#pragma unroll
      for (int j = 0; j < kFlGroup; ++j) {
        const int need = (int)R[j].c.z;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(seen < need) != 0, 0)) {
          unsigned spins = 0;
          do {
            seen = fl_ld(word);
            dead |= __builtin_amdgcn_readlane(seen, FL_FAILED) | (++spins > 4 * kFlSpins);
          } while (!dead && __builtin_amdgcn_ballot_w64(seen < need) != 0);
        }
        fl_fence();
        const char *const lds = reinterpret_cast<const char *>(all);
        auto at = [&](unsigned o) { return *reinterpret_cast<const VT *>(lds + o); };
        VT yv[4];
        yv[0] = at(R[j].c.x & 0xffffu);
        yv[1] = at(R[j].c.x >> 16);
        yv[2] = at(R[j].c.y & 0xffffu);
        yv[3] = at(R[j].c.y >> 16);
        double acc = (double)X[j];
#pragma unroll
        for (int d = 0; d < 4; ++d) acc -= R[j].val(d) * (double)yv[d];
        const double piv = fl_f64(R[j].pv.x, R[j].pv.y);
        double q = fl_div(acc, piv, fl_f64(R[j].pv.z, R[j].pv.w));
        // outside the refined division's range (a zero among them): divide
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(fl_out(acc, R[j].c.w)) != 0, 0)) {
          fl_fence();  // (kept a branch)
          q = acc / piv;
        }
        vals[k % kFlRing * kWave + j * kWave + lane] = (VT)q;
        fl_fence();
        fl_st(out, need);
        // (past the chunk's end: the following blocks, which are allocated)
        __builtin_amdgcn_sched_barrier(0);
        R[j].load(rb, lane * 16, (k + j + kFlGroup) * FlRec<AT>::bytes);
        fl_load_x(xb, lane, k + j + kFlGroup, &X[j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (dead) fail();
  } else if (wave == 1) {
    const int h0 = __builtin_amdgcn_readfirstlane(hbase[c]);
    const int nh = __builtin_amdgcn_readfirstlane(hbase[c + 1]) - h0;
    // Two looks at the inbox are in flight at a time, each at the two windows
    // of 64 entries from the first one missing when it was issued: a value is
    // seen half a round trip after it can be, not up to a whole one.
    int base = 0, at[2];
    FlBoxed<VT> w[2][2];
    auto look = [&](int s) {
      at[s] = base;
      // (past the inbox's end the buffer reads as zero, which is no tag)
      w[s][0].load(box, h0 + base + lane);
      w[s][1].load(box, h0 + base + kWave + lane);
    };
    if (nh > 0) {
      look(0);
      look(1);
    }
    unsigned spins = 0;
    while (base < nh) {
      bool stop = false;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int lim = min(nh, __builtin_amdgcn_readfirstlane(fl_ld(&prog.hcons)) + kFlHalo);
        const int i = at[s] + lane, i2 = i + kWave;
        const bool got = i < base || (i < lim && w[s][0].is(tag));
        const bool got2 = i2 < base || (i2 < lim && w[s][1].is(tag));
        const unsigned long long m = ~__builtin_amdgcn_ballot_w64(got);
        const unsigned long long m2 = ~__builtin_amdgcn_ballot_w64(got2);
        const int to = at[s] + (m ? __builtin_ctzll(m) : m2 ? kWave + __builtin_ctzll(m2) : 2 * kWave);
        if (to > base) {  // the leading run of values that are there
          VT *const buf = vals + kFlRing * kWave;
          if (i >= base && i < to) buf[i % kFlHalo] = w[s][0].value();
          if (i2 >= base && i2 < to) buf[i2 % kFlHalo] = w[s][1].value();
          fl_fence();
          base = to;
          if (lane == 0) fl_st(&prog.hready, base);
          spins = 0;
        } else {
          // (a chunk that the solve has not reached yet leaves the memory to
          // the others)
          if (spins > 8) __builtin_amdgcn_s_sleep(12);
          if (fl_ld(&prog.failed)) stop = true;
          if (++spins > kFlSpins) {
            fail();
            stop = true;
          } else if ((spins & 63u) == 0 &&
                     __hip_atomic_load(&state[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            if (lane < kFlTeam) fl_st(&progs[lane].failed, -1);
            stop = true;
          }
        }
        look(s);
      }
      if (__builtin_amdgcn_readfirstlane((int)stop)) break;
    }
  } else if (wave == 2) {
    const int e0 = __builtin_amdgcn_readfirstlane(ebase[c]);
    const int ne = __builtin_amdgcn_readfirstlane(ebase[c + 1]) - e0;
    const int2 none{0x7fffffff, 0};
    // the list is read kFlAhead windows ahead (a window is a few steps long,
    // less than a trip to memory)
    int2 win[kFlAhead];
#pragma unroll
    for (int w = 0; w < kFlAhead; ++w)
      win[w] = w * kWave + lane < ne ? exps[e0 + w * kWave + lane] : none;
    if (ne == 0 && lane == 0) fl_st(&prog.xdone, 0x3fffffff);
    unsigned spins = 0;
    bool stop = false;
    for (int b = 0; b < ne && !stop; b += kWave) {
      const int2 e = win[0];  // {local record, inbox entry}, ascending records
#pragma unroll
      for (int w = 0; w + 1 < kFlAhead; ++w) win[w] = win[w + 1];
      const int nb = b + kFlAhead * kWave + lane;
      win[kFlAhead - 1] = nb < ne ? exps[e0 + nb] : none;
      bool pending = e.x != none.x;
      for (;;) {
        const int cd = __builtin_amdgcn_readfirstlane(fl_ld(&prog.cdone));
        fl_fence();
        const bool now = pending && e.x < cd * kWave;
        const unsigned long long any = __builtin_amdgcn_ballot_w64(now);
        if (now) {
          fl_put(box, e.y, tag, vals[e.x % (kFlRing * kWave)]);
          pending = false;
        }
        const unsigned long long left = __builtin_amdgcn_ballot_w64(pending);
        // the first record still to be exported (of this window or the next)
        const int t = left ? __builtin_amdgcn_readlane(e.x, __builtin_ctzll(left))
                           : __builtin_amdgcn_readfirstlane(win[0].x);
        fl_fence();
        if (lane == 0) fl_st(&prog.xdone, t == none.x ? 0x3fffffff : t / kWave);
        if (!left) break;
        if (any) {
          spins = 0;
        } else {
          if (fl_ld(&prog.failed)) stop = true;
          if (++spins > 4 * kFlSpins) {
            fail();
            stop = true;
          }
          if (__builtin_amdgcn_readfirstlane((int)stop)) break;
          __builtin_amdgcn_s_sleep(1);
        }
      }
    }
  } else {
    bool stop = false;
    for (int k = 0; k < ns; k += kFlGroup) {
      unsigned spins = 0;
      while (__builtin_amdgcn_readfirstlane(fl_ld(&prog.cdone)) < k + kFlGroup) {
        if (fl_ld(&prog.failed)) stop = true;
        if (++spins > 4 * kFlSpins) {
          fail();
          stop = true;
        }
        if (__builtin_amdgcn_readfirstlane((int)stop)) break;
        __builtin_amdgcn_s_sleep(1);
      }
      if (__builtin_amdgcn_readfirstlane((int)stop)) break;
      fl_fence();
      VT v[kFlGroup];
#pragma unroll
      for (int j = 0; j < kFlGroup; ++j) v[j] = vals[k % kFlRing * kWave + j * kWave + lane];
      fl_fence();
      if (lane == 0) fl_st(&prog.ydone, k + kFlGroup);
#pragma unroll
      for (int j = 0; j < kFlGroup; ++j) st_nt(xk + (k + j) * kWave + lane, v[j]);
    }
  }
}

// xc[t] = x[map[t]]: the right-hand side in the order the compute waves read
// it (padding, map < 0, keeps the 1.0 it was given), and the next solve's tag.
// The rows of neighbouring schedule positions share lines of x, so each XCD
// (workgroups are dealt to the 8 XCDs round-robin) sweeps one contiguous
// eighth of the positions: its workgroups then read the same lines out of
// their own L2.  The grid is a multiple of 8.
template <class VT>
__global__ __launch_bounds__(kBlock) void k_fl_gather(int n, const int *__restrict__ map,
                                                      const VT *__restrict__ x,
                                                      VT *__restrict__ xc, unsigned *epoch,
                                                      const int *__restrict__ done) {
  if (done && *done) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) *epoch += 1u;
  const int xcd = blockIdx.x & 7, per = gridDim.x >> 3;
  const long long lo = (long long)n * xcd / 8, hi = (long long)n * (xcd + 1) / 8;
  for (long long t = lo + (long long)(blockIdx.x >> 3) * kBlock + threadIdx.x; t < hi;
       t += (long long)per * kBlock) {
    const int row = ld_nt(map + t);  // the map and xc are streamed; x lines are reused
    if (row >= 0) st_nt(xc + t, x[row]);
  }
}

// y[i] = xc[pos[i]]: a solve's results in row order (the same walk).
template <class VT>
__global__ __launch_bounds__(kBlock) void k_fl_spread(int n, const int *__restrict__ pos,
                                                      const VT *__restrict__ xc,
                                                      VT *__restrict__ y,
                                                      const int *__restrict__ done) {
  if (done && *done) return;
  const int xcd = blockIdx.x & 7, per = gridDim.x >> 3;
  const long long lo = (long long)n * xcd / 8, hi = (long long)n * (xcd + 1) / 8;
  for (long long i = lo + (long long)(blockIdx.x >> 3) * kBlock + threadIdx.x; i < hi;
       i += (long long)per * kBlock)
    st_nt(y + i, xc[ld_nt(pos + i)]);
}

// The same with what the caller does next in the same pass: y += the solve
// (ADD), and partials of r.y (part != null).  Rows are walked and summed as
// k_rw does it, so the partials are k_rw's bit for bit, in an order of the
// workgroups that keeps an XCD on one run of rows per round.  Bound by the
// gather, whose lines several XCDs read: at 97 x 110 x 83 the solve's copy back,
// axpy and dot product took 7.6 + 5.5 + 4.6 us, this 10.7; at 128^3 the copy back
// and dot product 14.0 + 8.8, this 20.4.
template <bool ADD>
__global__ __launch_bounds__(kBlock) void k_fl_tail(int n, const int *__restrict__ pos,
                                                    const double *__restrict__ xc, double *y,
                                                    const double *__restrict__ r, double *part,
                                                    int group, const int *__restrict__ done) {
  if (done && *done) return;
  __shared__ double red[kBlock / kWave];
  const int me = cls_block(blockIdx.x, group);
  const size_t stride = (size_t)gridDim.x * kBlock;
  double s = 0.0;
  constexpr int U = 4;  // rows in flight
  for (size_t i0 = (size_t)me * kBlock + threadIdx.x; i0 < (size_t)n; i0 += U * stride) {
    int at[U];
    double v[U], w[U], rv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * stride;
      at[u] = i < (size_t)n ? ld_nt(pos + i) : 0;
      w[u] = ADD && i < (size_t)n ? ld_nt(y + i) : 0.0;
      rv[u] = part && i < (size_t)n ? ld_nt(r + i) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = xc[at[u]];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t i = i0 + u * stride;
      if (i >= (size_t)n) continue;
      w[u] = ADD ? w[u] + 1.0 * v[u] : v[u];
      st_nt(y + i, w[u]);
      if (part) s += rv[u] * w[u];
    }
  }
  if (!part) return;
  const double t = block_sum<kBlock>(s, red);
  if (threadIdx.x == 0) part[me] = t;
}

// comp[t] = pos[map[t]]: a schedule's right-hand sides taken from another
// schedule's results.
__global__ __launch_bounds__(kBlock) void k_fl_compose(int n, const int *__restrict__ map,
                                                       const int *__restrict__ pos,
                                                       int *__restrict__ comp) {
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < n; t += gridDim.x * kBlock)
    comp[t] = map[t] < 0 ? -1 : pos[map[t]];
}

// The records for one set of values, and xc's padding.
template <class AT, class VT>
__global__ __launch_bounds__(kBlock) void k_fl_pack(int n, const int *__restrict__ cmap,
                                                    const int4 *__restrict__ desc,
                                                    const int *__restrict__ ja,
                                                    const AT *__restrict__ a,
                                                    const int2 *__restrict__ code,
                                                    const int2 *__restrict__ need,
                                                    const int *__restrict__ step_in_chunk,
                                                    char *__restrict__ rec,
                                                    VT *__restrict__ xc) {
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < n; t += gridDim.x * kBlock) {
    const int k = t / kWave, l = t % kWave;
    char *blk = rec + (size_t)k * FlRec<AT>::bytes;
    AT v[4] = {AT(0), AT(0), AT(0), AT(0)};
    AT piv = AT(1);
    const int m = cmap[t];
    if (m >= 0) {
      const int4 d = desc[m];
      int j = 0;
      for (int e = d.y; e < d.z; ++e) {
        if (ja[e] == d.x)
          piv = a[e];
        else if (j < 4)
          v[j++] = a[e];
      }
    }
    if (m < 0) xc[t] = VT(1);
    const int2 ce = code[t];  // LDS entries -> byte offsets
    const int2 cd{(int)((unsigned)ce.x * sizeof(VT)), (int)((unsigned)ce.y * sizeof(VT))};
    const int2 nd = need[k];
    const int low = -0x7fffffff;
    const int step = step_in_chunk[k];
    const int word = l == FL_HALO             ? nd.x
                     : l == FL_SIB            ? nd.y
                     : l == FL_X || l == FL_Y ? step - kFlRing + 1
                     : l == FL_FAILED         ? 0
                     : l == FL_DONE           ? step + 1
                                              : low;
    const double dp = (double)piv;
    const bool out = fl_out(dp, kFlBase);
    reinterpret_cast<int4 *>(blk)[l] = int4{cd.x, cd.y, word, (int)(out ? kFlNever : kFlBase)};
    const double2 pv{dp, out ? 0.0 : 1.0 / dp};
    if constexpr (sizeof(AT) == 8) {
      double2 *p = reinterpret_cast<double2 *>(blk + kWave * 16);
      p[l] = double2{v[0], v[1]};
      p[kWave + l] = double2{v[2], v[3]};
      p[2 * kWave + l] = pv;
    } else {
      reinterpret_cast<float4 *>(blk + kWave * 16)[l] = float4{v[0], v[1], v[2], v[3]};
      reinterpret_cast<double2 *>(blk + kWave * 32)[l] = pv;
    }
  }
}

int *sf_state() {  // [unused, error flag, unused, unused]
  static DevBufPtr buf;
  if (!buf) {
    buf = dev_alloc(4 * sizeof(int));
    if (buf) {
      LAP_HIP(hipMemsetAsync(buf->p, 0, 4 * sizeof(int), stream()));
      sync();
    }
  }
  return buf ? buf->as<int>() : nullptr;
}

using Key = std::tuple<const int *, const int *, int, int, bool>;
std::map<Key, std::unique_ptr<TriPlan>> g_plans;

}  // namespace

void release_tri_plans() { g_plans.clear(); }
void forget_tri_plans(const void *p) {
  for (auto it = g_plans.begin(); it != g_plans.end();) {
    if (std::get<0>(it->first) == p || std::get<1>(it->first) == p)
      it = g_plans.erase(it);
    else
      ++it;
  }
}

// ------------------------------------------------ chunked schedule (host)
//
// A partition of the rows into at most kFlPerCu kFlTeam chunks per CU is chosen among
// a few candidates by simulating the pipeline: every step of a chunk costs
// one unit, a value from another chunk of the workgroup kSibCost more, one
// from another workgroup kHopCost more (it goes through memory).  Candidates:
// contiguous ranges in solve order, and for matrices whose column offsets
// take few values (grids in lexicographic order) tiles over two of the offset
// strides, which keep the long dependency chains inside one chunk (e.g. the
// 256^3 grid's chains along z: 8 x 8 x 256 tiles, whose levels fill a step of
// 64 rows, 2 x 2 tiles to a workgroup).
constexpr int kHopCost = 18;
constexpr int kSibCost = 1;

// f(t0, t1) over contiguous ranges covering [0, n), one per host thread.
template <class F>
static void host_ranges(int n, F f, int grain = 65536) {
  const int T = std::max(1, std::min(host_threads(), n / grain + 1));
  std::vector<std::thread> th;
  for (int k = 1; k < T; ++k)
    th.emplace_back(f, (int)((long)n * k / T), (int)((long)n * (k + 1) / T));
  f(0, (int)((long)n / T));
  for (std::thread &t : th) t.join();
}

struct ChunkSched {
  int G = 0;  // chunks, a multiple of kFlTeam; kFlTeam consecutive ones share a workgroup
  std::vector<int> cstep;        // first step of each chunk (+ end), multiples of kFlGroup
  std::vector<int> crow, cmap;   // row and level-order position of each record, -1: padding
  std::vector<int> pos;          // record of each row (64 * step + lane)
  std::vector<int> slev;         // level of each step, kFlPadLevel: padding
  std::vector<int> owner;        // chunk of each step
  long long cost = -1;
  // How step k of chunk c gets the result of step kd: 0 through c's inbox, 1
  // from its own ring, 2 from the ring of another chunk of the workgroup.  The
  // step that overwrites kd's ring entries waits for step k (see need below);
  // that step has a higher level than k here, so all waits, like the
  // dependencies, lead from lower to higher levels and none can close a cycle.
  int how(int c, int k, int kd) const {
    const int cd = owner[(size_t)kd];
    if (cd == c) return k - kd < kFlRing ? 1 : 0;
    if (cd / kFlTeam != c / kFlTeam) return 0;
    const int over = kd + kFlRing;
    return over >= cstep[(size_t)cd + 1] || slev[(size_t)k] < slev[(size_t)over] ? 2 : 0;
  }
};
constexpr int kFlPadLevel = 0x7fffffff;

// The steps of a partition (each chunk's rows level by level, at most 64 rows
// a step) and its simulated length; false when padding would more than
// quadruple the records.
static bool sched_build(ChunkSched &S, const std::vector<int> &chunk_of, int G,
                        const std::vector<int> &ia, const std::vector<int> &ja,
                        const std::vector<int> &level, const std::vector<int> &order) {
  const int n = (int)chunk_of.size();
  S.G = G;
  std::vector<int> cbase((size_t)G + 1, 0);
  for (int i = 0; i < n; ++i) cbase[(size_t)chunk_of[(size_t)i] + 1]++;
  for (int c = 0; c < G; ++c) cbase[(size_t)c + 1] += cbase[(size_t)c];
  std::vector<int> at((size_t)n);  // level-order positions by (chunk, level, row)
  {
    std::vector<int> fill(cbase.begin(), cbase.end() - 1);
    for (int t = 0; t < n; ++t)
      at[(size_t)fill[(size_t)chunk_of[(size_t)order[(size_t)t]]]++] = t;
  }
  const long long most = 4ll * n + 65536;
  S.cstep.assign((size_t)G + 1, 0);
  S.slev.clear();
  S.crow.clear();
  S.cmap.clear();
  S.crow.reserve((size_t)n + (size_t)n / 8);
  S.cmap.reserve((size_t)n + (size_t)n / 8);
  S.pos.assign((size_t)n, 0);
  auto pad = [&](int upto) {
    S.crow.resize((size_t)upto, -1);
    S.cmap.resize((size_t)upto, -1);
  };
  for (int c = 0; c < G; ++c) {
    S.cstep[(size_t)c] = (int)S.slev.size();
    for (int t = cbase[(size_t)c]; t < cbase[(size_t)c + 1];) {
      const int lv = level[(size_t)order[(size_t)at[(size_t)t]]];
      const int p0 = (int)S.slev.size() * kWave;
      int l = 0;
      for (; l < kWave && t < cbase[(size_t)c + 1]; ++l, ++t) {
        const int m = at[(size_t)t], i = order[(size_t)m];
        if (level[(size_t)i] != lv) break;
        S.crow.push_back(i);
        S.cmap.push_back(m);
        S.pos[(size_t)i] = p0 + l;
      }
      S.slev.push_back(lv);
      pad(p0 + kWave);
    }
    while (S.slev.size() % kFlGroup) {
      S.slev.push_back(kFlPadLevel);
      pad((int)S.slev.size() * kWave);
    }
    if ((long long)S.crow.size() > most ||
        (int)S.slev.size() - S.cstep[(size_t)c] > kFlMaxSteps)
      return false;
  }
  const int nsteps = (int)S.slev.size();
  S.cstep[(size_t)G] = nsteps;
  S.owner.resize((size_t)nsteps);
  for (int c = 0; c < G; ++c)
    for (int k = S.cstep[(size_t)c]; k < S.cstep[(size_t)c + 1]; ++k) S.owner[(size_t)k] = c;
  // pipeline simulation, steps taken in level order (a dependency has a lower
  // level, so its step is already timed)
  int nlev = 0;
  for (int v : S.slev)
    if (v != kFlPadLevel) nlev = std::max(nlev, v + 1);
  std::vector<int> lcnt((size_t)nlev + 1, 0), byl;
  int real = 0;
  for (int v : S.slev)
    if (v != kFlPadLevel) lcnt[(size_t)v + 1]++, ++real;
  for (int l = 0; l < nlev; ++l) lcnt[(size_t)l + 1] += lcnt[(size_t)l];
  byl.resize((size_t)real);
  for (int k = 0; k < nsteps; ++k)
    if (S.slev[(size_t)k] != kFlPadLevel) byl[(size_t)lcnt[(size_t)S.slev[(size_t)k]]++] = k;
  std::vector<int> tdone((size_t)nsteps, 0);
  const int extra[3] = {kHopCost, 0, kSibCost};
  int cost = 0;
  for (int k : byl) {
    const int c = S.owner[(size_t)k];
    int t0 = k > S.cstep[(size_t)c] ? tdone[(size_t)k - 1] : 0;
    for (int l = 0; l < kWave; ++l) {
      const int i = S.crow[(size_t)k * kWave + l];
      if (i < 0) break;
      for (int e = ia[i]; e < ia[i + 1]; ++e) {
        if (ja[e] == i) continue;
        const int kd = S.pos[(size_t)ja[e]] / kWave;
        t0 = std::max(t0, tdone[(size_t)kd] + extra[S.how(c, k, kd)]);
      }
    }
    tdone[(size_t)k] = t0 + 1;
    cost = std::max(cost, t0 + 1);
  }
  S.cost = cost;
  return true;
}

// The chunked schedule of a triangle whose rows hold at most 4 entries beside
// the pivot (a record's dependencies).
static void tri_chunks_build(TriPlan &p, const std::vector<int> &ia, const std::vector<int> &ja,
                             const std::vector<int> &level, const std::vector<int> &order) {
  const int n = p.n;
  if (n <= 0 || p.max_row > 5 || !p.has_diag || !sf_state()) return;
  const int Gmax = std::max(1, device_cus() * kFlPerCu) * kFlTeam;
  const bool lower = p.lower;
  auto pos_of = [&](int i) { return lower ? i : n - 1 - i; };
  // candidate partitions: {chunk rows of a contiguous range} or {strides and
  // tile of a tiling}
  struct Cand {
    int C = 0, Oa = 0, nb = 0, Ti = 0, Tj = 0, gi = 0, gj = 0;
    int wi = 1, wj = 1, hi = 0, hj = 0;
    long est = 0;
  };
  std::vector<Cand> tiles, cands;
  std::vector<int> offs;
  for (int i = 0; i < n && offs.size() <= 16; ++i)
    for (int e = ia[i]; e < ia[i + 1]; ++e) {
      const int d = ja[e];
      if (d == i) continue;
      const int o = std::abs(i - d);
      if (std::find(offs.begin(), offs.end(), o) == offs.end()) offs.push_back(o);
    }
  int line = 0;  // the longest offset that divides n: ranges aligned to it
  if (offs.size() <= 16) {
    std::sort(offs.begin(), offs.end());
    for (size_t x = 0; x < offs.size(); ++x) {
      if (offs[x] >= 2 && n % offs[x] == 0) line = offs[x];
      for (size_t y = x + 1; y < offs.size(); ++y) {
        const int Oa = offs[x], Ob = offs[y];
        if (Oa < 2 || Ob % Oa || n % Ob) continue;
        const int nb = Ob / Oa;  // extent of the second coordinate
        for (int Ti = 2; Ti <= 64; Ti *= 2)
          for (int Tj = 2; Tj <= 64; Tj *= 2) {
            Cand t;
            t.Oa = Oa;
            t.nb = nb;
            t.Ti = std::min(Ti, Oa);
            t.Tj = std::min(Tj, nb);
            t.gi = (Oa + t.Ti - 1) / t.Ti;
            t.gj = (nb + t.Tj - 1) / t.Tj;
            if ((Ti > 2 * Oa) || (Tj > 2 * nb)) continue;
            const long sub = ((long)t.Ti * t.Tj + kWave - 1) / kWave;
            for (int wi = 1; wi <= kFlTeam; wi *= 2) {  // tiles of a workgroup
              t.wi = wi;
              t.wj = kFlTeam / wi;
              t.hi = (t.gi + t.wi - 1) / t.wi;
              t.hj = (t.gj + t.wj - 1) / t.wj;
              if ((long)t.hi * t.hj * kFlTeam > Gmax) continue;
              t.est = (Oa + nb + n / Ob) * sub + (long)(t.hi + t.hj - 2) * kHopCost +
                      (long)(t.gi - t.hi + t.gj - t.hj) * kSibCost;
              tiles.push_back(t);
            }
          }
      }
    }
  }
  std::stable_sort(tiles.begin(), tiles.end(),
                   [](const Cand &u, const Cand &v) { return u.est < v.est; });
  if (tiles.size() > 3) tiles.resize(3);
  auto ranges = [&](long C) {
    C = std::max(1l, std::min(C, (long)n));
    if ((n + C - 1) / C > Gmax) return;
    for (const Cand &o : cands)
      if (o.C == (int)C) return;
    Cand t;
    t.C = (int)C;
    cands.push_back(t);
  };
  auto round64 = [](long v) { return (v + 63) / 64 * 64; };
  ranges(round64((n + Gmax - 1) / Gmax));
  if (tiles.empty()) {
    for (int G = Gmax / 4; G >= 1; G /= 4) ranges(round64((n + G - 1) / G));
    if (line)
      for (long q = 16; q <= 64; q *= 2) ranges(q * line);
    const size_t most = n > 2000000 ? 3 : 8;
    if (cands.size() > most) cands.resize(most);
  }
  cands.insert(cands.end(), tiles.begin(), tiles.end());
  auto chunk_fn = [&](const Cand &t, std::vector<int> &co) {
    co.resize((size_t)n);
    for (int r = 0; r < n; ++r) {
      const int ps = pos_of(r);
      if (t.C) {
        co[(size_t)r] = ps / t.C;
        continue;
      }
      const int ti = (ps % t.Oa) / t.Ti, tj = (ps / t.Oa) % t.nb / t.Tj;
      co[(size_t)r] = ((tj / t.wj) * t.hi + ti / t.wi) * kFlTeam + tj % t.wj * t.wi + ti % t.wi;
    }
  };
  auto chunks_of = [&](const Cand &t) {
    return t.C ? ((n + t.C - 1) / t.C + kFlTeam - 1) / kFlTeam * kFlTeam
               : t.hi * t.hj * kFlTeam;
  };
  // the candidates are independent: one host thread each (the lowest cost
  // wins, ties to the earlier candidate, so the choice does not depend on
  // thread timing)
  std::vector<ChunkSched> built(cands.size());
  {
    std::atomic<size_t> next{0};
    auto work = [&]() {
      std::vector<int> co;
      for (size_t ci; (ci = next.fetch_add(1)) < cands.size();) {
        chunk_fn(cands[ci], co);
        if (!sched_build(built[ci], co, chunks_of(cands[ci]), ia, ja, level, order))
          built[ci] = ChunkSched();
      }
    };
    const int T = std::max(1, std::min(host_threads(), (int)cands.size()));
    std::vector<std::thread> th;
    for (int t = 1; t < T; ++t) th.emplace_back(work);
    work();
    for (std::thread &t : th) t.join();
  }
  size_t best_i = 0;
  for (size_t ci = 0; ci < cands.size(); ++ci)
    if (built[ci].cost >= 0 && (built[best_i].cost < 0 || built[ci].cost < built[best_i].cost))
      best_i = ci;
  if (cands.empty() || built[best_i].cost < 0) return;
  ChunkSched best = std::move(built[best_i]);
  built.clear();
  const int G = best.G, nsteps = (int)best.slev.size();
  // LDS entries of the dependencies: results in a ring of the workgroup are
  // read there, any other one comes through the chunk's inbox, one entry per
  // use, in the order the steps use them
  std::vector<int> hcnt((size_t)G + 1, 0);
  auto in_ring = [&](int c, int k, int d) {
    return best.how(c, k, best.pos[(size_t)d] / kWave) != 0;
  };
  host_ranges(G, [&](int c0, int c1) {
    for (int c = c0; c < c1; ++c) {
      int h = 0;
      for (int k = best.cstep[(size_t)c]; k < best.cstep[(size_t)c + 1]; ++k)
        for (int l = 0; l < kWave; ++l) {
          const int i = best.crow[(size_t)k * kWave + l];
          if (i < 0) break;
          for (int e = ia[i]; e < ia[i + 1]; ++e)
            if (ja[e] != i && !in_ring(c, k, ja[e])) ++h;
        }
      hcnt[(size_t)c + 1] = h;
    }
  }, 8);
  long long total = 0;
  for (int c = 0; c < G; ++c) total += hcnt[(size_t)c + 1];
  if (total > 0x7fffffell) return;  // the inbox stays below 2^31 bytes
  for (int c = 0; c < G; ++c) hcnt[(size_t)c + 1] += hcnt[(size_t)c];
  const size_t T = (size_t)nsteps * kWave;
  std::vector<unsigned> code(2 * T);
  std::vector<int> need(2 * (size_t)nsteps, 0), src((size_t)total);  // src: feeds an entry
  host_ranges(G, [&](int c0, int c1) {
    for (int c = c0; c < c1; ++c) {
      int h = 0;
      for (int k = best.cstep[(size_t)c]; k < best.cstep[(size_t)c + 1]; ++k) {
        for (int l = 0; l < kWave; ++l) {
          const size_t t = (size_t)k * kWave + l;
          unsigned cd[4] = {kFlZero, kFlZero, kFlZero, kFlZero};
          const int i = best.crow[t];
          if (i >= 0) {
            int j = 0;
            for (int e = ia[i]; e < ia[i + 1]; ++e) {
              const int d = ja[e];
              if (d == i) continue;
              const int pd = best.pos[(size_t)d];
              const int kd = pd / kWave, oc = best.owner[(size_t)kd];
              if (in_ring(c, k, d)) {
                cd[j++] = (unsigned)(oc % kFlTeam * kFlLds +
                                     (kd - best.cstep[(size_t)oc]) % kFlRing * kWave + pd % kWave);
                if (oc != c) {
                  int &nd = need[2 * (size_t)k + 1];
                  nd = std::max(nd, kd - best.cstep[(size_t)oc] + 1);
                }
              } else {
                src[(size_t)hcnt[(size_t)c] + h] = pd;
                cd[j++] = (unsigned)(c % kFlTeam * kFlLds + kFlRing * kWave + h % kFlHalo);
                ++h;
              }
            }
          }
          code[2 * t] = cd[0] | cd[1] << 16;
          code[2 * t + 1] = cd[2] | cd[3] << 16;
        }
        need[2 * (size_t)k] = h;
      }
    }
  }, 8);
  // a step that overwrites ring entries waits for their readers in the
  // workgroup's other chunks (one host thread per workgroup: its chunks only)
  host_ranges(G / kFlTeam, [&](int w0, int w1) {
    for (int c = w0 * kFlTeam; c < w1 * kFlTeam; ++c)
      for (int k = best.cstep[(size_t)c]; k < best.cstep[(size_t)c + 1]; ++k)
        for (int l = 0; l < kWave; ++l) {
          const int i = best.crow[(size_t)k * kWave + l];
          if (i < 0) break;
          for (int e = ia[i]; e < ia[i + 1]; ++e) {
            const int kd = best.pos[(size_t)ja[e]] / kWave, oc = best.owner[(size_t)kd];
            if (oc == c || best.how(c, k, kd) != 2) continue;
            const int over = kd + kFlRing;
            if (over >= best.cstep[(size_t)oc + 1]) continue;
            int &nd = need[2 * (size_t)over + 1];
            nd = std::max(nd, k - best.cstep[(size_t)c] + 1);
          }
        }
  }, 8);
  // exports by producing record: a chunk's are consecutive and in the order
  // its steps make them
  std::vector<int> first((size_t)nsteps + 1, 0), ebase((size_t)G + 1, 0);
  for (int t : src) first[(size_t)(t / kWave) + 1]++;
  for (int k = 0; k < nsteps; ++k) first[(size_t)k + 1] += first[(size_t)k];
  for (int c = 0; c <= G; ++c) ebase[(size_t)c] = first[(size_t)best.cstep[(size_t)c]];
  std::vector<int> exps(2 * (size_t)total + 2, 0);
  {
    std::vector<int> fill(first.begin(), first.end() - 1);
    for (size_t h = 0; h < src.size(); ++h) {
      const int k = src[h] / kWave, s = fill[(size_t)k]++;
      exps[2 * (size_t)s] = src[h] - best.cstep[(size_t)best.owner[(size_t)k]] * kWave;
      exps[2 * (size_t)s + 1] = (int)h;
    }
  }
  TriPlan::Chunks &ch = p.ch;
  ch.inbox = dev_alloc(16 * ((size_t)total + 1));
  ch.epoch = dev_alloc(16);
  if (!ch.inbox->p || !ch.epoch->p) return;
  LAP_HIP(hipMemsetAsync(ch.inbox->p, 0, 16 * ((size_t)total + 1), stream()));
  LAP_HIP(hipMemsetAsync(ch.epoch->p, 0, 16, stream()));
  std::vector<int> lstep((size_t)nsteps);
  for (int k = 0; k < nsteps; ++k)
    lstep[(size_t)k] = k - best.cstep[(size_t)best.owner[(size_t)k]];
  ch.cstep = dev_upload(best.cstep);
  ch.crow = dev_upload(best.crow);
  ch.cmap = dev_upload(best.cmap);
  ch.code = dev_upload(code);
  ch.need = dev_upload(need);
  ch.lstep = dev_upload(lstep);
  ch.pos = dev_upload(best.pos);
  ch.hbase = dev_upload(hcnt);
  ch.ebase = dev_upload(ebase);
  ch.exps = dev_upload(exps);
  for (const DevBufPtr &b : {ch.cstep, ch.crow, ch.cmap, ch.code, ch.need, ch.lstep, ch.pos, ch.hbase, ch.ebase,
                             ch.exps})
    if (!b->p) return;
  ch.nrec = (int)T;
  ch.nchunks = G;
  ch.cost = best.cost;
  if (getenv("LAP_SCHED_LOG"))
    fprintf(stderr, "[lapgfx] %s triangle n=%d: chunked schedule %zu of %zu, %d chunks, %d steps, "
            "%lld values between chunks, simulated length %lld (one launch per level: %d)\n",
            lower ? "lower" : "upper", n, best_i, cands.size(), G, nsteps, total, best.cost,
            p.nlevels);
}

// Host-side level analysis of a triangular CSR pattern.
std::unique_ptr<TriPlan> tri_analyse_host(int n, const std::vector<int> &ia,
                                        const std::vector<int> &ja, bool lower) {
  auto p = std::make_unique<TriPlan>();
  p->n = n;
  p->nnz = n ? ia[n] : 0;
  p->lower = lower;
  std::vector<int> level((size_t)n, 0);
  int nlev = 0;
  bool has_diag = true;
  for (int s = 0; s < n; ++s) {
    const int i = lower ? s : n - 1 - s;
    int lv = 0;
    bool diag = false;
    for (int e = ia[i]; e < ia[i + 1]; ++e) {
      const int c = ja[e];
      if (c < 0 || c >= n) {
        set_error(LAP_ERR_STRUCT, "triangular solve: column %d out of range in row %d", c, i);
        return nullptr;
      }
      if (c == i) {
        diag = true;
        continue;
      }
      if ((lower && c > i) || (!lower && c < i)) {
        set_error(LAP_ERR_STRUCT, "%s triangular solve: entry (%d,%d) on the wrong side",
                  lower ? "lower" : "upper", i, c);
        return nullptr;
      }
      lv = std::max(lv, level[c] + 1);
    }
    has_diag = has_diag && diag;
    level[i] = lv;
    nlev = std::max(nlev, lv + 1);
  }
  if (n == 0) nlev = 0;
  p->nlevels = nlev;
  p->has_diag = has_diag;
  p->level_ptr.assign((size_t)nlev + 1, 0);
  for (int i = 0; i < n; ++i) p->level_ptr[level[i] + 1]++;
  for (int l = 0; l < nlev; ++l) p->level_ptr[l + 1] += p->level_ptr[l];
  // within a level: the rows of at most kTriLongRow entries, then the rest,
  // each in row order
  std::vector<int> nshort((size_t)nlev, 0);
  for (int i = 0; i < n; ++i)
    if (ia[i + 1] - ia[i] <= kTriLongRow) nshort[level[i]]++;
  p->level_long.resize((size_t)nlev);
  std::vector<int> fill(p->level_ptr.begin(), p->level_ptr.end() - 1), fill_long((size_t)nlev),
      order((size_t)n);
  for (int l = 0; l < nlev; ++l) fill_long[l] = p->level_long[l] = p->level_ptr[l] + nshort[l];
  for (int i = 0; i < n; ++i) {
    if (ia[i + 1] - ia[i] <= kTriLongRow)
      order[fill[level[i]]++] = i;
    else
      order[fill_long[level[i]]++] = i;
  }
  for (int l = 0; l < nlev; ++l)
    p->max_level_rows = std::max(p->max_level_rows, p->level_ptr[l + 1] - p->level_ptr[l]);
  for (int i = 0; i < n; ++i) p->max_row = std::max(p->max_row, ia[i + 1] - ia[i]);
  p->order = dev_upload(order);
  std::vector<int> desc((size_t)n * 4);
  for (int t = 0; t < n; ++t) {
    const int i = order[(size_t)t];
    int piv = -1;  // the last diagonal entry, as the sequential loop keeps
    for (int e = ia[i]; e < ia[i + 1]; ++e)
      if (ja[e] == i) piv = e;
    desc[(size_t)t * 4] = i;
    desc[(size_t)t * 4 + 1] = ia[i];
    desc[(size_t)t * 4 + 2] = ia[i + 1];
    desc[(size_t)t * 4 + 3] = piv;
  }
  p->desc = dev_upload(desc);
  // segments of the long rows (tree-summed level launches)
  std::vector<int> segd;
  p->level_seg.assign((size_t)nlev + 1, 0);
  for (int l = 0; l < nlev; ++l) {
    for (int t = p->level_long[l]; t < p->level_ptr[l + 1]; ++t) {
      const int i = order[(size_t)t];
      const int ns = (ia[i + 1] - ia[i] + kTriSeg - 1) / kTriSeg;
      const int slot = (int)(segd.size() / 4);
      for (int g = 0; g < ns; ++g)
        segd.insert(segd.end(), {t - p->level_ptr[l], g, ns, slot});
    }
    p->level_seg[(size_t)l + 1] = (int)(segd.size() / 4);
  }
  const size_t nseg = segd.size() / 4;
  p->segd = dev_upload(segd);
  p->seg_part = dev_alloc(sizeof(double) * (nseg + 1));
  p->seg_tick = dev_upload(std::vector<int>(nseg + 1, 0));
  tri_chunks_build(*p, ia, ja, level, order);
  return p;
}

// The analysis of a device pattern (not cached).
static std::unique_ptr<TriPlan> tri_plan_make(int n, int nnz, const int *ia, const int *ja,
                                              bool lower) {
  if (n < 0 || nnz < 0) {
    set_error(LAP_ERR_ARG, "triangular solve: negative size");
    return nullptr;
  }
  std::vector<int> h_ia = dev_download(ia, (size_t)n + 1);
  const int total = n ? h_ia[n] : 0;
  if (n && (h_ia[0] != 0 || total < 0 || total > nnz)) {
    set_error(LAP_ERR_STRUCT, "triangular solve: row pointers inconsistent with nnz=%d", nnz);
    return nullptr;
  }
  std::vector<int> h_ja = dev_download(ja, (size_t)total);
  return tri_analyse_host(n, h_ia, h_ja, lower);
}

const TriPlan *tri_plan(int n, int nnz, const int *ia, const int *ja, bool lower) {
  Key key{ia, ja, n, nnz, lower};
  auto it = g_plans.find(key);
  if (it != g_plans.end()) return it->second.get();
  auto plan = tri_plan_make(n, nnz, ia, ja, lower);
  if (!plan) return nullptr;
  TriPlan *raw = plan.get();
  g_plans[key] = std::move(plan);
  return raw;
}

std::pair<std::unique_ptr<TriPlan>, std::unique_ptr<TriPlan>> tri_analyse_pair(
    int n, const std::vector<int> &lia, const std::vector<int> &lja,
    const std::vector<int> &uia, const std::vector<int> &uja) {
  // the shared device buffers are allocated lazily: before the threads
  sf_state();
  std::unique_ptr<TriPlan> up;
  std::thread tu([&] { up = tri_analyse_host(n, uia, uja, false); });
  auto lp = tri_analyse_host(n, lia, lja, true);
  tu.join();
  return {std::move(lp), std::move(up)};
}

void tri_plan_pair(int n, int nnzL, const int *lia, const int *lja, int nnzU, const int *uia,
                   const int *uja) {
  const Key kl{lia, lja, n, nnzL, true}, ku{uia, uja, n, nnzU, false};
  const bool need_l = !g_plans.count(kl), need_u = !g_plans.count(ku);
  if (!need_l || !need_u) {  // one (or none) to build
    tri_plan(n, nnzL, lia, lja, true);
    tri_plan(n, nnzU, uia, uja, false);
    return;
  }
  sf_state();
  std::unique_ptr<TriPlan> up;
  std::thread tu([&] { up = tri_plan_make(n, nnzU, uia, uja, false); });
  auto lp = tri_plan_make(n, nnzL, lia, lja, true);
  tu.join();
  if (lp) g_plans[kl] = std::move(lp);
  if (up) g_plans[ku] = std::move(up);
}

int tri_error() {
  int *st = sf_state();
  if (!st) return 0;
  int h = 0;
  LAP_HIP(hipMemcpy(&h, st + 1, sizeof(int), hipMemcpyDeviceToHost));
  return h;
}

void tri_clear_error() {
  int *st = sf_state();
  if (st) LAP_HIP(hipMemsetAsync(st, 0, 4 * sizeof(int), stream()));
}

// The chunked schedule's records for one set of values, and its right-hand
// side buffer, each with kFlGroup steps of room past the end.  false: there is no
// memory for them (the solve goes by levels).
template <class AT, class VT>
static bool tri_fl_pack(const TriPlan &p, const int *ja, const AT *a, DevBufPtr &rec,
                        DevBufPtr &xc) {
  const size_t steps = (size_t)p.ch.nrec / kWave + kFlGroup;
  const size_t rb = steps * FlRec<AT>::bytes, xb = steps * kWave * sizeof(VT);
  if (!rec || rec->bytes < rb) rec = dev_try(rb);
  if (!xc || xc->bytes < xb) xc = dev_try(xb);
  if (!rec || !xc) return false;
  const unsigned g = grid_for((size_t)p.ch.nrec, 1, kBlock, 65536);
  k_fl_pack<AT, VT><<<g, kBlock, 0, stream()>>>(
      p.ch.nrec, p.ch.cmap->as<int>(), p.desc->as<int4>(), ja, a, p.ch.code->as<int2>(),
      p.ch.need->as<int2>(), p.ch.lstep->as<int>(), rec->as<char>(), xc->as<VT>());
  return true;
}

// One solve over the chunks: the right-hand sides x[map[t]] (x in row order
// and map = crow, or another schedule's results and the composed map) into
// schedule order, then the chunks, which leave the results there.
template <class AT, class VT>
static void tri_fl_launch(const TriPlan &p, const DevBufPtr &rec, const DevBufPtr &xc,
                          const VT *x, const int *map, const int *done) {
  const TriPlan::Chunks &ch = p.ch;
  const unsigned g = std::min(2048u, 8u * ((unsigned)ch.nrec / (8u * kBlock) + 1u));
  k_fl_gather<VT><<<g, kBlock, 0, stream()>>>(ch.nrec, map, x, xc->as<VT>(),
                                              ch.epoch->as<unsigned>(), done);
  k_tri_flow<AT, VT><<<ch.nchunks / kFlTeam, 4 * kFlTeam * kWave, 0, stream()>>>(
      ch.cstep->as<int>(), rec->as<char>(), xc->as<VT>(), ch.hbase->as<int>(),
      ch.ebase->as<int>(), ch.exps->as<int2>(), ch.inbox->p, (int)ch.inbox->bytes,
      ch.epoch->as<unsigned>(), sf_state(), done);
}
template <class VT>
static void tri_fl_spread(const TriPlan &p, const DevBufPtr &xc, VT *y, const int *done) {
  const unsigned g = std::min(2048u, 8u * ((unsigned)p.n / (8u * kBlock) + 1u));
  k_fl_spread<VT><<<g, kBlock, 0, stream()>>>(p.n, p.ch.pos->as<int>(), xc->as<VT>(), y, done);
}

static void tri_fl_tail(const TriPlan &p, const DevBufPtr &xc, double *y, const TriTail &t,
                        const int *done) {
  auto *k = t.add ? k_fl_tail<true> : k_fl_tail<false>;
  k<<<t.grid, kBlock, 0, stream()>>>(p.n, p.ch.pos->as<int>(), xc->as<double>(), y, t.r, t.part,
                                     t.grid % 8 ? 1 : (int)t.grid / 8, done);
}

static void tri_choose(const TriPlan &p, const TriEll &e);

void tri_ell_build(const TriPlan &p, const int *ja, const double *a, TriEll &e) {
  e.w = 0;
  if (p.n <= 0 || p.max_row > 8) return;
  const int w = p.max_row <= 4 ? 4 : 8;
  e.ja = dev_try(sizeof(int) * (size_t)p.n * w);
  e.a = dev_try(sizeof(double) * (size_t)p.n * w);
  if (!e.ja || !e.a) return;
  const unsigned g = grid_for((size_t)p.n, 1, kBlock, 65536);
  if (w == 4)
    k_ell_pack<4><<<g, kBlock, 0, stream()>>>(p.n, p.desc->as<int4>(), ja, a, e.ja->as<int>(),
                                              e.a->as<double>());
  else
    k_ell_pack<8><<<g, kBlock, 0, stream()>>>(p.n, p.desc->as<int4>(), ja, a, e.ja->as<int>(),
                                              e.a->as<double>());
  e.w = w;
  if (p.ch.nchunks > 0 && tri_fl_pack<double, double>(p, ja, a, e.crec, e.xc)) tri_choose(p, e);
}

void tri_ch_pack32(const TriPlan &p, const int *ja, const float *a, TriChunks32 &c) {
  c.ok = p.n > 0 && p.ch.nchunks > 0 && tri_fl_pack<float, float>(p, ja, a, c.rec, c.xc);
}

// One launch per level: a lane per short row, then a workgroup per long row
// (sequential order) or per long-row segment (option sptrsv_long 1).
template <class AT, class VT>
static void tri_level_launch(const TriPlan &p, const int *ja, const AT *a, const double *diag,
                             const VT *x, VT *y, const int *done) {
  const int4 *desc = p.desc->as<int4>();
  const bool tree = options().sptrsv_long == 1;
  const int4 *segd = p.segd->as<int4>();
  double *part = p.seg_part->as<double>();
  int *tick = p.seg_tick->as<int>();
  for (int l = 0; l < p.nlevels; ++l) {
    const int cnt = p.level_long[l] - p.level_ptr[l];
    const int nlong = tree ? p.level_seg[(size_t)l + 1] - p.level_seg[(size_t)l]
                           : p.level_ptr[l + 1] - p.level_long[l];
    const unsigned g = (unsigned)((cnt + kBlock - 1) / kBlock + nlong);
    if (tree)
      k_tri_level<AT, VT, true><<<g, kBlock, 0, stream()>>>(cnt, nlong, desc + p.level_ptr[l],
                                                            ja, a, diag, x, y, done,
                                                            segd + p.level_seg[(size_t)l], part,
                                                            tick);
    else
      k_tri_level<AT, VT><<<g, kBlock, 0, stream()>>>(cnt, nlong, desc + p.level_ptr[l], ja, a,
                                                      diag, x, y, done, nullptr, nullptr,
                                                      nullptr);
  }
}

// One launch per level over the packed rows.
static void tri_ell_launch(const TriPlan &p, const TriEll &ell, const double *diag,
                           const double *x, double *y, const int *done) {
  const int *order = p.order->as<int>();
  for (int l = 0; l < p.nlevels; ++l) {
    const int l0 = p.level_ptr[l], cnt = p.level_ptr[l + 1] - l0;
    const unsigned g = (unsigned)((cnt + kBlock - 1) / kBlock);
    const size_t off = (size_t)l0 * ell.w;
    if (ell.w == 4)
      k_tri_level_ell<4><<<g, kBlock, 0, stream()>>>(cnt, order + l0, ell.ja->as<int>() + off,
                                                     ell.a->as<double>() + off, diag, x, y, done);
    else
      k_tri_level_ell<8><<<g, kBlock, 0, stream()>>>(cnt, order + l0, ell.ja->as<int>() + off,
                                                     ell.a->as<double>() + off, diag, x, y, done);
  }
}

// Which path tri_solve_launch takes.
enum TriPath { TRI_CHUNKS, TRI_LEVELS_ELL, TRI_LEVELS };

// Whether the option asks for chunks: 4, or 3 and they are not known to be slower.
static bool tri_mode_chunks(const TriPlan &p) {
  const int mode = options().sptrsv_mode;
  return mode == 4 || (mode == 3 && p.ch.taken != 0);
}

static TriPath tri_path(const TriPlan &p, const TriEll *ell, bool in_place) {
  if (tri_mode_chunks(p) && ell && ell->w && ell->crec && ell->xc && p.ch.nchunks > 0 &&
      sf_state())
    return TRI_CHUNKS;
  (void)in_place;  // the chunked kernel reads x from its own gathered copy
  if (ell && ell->w) return TRI_LEVELS_ELL;
  return TRI_LEVELS;
}

int tri_launches(const TriPlan &p, const TriEll *ell, bool in_place) {
  switch (tri_path(p, ell, in_place)) {
    case TRI_CHUNKS: return 3;
    default: return p.nlevels;
  }
}

void tri_solve_launch(const TriPlan &p, const int *ia, const int *ja, const double *a,
                      const double *diag, const double *x, double *y, const int *done,
                      const TriEll *ell) {
  (void)ia;  // the plan's descriptors carry every row's range
  const TriPath path = tri_path(p, ell, x == y);
  if (path == TRI_CHUNKS) {
    tri_fl_launch<double, double>(p, ell->crec, ell->xc, x, p.ch.crow->as<int>(), done);
    tri_fl_spread(p, ell->xc, y, done);
    return;
  }
  if (path == TRI_LEVELS_ELL) return tri_ell_launch(p, *ell, diag, x, y, done);
  tri_level_launch<double, double>(p, ja, a, diag, x, y, done);
}

// Chunks or a launch per level, found out at a triangle's first values: both give
// the same bits.  A triangle of wide levels without locality (nodes in random
// order, far neighbours) has few levels, and chunks that wait for each other at
// every step.  us per IC0 PCG iteration, chunks and levels: shuffled 100^2 grid (11
// levels, simulated length 137) 247 and 102, 200^2 (13, 216) 101 and 125, 1200^2
// (17, 345) 524 and 408, circulant of 500,000 rows with neighbours 23,000 and 70,000
// away (22, 554) 351 and 201.  The simulated length does not tell these apart, so
// where it is kTriSure times the levels or more the two are timed, once per plan;
// below (grids: 1 to 2) a level costs its launch, 1.8 to 3 us, against 0.2 us a
// step.  Up to 3 levels are no more launches than the chunks' three (100,000 rows
// of one entry 85 and 61).  In a solve the chunks save some 4 us more, which the
// timing does not see: two solves in a row skip a copy, the last copy does the axpy
// or the dot product (circulant of 50,000 rows with neighbours 2300 and 7000 away,
// 53 us either way alone, 134 and 170 an iteration).
constexpr int kTriSure = 4, kTriFew = 3, kTriTimed = 8192;
constexpr float kTriSaved = 4.f;
static void tri_choose(const TriPlan &p, const TriEll &e) {
  if (p.ch.taken >= 0 || options().sptrsv_mode != 3) return;
  p.ch.taken = p.nlevels > kTriFew;
  if (!p.ch.taken || p.ch.cost < (long long)kTriSure * p.nlevels || p.nlevels > kTriTimed) return;
  double *x = scratch_try("tri_time_x", (size_t)p.n), *y = scratch_try("tri_time_y", (size_t)p.n);
  hipEvent_t ev[2];
  if (!x || !y || !hip_try(hipEventCreate(&ev[0]))) return;
  if (!hip_try(hipEventCreate(&ev[1]))) {
    (void)hipEventDestroy(ev[0]);
    return;
  }
  launch_fill(p.n, 1.0, x);
  const int solves = std::max(1, std::min(4, 2048 / p.nlevels));
  float ms[2] = {0.f, 0.f};  // by levels, by chunks
  bool ok = true;
  for (int chunks = 0; ok && chunks < 2; ++chunks) {
    // as the solves run them: several in a graph
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    ok = hip_try(hipStreamBeginCapture(stream(), hipStreamCaptureModeThreadLocal));
    if (ok) {
      // (the copy back to row order does what the levels leave to another launch:
      // the next solve's gather, the axpy or the dot product)
      for (int s = 0; s < solves; ++s)
        if (chunks)
          tri_fl_launch<double, double>(p, e.crec, e.xc, x, p.ch.crow->as<int>(), nullptr);
        else
          tri_ell_launch(p, e, nullptr, x, y, nullptr);
      ok = hip_try(hipStreamEndCapture(stream(), &graph));
    }
    ok = ok && hip_try(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    for (int rep = 0; ok && rep < 2; ++rep) {  // (the first one apart)
      if (rep == 1) ok = hip_try(hipEventRecord(ev[0], stream()));
      ok = ok && hip_try(hipGraphLaunch(exec, stream()));
    }
    ok = ok && hip_try(hipEventRecord(ev[1], stream())) && hip_try(hipEventSynchronize(ev[1])) &&
         hip_try(hipEventElapsedTime(&ms[chunks], ev[0], ev[1]));
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
  }
  (void)hipEventDestroy(ev[0]);
  (void)hipEventDestroy(ev[1]);
  if (ok) p.ch.taken = ms[1] <= ms[0] + 1e-3f * solves * kTriSaved;
  if (getenv("LAP_SCHED_LOG"))
    fprintf(stderr, "[lapgfx] triangle n=%d: %.1f us by chunks, %.1f us by levels\n", p.n,
            ms[1] * 1e3f / solves, ms[0] * 1e3f / solves);
  if (tri_error()) {  // a wait ran out
    tri_clear_error();
    p.ch.taken = 0;
  }
}

bool tri_solve_tail_launch(const TriPlan &p, const double *x, double *y, const TriEll &ell,
                           const TriTail &tail, const int *done) {
  if (tri_path(p, &ell, x == y) != TRI_CHUNKS) return false;
  tri_fl_launch<double, double>(p, ell.crec, ell.xc, x, p.ch.crow->as<int>(), done);
  tri_fl_tail(p, ell.xc, y, tail, done);
  return true;
}

DevBufPtr tri_compose(const TriPlan &first, const TriPlan &second) {
  if (first.ch.nchunks <= 0 || second.ch.nchunks <= 0) return nullptr;
  DevBufPtr m = dev_try(sizeof(int) * (size_t)second.ch.nrec);
  if (!m) return nullptr;
  k_fl_compose<<<grid_for((size_t)second.ch.nrec, 4, kBlock, 4096), kBlock, 0, stream()>>>(
      second.ch.nrec, second.ch.crow->as<int>(), first.ch.pos->as<int>(), m->as<int>());
  return m;
}

bool tri_solve_two_launch(const TriPlan &p1, const TriEll &e1, const TriPlan &p2,
                          const TriEll &e2, const DevBufPtr &comp, const double *x, double *y,
                          const int *done, const TriTail *tail) {
  if (!comp || tri_path(p1, &e1, false) != TRI_CHUNKS || tri_path(p2, &e2, false) != TRI_CHUNKS)
    return false;
  tri_fl_launch<double, double>(p1, e1.crec, e1.xc, x, p1.ch.crow->as<int>(), done);
  tri_fl_launch<double, double>(p2, e2.crec, e2.xc, e1.xc->as<double>(), comp->as<int>(), done);
  if (tail)
    tri_fl_tail(p2, e2.xc, y, *tail, done);
  else
    tri_fl_spread(p2, e2.xc, y, done);
  return true;
}

template <class VT>
static void tri_mixed_launch(const TriPlan &p, const int *ja, const float *a, const VT *x, VT *y,
                             const int *done) {
  tri_level_launch<float, VT>(p, ja, a, nullptr, x, y, done);
}

static bool tri_chunks32_ready(const TriPlan &p, const TriChunks32 *c) {
  return c && c->ok && tri_mode_chunks(p) && p.ch.nchunks > 0 && sf_state();
}

int tri_launches32(const TriPlan &p, const TriChunks32 *c) {
  return tri_chunks32_ready(p, c) ? 3 : p.nlevels;
}

bool tri_solve32_two_launch(const TriPlan &p1, const TriChunks32 &c1, const TriPlan &p2,
                            const TriChunks32 &c2, const DevBufPtr &comp, const float *x,
                            float *y, const int *done) {
  if (!comp || !tri_chunks32_ready(p1, &c1) || !tri_chunks32_ready(p2, &c2)) return false;
  tri_fl_launch<float, float>(p1, c1.rec, c1.xc, x, p1.ch.crow->as<int>(), done);
  tri_fl_launch<float, float>(p2, c2.rec, c2.xc, c1.xc->as<float>(), comp->as<int>(), done);
  tri_fl_spread(p2, c2.xc, y, done);
  return true;
}

void tri_solve32_launch(const TriPlan &p, const int *ja, const float *a, const float *x, float *y,
                        const int *done, const TriChunks32 *c) {
  if (tri_chunks32_ready(p, c)) {
    tri_fl_launch<float, float>(p, c->rec, c->xc, x, p.ch.crow->as<int>(), done);
    tri_fl_spread(p, c->xc, y, done);
    return;
  }
  tri_mixed_launch<float>(p, ja, a, x, y, done);
}


static void tri_entry(int n, int nnz, const int *ia, const int *ja, const double *a,
                      const double *diag, const double *x, double *y, bool lower) {
  if (n <= 0) return;
  const char *fn = lower ? "hip_lower_triangular_solve" : "hip_upper_triangular_solve";
  if (!check_device(fn, {{ia, "ia", sizeof(int) * ((size_t)n + 1)},
                         {ja, "ja", sizeof(int) * (size_t)nnz},
                         {a, "values", sizeof(double) * (size_t)nnz},
                         {x, "x", sizeof(double) * (size_t)n},
                         {y, "result", sizeof(double) * (size_t)n}}))
    return;
  const TriPlan *p = tri_plan(n, nnz, ia, ja, lower);
  if (!p) return;
  // With the pivots inside the matrix (the GPU drivers' L+D / D+U layout)
  // `diagonal` is ignored, as rocSPARSE ignores it (hip_blas.cpp:534-591);
  // the reference drivers may pass a stale host pointer there
  // (cg_driver2.c:246-248).
  const double *dg = nullptr;
  if (!p->has_diag) {
    if (!check_device(fn, {{diag, "diagonal (rows without an in-row pivot)",
                            sizeof(double) * (size_t)n}}))
      return;
    dg = diag;
  }
  tri_solve_launch(*p, ia, ja, a, dg, x, y, nullptr);
  sync();
  if (options().sptrsv_mode != 0 && tri_error()) {
    set_error(LAP_ERR_NUMERIC, "triangular solve: a dependency wait ran out (result invalid)");
    tri_clear_error();
  }
}

}  // namespace lap

using namespace lap;

extern "C" {

void initialize_and_analyze_L_and_U_solve(const int n, const int nnzL, int *lia, int *lja,
                                          double *la, const int nnzU, int *uia, int *uja,
                                          double *ua) {
  (void)la;
  (void)ua;
  if (n <= 0) return;
  if (!check_device("initialize_and_analyze_L_and_U_solve",
                    {{lia, "lia"}, {lja, "lja"}, {uia, "uia"}, {uja, "uja"}}))
    return;
  g_plans.erase(Key{lia, lja, n, nnzL, true});  // explicit analysis rebuilds
  g_plans.erase(Key{uia, uja, n, nnzU, false});
  tri_plan_pair(n, nnzL, lia, lja, nnzU, uia, uja);
}

void hip_lower_triangular_solve(const int n, const int nnzL, const int *lia, const int *lja,
                                const double *la, const double *diagonal, const double *x,
                                double *result) {
  tri_entry(n, nnzL, lia, lja, la, diagonal, x, result, true);
}

void hip_upper_triangular_solve(const int n, const int nnzU, const int *uia, const int *uja,
                                const double *ua, const double *diagonal, const double *x,
                                double *result) {
  tri_entry(n, nnzU, uia, uja, ua, diagonal, x, result, false);
}

void lower_triangular_solve(const int n, const int nnz, const int *lia, const int *lja,
                            const double *la, const double *diag, const double *x,
                            double *result) {
  hip_lower_triangular_solve(n, nnz, lia, lja, la, diag, x, result);
}

void upper_triangular_solve(const int n, const int nnz, const int *uia, const int *uja,
                            const double *ua, const double *diag, const double *x,
                            double *result) {
  hip_upper_triangular_solve(n, nnz, uia, uja, ua, diag, x, result);
}

}  // extern "C"
