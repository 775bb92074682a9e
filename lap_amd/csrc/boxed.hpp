// boxed.hpp -- values passed between running workgroups, and the buffer
// accesses they use.
//
// A value travels in an aligned 8-byte word per 32-bit half, the half beside a
// 32-bit tag that no earlier value of that place had.  Such a word is written
// and read whole, so a matching tag means the half is the expected one: no
// flag, fence or store order is involved.  Stores and loads are agent-scope
// (sc1): past the CU's cache and the XCD's L2, about 3 us from the store to
// the first load that sees it.
#pragma once

#include <hip/hip_runtime.h>

namespace lap {

typedef __attribute__((ext_vector_type(4))) unsigned fl_u4;
typedef __attribute__((ext_vector_type(2))) unsigned fl_u2;

__device__ __forceinline__ double fl_f64(unsigned lo, unsigned hi) {
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// a buffer of `bytes` from p (gfx9 word 3: raw data, 32-bit); loads past its
// end give 0
__device__ __forceinline__ __amdgpu_buffer_rsrc_t fl_buffer(const void *p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00027000);
}

constexpr int kFlAgent = 16;  // sc1
__device__ __forceinline__ void fl_put(__amdgpu_buffer_rsrc_t box, int i, unsigned tag, double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  __builtin_amdgcn_raw_buffer_store_b128(fl_u4{(unsigned)b, tag, (unsigned)(b >> 32), tag}, box,
                                         i * 16, 0, kFlAgent);
}
__device__ __forceinline__ void fl_put(__amdgpu_buffer_rsrc_t box, int i, unsigned tag, float v) {
  __builtin_amdgcn_raw_buffer_store_b64(fl_u2{__float_as_uint(v), tag}, box, i * 8, 0, kFlAgent);
}
template <class VT>
struct FlBoxed;
template <>
struct FlBoxed<double> {
  fl_u4 w;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t box, int i) {
    w = __builtin_amdgcn_raw_buffer_load_b128(box, i * 16, 0, kFlAgent);
  }
  __device__ __forceinline__ bool is(unsigned tag) const { return w.y == tag && w.w == tag; }
  __device__ __forceinline__ double value() const { return fl_f64(w.x, w.z); }
};
template <>
struct FlBoxed<float> {
  fl_u2 w;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t box, int i) {
    w = __builtin_amdgcn_raw_buffer_load_b64(box, i * 8, 0, kFlAgent);
  }
  __device__ __forceinline__ bool is(unsigned tag) const { return w.y == tag; }
  __device__ __forceinline__ float value() const { return __uint_as_float(w.x); }
};

// The compiler may not move memory accesses across this.
__device__ __forceinline__ void fl_fence() { __atomic_signal_fence(__ATOMIC_SEQ_CST); }

}  // namespace lap
