// Device pieces shared by the resident CG kernels: published values, wave sums, barrier.
#pragma once
#include "fem_cell.h"
#include "fem_resident.h"

namespace fem {

constexpr int kResT = 512;              // threads per block
constexpr int kResWaves = kResT / 64;
constexpr int kResMaxBlocks = 256;      // one per CU
constexpr int kResCopies = 8;           // copies of a block's record
constexpr int kStaticLds = 1024;        // left for a kernel's static LDS; the rest of the device's limit may be dynamic
constexpr size_t kRecWords = (size_t)2 * kResCopies * 2 * kResMaxBlocks * 4;

// Lets a kernel take all the dynamic LDS there is.  The attribute belongs to the kernel, not to a
// launch: a value per launch would let one host thread lower it under the launch of another.
inline hipError_t res_dynamic_lds(const void* kernel, int maxlds) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, maxlds - kStaticLds);
}

typedef unsigned int U4 __attribute__((ext_vector_type(4)));
typedef unsigned int U2 __attribute__((ext_vector_type(2)));

// Published values: an FP64 value as 16 bytes (low half, tag, high half, tag), an FP32 value as
// 8 (bits, tag); each 8-byte word carries its own tag, so a reader may see the words of one
// value at different times.  The buffer forms with sc1 are the agent-scope relaxed accesses
// (write-through, and a read of what all XCDs share), 16 bytes wide.
constexpr int kAgent = 16;              // sc1
__device__ __forceinline__ void ll_put(__amdgpu_buffer_rsrc_t r, uint32_t at, double v, uint32_t tag) {
  const long long bits = __double_as_longlong(v);
  U4 q = {(uint32_t)bits, tag, (uint32_t)((unsigned long long)bits >> 32), tag};
  __builtin_amdgcn_raw_buffer_store_b128(q, r, (int)(at * 16u), 0, kAgent);
}
__device__ __forceinline__ void ll_put(__amdgpu_buffer_rsrc_t r, uint32_t at, float v, uint32_t tag) {
  U2 q = {__float_as_uint(v), tag};
  __builtin_amdgcn_raw_buffer_store_b64(q, r, (int)(at * 8u), 0, kAgent);
}
template <typename X>
struct LL;
template <>
struct LL<double> {
  typedef U4 W;
  static __device__ __forceinline__ W get(__amdgpu_buffer_rsrc_t r, uint32_t at) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, (int)(at * 16u), 0, kAgent);
  }
  static __device__ __forceinline__ bool ok(W v, uint32_t tag) { return v[1] == tag && v[3] == tag; }
  static __device__ __forceinline__ double val(W v) {
    return __longlong_as_double((long long)(((unsigned long long)v[2] << 32) | v[0]));
  }
};
template <>
struct LL<float> {
  typedef U2 W;
  static __device__ __forceinline__ W get(__amdgpu_buffer_rsrc_t r, uint32_t at) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, (int)(at * 8u), 0, kAgent);
  }
  static __device__ __forceinline__ bool ok(W v, uint32_t tag) { return v[1] == tag; }
  static __device__ __forceinline__ float val(W v) { return __uint_as_float(v[0]); }
};

// Sum over the wave by DPP row shifts and broadcasts, valid in lane 63 (fixed order).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8: sums of 16 lanes in the row's last lane
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
  return v;
}

// A value all lanes hold, in scalar registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uniform(double v) {
  const long long b = __double_as_longlong(v);
  return __longlong_as_double(((long long)uniform((int)(b >> 32)) << 32) | (unsigned int)uniform((int)b));
}

// Element of an LDS array at a byte offset.
template <typename X>
__device__ __forceinline__ X at_lds(const X* base, uint32_t boff) {
  return *reinterpret_cast<const X*>(reinterpret_cast<const char*>(base) + boff);
}

__device__ __forceinline__ void res_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The kernel's argument block, through a pointer the compiler cannot trace.
__device__ __forceinline__ const void* res_kernargs() {
  const void* p = (const void*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

}  // namespace fem
