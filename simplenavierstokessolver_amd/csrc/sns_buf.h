// sns_buf.h -- raw buffer accesses (gfx950).
//
// A buffer descriptor holds an array's base and size in four scalar
// registers; an access adds a 32-bit byte offset per lane and one that is
// uniform across the wave (a row), both in the instruction, so the rows of an
// array cost one scalar register each and no address arithmetic per lane.
// The hardware checks the range: loads past the end return 0 and stores past
// it are dropped.  Lanes and whole arrays are switched off that way (offset
// kOff, size 0) instead of by a branch, which keeps the loads of a stencil in
// one straight run of instructions.
#pragma once
#include <hip/hip_runtime.h>

namespace sns {

typedef __amdgpu_buffer_rsrc_t Buf;

// beyond every array: itot <= 8192 and jtot <= 16384 keep them under 2^31 bytes
constexpr unsigned kOff = 0x80000000u;

// stride 0, 32-bit data format: the range check is on bytes
__device__ __forceinline__ Buf buf_of(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000);
}

typedef unsigned buf_v2 __attribute__((ext_vector_type(2)));
typedef unsigned buf_v4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double bld(Buf b, unsigned lane, unsigned row) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, lane, row, 0));
}
__device__ __forceinline__ double2 bld2(Buf b, unsigned lane, unsigned row) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(b, lane, row, 0));
}
__device__ __forceinline__ void bst(Buf b, unsigned lane, unsigned row, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(buf_v2, v), b, lane, row, 0);
}
__device__ __forceinline__ void bst2(Buf b, unsigned lane, unsigned row, double2 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(buf_v4, v), b, lane, row, 0);
}

}  // namespace sns
