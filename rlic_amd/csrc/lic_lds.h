// What the replay kernels that stage a part of the image in LDS share.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lic_device.h"

namespace rlic {

// Buffer addressing covers arrays of fewer than 2^32 bytes.
inline bool fits_buffer(int64_t bytes) { return bytes > 0 && bytes <= 0xFFFFFFFFll; }

// Per-block LDS of the current device, in bytes.
inline int32_t lds_replay_limit_bytes() {
  int dev = 0, limit = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&limit, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
    return 0;
  return limit;
}

__device__ __forceinline__ int32_t wrap_index(int32_t c, int32_t n) {
  c %= n;
  return c < 0 ? c + n : c;
}

// A line's position while replaying: an LDS byte pointer into the staged
// box (LdsWalk) or a byte offset into the image, read with buffer loads
// (ImageWalk, the hybrid replay's steps past the box).  Either way each
// step is one add of a pair-table delta.
typedef const unsigned char __attribute__((address_space(3))) lds_byte;

template <typename T>
__device__ __forceinline__ T lds_value(lds_byte* at) {
  typedef const T __attribute__((address_space(3))) lds_t;
  return *reinterpret_cast<lds_t*>(at);
}

// kTableFirst: the replay loop reads the pair-table entries of all of a
// lane's lines before their gathers (LDS gathers are short; the early table
// reads hide their latency), or each line's just before its own gathers
// (image gathers are long; fewer registers live).
template <typename T>
struct LdsWalk {
  typedef lds_byte* Pos;
  static constexpr bool kTableFirst = true;
  __device__ __forceinline__ T operator()(Pos at) const { return lds_value<T>(at); }
};

template <typename T>
struct ImageWalk {
  typedef uint32_t Pos;
  static constexpr bool kTableFirst = false;
  __amdgpu_buffer_rsrc_t rsrc;  // the image, n elements with n * sizeof(T) < 2^32
  // base and size pass through readfirstlane: the descriptor must be
  // wave-uniform (scalar registers), which the compiler does not prove here
  __device__ __forceinline__ ImageWalk(const T* base, int64_t n) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32));
    const uint32_t bytes =
        __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(n * static_cast<int64_t>(sizeof(T))));
    rsrc = make_rsrc(reinterpret_cast<const void*>((uint64_t{hi} << 32) | lo), bytes);
  }
  __device__ __forceinline__ T operator()(Pos at) const {
    return buf_load(rsrc, at, static_cast<T*>(nullptr));
  }
};

}  // namespace rlic
