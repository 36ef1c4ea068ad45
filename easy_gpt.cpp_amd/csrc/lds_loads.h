// Loads that go from memory directly to LDS, and the wait for them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace egpt {

typedef __attribute__((address_space(3))) void lds_void;

// At most N of this wavefront's memory operations are still on their way (they end in the order in which they were made).
// The loads into LDS are written in assembly and have no result in registers; __syncthreads() alone does not wait for them.
template <int N>
__device__ __forceinline__ void arrived() { __builtin_amdgcn_s_waitcnt((N & 15) | 0x0f70 | (N >> 4) << 14); }

typedef __attribute__((ext_vector_type(4))) int r_i32x4;

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"        // (m0 is a reserved register; nothing else here uses it)
// 16 bytes a lane from `resource` at byte `offset` + `at` to LDS: `lds` (the same for the whole wavefront) + 16 x lane.
__device__ __forceinline__ void load_to_lds(r_i32x4 resource, int offset, int at, char* lds) {
    const unsigned to = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_void*)lds));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(offset), "s"(resource), "s"(at)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ r_i32x4 buffer_of(const void* p, size_t bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(p);
    return r_i32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(at)), __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32) & 0xffff),
                   __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
}

// Loads bounded by a buffer's bytes: what lies past them reads as zero, without a branch around the load.  `p` and `bytes` are the
// same for the whole wavefront, at most kNowhere.
constexpr int kNowhere = static_cast<int>(0x80000000u);
typedef __amdgpu_buffer_rsrc_t buffer_t;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
__device__ __forceinline__ buffer_t values_of(const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ uint32_t read2(buffer_t b, int offset) { return __builtin_amdgcn_raw_buffer_load_b16(b, offset, 0, 0); }
__device__ __forceinline__ uint32_t read4(buffer_t b, int offset) { return __builtin_amdgcn_raw_buffer_load_b32(b, offset, 0, 0); }
__device__ __forceinline__ u32x2 read8(buffer_t b, int offset) { return __builtin_amdgcn_raw_buffer_load_b64(b, offset, 0, 0); }
__device__ __forceinline__ u32x4 read16(buffer_t b, int offset) { return __builtin_amdgcn_raw_buffer_load_b128(b, offset, 0, 0); }

}  // namespace egpt
