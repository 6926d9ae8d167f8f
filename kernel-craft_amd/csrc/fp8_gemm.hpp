// fp8_gemm.hpp -- device helpers shared by the FP8 W8A8 GEMM kernels
// (fp8_gemm.hip: 256 x 256 tiles; fp8_gemm_small.hip: few tokens and grids
// that large tiles leave too small).
#pragma once

#include "kc_common.hpp"

namespace kc {
namespace fp8 {

typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void global_void;

constexpr int kBK = 128;       // bytes of K per step
constexpr int kE8M0One = 127;  // block scale 2^0
// instruction classes of __builtin_amdgcn_sched_group_barrier
constexpr int kSchedMfma = 0x008, kSchedDsRead = 0x100;

__device__ __forceinline__ int swizzle(int row) { return (row >> 1) & 7; }

// One global_load_lds_dwordx4: 16 bytes per lane from `g` into LDS at
// lds_base + 16 * lane.  Written as inline assembly so that the compiler's
// LDS-wait bookkeeping does not see it: with such a load in flight the
// compiler cannot count the ordinary LDS reads and drains them all before
// every use.  The kernel waits for these loads itself (vmcnt(0) before the
// barrier that publishes the buffer), and the "memory" clobber keeps LDS
// reads and writes on their side of it.
__device__ __forceinline__ void lds_dma16(const void* g, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_base)
                 : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_address(const uint8_t* p) {
    return static_cast<uint32_t>(reinterpret_cast<size_t>((lds_void*)p));
}

// Operand of the 16-row block at tile row r0: lane (i, kb) gets bytes
// 32 kb .. 32 kb + 31 of row r0 + i; with kvalid < 128 the 16-byte halves at
// or past kvalid read as zeros.
template <bool TAIL>
__device__ __forceinline__ i32x8 read_operand(const uint8_t* tile, int r0, int lane, int kvalid) {
    const int row = r0 + (lane & 15), kb = lane >> 4, sw = swizzle(row);
    const uint8_t* p = tile + row * kBK;
    u32x4 lo = *reinterpret_cast<const u32x4*>(p + 16 * ((2 * kb) ^ sw));
    u32x4 hi = *reinterpret_cast<const u32x4*>(p + 16 * ((2 * kb + 1) ^ sw));
    if constexpr (TAIL) {
        if (32 * kb >= kvalid) lo = u32x4{0u, 0u, 0u, 0u};
        if (32 * kb + 16 >= kvalid) hi = u32x4{0u, 0u, 0u, 0u};
    }
    return i32x8{static_cast<int32_t>(lo.x), static_cast<int32_t>(lo.y), static_cast<int32_t>(lo.z),
                 static_cast<int32_t>(lo.w), static_cast<int32_t>(hi.x), static_cast<int32_t>(hi.y),
                 static_cast<int32_t>(hi.z), static_cast<int32_t>(hi.w)};
}

// The GEMMs of fp8_gemm_small.hip (arguments checked by the caller, K > 0):
// false, nothing launched, for shapes that are left to the 256 x 256 tiles.
template <bool YBF16>
bool gemm_small(const char* fn, const int8_t* qx, const float* sx, const int8_t* qw, const float* sw, void* y,
                int64_t M, int64_t N, int64_t K, hipStream_t stream, int* status);

}  // namespace fp8
}  // namespace kc
