// int4_gemm.hpp -- the INT4 GEMM of int4_gemm_skinny.hip, called by the
// dispatch in int4_gemm_mfma.hip.
#pragma once

#include "kc_common.hpp"

namespace kc {
namespace int4 {

// M 2..64 (1..64), K a multiple of 128, group_size a power of two >= 128, on
// the reference layout also 64 or 32; 16-byte aligned packed and X.  -1
// (nothing launched) where another kernel is to be used.
template <bool SHUF>
int gemm_skinny(const char* fn, const uint8_t* packed, const float* scales, const uint8_t* zeros, const uint16_t* X,
                uint16_t* Y, int M, int N, int K, int group_size, hipStream_t stream);

}  // namespace int4
}  // namespace kc
