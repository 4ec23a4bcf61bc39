// What the attention kernels on the matrix cores share: fragment types, the layout of a tile of cache
// rows in LDS, the softmax's constants.
//
// A tile is an image of whole rows (pitch 2 * columns bytes) in 16-byte chunks; the chunk number of a
// row is XORed with a function of the row, so that both the row reads (16 rows, one chunk) and the
// transposed reads (4 rows, 64 bytes) of a wave fall on different banks, for row pitches of whole
// multiples of 256 bytes and of odd multiples of 128.
#pragma once
#include "hybrid_merge.h"
#include <type_traits>

namespace hyb {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

constexpr float LOG2E = 1.4426950408889634f;
constexpr float RESCALE = 6.f;      // log2 units: weights stay <= 64 between rescales

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

__device__ __forceinline__ uint16_t bf16_bits(float f) {
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}

// what the chunk number of a row is XORed with (see the header comment)
template <int DP>
__device__ __forceinline__ int swizzle(int row) {
    return DP % 128 == 0 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

}  // namespace hyb
