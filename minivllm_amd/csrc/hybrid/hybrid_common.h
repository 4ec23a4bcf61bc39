// Helpers shared by the kernels of hybrid decoders (fp32 residual stream, zero-centred or grouped
// norms, attention with a sink or a window, gated outer-product recurrences, expert routing).
// Activations are bfloat16 or float (template parameter), everything a norm, a softmax or a
// recurrence touches is fp32.
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hyb {

constexpr int kWave = 64;

// Between LDS that lanes of a wave have written and other lanes of it read, or the other way round: the hardware keeps a wave's
// LDS instructions in order, this keeps the compiler from moving them, to which lanes are threads of their own.  No
// instruction.
__device__ __forceinline__ void lanes_meet() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct bf16_t { uint16_t v; };

template <typename T> __device__ __forceinline__ float ld(const T* p);
template <> __device__ __forceinline__ float ld<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ld<bf16_t>(const bf16_t* p) {
    return __uint_as_float(((uint32_t)p->v) << 16);
}
template <typename T> __device__ __forceinline__ void st(T* p, float f);
template <> __device__ __forceinline__ void st<float>(float* p, float f) { *p = f; }
template <> __device__ __forceinline__ void st<bf16_t>(bf16_t* p, float f) {
    __bf16 b = (__bf16)f;                          // round to nearest even
    p->v = __builtin_bit_cast(uint16_t, b);
}

// The sum over each run of N lanes (a power of two up to 16, all of them active or none), the same bits in every lane:
// the additions of __shfl_xor by 1, 2, 4, .. in that order, by moves inside the vector unit instead of through LDS
// (some 10 cycles a step instead of 100).
template <int N>
__device__ __forceinline__ float run_sum(float v) {
#ifdef __HIP_DEVICE_COMPILE__
    static_assert(N == 1 || N == 2 || N == 4 || N == 8 || N == 16);
    auto moved = [&](auto ctrl) {
        return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    if constexpr (N >= 2) v += moved(std::integral_constant<int, 0xb1>{});       // quads 1 0 3 2
    if constexpr (N >= 4) v += moved(std::integral_constant<int, 0x4e>{});       // quads 2 3 0 1
    if constexpr (N >= 8) v += moved(std::integral_constant<int, 0x141>{});      // rows of 8 mirrored: a quad's lanes are alike
    if constexpr (N >= 16) v += moved(std::integral_constant<int, 0x140>{});     // rows of 16 mirrored
#endif
    return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

// sum over a workgroup of up to 1024 threads; `red` holds 16 floats of LDS; every thread gets it
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int w = threadIdx.x / kWave, nw = (blockDim.x + kWave - 1) / kWave;
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) red[w] = v;
    __syncthreads();
    float s = 0.f;
    for (int i = 0; i < nw; ++i) s += red[i];
    return s;
}
__device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int w = threadIdx.x / kWave, nw = (blockDim.x + kWave - 1) / kWave;
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) red[w] = v;
    __syncthreads();
    float s = red[0];
    for (int i = 1; i < nw; ++i) s = fmaxf(s, red[i]);
    return s;
}

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float siluf_(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }

// 0.5 z (1 + tanh(a)) = z sigmoid(2 a), a = sqrt(2/pi) (z + 0.044715 z^3)
__device__ __forceinline__ float gelu_tanh_(float z) {
    return z * sigmoidf_(1.5957691216057308f * (z + 0.044715f * z * z * z));
}

// four (Vec4) or N (load_run, N % 4 == 0) consecutive elements widened to fp32; the address must
// be aligned to the run of four (8 bytes for bfloat16, 16 for float)
template <typename T> struct Vec4;
template <> struct Vec4<float> {
    static __device__ __forceinline__ void load(const float* p, float* o) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    }
};
template <> struct Vec4<bf16_t> {
    static __device__ __forceinline__ void load(const bf16_t* p, float* o) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        o[0] = __uint_as_float(v.x << 16); o[1] = __uint_as_float(v.x & 0xffff0000u);
        o[2] = __uint_as_float(v.y << 16); o[3] = __uint_as_float(v.y & 0xffff0000u);
    }
};
template <typename T, int N> __device__ __forceinline__ void load_run(const T* p, float* o) {
#pragma unroll
    for (int i = 0; i < N; i += 4) Vec4<T>::load(p + i, o + i);
}

// eight consecutive elements narrowed from fp32 and stored as one run (16 bytes of bfloat16, two
// 16-byte stores of float); the address must be aligned to the run
template <typename T> __device__ __forceinline__ void store_run8(T* p, const float* v);
template <> __device__ __forceinline__ void store_run8<float>(float* p, const float* v) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
template <> __device__ __forceinline__ void store_run8<bf16_t>(bf16_t* p, const float* v) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const __bf16 lo = (__bf16)v[2 * i], hi = (__bf16)v[2 * i + 1];
        w[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Rows of a recurrence's output o [T, H, E] that no live sequence owns (ahead of the first sequence,
// behind the last, those of a sequence without a state slot) read as zeros: workgroup (b, h, columns
// [e0, e0 + cols)) of B sequences clears its share of them.
__device__ __forceinline__ void clear_unowned(float* o, const int* cu_q, const int* slots, int b, int B, long T,
                                              int H, int h, int E, int e0, int cols) {
    const int n = min(cols, E - e0);
    auto clear = [&](long from, long to) {
        for (long i = threadIdx.x; i < (to - from) * n; i += blockDim.x)
            o[((from + i / n) * H + h) * E + e0 + i % n] = 0.f;
    };
    if (b == 0 && cu_q) clear(0, cu_q[0]);
    if (b + 1 == B) clear(cu_q ? cu_q[B] : B, T);
    if (slots[b] < 0) clear(cu_q ? cu_q[b] : b, cu_q ? cu_q[b + 1] : b + 1);
}

#define HYB_DISPATCH(dt, ...)                                         \
    do {                                                              \
        if ((dt) == 0) { using T = hyb::bf16_t; __VA_ARGS__; }        \
        else if ((dt) == 2) { using T = float; __VA_ARGS__; }         \
        else return 1;                                                \
    } while (0)

#define HYB_LAUNCH_OK() (hipGetLastError() == hipSuccess ? 0 : 2)

}  // namespace hyb
