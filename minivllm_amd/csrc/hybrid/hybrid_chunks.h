// Recurrences over prompt portions in chunks of tokens on the matrix cores: the matrix LSTM's
// (hybrid_chunks.hip) and the delta rule's (hybrid_delta_chunks.hip); what their kernels share.
//
// An fp32 operand of a bf16 product is cut into three parts of eight bits, which hold all of its 24.  The parts are
// rounded, not cut off: what they leave is half as large and of either sign, so that the three products of parts
// that a product of two such operands leaves out (2^-27 of it in the mean, 2^-23 at most) do not add up over a sum.
#pragma once
#include "hybrid_tiles.h"

namespace hyb {

typedef __attribute__((ext_vector_type(4))) float f32x4;

// x and y rounded to eight bits each, side by side
__device__ __forceinline__ uint32_t rounded(float x, float y) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
// what the two parts `w` leave of x and y (exact)
__device__ __forceinline__ void rest(uint32_t w, float& x, float& y) {
    x -= __uint_as_float(w << 16);
    y -= __uint_as_float(w & 0xffff0000u);
}

// What the number of a row's 16-byte chunk is XORed with in images of 64 (rows of 128 bytes) or 128 columns that
// 16 x 16 products read.  LDS serves a wave's accesses in groups of lanes, and a group has to find its
// bytes in different banks (a line of 256 bytes, two rows of 64 columns):
//   rows, 16 bytes a lane: rows 0-3 and 12-15 of one chunk with 4-11 of the next: distinct XOR [4 <= row < 12];
//   transposed, 8 bytes a lane: 32 bytes of rows 0-7 (8-15), or of 0-3 and 8-11 (4-7 and 12-15): half of it distinct;
//   stores of 8 bytes a lane, a column's chunk of 16 rows: distinct.
// swizzle (hybrid_tiles.h), which is for transposed reads of 64 bytes of four rows, had every such read of 32
// bytes take twice as long: a third of the delta rule's LDS cycles (its walk 150 -> 147 us; the matrix LSTM's does not
// wait for them).
template <int DP>
__device__ __forceinline__ int rows16(int row) {
    if (DP % 128 == 0) return (((row ^ (row >> 1 & 4)) & 7) << 1) | (row >> 3 & 1);
    const int i = row >> 1;
    return (((i ^ (i >> 1 & 2)) & 3) << 1) | (i >> 2 & 1);
}

// eight numbers as three bfloat16 fragments whose sum they are
__device__ __forceinline__ void split8(const float* x, bf16x8* p) {
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float u = x[2 * j], v = x[2 * j + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            w[k][j] = rounded(u, v);
            if (k < 2) rest(w[k][j], u, v);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = __builtin_bit_cast(bf16x8, make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]));
}

#ifdef __HIP_DEVICE_COMPILE__
__device__ __forceinline__ s16x4 read_tr(const char* lds) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(
        (__attribute__((address_space(3))) char*)lds));
}
__device__ __forceinline__ bf16x8 join(s16x4 x, s16x4 y) {
    const s16x8 v = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// sum of the six products of parts that reach 24 bits, the small ones first
__device__ __forceinline__ f32x4 mfma6(const bf16x8* a, const bf16x8* b, f32x4 c) {
    c = mfma(a[2], b[0], c);
    c = mfma(a[0], b[2], c);
    c = mfma(a[1], b[1], c);
    c = mfma(a[1], b[0], c);
    c = mfma(a[0], b[1], c);
    return mfma(a[0], b[0], c);
}
// A product of fp32 operands: the six products of parts that reach 24 bits.  The small five have a sum of
// their own, so that a step rounds the result once and not six times.
struct Product {
    f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = {0.f, 0.f, 0.f, 0.f};
    __device__ __forceinline__ void add(const bf16x8* a, const bf16x8* b) {
        lo = mfma(a[2], b[0], lo);
        hi = mfma(a[0], b[0], hi);
        lo = mfma(a[0], b[2], lo);
        lo = mfma(a[1], b[1], lo);
        lo = mfma(a[1], b[0], lo);
        lo = mfma(a[0], b[1], lo);
    }
    __device__ __forceinline__ f32x4 sum() const { return hi + lo; }
};
#endif

#ifdef __HIP_DEVICE_COMPILE__
// A kernel's only argument, loaded again: what a rare path needs of it is not kept in registers all along.
template <class A>
__device__ __forceinline__ A arguments_anew() {
    uintptr_t p = (uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const __attribute__((address_space(4))) A*)p;
}
#endif

// four numbers of a lane as three runs of bfloat16; at(k): where part k goes
template <class F>
__device__ __forceinline__ void put_parts(f32x4 x, F&& at) {
    float a = x[0], b = x[1], c = x[2], d = x[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint2 w = make_uint2(rounded(a, b), rounded(c, d));
        *reinterpret_cast<uint2*>(at(k)) = w;
        rest(w.x, a, b);
        rest(w.y, c, d);
    }
}

// x of the lane N places before (behind) this one inside its row of 16, `none` where there is none
template <int N> __device__ __forceinline__ float from_left(float x, float none) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(none), __float_as_uint(x), 0x110 | N, 0xf, 0xf, false));
}
template <int N> __device__ __forceinline__ float from_right(float x, float none) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(none), __float_as_uint(x), 0x100 | N, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_of(float x, int lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), lane));
}

struct MlstmChunks {
    const void *q, *k, *v;          // rows of [*, H, D] / [*, H, E], element strides per token below
    long q_row, k_row, v_row;
    const void *gi, *gf;            // raw gate pre-activations [T, H]
    long g_row;
    const float *bi, *bf;           // [H]
    float cap;
    float *state, *nstate, *mstate; // [slots,H,D,E], [slots,H,ZG,D], [slots,H,ZG], ZG = ceil(E/16)
    const int *cu_q, *positions, *slots;
    float* o;                       // [T, H, E]
    void* ws;                       // mlstm_chunks_bytes
    long T;                         // rows of o; those of no sequence become zeros
    int B, H, D, E;
    float qscale;
};

// bytes of workspace, 0 where there is no such way: it takes portions (cu_q), up to 128 key channels, sizes in whole runs
// of eight and 16-byte addresses
long mlstm_chunks_bytes(const MlstmChunks& a, int dt);
// whether it is the faster one; longest: the longest portion's tokens, 0 if that is not known
bool mlstm_chunks_pay(const MlstmChunks& a, int longest, int dt);
int mlstm_chunks(const MlstmChunks& a, int dt, hipStream_t s);

struct DeltaChunks {
    const float *q, *k, *v;         // [T, G, D], [T, G, D], [T, H, E]
    const float *beta, *decay;      // [T, H]
    float* state;                   // [slots, H, D, E]
    const int *cu_q, *positions, *slots;
    float* o;                       // [T, H, E]
    char* ws;                       // what the first kernel leaves for the second: delta_chunks_bytes
    long T;
    int B, H, G, D, E;
};

// bytes of workspace for portions of these sizes, 0 when the recurrence is to be walked token by token
long delta_chunks_bytes(const DeltaChunks& a);
// correct: with the delta rule's correction term
int delta_chunks(const DeltaChunks& a, bool correct, hipStream_t s);

enum ChannelRule { CHANNEL_GLA = 0, CHANNEL_WKV = 1 };

struct ChannelChunks {
    const void *q, *k, *v, *a;      // rows of [*, H, D] / [*, H, E]; a: the decays' pre-activations [*, H*D]
    long q_row, k_row, v_row, a_row;
    const float *a_bias, *bonus;    // [H*D]
    float tau_inv, qscale;
    float* state;                   // [slots, H, D, E]
    const int *cu_q, *positions, *slots;
    float* ws;                      // channel_chunks_bytes
    float* o;                       // [T, H, E], or
    void* y;                        // [T, H*E]: the same normed and gated
    const void* gate; long gate_row;
    const float* norm_w;
    float eps;
    int sig, w_heads;
    long T;
    int B, H, D, E;
};

// bytes of workspace for portions of these sizes, 0 when the recurrence is to be walked token by token
long channel_chunks_bytes(const ChannelChunks& a, int dt);
int channel_chunks(const ChannelChunks& a, int rule, int dt, hipStream_t s);

// hybrid_delta.hip: single next tokens of the delta rule with a decay per key channel; false when the sizes have
// no instance
bool channel_delta_step(const void* qn, const void* kn, const void* vv, const void* beta, const void* decay, void* state,
                        const void* positions, const void* slots, void* o, long T_, int B, int H, int G, int D, int E,
                        hipStream_t s, int* rc);

}  // namespace hyb
