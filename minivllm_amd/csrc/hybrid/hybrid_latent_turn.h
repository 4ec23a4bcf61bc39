// A token of latent attention by one wave: the latent's norm and its cache row, the rotated parts of the cache row and of
// the queries.  Used by a kernel of its own (hybrid_branches.hip) and beside the products of few rows
// (hybrid_latent_rows.hip).
#pragma once
#include "hybrid_common.h"

namespace hyb {

template <typename T>
__device__ __forceinline__ void turned8(const T* r, int i, int dims, int neighbours, const float* cs,
                                        const float* sn, float* o) {
    const int half = dims >> 1;
    float x[8], y[8];
    load_run<T, 8>(r + i, x);
    if (i >= dims) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = x[e];
    } else if (neighbours) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const float c = cs[(i + e) >> 1], s = sn[(i + e) >> 1];
            o[e] = x[e] * c - x[e + 1] * s;
            o[e + 1] = x[e + 1] * c + x[e] * s;
        }
    } else {
        const int at = i < half ? i : i - half;
        load_run<T, 8>(r + (i < half ? i + half : i - half), y);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float s = i < half ? -sn[at + e] : sn[at + e];
            o[e] = x[e] * cs[at + e] + y[e] * s;
        }
    }
}

// `cs`: [dims] floats of LDS of this wave's own.  No barrier inside.
template <typename T>
__device__ __forceinline__ void latent_turn_store(long t, float* cs, const T* __restrict__ q, long q_row,
                                                  const T* __restrict__ dkv, long dkv_row, const float* __restrict__ w,
                                                  float eps, const int* __restrict__ positions,
                                                  const float* __restrict__ inv_freq, int dims, T* __restrict__ k_cache,
                                                  T* __restrict__ v_cache, const int* __restrict__ slot_mapping,
                                                  T* __restrict__ out, int H, int D, int P, int R, int neighbours, float mult) {
    const int half = dims / 2, lane = threadIdx.x & 63;
    float* sn = cs + half;
    const long slot = slot_mapping ? slot_mapping[t] : -1;
    const bool store = slot >= 0 && k_cache;
    const float p = (float)positions[t];
    const T* lr = dkv + t * dkv_row;
    float ss = 0.f, x[8];
    for (int c = lane * 8; c < R; c += 512) {
        load_run<T, 8>(lr + c, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
    }
    for (int i = lane; i < half; i += 64) {
        float s_, c_;
        sincosf(p * inv_freq[i], &s_, &c_);
        cs[i] = c_ * mult; sn[i] = s_ * mult;
    }
    lanes_meet();                                                   // cs / sn: written and read by this wave
    const float r = rsqrtf(wave_sum(ss) / (float)R + eps);
    const int DK = R + P;
    if (store) {
        for (int c = lane * 8; c < R; c += 512) {
            float g[8];
            load_run<T, 8>(lr + c, x);
            load_run<float, 8>(w + c, g);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = x[e] * r * g[e];
            store_run8<T>(k_cache + slot * DK + c, x);
            if (v_cache) store_run8<T>(v_cache + slot * R + c, x);
        }
        for (int i = lane * 8; i < P; i += 512) {
            turned8(lr + R, i, dims, neighbours, cs, sn, x);
            store_run8<T>(k_cache + slot * DK + R + i, x);
        }
    }
    for (int j = lane * 8; j < H * P; j += 512) {
        const int hh = j / P, c = j - hh * P;
        turned8(q + t * q_row + (long)hh * (D + P) + D, c, dims, neighbours, cs, sn, x);
        store_run8<T>(out + t * (long)(H * P) + j, x);
    }
}

}  // namespace hyb
