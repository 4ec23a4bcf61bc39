// Prompt portions of latent attention with keys and values formed: K[h] = c up_k[h]^T and V[h] = c up_v[h] for
// the cached latents c of every sequence of the step, then ordinary attention per head over
// [K | r] and V (hybrid_prompts.hip), r being the key part that the heads share, read from the cache.
//
// Against attention in the latents' own coordinates (hybrid_latent.hip), which for a query and a key takes
// 2 (R + P) + 4 R operations per head where this takes 2 (D + P) + 4 E (two parts per weight in both), and for a token
// as many for its query and its output as this for its key and value.  With R 512, P 64, D = E = 128: 3200
// against 896.  8 prompts of 512..1024 tokens, 16 heads: 267 -> 116 us for the layer (12.5 the store, 49 the forming, 61
// the attention, where the library's two batched products around the other form took 90 and its attention 182), one of 2048
// 188 -> 100, of 8192 1632 -> 536; 512 tokens behind 1536 146 -> 100.  Which of the two: the caller's rule.
//
// Formed rows: [H][formed_rows][D | E], a sequence's rows one after the other, its last tile of 32 filled up
// with zeros, the sequences in turn.
#include "hybrid_keys.h"
#include "hybrid_tiles.h"

using namespace hyb;

namespace {

struct FormArgs {
    const uint16_t* latents; int latent_row;       // cache rows [c | r]
    const int* tables; int max_blocks, block_size;
    const int *cu_q, *positions;
    const uint16_t *up_k, *up_v;                   // [H, D, R], [H, R, E]
    uint16_t *k, *v;
    long formed_rows;
    int nseq, D, E, R;
};

// A workgroup forms 256 rows (eight tiles of 32, each of one sequence and inside one page) of one head, keys by
// waves 0 to 3, values by 4 to 7, 64 rows by 128 columns each: K^T = up_k c^T and V^T = up_v^T c^T on
// v_mfma_f32_32x32x16_bf16, so that a lane's results are runs of one row's columns.  64 of R at a time go through
// registers to one of two LDS images, requested a step ahead (direct loads to LDS would be waited for ahead of
// every transposed read).  up_v lies with its columns innermost: its fragments are transposed LDS reads, and the rows they are
// multiplied with are read in the order of k that those give.
// 64 bytes a cycle from L2 to a CU are 256 x 64 of rows and 2 x 128 x 64 of weights in 1024 cycles, half of the 2048 the
// products take.   8 prompts of 512..1024 tokens, 16 heads, R 512: 49 us, 530 TFLOP/s (25 x 16
// workgroups are 1.6 for each CU; LDS moves as many bytes as it can in the time of the products).
constexpr int FM = 256, FK = 64, ROWS = FM * FK * 2, WK = 128 * FK * 2, WV = FK * 128 * 2, IMAGE = ROWS + WK + WV;

__global__ void __launch_bounds__(512, 2) latent_form_kernel(FormArgs a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    extern __shared__ __attribute__((aligned(256))) char smem[];
    __shared__ int s_live[8];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x;

    // ---- this wave's tile of rows: which sequence's, from which key on
    const int tile = blockIdx.y * 8 + wave;
    int b = -1, key0 = 0, ctx = 0;
    for (int i0 = 0, before = 0; i0 < a.nseq && b < 0; i0 += 64) {
        int n = 0, c = 0;
        if (i0 + lane < a.nseq) {
            const int r = a.cu_q[i0 + lane], len = a.cu_q[i0 + lane + 1] - r;
            if (len > 0) c = a.positions[r] + len;
            n = (c + 31) / 32;
        }
        int upto = n;                                // tiles of the sequences up to this lane's
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(upto, o, 64);
            if (lane >= o) upto += u;
        }
        const uint64_t past = __ballot(before + upto > tile);
        if (past) {
            const int src = __builtin_ctzll(past);
            b = i0 + src;
            ctx = __shfl(c, src, 64);
            key0 = (tile - before - __shfl(upto - n, src, 64)) * 32;
        }
        before += __shfl(upto, 63, 64);
    }
    b = __builtin_amdgcn_readfirstlane(b);
    ctx = __builtin_amdgcn_readfirstlane(ctx);
    key0 = __builtin_amdgcn_readfirstlane(key0);
    if (lane == 0) s_live[wave] = b >= 0 && (long)tile * 32 + 32 <= a.formed_rows;
    __syncthreads();
    if (!s_live[0]) return;                          // (the tiles behind it are not there either)

    // ---- sources: rows behind the context, and columns behind D, are out of a descriptor's range: zeros
    const uint16_t* rows = a.latents;
    int row_bytes = 0;
    if (b >= 0) {
        const int page = a.tables[(long)b * a.max_blocks + key0 / a.block_size];
        rows += ((long)page * a.block_size + key0 % a.block_size) * a.latent_row;
        row_bytes = min(32, ctx - key0) * a.latent_row * 2;
    }
    auto source = [](const uint16_t* p, int bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, bytes, 0x00020000);
    };
    const auto rs = source(rows, row_bytes);
    const auto ks = source(a.up_k + (long)h * a.D * a.R, a.D * a.R * 2);
    const auto vs = source(a.up_v + (long)h * a.R * a.E, a.R * a.E * 2);
    // 16-byte pieces of this thread: four of its wave's 32 rows, two of each weight
    int r_src[4], k_src[2], v_src[2], r_dst[4], k_dst[2], v_dst[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3), ch = lane & 7, row = wave * 32 + r;
        r_src[i] = r * a.latent_row * 2 + ch * 16;
        r_dst[i] = row * (FK * 2) + ((ch ^ swizzle<FK>(row)) << 4);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = i * 512 + tid, kr = c >> 3, kc = c & 7, vr = c >> 4, vc = c & 15;
        k_src[i] = kr * a.R * 2 + kc * 16;
        k_dst[i] = ROWS + kr * (FK * 2) + ((kc ^ swizzle<FK>(kr)) << 4);
        v_src[i] = vr * a.E * 2 + (vc * 8 < a.E ? vc * 16 : 0);       // (columns behind E: not stored)
        v_dst[i] = ROWS + WK + vr * 256 + ((vc ^ swizzle<128>(vr)) << 4);
    }
    typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
    u32x4 in[8];
    auto request = [&](int k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) in[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, r_src[i], k * 2, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            in[4 + i] = __builtin_amdgcn_raw_buffer_load_b128(ks, k_src[i], k * 2, 0);
            in[6 + i] = __builtin_amdgcn_raw_buffer_load_b128(vs, v_src[i], k * a.E * 2, 0);
        }
    };
    auto keep = [&](char* image) {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(image + r_dst[i]) = in[i];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<u32x4*>(image + k_dst[i]) = in[4 + i];
            *reinterpret_cast<u32x4*>(image + v_dst[i]) = in[6 + i];
        }
    };

    const int wm = wave & 3;
    const bool values = wave >= 4;
    f32x16 acc[4][2];                                // [block of 32 columns][block of 32 rows]
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[m][j][e] = 0.f;
    auto products = [&](const bf16x8 (&w)[4], const bf16x8 (&x)[2]) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[m], x[j], acc[m][j], 0, 0, 0);
    };
    const int i16 = lane & 15;
    auto read_keys = [&](const char* image, int s, bf16x8 (&w)[4], bf16x8 (&x)[2]) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int r = 32 * m + l32;
            w[m] = *reinterpret_cast<const bf16x8*>(image + ROWS + r * (FK * 2) + (((2 * s + half) ^ swizzle<FK>(r)) << 4));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 64 * wm + 32 * j + l32;
            x[j] = *reinterpret_cast<const bf16x8*>(image + r * (FK * 2) + (((2 * s + half) ^ swizzle<FK>(r)) << 4));
        }
    };
    auto read_values = [&](const char* image, int s, bf16x8 (&w)[4], bf16x8 (&x)[2]) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            s16x4 part[2];
#pragma unroll
            for (int hi = 0; hi < 2; ++hi) {         // k = 16 s + 8 hi + 4 half + 0 .. 3 of column 32 m + l32
                const int r = 16 * s + 8 * hi + 4 * half + (i16 >> 2);
                const int ch = 4 * m + 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1);
                part[hi] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4*)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)
                        (image + ROWS + WK + r * 256 + ((ch ^ swizzle<128>(r)) << 4) + (i16 & 1) * 8));
            }
            w[m] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 64 * wm + 32 * j + l32;
            const char* p = image + r * (FK * 2) + 8 * half;
            const s16x4 lo = *reinterpret_cast<const s16x4*>(p + (((2 * s) ^ swizzle<FK>(r)) << 4));
            const s16x4 hi = *reinterpret_cast<const s16x4*>(p + (((2 * s + 1) ^ swizzle<FK>(r)) << 4));
            x[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    auto walk = [&](auto&& read) {
        for (int k = 0; k < a.R; k += FK) {
            char* image = smem + (k / FK & 1) * IMAGE;
            if (k + FK < a.R) request(k + FK);
            bf16x8 w[2][4], x[2][2];
            read(image, 0, w[0], x[0]);
#pragma unroll
            for (int s = 0; s < FK / 16; ++s) {
                if (s + 1 < FK / 16) read(image, s + 1, w[(s + 1) & 1], x[(s + 1) & 1]);
                products(w[s & 1], x[s & 1]);
            }
            if (k + FK < a.R) keep(smem + ((k / FK + 1) & 1) * IMAGE);   // (last read before the previous barrier)
            __syncthreads();
        }
    };
    request(0);
    keep(smem);
    __syncthreads();
    if (values) walk(read_values); else walk(read_keys);

    // ---- a lane's row 64 wm + 32 j + l32: columns 32 m + 8 (e / 4) + 4 half + e % 4; the halves swap runs of four
    const int n = values ? a.E : a.D;
    uint16_t* out = (values ? a.v : a.k) + (h * a.formed_rows + blockIdx.y * (long)FM) * n;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (!s_live[2 * wm + j]) continue;
        uint16_t* row = out + (long)(64 * wm + 32 * j + l32) * n;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                uint32_t w[4];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    w[k] = (uint32_t)bf16_bits(acc[m][j][4 * r + 2 * k]) |
                           ((uint32_t)bf16_bits(acc[m][j][4 * r + 2 * k + 1]) << 16);
                const auto r0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
                const auto r1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
                const int c = 32 * m + 8 * r + 8 * half;
                if (c < n) *reinterpret_cast<uint4*>(row + c) = make_uint4(r0[0], r1[0], r0[1], r1[1]);
            }
    }
#endif
}

}  // namespace

extern "C" {

int hyb_latent_attention_ok(int R, int P);           // hybrid_latent.hip

// 1 when keys of D and values of E numbers can be formed from latents of R and attended to with P shared ones.
// R: the ranks of hybrid_latent.hip (up to 512), whose weights are in two parts as they are here; latents of higher
// ranks are attended to by kernels with weights of 24 bits and more, which forming would take bits from.
int hyb_latent_formed_ok(int D, int E, int R, int P, int block_size, int max_blocks) {
    if (D < 8 || D > 128 || E < 8 || E > 128 || P < 8 || P > 128 || (D | E | P) % 8) return 0;
    if (R < 64 || R % 64 || !hyb_latent_attention_ok(R, P) || block_size % 32) return 0;
    return latent_prompts_pages_ok(block_size, max_blocks, R + P);
}

// q [rows, H, D + P] (its first D numbers of a head are used), qr [rows, H, P] turned, cache rows [c | r] of R + P
// numbers; sequence b of nseq owns rows cu_q[b] .. cu_q[b + 1] at positions[cu_q[b]] .., with block table row b; max_q: the
// longest portion.  k, v: [H][formed_rows][D | E], formed_rows a multiple of 32 and no fewer than the sequences'
// contexts, each rounded up to 32, together.  out [rows, H, E], contiguous.
int hyb_latent_formed_prompts(const void* q, long q_row, long q_head, const void* qr, long qr_row, const void* cache,
                              const void* tables, int max_blocks, int block_size, const void* cu_q,
                              const void* positions, const void* up_k, const void* up_v, const void* sink, void* k,
                              void* v, long formed_rows, void* out, float scale, int nseq, int max_q, int H, int D, int E,
                              int R, int P, int window, hipStream_t s) {
    if (nseq <= 0 || max_q <= 0) return 0;
    if (!hyb_latent_formed_ok(D, E, R, P, block_size, max_blocks) || H <= 0 || formed_rows <= 0 || formed_rows % 32) return 1;
    if (((size_t)q | (size_t)qr | (size_t)cache | (size_t)up_k | (size_t)up_v | (size_t)k | (size_t)v | (size_t)out) % 16) return 1;
    if (q_row % 8 || q_head % 8 || qr_row % 8) return 1;
    if (nseq > 65535 || (max_q + 127) / 128 > 65535 || (formed_rows + FM - 1) / FM > 65535) return 1;
    static const hipError_t once = hipFuncSetAttribute((const void*)latent_form_kernel,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 2 * IMAGE);
    if (once != hipSuccess) return 2;
    const FormArgs a{(const uint16_t*)cache, R + P, (const int*)tables, max_blocks, block_size, (const int*)cu_q,
                     (const int*)positions, (const uint16_t*)up_k, (const uint16_t*)up_v, (uint16_t*)k, (uint16_t*)v,
                     formed_rows, nseq, D, E, R};
    hipLaunchKernelGGL(latent_form_kernel, dim3(H, (formed_rows + FM - 1) / FM), dim3(512), 2 * IMAGE, s, a);
    if (HYB_LAUNCH_OK()) return 2;
    return latent_prompts(q, q_row, q_head, qr, qr_row, cache, tables, max_blocks, block_size, cu_q, positions, sink, k, v,
                          formed_rows, out, scale, nseq, max_q, H, D, E, R, P, window, s);
}

}  // extern "C"
