// Latent attention of steps with few rows (single next tokens, short prompts) in the latents' coordinates, three kernels:
//
//   latent_absorb_kernel  a_h = W_uk_h^T q_h for every row and head, and beside it, in workgroups of their own, the
//                         latent's norm, the rotations and the cache rows (hybrid_latent_turn.h)
//   latent_attention      hybrid_latent.hip
//   latent_expand_kernel  the partial results of a split context folded, then W_uv_h times the sum of latents
//
// The products are one read of the weights (4 MB for 16 heads of 128, R 512) under at most a few hundred rows: bound by the
// chain load -> LDS -> product -> store of one workgroup, and with it by how many kernels stand behind each other.  As
// two library products, rotation and store, attention and merge (five kernels, 12 us of the host each for the library's two),
// one token with 432 keys, 16 heads, R 128: 88 us a call,
// 30 of them on the card; now 27 (the limits: latent_rows_pay in ops/hip_hybrid.py).
#include "hybrid_chunks.h"
#include "hybrid_latent.h"
#include "hybrid_latent_turn.h"

using namespace hyb;

namespace {

// image of rows of 64 bfloat16 (128 bytes) in 16-byte chunks
__device__ __forceinline__ int at64(int row, int chunk) { return row * 128 + ((chunk ^ rows16<64>(row)) << 4); }

struct RowsArgs {
    const uint16_t* q; long q_row;                 // [T, H, D + P]
    const uint16_t* dkv; long dkv_row;
    const float* w; float eps;
    const int* positions;
    const float* inv_freq; int dims, neighbours; float mult;
    uint16_t* cache;
    const int* slots;
    const uint16_t *up_k, *up_v;                   // [H, D, R], [H, R, E]
    uint16_t *qa, *qr, *o;                         // [H, T, R], [T, H, P], [T, H, R]
    const float* part;                             // [T, H, splits][R + 2] where splits > 1
    const float* sink;
    const int* lens;                               // single next tokens: their contexts
    uint16_t* out;                                 // [T, H, E]
    int T, H, D, P, R, E, splits;
};

// 64 columns of W (row-major, `cols` of them, from c0) and rows 0 .. n - 1 into an image, zeros up to `rows`
__device__ __forceinline__ void stage64(char* lds, const uint16_t* w, int n, int rows, int cols, int c0) {
    for (int i = threadIdx.x; i < rows * 8; i += 256) {
        const int row = i >> 3, c = c0 + (i & 7) * 8;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (row < n && c < cols) x = *reinterpret_cast<const uint4*>(w + (long)row * cols + c);
        *reinterpret_cast<uint4*>(lds + at64(row, i & 7)) = x;
    }
}

// Workgroup = 64 columns of W_uk of a head under 64 rows (wave = 16 columns); behind them one for every four tokens.
__global__ void __launch_bounds__(256) latent_absorb_kernel(const RowsArgs a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const int nrb = (a.R + 63) >> 6, ntb = (a.T + 63) >> 6, products = nrb * ntb * a.H;
    if ((int)blockIdx.x >= products) {
        const long t = (long)(blockIdx.x - products) * 4 + (threadIdx.x >> 6);
        if (t < a.T)
            latent_turn_store((long)t, reinterpret_cast<float*>(smem) + (threadIdx.x >> 6) * a.dims, (const bf16_t*)a.q, a.q_row,
                              (const bf16_t*)a.dkv, a.dkv_row, a.w, a.eps, a.positions, a.inv_freq, a.dims, (bf16_t*)a.cache,
                              (bf16_t*)nullptr, a.slots, (bf16_t*)a.qr, a.H, a.D, a.P, a.R, a.neighbours, a.mult);
        return;
    }
    const int rb = blockIdx.x % nrb, tb = blockIdx.x / nrb % ntb, h = blockIdx.x / (nrb * ntb);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, q4 = lane >> 4;
    const int steps = (a.D + 31) >> 5;
    stage64(smem, a.up_k + (long)h * a.D * a.R, a.D, 32 * steps, a.R, 64 * rb);
    __syncthreads();
    const int r0 = 64 * rb + 16 * w;
    if (r0 >= a.R) return;
    for (int t0 = 64 * tb; t0 < min(a.T, 64 * tb + 64); t0 += 16) {
        const int t = t0 + l16;
        const uint16_t* qp = a.q + (long)min(t, a.T - 1) * a.q_row + (long)h * (a.D + a.P);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < steps; ++s) {
            const int d = 32 * s + 8 * q4, row = d + (l16 >> 2), chunk = 2 * w + ((l16 & 3) >> 1);
            uint4 x = make_uint4(0, 0, 0, 0);
            if (d < a.D) x = *reinterpret_cast<const uint4*>(qp + d);
            const bf16x8 wf = join(read_tr(smem + at64(row, chunk) + (l16 & 1) * 8), read_tr(smem + at64(row + 4, chunk) + (l16 & 1) * 8));
            acc = mfma(wf, __builtin_bit_cast(bf16x8, x), acc);
        }
        if (t < a.T && r0 + 4 * q4 < a.R)
            *reinterpret_cast<uint2*>(a.qa + ((long)h * a.T + t) * a.R + r0 + 4 * q4) = make_uint2(rounded(acc[0], acc[1]), rounded(acc[2], acc[3]));
    }
#endif
}

// Workgroup = 64 columns of W_uv of a head (wave = 16) and 16 rows.
template <bool MERGE>
__global__ void __launch_bounds__(256) latent_expand_kernel(const RowsArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const int neb = (a.E + 63) >> 6, eb = blockIdx.x % neb, h = blockIdx.x / neb % a.H, t0 = blockIdx.x / (neb * a.H) * 16;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, q4 = lane >> 4;
    const int steps = (a.R + 31) >> 5, R = a.R, splits = a.splits;
    char* rows = smem + 32 * steps * 128;                       // [16] folded rows, padded by a chunk
    const int pitch = 32 * steps * 2 + 16;
    float* fac = reinterpret_cast<float*>(rows + 16 * pitch);   // [16][17]: a split's factor, the row's
    float* ml = fac + 16 * 17;                                  // [16][16][2]
    if (MERGE) {
        const int t = tid >> 4, s = tid & 15, tt = min(t0 + t, a.T - 1);
        const float* p = a.part + (((long)tt * a.H + h) * splits + min(s, splits - 1)) * (R + 2);
        *reinterpret_cast<float2*>(ml + (t * 16 + s) * 2) = *reinterpret_cast<const float2*>(p);
    }
    stage64(smem, a.up_v + (long)h * R * a.E, R, 32 * steps, a.E, 64 * eb);
    __syncthreads();
    if (MERGE) {
        {   // as sink_attention_merge_kernel
            const int t = tid >> 4, s = tid & 15;
            const float* x = ml + t * 32;
            float M = a.sink ? a.sink[h] : NO_SINK_MAX;
            for (int i = 0; i < splits; ++i) M = fmaxf(M, x[2 * i]);
            float L = a.sink ? expf(a.sink[h] - M) : 0.f;
            for (int i = 0; i < splits; ++i) L += x[2 * i + 1] * expf(x[2 * i] - M);
            if (s < splits) fac[t * 17 + s] = expf(x[2 * s] - M);
            if (s == 0) fac[t * 17 + 16] = 1.f / L;
        }
        __syncthreads();
        for (int i = tid; i < 16 * 16 * steps; i += 256) {      // two neighbouring numbers of a row
            const int t = i / (16 * steps), r = i % (16 * steps) * 2;
            float x = 0.f, y = 0.f;
            if (t0 + t < a.T && r < R) {
                const float* p = a.part + ((long)(t0 + t) * a.H + h) * splits * (R + 2) + 2 + r;
                for (int s = 0; s < splits; ++s) {
                    const float2 v = *reinterpret_cast<const float2*>(p + (long)s * (R + 2));
                    x += v.x * fac[t * 17 + s];
                    y += v.y * fac[t * 17 + s];
                }
            }
            *reinterpret_cast<uint32_t*>(rows + t * pitch + r * 2) = rounded(x * fac[t * 17 + 16], y * fac[t * 17 + 16]);
        }
        __syncthreads();
    }
    const int e0 = 64 * eb + 16 * w, t = t0 + l16;
    if (e0 >= a.E) return;
    const uint16_t* op = a.o + ((long)min(t, a.T - 1) * a.H + h) * R;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < steps; ++s) {
        const int r = 32 * s + 8 * q4, row = r + (l16 >> 2), chunk = 2 * w + ((l16 & 3) >> 1);
        uint4 x = make_uint4(0, 0, 0, 0);
        if (MERGE) x = *reinterpret_cast<const uint4*>(rows + l16 * pitch + r * 2);
        else if (r < R) x = *reinterpret_cast<const uint4*>(op + r);
        const bf16x8 wf = join(read_tr(smem + at64(row, chunk) + (l16 & 1) * 8), read_tr(smem + at64(row + 4, chunk) + (l16 & 1) * 8));
        acc = mfma(wf, __builtin_bit_cast(bf16x8, x), acc);
    }
    if (t >= a.T || e0 + 4 * q4 >= a.E) return;
    if (a.lens && a.lens[t] <= 0) acc = {0.f, 0.f, 0.f, 0.f};   // no sequence's row
    *reinterpret_cast<uint2*>(a.out + ((long)t * a.H + h) * a.E + e0 + 4 * q4) = make_uint2(rounded(acc[0], acc[1]), rounded(acc[2], acc[3]));
#endif
}

constexpr long align256(long n) { return (n + 255) & ~255L; }

}  // namespace

extern "C" {

int hyb_latent_attention_ok(int R, int P);

// Whether hyb_latent_rows takes these sizes (addresses and row strides: whole runs of eight).
int hyb_latent_rows_ok(int H, int D, int P, int R, int E, int dims, int neighbours) {
    if (H <= 0 || H > 4096 || D < 8 || D > 256 || D % 8 || E < 8 || E % 8 || P <= 0) return 0;
    return dims >= 0 && dims <= P && dims % (neighbours ? 8 : 16) == 0 && hyb_latent_attention_ok(R, P);
}

// Bytes of workspace: absorbed queries, rotated parts, sums of latents, partial results of split contexts.
long hyb_latent_rows_ws(long T_, int H, int P, int R, int splits) {
    return align256(T_ * H * R * 2) * 2 + align256(T_ * H * P * 2) + (splits > 1 ? T_ * H * splits * (R + 2L) * 4 : 0);
}

// A step's rows: prompt portions (cu_q and positions: sequence b owns rows cu_q[b] .. cu_q[b + 1], max_q the longest) or
// single next tokens (lens: row b is sequence b, its context its own token included).  out [T, H, E].
int hyb_latent_rows(const void* q, long q_row, const void* dkv, long dkv_row, const void* w, float eps, const void* positions,
                    const void* inv_freq, int dims, int neighbours, float mult, void* cache, const void* slot_mapping,
                    const void* up_k, const void* up_v, const void* tables, int max_blocks, int block_size, const void* cu_q,
                    const void* lens, const void* sink, void* ws, void* out, float scale, long T_, int nseq, int max_q, int H,
                    int D, int P, int R, int E, int window, int splits, hipStream_t s) {
    if (T_ <= 0 || nseq <= 0 || max_q <= 0) return 0;
    if (!hyb_latent_rows_ok(H, D, P, R, E, dims, neighbours) || block_size <= 0 || splits < 1 || splits > 16 || T_ > 1 << 20) return 1;
    if (cu_q ? splits != 1 : (!lens || max_q != 1 || nseq != T_)) return 1;
    if (((size_t)q | (size_t)dkv | (size_t)w | (size_t)cache | (size_t)up_k | (size_t)up_v | (size_t)ws | (size_t)out) % 16) return 1;
    if (q_row % 8 || dkv_row % 8 || !cache || !slot_mapping || (long)max_q * H > 0x3fffffffL) return 1;
    char* p = (char*)ws;
    RowsArgs a{(const uint16_t*)q, q_row, (const uint16_t*)dkv, dkv_row, (const float*)w, eps, (const int*)positions,
               (const float*)inv_freq, dims, neighbours, mult, (uint16_t*)cache, (const int*)slot_mapping,
               (const uint16_t*)up_k, (const uint16_t*)up_v, nullptr, nullptr, nullptr, nullptr, (const float*)sink,
               (const int*)lens, (uint16_t*)out, (int)T_, H, D, P, R, E, splits};
    a.qa = (uint16_t*)p;
    p += align256(T_ * H * R * 2);
    a.o = (uint16_t*)p;
    p += align256(T_ * H * R * 2);
    a.qr = (uint16_t*)p;
    p += align256(T_ * H * P * 2);
    a.part = (const float*)p;
    const int products = ((R + 63) / 64) * (int)((T_ + 63) / 64) * H;
    const size_t lds1 = (size_t)((D + 31) / 32) * 32 * 128;
    if (4 * (size_t)dims * 4 > 64 * 1024) return 1;
    hipLaunchKernelGGL(latent_absorb_kernel, dim3(products + (T_ + 3) / 4), dim3(256), lds1 > 16 * (size_t)dims ? lds1 : 16 * (size_t)dims,
                       s, a);
    const hyb_latent::LatentArgs l{a.qa, R, T_ * R, a.qr, (long)H * P, P, a.cache, (const int*)tables, max_blocks, block_size,
                                   (const int*)cu_q, (const int*)positions, (const int*)lens, a.sink, a.o, (long)H * R, R,
                                   (float*)p, scale, H, R, P, window, splits};
    const int rc = hyb_latent::dispatch(l, nseq, max_q * H, max_q * H > 64, s);
    if (rc) return rc;
    const int steps = (R + 31) / 32;
    const size_t lds2 = (size_t)steps * 32 * 128 + (splits > 1 ? 16 * (steps * 64 + 16) + (16 * 17 + 512) * 4 : 0);
    if (lds2 > 64 * 1024) {
        static const bool ok = hipFuncSetAttribute((const void*)latent_expand_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   96 * 1024) == hipSuccess &&
                               hipFuncSetAttribute((const void*)latent_expand_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   96 * 1024) == hipSuccess;
        if (!ok || lds2 > 96 * 1024) return 2;
    }
    const dim3 grid((unsigned)(((E + 63) / 64) * H * ((T_ + 15) / 16)));
    if (splits > 1) hipLaunchKernelGGL(latent_expand_kernel<true>, grid, dim3(256), lds2, s, a);
    else hipLaunchKernelGGL(latent_expand_kernel<false>, grid, dim3(256), lds2, s, a);
    return HYB_LAUNCH_OK();
}

}  // extern "C"
