// Residual-add + RMSNorm fused into the weight-streaming GEMM of a decode step, for weights
// that already carry the norm's scale vector (W' = W * gamma along K, folded once at load time):
//
//     r   = x + residual                      (rounded to the storage dtype, as add_rms_norm does)
//     out = rsqrt(mean(r^2) + eps) * (r . W'^T)            [optionally through SwiGLU]
//
// At decode sizes the norm kernel in front of a projection is pure launch latency (a few KB of
// data, ~5 us with its launch gap, twice per layer).  Because the per-row factor commutes with
// the matrix product, nothing has to be normalised BEFORE the k-loop:
//
//  * the A fragment of every k-step is formed in registers as x + residual (two 16-byte loads);
//  * the sum of squares comes from the matrix core as well: the A fragment of lane (m, q) is
//    bit-for-bit the B fragment of r^T, so one extra MFMA per k-step accumulates the Gram
//    matrix r r^T, whose diagonal is sum_k r[m][k]^2 - no VALU reduction, no extra pass;
//  * the epilogue multiplies the split-K-reduced sums by rsqrt(diag / K + eps);
//  * workgroup 0 also writes r (the new residual stream) to `res_out`, a buffer distinct from
//    the inputs, which the other workgroups are still reading.
#include "common.h"

using namespace mvl;

namespace {

constexpr int kCus = 256;
constexpr size_t kStagedLds = 112 * 1024;     // rows in LDS, besides at most 20 KB of partial sums
constexpr int kUnroll = 4;       // 4 k-steps in flight keep the kernel under 96 VGPRs (>= 2 workgroups per CU)

template <int CODE>
__device__ __forceinline__ u32x4_t add_round(u32x4_t a, u32x4_t b) {
    float fa[8], fb[8];
    unpack8<CODE>(a, fa);
    unpack8<CODE>(b, fb);
#pragma unroll
    for (int j = 0; j < 8; ++j) fa[j] += fb[j];
    return pack8<CODE>(fa);
}

// Sums of the waves' K slices, the row factor rsqrt(mean(r^2) + eps) from the Gram diagonals, bias
// and SwiGLU, store.
template <int CODE, int EPI, int WAVES>
__device__ __forceinline__ void finish_rows(
        float (&red)[WAVES][EPI == 1 ? 2 : 1][16][17], float (&diag)[WAVES][16],
        const f32x4_t (&acc)[EPI == 1 ? 2 : 1], const f32x4_t gram, int lane, int wv, int M, int K, float eps,
        const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, long o_stride, int n0, int up_row_offset) {
    using DT = DType<CODE>;
    constexpr int NB = EPI == 1 ? 2 : 1;
    const int c16 = lane & 15, q4 = lane >> 4;
    // split-K reduction; accumulator layout: col n = lane & 15, row m = 4 q + r.  The diagonal of
    // the Gram tile (row == col) sits in the lanes with 4 q <= c16 < 4 q + 4.
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wv][b][4 * q4 + r][c16] = acc[b][r];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (c16 == 4 * q4 + r) diag[wv][c16] = gram[r];
    __syncthreads();
    if (threadIdx.x < 256) {
        const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
        if (m < M) {
            float s[NB], ss = 0.f;
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) ss += diag[ww][m];
            const float rstd = rsqrtf(ss / (float)K + eps);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                s[b] = 0.f;
#pragma unroll
                for (int ww = 0; ww < WAVES; ++ww) s[b] += red[ww][b][m][n];
                s[b] *= rstd;
            }
            float r;
            if (EPI == 1) {
                if (bias != nullptr) {
                    s[0] += DT::to_float(bias[n0 + n]);
                    s[NB - 1] += DT::to_float(bias[up_row_offset + n0 + n]);
                }
                r = s[0] / (1.f + __expf(-s[0])) * s[NB - 1];
            } else {
                r = s[0] + (bias != nullptr ? DT::to_float(bias[n0 + n]) : 0.f);
            }
            out[(long)m * o_stride + n0 + n] = DT::from_float(r);
        }
    }
}

template <int CODE, int EPI, int WAVES, bool HAS_RES>
__global__ __launch_bounds__(WAVES * 64) void skinny_norm_gemm_kernel(
        const uint16_t* __restrict__ x, long x_stride, const uint16_t* __restrict__ res_in,
        long ri_stride, uint16_t* __restrict__ res_out, long ro_stride, float eps,
        const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
        uint16_t* __restrict__ out, long o_stride, int M, int K, int up_row_offset) {
    using DT = DType<CODE>;
    using vec8 = typename DT::vec8;
    constexpr int NB = EPI == 1 ? 2 : 1;
    __shared__ float red[WAVES][NB][16][17];
    __shared__ float diag[WAVES][16];

    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, q4 = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const int kslice = K / WAVES;
    const long koff = (long)wv * kslice + 8 * q4;
    const int row = min(c16, M - 1);
    const uint16_t* wp0 = w + (long)(n0 + c16) * K + koff;
    const uint16_t* wp1 = w + (long)(up_row_offset + n0 + c16) * K + koff;
    const uint16_t* xp = x + (long)row * x_stride + koff;
    const uint16_t* rp = HAS_RES ? res_in + (long)row * ri_stride + koff : nullptr;
    // workgroup 0 publishes r in a pass of its own, so that the k-loop carries no stores
    if (HAS_RES && res_out != nullptr && blockIdx.x == 0) {
        const int nchunk = K >> 3;
        for (int m = 0; m < M; ++m)
            for (int c = threadIdx.x; c < nchunk; c += WAVES * 64)
                reinterpret_cast<u32x4_t*>(res_out + m * ro_stride)[c] = add_round<CODE>(
                    reinterpret_cast<const u32x4_t*>(x + m * x_stride)[c],
                    reinterpret_cast<const u32x4_t*>(res_in + m * ri_stride)[c]);
    }

    f32x4_t acc[NB], gram = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    int k = 0;
    for (; k + 32 * kUnroll <= kslice; k += 32 * kUnroll) {
        u32x4_t bw[NB][kUnroll], ax[kUnroll], ar[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            bw[0][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wp0 + k + 32 * u));
            if (NB == 2)
                bw[NB - 1][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wp1 + k + 32 * u));
            ax[u] = *reinterpret_cast<const u32x4_t*>(xp + k + 32 * u);
            if (HAS_RES) ar[u] = *reinterpret_cast<const u32x4_t*>(rp + k + 32 * u);
        }
        __builtin_amdgcn_sched_barrier(0);          // all loads issued before the first use
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const u32x4_t r = HAS_RES ? add_round<CODE>(ax[u], ar[u]) : ax[u];
            const vec8 a = __builtin_bit_cast(vec8, r);
            gram = DT::mfma16(a, a, gram);
#pragma unroll
            for (int b = 0; b < NB; ++b)
                acc[b] = DT::mfma16(a, __builtin_bit_cast(vec8, bw[b][u]), acc[b]);
        }
    }
    for (; k < kslice; k += 32) {
        u32x4_t r = *reinterpret_cast<const u32x4_t*>(xp + k);
        if (HAS_RES) r = add_round<CODE>(r, *reinterpret_cast<const u32x4_t*>(rp + k));
        const vec8 a = __builtin_bit_cast(vec8, r);
        gram = DT::mfma16(a, a, gram);
        acc[0] = DT::mfma16(a, __builtin_bit_cast(vec8, *reinterpret_cast<const u32x4_t*>(wp0 + k)), acc[0]);
        if (NB == 2)
            acc[NB - 1] = DT::mfma16(a, __builtin_bit_cast(vec8, *reinterpret_cast<const u32x4_t*>(wp1 + k)),
                                     acc[NB - 1]);
    }

    finish_rows<CODE, EPI, WAVES>(red, diag, acc, gram, lane, wv, M, K, eps, bias, out, o_stride, n0, up_row_offset);
}

// The same with the rows formed once per workgroup instead of once per k-step and wave: every
// thread adds up some 16-byte chunks of x (or of the SLABS fp32 K-slices a split projection left,
// plus that projection's bias) and of the residual, rounds them, and stores them to LDS, from
// where the waves take their A fragments; the first weights are requested ahead of that and fly
// meanwhile, those of the next block of k-steps during the products of the present one.  There is a workgroup for
// every CU at most (132 registers and more: no second one fits beside it), which takes its 16 columns and those 256
// tiles on in turn: as many workgroups as tiles form the rows again for every round of 256.
//
// Bound by latency: at 8 rows, N = 4096, K = 1024 the weights (8 MB) take 1.6 us at the rate of a large
// copy, a launch 2, the whole 5.4 (5.6 with two slices to sum, where a norm kernel that sums them and the plain
// product take 8.4).  us with two slices, K = 1024, a workgroup per tile / per CU (norm kernel + product): 16 rows, N = 4096
// 8.5 / 6.8 (10.1), 4112 13.7 / 8.1 (10.4), 8192 15.2 / 8.9 (10.9); 1 row, N = 8192 8.5 / 6.8 (8.3); 16 rows from a
// tensor, N = 8192 11.3 / 8.6 (11.2).  Rows of 4096 are too much for every workgroup to form: 24 us at 4 rows and N = 6144 against 17.
template <int CODE, int EPI, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void skinny_norm_staged_kernel(
        const uint16_t* __restrict__ x, long x_stride, const float* __restrict__ slabs, int n_slabs,
        const uint16_t* __restrict__ x_bias, const uint16_t* __restrict__ res_in, long ri_stride,
        uint16_t* __restrict__ res_out, long ro_stride, float eps,
        const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias,
        uint16_t* __restrict__ out, long o_stride, int M, int K, int up_row_offset, int tiles) {
    using DT = DType<CODE>;
    using vec8 = typename DT::vec8;
    constexpr int NB = EPI == 1 ? 2 : 1;
    constexpr int U = 8 / NB;                    // k-steps per block: 8 weight loads in flight per lane
    __shared__ float red[WAVES][NB][16][17];
    __shared__ float diag[WAVES][16];
    extern __shared__ __attribute__((aligned(16))) uint16_t rows[];     // [M][K + 8]

    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, q4 = lane >> 4;
    const int kslice = K / WAVES;                // a multiple of 32
    const uint16_t* wp[NB];
    auto point = [&](int tile) {                 // this lane's weights of 16 columns
        wp[0] = w + (long)(16 * tile + c16) * K + (long)wv * kslice + 8 * q4;
        if (NB == 2) wp[NB - 1] = w + (long)(up_row_offset + 16 * tile + c16) * K + (long)wv * kslice + 8 * q4;
    };
    auto request = [&](int k, u32x4_t (&bw)[NB][U]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (k + 32 * u < kslice)         // uniform
                    bw[b][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wp[b] + k + 32 * u));
    };
    u32x4_t bw[NB][U];
    point(blockIdx.x);
    request(0, bw);

    const int per_row = K >> 3, pitch = K + 8;
    const long slab = (long)M * K;
    for (int i = threadIdx.x; i < M * per_row; i += WAVES * 64) {
        const int m = i / per_row, c = i - m * per_row;
        u32x4_t r;
        if (slabs != nullptr) {
            const float* p = slabs + (long)m * K + 8 * c;
            f32x4_t lo[4], hi[4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s < n_slabs) {               // uniform
                    lo[s] = *reinterpret_cast<const f32x4_t*>(p + s * slab);
                    hi[s] = *reinterpret_cast<const f32x4_t*>(p + s * slab + 4);
                }
            float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (res_in != nullptr)
                unpack8<CODE>(reinterpret_cast<const u32x4_t*>(res_in + m * ri_stride)[c], f);
            if (x_bias != nullptr) {
                float b[8];
                unpack8<CODE>(reinterpret_cast<const u32x4_t*>(x_bias)[c], b);
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] += b[j];
            }
#pragma unroll
            for (int s = 1; s < 4; ++s)
                if (s < n_slabs) { lo[0] += lo[s]; hi[0] += hi[s]; }
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] += j < 4 ? lo[0][j] : hi[0][j - 4];
            r = pack8<CODE>(f);
        } else {
            r = reinterpret_cast<const u32x4_t*>(x + m * x_stride)[c];
            if (res_in != nullptr)
                r = add_round<CODE>(r, reinterpret_cast<const u32x4_t*>(res_in + m * ri_stride)[c]);
        }
        *reinterpret_cast<u32x4_t*>(rows + m * pitch + 8 * c) = r;
        if (res_out != nullptr && blockIdx.x == 0)
            reinterpret_cast<u32x4_t*>(res_out + m * ro_stride)[c] = r;
    }
    __syncthreads();

    const uint16_t* rp = rows + min(c16, M - 1) * pitch + wv * kslice + 8 * q4;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {      // uniform
        f32x4_t acc[NB], gram = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < kslice; k += 32 * U) {
            u32x4_t next[NB][U];
            request(k + 32 * U, next);
            __builtin_amdgcn_sched_barrier(0);   // the next block's loads ahead of this one's waits
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + 32 * u < kslice) {       // uniform
                    const vec8 a = __builtin_bit_cast(vec8, *reinterpret_cast<const u32x4_t*>(rp + k + 32 * u));
                    gram = DT::mfma16(a, a, gram);
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        acc[b] = DT::mfma16(a, __builtin_bit_cast(vec8, bw[b][u]), acc[b]);
                }
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < U; ++u) bw[b][u] = next[b][u];
        }
        const bool more = tile + (int)gridDim.x < tiles;
        if (more) {
            point(tile + gridDim.x);
            request(0, bw);
        }
        finish_rows<CODE, EPI, WAVES>(red, diag, acc, gram, lane, wv, M, K, eps, bias, out, o_stride, 16 * tile,
                                      up_row_offset);
        if (more) __syncthreads();               // the sums have been read before the next columns' are written
    }
}

template <int CODE, int EPI, bool HAS_RES>
int launch(const void* x, long xs, const void* ri, long ris, void* ro, long ros, float eps,
           const void* w, const void* bias, void* out, long os, int M, int tiles, int K, int up_off,
           hipStream_t st) {
    auto X = (const uint16_t*)x; auto RI = (const uint16_t*)ri; auto RO = (uint16_t*)ro;
    auto W = (const uint16_t*)w; auto B = (const uint16_t*)bias; auto O = (uint16_t*)out;
    if (K % 256 == 0)
        skinny_norm_gemm_kernel<CODE, EPI, 8, HAS_RES><<<tiles, 8 * 64, 0, st>>>(
            X, xs, RI, ris, RO, ros, eps, W, B, O, os, M, K, up_off);
    else if (K % 128 == 0)
        skinny_norm_gemm_kernel<CODE, EPI, 4, HAS_RES><<<tiles, 4 * 64, 0, st>>>(
            X, xs, RI, ris, RO, ros, eps, W, B, O, os, M, K, up_off);
    else
        return -1;
    return MVL_CHECK_LAUNCH();
}

template <int CODE, int EPI>
int launch_r(const void* x, long xs, const void* slabs, int n_slabs, const void* xb, const void* ri, long ris,
             void* ro, long ros, float eps, const void* w, const void* bias, void* out, long os, int M, int tiles,
             int K, int up_off, hipStream_t st) {
    const size_t lds = (size_t)M * (K + 8) * 2;
    // up to 4 rows the loads of x and residual beside the weights cost less than the pass through LDS
    // and its barrier (us, per k-step / staged, N = 4096, K = 1024: 4.2 / 4.8 at 2 rows, 4.9 / 4.9 at 4, 6.1 / 5.4 at 8, 8.4 /
    // 6.4 at 16; K = 2048 6.7 / 7.2, 7.3 / 7.7, 8.2 / 8.4, 11.4 / 10.7)
    if ((slabs != nullptr || M > 4) && K % 256 == 0 && lds <= kStagedLds) {
        auto kern = skinny_norm_staged_kernel<CODE, EPI, 8>;
        static const hipError_t once = hipFuncSetAttribute(
            (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStagedLds);
        if (once != hipSuccess) return -1;
        kern<<<min(tiles, kCus), 8 * 64, lds, st>>>(
            (const uint16_t*)x, xs, (const float*)slabs, n_slabs, (const uint16_t*)xb, (const uint16_t*)ri, ris,
            (uint16_t*)ro, ros, eps, (const uint16_t*)w, (const uint16_t*)bias, (uint16_t*)out, os, M, K, up_off, tiles);
        return MVL_CHECK_LAUNCH();
    }
    if (slabs != nullptr) return -1;
    return ri != nullptr
        ? launch<CODE, EPI, true>(x, xs, ri, ris, ro, ros, eps, w, bias, out, os, M, tiles, K, up_off, st)
        : launch<CODE, EPI, false>(x, xs, ri, ris, ro, ros, eps, w, bias, out, os, M, tiles, K, up_off, st);
}

}  // namespace

// w: the projection weights with the norm's scale vector folded in.  res_in may be null (no
// residual yet: r = x); res_out may be null (r is not wanted) and must not alias x or res_in.
// Other arguments as mvl_skinny_gemm; M <= 16.  slabs != null: in place of x the n_slabs (1..4) fp32
// K-slices [n_slabs][M][K] of the projection before, x_bias (may be null) its bias; K a multiple of 256,
// M (K + 8) at most 57344.
extern "C" int mvl_skinny_norm_gemm(const void* x, long x_stride, const void* slabs, int n_slabs,
                                    const void* x_bias, const void* res_in, long ri_stride,
                                    void* res_out, long ro_stride, float eps, const void* w,
                                    const void* bias, void* out, long o_stride, int M, int N, int K,
                                    int epilogue, int dtype, void* stream) {
    if (M == 0) return 0;
    if (M > 16 || K % 128 != 0) return -1;
    if (slabs != nullptr && (n_slabs < 1 || n_slabs > 4)) return -1;
    if (res_out != nullptr && (res_out == x || res_out == res_in)) return -1;
    if (epilogue == 0 ? N % 16 != 0 : N % 32 != 0) return -1;
    auto st = (hipStream_t)stream;
    const int inter = N / 2;
#define MVL_SN(CODE) (epilogue == 0                                                                              \
        ? launch_r<CODE, 0>(x, x_stride, slabs, n_slabs, x_bias, res_in, ri_stride, res_out, ro_stride, eps, w,  \
                            bias, out, o_stride, M, N / 16, K, 0, st)                                            \
        : launch_r<CODE, 1>(x, x_stride, slabs, n_slabs, x_bias, res_in, ri_stride, res_out, ro_stride, eps, w,  \
                            bias, out, o_stride, M, inter / 16, K, inter, st))
    return dtype == 0 ? MVL_SN(0) : MVL_SN(1);
#undef MVL_SN
}
