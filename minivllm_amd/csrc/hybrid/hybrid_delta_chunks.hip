// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form
// The gated delta rule over prompt portions in chunks of 64 tokens on the matrix cores
// (hybrid_delta.hip has the recurrence itself and takes everything else):
//
//   S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
// With c_t = g_1 .. g_t (from the chunk's start) and W_ti = g_(i+1) .. g_t for i <= t, a chunk is
//
//   (I + L) U = diag(beta) (V - diag(c) K S_0),  L_ti = beta_t W_ti k_t . k_i below the diagonal;
//   O = diag(c) Q S_0 + A U,  A = (Q K^T) o W;   S_end = c_end S_0 + K^T diag(W_end) U
//
// (without the correction term U = diag(beta) V).  Every factor is a product of the decays the
// recurrence multiplies by, as in hybrid_chunks.hip.
//
// delta_weights_kernel, one workgroup per (chunk, group of heads): A and M = (I + L)^-1 diag(beta), which
// depend on no state, as operand fragments in three parts, and c, W_end.  The inverse goes by
// blocks of 16: those on the diagonal by substitution, the others by products of the fp32 instruction.
// delta_chunks_kernel, one workgroup of 8 waves per (sequence, head, 32 ET state columns), walks the
// chunks: U = M (V - diag(c) K S), O, S.  Wave w owns tokens 16 (w % 4) .. + 15, for which the first four
// waves form U and the others O, and of the state a quarter of the channels and half of the columns.  The
// state stays in registers; its parts, those of K and of the updates go through LDS; the next chunk's
// rows are on their way all the while.
//
// Everything is fp32 here, so every operand is cut into three parts of eight bits and a product is the sum
// of the six largest products of parts, on v_mfma_f32_16x16x32_bf16 with fp32 sums (2.7 times the rate of the
// fp32 instruction).  An instruction rounds its sum once, so the small products are summed apart from, or
// ahead of, the large one.  From 64 bits, 4 portions of 1024 tokens, decays of a trained range: outputs 1.0e-7,
// state 6.9e-8, against 1.1e-7 and 7.2e-8 token by token (2.3e-7 and 1.4e-7 with parts cut off and one sum for
// all products).
//
// An infinity or a NaN in a row of a chunk meets the zero weights of the tokens ahead of it, and its parts are NaN.
// It stays in the sums once it is there, so a portion whose outputs and state come out finite met none; any other is
// walked again from its first token by the recurrence itself (same workgroup, its own columns).
//
// 8 portions of 512..1024 tokens, 16 / 8 heads of 128: 37 + 150 us, against 645 us token by token.  The walk
// takes 9.7 us a chunk of 64 columns; its six phases between barriers use the matrix units, the
// vector units (cutting) and the LDS for about 2.5 us each and hardly overlap: one workgroup per CU is all that
// LDS and registers hold.  32 columns per workgroup 160 us; all waves in both roles, two workgroups per CU
// 213 us (registers spill); k's rows fetched a whole chunk ahead 193 us (spill).
#include "hybrid_chunks.h"

using namespace hyb;

namespace {

constexpr int C = 64;
constexpr int PAIRS = 6;                         // (16 queries, 32 keys) blocks at or below the diagonal
constexpr int FRAG = PAIRS * 3 * 1024;           // bytes of a C x C matrix as fragments in three parts
constexpr int SLOT = 2 * FRAG + 2 * C * 4;       // per (chunk, head): A, M, c, W_end
constexpr int NOWHERE = 0x7fffffff;

__device__ __forceinline__ int pair_of(int tb, int s) { return s ? 2 + tb : tb; }

#ifdef __HIP_DEVICE_COMPILE__
// eight neighbouring floats at a byte offset of a buffer (zeros out of its range)
__device__ __forceinline__ void load8(__amdgpu_buffer_rsrc_t b, int off, float* x) {
    const int4 u = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
    const int4 v = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 16, 0));
    x[0] = __int_as_float(u.x); x[1] = __int_as_float(u.y); x[2] = __int_as_float(u.z); x[3] = __int_as_float(u.w);
    x[4] = __int_as_float(v.x); x[5] = __int_as_float(v.y); x[6] = __int_as_float(v.z); x[7] = __int_as_float(v.w);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const float* p, int row, int nt, int width) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, ((nt - 1) * row + width) * 4, 0x00020000);
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

// bytes of delta_weights_kernel's LDS that hold first the k rows, then the triangular systems
template <int DP>
constexpr int weights_room() {
    constexpr int rows = 3 * C * DP * 2, systems = 2 * C * (C + 4) * 4;
    return rows > systems ? rows : systems;
}

template <int DP, bool DELTA>
__global__ void __launch_bounds__(256, 2)
delta_weights_kernel(DeltaChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KS = DP / 32, PITCH = C + 4;
    extern __shared__ __attribute__((aligned(256))) char smem[];
    // the k rows' images make room for the triangular systems: with both at once (86 KB) one workgroup was all a
    // CU held, and 112 chunks of 8 groups of two heads of 128 took 53 us instead of 37
    char* kparts = smem;                                         // [3] images of the chunk's k rows
    float* Lm = reinterpret_cast<float*>(smem);                  // [C][PITCH]
    float* Tm = Lm + C * PITCH;                                  // [C][PITCH]
    const int tid = threadIdx.x, lane = tid & 63, tb = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4;
    float* suf = reinterpret_cast<float*>(smem + weights_room<DP>()) + tb * 2 * C;   // per wave: [C] W to a block's end, [C] decays
    float* dec = suf + C;
    const int H = a.H, G = a.G, D = a.D, R = H / G, g = blockIdx.y;

    // the chunk's sequence: chunk c of sequence b has number cu_q[b] / C + b + c
    int b = -1;
    for (int i = 0; i < a.B; i += 64) {
        const bool before = i + lane < a.B && a.cu_q[min(i + lane, a.B - 1)] / C + i + lane <= (int)blockIdx.x;
        b += __popcll(__ballot(before));
    }
    if (b < 0 || a.slots[b] < 0) return;
    const int first = a.cu_q[b], n = a.cu_q[b + 1] - first, ch = blockIdx.x - (first / C + b);
    const int nt = min(C, n - ch * C);
    if (nt <= 0) return;
    const long t0 = (long)first + ch * C;

    const int t = 16 * tb + l16;
    f32x4 kk[4], qk[4];
    {
        const __amdgpu_buffer_rsrc_t kb = rows_of(a.k + t0 * G * D + (long)g * D, G * D, nt, D);
        const __amdgpu_buffer_rsrc_t qb = rows_of(a.q + t0 * G * D + (long)g * D, G * D, nt, D);
        bf16x8 kf[KS][3], qf[KS][3];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 32 * s + 8 * q4, off = d < D ? (t * G * D + d) * 4 : NOWHERE;
            float x[8], y[8];
            load8(kb, off, x);
            load8(qb, off, y);
            split8(x, kf[s]);
            split8(y, qf[s]);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<bf16x8*>(kparts + p * C * DP * 2 + t * DP * 2 + (((4 * s + q4) ^ rows16<DP>(t)) << 4)) = kf[s][p];
        }
        __syncthreads();
#pragma unroll
        for (int kb2 = 0; kb2 < 4; ++kb2) {
            kk[kb2] = {0.f, 0.f, 0.f, 0.f};
            qk[kb2] = kk[kb2];
            if (kb2 > tb) continue;
            const int row = 16 * kb2 + l16;
            Product pk, pq;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                bf16x8 x[3];
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    x[p] = *reinterpret_cast<const bf16x8*>(kparts + p * C * DP * 2 + row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4));
                if (DELTA) pk.add(x, kf[s]);
                pq.add(x, qf[s]);
            }
            kk[kb2] = pk.sum();
            qk[kb2] = pq.sum();
        }
    }
    for (int r = 0; r < R; ++r) {
        const int h = g * R + r;
        char* ws = a.ws + ((long)blockIdx.x * H + h) * SLOT;
        // lane = token: products of the decays inside blocks of 16; tokens behind the portion change nothing
        const float dc = lane < nt ? a.decay[(t0 + lane) * H + h] : 1.f;
        const float bt = lane < nt ? a.beta[(t0 + lane) * H + h] : 0.f;
        float pre = dc, sf = dc;
        static_for<0, 4>([&](auto ic) {
            constexpr int d = 1 << decltype(ic)::value;
            pre *= from_left<d>(pre, 1.f);
            sf *= from_right<d>(sf, 1.f);
        });
        sf = from_right<1>(sf, 1.f);
        float blk[4], ahead = 1.f, behind = 1.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            blk[k] = lane_of(pre, 16 * k + 15);
            if (k < q4) ahead *= blk[k];
            if (k > q4) behind *= blk[k];
        }
        if (tb == 0) {
            float* cw = reinterpret_cast<float*>(ws + 2 * FRAG);
            cw[lane] = pre * ahead;
            cw[C + lane] = sf * behind;
        }
        suf[lane] = sf;
        dec[lane] = dc;
        const float pt = __shfl(pre, t, kWave), beta_t = __shfl(bt, t, kWave);
        // W of this lane's query and keys 16 kb + 4 q4 + i
        float w[4][4], mid = 1.f;
#pragma unroll
        for (int kb = 3; kb >= 0; --kb) {
            if (kb > tb) {
#pragma unroll
                for (int i = 0; i < 4; ++i) w[kb][i] = 0.f;
            } else if (kb == tb) {
                const int i3 = 4 * q4 + 3;
                float ga[16];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float4 x = reinterpret_cast<const float4*>(dec + 16 * kb)[j];
                    ga[4 * j] = x.x; ga[4 * j + 1] = x.y; ga[4 * j + 2] = x.z; ga[4 * j + 3] = x.w;
                }
                float p = 1.f;
#pragma unroll
                for (int j = 4; j < 16; ++j) p *= ((j > i3) & (j <= l16)) ? ga[j] : 1.f;
                const float4 x = reinterpret_cast<const float4*>(dec + 16 * kb)[q4];
                const float ar[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int i = 3; i >= 0; --i) {
                    const bool seen = 4 * q4 + i <= l16;
                    w[kb][i] = seen ? p : 0.f;
                    p *= seen ? ar[i] : 1.f;
                }
            } else {
                const float f = pt * mid;
                const float4 x = reinterpret_cast<const float4*>(suf + 16 * kb)[q4];
                w[kb][0] = f * x.x; w[kb][1] = f * x.y; w[kb][2] = f * x.z; w[kb][3] = f * x.w;
                mid *= blk[kb];
            }
        }
        // a block of 16 queries and 32 keys as a fragment, in three parts
        auto put = [&](char* to, int s, const float* x) {
            bf16x8 p[3];
            split8(x, p);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                *reinterpret_cast<bf16x8*>(to + (pair_of(tb, s) * 3 + k) * 1024 + lane * 16) = p[k];
        };
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (2 * s > tb) continue;
            float x[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = qk[2 * s][i] * w[2 * s][i];
                x[4 + i] = qk[2 * s + 1][i] * w[2 * s + 1][i];
            }
            put(ws, s, x);
        }
        if constexpr (DELTA) {
            __syncthreads();                              // the images, or the last head's inverse, have been read
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                if (kb <= tb) {
                    float x[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x[i] = (kb < tb || 4 * q4 + i < l16) ? beta_t * w[kb][i] * kk[kb][i] : 0.f;
                    *reinterpret_cast<float4*>(Lm + t * PITCH + 16 * kb + 4 * q4) = make_float4(x[0], x[1], x[2], x[3]);
                }
            // the inverse of the block on the diagonal, a column per lane (four lanes share one)
            {
                float x[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float s0 = 0.f, s1 = 0.f;
                    float row[16];
#pragma unroll
                    for (int j = 0; j < (i + 3) / 4; ++j) {
                        const float4 y = reinterpret_cast<const float4*>(Lm + (16 * tb + i) * PITCH + 16 * tb)[j];
                        row[4 * j] = y.x; row[4 * j + 1] = y.y; row[4 * j + 2] = y.z; row[4 * j + 3] = y.w;
                    }
#pragma unroll
                    for (int m = 0; m < i; ++m) {
                        if (m & 1) s1 += row[m] * x[m];
                        else s0 += row[m] * x[m];
                    }
                    x[i] = (i == l16 ? 1.f : 0.f) - (s0 + s1);
                }
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (i / 4 == q4) Tm[(16 * tb + i) * PITCH + 16 * tb + l16] = x[i];
            }
            // the blocks below it, one diagonal after the other: -T_bb sum_m L_bm T_mk
            const float4 tt = reinterpret_cast<const float4*>(Tm + t * PITCH + 16 * tb)[q4];
            const float tbb[4] = {tt.x, tt.y, tt.z, tt.w};
#pragma unroll
            for (int lv = 1; lv < 4; ++lv) {
                __syncthreads();
                if (tb >= lv) {
                    const int k0 = tb - lv;
                    f32x4 p = {0.f, 0.f, 0.f, 0.f};
                    for (int m = k0; m < tb; ++m) {
                        const float4 l4 = reinterpret_cast<const float4*>(Lm + t * PITCH + 16 * m)[q4];
                        const float la[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            p = __builtin_amdgcn_mfma_f32_16x16x4f32(la[i], Tm[(16 * m + 4 * q4 + i) * PITCH + 16 * k0 + l16], p, 0, 0, 0);
                    }
                    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < 4; ++i) y = __builtin_amdgcn_mfma_f32_16x16x4f32(tbb[i], p[i], y, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) Tm[(16 * tb + 4 * q4 + i) * PITCH + 16 * k0 + l16] = -y[i];
                }
            }
            // M = inverse times beta of the column's token (this wave's rows are its own)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (2 * s > tb) continue;
                float x[8];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int kb = 2 * s + k;
                    const float4 y = kb <= tb ? reinterpret_cast<const float4*>(Tm + t * PITCH + 16 * kb)[q4] : make_float4(0.f, 0.f, 0.f, 0.f);
                    const float row[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[4 * k + i] = row[i] * __shfl(bt, 16 * kb + 4 * q4 + i, kWave);
                }
                put(ws + FRAG, s, x);
            }
        }
    }
#endif
}

template <int DP, int ET>
struct Lds {
    static constexpr int EB = 32 * ET, ROW = EB * 2;
    char k[3][C * DP * 2];             // images (rows16) of the chunk's k rows, in parts
    union {
        char s[3][EB * DP * 2];        // the state's parts, a row per state column
        struct { char x[3][C * ROW], u[3][C * ROW]; };   // rows of tokens: V - diag(c) K S, later diag(W_end) U; U
    };
    int lost;                          // an output or a state is not finite
};

// The portion's tokens one after the other: a thread has a column and some of the channels, sums through LDS
// (`red`: 4 KB).
template <int DP, int EB, bool DELTA>
__device__ __forceinline__ void walk_tokens(const DeltaChunks a, float* red) {
    constexpr int NS = 512 / EB, CH = DP / NS;
    const int b = blockIdx.x, h = blockIdx.y, slot = a.slots[b], first = a.cu_q[b], n = a.cu_q[b + 1] - first;
    const bool has_past = a.positions[first] > 0;
    const int c = threadIdx.x % EB, r = threadIdx.x / EB, e = blockIdx.z * EB + c, d0 = r * CH;
    const int H = a.H, G = a.G, D = a.D, E = a.E, g = h / (H / G);
    float* sp = a.state + ((long)slot * H + h) * D * E;
    float S[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) S[i] = has_past && d0 + i < D && e < E ? sp[(long)(d0 + i) * E + e] : 0.f;
    auto column_sum = [&](float* at, float x) {
        at[r * EB + c] = x;
        __syncthreads();
        x = 0.f;
        for (int i = 0; i < NS; ++i) x += at[i * EB + c];
        return x;
    };
    for (long t = first; t < first + n; ++t) {
        const float* kp = a.k + (t * G + g) * D + d0;
        const float* qp = a.q + (t * G + g) * D + d0;
        const float dec = a.decay[t * H + h];
        float u = e < E ? a.v[(t * H + h) * E + e] : 0.f, dot = 0.f, po = 0.f;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            S[i] *= dec;
            if (DELTA && d0 + i < D) dot += S[i] * kp[i];
        }
        if (DELTA) u -= column_sum(red, dot);
        u *= a.beta[t * H + h];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (d0 + i >= D) continue;
            S[i] += kp[i] * u;
            po += S[i] * qp[i];
        }
        // (the barriers of this sum and of the one above stand between a sum's reads and the next token's writes; with
        // this one alone two places take turns)
        po = column_sum(red + (DELTA ? 512 : (t & 1) * 512), po);
        if (r == 0 && e < E) a.o[(t * H + h) * E + e] = po;
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
        if (d0 + i < D && e < E) sp[(long)(d0 + i) * E + e] = S[i];
}

template <int DP, int ET, bool DELTA>
__global__ void __launch_bounds__(512, 2)
delta_chunks_kernel(DeltaChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KS = DP / 32, DT = DP / 64;
    using Mem = Lds<DP, ET>;
    constexpr int EB = Mem::EB, ROW = Mem::ROW;
    extern __shared__ __attribute__((aligned(256))) char smem[];
    Mem& L = *reinterpret_cast<Mem*>(smem);
    const int b = blockIdx.x, h = blockIdx.y, e0 = blockIdx.z * EB;
    const int H = a.H, G = a.G, D = a.D, E = a.E, g = h / (H / G);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tb = wave & 3, eh = wave >> 2;
    const int l16 = lane & 15, q4 = lane >> 4;
    clear_unowned(a.o, a.cu_q, a.slots, b, gridDim.x, a.T, H, h, E, e0, EB);
    const int slot = a.slots[b];
    const int first = a.cu_q[b], n = a.cu_q[b + 1] - first;
    if (slot < 0 || n <= 0) return;
    const bool has_past = a.positions[first] > 0;

    // S[j][x]: channels 16 (tb + 4 j) + 4 q4 + r of column e0 + 16 (eh ET + x) + l16
    f32x4 S[DT][ET];
    float* sp = a.state + ((long)slot * H + h) * D * E;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int x = 0; x < ET; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int d = 16 * (tb + 4 * j) + 4 * q4 + r, e = e0 + 16 * (eh * ET + x) + l16;
                S[j][x][r] = has_past && d < D && e < E ? sp[(long)d * E + e] : 0.f;
            }

    // `update` waves hold k and form U, the others hold q and form O
    const bool update = eh == 0;
    const int t = 16 * tb + l16;
    float raw[KS][8];
    bf16x8 xp[KS][3];                                // the chunk's k (or q) rows as operand, in parts
    // (addresses worked out ahead of the loop, for every phase, cost the registers that the products need: each phase
    // works its own out)
    auto again = [](int x) {
        asm volatile("" : "+v"(x));
        return x;
    };
    auto fetch = [&](int ch) {
        const int nt = min(C, n - ch * C);
        const __amdgpu_buffer_rsrc_t rows = rows_of((update ? a.k : a.q) + ((long)first + ch * C) * G * D + (long)g * D, G * D, nt, D);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 32 * s + 8 * q4;
            load8(rows, d < D ? (t * G * D + d) * 4 : NOWHERE, raw[s]);
        }
    };
    // the state's parts
    auto publish = [&]() {
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int x = 0; x < ET; ++x) {
                const int d = 16 * (tb + 4 * j) + 4 * q4, row = 16 * (eh * ET + x) + l16;
                put_parts(S[j][x], [&](int k) { return L.s[k] + row * DP * 2 + (((d >> 3) ^ rows16<DP>(row)) << 4) + (d & 4) * 2; });
            }
    };
    auto stash = [&]() {
        const int ln = again(lane), t = 16 * tb + (ln & 15), q4 = ln >> 4;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            split8(raw[s], xp[s]);
            if (update)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    *reinterpret_cast<bf16x8*>(L.k[k] + t * DP * 2 + (((4 * s + q4) ^ rows16<DP>(t)) << 4)) = xp[s][k];
        }
    };
    // a token row's 16-byte chunk in the x / u images
    auto place = [&](int row, int chunk) {
        return row * ROW + ((chunk ^ (ET == 1 ? (row >> 1 & 2) | (row >> 3 & 1) : rows16<64>(row))) << 4);
    };
    auto put_cols = [&](char (*im)[C * ROW], int x, f32x4 v) {        // this lane's token, four of the columns 16 x ..
        const int at = place(t, 2 * x + (q4 >> 1)) + (q4 & 1) * 8;
        put_parts(v, [&](int k) { return im[k] + at; });
    };
    // the parts of columns 16 x .. of an image as operand: rows row0 + 4 (quarter of the wave's lanes) + j, then
    // those `step` behind them
    auto get_cols = [&](char (*im)[C * ROW], int ln, int x, int row0, int step, bf16x8* p) {
        const int l16 = ln & 15, r0 = row0 + 4 * (ln >> 4) + (l16 >> 2), r1 = r0 + step, ch = 2 * x + ((l16 & 3) >> 1);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            p[k] = join(read_tr(im[k] + place(r0, ch) + (l16 & 1) * 8), read_tr(im[k] + place(r1, ch) + (l16 & 1) * 8));
    };
    constexpr int NE = 2 * ET;                       // 16-wide blocks of columns
    // the fragments m (of M or A) times columns 16 x .. of an image: the small products of parts first, so that
    // two steps round the whole sum
    auto chunk_product = [&](char (*im)[C * ROW], int ln, int x, const bf16x8 (*m)[3]) {
        bf16x8 p[2][3];
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s)
            if (2 * s <= tb) {
                get_cols(im, ln, x, 32 * s, 16, p[s]);
                y = mfma(p[s][2], m[s][0], y);
                y = mfma(p[s][0], m[s][2], y);
                y = mfma(p[s][1], m[s][1], y);
                y = mfma(p[s][1], m[s][0], y);
                y = mfma(p[s][0], m[s][1], y);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int s = 0; s < 2; ++s)
            if (2 * s <= tb) y = mfma(p[s][0], m[s][0], y);
        __builtin_amdgcn_sched_barrier(0);
        return y;
    };

    const int nchunks = (n + C - 1) / C;
    float seen = 0.f;                                // the sum of all outputs and states: finite if they are
    if (tid == 0) L.lost = 0;
    fetch(0);
    stash();
    publish();
    for (int ch = 0; ch < nchunks; ++ch) {
        const int left = n - ch * C;
        const long t0 = (long)first + ch * C;
        const char* ws = a.ws + ((long)(first / C + b + ch) * H + h) * SLOT;
        const float* cw = reinterpret_cast<const float*>(ws + 2 * FRAG);
        const float ct = cw[t], wt = cw[C + t], ce = cw[C - 1];
        f32x4 v[NE];
        bf16x8 mf[2][3];                                     // M for the update waves, A for the others
        if (update) {
            const __amdgpu_buffer_rsrc_t vb = rows_of(a.v + (t0 * H + h) * E + e0, H * E, min(C, left), E - e0);
#pragma unroll
            for (int x = 0; x < NE; ++x) {
                const int e = 16 * x + 4 * q4;
                v[x] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(vb, e0 + e < E ? (t * H * E + e) * 4 : NOWHERE, 0, 0));
            }
        }
        if (DELTA || !update)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (2 * s <= tb)
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        mf[s][k] = *reinterpret_cast<const bf16x8*>(ws + (update ? FRAG : 0) + (pair_of(tb, s) * 3 + k) * 1024 + lane * 16);
        const float bt = !DELTA && update && t < left ? a.beta[(t0 + t) * H + h] : 0.f;
        __syncthreads();                                     // the images of k and of the state are there
        f32x4 X[NE];                                         // K S (Q S)
        if (DELTA || !update) {
            const int ln = again(lane), l16 = ln & 15, q4 = ln >> 4;
#pragma unroll
            for (int x = 0; x < NE; ++x) {
                Product p;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const int row = 16 * x + l16;
                    bf16x8 sf[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        sf[k] = *reinterpret_cast<const bf16x8*>(L.s[k] + row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4));
                    p.add(sf, xp[s]);
                    __builtin_amdgcn_sched_barrier(0);       // (reads hoisted over the products cost registers)
                }
                X[x] = p.sum();
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ch + 1 < nchunks) fetch(ch + 1);                 // (into the registers of the operand)
        __syncthreads();                                     // the state's image has been read
        f32x4 U[NE];
        if constexpr (DELTA) {
            if (update)
#pragma unroll
                for (int x = 0; x < NE; ++x) put_cols(L.x, x, v[x] - ct * X[x]);
            __syncthreads();
            if (update) {
                const int ln = again(lane);
#pragma unroll
                for (int x = 0; x < NE; ++x) U[x] = chunk_product(L.x, ln, x, mf);
            }
        } else if (update) {
#pragma unroll
            for (int x = 0; x < NE; ++x) U[x] = bt * v[x];
        }
        if (update)
#pragma unroll
            for (int x = 0; x < NE; ++x) put_cols(L.u, x, U[x]);
        __syncthreads();                                     // U is there, x has been read
        if (update) {
#pragma unroll
            for (int x = 0; x < NE; ++x) put_cols(L.x, x, wt * U[x]);
        } else {
            const int ln = again(lane);
#pragma unroll
            for (int x = 0; x < NE; ++x) X[x] = ct * X[x] + chunk_product(L.u, ln, x, mf);
#pragma unroll
            for (int x = 0; x < NE; ++x) seen += (X[x][0] + X[x][1]) + (X[x][2] + X[x][3]);      // (zeros behind the portion)
            if (t < left)
#pragma unroll
                for (int x = 0; x < NE; ++x) {
                    const int e = e0 + 16 * x + 4 * q4;
                    if (e < E) *reinterpret_cast<f32x4*>(a.o + ((t0 + t) * H + h) * E + e) = X[x];
                }
        }
        __syncthreads();                                     // diag(W_end) U is there
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int x = 0; x < ET; ++x) S[j][x] *= ce;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int ln = again(lane), l16 = ln & 15, q4 = ln >> 4;
            bf16x8 up[ET][3];
#pragma unroll
            for (int x = 0; x < ET; ++x) get_cols(L.x, ln, eh * ET + x, 32 * s, 16, up[x]);
            const int row = 32 * s + 4 * q4 + (l16 >> 2);
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const int chunk = 2 * (tb + 4 * j) + ((l16 & 3) >> 1);
                bf16x8 kp[3];
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    kp[k] = join(read_tr(L.k[k] + row * DP * 2 + ((chunk ^ rows16<DP>(row)) << 4) + (l16 & 1) * 8),
                                 read_tr(L.k[k] + (row + 16) * DP * 2 + ((chunk ^ rows16<DP>(row + 16)) << 4) + (l16 & 1) * 8));
#pragma unroll
                for (int x = 0; x < ET; ++x) S[j][x] = mfma6(kp, up[x], S[j][x]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (ch + 1 < nchunks) {
            __syncthreads();                                 // k's and the updates' images have been read
            publish();
            __builtin_amdgcn_sched_barrier(0);
            stash();
        }
    }
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int x = 0; x < ET; ++x) seen += (S[j][x][0] + S[j][x][1]) + (S[j][x][2] + S[j][x][3]);
    if (seen * 0.f != 0.f) L.lost = 1;
    __syncthreads();
    if (L.lost) {
        __threadfence();                                     // (the outputs are written again, by other waves)
        __syncthreads();
        walk_tokens<DP, EB, DELTA>(arguments_anew<DeltaChunks>(), reinterpret_cast<float*>(smem));
        return;
    }
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int x = 0; x < ET; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int d = 16 * (tb + 4 * j) + 4 * q4 + r, e = e0 + 16 * (eh * ET + x) + l16;
                if (d < D && e < E) sp[(long)d * E + e] = S[j][x][r];
            }
#endif
}

template <class F>
int allow_lds(F* kernel, int bytes) {
    return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess ? 0 : 2;
}

template <int DP, bool DELTA>
int launch(const DeltaChunks& a, hipStream_t s) {
    constexpr int lds1 = weights_room<DP>() + 4 * 2 * C * 4;
    static const int ok1 = allow_lds(delta_weights_kernel<DP, DELTA>, lds1);
    if (ok1) return ok1;
    hipLaunchKernelGGL((delta_weights_kernel<DP, DELTA>), dim3(a.T / C + a.B, a.G), dim3(256), lds1, s, a);
    if (hipGetLastError() != hipSuccess) return 2;
#define WALK(ET)                                                                                       \
    do {                                                                                               \
        constexpr int lds = sizeof(Lds<DP, ET>);                                                       \
        static_assert(lds <= 160 * 1024);                                                              \
        static const int ok = allow_lds(delta_chunks_kernel<DP, ET, DELTA>, lds);                       \
        if (ok) return ok;                                                                             \
        hipLaunchKernelGGL((delta_chunks_kernel<DP, ET, DELTA>), dim3(a.B, a.H, (a.E + 32 * ET - 1) / (32 * ET)), \
                           dim3(512), lds, s, a);                                                      \
    } while (0)
    // 64 columns per workgroup share the cutting of k and q (307 us in all against 336 at 256 workgroups of
    // 64), where that leaves a workgroup for every CU; fewer are as fast with 32
    if (a.E > 32 && (long)a.B * a.H * ((a.E + 63) / 64) >= 256) WALK(2); else WALK(1);
#undef WALK
    return HYB_LAUNCH_OK();
}

}  // namespace

namespace hyb {

// A portion costs at least a chunk and a second launch: 64 sequences of 16 tokens (16 heads of 128) take 153 us
// against 158 token by token, of 64 tokens 226 against 430; one of 256 below the launches' 60 against 181,
// one of 16 no less than before.  So 20 rows per sequence, or a thousand beyond the first of each (a prompt
// next to many single tokens: the literal kernel walks it in 0.65 us a token).
long delta_chunks_bytes(const DeltaChunks& a) {
    if (a.T < 20L * a.B && a.T - a.B < 1024) return 0;
    if (!a.cu_q || a.B <= 0 || a.G <= 0 || a.H % a.G || a.D < 8 || a.D > 128 || a.D % 8 || a.E % 4 || a.E < 4) return 0;
    if (a.H > 65535 || a.T >= 1L << 30 || (long)a.G * a.D >= 1 << 22 || (long)a.H * a.E >= 1 << 22) return 0;
    if (((size_t)a.q | (size_t)a.k | (size_t)a.v | (size_t)a.o) % 16) return 0;
    return (a.T / C + a.B) * a.H * (long)SLOT;
}

int delta_chunks(const DeltaChunks& a, bool correct, hipStream_t s) {
    if (a.D <= 64) return correct ? launch<64, true>(a, s) : launch<64, false>(a, s);
    return correct ? launch<128, true>(a, s) : launch<128, false>(a, s);
}

}  // namespace hyb
