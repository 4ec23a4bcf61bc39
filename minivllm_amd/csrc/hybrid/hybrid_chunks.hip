// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form
// The matrix LSTM's recurrence over prompt portions in chunks of 64 tokens on the matrix cores
// (hybrid_recurrent.hip has the recurrence itself and takes everything else):
//
//   m_t = max(f_t + m_(t-1), i_t);  a_t = e^(f_t + m_(t-1) - m_t), b_t = e^(i_t - m_t);
//   S_t = a_t S_(t-1) + b_t k_t v_t^T,  n_t likewise with k_t alone;
//   o_t = S_t^T q_t / (max(|n_t . q_t|, e^(-m_t)) + 1e-6)
//
// With c_t = a_1 .. a_t (from the chunk's start) and W_ti = b_i a_(i+1) .. a_t for i <= t:
//
//   A = (Q K^T) o W;  O = diag(c) Q S_0 + A V;  n . q = c_t n_0 . q_t + sum_i A_ti
//   S_end = c_end S_0 + K^T diag(W_end) V,  n_end = c_end n_0 + K^T W_end
//
// Two kernels.  mlstm_weights_kernel, a workgroup per (chunk, head, 128 columns), takes m' of a chunk that begins with m =
// -inf, and so depends on no state: A' = (Q K^T) o W', A' V, the sums of A', W'_end.  With F_t = f_1 + .. + f_t, where the chunk
// follows a maximum m it is m_t = max(m + F_t, m'_t), c_t = e^(m + F_t - m_t) and W = e^(m'_t - m_t) W', one of the two
// factors being 1.  mlstm_chunks_kernel, a workgroup per (sequence, head, 32 state columns), walks the chunks.  Many small heads
// in bfloat16 are one kernel's, mlstm_whole_kernel.
//
// Every factor inside a chunk is a product of a and b, all <= 1: no quotients, no logarithms of products.  W' comes from the
// products inside blocks of 16 tokens: in a pair of different blocks it is (a .. to t inside its block) (whole blocks between)
// (a .. from i to its block's end) b_i, on the diagonal the running product.
//
// bfloat16 q, k, v are operands as they are; what is fp32 (floats, the weighted scores, the state, the weighted values) is cut
// into three parts of eight bits, all of its 24, and multiplied part by part on v_mfma_f32_16x16x32_bf16 with fp32 sums.
//
// The walk's workgroup is 16 waves: eight keep the state (wave w a quarter of the key channels, 16 of the columns, in
// registers) and lay its parts, the chunk's k and W_end v out in LDS, eight form the outputs (16 queries, 16 columns each) from
// the same images a chunk's turn later.  With two sets of images a chunk has one barrier.
//
// An infinity or a NaN in a row of a chunk meets the zero weights of the tokens ahead of it, and its parts are NaN.
// It stays in the sums once it is there, so a portion whose outputs and state come out finite met none; any other is
// walked again from its first token by the recurrence itself (same workgroup, its own columns).
//
// Bound by the vector instructions of the walk (splitting, addresses, exponentials: 270 a chunk in a wave of the state, 200 in
// the others, four waves per SIMD), 2.1 us a chunk.  8 portions of 512..1024 tokens, 8 heads of 128, bfloat16: 38 + 19 us and 11
// of the norm behind them, against 70 + 11 when one kernel did it all in every workgroup (the weights in each of its four
// column blocks, and twice in each: 4.4 us a chunk); floats 93 + 30 + 14 against 620 token by token.  The walk with both roles
// in eight waves: 45 us, floats 79.
#include "hybrid_chunks.h"

using namespace hyb;

namespace {

constexpr int C = 64;                  // tokens per chunk
constexpr int EB = 32;                 // state columns per workgroup of the walk
constexpr int EV = 128;                // value columns per workgroup of the first kernel
constexpr float NEG_INF = -__builtin_inff();
constexpr int NOWHERE = 0x7fffffff;

// what the first kernel leaves per (chunk, head) beside its outputs
struct Slot {
    float sum[C];              // sum_i A'_ti
    float F[C];                // f up to the token from the chunk's start
    float m[C];                // m'
    float wl[C];               // W'_end
};

__device__ __forceinline__ float logsigmoid_(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

#ifdef __HIP_DEVICE_COMPILE__
// Eight neighbouring elements of a row, as they come and as operands: bfloat16 is one, a float is cut into three parts.
template <typename T> struct Run;
template <> struct Run<bf16_t> {
    static constexpr int PARTS = 1;
    uint4 raw;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int off) {
        raw = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
    }
    __device__ __forceinline__ void parts(bf16x8* p) const { p[0] = __builtin_bit_cast(bf16x8, raw); }
};
template <> struct Run<float> {
    static constexpr int PARTS = 3;
    float x[8];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int off) {
        const int4 u = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
        const int4 v = __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(b, off, 16, 0));
        x[0] = __int_as_float(u.x); x[1] = __int_as_float(u.y); x[2] = __int_as_float(u.z); x[3] = __int_as_float(u.w);
        x[4] = __int_as_float(v.x); x[5] = __int_as_float(v.y); x[6] = __int_as_float(v.z); x[7] = __int_as_float(v.w);
    }
    __device__ __forceinline__ void parts(bf16x8* p) const { split8(x, p); }
};
// rows of `width` elements, `row` apart, `nt` of them; out of their range loads give zeros
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const void* p, long at, long row, int nt, int width) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>((const T*)p + at), 0, (int)(((nt - 1) * row + width) * sizeof(T)), 0x00020000);
}
// a product of the parts of an fp32 operand (a) and of one of T (b); small products have a sum of their own
template <typename T> struct Sum {
    Product p;
    __device__ __forceinline__ void add(const bf16x8* a, const bf16x8* b) {
        if constexpr (sizeof(T) == 2) {
            p.lo = mfma(a[2], b[0], p.lo);
            p.hi = mfma(a[0], b[0], p.hi);
            p.lo = mfma(a[1], b[0], p.lo);
        } else {
            p.add(a, b);
        }
    }
    __device__ __forceinline__ f32x4 sum() const { return p.sum(); }
};
#endif

// ---- what depends on no state: O' = A' V, the sums of A', F, m', W'_end
template <typename T, int DP>
__global__ void __launch_bounds__(256, sizeof(T) == 2 ? 3 : 2)
mlstm_weights_kernel(MlstmChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KS = DP / 32, NP = Run<T>::PARTS, KIM = C * DP * 2, VIM = C * EV * 2, VP = C * EV / 8 / 256;
    constexpr int ES = sizeof(T);
    extern __shared__ __attribute__((aligned(256))) char smem[];
    // [NP] images (rows16) of the chunk's k and v rows; three parts of both would leave a CU to one workgroup, so
    // those of v come after those of k
    char *kim = smem, *vim = NP == 1 ? smem + KIM : smem;
    __shared__ __attribute__((aligned(16))) float ga[C], gb[C], gbs[C];    // decay; input; input times the decays behind it in its block of 16
    __shared__ float gpre[C], gblk[4];                                     // decays up to the token in its block; a block's
    const int tid = threadIdx.x, lane = tid & 63, tb = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4, h = blockIdx.y, e0 = blockIdx.z * EV;
    const int H = a.H, D = a.D, E = a.E;
    // the chunk's sequence: chunk c of sequence b has number cu_q[b] / C + b + c
    int b = -1;
    for (int i = 0; i < a.B; i += 64) {
        const bool before = i + lane < a.B && a.cu_q[min(i + lane, a.B - 1)] / C + i + lane <= (int)blockIdx.x;
        b += __popcll(__ballot(before));
    }
    if (b < 0 || a.slots[b] < 0) return;
    const int first = a.cu_q[b], ch = blockIdx.x - (first / C + b);
    const int nt = min(C, a.cu_q[b + 1] - first - ch * C);
    if (nt <= 0) return;
    const long t0 = (long)first + ch * C;
    Slot& ws = reinterpret_cast<Slot*>(a.ws)[(long)blockIdx.x * H + h];

    const int t = 16 * tb + l16;
    const __amdgpu_buffer_rsrc_t qb = rows_of<T>(a.q, t0 * a.q_row + h * D, a.q_row, nt, D);
    const __amdgpu_buffer_rsrc_t kb = rows_of<T>(a.k, t0 * a.k_row + h * D, a.k_row, nt, D);
    const __amdgpu_buffer_rsrc_t vb = rows_of<T>(a.v, t0 * a.v_row + (long)h * E + e0, a.v_row, nt, E - e0);
    Run<T> qr[KS], kr[KS], vr[VP];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int d = 32 * s + 8 * q4;
        kr[s].load(kb, d < D ? (t * (int)a.k_row + d) * ES : NOWHERE);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int d = 32 * s + 8 * q4;
        qr[s].load(qb, d < D ? (t * (int)a.q_row + d) * ES : NOWHERE);
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
        const int c = i * 256 + tid, row = c / (EV / 8), e = c % (EV / 8) * 8;
        vr[i].load(vb, e0 + e < E ? (row * (int)a.v_row + e) * ES : NOWHERE);
    }
    auto put_v = [&]() {
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int c = i * 256 + tid, row = c / (EV / 8);
            bf16x8 p[NP];
            vr[i].parts(p);
#pragma unroll
            for (int k = 0; k < NP; ++k)
                *reinterpret_cast<bf16x8*>(vim + k * VIM + row * EV * 2 + (((c % (EV / 8)) ^ rows16<EV>(row)) << 4)) = p[k];
        }
    };
    if (tb == 0) {                                 // (the wave with the fewest keys) lane = token; those behind the portion change nothing
        const bool ok = lane < nt;
        const long at = (t0 + min(lane, nt - 1)) * a.g_row + h;
        const float i = ok ? a.cap * tanhf((ld((const T*)a.gi + at) + a.bi[h]) / a.cap) : NEG_INF;
        const float f = ok ? logsigmoid_(a.cap * tanhf((ld((const T*)a.gf + at) + a.bf[h]) / a.cap)) : 0.f;
        float F = f, M = i;                                    // inclusive scan of (sum of f, max), 16 tokens at a time
        static_for<0, 4>([&](auto dc) {
            constexpr int d = 1 << decltype(dc)::value;
            M = fmaxf(M, from_left<d>(M, NEG_INF) + F);
            F += from_left<d>(F, 0.f);
        });
        float before = NEG_INF, m0 = before, sum = 0.f, F0 = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k == q4) { m0 = before; F0 = sum; }
            const float Fk = lane_of(F, 16 * k + 15);
            before = fmaxf(lane_of(M, 16 * k + 15), before + Fk);
            sum += Fk;
        }
        const float m = fmaxf(M, m0 + F), mp = from_left<1>(m, m0);
        // (of the difference that decides the maximum, as in the recurrence, and not of m, whose own rounding would
        // come on top; not by fminf, which would lose a NaN)
        const float x = f + mp - i;
        const float fa = ok ? expf(x >= 0.f ? 0.f : x) : 1.f, fb = ok ? expf(x <= 0.f ? 0.f : -x) : 0.f;
        float pre = fa, suf = fa;
        static_for<0, 4>([&](auto dc) {
            constexpr int d = 1 << decltype(dc)::value;
            pre *= from_left<d>(pre, 1.f);
            suf *= from_right<d>(suf, 1.f);
        });
        suf = from_right<1>(suf, 1.f);
        float behind = 1.f;
#pragma unroll
        for (int k = 1; k < 4; ++k) {
            const float bk = lane_of(pre, 16 * k + 15);
            if (k > q4) behind *= bk;
        }
        ga[lane] = fa;
        gb[lane] = fb;
        gbs[lane] = fb * suf;
        gpre[lane] = pre;
        if (l16 == 15) gblk[q4] = pre;
        if (e0 == 0) {
            ws.F[lane] = F0 + F;
            ws.m[lane] = m;
            ws.wl[lane] = fb * suf * behind;
        }
    }
    bf16x8 qf[KS][NP];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        bf16x8 p[NP];
        kr[s].parts(p);
        qr[s].parts(qf[s]);
#pragma unroll
        for (int k = 0; k < NP; ++k)
            *reinterpret_cast<bf16x8*>(kim + k * KIM + t * DP * 2 + (((4 * s + q4) ^ rows16<DP>(t)) << 4)) = p[k];
    }
    if (NP == 1) put_v();
    __syncthreads();
    // ---- this wave's 16 queries against the key blocks from the diagonal down
    bf16x8 pf[2][3];
    float sum = 0.f, mid = 1.f;
    const float pre = gpre[t] * a.qscale;
    auto weighted = [&](int kb, float* x) {                               // x[r]: key 16 kb + 4 q4 + r
        const int row = 16 * kb + l16;
        f32x4 sc;
        if constexpr (NP == 1) {
            sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s)
                sc = mfma(*reinterpret_cast<const bf16x8*>(kim + row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4)), qf[s][0], sc);
        } else {
            Product p;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                bf16x8 kf[3];
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    kf[k] = *reinterpret_cast<const bf16x8*>(kim + k * KIM + row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4));
                p.add(kf, qf[s]);
            }
            sc = p.sum();
        }
        float w[4];
        if (kb == tb) {
            const int i3 = 4 * q4 + 3;
            float g[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 x4 = reinterpret_cast<const float4*>(ga + 16 * kb)[j];
                g[4 * j] = x4.x; g[4 * j + 1] = x4.y; g[4 * j + 2] = x4.z; g[4 * j + 3] = x4.w;
            }
            float p = 1.f;
#pragma unroll
            for (int j = 4; j < 16; ++j) p *= ((j > i3) & (j <= l16)) ? g[j] : 1.f;
            const float4 a4 = reinterpret_cast<const float4*>(ga + 16 * kb)[q4];
            const float4 b4 = reinterpret_cast<const float4*>(gb + 16 * kb)[q4];
            const float ar[4] = {a4.x, a4.y, a4.z, a4.w}, br[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int r = 3; r >= 0; --r) {
                const bool seen = 4 * q4 + r <= l16;
                w[r] = seen ? br[r] * p * a.qscale : 0.f;
                p *= seen ? ar[r] : 1.f;
            }
        } else {
            const float f = pre * mid;
            const float4 b4 = reinterpret_cast<const float4*>(gbs + 16 * kb)[q4];
            w[0] = f * b4.x; w[1] = f * b4.y; w[2] = f * b4.z; w[3] = f * b4.w;
            mid *= gblk[kb];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            x[r] = sc[r] * w[r];
            sum += x[r];
        }
    };
#pragma unroll
    for (int s = 1; s >= 0; --s) {
        if (2 * s > tb) continue;
        float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (2 * s + 1 <= tb) weighted(2 * s + 1, x + 4);
        weighted(2 * s, x);
        split8(x, pf[s]);
    }
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    if (q4 == 0 && e0 == 0) ws.sum[t] = sum;
    if (NP == 3) {
        __syncthreads();                                       // k's images have been read
        put_v();
        __syncthreads();
    }
    // ---- O': columns 16 n + 4 q4 + r of query t
#pragma unroll
    for (int n = 0; n < EV / 16; ++n) {
        if (e0 + 16 * n >= E) break;
        f32x4 O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 1; s >= 0; --s) {
            if (2 * s > tb) continue;
            const int row = 32 * s + 4 * q4 + (l16 >> 2), c = 2 * n + ((l16 & 3) >> 1);
            bf16x8 vf[NP];
#pragma unroll
            for (int k = 0; k < NP; ++k)
                vf[k] = join(read_tr(vim + k * VIM + row * EV * 2 + ((c ^ rows16<EV>(row)) << 4) + (l16 & 1) * 8),
                             read_tr(vim + k * VIM + (row + 16) * EV * 2 + ((c ^ rows16<EV>(row + 16)) << 4) + (l16 & 1) * 8));
            if constexpr (NP == 1) {
#pragma unroll
                for (int k = 2; k >= 0; --k) O = mfma(vf[0], pf[s][k], O);
            } else {
                O = mfma6(vf, pf[s], O);
            }
        }
        if (t < nt && e0 + 16 * n + 4 * q4 < E)
            *reinterpret_cast<f32x4*>(a.o + ((t0 + t) * H + h) * (long)E + e0 + 16 * n + 4 * q4) = O;
    }
#endif
}

template <int DP, int NP>
struct Lds {
    char k[NP][C * DP * 2];                // images (rows16) of the chunk's k rows
    char wv[3][C * EB * 2];                // W_end v in three parts, rows of 64 bytes, halves swapped where wv_at says so
    char s[3][EB * DP * 2];                // the state's parts, a row per state column
    char n[3][DP * 2];                     // the normaliser's parts
    alignas(16) uint16_t wp[4][C];         // W_end in three parts, zeros
};

// Place of a byte of a row of wv.  Transposed reads take 32 bytes of rows 0-7 (of 0-3 and 8-11): the halves of the
// second four are swapped, so that they are in the banks that the first four leave.
__device__ __forceinline__ int wv_at(int row, int byte) { return row * (EB * 2) + (byte ^ (row << 2 & 32)); }

// The portion's tokens one after the other: thread = a column and a GROUPS-th of the channels, sums through LDS
// (`red`: 16 bytes a thread).
template <typename T, int DP, int THREADS>
__device__ __forceinline__ void walk_tokens(const MlstmChunks a, float* red) {
    constexpr int GROUPS = THREADS / 32, CH = DP / GROUPS;
    const int b = blockIdx.x, h = blockIdx.y, e0 = blockIdx.z * EB, slot = a.slots[b];
    const long first = a.cu_q[b];
    const int n = a.cu_q[b + 1] - (int)first;
    const bool has_past = a.positions[first] > 0;
    const int c = threadIdx.x & 31, r = threadIdx.x >> 5, e = e0 + c, d0 = r * CH;
    const int H = a.H, D = a.D, E = a.E, ZG = (E + 15) / 16, z = e0 / 16;
    float* sp = a.state + ((long)slot * H + h) * D * E;
    float* np = a.nstate + (((long)slot * H + h) * ZG + z) * D;
    float* mp = a.mstate + ((long)slot * H + h) * ZG + z;
    float S[CH], N[CH], m = has_past ? *mp : 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        S[i] = has_past && d0 + i < D && e < E ? sp[(long)(d0 + i) * E + e] : 0.f;
        N[i] = has_past && d0 + i < D ? np[d0 + i] : 0.f;
    }
    for (int x = 0; x < n; ++x) {
        const long t = first + x;
        const float gi = a.cap * tanhf((ld((const T*)a.gi + t * a.g_row + h) + a.bi[h]) / a.cap);
        const float gf = logsigmoid_(a.cap * tanhf((ld((const T*)a.gf + t * a.g_row + h) + a.bf[h]) / a.cap));
        const float m2 = fmaxf(gf + m, gi), fs = expf(gf + m - m2), is = expf(gi - m2);
        m = m2;
        const float kv = e < E ? is * ld((const T*)a.v + t * a.v_row + (long)h * E + e) : 0.f;
        float po = 0.f, pn = 0.f;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (d0 + i >= D) continue;
            const float k = ld((const T*)a.k + t * a.k_row + (long)h * D + d0 + i);
            const float q = ld((const T*)a.q + t * a.q_row + (long)h * D + d0 + i) * a.qscale;
            S[i] = fs * S[i] + k * kv;
            po += S[i] * q;
            N[i] = fs * N[i] + is * k;
            pn += N[i] * q;
        }
        float* at = red + (x & 1) * (2 * THREADS);              // two of them: one barrier per token
        at[r * 32 + c] = po;
        at[THREADS + r * 32 + c] = pn;
        __syncthreads();
        if (r == 0 && e < E) {
            po = pn = 0.f;
            for (int i = 0; i < GROUPS; ++i) {
                po += at[i * 32 + c];
                pn += at[THREADS + i * 32 + c];
            }
            a.o[(t * H + h) * (long)E + e] = po / (fmaxf(fabsf(pn), expf(-m)) + 1e-6f);
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if (d0 + i >= D) continue;
        if (e < E) sp[(long)(d0 + i) * E + e] = S[i];
        if (c < 2 && z + c < ZG) np[c * D + d0 + i] = N[i];
    }
    if (r == 0 && c < 2 && z + c < ZG) mp[c] = m;
}

template <typename T, int DP>
__global__ void __launch_bounds__(1024)
mlstm_chunks_kernel(MlstmChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KS = DP / 32, DT = DP / 64, NP = Run<T>::PARTS, ES = sizeof(T);
    constexpr int PIECES = C * DP / 8 / 512;       // runs of a k image per thread
    constexpr int SETS = sizeof(Lds<DP, NP>) <= 56 * 1024 ? 2 : 1;     // of images
    extern __shared__ __attribute__((aligned(256))) char smem[];
    Lds<DP, NP>* L = reinterpret_cast<Lds<DP, NP>*>(smem);
    __shared__ int lost;                           // an output or a state is not finite
    const int b = blockIdx.x, h = blockIdx.y, e0 = blockIdx.z * EB;
    const int H = a.H, D = a.D, E = a.E;
    const int tid = threadIdx.x & 511, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool states = wave < 8;                  // keeps the state; the others form the outputs
    const int tb = wave & 3, et = wave >> 2 & 1;   // this wave's channels or queries; its 16 state columns
    const int l16 = lane & 15, q4 = lane >> 4;
    const int slot = a.slots[b];
    const long first = a.cu_q[b];
    const int n = a.cu_q[b + 1] - (int)first;
    clear_unowned(a.o, a.cu_q, a.slots, b, gridDim.x, a.T, H, h, E, e0, EB);
    if (slot < 0 || n <= 0) return;
    const bool has_past = a.positions[first] > 0;
    const int ZG = (E + 15) / 16, nchunks = (n + C - 1) / C;
    const int e = e0 + 16 * et + l16;
    float* sp = a.state + ((long)slot * H + h) * D * E;
    float* np = a.nstate + (((long)slot * H + h) * ZG + e0 / 16) * D;
    float m_run = has_past ? a.mstate[((long)slot * H + h) * ZG + e0 / 16] : 0.f;
    float seen = 0.f;                              // the sum of all outputs or states: finite if they are
    if (threadIdx.x == 0) lost = 0;
    auto slot_of = [&](int ch) -> const Slot& { return reinterpret_cast<const Slot*>(a.ws)[(first / C + b + ch) * H + h]; };
    // what the state of maximum m_run and the chunk's part are multiplied by, where the part's own maximum m is behind a
    // sum F of f (of the difference that decides, as in the recurrence; a NaN stays one)
    auto of_state = [&](float F, float m) { const float x = m_run + F - m; return expf(x >= 0.f ? 0.f : x); };
    auto of_chunk = [&](float F, float m) { const float x = m_run + F - m; return expf(x <= 0.f ? 0.f : -x); };
    f32x4 S[DT], N[DT];
    if (states) {
        // ---- S[j] holds channels 16 (tb + 4 j) + 4 q4 + r of column e, the first column of N a channel's normaliser (the
        // waves of the first 16 columns keep it)
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int d = 16 * (tb + 4 * j) + 4 * q4 + r;
                S[j][r] = has_past && d < D && e < E ? sp[(long)d * E + e] : 0.f;
                N[j][r] = has_past && d < D && l16 == 0 ? np[d] : 0.f;
            }
        // the next chunk on its way: rows behind the portion and columns behind a head are out of the buffers' range and
        // read as zeros
        constexpr int WP = 4;                      // the wave that lays out W_end (few products: no N)
        Run<T> kr[PIECES];
        f32x4 vr;
        float w_row, w_lane, F_e, m_e, c_end;
        int k_off[PIECES];
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int c = i * 512 + tid, row = c / (DP / 8), d = c % (DP / 8) * 8;
            k_off[i] = d < D ? (row * (int)a.k_row + d) * ES : NOWHERE;
        }
        const int v_off = e0 + (tid & 7) * 4 < E ? ((tid >> 3) * (int)a.v_row + (tid & 7) * 4) * ES : NOWHERE;
        auto fetch = [&](int ch) {
            const int nt = min(C, n - ch * C);
            const long t0 = first + (long)ch * C;
            const __amdgpu_buffer_rsrc_t kb = rows_of<T>(a.k, t0 * a.k_row + h * D, a.k_row, nt, D);
            const __amdgpu_buffer_rsrc_t vb = rows_of<T>(a.v, t0 * a.v_row + (long)h * E + e0, a.v_row, nt, E - e0);
            const Slot& w = slot_of(ch);
            F_e = w.F[C - 1];
            m_e = w.m[C - 1];
            w_row = w.wl[tid >> 3];
            if (wave == WP) w_lane = w.wl[lane];
#pragma unroll
            for (int i = 0; i < PIECES; ++i) kr[i].load(kb, k_off[i]);
            if constexpr (NP == 1) {
                const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(vb, v_off, 0, 0));
                vr = __builtin_bit_cast(f32x4, make_uint4(x.x, x.y, 0, 0));
            } else {
                vr = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(vb, v_off, 0, 0));
            }
        };
        // what was fetched last into LDS, and m_run behind it
        auto stash = [&](Lds<DP, NP>& l) {
            const float ahead = m_run + F_e - m_e, z = (lane & 1) ? -ahead : ahead, f = expf(z >= 0.f ? 0.f : z);
            c_end = lane_of(f, 0);
            const float r_end = lane_of(f, 1);
            m_run = fmaxf(m_run + F_e, m_e);
#pragma unroll
            for (int i = 0; i < PIECES; ++i) {
                const int c = i * 512 + tid, row = c / (DP / 8), at = row * DP * 2 + (((c % (DP / 8)) ^ rows16<DP>(row)) << 4);
                bf16x8 p[NP];
                kr[i].parts(p);
#pragma unroll
                for (int k = 0; k < NP; ++k) *reinterpret_cast<bf16x8*>(l.k[k] + at) = p[k];
            }
            f32x4 x = vr;                          // W_end v, four columns of a token per thread
            if constexpr (NP == 1) {
                const uint4 raw = __builtin_bit_cast(uint4, vr);
                x = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                     __uint_as_float(raw.y & 0xffff0000u)};
            }
            put_parts(x * (w_row * r_end), [&](int k) { return l.wv[k] + wv_at(tid >> 3, (tid & 7) * 8); });
            if (wave == WP) {
                float x = w_lane * r_end, y = 0.f;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const uint32_t w = rounded(x, y);
                    l.wp[k][lane] = (uint16_t)w;
                    rest(w, x, y);
                }
                l.wp[3][lane] = 0;
            }
        };
        // the state's parts: a row per column of the state
        auto publish = [&](Lds<DP, NP>& l) {
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const int d = 16 * (tb + 4 * j) + 4 * q4, row = 16 * et + l16;
                put_parts(S[j], [&](int k) { return l.s[k] + row * DP * 2 + (((d >> 3) ^ rows16<DP>(row)) << 4) + (d & 4) * 2; });
                if (et == 0 && l16 == 0) put_parts(N[j], [&](int k) { return l.n[k] + d * 2; });
            }
        };
        fetch(0);
        stash(L[0]);
        publish(L[0]);
        for (int ch = 0; ch < nchunks; ++ch) {
            Lds<DP, NP>& l = L[SETS == 2 ? ch & 1 : 0];
            __syncthreads();                                // the images are there; with two sets, the other has been read
            if (ch + 1 < nchunks) fetch(ch + 1);
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                S[j] *= c_end;
                N[j] *= c_end;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int row = 32 * s + 8 * q4 + (l16 >> 2);
                bf16x8 wf[3], pf[3], kf[DT][NP];            // pf: W_end in the first column, zeros in the others
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const char* at = l.wv[k] + wv_at(row, et * 32 + (l16 & 3) * 8);
                    wf[k] = join(read_tr(at), read_tr(at + 4 * EB * 2));
                    pf[k] = *reinterpret_cast<const bf16x8*>(&l.wp[l16 == 0 ? k : 3][32 * s + 8 * q4]);
                }
#pragma unroll
                for (int j = 0; j < DT; ++j) {
                    const int chunk = 2 * (tb + 4 * j) + ((l16 & 3) >> 1);
#pragma unroll
                    for (int k = 0; k < NP; ++k)
                        kf[j][k] = join(read_tr(l.k[k] + row * DP * 2 + ((chunk ^ rows16<DP>(row)) << 4) + (l16 & 1) * 8),
                                        read_tr(l.k[k] + (row + 4) * DP * 2 + ((chunk ^ rows16<DP>(row + 4)) << 4) + (l16 & 1) * 8));
                }
                // the products of parts, the small ones first; the sums in turn, as each waits for its last product.  (N in
                // all waves: a branch around it keeps its products apart from the others)
                constexpr int ORDER[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
                for (int i = 0; i < 6; ++i) {
                    const int x = ORDER[i][0], y = ORDER[i][1];
                    if (x >= NP) continue;
#pragma unroll
                    for (int j = 0; j < DT; ++j) {
                        S[j] = mfma(kf[j][x], wf[y], S[j]);
                        N[j] = mfma(kf[j][x], pf[y], N[j]);
                    }
                }
            }
            if (SETS == 1) __syncthreads();                 // everybody has read this chunk's images
            if (ch + 1 < nchunks) {
                Lds<DP, NP>& other = L[SETS == 2 ? ~ch & 1 : 0];
                stash(other);
                publish(other);
            }
        }
    } else {
        const int t = 16 * tb + l16;               // this wave's queries
        Run<T> qr[KS], qc[KS];
        f32x4 next_o, o_c;
        float sum_n, F_t, m_t, F_e, m_e, c_t, r_t, em, sum_c;
        int q_off[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) q_off[s] = 32 * s + 8 * q4 < D ? (t * (int)a.q_row + 32 * s + 8 * q4) * ES : NOWHERE;
        const int o_off = e0 + 16 * et + 4 * q4 < E ? (t * H * E + 16 * et + 4 * q4) * 4 : NOWHERE;
        auto fetch = [&](int ch) {
            const int nt = min(C, n - ch * C);
            const long t0 = first + (long)ch * C;
            const __amdgpu_buffer_rsrc_t qb = rows_of<T>(a.q, t0 * a.q_row + h * D, a.q_row, nt, D);
            const __amdgpu_buffer_rsrc_t ob = rows_of<float>(a.o, (t0 * H + h) * E + e0, (long)H * E, nt, E - e0);
            const Slot& w = slot_of(ch);
            F_t = w.F[t];
            m_t = w.m[t];
            sum_n = w.sum[t];
            F_e = w.F[C - 1];
            m_e = w.m[C - 1];
#pragma unroll
            for (int s = 0; s < KS; ++s) qr[s].load(qb, q_off[s]);
            next_o = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ob, o_off, 0, 0));
        };
        auto take = [&]() {
            c_t = of_state(F_t, m_t) * a.qscale;
            r_t = of_chunk(F_t, m_t);
            em = expf(-fmaxf(m_run + F_t, m_t));
            sum_c = sum_n * r_t;
            o_c = next_o * r_t;
            m_run = fmaxf(m_run + F_e, m_e);
#pragma unroll
            for (int s = 0; s < KS; ++s) qc[s] = qr[s];
        };
        fetch(0);
        take();
        for (int ch = 0; ch < nchunks; ++ch) {
            const Lds<DP, NP>& l = L[SETS == 2 ? ch & 1 : 0];
            __syncthreads();
            if (ch + 1 < nchunks) fetch(ch + 1);
            const int left = n - ch * C;
            f32x4 O = {0.f, 0.f, 0.f, 0.f};
            if (16 * tb < left) {
                Sum<T> qs;
                f32x4 nq = {0.f, 0.f, 0.f, 0.f};
                const int row = 16 * et + l16;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const int at = row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4);
                    bf16x8 sf[3], qf[NP];
                    qc[s].parts(qf);
#pragma unroll
                    for (int k = 0; k < 3; ++k) sf[k] = *reinterpret_cast<const bf16x8*>(l.s[k] + at);
                    const bf16x8 nf = *reinterpret_cast<const bf16x8*>(l.n[min(l16, 2)] + (4 * s + q4) * 16);
                    qs.add(sf, qf);
#pragma unroll
                    for (int k = NP - 1; k >= 0; --k) nq = mfma(nf, qf[k], nq);
                }
                const float nn = __shfl(nq[0] + (nq[1] + nq[2]), l16, kWave) * c_t;          // rows 0 .. 2 lie in lanes 0 .. 15
                const float den = 1.f / (fmaxf(fabsf(nn + sum_c), em) + 1e-6f);
                O = (qs.sum() * c_t + o_c) * den;
            }
            if (ch + 1 < nchunks) take();                   // (ahead of the store, which would be waited for as well)
            if (t < left) {
                if (e0 + 16 * et + 4 * q4 < E)
                    *reinterpret_cast<f32x4*>(a.o + ((first + ch * C + t) * H + h) * (long)E + e0 + 16 * et + 4 * q4) = O;
                seen += (O[0] + O[1]) + (O[2] + O[3]);
            }
            if (SETS == 1) __syncthreads();
        }
    }
    if (states)
#pragma unroll
    for (int j = 0; j < DT; ++j) seen += (S[j][0] + S[j][1]) + (S[j][2] + S[j][3]);
    if (seen * 0.f != 0.f) lost = 1;
    __syncthreads();
    if (lost) {
        __threadfence();                                    // (the outputs are written again, by other waves)
        __syncthreads();
        walk_tokens<T, DP, 1024>(arguments_anew<MlstmChunks>(), reinterpret_cast<float*>(smem));
        return;
    }
    // ---- the state after the portion
    if (!states) return;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * (tb + 4 * j) + 4 * q4 + r;
            if (d < D && e < E) sp[(long)d * E + e] = S[j][r];
            if (et == 0 && l16 == 0 && d < D) {
                np[d] = N[j][r];
                if (e0 / 16 + 1 < ZG) np[D + d] = N[j][r];
            }
        }
    if (wave == 0 && lane < 2 && e0 / 16 + lane < ZG) a.mstate[((long)slot * H + h) * ZG + e0 / 16 + lane] = m_run;
#endif
}

// ---- All of a portion in one kernel, for bfloat16 heads of up to 64 channels (`whole` has when): every workgroup of 32 columns
// works the weights out for itself, in eight waves that both keep the state and form the outputs, but two of it share a CU,
// which the walk above, with 16 waves of 82 registers, has to itself (at 64 registers it spills: 64 portions of 64, 16 heads of
// 64 x 64, 63 us; this 52).  Bound by the vector instructions around the products.
// per token of a chunk, in LDS
struct Gates {
    alignas(16) float a[C], b[C];          // decay, input
    alignas(16) float bs[C];               // b times the decays behind the token inside its block of 16
    float pre[C];              // the decays up to the token inside its block
    float c[C];                // ... from the chunk's start
    float wl[C];               // W_end
    float em[C];               // e^(-m)
    float blk[4];              // a block's decays
    alignas(16) uint16_t wp[3][C];         // wl in three parts
};

struct WholeLds {
    static constexpr int DP = 64;
    char q[C * DP * 2], k[C * DP * 2];     // images (rows16) of the chunk's rows
    char v[C * EB * 2];                    // rows of 64 bytes, halves swapped where v_at says so
    char wv[3][C * EB * 2];                // W_end v in three parts, likewise
    char s[3][EB * DP * 2];                // the state's parts, a row per state column
    char n[3][DP * 2];                     // the normaliser's parts
    Gates g;
    int lost;                              // an output or a state is not finite
};

// Place of a byte of a row of v (wv).  Transposed reads take 32 bytes of rows 0-7 (of 0-3 and 8-11): the halves of the
// second four are swapped, so that they are in the banks that the first four leave.
__device__ __forceinline__ int v_at(int row, int byte) { return row * (EB * 2) + (byte ^ (row << 3 & 32)); }
__global__ void __launch_bounds__(512, 4)                   // (two workgroups on a CU)
mlstm_whole_kernel(MlstmChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int DP = 64, KS = DP / 32;           // key channels; steps over them
    static_assert(C * DP / 8 == 512);              // a piece of 16 bytes of a q (or k) image per thread
    extern __shared__ __attribute__((aligned(256))) char smem[];
    WholeLds& L = *reinterpret_cast<WholeLds*>(smem);
    const int b = blockIdx.x, h = blockIdx.y, e0 = blockIdx.z * EB;
    const int H = a.H, D = a.D, E = a.E;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tb = wave & 3, et = wave >> 2;       // this wave's queries and channels; its 16 state columns
    const int l16 = lane & 15, q4 = lane >> 4;
    const int slot = a.slots[b];
    const long first = a.cu_q[b];
    const int n = a.cu_q[b + 1] - (int)first;
    clear_unowned(a.o, a.cu_q, a.slots, b, gridDim.x, a.T, H, h, E, e0, EB);
    if (slot < 0 || n <= 0) return;
    const bool has_past = a.positions[first] > 0;
    const int ZG = (E + 15) / 16;

    // ---- the state: S holds channels 16 tb + 4 q4 + r of column e, the first column of N a channel's normaliser (the waves of
    // the first 16 columns keep it)
    const int e = e0 + 16 * et + l16;
    f32x4 S, N;
    float* sp = a.state + ((long)slot * H + h) * D * E;
    float* np = a.nstate + (((long)slot * H + h) * ZG + e0 / 16) * D;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int d = 16 * tb + 4 * q4 + r;
        S[r] = has_past && d < D && e < E ? sp[(long)d * E + e] : 0.f;
        N[r] = has_past && d < D && l16 == 0 ? np[d] : 0.f;
    }
    float m_run = has_past ? a.mstate[((long)slot * H + h) * ZG + e0 / 16] : 0.f;

    // ---- the next chunk on its way: rows behind the portion and columns behind a head are out of the
    // buffers' range and read as zeros
    uint4 qr, kr;
    uint2 vr;
    float gi = 0.f, gf = 0.f;
    const int row = tid / (DP / 8), piece = tid % (DP / 8), d = piece * 8;
    const int q_off = d < D ? (row * (int)a.q_row + d) * 2 : NOWHERE, k_off = d < D ? (row * (int)a.k_row + d) * 2 : NOWHERE;
    const int v_off = e0 + (tid & 7) * 4 < E ? ((tid >> 3) * (int)a.v_row + (tid & 7) * 4) * 2 : NOWHERE;
    constexpr int GATES = 4;                       // the wave that works the gates out (few key blocks, no N)
    auto fetch = [&](int ch) {
        const int nt = min(C, n - ch * C);
        const long t0 = first + (long)ch * C;
        const __amdgpu_buffer_rsrc_t qb = rows_of<bf16_t>(a.q, t0 * a.q_row + h * D, a.q_row, nt, D);
        const __amdgpu_buffer_rsrc_t kb = rows_of<bf16_t>(a.k, t0 * a.k_row + h * D, a.k_row, nt, D);
        const __amdgpu_buffer_rsrc_t vb = rows_of<bf16_t>(a.v, t0 * a.v_row + (long)h * E + e0, a.v_row, nt, E - e0);
        qr = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qb, q_off, 0, 0));
        kr = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kb, k_off, 0, 0));
        vr = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(vb, v_off, 0, 0));
        if (wave == GATES) {
            const long t = t0 + min(lane, nt - 1);
            gi = ld((const bf16_t*)a.gi + t * a.g_row + h);
            gf = ld((const bf16_t*)a.gf + t * a.g_row + h);
        }
    };
    const float bi = a.bi[h], bf = a.bf[h];
    struct { float a, b, bs, pre, c, wl, em; } G;
    // the factors of every token of the chunk fetched last (lane = token)
    auto gates = [&](int ch) {
        const bool ok = lane < min(C, n - ch * C);             // tokens behind the portion change nothing
        const float i = ok ? a.cap * tanhf((gi + bi) / a.cap) : NEG_INF;
        const float f = ok ? logsigmoid_(a.cap * tanhf((gf + bf) / a.cap)) : 0.f;
        float F = f, M = i;                                    // inclusive scan of (sum of f, max), 16 tokens at a time
        static_for<0, 4>([&](auto dc) {
            constexpr int d = 1 << decltype(dc)::value;
            M = fmaxf(M, from_left<d>(M, NEG_INF) + F);
            F += from_left<d>(F, 0.f);
        });
        float before = m_run, m0 = m_run;                      // the maximum ahead of this lane's block
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k == q4) m0 = before;
            before = fmaxf(lane_of(M, 16 * k + 15), before + lane_of(F, 16 * k + 15));
        }
        m_run = before;
        const float m = fmaxf(M, m0 + F), mp = from_left<1>(m, m0);
        // (of the difference that decides the maximum, as in the recurrence, and not of m, whose own rounding would
        // come on top; not by fminf, which would lose a NaN)
        const float x = f + mp - i;
        const float fa = ok ? expf(x >= 0.f ? 0.f : x) : 1.f, fb = ok ? expf(x <= 0.f ? 0.f : -x) : 0.f;
        float pre = fa, suf = fa;
        static_for<0, 4>([&](auto dc) {
            constexpr int d = 1 << decltype(dc)::value;
            pre *= from_left<d>(pre, 1.f);
            suf *= from_right<d>(suf, 1.f);
        });
        suf = from_right<1>(suf, 1.f);
        float ahead = 1.f, behind = 1.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float bk = lane_of(pre, 16 * k + 15);
            if (k < q4) ahead *= bk;
            if (k > q4) behind *= bk;
        }
        G.a = fa; G.b = fb; G.bs = fb * suf; G.pre = pre; G.c = pre * ahead; G.wl = fb * suf * behind;
        G.em = expf(-m);
    };
    auto publish_gates = [&]() {
        Gates& g = L.g;
        g.a[lane] = G.a;
        g.b[lane] = G.b;
        g.bs[lane] = G.bs;
        g.pre[lane] = G.pre;
        g.c[lane] = G.c;
        g.wl[lane] = G.wl;
        g.em[lane] = G.em;
        if (l16 == 15) g.blk[q4] = G.pre;
        float x = G.wl, y = 0.f;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t w = rounded(x, y);
            g.wp[k][lane] = (uint16_t)w;
            rest(w, x, y);
        }
    };
    // what was fetched last into LDS
    auto stash = [&]() {
        const int at = row * DP * 2 + ((piece ^ rows16<DP>(row)) << 4);
        *reinterpret_cast<uint4*>(L.q + at) = qr;
        *reinterpret_cast<uint4*>(L.k + at) = kr;
        *reinterpret_cast<uint2*>(L.v + v_at(tid >> 3, (tid & 7) * 8)) = vr;
    };
    // the state's parts: a row per column of the state
    auto publish = [&]() {
        const int d = 16 * tb + 4 * q4, row = 16 * et + l16;
        put_parts(S, [&](int k) { return L.s[k] + row * DP * 2 + (((d >> 3) ^ rows16<DP>(row)) << 4) + (d & 4) * 2; });
        if (et == 0 && l16 == 0) put_parts(N, [&](int k) { return L.n[k] + d * 2; });
    };

    const int nchunks = (n + C - 1) / C;
    float seen = 0.f;                              // the sum of all outputs and states: finite if they are
    if (tid == 0) L.lost = 0;
    fetch(0);
    if (wave == GATES) {
        gates(0);
        publish_gates();
    }
    stash();
    publish();
    __syncthreads();
    for (int ch = 0; ch < nchunks; ++ch) {
        const Gates& g = L.g;
        if (ch + 1 < nchunks) fetch(ch + 1);
        {   // W_end v, four columns of a token per thread
            const uint2 raw = *reinterpret_cast<const uint2*>(L.v + v_at(tid >> 3, (tid & 7) * 8));
            const float w = g.wl[tid >> 3];
            const f32x4 x = {w * __uint_as_float(raw.x << 16), w * __uint_as_float(raw.x & 0xffff0000u),
                             w * __uint_as_float(raw.y << 16), w * __uint_as_float(raw.y & 0xffff0000u)};
            put_parts(x, [&](int k) { return L.wv[k] + wv_at(tid >> 3, (tid & 7) * 8); });
        }
        // ---- this wave's 16 queries: t = 16 tb + l16
        const int t = 16 * tb + l16, left = n - ch * C;
        if (16 * tb < left) {
        bf16x8 qf[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s)
            qf[s] = *reinterpret_cast<const bf16x8*>(L.q + t * DP * 2 + (((4 * s + q4) ^ rows16<DP>(t)) << 4));
        f32x4 O = {0.f, 0.f, 0.f, 0.f}, O1 = O, O2 = O, nq = O;
        {
            const int row = 16 * et + l16;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int at = row * DP * 2 + (((4 * s + q4) ^ rows16<DP>(row)) << 4);
                O2 = mfma(*reinterpret_cast<const bf16x8*>(L.s[2] + at), qf[s], O2);
                O1 = mfma(*reinterpret_cast<const bf16x8*>(L.s[1] + at), qf[s], O1);
                O = mfma(*reinterpret_cast<const bf16x8*>(L.s[0] + at), qf[s], O);
                nq = mfma(*reinterpret_cast<const bf16x8*>(L.n[min(l16, 2)] + (4 * s + q4) * 16), qf[s], nq);
            }
        }
        const float ct = g.c[t] * a.qscale;
        O = (O + (O1 + O2)) * ct;
        float den = __shfl(nq[0] + (nq[1] + nq[2]), l16, kWave) * ct;         // rows 0 .. 2 lie in lanes 0 .. 15
        float sum = 0.f, mid = 1.f;
        // key blocks from the diagonal down, two of 16 per step of the value product
        const float pre = g.pre[t] * a.qscale;
        auto weighted = [&](int kb, float* x) {                               // x[r]: key 16 kb + 4 q4 + r
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
            const int row = 16 * kb + l16;
#pragma unroll
            for (int i = 0; i < KS; ++i)
                s = mfma(*reinterpret_cast<const bf16x8*>(L.k + row * DP * 2 + (((4 * i + q4) ^ rows16<DP>(row)) << 4)), qf[i], s);
            float w[4];
            if (kb == tb) {
                const int i3 = 4 * q4 + 3;
                float ga[16];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float4 x4 = reinterpret_cast<const float4*>(g.a + 16 * kb)[j];
                    ga[4 * j] = x4.x; ga[4 * j + 1] = x4.y; ga[4 * j + 2] = x4.z; ga[4 * j + 3] = x4.w;
                }
                float p = 1.f;
#pragma unroll
                for (int j = 4; j < 16; ++j) p *= ((j > i3) & (j <= l16)) ? ga[j] : 1.f;
                const float4 a4 = reinterpret_cast<const float4*>(g.a + 16 * kb)[q4];
                const float4 b4 = reinterpret_cast<const float4*>(g.b + 16 * kb)[q4];
                const float ar[4] = {a4.x, a4.y, a4.z, a4.w}, br[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                for (int r = 3; r >= 0; --r) {
                    const bool seen = 4 * q4 + r <= l16;
                    w[r] = seen ? br[r] * p * a.qscale : 0.f;
                    p *= seen ? ar[r] : 1.f;
                }
            } else {
                const float f = pre * mid;
                const float4 b4 = reinterpret_cast<const float4*>(g.bs + 16 * kb)[q4];
                w[0] = f * b4.x; w[1] = f * b4.y; w[2] = f * b4.z; w[3] = f * b4.w;
                mid *= g.blk[kb];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x[r] = s[r] * w[r];
                sum += x[r];
            }
        };
        for (int s = tb >> 1; s >= 0; --s) {
            float x[8];
            if (2 * s + 1 <= tb) weighted(2 * s + 1, x + 4);
            else { x[4] = 0.f; x[5] = 0.f; x[6] = 0.f; x[7] = 0.f; }
            weighted(2 * s, x);
            bf16x8 p[3];
            split8(x, p);
            const char* at = L.v + v_at(32 * s + 4 * q4 + (l16 >> 2), et * 32 + (l16 & 3) * 8);
            const bf16x8 vf = join(read_tr(at), read_tr(at + 16 * EB * 2));
#pragma unroll
            for (int k = 2; k >= 0; --k) O = mfma(vf, p[k], O);
        }
        sum += __shfl_xor(sum, 16, kWave);
        sum += __shfl_xor(sum, 32, kWave);
        den = 1.f / (fmaxf(fabsf(den + sum), g.em[t]) + 1e-6f);
        O *= den;
        if (t < left && e0 + 16 * et + 4 * q4 < E)
            *reinterpret_cast<f32x4*>(a.o + ((first + ch * C + t) * H + h) * (long)E + e0 + 16 * et + 4 * q4) = O;
        seen += (O[0] + O[1]) + (O[2] + O[3]);              // (zeros behind the portion, as q is)
        }
        if (wave == GATES && ch + 1 < nchunks) gates(ch + 1);
        __syncthreads();                                    // W_end v is there
        const float ce = g.c[C - 1];
        f32x4 n = {0.f, 0.f, 0.f, 0.f};                     // the chunk's, a column for each part of W_end
        S *= ce;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int row = 32 * s + 8 * q4 + (l16 >> 2), piece = 2 * tb + ((l16 & 3) >> 1);
            bf16x8 wf[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const char* at = L.wv[k] + wv_at(row, et * 32 + (l16 & 3) * 8);
                wf[k] = join(read_tr(at), read_tr(at + 4 * EB * 2));
            }
            const bf16x8 kf = join(read_tr(L.k + row * DP * 2 + ((piece ^ rows16<DP>(row)) << 4) + (l16 & 1) * 8),
                                   read_tr(L.k + (row + 4) * DP * 2 + ((piece ^ rows16<DP>(row + 4)) << 4) + (l16 & 1) * 8));
#pragma unroll
            for (int k = 2; k >= 0; --k) S = mfma(kf, wf[k], S);
            if (et == 0) n = mfma(kf, *reinterpret_cast<const bf16x8*>(&g.wp[min(l16, 2)][32 * s + 8 * q4]), n);
        }
        if (et == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {                   // (what the first sum rounds off goes with the small ones)
                const float x = fmaf(N[r], ce, n[r]), off = fmaf(N[r], ce, n[r] - x);
                N[r] = x + (off + (from_right<1>(n[r], 0.f) + from_right<2>(n[r], 0.f)));
            }
        }
        if (ch + 1 < nchunks) {
            __syncthreads();                                // everybody has read this chunk's images
            if (wave == GATES) publish_gates();
            stash();
            publish();
            __syncthreads();
        }
    }
    seen += (S[0] + S[1]) + (S[2] + S[3]);
    if (et == 0 && l16 == 0) seen += (N[0] + N[1]) + (N[2] + N[3]);
    if (seen * 0.f != 0.f) L.lost = 1;
    __syncthreads();
    if (L.lost) {
        __threadfence();                                    // (the outputs are written again, by other waves)
        __syncthreads();
        walk_tokens<bf16_t, DP, 512>(arguments_anew<MlstmChunks>(), reinterpret_cast<float*>(smem));
        return;
    }
    // ---- the state after the portion
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int d = 16 * tb + 4 * q4 + r;
        if (d < D && e < E) sp[(long)d * E + e] = S[r];
        if (et == 0 && l16 == 0 && d < D) {
            np[d] = N[r];
            if (e0 / 16 + 1 < ZG) np[D + d] = N[r];
        }
    }
    if (wave == GATES && lane < 2 && e0 / 16 + lane < ZG) a.mstate[((long)slot * H + h) * ZG + e0 / 16 + lane] = m_run;
#endif
}

template <typename T, int DP>
int launch(const MlstmChunks& a, int B, hipStream_t s) {
    constexpr int NP = sizeof(T) == 2 ? 1 : 3, images = sizeof(Lds<DP, NP>), lds = images <= 56 * 1024 ? 2 * images : images;
    constexpr int rows = C * (DP > EV ? DP : EV) * 2, lds1 = NP == 1 ? C * (DP + EV) * 2 : 3 * rows;
    static_assert(lds <= 112 * 1024 && lds >= 16 * 1024 && lds1 <= 64 * 1024 - 2048);
    if (lds > 63 * 1024) {
        static const hipError_t once = hipFuncSetAttribute((const void*)mlstm_chunks_kernel<T, DP>,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (once != hipSuccess) return 2;
    }
    hipLaunchKernelGGL((mlstm_weights_kernel<T, DP>), dim3((unsigned)(a.T / C + B), a.H, (a.E + EV - 1) / EV), dim3(256), lds1, s, a);
    hipLaunchKernelGGL((mlstm_chunks_kernel<T, DP>), dim3(B, a.H, (a.E + EB - 1) / EB), dim3(1024), lds, s, a);
    return HYB_LAUNCH_OK();
}

int launch_whole(const MlstmChunks& a, hipStream_t s) {
    static_assert(sizeof(WholeLds) <= 64 * 1024);
    hipLaunchKernelGGL(mlstm_whole_kernel, dim3(a.B, a.H, (a.E + EB - 1) / EB), dim3(512), sizeof(WholeLds), s, a);
    return HYB_LAUNCH_OK();
}

long walks_of(const MlstmChunks& a) { return (long)a.B * a.H * ((a.E + EB - 1) / EB); }

// Whether one kernel does it all: where the walks are more than the CUs.  bfloat16, us, one / two kernels: 4 heads of 64 x 256
// (32 walks a sequence) 16 portions of 100 24 / 31, of 256 36 / 44, 64 of 32 42 / 50, of 128 72 / 74; 16 heads of 64 x 64 16 of
// 512 59 / 71, 64 of 64 52 / 66; 256 of 32, 4 heads of 48 x 40 40 / 49.  256 walks: 8 of 512, 16 heads of 64 x 64 47 / 41.
bool whole(const MlstmChunks& a, int dt) { return dt == 0 && a.D <= 64 && walks_of(a) > 256; }

}  // namespace

namespace hyb {

// A portion of a few tokens costs a whole chunk, so the rows must make up for the portions: by the walks (workgroups of
// mlstm_chunks_kernel), as few of either way take a call's 21 to 26 us and a token 0.3 us of it, and by how fast either way
// is.  Or one portion is long beside many short ones, and walked at 0.6 us a token.  us, chunks / tokens:
//   64 < D, bfloat16: 32 walks 24 tokens a portion 27 / 25, 32 26 / 28; 256 16 27 / 22, 24 27 / 28; 512 12 27 / 24, 16 26 / 26; 1024 10 35 /
//   37; 4096 10 97 / 124; 8192 8 178 / 214; floats: 32 walks 16 26 / 26, 24 26 / 31; 256 12 26 / 25, 16 26 / 28; 512 10 32 / 32; 1024
//   10 46 / 56; 8192 8 245 / 346
//   up to 64, bfloat16: 256 walks 32 27 / 26, 48 26 / 33; 512 16 24 / 21, 24 24 / 26; 1024 16 25 / 24, 24 26 / 32; 2048 12 38 / 35, 16
//   38 / 39; 8192 16 121 / 127; floats: 128 32 28 / 25, 48 26 / 33; 512 24 26 / 28; 1024 24 38 / 33, 32 38 / 38; 4096 16 106 / 84, 24 109 / 110
//   one portion beside single tokens: 255 of these, 8 heads of 128 x 128, bfloat16, one of 64 176 / 235, of 256 198 / 597; 127 and 4
//   of 48 x 40 one of 64 24 / 53, of 1024 81 / 666; 255 and 16 of 64 x 64, floats, one of 96 197 / 144, of 1024 329 / 794
static long tokens_that_pay(const MlstmChunks& a, int dt) {
    const long walks = walks_of(a);
    if (a.D > 64) {
        if (walks >= 512) return walks >= 4096 ? 8 : walks >= 1024 || dt == 2 ? 10 : 16;
        return dt == 2 ? (walks >= 256 ? 16 : 24) : (walks >= 256 ? 24 : 32);
    }
    if (dt == 2) return walks >= 256 ? 32 : 40;
    return walks > 1024 ? 16 : walks > 256 ? 24 : 40;
}

bool mlstm_chunks_pay(const MlstmChunks& a, int longest, int dt) {
    const long walks = walks_of(a), alone = 40 + walks / (dt == 2 && a.D <= 64 ? 64 : 200);
    return a.T >= tokens_that_pay(a, dt) * a.B || (longest > 0 ? longest >= alone : a.T - a.B >= 1024);
}

long mlstm_chunks_bytes(const MlstmChunks& a, int dt) {
    const int B = a.B;
    if (!a.cu_q || B <= 0 || a.D < 8 || a.D > 128 || a.D % 8 || a.E % 8 || a.H > 65535 || (dt != 0 && dt != 2)) return 0;
    if (((size_t)a.q | (size_t)a.k | (size_t)a.v) % 16) return 0;
    for (long row : {a.q_row, a.k_row, a.v_row})
        if (row % (dt == 0 ? 8 : 4) || row < 0 || row >= (dt == 0 ? 1 << 23 : 1 << 22)) return 0;      // (64 rows are addressed in 31 bits)
    if ((long)a.H * a.E >= 1 << 22) return 0;
    return whole(a, dt) ? 256 : (a.T / C + B) * (long)a.H * (long)sizeof(Slot);
}

int mlstm_chunks(const MlstmChunks& a, int dt, hipStream_t s) {
    if (whole(a, dt)) return launch_whole(a, s);
    if (dt == 0) return a.D <= 64 ? launch<bf16_t, 64>(a, a.B, s) : launch<bf16_t, 128>(a, a.B, s);
    return a.D <= 64 ? launch<float, 64>(a, a.B, s) : launch<float, 128>(a, a.B, s);
}

}  // namespace hyb
