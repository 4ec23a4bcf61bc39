// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form
// Recurrences with a decay per key channel over prompt portions, in chunks of 64 tokens, all chunks side by side
// (hybrid_recurrent.hip has the recurrences themselves and takes everything else):
//
//   GLA     S_t = diag(g_t) S_(t-1) + k_t v_t^T;   o_t = S_t^T q_t
//   WKV     o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t;   S_t = diag(g_t) S_(t-1) + k_t v_t^T
//
// With P_d(s..t) = g_(s+1)d .. g_td (GLA; WKV: without g_t) and c_t = P(start..t), a chunk is
//
//   A_ts = sum_d q_td k_sd P_d(s..t),  s <= t   (WKV: s < t, and sum_d q_td u_d k_td on the diagonal);
//   O = A V + (Q o c) S_0;   S_end = diag(c_end) S_0 + (K o P(..end))^T V
//
// Three kernels: channel_chunk_kernel, a workgroup per (chunk, head), forms A V, Q o c and (K o P)^T V, none of which
// depend on a state; channel_state_kernel runs over the chunks of a sequence, element by element of the state, and leaves
// every chunk's S_0; channel_out_kernel adds (Q o c) S_0 and, where asked for, norms and gates the heads' outputs.
//
// Every P is a product of decays, all <= 1: no quotients, no logarithms of products.  For tokens of different blocks of
// 16 it is (.. to t inside its block) (whole blocks between) (.. from s to its block's end), factors that go to q and
// k, and the sum over d is a matrix product; inside a block it is the running product, on the vector units.
//
// What is fp32 (weighted q, k, scores, state) is cut into three parts of eight bits, all of its 24, and multiplied part by
// part on v_mfma_f32_16x16x32_bf16, as in hybrid_delta_chunks.hip; v is bfloat16 as it is, or cut likewise.
//
// An infinity or a NaN meets the zero weights of the tokens ahead of it, and its parts are NaN.  So the first two kernels
// look at what goes in: with every operand up to LARGE and every S_0 up to LARGE_STATE all sums are finite, here and token
// by token.  A portion with any other is walked by the recurrence itself, in the third kernel, by the workgroup of its
// first chunk.  (A flag of the third kernel's own would have to be seen by a workgroup behind all others: with a fence and
// a ticket in each that kernel took 115 us instead of 26, a fourth kernel is 3 us more.)
//
// 8 portions of 512..1024 tokens, 8 heads of 64 x 128, layer with its norm: 333 us token by token, now 80 (38 + 12 + 26 in the
// kernels: decays, scores inside blocks and cutting on the vector units; 5 TB/s; 4.6 TB/s over 120 MB); one of 1024
// 308 -> 38.  WKV, 16 heads of 64: 334 -> 100, 310 -> 41.  From 64 bits: outputs 1.5e-7, state 1.2e-7, token by token 1.6e-7
// and 1.3e-7.
#include "hybrid_chunks.h"

using namespace hyb;

namespace {

constexpr int C = 64;

// ---- the workspace of a (chunk, head), in floats
template <int DP, int EP>
struct Item {
    static constexpr int Q = 0;                    // Q o c as operands: [block of 16 tokens][32 channels][lane][8]
    static constexpr int O = Q + C * DP;           // A V: [block of 16 tokens][16 columns][lane][4]
    static constexpr int S = O + C * EP;           // the chunk's own part of S_end, then S_0: [16 channels][16 columns][lane][4]
    static constexpr int CE = S + DP * EP;         // c_end
    static constexpr int FLAG = CE + DP;           // an operand that is not finite, or large, was met
    static constexpr int SIZE = FLAG + 4;
};
__host__ __device__ inline long item_count(long T, int B) { return T / C + B; }

constexpr float LARGE = 1e9f, LARGE_STATE = 1e25f;      // 64 channels of q u k v: 6e37

// sigmoid(z)^(1/tau) and exp(-exp(z)), as the recurrence has them: log1pf and not the logarithm of 1 + e^-|z|, whose rounding is
// the whole of a slow decay's error and adds up over a portion (600 tokens of one decay each, tau 0.25: outputs 2.7e-5 from 64 bits,
// 4.3e-6 with log1pf and token by token; the layer's call below 73 us and 80).
template <int RULE>
__device__ __forceinline__ float decay_of(float z, float tau_inv) {
    if (RULE == CHANNEL_WKV) return expf(-expf(z));
    return expf((fminf(z, 0.f) - log1pf(expf(-fabsf(z)))) * tau_inv);
}

// the sequence that chunk slot `i` belongs to (chunk c of sequence b has slot cu_q[b] / C + b + c), -1: none
__device__ __forceinline__ int sequence_of(const int* cu_q, int B, int i) {
    const int lane = threadIdx.x & 63;
    int b = -1;
    for (int x = 0; x < B; x += 64) {
        const bool before = x + lane < B && cu_q[min(x + lane, B - 1)] / C + x + lane <= i;
        b += __popcll(__ballot(before));
    }
    return b;
}

#ifdef __HIP_DEVICE_COMPILE__
// image of rows of 64 numbers (128 bytes) in 16-byte chunks
__device__ __forceinline__ int at64(int row, int chunk) { return row * 128 + ((chunk ^ rows16<64>(row)) << 4); }
template <int EP>
__device__ __forceinline__ int at_v(int row, int chunk) { return row * EP * 2 + ((chunk ^ rows16<EP>(row)) << 4); }
#endif

template <typename TI, int RULE, int DP, int EP>
struct ChunkLds {
    static constexpr int P = DP + 4, NP = sizeof(TI) == 2 ? 1 : 3;
    union {
        float q[4][16][P];                         // q, then q with the decays from its block's start
        char v[C * EP * 2];                        // v where it is bfloat16
    };
    char vp[NP == 1 ? 1 : 3][NP == 1 ? 16 : C * EP * 2];       // v in parts
    union {
        float ka[4][2][16][P];                     // k and the decays
        char kt[3][DP * 128];                      // k with decays to a block's (then the chunk's) end: parts, a row per channel
    };
    float blk[4][DP];                              // a block's decays
    alignas(16) float diag[4][16][20];             // scores inside a block [t][s]
};

template <typename TI, int RULE, int DP, int EP>
__global__ void __launch_bounds__(256, sizeof(TI) == 2 ? 3 : 2)
channel_chunk_kernel(const ChannelChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    using Mem = ChunkLds<TI, RULE, DP, EP>;
    using It = Item<DP, EP>;
    constexpr int P = Mem::P, NP = Mem::NP, NC = DP / 64, KS = DP / 32, DC = DP / 4;
    extern __shared__ __attribute__((aligned(256))) char smem[];
    Mem& L = *reinterpret_cast<Mem*>(smem);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4, h = blockIdx.y;
    const int H = a.H, D = a.D, E = a.E;
    const int b = sequence_of(a.cu_q, a.B, blockIdx.x);
    if (b < 0 || a.slots[b] < 0) return;
    const int first = a.cu_q[b], n = a.cu_q[b + 1] - first, ch = blockIdx.x - (first / C + b);
    const int nt = min(C, n - ch * C);
    if (nt <= 0) return;
    const long t0 = (long)first + ch * C;
    float* ws = a.ws + ((long)blockIdx.x * H + h) * It::SIZE;
    // the largest magnitude met, as bits: infinities and NaN are larger than any number
    uint32_t top = 0;
    auto see = [&](float x) { top = max(top, __float_as_uint(x) & 0x7fffffffu); };

    // ---- rows: lane = channel, wave = block of 16 tokens; tokens behind the portion change nothing
    const TI* qp = (const TI*)a.q + t0 * a.q_row + (long)h * D;
    const TI* kp = (const TI*)a.k + t0 * a.k_row + (long)h * D;
    const TI* ap = (const TI*)a.a + t0 * a.a_row + (long)h * D;
    const TI* vp = (const TI*)a.v + t0 * a.v_row + (long)h * E;
    float k[NC][16], g[NC][16];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int d = lane + 64 * i, dd = min(d, D - 1);
        TI qr[16], kr[16], ar[16];
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const int t = min(16 * w + x, nt - 1);
            qr[x] = qp[t * a.q_row + dd];
            kr[x] = kp[t * a.k_row + dd];
            ar[x] = ap[t * a.a_row + dd];
        }
        const float bias = a.a_bias[h * D + dd];
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const bool in = 16 * w + x < nt && d < D;
            k[i][x] = in ? ld(kr + x) : 0.f;
            g[i][x] = in ? decay_of<RULE>(ld(ar + x) + bias, a.tau_inv) : 1.f;
            const float q = in ? ld(qr + x) * a.qscale : 0.f;
            see(q);
            see(k[i][x]);
            see(g[i][x]);
            L.q[w][x][d] = q;
            L.ka[w][0][x][d] = k[i][x];
            L.ka[w][1][x][d] = g[i][x];
        }
    }
    // v, eight columns a thread and step: bfloat16 stays in registers until q's rows make room for it
    constexpr int VP = C * EP / 8 / 256;
    uint4 vr[NP == 1 ? VP : 1];
#pragma unroll
    for (int i = 0; i < VP; ++i) {
        const int c = tid + 256 * i, row = c / (EP / 8), e = c % (EP / 8) * 8;
        const bool in = row < nt && e < E;
        if constexpr (NP == 1) {
            vr[i] = make_uint4(0, 0, 0, 0);
            if (in) vr[i] = *reinterpret_cast<const uint4*>(vp + row * a.v_row + e);
        } else {
            float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (in) load_run<TI, 8>(vp + row * a.v_row + e, x);
#pragma unroll
            for (int y = 0; y < 8; ++y) see(x[y]);
            bf16x8 p[3];
            split8(x, p);
#pragma unroll
            for (int y = 0; y < 3; ++y) *reinterpret_cast<bf16x8*>(L.vp[y] + at_v<EP>(row, e >> 3)) = p[y];
        }
    }
    lanes_meet();                                               // (a wave reads its own block's rows)
    // ---- scores inside the block: lane = (key s, a quarter of the channels), s + j is the query of step j
    {
        float kd[DC], p[16];
        const int s = l16, c0 = q4 * DC;
#pragma unroll
        for (int d = 0; d < DC; d += 4) *reinterpret_cast<float4*>(kd + d) = *reinterpret_cast<const float4*>(&L.ka[w][0][s][c0 + d]);
        if constexpr (RULE == CHANNEL_WKV) {
            float x = 0.f;
#pragma unroll
            for (int d = 0; d < DC; ++d) {
                const float u = a.bonus[h * D + min(c0 + d, D - 1)];
                see(u);
                x += L.q[w][s][c0 + d] * u * kd[d];
            }
            p[0] = x;
        }
#pragma unroll
        for (int j = RULE == CHANNEL_WKV ? 1 : 0; j < 16; ++j) {
            const int t = min(s + j, 15);                       // (queries behind the block are left out below)
            const int dt = RULE == CHANNEL_WKV ? t - 1 : t;     // the last decay between s and t
            float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < DC; d += 4) {
                const float4 q = *reinterpret_cast<const float4*>(&L.q[w][t][c0 + d]);
                if (j > (RULE == CHANNEL_WKV ? 1 : 0)) {
                    const float4 y = *reinterpret_cast<const float4*>(&L.ka[w][1][dt][c0 + d]);
                    kd[d] *= y.x; kd[d + 1] *= y.y; kd[d + 2] *= y.z; kd[d + 3] *= y.w;
                }
                x[0] += q.x * kd[d]; x[1] += q.y * kd[d + 1]; x[2] += q.z * kd[d + 2]; x[3] += q.w * kd[d + 3];
            }
            p[j] = (x[0] + x[1]) + (x[2] + x[3]);
            if (j & 1) __builtin_amdgcn_sched_barrier(0);
        }
        // the sum of the four quarters: a lane ends up with four of the sixteen queries
        float p8[8], p4[4];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float keep = q4 & 2 ? p[8 + j] : p[j], give = q4 & 2 ? p[j] : p[8 + j];
            p8[j] = keep + __shfl_xor(give, 32, kWave);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float keep = q4 & 1 ? p8[4 + j] : p8[j], give = q4 & 1 ? p8[j] : p8[4 + j];
            p4[j] = keep + __shfl_xor(give, 16, kWave);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = s + 4 * q4 + j;                       // (q4 & 2: steps 8 .., q4 & 1: four more)
            if (t < 16) L.diag[w][t][s] = p4[j];
        }
    }
    lanes_meet();                                               // q's rows are about to change
    // ---- q with the decays from its block's start, k with those to its block's end
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int d = lane + 64 * i;
        float f = 1.f;
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            if (RULE != CHANNEL_WKV) f *= g[i][x];
            L.q[w][x][d] *= f;
            if (RULE == CHANNEL_WKV) f *= g[i][x];
        }
        L.blk[w][d] = f;
        f = 1.f;
#pragma unroll
        for (int x = 15; x >= 0; --x) {
            k[i][x] *= f;
            f *= g[i][x];
        }
    }
    __syncthreads();                                            // k's and the decays' rows have been read
    auto put_k = [&]() {
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                bf16x8 p[3];
                split8(k[i] + 8 * y, p);
#pragma unroll
                for (int z = 0; z < 3; ++z) *reinterpret_cast<bf16x8*>(L.kt[z] + at64(lane + 64 * i, 2 * w + y)) = p[z];
            }
    };
    put_k();
    __syncthreads();
    // ---- scores of this wave's queries t = 16 w + l16 and the blocks ahead; a lane has keys 16 kb + 4 q4 + r of each block
    f32x4 x[4];
    {
        float qf[KS][8];                                        // channels 32 s + 4 q4 .. and 16 behind them
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            *reinterpret_cast<float4*>(qf[s]) = *reinterpret_cast<const float4*>(&L.q[w][l16][32 * s + 4 * q4]);
            *reinterpret_cast<float4*>(qf[s] + 4) = *reinterpret_cast<const float4*>(&L.q[w][l16][32 * s + 16 + 4 * q4]);
        }
        const float4 dg = *reinterpret_cast<const float4*>(&L.diag[w][l16][4 * q4]);
        const float dr[4] = {dg.x, dg.y, dg.z, dg.w};
#pragma unroll
        for (int kb = 3; kb >= 0; --kb) {
            x[kb] = {0.f, 0.f, 0.f, 0.f};
            if (kb > w) continue;
            if (kb == w) {
#pragma unroll
                for (int r = 0; r < 4; ++r) x[kb][r] = 4 * q4 + r <= l16 ? dr[r] : 0.f;
                continue;
            }
            Product pr;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                bf16x8 qs[3], ks[3];
                split8(qf[s], qs);
                const int row = 32 * s + 4 * q4 + (l16 >> 2), chunk = 2 * kb + ((l16 & 3) >> 1);
#pragma unroll
                for (int z = 0; z < 3; ++z)
                    ks[z] = join(read_tr(L.kt[z] + at64(row, chunk) + (l16 & 1) * 8), read_tr(L.kt[z] + at64(row + 16, chunk) + (l16 & 1) * 8));
                pr.add(ks, qs);
            }
            x[kb] = pr.sum();
            // on to the block ahead
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const float4 f = *reinterpret_cast<const float4*>(&L.blk[kb][32 * s + 4 * q4]), f2 = *reinterpret_cast<const float4*>(&L.blk[kb][32 * s + 16 + 4 * q4]);
                qf[s][0] *= f.x; qf[s][1] *= f.y; qf[s][2] *= f.z; qf[s][3] *= f.w;
                qf[s][4] *= f2.x; qf[s][5] *= f2.y; qf[s][6] *= f2.z; qf[s][7] *= f2.w;
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float4* to = reinterpret_cast<float4*>(ws + It::Q + ((w * KS + s) * 64 + lane) * 8);
            to[0] = make_float4(qf[s][0], qf[s][1], qf[s][2], qf[s][3]);
            to[1] = make_float4(qf[s][4], qf[s][5], qf[s][6], qf[s][7]);
        }
    }
    if constexpr (NP == 1) {
        __syncthreads();                                        // q's rows have been read
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int c = tid + 256 * i;
            *reinterpret_cast<uint4*>(L.v + at_v<EP>(c / (EP / 8), c % (EP / 8))) = vr[i];
            const uint32_t y[4] = {vr[i].x, vr[i].y, vr[i].z, vr[i].w};
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                see(__uint_as_float(y[z] << 16));
                see(__uint_as_float(y[z] & 0xffff0000u));
            }
        }
        __syncthreads();
    }
    auto v_part = [&](int z) { return NP == 1 ? L.v : L.vp[z]; };
    // ---- A V
    {
        bf16x8 p[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float y[8] = {x[2 * s][0], x[2 * s][1], x[2 * s][2], x[2 * s][3],
                                x[2 * s + 1][0], x[2 * s + 1][1], x[2 * s + 1][2], x[2 * s + 1][3]};
            split8(y, p[s]);
        }
        for (int eb = 0; eb < EP / 16; ++eb) {
            f32x4 o = {0.f, 0.f, 0.f, 0.f}, lo = o;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (2 * s > w) continue;
                const int row = 32 * s + 4 * q4 + (l16 >> 2), chunk = 2 * eb + ((l16 & 3) >> 1);
                bf16x8 vf[NP];
#pragma unroll
                for (int z = 0; z < NP; ++z)
                    vf[z] = join(read_tr(v_part(z) + at_v<EP>(row, chunk) + (l16 & 1) * 8), read_tr(v_part(z) + at_v<EP>(row + 16, chunk) + (l16 & 1) * 8));
                if constexpr (NP == 1) {
                    lo = mfma(vf[0], p[s][2], lo);
                    o = mfma(vf[0], p[s][0], o);
                    lo = mfma(vf[0], p[s][1], lo);
                } else {
                    lo = mfma(vf[2], p[s][0], lo);
                    o = mfma(vf[0], p[s][0], o);
                    lo = mfma(vf[0], p[s][2], lo);
                    lo = mfma(vf[1], p[s][1], lo);
                    lo = mfma(vf[1], p[s][0], lo);
                    lo = mfma(vf[0], p[s][1], lo);
                }
            }
            *reinterpret_cast<f32x4*>(ws + It::O + ((w * (EP / 16) + eb) * 64 + lane) * 4) = o + lo;
        }
    }
    // ---- (K o P)^T V: k with the decays to the chunk's end
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        float f = 1.f;
        for (int m = w + 1; m < 4; ++m) f *= L.blk[m][lane + 64 * i];
#pragma unroll
        for (int y = 0; y < 16; ++y) k[i][y] *= f;
        if (w == 0) ws[It::CE + lane + 64 * i] = L.blk[0][lane + 64 * i] * f;
    }
    const bool any_bad = __syncthreads_or(top > __float_as_uint(LARGE));     // (k's images have been read)
    if (tid == 0) reinterpret_cast<int*>(ws)[It::FLAG] = any_bad;
    put_k();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int db = w + 4 * i;                               // this wave's channels 16 db ..
        bf16x8 kf[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int z = 0; z < 3; ++z) kf[s][z] = *reinterpret_cast<const bf16x8*>(L.kt[z] + at64(16 * db + l16, 4 * s + q4));
        for (int eb = 0; eb < EP / 16; ++eb) {
            f32x4 o = {0.f, 0.f, 0.f, 0.f}, lo = o;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int row = 32 * s + 8 * q4 + (l16 >> 2), chunk = 2 * eb + ((l16 & 3) >> 1);
                bf16x8 vf[NP];
#pragma unroll
                for (int z = 0; z < NP; ++z)
                    vf[z] = join(read_tr(v_part(z) + at_v<EP>(row, chunk) + (l16 & 1) * 8), read_tr(v_part(z) + at_v<EP>(row + 4, chunk) + (l16 & 1) * 8));
                if constexpr (NP == 1) {
                    lo = mfma(kf[s][2], vf[0], lo);
                    o = mfma(kf[s][0], vf[0], o);
                    lo = mfma(kf[s][1], vf[0], lo);
                } else {
                    lo = mfma(kf[s][2], vf[0], lo);
                    o = mfma(kf[s][0], vf[0], o);
                    lo = mfma(kf[s][0], vf[2], lo);
                    lo = mfma(kf[s][1], vf[1], lo);
                    lo = mfma(kf[s][1], vf[0], lo);
                    lo = mfma(kf[s][0], vf[1], lo);
                }
            }
            *reinterpret_cast<f32x4*>(ws + It::S + ((db * (EP / 16) + eb) * 64 + lane) * 4) = o + lo;
        }
    }
#endif
}

// One thread per run of four channels of a state column: over the chunks of its sequence, S_0 of each into the place of
// the chunk's own part, the state behind the portion into its slot.
template <int DP, int EP>
__global__ void __launch_bounds__(256) channel_state_kernel(const ChannelChunks a) {
    using It = Item<DP, EP>;
    constexpr int AHEAD = 8;
    const int b = blockIdx.x, h = blockIdx.y, i = blockIdx.z * 256 + threadIdx.x;      // [16 channels][16 columns][lane]
    const int slot = a.slots[b], first = a.cu_q[b], n = a.cu_q[b + 1] - first, H = a.H;
    if (slot < 0 || n <= 0 || i >= DP * EP / 4) return;
    const int ln = i & 63, eb = (i >> 6) % (EP / 16), db = (i >> 6) / (EP / 16);
    const int d = 16 * db + 4 * (ln >> 4), e = 16 * eb + (ln & 15);
    float* sp = a.state + (((long)slot * H + h) * a.D + d) * a.E + e;
    const bool col = e < a.E, has_past = a.positions[first] > 0;
    float4 S = make_float4(0.f, 0.f, 0.f, 0.f);
    if (has_past && col) {
        if (d < a.D) S.x = sp[0];
        if (d + 1 < a.D) S.y = sp[a.E];
        if (d + 2 < a.D) S.z = sp[2 * a.E];
        if (d + 3 < a.D) S.w = sp[3 * a.E];
    }
    bool bad = false;
    const int chunks = (n + C - 1) / C;
    const long step = (long)H * It::SIZE;
    float* ws = a.ws + ((long)(first / C + b) * H + h) * It::SIZE;
    for (int c0 = 0; c0 < chunks; c0 += AHEAD) {
        float4 own[AHEAD], ce[AHEAD];
#pragma unroll
        for (int c = 0; c < AHEAD; ++c)
            if (c0 + c < chunks) {
                own[c] = *reinterpret_cast<const float4*>(ws + (c0 + c) * step + It::S + i * 4);
                ce[c] = *reinterpret_cast<const float4*>(ws + (c0 + c) * step + It::CE + d);
            }
#pragma unroll
        for (int c = 0; c < AHEAD; ++c)
            if (c0 + c < chunks) {
                *reinterpret_cast<float4*>(ws + (c0 + c) * step + It::S + i * 4) = S;
                bad |= !(fabsf(S.x) + fabsf(S.y) + fabsf(S.z) + fabsf(S.w) <= LARGE_STATE);
                S.x = fmaf(ce[c].x, S.x, own[c].x);
                S.y = fmaf(ce[c].y, S.y, own[c].y);
                S.z = fmaf(ce[c].z, S.z, own[c].z);
                S.w = fmaf(ce[c].w, S.w, own[c].w);
            }
    }
    if (col) {
        if (d < a.D) sp[0] = S.x;
        if (d + 1 < a.D) sp[a.E] = S.y;
        if (d + 2 < a.D) sp[2 * a.E] = S.z;
        if (d + 3 < a.D) sp[3 * a.E] = S.w;
        bad |= !(fabsf(S.x) + fabsf(S.y) + fabsf(S.z) + fabsf(S.w) <= LARGE_STATE);
    }
    if (bad) reinterpret_cast<int*>(ws)[It::FLAG] = 1;
}

template <typename TI, bool NORM>
__device__ __forceinline__ void put_row(const ChannelChunks& a, long t, int h, int e, float o, float r) {
    if constexpr (NORM) {
        const float z = ld((const TI*)a.gate + t * a.gate_row + (long)h * a.E + e);
        st((TI*)a.y + (t * a.H + h) * a.E + e, o * (r * a.norm_w[(a.w_heads ? h * a.E : 0) + e] * (a.sig ? sigmoidf_(z) : siluf_(z))));
    } else {
        a.o[(t * a.H + h) * (long)a.E + e] = o;
    }
}

// A portion's tokens one after the other, from the first chunk's S_0: a thread has a column and some of the channels.
template <typename TI, int RULE, int DP, int EP, bool NORM>
__device__ __forceinline__ void walk_tokens(const ChannelChunks a, int b, int h, float* sm) {
    using It = Item<DP, EP>;
    constexpr int NS = 256 / EP, CH = DP / NS;
    const int first = a.cu_q[b], n = a.cu_q[b + 1] - first, H = a.H, D = a.D, E = a.E;
    const int c = threadIdx.x % EP, r = threadIdx.x / EP, d0 = r * CH;
    const float* s0 = a.ws + ((long)(first / C + b) * H + h) * It::SIZE + It::S;
    float* sp = a.state + ((long)a.slots[b] * H + h) * D * E;
    float *q = sm, *k = q + DP, *g = k + DP, *part = g + DP, *os = part + NS * EP;
    float S[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int d = d0 + i;
        S[i] = s0[(((d >> 4) * (EP / 16) + (c >> 4)) * 64 + (d >> 2 & 3) * 16 + (c & 15)) * 4 + (d & 3)];
    }
    for (long t = first; t < first + n; ++t) {
        __syncthreads();
        for (int d = threadIdx.x; d < DP; d += 256) {
            const bool in = d < D;
            q[d] = in ? ld((const TI*)a.q + t * a.q_row + (long)h * D + d) * a.qscale : 0.f;
            k[d] = in ? ld((const TI*)a.k + t * a.k_row + (long)h * D + d) : 0.f;
            g[d] = in ? decay_of<RULE>(ld((const TI*)a.a + t * a.a_row + (long)h * D + d) + a.a_bias[h * D + d], a.tau_inv) : 1.f;
        }
        const float v = c < E ? ld((const TI*)a.v + t * a.v_row + (long)h * E + c) : 0.f;
        __syncthreads();
        float po = 0.f, dot = 0.f;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int d = d0 + i;
            if (d >= D) continue;
            if constexpr (RULE == CHANNEL_WKV) {
                po += S[i] * q[d];
                S[i] = g[d] * S[i] + k[d] * v;
            } else {
                S[i] = g[d] * S[i] + k[d] * v;
                po += S[i] * q[d];
            }
        }
        part[r * EP + c] = po;
        __syncthreads();
        if (r == 0) {
            po = 0.f;
            for (int i = 0; i < NS; ++i) po += part[i * EP + c];
            if constexpr (RULE == CHANNEL_WKV) {
                for (int d = 0; d < D; ++d) dot += k[d] * q[d] * a.bonus[h * D + d];
                po += dot * v;
            }
            os[c] = c < E ? po : 0.f;
        }
        __syncthreads();
        if (r == 0 && c < E) {
            float s = 0.f;
            if constexpr (NORM)
                for (int e = 0; e < E; ++e) s += os[e] * os[e];
            put_row<TI, NORM>(a, t, h, c, po, rsqrtf(s / (float)E + a.eps));
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
        if (d0 + i < D && c < E) sp[(long)(d0 + i) * E + c] = S[i];
}

// wave = 16 tokens of a chunk; a lane has columns 16 eb + 4 q4 .. + 3 of token l16
template <typename TI, int RULE, int DP, int EP, bool NORM>
__global__ void __launch_bounds__(256, 2) channel_out_kernel(const ChannelChunks a) {
#ifdef __HIP_DEVICE_COMPILE__
    using It = Item<DP, EP>;
    constexpr int KS = DP / 32, NB = EP / 16;
    __shared__ __attribute__((aligned(16))) float sm[3 * DP + 256 + EP];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4, h = blockIdx.y, H = a.H, E = a.E;
    auto clear = [&](long from, long to) {                      // rows of no sequence
        for (long i = tid; i < (to - from) * E; i += 256) {
            const long at = ((from + i / E) * H + h) * E + i % E;
            if constexpr (NORM) st((TI*)a.y + at, 0.f);
            else a.o[at] = 0.f;
        }
    };
    if (blockIdx.x == 0) {
        clear(0, a.cu_q[0]);
        clear(a.cu_q[a.B], a.T);
    }
    const int b = sequence_of(a.cu_q, a.B, blockIdx.x);
    if (b < 0) return;
    const int first = a.cu_q[b], n = a.cu_q[b + 1] - first, ch = blockIdx.x - (first / C + b);
    const int nt = min(C, n - ch * C);
    if (nt <= 0) return;
    const long t0 = (long)first + ch * C;
    if (a.slots[b] < 0) return clear(t0, t0 + nt);
    const float* ws = a.ws + ((long)blockIdx.x * H + h) * It::SIZE;
    bool bad = false;                                           // (the same for all of the portion's workgroups)
    for (int c = lane; c < (n + C - 1) / C; c += 64) bad |= reinterpret_cast<const int*>(ws)[(long)(c - ch) * H * It::SIZE + It::FLAG] != 0;
    if (__any(bad)) {
        if (ch == 0) walk_tokens<TI, RULE, DP, EP, NORM>(arguments_anew<ChannelChunks>(), b, h, sm);
        return;
    }
    const int t = 16 * w + l16;
    if (16 * w < nt) {
        bf16x8 qf[KS][3];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float x[8];
            load_run<float, 8>(ws + It::Q + ((w * KS + s) * 64 + lane) * 8, x);
            split8(x, qf[s]);
        }
        f32x4 o[NB];
        float sq = 0.f;
#pragma unroll
        for (int eb = 0; eb < NB; ++eb) {
            Product p;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                float x[8];
                load_run<float, 4>(ws + It::S + ((2 * s * NB + eb) * 64 + lane) * 4, x);
                load_run<float, 4>(ws + It::S + (((2 * s + 1) * NB + eb) * 64 + lane) * 4, x + 4);
                bf16x8 sf[3];
                split8(x, sf);
                p.add(sf, qf[s]);
            }
            o[eb] = *reinterpret_cast<const f32x4*>(ws + It::O + ((w * NB + eb) * 64 + lane) * 4) + p.sum();
            sq += (o[eb][0] * o[eb][0] + o[eb][1] * o[eb][1]) + (o[eb][2] * o[eb][2] + o[eb][3] * o[eb][3]);
        }
        if constexpr (NORM) {
            sq += __shfl_xor(sq, 16, kWave);
            sq += __shfl_xor(sq, 32, kWave);
        }
        const float r = rsqrtf(sq / (float)E + a.eps);
        if (t < nt)
#pragma unroll
            for (int eb = 0; eb < NB; ++eb) {
                const int e = 16 * eb + 4 * q4;
                if (e >= E) continue;
                if constexpr (NORM) {
                    float z[4], nw[4], y[4];
                    Vec4<TI>::load((const TI*)a.gate + (t0 + t) * a.gate_row + (long)h * E + e, z);
                    Vec4<float>::load(a.norm_w + (a.w_heads ? h * E : 0) + e, nw);
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = o[eb][i] * (r * nw[i] * (a.sig ? sigmoidf_(z[i]) : siluf_(z[i])));
                    TI* to = (TI*)a.y + ((t0 + t) * H + h) * E + e;
                    if constexpr (sizeof(TI) == 2) *reinterpret_cast<uint2*>(to) = make_uint2(rounded(y[0], y[1]), rounded(y[2], y[3]));
                    else *reinterpret_cast<float4*>(to) = make_float4(y[0], y[1], y[2], y[3]);
                } else {
                    *reinterpret_cast<f32x4*>(a.o + ((t0 + t) * H + h) * (long)E + e) = o[eb];
                }
            }
    }
#endif
}

template <typename TI, int RULE, int DP, int EP>
int launch(const ChannelChunks& a, hipStream_t s) {
    constexpr int lds = sizeof(ChunkLds<TI, RULE, DP, EP>);
    static_assert(lds <= 160 * 1024);
    static const hipError_t once = hipFuncSetAttribute((const void*)channel_chunk_kernel<TI, RULE, DP, EP>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (once != hipSuccess) return 2;
    const unsigned items = (unsigned)item_count(a.T, a.B);
    hipLaunchKernelGGL((channel_chunk_kernel<TI, RULE, DP, EP>), dim3(items, a.H), dim3(256), lds, s, a);
    hipLaunchKernelGGL((channel_state_kernel<DP, EP>), dim3(a.B, a.H, (DP * EP / 4 + 255) / 256), dim3(256), 0, s, a);
    if (a.y) hipLaunchKernelGGL((channel_out_kernel<TI, RULE, DP, EP, true>), dim3(items, a.H), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((channel_out_kernel<TI, RULE, DP, EP, false>), dim3(items, a.H), dim3(256), 0, s, a);
    return HYB_LAUNCH_OK();
}

}  // namespace

namespace hyb {

// Three kernels, of which each portion costs at least a chunk, against a token after the other, by what both take on the
// card, us: the tokens a walk as long as the longest portion and their share of the card (by rows of the outputs and by states),
// the chunks a share by their number.  Layer of 8 heads of 64 x 128, bfloat16, with the norm, us, chunks / tokens: 8 portions of 32
// 30.5 / 26.9, of 64 31.6 / 30.6, of 128 32.8 / 51.8; 64 of 17 57 / 33, of 64 74 / 78, of 128 97 / 141; 63 single tokens
// and one of 128 54 / 84; 255 and one of 128 132 / 101, of 512 135 / 323.  Without it, 16 heads of 64 x 64: 8 of 96 36 / 41, 32
// of 64 59 / 44, of 128 74 / 75, 128 of 64 194 / 144; 8 heads of 32 x 32, 256 of 64, up to 3.9 times as long.  Over 1342
// steps of either (1 to 256 portions of 16 to 1024 tokens, 4 to 32 heads of 32 to 64 x 32 to 128, both types) the rule's way takes
// 1.009 of the shorter one in the mean, and 1.16 of the tokens' at the most; below `each` tokens a portion and half a
// token for every portion it was not measured, and is the tokens'.  longest 0: not known.
static bool channel_chunks_pay(const ChannelChunks& a, int longest, int dt) {
    const long each = a.y ? 64 : 96;
    if (a.T < each * a.B && 2L * longest < 2 * each + a.B) return false;
    const bool f32 = dt == 2, wide = a.E > 64;
    const float n = longest > 0 ? (float)longest : (float)a.T / a.B, T = (float)a.T, B = (float)a.B;
    const float columns = a.H * ((a.E + 15) / 16) / 4.f;       // in 64s
    const float tokens = a.D <= 32 ? 12.f + .22f * n + columns * (.00027f * T + .0136f * B)
                             : f32 ? 9.f + .25f * n + columns * (.0012f * T + .0415f * B)
                                   : 11.f + .28f * n + columns * (.0005f * T + .009f * B);
    const float share = f32 ? (wide ? .084f : .059f) : (wide ? .053f : .0355f);
    const float chunks = (wide ? 29.f : 25.5f) + (a.y ? 0.f : 2.f) + share * a.H * (T / 64.f + B);
    return chunks * 1.03f < tokens;
}

long channel_chunks_bytes(const ChannelChunks& a, int dt) {
    if (!a.cu_q || a.B <= 0 || a.D < 4 || a.D > 64 || a.E % 8 || a.E < 8 || a.E > 128) return 0;
    if (a.H <= 0 || a.H > 65535 || a.B > 65535 || a.T >= 1L << 30) return 0;
    const int run = dt == 0 ? 8 : 4;               // v comes in runs of eight, gates of four
    if ((size_t)a.v % 16 || a.v_row % run || ((size_t)a.o | (size_t)a.y) % 16) return 0;
    if (a.y && ((size_t)a.gate % 16 || a.gate_row % 4 || (size_t)a.norm_w % 16)) return 0;
    const long size = a.E <= 64 ? Item<64, 64>::SIZE : Item<64, 128>::SIZE;
    return item_count(a.T, a.B) * a.H * size * 4;
}

int channel_chunks(const ChannelChunks& a, int rule, int dt, hipStream_t s) {
#define RUN(RULE)                                                                         \
    do {                                                                                  \
        if (a.E <= 64) HYB_DISPATCH(dt, return (launch<T, RULE, 64, 64>(a, s)));          \
        else HYB_DISPATCH(dt, return (launch<T, RULE, 64, 128>(a, s)));                   \
    } while (0)
    if (rule == CHANNEL_GLA) RUN(CHANNEL_GLA);
    else RUN(CHANNEL_WKV);
#undef RUN
    return 1;
}

}  // namespace hyb

extern "C" {

// Bytes of workspace hyb_channel_chunks wants (0: it does not take the call).  `aligned`: v, gate and norm_w on 16 bytes,
// v in rows of whole runs of eight, gates of four; longest: the longest portion's tokens, 0 if that is not known, -1 for what it
// would want of any step of that size
long hyb_channel_chunks_bytes(long T_, int B, int longest, int H, int D, int E, int aligned, int norm, int dt) {
    ChannelChunks a{};
    a.cu_q = (const int*)256;
    a.T = T_; a.B = B; a.H = H; a.D = D; a.E = E;
    if (!aligned) return 0;
    if (norm) a.y = (void*)256;
    return longest < 0 || channel_chunks_pay(a, longest, dt) ? channel_chunks_bytes(a, dt) : 0;
}

// rule 0: GLA (tau; bonus null), 1: WKV (bonus [H*D]).  y null: o [T, H, E] fp32; else y [T, H*E] of the activation type,
// every head's outputs divided by their root mean square, times norm_w ([E] or, w_heads, [H*E]), times silu (sig:
// sigmoid) of gate.  ws: hyb_channel_chunks_bytes.
int hyb_channel_chunks(int rule, const void* q, const void* k, const void* v, long q_row, long k_row, long v_row,
                       const void* a_raw, long a_row, const void* a_bias, const void* bonus, float tau, float qscale,
                       void* state, const void* cu_q, const void* positions, const void* slots, void* ws, void* o, void* y,
                       const void* gate, long gate_row, const void* norm_w, int w_heads, float eps, int sig, long T_, int B,
                       int H, int D, int E, int dt, hipStream_t s) {
    const ChannelChunks a{q, k, v, a_raw, q_row, k_row, v_row, a_row, (const float*)a_bias, (const float*)bonus, 1.f / tau,
                          qscale, (float*)state, (const int*)cu_q, (const int*)positions, (const int*)slots, (float*)ws,
                          (float*)o, y, gate, gate_row, (const float*)norm_w, eps, sig, w_heads, T_, B, H, D, E};
    if (!ws || (!o && !y) || (rule != CHANNEL_GLA && rule != CHANNEL_WKV) || (rule == CHANNEL_WKV && !bonus)) return 1;
    if ((dt != 0 && dt != 2) || !channel_chunks_bytes(a, dt)) return 1;
    return channel_chunks(a, rule, dt, s);
}

}  // extern "C"
