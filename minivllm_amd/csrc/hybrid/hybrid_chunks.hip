// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form
// The matrix LSTM's recurrence over prompt portions in chunks of 64 tokens on the matrix cores
// (bfloat16 projections; hybrid_recurrent.hip has the recurrence itself and takes everything else).
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
// Every factor is a product of the same a and b the recurrence multiplies by, all <= 1: no quotients, no
// logarithms of products.  W comes from the products inside blocks of 16 tokens: in a pair of different blocks it
// is (a .. to t inside its block) (whole blocks between) (a .. from i to its block's end) b_i, on the diagonal the
// running product.
//
// q, k, v ARE bfloat16; what is fp32 (the weighted scores, the state, the weighted values) is cut into
// three parts of eight bits, all of its 24, and multiplied part by part on
// v_mfma_f32_16x16x32_bf16 with fp32 sums.
//
// Workgroup = 8 waves on 32 state columns of one (sequence, head).  Wave w owns the chunk's
// tokens 16 (w % 4) .. + 15 as queries, a quarter of the key channels of the state and 16 of the
// columns; its part of the state stays in its registers, whose parts go through LDS once per chunk
// as operands for all waves.  The next chunk's q, k, v and gates are in registers while this one
// is worked on; three barriers per chunk.
//
// An infinity or a NaN in a row of a chunk meets the zero weights of the tokens ahead of it, and its parts are NaN.
// It stays in the sums once it is there, so a portion whose outputs and state come out finite met none; any other is
// walked again from its first token by the recurrence itself (same workgroup, its own columns).
//
// Bound by the vector instructions around the products (splitting, weights, addresses: 1300 per wave
// and chunk at two waves per SIMD), 4.4 us a chunk.  8 portions of 512..1024 tokens, 8 heads of
// 128: 70 us of 83 with the norm behind it, against 602 of 622 token by token.  With four waves of twice the
// columns 112 us; two workgroups per CU (128 registers) spill: 177 us.
#include "hybrid_chunks.h"

using namespace hyb;

namespace {

constexpr int C = 64;                  // tokens per chunk
constexpr int EB = 32;                 // state columns per workgroup
constexpr float NEG_INF = -__builtin_inff();

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

template <int DP>
struct Lds {
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
__device__ __forceinline__ int wv_at(int row, int byte) { return row * (EB * 2) + (byte ^ (row << 2 & 32)); }

__device__ __forceinline__ float logsigmoid_(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// The portion's tokens one after the other: thread = a column and a sixteenth of the channels, sums through LDS
// (`red`: 8 KB).
template <int DP>
__device__ __forceinline__ void walk_tokens(const MlstmChunks a, float* red) {
    constexpr int CH = DP / 16;
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
        const float gi = a.cap * tanhf((ld(a.gi + t * a.g_row + h) + a.bi[h]) / a.cap);
        const float gf = logsigmoid_(a.cap * tanhf((ld(a.gf + t * a.g_row + h) + a.bf[h]) / a.cap));
        const float m2 = fmaxf(gf + m, gi), fs = expf(gf + m - m2), is = expf(gi - m2);
        m = m2;
        const float kv = e < E ? is * ld((const bf16_t*)a.v + t * a.v_row + (long)h * E + e) : 0.f;
        float po = 0.f, pn = 0.f;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (d0 + i >= D) continue;
            const float k = ld((const bf16_t*)a.k + t * a.k_row + (long)h * D + d0 + i);
            const float q = ld((const bf16_t*)a.q + t * a.q_row + (long)h * D + d0 + i) * a.qscale;
            S[i] = fs * S[i] + k * kv;
            po += S[i] * q;
            N[i] = fs * N[i] + is * k;
            pn += N[i] * q;
        }
        float* at = red + (x & 1) * 1024;              // two of them: one barrier per token
        at[r * 32 + c] = po;
        at[512 + r * 32 + c] = pn;
        __syncthreads();
        if (r == 0 && e < E) {
            po = pn = 0.f;
            for (int i = 0; i < 16; ++i) {
                po += at[i * 32 + c];
                pn += at[512 + i * 32 + c];
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

template <int DP>
__global__ void __launch_bounds__(512, DP > 64 ? 2 : 4)      // (two workgroups on a CU where the LDS has room for them)
mlstm_chunks_kernel(MlstmChunks a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KS = DP / 32, DT = DP / 64;      // steps over the key channels; a wave's 16-wide blocks of them
    constexpr int PIECES = C * DP / 8 / 512;       // 16-byte pieces of a q (or k) image per thread
    extern __shared__ __attribute__((aligned(256))) char smem[];
    Lds<DP>& L = *reinterpret_cast<Lds<DP>*>(smem);
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

    // ---- the state: S[j] holds channels 16 (tb + 4 j) + 4 q4 + r of column e; a channel's normaliser is
    // the sum of N over the columns of its row (the waves of the first 16 columns keep it)
    const int e = e0 + 16 * et + l16;
    f32x4 S[DT], N[DT];
    float* sp = a.state + ((long)slot * H + h) * D * E;
    float* np = a.nstate + (((long)slot * H + h) * ZG + e0 / 16) * D;
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * (tb + 4 * j) + 4 * q4 + r;
            S[j][r] = has_past && d < D && e < E ? sp[(long)d * E + e] : 0.f;
            N[j][r] = has_past && d < D && l16 == 0 ? np[d] : 0.f;
        }
    float m_run = has_past ? a.mstate[((long)slot * H + h) * ZG + e0 / 16] : 0.f;

    // ---- the next chunk on its way: rows behind the portion and columns behind a head are out of the
    // buffers' range and read as zeros
    uint4 qr[PIECES], kr[PIECES];
    uint2 vr;
    float gi = 0.f, gf = 0.f;
    int q_off[PIECES], k_off[PIECES];
    constexpr int NOWHERE = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int c = i * 512 + tid, row = c / (DP / 8), d = c % (DP / 8) * 8;
        q_off[i] = d < D ? (row * (int)a.q_row + d) * 2 : NOWHERE;
        k_off[i] = d < D ? (row * (int)a.k_row + d) * 2 : NOWHERE;
    }
    const int v_off = e0 + (tid & 7) * 4 < E ? ((tid >> 3) * (int)a.v_row + (tid & 7) * 4) * 2 : NOWHERE;
    auto rows_of = [&](const uint16_t* p, long row, long t0, int nt, int col, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p + t0 * row + col), 0,
                                                 ((nt - 1) * (int)row + width) * 2, 0x00020000);
    };
    constexpr int GATES = 4;                       // the wave that works the gates out (few key blocks, no N)
    auto fetch = [&](int ch) {
        const int nt = min(C, n - ch * C);
        const long t0 = first + (long)ch * C;
        const __amdgpu_buffer_rsrc_t qb = rows_of(a.q, a.q_row, t0, nt, h * D, D), kb = rows_of(a.k, a.k_row, t0, nt, h * D, D),
                                     vb = rows_of(a.v, a.v_row, t0, nt, h * E + e0, E - e0);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            qr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qb, q_off[i], 0, 0));
            kr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kb, k_off[i], 0, 0));
        }
        vr = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(vb, v_off, 0, 0));
        if (wave == GATES) {
            const long t = t0 + min(lane, nt - 1);
            gi = ld(a.gi + t * a.g_row + h);
            gf = ld(a.gf + t * a.g_row + h);
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
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int c = i * 512 + tid, row = c / (DP / 8), ch = (c % (DP / 8)) ^ rows16<DP>(row);
            *reinterpret_cast<uint4*>(L.q + row * DP * 2 + ch * 16) = qr[i];
            *reinterpret_cast<uint4*>(L.k + row * DP * 2 + ch * 16) = kr[i];
        }
        *reinterpret_cast<uint2*>(L.v + v_at(tid >> 3, (tid & 7) * 8)) = vr;
    };
    // the state's parts: a row per column of the state
    auto publish = [&]() {
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            const int d = 16 * (tb + 4 * j) + 4 * q4, row = 16 * et + l16;
            put_parts(S[j], [&](int k) { return L.s[k] + row * DP * 2 + (((d >> 3) ^ rows16<DP>(row)) << 4) + (d & 4) * 2; });
            if (et == 0 && l16 == 0) put_parts(N[j], [&](int k) { return L.n[k] + d * 2; });
        }
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
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            S[j] *= ce;
            N[j] *= ce;
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int row = 32 * s + 8 * q4 + (l16 >> 2);
            bf16x8 wf[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const char* at = L.wv[k] + wv_at(row, et * 32 + (l16 & 3) * 8);
                wf[k] = join(read_tr(at), read_tr(at + 4 * EB * 2));
            }
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const int chunk = 2 * (tb + 4 * j) + ((l16 & 3) >> 1);
                const bf16x8 kf = join(read_tr(L.k + row * DP * 2 + ((chunk ^ rows16<DP>(row)) << 4) + (l16 & 1) * 8),
                                       read_tr(L.k + (row + 4) * DP * 2 + ((chunk ^ rows16<DP>(row + 4)) << 4) + (l16 & 1) * 8));
#pragma unroll
                for (int k = 2; k >= 0; --k) S[j] = mfma(kf, wf[k], S[j]);
                if (et == 0) N[j] = mfma(kf, *reinterpret_cast<const bf16x8*>(&g.wp[min(l16, 2)][32 * s + 8 * q4]), N[j]);
            }
        }
        if (et == 0) {
            // the sum of n's three columns goes on in the first
#pragma unroll
            for (int j = 0; j < DT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float y = from_right<1>(N[j][r], 0.f), z = from_right<2>(N[j][r], 0.f);
                    N[j][r] = l16 == 0 ? N[j][r] + (y + z) : 0.f;
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
#pragma unroll
    for (int j = 0; j < DT; ++j) seen += (S[j][0] + S[j][1]) + (S[j][2] + S[j][3]);
    if (seen * 0.f != 0.f) L.lost = 1;
    __syncthreads();
    if (L.lost) {
        __threadfence();                                    // (the outputs are written again, by other waves)
        __syncthreads();
        walk_tokens<DP>(arguments_anew<MlstmChunks>(), reinterpret_cast<float*>(smem));
        return;
    }
    // ---- the state after the portion
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
    if (wave == GATES && lane < 2 && e0 / 16 + lane < ZG) a.mstate[((long)slot * H + h) * ZG + e0 / 16 + lane] = m_run;
#endif
}

template <int DP>
int launch(const MlstmChunks& a, int B, hipStream_t s) {
    constexpr int lds = sizeof(Lds<DP>);
    static_assert(lds <= 80 * 1024);
    if (lds > 64 * 1024) {
        static const hipError_t once = hipFuncSetAttribute((const void*)mlstm_chunks_kernel<DP>,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (once != hipSuccess) return 2;
    }
    hipLaunchKernelGGL(mlstm_chunks_kernel<DP>, dim3(B, a.H, (a.E + EB - 1) / EB), dim3(512), lds, s, a);
    return HYB_LAUNCH_OK();
}

}  // namespace

namespace hyb {

// A portion of a few tokens costs a whole chunk (64 sequences of 4 tokens, 8 heads of 128: 61 us against
// the literal kernel's 50; of 16 tokens: 62 against 83; of 128: 126 against 453; one of 300: below the
// launch, against 161), so the rows must make up for the sequences: ten per sequence, or a thousand beyond
// the first of each, as with a prompt next to many single tokens, which the literal kernel walks in 0.5 us a token.
bool mlstm_chunks_ok(const MlstmChunks& a, int B) {
    if (a.T < 10L * B && a.T - B < 1024) return false;
    if (!a.cu_q || a.D < 8 || a.D > 128 || a.D % 8 || a.E % 8 || a.H > 65535) return false;
    if (((size_t)a.q | (size_t)a.k | (size_t)a.v | (size_t)a.o) % 16) return false;
    for (long row : {a.q_row, a.k_row, a.v_row})
        if (row % 8 || row < 0 || row >= 1 << 23) return false;      // (64 rows are addressed in 31 bits)
    return true;
}

int mlstm_chunks(const MlstmChunks& a, int B, hipStream_t s) {
    return a.D <= 64 ? launch<64>(a, B, s) : launch<128>(a, B, s);
}

}  // namespace hyb
