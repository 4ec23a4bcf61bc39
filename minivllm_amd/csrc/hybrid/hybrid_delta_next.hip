// Gated delta rule, single next tokens (row b is sequence b), all of a layer between its projections in one kernel:
// the short convolution and its tail, unit vectors, beta and decay, the recurrence's step, the gated norm of the heads.
//
// Workgroup = one (sequence, key head): the key head's q and k channels and the v channels of its TEAMS value heads,
// so that every channel's tail is read and written by one workgroup alone, and a team of 256 threads per value head
// for the state, as in delta_step_kernel (hybrid_delta.hip): E / 4 neighbouring threads cover a row of S, a thread
// keeps RPT rows of its four columns.  The sums are those of delta_prepare_rows_kernel, delta_step_kernel and
// gated_head_norm_runs_kernel, in their order.
//
// Bound by memory where there are many sequences (the state, read and written once); with few of them by the chain
// slot -> state and row -> convolution -> two sums over the rows -> norm, and by the launch.  64 sequences, 16 / 8 heads
// of 128 x 128 (134 MB of state): 28.6 us a call; the three kernels took 37 us on the card (7.6 + 25.9 + 3.9) and 47 a
// call, of which the host was half, for 6 sequences as well.
#include "hybrid_chunks.h"

using namespace hyb;

struct DeltaNext {
    const void* proj; long row; int b_off;         // [q (G*D) | k (G*D) | v (H*E) | ..], beta's pre-activation at b_off
    const void* a; long a_row; int DC;             // the decay's: DC entries per head (1 or D)
    const void* gate; long gate_row;               // [T, H*E]
    const float *conv_w, *a_log, *dt_bias, *norm_w;
    float *conv_state, *state;
    const int *positions, *slots;
    void* out;                                     // [T, H*E]
    float eps;
    int taps, H, G, D, E, sig, w_heads;
};

constexpr int NEXT_TAPS = 4;

// rows that `groups` row groups (and the idle threads behind them, one group more) walk, in whole runs of four
__host__ __device__ inline int next_rows(int rpt, int groups) { return (rpt * groups + 1 + 3) & ~3; }

template <typename T, int TEAMS, int RPT, bool CHANNEL>
__global__ void __launch_bounds__(256 * TEAMS, 4) delta_next_kernel(const DeltaNext p) {
    extern __shared__ float sm[];
    constexpr int NT = 256 * TEAMS;
    const int b = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, h0 = g * TEAMS;
    const int H = p.H, D = p.D, E = p.E, GD = p.G * D, C = 2 * GD + H * E, taps = p.taps, n = 2 * D + TEAMS * E;
    T* out = (T*)p.out + ((long)b * H + h0) * E;
    const int slot = p.slots[b];
    if (slot < 0) {                                // no sequence's row reads as zeros
        if (tid < TEAMS * E) st(out + tid, 0.f);
        return;
    }
    const bool has_past = p.positions[b] > 0;
    const T* row = (const T*)p.proj + (long)b * p.row;
    float* tail = p.conv_state + (long)slot * (taps - 1) * C;
    const int team = tid >> 8, t = tid & 255, lanes = E >> 2, groups = 256 / lanes, padded = (groups + 3) & ~3;
    const int grp = t / lanes, e = t % lanes * 4;
    const bool in_state = grp < groups;
    // q, k and decays in LDS behind D: zeros up to the rows that the row groups walk
    const int DP = next_rows(RPT, groups), step = groups * E;
    float* ys = sm;                                // as convolved: [q (DP) | k (DP) | v (TEAMS * E)]
    float* vs = ys + 2 * DP;
    float* dec = vs + TEAMS * E;                   // [TEAMS][DP] or [TEAMS], in whole runs of four
    float* bt_ = dec + (CHANNEL ? TEAMS * DP : 4); // [TEAMS]
    float* rn = bt_ + 4;                           // [TEAMS]: the norm's factors
    float* os = rn + 4;                            // [TEAMS][E]
    float* sums = os + TEAMS * E + team * 2 * padded * E;           // [padded][E] twice

    // ---- loads: the row's channels first, the state behind them (loads arrive in order)
    float x[NEXT_TAPS], w[NEXT_TAPS];
    auto channel = [&](int c) { return c < 2 * D ? (c < D ? g * D + c : GD + g * D + c - D) : 2 * GD + h0 * E + c - 2 * D; };
    auto fetch = [&](int c) {
        const int ch = channel(c);
#pragma unroll
        for (int j = 0; j < NEXT_TAPS; ++j) {
            x[j] = w[j] = 0.f;
            if (j < taps) {
                w[j] = p.conv_w[(long)ch * taps + j];
                if (j == taps - 1) x[j] = ld(row + ch);
                else if (has_past) x[j] = tail[(long)j * C + ch];
            }
        }
    };
    if (tid < n) fetch(tid);
    const float z = tid < TEAMS * E ? ld((const T*)p.gate + (long)b * p.gate_row + (long)h0 * E + tid) : 0.f;
    const float nw = tid < TEAMS * E ? p.norm_w[p.w_heads ? h0 * E + tid : tid % E] : 0.f;
    float4 S[RPT];
    float* sp = p.state + (((long)slot * H + h0 + team) * D + grp) * E + e;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int d = grp + i * groups;
        S[i] = has_past && in_state && d < D ? *reinterpret_cast<const float4*>(sp + i * step) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // ---- convolution, gates
    for (int c = tid; c < n; c += NT) {
        if (c >= NT) fetch(c);
        const int ch = channel(c);
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < NEXT_TAPS; ++j)
            if (j < taps) s += x[j] * w[j];
        // (the kernels of hybrid_delta.hip have filter_silu here: the same bits in 18 vector instructions instead of 25)
        (c < 2 * D ? ys + c + (c < D ? 0 : DP - D) : vs + c - 2 * D)[0] = siluf_(s);
#pragma unroll
        for (int j = 0; j < NEXT_TAPS - 1; ++j)
            if (j < taps - 1) tail[(long)j * C + ch] = x[j + 1];
    }
    for (int i = tid; i < TEAMS * p.DC; i += NT) {
        const int h = h0 + i / p.DC;
        const float spl = softplusf_(ld((const T*)p.a + (long)b * p.a_row + (long)h0 * p.DC + i) + p.dt_bias[h0 * p.DC + i]);
        dec[CHANNEL ? i / D * DP + i % D : i] = expf(-expf(p.a_log[h]) * spl);
        if (i % p.DC == 0) bt_[i / p.DC] = sigmoidf_(ld(row + p.b_off + h));
    }
    for (int i = tid; i < (2 + (CHANNEL ? TEAMS : 0)) * (DP - D); i += NT) {
        const int which = i / (DP - D), at = D + i % (DP - D);
        (which < 2 ? ys + which * DP : dec + (which - 2) * DP)[at] = 0.f;
    }
    // no rows: the sums over the row groups run by whole fours
    for (int i = tid; i < (padded - groups) * E * 2 * TEAMS; i += NT) {
        const int which = i / ((padded - groups) * E), at = i % ((padded - groups) * E);
        os[TEAMS * E + which * padded * E + groups * E + at] = 0.f;
    }
    __syncthreads();
    // ---- unit vectors: wave 0 q, wave 1 k, eight channels a lane
    if (tid < 128) {
        const int lane = tid & 63, runs = D >> 3;
        float* y = ys + (tid >> 6) * DP + lane * 8;
        float v[8], sq = 0.f;
        if (lane < runs) {
#pragma unroll
            for (int i = 0; i < 8; ++i) { v[i] = y[i]; sq += v[i] * v[i]; }
        }
        if ((runs & (runs - 1)) == 0) {
            for (int o = 1; o < runs; o <<= 1) sq += __shfl_xor(sq, o, kWave);
        } else {
            float s = 0.f;
            for (int i = 0; i < runs; ++i) s += __shfl(sq, i, kWave);
            sq = s;
        }
        float r = rsqrtf(sq + 1e-6f);
        if (tid < 64) r *= rsqrtf((float)D);
        if (lane < runs) {
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = v[i] * r;
        }
    }
    __syncthreads();
    // ---- the step (delta_step_kernel)
    const float bt = bt_[team], gh = CHANNEL ? 1.f : dec[team];
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (in_state) v = *reinterpret_cast<const float4*>(vs + team * E + e);
    if (CHANNEL)
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const float gd = dec[team * DP + grp + i * groups];
            S[i].x *= gd; S[i].y *= gd; S[i].z *= gd; S[i].w *= gd;
        }
    auto plus = [](float4 a, float4 c) { return make_float4(a.x + c.x, a.y + c.y, a.z + c.z, a.w + c.w); };
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    auto column_sums = [&](const float* vec, float* at) {
        float4 mine = zero;
#pragma unroll
        for (int i = 0; i < RPT; i += 4) {
            float4 four = zero;
#pragma unroll
            for (int j = i; j < min(i + 4, RPT); ++j) {
                const float f = vec[grp + j * groups];
                four.x += S[j].x * f; four.y += S[j].y * f; four.z += S[j].z * f; four.w += S[j].w * f;
            }
            mine = plus(mine, four);
        }
        if (in_state) *reinterpret_cast<float4*>(at + grp * E + e) = mine;
        __syncthreads();
        auto of = [&](int i) { return *reinterpret_cast<const float4*>(at + i * E + e); };
        float4 all[4] = {zero, zero, zero, zero};
        for (int i = 0; i < padded; i += 16)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i + 4 * j < padded) {
                    const int r = i + 4 * j;
                    all[j] = plus(all[j], plus(plus(of(r), of(r + 1)), plus(of(r + 2), of(r + 3))));
                }
        return plus(plus(all[0], all[1]), plus(all[2], all[3]));
    };
    const float4 sk = column_sums(ys + DP, sums);
    const float4 u = make_float4(bt * (v.x - gh * sk.x), bt * (v.y - gh * sk.y), bt * (v.z - gh * sk.z), bt * (v.w - gh * sk.w));
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int d = grp + i * groups;
        const float k = ys[DP + d];
        S[i].x = fmaf(gh, S[i].x, k * u.x); S[i].y = fmaf(gh, S[i].y, k * u.y);
        S[i].z = fmaf(gh, S[i].z, k * u.z); S[i].w = fmaf(gh, S[i].w, k * u.w);
        if (in_state && d < D) *reinterpret_cast<float4*>(sp + i * step) = S[i];
    }
    const float4 so = column_sums(ys, sums + padded * E);
    if (grp == 0) *reinterpret_cast<float4*>(os + team * E + e) = so;
    __syncthreads();
    // ---- gated norm of every head: its sum of squares by runs of eight, as lanes share them
    int lph = 4;
    while (lph * 8 < E) lph *= 2;
    if (tid < TEAMS * lph) {
        const int hd = tid / lph, c = tid % lph * 8;
        float s = 0.f;
        if (c < E)
#pragma unroll
            for (int i = 0; i < 8; ++i) { const float y = os[hd * E + c + i]; s += y * y; }
        for (int o = 1; o < lph; o <<= 1) s += __shfl_xor(s, o, kWave);
        if (c == 0) rn[hd] = rsqrtf(s / (float)E + p.eps);
    }
    __syncthreads();
    if (tid < TEAMS * E) st(out + tid, os[tid] * (rn[tid / E] * nw * (p.sig ? sigmoidf_(z) : siluf_(z))));
}

template <typename T, int TEAMS>
static int delta_next(const DeltaNext& p, int B, hipStream_t s) {
    const int groups = 256 / (p.E / 4), padded = (groups + 3) & ~3, rpt = (p.D + groups - 1) / groups;
    const bool channel = p.DC > 1;
#define NEXT(RPT)                                                                                                        \
    do {                                                                                                                 \
        const int DP = next_rows(RPT, groups);                                                                           \
        const size_t lds = (2 * DP + 2 * TEAMS * p.E + (channel ? TEAMS * DP : 4) + 8 + TEAMS * 2 * padded * p.E) * sizeof(float); \
        if (lds > 64 * 1024) return 1;                                                                                   \
        if (channel)                                                                                                     \
            hipLaunchKernelGGL((delta_next_kernel<T, TEAMS, RPT, true>), dim3(B, p.G), dim3(256 * TEAMS), lds, s, p);    \
        else                                                                                                             \
            hipLaunchKernelGGL((delta_next_kernel<T, TEAMS, RPT, false>), dim3(B, p.G), dim3(256 * TEAMS), lds, s, p);   \
    } while (0)
    if (rpt <= 2) NEXT(2);
    else if (rpt <= 4) NEXT(4);
    else if (rpt <= 8) NEXT(8);
    else NEXT(16);
#undef NEXT
    return HYB_LAUNCH_OK();
}

extern "C" {

// Whether hyb_delta_next takes these sizes: up to four value heads per key head, heads in whole runs of eight, a value
// row of 16 to 256 columns and no more than 16 rows of the state per thread, up to four taps.
int hyb_delta_next_ok(int H, int G, int D, int E, int taps) {
    if (G <= 0 || H % G || H / G > 4 || G > 65535 || taps < 1 || taps > NEXT_TAPS) return 0;
    if (D < 8 || D % 8 || D > 256 || E % 8 || E < 16 || E > 256) return 0;
    return D <= 16 * (256 / (E / 4));
}

// proj, a, gate and out are of the activation type, everything else fp32; B rows, row b is sequence b
int hyb_delta_next(const void* proj, long row, int b_off, const void* a, long a_row, int DC, const void* gate, long gate_row,
                   const void* conv_w, int taps, const void* a_log, const void* dt_bias, const void* norm_w, int w_heads,
                   void* conv_state, void* state, const void* positions, const void* slots, void* out, float eps, int sig,
                   int B, int H, int G, int D, int E, int dt, hipStream_t s) {
    if (B <= 0) return 0;
    if (!hyb_delta_next_ok(H, G, D, E, taps) || (DC != 1 && DC != D) || (size_t)state % 16) return 1;
    const DeltaNext p{proj, row, b_off, a, a_row, DC, gate, gate_row, (const float*)conv_w, (const float*)a_log,
                      (const float*)dt_bias, (const float*)norm_w, (float*)conv_state, (float*)state, (const int*)positions,
                      (const int*)slots, out, eps, taps, H, G, D, E, sig, w_heads};
    switch (H / G) {
        case 1: HYB_DISPATCH(dt, return (delta_next<T, 1>(p, B, s)));
        case 2: HYB_DISPATCH(dt, return (delta_next<T, 2>(p, B, s)));
        case 3: HYB_DISPATCH(dt, return (delta_next<T, 3>(p, B, s)));
        default: HYB_DISPATCH(dt, return (delta_next<T, 4>(p, B, s)));
    }
}

}  // extern "C"
