// Single next tokens of paged attention with the options of hybrid_attention.hip but pooled rows, temperatures and soft
// caps, over bfloat16 caches: fp32 scores, weights and sums on the bf16 matrix instruction.
//
// Workgroup = the query heads of one (sequence, KV head), up to 16, as columns of a product: S^T = K Q^T puts the head on
// the lane, which is the operand layout of O^T = V^T P^T as it stands; the weights are cut into three parts of eight
// bits, all of an fp32 weight.  Its waves walk their own tiles of 32 keys, each through an LDS image of its own
// that is filled from registers requested a tile ahead, and meet once, at the end: no barrier in the loop.  Keys that
// the token does not see (behind the context, outside the window) are zeros in the images.  A row that comes out with an
// infinity or a NaN is worked out again key by key.
//
// Reading the keys and values bounds it.  A workgroup that has a context to itself writes the result; the splits of a
// context are folded by a second kernel (how many: next_splits).  A page is looked up two tiles ahead of its use: one
// ahead, the rows behind it are asked for late (64 x 1024 keys two us more).
// 64 sequences of about 1024 keys, 16 / 8 heads of 128: 44.4 us a call among many (4.7 TB/s; the kernel alone 43).  A call among
// eight, in us, against the kernel on the vector units (scores by exchanges between 16 lanes) and its fold: 64 x 1024 keys
// 47 and 52, 128 x 1024 84 and 91, 32 x 1024 27 and 33, 16 x 2048 30 and 35, 64 of 200 and one of 8192 94 and 157, 1 x 512 19 and
// 25, 64 x 1024 under a window of 128 20 and 25, 1 x 2048 24 and 25 (both the launches).  Where the vector units are ahead:
// next_pays in ops/hip_hybrid.py.  Error 1.7e-3 of the result, its rounding, in both.
#include "hybrid_chunks.h"
#include "hybrid_row_by_keys.h"

using namespace hyb;

namespace {

struct NextArgs {
    const uint16_t* q; long q_row, q_head;
    const uint16_t *k_cache, *v_cache;
    const int* tables; int max_blocks, block_size;
    const int* lens;
    const float* sink;
    const bf16_t* gate; long gate_row;
    bf16_t* out;
    float* ws;                                     // splits > 1: [sequence, head, split][E + 2]: largest score, sum, row
    float scale;
    int H, G, splits, clear;
    KeyRule rule;
};

constexpr int TK = 32;

template <int CPR>
__device__ __forceinline__ int place(int row, int ch) {
    const int x = (((row & 7) << 1) | ((row >> 2) & 1)) & (CPR - 1);
    return row * (CPR * 16) + ((ch ^ x) << 4);
}

__device__ __forceinline__ void by_keys(const NextArgs& a, int b, int h, int L, int D, int E) {
    const int g = h / (a.H / a.G);
    row_by_keys<bf16_t, false>((const bf16_t*)a.q + (long)b * a.q_row + (long)h * a.q_head, (const bf16_t*)a.k_cache,
                               (const bf16_t*)a.v_cache, a.tables + (long)b * a.max_blocks, a.block_size, L, a.scale,
                               a.rule.slopes ? a.rule.slopes[h] : 0.f, a.sink, a.gate ? a.gate + (long)b * a.gate_row + h : nullptr,
                               a.out + ((long)b * a.H + h) * E, a.G, g, h, D, E, a.rule);
}

template <int D, int E, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, 2) next_attention_kernel(const NextArgs a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int KC = D / 8, VC = E / 8, KIT = TK * KC / 64, VIT = TK * VC / 64, KS = D / 32, NB = E / 16;
    constexpr int WAVE = TK * (D + E) * 2, LD = E + 4;
    static_assert(16 * LD * 4 + 128 <= WAVE);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ uint32_t lost;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c16 = lane & 15, q4 = lane >> 4;
    char *kim = smem + w * WAVE, *vim = kim + TK * D * 2;
    const int H = a.H, G = a.G, R = H / G, chunks = (R + 15) >> 4;
    // the heads of a context next to each other: their rows of a key are
    const int split = blockIdx.x % a.splits, chunk = blockIdx.x / a.splits % (G * chunks), b = blockIdx.x / a.splits / (G * chunks);
    const int g = chunk / chunks, h0 = g * R + (chunk - g * chunks) * 16, heads = min(16, g * R + R - h0);
    const int L = a.lens[b];
    if (L <= 0) {                                  // no sequence's row
        if (a.clear && split == 0)
            for (int i = threadIdx.x; i < heads * E; i += 64 * WAVES) st(a.out + ((long)b * H + h0) * E + i, 0.f);
        return;
    }
    const KeyRule& rule = a.rule;
    const int lo = rule.first_key(L - 1), keep = rule.keep_first, first_tile = lo / TK;
    const int ktiles = min((keep + TK - 1) / TK, first_tile);
    const int n_tiles = ktiles + (L + TK - 1) / TK - first_tile, per = (n_tiles + a.splits - 1) / a.splits;
    const int t1 = min(n_tiles, split * per + per);
    auto key_of = [&](int t) { return (t < ktiles ? t : t - ktiles + first_tile) * TK; };
    auto sees = [&](int key) { return key < L && (key >= lo || key < keep); };

    bf16x8 qf[KS];
    {
        const uint16_t* qp = a.q + (long)b * a.q_row + (long)(h0 + min(c16, heads - 1)) * a.q_head;
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + 32 * s + 8 * q4));
    }
    const float slope = rule.slopes ? rule.slopes[h0 + min(c16, heads - 1)] : 0.f;
    const int* table = a.tables + (long)b * a.max_blocks;
    const int shift = (a.block_size & (a.block_size - 1)) == 0 ? __builtin_ctz(a.block_size) : -1;
    const long krow = (long)G * D, vrow = (long)G * rule.v_stride;
    const uint16_t *kh = a.k_cache + g * D, *vh = a.v_cache + (long)g * rule.v_stride;
    auto page_of = [&](int key) { return shift >= 0 ? key >> shift : key / a.block_size; };
    typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
    u32x4 kr[KIT], vr[VIT];
    // pages of a tile's rows, looked up a tile ahead of the rows (as they come: arithmetic on them here would be waited for,
    // and with it all rows in flight)
    int kp[KIT], vp[E == D ? 1 : VIT];
    auto look = [&](int t) {
        const int k0 = key_of(t);
#pragma unroll
        for (int i = 0; i < KIT; ++i) kp[i] = table[page_of(min(k0 + (i * 64 + lane) / KC, L - 1))];
        if constexpr (E != D)
#pragma unroll
            for (int i = 0; i < VIT; ++i) vp[i] = table[page_of(min(k0 + (i * 64 + lane) / VC, L - 1))];
    };
    auto fetch = [&](int t) {
        const int k0 = key_of(t);
        auto slot = [&](int page, int row) {
            const int key = min(k0 + row, L - 1);
            return (long)page * a.block_size + (key - page_of(key) * a.block_size);
        };
#pragma unroll
        for (int i = 0; i < KIT; ++i)
            kr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kh + slot(kp[i], (i * 64 + lane) / KC) * krow + (i * 64 + lane) % KC * 8));
#pragma unroll
        for (int i = 0; i < VIT; ++i)
            vr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
                vh + slot(E == D ? kp[i] : vp[E == D ? 0 : i], (i * 64 + lane) / VC) * vrow + (i * 64 + lane) % VC * 8));
    };
    float m_run = NO_SINK_MAX, l_run = 0.f;
    f32x4 acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n] = {0.f, 0.f, 0.f, 0.f};
    int t = split * per + w;
    if (t < t1) {
        look(t);
        fetch(t);
        if (t + WAVES < t1) look(t + WAVES);
    }
    for (; t < t1; t += WAVES) {
        const int k0 = key_of(t);
        const bool whole = k0 + TK <= L && (k0 >= lo || k0 + TK <= keep);       // (uniform)
#pragma unroll
        for (int i = 0; i < KIT; ++i) {
            const int c = i * 64 + lane;
            u32x4 x = kr[i];
            if (!whole && !sees(k0 + c / KC)) x = u32x4{0, 0, 0, 0};
            *reinterpret_cast<u32x4*>(kim + place<KC>(c / KC, c % KC)) = x;
        }
#pragma unroll
        for (int i = 0; i < VIT; ++i) {
            const int c = i * 64 + lane;
            u32x4 x = vr[i];
            if (!whole && !sees(k0 + c / VC)) x = u32x4{0, 0, 0, 0};
            *reinterpret_cast<u32x4*>(vim + place<VC>(c / VC, c % VC)) = x;
        }
        if (t + WAVES < t1) {
            fetch(t + WAVES);
            if (t + 2 * WAVES < t1) look(t + 2 * WAVES);
        }
        lanes_meet();                              // the images are there
        // scores of two blocks of 16 keys: lane = head c16, keys 16 x + 4 q4 + r.  Sums of 32 channels stay apart to the end, and
        // log2(e) comes to the difference from the largest: as one chain, and with it in the scores, they were 1.2 to 1.3 times as
        // far from 64 bits as on the vector units where a context has few large weights; now 0.84 to 1.02 times (1 % of the time)
        float p[8], top = -INFINITY;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            f32x4 part[KS];
#pragma unroll
            for (int i = 0; i < KS; ++i)
                part[i] = mfma(*reinterpret_cast<const bf16x8*>(kim + place<KC>(16 * x + c16, 4 * i + q4)), qf[i], f32x4{0.f, 0.f, 0.f, 0.f});
            const f32x4 s = KS == 2 ? part[0] + part[1] : (part[0] + part[1]) + (part[KS - 2] + part[KS - 1]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = k0 + 16 * x + 4 * q4 + r;
                float v = s[r] * a.scale;
                if (rule.slopes) v -= slope * (float)(L - 1 - key);
                if (!whole && !sees(key)) v = -INFINITY;
                p[4 * x + r] = v;
                top = fmaxf(top, v);
            }
        }
        top = fmaxf(top, __shfl_xor(top, 16, kWave));
        top = fmaxf(top, __shfl_xor(top, 32, kWave));
        const float m_new = fmaxf(m_run, top), f = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
        l_run *= f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = __builtin_amdgcn_exp2f((p[j] - m_new) * LOG2E);
            l_run += p[j];
        }
        m_run = m_new;
        bf16x8 pf[3];
        split8(p, pf);
        if (__builtin_amdgcn_ballot_w64(f != 1.f) != 0) {
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[n] *= f;
        }
        const int row = 4 * q4 + (c16 >> 2);
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int ch = 2 * n + ((c16 & 3) >> 1);
            const bf16x8 vf = join(read_tr(vim + place<VC>(row, ch) + (c16 & 1) * 8), read_tr(vim + place<VC>(16 + row, ch) + (c16 & 1) * 8));
#pragma unroll
            for (int k = 2; k >= 0; --k) acc[n] = mfma(vf, pf[k], acc[n]);
        }
        lanes_meet();                              // and have been read
    }
    // ---- the waves' sums through LDS, each in its own place
    l_run += __shfl_xor(l_run, 16, kWave);
    l_run += __shfl_xor(l_run, 32, kWave);
    float* mine = reinterpret_cast<float*>(kim);
    if (q4 == 0) { mine[c16] = m_run; mine[16 + c16] = l_run; }
#pragma unroll
    for (int n = 0; n < NB; ++n) *reinterpret_cast<f32x4*>(mine + 32 + c16 * LD + 16 * n + 4 * q4) = acc[n];
    if (threadIdx.x == 0) lost = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < heads * E; i += 64 * WAVES) {
        const int c = i / E, d = i - c * E, h = h0 + c;
        float M = NO_SINK_MAX, o = 0.f, l = 0.f;
#pragma unroll
        for (int x = 0; x < WAVES; ++x) M = fmaxf(M, reinterpret_cast<const float*>(smem + x * WAVE)[c]);
#pragma unroll
        for (int x = 0; x < WAVES; ++x) {
            const float* y = reinterpret_cast<const float*>(smem + x * WAVE);
            const float f = expf(y[c] - M);
            o += y[32 + c * LD + d] * f;
            l += y[16 + c] * f;
        }
        if (a.splits > 1) {
            float* to = a.ws + (((long)b * H + h) * a.splits + split) * (E + 2);
            if (d == 0) { to[0] = M; to[1] = l; }
            to[2 + d] = o;
        } else {
            float f = 1.f;
            if (a.sink) {
                const float sk = a.sink[h], top = fmaxf(M, sk);
                f = expf(M - top);
                l = l * f + expf(sk - top);
            }
            f = f / l;
            if (a.gate) f *= sigmoidf_(ld(a.gate + (long)b * a.gate_row + h));
            o *= f;
            if (o * 0.f != 0.f) atomicOr(&lost, 1u << c);
            st(a.out + ((long)b * H + h) * E + d, o);
        }
    }
    if (a.splits > 1) return;
    __syncthreads();
    for (uint32_t left = lost, n = 0; left; left &= left - 1, ++n)
        if ((int)(n % WAVES) == w) by_keys(a, b, h0 + __builtin_ctz(left), L, D, E);
#endif
}

// the splits' partial results of a (sequence, head); E threads
template <int D, int E>
__global__ void __launch_bounds__(E) next_fold_kernel(const NextArgs a) {
    const int b = blockIdx.x / a.H, h = blockIdx.x % a.H, e = threadIdx.x, L = a.lens[b];
    if (L <= 0) return;                            // (cleared where asked for)
    const float* p = a.ws + ((long)b * a.H + h) * a.splits * (E + 2);
    const float sk = a.sink ? a.sink[h] : 0.f;
    float M = a.sink ? sk : NO_SINK_MAX;
    for (int s = 0; s < a.splits; ++s) M = fmaxf(M, p[s * (E + 2)]);
    float l = a.sink ? expf(sk - M) : 0.f, o = 0.f;
    for (int s = 0; s < a.splits; ++s) {
        const float f = expf(p[s * (E + 2)] - M);
        l += p[s * (E + 2) + 1] * f;
        o += p[s * (E + 2) + 2 + e] * f;
    }
    float f = 1.f / l;
    if (a.gate) f *= sigmoidf_(ld(a.gate + (long)b * a.gate_row + h));
    o *= f;
    const bool lost = __syncthreads_or(o * 0.f != 0.f);
    st(a.out + ((long)b * a.H + h) * E + e, o);
    if (!lost) return;
    __syncthreads();
    if (e < 64) by_keys(a, b, h, L, D, E);
}

template <int D, int E, int WAVES>
int launch(const NextArgs& a, int B, hipStream_t s) {
    constexpr int lds = WAVES * TK * (D + E) * 2;
    if constexpr (lds + 64 > 64 * 1024) {              // (the kernel has a few bytes of its own)
        static const hipError_t once = hipFuncSetAttribute((const void*)next_attention_kernel<D, E, WAVES>,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (once != hipSuccess) return 2;
    }
    const int chunks = (a.H / a.G + 15) / 16;
    hipLaunchKernelGGL((next_attention_kernel<D, E, WAVES>), dim3((unsigned)a.splits * a.G * chunks * B), dim3(64 * WAVES), lds, s, a);
    if (a.splits > 1) hipLaunchKernelGGL((next_fold_kernel<D, E>), dim3((unsigned)B * a.H), dim3(E), 0, s, a);
    return HYB_LAUNCH_OK();
}

}  // namespace

extern "C" {

int hyb_next_attention_ok(int D, int E) { return (D == 64 || D == 128) && (E == 64 || E == 128); }

// Row b is sequence b with lens[b] keys.  ws: B * H * splits * (E + 2) floats where splits > 1; clear: rows without a
// context become zeros.  Caches, gate and out as hyb_sink_attention_split, in bfloat16.
int hyb_next_attention(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache, const void* tables,
                       int max_blocks, int block_size, const void* lens, const void* sink, const void* gate, long gate_row,
                       void* out, void* ws, float scale, int B, int H, int G, int D, int E, int splits, int window,
                       int keep_first, const void* slopes, int v_stride, int chunk, int clear, hipStream_t s) {
    KeyRule rule{};
    rule.window = window; rule.keep_first = keep_first; rule.slopes = (const float*)slopes;
    rule.v_stride = v_stride > 0 ? v_stride : E; rule.chunk = chunk;
    if (B <= 0) return 0;
    if (!hyb_next_attention_ok(D, E) || !chunk_rule_ok(rule) || G <= 0 || H % G || splits < 1 || splits > 64 || block_size <= 0) return 1;
    if (rule.v_stride < E || rule.v_stride % 8 || (splits > 1 && !ws)) return 1;
    if (((size_t)q | (size_t)k_cache | (size_t)v_cache) % 16 || q_row % 8 || q_head % 8) return 1;
    const NextArgs a{(const uint16_t*)q, q_row, q_head, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (const int*)tables,
                     max_blocks, block_size, (const int*)lens, (const float*)sink, (const bf16_t*)gate, gate_row, (bf16_t*)out,
                     (float*)ws, scale, H, G, splits, clear, rule};
    // eight waves where every workgroup finds a CU of its own
    const bool wide = (long)splits * G * ((H / G + 15) / 16) * B <= 256;
#define NEXT(D_, E_) if (D == D_ && E == E_) return wide ? launch<D_, E_, 8>(a, B, s) : launch<D_, E_, 4>(a, B, s)
    NEXT(128, 128);
    NEXT(64, 64);
    NEXT(128, 64);
    NEXT(64, 128);
#undef NEXT
    return 1;
}

}  // extern "C"
