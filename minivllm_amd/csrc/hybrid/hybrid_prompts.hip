// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form
// (the flag: results of matrix products stay in ordinary vector registers, where the softmax rescales them)
// Prompt portions of paged attention with the options of hybrid_attention.hip, for bfloat16 caches:
// fp32 scores, weights and sums on the bf16 matrix instruction.
//
//   S^T = K Q^T on v_mfma_f32_32x32x16_bf16 (a lane owns one query and 16 of a step's 32 keys),
//   softmax with a running reference per lane, O^T += V^T P^T on the same instruction.
//
// The operands of the scores ARE bfloat16, so their products are exact.  The weights stay fp32: each
// is cut into parts of eight bits (PARTS of them; three hold all 24) that are multiplied one after the
// other.  The score accumulators are the B operand as they stand, V^T fragments are transposed LDS reads.
//
// Workgroup = 4 waves x 32 consecutive queries of one (sequence, query head); keys in tiles of TK, K and
// V each an LDS image filled by direct global -> LDS loads, two buffers, the next tile requested
// before the current one's products.  A page that holds whole tiles is read through one buffer
// descriptor per tile (rows behind the context are out of its range and read as zeros); smaller pages
// and pooled rows look every row up.  Heads of one KV head go to one XCD, long contexts start first.
//
// Bound by the wave's own chain of score product, softmax and value product with two waves per SIMD
// (about 220 registers).  8 prompts of 512..1024 tokens, 16 / 8 heads of 128, sink and gate: 69 us
// = 350 TFLOP/s of the products a bf16 softmax would need, against 566 us of the fp32 instruction over
// tiles widened to fp32 in LDS and loaded between two barriers.  Two parts per weight instead of three
// would take 58 us and hold 16 bits of it; key tiles of 32 take 70 us, the two halves of a tile of 64
// unrolled 73 us (registers spill).
#include "hybrid_keys.h"
#include "hybrid_chunks.h"

using namespace hyb;

namespace {

constexpr int PARTS = 3;

struct PromptArgs {
    const uint16_t* q; long q_row, q_head;
    const uint16_t *k_cache, *v_cache;
    const int* tables; int max_blocks, block_size;
    const int *cu_q, *positions;
    const float* sink;
    const bf16_t* gate; long gate_row;
    uint16_t* out;
    float scale;
    int H, G, D, E, seq0;
    KeyRule rule;
};

// rows of the wave (lane: a row and half of its columns, acc times f) with an infinity or a NaN
template <int NB>
__device__ __forceinline__ uint32_t rows_not_finite(const f32x16* acc, float f, bool ok) {
    f32x16 sum = acc[0];
#pragma unroll
    for (int n = 1; n < NB; ++n) sum += acc[n];
#pragma unroll
    for (int w = 8; w > 0; w >>= 1)
#pragma unroll
        for (int e = 0; e < w; ++e) sum[e] += sum[e + w];
    const uint64_t odd = __ballot(ok && sum[0] * f * 0.f != 0.f);
    return (uint32_t)odd | (uint32_t)(odd >> 32);
}

// Infinities and NaN.  A key may be infinite without the row being lost (its score is -infinity and its weight
// zero), and so may a value (the row's entry in that column is infinite, and no other row's); but part times
// part, padding column times anything, and zero weight times what no query sees would make NaN of them.  NaN and
// infinities stay in a row's sums once they are there, so a row that comes out finite met none, and the others are
// worked out again by all lanes of their wave: one query, key after key, nothing in parts.
template <typename T, bool EXT>
__device__ void row_by_keys(const T* q, const T* k_cache, const T* v_cache, const int* table, int block_size, int ctx,
                            float scale, float slope, const float* sink, const T* gate, T* out, int G, int g, int h,
                            int D, int E, const KeyRule& rule) {
    constexpr int N = 256 / kWave;                 // of up to 256 columns, lane + 64 i are this lane's
    const int lane = threadIdx.x & 63;
    const VisibleKeys vis(ctx, rule);
    float qf[N], acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        qf[i] = lane + 64 * i < D ? ld(q + lane + 64 * i) * scale : 0.f;
        acc[i] = 0.f;
    }
    float m = sink ? sink[h] : NO_SINK_MAX, l = sink ? 1.f : 0.f;
    for (int v = 0; v < vis.count; ++v) {
        const long row = vis.row(v, table, block_size, rule) * G + g;
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (lane + 64 * i < D) s += ld(k_cache + row * D + lane + 64 * i) * qf[i];
        s = wave_sum(s);
        if (EXT) s = rule.capped(s);
        s -= slope * (float)(ctx - 1 - vis.key(v));
        const float top = fmaxf(m, s), f = expf(m - top), w = expf(s - top);
        l = l * f + w;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int e = lane + 64 * i;
            acc[i] = acc[i] * f + w * (e < E ? ld(v_cache + row * (long)rule.v_stride + e) : 0.f);
        }
        m = top;
    }
    float f = 1.f / l;
    if (gate) f *= sigmoidf_(ld(gate));
#pragma unroll
    for (int i = 0; i < N; ++i)
        if (lane + 64 * i < E) st(out + lane + 64 * i, acc[i] * f);
}

template <int DP, int EP, int TK, bool EXT>
__global__ void __launch_bounds__(256, DP + EP > 256 ? 1 : 2)
prompt_attention_kernel(PromptArgs a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    static_assert(DP % 64 == 0 && EP % 64 == 0 && TK % 32 == 0);
    constexpr int KS = DP / 16, NB = EP / 32;      // steps of the score product; 32-wide value blocks
    constexpr int KT = TK * DP * 2, VT = TK * EP * 2, BUF = KT + VT;          // bytes
    constexpr int KIT = KT / 4096, VIT = VT / 4096;                           // 16-byte pieces per thread
    constexpr int KSW = DP % 128 == 0 ? 16 : 8, VSW = EP % 128 == 0 ? 16 : 8; // chunks a swizzle permutes
    extern __shared__ __attribute__((aligned(256))) char smem[];

    const int H = a.H, hx = blockIdx.x;
    const int h = H % 8 == 0 ? (hx & 7) * (H >> 3) + (hx >> 3) : hx;
    const int b = blockIdx.y + a.seq0, tile_q0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * 128;
    const int row0 = a.cu_q[b], qlen = a.cu_q[b + 1] - row0;
    if (tile_q0 >= qlen) return;
    const int start = a.positions[row0], G = a.G, g = h / (H / G);
    const int* table = a.tables + (long)b * a.max_blocks;
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int wq0 = tile_q0 + wave * 32, qi = wq0 + l32;
    const bool qok = qi < qlen, wave_live = wq0 < qlen;
    const int qpos = start + qi;
    bf16x8 qf[KS];
    {
        const uint16_t* qp = a.q + (long)(row0 + min(qi, qlen - 1)) * a.q_row + (long)h * a.q_head;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 16 * s + 8 * half;
            uint4 raw = make_uint4(0, 0, 0, 0);                     // columns from D on: zeros
            if (d < a.D) raw = *reinterpret_cast<const uint4*>(qp + d);
            qf[s] = __builtin_bit_cast(bf16x8, raw);
        }
    }

    // ---- the tiles this workgroup walks: pooled rows, kept first tokens, the tokens its window reaches
    const KeyRule& rule = a.rule;
    const int wg_ctx = start + min(qlen, tile_q0 + 128);
    const int wave_first = start + wq0, wave_last = start + min(qlen - 1, wq0 + 31);
    const int wg_lo = rule.first_key(start + tile_q0), wave_lo = rule.first_key(wave_first);
    const int q_lo = rule.first_key(qpos);
    const int wave_top = rule.first_key(wave_last);      // every query of the wave sees the keys from here on
    const int wg_nb = EXT ? rule.pooled_for(wg_ctx) : 0, wave_nb = EXT ? rule.pooled_for(wave_last + 1) : 0;
    const int q_nb = EXT ? rule.pooled_for(qpos + 1) : 0;
    const int ptiles = (wg_nb + TK - 1) / TK, first_tile = wg_lo / TK;
    const int ktiles = min((rule.keep_first + TK - 1) / TK, first_tile);
    const int n_tiles = ptiles + ktiles + (wg_ctx + TK - 1) / TK - first_tile;
    auto tile_key = [&](int t) { return (t < ptiles ? t : t < ptiles + ktiles ? t - ptiles : t - ptiles - ktiles + first_tile) * TK; };

    // ---- staging: slot c of an image (row c / chunks per row) receives the chunk that the swizzle puts
    // there; chunks behind a row's end repeat chunk 0 (their queries are zeros, their columns not stored)
    const int krow = G * a.D * 2, vrow = G * rule.v_stride * 2;     // bytes from one token's row to the next
    int k_off[KIT], v_off[VIT];
#pragma unroll
    for (int i = 0; i < KIT; ++i) {
        const int c = i * 256 + tid, row = c / (DP / 8);
        int ch = (c % (DP / 8)) ^ swizzle<DP>(row);
        if (ch * 8 >= a.D) ch = 0;
        k_off[i] = row * krow + ch * 16;
    }
#pragma unroll
    for (int i = 0; i < VIT; ++i) {
        const int c = i * 256 + tid, row = c / (EP / 8);
        int ch = (c % (EP / 8)) ^ swizzle<EP>(row);
        if (ch * 8 >= a.E) ch = 0;
        v_off[i] = row * vrow + ch * 16;
    }
    const bool whole = a.block_size % TK == 0;           // a tile of tokens lies in one page
    typedef const __attribute__((address_space(4))) int* const_int_p;
    auto page_of = [&](int t) {                          // through the scalar unit (the table is read-only here)
        return *(const_int_p)(uintptr_t)(table + min(tile_key(t), wg_ctx - 1) / a.block_size);
    };
    int page = 0;                                        // of the tile to be staged next
    auto stage = [&](int t, int buf) {
        const int key0 = tile_key(t);
        const bool pooled = EXT && t < ptiles;
        char* dst = smem + buf * BUF + wave * 1024;
        if (whole && !pooled) {
            const long slot = (long)page * a.block_size + key0 % a.block_size;
            const int rows = min(TK, wg_ctx - key0) - 1;
            const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint16_t*>(a.k_cache + (slot * G + g) * a.D), 0, rows * krow + a.D * 2, 0x00020000);
            const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint16_t*>(a.v_cache + (slot * G + g) * rule.v_stride), 0, rows * vrow + a.E * 2, 0x00020000);
#pragma unroll
            for (int i = 0; i < KIT; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    kr, (__attribute__((address_space(3))) void*)(dst + i * 4096), 16, k_off[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < VIT; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    vr, (__attribute__((address_space(3))) void*)(dst + KT + i * 4096), 16, v_off[i], 0, 0, 0);
        } else {
            const int lim = (pooled ? wg_nb : wg_ctx) - 1;
            auto cache_row = [&](int j) -> long {
                return pooled ? rule.pooled_row(table, j) : (long)table[j / a.block_size] * a.block_size + j % a.block_size;
            };
#pragma unroll
            for (int i = 0; i < KIT; ++i) {
                const int row = (i * 256 + tid) / (DP / 8);
                const char* src = reinterpret_cast<const char*>(a.k_cache) +
                                  (cache_row(min(key0 + row, lim)) * G + g) * a.D * 2 + (k_off[i] - row * krow);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)(dst + i * 4096), 16, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < VIT; ++i) {
                const int row = (i * 256 + tid) / (EP / 8);
                const char* src = reinterpret_cast<const char*>(a.v_cache) +
                                  (cache_row(min(key0 + row, lim)) * G + g) * (long)rule.v_stride * 2 + (v_off[i] - row * vrow);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)(dst + KT + i * 4096), 16, 0, 0);
            }
        }
    };

    // ---- LDS addresses of this lane's fragments inside a buffer
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)smem;
    uint32_t k_addr[KSW / 2];                       // row l32, chunk 2 s + half: distinct for s < KSW / 2
#pragma unroll
    for (int s = 0; s < KSW / 2; ++s) k_addr[s] = lds0 + l32 * (DP * 2) + (((2 * s + half) ^ swizzle<DP>(l32)) << 4);
    // transposed reads: 16 lanes take 4 key rows x 16 columns and return 4 keys of one column each
    constexpr int NA = NB < VSW / 4 ? NB : VSW / 4; // value blocks with addresses of their own
    const int i16 = lane & 15, tr_row = 4 * half + (i16 >> 2);
    const int tr_chunk = 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1);
    uint32_t v_addr[NA][2];
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            const int row = tr_row + 8 * hi;
            v_addr[n][hi] = lds0 + KT + row * (EP * 2) + (((4 * n + tr_chunk) ^ swizzle<EP>(row)) << 4) + (i16 & 1) * 8;
        }

    f32x16 acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[n][e] = 0.f;
    float m_run = NO_SINK_MAX, l_run = 0.f;         // in log2 units of the scores
    const float sc = (EXT ? rule.head_scale(a.scale, h) : a.scale) * (EXT ? 1.f : LOG2E);
    const float slope = rule.slopes ? rule.slopes[h] * LOG2E : 0.f;

    page = page_of(0);
    stage(0, 0);
    if (n_tiles > 1) page = page_of(1);
    __syncthreads();
    for (int t = 0, buf = 0; t < n_tiles; ++t, buf ^= 1) {
        if (t + 1 < n_tiles) {
            stage(t + 1, buf ^ 1);
            if (t + 2 < n_tiles) page = page_of(t + 2);
        }
        const int key0 = tile_key(t);
        const bool pooled = EXT && t < ptiles;
#pragma unroll 1
        for (int j = 0; j < TK / 32; ++j) {
            const int k0 = key0 + 32 * j;
            const bool live = wave_live && (pooled ? k0 < wave_nb
                                                   : (k0 <= wave_last && (k0 < rule.keep_first || k0 + 32 > wave_lo)));
            if (!live) continue;                                     // (uniform per wave)
            f32x16 s_acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) s_acc[e] = 0.f;
            uint32_t ka[KSW / 2];
#pragma unroll
            for (int s = 0; s < KSW / 2; ++s) ka[s] = k_addr[s] + buf * BUF + j * (32 * DP * 2);
            // (inline asm: through the builtin the compiler would wait for the stage's loads in flight
            // ahead of the first read; AHEAD reads are in flight)
            constexpr int KA = 4;
            s16x8 kf[KS];
            auto read_k = [&](auto ic) {
                constexpr int i = decltype(ic)::value;
                constexpr int off = (i / (KSW / 2)) * (KSW * 16);
                const uint32_t a0 = ka[i % (KSW / 2)];
                s16x8 x;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x) : "v"(a0), "n"(off));
                kf[i] = x;
            };
            static_for<0, (KA < KS ? KA : KS)>(read_k);
            static_for<0, KS>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i + KA < KS) read_k(std::integral_constant<int, i + KA>{});
                constexpr int left = KS - 1 - i < KA ? KS - 1 - i : KA;      // reads still in flight
                s16x8 x = kf[i];
                asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(x) : "n"(left));
                s_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), qf[i], s_acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            // lane: query qi, keys k0 + (e & 3) + 8 (e >> 2) + 4 half
#pragma unroll
            for (int e = 0; e < 16; ++e) s_acc[e] = EXT ? rule.capped(s_acc[e] * sc) * LOG2E : s_acc[e] * sc;
            if (rule.slopes && !pooled) {
#pragma unroll
                for (int e = 0; e < 16; ++e) s_acc[e] -= slope * (float)(qpos - (k0 + (e & 3) + 8 * (e >> 2) + 4 * half));
            }
            const bool all_seen = pooled ? k0 + 32 <= rule.pooled_for(wave_first + 1)
                                         : k0 + 31 <= wave_first && k0 >= wave_top;
            if (!all_seen) {                                         // (one uniform branch, not one per score)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = k0 + (e & 3) + 8 * (e >> 2) + 4 * half;
                    const bool seen = pooled ? key < q_nb : (key <= qpos) & ((key >= q_lo) | (key < rule.keep_first));
                    s_acc[e] = seen ? s_acc[e] : -INFINITY;
                }
            }
            float mt = s_acc[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mt = fmaxf(mt, s_acc[e]);
            mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
            // the reference of the exponentials only moves when some row outgrows it by RESCALE
            if (!__all(mt - m_run <= RESCALE)) {
                const float m_new = fmaxf(m_run, mt);
                const float f = __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= f;
#pragma unroll
                for (int n = 0; n < NB; ++n) acc[n] *= f;
                m_run = m_new;
            }
            // part k of a pair of weights: the upper halves of what the parts before it left over
            bf16x8 p[PARTS][2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t w[PARTS][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float x = __builtin_amdgcn_exp2f(s_acc[8 * s + 2 * j] - m_run);
                    float y = __builtin_amdgcn_exp2f(s_acc[8 * s + 2 * j + 1] - m_run);
                    l_run += x;
                    l_run += y;
#pragma unroll
                    for (int k = 0; k < PARTS; ++k) {
                        const uint32_t ux = __float_as_uint(x), uy = __float_as_uint(y);
                        w[k][j] = __builtin_amdgcn_perm(uy, ux, 0x07060302);
                        if (k + 1 < PARTS) {
                            x -= __uint_as_float(ux & 0xffff0000u);
                            y -= __uint_as_float(uy & 0xffff0000u);
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < PARTS; ++k)
                    p[k][s] = __builtin_bit_cast(bf16x8, make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]));
            }
            // step i: value block i / 2, keys 16 (i & 1) .. of the 32; requested AHEAD steps early
            constexpr int STEPS = 2 * NB, AHEAD = STEPS < 4 ? STEPS : 4;
            s16x4 lo4[STEPS], hi4[STEPS];
            uint32_t va[NA][2];
#pragma unroll
            for (int n = 0; n < NA; ++n) {
                va[n][0] = v_addr[n][0] + buf * BUF + j * (32 * EP * 2);
                va[n][1] = v_addr[n][1] + buf * BUF + j * (32 * EP * 2);
            }
            auto read_v = [&](auto ic) {
                constexpr int i = decltype(ic)::value, n = i >> 1, s = i & 1;
                constexpr int off = (n / NA) * NA * 64 + s * 16 * EP * 2;
                const uint32_t a0 = va[n % NA][0], a1 = va[n % NA][1];
                s16x4 x, y;
                asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(x) : "v"(a0), "n"(off));
                asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(y) : "v"(a1), "n"(off));
                lo4[i] = x;
                hi4[i] = y;
            };
            static_for<0, AHEAD>(read_v);
            static_for<0, STEPS>([&](auto ic) {
                constexpr int i = decltype(ic)::value, n = i >> 1, s = i & 1;
                if constexpr (i + AHEAD < STEPS) read_v(std::integral_constant<int, i + AHEAD>{});
                constexpr int left = 2 * (STEPS - 1 - i < AHEAD ? STEPS - 1 - i : AHEAD);   // reads still in flight
                s16x4 x = lo4[i], y = hi4[i];
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(x), "+v"(y) : "n"(left));
                const s16x8 v = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                const bf16x8 vf = __builtin_bit_cast(bf16x8, v);
#pragma unroll
                for (int k = 0; k < PARTS; ++k)
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, p[k][s], acc[n], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        __syncthreads();
    }
    if (!wave_live) return;
    l_run += __shfl_xor(l_run, 32, kWave);
    float f;
    if (a.sink) {
        const float sk = a.sink[h] * LOG2E, M = fmaxf(m_run, sk);
        f = __builtin_amdgcn_exp2f(m_run - M);
        f = f / (l_run * f + __builtin_amdgcn_exp2f(sk - M));
    } else {
        f = 1.f / l_run;
    }
    const long row = row0 + min(qi, qlen - 1);
    if (a.gate) f *= sigmoidf_(ld(a.gate + row * a.gate_row + h));
    uint32_t lost = rows_not_finite<NB>(acc, f, qok);
    // both halves of the wave hold every second run of four columns of a row: swapped so that a
    // lane stores eight neighbouring ones
    uint16_t* op = a.out + (row * H + h) * a.E;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                w[k] = (uint32_t)bf16_bits(acc[n][4 * r + 2 * k] * f) |
                       ((uint32_t)bf16_bits(acc[n][4 * r + 2 * k + 1] * f) << 16);
            const uint32_t s0 = half ? w[0] : w[2], s1 = half ? w[1] : w[3];
            const uint32_t g0 = __shfl_xor(s0, 32, kWave), g1 = __shfl_xor(s1, 32, kWave);
            const uint4 v = half ? make_uint4(g0, g1, w[2], w[3]) : make_uint4(w[0], w[1], g0, g1);
            const int e = 32 * n + 8 * r + 8 * half;
            if (qok && e < a.E && !(lost >> l32 & 1)) *reinterpret_cast<uint4*>(op + e) = v;
        }
    for (; lost; lost &= lost - 1) {
        const int i = __builtin_ctz(lost);
        const long r = row0 + wq0 + i;
        row_by_keys<bf16_t, EXT>((const bf16_t*)a.q + r * a.q_row + (long)h * a.q_head, (const bf16_t*)a.k_cache,
                                 (const bf16_t*)a.v_cache, table, a.block_size, start + wq0 + i + 1,
                                 EXT ? rule.head_scale(a.scale, h) : a.scale, rule.slopes ? rule.slopes[h] : 0.f, a.sink,
                                 a.gate ? a.gate + r * a.gate_row + h : nullptr, (bf16_t*)a.out + (r * H + h) * a.E, G, g,
                                 h, a.D, a.E, rule);
    }
#endif
}

// The same over float caches: keys, values, queries and weights all fp32, each cut into three parts; a
// product is the sum of the six largest products of parts.  Key tiles of 32; K and V are
// in registers a tile ahead and go to LDS as images of their parts, one buffer.  Exponentials are expf of
// the difference, as in the general kernel.
// Against the fp32 instruction (2.7 times the cycles) behind loads that nothing hid: 3 prompts of 300..611
// tokens, window 256, 8 heads of 64: 90 -> 39 us with the fill of the output ahead of it, 1.9e-7 from 64 bits
// instead of 2.7e-7.
struct PromptArgs32 {
    const float* q; long q_row, q_head;
    const float *k_cache, *v_cache;
    const int* tables; int max_blocks, block_size;
    const int *cu_q, *positions;
    const float* sink;
    const float* gate; long gate_row;
    float* out;
    float scale;
    int H, G, D, E, seq0;
    KeyRule rule;
};

template <int DP, int EP, bool EXT>
__global__ void __launch_bounds__(256, 1)
prompt_attention_f32_kernel(PromptArgs32 a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int TK = 32, KS = DP / 16, NB = EP / 32;
    constexpr int KT = TK * DP * 2, VT = TK * EP * 2;                         // bytes of a part's image
    constexpr int KIT = TK * DP / 8 / 256, VIT = TK * EP / 8 / 256;           // runs of eight per thread
    extern __shared__ __attribute__((aligned(256))) char smem[];
    char *kim = smem, *vim = smem + 3 * KT;

    const int H = a.H, hx = blockIdx.x;
    const int h = H % 8 == 0 ? (hx & 7) * (H >> 3) + (hx >> 3) : hx;
    const int b = blockIdx.y + a.seq0, tile_q0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * 128;
    const int row0 = a.cu_q[b], qlen = a.cu_q[b + 1] - row0;
    if (tile_q0 >= qlen) return;
    const int start = a.positions[row0], G = a.G, g = h / (H / G);
    const int* table = a.tables + (long)b * a.max_blocks;
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq0 = tile_q0 + wave * 32, qi = wq0 + l32;
    const bool qok = qi < qlen, wave_live = wq0 < qlen;
    const int qpos = start + qi;
    const float sc = EXT ? a.rule.head_scale(a.scale, h) : a.scale;
    bf16x8 qf[KS][3];
    {
        const float* qp = a.q + (long)(row0 + min(qi, qlen - 1)) * a.q_row + (long)h * a.q_head;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 16 * s + 8 * half;
            float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (d < a.D) load_run<float, 8>(qp + d, x);
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] *= sc;
            split8(x, qf[s]);
        }
    }
    const KeyRule& rule = a.rule;
    const int wg_ctx = start + min(qlen, tile_q0 + 128);
    const int wave_first = start + wq0, wave_last = start + min(qlen - 1, wq0 + 31);
    const int wg_lo = rule.first_key(start + tile_q0), wave_lo = rule.first_key(wave_first);
    const int q_lo = rule.first_key(qpos), wave_top = rule.first_key(wave_last);
    const int wg_nb = EXT ? rule.pooled_for(wg_ctx) : 0, wave_nb = EXT ? rule.pooled_for(wave_last + 1) : 0;
    const int q_nb = EXT ? rule.pooled_for(qpos + 1) : 0;
    const int ptiles = (wg_nb + TK - 1) / TK, first_tile = wg_lo / TK;
    const int ktiles = min((rule.keep_first + TK - 1) / TK, first_tile);
    const int n_tiles = ptiles + ktiles + (wg_ctx + TK - 1) / TK - first_tile;
    auto tile_key = [&](int t) { return (t < ptiles ? t : t < ptiles + ktiles ? t - ptiles : t - ptiles - ktiles + first_tile) * TK; };
    const bool whole = a.block_size % TK == 0;
    typedef const __attribute__((address_space(4))) int* const_int_p;
    auto page_of = [&](int t) { return *(const_int_p)(uintptr_t)(table + min(tile_key(t), wg_ctx - 1) / a.block_size); };
    int page = page_of(0);
    float kr[KIT][8], vr[VIT][8];
    auto fetch = [&](int t) {
        const int key0 = tile_key(t);
        const bool pooled = EXT && t < ptiles;
        const int lim = (pooled ? wg_nb : wg_ctx) - 1;               // (keys behind it repeat the last: masked)
        const long base = (long)page * a.block_size + key0 % a.block_size - key0;
        auto cache_row = [&](int j) -> long {
            if (whole && !pooled) return base + j;
            return pooled ? rule.pooled_row(table, j) : (long)table[j / a.block_size] * a.block_size + j % a.block_size;
        };
#pragma unroll
        for (int i = 0; i < KIT; ++i) {
            const int c = i * 256 + tid, d = c % (DP / 8) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) kr[i][j] = 0.f;
            if (d < a.D) load_run<float, 8>(a.k_cache + (cache_row(min(key0 + c / (DP / 8), lim)) * G + g) * a.D + d, kr[i]);
        }
#pragma unroll
        for (int i = 0; i < VIT; ++i) {
            const int c = i * 256 + tid, d = c % (EP / 8) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) vr[i][j] = 0.f;
            if (d < a.E)
                load_run<float, 8>(a.v_cache + (cache_row(min(key0 + c / (EP / 8), lim)) * G + g) * rule.v_stride + d, vr[i]);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int i = 0; i < KIT; ++i) {
            const int c = i * 256 + tid, row = c / (DP / 8), ch = (c % (DP / 8)) ^ swizzle<DP>(row);
            bf16x8 p[3];
            split8(kr[i], p);
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(kim + k * KT + row * DP * 2 + ch * 16) = p[k];
        }
#pragma unroll
        for (int i = 0; i < VIT; ++i) {
            const int c = i * 256 + tid, row = c / (EP / 8), ch = (c % (EP / 8)) ^ swizzle<EP>(row);
            bf16x8 p[3];
            split8(vr[i], p);
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(vim + k * VT + row * EP * 2 + ch * 16) = p[k];
        }
    };
    const int i16 = lane & 15, tr_row = 4 * half + (i16 >> 2);
    const int tr_chunk = 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1);

    f32x16 acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[n][e] = 0.f;
    float m_run = NO_SINK_MAX, l_run = 0.f;
    const float slope = rule.slopes ? rule.slopes[h] : 0.f;
    fetch(0);
    for (int t = 0; t < n_tiles; ++t) {
        if (t > 0) __syncthreads();                                  // the images have been read
        stash();
        if (t + 1 < n_tiles) {
            page = page_of(t + 1);
            fetch(t + 1);
        }
        __syncthreads();
        const int k0 = tile_key(t);
        const bool pooled = EXT && t < ptiles;
        const bool live = wave_live && (pooled ? k0 < wave_nb
                                               : (k0 <= wave_last && (k0 < rule.keep_first || k0 + 32 > wave_lo)));
        if (!live) continue;                                         // (uniform per wave)
        f32x16 s_hi, s_lo;
#pragma unroll
        for (int e = 0; e < 16; ++e) { s_hi[e] = 0.f; s_lo[e] = 0.f; }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            bf16x8 kf[3];
#pragma unroll
            for (int k = 0; k < 3; ++k)
                kf[k] = *reinterpret_cast<const bf16x8*>(kim + k * KT + l32 * DP * 2 + (((2 * s + half) ^ swizzle<DP>(l32)) << 4));
            s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[2], qf[s][0], s_lo, 0, 0, 0);
            s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[s][2], s_lo, 0, 0, 0);
            s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[s][1], s_lo, 0, 0, 0);
            s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[1], qf[s][0], s_lo, 0, 0, 0);
            s_lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[s][1], s_lo, 0, 0, 0);
            s_hi = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[s][0], s_hi, 0, 0, 0);
        }
        float z[16], mt = -INFINITY;
        const bool all_seen = pooled ? k0 + 32 <= rule.pooled_for(wave_first + 1) : k0 + 31 <= wave_first && k0 >= wave_top;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int key = k0 + (e & 3) + 8 * (e >> 2) + 4 * half;
            float v = s_hi[e] + s_lo[e];
            if (EXT) v = rule.capped(v);
            if (!pooled) v -= slope * (float)(qpos - key);
            if (!all_seen) {
                const bool seen = pooled ? key < q_nb : (key <= qpos) & ((key >= q_lo) | (key < rule.keep_first));
                v = seen ? v : -INFINITY;
            }
            z[e] = v;
            mt = fmaxf(mt, v);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
        if (!__all(mt - m_run <= 4.f)) {                             // the reference moves when a row outgrows it
            const float m_new = fmaxf(m_run, mt), f = expf(m_run - m_new);
            l_run *= f;
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[n] *= f;
            m_run = m_new;
        }
        bf16x8 p[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x[j] = expf(z[8 * s + j] - m_run);
                l_run += x[j];
            }
            split8(x, p[s]);
        }
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                bf16x8 vf[3];
                const int r0 = 16 * s + tr_row, ch = 4 * n + tr_chunk;
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    vf[k] = join(read_tr(vim + k * VT + r0 * EP * 2 + ((ch ^ swizzle<EP>(r0)) << 4) + (i16 & 1) * 8),
                                 read_tr(vim + k * VT + (r0 + 8) * EP * 2 + ((ch ^ swizzle<EP>(r0 + 8)) << 4) + (i16 & 1) * 8));
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[2], p[s][0], acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[0], p[s][2], acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[1], p[s][1], acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[1], p[s][0], acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[0], p[s][1], acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[0], p[s][0], acc[n], 0, 0, 0);
            }
    }
    if (!wave_live) return;
    l_run += __shfl_xor(l_run, 32, kWave);
    float f;
    if (a.sink) {
        const float M = fmaxf(m_run, a.sink[h]);
        f = expf(m_run - M);
        f = f / (l_run * f + expf(a.sink[h] - M));
    } else {
        f = 1.f / l_run;
    }
    const long row = row0 + min(qi, qlen - 1);
    if (a.gate) f *= sigmoidf_(a.gate[row * a.gate_row + h]);
    uint32_t lost = rows_not_finite<NB>(acc, f, qok);
    float* op = a.out + (row * H + h) * a.E;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = 32 * n + 8 * r + 4 * half;
            if (qok && e < a.E && !(lost >> l32 & 1))
                *reinterpret_cast<float4*>(op + e) = make_float4(acc[n][4 * r] * f, acc[n][4 * r + 1] * f,
                                                                 acc[n][4 * r + 2] * f, acc[n][4 * r + 3] * f);
        }
    for (; lost; lost &= lost - 1) {
        const int i = __builtin_ctz(lost);
        const long r = row0 + wq0 + i;
        row_by_keys<float, EXT>(a.q + r * a.q_row + (long)h * a.q_head, a.k_cache, a.v_cache, table, a.block_size,
                                start + wq0 + i + 1, sc, slope, a.sink, a.gate ? a.gate + r * a.gate_row + h : nullptr,
                                a.out + (r * H + h) * a.E, G, g, h, a.D, a.E, rule);
    }
#endif
}

template <int DP, int EP>
int launch_f32(const PromptArgs32& a, int nseq, int max_q, hipStream_t s) {
    constexpr int lds = 3 * 32 * (DP + EP) * 2;
    static_assert(lds <= 64 * 1024);
    const dim3 grid(a.H, nseq, (max_q + 127) / 128);
    if (a.rule.temps || a.rule.softcap > 0.f || a.rule.pool > 0)
        hipLaunchKernelGGL((prompt_attention_f32_kernel<DP, EP, true>), grid, dim3(256), lds, s, a);
    else
        hipLaunchKernelGGL((prompt_attention_f32_kernel<DP, EP, false>), grid, dim3(256), lds, s, a);
    return HYB_LAUNCH_OK();
}

template <int DP, int EP>
int launch(const PromptArgs& a, int nseq, int max_q, hipStream_t s) {
    constexpr int TK = DP + EP <= 256 ? 64 : 32, lds = 2 * TK * (DP + EP) * 2;
    static_assert(lds <= 64 * 1024);
    const dim3 grid(a.H, nseq, (max_q + 127) / 128);
    if (a.rule.temps || a.rule.softcap > 0.f || a.rule.pool > 0)
        hipLaunchKernelGGL((prompt_attention_kernel<DP, EP, TK, true>), grid, dim3(256), lds, s, a);
    else
        hipLaunchKernelGGL((prompt_attention_kernel<DP, EP, TK, false>), grid, dim3(256), lds, s, a);
    return HYB_LAUNCH_OK();
}

}  // namespace

namespace hyb {

bool prompt_attention_ok(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                         const void* out, int nseq, int max_q, int D, int E, int v_stride, bool f32) {
    if (f32 && (D > 128 || E > 128)) return false;                    // (the queries' parts fill the registers)
    if (D < 8 || E < 8 || D % 8 || E % 8 || v_stride % 8 || D > 256 || E > 256 || (D > 128 && E > 128)) return false;
    if (((size_t)q | (size_t)k_cache | (size_t)v_cache | (size_t)out) % 16 || q_row % 8 || q_head % 8) return false;
    return nseq <= 65535 && (max_q + 127) / 128 <= 65535;             // (the grid)
}

int prompt_attention(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                     const void* block_tables, int max_blocks, int block_size, const void* cu_q,
                     const void* positions, const void* sink, const void* gate, long gate_row, void* out,
                     float scale, int nseq, int seq0, int max_q, int H, int G, int D, int E,
                     const KeyRule& rule, hipStream_t s) {
    const PromptArgs a{(const uint16_t*)q, q_row, q_head, (const uint16_t*)k_cache, (const uint16_t*)v_cache,
                       (const int*)block_tables, max_blocks, block_size, (const int*)cu_q, (const int*)positions,
                       (const float*)sink, (const bf16_t*)gate, gate_row, (uint16_t*)out, scale, H, G, D, E, seq0, rule};
#define PICK(DP, EP) if (D <= DP && E <= EP) return launch<DP, EP>(a, nseq, max_q, s)
    PICK(64, 64);
    PICK(64, 128);
    PICK(64, 256);
    PICK(128, 64);
    PICK(128, 128);
    PICK(128, 256);
    PICK(256, 64);
    PICK(256, 128);
#undef PICK
    return 1;
}

int prompt_attention_f32(const void* q, long q_row, long q_head, const void* k_cache, const void* v_cache,
                         const void* block_tables, int max_blocks, int block_size, const void* cu_q,
                         const void* positions, const void* sink, const void* gate, long gate_row, void* out,
                         float scale, int nseq, int seq0, int max_q, int H, int G, int D, int E,
                         const KeyRule& rule, hipStream_t s) {
    const PromptArgs32 a{(const float*)q, q_row, q_head, (const float*)k_cache, (const float*)v_cache,
                         (const int*)block_tables, max_blocks, block_size, (const int*)cu_q, (const int*)positions,
                         (const float*)sink, (const float*)gate, gate_row, (float*)out, scale, H, G, D, E, seq0, rule};
    if (D <= 64) return E <= 64 ? launch_f32<64, 64>(a, nseq, max_q, s) : launch_f32<64, 128>(a, nseq, max_q, s);
    return E <= 64 ? launch_f32<128, 64>(a, nseq, max_q, s) : launch_f32<128, 128>(a, nseq, max_q, s);
}

}  // namespace hyb
