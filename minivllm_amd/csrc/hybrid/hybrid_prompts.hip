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
// Workgroup = 4 waves x 32 consecutive queries of one (sequence, query head); keys in tiles of 32, K and V each an
// LDS image filled by direct global -> LDS loads two tiles ahead (three buffers of keys, four of values: a tile's
// values are read a tile later than its keys).  Where a page holds whole tiles (WHOLE) a tile is read through one
// buffer descriptor, where it holds runs of eight tokens a wave's rows are (rows behind the context are out of its
// range and read as zeros); other pages and pooled rows look every row up.  Heads of one KV head go to one XCD, long
// contexts start first.
//
// A wave issues in order, and a matrix instruction leaves the unit busy for 32 cycles after the 8 of its issue: what
// the softmax does in vector instructions has to stand between them.  So a tile's exponentials and the first half
// of its parts are formed between the value products of the tile BEFORE, the second half between the score products of
// the tile AFTER, a few instructions behind each product.  No maximum is formed ahead of the exponentials: they are
// taken against the last reference, and formed again where that turns out too low.  The scalar work of a tile
// (where the next lies) was a fifth of its time as expressions of the tile's number: it is kept up instead.
//
// 8 prompts of 512..1024 tokens, 16 / 8 heads of 128, sink and gate: 68 -> 59 us for the layer, 65 of which as long as a
// fill of the output ran ahead of it; one of 1024 tokens alone 46 -> 36 (a tile in 2260 cycles of a lone wave: 1024 of products,
// some 1000 of vector issue beside them; two waves on a SIMD take 1600 each).  Before that the waves formed score
// product, softmax and value product one after the other (a tile of 32 in 3350 cycles).  What is left: the clock (1.9
// GHz under this load), 6 us at the two ends of a workgroup, and the last workgroups, of which not all CUs have one.
// Two parts per weight instead of three would hold 16 bits of it.
#include "hybrid_row_by_keys.h"
#include "hybrid_chunks.h"
#include <algorithm>

using namespace hyb;

namespace {

struct PromptArgs {
    const uint16_t* q; long q_row, q_head;
    const uint16_t *k_cache, *v_cache;             // latent attention: the formed keys and values [H, formed_rows, D | E]
    const int* tables; int max_blocks, block_size;
    const int *cu_q, *positions;
    const float* sink;
    const bf16_t* gate; long gate_row;
    uint16_t* out;
    float scale;
    int H, G, D, E, seq0;
    KeyRule rule;
    // latent attention: the turned key part of a token (its cache row's last P numbers) and of the queries
    const uint16_t* q_turned; long turned_row;     // [T, H, P]
    const uint16_t* latents; int latent_row, P;    // cache rows of latent_row numbers
    long formed_rows;
    RowSpan clear;
    uint32_t page_magic;                           // key / block_size == key * page_magic >> 32 for every key there can be (0: none)
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

// tiles of 32 keys that the sequences ahead of b have (by all lanes of a wave)
__device__ __forceinline__ int formed_tiles_before(const int* cu_q, const int* positions, int b, int lane) {
    int n = 0;
    for (int i = lane; i < b; i += 64) {
        const int r = cu_q[i], len = cu_q[i + 1] - r;
        if (len > 0) n += (positions[r] + len + 31) / 32;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) n += __shfl_xor(n, o, kWave);
    return __builtin_amdgcn_readfirstlane(n);
}

// DP, EP: columns of the K and V images; RP: columns of a second key image (0: none), the shared key part of
// latent attention; PARTS: parts a weight is cut into.
// KG: groups of four waves on the same queries, each with its run of the key tiles and buffers of its own.
template <int DP, int RP, int EP, int PARTS, bool EXT, bool WHOLE, int KG>
__global__ void __launch_bounds__(256 * KG, KG > 1 || DP + RP + EP <= 256 + (RP ? 128 : 0) ? 2 : 1)
prompt_attention_kernel(PromptArgs a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    static_assert(DP % 64 == 0 && EP % 64 == 0 && RP % 64 == 0 && (PARTS == 2 || PARTS == 3) && !(RP && !WHOLE) && !(EXT && WHOLE));
    constexpr bool LAT = RP > 0;
    constexpr int TK = 32, KS = DP / 16, RS = RP / 16, NB = EP / 32;  // steps of the score product; 32-wide value blocks
    constexpr int KT = TK * DP * 2, RT = TK * RP * 2, VT = TK * EP * 2;                     // bytes of an image
    constexpr int KIT = KT / 4096, RIT = RT / 4096, VIT = VT / 4096, LOADS = KIT + RIT + VIT; // 16-byte pieces per thread
    constexpr int KSW = DP % 128 == 0 ? 16 : 8, RSW = RP % 128 == 0 ? 16 : 8, VSW = EP % 128 == 0 ? 16 : 8; // chunks a swizzle permutes
    constexpr int R_AT = 3 * KT, V_AT = 3 * (KT + RT);                // three buffers of keys, four of values
    constexpr int GROUP = V_AT + 4 * VT;                              // a group's buffers
    extern __shared__ __attribute__((aligned(256))) char shared[];
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    char* const smem = shared + kg * GROUP;

    const int H = a.H, hx = blockIdx.x;
    const int h = H % 8 == 0 ? (hx & 7) * (H >> 3) + (hx >> 3) : hx;
    const int b = blockIdx.y + a.seq0, tile_q0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * 128;
    if (a.clear.end > 0) clear_rest(a.out, a.cu_q + a.seq0, a.clear, h, H, a.E);
    const int row0 = __builtin_amdgcn_readfirstlane(a.cu_q[b]), qlen = __builtin_amdgcn_readfirstlane(a.cu_q[b + 1]) - row0;
    if (tile_q0 >= qlen) return;
    const int start = __builtin_amdgcn_readfirstlane(a.positions[row0]), G = a.G, g = h / (H / G);
    const int* table = a.tables + (long)b * a.max_blocks;
    const int tid = threadIdx.x & 255, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int wq0 = tile_q0 + wave * 32, qi = wq0 + l32;
    const bool qok = qi < qlen, wave_live = wq0 < qlen;
    const int qpos = start + qi;
    bf16x8 qf[KS + RS];
    {
        const uint16_t* qp = a.q + (long)(row0 + min(qi, qlen - 1)) * a.q_row + (long)h * a.q_head;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 16 * s + 8 * half;
            uint4 raw = make_uint4(0, 0, 0, 0);                     // columns from D on: zeros
            if (d < a.D) raw = *reinterpret_cast<const uint4*>(qp + d);
            qf[s] = __builtin_bit_cast(bf16x8, raw);
        }
        if constexpr (LAT) {
            const uint16_t* rp = a.q_turned + (long)(row0 + min(qi, qlen - 1)) * a.turned_row + (long)h * a.P;
#pragma unroll
            for (int s = 0; s < RS; ++s) {
                const int d = 16 * s + 8 * half;
                uint4 raw = make_uint4(0, 0, 0, 0);
                if (d < a.P) raw = *reinterpret_cast<const uint4*>(rp + d);
                qf[KS + s] = __builtin_bit_cast(bf16x8, raw);
            }
        }
    }

    // (asked for here: at the end they would be waited for)
    const float gate = a.gate ? ld(a.gate + (long)(row0 + min(qi, qlen - 1)) * a.gate_row + h) : 0.f;
    const float sink = a.sink ? a.sink[h] * LOG2E : 0.f;

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
    // this group's: one run of them, of up to `per`
    const int per = (n_tiles + KG - 1) / KG, t_begin = kg * per, t_end = min(n_tiles, t_begin + per);
    auto tile_key = [&](int t) { return (t < ptiles ? t : t < ptiles + ktiles ? t - ptiles : t - ptiles - ktiles + first_tile) * TK; };

    // ---- staging: slot c of an image (row c / chunks per row) receives the chunk that the swizzle puts
    // there; chunks behind a row's end repeat chunk 0 (their queries are zeros, their columns not stored).
    // A wave's piece of an image is a whole number of rows: they lie in one page where a page holds whole runs of
    // eight tokens, and a descriptor reads them (rows behind the context are out of its range and read as zeros);
    // where it holds whole tiles (WHOLE), one descriptor does for all pieces.
    const int cols_k = a.D, cols_v = a.E;
    const int krow = G * a.D * 2, vrow = G * rule.v_stride * 2;     // bytes from one token's row to the next
    const int rrow = LAT ? a.latent_row * 2 : 0;
    int k_off[KIT], v_off[VIT], r_off[RIT > 0 ? RIT : 1];
    auto slot_of = [&](auto cols, int i, int n, int row_bytes) {    // lane's source offset from the tile's first row
        constexpr int C = decltype(cols)::value;
        const int c = i * 256 + tid, row = c / (C / 8);
        int ch = (c % (C / 8)) ^ swizzle<C>(row);
        if (ch * 8 >= n) ch = 0;
        return row * row_bytes + ch * 16;
    };
#pragma unroll
    for (int i = 0; i < KIT; ++i) k_off[i] = slot_of(std::integral_constant<int, DP>{}, i, cols_k, LAT ? a.D * 2 : krow);
#pragma unroll
    for (int i = 0; i < VIT; ++i) v_off[i] = slot_of(std::integral_constant<int, EP>{}, i, cols_v, LAT ? a.E * 2 : vrow);
    if constexpr (LAT) {
#pragma unroll
        for (int i = 0; i < RIT; ++i) r_off[i] = slot_of(std::integral_constant<int, RP>{}, i, a.P, rrow);
    }
    const bool runs = WHOLE || (a.page_magic && a.block_size % 8 == 0);
    // (a division is some 40 instructions of a tile's 400)
    auto page_index = [&](int key) { return (int)__umulhi((uint32_t)key, a.page_magic); };
    auto in_page = [&](int key) { return key - page_index(key) * a.block_size; };
    // bytes of a row inside a page (page_magic: a page's bytes fit 31 bits)
    auto place = [&](int page, int in, int row_bytes) {
        return (uint64_t)(uint32_t)page * (uint32_t)(a.block_size * row_bytes) + (uint32_t)(in * row_bytes);
    };
    const char* k_head = reinterpret_cast<const char*>(a.k_cache) + g * a.D * 2;
    const char* v_head = reinterpret_cast<const char*>(a.v_cache) + (long)g * rule.v_stride * 2;
    typedef const __attribute__((address_space(4))) int* const_int_p;
    auto page_of = [&](int key) {                        // through the scalar unit (the table is read-only here)
        return *(const_int_p)(uintptr_t)(table + page_index(min(key, wg_ctx - 1)));
    };
    const int last_page = page_index(wg_ctx - 1);
    // LAT: rows of the formed keys and values ahead of this sequence's
    long formed0 = 0;
    if constexpr (LAT) {
        formed0 = (long)formed_tiles_before(a.cu_q, a.positions, b, lane) * 32;
        if (formed0 + (wg_ctx + 31) / 32 * 32 > a.formed_rows) return;      // (a longest context given too short: nothing there)
    }
    constexpr int RPK = 512 / (LAT ? RP : DP), RPV = 512 / EP;   // rows of a piece that is looked up by page
    constexpr int PIT = LAT ? RIT : KIT;
    // the tile to be staged next, kept up from tile to tile (as expressions of its number they were a fifth of the
    // loop's time): its number, its first key, its LDS buffers; WHOLE: where it lies, tiles until the page or the run ends
    int ahead = t_begin, s_key = 0, s_kbuf = 0, s_vbuf = 0, s_run = 0;
    const char *s_k = nullptr, *s_v = nullptr, *s_r = nullptr;
    int kpage[PIT], vpage[VIT];                          // requested ahead
    auto locate = [&]() {                                // WHOLE: tile `ahead` begins a page, a run of tiles or the work
        const int page = *(const_int_p)(uintptr_t)(table + min(page_index(s_key), last_page)), in = in_page(s_key);
        s_run = (a.block_size - in) / TK;
        if (ahead < ktiles) s_run = min(s_run, ktiles - ahead);
        if constexpr (LAT) {
            s_r = reinterpret_cast<const char*>(a.latents) + place(page, in, rrow) + rrow - a.P * 2;
        } else {
            s_k = k_head + place(page, in, krow);
            s_v = v_head + place(page, in, vrow);
        }
    };
    auto fetch_pages = [&]() {
        if constexpr (!WHOLE) {
            if (!runs || (EXT && ahead < ptiles)) return;
#pragma unroll
            for (int i = 0; i < PIT; ++i) kpage[i] = page_of(s_key + (4 * i + wave) * RPK);
#pragma unroll
            for (int i = 0; i < VIT; ++i) vpage[i] = page_of(s_key + (4 * i + wave) * RPV);
        }
    };
    auto next_tile = [&]() {
        ++ahead;
        s_kbuf = s_kbuf == 2 * KT ? 0 : s_kbuf + KT;
        s_vbuf = s_vbuf == 3 * VT ? 0 : s_vbuf + VT;
        if constexpr (WHOLE) {
            s_key += TK;
            if constexpr (LAT) {
                s_r += TK * rrow;
                s_k += TK * a.D * 2;
                s_v += TK * a.E * 2;
            } else {
                s_k += TK * krow;
                s_v += TK * vrow;
            }
            if (--s_run == 0) {
                const int jump = tile_key(ahead) - s_key;
                s_key += jump;
                if constexpr (LAT) {
                    s_k += (long)jump * a.D * 2;
                    s_v += (long)jump * a.E * 2;
                }
                locate();
            }
        } else {
            s_key = tile_key(ahead);
            fetch_pages();
        }
    };
    // rows of a tile: `first` lies `rb` rows into it, `left` rows from the tile's start are there
    auto source = [](const char* first, int rb, int left, int row_bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(first - (long)rb * row_bytes), 0, left * row_bytes, 0x00020000);
    };
    auto to_lds = [](__amdgpu_buffer_rsrc_t r, char* dst, int off) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
    };
    auto stage = [&]() {
        const int key0 = s_key;
        int left = min(TK, wg_ctx - key0);                           // (behind the last tile: zeros are staged)
        asm volatile("" : "+s"(left));                               // (min and max in one are a vector instruction)
        left = max(left, 0);
        const bool pooled = EXT && ahead < ptiles;
        char* kd = smem + s_kbuf + wave * 1024;
        char* vd = smem + V_AT + s_vbuf + wave * 1024;
        if constexpr (WHOLE) {
            const int rows = !LAT ? left : left > 0 ? TK : 0;        // (formed rows fill their last tile)
            const auto kr = source(s_k, 0, rows, LAT ? a.D * 2 : krow), vr = source(s_v, 0, rows, LAT ? a.E * 2 : vrow);
#pragma unroll
            for (int i = 0; i < KIT; ++i) to_lds(kr, kd + i * 4096, k_off[i]);
#pragma unroll
            for (int i = 0; i < VIT; ++i) to_lds(vr, vd + i * 4096, v_off[i]);
            if constexpr (LAT) {
                const auto rr = source(s_r, 0, left, rrow);
                char* rd = smem + R_AT + s_kbuf / KT * RT + wave * 1024;
#pragma unroll
                for (int i = 0; i < RIT; ++i) to_lds(rr, rd + i * 4096, r_off[i]);
            }
        } else if (runs && !pooled) {
#pragma unroll
            for (int i = 0; i < KIT; ++i) {
                const int rb = (4 * i + wave) * RPK;
                to_lds(source(k_head + place(kpage[i], in_page(key0 + rb), krow), rb, left, krow), kd + i * 4096, k_off[i]);
            }
#pragma unroll
            for (int i = 0; i < VIT; ++i) {
                const int rb = (4 * i + wave) * RPV;
                to_lds(source(v_head + place(vpage[i], in_page(key0 + rb), vrow), rb, left, vrow), vd + i * 4096, v_off[i]);
            }
        } else {
            const int lim = (pooled ? wg_nb : wg_ctx) - 1;
            auto cache_row = [&](int j) -> long {
                return pooled ? rule.pooled_row(table, j) : (long)table[j / a.block_size] * a.block_size + j % a.block_size;
            };
            int me = tid;
            asm volatile("" : "+v"(me));                             // (worked out ahead of the loop it costs registers)
#pragma unroll
            for (int i = 0; i < KIT; ++i) {
                const int row = (i * 256 + me) / (DP / 8);
                const char* src = reinterpret_cast<const char*>(a.k_cache) +
                                  (cache_row(min(key0 + row, lim)) * G + g) * a.D * 2 + (k_off[i] - row * krow);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)(kd + i * 4096), 16, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < VIT; ++i) {
                const int row = (i * 256 + me) / (EP / 8);
                const char* src = reinterpret_cast<const char*>(a.v_cache) +
                                  (cache_row(min(key0 + row, lim)) * G + g) * (long)rule.v_stride * 2 + (v_off[i] - row * vrow);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)(vd + i * 4096), 16, 0, 0);
            }
        }
    };
    // all but the last tile's requests have landed, for all waves
    auto tile_done = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(LOADS) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- LDS addresses of this lane's fragments inside a buffer
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)smem;
    uint32_t k_addr[KSW / 2], r_addr[LAT ? RSW / 2 : 1]; // row l32, chunk 2 s + half: distinct for s < KSW / 2
#pragma unroll
    for (int s = 0; s < KSW / 2; ++s) k_addr[s] = lds0 + l32 * (DP * 2) + (((2 * s + half) ^ swizzle<DP>(l32)) << 4);
    if constexpr (LAT) {
#pragma unroll
        for (int s = 0; s < RSW / 2; ++s) r_addr[s] = lds0 + R_AT + l32 * (RP * 2) + (((2 * s + half) ^ swizzle<RP>(l32)) << 4);
    }
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
            v_addr[n][hi] = lds0 + V_AT + row * (EP * 2) + (((4 * n + tr_chunk) ^ swizzle<EP>(row)) << 4) + (i16 & 1) * 8;
        }

    f32x16 acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[n][e] = 0.f;
    float m_run = NO_SINK_MAX, l_run = 0.f;         // in log2 units of the scores
    const float slope = rule.slopes ? rule.slopes[h] * LOG2E : 0.f;
    // scores are scaled inside the exponential's argument where nothing but a positive factor is between
    const float sc_all = (EXT ? rule.head_scale(a.scale, h) : a.scale) * (EXT ? 1.f : LOG2E);
    const bool scaled_first = EXT || rule.slopes || !(sc_all > 0.f);
    const float sc = scaled_first ? 1.f : sc_all;

    // ---- a tile's weights: the exponentials of both halves of its keys (e < 8, e >= 8 of a lane's 16) and the parts
    // of the first are formed between the value products of the tile before, the parts of the second between the
    // score products of the tile after
    uint32_t pw[PARTS][2][4];                       // [part][half][pair]: the operand of the value products
    float late[8];                                  // weights of the second half, not yet in parts
    auto stay = [](auto& x, auto& y) { asm volatile("" : "+v"(x), "+v"(y)); };     // (the compiler would sink it all to its use)
    constexpr int SPLITS = 4 * (PARTS - 1);         // steps in which a half's weights are cut
    auto cut = [&](auto ic, float* w, int s) {      // step i: pair i / (PARTS - 1)
        constexpr int i = decltype(ic)::value, j = i / (PARTS - 1), k = i % (PARTS - 1);
        float x = w[2 * j], y = w[2 * j + 1];
        if constexpr (PARTS == 3) {                 // the upper halves of what the parts before left over
            if constexpr (k == 0) pw[0][s][j] = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302);
            x -= __uint_as_float(__float_as_uint(x) & 0xffff0000u);
            y -= __uint_as_float(__float_as_uint(y) & 0xffff0000u);
            pw[k + 1][s][j] = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302);
            w[2 * j] = x;
            w[2 * j + 1] = y;
            stay(pw[0][s][j], pw[k + 1][s][j]);
        } else {                                    // rounded parts
            pw[0][s][j] = rounded(x, y);
            rest(pw[0][s][j], x, y);
            pw[1][s][j] = rounded(x, y);
            stay(pw[0][s][j], pw[1][s][j]);
        }
    };
    auto part = [&](int k, int s) { return __builtin_bit_cast(bf16x8, make_uint4(pw[k][s][0], pw[k][s][1], pw[k][s][2], pw[k][s][3])); };
    // step i of n takes its share of the `of` pieces of work
    auto share = [](auto ic, auto nc, auto ofc, auto&& f) {
        constexpr int i = decltype(ic)::value, n = decltype(nc)::value, of = decltype(ofc)::value;
        static_for<i * of / n, (i + 1) * of / n>(f);
    };
    // value products of the tile whose values lie at va, half s of its keys after the other; between them work(step)
    // (inline asm: through the builtin the compiler would wait for the stage's loads in flight ahead of the first
    // read; a pair of blocks is requested ahead)
    constexpr int PAIRS = NB / 2, HALF = NB * PARTS, STEPS = 2 * HALF;
    s16x4 vlo[2][2], vhi[2][2];
    uint32_t va[NA][2];
    auto read_v = [&](auto gc) {                    // group g: half g / PAIRS, blocks 2 (g % PAIRS) ..
        constexpr int gi = decltype(gc)::value, s = gi / PAIRS;
        static_for<0, 2>([&](auto dc) {
            constexpr int d = decltype(dc)::value, n = 2 * (gi % PAIRS) + d;
            constexpr int off = (n / NA) * NA * 64 + s * 16 * EP * 2;
            const uint32_t a0 = va[n % NA][0], a1 = va[n % NA][1];
            s16x4 x, y;
            asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(x) : "v"(a0), "n"(off));
            asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(y) : "v"(a1), "n"(off));
            vlo[gi & 1][d] = x;
            vhi[gi & 1][d] = y;
        });
    };
    auto open_values = [&](int buf) {               // (ahead of value_products, as soon as the addresses are free)
#pragma unroll
        for (int n = 0; n < NA; ++n) {
            va[n][0] = v_addr[n][0] + buf;
            va[n][1] = v_addr[n][1] + buf;
        }
        read_v(std::integral_constant<int, 0>{});
    };
    auto value_products = [&](auto&& work) {
        static_for<0, 2 * PAIRS>([&](auto gc) {
            constexpr int gi = decltype(gc)::value, s = gi / PAIRS, n0 = 2 * (gi % PAIRS);
            if constexpr (gi + 1 < 2 * PAIRS) read_v(std::integral_constant<int, gi + 1>{});
            s16x4 x0 = vlo[gi & 1][0], y0 = vhi[gi & 1][0], x1 = vlo[gi & 1][1], y1 = vhi[gi & 1][1];
            asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1) : "n"(gi + 1 < 2 * PAIRS ? 4 : 0));
            const bf16x8 v0 = join(x0, y0), v1 = join(x1, y1);
            static_for<0, 2 * PARTS>([&](auto ic) {
                constexpr int i = decltype(ic)::value, k = i / 2, d = i % 2;
                acc[n0 + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(d ? v1 : v0, part(k, s), acc[n0 + d], 0, 0, 0);
                work(std::integral_constant<int, gi * 2 * PARTS + i>{});
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };

    // (behind the last tile more are requested, of keys that are not there: the pages stay those of the table)
    if constexpr (LAT) {
        const long at = h * a.formed_rows + formed0 + tile_key(t_begin);
        s_k = reinterpret_cast<const char*>(a.k_cache) + at * a.D * 2;
        s_v = reinterpret_cast<const char*>(a.v_cache) + at * a.E * 2;
    }
    s_key = tile_key(t_begin);
    if constexpr (WHOLE) locate(); else fetch_pages();
    stage();
    next_tile();
    stage();
    next_tile();
    tile_done();
    // the tiles this wave has a share in (uniform): of the pooled ones the first, then those with kept first tokens,
    // then from the first its window reaches to that of its last query
    const int p_end = EXT ? (wave_nb + TK - 1) / TK : 0, keep_end = ptiles + (rule.keep_first + TK - 1) / TK;
    const int win_begin = ptiles + ktiles + wave_lo / TK - first_tile, win_end = ptiles + ktiles + wave_last / TK - first_tile;
    auto live_tile = [&](int t) -> int {
        return wave_live && (EXT && t < ptiles ? t < p_end : (t < keep_end || t >= win_begin) && t <= win_end);
    };
    // buffers of the current tile; that of the tile whose value products are still to come (< 0: none)
    int kbuf = 0, vbuf = 0, open = -1, t = t_begin;
    auto turn = [&]() {
        tile_done();
        kbuf = kbuf == 2 * KT ? 0 : kbuf + KT;
        vbuf = vbuf == 3 * VT ? 0 : vbuf + VT;
        ++t;
    };
    while (true) {
        for (; t < t_end && !live_tile(t); turn()) {
            stage();
            next_tile();
        }
        if (t >= t_end) break;
#pragma unroll
        for (int k = 0; k < PARTS; ++k)
#pragma unroll
            for (int i = 0; i < 8; ++i) pw[k][i / 4][i % 4] = 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i) late[i] = 0.f;
        open = -1;
        do {
            const int k0 = tile_key(t);
            const bool pooled = EXT && t < ptiles;
            if constexpr (!WHOLE) stage();
            // (K reads: inline asm, as through the builtin the compiler would wait for the stage's loads in flight ahead
            // of the first; KA of them are in flight)
            constexpr int N = KS + RS, KA = N < 8 ? N : 8;
            s16x8 kf[N];
            uint32_t ka[KSW / 2], ra[LAT ? RSW / 2 : 1];
            auto read_k = [&](auto ic) {
                constexpr int i = decltype(ic)::value, j = i < KS ? i : i - KS;
                constexpr int off = i < KS ? (j / (KSW / 2)) * (KSW * 16) : (j / (RSW / 2)) * (RSW * 16);
                const uint32_t a0 = i < KS ? ka[j % (KSW / 2)] : ra[LAT ? j % (RSW / 2) : 0];
                s16x8 x;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x) : "v"(a0), "n"(off));
                kf[i] = x;
            };
            {
#pragma unroll
                for (int s = 0; s < KSW / 2; ++s) ka[s] = k_addr[s] + kbuf;
                if constexpr (LAT) {
#pragma unroll
                    for (int s = 0; s < RSW / 2; ++s) ra[s] = r_addr[s] + kbuf / KT * RT;
                }
                static_for<0, KA>(read_k);
            }
            if constexpr (WHOLE) stage();                // (while the first reads are on their way)
            f32x16 s_acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) s_acc[e] = 0.f;
            static_for<0, N>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i + KA < N) read_k(std::integral_constant<int, i + KA>{});
                constexpr int left = N - 1 - i < KA ? N - 1 - i : KA;        // reads still in flight
                s16x8 x = kf[i];
                asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(x) : "n"(left));
                s_acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), qf[i], s_acc, 0, 0, 0);
                share(ic, std::integral_constant<int, N>{}, std::integral_constant<int, SPLITS>{},
                      [&](auto jc) { cut(jc, late, 1); });
                __builtin_amdgcn_sched_barrier(0);
            });
            // (nothing open: the weights are zeros, of any values that are there)
            open_values(open < 0 ? vbuf : open);
            __builtin_amdgcn_sched_barrier(0);
            // lane: query qi, keys k0 + (e & 3) + 8 (e >> 2) + 4 half
            if (scaled_first) {
#pragma unroll
                for (int e = 0; e < 16; ++e) s_acc[e] = EXT ? rule.capped(s_acc[e] * sc_all) * LOG2E : s_acc[e] * sc_all;
                if (rule.slopes && !pooled) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) s_acc[e] -= slope * (float)(qpos - (k0 + (e & 3) + 8 * (e >> 2) + 4 * half));
                }
            }
            const bool all_seen = pooled ? k0 + TK <= rule.pooled_for(wave_first + 1)
                                         : k0 + TK - 1 <= wave_first && k0 >= wave_top;
            if (!all_seen) {                                             // (one uniform branch, not one per score)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = k0 + (e & 3) + 8 * (e >> 2) + 4 * half;
                    const bool seen = pooled ? key < q_nb : (key <= qpos) & ((key >= q_lo) | (key < rule.keep_first));
                    s_acc[e] = seen ? s_acc[e] : -INFINITY;
                }
            }
            float w[16], l_new = 0.f, top = 0.f, f = 1.f;
            bool grows = false;
            const float neg = -m_run;
            value_products([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i < HALF) {
                    share(ic, std::integral_constant<int, HALF>{}, std::integral_constant<int, 8>{}, [&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        w[2 * j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[2 * j], sc, neg));
                        w[2 * j + 1] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[2 * j + 1], sc, neg));
                        stay(w[2 * j], w[2 * j + 1]);
                        l_new += w[2 * j];
                        l_new += w[2 * j + 1];
                        top = fmaxf(top, fmaxf(w[2 * j], w[2 * j + 1]));
                        stay(l_new, top);
                    });
                    // The reference of the exponentials only moves when some row outgrows it by RESCALE (a tile's weights
                    // are NaN or infinite or too large, so is the first one's): they are formed again.  The sums follow
                    // once the products of the tile before are in them.
                    if constexpr (i == HALF - 1) {
                        grows = !__all(top <= 64.f && l_new == l_new);       // (2^RESCALE)
                        if (grows) {
                            float mt = s_acc[0];
#pragma unroll
                            for (int e = 1; e < 16; ++e) mt = fmaxf(mt, s_acc[e]);
                            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
                            const float m_new = fmaxf(m_run, fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * sc);
                            f = __builtin_amdgcn_exp2f(m_run - m_new);
                            l_run *= f;
                            m_run = m_new;
                            l_new = 0.f;
#pragma unroll
                            for (int e = 0; e < 16; ++e) {
                                w[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[e], sc, -m_new));
                                l_new += w[e];
                            }
                        }
                        l_run += l_new;
                    }
                }
                if constexpr (i >= HALF)
                    share(std::integral_constant<int, i - HALF>{}, std::integral_constant<int, HALF>{},
                          std::integral_constant<int, SPLITS>{}, [&](auto jc) { cut(jc, w, 0); });
            });
#pragma unroll
            for (int i = 0; i < 8; ++i) late[i] = w[8 + i];
            if constexpr (WHOLE) next_tile();
            if (grows) {
#pragma unroll
                for (int n = 0; n < NB; ++n) acc[n] *= f;
            }
            open = vbuf;
            if constexpr (!WHOLE) next_tile();
            turn();
        } while (t < t_end && live_tile(t));
        // tiles that are not this wave's may follow, and its values' buffer be used again: the products now
        static_for<0, SPLITS>([&](auto jc) { cut(jc, late, 1); });
        open_values(open);
        value_products([](auto) {});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // (the requests behind the last tile)
    l_run += __shfl_xor(l_run, 32, kWave);
    if constexpr (KG > 1) {                                          // the other groups' sums through LDS to the first
        constexpr int PART = (NB * 16 + 2) * 64;                     // floats of a wave
        static_assert((KG - 1) * 4 * PART * 4 <= KG * GROUP);
        for (int i = t_end - t_begin < 0 ? 0 : t_end - t_begin; i < per; ++i) __builtin_amdgcn_s_barrier();     // (turns of a run that is shorter)
        __syncthreads();
        float* x = reinterpret_cast<float*>(shared) + lane;
        if (kg > 0 && wave_live) {
            float* o = x + ((kg - 1) * 4 + wave) * PART;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[(n * 16 + e) * 64] = acc[n][e];
            o[NB * 16 * 64] = m_run;
            o[(NB * 16 + 1) * 64] = l_run;
        }
        __syncthreads();
        if (kg > 0) return;
        if (wave_live)
            for (int i = 0; i < KG - 1; ++i) {
                const float* o = x + (i * 4 + wave) * PART;
                const float m2 = o[NB * 16 * 64], M = fmaxf(m_run, m2);
                const float f1 = __builtin_amdgcn_exp2f(m_run - M), f2 = __builtin_amdgcn_exp2f(m2 - M);
                l_run = l_run * f1 + o[(NB * 16 + 1) * 64] * f2;
                m_run = M;
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[n][e] = acc[n][e] * f1 + o[(n * 16 + e) * 64] * f2;
            }
    }
    if (!wave_live) return;
    const PromptArgs z = arguments_anew<PromptArgs>();
    float f;
    if (z.sink) {
        const float M = fmaxf(m_run, sink);
        f = __builtin_amdgcn_exp2f(m_run - M);
        f = f / (l_run * f + __builtin_amdgcn_exp2f(sink - M));
    } else {
        f = 1.f / l_run;
    }
    const long row = row0 + min(qi, qlen - 1);
    if (z.gate) f *= sigmoidf_(gate);
    uint32_t lost = rows_not_finite<NB>(acc, f, qok);
    // both halves of the wave hold every second run of four columns of a row: swapped so that a
    // lane stores eight neighbouring ones
    uint16_t* op = z.out + (row * z.H + h) * z.E;
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                w[k] = (uint32_t)bf16_bits(acc[n][4 * r + 2 * k] * f) |
                       ((uint32_t)bf16_bits(acc[n][4 * r + 2 * k + 1] * f) << 16);
            const auto r0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
            const auto r1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
            const int e = 32 * n + 8 * r + 8 * half;
            if (qok && e < z.E && !(lost >> l32 & 1)) *reinterpret_cast<uint4*>(op + e) = make_uint4(r0[0], r1[0], r0[1], r1[1]);
        }
    for (; lost; lost &= lost - 1) {
        const int i = __builtin_ctz(lost);
        const long r = row0 + wq0 + i;
        const float scale = EXT ? z.rule.head_scale(z.scale, h) : z.scale;
        if constexpr (LAT) {
            const long at = h * z.formed_rows + formed0;
            row_by_keys<bf16_t, false>((const bf16_t*)z.q + r * z.q_row + (long)h * z.q_head, (const bf16_t*)z.k_cache + at * z.D,
                                       (const bf16_t*)z.v_cache + at * z.E, nullptr, 0, start + wq0 + i + 1, scale, 0.f,
                                       z.sink, nullptr, (bf16_t*)z.out + (r * z.H + h) * z.E, 1, 0, h, z.D, z.E, z.rule,
                                       LatentTail{(const bf16_t*)z.q_turned + r * z.turned_row + (long)h * z.P,
                                                  (const bf16_t*)z.latents, z.latent_row, z.P, table, z.block_size});
        } else {
            row_by_keys<bf16_t, EXT>((const bf16_t*)z.q + r * z.q_row + (long)h * z.q_head, (const bf16_t*)z.k_cache,
                                     (const bf16_t*)z.v_cache, table, z.block_size, start + wq0 + i + 1, scale,
                                     z.rule.slopes ? z.rule.slopes[h] : 0.f, z.sink,
                                     z.gate ? z.gate + r * z.gate_row + h : nullptr, (bf16_t*)z.out + (r * z.H + h) * z.E, z.G, g,
                                     h, z.D, z.E, z.rule);
        }
    }
#endif
}

// The same over float caches: keys, values, queries and weights all fp32, each cut into three parts; a
// product is the sum of the six largest products of parts.  Key tiles of 32; K and V are
// in registers a tile ahead and go to LDS as images of their parts, one buffer.  Exponentials are expf of
// the difference, as in the general kernel.
// Workgroup = KG groups of QW waves on 32 QW queries: group x takes tiles x, x + KG, .., each in images of its own, and the
// groups' sums meet in LDS at the end.  A tile is a chain of cutting, barrier, products, softmax, products, which a lone wave on
// a SIMD walks in 2.6 us, products 0.6 of them: a second wave fills it, and where there are fewer workgroups than CUs
// the chain itself is shorter.  (Chains of sums are shorter too: 1.3e-7 from 64 bits instead of 1.9e-7.)
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
    RowSpan clear;
};

template <int DP, int EP, bool EXT, int QW, int KG>
__global__ void __launch_bounds__(64 * QW * KG, 1)
prompt_attention_f32_kernel(PromptArgs32 a) {
#ifdef __HIP_DEVICE_COMPILE__       // (the host pass only needs the launch stub)
    constexpr int TK = 32, KS = DP / 16, NB = EP / 32;
    constexpr int KT = TK * DP * 2, VT = TK * EP * 2;                         // bytes of a part's image
    constexpr int GT = 64 * QW;                                               // threads of a group
    constexpr int KIT = TK * DP / 8 / GT, VIT = TK * EP / 8 / GT;             // runs of eight per thread
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
    char *kim = smem + kg * 3 * (KT + VT), *vim = kim + 3 * KT;

    const int H = a.H, hx = blockIdx.x;
    const int h = H % 8 == 0 ? (hx & 7) * (H >> 3) + (hx >> 3) : hx;
    const int b = blockIdx.y + a.seq0, tile_q0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * (32 * QW);
    if (a.clear.end > 0) clear_rest(a.out, a.cu_q + a.seq0, a.clear, h, H, a.E);
    const int row0 = a.cu_q[b], qlen = a.cu_q[b + 1] - row0;
    if (tile_q0 >= qlen) return;
    const int start = a.positions[row0], G = a.G, g = h / (H / G);
    const int* table = a.tables + (long)b * a.max_blocks;
    const int tid = threadIdx.x - kg * GT, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
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
    const int wg_ctx = start + min(qlen, tile_q0 + 32 * QW);
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
    int page = kg < n_tiles ? page_of(kg) : 0;
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
            const int c = i * GT + tid, d = c % (DP / 8) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) kr[i][j] = 0.f;
            if (d < a.D) load_run<float, 8>(a.k_cache + (cache_row(min(key0 + c / (DP / 8), lim)) * G + g) * a.D + d, kr[i]);
        }
#pragma unroll
        for (int i = 0; i < VIT; ++i) {
            const int c = i * GT + tid, d = c % (EP / 8) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) vr[i][j] = 0.f;
            if (d < a.E)
                load_run<float, 8>(a.v_cache + (cache_row(min(key0 + c / (EP / 8), lim)) * G + g) * rule.v_stride + d, vr[i]);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int i = 0; i < KIT; ++i) {
            const int c = i * GT + tid, row = c / (DP / 8), ch = (c % (DP / 8)) ^ swizzle<DP>(row);
            bf16x8 p[3];
            split8(kr[i], p);
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(kim + k * KT + row * DP * 2 + ch * 16) = p[k];
        }
#pragma unroll
        for (int i = 0; i < VIT; ++i) {
            const int c = i * GT + tid, row = c / (EP / 8), ch = (c % (EP / 8)) ^ swizzle<EP>(row);
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
    if (kg < n_tiles) fetch(kg);
    for (int t0 = 0; t0 < n_tiles; t0 += KG) {                       // (all groups meet at the barriers)
        const int t = t0 + kg;
        if (t0 > 0) __syncthreads();                                 // the images have been read
        if (t < n_tiles) stash();
        if (t + KG < n_tiles) {
            page = page_of(t + KG);
            fetch(t + KG);
        }
        __syncthreads();
        if (t >= n_tiles) continue;
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
    l_run += __shfl_xor(l_run, 32, kWave);
    if constexpr (KG > 1) {                                          // the other groups' parts through LDS to the first
        constexpr int PART = (NB * 16 + 2) * 64;                     // floats of a wave
        float* part = reinterpret_cast<float*>(smem);
        __syncthreads();                                             // the images have been read
        if (kg > 0 && wave_live) {
            float* o = part + ((kg - 1) * QW + wave) * PART + lane;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[(n * 16 + e) * 64] = acc[n][e];
            o[NB * 16 * 64] = m_run;
            o[(NB * 16 + 1) * 64] = l_run;
        }
        __syncthreads();
        if (kg > 0) return;
        if (wave_live)
            for (int x = 0; x < KG - 1; ++x) {
                const float* o = part + (x * QW + wave) * PART + lane;
                const float m2 = o[NB * 16 * 64], M = fmaxf(m_run, m2), f1 = expf(m_run - M), f2 = expf(m2 - M);
                l_run = l_run * f1 + o[(NB * 16 + 1) * 64] * f2;
                m_run = M;
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[n][e] = acc[n][e] * f1 + o[(n * 16 + e) * 64] * f2;
            }
    }
    if (!wave_live) return;
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

// floor(2^32 / n) + 1 is off by less than n / 2^32 of itself: exact below 2^32 / n
uint32_t page_magic(int n, int max_blocks, long row_bytes) {
    return n > 1 && (long)max_blocks * n * n < (1L << 32) && n * row_bytes < (1L << 31) ? (uint32_t)((1ull << 32) / n + 1) : 0;
}

template <int DP, int EP, bool EXT, int QW, int KG>
int launch_f32_as(const PromptArgs32& a, int nseq, int max_q, hipStream_t s) {
    constexpr int images = KG * 3 * 32 * (DP + EP) * 2, parts = (KG - 1) * QW * (EP / 2 + 2) * 256;
    constexpr int lds = images > parts ? images : parts;
    static_assert(lds <= 160 * 1024 && DP >= 32 * QW / 4 && EP >= 32 * QW / 4);
    auto* kernel = prompt_attention_f32_kernel<DP, EP, EXT, QW, KG>;
    if constexpr (lds > 64 * 1024) {
        static const hipError_t once = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (once != hipSuccess) return 2;
    }
    hipLaunchKernelGGL(kernel, dim3(a.H, nseq, (max_q + 32 * QW - 1) / (32 * QW)), dim3(64 * QW * KG), lds, s, a);
    return HYB_LAUNCH_OK();
}

// The most keys that a workgroup walks: contexts fit their pages, and queries see no more than a window or a chunk has.
long longest_walk(int max_blocks, int block_size, const KeyRule& rule) {
    long n = (long)max_blocks * block_size;
    if (rule.window > 0) n = std::min(n, (long)rule.window + rule.keep_first + 127);
    if (rule.chunk > 0) n = std::min(n, (long)rule.chunk + 127);
    return n;
}

// Which form takes a launch of float rows, F32_QUERIES * 10 + F32_GROUPS: 41, one group of four waves; 42, two groups; 22 and 24,
// two and four groups of two waves on 64 queries.  rows: of the step, 0 if that is not known.
//
// More groups shorten the chain of a workgroup and cost their meeting, LDS and, with 24 and 42, the second workgroup of a CU;
// they pay for long walks and where there is at most a workgroup for every CU.  us, 41 / 42 / 24 / 22, 8 heads, prompts of
// equal length, 64 + 64, 128 + 64 and (41 / 42 / 22) 128 + 128 columns:
//   4 of 128 keys                  14 / 14 / 11 / 11      18 / 18 / 16 / 14      21 / 22 / 17
//   32 of 128                      16 / 15 / 19 / 13      21 / 21 / 33 / 26      26 / 29 / 34
//   64 of 128                      23 / 30 / 39 / 24      31 / 39 / 63 / 50      49 / 54 / 67
//   256 of 32                      28 / 51 / 59 / 30      35 / 68 / 84 / 66      68 / 89 / 81
//   4 of 512                       45 / 35 / 24 / 29      58 / 44 / 33 / 38      69 / 56 / 46
//   16 of 512                      49 / 48 / 62 / 48      64 / 64 / 91 / 91      92 / 87 / 113
//   2 of 2048                     165 / 118 / 83 / 101   216 / 148 / 114 / 143  253 / 186 / 177
//   4 of 2048                     168 / 133 / 157 / 148  222 / 173 / 222 / 278  276 / 236 / 342
//   16 of 2048                    487 / 526 / 627 / 546  658 / 700 / 894 / 1107 1097 / 953 / 1366
// Over 420 such launches (32 to 2048 keys, 24 to 2048 tiles of 128 queries, also of uneven lengths) the choice below is at worst
// 1.02 times as slow as 41 and in the mean 1.01 times the best of the four; by the number of tiles alone it was 1.16, and
// up to 1.9 times 41 for many short prompts.
int f32_form(int columns, long keys, int H, int nseq, int max_q, long rows) {
    auto tiles = [&](int q) {
        const long most = (long)H * nseq * ((max_q + q - 1) / q);
        return rows > 0 ? std::min(most, H * (rows / q + (nseq + 1) / 2)) : most;
    };
    const bool wide = columns > 192;
    const long t64 = tiles(64), t128 = tiles(128);
    if (keys <= 32) return 41;
    if (t64 <= 256) return !wide && keys >= (columns > 128 ? 256 : 96) ? 24 : 22;
    if (t64 <= 512 && (keys >= 192 || columns <= 128)) return !wide && (keys >= 1024 || (keys >= 512 && t64 <= 384)) ? 24 : 22;
    if (wide) return keys >= 384 ? 42 : 41;
    return (keys >= 384 && t128 <= 384) || (keys >= 512 && t128 <= 512) || (keys >= 1024 && t128 <= 640) ? 42 : 41;
}

template <int DP, int EP>
int launch_f32(const PromptArgs32& a, int nseq, int max_q, hipStream_t s) {
    if (a.rule.temps || a.rule.softcap > 0.f || a.rule.pool > 0) return launch_f32_as<DP, EP, true, 4, 1>(a, nseq, max_q, s);
    switch (f32_form(DP + EP, longest_walk(a.max_blocks, a.block_size, a.rule), a.H, nseq, max_q, a.clear.end - a.clear.first)) {
        case 24: if constexpr (DP + EP <= 192) return launch_f32_as<DP, EP, false, 2, 4>(a, nseq, max_q, s);
        case 22: return launch_f32_as<DP, EP, false, 2, 2>(a, nseq, max_q, s);
        case 42: return launch_f32_as<DP, EP, false, 4, 2>(a, nseq, max_q, s);
        default: return launch_f32_as<DP, EP, false, 4, 1>(a, nseq, max_q, s);
    }
}

template <int DP, int RP, int EP, int PARTS, bool EXT, bool WHOLE, int KG>
int launch_groups(const PromptArgs& a, int nseq, int max_q, hipStream_t s) {
    constexpr int lds = KG * 32 * 2 * (3 * (DP + RP) + 4 * EP);
    static_assert(lds <= 160 * 1024);
    auto* kernel = prompt_attention_kernel<DP, RP, EP, PARTS, EXT, WHOLE, KG>;
    if (lds > 64 * 1024) {
        static const hipError_t once = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (once != hipSuccess) return 2;
    }
    hipLaunchKernelGGL(kernel, dim3(a.H, nseq, (max_q + 127) / 128), dim3(256 * KG), lds, s, a);
    return HYB_LAUNCH_OK();
}

// Groups of waves on a workgroup's queries, for images of so many key and value columns (`columns`: both).  A second group shortens each one's
// run of tiles; it pays where there is a workgroup for every CU at most, and where the run is long enough for the groups'
// meeting.  us, one group / two, 8 heads, prompts of equal length, 128 workgroups:
//   keys a prompt      64        128       256       384       512       1024      2048
//   64 + 64           10 / 9    10 / 10   13 / 12   16 / 14   18 / 16   31 / 25   55 / 41
//   128 + 128         10 / 10   11 / 13   15 / 16   19 / 18   23 / 21   38 / 32   68 / 53
//   64 + 256          11 / 14   15 / 19   20 / 23   25 / 26   30 / 30   50 / 45   89 / 77
//   256 + 128         10 / 12   13 / 16   17 / 19   22 / 23   26 / 26   43 / 39   76 / 65
// The two last spill some 20 registers with two groups of waves on a CU, which one group has room for.  Keys and values formed
// from latents, 16 heads: 4 of 256 41.7 / 41.8, 5 of 384 50 / 48.5, one of 1024 68.5 / 62.
int groups_of(int columns, int value_columns, long keys, long workgroups) {
    const bool spills = value_columns > 128 || columns > 320;
    return workgroups <= 256 && keys >= (spills ? 640 : 384) ? 2 : 1;
}

template <int DP, int RP, int EP, int PARTS, bool EXT, bool WHOLE>
int launch_form(const PromptArgs& a, int nseq, int max_q, hipStream_t s) {
    if constexpr (!EXT && 2 * 32 * 2 * (3 * (DP + RP) + 4 * EP) <= 160 * 1024) {
        if (groups_of(DP + EP, EP, longest_walk(a.max_blocks, a.block_size, a.rule), (long)a.H * nseq * ((max_q + 127) / 128)) == 2)
            return launch_groups<DP, RP, EP, PARTS, EXT, WHOLE, 2>(a, nseq, max_q, s);
    }
    return launch_groups<DP, RP, EP, PARTS, EXT, WHOLE, 1>(a, nseq, max_q, s);
}

template <int DP, int EP>
int launch(const PromptArgs& a, int nseq, int max_q, hipStream_t s) {
    if (a.rule.temps || a.rule.softcap > 0.f || a.rule.pool > 0) return launch_form<DP, 0, EP, 3, true, false>(a, nseq, max_q, s);
    return a.page_magic && a.block_size % 32 == 0 ? launch_form<DP, 0, EP, 3, false, true>(a, nseq, max_q, s)
                                                  : launch_form<DP, 0, EP, 3, false, false>(a, nseq, max_q, s);
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
                     const KeyRule& rule, RowSpan clear, hipStream_t s) {
    const PromptArgs a{(const uint16_t*)q, q_row, q_head, (const uint16_t*)k_cache, (const uint16_t*)v_cache,
                       (const int*)block_tables, max_blocks, block_size, (const int*)cu_q, (const int*)positions,
                       (const float*)sink, (const bf16_t*)gate, gate_row, (uint16_t*)out, scale, H, G, D, E, seq0, rule, nullptr, 0, nullptr, 0, 0, 0, clear,
                       page_magic(block_size, max_blocks, 2L * G * (D > rule.v_stride ? D : rule.v_stride))};
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
                         const KeyRule& rule, RowSpan clear, hipStream_t s) {
    const PromptArgs32 a{(const float*)q, q_row, q_head, (const float*)k_cache, (const float*)v_cache,
                         (const int*)block_tables, max_blocks, block_size, (const int*)cu_q, (const int*)positions,
                         (const float*)sink, (const float*)gate, gate_row, (float*)out, scale, H, G, D, E, seq0, rule, clear};
    if (D <= 64) return E <= 64 ? launch_f32<64, 64>(a, nseq, max_q, s) : launch_f32<64, 128>(a, nseq, max_q, s);
    return E <= 64 ? launch_f32<128, 64>(a, nseq, max_q, s) : launch_f32<128, 128>(a, nseq, max_q, s);
}

bool latent_prompts_pages_ok(int block_size, int max_blocks, int latent_row) {
    return block_size > 0 && block_size % 32 == 0 && page_magic(block_size, max_blocks, 2L * latent_row) != 0;
}

int latent_prompts(const void* q, long q_row, long q_head, const void* qr, long qr_row, const void* cache,
                   const void* block_tables, int max_blocks, int block_size, const void* cu_q, const void* positions,
                   const void* sink, const void* k, const void* v, long formed_rows, void* out, float scale, int nseq,
                   int max_q, int H, int D, int E, int R, int P, int window, hipStream_t s) {
    if (!latent_prompts_pages_ok(block_size, max_blocks, R + P)) return 1;
    KeyRule rule{};
    rule.window = window;
    rule.v_stride = E;
    const PromptArgs a{(const uint16_t*)q, q_row, q_head, (const uint16_t*)k, (const uint16_t*)v,
                       (const int*)block_tables, max_blocks, block_size, (const int*)cu_q, (const int*)positions,
                       (const float*)sink, nullptr, 0, (uint16_t*)out, scale, H, 1, D, E, 0, rule,
                       (const uint16_t*)qr, qr_row, (const uint16_t*)cache, R + P, P, formed_rows,
                       RowSpan{0, 0}, page_magic(block_size, max_blocks, 2L * (R + P))};
    return P <= 64 ? launch_form<128, 64, 128, 2, false, true>(a, nseq, max_q, s)
                   : launch_form<128, 128, 128, 2, false, true>(a, nseq, max_q, s);
}

}  // namespace hyb

extern "C" {

// The rules above, for tests of where their lines lie.
int hyb_prompt_f32_form(int columns, long keys, int H, int nseq, int max_q, long rows) {
    return f32_form(columns, keys, H, nseq, max_q, rows);
}
int hyb_prompt_groups(int columns, int value_columns, long keys, long workgroups) {
    return groups_of(columns, value_columns, keys, workgroups);
}
int hyb_prompt_longest_walk(int max_blocks, int block_size, int window, int keep_first, int chunk) {
    KeyRule rule{};
    rule.window = window; rule.keep_first = keep_first; rule.chunk = chunk;
    return (int)std::min(longest_walk(max_blocks, block_size, rule), 1L << 30);
}

}  // extern "C"
