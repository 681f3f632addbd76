// Paged attention on the gfx950 matrix cores, bfloat16 cache, for prompt portions and decoded
// tokens alike.
//
// Work is cut the same way whatever the batch: the keys of a request are split into partitions
// of 256 positions (0..255, 256..511, ...), each of four units of 64.  A workgroup takes one
// partition, one kv head and one block of query columns (a column = one query head of one token;
// all columns of a block share the request and the kv head): one wave that walks the four units, or,
// where that would leave the chip idle, four waves with a unit each.  Either way a unit starts from
// a fresh state and the units' results (running maximum m, sum l, unnormalised output o, float32)
// are merged in ascending order through one chain of operations, so both give the same bits.  A
// second kernel merges a token's partitions in ascending order.  Where column blocks are many and partitions few, a
// workgroup of eight waves takes all of a block's partitions and does that itself, in the same order.  Since the columns of a matrix product do not influence each
// other, a token's result does not depend on how the sequence was cut into steps or on what
// else was in the batch.
//
// Inside a wave (S^T = K Q^T, O^T = V^T P^T, all with v_mfma_f32_16x16x32_bf16):
//  * 32 keys a step, in two products of 16.  A operand of S^T: K rows [key][hd], 16 bytes a lane;
//    B operand: Q [column][hd], loaded once.  Row m of product kb is key 8 (m/4) + 4 kb + m % 4.
//  * A result tile gives lane (column = l % 16, group g = l / 16) rows 4g..4g+3, so over both
//    products the lane holds the scores of keys 8g..8g+7 in order.  After masking, running max
//    and exp these eight values are, as they lie, the lane's part of the B operand P^T of the
//    second product (k = 8g + i), and the A operand V^T is one 16-byte load of eight consecutive
//    positions of a channel from the transposed V page.
//  * No transposes, no barriers, LDS only for K rows on their way; K rows and V columns of the next step are loaded
//    while the current step computes, with streaming (non-temporal) loads: a step of single tokens
//    reads every key once.
//
// Cache layout: K [page][kv_head][offset][hd], V [page][kv_head][hd][offset]; the page size
// must be a multiple of 16 and the head size a multiple of 8 (the host falls back to the
// general kernel otherwise).
#include "common.h"
#include <math.h>
#include <mutex>

namespace {
constexpr int PART = 256;

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// What the kernel does itself, for heads of 64 channels, when it is handed the projected rows
// [q heads | k heads | v heads] of a step of single tokens instead of finished queries: the per-head
// RMSNorm of q and k, the half-split rotation, and the write of the token's key and value into the
// cache (by the workgroup whose partition holds the token's position, before it reads its keys).
// The arithmetic is that of the kernel that does this for prompt portions (qkv_post64_kernel), sum
// for sum, so a key in the cache does not tell which of the two wrote it.
struct FusedQKV {
    const void* q_norm_w = nullptr;        // [64] each, float32 or bfloat16 (norm_dt); null: no norm
    const void* k_norm_w = nullptr;
    int norm_dt = DT_F32;
    float eps = 0.f;
    const float* inv_freq = nullptr;       // [32]
    const float* angles = nullptr;         // [n_angles][2][32]: cosines and sines of pos * inv_freq, or null
    int n_angles = 0;
    const int* slot_mapping = nullptr;     // [tokens]; null: the cache is only read
    // (not of the fused form, but of every form: it travels here)  A distance slope per head [H], or null:
    // slopes[h] * (position - key) is taken off head h's scaled scores.
    const float* slopes = nullptr;
    int group = 1;                         // query heads a kv head
};

// cosine and sine of pos * inv_freq[j]: from the table where it reaches, else computed (the same bits)
__device__ __forceinline__ void angle(const FusedQKV& fq, int pos, int j, float& rc, float& rs) {
    if (pos < fq.n_angles) {
        rc = fq.angles[((long long)pos * 2) * 32 + j];
        rs = fq.angles[((long long)pos * 2 + 1) * 32 + j];
    } else {
        const float a = (float)pos * fq.inv_freq[j];
        rc = cosf(a);
        rs = sinf(a);
    }
}

// The same of N neighbours from j on, and N norm weights of either type from i on, both multiples of N: whole pieces at a
// time, one branch.
typedef f32x4 f32x4_any __attribute__((aligned(4)));       // (tables and weights may start anywhere)
typedef bf16x4 bf16x4_any __attribute__((aligned(2)));
template <int N>
__device__ __forceinline__ void angles(const FusedQKV& fq, int pos, int j, float (&rc)[N], float (&rs)[N]) {
    if (pos < fq.n_angles) {
        const float* at = fq.angles + (long long)pos * 64 + j;
#pragma unroll
        for (int e = 0; e < N; e += 4) {
            const f32x4 c = *(const f32x4_any*)(at + e), s = *(const f32x4_any*)(at + 32 + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) { rc[e + i] = c[i]; rs[e + i] = s[i]; }
        }
    } else {
#pragma nounroll
        for (int e = 0; e < N; ++e) {
            float c, s;
            angle(fq, pos, j + e, c, s);
#pragma unroll
            for (int i = 0; i < N; ++i) { rc[i] = i == e ? c : rc[i]; rs[i] = i == e ? s : rs[i]; }
        }
    }
}

template <int N>
__device__ __forceinline__ void norm_weights(const void* w, int dt, int i, float (&out)[N]) {
    if (dt == DT_F32) {
#pragma unroll
        for (int e = 0; e < N; e += 4) {
            const f32x4 x = *(const f32x4_any*)((const float*)w + i + e);
#pragma unroll
            for (int k = 0; k < 4; ++k) out[e + k] = x[k];
        }
    } else {
#pragma unroll
        for (int e = 0; e < N; e += 4) {
            const bf16x4 x = *(const bf16x4_any*)((const bf16_t*)w + i + e);
#pragma unroll
            for (int k = 0; k < 4; ++k) out[e + k] = (float)x[k];
        }
    }
}

// One partial result (m, l, o) merged into a running one, element by element:
//   m' = max(m, mu);  l' = l e^(m - m') + lu e^(mu - m');  o' likewise.
// Both forms of the kernel (one wave or four a partition) merge a partition's four units of 64 keys
// through this, in ascending order, so they give the same bits.
__device__ __forceinline__ void merge_weights(float m, float mu, float& m_new, float& ca, float& cb) {
    m_new = fmaxf(m, mu);
    const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
    ca = __expf(m - m_safe);               // 0 while nothing was seen
    cb = __expf(mu - m_safe);
}

// a ca + b cb as one product and one fused multiply-add, spelled out: left to the compiler, two
// instantiations of the kernel may fuse the other product and differ in the last bit
__device__ __forceinline__ float merged(float a, float ca, float b, float cb) { return fmaf(b, cb, a * ca); }

// a b rounded, whatever is taken from it afterwards
__device__ __forceinline__ float product(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

constexpr int UNIT = 64;                   // keys a unit: two steps of 32
constexpr int UNITS = PART / UNIT;

// How many pages the partition that starts at key_begin (a multiple of PART) touches: one lane of the
// wave fetches each page's number.  A partition that starts inside a page (page sizes that do not divide
// PART) touches one page more than PART / page_size rounded up.
__host__ __device__ inline int partition_pages(int key_begin, int page_size) {
    return (key_begin + PART - 1) / page_size - key_begin / page_size + 1;
}

// NW: waves a workgroup (1: the wave walks the partition's four units; 4: a unit a wave, merged through LDS; more: the workgroup
// takes all partitions of its column block, its waves the units in turn, merges them and writes the finished rows, no kernel after it).
template <int HDP, int NB, int NW, bool FUSED, bool STREAM_V, bool STAGE_K = false>
__global__ __launch_bounds__(NW * WAVE) void attn_partition_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache,
    float* __restrict__ ws_o, float* __restrict__ ws_ml,
    const int* __restrict__ block_table, int max_blocks,
    const int2* __restrict__ blk, const int4* __restrict__ req_info,
    int H, int Hkv, int hd, int page_size, int window, float scale, int n_parts, FusedQKV fq, int kv_fast,
    bf16_t* __restrict__ out, const float* __restrict__ sinks) {
    constexpr bool WHOLE = NW > UNITS;     // out and sinks are this form's; ws_o and ws_ml the others'
    static_assert(NW == 1 || NW % UNITS == 0, "one wave a partition, one a unit, or whole partitions side by side");
    static_assert(!WHOLE || (HDP == 64 && NB == 1), "all partitions a workgroup: heads of up to 64 and one column block");
    static_assert(!FUSED || (HDP == 64 && NB == 1), "the fused form is for heads of 64 and one column block");
    constexpr int KC = HDP / 32;          // 32-wide chunks of the head dimension
    constexpr int DB = HDP / 16;          // 16-wide blocks of output channels
    const int ps = STREAM_V ? 16 : page_size;              // (STREAM_V: pages of sixteen; what is divided by them is shifted)
    const int HD = FUSED ? 64 : hd;
    // Workgroups that run side by side read neighbouring memory when the kv head is what changes fastest
    // from one to the next (a page holds its kv heads one after the other): that order for launches of
    // several rounds of waves, partitions first for the others.
    const int part = WHOLE ? 0 : kv_fast ? blockIdx.x / Hkv : blockIdx.x, qb = blockIdx.y, kvh = kv_fast ? (int)blockIdx.x - part * Hkv : blockIdx.z;
    const int lane = threadIdx.x % WAVE, n16 = lane % 16, g = lane / 16;
    const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int G = fq.group;
    // Every load that depends on another costs a trip to memory, so the chain is kept short: block -> request record (start,
    // length, first position: a portion's positions are consecutive), and beside it the page numbers, all at once -> keys and
    // values.
    int r = qb, col0 = 0;                  // without a block list every request is one block
    if (blk) { const int2 b = blk[qb]; r = b.x; col0 = b.y; }
    const int4 info = req_info[r];         // (first token of the request in the step, tokens, first position, -)
    const int* table = block_table + (long long)r * max_blocks;
    const int t0 = info.x, ncols = FUSED ? G : info.y * G, pos0 = info.z;
    // the block's range of keys (fused: a block is one token's columns)
    const int last_col = FUSED ? G - 1 : min(ncols, col0 + NB * 16) - 1;
    const int pos_max = FUSED ? pos0 : pos0 + last_col / G;
    const int lo_min = window > 0 ? max(0, pos0 + (FUSED ? 0 : col0 / G) - window + 1) : 0;
    const int key_begin = WHOLE ? lo_min / PART * PART : part * PART;
    const int first_page = key_begin / ps;
    int my_page = 0;                       // lane i: the page of the partition's i-th block of page_size keys
    if constexpr (WHOLE) {
        // lane 8 j + i: the page of the i-th such block of the wave's unit of turn j (a unit touches at most four)
        const int block = (key_begin + (lane / 8 * NW + wave) * UNIT) / ps + lane % 8;
        if (block < max_blocks) my_page = table[block];
    } else {
        if (lane < partition_pages(key_begin, ps) && first_page + lane < max_blocks) my_page = table[first_page + lane];
        if (key_begin > pos_max || key_begin + PART <= lo_min) return;
    }
    const int key_end = WHOLE ? pos_max + 1 : min(key_begin + PART, pos_max + 1);

    // (of the whole form, the wave that reads the token's key writes it)
    auto write_token = [&]() {
        const long long slot = fq.slot_mapping[t0];
        if (slot >= 0) {
            const long long page = slot / ps, off = slot % ps;
            const int row_width = (H + 2 * Hkv) * 64;
            const bf16_t* row = q + (long long)t0 * row_width;
            const int l = lane % 16;
            const bf16_t value = row[(H + Hkv + kvh) * 64 + lane];
            const bf16x4 raw = *(const bf16x4*)(row + (H + kvh) * 64 + 4 * l);
            float rc[4], rs[4], nw[4] = {};
            if (fq.k_norm_w != nullptr) norm_weights<4>(fq.k_norm_w, fq.norm_dt, 4 * l, nw);
            angles<4>(fq, pos0, (4 * l) & 31, rc, rs);
            // value: lane = channel, as projected
            v_cache[((page * Hkv + kvh) * 64 + lane) * ps + off] = value;
            // key: sixteen lanes hold four channels each (the other lanes do the same work again)
            float v[4] = {(float)raw[0], (float)raw[1], (float)raw[2], (float)raw[3]};
            float ss = v[0] * v[0];
            ss = fmaf(v[1], v[1], ss);
            ss = fmaf(v[2], v[2], ss);
            ss = fmaf(v[3], v[3], ss);
            ss = row_sum_down(ss);
            if (fq.k_norm_w != nullptr) {
                const float inv = 1.0f / sqrtf(ss / 64.0f + fq.eps);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = v[e] * inv * nw[e];
            }
            const bool first = l < 8;
            bf16x4 o4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float other = lane_xor8(v[e]);
                const float x0 = first ? v[e] : other, x1 = first ? other : v[e];
                o4[e] = (bf16_t)(first ? (x0 * rc[e] - x1 * rs[e]) : (x0 * rs[e] + x1 * rc[e]));
            }
            if (lane < 16) *(bf16x4*)(k_cache + ((page * Hkv + kvh) * ps + off) * 64 + 4 * l) = o4;
        }
    };
    if constexpr (FUSED) {
        // the token's key and value go into the cache before anybody reads the partition that holds them
        if constexpr (WHOLE) {
            if (fq.slot_mapping != nullptr && wave == (pos0 - key_begin) / UNIT % NW) {
                write_token();
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");      // for the other lanes of this wave, which reads them
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            }
        } else if (fq.slot_mapping != nullptr && pos0 / PART == part) {
            if (wave == 0) write_token();
            __syncthreads();               // the stores have landed before a wave of this workgroup loads the keys
        }
    }

    // the unit under way, and the partition's result so far
    float m_run[NB], l_run[NB];
    f32x4 o[DB][NB];
    float m_acc[NB], l_acc[NB];
    f32x4 o_acc[DB][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m_acc[nb] = -INFINITY;
        l_acc[nb] = 0.f;
#pragma unroll
        for (int db = 0; db < DB; ++db) o_acc[db][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // One step covers 32 keys, two halves of 16 that each lie in one page.  The two S^T products
    // of a step do not take the keys in order: row m of product kb is key 8 (m / 4) + 4 kb + m % 4
    // of the step, so that lane group g ends up with the scores of keys 8g .. 8g+7, which is what
    // the second product's operands hold for k = 8g + i.  A step's K rows and V columns are loaded
    // into registers a step ahead of their use (where the head size leaves room for it); large
    // tiles (head size x columns) load as they go.
    //
    // What bounds it: a wave issues an instruction in about five cycles, so with three waves a SIMD the instructions around the loads
    // and products count as much as the bytes, until they are few: 64 requests of 8,192 keys then move 5.95 TB/s (counters: two
    // thirds of a wave's time its instructions wait for the memory side to take them), one request is the chain of its trips.  Hence no branch but those a whole wave takes, every lane loads
    // from a page that holds keys of the request whatever its own are, only steps at an end of the keys look at single keys,
    // and pages of sixteen (STREAM_V) are shifted, not divided: a step of 32 keys in some 170 instructions instead of 670.  One
    // layer's attention, 32 heads on 8: 64 requests of 8,192 keys 201 -> 184 us (5.8 TB/s), 8 of 8,192 29.7 -> 25, one of 256
    // 8.6 -> 6.4; heads of 128, 32 requests of 4,000 116 -> 95, of 256 (16 on 4) 107 -> 98.
    constexpr bool AHEAD = HDP * NB <= 256;
    // STAGE_K (heads of up to 64 channels): a step's keys are asked for as they lie in memory, 1 KB an instruction (the
    // 16 keys of a half are one run of 16 hd elements), and go through LDS into the order of the matrix operands.  Asked
    // for in that order at once, an instruction touches half of each of sixteen lines and every line is asked for twice:
    // whole lines are 2 to 6 % of a decode step faster wherever waves walk a partition by themselves.
    static_assert(!STAGE_K || (HDP == 64 && HDP * NB <= 256 && NW != UNITS), "staged keys: heads of up to 64, not with a unit a wave");
    constexpr bool STAGE = STAGE_K;
    __shared__ __attribute__((aligned(16))) bf16_t k_stage[STAGE ? NW : 1][STAGE ? 32 * 64 : 8];
    // where the 16-byte piece `chunk` of key `key` of the step lies in the wave's 4 KB: rows of 128 bytes, the pieces of
    // a row exchanged so that the sixteen rows an operand read takes its pieces from fall into different banks
    auto stage_at = [&](int key, int chunk) { return key * 64 + ((chunk ^ (((key >> 1) & 1) | (((key >> 3) & 3) << 1))) * 8); };
    const int row_pieces = HD / 8;                                   // 16-byte pieces of a key
    int stage_to[2][2];                                              // where this lane's four pieces of a step go (-1: no piece)
    if constexpr (STAGE) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int piece = 64 * i + lane;
                stage_to[h][i] = piece < 16 * row_pieces ? stage_at(16 * h + piece / row_pieces, piece % row_pieces) : -1;
            }
    }
    struct Tile {
        bf16x8 kf[2][AHEAD ? KC : 1];
        bf16x8 vx[AHEAD ? DB : 1];
        const bf16_t *k_at, *v_at;         // (not AHEAD) where this lane's parts of the keys and values begin
    };
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    // Channels beyond the head are asked for as its first ones.  The keys' are zero before a product reads them, as the query's
    // are (an infinite key times the query's zero is none); the values' give results that nobody takes.
    const bool narrow = HD < HDP;
    using place_t = std::conditional_t<STREAM_V, unsigned, unsigned long long>;        // (pages of sixteen: 32 bits hold any place in one)
    const place_t page_elems = (place_t)Hkv * ps * HD;
    // this lane's place in a half's keys and values: key 8 ((n16 / 4) % 2) + n16 % 4 (+ 4 kb) of half n16 / 8; channel n16
    // (+ 16 db), positions 8 (g % 2) of half g / 2
    const bf16_t* const k_mine = k_cache + (long long)kvh * ps * HD + (8 * ((n16 / 4) % 2) + n16 % 4) * HD;
    const bf16_t* const v_mine = v_cache + (long long)kvh * ps * HD + (g % 2) * 8;
    auto k_frag = [&](const bf16_t* at, int kb, int kc, bool narrow) {
        const int k = kc * 32 + g * 8;
        return __builtin_nontemporal_load((const bf16x8*)(at + 4 * kb * HD + (!narrow || k < HD ? k : 0)));
    };
    // A page's V^T rows are 2 * page_size bytes: with pages of 16 positions a step of 32 keys reads whole rows and
    // never comes back to them; with larger pages it reads a part of each row's cache lines and the steps after it
    // read the rest, so those loads are ordinary ones (a line asked for as streaming does not wait for them):
    // STREAM_V is page_size == 16.
    auto v_frag = [&](const bf16_t* at, int db) {
        const int dim = db * 16 + n16;
        const bf16x8* from = (const bf16x8*)(at + (place_t)(!narrow || dim < HD ? dim : 0) * ps);
        if constexpr (STREAM_V) return __builtin_nontemporal_load(from); else return *from;
    };
    // the page that holds block `block` of page_size keys; key: one of the step's
    auto page_of = [&](int block, int key) {
        int holder = block - first_page;
        if constexpr (WHOLE) {
            const int unit = (key - key_begin) / UNIT;
            holder = unit / NW * 8 + block - (key_begin + unit * UNIT) / ps;
        }
        return (unsigned)__builtin_amdgcn_readlane(my_page, holder & (WAVE - 1));
    };
    if constexpr (STAGE) {
        // the pieces beyond the head, which no step's keys go to
        if (narrow)
            for (int i = lane; i < 32 * 8; i += WAVE)
                if (i % 8 >= row_pieces) *(bf16x8*)(k_stage[wave] + stage_at(i / 8, i % 8)) = zero8;
    }
    auto load_tile = [&](int key0, Tile& t) {
        // a half without a key that some column may see: the other half's keys in its place (their weights are zero), and
        // where both are, the first page's (the cache's own first one where that is no longer held)
        const bool live0 = key0 <= pos_max && key0 + 15 >= lo_min, live1 = key0 + 16 <= pos_max && key0 + 31 >= lo_min;
        const int h0 = live0 ? key0 : key0 + 16, h1 = live1 ? key0 + 16 : key0;
        const bool any = live0 || live1;
        const unsigned at0 = page_of(h0 / ps, key0), at1 = page_of(h1 / ps, key0);
        const unsigned none = max(__builtin_amdgcn_readlane(my_page, 0), 0);
        const unsigned p0 = any ? at0 : none, p1 = any ? at1 : none;
        const int off0 = any ? h0 % ps : 0, off1 = any ? h1 % ps : 0;      // multiples of 16
        if constexpr (STAGE) {
            // kf[h][i]: pieces 64 i + lane of half h, as they lie in memory
            const bf16_t* const at[2] = {k_cache + ((unsigned long long)p0 * page_elems + ((place_t)kvh * ps + off0) * HD),
                                         k_cache + ((unsigned long long)p1 * page_elems + ((place_t)kvh * ps + off1) * HD)};
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int piece = 64 * i + lane;
                    t.kf[h][i] = __builtin_nontemporal_load((const bf16x8*)(at[h] + (!narrow || piece < 16 * row_pieces ? piece : 0) * 8));
                }
        }
        const bf16_t* const v_at = v_mine + ((unsigned long long)(g / 2 ? p1 : p0) * page_elems + (place_t)(g / 2 ? off1 : off0));
        if constexpr (AHEAD) {
            if constexpr (!STAGE) {
                const bf16_t* const k_at = k_mine + ((unsigned long long)(n16 / 8 ? p1 : p0) * page_elems + (place_t)(n16 / 8 ? off1 : off0) * HD);
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc) t.kf[kb][kc] = k_frag(k_at, kb, kc, narrow);
            }
#pragma unroll
            for (int db = 0; db < DB; ++db) t.vx[db] = v_frag(v_at, db);
        } else {
            t.k_at = k_mine + ((unsigned long long)(n16 / 8 ? p1 : p0) * page_elems + (place_t)(n16 / 8 ? off1 : off0) * HD);
            t.v_at = v_at;
        }
    };
    // The first keys and values are asked for before the queries are prepared: they depend on the page
    // numbers alone, and the queries' norm and rotation (in the fused form) then run while the keys are on their way.  What the
    // queries are made of is asked for ahead of them: loads of a CU come back in the order they were asked for (32 heads on 8, kernel and
    // merge: one request of 256 keys 7.56 -> 7.15 us, 8 of 256 6.5 -> 6.3, 8 of 3,000 14.3 -> 13.2, one of 30,000 21.3 -> 20.7, with no divisions where
    // a block is one token; one of 900 7.9 -> 8.0).
    // (of the whole form, the wave after the one that writes the token prepares the queries, the others read them from LDS)
    __shared__ __attribute__((aligned(16))) bf16_t q_stage[WHOLE && FUSED ? KC * WAVE * 8 : 8];
    const bool prepares = !(WHOLE && FUSED) || wave == ((pos0 - key_begin) / UNIT + 1) % NW;
    struct Raw { bf16x8 r0, r1; float rc[8], rs[8], w0[8], w1[8]; };
    Raw raw;
    if constexpr (FUSED) {
        if (prepares) {
            // channels 8g .. 8g+7 and 32 + 8g .. 32 + 8g+7 of the head: partners of the rotation sit in one lane
            const bf16_t* src = q + (long long)t0 * ((H + 2 * Hkv) * 64) + (kvh * G + (n16 < G ? n16 : 0)) * 64 + g * 8;
            raw.r0 = *(const bf16x8*)src;
            raw.r1 = *(const bf16x8*)(src + 32);
            if (fq.q_norm_w != nullptr) {
                norm_weights<8>(fq.q_norm_w, fq.norm_dt, g * 8, raw.w0);
                norm_weights<8>(fq.q_norm_w, fq.norm_dt, 32 + g * 8, raw.w1);
            }
            angles<8>(fq, pos0, g * 8, raw.rc, raw.rs);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    Tile ta, tb;
    const int key_first = NW == 1 ? key_begin : key_begin + wave * UNIT;
    if constexpr (AHEAD) {
        if (NW == 1 || key_first < key_end) {
            load_tile(key_first, ta);
            if (NW > 1 && !WHOLE) load_tile(key_first + 32, tb);
        }
    }

    // this lane's columns
    int pos_c[NB], lo_c[NB];
    float slope_c[NB];
    const bool has_slopes = !FUSED && fq.slopes != nullptr;
    long long qrow[NB];                    // row of the column in the work space; -1: no column
    bf16x8 qf[NB][KC];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int c = col0 + nb * 16 + n16;
        const bool valid = c < ncols;
        const int cc = valid ? c : col0;   // no column: another one's query, whose result nobody takes
        const int tok = FUSED ? t0 : t0 + cc / G;
        const int head = kvh * G + (FUSED ? cc : cc % G);
        slope_c[nb] = has_slopes ? fq.slopes[head] : 0.f;
        pos_c[nb] = FUSED ? pos0 : pos0 + cc / G;
        lo_c[nb] = window > 0 ? max(0, pos_c[nb] - window + 1) : 0;
        qrow[nb] = valid ? (long long)tok * H + head : -1;
        if constexpr (FUSED) {
            if (!prepares) continue;
            float v0[8], v1[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) { v0[e] = (float)raw.r0[e]; v1[e] = (float)raw.r1[e]; }
            // sums of squares of four channels each, then the butterfly of sixteen such sums in the order
            // of the kernel for portions (partners 32, 16, 8 and 4 channels away)
            float p[2][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float a = v0[4 * h] * v0[4 * h], b = v1[4 * h] * v1[4 * h];
#pragma unroll
                for (int e = 1; e < 4; ++e) { a = fmaf(v0[4 * h + e], v0[4 * h + e], a); b = fmaf(v1[4 * h + e], v1[4 * h + e], b); }
                p[0][h] = a; p[1][h] = b;
            }
            float s0 = p[0][0] + p[1][0], s1 = p[0][1] + p[1][1];
            s0 = butterfly_sum<16>(butterfly_sum<32>(s0)); s1 = butterfly_sum<16>(butterfly_sum<32>(s1));
            const float ss = s0 + s1;
            if (fq.q_norm_w != nullptr) {
                const float inv = 1.0f / sqrtf(ss / 64.0f + fq.eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v0[e] = v0[e] * inv * raw.w0[e];
                    v1[e] = v1[e] * inv * raw.w1[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x0 = v0[e], x1 = v1[e];
                // (the fused product spelled out: left to the compiler, the forms of the kernel choose differently)
                qf[nb][0][e] = (bf16_t)fmaf(x0, raw.rc[e], -product(x1, raw.rs[e]));
                qf[nb][1][e] = (bf16_t)fmaf(x0, raw.rs[e], product(x1, raw.rc[e]));
            }
        } else {
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) {
                const int k = kc * 32 + g * 8;
                qf[nb][kc] = k < HD ? *(const bf16x8*)(q + ((long long)tok * H + head) * HD + k) : zero8;
            }
        }
    }
    if constexpr (WHOLE) {
        if (key_first + 32 < key_end) load_tile(key_first + 32, tb);
    }
    if constexpr (WHOLE && FUSED) {
        if (prepares) {
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) *(bf16x8*)(q_stage + (kc * WAVE + lane) * 8) = qf[0][kc];
        }
        lds_barrier();
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) qf[0][kc] = *(const bf16x8*)(q_stage + (kc * WAVE + lane) * 8);
    }

    // Scores stay as the products leave them, and their scale goes into the base of the exponential: e^(scale (s - max)) is
    // 2^(log2s s - log2s max).  With distance slopes (or a scale that turns the order round) they are scaled first.
    const bool scaled = has_slopes || !(scale > 0.f);
    const float to_m = scaled ? 1.f : scale, log2s = to_m * 1.44269504088896340736f;
    auto exp2_of = [](float x) { return __builtin_amdgcn_exp2f(x); };
    // what every column of the block sees: a step within it takes all its keys as they are
    const int all_lo = window > 0 ? max(0, pos_max - window + 1) : 0, all_hi = FUSED ? pos0 : pos0 + col0 / G;
    // FIRST: the unit's first step, which finds nothing to scale
    auto compute = [&](int key0, Tile& t, auto FIRST) {
        // ---- S^T = K Q^T, twice 16 keys
        f32x4 s[2][NB];
        bf16_t* stage = k_stage[STAGE ? wave : 0];
        if constexpr (STAGE) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (!narrow || stage_to[h][i] >= 0) *(bf16x8*)(stage + stage_to[h][i]) = t.kf[h][i];
                }
            __builtin_amdgcn_wave_barrier();       // the wave's LDS accesses run in the order of the program
        }
        auto scores = [&](auto NARROW) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) s[kb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kc = 0; kc < KC; ++kc) {
                    bf16x8 kf;
                    const int chunk = kc * 4 + g;
                    if constexpr (STAGE) kf = *(const bf16x8*)(stage + stage_at(8 * (n16 / 4) + 4 * kb + n16 % 4, chunk));
                    else if constexpr (AHEAD) kf = t.kf[kb][kc];
                    else kf = k_frag(t.k_at, kb, kc, decltype(NARROW)::value);
                    if (decltype(NARROW)::value && chunk * 8 >= HD) kf = zero8;
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) s[kb][nb] = mfma32(kf, qf[nb][kc], s[kb][nb]);
                }
            }
        };
        // (staged, the pieces beyond the head lie in LDS as zeros)
        if constexpr (AHEAD) {
            if (!STAGE && narrow) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc)
                        if ((kc * 4 + g) * 8 >= HD) t.kf[kb][kc] = zero8;
            }
            scores(std::false_type());
        } else if (narrow) scores(std::true_type());
        else scores(std::false_type());
        // ---- mask, running maximum, exp; P^T stays in registers as the next B operand
        const bool whole_step = key0 >= all_lo && key0 + 31 <= all_hi;
        bf16x8 pf[NB];
        float corr[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = s[i / 4][nb][i % 4];
            if (scaled) {
                // (the distance as an integer first: far positions lose no bits)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = fmaf(v[i], scale, slope_c[nb] * (float)(key0 + 8 * g + i - pos_c[nb]));
            }
            if (!whole_step) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int key = key0 + 8 * g + i;
                    v[i] = key <= pos_c[nb] && key >= lo_c[nb] ? v[i] : -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
            mx = butterfly_max<32>(butterfly_max<16>(mx));
            const float m_new = FIRST ? mx : fmaxf(m_run[nb], mx);
            const float m_safe = (m_new == -INFINITY) ? 0.f : product(m_new, log2s);
            if constexpr (!FIRST) corr[nb] = exp2_of(fmaf(m_run[nb], log2s, -m_safe));      // 0 while nothing was seen yet
            float p[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                p[i] = exp2_of(fmaf(v[i], log2s, -m_safe));
                pf[nb][i] = (bf16_t)p[i];
            }
            const float sum = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            if constexpr (FIRST) l_run[nb] = sum; else l_run[nb] = fmaf(l_run[nb], corr[nb], sum);
            m_run[nb] = m_new;
        }
        // ---- O^T = O^T * corr + V^T P^T
        // values of keys that no column sees may be anything (beyond pos_max none was written)
        const bool tail = key0 + 31 > pos_max || key0 < lo_min;
        auto clear_unseen = [&](bf16x8& vf) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int key = key0 + 8 * g + i;
                if (key > pos_max || key < lo_min) vf[i] = (bf16_t)0.f;
            }
        };
        if (AHEAD && tail) {
#pragma unroll
            for (int db = 0; db < (AHEAD ? DB : 1); ++db) clear_unseen(t.vx[db]);
        }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            bf16x8 vf;
            if constexpr (AHEAD) vf = t.vx[db];
            else {
                vf = v_frag(t.v_at, db);
                if (tail) clear_unseen(vf);
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                if constexpr (!FIRST) {
                    acc = o[db][nb];
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] *= corr[nb];
                }
                o[db][nb] = mfma32(vf, pf[nb], acc);
            }
        }
    };
    constexpr std::true_type first_step;
    constexpr std::false_type later_step;
    auto begin_unit = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            m_run[nb] = -INFINITY;
            l_run[nb] = 0.f;
#pragma unroll
            for (int db = 0; db < DB; ++db) o[db][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // the unit's sum of a column is spread over the four lane groups until here, and its maximum is one of scores
    auto unit_sums = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            l_run[nb] = butterfly_sum<32>(butterfly_sum<16>(l_run[nb]));
            m_run[nb] = product(m_run[nb], to_m);
        }
    };

    // Heads wider than 128 channels have no form of four waves to agree with, and a second set of accumulators does
    // not fit beside the first in a wave's registers: the partition is walked as one unit.
    constexpr bool ONE_UNIT = HDP > 128;
    if constexpr (WHOLE) {
        // Every wave takes a unit of each turn of NW; a turn's units are merged into partitions through LDS, a wave a column
        // of a partition at a time, and the partitions at the end, each element through the chains of the other forms and of
        // their merge.  The next turn's keys are asked for before this one's are merged.
        extern __shared__ __attribute__((aligned(16))) float whole_lds[];
        const int cols = FUSED ? G : 16, n_cols = last_col + 1 - col0, n_units = (pos_max - key_begin) / UNIT + 1;
        float* const u_o = whole_lds;                      // [NW][cols][64]
        float* const p_o = u_o + NW * cols * 64;           // [n_parts][cols][64]
        float* const u_ml = p_o + n_parts * cols * 64;     // [NW][cols][2]
        float* const p_ml = u_ml + NW * cols * 2;          // [n_parts][cols][2]
        for (int first = 0; first < n_units; first += NW) {
            const int u = first + wave, key0 = key_begin + u * UNIT, key_next = key0 + NW * UNIT;
            if (u < n_units) {
                compute(key0, ta, first_step);
                if (key_next < key_end) load_tile(key_next, ta);
                if (key0 + 32 < key_end) compute(key0 + 32, tb, later_step);
                if (key_next + 32 < key_end) load_tile(key_next + 32, tb);
                unit_sums();
            }
            if (first > 0) lds_barrier();                  // the turn before has been read
            if (u < n_units && n16 < n_cols) {
                if (g == 0) { u_ml[(wave * cols + n16) * 2] = m_run[0]; u_ml[(wave * cols + n16) * 2 + 1] = l_run[0]; }
#pragma unroll
                for (int db = 0; db < DB; ++db) *(f32x4*)(u_o + (wave * cols + n16) * 64 + db * 16 + 4 * g) = o[db][0];
            }
            lds_barrier();
            const int units = min(NW, n_units - first), jobs = (units + UNITS - 1) / UNITS * n_cols;
            for (int job = wave; job < jobs; job += NW) {
                const int p = job / n_cols, c = job % n_cols;
                float m = -INFINITY, l = 0.f, acc = 0.f;
#pragma unroll
                for (int i = 0; i < UNITS; ++i) {
                    const int v = p * UNITS + i;
                    if (v < units) {
                        float m_new, ca, cb;
                        merge_weights(m, u_ml[(v * cols + c) * 2], m_new, ca, cb);
                        l = merged(l, ca, u_ml[(v * cols + c) * 2 + 1], cb);
                        acc = merged(acc, ca, u_o[(v * cols + c) * 64 + lane], cb);
                        m = m_new;
                    }
                }
                const int at = (first / UNITS + p) * cols + c;
                if (lane == 0) { p_ml[at * 2] = m; p_ml[at * 2 + 1] = l; }
                p_o[at * 64 + lane] = acc;
            }
        }
        lds_barrier();
        const int parts = (n_units + UNITS - 1) / UNITS;
        for (int c = wave; c < n_cols; c += NW) {
            const int head = kvh * G + (FUSED ? c : (col0 + c) % G);
            const float sink = sinks ? sinks[head] : -INFINITY;
            float m_l = -INFINITY, l_l = 0.f;              // of partition `lane`
            if (lane < parts) { m_l = p_ml[(lane * cols + c) * 2]; l_l = p_ml[(lane * cols + c) * 2 + 1]; }
            const float M = fmaxf(wave_max(l_l > 0.f ? m_l : -INFINITY), sink);
            const float w_l = l_l > 0.f ? __expf(m_l - M) : 0.f, wl_l = w_l * l_l;
            float L = 0.f, acc = 0.f;
            for (int p = 0; p < parts; ++p) {
                const float w = lane_of(w_l, p);
                L += lane_of(wl_l, p);
                if (w > 0.f) acc = fmaf(w, p_o[(p * cols + c) * 64 + lane], acc);
            }
            if (sinks) L += __expf(sink - M);
            if (lane < hd) out[((long long)(FUSED ? t0 : t0 + (col0 + c) / G) * H + head) * hd + lane] = (bf16_t)(acc * (1.0f / L));
        }
        return;
    } else if constexpr (NW == 1 && ONE_UNIT) {
        begin_unit();
        for (int key0 = key_begin; key0 < key_end; key0 += UNIT) {
            if constexpr (AHEAD) {
                const bool more = key0 + 32 < key_end;
                if (more) load_tile(key0 + 32, tb);
                compute(key0, ta, later_step);
                if (more) {
                    if (key0 + UNIT < key_end) load_tile(key0 + UNIT, ta);
                    compute(key0 + 32, tb, later_step);
                }
            } else {
                for (int k2 = key0; k2 < min(key0 + UNIT, key_end); k2 += 32) {
                    load_tile(k2, ta);
                    compute(k2, ta, later_step);
                }
            }
        }
        unit_sums();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            m_acc[nb] = m_run[nb];
            l_acc[nb] = l_run[nb];
#pragma unroll
            for (int db = 0; db < DB; ++db) o_acc[db][nb] = o[db][nb];
        }
    } else if constexpr (NW == 1) {
        // units in ascending order, each from a fresh state, merged into the partition's result as they end.  (A step's loads
        // are never left out, nor is one step's work between two others' loads: where they may be, the compiler no longer
        // knows how many are under way and waits for all of them.)
        auto end_unit = [&]() {
            unit_sums();
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                float m_new, ca, cb;
                merge_weights(m_acc[nb], m_run[nb], m_new, ca, cb);
                l_acc[nb] = merged(l_acc[nb], ca, l_run[nb], cb);
                m_acc[nb] = m_new;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[db][nb][e] = merged(o_acc[db][nb][e], ca, o[db][nb][e], cb);
            }
        };
        if constexpr (AHEAD) {
            int key0 = key_begin;
            for (; key0 + 32 < key_end; key0 += UNIT) {
                load_tile(key0 + 32, tb);
                compute(key0, ta, first_step);
                load_tile(key0 + UNIT, ta);
                compute(key0 + 32, tb, later_step);
                end_unit();
            }
            if (key0 < key_end) {          // a unit of one step
                compute(key0, ta, first_step);
                end_unit();
            }
        } else {
            for (int key0 = key_begin; key0 < key_end; key0 += UNIT) {
                load_tile(key0, ta);
                compute(key0, ta, first_step);
                if (key0 + 32 < key_end) {
                    load_tile(key0 + 32, ta);
                    compute(key0 + 32, ta, later_step);
                }
                end_unit();
            }
        }
    } else {
        // a unit a wave; the waves' results go through LDS and every wave merges a share of the elements,
        // each element through the same chain as above
        __shared__ float u_ml[UNITS][NB][16][2];
        __shared__ __attribute__((aligned(16))) float u_o[UNITS][NB][DB][WAVE][4];
        const int key0 = key_begin + wave * UNIT;
        begin_unit();
        if (key0 < key_end) {
            const bool more = key0 + 32 < key_end;
            if constexpr (!AHEAD) load_tile(key0, ta);
            compute(key0, ta, first_step);
            if (more) {
                if constexpr (!AHEAD) { load_tile(key0 + 32, ta); compute(key0 + 32, ta, later_step); }
                else compute(key0 + 32, tb, later_step);
            }
            unit_sums();
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (g == 0) { u_ml[wave][nb][n16][0] = m_run[nb]; u_ml[wave][nb][n16][1] = l_run[nb]; }
#pragma unroll
            for (int db = 0; db < DB; ++db) *(f32x4*)u_o[wave][nb][db][lane] = o[db][nb];
        }
        __syncthreads();
        // wave w finishes the channel blocks db = w, w + 4, ... of every column block
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int u = 0; u < UNITS; ++u) {
                const float mu = u_ml[u][nb][n16][0], lu = u_ml[u][nb][n16][1];
                float m_new, ca, cb;
                merge_weights(m_acc[nb], mu, m_new, ca, cb);
                l_acc[nb] = merged(l_acc[nb], ca, lu, cb);
                m_acc[nb] = m_new;
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    if (db % NW != wave) continue;
                    const f32x4 ou = *(const f32x4*)u_o[u][nb][db][lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o_acc[db][nb][e] = merged(o_acc[db][nb][e], ca, ou[e], cb);
                }
            }
        }
    }

    // ---- the partition's result per column
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (qrow[nb] < 0) continue;
        const long long slot = qrow[nb] * n_parts + part;
        if (g == 0 && wave == 0) { ws_ml[slot * 2] = m_acc[nb]; ws_ml[slot * 2 + 1] = l_acc[nb]; }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (NW > 1 && db % NW != wave) continue;
            const int dim = db * 16 + 4 * g;
            if (dim < hd) *(f32x4*)(ws_o + slot * hd + dim) = o_acc[db][nb];
        }
    }
}

// Merges the partitions of one (token, head) and writes the bfloat16 row:
//   M = max_p m_p;  w_p = exp(m_p - M);  out = (sum_p w_p o_p) / (sum_p w_p l_p),
// both sums over p in ascending order, so the result depends on the token's position only.
constexpr int COMBINE_MAX_PARTS = 2048;

// Up to 64 partitions: lane p keeps (m_p, l_p) in registers, weights are read out of its lane; no LDS.
// Same arithmetic as the general kernel below.  PER: channels a lane (head size / 64, rounded up);
// the partial outputs of BATCH partitions are asked for at once, so that a context of 16,384 positions
// with heads of 64 is one trip to memory (36 partitions of 256 rows: 7.5 -> 4.8 us).
template <int PER, int BATCH>
__global__ __launch_bounds__(WAVE) void attn_combine64_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                              bf16_t* __restrict__ out, const int* __restrict__ positions,
                                                              int H, int hd, int window, int n_parts, int part_keys,
                                                              const float* __restrict__ sinks) {
    const long long row = blockIdx.x;                      // token * H + head
    const int lane = threadIdx.x;
    const unsigned token = blockIdx.x / (unsigned)H;
    // a head's sink: a logit without key or value that counts once in the denominator (none: -inf, which adds 0)
    const float sink = sinks ? sinks[blockIdx.x - token * H] : -INFINITY;
    float m_l = -INFINITY, l_l = 0.f;
    if (lane < n_parts) {                                  // read before the position is known: rows exist for all partitions
        const float* ml = ws_ml + (row * n_parts + lane) * 2;
        m_l = ml[0];
        l_l = ml[1];
    }
    const int pos = positions[token];
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int p_lo = (unsigned)lo / (unsigned)part_keys, p_hi = (unsigned)pos / (unsigned)part_keys;
    const bool valid = lane >= p_lo && lane <= p_hi && l_l > 0.f;
    const float M = fmaxf(wave_max(valid ? m_l : -INFINITY), sink);
    const float w_l = valid ? __expf(m_l - M) : 0.f;
    const float wl_l = w_l * (valid ? l_l : 0.f);
    const buffer_t obuf = make_buffer(ws_o + row * n_parts * hd, n_parts * hd * 4);
    float acc[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) acc[j] = 0.f;
    float L = 0.f;                                         // both sums run over p in ascending order
    // The loads below do not wait for the position: rows of partitions the token does not have
    // exist too (unwritten); their weight is zero and they are skipped by a select, not a product.
    for (int i0 = 0; i0 < n_parts; i0 += BATCH) {
        float ov[BATCH][PER];
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int d = lane + j * WAVE;
                ov[u][j] = load_buffer_float(obuf, d < hd ? ((i0 + u) * hd + d) * 4 : NOWHERE, 0);     // (beyond the last partition: zero)
            }
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const float w = lane_of(w_l, i0 + u);
            L += lane_of(wl_l, i0 + u);
            if (w > 0.f) {
#pragma unroll
                for (int j = 0; j < PER; ++j) acc[j] = fmaf(w, ov[u][j], acc[j]);
            }
        }
    }
    if (sinks) L += __expf(sink - M);
    const float inv = 1.0f / L;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int d = lane + j * WAVE;
        if (d < hd) out[row * hd + d] = (bf16_t)(acc[j] * inv);
    }
}

// More than 64 partitions (contexts beyond 16,384 keys): the partitions are taken in groups of 64 by
// their absolute numbers (0..63, 64..127, ...); a wave sums a group in ascending order as above, the
// waves of the workgroup take the groups in turn, and the groups' sums are added in ascending order.
// The grouping is by absolute partition number, so the result still depends on the token's position only.
constexpr int COMBINE_WAVES = 8;
constexpr int COMBINE_GROUP = 64;
constexpr int COMBINE_MAX_GROUPS = COMBINE_MAX_PARTS / COMBINE_GROUP;

// NARROW: heads of up to 64 channels.  The maxima and sums are asked for with the position; when that is known a wave asks for
// all partial outputs of the group of its own number at once, as far as the token sees them, and takes the weights meanwhile: two
// trips to memory instead of six one after the other.  A wave with few of them (a short request beside a long one, a
// window) fetches them behind the weights, sixteen at a time, in less code.  94 registers: two workgroups a CU (one, with 144,
// takes half as long again where rows are many).  32 heads, the whole attention: 3 requests of 30,000 keys 51.1 -> 46.6 us, one of
// 30,000 beside 63 of 256 66.8 -> 60.4, 64 requests with a window of 1,024 and room for 30,000 65.5 -> 61.1 (everything asked for
// before the position, whatever the row: 46.9, 88.9 and 89.3).
template <bool NARROW>
__global__ __launch_bounds__(COMBINE_WAVES * WAVE) void attn_combine_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                                            bf16_t* __restrict__ out, const int* __restrict__ positions,
                                                                            int H, int hd, int window, int n_parts, int part_keys,
                                                                            const float* __restrict__ sinks) {
    constexpr int PER_THREAD = COMBINE_MAX_PARTS / (COMBINE_WAVES * WAVE);
    constexpr int PER = NARROW ? 1 : 4;                    // channels a lane, at most
    constexpr int AHEAD = NARROW ? COMBINE_GROUP : 1;
    constexpr int FEW = 16;                                // partitions a trip below
    __shared__ float wts[COMBINE_MAX_PARTS], wls[COMBINE_MAX_PARTS];
    __shared__ float grp_acc[COMBINE_MAX_GROUPS][NARROW ? WAVE : 256], grp_l[COMBINE_MAX_GROUPS];
    __shared__ float red[COMBINE_WAVES];
    const long long row = blockIdx.x;                      // token * H + head
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const unsigned token = blockIdx.x / (unsigned)H;
    const int pos = positions[token];
    const buffer_t mbuf = make_buffer(ws_ml + row * n_parts * 2, n_parts * 8);
    const buffer_t obuf = make_buffer(ws_o + row * n_parts * hd, n_parts * hd * 4);
    float m_p[PER_THREAD], l_p[PER_THREAD];                // of the partitions tid, tid + 512, ...; beyond the last: zero
#pragma unroll
    for (int k = 0; k < PER_THREAD; ++k) {
        m_p[k] = load_buffer_float(mbuf, (tid + k * COMBINE_WAVES * WAVE) * 8, 0);
        l_p[k] = load_buffer_float(mbuf, (tid + k * COMBINE_WAVES * WAVE) * 8 + 4, 0);
    }
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int p_lo = (unsigned)lo / (unsigned)part_keys, p_hi = (unsigned)pos / (unsigned)part_keys;          // the token's partitions, absolute numbers
    float first[AHEAD];                                    // the partial outputs of group `wave`
    const int first_lo = max(p_lo, wave * COMBINE_GROUP), first_hi = min(p_hi, wave * COMBINE_GROUP + COMBINE_GROUP - 1);
    const bool ahead = NARROW && first_hi - first_lo >= FEW;
    if (ahead) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int p = wave * COMBINE_GROUP + u;
            first[u] = load_buffer_float(obuf, p >= first_lo && p <= first_hi && lane < hd ? (p * hd + lane) * 4 : NOWHERE, 0);
        }
    }
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < PER_THREAD; ++k) {
        const int p = tid + k * COMBINE_WAVES * WAVE;
        if (p < p_lo || p > p_hi) l_p[k] = 0.f;
        M = fmaxf(M, l_p[k] > 0.f ? m_p[k] : -INFINITY);
    }
    M = wave_max(M);
    if (lane == 0) red[wave] = M;
    lds_barrier();
#pragma unroll
    for (int w = 0; w < COMBINE_WAVES; ++w) M = fmaxf(M, red[w]);
    const float sink = sinks ? sinks[blockIdx.x - token * H] : -INFINITY;
    M = fmaxf(M, sink);
#pragma unroll
    for (int k = 0; k < PER_THREAD; ++k) {
        const int p = tid + k * COMBINE_WAVES * WAVE;
        const float w = l_p[k] > 0.f ? __expf(m_p[k] - M) : 0.f;
        wts[p] = w;
        wls[p] = w * (l_p[k] > 0.f ? l_p[k] : 0.f);
    }
    lds_barrier();
    const int g_lo = p_lo / COMBINE_GROUP, g_hi = p_hi / COMBINE_GROUP;
    const int per = (hd + WAVE - 1) / WAVE;                // channels a lane
    const float* o = ws_o + row * n_parts * hd;
    for (int grp = wave; grp <= g_hi; grp += COMBINE_WAVES) {
        if (grp < g_lo) continue;
        const int a = max(p_lo, grp * COMBINE_GROUP), b = min(p_hi, grp * COMBINE_GROUP + COMBINE_GROUP - 1);
        float acc[PER] = {};
        float L = 0.f;
        if (ahead && grp == wave) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int p = grp * COMBINE_GROUP + u;
                if (p >= a && p <= b) {
                    const float w = wts[p];
                    L += wls[p];
                    if (w > 0.f) acc[0] = fmaf(w, first[u], acc[0]);       // a partition without weight may hold anything
                }
            }
        } else {
            // the partial outputs of sixteen partitions are asked for together; the sums run in ascending order
            for (int i0 = a; i0 <= b; i0 += 16) {
                float ov[16][PER];
#pragma unroll
                for (int u = 0; u < 16; ++u)
#pragma unroll
                    for (int j = 0; j < PER; ++j) {
                        const int d = lane + j * WAVE;
                        ov[u][j] = (j < per && i0 + u <= b && d < hd) ? o[(long long)(i0 + u) * hd + d] : 0.f;
                    }
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    if (i0 + u <= b) {
                        const float w = wts[i0 + u];
                        L += wls[i0 + u];
                        if (w > 0.f) {                     // a partition without weight may hold anything
#pragma unroll
                            for (int j = 0; j < PER; ++j) acc[j] = fmaf(w, ov[u][j], acc[j]);
                        }
                    }
            }
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int d = lane + j * WAVE;
            if (d < hd) grp_acc[grp][d] = acc[j];
        }
        if (lane == 0) grp_l[grp] = L;
    }
    __syncthreads();
    if (wave == 0) {
        float acc[PER] = {};
        float L = 0.f;
        for (int grp = g_lo; grp <= g_hi; ++grp) {
            L += grp_l[grp];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int d = lane + j * WAVE;
                if (d < hd) acc[j] += grp_acc[grp][d];
            }
        }
        if (sinks) L += __expf(sink - M);
        const float inv = 1.0f / L;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int d = lane + j * WAVE;
            if (d < hd) out[row * hd + d] = (bf16_t)(acc[j] * inv);
        }
    }
}

// Workgroups of four waves where one wave a partition would leave most of the chip idle (a step of a
// few single tokens); the result is the same bit for bit.
int few_waves = 2048;
// From how many workgroups on the kv head is the fastest-changing part of a workgroup's number: decode steps with it / without:
// 8 requests of 20,000 keys 955 / 985 us, 3 of 30,001 838 / 848, one of 20,000 (632 workgroups) 699 / 706; heads of 128, 32 requests
// of 4,000 95 / 101 us an operation.  With fewer workgroups there is nothing in it.
int kv_fast_waves = 512;
// From how many workgroups on the keys of heads of up to 64 channels go through LDS (STAGE_K of the kernel): 3 requests of
// 30,001 keys (2,832) 870 -> 848 us a step, 12 of 8,000 913 -> 886, 8 of 3,800 (960) 736 -> 722, one of 20,000 (632) 709 -> 706.
int stage_k_waves = 512;

// Eight waves a workgroup that take all partitions of a column block and write the finished rows, no merge after them: for
// launches of few partitions with work for the chip all the same.  A workgroup's share of a CU must be most of what there is: with
// more than four partitions (a launch knows the room for keys, not the keys) the blocks have to fill a round of 256, and the last
// round where they are more; with up to four, where the merge is the larger part, a quarter of a round is enough, and a second
// round that is half empty loses at the most keys of the room what it gains at the least.  And the more columns a block has, whose
// sums all go through LDS, the less is gained.
// 32 heads on 8, kernel and merge against the one kernel, us, at 200, 600 and 1,000 keys of room for 1,024:
//   64 blocks 9.8 / 6.5, 9.6 / 9.2 and 10.6 / 12.1; 128 10.8 / 7.0, 11.2 / 9.6 and 12.5 / 12.8; 256 12.1 / 7.5, 13.7 / 11.5 and 17.5 / 16.1;
//   384 15.0 / 11.9, 18.0 / 18.6 and 23.2 / 26.9; 512 16.3 / 12.8, 22.6 / 21.2 and 28.2 / 29.4; 576 19.4 / 16.8, 26.3 / 26.8 and 32.8 / 37.7;
// at 1,100 and 2,000 of room for 2,048:
//   128 13.5 / 14.1 and 16.7 / 21.3; 160 15.9 / 14.5 and 20.4 / 21.4; 192 17.6 / 15.3 and 22.4 / 22.7; 256 21.2 / 17.3 and 27.4 / 26.1;
//   384 29.3 / 27.3 and 38.1 / 44.1; 512 32.2 / 31.4 and 49.3 / 48.7; 576 37.8 / 39.7 and 57.1 / 63.0; 768 46.5 / 45.2 and 72.2 / 71.9.
// 64 heads on 8: room for 1,024, 384 blocks 15.6 / 12.9, 19.8 / 21.2 and 24.6 / 29.9, 512 17.5 / 13.9, 24.2 / 23.4 and 29.7 / 32.6; for 2,048, 256
// 22.5 / 18.7 and 28.2 / 28.5, 512 34.7 / 34.7 and 52.5 / 53.0.  128 on 8: for 1,024, 128 11.6 / 8.2, 12.3 / 13.1 and 13.5 / 17.8, 256 13.5 / 9.1,
// 16.2 / 15.1 and 19.8 / 20.9, 512 19.1 / 16.6, 26.6 / 27.9 and 32.7 / 39.2; for 2,048, 256 24.2 / 22.1 and 30.8 / 34.0.  Whole decode steps of 16
// layers of which 6 attend: 24 requests of 1,100 919 / 901, 32 of 1,650 995 / 981, 56 of 1,650 1,203 / 1,198, 48 of 100 1,007 / 987, but 48 of 1,650
// 1,125 / 1,147 and 36 1,076 / 1,119.
constexpr int WHOLE_WAVES = 8;
bool takes_whole(long long blocks, int n_parts, int columns) {
    constexpr int ROUND = 256, MOST_OF_IT = 176;
    const bool filled = (blocks - 1) % ROUND + 1 >= MOST_OF_IT;
    if (n_parts > 8) return false;
    if (n_parts > 4) return filled && (columns <= 4 || (columns <= 8 && blocks <= ROUND));
    if (columns <= 4) return blocks >= ROUND / 4 && (blocks <= 2 * ROUND || filled);
    if (columns <= 8) return (blocks >= ROUND / 4 && blocks <= ROUND) || (filled && blocks <= 2 * ROUND);
    return filled && blocks <= ROUND;
}

template <bool FUSED, bool STREAM_V = true>
int launch_whole(dim3 grid, hipStream_t stream, const bf16_t* q, bf16_t* kc, bf16_t* vc, const int* bt, int max_blocks, const int2* blk,
                 const int4* req_info, int H, int Hkv, int hd, int ps, int window, float scale, int n_parts, const FusedQKV& fq,
                 bf16_t* out, const float* sinks) {
    if constexpr (STREAM_V) {
        if (ps > 16)
            return launch_whole<FUSED, false>(grid, stream, q, kc, vc, bt, max_blocks, blk, req_info, H, Hkv, hd, ps, window, scale, n_parts,
                                              fq, out, sinks);
    }
    auto kern = attn_partition_kernel<64, 1, WHOLE_WAVES, FUSED, STREAM_V, true>;
    const int lds = (WHOLE_WAVES + n_parts) * (FUSED ? H / Hkv : 16) * (64 + 2) * 4;       // at most 67,584 bytes
    static bool set = false;
    if (!set) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * WHOLE_WAVES * 16 * (64 + 2) * 4) != hipSuccess) return -1;
        set = true;
    }
    hipLaunchKernelGGL(kern, grid, dim3(WHOLE_WAVES * WAVE), lds, stream, q, kc, vc, nullptr, nullptr, bt, max_blocks, blk, req_info, H, Hkv,
                       hd, ps, window, scale, n_parts, fq, 0, out, sinks);
    return launch_status();
}

template <int HDP, int NB, bool FUSED, bool STREAM_V = true>
void launch_partition(dim3 grid, hipStream_t stream, const bf16_t* q, bf16_t* kc, bf16_t* vc, float* ws_o,
                      float* ws_ml, const int* bt, int max_blocks, const int2* blk, const int4* req_info,
                      int H, int Hkv, int hd, int ps, int window, float scale, int n_parts, const FusedQKV& fq) {
    if constexpr (STREAM_V) {
        if (ps > 16) {
            launch_partition<HDP, NB, FUSED, false>(grid, stream, q, kc, vc, ws_o, ws_ml, bt, max_blocks, blk, req_info, H, Hkv, hd,
                                                    ps, window, scale, n_parts, fq);
            return;
        }
    }
    const long long waves = (long long)grid.x * grid.y * grid.z;
    const int kv_fast = waves >= kv_fast_waves ? 1 : 0;
    if (kv_fast) grid = dim3(grid.x * grid.z, grid.y, 1);
    if constexpr (HDP * NB <= 128) {
        // the fused form prepares its queries in every wave, and four waves pay for that four times: one of 30,000 keys (944
        // workgroups) 758 us a step with four, 731 with one; one of 8,000 (256) 653 and 662
        if (waves < (FUSED ? few_waves / 4 : few_waves)) {
            hipLaunchKernelGGL((attn_partition_kernel<HDP, NB, UNITS, FUSED, STREAM_V>), grid, dim3(UNITS * WAVE), 0, stream, q, kc, vc, ws_o,
                               ws_ml, bt, max_blocks, blk, req_info, H, Hkv, hd, ps, window, scale, n_parts, fq, kv_fast, nullptr, nullptr);
            return;
        }
    }
    if constexpr (HDP == 64 && HDP * NB <= 256) {
        if (waves >= stage_k_waves) {
            hipLaunchKernelGGL((attn_partition_kernel<HDP, NB, 1, FUSED, STREAM_V, true>), grid, dim3(WAVE), 0, stream, q, kc, vc, ws_o,
                               ws_ml, bt, max_blocks, blk, req_info, H, Hkv, hd, ps, window, scale, n_parts, fq, kv_fast, nullptr, nullptr);
            return;
        }
    }
    hipLaunchKernelGGL((attn_partition_kernel<HDP, NB, 1, FUSED, STREAM_V>), grid, dim3(WAVE), 0, stream, q, kc, vc, ws_o, ws_ml, bt,
                       max_blocks, blk, req_info, H, Hkv, hd, ps, window, scale, n_parts, fq, kv_fast, nullptr, nullptr);
}
}  // namespace

// Merges, for every (token, head) of n_tokens tokens, the partial results of its partitions of
// part_keys keys each.
static int launch_merge(const float* ws_o, const float* ws_ml, bf16_t* out, const int* positions, int n_tokens, int H, int hd,
                 int window, int n_parts, int part_keys, hipStream_t stream, const float* sinks = nullptr) {
    const dim3 grid((unsigned)((long long)n_tokens * H));
    if (n_parts <= WAVE) {
#define COMBINE(PER, BATCH) hipLaunchKernelGGL((attn_combine64_kernel<PER, BATCH>), grid, dim3(WAVE), 0, stream, ws_o, ws_ml, out, \
                                               positions, H, hd, window, n_parts, part_keys, sinks)
        if (hd <= 64) { if (n_parts <= 8) COMBINE(1, 8); else if (n_parts <= 16) COMBINE(1, 16); else if (n_parts <= 32) COMBINE(1, 32); else COMBINE(1, 64); }
        else if (hd <= 128) { if (n_parts <= 8) COMBINE(2, 8); else COMBINE(2, 16); }
        else COMBINE(4, 8);
#undef COMBINE
    } else {
#define COMBINE_WIDE(NARROW) hipLaunchKernelGGL(attn_combine_kernel<NARROW>, grid, dim3(COMBINE_WAVES * WAVE), 0, stream, ws_o, ws_ml, \
                                                out, positions, H, hd, window, n_parts, part_keys, sinks)
        if (hd <= WAVE) COMBINE_WIDE(true); else COMBINE_WIDE(false);
#undef COMBINE_WIDE
    }
    return launch_status();
}

// Query blocks are listed by the host: block b holds the columns blk[b].y .. +16*nb-1 of request
// blk[b].x (a request's columns are numbered (token - its first token) * G + head within the kv
// group); blk == null: block b is request b from column 0 (every request fits one block).
// req_info [R]: (first token of the request in the step, its tokens, position of the first, -).
// positions [n_tokens]: every token's position (read by the merge).
// ws_o: float32 [n_tokens * H * n_parts * hd], ws_ml: float32 [n_tokens * H * n_parts * 2].
// n_parts >= ceil((largest position + 1) / 256).  nb: 1, 2 or 4 column blocks a wave.
static int launch_attention(const void* q, const void* k_cache, const void* v_cache, void* out,
                            float* ws_o, float* ws_ml, const int* block_table, int max_blocks,
                            const int* blk, int n_qblocks, int nb, const int* req_info, const int* positions,
                            int n_tokens, int H, int Hkv, int hd, int page_size, int window, float scale,
                            int n_parts, hipStream_t stream, const float* sinks = nullptr, const float* slopes = nullptr) {
    if (n_tokens <= 0 || n_qblocks <= 0) return 0;
    if (hd > 256 || hd % 8 != 0 || page_size % 16 != 0 || Hkv <= 0 || H % Hkv != 0 || n_parts < 1) return -2;
    if (Hkv > 65535 || n_qblocks > 65535 || n_parts > COMBINE_MAX_PARTS) return -2;
    const bf16_t* Q = (const bf16_t*)q;
    bf16_t* K = (bf16_t*)k_cache;                                        // read only without the fused form
    bf16_t* V = (bf16_t*)v_cache;
    dim3 grid(n_parts, n_qblocks, Hkv);
    FusedQKV plain_form;
    plain_form.slopes = slopes;
    plain_form.group = H / Hkv;
    // (as many blocks as tokens: a token a block, of up to eight columns)
    if (nb == 1 && hd > 32 && hd <= 64 && takes_whole((long long)n_qblocks * Hkv, n_parts, n_qblocks == n_tokens ? H / Hkv : 16))
        return launch_whole<false>(dim3(1, n_qblocks, Hkv), stream, Q, K, V, block_table, max_blocks, (const int2*)blk, (const int4*)req_info,
                                   H, Hkv, hd, page_size, window, scale, n_parts, plain_form, (bf16_t*)out, sinks);
#define GO(HDP, NB) launch_partition<HDP, NB, false>(grid, stream, Q, K, V, ws_o, ws_ml, block_table, max_blocks, (const int2*)blk, \
                                                     (const int4*)req_info, H, Hkv, hd, page_size, window, scale, n_parts, plain_form)
#define BY_NB(HDP) do { if (nb == 1) GO(HDP, 1); else if (nb == 2) GO(HDP, 2); else if (nb == 4) GO(HDP, 4); else return -2; } while (0)
    if (hd <= 32) BY_NB(32);
    else if (hd <= 64) BY_NB(64);
    else if (hd <= 96) BY_NB(96);
    else if (hd <= 128) BY_NB(128);
    else { if (nb == 1) GO(256, 1); else if (nb == 2) GO(256, 2); else return -2; }
#undef BY_NB
#undef GO
    int rc = launch_status();
    if (rc) return rc;
    return launch_merge((const float*)ws_o, (const float*)ws_ml, (bf16_t*)out, positions, n_tokens, H, hd, window, n_parts, PART,
                        stream, sinks);
}

// The same with a sink per head and a distance slope per head (each float32 [H], or null): slopes[h] * (position - key)
// is taken off head h's scaled scores.
TUFF_EXPORT int tuff_attention_mfma_biased(const void* q, const void* k_cache, const void* v_cache, void* out,
                                           float* ws_o, float* ws_ml, const int* block_table, int max_blocks,
                                           const int* blk, int n_qblocks, int nb, const int* req_info, const int* positions,
                                           int n_tokens, int H, int Hkv, int hd, int page_size, int window, float scale,
                                           int n_parts, const float* sinks, const float* slopes, hipStream_t stream) {
    return launch_attention(q, k_cache, v_cache, out, ws_o, ws_ml, block_table, max_blocks, blk, n_qblocks, nb, req_info,
                            positions, n_tokens, H, Hkv, hd, page_size, window, scale, n_parts, stream, sinks, slopes);
}

// The number of lanes of a wave that fetch page numbers for partition `part` with pages of page_size
// positions (what the kernel computes; host arithmetic, for checks).
TUFF_EXPORT int tuff_attention_partition_pages(int part, int page_size) {
    if (part < 0 || page_size <= 0 || (long long)part * PART + PART > 0x7fffffffll) return -2;
    return partition_pages(part * PART, page_size);
}

// Below how many workgroups a step's partitions get four waves each (0: never).  For measurements and
// tests; the result of the attention does not depend on it.  Returns the value before.
TUFF_EXPORT int tuff_attention_few_waves(int n) {
    const int old = few_waves;
    if (n >= 0) few_waves = n;
    return old;
}

// From how many workgroups on the kv head changes fastest in the order of the workgroups.  For
// measurements and tests; the result does not depend on it.  Returns the value before.
// From how many workgroups on keys are asked for in whole lines and go through LDS.  For measurements and tests; the
// result does not depend on it.  Returns the value before.
TUFF_EXPORT int tuff_attention_stage_k_waves(int n) {
    const int old = stage_k_waves;
    if (n >= 0) stage_k_waves = n;
    return old;
}

TUFF_EXPORT int tuff_attention_takes_whole(long long blocks, int n_parts, int columns) { return takes_whole(blocks, n_parts, columns); }

TUFF_EXPORT int tuff_attention_kv_fast_waves(int n) {
    const int old = kv_fast_waves;
    if (n >= 0) kv_fast_waves = n;
    return old;
}

TUFF_EXPORT int tuff_attention_mfma(const void* q, const void* k_cache, const void* v_cache, void* out,
                                    float* ws_o, float* ws_ml, const int* block_table, int max_blocks,
                                    const int* blk, int n_qblocks, int nb, const int* req_info, const int* positions,
                                    int n_tokens, int H, int Hkv, int hd, int page_size, int window, float scale,
                                    int n_parts, hipStream_t stream) {
    return launch_attention(q, k_cache, v_cache, out, ws_o, ws_ml, block_table, max_blocks, blk, n_qblocks, nb, req_info,
                            positions, n_tokens, H, Hkv, hd, page_size, window, scale, n_parts, stream);
}

// The same with a sink per head (sinks float32 [H], or null): a logit that has neither key nor value and
// counts once, unscaled, in the softmax's denominator.  It enters where a row's partitions are merged.
TUFF_EXPORT int tuff_attention_mfma_sinks(const void* q, const void* k_cache, const void* v_cache, void* out,
                                          float* ws_o, float* ws_ml, const int* block_table, int max_blocks,
                                          const int* blk, int n_qblocks, int nb, const int* req_info, const int* positions,
                                          int n_tokens, int H, int Hkv, int hd, int page_size, int window, float scale,
                                          int n_parts, const float* sinks, hipStream_t stream) {
    return launch_attention(q, k_cache, v_cache, out, ws_o, ws_ml, block_table, max_blocks, blk, n_qblocks, nb, req_info,
                            positions, n_tokens, H, Hkv, hd, page_size, window, scale, n_parts, stream, sinks);
}

// A step of single tokens (request r's token is row r) over heads of 64 channels, from the projected
// rows qkv [n_tokens, (H + 2 Hkv) * 64]: per-head RMSNorm of q and k (weights [64] of type norm_dt, or
// null), half-split rotation over the whole head by inv_freq [32] (angles [n_angles][2][32]: the
// cosines and sines of the first n_angles positions as tuff_rope_table makes them, or null), the token's key and value written
// to the cache at slot_mapping[r] (null: the cache is only read), attention, merge.  The query heads
// of a kv head must fit one block of sixteen columns (H / Hkv <= 16).
TUFF_EXPORT int tuff_attention_decode_fused(const void* qkv, void* k_cache, void* v_cache, void* out,
                                            float* ws_o, float* ws_ml, const int* block_table, int max_blocks,
                                            const int* req_info, const int* positions, const int* slot_mapping,
                                            const void* q_norm_w, const void* k_norm_w, int norm_dt, float eps,
                                            const float* inv_freq, const float* angles, int n_angles,
                                            int n_tokens, int H, int Hkv, int page_size,
                                            int window, float scale, int n_parts, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (page_size % 16 != 0 || Hkv <= 0 || H % Hkv != 0 || H / Hkv > 16 || n_parts < 1 || !inv_freq) return -2;
    if ((q_norm_w == nullptr) != (k_norm_w == nullptr)) return -2;
    if (Hkv > 65535 || n_tokens > 65535 || n_parts > COMBINE_MAX_PARTS) return -2;
    FusedQKV fq;
    fq.q_norm_w = q_norm_w; fq.k_norm_w = k_norm_w; fq.norm_dt = norm_dt; fq.eps = eps;
    fq.inv_freq = inv_freq; fq.slot_mapping = slot_mapping;
    fq.angles = angles; fq.n_angles = angles ? n_angles : 0;
    fq.group = H / Hkv;
    if (takes_whole((long long)n_tokens * Hkv, n_parts, H / Hkv))
        return launch_whole<true>(dim3(1, n_tokens, Hkv), stream, (const bf16_t*)qkv, (bf16_t*)k_cache, (bf16_t*)v_cache, block_table,
                                  max_blocks, nullptr, (const int4*)req_info, H, Hkv, 64, page_size, window, scale, n_parts, fq,
                                  (bf16_t*)out, nullptr);
    launch_partition<64, 1, true>(dim3(n_parts, n_tokens, Hkv), stream, (const bf16_t*)qkv, (bf16_t*)k_cache, (bf16_t*)v_cache,
                                  ws_o, ws_ml, block_table, max_blocks, nullptr, (const int4*)req_info, H, Hkv, 64, page_size,
                                  window, scale, n_parts, fq);
    int rc = launch_status();
    if (rc) return rc;
    return launch_merge((const float*)ws_o, (const float*)ws_ml, (bf16_t*)out, positions, n_tokens, H, 64, window, n_parts, PART,
                        stream);
}

// The merge alone, for partial results that another kernel left in the same layout (ws_o
// [tokens * H * n_parts * hd], ws_ml [tokens * H * n_parts * 2] = (reference exponent, sum); partition
// p of a row holds the keys p * part_keys .. (p + 1) * part_keys - 1).
TUFF_EXPORT int tuff_attention_merge(const float* ws_o, const float* ws_ml, void* out, const int* positions, int n_tokens,
                                     int H, int hd, int window, int n_parts, int part_keys, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (hd > 256 || n_parts < 1 || n_parts > COMBINE_MAX_PARTS || part_keys < 1) return -2;
    return launch_merge(ws_o, ws_ml, (bf16_t*)out, positions, n_tokens, H, hd, window, n_parts, part_keys, stream);
}

// The same with a sink per head (sinks float32 [H], or null): exp(sink) joins every row's denominator.
TUFF_EXPORT int tuff_attention_merge_sinks(const float* ws_o, const float* ws_ml, void* out, const int* positions, int n_tokens,
                                           int H, int hd, int window, int n_parts, int part_keys, const float* sinks,
                                           hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (hd > 256 || n_parts < 1 || n_parts > COMBINE_MAX_PARTS || part_keys < 1) return -2;
    return launch_merge(ws_o, ws_ml, (bf16_t*)out, positions, n_tokens, H, hd, window, n_parts, part_keys, stream, sinks);
}

// ------------------------------------------------- the same attention without an allocation
// tuff_attention_mfma_static: tuff_attention_mfma with the partitions' partial results kept in an
// array of this library instead of a work space the caller brings, for callers that cannot
// allocate (a HIP graph under capture, a serving loop that must not call the allocator).  It calls
// no hipMalloc, hipFree or allocating library routine.
//
// The array is STATIC_SCRATCH_FLOATS floats (16 MiB) of device memory on every GPU the library is
// loaded on, held until the process ends.  A call needs n_tokens * H * n_parts * (hd + 2) floats
// (rounded up to 64 for the first of its two parts) and is refused with TUFF_STATIC_TOO_LARGE
// beyond that.  All calls on one GPU share that GPU's array: it keeps the last call's contents
// (nothing has to start at zero: a row of a partition that a token does not have is never used),
// and two calls that overlap on one GPU, on different streams or from different threads, race.
//
// In host code the array's name stands for the symbol, not for device memory; the address on the
// current device comes from hipGetSymbolAddress, once per device, and only that pointer is handed
// to the kernels.
constexpr long long STATIC_SCRATCH_FLOATS = 4ll << 20;
constexpr int STATIC_MAX_DEVICES = 64;
enum : int { TUFF_STATIC_TOO_LARGE = -7, TUFF_STATIC_NO_DEVICE = -8 };

static __device__ __align__(256) float static_scratch[STATIC_SCRATCH_FLOATS];
static float* static_scratch_ptr[STATIC_MAX_DEVICES];      // per device; written once, under the lock

static std::mutex static_scratch_lock;

// The array's address on the current device; looked up at the first call on that device.
static int static_scratch_of_current_device(float** ptr) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= STATIC_MAX_DEVICES) return TUFF_STATIC_NO_DEVICE;
    std::lock_guard<std::mutex> guard(static_scratch_lock);
    if (!static_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(static_scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return TUFF_STATIC_NO_DEVICE;
        static_scratch_ptr[dev] = (float*)p;
    }
    *ptr = static_scratch_ptr[dev];
    return 0;
}

// Looks the array up on the current device, so that the first attention call there does nothing
// but launch.  Returns 0, or a HIP error code.
TUFF_EXPORT int tuff_attention_static_setup(void) {
    float* p = nullptr;
    return static_scratch_of_current_device(&p);
}

// Floats of the static array a call of these sizes needs, and (*capacity) how many there are.
TUFF_EXPORT long long tuff_attention_static_floats(int n_tokens, int H, int hd, int n_parts, long long* capacity) {
    if (capacity) *capacity = STATIC_SCRATCH_FLOATS;
    const long long rows = (long long)n_tokens * H * n_parts;
    return (rows * hd + 63) / 64 * 64 + rows * 2;
}

TUFF_EXPORT int tuff_attention_mfma_static(const void* q, const void* k_cache, const void* v_cache, void* out,
                                           const int* block_table, int max_blocks,
                                           const int* blk, int n_qblocks, int nb, const int* req_info, const int* positions,
                                           int n_tokens, int H, int Hkv, int hd, int page_size, int window, float scale,
                                           int n_parts, hipStream_t stream) {
    if (n_tokens <= 0 || n_qblocks <= 0) return 0;
    if (H <= 0 || hd <= 0 || n_parts < 1) return -2;
    if (tuff_attention_static_floats(n_tokens, H, hd, n_parts, nullptr) > STATIC_SCRATCH_FLOATS) return TUFF_STATIC_TOO_LARGE;
    float* base = nullptr;
    const int rc = static_scratch_of_current_device(&base);
    if (rc) return rc;
    const long long rows = (long long)n_tokens * H * n_parts;
    float* ws_o = base;
    float* ws_ml = base + (rows * hd + 63) / 64 * 64;
    return launch_attention(q, k_cache, v_cache, out, ws_o, ws_ml, block_table, max_blocks, blk, n_qblocks, nb, req_info,
                            positions, n_tokens, H, Hkv, hd, page_size, window, scale, n_parts, stream);
}
