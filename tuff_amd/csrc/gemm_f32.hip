// True float32 matrix product  Y[M,N] (=|+=) X[M,K] * W[N,K]^T.
//
// Every output element is one chain  acc = fma(x[m,k], w[n,k], acc)  over k = 0..K-1
// in ascending order, whatever kernel or tile it falls into, so a row of Y does not depend
// on how many other rows were in the call.  No reduced precision.
//
//  * chain    an inner size that is a multiple of 32: the chain on the matrix cores.
//    v_mfma_f32_16x16x4_f32 adds its four products to an element one after the other, each fused and
//    rounded to float32, in ascending order of the lane group that brings them, so with k = 4 i + group
//    in instruction i an element is the same chain, bit for bit, denormal numbers included
//    (test_gemm_f32_matrix_cores compares the two kernels).
//  * general  other inner sizes, or operands off a 16-byte border: plain FMAs.
#include "common.h"

namespace {
// ------------------------------------------------------------------------------------------ general
constexpr int BM = 64, BN = 64, BK = 16, TM = 4, TN = 4, NT = 256;

template <bool ACCUM>
__global__ __launch_bounds__(NT) void gemm_f32_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                      float* __restrict__ Y, int M, int N, int K) {
    __shared__ float Xs[BK][BM + 4];
    __shared__ float Ws[BK][BN + 4];
    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
        for (int i = 0; i < (BM * BK) / NT; ++i) {
            const int idx = tid + i * NT;
            const int row = idx / BK, kk = idx % BK;
            const int gm = m0 + row, gn = n0 + row, gk = k0 + kk;
            Xs[kk][row] = (gm < M && gk < K) ? X[(long long)gm * K + gk] : 0.f;
            Ws[kk][row] = (gn < N && gk < K) ? W[(long long)gn * K + gk] : 0.f;
        }
        __syncthreads();
        const int kmax = min(BK, K - k0);      // zero padding would be harmless; skip it anyway
        for (int kk = 0; kk < kmax; ++kk) {
            float a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = Xs[kk][ty * TM + i];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = Ws[kk][tx * TN + j];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int gm = m0 + ty * TM + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int gn = n0 + tx * TN + j;
            if (gn >= N) continue;
            float* y = Y + (long long)gm * N + gn;
            if (ACCUM) *y = *y + acc[i][j]; else *y = acc[i][j];
        }
    }
}

// -------------------------------------------------------------------------------------------- chain
// A block of Y of 2 x 2 waves, T x T tiles of 16x16 each.  K is walked in steps of 32, which go from memory
// straight into LDS, STAGES buffers: the operands of STAGES - 1 steps are under way.  A step
// of a row is 128 bytes, eight pieces of 16; piece p of row r lies at position p ^ (r % 8), so the rows a fragment read
// touches spread over the banks.  A wave's load instruction fills 1 KB, eight rows.  For instruction i of a step a lane
// (row r16 = lane % 16, group g = lane / 16) reads element g of piece i of its row: k = 4 i + g.
//
// More than 16 rows: blocks of 64x64 or, where those leave CUs idle, of 32x32; see block_cycles.  What bounds it: a matrix
// instruction takes 32 cycles (157 TFLOP/s); 500 rows, 16,384 x 2,048: 283 us, 119 TFLOP/s, the general kernel 577; 2,048 x
// 8,192: 160 us against 1,480.
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int STEP = 32;

constexpr int WAVES = 2;

// SWIGLU, in all three kernels on whole chains: W holds N / 2 gate rows and then as many up rows, a block takes as many of each,
// and of the two chains of a column, which lie in one lane or in two of one wave, swiglu_value leaves Y [M, N / 2].  As a
// kernel of its own it wrote and read [M, N] once more.  Two kernels / one, us: 16,384 x 2,048 of 4 rows 31.2 and 29.6, 39 46.7 and
// 43.9, 500 286.1 and 281.9; 13,824 x 1,536 20.0 and 18.1, 35.8 and 33.8, 193.8 and 186.2; 2,048 x 512 7.0 and 5.1, 8.3 and
// 6.6, 17.8 and 13.9.
__device__ __forceinline__ float swiglu_value(float gate, float up) { return gate / (1.0f + expf(-gate)) * up; }

template <int T, int STAGES, bool SWIGLU>
__global__ __launch_bounds__(WAVES * WAVES * WAVE) void gemm_f32_chain_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                                              float* __restrict__ Y, int M, int N, int K, int accumulate) {
    constexpr int SIDE = 16 * T * WAVES;                  // rows and columns of the block
    constexpr int IN = SIDE / 8 / (WAVES * WAVES);        // load instructions a wave issues a step, for X and for W each
    static_assert(SIDE % (8 * WAVES * WAVES) == 0 && 2 * IN * (STAGES - 2) < 64, "whole instructions, and a count that s_waitcnt can hold");
    extern __shared__ __attribute__((aligned(16))) float tiles[];      // [STAGES][SIDE * STEP] of X, then of W
    float* Xs = tiles;
    float* Ws = tiles + STAGES * SIDE * STEP;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wm = (wave / WAVES) * (16 * T), wn = (wave % WAVES) * (16 * T);
    const int r16 = lane % 16, g = lane / 16;
    const long long m0 = (long long)blockIdx.y * SIDE, n0 = (long long)blockIdx.x * SIDE;
    const int last_m = (int)min((long long)SIDE - 1, (long long)M - 1 - m0);
    // SWIGLU: half the block's rows of W are gate rows, tile by tile (T = 2) or eight by eight, and their up rows follow them
    constexpr int RUN = T == 2 ? 16 : 8;
    const long long h0 = n0 / 2;
    const int last_n = SWIGLU ? (int)min((long long)SIDE / 2 - 1, (long long)N / 2 - 1 - h0) : (int)min((long long)SIDE - 1, (long long)N - 1 - n0);
    // (rows beyond the matrix read its last row instead: their results are never stored)
    int offx[IN], offw[IN];                               // bytes from the block's first row
#pragma unroll
    for (int i = 0; i < IN; ++i) {
        const int row = (wave * IN + i) * 8 + lane / 8, piece = (lane % 8) ^ (lane / 8);
        offx[i] = (min(row, last_m) * K + piece * 4) * 4;
        const int up = SWIGLU && row / RUN % 2 ? N / 2 : 0;
        offw[i] = ((up + min(SWIGLU ? row / (2 * RUN) * RUN + row % RUN : row, last_n)) * K + piece * 4) * 4;
    }
    const buffer_t xbuf = make_buffer(X + m0 * K, (last_m + 1) * K * 4);
    const buffer_t wbuf = make_buffer(W + (SWIGLU ? h0 : n0) * K, ((SWIGLU ? N / 2 : 0) + last_n + 1) * K * 4);
    const int steps = K / STEP;
    auto issue = [&](int buf, int s) {
#pragma unroll
        for (int i = 0; i < IN; ++i) load_to_lds(xbuf, Xs + buf * SIDE * STEP + (wave * IN + i) * 256, offx[i], s * (STEP * 4));
#pragma unroll
        for (int i = 0; i < IN; ++i) load_to_lds(wbuf, Ws + buf * SIDE * STEP + (wave * IN + i) * 256, offw[i], s * (STEP * 4));
    };
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    f32x4 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = z;
    // The operands of half a step (four instructions) are read into one of two register sets while the other set is
    // multiplied, also across the barrier between two steps.
    float x[2][4][T], w[2][4][T];
    int at[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) at[i] = r16 * STEP + ((i ^ (r16 % 8)) * 4 + g);
    auto read_half = [&](int buf, auto half) {
        constexpr int h = decltype(half)::value;
        const float* xb = Xs + buf * SIDE * STEP + wm * STEP;
        const float* wb = Ws + buf * SIDE * STEP + wn * STEP;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < T; ++t) {
                x[h][i][t] = xb[at[h * 4 + i] + t * 16 * STEP];
                w[h][i][t] = wb[at[h * 4 + i] + t * 16 * STEP];
            }
    };
    auto multiply = [&](auto half) {
        constexpr int h = decltype(half)::value;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j) acc[i][j] = mfma_f32(w[h][e][j], x[h][e][i], acc[i][j]);
    };
    // asks the instruction scheduler to spread the reads of half a step among the matrix instructions of the other
    auto spread = [&]() {
        static_for<4>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * T, 0);     // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, T * T, 0);     // matrix instructions
        });
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t) x[1][i][t] = w[1][i][t] = 0.f;
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st)
        if (st < steps) issue(st, st);
    auto products = [&](int buf) {
        read_half(buf, H0());
        multiply(H1());                                   // of the step before (products of zeros at first)
        spread();
        read_half(buf, H1());
        multiply(H0());
        spread();
    };
    // All loads but those of the steps after this one have landed; the barrier then says so of every wave's, and that nobody
    // reads the buffer that the next loads go into.  (Two loops without a branch inside: the compiler keeps count of what it
    // waits for.)
    int buf = 0, s = 0;
    for (; s + STAGES - 1 < steps; ++s) {
        wait_loads_and_lds<2 * IN * (STAGES - 2)>();
        __builtin_amdgcn_s_barrier();
        issue(buf == 0 ? STAGES - 1 : buf - 1, s + STAGES - 1);
        products(buf);
        buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
    static_for<STAGES - 1>([&](auto i) {                  // the last STAGES - 1 steps, fewer if there are fewer
        constexpr int later = STAGES - 2 - decltype(i)::value;
        if (s < steps - later) {
            wait_loads_and_lds<2 * IN * later>();
            __builtin_amdgcn_s_barrier();
            products(buf);
            buf = buf + 1 == STAGES ? 0 : buf + 1;
            ++s;
        }
    });
    multiply(H1());
    if constexpr (SWIGLU) {
        const int half_n = N / 2;
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const long long row = m0 + wm + i * 16 + r16;
            const long long col = h0 + wn / 2 + g * 4;
            f32x4 gate = acc[i][0], up;
            if constexpr (T == 2) up = acc[i][T - 1];
            else
#pragma unroll
                for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(gate[e], 32);      // (lane groups 0 and 1: gate, 2 and 3: up)
            if (row >= M || (T == 1 && g >= 2)) continue;
            float* y = Y + row * half_n + col;
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = swiglu_value(gate[e], up[e]);
            if (half_n % 4 == 0 && col + 3 < half_n) *(f32x4*)y = o;
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < half_n) y[e] = o[e];
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const long long row = m0 + wm + i * 16 + r16;
        if (row >= M) continue;
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const long long col = n0 + wn + j * 16 + g * 4;
            float* y = Y + row * N + col;
            f32x4 o = acc[i][j];
            if (N % 4 == 0 && col + 3 < N) {
                if (accumulate) { const f32x4 old = *(const f32x4*)y; o[0] = old[0] + o[0]; o[1] = old[1] + o[1]; o[2] = old[2] + o[2]; o[3] = old[3] + o[3]; }
                *(f32x4*)y = o;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < N) y[e] = accumulate ? y[e] + o[e] : o[e];
            }
        }
    }
}

// ---------------------------------------------------------------------------------------- few rows
// Up to 16 rows: a wave a workgroup, 16 columns, the same chain and the same tiles in LDS as above.  With one tile a wave the
// chain sets the pace, one matrix instruction after the other (33 cycles each with nothing between them): the operands of a
// whole step (eight instructions) are read from LDS into one of two register sets while the other is multiplied, and all reads
// are waited for at once, where they have long arrived, so that no product waits for LDS (the kernel above, half a step ahead:
// 2,048 x 8,192 of 16 rows 58 us, this one 49; 65,536 x 2,048 of 8 rows 113 and 109, 4.9 TB/s).  Rows beyond X are not
// fetched.  STAGES: steps of 32 k in LDS, 16 where two workgroups fill a CU's share of the launch anyway.
template <int STAGES, bool SWIGLU>
__global__ __launch_bounds__(WAVE) void gemm_f32_rows_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                             float* __restrict__ Y, int M, int N, int K, int accumulate) {
    constexpr int TILE = 16 * STEP, PER = 4;              // floats of a tile; load instructions a step
    static_assert(STAGES % 2 == 0 && PER * (STAGES - 2) < 64, "pairs of steps, and a count that s_waitcnt can hold");
    extern __shared__ __attribute__((aligned(16))) float tiles[];      // [STAGES][X, W][TILE]
    const int lane = threadIdx.x, r16 = lane % 16, g = lane / 16;
    const long long n0 = (long long)blockIdx.x * 16;
    const long long h0 = n0 / 2;                          // SWIGLU: eight gate rows, then their up rows
    const int rows_n = SWIGLU ? (int)min(8ll, (long long)N / 2 - h0) : (int)min(16ll, (long long)N - n0);
    const buffer_t xbuf = make_buffer(X, M * K * 4), wbuf = make_buffer(W + (SWIGLU ? h0 : n0) * K, ((SWIGLU ? N / 2 : 0) + rows_n) * K * 4);
    int offx[2], offw[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = i * 8 + lane / 8, piece = (lane % 8) ^ (lane / 8);
        offx[i] = row < M ? (row * K + piece * 4) * 4 : NOWHERE;
        const int wrow = SWIGLU ? row % 8 : row;
        offw[i] = wrow < rows_n ? (((SWIGLU && row >= 8 ? N / 2 : 0) + wrow) * K + piece * 4) * 4 : NOWHERE;
    }
    const int steps = K / STEP;
    auto issue = [&](int s) {
        float* to = tiles + s % STAGES * (2 * TILE);
#pragma unroll
        for (int i = 0; i < 2; ++i) load_to_lds(xbuf, to + i * 256, offx[i], s * (STEP * 4));
#pragma unroll
        for (int i = 0; i < 2; ++i) load_to_lds(wbuf, to + TILE + i * 256, offw[i], s * (STEP * 4));
    };
    int at[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) at[i] = r16 * STEP + ((i ^ (r16 % 8)) * 4 + g);
    float x[2][8], w[2][8];
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto read = [&](auto set, int s) {
        const float* from = tiles + s % STAGES * (2 * TILE);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            w[decltype(set)::value][i] = from[TILE + at[i]];
            x[decltype(set)::value][i] = from[at[i]];
        }
    };
    auto multiply = [&](auto set) {
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = mfma_f32(w[decltype(set)::value][i], x[decltype(set)::value][i], acc);
    };
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;
    // (reads of step s + 1, products of step s)
    auto turn = [&](auto set, int s) {
        read(std::integral_constant<int, 1 - decltype(set)::value>(), s + 1);
        multiply(set);
        static_for<8>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);         // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);         // a matrix instruction
        });
    };
    for (int st = 0; st < min(STAGES - 1, steps); ++st) issue(st);
    int s = 0;
    if (steps < STAGES) wait_loads_and_lds<0>();
    wait_loads_and_lds<PER * (STAGES - 2)>();
    read(Set0(), 0);
    if (steps % 2) {                                      // an odd number of steps: one by itself, then pairs
        if (STAGES - 1 < steps) issue(STAGES - 1); else wait_loads_and_lds<0>();
        wait_loads_and_lds<PER * (STAGES - 2)>();
        if (steps > 1) {
            turn(Set0(), 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) { x[0][i] = x[1][i]; w[0][i] = w[1][i]; }
        } else multiply(Set0());
        s = 1;
    }
    for (; steps - s > STAGES; s += 2) {
        issue(s + STAGES - 1);
        wait_loads_and_lds<PER * (STAGES - 2)>();                 // all but those of steps s + 2 and later
        turn(Set0(), s);
        issue(s + STAGES);
        wait_loads_and_lds<PER * (STAGES - 2)>();
        turn(Set1(), s + 1);
    }
    static_for<STAGES>([&](auto i) {                      // the last STAGES steps, fewer if there are fewer; an even number
        constexpr int later = STAGES - 1 - decltype(i)::value;
        using Set = std::integral_constant<int, 1 - later % 2>;
        if (steps - s <= later) return;
        if constexpr (later == STAGES - 1) issue(s + later);
        if constexpr (later > 0) {
            wait_loads_and_lds<PER * (later - 1)>();
            turn(Set(), s);
        } else multiply(Set());
        ++s;
    });
    const int row = r16;
    if constexpr (SWIGLU) {
        const int half_n = N / 2;
        f32x4 up;
#pragma unroll
        for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(acc[e], 32);               // (lane groups 0 and 1: gate, 2 and 3: up)
        if (row >= M || g >= 2) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const long long col = h0 + g * 4 + e;
            if (col < half_n) Y[(long long)row * half_n + col] = swiglu_value(acc[e], up[e]);
        }
        return;
    }
    if (row >= M) return;
    const long long col = n0 + g * 4;
    float* y = Y + (long long)row * N + col;
    if (N % 4 == 0 && col + 3 < N) {
        if (accumulate) { const f32x4 old = *(const f32x4*)y; acc[0] = old[0] + acc[0]; acc[1] = old[1] + acc[1]; acc[2] = old[2] + acc[2]; acc[3] = old[3] + acc[3]; }
        *(f32x4*)y = acc;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e < N) y[e] = accumulate ? y[e] + acc[e] : acc[e];
    }
}

// ---------------------------------------------------------------------------------------- four rows
// Four rows by 16 columns a workgroup of two waves, the chain on the vector unit: lane (row g, column r16) of the first wave has one
// element, v_fmac_f32 takes its x from a lane of the row's sixteen (row_newbcast), so 64 k of X are four registers, and its w from
// the lane's own column.  A fused multiply-add waits 6 cycles for the one before it, four of them 24, where a matrix instruction of
// four k takes 33 and in a loop with its reads 50: where nothing but the chain's length counts, this is the shorter one.  A lone wave
// issues an instruction in four to five cycles, so the first wave's loop holds next to nothing but the chain and, one between
// four links, its reads of the next step; the second wave, on another SIMD, does the loads into LDS and says by a barrier a step
// that they have landed.
// K in steps of 64: X rows of 256 bytes as they lie; W rows of 256 bytes, piece p (16 bytes) of column c at p ^ c.
// What bounds it: a step of 64 k takes some 530 cycles, of them 64 links of 6 to 6.5 and 17 reads of 4 (measured alone: a dependent link 6 to 7
// cycles, an instruction between two of them 3 to 4 more).  4 rows, us, one wave that did the loads itself / two: 2,048 x 8,192 35.6 and
// 31.8 (rows kernel 49), 2,048 x 2,048 11.4 and 10.1 (13.9), 3,072 x 2,048 11.4 and 10.3, 6,144 x 2,048 13.3 and 12.3 (15.7), 1,536 x 6,912 30.2
// and 26.9; 16 rows of 2,048 x 8,192 40.0 and 34.0; from 16,384 columns on the memory sets the time of both.
// A DPP operand that a vector instruction has just written is read too early unless two wait states lie between, and the compiler,
// which keeps that distance for its own instructions, does not look into these.  x comes from LDS, which is waited for; should the
// compiler move it behind that, then ahead of a step's first link, which stands behind s_nop in one piece with it.  (x as an operand
// that each link hands on would pin it, and costs four moves a step.)  That no move stands between the links either is looked for
// in the assembly by tests/test_kernel_bounds.py.
template <int LANE>
__device__ __forceinline__ void chain4(float& acc, const f32x4& x, const f32x4& w) {
#ifdef __HIP_DEVICE_COMPILE__
    // k = 4 LANE + e: register e of lane LANE
#define TUFF_FOUR_LINKS(FIRST) \
    asm(FIRST "v_fmac_f32_dpp %0, %1, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n" \
              "v_fmac_f32_dpp %0, %2, %6 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n" \
              "v_fmac_f32_dpp %0, %3, %7 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n" \
              "v_fmac_f32_dpp %0, %4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf" \
        : "+v"(acc) \
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(LANE))
    if constexpr (LANE == 0) TUFF_FOUR_LINKS("s_nop 1\n");
    else TUFF_FOUR_LINKS("");
#undef TUFF_FOUR_LINKS
#endif
}

constexpr int LONG_STEP = 64;

// `row_groups` workgroups of one column block on one XCD (numbers eight apart), so that its L2 serves W again.
template <int STAGES, bool SWIGLU>
__global__ __launch_bounds__(2 * WAVE) void gemm_f32_quad_kernel(const float* __restrict__ X, const float* __restrict__ W,
                                                                 float* __restrict__ Y, int M, int N, int K, int row_groups, int accumulate) {
    constexpr int WTILE = 16 * LONG_STEP, XTILE = 4 * LONG_STEP, STAGE = WTILE + XTILE;
    constexpr int PER = 5;                                // load instructions a step
    static_assert(PER * (STAGES - 2) < 64, "a count that s_waitcnt can hold");
    static_assert(STAGES % 2 == 0, "two sets of registers in turn");
    extern __shared__ __attribute__((aligned(16))) float tiles[];      // [STAGES][W, X]
    const int lane = threadIdx.x % WAVE, r16 = lane % 16, g = lane / 16;
    const bool brings = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) != 0;
    const int id = blockIdx.x, group = id / 8 % row_groups, block = id / (8 * row_groups) * 8 + id % 8;
    const long long n0 = (long long)block * 16;
    const int m0 = group * 4;
    if (n0 >= N) return;
    const long long j0 = n0 / 2;                          // SWIGLU: eight gate rows, then their up rows
    const int rows_m = min(4, M - m0), rows_n = SWIGLU ? (int)min(8ll, (long long)N / 2 - j0) : (int)min(16ll, (long long)N - n0);
    const int steps = K / LONG_STEP;
    auto turn = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    // Step s lies in buffer s % STAGES.  Behind turn s step s has landed, and the reads of step s - 1 are done: step s - 1 + STAGES
    // goes into its buffer.
    if (brings) {
        const int offx = g < rows_m ? (g * K + r16 * 4) * 4 : NOWHERE;
        int offw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = i * 4 + g, wrow = SWIGLU ? row % 8 : row;
            offw[i] = wrow < rows_n ? (((SWIGLU && row >= 8 ? N / 2 : 0) + wrow) * K + (r16 ^ row) * 4) * 4 : NOWHERE;
        }
        const float* xrows = X + (long long)m0 * K;
        const float* wrows = W + (SWIGLU ? j0 : n0) * K;
        const int bytes_w = ((SWIGLU ? N / 2 : 0) + rows_n) * K * 4;
        // Steps beyond the last are asked for too, of buffers without bytes (zeros, no traffic): the count of loads under way is then
        // the same in every step.
        auto issue = [&](int buf, int s) {
            const bool there = s < steps;
            const buffer_t xbuf = make_buffer(xrows, there ? rows_m * K * 4 : 0), wbuf = make_buffer(wrows, there ? bytes_w : 0);
            const int at = there ? s * (LONG_STEP * 4) : 0;
            float* to = tiles + buf * STAGE;
            load_to_lds(xbuf, to + WTILE, offx, at);
#pragma unroll
            for (int i = 0; i < 4; ++i) load_to_lds(wbuf, to + i * 256, offw[i], at);
        };
        for (int s = 0; s < STAGES; ++s) issue(s, s);
        int buf = STAGES - 1;
        for (int s = 0; s < steps; ++s) {
            wait_loads_and_lds<PER * (STAGES - 2)>();
            turn();
            if (s > 0) issue(buf, s - 1 + STAGES);
            buf = buf + 1 == STAGES ? 0 : buf + 1;
        }
        wait_loads_and_lds<0>();                          // nothing may land in LDS that is another workgroup's by then
        return;
    }
    const bool mine = g < rows_m && r16 < rows_n && !(SWIGLU && r16 >= 8);
    float* const y = Y + (SWIGLU ? (long long)(m0 + g) * (N / 2) + j0 + r16 : (long long)(m0 + g) * N + n0 + r16);
    float old = 0.f;
    if (!SWIGLU && accumulate && mine) old = *y;
    int atw[16];                                          // of every piece of the lane's row of W: where it lies
#pragma unroll
    for (int i = 0; i < 16; ++i) atw[i] = r16 * LONG_STEP + (i ^ r16) * 4;
    const int atx = WTILE + lane * 4;
    struct Step { f32x4 w[16]; f32x4 x; };
    Step r0, r1;
    float acc = 0.f;
    turn();                                               // step 0
    r0.x = *(const f32x4*)(tiles + atx);
#pragma unroll
    for (int i = 0; i < 16; ++i) r0.w[i] = *(const f32x4*)(tiles + atw[i]);
    auto step = [&](const Step& now, Step& next, auto buf, bool more) {       // buf: the next step's
        const float* from = tiles + decltype(buf)::value * STAGE;
        __builtin_amdgcn_s_waitcnt(0xC07F);               // lgkmcnt(0): this step's reads
        if (more) {
            turn();
            next.x = *(const f32x4*)(from + atx);
            static_for<16>([&](auto i) {
                chain4<decltype(i)::value>(acc, now.x, now.w[decltype(i)::value]);
                __builtin_amdgcn_sched_barrier(0);
                next.w[decltype(i)::value] = *(const f32x4*)(from + atw[decltype(i)::value]);
                __builtin_amdgcn_sched_barrier(0);
            });
        } else static_for<16>([&](auto i) { chain4<decltype(i)::value>(acc, now.x, now.w[decltype(i)::value]); });
    };
    // whole turns of the ring with a step to read behind every one of theirs, then what is left
    auto ring = [&](int s0, auto whole) {
        static_for<STAGES>([&](auto b) {
            constexpr int at = decltype(b)::value;
            if (!decltype(whole)::value && s0 + at >= steps) return;
            const bool more = decltype(whole)::value || s0 + at + 1 < steps;
            std::integral_constant<int, (at + 1) % STAGES> next;
            if constexpr (at % 2 == 0) step(r0, r1, next, more);
            else step(r1, r0, next, more);
        });
    };
    int s0 = 0;
    for (; s0 + STAGES < steps; s0 += STAGES) ring(s0, std::true_type());
    ring(s0, std::false_type());
    if constexpr (SWIGLU) {
        const float up = __shfl_xor(acc, 8);
        if (mine) *y = swiglu_value(acc, up);
        return;
    }
    if (mine) *y = accumulate ? old + acc : acc;
}

// What the slowest CU takes for four k, in cycles, as measured over 17 to 2,048 rows and 2,048 to 65,536 columns: a round
// of 64x64 blocks (four tiles a wave) 170 to 185 whether a CU holds one block or shares its time among several, 32x32 blocks
// (one tile a wave) 62 to 70 each and 71 at least.  The fewer: 300 rows of 2,048 x 2,048 36 us in 32x32 and 41 in 64x64 blocks, 500
// rows 46 and 42, 39 rows of 16,384 columns 60 and 44.
long long block_cycles(int M, int N, int side) {
    constexpr long long CUS = 256;
    const long long blocks = ceil_div_ll(M, side) * ceil_div_ll(N, side);
    return side == 64 ? ceil_div_ll(blocks, CUS) * 170 : max(71ll, blocks * 62 / CUS);
}

template <bool SWIGLU, int STAGES>
int launch_quad(const float* X, const float* W, float* Y, int M, int N, int K, int accumulate, hipStream_t stream) {
    constexpr int lds = STAGES * 20 * LONG_STEP * (int)sizeof(float);
    static_assert(lds <= 65536, "without asking for more");
    const int row_groups = ceil_div(M, 4);
    hipLaunchKernelGGL((gemm_f32_quad_kernel<STAGES, SWIGLU>), dim3(ceil_div(ceil_div(N, 16), 8) * 8 * row_groups), dim3(2 * WAVE), lds, stream,
                       X, W, Y, M, N, K, row_groups, accumulate);
    return launch_status();
}

template <bool SWIGLU, int STAGES>
int launch_rows(const float* X, const float* W, float* Y, int M, int N, int K, int accumulate, hipStream_t stream) {
    constexpr int lds = STAGES * 2 * 16 * STEP * (int)sizeof(float);
    static_assert(lds <= 65536, "without asking for more");
    hipLaunchKernelGGL((gemm_f32_rows_kernel<STAGES, SWIGLU>), dim3(ceil_div(N, 16)), dim3(WAVE), lds, stream, X, W, Y, M, N, K, accumulate);
    return launch_status();
}

template <bool SWIGLU, int T, int STAGES>
int launch_chain(const float* X, const float* W, float* Y, int M, int N, int K, int accumulate, hipStream_t stream) {
    constexpr int side = 16 * T * WAVES, lds = STAGES * side * STEP * 2 * (int)sizeof(float);
    static_assert(lds <= 65536, "without asking for more");
    dim3 grid(ceil_div(N, side), ceil_div(M, side));
    if (grid.y > 65535) return -2;
    hipLaunchKernelGGL((gemm_f32_chain_kernel<T, STAGES, SWIGLU>), grid, dim3(WAVES * WAVES * WAVE), lds, stream, X, W, Y, M, N, K, accumulate);
    return launch_status();
}
constexpr int LARGEST = 1 << 22;                          // K of the chain kernels (they count the bytes of 64 rows in 31 bits)

constexpr long long SWIGLU_LARGEST = 1ll << 28;           // elements of W (the bytes up to an up row are counted in 31 bits)

// How many steps of 64 k the four-row kernel keeps in LDS for a product of up to 16 rows; 0: another kernel takes it.
// Four rows a wave as long as one trip over W serves all rows, or the waves are few enough to run side by side, two a CU (16
// rows, 2,048 x 8,192: 42 us, 49 through the rows kernel; 3,072 x 2,048, 768 waves: 23 and 14), and K is not so short that
// the empty steps it begins with count (4 rows, 2,048 x 64: 3.2 us and 2.7, x 192 3.6 and 3.5, 32,768 x 192 6.4 and 7.2).
// Steps: twelve where a CU has one workgroup, six where it has two (4,608 x 1,536 9.4 us, with four 10.4), and four beyond, where the
// loads under way are more than enough and the workgroups side by side count (4 rows, four / six / twelve: 16,384 x 2,048 with
// SwiGLU 30.3, 30.9 and 39.4 us, 9,216 x 2,048 17.5, 18.0 and 24.7, 24,576 x 3,072 59.1, 69.1 and 63.2, 65,536 x 1,024 52.8, 53.9 and 57.4, x 1,536 75.4,
// 76.2 and 78.4, x 2,304 110.1, 111.9 and 111.9, 40,960 x 2,560 79.6, 81.3 and 82.2, x 2,944 90.5, 92.8 and 92.5).
// But twelve again for eight workgroups a CU and more, which begin and end at different times, where K is long: the columns'
// rows are then so far apart that with few steps under way they are waited for (65,536 x 3,584 169.5, 170.8 and 165.8, x 4,608 216.5, 214.7 and 211.0, x
// 6,144 297.4, 294.4 and 272.6, x 12,288 566, 574 and 544, 32,768 x 4,608 117.3, 116.5 and 111.8, x 24,576 614, 598 and 550), and earlier where they are whole 4 KB
// apart (32,768 x 2,048 57.9, 57.4 and 56.0, 65,536 x 2,048 105.5, 105.3 and 100.9, x 3,072 156.0, 155.3 and 147.7).  Rows 32 KB apart or any larger power of two
// are slow however many steps are under way, and slower with more (65,536 x 8,192 419, 424 and 460, 1 row 415, 426 and 475, 40,960 x 8,192 268,
// 287 and 291, 65,536 x 16,384 782, 780 and 842).
int quad_steps(int M, int N, int K) {
    const long long waves = ceil_div_ll(N, 16) * ceil_div(M, 4);
    if (M > 16 || K % LONG_STEP != 0 || K < 192 || (M > 4 && waves > 512)) return 0;
    const bool long_rows = (K % 1024 == 0 ? K >= 2048 : K >= 3072) && !(K >= 8192 && (K & (K - 1)) == 0);
    return waves <= 256 || (waves >= 2048 && long_rows) ? 12 : waves <= 512 ? 6 : 4;
}

// Which of the kernels on whole chains (K a multiple of STEP, operands on 16-byte borders).
template <bool SWIGLU>
int launch_whole_chain(const float* X, const float* W, float* Y, int M, int N, int K, int accumulate, hipStream_t stream) {
    if (M <= 16) {
        switch (quad_steps(M, N, K)) {
            case 12: return launch_quad<SWIGLU, 12>(X, W, Y, M, N, K, accumulate, stream);
            case 6: return launch_quad<SWIGLU, 6>(X, W, Y, M, N, K, accumulate, stream);
            case 4: return launch_quad<SWIGLU, 4>(X, W, Y, M, N, K, accumulate, stream);
        }
        if (N <= 4096) return launch_rows<SWIGLU, 16>(X, W, Y, M, N, K, accumulate, stream);
        return launch_rows<SWIGLU, 8>(X, W, Y, M, N, K, accumulate, stream);
    }
    constexpr int MOST_BLOCKS = 65535;                    // of rows in a grid
    if (ceil_div(M, 32) <= MOST_BLOCKS && block_cycles(M, N, 32) < block_cycles(M, N, 64))
        return launch_chain<SWIGLU, 1, 4>(X, W, Y, M, N, K, accumulate, stream);
    return launch_chain<SWIGLU, 2, 4>(X, W, Y, M, N, K, accumulate, stream);
}
}  // namespace

// quad_steps, for tests.
TUFF_EXPORT int tuff_gemm_f32_quad_steps(int M, int N, int K) { return quad_steps(M, N, K); }

// accumulate != 0: Y += X W^T (the residual add of the reference, src/lfm25_gpu.cu:171).
TUFF_EXPORT int tuff_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K,
                              int accumulate, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const bool aligned = (((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) & 15) == 0;
    if (K % STEP != 0 || K <= 0 || K > LARGEST || !aligned) {
        dim3 grid(ceil_div(N, BN), ceil_div(M, BM)), block(NT);
        if (accumulate) hipLaunchKernelGGL(gemm_f32_kernel<true>, grid, block, 0, stream, X, W, Y, M, N, K);
        else hipLaunchKernelGGL(gemm_f32_kernel<false>, grid, block, 0, stream, X, W, Y, M, N, K);
        return launch_status();
    }
    return launch_whole_chain<false>(X, W, Y, M, N, K, accumulate, stream);
}

// Y [M, F] = silu(X Wg^T) * (X Wu^T), W [2 F, K]: the gate rows Wg, then the up rows Wu; the bits of tuff_gemm_f32 and the
// kernel that applies SwiGLU.  -2 where the product is not one of whole chains.
TUFF_EXPORT int tuff_gemm_f32_swiglu(const float* X, const float* W, float* Y, int M, int F, int K, hipStream_t stream) {
    if (K % STEP != 0 || K <= 0 || K > LARGEST || (long long)2 * F * K > SWIGLU_LARGEST || (((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) & 15) != 0) return -2;
    if (M <= 0 || F <= 0) return 0;
    return launch_whole_chain<true>(X, W, Y, M, 2 * F, K, 0, stream);
}
