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
// A block of Y of WAVES x WAVES waves, T x T tiles of 16x16 each.  K is walked in steps of 32, which go from memory
// straight into LDS, STAGES buffers: the operands of STAGES - 1 steps are under way.  A step
// of a row is 128 bytes, eight pieces of 16; piece p of row r lies at position p ^ (r % 8), so the rows a fragment read
// touches spread over the banks.  A wave's load instruction fills 1 KB, eight rows.  For instruction i of a step a lane
// (row r16 = lane % 16, group g = lane / 16) reads element g of piece i of its row: k = 4 i + g.
//
// What bounds it: a matrix instruction takes 32 cycles (157 TFLOP/s), and one that waits for the one before it in its
// chain 48 or more: with one tile a wave K = 8,192 takes 61 us, whatever the number of rows.  Up to 16 rows: blocks of 16x16,
// a wave a workgroup (2,048 x 8,192: 61 us; 16,384 x 2,048 of 4 rows: 30 us, 4.4 TB/s; 65,536 x 2,048: 107 us, 5.0 TB/s.  The
// general kernel: 825, 345 and 432 us).  More rows: blocks of 64x64 or, where those leave CUs idle, of 32x32; see
// block_cycles (500 rows, 16,384 x 2,048: 283 us, 119 TFLOP/s, the general kernel 577; 2,048 x 8,192: 160 us against 1,480).
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int STEP = 32;

template <int T, int WAVES, int STAGES>
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
    const int last_n = (int)min((long long)SIDE - 1, (long long)N - 1 - n0);
    // (rows beyond the matrix read its last row instead: their results are never stored)
    int offx[IN], offw[IN];                               // bytes from the block's first row
#pragma unroll
    for (int i = 0; i < IN; ++i) {
        const int row = (wave * IN + i) * 8 + lane / 8, piece = (lane % 8) ^ (lane / 8);
        offx[i] = (min(row, last_m) * K + piece * 4) * 4;
        offw[i] = (min(row, last_n) * K + piece * 4) * 4;
    }
    const buffer_t xbuf = make_buffer(X + m0 * K, (last_m + 1) * K * 4), wbuf = make_buffer(W + n0 * K, (last_n + 1) * K * 4);
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
        if (WAVES > 1) __builtin_amdgcn_s_barrier();
        issue(buf == 0 ? STAGES - 1 : buf - 1, s + STAGES - 1);
        products(buf);
        buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
    static_for<STAGES - 1>([&](auto i) {                  // the last STAGES - 1 steps, fewer if there are fewer
        constexpr int later = STAGES - 2 - decltype(i)::value;
        if (s < steps - later) {
            wait_loads_and_lds<2 * IN * later>();
            if (WAVES > 1) __builtin_amdgcn_s_barrier();
            products(buf);
            buf = buf + 1 == STAGES ? 0 : buf + 1;
            ++s;
        }
    });
    multiply(H1());
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

// What the slowest CU takes for four k, in cycles, as measured over 17 to 2,048 rows and 2,048 to 65,536 columns: a round
// of 64x64 blocks (four tiles a wave) 170 to 185 whether a CU holds one block or shares its time among several, 32x32 blocks
// (one tile a wave) 62 to 70 each and 71 at least.  The fewer: 300 rows of 2,048 x 2,048 36 us in 32x32 and 41 in 64x64 blocks, 500
// rows 46 and 42, 39 rows of 16,384 columns 60 and 44.
long long block_cycles(int M, int N, int side) {
    constexpr long long CUS = 256;
    const long long blocks = ceil_div_ll(M, side) * ceil_div_ll(N, side);
    return side == 64 ? ceil_div_ll(blocks, CUS) * 170 : max(71ll, blocks * 62 / CUS);
}

template <int T, int WAVES, int STAGES>
int launch_chain(const float* X, const float* W, float* Y, int M, int N, int K, int accumulate, hipStream_t stream) {
    constexpr int side = 16 * T * WAVES, lds = STAGES * side * STEP * 2 * (int)sizeof(float);
    static_assert(lds <= 65536, "without asking for more");
    dim3 grid(ceil_div(N, side), ceil_div(M, side));
    if (grid.y > 65535) return -2;
    hipLaunchKernelGGL((gemm_f32_chain_kernel<T, WAVES, STAGES>), grid, dim3(WAVES * WAVES * WAVE), lds, stream, X, W, Y, M, N, K, accumulate);
    return launch_status();
}
}  // namespace

// accumulate != 0: Y += X W^T (the residual add of the reference, src/lfm25_gpu.cu:171).
TUFF_EXPORT int tuff_gemm_f32(const float* X, const float* W, float* Y, int M, int N, int K,
                              int accumulate, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const bool aligned = (((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) & 15) == 0;
    constexpr int LARGEST = 1 << 22;                      // (the chain kernel counts the bytes of 64 rows in 31 bits)
    if (K % STEP != 0 || K <= 0 || K > LARGEST || !aligned) {
        dim3 grid(ceil_div(N, BN), ceil_div(M, BM)), block(NT);
        if (accumulate) hipLaunchKernelGGL(gemm_f32_kernel<true>, grid, block, 0, stream, X, W, Y, M, N, K);
        else hipLaunchKernelGGL(gemm_f32_kernel<false>, grid, block, 0, stream, X, W, Y, M, N, K);
        return launch_status();
    }
    if (M <= 16) return launch_chain<1, 1, 8>(X, W, Y, M, N, K, accumulate, stream);
    constexpr int MOST_BLOCKS = 65535;                    // of rows in a grid
    if (ceil_div(M, 32) <= MOST_BLOCKS && block_cycles(M, N, 32) < block_cycles(M, N, 64))
        return launch_chain<1, 2, 4>(X, W, Y, M, N, K, accumulate, stream);
    return launch_chain<2, 2, 4>(X, W, Y, M, N, K, accumulate, stream);
}
