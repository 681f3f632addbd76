// bfloat16 matrix products on the gfx950 matrix cores:  Y[M,N] (=|+=) X[M,K] * W[N,K]^T,
// X bfloat16 with K contiguous, products accumulated in float32.
//
// W is stored tile-major: [ceil(N/16)][ceil(K/32)] blocks of 16 rows x 32 k, each block 1 KB in
// the order a wave's MFMA operand wants it (piece l of 16 bytes = row l % 16, k 8 (l / 16) .. + 7),
// rows and k beyond the matrix zero.  One load instruction of a wave then reads 1 KB in one run
// instead of 64 bytes from each of sixteen rows that lie a whole row apart; measured on streams of
// the shapes of a decode step, the run-wise reads are 17 % faster.
//
// Three kernels, chosen by the sizes on the host:
//  * tiled     M > 64: 128x128 or 256x256 block tiles staged through LDS (compute bound), in two
//    forms: operands loaded straight into LDS (K a multiple of 64, up to 2^22) or through registers (other K);
//  * skinny64  up to 64 rows that skinny16 does not take: a workgroup owns 64 rows of W, one MFMA column
//    tile a wave; the activations of a K chunk are staged once in LDS for all four waves (bandwidth bound);
//  * skinny16  M <= 16, and up to 32 rows (two row tiles a wave) where few_rows_kernel() says so:
//    a workgroup owns 8 to 64 rows of W; its waves split K (bandwidth bound), no barrier in the loop.  Some products
//    of up to 16 rows whose sizes divide evenly have a kernel of their own with its cut and its bits (gemm_bf16_lean.h;
//    launch_lean16() says which).
// The skinny kernels stream each weight byte once from HBM straight into MFMA operands.  Where
// N alone gives too little parallelism to fill 256 CUs, skinny16 uses more waves a workgroup
// (8 or 16, partials added in wave order through LDS) and skinny64 splits K over workgroups
// (partial tiles in a work space, added in slice order by a second kernel, which also does the
// epilogue).  Within a kernel the cut depends on N and K only (and on whether M is beyond 16), so the
// order of additions is fixed.
//
// All use v_mfma_f32_16x16x32_bf16.  Lane l of a wave supplies row (l % 16) of an operand tile
// and eight consecutive k at 8 * (l / 16); it receives rows 4 * (l / 16) + 0..3, column (l % 16)
// of the 16x16 result.
#include "common.h"
#include <stdlib.h>

// OUT_SWIGLU: the rows of W are gate and up rows interleaved (2f: gate f, 2f+1: up f); the
// output is bfloat16 [M, N/2] with y[m, f] = silu(g) * u, silu(g) = g / (1 + exp(-g)).
// OUT_CONV (at most 16 rows, one token a row): W is the input projection of a gated short convolution
// with its rows regrouped, sixteen channels a group, as [B of the group | C of the group | X of the
// group]; the epilogue forms u = B * X, runs the convolution over the row's state, writes
// bfloat16 C * y [M, N/3] and shifts u into the state.  No projected row ever reaches memory.
enum : int { OUT_BF16 = 0, OUT_F32 = 1, OUT_F32_ACCUM = 2, OUT_SWIGLU = 3, OUT_CONV = 4 };

namespace {

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

template <int MODE>
__device__ __forceinline__ void store_out(void* Y, long long idx, float v) {
    if (MODE == OUT_BF16) ((bf16_t*)Y)[idx] = (bf16_t)v;
    else if (MODE == OUT_F32) ((float*)Y)[idx] = v;
    else ((float*)Y)[idx] += v;
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Stores element (row, col) of the product.  For OUT_SWIGLU `partner` is the value of column
// col ^ 1 of the same row; even columns (the gates) write.  Every lane must call it.
template <int MODE>
__device__ __forceinline__ void store_elem(void* Y, long long row, long long col, int M, int N, float v, float partner) {
    if (MODE == OUT_SWIGLU) {
        if ((col & 1) == 0 && row < M && col < N) ((bf16_t*)Y)[row * (N / 2) + col / 2] = (bf16_t)silu_mul(v, partner);
    } else {
        if (row < M && col < N) store_out<MODE>(Y, row * N + col, v);
    }
}

// ------------------------------------------------------------------ tiled kernel
// A workgroup of WAVES_M x WAVES_N waves computes a block of Y; each wave a (16 TM) x (16 TN) part
// of it as TM x TN MFMA tiles.  K is walked in steps of 64 through two LDS buffers: while a step
// is multiplied out of one buffer, the next step's operands travel from memory to registers and,
// piece by piece between the MFMAs, into the other buffer; one barrier a step.
//
// What the shapes answer to, measured on this part: one wave per SIMD issues MFMAs at little more
// than half the rate two waves reach, the LDS takes about 170 bytes/ns per CU and gives 350 to
// 430, against 8600 flop/ns per CU of the matrix cores.  So
//   large:  256 x 256 blocks of eight waves (2 x 4, 128 x 64 each), 128 KB of LDS: two waves per
//           SIMD, and per flop the least LDS traffic two buffers of 160 KB allow;
//   small:  128 x 128 blocks of eight waves (2 x 4, 64 x 32 each), 64 KB of LDS, where the product
//           has too few large blocks to give every CU one.
// The MFMA takes W as its first operand, so a lane ends up with four neighbouring columns of one
// row of Y and stores them as one piece.
constexpr int TBK = 64;
constexpr int CHUNKS = TBK / 8;                     // 16-byte chunks in one row of a tile

// Chunk c of row r lives at chunk position c ^ (r % CHUNKS): the sixteen lanes that
// read one k-chunk of sixteen rows then hit different LDS banks.
__device__ __forceinline__ int swz(int r, int c) { return r * TBK + ((c ^ (r % CHUNKS)) * 8); }

template <int MODE>
__device__ __forceinline__ void store_quad(void* Y, long long row, long long col, int M, int N, f32x4 v) {
    if (row >= M) return;
    if (MODE == OUT_SWIGLU) {
        bf16_t* out = (bf16_t*)Y + row * (N / 2) + col / 2;
        if (col + 3 < N && N % 4 == 0) {
            bf16x2 o = {(bf16_t)silu_mul(v[0], v[1]), (bf16_t)silu_mul(v[2], v[3])};
            *(bf16x2*)out = o;
        } else {
            if (col + 1 < N) out[0] = (bf16_t)silu_mul(v[0], v[1]);
            if (col + 3 < N) out[1] = (bf16_t)silu_mul(v[2], v[3]);
        }
    } else if (col + 3 < N && N % 4 == 0) {
        if (MODE == OUT_BF16) {
            bf16x4 o = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
            *(bf16x4*)((bf16_t*)Y + row * N + col) = o;
        } else {
            f32x4* out = (f32x4*)((float*)Y + row * N + col);
            if (MODE == OUT_F32_ACCUM) { const f32x4 old = *out; v[0] += old[0]; v[1] += old[1]; v[2] += old[2]; v[3] += old[3]; }
            *out = v;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e < N) store_out<MODE>(Y, row * N + col + e, v[e]);
    }
}

// What the tiled product can do around an RMSNorm, as the skinny products do (described with them below):
// TILED_SCALED: X is bf16(x * norm weight) and ss_in [n_ss][M] holds sums of squares of each row of x over
// n_ss groups of columns; every row of the result is scaled by 1 / sqrt(sum / K + eps).  TILED_EMIT (adding
// into the float32 residual stream Y): the new Y is also written as bf16(Y * emit_nw[col]) to emit_xw, and
// each workgroup leaves the sums of squares of its rows over its columns in emit_ss [block column][M] (the
// waves that share rows add theirs in the order of their columns).
struct TiledExtra {
    const float* ss_in = nullptr; int n_ss = 0; float eps = 0.f;
    int ss_rows = 0;                      // rows of a group of sums in ss_in (0: M; 64 where a product of at most 64 rows left them)
    const float* emit_nw = nullptr; bf16_t* emit_xw = nullptr; float* emit_ss = nullptr;
    int bands = 0;                        // the order of the blocks (bands_of_rows)
    const float* bias = nullptr;          // TILED_BIAS, TILED_RELU2: [N] or null
};
// TILED_BIAS: v + bias[column], rounded to bfloat16; TILED_RELU2: the square of its positive part, rounded.  As a kernel of their
// own each wrote and read the float32 sums once more (2,048 rows of 5,632 columns: 15 us beside a product of 50).
// TILED_EMIT_FAR: TILED_EMIT for rows of 2^25 columns and more, of which sixteen are 2^31 bytes: its epilogue goes by address and not
// through buffers (both in one kernel cost the others 0.25 us of 10 to 27).
enum : int { TILED_PLAIN = 0, TILED_SCALED = 1, TILED_EMIT = 2, TILED_BIAS = 3, TILED_RELU2 = 4, TILED_EMIT_FAR = 5 };

template <int TM, int TN, int WAVES_M, int WAVES_N, int AHEAD, int MODE>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_bf16_tiled_kernel(
        const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K,
        int steps_per_slice, float* __restrict__ ws) {
    constexpr int NT = 64 * WAVES_M * WAVES_N;
    constexpr int BM = 16 * TM * WAVES_M, BN = 16 * TN * WAVES_N;
    constexpr int PA = BM * CHUNKS / NT, PB = BN * CHUNKS / NT;     // 16-byte pieces of X and of W a thread moves a step
    constexpr int ROWS_PER_PIECE = NT / CHUNKS;
    static_assert(BM * CHUNKS % NT == 0 && BN * CHUNKS % NT == 0, "whole pieces");
    static_assert(TN <= TM, "the fragments of W are fetched over TM inner steps");
    extern __shared__ __attribute__((aligned(16))) bf16_t tiles[];       // [2][BM * TBK] of X then [2][BN * TBK] of W
    bf16_t* As = tiles;
    bf16_t* Bs = tiles + 2 * BM * TBK;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const int wm = (wave / WAVES_N) * 16 * TM, wn = (wave % WAVES_N) * 16 * TN;
    const int r16 = lane % 16, g = lane / 16;
    const long long m0 = (long long)blockIdx.y * BM, n0 = (long long)blockIdx.x * BN;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Rows beyond the matrix read its last row instead (their results are never stored), so the
    // loads of a full step need no guard.  Offsets are relative to the block's first row.
    // Of W a step holds two blocks (k 0..31, 32..63) of each of the BN / 16 row tiles; thread tid moves
    // piece tid % 64 of block (tid / 64) % 2 of row tile tid / 128, and the same NT / 128 tiles further.
    const int kb = (K + 31) / 32;
    const bf16_t* Xb = X + m0 * K;
    const bf16_t* Wb = W + (n0 / 16) * (long long)kb * 512;
    const int row0 = tid / CHUNKS, c0 = tid % CHUNKS;
    const int last_a = (int)min((long long)BM - 1, (long long)M - 1 - m0);
    const int last_tile = (int)min((long long)BN / 16 - 1, (N - 1 - n0) / 16);
    const int wpiece = tid % 64, wh = (tid / 64) % 2, wtile = tid / 128;
    static_assert(NT % 128 == 0 && ROWS_PER_PIECE == (NT / 128) * 16, "pieces of X and of W advance by the same rows");
    unsigned offa[PA], offb[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) offa[i] = (unsigned)min(row0 + i * ROWS_PER_PIECE, last_a) * (unsigned)K + c0 * 8;
#pragma unroll
    for (int i = 0; i < PB; ++i)
        offb[i] = ((unsigned)min(wtile + i * (NT / 128), last_tile) * (unsigned)kb + wh) * 512u + wpiece * 8;
    const int lds_st = swz(row0, c0);                    // piece i goes ROWS_PER_PIECE * TBK * i further
    const int lds_st_b = swz(wtile * 16 + wpiece % 16, wh * 4 + wpiece / 16);
    // Memory answers later than a step lasts, so the operands of AHEAD steps are on their way at
    // any time, each in a register set of its own; a set is free again once it went into LDS.
    bf16x8 ra[AHEAD][PA], rb[AHEAD][PB];
    // gridDim.z > 1: the block walks only its slice of K and leaves a float32 partial block in the work
    // space, ws[slice][row][col]; splitk_finish_kernel adds the slices and does the epilogue.
    const int nk = (K + TBK - 1) / TBK;
    const int kt_begin = blockIdx.z * steps_per_slice, kt_end = min(nk, kt_begin + steps_per_slice);

    auto load_global = [&](auto set_tag, int kt) {
        constexpr int set = decltype(set_tag)::value;
        const int k0 = min(kt, nk - 1) * TBK;            // steps past the end read the last one again; nobody uses them
        const unsigned w0 = (unsigned)(k0 / 32) * 512u;  // W: two blocks a step
        if (k0 + TBK <= K) {
#pragma unroll
            for (int i = 0; i < PA; ++i) ra[set][i] = *(const bf16x8*)(Xb + k0 + offa[i]);
#pragma unroll
            for (int i = 0; i < PB; ++i) rb[set][i] = *(const bf16x8*)(Wb + w0 + offb[i]);
        } else {                                         // the last, partial step: zeros beyond K
            const bool in = k0 + c0 * 8 < K, in_w = k0 / 32 + wh < kb;
            const bf16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < PA; ++i) ra[set][i] = in ? *(const bf16x8*)(Xb + k0 + offa[i]) : z;
#pragma unroll
            for (int i = 0; i < PB; ++i) rb[set][i] = in_w ? *(const bf16x8*)(Wb + w0 + offb[i]) : z;
        }
    };
    auto store_piece = [&](auto set_tag, int buf, int p) {             // p counts the pieces of X, then those of W
        constexpr int set = decltype(set_tag)::value;
        if (p < PA) *(bf16x8*)(&As[buf * BM * TBK + lds_st + p * ROWS_PER_PIECE * TBK]) = ra[set][p < PA ? p : 0];
        else *(bf16x8*)(&Bs[buf * BN * TBK + lds_st_b + (p - PA) * ROWS_PER_PIECE * TBK]) = rb[set][p < PA ? 0 : p - PA];
    };
    // fragment offsets inside a buffer: row r16 of MFMA tile 0 of this wave, k-chunk g (+4 for the second half)
    const int fa0 = swz(wm + r16, g), fa1 = swz(wm + r16, 4 + g);
    const int fb0 = swz(wn + r16, g), fb1 = swz(wn + r16, 4 + g);

    // One step out of buffer `buf`: two halves (k 0..31, 32..63) of TM inner steps.  An inner step
    // multiplies one fragment of X with the TN fragments of W; meanwhile the next fragment of X
    // and, in the first half, the fragments of W for the second half are on their way from LDS,
    // and in the second half the pieces of register set `fill` go into the other buffer.
    auto multiply = [&](int buf, auto fill) {
        const bf16_t* Ab = As + buf * BM * TBK;
        const bf16_t* Bb = Bs + buf * BN * TBK;
        bf16x8 b[TN], bn[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = *(const bf16x8*)(Bb + fb0 + j * 16 * TBK);
        bf16x8 a = *(const bf16x8*)(Ab + fa0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const bf16x8 an = *(const bf16x8*)(Ab + (i + 1 < TM ? fa0 + (i + 1) * 16 * TBK : fa1));
            if (i < TN) bn[i] = *(const bf16x8*)(Bb + fb1 + i * 16 * TBK);
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(b[j], a, acc[i][j]);
            a = an;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            bf16x8 an = a;
            if (i + 1 < TM) an = *(const bf16x8*)(Ab + fa1 + (i + 1) * 16 * TBK);
#pragma unroll
            for (int p = 0; p < PA + PB; ++p)
                if (p * TM / (PA + PB) == i) store_piece(fill, buf ^ 1, p);
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(bn[j], a, acc[i][j]);
            a = an;
        }
    };

    // set s holds step s, later step s + AHEAD, ...; step kt + 1 is filled in while step kt is multiplied
    static_for<AHEAD>([&](auto s) { load_global(s, kt_begin + decltype(s)::value); });
#pragma unroll
    for (int p = 0; p < PA + PB; ++p) store_piece(std::integral_constant<int, 0>(), 0, p);
    __syncthreads();
    for (int kt0 = kt_begin; kt0 < kt_end; kt0 += AHEAD) {
        static_for<AHEAD>([&](auto u) {
            constexpr int set = decltype(u)::value;
            const int kt = kt0 + set;
            if (kt < kt_end) {
                load_global(u, kt + AHEAD);
                multiply((kt - kt_begin) & 1, std::integral_constant<int, (set + 1) % AHEAD>());
                __syncthreads();
            }
        });
    }

    if (gridDim.z > 1) {
        float* mine = ws + (long long)blockIdx.z * M * N;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                store_quad<OUT_F32>(mine, m0 + wm + i * 16 + r16, n0 + wn + j * 16 + g * 4, M, N, acc[i][j]);
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            store_quad<MODE>(Y, m0 + wm + i * 16 + r16, n0 + wn + j * 16 + g * 4, M, N, acc[i][j]);
}

// The same product with the operands going from memory straight into LDS (load_to_lds),
// without a stop in registers; used where K is a multiple of 64.  A wave's load instruction fills
// 1 KB of LDS, lane l the 16 bytes at 16 l.  X keeps the swizzled row-major layout above: an
// instruction covers eight rows of 128 bytes, and the lane that fills chunk position p of row r
// fetches chunk p ^ (r % 8) of that row.  W lies in LDS as in memory, one block of 1 KB per (row
// tile, k 32): the fragment of lane l is at 16 l.  STAGES buffers of a step of 64 k each: the
// operands of STAGES - 1 steps are on their way while one is multiplied.
// Measured against the kernel above (M = 2048; N x K): 3072 x 2048 42.8 -> 32.9 us, 2048 x 2048
// 35.1 -> 27.4, 2048 x 8192 102.7 -> 81.3, 16384 x 2048 157.6 -> 148.6, 6144 x 2048 69.0 -> 61.2.
// With all CUs busy and random operands the clock, not the instruction stream, sets the pace: the
// same loop over constant data runs a quarter faster.
//
// BUFFER: the loads go through buffers, which leaves the compiler its count of the LDS reads under way (load_to_lds); else they are
// global loads, and it waits for more of them.  Buffers win where the whole grid runs side by side, one block a CU, and K is
// short, and with the blocks of 256 x 256; they lose a little where the operands come slower than the waves could go on:
// see dma_through_buffer.
template <int TM, int TN, int WAVES_M, int WAVES_N, int STAGES, bool BUFFER, bool FOLDS, int MODE, int AROUND>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void gemm_bf16_dma_kernel(
        const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K,
        int steps_per_slice, float* __restrict__ ws, TiledExtra ex) {
    static_assert(!(AROUND == TILED_EMIT || AROUND == TILED_EMIT_FAR) || MODE == OUT_F32_ACCUM, "the emitting epilogue adds into the residual stream");
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int BM = 16 * TM * WAVES_M, BN = 16 * TN * WAVES_N;
    constexpr int IA = BM / 8 / NW, IB = BN / 8 / NW;                  // load instructions of X and of W a wave issues a step
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole instructions");
    // all arguments in one trip (left alone they are asked for one by one, where they are first needed)
    asm volatile("" ::"s"(X), "s"(W), "s"(Y), "s"(M), "s"(N), "s"(K), "s"(steps_per_slice));
    if constexpr (AROUND == TILED_SCALED) asm volatile("" ::"s"(ex.ss_in), "s"(ex.n_ss), "s"(ex.ss_rows), "s"(ex.eps));
    extern __shared__ __attribute__((aligned(16))) bf16_t tiles[];       // [STAGES][BM * TBK] of X then [STAGES][BN * TBK] of W
    bf16_t* As = tiles;
    bf16_t* Bs = tiles + STAGES * BM * TBK;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = (wave / WAVES_N) * 16 * TM, wn = (wave % WAVES_N) * 16 * TN;
    const int r16 = lane % 16, g = lane / 16;
    constexpr bool BANDS = BM >= 256 || BN >= 256;
    // ex.bands (bands_of_rows): an eighth of the blocks, one behind the other, an XCD (block id % 8), bands of eight row blocks,
    // in a band column by column
    unsigned bx = blockIdx.x, by = blockIdx.y;
    if (BANDS && ex.bands) {
        const unsigned all = gridDim.x * gridDim.y, id = bx + gridDim.x * by, xcd = id % 8;
        const unsigned at = xcd * (all / 8) + min(xcd, all % 8) + id / 8;
        const unsigned band = at / (8 * gridDim.x), rest = at - band * (8 * gridDim.x), rows = min(8u, gridDim.y - 8 * band);
        bx = rest / rows;
        by = 8 * band + rest % rows;
    }
    const long long m0 = (long long)by * BM, n0 = (long long)bx * BN;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // FOLDS: a block in the place of slices of K adds them itself: a sum each, in the order of the kernel that adds slices, so
    // the same bits.
    f32x4 folded[FOLDS ? TM : 1][FOLDS ? TN : 1];
#pragma unroll
    for (int i = 0; i < (FOLDS ? TM : 1); ++i)
#pragma unroll
        for (int j = 0; j < (FOLDS ? TN : 1); ++j) folded[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int kb = (int)((unsigned)K / 32u);
    const int last_a = min(BM - 1, M - 1 - (int)m0);
    const int last_tile = min(BN / 16 - 1, (int)((unsigned)(N - 1 - (int)n0) / 16u));
    // instruction q of X (q = wave + NW i) fills rows 8 q .. 8 q + 7; instruction q of W fills block q % 2 of row tile q / 2;
    // offsets from the block's first row (tile), in bytes (global loads: in elements).  Rows and tiles beyond the matrix have results
    // that are never stored.  Through buffers they are not fetched: if they read the last one instead, all blocks ask for the same
    // line again and again, and 160 rows took longer than 256 (2,048 x 5,632: 20.1 us against 18.1, now 15.5).
    unsigned offa[IA], offb[IB];
#pragma unroll
    for (int i = 0; i < IA; ++i) {
        const int row = (wave + NW * i) * 8 + lane / 8, piece = ((lane % 8) ^ (lane / 8)) * 8;
        if (BUFFER) offa[i] = row <= last_a ? (unsigned)(row * K + piece) * 2 : (unsigned)NOWHERE;
        else offa[i] = (unsigned)min(row, last_a) * (unsigned)K + piece;
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        const int q = wave + NW * i, tile = q / 2;
        if (BUFFER) offb[i] = tile <= last_tile ? (unsigned)(tile * kb + q % 2) * 1024 + lane * 16 : (unsigned)NOWHERE;
        else offb[i] = ((unsigned)min(tile, last_tile) * (unsigned)kb + q % 2) * 512 + lane * 8;
    }
    const buffer_t xbuf = make_buffer(X + m0 * K, (last_a + 1) * K * 2);
    const buffer_t wbuf = make_buffer(W + (n0 / 16) * (long long)kb * 512, (last_tile + 1) * kb * 1024);
    const int nk = (int)((unsigned)K / (unsigned)TBK);
    const int kt_begin = blockIdx.z * steps_per_slice, kt_end = FOLDS ? nk : min(nk, kt_begin + steps_per_slice);
    int fold_at = kt_begin + steps_per_slice;                          // the step that the next slice begins with (FOLDS)

    const bf16_t* Xb = X + m0 * K;
    const bf16_t* Wb = W + (n0 / 16) * (long long)kb * 512;
    // TILED_EMIT, small blocks: what the epilogue adds to and multiplies with is asked for ahead of the operands (rows beyond
    // the matrix: the last one's, never used); behind the loop it would be a trip to memory more
    // (512 rows, 2,048 x 2,048 11.1 and 10.9 us, x 4,096 17.0 and 16.9; 128 x 128 blocks are no faster for it).
    constexpr bool EARLY = AROUND == TILED_EMIT && BM == 64;
    f32x4 y_old[EARLY ? TM : 1][EARLY ? TN : 1], next_w[EARLY ? TN : 1];
    if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            next_w[j] = *(const f32x4*)(ex.emit_nw + n0 + wn + j * 16 + g * 4);
#pragma unroll
            for (int i = 0; i < TM; ++i)
                y_old[i][j] = *(const f32x4*)((const float*)Y + min(m0 + wm + i * 16 + r16, (long long)M - 1) * N + n0 + wn + j * 16 + g * 4);
        }
    }
    auto issue = [&](int buf, int kt) {
#pragma unroll
        for (int i = 0; i < IA; ++i) {
            bf16_t* to = As + buf * BM * TBK + (wave + NW * i) * 512;
            if constexpr (BUFFER) load_to_lds(xbuf, to, (int)offa[i], kt * (TBK * 2));
            else load_to_lds(Xb + kt * TBK + offa[i], to);
        }
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            bf16_t* to = Bs + buf * BN * TBK + (wave + NW * i) * 512;
            if constexpr (BUFFER) load_to_lds(wbuf, to, (int)offb[i], kt * 2048);
            else load_to_lds(Wb + (unsigned)(kt * 2) * 512u + offb[i], to);
        }
    };
    const int fa0 = swz(wm + r16, g), fa1 = swz(wm + r16, 4 + g);
    const int fb = (wn / 16) * 1024 + lane * 8;                        // block h of MFMA tile j: + (2 j + h) * 512

    // The fragments of half a step (k 0..31 or 32..63: TM of X, TN of W) are read at once into one of
    // two register sets, half a step before the MFMAs that use them: while one set is multiplied the
    // other is on its way from LDS, also across the barrier between two steps.
    bf16x8 fx[2][TM], fw[2][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) fx[1][i] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < TN; ++j) fw[1][j] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    auto read_half = [&](auto set_tag, int buf, auto half_tag) {
        constexpr int set = decltype(set_tag)::value, h = decltype(half_tag)::value;
        const bf16_t* Ab = As + buf * BM * TBK + (h ? fa1 : fa0);
        const bf16_t* Bb = Bs + buf * BN * TBK + fb + h * 512;
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[set][j] = *(const bf16x8*)(Bb + 2 * j * 512);
#pragma unroll
        for (int i = 0; i < TM; ++i) fx[set][i] = *(const bf16x8*)(Ab + i * 16 * TBK);
    };
    auto mult = [&](auto set_tag) {
        constexpr int set = decltype(set_tag)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = mfma16(fw[set][j], fx[set][i], acc[i][j]);
    };
    // asks the instruction scheduler to spread the LDS reads of a half step evenly among its MFMAs
    auto spread = [&]() {
        constexpr int R = TM + TN, Q = TM * TN;
        static_for<R>([&](auto r) {
            constexpr int n = Q / R + (decltype(r)::value < Q % R ? 1 : 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);         // one LDS read
            __builtin_amdgcn_sched_group_barrier(0x008, n, 0);         // n MFMAs
        });
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;

    // Step kt lives in buffer (kt - kt_begin) % STAGES.  Before step kt is multiplied the loads of
    // steps kt .. kt + STAGES - 2 are under way; a wave waits until all but those of the later steps
    // have landed, the barrier then says the same of everybody's and that nobody reads the buffer
    // of step kt - 1 any more, which the loads of step kt + STAGES - 1 go into.  Two loops, of the steps with loads to issue
    // and of the last ones, with no branch inside: with the loads through buffers (load_to_lds) the compiler then counts the
    // fragment reads under way and waits for the ones it needs, where it waited for all of them, those just issued among
    // them, before every group of MFMAs.
    // TILED_SCALED: the scale of each of the block's rows out of its sums of squares over groups of columns.  Up to 32 groups (as products of
    // 64 and more columns a block leave them): a thread a row asks for all of them ahead of the operands and has the scale before they
    // are there.  Behind the operands, and one condition a load, the sums came when all that had been asked for was there, and the
    // loop began 0.3 to 0.5 us later.
    constexpr int SS_PARTS = (64 * NW) / BM >= 4 ? 4 : (64 * NW) / BM >= 2 ? 2 : 1;
    constexpr int SS_AT_ONCE = 32;
    __shared__ float row_ss[AROUND == TILED_SCALED ? SS_PARTS : 1][AROUND == TILED_SCALED ? BM : 1];
    __shared__ float row_scale[AROUND == TILED_SCALED ? BM : 1];
    const int ss_rows = ex.ss_rows ? ex.ss_rows : M;
    const bool at_once = AROUND == TILED_SCALED && ex.n_ss <= SS_AT_ONCE && ss_rows < (1 << 23) && gridDim.z == 1;
    const bool sums = at_once && wave < BM / 64;
    float ss_v[AROUND == TILED_SCALED ? SS_AT_ONCE : 1];
    if constexpr (AROUND == TILED_SCALED) {
#pragma unroll
        for (int u = 0; u < SS_AT_ONCE; ++u) ss_v[u] = 0.f;
        if (sums) {
            // (rows beyond the matrix and groups that are none lie behind the buffer: zeros)
            const buffer_t sbuf = make_buffer(ex.ss_in + m0, ((ex.n_ss - 1) * ss_rows + last_a + 1) * 4);
            const int at = tid <= last_a ? tid * 4 : NOWHERE;
#pragma unroll
            for (int u = 0; u < SS_AT_ONCE / 2; ++u) ss_v[u] = load_buffer_float(sbuf, u < ex.n_ss ? at : NOWHERE, u < ex.n_ss ? u * ss_rows * 4 : 0);
            if (ex.n_ss > SS_AT_ONCE / 2) {
#pragma unroll
                for (int u = SS_AT_ONCE / 2; u < SS_AT_ONCE; ++u)
                    ss_v[u] = load_buffer_float(sbuf, u < ex.n_ss ? at : NOWHERE, u < ex.n_ss ? u * ss_rows * 4 : 0);
            }
        }
    }
    // (steps that are none: the last one's operands again, so that the count of loads under way is known; without an inner size there is
    // not even that one: buffers of no bytes, and no global loads)
    static_for<STAGES - 1>([&](auto s) {
        constexpr int st = decltype(s)::value;
        if (BUFFER || nk > 0) issue(st, max(0, min(kt_begin + st, kt_end - 1)));
    });
    // (a product cut along K leaves the scales to the kernel that adds the slices)
    if constexpr (AROUND == TILED_SCALED) {
        if (sums) {
            float t;
            if (ex.n_ss <= 16) {
                t = ss_v[0];
#pragma unroll
                for (int u = 1; u < 16; ++u) t += ss_v[u];
            } else {
                // in parts as below, so the same bits
                float part[SS_PARTS];
#pragma unroll
                for (int q = 0; q < SS_PARTS; ++q) {
                    part[q] = ss_v[q];
#pragma unroll
                    for (int u = q + SS_PARTS; u < SS_AT_ONCE; u += SS_PARTS) part[q] += ss_v[u];
                }
                t = part[0];
#pragma unroll
                for (int q = 1; q < SS_PARTS; ++q) t += part[q];
            }
            row_scale[tid] = 1.0f / sqrtf(t / (float)K + ex.eps);      // (read in the epilogue, behind the barriers of the loop)
        } else if (!at_once && tid < SS_PARTS * BM && gridDim.z == 1) {
            // More groups: SS_PARTS parts, thread (part, row) adds the groups part, part + SS_PARTS, ... in that order, sixteen loads at a
            // time (one after the other would be as many trips to memory); behind the loop the parts of a row are added in their
            // order and the row's scale is left for the epilogue.
            const int r = tid % BM, part = tid / BM;
            const long long row = m0 + r;
            float t = 0.f;
            if (row < M) {
                for (int j0 = part; j0 < ex.n_ss; j0 += 16 * SS_PARTS) {
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int j = j0 + u * SS_PARTS;
                        v[u] = j < ex.n_ss ? ex.ss_in[(long long)j * ss_rows + row] : 0.f;
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) t += v[u];
                }
            }
            row_ss[part][r] = t;
        }
        // read in the epilogue, behind the barriers of the loop (every wave waits for its LDS writes before each)
    }
    auto fold = [&]() {
        if constexpr (FOLDS) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    folded[i][j] += acc[i][j];
                    acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            fold_at += steps_per_slice;
        }
    };
    auto products = [&](int buf, auto first_of_slice) {
        read_half(S0(), buf, S0());
        mult(S1());                                            // the second half of the step before (zeros at first)
        spread();
        if constexpr (decltype(first_of_slice)::value) fold();
        read_half(S1(), buf, S1());
        mult(S0());
        spread();
    };
    int buf = 0, kt = kt_begin;
    auto step = [&](auto first_of_slice) {
        wait_loads_and_lds<(STAGES - 2) * (IA + IB)>();
        __builtin_amdgcn_s_barrier();
        issue(buf == 0 ? STAGES - 1 : buf - 1, kt + STAGES - 1);
        products(buf, first_of_slice);
        buf = buf + 1 == STAGES ? 0 : buf + 1;
        ++kt;
    };
    const int steady = kt_end - (STAGES - 1);                  // the steps before it have loads to issue
    if constexpr (FOLDS) {
        while (kt < steady) {
            if (kt == fold_at) step(std::true_type());
            const int until = min(steady, fold_at);
            while (kt < until) step(std::false_type());
        }
    } else {
        while (kt < steady) step(std::false_type());
    }
    static_for<STAGES - 1>([&](auto i) {                       // the last STAGES - 1 steps, fewer if there are fewer
        constexpr int later = STAGES - 2 - decltype(i)::value;
        if (kt < kt_end - later) {
            wait_loads_and_lds<later * (IA + IB)>();
            __builtin_amdgcn_s_barrier();
            if (FOLDS && kt == fold_at) products(buf, std::true_type());
            else products(buf, std::false_type());
            buf = buf + 1 == STAGES ? 0 : buf + 1;
            ++kt;
        }
    });
    if (kt_begin < kt_end) mult(S1());
    else {                                                     // no step has waited for the loads into LDS and for the rows' scales
        wait_loads_and_lds<0>();
        __builtin_amdgcn_s_barrier();
    }
    if constexpr (FOLDS) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = folded[i][j] + acc[i][j];
    }

    if (gridDim.z > 1) {
        float* mine = ws + (long long)blockIdx.z * M * N;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                store_quad<OUT_F32>(mine, m0 + wm + i * 16 + r16, n0 + wn + j * 16 + g * 4, M, N, acc[i][j]);
        return;
    }
    if constexpr (AROUND == TILED_SCALED) {
        if (!at_once) {                                        // (the parts were written before the loop's first barrier)
            if (tid < BM) {
                float t = row_ss[0][tid];
#pragma unroll
                for (int q = 1; q < SS_PARTS; ++q) t += row_ss[q][tid];
                row_scale[tid] = 1.0f / sqrtf(t / (float)K + ex.eps);
            }
            __syncthreads();
        }
    }
    if constexpr (AROUND == TILED_EMIT || AROUND == TILED_EMIT_FAR) {
        constexpr bool FAR = AROUND == TILED_EMIT_FAR;
        // whole blocks of columns only (the host sees to it): Y += acc, the next norm's operand, the row's sum of squares.  Sixteen rows a
        // buffer: those beyond the matrix lie behind it (nothing is fetched or written), and a lane's place is the same in every one.
        const int at = FAR ? 0 : r16 * N + (int)n0 + wn + g * 4;
        float wave_sq[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float sq = 0.f;
            const int row0 = wm + i * 16, rows = max(0, min(16, last_a + 1 - row0));
            const long long first = (m0 + (rows > 0 ? row0 : 0)) * N;
            const buffer_t ybuf = make_buffer((float*)Y + first, FAR ? 0 : rows * N * 4), xwbuf = make_buffer(ex.emit_xw + first, FAR ? 0 : rows * N * 2);
            const long long far = first + (long long)r16 * N + n0 + wn + g * 4;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 y, nw;
                if constexpr (EARLY) { y = y_old[i][j]; nw = next_w[j]; }
                else {
                    if constexpr (FAR) y = r16 < rows ? *(const f32x4*)((const float*)Y + far + j * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
                    else y = load_buffer_f32x4(ybuf, at * 4 + j * 64, 0);
                    nw = *(const f32x4*)(ex.emit_nw + n0 + wn + j * 16 + g * 4);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] += acc[i][j][e];
                if constexpr (!FAR) store_buffer(ybuf, at * 4 + j * 64, 0, y);
                const bf16x4 o = {(bf16_t)(y[0] * nw[0]), (bf16_t)(y[1] * nw[1]), (bf16_t)(y[2] * nw[2]), (bf16_t)(y[3] * nw[3])};
                if constexpr (!FAR) store_buffer(xwbuf, at * 2 + j * 32, 0, o);
                else if (r16 < rows) {
                    *(f32x4*)((float*)Y + far + j * 16) = y;
                    *(bf16x4*)(ex.emit_xw + far + j * 16) = o;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) sq = fmaf(y[e], y[e], sq);
            }
            sq = r16 < rows ? sq : 0.f;
            sq = butterfly_sum<32>(butterfly_sum<16>(sq));
            wave_sq[i] = sq;
        }
        // the waves that share rows add their sums in the order of their columns, through the LDS the operands
        // have left: one sum per row and block of columns, so that whoever reads them asks only once
        float* red = (float*)tiles;                            // [WAVES_N][BM]
        __syncthreads();                                       // nobody reads operands any more
        if (g == 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i) red[(wave % WAVES_N) * BM + wm + i * 16 + r16] = wave_sq[i];
        }
        __syncthreads();
        for (int r = tid; r < BM; r += 64 * NW) {
            float t = red[r];
#pragma unroll
            for (int w = 1; w < WAVES_N; ++w) t += red[w * BM + r];
            if (m0 + r < M) ex.emit_ss[(long long)bx * M + m0 + r] = t;
        }
        return;
    }
    f32x4 col_bias[AROUND == TILED_BIAS || AROUND == TILED_RELU2 ? TN : 1];
    if constexpr (AROUND == TILED_BIAS || AROUND == TILED_RELU2) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const long long col = n0 + wn + j * 16 + g * 4 + e;
                col_bias[j][e] = ex.bias && col < N ? ex.bias[col] : 0.f;
            }
    }
    // whole blocks of columns: through buffers, as above
    const bool whole = N % BN == 0 && N < (1 << 25);
    constexpr int SIZE = MODE == OUT_BF16 || MODE == OUT_SWIGLU ? 2 : 4, PER = MODE == OUT_SWIGLU ? 2 : 1;      // bytes an output, columns an output
    const int at = (r16 * (N / PER) + ((int)n0 + wn + g * 4) / PER) * SIZE;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        float sc = 1.f;
        if constexpr (AROUND == TILED_SCALED) sc = row_scale[wm + i * 16 + r16];
        const int row0 = wm + i * 16, rows = whole ? max(0, min(16, last_a + 1 - row0)) : 0;
        const buffer_t ybuf = make_buffer((char*)Y + (m0 + (rows > 0 ? row0 : 0)) * (N / PER) * SIZE, rows * (N / PER) * SIZE);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            f32x4 v = acc[i][j];
            if constexpr (AROUND == TILED_SCALED) { v[0] *= sc; v[1] *= sc; v[2] *= sc; v[3] *= sc; }
            if constexpr (AROUND == TILED_BIAS || AROUND == TILED_RELU2) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] += col_bias[j][e];
                    if constexpr (AROUND == TILED_RELU2) { v[e] = fmaxf(v[e], 0.f); v[e] *= v[e]; }
                }
            }
            if (whole) {
                const int here = at + j * 16 / PER * SIZE;
                if constexpr (MODE == OUT_SWIGLU) store_buffer(ybuf, here, 0, bf16x2{(bf16_t)silu_mul(v[0], v[1]), (bf16_t)silu_mul(v[2], v[3])});
                else if constexpr (MODE == OUT_BF16) store_buffer(ybuf, here, 0, bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]});
                else {
                    if constexpr (MODE == OUT_F32_ACCUM) v += load_buffer_f32x4(ybuf, here, 0);
                    store_buffer(ybuf, here, 0, v);
                }
            } else store_quad<MODE>(Y, m0 + wm + i * 16 + r16, n0 + wn + j * 16 + g * 4, M, N, v);
        }
    }
}

// ----------------------------------------------------------------- skinny kernels
constexpr int SK_CHUNK = 128;

// M <= 16.  grid: tiles of 16 columns.  The NW waves of a workgroup split K: wave w takes the
// chunks w, w + NW, w + 2 NW, ... of 128; in a chunk the wave reads four blocks of its row tile of W
// (1 KB each) and 256 bytes of each of the 16 X rows (four loads of 16 rows x 64 contiguous bytes)
// and issues four MFMAs.
// The loads of two chunks are under way.  The wave partials are added in wave order through LDS.  NW is
// chosen from N and K only.
//
// The product may be taken of the RMSNorm of the float32 residual stream x,
//   y[m, n] = (1 / sqrt(mean_k x[m,k]^2 + eps)) * sum_k bf16(x[m,k] * w[k]) W[n,k]:
// the norm weight is applied to the operand, the row's scale to the result.
//  * NORM_INSIDE: X is x itself; the operand is formed and the sum of squares taken from the
//    values the workgroup loads anyway (lane partials in a fixed butterfly, waves in wave
//    order).  `rows` (optional) gathers rows of x.
//  * NORM_SCALED: X is bf16(x * w), made by the product that last added into x (below), and
//    ss_in [n_ss][16] holds that product's per-tile sums of squares of each row; this kernel
//    adds them in tile order and scales its result.  Costs no more than the plain product.
// EMIT (with OUT_F32_ACCUM): after y += ..., the new y is also written as bf16(y * emit_nw[col])
// to emit_xw [M, N], and the tile's sums of squares of each row to emit_ss [tile][16], for the
// NORM_SCALED product that follows.
enum : int { NORM_NONE = 0, NORM_INSIDE = 1, NORM_SCALED = 2 };

// What the OUT_CONV epilogue needs beside the product: the taps [d][taps] (float32 or bfloat16), the
// float32 state [slots][taps - 1][d] and each row's slot.
constexpr int CONV_MAX_TAPS = 16;
struct ConvTail {
    const void* taps_w = nullptr; int taps_dt = DT_F32; int taps = 0;
    float* state = nullptr; const int* state_slot = nullptr;
    __device__ __forceinline__ float tap(int ch, int k) const {
        const long long i = (long long)ch * taps + k;
        return taps_dt == DT_F32 ? ((const float*)taps_w)[i] : (float)((const bf16_t*)taps_w)[i];
    }
};

// MT: row tiles of 16 (1: up to 16 rows, 2: up to 32).  With two, a wave multiplies every block of W
// with two tiles of X rows; the sums of squares that go from product to product then have 64 rows a tile
// in memory (SS_ROWS), as for every product of 17 to 64 rows.
constexpr int SS_ROWS_WIDE = 64;

// How many chunks the waves of a workgroup have: at most one; one or two; two or more.  Each is a kernel of its own, without
// the others' code and operands, and with the norm inside its barrier where every wave passes.
enum : int { SHARE_ONE = 0, SHARE_TWO = 1, SHARE_MANY = 2 };

// Waves a SIMD has to hold.  Eight waves over 32 columns: two workgroups a CU (at most 128 registers a lane), so that the 512
// workgroups of 16,384 columns run side by side and not in two rounds.
constexpr int skinny16_waves_a_simd(int NW, int COLS, int MT, int MODE, int SHARE) {
    return NW == 8 && COLS == 32 && MT == 1 && !(MODE == OUT_F32_ACCUM && SHARE == SHARE_MANY) ? 4 : 1;      // (that one would spill)
}

// XL: the rows of X lie in LDS, in whole.  A workgroup reads all of them either way; in the order of the operands every load of a
// wave touches sixteen rows for 64 bytes each, however few rows there are, and there are as many of them as loads of W.  As they
// lie, one row of 8,192 is one load a wave instead of sixteen.  At most so many pieces of 16 bytes a thread:
constexpr int skinny16_pieces(int MT) { return MT == 1 ? 9 : 12; }

template <int NW, int MODE, int NORM, bool EMIT, int COLS, int MT, int SHARE, bool XL>
__global__ __launch_bounds__(NW * WAVE, skinny16_waves_a_simd(NW, COLS, MT, MODE, SHARE)) void gemm_bf16_skinny16_kernel(const void* __restrict__ Xv, const bf16_t* __restrict__ W,
                                                                       void* __restrict__ Y, int M, int N, int K,
                                                                       const float* __restrict__ norm_w, float eps,
                                                                       const int* __restrict__ rows, long long ldx,
                                                                       const float* __restrict__ ss_in, int n_ss,
                                                                       const float* __restrict__ emit_nw,
                                                                       bf16_t* __restrict__ emit_xw, float* __restrict__ emit_ss,
                                                                       ConvTail cv) {
    constexpr bool CONV = MODE == OUT_CONV;
    // Neighbouring columns on one XCD (workgroups go round the eight of them) where all workgroups run side by side, of up to 16
    // columns each: 2,048 x 8,192 of 8 rows 9.9 -> 9.6 us, 2,048 x 2,048 4.7 -> 4.5.  Wider ones read enough of W by themselves and are faster
    // as the grid counts them (16,384 x 2,048 of 8 rows 13.4 us and 12.9); with two row tiles a decode step of 23 rows is 1 % slower.
    // All workgroups begin at the first chunk: beginning at chunks of their own was slower whatever the shape (65,536 x 2,048 of 8 rows
    // 44.9 -> 44.2, 32,768 x 2,048 25.8 -> 23.8, 6,144 x 2,048 of 32 rows 11.5 -> 11.1, 2,048 x 8,192 of 12 12.2 -> 11.7).
    const unsigned block = MT == 1 && COLS < 32 && gridDim.x <= 512 && gridDim.x % 8 == 0 ? blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    static_assert(!CONV || COLS == 8, "the convolution's epilogue takes eight channels a workgroup");
    static_assert(MT == 1 || NORM != NORM_INSIDE, "the norm inside is for at most 16 rows");
    constexpr int TN = CONV ? 3 : (COLS > 16 ? COLS / 16 : 1);           // MFMA tiles side by side: they share the rows of X
    static_assert(!EMIT || TN == 1, "the emitting epilogue works on one tile");
    constexpr int ROWS = 16 * MT;
    constexpr int SSR = MT == 1 ? 16 : SS_ROWS_WIDE;                     // rows of a tile of sums of squares in memory
    constexpr int NT_ = NW * WAVE;
    constexpr int PAIRS = (16 * ROWS + NT_ - 1) / NT_;                   // (row, part) sums a thread adds for NORM_SCALED
    __shared__ float red[MT][TN][NW][WAVE][4];
    __shared__ float ssq[16][ROWS];                                      // [wave or part][row]
    extern __shared__ __attribute__((aligned(16))) float nw_lds[];       // NORM_INSIDE: the norm weight, K floats
    bf16_t* const x_lds = (bf16_t*)nw_lds;                               // XL: [M][K + 8], eight zeros behind every row
    static_assert(!XL || NORM != NORM_INSIDE, "rows in LDS are bfloat16");
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int r16 = lane % 16, g = lane / 16;
    // OUT_CONV: workgroup b takes the channels 8 b .. 8 b + 7: half (b % 2) of the three row tiles of group b / 2
    const long long n0 = CONV ? (long long)(block / 2) * 48 + (block % 2) * 8 : (long long)block * COLS;
    const int nchunks = (K + SK_CHUNK - 1) / SK_CHUNK;
    const long long w_rows = min((long long)N, n0 + COLS);               // this tile's rows of W end here
    // tile-major W: this lane's piece of a block; a workgroup of 8 columns owns half a row tile
    const int kb = (K + 31) / 32, n_tiles16 = (N + 15) / 16;
    const long long tile0 = n0 / 16;
    const int wpiece = COLS == 8 ? g * 16 + (int)(n0 % 16) + r16 : lane;
    const bool wlane = COLS == 8 ? r16 < 8 : true;
    // NORM_INSIDE: this lane's row of x; a lane without one reads row 0 and its values count as zero
    const bool xlane = r16 < M;
    const int xr = NORM == NORM_INSIDE && xlane ? (rows ? rows[r16] : r16) : 0;
    const float* xrow = (const float*)Xv + (NORM == NORM_INSIDE ? (long long)xr * ldx : 0);

    // What the epilogue adds to is read now, not after the last product: a load at the end would
    // cost one more trip to memory.  (Thread t of every 256 -> element (row (t / 64) * 4 + t % 4,
    // column (t / 4) % 16) of a 16 x 16 tile; the groups of 256 threads take the row tiles in turn.)
    constexpr int EPI_GROUPS = NT_ / 256;                                // groups of 256 threads a workgroup
    constexpr int EPI_TILES = (MT + EPI_GROUPS - 1) / EPI_GROUPS;        // row tiles a group finishes
    float y_old[EPI_TILES][TN], emit_w = 0.f;
#pragma unroll
    for (int i = 0; i < EPI_TILES; ++i) {
        const int mt = tid / 256 + i * EPI_GROUPS;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
            y_old[i][tn] = 0.f;
            if (MODE == OUT_F32_ACCUM && mt < MT) {
                const int t = tid % 256;
                const long long row = mt * 16 + (t / 64) * 4 + t % 4, col = n0 + tn * 16 + (t / 4) % 16;
                if (row < M && col < w_rows) {
                    y_old[i][tn] = ((const float*)Y)[row * N + col];
                    if (EMIT) emit_w = emit_nw[col];
                }
            }
        }
    }

    // OUT_CONV: likewise the taps and the rows of the state that the convolution reads: the first CONV_AHEAD rows, which is
    // all of them up to a kernel length of CONV_AHEAD + 1, and the last tap.  Slot -> state are two trips to memory one after
    // the other: the slot is asked for before the first operands of the product and the state's rows behind them.
    constexpr int CONV_AHEAD = 4;
    float st_ahead[CONV ? EPI_TILES : 1][CONV_AHEAD], tap_ahead[CONV ? EPI_TILES : 1][CONV_AHEAD + 1];
    int slot_ahead[CONV ? EPI_TILES : 1];
    if constexpr (CONV) {
#pragma unroll
        for (int i = 0; i < EPI_TILES; ++i) {
            const int mt = tid / 256 + i * EPI_GROUPS, t = tid % 256, l = t / 4;
            const int row = mt * 16 + (l / 16) * 4 + t % 4, ch = (int)block * 8 + (l % 16), d = N / 3, Kc = cv.taps;
#pragma unroll
            for (int k = 0; k <= CONV_AHEAD; ++k) tap_ahead[i][k] = 0.f;
            slot_ahead[i] = cv.state_slot[min(row, M - 1)];
            if (mt < MT && (l % 16) < 8 && row < M && ch < d) {
#pragma unroll
                for (int k = 0; k < CONV_AHEAD; ++k)
                    if (k < Kc - 1) tap_ahead[i][k] = cv.tap(ch, k);
                tap_ahead[i][CONV_AHEAD] = cv.tap(ch, Kc - 1);
            }
        }
    }

    f32x4 acc[MT][TN];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[mt][tn] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
    struct Operands { bf16x8 a[XL ? 1 : MT][XL ? 1 : 4]; bf16x8 b[TN][4]; f32x4 x[NORM == NORM_INSIDE ? 4 : 1][2]; };
    Operands o0, o1;
    // The operands come through buffer loads; an offset beyond the buffer, for rows, columns and k that are not
    // there, reads as zero and fetches nothing.  With no branch around a load the compiler counts the loads under way and
    // waits for a chunk's own while the next one's are on their way; with the loads under conditions it waited for all.
    const int w_tiles = (int)min((long long)TN, n_tiles16 - tile0);
    const buffer_t wbuf = make_buffer(W + tile0 * kb * 512, w_tiles * kb * 1024);
    const buffer_t xbuf = make_buffer(Xv, NORM == NORM_INSIDE ? 0 : M * K * 2);
    const int w_at = wlane ? wpiece * 16 : NOWHERE;
    auto load = [&](int c, Operands& o) {
        // instruction j of the wave reads block 4 c + j of its row tile (1 KB) and bytes 64 j .. 64 j + 63 of
        // the chunk of each of the rows of X
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = tn < w_tiles && c * 4 + j < kb;
                o.b[tn][j] = load_buffer<true>(wbuf, in ? w_at : NOWHERE, in ? (tn * kb + c * 4 + j) * 1024 : 0);
            }
#pragma unroll
        for (int j = 0; j < (XL ? 0 : 4); ++j) {
            const int kj = c * SK_CHUNK + j * 32 + g * 8;
            if (COLS == 32 && MT == 1 && NORM != NORM_INSIDE) {
                // (lanes without a row are switched off: here, where the rows of X are half as many bytes as W, one that reads
                // nothing still takes its time: 16,384 x 2,048 of 1 row 14.4 us with them on, 13.7 off; narrower tiles no gain)
                o.a[0][j] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if (r16 < M) o.a[0][j] = load_buffer<false>(xbuf, kj < K ? (r16 * K + g * 8) * 2 : NOWHERE, min(c * SK_CHUNK + j * 32, K - 8) * 2);
            } else if (NORM == NORM_INSIDE) {
                const float* xp = xrow + min(kj, K - 8);
                o.x[j][0] = *(const f32x4*)xp;
                o.x[j][1] = *(const f32x4*)(xp + 4);
            } else {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    o.a[mt][j] = load_buffer<false>(xbuf, kj < K ? ((mt * 16 + r16) * K + g * 8) * 2 : NOWHERE, min(c * SK_CHUNK + j * 32, K - 8) * 2);
            }
        }
    };
    constexpr int PIECES = skinny16_pieces(MT);
    bf16x8 x_piece[XL ? PIECES : 1];
    const int n_pieces = XL ? M * K / 8 : 0;
    auto fetch_x = [&]() {
        if constexpr (XL) {
#pragma unroll
            for (int u = 0; u < PIECES; ++u)
                if (u * NT_ < n_pieces) x_piece[u] = load_buffer<false>(xbuf, (tid + u * NT_) * 16, 0);
        }
    };
    auto keep_x = [&]() {
        if constexpr (XL) {
            const unsigned per_row = (unsigned)K / 8, inverse = 0xFFFFFFFFu / per_row + 1;       // (exact for 2 to 2^16 a row, up to 2^16 pieces)
#pragma unroll
            for (int u = 0; u < PIECES; ++u)
                if (u * NT_ < n_pieces) {
                    const unsigned i = tid + u * NT_, row = __umulhi(i, inverse);
                    if (i < (unsigned)n_pieces) *(bf16x8*)(x_lds + 8 * (i + row)) = x_piece[u];
                }
            if (tid < M) *(bf16x8*)(x_lds + (tid + 1) * (K + 8) - 8) = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
            lds_barrier();
        }
    };
    auto multiply = [&](int c, Operands& o) {
        if constexpr (XL) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const bf16_t* row = x_lds + min(mt * 16 + r16, M - 1) * (K + 8);             // (no row: another one's, its result is not taken)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bf16x8 a = *(const bf16x8*)(row + min(c * SK_CHUNK + j * 32 + g * 8, K));
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn) acc[mt][tn] = mfma16(a, o.b[tn][j], acc[mt][tn]);
                }
            }
            return;
        }
        if (NORM == NORM_INSIDE) {
            const int k0 = c * SK_CHUNK + g * 8;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = min(k0 + j * 32, K - 8);
                const bool in = xlane && k0 + j * 32 < K;
                const f32x4 w0 = *(const f32x4*)(&nw_lds[k]), w1 = *(const f32x4*)(&nw_lds[k + 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x0 = in ? o.x[j][0][e] : 0.f, x1 = in ? o.x[j][1][e] : 0.f;
                    ss = fmaf(x0, x0, ss);
                    ss = fmaf(x1, x1, ss);
                    o.a[0][j][e] = (bf16_t)(x0 * w0[e]);
                    o.a[0][j][4 + e] = (bf16_t)(x1 * w1[e]);
                }
            }
        }
#pragma unroll
        for (int mt = 0; mt < (XL ? 0 : MT); ++mt)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[mt][tn] = mfma16(o.a[mt][j], o.b[tn][j], acc[mt][tn]);
    };
    // NORM_SCALED: 16 parts x ROWS rows; part p adds the tiles p, p + 16, ... of its row.  The first
    // sixteen of them are only asked for here and added after the products, when they have long
    // arrived; a wider matrix adds the rest right away.
    float ss_part[PAIRS][16], ss_rest[PAIRS];
    const buffer_t sbuf = make_buffer(ss_in, NORM == NORM_SCALED ? n_ss * SSR * 4 : 0);
    if (NORM == NORM_SCALED) {
#pragma unroll
        for (int q = 0; q < PAIRS; ++q) {
            const int pr = tid + q * NT_;
            ss_rest[q] = 0.f;
            if (n_ss > 256 && pr < 16 * ROWS)
                for (int j = pr / ROWS + 256; j < n_ss; j += 16) ss_rest[q] += ss_in[(long long)j * SSR + pr % ROWS];
        }
    }
    // What is asked for behind the first operands.
    auto behind = [&]() {
        if (NORM == NORM_SCALED) {
#pragma unroll
            for (int q = 0; q < PAIRS; ++q) {
                const int pr = tid + q * NT_;
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    ss_part[q][u] = load_buffer_float(sbuf, pr < 16 * ROWS ? ((pr / ROWS + 16 * u) * SSR + pr % ROWS) * 4 : NOWHERE, 0);
            }
        }
        if constexpr (CONV) {
#pragma unroll
            for (int i = 0; i < EPI_TILES; ++i) {
                const int t = tid % 256, l = t / 4, ch = (int)block * 8 + (l % 16), d = N / 3, Kc = cv.taps;
                const float* st = cv.state + (long long)slot_ahead[i] * (Kc - 1) * d + min(ch, d - 1);
#pragma unroll
                for (int k = 0; k < CONV_AHEAD; ++k) st_ahead[i][k] = st[(long long)min(k, Kc - 2) * d];
            }
        }
    };
    // The norm weight goes to LDS while the first operands are on their way from HBM.  (Holds a barrier: it stands where every
    // wave passes, whatever its number of chunks.)
    auto norm_weight = [&]() {
        for (int k = tid * 4; k < K; k += NW * WAVE * 4) *(f32x4*)(&nw_lds[k]) = *(const f32x4*)(norm_w + k);
        __syncthreads();
    };
    // The wave's chunks, two sets of operands in turn; every way through has its loads and products in straight order.
    const int n = (nchunks - wave + NW - 1) / NW;
    auto nth = [&](int i) { return wave + i * NW; };
    // Loads are issued where they stand.  Left alone, the instruction scheduler puts off the last ones of a chunk until the first
    // have arrived and their registers are free again: a second trip to memory (2,048 x 2,048, one chunk a wave, 1 row: 4.64 us,
    // with this 4.15; 16 rows 5.7 and 5.1).
    auto issued = [&]() { __builtin_amdgcn_sched_barrier(0); };
    if constexpr (SHARE == SHARE_ONE) {
        const int c = n > 0 ? nth(0) : nchunks;        // (a wave without a chunk, K up to 384: the one behind the last is all zeros)
        fetch_x();
        load(c, o0);
        issued();
        behind();
        issued();
        if constexpr (NORM == NORM_INSIDE) norm_weight();
        keep_x();
        multiply(c, o0);
    } else if constexpr (SHARE == SHARE_TWO && NORM == NORM_INSIDE) {
        load(nth(0), o0);
        if (n > 1) load(nth(1), o1);
        issued();
        behind();
        issued();
        norm_weight();
        multiply(nth(0), o0);
        if (n > 1) multiply(nth(1), o1);
    } else if constexpr (SHARE == SHARE_TWO) {
        static_assert(!XL, "rows in LDS: one chunk a wave or many");
        if (n > 1) {
            load(nth(0), o0);
            load(nth(1), o1);
            issued();
            behind();
            issued();
            multiply(nth(0), o0);
            multiply(nth(1), o1);
        } else {
            load(nth(0), o0);
            issued();
            behind();
            issued();
            multiply(nth(0), o0);
        }
    } else {
        // (two sets of operands over 32 columns and the sums of squares are more than 128 registers: there the sums are asked
        // for where one of the sets is used up)
        constexpr bool LATE = NORM == NORM_SCALED && COLS == 32;
        fetch_x();
        load(nth(0), o0);
        load(nth(1), o1);
        issued();
        if (!LATE) behind();
        issued();
        if constexpr (NORM == NORM_INSIDE) norm_weight();
        keep_x();
        int i = 0;
        for (; i + 3 < n; i += 2) {
            multiply(nth(i), o0);
            load(nth(i + 2), o0);
            issued();
            multiply(nth(i + 1), o1);
            load(nth(i + 3), o1);
            issued();
        }
        multiply(nth(i), o0);
        if (i + 2 < n) {
            load(nth(i + 2), o0);
            issued();
            multiply(nth(i + 1), o1);
            if (LATE) { issued(); behind(); issued(); }
            multiply(nth(i + 2), o0);
        } else {
            if (LATE) { issued(); behind(); issued(); }
            multiply(nth(i + 1), o1);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[mt][tn][wave][lane][e] = acc[mt][tn][e];
    if (NORM == NORM_SCALED) {
#pragma unroll
        for (int q = 0; q < PAIRS; ++q) {
            const int pr = tid + q * NT_;
            if (pr < 16 * ROWS) {
                float t = ss_rest[q];
#pragma unroll
                for (int u = 0; u < 16; ++u) t += ss_part[q][u];
                ssq[pr / ROWS][pr % ROWS] = t;
            }
        }
    }
    if (NORM == NORM_INSIDE) {
        ss = butterfly_sum<32>(butterfly_sum<16>(ss));
        if (g == 0) ssq[wave][r16] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int ei = 0; ei < EPI_TILES; ++ei) {
        const int mt = tid / 256 + ei * EPI_GROUPS;
        if (mt >= MT) break;
        // thread -> (lane l, element e) of each 16x16 tile; the wave partials in wave order
        const int t256 = tid % 256;
        const int e = t256 % 4, l = t256 / 4;
        const int trow = mt * 16 + (l / 16) * 4 + e;                     // the thread's row of the product
        float scale = 1.f;
        if (NORM != NORM_NONE) {
            constexpr int PARTS = NORM == NORM_INSIDE ? NW : 16;
            float total = ssq[0][trow];
#pragma unroll
            for (int w = 1; w < PARTS; ++w) total += ssq[w][trow];
            scale = 1.0f / sqrtf(total / (float)K + eps);
        }
        if constexpr (CONV) {
            // (row, channel): the three tiles hold B, C and X of the channel; the convolution as the kernel
            // for single tokens does it, on the values rounded to bfloat16 as a projected row would hold them
            float bcx[3];
#pragma unroll
            for (int tn = 0; tn < 3; ++tn) {
                float v = red[mt][tn][0][l][e];
#pragma unroll
                for (int w = 1; w < NW; ++w) v += red[mt][tn][w][l][e];
                if (NORM != NORM_NONE) v *= scale;
                bcx[tn] = (float)(bf16_t)v;
            }
            const int row = trow, d = N / 3, Kc = cv.taps;
            const int ch = (int)(block) * 8 + (l % 16);
            if ((l % 16) < 8 && row < M && ch < d) {
                float* st = cv.state + (long long)slot_ahead[ei] * (Kc - 1) * d;
                float sv[CONV_MAX_TAPS], wv[CONV_MAX_TAPS];
#pragma unroll
                for (int k = 0; k < CONV_MAX_TAPS; ++k) {
                    if (k < CONV_AHEAD) { sv[k] = st_ahead[ei][k]; wv[k] = tap_ahead[ei][k]; continue; }   // (not used beyond Kc - 1)
                    sv[k] = k < Kc - 1 ? st[(long long)k * d + ch] : 0.f;
                    wv[k] = k < Kc - 1 ? cv.tap(ch, k) : 0.f;
                }
                const float w_last = tap_ahead[ei][CONV_AHEAD];
                const float u = bcx[0] * bcx[2];
                float y = 0.f;
#pragma unroll
                for (int k = 0; k < CONV_MAX_TAPS; ++k)
                    if (k < Kc - 1) y = (k == 0) ? sv[k] * wv[k] : fmaf(sv[k], wv[k], y);
                y = fmaf(u, w_last, y);
#pragma unroll
                for (int k = 1; k < CONV_MAX_TAPS; ++k)
                    if (k < Kc - 1) st[(long long)(k - 1) * d + ch] = sv[k];
                st[(long long)(Kc - 2) * d + ch] = u;
                ((bf16_t*)Y)[(long long)row * d + ch] = (bf16_t)(bcx[1] * y);
            }
            continue;
        }
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
            float v = red[mt][tn][0][l][e];
#pragma unroll
            for (int w = 1; w < NW; ++w) v += red[mt][tn][w][l][e];
            const long long col = n0 + tn * 16 + (l % 16);
            const long long row = col < w_rows ? trow : ROWS;                // columns beyond the tile: no row
            if (NORM != NORM_NONE) v *= scale;
            if (EMIT) {
                // y += v; the new y also as the next norm's operand, and its square into the row's tile sum
                float y = 0.f;
                if (row < M && col < N) {
                    y = y_old[ei][tn] + v;
                    ((float*)Y)[row * N + col] = y;
                    emit_xw[row * N + col] = (bf16_t)(y * emit_w);
                }
                float sq = y * y;                       // t256 = (16 q + c) * 4 + e: the 16 columns c are its bits 2..5
                sq += __shfl_xor(sq, 4, WAVE);
                sq = butterfly_sum<32>(butterfly_sum<16>(butterfly_sum<8>(sq)));
                if ((l % 16) == 0 && row < ROWS) emit_ss[(long long)block * SSR + row] = sq;
            } else if (MODE == OUT_F32_ACCUM) {
                if (row < M && col < N) ((float*)Y)[row * N + col] = y_old[ei][tn] + v;
            } else {
                const float partner = (MODE == OUT_SWIGLU) ? __shfl_xor(v, 4, WAVE) : 0.f;   // thread t ^ 4 holds column col ^ 1
                store_elem<MODE>(Y, row, col, min(M, ROWS), N, v, partner);
            }
        }
    }
}

}  // namespace
#include "gemm_bf16_lean.h"
namespace {

// 16 < M <= 64.  grid (tiles of 64 columns, K slices).  Wave w owns columns 16w..16w+15 of the
// tile and all MT row tiles.  The X rows of a K chunk (128 wide) go through LDS once for the
// four waves, double buffered; the loads of two chunks are under way.  With more than
// one K slice, or when the epilogue has to leave the next norm's operand, the partial tiles go to
// a work space and splitk_finish_kernel adds them in slice order and does the epilogue.
// NORM_SCALED as above, with the sums of squares per tile of 64 columns: ss_in [n_ss][64].
constexpr int SK_NT = 256;
constexpr int XS_STRIDE = SK_CHUNK + 16;            // bf16 elements; 288 bytes, an odd multiple of 32: conflict-free 16-byte reads

template <int MT, int MODE, int NORM>
__global__ __launch_bounds__(SK_NT) void gemm_bf16_skinny64_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                   void* __restrict__ Y, int M, int N, int K, int chunks_per_slice,
                                                                   float* __restrict__ ws, bool to_ws,
                                                                   const float* __restrict__ ss_in, int n_ss, float eps) {
    static_assert(NORM != NORM_INSIDE, "the norm inside is for at most 16 rows");
    __shared__ __attribute__((aligned(16))) bf16_t xs[2][MT * 16 * XS_STRIDE];
    __shared__ float ss_parts[4][64];
    __shared__ float scale_lds[64];
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int r16 = lane % 16, g = lane / 16;
    const int tile = blockIdx.x, slice = blockIdx.y, n_slices = gridDim.y;
    const long long tile16 = (long long)tile * 4 + wave;                 // this wave's row tile of W
    const int kb = (K + 31) / 32;
    const bool tile_ok = tile16 < (N + 15) / 16;
    const int nchunks = (K + SK_CHUNK - 1) / SK_CHUNK;
    const int c_begin = slice * chunks_per_slice, c_end = min(nchunks, c_begin + chunks_per_slice);

    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // X chunk: MT*16 rows x 16 pieces of 16 bytes = MT*256 pieces, MT a thread.  Loads through buffers, at an offset beyond them
    // for what is not there: two chunks' operands are on their way and each is waited for by itself.
    const buffer_t xbuf = make_buffer(X, M * K * 2);
    const buffer_t wbuf = make_buffer(W + (tile_ok ? tile16 : 0) * kb * 512, tile_ok ? kb * 1024 : 0);
    bf16x8 x0[MT], x1[MT], b0[4], b1[4];
    auto load_x = [&](int c, bf16x8* xr) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int id = tid + i * SK_NT, k = c * SK_CHUNK + (id % 16) * 8;
            xr[i] = load_buffer<false>(xbuf, c < c_end && k < K ? (id / 16 * K + k) * 2 : NOWHERE, 0);
        }
    };
    auto store_x = [&](int buf, const bf16x8* xr) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int id = tid + i * SK_NT;
            *(bf16x8*)(&xs[buf][(id / 16) * XS_STRIDE + (id % 16) * 8]) = xr[i];
        }
    };
    auto load_w4 = [&](int c, bf16x8* b) {
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = load_buffer<true>(wbuf, c < c_end && c * 4 + j < kb ? lane * 16 : NOWHERE, c < c_end && c * 4 + j < kb ? (c * 4 + j) * 1024 : 0);
    };
    auto compute = [&](int buf, const bf16x8* b) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bf16x8 a = *(const bf16x8*)(&xs[buf][(i * 16 + r16) * XS_STRIDE + j * 32 + g * 8]);
                acc[i] = mfma16(a, b[j], acc[i]);
            }
    };

    if (c_begin < c_end) {
        load_x(c_begin, x0);
        load_w4(c_begin, b0);
        load_x(c_begin + 1, x1);
        load_w4(c_begin + 1, b1);
    }
    if (NORM == NORM_SCALED && !to_ws) {
        // thread -> (row tid % 64, part tid / 64): part p adds the tiles p, p + 4, ... of its row
        float t = 0.f;
        for (int j = tid / 64; j < n_ss; j += 4) t += ss_in[(long long)j * 64 + tid % 64];
        ss_parts[tid / 64][tid % 64] = t;
        __syncthreads();
        if (tid < 64)                                 // read in the epilogue, behind the barriers of the loop
            scale_lds[tid] = 1.0f / sqrtf((ss_parts[0][tid] + ss_parts[1][tid] + ss_parts[2][tid] + ss_parts[3][tid]) / (float)K + eps);
    }
    // Chunk c from buffer 0 / b0, chunk c + 1 from buffer 1 / b1.  The barriers wait for LDS only; a buffer is written again
    // behind the barrier of the chunk after it, which every wave reaches when it has used it.
    int c = c_begin;
    for (; c + 2 < c_end; c += 2) {
        store_x(0, x0);
        lds_barrier();
        load_x(c + 2, x0);
        compute(0, b0);
        load_w4(c + 2, b0);
        store_x(1, x1);
        lds_barrier();
        load_x(c + 3, x1);
        compute(1, b1);
        load_w4(c + 3, b1);
    }
    if (c < c_end) {
        store_x(0, x0);
        lds_barrier();
        compute(0, b0);
    }
    if (c + 1 < c_end) {
        store_x(1, x1);
        lds_barrier();
        compute(1, b1);
    }
    if (NORM == NORM_SCALED && !to_ws) lds_barrier();             // (a slice without a chunk has had no barrier)

    const long long col = (long long)tile * 64 + wave * 16 + r16;
    if (to_ws) {
        // partial tile of this slice: ws[slice][row][col]
        if (col >= N) return;
        float* mine = ws + (long long)slice * (MT * 16) * N;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[(long long)(i * 16 + g * 4 + e) * N + col] = acc[i][e];
        return;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const long long row = i * 16 + g * 4 + e;
            float v = acc[i][e];
            if (NORM == NORM_SCALED) v *= scale_lds[row];
            const float partner = (MODE == OUT_SWIGLU) ? lane_xor1(v) : 0.f;
            store_elem<MODE>(Y, row, col, M, N, v, partner);
        }
}

// Finishes a product whose partial tiles lie in the work space: v = sum over slices, in slice
// order, of ws[slice][row][col] (rows_padded rows a slice), scaled per row for NORM_SCALED, then the
// epilogue of MODE; with EMIT, Y += v and from the new Y the operand of the norm that follows, as
// in the kernel for at most 16 rows, with sums of squares per tile of 64 columns: emit_ss [tiles][64].
// grid (tiles of 64 columns, groups of 16 rows), 256 threads: thread -> row tid / 16 of the group and
// four neighbouring columns.
struct FinishExtra {
    const float* ss_in = nullptr; int n_ss = 0; float eps = 0.f; int K = 0;                 // NORM_SCALED
    const float* emit_nw = nullptr; bf16_t* emit_xw = nullptr; float* emit_ss = nullptr;   // EMIT
    int ss_rows = 64;                     // rows of a tile of sums of squares, read or written: 64, or M for the tiled product
};

template <int MODE, int NORM, bool EMIT>
__global__ __launch_bounds__(256) void splitk_finish_kernel(const float* __restrict__ ws, void* __restrict__ Y, int M, int N,
                                                            int rows_padded, int n_slices, FinishExtra ex) {
    static_assert(!EMIT || MODE == OUT_F32_ACCUM, "the emitting epilogue adds into the residual stream");
    // Slices asked for together, sixteen (all of them, as a rule) or, for the plain epilogues, eight (23 rows, 2,048 x 2,048: 7.13 us
    // with eight, 7.47 with sixteen, product and sum; 64 rows of 3,072 columns behind a norm 10.4 and 10.7)
    constexpr int TOGETHER = EMIT ? 16 : 8;
    const int tid = threadIdx.x, q = tid % 16;
    const long long row = (long long)blockIdx.y * 16 + tid / 16;
    const long long col = (long long)blockIdx.x * 64 + q * 4;
    float scale = 1.f;
    if (NORM == NORM_SCALED) {
        // the sixteen threads of a row add the tiles q, q + 16, ... and then each other, in a fixed butterfly
        float t = 0.f;
        if (row < ex.ss_rows)
            for (int j = q; j < ex.n_ss; j += 16) t += ex.ss_in[(long long)j * ex.ss_rows + row];
        t = row_sum_up(t);
        scale = 1.0f / sqrtf(t / (float)ex.K + ex.eps);
    }
    const bool whole = N % 4 == 0 && col + 3 < N;
    // What the emitting epilogue adds to and multiplies with is asked for ahead of the slices: behind them it would be another
    // trip to memory (23 rows, 2,048 columns, 16 slices of K = 8,192: 4.8 us, with them ahead 4.3).
    f32x4 y_old = {0.f, 0.f, 0.f, 0.f}, nw = {0.f, 0.f, 0.f, 0.f};
    const bool fours = EMIT && whole && (((uintptr_t)Y | (uintptr_t)ex.emit_nw) & 15) == 0 && ((uintptr_t)ex.emit_xw & 7) == 0;
    if (fours && row < M) {
        y_old = *(const f32x4*)((const float*)Y + row * N + col);
        nw = *(const f32x4*)(ex.emit_nw + col);
    }
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (row < M) {
        if (whole) {
            // the slices of a step of TOGETHER are asked for together and added in their order
            const long long stride = (long long)rows_padded * N;
            const float* p0 = ws + row * N + col;
            for (int s0 = 0; s0 < n_slices; s0 += TOGETHER) {
                f32x4 t[TOGETHER];
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u)
                    if (s0 + u < n_slices) t[u] = *(const f32x4*)(p0 + (s0 + u) * stride);
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u)
                    if (s0 + u < n_slices) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] += t[u][e];
                    }
            }
        } else {
            for (int s = 0; s < n_slices; ++s) {
                const float* p = ws + ((long long)s * rows_padded + row) * N + col;
#pragma unroll
                for (int e = 0; e < 4; ++e) if (col + e < N) v[e] += p[e];
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= scale;
    float sq = 0.f;
    if (row < M) {
        if (MODE == OUT_SWIGLU) {
            bf16_t* out = (bf16_t*)Y + row * (N / 2) + col / 2;
            if (col + 1 < N) out[0] = (bf16_t)silu_mul(v[0], v[1]);
            if (col + 3 < N) out[1] = (bf16_t)silu_mul(v[2], v[3]);
        } else if (fours) {
            f32x4 y;
            bf16x4 xw;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = y_old[e] + v[e];
                xw[e] = (bf16_t)(y[e] * nw[e]);
                sq = fmaf(y[e], y[e], sq);
            }
            *(f32x4*)((float*)Y + row * N + col) = y;
            *(bf16x4*)(ex.emit_xw + row * N + col) = xw;
        } else if (EMIT) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < N) {
                    const float y = ((const float*)Y)[row * N + col + e] + v[e];
                    ((float*)Y)[row * N + col + e] = y;
                    ex.emit_xw[row * N + col + e] = (bf16_t)(y * ex.emit_nw[col + e]);
                    sq = fmaf(y, y, sq);
                }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (col + e < N) store_out<MODE>(Y, row * N + col + e, v[e]);
        }
    }
    if (EMIT) {
        sq = row_sum_up(sq);
        if (q == 0 && row < ex.ss_rows) ex.emit_ss[(long long)blockIdx.x * ex.ss_rows + row] = sq;   // rows beyond M: zero
    }
}

// The same for the input projection of a gated short convolution over 17 to 64 single tokens (row r is
// request r's token): from the partial tiles of the projection [3 d] wide (B | C | X, as the checkpoint
// has them) the thread of (row, four channels) adds the slices of its twelve columns in slice order,
// scales and rounds them to bfloat16 as a projected row would hold them, and then does what the kernel
// for single tokens does: y = C * (taps . (state, B * X)), the state shifted by one.  The projected
// rows are never written.  grid (tiles of 64 channels, groups of 4 rows), one wave a workgroup: with twelve
// columns a thread there is three times the work of the kernel above in a thread, so more and smaller
// workgroups.  Two trips to memory one after the other remain (the row's slot, then its state beside the
// slices): 7.1 us at 64 rows of 2,048 channels, where the kernel above and the convolution's own took 9.5.
constexpr int FC_ROWS = 4;
template <int NORM>
__global__ __launch_bounds__(FC_ROWS * 16) void splitk_finish_conv_kernel(const float* __restrict__ ws, bf16_t* __restrict__ Y, int M, int d,
                                                                 int rows_padded, int n_slices, FinishExtra ex, ConvTail cv) {
    const int tid = threadIdx.x, q = tid % 16;
    const long long row = (long long)blockIdx.y * FC_ROWS + tid / 16;
    const long long ch0 = (long long)blockIdx.x * 64 + q * 4;
    const int N = 3 * d;
    float scale = 1.f;
    if (NORM == NORM_SCALED) {
        float t = 0.f;
        if (row < ex.ss_rows)
            for (int j = q; j < ex.n_ss; j += 16) t += ex.ss_in[(long long)j * ex.ss_rows + row];
        t = row_sum_up(t);
        scale = 1.0f / sqrtf(t / (float)ex.K + ex.eps);
    }
    if (row >= M || ch0 >= d) return;                      // d is a multiple of 16: four channels or none
    // The state's rows and the taps are asked for now, before the slices: they depend on nothing that is
    // computed here, and a load at the end would cost another trip to memory.  (Up to four older rows are
    // kept in registers; a longer convolution reads the rest when it needs them.)
    const int Kc = cv.taps;
    float* st = cv.state + (long long)cv.state_slot[row] * (Kc - 1) * d;
    constexpr int KEEP = 4;
    f32x4 sv[KEEP];
    float wv[KEEP + 1][4];
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
        sv[k] = k < Kc - 1 ? *(const f32x4*)(st + (long long)k * d + ch0) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) wv[k][e] = k < Kc - 1 ? cv.tap((int)ch0 + e, k) : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) wv[KEEP][e] = cv.tap((int)ch0 + e, Kc - 1);
    float v[3][4];
    const long long stride = (long long)rows_padded * N;
#pragma unroll
    for (int part = 0; part < 3; ++part) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[part][e] = 0.f;
        const float* p0 = ws + row * N + (long long)part * d + ch0;
        for (int s0 = 0; s0 < n_slices; s0 += 8) {         // as the kernel above: eight slices asked for together, added in order
            f32x4 t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < n_slices) t[u] = *(const f32x4*)(p0 + (s0 + u) * stride);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < n_slices) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[part][e] += t[u][e];
                }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[part][e] = (float)(bf16_t)(v[part][e] * scale);
    }
    f32x4 y, u4;
#pragma unroll
    for (int e = 0; e < 4; ++e) { u4[e] = v[0][e] * v[2][e]; y[e] = 0.f; }
    // y = taps . (state rows in order, then u), one chain of operations a channel; row k moves to k - 1
#pragma unroll
    for (int k = 0; k < KEEP; ++k)
        if (k < Kc - 1) {
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = (k == 0) ? sv[k][e] * wv[k][e] : fmaf(sv[k][e], wv[k][e], y[e]);
            if (k > 0) *(f32x4*)(st + (long long)(k - 1) * d + ch0) = sv[k];
        }
    for (int k = KEEP; k < Kc - 1; ++k) {
        const f32x4 s4 = *(const f32x4*)(st + (long long)k * d + ch0);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = fmaf(s4[e], cv.tap((int)ch0 + e, k), y[e]);
        *(f32x4*)(st + (long long)(k - 1) * d + ch0) = s4;
    }
    bf16x4 o4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        y[e] = fmaf(u4[e], wv[KEEP][e], y[e]);
        o4[e] = (bf16_t)(v[1][e] * y[e]);
    }
    *(f32x4*)(st + (long long)(Kc - 2) * d + ch0) = u4;
    *(bf16x4*)(Y + row * d + ch0) = o4;
}

struct SkinnyPlan { int tiles, waves, slices, chunks_per_slice, cols; long long ws_floats; };

// The kernels count bytes inside a buffer, which is a block's rows of X or of W, in 31 bits: 64 rows at most in those for few rows,
// 256 in the tiled one that loads straight into LDS.  The one through registers counts elements in 32.
constexpr int LARGEST_K = (1 << 24) - 64, LARGEST_K_DMA = (1 << 22) - TBK;
bool inner_ok(int K) { return K % 8 == 0 && K <= LARGEST_K; }
bool dma_ok(int K) { return K % TBK == 0 && K <= LARGEST_K_DMA; }

constexpr int SKINNY_ROWS = 32;     // the most rows of the kernel whose waves split K inside the workgroup (two row tiles)

// 17 to 64 rows and a wide output with a short K (gate and up of a feed-forward): the tiled product with one
// block of 64 x 64 for every 64 columns gives every CU a workgroup without slices of K, so no second kernel
// adds partial tiles, and its time is that of streaming W whatever the rows.  Measured against the two ways
// for few rows, SwiGLU epilogue, 17 to 64 rows: 16,384 x 2,048 18 to 22 us -> 15.5 to 16.5, 13,824 x 1,536 14 to
// 17 -> 11.5, 9,216 x 1,536 12 to 14 -> 11, 24,576 x 2,048 26 to 28.5 -> 24 to 27; no gain at 6,144 and 8,192
// columns nor at 32,768.
int wide64_min_n = 9216, wide64_max_n = 24576, wide64_min_m = 17;      // measurements may move them
bool wide64_shape(int N, int K) { return N >= wide64_min_n && N <= wide64_max_n && K % TBK == 0 && K / TBK <= 48; }
bool rows64_tiled(int M, int N, int K) { return M >= wide64_min_m && M <= 64 && wide64_shape(N, K); }

// Whether a product of M rows goes through that kernel (else, up to 64 rows: K cut over workgroups and a
// second kernel that adds the slices).  Up to 16 rows always.  17 to 32 rows: every workgroup reads all M
// rows of X again, M / (its columns) times the bytes of its share of W, and has half the waves.  Measured
// on the shapes of a 1.2B model (against the two kernels of the other way, at 32 rows): 3,072 columns 8.8 us
// against 10.7, a conv's input projection with the convolution 12.5 against 15.2, 16,384 columns 21.7 against
// 21.3, 65,536 columns 67.7 against 52.2, at 17 rows it wins.  So: medium outputs up to 32 rows, wide ones up to 24 (where
// the tiled product does not take them, above).  Outputs of up to 2,048 columns: up to 20 rows with a short K, where the
// second launch costs more than the rows read again (20 rows, this way and the other: 1,024 x 1,024 4.1 us and 5.1, 2,048 x
// 1,024 4.3 and 5.3, 2,048 x 2,048 5.7 and 6.2, 2,048 x 3,072 8.2 and 7.3, x 8,192 16.2 and 11.4), at 32 rows it
// loses from K = 1,024 on (2,048 x 2,048 7.5 and 7.3).  One that leaves the next norm its sums leaves a group a workgroup,
// up to 256 instead of 32, which the product after it adds up: only up to K = 1,024 (1,024 x 1,024 and a product of 3,072
// columns behind it 9.4 and 11.1, 2,048 x 2,048 14.1 and 13.9).
// Less than 1,024 columns are too few workgroups for K = 2,048 (512 columns 5.5 and 5.2).
constexpr int NARROW_SHORT_K = 2048, NARROW_SHORT_K_EMIT = 1024;
bool few_rows_kernel(int M, int N, int K, bool conv = false, bool emit = false) {
    if (M <= 16) return true;
    if (M > SKINNY_ROWS) return false;
    if (conv) return true;
    if (rows64_tiled(M, N, K)) return false;
    return N <= 2048 ? M <= 20 && K <= (emit || N < 1024 ? NARROW_SHORT_K_EMIT : NARROW_SHORT_K) : N <= 8192 ? true : M <= 24;
}

// How a skinny product is cut.  Depends on N and K (and on which of the two kernels M selects).
SkinnyPlan plan_skinny(int M, int N, int K, int max_waves = 16, bool emit = false, bool conv = false) {
    const int nchunks = ceil_div(K, SK_CHUNK);
    SkinnyPlan p;
    p.slices = 1; p.chunks_per_slice = nchunks; p.ws_floats = 0; p.waves = 4;
    p.cols = 16;
    if (few_rows_kernel(M, N, K, conv, emit)) {
        // Narrow outputs: tiles of 8 columns, where 16 would leave CUs without a workgroup (half of
        // each MFMA idles, which costs nothing here: these products wait for memory).  Wide outputs:
        // 32 or 64 columns, whose MFMA tiles share the rows of X: with 16 columns the rows of X
        // (from the L2, again for every workgroup) are up to as many bytes again as the weights.
        const int tiles16 = ceil_div(N, 16);
        if (tiles16 <= 128) p.cols = 8;
        else if (tiles16 >= 4096) p.cols = 64;
        else if (tiles16 >= 512) p.cols = 32;
        if ((max_waves < 16 || emit) && p.cols > 16) p.cols = 16;       // the norm inside keeps float32 rows in registers (an output head: launch_skinny16);
                                                                        // the emitting epilogue works on one tile
        if (M > 16) {
            // two row tiles: twice the operands of X a wave, so at most two tiles of W side by side and eight waves
            p.cols = min(p.cols, 32);
            max_waves = min(max_waves, 8);
        }
        p.tiles = ceil_div(N, p.cols);
        // enough waves in flight to cover the latency of HBM, at least one chunk a wave
        while (p.waves < max_waves && p.tiles * p.waves < 3072 && nchunks >= 2 * p.waves) p.waves *= 2;
    } else {
        const int mt = ceil_div(M, 16);
        p.tiles = ceil_div(N, 64);
        int s = ceil_div(512, p.tiles);
        s = max(1, min(s, nchunks / 2));
        p.chunks_per_slice = ceil_div(nchunks, s);
        p.slices = ceil_div(nchunks, p.chunks_per_slice);
        p.ws_floats = (p.slices > 1 || emit) ? (long long)p.slices * mt * 16 * N : 0;
    }
    return p;
}

// How a product of more than 64 rows is cut: shape 0: 256 x 256 blocks; 1: 128 x 128 blocks, two a CU;
// 2: 128 x 128 blocks, one a CU, four steps of operands under way; 3: 64 x 64 blocks of four waves;
// 4: 256 x 192 blocks; 5: 128 x 256 blocks, three steps under way; 6: 64 x 128 blocks of four waves.
// Depends on the sizes only.  One slice of fewer steps than K has: the block adds the slices itself (shape 3).
struct TiledPlan { int shape, slices, steps_per_slice; long long ws_floats; };

int tiled_shape_forced = -1;       // >= 0: every tiled product takes this shape (measurements only)

TiledPlan plan_tiled(int M, int N, int K) {
    const long long large = (long long)ceil_div(N, 256) * ceil_div(M, 256);
    const long long small = (long long)ceil_div(N, 128) * ceil_div(M, 128);
    const int nk = ceil_div(K, TBK);
    TiledPlan t;
    t.shape = large >= 160 ? 0 : small > 256 ? 1 : 2;
    t.slices = 1; t.steps_per_slice = nk; t.ws_floats = 0;
    if (tiled_shape_forced >= 0 && dma_ok(K)) { t.shape = tiled_shape_forced; return t; }
    if ((t.shape == 0 || (t.shape == 1 && small > 512)) && dma_ok(K)) {
        const long long wide = (long long)ceil_div(N, 192) * ceil_div(M, 256);
        // blocks of 256 x 192 where they need fewer rounds of 256 workgroups times columns than 256 x 256
        // (6144 columns and 2048 rows: 256 blocks, one round, instead of 192 blocks that leave a quarter of the CUs idle), and for
        // a little more than one round of pairs of 128 x 128 blocks (512 of them side by side), where the blocks beyond the round
        // would run a second one almost alone (4608 columns and 2048 rows, K = 1536: 37.1 us instead of 43.8; 256 x 256: 45.7)
        if (t.shape == 0 ? ceil_div(wide, 256) * 192 < ceil_div(large, 256) * 256 : wide <= 256) t.shape = 4;
        // Whole blocks of 128 x 256: the shape whose rounds cost least, of 256 x 256, 256 x 192 and 128 x 256 blocks, as measured a
        // round and step 1.72, 1.39 and 0.97 us (alike with 1,536 to 8,192 of K; a smaller block reads its operands for
        // fewer products).  Halves of a round instead of a round almost empty: 1,050 rows 13,824 x 1,536 64.5 -> 48.7 us, 21,504 x 2,048 106 ->
        // 96, 1,300 rows 16,384 x 2,048 108 -> 90, 1,536 109 -> 94; 256 x 192 instead of 256 x 256, 1,050 rows, 96.5 -> 84.
        if (N % 256 == 0) {
            const long long cost0 = 17 * ceil_div(large, 256), cost4 = 14 * ceil_div(wide, 256);
            const long long cost5 = 10 * ceil_div((long long)(N / 256) * ceil_div(M, 128), 256);
            t.shape = cost5 < cost0 && cost5 < cost4 ? 5 : cost4 < cost0 ? 4 : 0;
        }
        return t;
    }
    // One round of 128 x 256 blocks in the place of one of pairs of 128 x 128, which read an operand once more and wait for it: 2,048 x 8,192
    // of 2,560 rows 112 -> 103 us, 4,096 131 -> 110; 3,072 x 2,048 of 1,536 rows 32.0 -> 30.1, 2,048 33.4 -> 30.9; 2,048 x 2,048 of 2,560
    // rows into the stream 40.1 -> 37.3; 13,824 x 1,536 with SwiGLU of 512 rows 30.7 -> 28.9, 400 29.4 -> 26.7, 384 27.8 and 28.0.
    if (t.shape == 1 && dma_ok(K) && N % 256 == 0) { t.shape = 5; return t; }
    // few blocks and a short K: blocks of 64 x 64 give enough workgroups without slices of K, whose partial
    // tiles cost a second kernel and as much traffic as the product's own (K = 1536 .. 2048, 96 to 512
    // rows: 9 to 14 us instead of 11 to 19); beyond 48 steps the slices win
    const long long least = (long long)ceil_div(N, 64) * ceil_div(M, 64);
    if (t.shape == 2 && small <= 128 && dma_ok(K) && nk <= 48) {
        // where they are well beyond a round, one block of 64 x 128 a CU: the second round's blocks take as long as the first's (64 x 64 and
        // 64 x 128, us: 400 rows, 4,608 x 1,536 (504 blocks of 64 x 64) 14.3 and 11.2, 300 rows, 6,144 x 2,048 (480) 17.7 and 16.5, 100 rows,
        // 16,384 x 2,048 (512) 22.2 and 20.3; 512 rows, 2,560 x 1,536 (320) 11.7 and 13.0, 256 rows, 5,632 x 2,048 (352) 15.2 and 17.5, 512
        // rows, 3,072 x 2,048 (384) 14.4 and 15.8, 400 rows, 3,584 x 2,048 (392) 14.4 and 14.6)
        t.shape = least > 400 && N % 128 == 0 && (long long)(N / 128) * ceil_div(M, 64) <= 256 ? 6 : 3;
        return t;
    }
    if (t.shape == 2 && small <= 128) {
        // as many slices as give every CU at most one block, at least eight steps a slice
        int s = max(1, min((int)(256 / small), nk / 8));
        t.steps_per_slice = ceil_div(nk, s);
        t.slices = ceil_div(nk, t.steps_per_slice);
        // A longer K still in blocks of 64 x 64 that add the slices themselves, where the partial tiles would cost more (their bytes grow
        // with rows and columns, a block's time with K).  Slices and 64 x 64 into the residual stream, us: 2,048 x 3,584 of 100 rows 13.6 and
        // 14.0, 200 16.1 and 14.4, 512 19.9 and 15.9; x 4,096 of 100 rows 14.5 and 14.9, 200 16.4 and 15.4, 512 20.4 and 16.9; x 5,632 of 300
        // rows 19.2 and 20.3, 400 21.4 and 20.9, 512 24.5 and 21.8; 1,536 x 6,912 of 300 rows 21.7 and 22.9, 600 27.0 and 24.6;
        // 2,048 x 8,192 of 400 rows 25.2 and 28.1, 512 28.6 and 29.2.
        if (dma_ok(K) && N % 64 == 0 && least <= 256 && 2 * least > 5 * (nk - 24)) { t.shape = 3; t.slices = 1; return t; }
        if (t.slices > 1) t.ws_floats = (long long)t.slices * M * N;
    }
    return t;
}

// Which loads the kernel straight into LDS takes (see there).  Measured through buffers and globally, us: blocks of 64 x 64, up to
// one a CU 9.7 and 10.0 (300 rows, 2,560 x 2,560), 8.7 and 9.0 (500, 2,048 x 2,048), more 13.6 and 12.8 (400, 2,560 x 2,560), 12.3
// and 11.8 (512, 2,560 x 2,048), but two on every CU 16.7 and 17.2 (512, 4,096 x 2,048); 128 x 128, one a CU, K = 2,048 16.1 and 17.6 (1,024 rows, 2,048 columns), K = 5,632 48.2 and 47.2, K =
// 6,912 58.4 and 56.2; 256 x 192 45.0 and 43.7 (1,500, 6,144 x 2,048), 35.7 and 34.0 (2,048, 4,608 x 1,536); 256 x 256 111.7 and 114.2 (2,048,
// 16,384 x 2,048); 128 x 128, two a CU, within 1 %.
bool dma_through_buffer(const TiledPlan& t, int M, int N) {
    if (t.shape == 4) return false;
    if (t.shape == 5 || t.shape == 6) return true;
    if (t.shape == 3) {
        const long long blocks = (long long)ceil_div(M, 64) * ceil_div(N, 64);
        return blocks <= 256 || blocks > 448;
    }
    return t.shape != 2 || t.steps_per_slice <= 64;
}

// The order of the blocks of 256 rows or columns.  As the grid counts them an XCD takes every eighth: the same columns again and again
// where their number is a multiple of eight, else a new mixture a row, and each XCD's L2 reads nearly all of W.  In bands of
// eight row blocks an XCD has neighbours in both directions.  As counted / in bands, us: 1,050 rows, 16,384 x 2,048 (86 blocks
// of columns) 96.2 and 84.0; 20,001 rows, 13,824 x 1,536 791 and 741, 6,144 x 2,048 512 and 461, 2,048 x 2,048 171 and 160; 8,192 rows,
// 2,048 x 8,192 241 and 200.  Few rows and a multiple of eight: 3,000 rows, 6,144 x 2,048 81.0 and 83.9, 520 rows, 16,384 x 2,048 53.4 and
// 54.6.  The smaller blocks lose (128 x 128 2 to 5 % up to 2,000 rows, 64 x 64 up to 10).
bool bands_of_rows(const TiledPlan& t, int M, int N) {
    if (t.shape != 0 && t.shape != 4 && t.shape != 5) return false;
    return ceil_div(N, t.shape == 4 ? 192 : 256) % 8 != 0 || ceil_div(M, t.shape == 5 ? 128 : 256) >= 16;
}

struct Skinny16Extra {
    const float* norm_w = nullptr; float eps = 0.f; const int* rows = nullptr; long long ldx = 0;       // NORM_INSIDE (ldx: rows of X that far apart)
    const float* ss_in = nullptr; int n_ss = 0;                                      // NORM_SCALED (+ eps)
    const float* emit_nw = nullptr; bf16_t* emit_xw = nullptr; float* emit_ss = nullptr;   // EMIT
    ConvTail conv;                                                                   // OUT_CONV
};

// LDS that is left for the rows of X beside the partial sums (up to 16 columns a workgroup).
constexpr int skinny16_lds_left(int NW, int MT) { return 160 * 1024 - MT * NW * 1024 - 16 * 16 * MT * 4; }
// Where the waves have many chunks, X goes through LDS as far as it fits; where they have one each, a barrier before its product
// costs a few rows more than it saves.  Rows from memory / in LDS, us: 2,048 x 8,192 of 1 row 8.9 and 7.8, 4 9.2 and 8.1, 8 9.6 and
// 8.8; one chunk a wave, 2,048 x 2,048 of 1 row 4.2 and 4.3, 8 4.5 and 4.4, 16 5.2 and 4.7, 3,072 x 2,048 4.8 and 5.2, 5.4 and 5.5, 6.0
// and 5.7; two row tiles, 17 rows, 3,072 x 2,560 6.9 and 6.0, 6,144 x 2,560 11.7 and 10.3, 20 rows, 8,176 x 2,304 12.2 and 11.1.  (Two
// chunks a wave lose: 6,144 x 2,048 with the convolution 7.5 and 8.1, 16,384 x 2,048 13.0 and 13.1.)
bool skinny16_rows_in_lds(int NW, int MT, int SHARE, int M, int K) {
    if (K < 256 || (SHARE == SHARE_ONE && M <= 8)) return false;
    return (long long)M * (K + 8) * 2 <= skinny16_lds_left(NW, MT) && (long long)M * K / 8 <= (long long)skinny16_pieces(MT) * NW * WAVE;
}

// The waves of the product with the convolution in its epilogue, eight channels a workgroup (three half tiles); they split K as
// always, at most eight of them: sixteen would leave a wave 128 registers, too few for three tiles' operands of two chunks.
int skinny16_conv_waves(int N, int K) {
    const int groups = N / 3 / 8, chunks = ceil_div(K, SK_CHUNK);
    int waves = 4;
    while (waves < 8 && groups * waves < 3072 && chunks >= 2 * waves) waves *= 2;
    return waves;
}

// Whether the kernel for sizes that divide evenly takes a product (cut as p says), and launches it: 1 launched, 0 not taken, else an
// error (negative).  Chunks a wave: up to six, whose operands are all under way at once; SwiGLU and the convolution, with two and three
// tiles of W, two.  From three on X lies in LDS whole or the product is not taken: into the stream up to 8 rows of K = 8,192, 10 of
// 6,912, 6 of 10,752.
template <int MODE, int NORM, bool EMIT>
int launch_lean16(const SkinnyPlan& p, const void* X, const bf16_t* W, void* Y, int M, int N, int K, const Skinny16Extra& x, hipStream_t stream) {
    constexpr bool CONV = MODE == OUT_CONV, SCALED = NORM == NORM_SCALED;
    const int chunks = K / SK_CHUNK, share = ceil_div(chunks, p.waves), grid = CONV ? N / 24 : N / p.cols;
    if (M > 16 || K % SK_CHUNK != 0 || chunks < 8 || (!CONV && N % p.cols != 0) || grid > 8192 || share > 6) return 0;
    if (SCALED && (x.n_ss > 256 || (uintptr_t)x.ss_in % 16 != 0)) return 0;      // (sums of squares go into LDS in pieces of 16 bytes)
    // Rows of X in LDS: see skinny16_rows_in_lds.
    const bool rows_in_lds = share > 2 || (share == 1 && M > 8 && p.cols < 32 && !CONV);
    constexpr int static_lds = 16 * 1024 + (SCALED ? 17 * 1024 + 512 : 512), lds_left = 160 * 1024 - static_lds;
    const int lds = rows_in_lds ? M * (K + 8) * (int)sizeof(bf16_t) : 0;
    if (rows_in_lds && (lds > lds_left || p.cols > 16 || CONV)) return 0;
    Lean16Args a;
    a.X = (const bf16_t*)X; a.W = W; a.Y = Y; a.ss_in = x.ss_in; a.emit_nw = x.emit_nw; a.emit_xw = x.emit_xw; a.emit_ss = x.emit_ss;
    a.M = M; a.N = N; a.K = K; a.n_ss = x.n_ss; a.eps = x.eps;
    a.per_xcd = (CONV || p.cols < 32) && grid <= 512 && grid % 8 == 0 ? grid / 8 : 0;
    a.pieces_inverse = 0xFFFFFFFFu / (unsigned)ceil_div(K, 512) + 1;
    a.cv = x.conv;
#define LEAN(NW, COLS, CH, XL) do { \
        auto kern = gemm_bf16_lean16_kernel<NW, MODE, SCALED, EMIT, COLS, CH, XL>; \
        if constexpr (XL) { \
            static bool set = false; \
            if (!set) { \
                if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_left) != hipSuccess) return -1; \
                set = true; \
            } \
        } \
        hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * WAVE), lds, stream, a); \
        return 1; \
    } while (0)
    if constexpr (CONV) {
        if (p.waves != 8) return 0;
        if (share == 1) LEAN(8, 8, 1, false);
        if (share == 2) LEAN(8, 8, 2, false);
    } else if constexpr (MODE == OUT_SWIGLU) {
        if (p.waves == 8 && p.cols == 32) {
            if (share == 1) LEAN(8, 32, 1, false);
            if (share == 2) LEAN(8, 32, 2, false);
        }
    } else {
#define LEAN_COLS(NW, COLS) do { \
        if (share == 1) { if (rows_in_lds) LEAN(NW, COLS, 1, true); else LEAN(NW, COLS, 1, false); } \
        else if (share == 2) LEAN(NW, COLS, 2, false); \
        else if (share <= 4) LEAN(NW, COLS, 4, true); \
        else LEAN(NW, COLS, 6, true); \
    } while (0)
        if (p.cols == 8) { if (p.waves == 8) LEAN_COLS(8, 8); else if (p.waves == 16) LEAN_COLS(16, 8); }
        else if (p.cols == 16) { if (p.waves == 8) LEAN_COLS(8, 16); else if (p.waves == 16) LEAN_COLS(16, 16); }
#undef LEAN_COLS
    }
#undef LEAN
    return 0;
}

template <int MODE, int NORM, bool EMIT>
int launch_skinny16(const void* X, const bf16_t* W, void* Y, int M, int N, int K, const Skinny16Extra& x, hipStream_t stream) {
    // the in-kernel norm needs more registers a wave: at most 8 waves a workgroup
    SkinnyPlan p = plan_skinny(M, N, K, NORM == NORM_INSIDE ? 8 : 16, EMIT, MODE == OUT_CONV);
    size_t lds = NORM == NORM_INSIDE ? (size_t)K * sizeof(float) : 0;
    const int mt = M > 16 ? 2 : 1, chunks = ceil_div(K, SK_CHUNK);
    if constexpr (MODE == OUT_CONV) p.waves = skinny16_conv_waves(N, K);
    if constexpr (NORM == NORM_INSIDE && MODE == OUT_F32) {
        // An output head behind the norm, four waves a workgroup: wide tiles, whose workgroups read and norm the rows fewer times, as float32
        // twice the bytes that the other products read.  16 columns a workgroup / wide ones, us: 65,536 x 2,048 of 1 row 47.7 / 45.2, 8 rows 61.3 /
        // 47.3, 16 rows 83.2 / 51.7; 32,768 x 2,048 27.1 / 24.5, 33.1 / 26.6 and 43.2 / 31.7.  Up to three rows of a short K have nothing to save
        // (65,536 x 1,024 of 2 rows 25.0 / 25.3, 16 rows 42.3 / 28.9); 16,384 columns are too few workgroups (1 row 15.9 / 24.0).  The waves cut K as before: the same bits.
        if (p.cols == 16 && p.waves == 4 && p.tiles >= 1536 && (M > 3 || K >= 1536)) {
            p.cols = p.tiles >= 4096 ? 64 : 32;
            p.tiles = ceil_div(N, p.cols);
        }
    }
    if constexpr ((NORM == NORM_SCALED && (MODE == OUT_BF16 || MODE == OUT_SWIGLU || MODE == OUT_CONV)) || EMIT) {
        const int rc = launch_lean16<MODE, NORM, EMIT>(p, X, W, Y, M, N, K, x, stream);
        if (rc) return rc < 0 ? rc : launch_status();
    }
#define GO_XL(NW, COLS, MT, SHARE, XL) hipLaunchKernelGGL((gemm_bf16_skinny16_kernel<NW, MODE, NORM, EMIT, COLS, MT, SHARE, XL>), grid, dim3(NW * WAVE), lds, stream, \
                                        X, W, Y, M, N, K, x.norm_w, x.eps, x.rows, x.ldx ? x.ldx : (long long)K, x.ss_in, x.n_ss, x.emit_nw, x.emit_xw, x.emit_ss, \
                                        x.conv)
#define GO_SHARE(NW, COLS, MT, SHARE) do { \
        if constexpr (NORM != NORM_INSIDE && COLS < 32 && MODE != OUT_CONV && (SHARE == SHARE_MANY || (SHARE == SHARE_ONE && MT == 1))) { \
            if (skinny16_rows_in_lds(NW, MT, SHARE, M, K)) { \
                lds = (size_t)M * (K + 8) * sizeof(bf16_t); \
                static bool set = false; \
                if (!set) { \
                    if (hipFuncSetAttribute((const void*)gemm_bf16_skinny16_kernel<NW, MODE, NORM, EMIT, COLS, MT, SHARE, true>, \
                                            hipFuncAttributeMaxDynamicSharedMemorySize, skinny16_lds_left(NW, MT)) != hipSuccess) return -1; \
                    set = true; \
                } \
                GO_XL(NW, COLS, MT, SHARE, true); \
                break; \
            } \
        } \
        GO_XL(NW, COLS, MT, SHARE, false); \
    } while (0)
#define GO_MT(NW, COLS, MT) do { \
        if (chunks <= NW) GO_SHARE(NW, COLS, MT, SHARE_ONE); \
        else if (chunks <= 2 * NW) GO_SHARE(NW, COLS, MT, SHARE_TWO); \
        else GO_SHARE(NW, COLS, MT, SHARE_MANY); \
    } while (0)
#define GO(NW, COLS) do { \
        if (mt == 1) GO_MT(NW, COLS, 1); \
        else if constexpr (NW <= 8 && COLS <= 32 && NORM != NORM_INSIDE) GO_MT(NW, COLS, 2); \
        else return -3; \
    } while (0)
#define GO16(COLS) do { if constexpr (NORM != NORM_INSIDE) GO(16, COLS); else return -3; } while (0)
    if constexpr (MODE == OUT_CONV) {
        dim3 grid(N / 3 / 8);
        if (p.waves == 4) GO(4, 8); else GO(8, 8);
    } else {
        dim3 grid(p.tiles);
        if (p.cols == 16) { if (p.waves == 4) GO(4, 16); else if (p.waves == 8) GO(8, 16); else GO16(16); }
        else if (p.cols == 8) { if (p.waves == 4) GO(4, 8); else if (p.waves == 8) GO(8, 8); else GO16(8); }
        else if constexpr (!EMIT && NORM != NORM_INSIDE) {
            if (p.cols == 32) { if (p.waves == 4) GO(4, 32); else if (p.waves == 8) GO(8, 32); else GO(16, 32); }
            else if (p.cols == 64 && p.waves == 4) GO(4, 64);      // (1,024 tiles or more: four waves)
            else return -3;
        } else if constexpr (NORM == NORM_INSIDE && MODE == OUT_F32) {
            if (p.cols == 32 && p.waves == 4) GO(4, 32);
            else if (p.cols == 64 && p.waves == 4) GO(4, 64);
            else return -3;
        } else return -3;
    }
#undef GO16
#undef GO
#undef GO_MT
#undef GO_SHARE
#undef GO_XL
    return launch_status();
}

template <int NORM>
int launch_skinny16_mode(const void* X, const bf16_t* W, void* Y, int M, int N, int K, int mode, const Skinny16Extra& x,
                         hipStream_t stream) {
    if (mode == OUT_BF16) return launch_skinny16<OUT_BF16, NORM, false>(X, W, Y, M, N, K, x, stream);
    if (mode == OUT_F32) return launch_skinny16<OUT_F32, NORM, false>(X, W, Y, M, N, K, x, stream);
    if (mode == OUT_F32_ACCUM) return launch_skinny16<OUT_F32_ACCUM, NORM, false>(X, W, Y, M, N, K, x, stream);
    if (mode == OUT_SWIGLU) {
        if (N % 2) return -2;
        return launch_skinny16<OUT_SWIGLU, NORM, false>(X, W, Y, M, N, K, x, stream);
    }
    return -3;
}

// 16 < M <= 64.  ws: the work space tuff_gemm_bf16_workspace asks for.
template <int MODE, int NORM, bool EMIT>
int launch_skinny64(const bf16_t* X, const bf16_t* W, void* Y, int M, int N, int K, float* ws, const FinishExtra& ex,
                    hipStream_t stream) {
    const SkinnyPlan p = plan_skinny(M, N, K, 16, EMIT);
    dim3 grid(p.tiles, p.slices), block(SK_NT);
    const bool to_ws = p.ws_floats > 0;
    if (to_ws && !ws) return -4;
    const int mt = ceil_div(M, 16);
#define GO(MT) hipLaunchKernelGGL((gemm_bf16_skinny64_kernel<MT, MODE, NORM>), grid, block, 0, stream, X, W, Y, M, N, K, \
                                  p.chunks_per_slice, ws, to_ws, ex.ss_in, ex.n_ss, ex.eps)
    if (mt == 2) GO(2); else if (mt == 3) GO(3); else GO(4);
#undef GO
    if (to_ws) {
        int rc = launch_status();
        if (rc) return rc;
        // the emitting epilogue writes the sums of squares of all 64 rows of a tile (zero beyond M)
        hipLaunchKernelGGL((splitk_finish_kernel<MODE, NORM, EMIT>), dim3(p.tiles, EMIT ? 4 : mt), dim3(256), 0, stream,
                           (const float*)ws, Y, M, N, mt * 16, p.slices, ex);
    }
    return launch_status();
}

// 16 < M <= 64: the projection's partial tiles into the work space (always: also with one slice), then the
// kernel that adds them and runs the convolution.
template <int NORM>
int launch_skinny64_conv(const bf16_t* X, const bf16_t* W, bf16_t* Y, int M, int d, int K, float* ws, const FinishExtra& ex,
                         const ConvTail& cv, hipStream_t stream) {
    const int N = 3 * d;
    const SkinnyPlan p = plan_skinny(M, N, K, 16, true);
    if (!ws) return -4;
    const int mt = ceil_div(M, 16);
    dim3 grid(p.tiles, p.slices), block(SK_NT);
#define GO(MT) hipLaunchKernelGGL((gemm_bf16_skinny64_kernel<MT, OUT_BF16, NORM_NONE>), grid, block, 0, stream, X, W, (void*)nullptr, \
                                  M, N, K, p.chunks_per_slice, ws, true, (const float*)nullptr, 0, 0.f)
    if (mt == 2) GO(2); else if (mt == 3) GO(3); else GO(4);
#undef GO
    int rc = launch_status();
    if (rc) return rc;
    hipLaunchKernelGGL((splitk_finish_conv_kernel<NORM>), dim3(ceil_div(d, 64), ceil_div(M, FC_ROWS)), dim3(FC_ROWS * 16), 0, stream,
                       (const float*)ws, Y, M, d, mt * 16, p.slices, ex, cv);
    return launch_status();
}

template <int NORM>
int launch_skinny64_mode(const bf16_t* X, const bf16_t* W, void* Y, int M, int N, int K, int mode, float* ws,
                         const FinishExtra& ex, hipStream_t stream) {
    if (mode == OUT_BF16) return launch_skinny64<OUT_BF16, NORM, false>(X, W, Y, M, N, K, ws, ex, stream);
    if (mode == OUT_F32) return launch_skinny64<OUT_F32, NORM, false>(X, W, Y, M, N, K, ws, ex, stream);
    if (mode == OUT_F32_ACCUM) return launch_skinny64<OUT_F32_ACCUM, NORM, false>(X, W, Y, M, N, K, ws, ex, stream);
    if (mode == OUT_SWIGLU) {
        if (N % 2) return -2;
        return launch_skinny64<OUT_SWIGLU, NORM, false>(X, W, Y, M, N, K, ws, ex, stream);
    }
    return -3;
}

// How the sums of squares of a tiled product with the emitting epilogue are grouped: columns a group, or 0
// where this product cannot emit (K no multiple of 64, K cut into slices, N no whole number of blocks).
int tiled_emit_group(int M, int N, int K) {
    const TiledPlan t = plan_tiled(M, N, K);
    if (t.slices > 1) return 64;                        // the kernel that adds the slices emits, 64 columns a workgroup
    if (!dma_ok(K)) return 0;
    const int bn = t.shape == 0 || t.shape == 5 ? 256 : t.shape == 4 ? 192 : t.shape == 3 ? 64 : 128;
    if (N % bn != 0) return 0;
    return bn;                                          // a workgroup's columns
}

// A product of more than 64 rows in one piece can add a bias to its sums and take the square of their positive part.
bool tiled_bias_ok(int M, int N, int K) { return M > 64 && dma_ok(K) && plan_tiled(M, N, K).slices <= 1; }

bool tiled_scaled_ok(int M, int N, int K) { return dma_ok(K) || plan_tiled(M, N, K).slices > 1; }

template <int MODE, int AROUND = TILED_PLAIN>
int launch_mode(const bf16_t* X, const bf16_t* W, void* Y, int M, int N, int K, float* ws, hipStream_t stream,
                TiledExtra ex = TiledExtra()) {
    if constexpr (AROUND == TILED_PLAIN) {
        if (few_rows_kernel(M, N, K)) return launch_skinny16<MODE, NORM_NONE, false>(X, W, Y, M, N, K, Skinny16Extra(), stream);
        if (M <= 64 && !rows64_tiled(M, N, K)) return launch_skinny64<MODE, NORM_NONE, false>(X, W, Y, M, N, K, ws, FinishExtra(), stream);
    }
    {
        // Large blocks where they give most CUs one.  Of the small ones a CU holds two if there are
        // enough; if not, a block is alone on its CU and hides the memory's latency by itself, with
        // the operands of four steps under way.  Where even the small blocks are fewer than half the
        // CUs (few rows, narrow output), blocks of 64 x 64 take over if K is short, else K is cut into
        // slices, a block a slice.
        TiledPlan t = plan_tiled(M, N, K);
        if (rows64_tiled(M, N, K)) { t.shape = 3; t.slices = 1; t.steps_per_slice = ceil_div(K, TBK); t.ws_floats = 0; }
        if (t.slices > 1 && !ws) return -4;
        ex.bands = bands_of_rows(t, M, N);
#define TILED(TM, TN, WM, WN, AHEAD) do { \
            auto kern = gemm_bf16_tiled_kernel<TM, TN, WM, WN, AHEAD, MODE>; \
            constexpr int bm = 16 * TM * WM, bn = 16 * TN * WN, lds = 2 * (bm + bn) * TBK * 2; \
            static bool set = false; \
            if (!set) { \
                if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return -1; \
                set = true; \
            } \
            hipLaunchKernelGGL(kern, dim3(ceil_div(N, bn), ceil_div(M, bm), t.slices), dim3(64 * WM * WN), lds, stream, \
                               X, W, Y, M, N, K, t.steps_per_slice, ws); \
        } while (0)
#define TILED_DMA(TM, TN, WM, WN, STAGES, BUFFER, FOLDS) do { \
            auto kern = gemm_bf16_dma_kernel<TM, TN, WM, WN, STAGES, BUFFER, FOLDS, MODE, AROUND>; \
            constexpr int bm = 16 * TM * WM, bn = 16 * TN * WN, lds = STAGES * (bm + bn) * TBK * 2; \
            static bool set = false; \
            if (!set) { \
                if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return -1; \
                set = true; \
            } \
            hipLaunchKernelGGL(kern, dim3(ceil_div(N, bn), ceil_div(M, bm), t.slices), dim3(64 * WM * WN), lds, stream, \
                               X, W, Y, M, N, K, t.steps_per_slice, ws, ex); \
        } while (0)
        if constexpr (AROUND == TILED_BIAS || AROUND == TILED_RELU2) {
            if (!dma_ok(K) || t.slices > 1) return -2;
        }
        if constexpr (AROUND != TILED_PLAIN) {
            if (!dma_ok(K) && t.slices == 1) return -2;            // a product in slices is finished by the kernel that adds them
        }
        if constexpr (AROUND == TILED_EMIT_FAR) {
            // (so many columns are many large blocks)
            if (t.shape == 4) TILED_DMA(8, 3, 2, 4, 2, false, false);
            else if (t.shape == 0) TILED_DMA(8, 4, 2, 4, 2, true, false);
            else if (t.shape == 5) TILED_DMA(4, 4, 2, 4, 3, true, false);
            else return -3;                                            // (a shape forced for a measurement)
        } else if (dma_ok(K)) {
            const bool buffer = dma_through_buffer(t, M, N);
            if (t.shape == 3 && t.steps_per_slice < ceil_div(K, TBK)) TILED_DMA(2, 2, 2, 2, 4, true, true);
            else if (t.shape == 3) { if (buffer) TILED_DMA(2, 2, 2, 2, 4, true, false); else TILED_DMA(2, 2, 2, 2, 4, false, false); }
            else if (t.shape == 4) TILED_DMA(8, 3, 2, 4, 2, false, false);
            else if (t.shape == 0) TILED_DMA(8, 4, 2, 4, 2, true, false);
            else if (t.shape == 1) TILED_DMA(4, 2, 2, 4, 2, true, false);
            else if (t.shape == 5) TILED_DMA(4, 4, 2, 4, 3, true, false);
            else if (t.shape == 6) TILED_DMA(4, 2, 1, 4, 4, true, false);
            else if (buffer) TILED_DMA(4, 2, 2, 4, 4, true, false);
            else TILED_DMA(4, 2, 2, 4, 4, false, false);
        }
        else if (t.shape == 0) TILED(8, 4, 2, 4, 1);
        else if (t.shape == 1) TILED(4, 2, 2, 4, 1);
        else TILED(4, 2, 2, 4, 4);
#undef TILED_DMA
#undef TILED
        if constexpr (AROUND != TILED_BIAS && AROUND != TILED_RELU2) if (t.slices > 1) {
            int rc = launch_status();
            if (rc) return rc;
            FinishExtra fx;
            fx.ss_rows = M;
            fx.ss_in = ex.ss_in; fx.n_ss = ex.n_ss; fx.eps = ex.eps; fx.K = K;
            fx.emit_nw = ex.emit_nw; fx.emit_xw = ex.emit_xw; fx.emit_ss = ex.emit_ss;
            constexpr int FN = AROUND == TILED_SCALED ? NORM_SCALED : NORM_NONE;
            hipLaunchKernelGGL((splitk_finish_kernel<MODE, FN, AROUND == TILED_EMIT || AROUND == TILED_EMIT_FAR>), dim3(ceil_div(N, 64), ceil_div(M, 16)),
                               dim3(256), 0, stream, (const float*)ws, Y, M, N, M, t.slices, fx);
        }
    }
    return launch_status();
}
}  // namespace

// For measurements: for how many columns and from how many rows on a product of at most 64 rows with a short K
// takes blocks of 64 x 64 instead of slices of K.  Returns the least number of columns before.
TUFF_EXPORT int tuff_gemm_bf16_wide64(int min_n, int max_n, int min_m) {
    const int old = wide64_min_n;
    if (min_n > 0) wide64_min_n = min_n;
    if (max_n > 0) wide64_max_n = max_n;
    if (min_m > 0) wide64_min_m = min_m;
    return old;
}

// For measurements: forces the block shape of every product of more than 64 rows whose K is a multiple
// of 64 (0: 256 x 256, 1: 128 x 128 two a CU, 2: 128 x 128 one a CU, 3: 64 x 64, 4: 256 x 192, 5: 128 x 256, 6: 64 x 128; -1: by size).
// Returns the value before.
TUFF_EXPORT int tuff_gemm_bf16_force_tiled_shape(int shape) {
    const int old = tiled_shape_forced;
    tiled_shape_forced = shape;
    return old;
}

// How the sums of squares of tuff_gemm_bf16_accum_emit are laid out for a product of M rows:
// *tiles tiles of columns, *rows rows each (16 for M <= 16, 64 for M <= 64).
TUFF_EXPORT int tuff_gemm_bf16_emit_layout(int M, int N, int K, int* tiles, int* rows) {
    if (M > 64) {
        // the tiled product: a group of columns a wave, M rows each; *tiles = 0 where it cannot emit
        const int group = tiled_emit_group(M, N, K);
        *tiles = group ? ceil_div(N, group) : 0;        // (a product in slices may end in a partial group of columns)
        *rows = M;
        return 0;
    }
    *tiles = plan_skinny(M, N, K, 16, true).tiles;
    *rows = M <= 16 ? 16 : 64;                          // (17 to 32 rows: the kernel for few rows, with tiles of 64 rows)
    return 0;
}

// 1 if tuff_gemm_bf16_scaled takes a product of these sizes (always for M <= 64; for more rows where the
// tiled product runs it in one piece), else 0.
TUFF_EXPORT int tuff_gemm_bf16_scaled_supported(int M, int N, int K) {
    if (!inner_ok(K) || M <= 0 || N <= 0) return 0;
    return M <= 64 || tiled_scaled_ok(M, N, K) ? 1 : 0;
}

// Work space a product of this shape needs: *ws_floats float32 for partial tiles (0: none).
// emit: for tuff_gemm_bf16_accum_emit.
TUFF_EXPORT int tuff_gemm_bf16_workspace(int M, int N, int K, int emit, long long* ws_floats) {
    *ws_floats = 0;
    if (N <= 0 || few_rows_kernel(M, N, K, false, emit != 0)) return 0;
    // (a wide product of few rows that the tiled kernel takes needs none, but only some of its epilogues go that way)
    *ws_floats = M <= 64 ? plan_skinny(M, N, K, 16, emit != 0).ws_floats : plan_tiled(M, N, K).ws_floats;
    return 0;
}

// W: tile-major, as described at the head of this file (ceil(N/16) * ceil(K/32) blocks of 1 KB).
// K must be a multiple of 8 (16-byte operand loads), here and below, and at most 2^24 - 64 (else -2); the host wrapper refuses other K.
// Y = bf16(X W^T + bias), or with square_positive bf16(max(X W^T + bias, 0)^2), for the products of which
// tuff_gemm_bf16_bias_supported says so.  bias float32 [N] or null.
TUFF_EXPORT int tuff_gemm_bf16_bias_supported(int M, int N, int K) {
    return M > 0 && N > 0 && inner_ok(K) && tiled_bias_ok(M, N, K) ? 1 : 0;
}
TUFF_EXPORT int tuff_gemm_bf16_bias(const void* X, const void* W, void* Y, int M, int N, int K, const float* bias, int square_positive,
                                    hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!inner_ok(K) || !tiled_bias_ok(M, N, K)) return -2;
    TiledExtra ex;
    ex.bias = bias;
    if (square_positive) return launch_mode<OUT_BF16, TILED_RELU2>((const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, nullptr, stream, ex);
    return launch_mode<OUT_BF16, TILED_BIAS>((const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, nullptr, stream, ex);
}

TUFF_EXPORT int tuff_gemm_bf16(const void* X, const void* W, void* Y, int M, int N, int K, int mode,
                               float* ws, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!inner_ok(K)) return -2;
    const bf16_t* x = (const bf16_t*)X;
    const bf16_t* w = (const bf16_t*)W;
    if (mode == OUT_BF16) return launch_mode<OUT_BF16>(x, w, Y, M, N, K, ws, stream);
    if (mode == OUT_F32) return launch_mode<OUT_F32>(x, w, Y, M, N, K, ws, stream);
    if (mode == OUT_F32_ACCUM) return launch_mode<OUT_F32_ACCUM>(x, w, Y, M, N, K, ws, stream);
    if (mode == OUT_SWIGLU) {
        if (N % 2) return -2;
        return launch_mode<OUT_SWIGLU>(x, w, Y, M, N, K, ws, stream);
    }
    return -3;
}

// Y (=|+=) RMSNorm(X[rows]) * W^T for M <= 16 rows: X float32 [*, K], rows ldx elements apart (a multiple of 4, rows on
// 16-byte borders), norm_w float32 [K], rows optional int32 [M].  K must be a multiple of 8 and at most 8192 (the norm
// weight sits in LDS).
TUFF_EXPORT int tuff_gemm_bf16_normed(const float* X, const int* rows, long long ldx, const float* norm_w, float eps, const void* W,
                                      void* Y, int M, int N, int K, int mode, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!inner_ok(K) || K > 8192 || M > 16 || ldx < K || ldx % 4 || (uintptr_t)X % 16) return -2;
    Skinny16Extra x;
    x.norm_w = norm_w; x.eps = eps; x.rows = rows; x.ldx = ldx;
    return launch_skinny16_mode<NORM_INSIDE>(X, (const bf16_t*)W, Y, M, N, K, mode, x, stream);
}

// Y += X W^T, and from the new Y (the residual stream, float32 [M, N]) the
// operand of the RMSNorm that follows: xw = bf16(Y * next_norm_w) [M, N] and ss [tiles][rows] (as
// tuff_gemm_bf16_emit_layout says; 0 tiles: this product cannot, -2), the sums of squares of each row
// over each tile of columns.
// ws: for M > 16, the work space tuff_gemm_bf16_workspace(M, N, K, 1) asks for.
TUFF_EXPORT int tuff_gemm_bf16_accum_emit(const void* X, const void* W, float* Y, int M, int N, int K,
                                          const float* next_norm_w, void* xw, float* ss, float* ws, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!inner_ok(K)) return -2;
    if (M > 64) {
        if (!tiled_emit_group(M, N, K)) return -2;
        TiledExtra t;
        t.emit_nw = next_norm_w; t.emit_xw = (bf16_t*)xw; t.emit_ss = ss;
        if (N >= 1 << 25) return launch_mode<OUT_F32_ACCUM, TILED_EMIT_FAR>((const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, ws, stream, t);
        return launch_mode<OUT_F32_ACCUM, TILED_EMIT>((const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, ws, stream, t);
    }
    if (few_rows_kernel(M, N, K, false, true)) {
        Skinny16Extra x;
        x.emit_nw = next_norm_w; x.emit_xw = (bf16_t*)xw; x.emit_ss = ss;
        return launch_skinny16<OUT_F32_ACCUM, NORM_NONE, true>(X, (const bf16_t*)W, Y, M, N, K, x, stream);
    }
    FinishExtra x;
    x.emit_nw = next_norm_w; x.emit_xw = (bf16_t*)xw; x.emit_ss = ss;
    return launch_skinny64<OUT_F32_ACCUM, NORM_NONE, true>((const bf16_t*)X, (const bf16_t*)W, Y, M, N, K, ws, x, stream);
}

// Y (=|+=) (XW W^T) scaled per row by 1 / sqrt(sum_t ss[t][row] / K + eps), with
// XW and ss as tuff_gemm_bf16_accum_emit leaves them for the same M (n_ss tiles); see
// tuff_gemm_bf16_scaled_supported for M > 64.
// ws: for M > 16, the work space tuff_gemm_bf16_workspace(M, N, K, 0) asks for.
TUFF_EXPORT int tuff_gemm_bf16_scaled(const void* XW, const float* ss, int n_ss, float eps, const void* W, void* Y,
                                      int M, int N, int K, int mode, float* ws, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (!inner_ok(K) || n_ss < 1) return -2;
    if (M > 64 || (rows64_tiled(M, N, K) && (mode == OUT_BF16 || mode == OUT_SWIGLU))) {
        // ss [n_ss][M] ([n_ss][64] from a product of at most 64 rows); bfloat16 and SwiGLU outputs (what reads a norm in a layer)
        if (!tiled_scaled_ok(M, N, K)) return -2;
        TiledExtra t;
        t.ss_in = ss; t.n_ss = n_ss; t.eps = eps; t.ss_rows = M > 64 ? 0 : 64;
        const bf16_t* x = (const bf16_t*)XW;
        const bf16_t* w = (const bf16_t*)W;
        if (mode == OUT_BF16) return launch_mode<OUT_BF16, TILED_SCALED>(x, w, Y, M, N, K, ws, stream, t);
        if (mode == OUT_SWIGLU) {
            if (N % 2) return -2;
            return launch_mode<OUT_SWIGLU, TILED_SCALED>(x, w, Y, M, N, K, ws, stream, t);
        }
        return -3;
    }
    if (few_rows_kernel(M, N, K)) {
        Skinny16Extra x;
        x.ss_in = ss; x.n_ss = n_ss; x.eps = eps;
        return launch_skinny16_mode<NORM_SCALED>(XW, (const bf16_t*)W, Y, M, N, K, mode, x, stream);
    }
    FinishExtra x;
    x.ss_in = ss; x.n_ss = n_ss; x.eps = eps; x.K = K;
    return launch_skinny64_mode<NORM_SCALED>((const bf16_t*)XW, (const bf16_t*)W, Y, M, N, K, mode, ws, x, stream);
}

// For M <= 16 rows, one token a row: the input projection of a gated short convolution and the
// convolution itself in one kernel.  W: the projection [3 d, K] with its rows regrouped (sixteen
// channels a group: B, C, X of the group), tile-major; d must be a multiple of 16.  Y: bfloat16 [M, d]
// = C * conv(B * X).  taps [d][n_taps] (taps_dt), state float32 [slots][n_taps - 1][d], state_slot [M].
// norm_kind 0: X is bfloat16 [M, K];  1: X is the float32 residual stream and the RMSNorm (norm_w,
// eps; K <= 8192) runs inside;  2: X is bf16(x * norm weight) and ss [n_ss][16] the sums of squares
// that tuff_gemm_bf16_accum_emit left.
// The same for 17 to 64 rows, in two kernels (the projection's partial tiles, then the kernel that adds
// them and runs the convolution), from the projection as the checkpoint has it: W [3 d, K] tile-major,
// rows B | C | X.  X: bfloat16 [M, K], or with ss [n_ss][64] (and eps) bf16(x * norm weight) and the sums of
// squares that tuff_gemm_bf16_accum_emit left for these M rows.  ws: tuff_gemm_bf16_workspace(M, 3 d, K, 1).
TUFF_EXPORT int tuff_gemm_bf16_conv64(const void* X, const float* ss, int n_ss, float eps, const void* W, void* Y,
                                      int M, int d, int K, const void* taps, int taps_dt, int n_taps, float* state,
                                      const int* state_slot, float* ws, hipStream_t stream) {
    if (M <= 0 || d <= 0) return 0;
    if (!inner_ok(K) || M <= SKINNY_ROWS || M > 64 || d % 16 != 0 || n_taps < 2 || n_taps - 1 > CONV_MAX_TAPS) return -2;
    ConvTail cv;
    cv.taps_w = taps; cv.taps_dt = taps_dt; cv.taps = n_taps; cv.state = state; cv.state_slot = state_slot;
    FinishExtra x;
    if (ss) {
        if (n_ss < 1) return -2;
        x.ss_in = ss; x.n_ss = n_ss; x.eps = eps; x.K = K;
        return launch_skinny64_conv<NORM_SCALED>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)Y, M, d, K, ws, x, cv, stream);
    }
    return launch_skinny64_conv<NORM_NONE>((const bf16_t*)X, (const bf16_t*)W, (bf16_t*)Y, M, d, K, ws, x, cv, stream);
}

TUFF_EXPORT int tuff_gemm_bf16_conv(const void* X, int norm_kind, const float* norm_w, float eps, const float* ss, int n_ss,
                                    const void* W, void* Y, int M, int d, int K,
                                    const void* taps, int taps_dt, int n_taps, float* state, const int* state_slot,
                                    hipStream_t stream) {
    if (M <= 0 || d <= 0) return 0;
    if (!inner_ok(K) || M > SKINNY_ROWS || d % 16 != 0 || n_taps < 2 || n_taps - 1 > CONV_MAX_TAPS) return -2;
    if (norm_kind == 1 && M > 16) return -2;
    Skinny16Extra x;
    x.conv.taps_w = taps; x.conv.taps_dt = taps_dt; x.conv.taps = n_taps; x.conv.state = state; x.conv.state_slot = state_slot;
    const bf16_t* w = (const bf16_t*)W;
    if (norm_kind == 0) return launch_skinny16<OUT_CONV, NORM_NONE, false>(X, w, Y, M, 3 * d, K, x, stream);
    if (norm_kind == 1) {
        if (K > 8192) return -2;
        x.norm_w = norm_w; x.eps = eps;
        return launch_skinny16<OUT_CONV, NORM_INSIDE, false>(X, w, Y, M, 3 * d, K, x, stream);
    }
    if (norm_kind == 2) {
        if (n_ss < 1) return -2;
        x.ss_in = ss; x.n_ss = n_ss; x.eps = eps;
        return launch_skinny16<OUT_CONV, NORM_SCALED, false>(X, w, Y, M, 3 * d, K, x, stream);
    }
    return -3;
}
