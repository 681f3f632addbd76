// Part of gemm_bf16.hip: the products of up to 16 rows whose sizes divide evenly.
#pragma once

namespace {

// The skinny16 product (described in gemm_bf16.hip) for K in whole chunks of 128, N in whole workgroups and at most CH chunks a
// wave: the same cut, the same order of additions, the same bits.
//
// What bounds it: the bytes of W, and beside them what no workgroup overlaps with another's, since all begin and end together.  By
// time stamps in the kernel for any sizes (gate and up, 16,384 x 2,048, 8 rows, 14 us): 0.44 us to the first load (bounds of every load, a
// division, two waits for arguments), 0.76 from the last barrier to the end (sums of squares asked for behind the operands,
// root and division in every thread); here 0.12 and 0.32.  Loads wait for their place once some 64 to 100 KB of a CU's are
// under way, so a wave is held up where it asks, and what is needed first is asked for first: sums of squares (straight into
// LDS), a first share of W, X, then the rows' scales are worked out while those are on their way, then the rest of W.  X ahead
// of W where no sums are (2,048 x 2,048 of 8 rows 4.28 us and 4.13), behind it where they are (3,072 x 2,048 4.81 and 4.57); all of W
// at once, ahead of the wait for X in LDS: 2,048 x 8,192 of 8 rows 9.4 us, two chunks a wave ahead 8.3.
// The kernel for any sizes / this one, us, 1, 8 and 16 rows: 16,384 x 2,048 with SwiGLU 13.7 / 12.5, 13.7 / 13.0 and 15.6 / 14.2;
// 3,072 x 2,048 behind a norm 4.8 / 4.4, 5.1 / 4.6 and 5.5 / 4.7; 6,144 x 2,048 with the convolution 7.4 / 7.2, 7.6 / 7.2 and 8.5 / 8.0;
// into the stream 2,048 x 2,048 4.1 / 3.95, 4.4 / 4.15 and 4.6 / 4.3, x 8,192 of 1, 3 and 8 rows 8.1 / 7.6, 8.5 / 8.0 and 9.0 / 8.4.
struct Lean16Args {
    const bf16_t* X; const bf16_t* W; void* Y;
    const float* ss_in; const float* emit_nw; bf16_t* emit_xw; float* emit_ss;
    int M, N, K, n_ss;
    float eps;
    unsigned per_xcd;          // workgroups an XCD, neighbours' columns one after the other; 0: as the grid counts them
    unsigned pieces_inverse;   // XL: 2^32 / the kilobytes that a row of X takes, both rounded up: quotients of numbers below 2^16
    ConvTail cv;
};

constexpr int lean16_waves_a_simd(int NW, int COLS) { return NW == 8 && COLS == 32 ? 4 : 1; }

template <int NW, int MODE, bool SCALED, bool EMIT, int COLS, int CH, bool XL>
__global__ __launch_bounds__(NW * WAVE, lean16_waves_a_simd(NW, COLS)) void gemm_bf16_lean16_kernel(Lean16Args a) {
    constexpr bool CONV = MODE == OUT_CONV;
    constexpr int TN = CONV ? 3 : COLS > 16 ? COLS / 16 : 1;
    static_assert(EMIT == (MODE == OUT_F32_ACCUM) && (!EMIT || TN == 1), "into the residual stream with the emitting epilogue, one tile");
    static_assert(!CONV || COLS == 8, "the convolution's epilogue takes eight channels a workgroup");
    static_assert(TN == 1 || CONV || NW * WAVE >= 256 * TN, "256 threads finish a tile");
    __shared__ __attribute__((aligned(16))) float red[TN][NW][WAVE][4];
    __shared__ __attribute__((aligned(16))) float ss_lds[SCALED ? 256 * 16 : 4];
    __shared__ float ssq[SCALED ? 16 : 1][16];
    __shared__ float scale_lds[16];
    extern __shared__ __attribute__((aligned(16))) bf16_t x_lds[];       // XL: [M][K + 8]
    const unsigned block = a.per_xcd ? blockIdx.x % 8 * a.per_xcd + blockIdx.x / 8 : blockIdx.x;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int r16 = lane % 16, g = lane / 16;
    const int M = a.M, N = a.N, K = a.K, nchunks = K / SK_CHUNK, kb = K / 32;
    // (OUT_CONV: half (b % 2) of the three row tiles of group b / 2)
    const unsigned half = COLS == 8 ? block % 2 * 8 : 0;                 // the tile's first row of W that this workgroup owns
    const unsigned tile0 = CONV ? block / 2 * 3 : COLS == 8 ? block / 2 : block * (COLS / 16);
    const int w_at = COLS == 8 ? (r16 < 8 ? (g * 16 + (int)half + r16) * 16 : NOWHERE) : lane * 16;
    const buffer_t wbuf = make_buffer(a.W + (long long)tile0 * kb * 512, TN * kb * 1024);
    const buffer_t xbuf = make_buffer(a.X, M * K * 2);

    // the thread's place in a tile: element (row, column) of its 256 threads
    const int t256 = tid % 256, e = t256 % 4, l = t256 / 4, trow = (l / 16) * 4 + e, tn_mine = CONV ? 0 : tid / 256;
    const int col = (int)(tile0 * 16 + half) + tn_mine * 16 + l % 16;
    const bool mine = tn_mine < TN && trow < M && (COLS != 8 || l % 16 < 8);

    // ---- what is asked for ahead of the operands: sums of squares, what the epilogue adds to, the convolution's slot and taps
    float y_old = 0.f, emit_w = 0.f;
    if constexpr (EMIT) {
        if (mine) {
            y_old = ((const float*)a.Y)[(long long)trow * N + col];
            emit_w = a.emit_nw[col];
        }
    }
    constexpr int CONV_AHEAD = 4;
    float st_ahead[CONV ? CONV_AHEAD : 1], tap_ahead[CONV ? CONV_AHEAD + 1 : 1];
    int slot = 0;
    const int d = N / 3, ch = (int)block * 8 + l % 16;
    if constexpr (CONV) {
        const int Kc = a.cv.taps;
        slot = a.cv.state_slot[min(trow, M - 1)];
#pragma unroll
        for (int k = 0; k <= CONV_AHEAD; ++k) tap_ahead[k] = 0.f;
        if (mine && tid < 256) {
#pragma unroll
            for (int k = 0; k < CONV_AHEAD; ++k)
                if (k < Kc - 1) tap_ahead[k] = a.cv.tap(ch, k);
            tap_ahead[CONV_AHEAD] = a.cv.tap(ch, Kc - 1);
        }
    }
    if constexpr (SCALED) {
        const buffer_t sbuf = make_buffer(a.ss_in, a.n_ss * 64);
#pragma unroll
        for (int i = 0; i < 16 / NW; ++i) load_to_lds(sbuf, ss_lds + (wave + i * NW) * 256, (wave + i * NW) * 1024 + lane * 16, 0);
    }
    if constexpr (XL) {
        const unsigned per_row = (unsigned)(K + 511) / 512;
        for (unsigned i = wave; i < M * per_row; i += NW) {
            const unsigned row = __umulhi(i, a.pieces_inverse), at = (i - row * per_row) * 512;
            if (at + lane * 8 < (unsigned)K) load_to_lds(xbuf, x_lds + row * (K + 8) + at, (int)(row * K + at) * 2 + lane * 16, 0);
        }
    }

    // ---- the operands of all the wave's chunks
    bool there[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) there[i] = wave + i * NW < nchunks;
    bf16x8 w[CH][TN][4], x[XL ? 1 : CH][4];
    auto load_w = [&](int i) {
        const int at = there[i] ? w_at : NOWHERE, from = there[i] ? (wave + i * NW) * 4096 : 0;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int j = 0; j < 4; ++j) w[i][tn][j] = load_buffer<true>(wbuf, at + j * 1024, from + (there[i] ? tn * kb * 1024 : 0));
    };
    auto load_x = [&]() {
        if constexpr (XL) return;
#pragma unroll
        for (int i = 0; i < (XL ? 0 : CH); ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) x[i][j] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (r16 < M) {                             // (lanes without a row are switched off: one that reads nothing still takes its time)
            const int at = (r16 * K + g * 8) * 2;
#pragma unroll
            for (int i = 0; i < (XL ? 0 : CH); ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) x[i][j] = load_buffer<false>(xbuf, at + j * 64, there[i] ? (wave + i * NW) * 256 : 0);
        }
    };
    constexpr int FIRST = CH > 2 ? 2 : 1;
    constexpr int W_LOADS = FIRST * 4 * TN, X_LOADS = XL ? 0 : CH * 4;
    if (!SCALED) load_x();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < FIRST; ++i) load_w(i);
    __builtin_amdgcn_sched_barrier(0);
    if (SCALED) load_x();
    __builtin_amdgcn_sched_barrier(0);
    // ---- while they are on their way: the rows' scales, or the rows of X into place
    if constexpr (SCALED) {
        wait_loads_and_lds<W_LOADS + X_LOADS>();           // the sums were asked for before those
        lds_barrier();
        if (tid < 256) {
            const int p = tid / 16, row = tid % 16;
            float t = 0.f;
#pragma unroll
            for (int u = 0; u < 16; ++u) t += ss_lds[(p + 16 * u) * 16 + row];
            ssq[p][row] = t;
        }
        lds_barrier();
        if (tid < 16) {
            float total = ssq[0][tid];
#pragma unroll
            for (int p = 1; p < 16; ++p) total += ssq[p][tid];
            scale_lds[tid] = 1.0f / sqrtf(total / (float)K + a.eps);
        }
    }
    if constexpr (XL) {
        wait_loads_and_lds<W_LOADS>();
        lds_barrier();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = FIRST; i < CH; ++i) load_w(i);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (CONV) {
        const float* st = a.cv.state + (long long)slot * (a.cv.taps - 1) * d + min(ch, d - 1);
#pragma unroll
        for (int k = 0; k < CONV_AHEAD; ++k) st_ahead[k] = st[(long long)min(k, a.cv.taps - 2) * d];
        __builtin_amdgcn_sched_barrier(0);
    }

    f32x4 acc[TN];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[tn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if (!there[i]) break;
        const bf16_t* row = x_lds + min(r16, M - 1) * (K + 8) + (wave + i * NW) * SK_CHUNK + g * 8;     // (no row: another one's, its result is not taken)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (XL) acc[tn] = mfma16(*(const bf16x8*)(row + j * 32), w[i][tn][j], acc[tn]);
                else acc[tn] = mfma16(x[i][j], w[i][tn][j], acc[tn]);
            }
    }
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) *(f32x4*)red[tn][wave][lane] = acc[tn];
    lds_barrier();
    if (tid >= (CONV ? 256 : 256 * TN)) return;

    if constexpr (CONV) {
        // as the kernel for any sizes does it
        const float scale = SCALED ? scale_lds[trow] : 1.f;
        float bcx[3];
#pragma unroll
        for (int tn = 0; tn < 3; ++tn) {
            float v = red[tn][0][l][e];
#pragma unroll
            for (int u = 1; u < NW; ++u) v += red[tn][u][l][e];
            if (SCALED) v *= scale;
            bcx[tn] = (float)(bf16_t)v;
        }
        const int Kc = a.cv.taps;
        if (mine && ch < d) {
            float* st = a.cv.state + (long long)slot * (Kc - 1) * d;
            float sv[CONV_MAX_TAPS], wv[CONV_MAX_TAPS];
#pragma unroll
            for (int k = 0; k < CONV_MAX_TAPS; ++k) {
                if (k < CONV_AHEAD) { sv[k] = st_ahead[k]; wv[k] = tap_ahead[k]; continue; }
                sv[k] = k < Kc - 1 ? st[(long long)k * d + ch] : 0.f;
                wv[k] = k < Kc - 1 ? a.cv.tap(ch, k) : 0.f;
            }
            const float u = bcx[0] * bcx[2];
            float y = 0.f;
#pragma unroll
            for (int k = 0; k < CONV_MAX_TAPS; ++k)
                if (k < Kc - 1) y = (k == 0) ? sv[k] * wv[k] : fmaf(sv[k], wv[k], y);
            y = fmaf(u, tap_ahead[CONV_AHEAD], y);
#pragma unroll
            for (int k = 1; k < CONV_MAX_TAPS; ++k)
                if (k < Kc - 1) st[(long long)(k - 1) * d + ch] = sv[k];
            st[(long long)(Kc - 2) * d + ch] = u;
            ((bf16_t*)a.Y)[(long long)trow * d + ch] = (bf16_t)(bcx[1] * y);
        }
        return;
    }
    float v = red[tn_mine][0][l][e];
#pragma unroll
    for (int u = 1; u < NW; ++u) v += red[tn_mine][u][l][e];
    if (SCALED) v *= scale_lds[trow];
    if constexpr (EMIT) {
        float y = 0.f;
        if (mine) {
            y = y_old + v;
            ((float*)a.Y)[(long long)trow * N + col] = y;
            a.emit_xw[(long long)trow * N + col] = (bf16_t)(y * emit_w);
        }
        float sq = y * y;
        sq += lane_xor4(sq);
        sq = butterfly_sum<32>(butterfly_sum<16>(butterfly_sum<8>(sq)));
        if (l % 16 == 0) a.emit_ss[(long long)block * 16 + trow] = sq;
    } else if constexpr (MODE == OUT_SWIGLU) {
        const float partner = lane_xor4(v);
        if (mine && (col & 1) == 0) ((bf16_t*)a.Y)[(long long)trow * (N / 2) + col / 2] = (bf16_t)silu_mul(v, partner);
    } else {
        if (mine) store_out<MODE>(a.Y, (long long)trow * N + col, v);
    }
}
}  // namespace
