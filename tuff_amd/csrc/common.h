// Shared helpers of the gfx950 kernels: element types, wave reductions, launch checks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#define TUFF_EXPORT extern "C" __attribute__((visibility("default")))

typedef __bf16 bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int WAVE = 64;

// Element type codes shared with the Python side.
enum : int { DT_F32 = 0, DT_BF16 = 1 };

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return (bf16_t)v; }

// For a step of a butterfly over the wave, 32 first: this lane's value and that of lane ^ M, in either order.  Through registers: a
// shuffle goes through LDS, and the steps wait for one another (six of them some 700 cycles, this way 100).  M = 4 takes
// lane + 4 of the sixteen, which after the step of 8 holds what lane ^ 4 holds.
struct LanePair { float a, b; };
template <int M>
__device__ __forceinline__ LanePair butterfly_pair(float v) {
#ifdef __HIP_DEVICE_COMPILE__
    const unsigned u = __float_as_uint(v);
    if constexpr (M == 32) {                               // the halves of two copies change places: (low, low) and (high, high)
        const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return {__uint_as_float(p[0]), __uint_as_float(p[1])};
    } else if constexpr (M == 16) {                        // and rows of sixteen
        const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return {__uint_as_float(p[0]), __uint_as_float(p[1])};
    } else {
        constexpr int CTRL = M == 8 ? 0x128 : M == 4 ? 0x124 : M == 2 ? 0x4E : 0xB1;
        return {v, __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xF, 0xF, true))};
    }
#else
    return {v, v};
#endif
}
template <int M>
__device__ __forceinline__ float butterfly_sum(float v) { const LanePair p = butterfly_pair<M>(v); return p.a + p.b; }
template <int M>
__device__ __forceinline__ float butterfly_max(float v) { const LanePair p = butterfly_pair<M>(v); return fmaxf(p.a, p.b); }

// The value of lane ^ 8, ^ 1, among the sixteen lanes of a row.
__device__ __forceinline__ float lane_xor8(float v) { return butterfly_pair<8>(v).b; }
__device__ __forceinline__ float lane_xor1(float v) { return butterfly_pair<1>(v).b; }
// and of lane ^ 4: lane ^ 7 of eight, of which lane ^ 3 of four.
__device__ __forceinline__ float lane_xor4(float v) {
#ifdef __HIP_DEVICE_COMPILE__
    const int u = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true);
    return __int_as_float(__builtin_amdgcn_update_dpp(0, u, 0x1B, 0xF, 0xF, true));
#else
    return v;
#endif
}
// The sum over the sixteen lanes of a row, steps 8, 4, 2, 1; and in steps 1, 2, 4, 8, where the step of 4 takes a lane of the other
// four of eight: the two before it have left the same in all four.
__device__ __forceinline__ float row_sum_down(float v) { return butterfly_sum<1>(butterfly_sum<2>(butterfly_sum<4>(butterfly_sum<8>(v)))); }
__device__ __forceinline__ float row_sum_up(float v) {
    v = butterfly_sum<2>(butterfly_sum<1>(v));
#ifdef __HIP_DEVICE_COMPILE__
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));      // lane 7 - i of eight
#endif
    return butterfly_sum<8>(v);
}

// Sum over the 64 lanes of a wave (all of them active); every lane receives the total.  The order of
// the butterfly is fixed, so the result does not depend on anything but the inputs.
__device__ __forceinline__ float wave_sum(float v) {
    return butterfly_sum<1>(butterfly_sum<2>(butterfly_sum<4>(butterfly_sum<8>(butterfly_sum<16>(butterfly_sum<32>(v))))));
}
__device__ __forceinline__ float wave_max(float v) {
    return butterfly_max<1>(butterfly_max<2>(butterfly_max<4>(butterfly_max<8>(butterfly_max<16>(butterfly_max<32>(v))))));
}

// Sum over a workgroup of NWAVES waves; `scratch` holds NWAVES floats of LDS.
// Wave partials are added in wave order.  Ends with the total in every thread.
template <int NWAVES>
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    v = wave_sum(v);
    const int wave = threadIdx.x / WAVE;
    __syncthreads();
    if ((threadIdx.x % WAVE) == 0) scratch[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NWAVES; ++i) t += scratch[i];
    return t;
}

// f(std::integral_constant<int, 0>()), ..., f(std::integral_constant<int, N - 1>()): a loop whose
// index is a compile-time constant inside the body (register arrays stay registers).
template <int N, typename F, int I = 0>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<N, F, I + 1>(static_cast<F&&>(f));
    }
}

// Memory straight into LDS through a buffer: lane l's 16 bytes at `offset` bytes (a lane's) + `scalar` bytes (the wave's)
// of the buffer go to lds + 16 l.  Bytes beyond the buffer read as zero and are not fetched.  A buffer load and not a global
// one: behind a global load into LDS the compiler no longer knows which counter stands for what, and waits for every read
// of LDS under way whenever it needs one of them.
typedef __amdgpu_buffer_rsrc_t buffer_t;
__device__ __forceinline__ buffer_t make_buffer(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00027000);
}
__device__ __forceinline__ void load_to_lds(buffer_t buf, void* lds, int offset, int scalar) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, (__attribute__((address_space(3))) void*)lds, 16, offset, scalar, 0, 0);
#endif
}

// The same from this lane's address, through a global load.
__device__ __forceinline__ void load_to_lds(const void* from, void* lds) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
#endif
}

// An offset that lies beyond every buffer: the lane reads zero.  (A lane's offset is held against the buffer's size less the
// wave's scalar offset, so that one must not be larger than the buffer even where no lane reads.)
constexpr int NOWHERE = (int)0x80000000;
// 16 bytes, or one float, at `offset` (a lane's) + `scalar` (the wave's) bytes of the buffer.  STREAMING: read once and never again.
template <bool STREAMING>
__device__ __forceinline__ bf16x8 load_buffer(buffer_t buf, int offset, int scalar) {
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(buf, offset, scalar, STREAMING ? 2 : 0));
}
__device__ __forceinline__ float load_buffer_float(buffer_t buf, int offset, int scalar) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buf, offset, scalar, 0));
}
__device__ __forceinline__ f32x4 load_buffer_f32x4(buffer_t buf, int offset, int scalar) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buf, offset, scalar, 0));
}
// 4, 8 or 16 bytes to `offset` (a lane's) + `scalar` (the wave's) bytes of the buffer; nothing beyond it is written.
template <typename T>
__device__ __forceinline__ void store_buffer(buffer_t buf, int offset, int scalar, T v) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8 || sizeof(T) == 16, "a whole store");
    typedef unsigned words2 __attribute__((ext_vector_type(2)));
    typedef unsigned words4 __attribute__((ext_vector_type(4)));
    if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), buf, offset, scalar, 0);
    else if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(words2, v), buf, offset, scalar, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(words4, v), buf, offset, scalar, 0);
}
// The value of lane `lane` (the same for the whole wave).
__device__ __forceinline__ float lane_of(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// s_waitcnt vmcnt(VM) lgkmcnt(0)
template <int VM>
__device__ __forceinline__ void wait_loads_and_lds() {
    static_assert(VM >= 0 && VM < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | 0x0070);
}

// A workgroup's barrier for LDS that lets loads from memory stay under way.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

static inline int launch_status() { return (int)hipGetLastError(); }

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
static inline long long ceil_div_ll(long long a, long long b) { return (a + b - 1) / b; }
