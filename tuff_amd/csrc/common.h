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

// Sum over the 64 lanes of a wave; every lane receives the total.  The order of
// the butterfly is fixed, so the result does not depend on anything but the inputs.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = WAVE / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, WAVE);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = WAVE / 2; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, WAVE));
    return v;
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
