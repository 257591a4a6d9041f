// What the kernels around the attention share: conversions and one value of the rotary embedding.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

namespace tl {

template <typename T> __device__ __forceinline__ float to_f(T v);
template <> __device__ __forceinline__ float to_f<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f<__half>(__half v) { return __half2float(v); }
template <typename T> __device__ __forceinline__ T from_f(float v);
template <> __device__ __forceinline__ float from_f<float>(float v) { return v; }
template <> __device__ __forceinline__ __half from_f<__half>(float v) { return __float2half(v); }

// One value of the rotate-half rotary embedding: x at dimension d, xp its partner half a head away, sgn = -1
// below the middle and +1 above.  One explicit fma whose fp32 result is kept apart from the conversion that
// follows it, so that every kernel rounds the same way: left to the compiler, some uses become an fma that
// rounds straight to fp16 (v_fma_mixlo_f16) and others an fp32 fma plus a conversion, which differ on near-ties.
__device__ __forceinline__ float rope_value(float x, float xp, float c, float s, float sgn)
{
    float r = fmaf(sgn * xp, s, x * c);
    asm volatile("" : "+v"(r));
    return r;
}

}  // namespace tl
