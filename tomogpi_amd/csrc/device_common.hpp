// device_common.hpp - device helpers shared by the kernel files.
//
// Arithmetic contract: every file is compiled with -ffp-contract=off and
// correctly rounded FP32 division / square root, so each fused multiply-add
// below is an explicit fmaf()/fma() call.  The CPU oracle restates the same
// operations in the same order, which makes the FP32 forms bit-comparable.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>

#include <cstdint>

#include "tomo_internal.hpp"

namespace tomo {

// ---- storage types: value = (float)stored * inv_scale; stored = value*scale
// (FP32 storage is unscaled).
template <typename T> struct Storage;
template <> struct Storage<float> {
    __device__ __forceinline__ static float load(const float* p, uint64_t i, float) { return p[i]; }
    __device__ __forceinline__ static void store(float* p, uint64_t i, float v, float) { p[i] = v; }
};
template <> struct Storage<__half> {
    __device__ __forceinline__ static float load(const __half* p, uint64_t i, float inv) {
        return __half2float(p[i]) * inv;
    }
    __device__ __forceinline__ static void store(__half* p, uint64_t i, float v, float scale) {
        p[i] = __float2half_rn(v * scale);
    }
};
template <> struct Storage<__hip_bfloat16> {
    __device__ __forceinline__ static float load(const __hip_bfloat16* p, uint64_t i, float inv) {
        return __bfloat162float(p[i]) * inv;
    }
    __device__ __forceinline__ static void store(__hip_bfloat16* p, uint64_t i, float v, float scale) {
        p[i] = __float2bfloat16(v * scale);
    }
};

// Raw (untyped) buffer access: descriptor word 3 for gfx9-family parts.  A
// buffer resource covers `bytes` bytes (below 4 GiB) from `p`; loads take a
// per-lane 32-bit byte offset plus a wave-uniform one, and read 0 past the
// end.
constexpr int kBufferWord3 = 0x00020000;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)bytes, kBufferWord3);
}

// The two 16-bit values of a packed word as float, low half first.
template <typename T> struct Unpack16;
template <> struct Unpack16<__half> {
    __device__ __forceinline__ static float lo(uint32_t w) {
        return __half2float(__builtin_bit_cast(__half, (unsigned short)(w & 0xffffu)));
    }
    __device__ __forceinline__ static float hi(uint32_t w) {
        return __half2float(__builtin_bit_cast(__half, (unsigned short)(w >> 16)));
    }
};
template <> struct Unpack16<__hip_bfloat16> {
    __device__ __forceinline__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
    __device__ __forceinline__ static float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};

// Whether work given to the stream is being captured into a graph.
inline bool stream_captures(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &status) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return status != hipStreamCaptureStatusNone;
}
inline unsigned ceil_div(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

// A grid of `tiles` workgroups of `threads` in x and, where that would be 2^32 work
// items or more, which HIP refuses, in y; `z` of them.  The last row may hold tiles
// past the end.
inline dim3 tile_grid(size_t tiles, unsigned threads, unsigned z = 1) {
    const unsigned y = ceil_div(tiles * threads, 0xffffffffu);
    return dim3(ceil_div(tiles, y), y, z);
}
__device__ __forceinline__ uint32_t tile_index() { return blockIdx.x + gridDim.x * blockIdx.y; }

// Dispatch a templated launcher on a TOMO_F32/F16/BF16 code.
#define TOMO_DISPATCH_STORAGE(code, T, ...)                        \
    switch (code) {                                                \
        case TOMO_F32: { using T = float; __VA_ARGS__; break; }    \
        case TOMO_F16: { using T = __half; __VA_ARGS__; break; }   \
        case TOMO_BF16: { using T = __hip_bfloat16; __VA_ARGS__; break; } \
        default: return fail(TOMO_ERR_UNSUPPORTED, "unsupported element type"); \
    }

}  // namespace tomo
