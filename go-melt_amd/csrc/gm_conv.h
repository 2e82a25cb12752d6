// Types and helpers shared by the convolution kernels (gm_conv.hip,
// gm_conv_march.hip, gm_conv_wgrad.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gm_internal.h"

namespace gm {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
    // round to nearest even (finite inputs)
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

struct ConvDims {
    int nb, D, H, W;  // batch and spatial extent
    int ci, co;       // channels (multiples of 16)
    int64_t nvox;     // nb * D * H * W
};

#define CONV_OOB 0x80000000u  // a byte offset past the end of every buffer
#define CONV_DW3 0x00020000   // buffer resource word 3 (raw access)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t conv_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, CONV_DW3);
}

// The marching convolution (gm_conv_march.hip).  conv_march_ok: whether it
// takes these operands; the sums of every output run in the same order as
// the other kernels', so both give the same bits.
bool conv_march_ok(const ConvDims& c, const void* X, const void* Wk, const void* Y,
                   const void* Ybf);
void launch_conv_march(const ConvDims& c, const uint16_t* X, const uint16_t* Wk,
                       const float* bias, int relu, float* Y, uint16_t* Ybf, hipStream_t s);

// The weight gradient on transposing LDS reads (gm_conv_wgrad.hip).
bool conv_wgrad_tr_ok(const ConvDims& c, const void* X, const void* dY);
void launch_conv_wgrad_tr(const ConvDims& c, const uint16_t* X, const uint16_t* dY, float* dW,
                          hipStream_t s);

}  // namespace gm
