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

// The marching convolution (gm_conv_march.hip): tile shape, cut of the volume
// and estimated time of a launch.
struct MarchCfg {
    int xt, yw, nt, wv, s;
    double lat;  // latency of a step, us (see march_plan)
};
// columns of a volume (x fastest, then y, z segments, batch) and output tiles
struct TileGrid {
    int nx, ny, nz, nt;
    int zs;  // planes of a segment
};
struct MarchPlan {
    MarchCfg g;
    TileGrid tg;
    int64_t blocks = 0;
    size_t lds = 0;
    double us = 0.0;
};
// whether the kernel takes these operands, and how.  Every output's sum runs
// tap by tap, the channels inner, as in the unsplit k_conv_fwd32: the same
// bits from both.
bool conv_march_plan(const ConvDims& c, const void* X, const void* Wk, const void* Y,
                     const void* Ybf, MarchPlan* p);
void launch_conv_march(const MarchPlan& p, const ConvDims& c, const uint16_t* X,
                       const uint16_t* Wk, const float* bias, int relu, float* Y, uint16_t* Ybf,
                       hipStream_t s);

// The weight gradient on transposing LDS reads (gm_conv_wgrad.hip).
struct WgGrid {
    int nx, ny, nz, zs;  // columns per axis, z segments of zs planes
    int units;           // nb * nx * ny * nz
};
struct WgTrPlan {
    int xt;     // column width
    bool wide;  // 32 inputs a block
    WgGrid g;
    int gx;     // blocks a channel tile
    double us;  // estimated time
};
// whether the kernel takes these operands, and how
bool conv_wgrad_tr_plan(const ConvDims& c, const void* X, const void* dY, WgTrPlan* p);
void launch_conv_wgrad_tr(const WgTrPlan& p, const ConvDims& c, const uint16_t* X,
                          const uint16_t* dY, float* dW, hipStream_t s);

}  // namespace gm
