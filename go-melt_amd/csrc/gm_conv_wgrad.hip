// Weight gradient of the learned L3 operator's 3x3x3 convolutions (layouts in
// gm_conv.hip).
#include <algorithm>
#include <type_traits>

#include "gm_conv.h"

namespace gm {

// ---------------------------------------------------------------------------
// Weight gradient dW[tap][o][i] += sum_v dY[v][o] X[v + s(tap)][i].
//
// A block of two groups of three waves (one per dy) sums 16 outputs x 16*IT
// inputs of all 27 taps.  A group takes columns of XT x YT voxels, plane by
// plane: plane p of X with its halo and planes p-1, p, p+1 of dY are in LDS,
// so X and dY are read once per channel tile instead of once per tap.  Both operands are
// channels last and the sum runs over voxels, so the fragments (8 voxels of
// one channel per lane) come from transposing LDS reads
// (ds_read_b64_tr_b16: 4 rows of 16 channels per 16 lanes).  A fragment of X
// at one dx feeds the three dz taps.  Rows are 96 bytes apart: the 32-byte
// pieces of four consecutive rows hit distinct banks.  Positions of a tile
// past the volume read zero rows for both operands.  After each column segment
// (32 planes, 2048 voxels, or fewer) the group adds its sums to the block's in LDS, which
// go to dW with FP32 atomics once at the end: short serial sums, and few
// atomics.
// ---------------------------------------------------------------------------
#define WG_ROW 96

template <int XT>
struct WgTile {
    static constexpr int YT = 64 / XT;  // 64 voxels of a plane
    static constexpr int HX = XT + 2, HY = YT + 2, PL = HX * HY;
    static constexpr int ZR = 2 * HX + 3;  // zero rows: any tap offset stays inside
};

template <int XT, int IT>
__global__ void __launch_bounds__(384, 2)
    k_conv_wgrad_tr(ConvDims c, WgGrid g, const uint16_t* __restrict__ X,
                    const uint16_t* __restrict__ dY, float* __restrict__ dW) {
    using G = WgTile<XT>;
    constexpr int NX = (G::PL * 4 + 191) / 192;  // 16-byte loads of X per thread and plane
    constexpr int ND = (64 * 2 + 191) / 192;     // and of dY (two per row: 16 outputs)
    constexpr int XB = G::PL * WG_ROW, DB = 64 * WG_ROW, GB = 2 * XB + 4 * DB;
    __shared__ __align__(16) uint8_t lds[2 * GB + G::ZR * WG_ROW];
    __shared__ v4f sums[27 * IT * 64];  // of the block, in the MFMA's lane order
    const int grp = threadIdx.x >= 192, tid = threadIdx.x - 192 * grp;
    uint8_t* sX = lds + grp * GB;
    uint8_t* sD = sX + 2 * XB;
    uint8_t* sZ = lds + 2 * GB;
    const int lane = tid & 63, dy = tid >> 6;
    const int o0 = blockIdx.y * 16, i0 = blockIdx.z * 16 * IT;
    const int slot = tid & 3, row0 = tid >> 2;   // X rows row0 + 48 q
    const int dslot = tid & 1, drow0 = tid >> 1;  // dY rows drow0 + 96 q
    const uint32_t xvb = (uint32_t)c.ci * 2u, dvb = (uint32_t)c.co * 2u;
    const uint32_t hw = (uint32_t)(c.H * c.W);
    // input channels past cin read zero
    const bool xok = slot * 8 < 16 * IT && i0 + slot * 8 < c.ci;
    for (int r = threadIdx.x; r < G::ZR * WG_ROW / 16; r += 384) *(v4u*)&sZ[r * 16] = v4u{0, 0, 0, 0};
    for (int r = threadIdx.x; r < 27 * IT * 64; r += 384) sums[r] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    v4f acc[3][3][IT];  // [dz][dx]
#pragma unroll
    for (int a = 0; a < 9; ++a)
#pragma unroll
        for (int i = 0; i < IT; ++i) acc[a / 3][a % 3][i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // the barriers are the block's: both groups run every round and plane slot
    const int step = 2 * gridDim.x, rounds = (g.units + step - 1) / step;
    for (int rd = 0; rd < rounds; ++rd) {
        const int u = rd * step + 2 * blockIdx.x + grp;
        const bool uok = u < g.units;
        int t = uok ? u : 0;
        const int x0 = (t % g.nx) * XT;
        t /= g.nx;
        const int y0 = (t % g.ny) * G::YT;
        t /= g.ny;
        const int za = (t % g.nz) * g.zs, b = t / g.nz;
        const int zb = za + g.zs < c.D ? za + g.zs : c.D;
        const auto rX = conv_rsrc(X + (int64_t)b * c.D * hw * c.ci, (uint32_t)c.D * hw * xvb);
        const auto rD = conv_rsrc(dY + (int64_t)b * c.D * hw * c.co, (uint32_t)c.D * hw * dvb);
        uint32_t xoff[NX], doff[ND];
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            const int row = row0 + 48 * q, hy = row / G::HX, hx = row - hy * G::HX;
            const int x = x0 - 1 + hx, y = y0 - 1 + hy;
            const bool ok = xok && row < G::PL && x >= 0 && x < c.W && y >= 0 && y < c.H;
            xoff[q] = ok ? (uint32_t)(y * c.W + x) * xvb + (uint32_t)(i0 * 2 + slot * 16) : CONV_OOB;
        }
#pragma unroll
        for (int q = 0; q < ND; ++q) {
            const int row = drow0 + 96 * q, y = y0 + row / XT, x = x0 + row % XT;
            const bool ok = row < 64 && x < c.W && y < c.H;
            doff[q] = ok ? (uint32_t)(y * c.W + x) * dvb + (uint32_t)(o0 * 2 + dslot * 16) : CONV_OOB;
        }
        auto load_x = [&](int p, v4u* r) {
#pragma unroll
            for (int q = 0; q < NX; ++q)
                r[q] = __builtin_amdgcn_raw_buffer_load_b128(rX, xoff[q], (uint32_t)p * hw * xvb, 0);
        };
        auto put_x = [&](int p, const v4u* r) {
#pragma unroll
            for (int q = 0; q < NX; ++q)
                if (row0 + 48 * q < G::PL)
                    *(v4u*)&sX[(p & 1) * XB + (row0 + 48 * q) * WG_ROW + slot * 16] = r[q];
        };
        auto load_d = [&](int z, v4u* r) {
#pragma unroll
            for (int q = 0; q < ND; ++q)
                r[q] = __builtin_amdgcn_raw_buffer_load_b128(rD, doff[q], (uint32_t)z * hw * dvb, 0);
        };
        auto put_d = [&](int z, const v4u* r) {
#pragma unroll
            for (int q = 0; q < ND; ++q)
                if (drow0 + 96 * q < 64)
                    *(v4u*)&sD[(z & 3) * DB + (drow0 + 96 * q) * WG_ROW + dslot * 16] = r[q];
        };
        // this lane's voxel of each 16-voxel read: row of X (tap dy, dx = -1)
        // and of dY; a voxel past the volume reads zero rows
        const uint8_t* px[4];
        const uint8_t* pd[4];
        uint32_t xs[4], ds[4];  // strides of the plane buffers (0 in the zero rows)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int vi = k * 16 + (lane >> 2), x = vi % XT, y = vi / XT;
            const bool ok = x0 + x < c.W && y0 + y < c.H;
            px[k] = (ok ? sX + ((y + dy) * G::HX + x) * WG_ROW : sZ) + (lane & 3) * 8;
            pd[k] = (ok ? sD + vi * WG_ROW : sZ) + (lane & 3) * 8;
            xs[k] = ok ? XB : 0;
            ds[k] = ok ? DB : 0;
        }
        const int p0 = za > 0 ? za - 1 : 0, p1 = uok ? (zb < c.D ? zb : c.D - 1) : -1;
        __syncthreads();  // the last round's reads are done
        if (uok) {
            v4u r[NX], d[ND];
            load_x(p0, r);
            for (int z = p0; z <= p0 + 1; ++z)
                if (z >= za && z < zb) {
                    load_d(z, d);
                    put_d(z, d);
                }
            put_x(p0, r);
        }
        __syncthreads();
        // plane p of X; bit d of M: dY plane p + 1 - d is in the segment
        auto plane = [&](auto mc, int p) {
            constexpr int M = decltype(mc)::value;
            v4u r[NX], dd[ND];
            const bool mx = p < p1, md = p + 2 < zb;
            if (mx) load_x(p + 1, r);
            if (md) load_d(p + 2, dd);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                typedef __attribute__((address_space(3))) v4s* lp;
                auto frag = [&](const uint8_t* a, const uint8_t* b2) {
                    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(void*)a);
                    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(void*)b2);
                    return __builtin_bit_cast(
                        v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                };
                v8bf fd[3];
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if ((M >> d) & 1)
                        fd[d] = frag(pd[2 * ks] + ((p + 1 - d) & 3) * ds[2 * ks],
                                     pd[2 * ks + 1] + ((p + 1 - d) & 3) * ds[2 * ks + 1]);
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int i = 0; i < IT; ++i) {
                        const v8bf fx =
                            frag(px[2 * ks] + (p & 1) * xs[2 * ks] + dx * WG_ROW + i * 32,
                                 px[2 * ks + 1] + (p & 1) * xs[2 * ks + 1] + dx * WG_ROW + i * 32);
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                            if ((M >> d) & 1)
                                acc[d][dx][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    fd[d], fx, acc[d][dx][i], 0, 0, 0);
                    }
            }
            if (mx) put_x(p + 1, r);
            if (md) put_d(p + 2, dd);
        };
        for (int k = 0; k < g.zs + 2; ++k) {
            const int p = p0 + k;
            const int m = p > p1 ? 0
                                 : (p + 1 >= za && p + 1 < zb ? 1 : 0) |
                                       (p >= za && p < zb ? 2 : 0) |
                                       (p - 1 >= za && p - 1 < zb ? 4 : 0);
            if (m == 7) plane(std::integral_constant<int, 7>{}, p);
            else if (m == 3) plane(std::integral_constant<int, 3>{}, p);
            else if (m == 6) plane(std::integral_constant<int, 6>{}, p);
            else if (m == 1) plane(std::integral_constant<int, 1>{}, p);
            else if (m == 2) plane(std::integral_constant<int, 2>{}, p);
            else if (m == 4) plane(std::integral_constant<int, 4>{}, p);
            __syncthreads();
        }
        // one group after the other adds its sums to the block's (in this
        // order; LDS float atomics took 36 us a segment)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (grp == h && uok) {
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int i = 0; i < IT; ++i) {
                            sums[((d * 9 + dy * 3 + dx) * IT + i) * 64 + lane] += acc[d][dx][i];
                            acc[d][dx][i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                        }
            }
            __syncthreads();
        }
    }
    // lane ln of a tile: outputs (ln >> 4) * 4 + r, input ln & 15
    for (int q = threadIdx.x; q < 27 * IT * 64; q += 384) {
        const int ln = q & 63, k = q >> 6, tap = k / IT;
        const int i = i0 + (k % IT) * 16 + (ln & 15), o = o0 + (ln >> 4) * 4;
        if (i >= c.ci) continue;
        float* w = dW + ((int64_t)tap * c.co + o) * c.ci + i;
        const v4f v = sums[q];
#pragma unroll
        for (int r = 0; r < 4; ++r) atomicAdd(w + (int64_t)r * c.ci, v[r]);
    }
}

template <int XT, int IT>
static void launch_wg(const WgTrPlan& p, const ConvDims& c, const uint16_t* X, const uint16_t* dY,
                      float* dW, hipStream_t s) {
    hipLaunchKernelGGL((k_conv_wgrad_tr<XT, IT>),
                       dim3((unsigned)p.gx, (unsigned)(c.co / 16),
                            (unsigned)((c.ci + 16 * IT - 1) / (16 * IT))),
                       dim3(384), 0, s, c, p.g, X, dY, dW);
}

// 32-bit byte offsets within an image, 16-byte loads, grid limits.
//
// Tile: the x-y shape that pads the volume least; 32 inputs where cin is a
// multiple of 32 and the tiles still fill the chip (one block a CU).  Segments
// of up to 32 planes, shorter where there are fewer than two groups a CU.
// Measured on one MI355X, tap by tap (27 taps over re-read rows) and now, us: 16
// windows 64x64x32, 32 -> 32 573 and 191, 96 -> 32 1980 and 590, 16 -> 32 514
// and 147; 16 of 32x32x16, 64 -> 64 193 and 107, 192 -> 64 550 and 315; 16 of
// 16x16x8, 128 -> 128 101 and 65; 3 of 35x27x13, 48 -> 80 102 and 38.  The relative
// error of the sums fell by half (32 -> 32: 8.6e-7 to 3.7e-7).
// Estimate: the planes a block walks one after the other, fitted to 411 shapes
// of 200 to 6e5 voxels (within 10%, one standard deviation).
bool conv_wgrad_tr_plan(const ConvDims& c, const void* X, const void* dY, WgTrPlan* p) {
    const int64_t vox = (int64_t)c.D * c.H * c.W, lim = (int64_t)1 << 31;
    if ((((uintptr_t)X | (uintptr_t)dY) & 15) || vox * c.ci * 2 >= lim || vox * c.co * 2 >= lim ||
        c.nvox >= lim / 2 || c.ci / 16 >= 65536 || c.co / 16 >= 65536)
        return false;
    const auto pad = [&](int xt) {
        const int yt = 64 / xt;
        return (int64_t)((c.W + xt - 1) / xt * xt) * ((c.H + yt - 1) / yt * yt);
    };
    p->xt = pad(8) < pad(16) ? 8 : 16;
    WgGrid& g = p->g;
    g.nx = (c.W + p->xt - 1) / p->xt;
    g.ny = (c.H + 64 / p->xt - 1) / (64 / p->xt);
    int64_t nt = 1;  // channel tiles
    const auto cut = [&](int it) {  // blocks of one round
        nt = (int64_t)(c.co / 16) * ((c.ci + 16 * it - 1) / (16 * it));
        g.zs = std::min(c.D, 32);
        for (;;) {
            g.nz = (c.D + g.zs - 1) / g.zs;
            g.units = c.nb * g.nx * g.ny * g.nz;
            const int64_t blocks = (g.units + 1) / 2 * nt;
            if (blocks >= 256 || g.zs <= 8) return blocks;
            g.zs = (g.zs + 1) / 2;
        }
    };
    p->wide = c.ci % 32 == 0 && cut(2) >= 128;
    if (!p->wide) cut(1);
    p->gx = std::min((g.units + 1) / 2, (int)std::max<int64_t>(1, 256 / nt));
    const int64_t rounds = (g.units + 2 * p->gx - 1) / (2 * p->gx);
    const int64_t planes = (p->gx * nt + 255) / 256 * rounds * (g.zs + 2);
    p->us = p->wide ? 9.5 + 1.25 * planes : 5.0 + 1.0 * planes;
    return true;
}

void launch_conv_wgrad_tr(const WgTrPlan& p, const ConvDims& c, const uint16_t* X,
                          const uint16_t* dY, float* dW, hipStream_t s) {
    if (p.xt == 16) {
        if (p.wide) launch_wg<16, 2>(p, c, X, dY, dW, s);
        else launch_wg<16, 1>(p, c, X, dY, dW, s);
    } else {
        if (p.wide) launch_wg<8, 2>(p, c, X, dY, dW, s);
        else launch_wg<8, 1>(p, c, X, dY, dW, s);
    }
}

}  // namespace gm
