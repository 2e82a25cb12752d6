// 3x3x3 convolutions of the learned L3 operator, marching along z (layouts in
// gm_conv.hip): the forward pass and, with the flipped weights, the gradient
// of the input, for input channels in multiples of 32.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "gm_conv.h"

namespace gm {

#define CONV_ROW 64  // LDS bytes of a row of 32 channels

// ---------------------------------------------------------------------------
// Forward (and input-gradient) convolution marching along z.
//
// A block of four waves computes an XT x YT column of voxels x 16*NT outputs
// over the planes za .. zb-1.  Plane p and its halo are in LDS once, with all
// channels; each fragment (16 voxels x 32 channels at one (dy, dx)) is read
// once and feeds the three output planes it belongs to: p+1 (dz = -1), p and
// p-1 (dz = +1), whose sums rotate through three accumulator sets.  Every
// output's sum therefore runs tap by tap in increasing order, the channels
// inner: the same bits whatever the tile shape.  The weights of a stage
// (three steps of one (dy, dx) x 32 channels, 3 dz x outputs each) pass
// through a double LDS buffer; the next stage's weights and a share of the
// next plane are in flight during the MFMAs.  RES (32 input channels): all
// weights stay in LDS and a plane is one stage.  The weights are the MFMA's A operand, so a lane ends with four
// consecutive outputs of one voxel: 16-byte stores.  LDS rows are 64 bytes
// with their 16-byte slots swizzled by (row >> 1) & 3, so the reads of eight
// consecutive rows hit distinct banks.
// ---------------------------------------------------------------------------
template <int XT, int YW, int WV>
struct ConvTile {
    static constexpr int YF = 16 / XT;       // y rows of a 16-voxel fragment
    static constexpr int YT = WV * YF * YW;  // y rows of a block of WV waves
    static constexpr int HX = XT + 2, HY = YT + 2;
    static constexpr int PL = HX * HY;  // halo rows of a plane
};

extern __shared__ __align__(16) uint8_t conv_lds[];

template <int XT, int YW, int NT, int WV, int S>
__global__ void __launch_bounds__(64 * WV, 2)
    k_conv_march(ConvDims c, TileGrid tg, const uint16_t* __restrict__ X,
                 const uint16_t* __restrict__ Wk, const float* __restrict__ bias, int relu,
                 float* __restrict__ Y, uint16_t* __restrict__ Ybf) {
    using G = ConvTile<XT, YW, WV>;
    constexpr bool RES = S == 9;
    constexpr int NTHR = 64 * WV, RP = NTHR / 4;    // rows of a load pass
    constexpr int NO = 16 * NT;                     // outputs of the block
    constexpr int NA = (G::PL + RP - 1) / RP;       // plane load passes per 32 channels
    constexpr int BR = 3 * NO;                      // weight rows of a step
    constexpr int BRS = S * BR;                     // and of a stage
    constexpr int NB = (BRS + RP - 1) / RP;
    constexpr int PB = G::PL * CONV_ROW;            // bytes of a plane of 32 channels
    constexpr int APS = (NA * S + 8) / 9;           // plane load passes per stage
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nch = RES ? 1 : c.ci / 32;
    uint8_t* sB = conv_lds + 2 * nch * PB;  // after the two plane buffers
    // a run of consecutive columns (with all their output tiles) per XCD
    int t = xcd_tile(blockIdx.x, gridDim.x);
    const int n0 = (t % tg.nt) * NO;
    t /= tg.nt;
    const int x0 = (t % tg.nx) * XT;
    t /= tg.nx;
    const int y0 = (t % tg.ny) * G::YT;
    t /= tg.ny;
    const int za = (t % tg.nz) * tg.zs, b = t / tg.nz;
    const int zb = za + tg.zs < c.D ? za + tg.zs : c.D;
    const int slot = tid & 3, row0 = tid >> 2;
    const int bslot = slot ^ ((row0 >> 1) & 3);  // the same for rows row0 + 64 q

    const uint32_t vb = (uint32_t)c.ci * 2u, plane_b = (uint32_t)(c.H * c.W) * vb;
    const auto rX = conv_rsrc(X + (int64_t)b * c.D * c.H * c.W * c.ci, plane_b * (uint32_t)c.D);
    const auto rW = conv_rsrc(Wk, (uint32_t)(27 * c.co) * vb);
    uint32_t aoff[NA];  // byte offsets of this thread's halo rows in a plane
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        const int row = row0 + RP * q;
        const int hy = row / G::HX, hx = row - hy * G::HX;
        const int x = x0 - 1 + hx, y = y0 - 1 + hy;
        const bool ok = row < G::PL && x >= 0 && x < c.W && y >= 0 && y < c.H;
        aoff[q] = ok ? (uint32_t)(y * c.W + x) * vb + slot * 16 : CONV_OOB;
    }
    // its weight rows (step k of the stage, dz, output): byte offsets at the
    // first step; step (ph, ch) adds ph * wph + 64 ch.  Steps run over
    // (dy, dx) outer, 32-channel stage inner.
    const uint32_t wph = (uint32_t)c.co * vb;
    uint32_t boff[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int row = row0 + RP * q, r2 = row % BR, dz = r2 / NO, n = r2 - dz * NO;
        boff[q] = row < BRS && n0 + n < c.co
                      ? (uint32_t)(dz * 9 * c.co + n0 + n) * vb + slot * 16 +
                            (RES ? (row / BR) * wph : 0u)
                      : CONV_OOB;
    }
    auto load_b = [&](const uint32_t* so, v4u* rb) {  // so[k]: the offset of step k
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            uint32_t o = boff[q];
            if constexpr (!RES) {
                // the steps that the rows of pass q belong to
                const int k0 = RP * q / BR, k1 = (RP * q + RP - 1) / BR;
                uint32_t s = so[k0 < S ? k0 : S - 1];
#pragma unroll
                for (int k = k0 + 1; k <= k1 && k < S; ++k)
                    if (row0 + RP * q >= k * BR) s = so[k];
                if (o != CONV_OOB) o += s;
            }
            rb[q] = __builtin_amdgcn_raw_buffer_load_b128(rW, o, 0, 0);
        }
    };
    auto put_b = [&](int buf, const v4u* rb) {
#pragma unroll
        for (int q = 0; q < NB; ++q)
            if ((q + 1) * RP <= BRS || row0 + RP * q < BRS)
                *(v4u*)&sB[(buf * BRS + row0 + RP * q) * CONV_ROW + bslot * 16] = rb[q];
    };
    auto load_a = [&](int p, int ch, int q) {
        return __builtin_amdgcn_raw_buffer_load_b128(rX, aoff[q], (uint32_t)p * plane_b + ch * 64, 0);
    };
    auto put_a = [&](int p, int ch, int q, v4u v) {
        if ((q + 1) * RP <= G::PL || row0 + RP * q < G::PL)
            *(v4u*)&conv_lds[((p & 1) * nch + ch) * PB + (row0 + RP * q) * CONV_ROW + bslot * 16] =
                v;
    };
    v4f acc[3][YW][NT];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < YW; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[d][j][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    // this lane's voxel of the fragments (column of the product) and k slot
    const int fx = lane & (XT - 1), fy = wave * (G::YF * YW) + ((lane & 15) / XT);
    const int frow = fy * G::HX + fx, fk = lane >> 4;
    const uint8_t* pb0 = sB + (lane & 15) * CONV_ROW + (fk ^ ((lane >> 1) & 3)) * 16;
    const int x = x0 + fx, og = n0 + (lane >> 4) * 4;

    // finished plane z: lane holds outputs og + 16 n .. + 3 of its voxels
    auto store = [&](int z, v4f(&a)[YW][NT]) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int o = og + n * 16;
            const bool nok = x < c.W && n0 + n * 16 < c.co;
            v4f bv = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (bias && nok) bv = v4f{bias[o], bias[o + 1], bias[o + 2], bias[o + 3]};
#pragma unroll
            for (int j = 0; j < YW; ++j) {
                const int y = y0 + fy + j * G::YF;
                v4f v = a[j][n] + bv;
                a[j][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                if (!nok || y >= c.H) continue;
                const int64_t i = ((((int64_t)b * c.D + z) * c.H + y) * c.W + x) * c.co + o;
                if (relu) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (v[r] < 0.0f) v[r] = 0.0f;
                }
                if (Y) *(v4f*)(Y + i) = v;
                if (Ybf) {
                    uint2 h;
                    h.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
                    h.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
                    *(uint2*)(Ybf + i) = h;
                }
            }
        }
    };
    const int p0 = za > 0 ? za - 1 : 0, p1 = zb < c.D ? zb : c.D - 1;
    {  // the first plane and weights
        v4u rb[NB];
        uint32_t so[S];
        for (int k = 0, ph = 0, ch = 0; k < S; ++k) {
            so[k] = ph * wph + ch * 64;
            if (++ch == nch) ch = 0, ++ph;
        }
        load_b(so, rb);
        for (int ch = 0; ch < nch; ++ch) {
            v4u ra[NA];
#pragma unroll
            for (int q = 0; q < NA; ++q) ra[q] = load_a(p0, ch, q);
#pragma unroll
            for (int q = 0; q < NA; ++q) put_a(p0, ch, q, ra[q]);
        }
        put_b(0, rb);
    }
    __syncthreads();
    int buf = 0;
    // plane p; its outputs p+1, p, p-1 are in sets R+1, R, R+2 (mod 3).  M: the
    // outputs summed (bit d: p+1-d).  The planes at the ends of a segment sum
    // one output too many rather than branch inside the products: it is never
    // stored, and a set is cleared when its plane has passed.
    auto plane = [&](auto rc, auto mc, int p) {
        constexpr int R = decltype(rc)::value, M = decltype(mc)::value;
        auto step = [&](int ph, int ch, int kb) {
            const int dy = ph / 3, dx = ph - dy * 3;
            const uint8_t* pa = conv_lds + ((p & 1) * nch + ch) * PB;
            const uint8_t* pb = pb0 + kb * BR * CONV_ROW;
            v8bf fw[3][NT], fv[YW];
#pragma unroll
            for (int j = 0; j < YW; ++j) {
                const int ar = frow + (j * G::YF + dy) * G::HX + dx;
                fv[j] = __builtin_bit_cast(
                    v8bf, *(const v4u*)(pa + ar * CONV_ROW + (fk ^ ((ar >> 1) & 3)) * 16));
            }
#pragma unroll
            for (int d = 0; d < 3; ++d)
                if ((M >> d) & 1)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        fw[d][n] = __builtin_bit_cast(
                            v8bf, *(const v4u*)(pb + (d * NO + n * 16) * CONV_ROW));
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if (!((M >> d) & 1)) continue;
#pragma unroll
                for (int j = 0; j < YW; ++j)
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        v4f& s = acc[(R + 4 - d) % 3][j][n];
                        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[d][n], fv[j], s, 0, 0, 0);
                    }
            }
        };
        if constexpr (RES) {
            v4u ra[NA];
            if (p < p1)
#pragma unroll
                for (int q = 0; q < NA; ++q) ra[q] = load_a(p + 1, 0, q);
#pragma unroll
            for (int ph = 0; ph < 9; ++ph) step(ph, 0, ph);
            if (p < p1)
#pragma unroll
                for (int q = 0; q < NA; ++q) put_a(p + 1, 0, q, ra[q]);
            __syncthreads();
        } else {
            int ph = 0, ch = 0, phn = S / nch, chn = S % nch;  // this stage's step, the next's
            for (int c3 = 0; c3 < nch; ++c3) {
#pragma unroll
                for (int r = 0; r < 9 / S; ++r) {
                    // in flight during the products: the next stage's weights
                    // and a share of the next plane
                    v4u rb[NB], ra[APS];
                    uint32_t so[S];
                    if (phn >= 9) phn = 0, chn = 0;  // the next plane's first
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        so[k] = phn * wph + chn * 64;
                        if (++chn == nch) chn = 0, ++phn;
                    }
                    load_b(so, rb);
                    if (p < p1)
#pragma unroll
                        for (int k = 0; k < APS; ++k)
                            if (r * APS + k < NA) ra[k] = load_a(p + 1, c3, r * APS + k);
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        step(ph, ch, buf * S + k);
                        if (++ch == nch) ch = 0, ++ph;
                    }
                    put_b(buf ^ 1, rb);
                    if (p < p1)
#pragma unroll
                        for (int k = 0; k < APS; ++k)
                            if (r * APS + k < NA) put_a(p + 1, c3, r * APS + k, ra[k]);
                    __syncthreads();
                    buf ^= 1;
                }
            }
        }
        if (p - 1 >= za) {
            store(p - 1, acc[(R + 2) % 3]);
        } else {
#pragma unroll
            for (int j = 0; j < YW; ++j)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[(R + 2) % 3][j][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if (p == c.D - 1 && p < zb) store(p, acc[R]);
    };
    auto rotate = [&](auto rc, int p) {
        if (p <= za) plane(rc, std::integral_constant<int, 3>{}, p);
        else if (p >= zb - 1) plane(rc, std::integral_constant<int, 6>{}, p);
        else plane(rc, std::integral_constant<int, 7>{}, p);
    };
    for (int p = p0; p <= p1; ++p) {
        const int r = p % 3;
        if (r == 0) rotate(std::integral_constant<int, 0>{}, p);
        else if (r == 1) rotate(std::integral_constant<int, 1>{}, p);
        else rotate(std::integral_constant<int, 2>{}, p);
    }
}

// All shapes the launcher instantiates.  s = 9: 32 input channels, weights
// resident in LDS.
static const MarchCfg kMarch[] = {
    {16, 2, 2, 8, 9, 0.02}, {16, 4, 1, 4, 9, 0.02}, {16, 2, 1, 4, 9, 0.02}, {8, 1, 2, 4, 9, 0.02},
    {8, 1, 1, 4, 9, 0.02},  {16, 2, 2, 8, 3, 0.13}, {16, 1, 4, 8, 1, 0.23}, {16, 1, 2, 8, 3, 0.10},
    {16, 1, 2, 4, 3, 0.16}, {16, 2, 1, 4, 3, 0.11}, {8, 1, 2, 4, 3, 0.16},  {8, 1, 1, 4, 3, 0.11}};

static const size_t kLds = 160 * 1024;

// Shape and z segments by estimated time: a block runs its planes (a segment
// and its two neighbours, 1.2 us each for the stores and the first reads) in
// 9 steps per 32 channels, each the shape's latency (LDS reads, barriers)
// plus 12 ns per MFMA of the waves that share a SIMD.  Measured on one MI355X (us, FP32 and bf16 outputs;
// the tap-by-tap kernel before it in brackets): 16 windows of 64x64x32,
// 32 -> 32 {16,2,2,8,9} 160 (446), 96 -> 32 {16,2,2,8,3} 430 (1200, 0.50 us a
// step); 16 of 32x32x16, 64 -> 64 {16,2,2,8,3} 83 (151), 192 -> 64 {16,1,4,8,1}
// 296 (470, 0.55 us a step); 16 of 16x16x8, 128 -> 128 {16,1,2,8,3} 57 (95),
// 256 -> 128 {16,1,2,4,3} 147 (180); 16 of 8x8x4, 128 -> 128 {8,1,1,4,3} 24 (51);
// one window 64x64x32, 32 -> 32 {16,2,1,4,9} 16 (40), 96 -> 32 {16,2,2,8,3} 46
// (101); 32x32x16, 192 -> 64 {16,2,1,4,3} 48 (75).
static bool march_plan(const ConvDims& c, MarchPlan* best) {
    const int nch = c.ci / 32;
    bool found = false;
    for (const MarchCfg& g : kMarch) {
        if ((g.s == 9) != (nch == 1) || (g.nt > 1 && c.co % (16 * g.nt))) continue;
        const int yf = 16 / g.xt, yt = g.wv * yf * g.yw, pl = (g.xt + 2) * (yt + 2);
        MarchPlan p;
        p.g = g;
        p.lds = (size_t)2 * nch * pl * CONV_ROW + (size_t)(g.s == 9 ? 9 : 2 * g.s) * 48 * g.nt * CONV_ROW;
        if (p.lds > kLds) continue;
        const int res = std::max(1, std::min(8 / g.wv, (int)(kLds / p.lds)));
        p.tg.nx = (c.W + g.xt - 1) / g.xt;
        p.tg.ny = (c.H + yt - 1) / yt;
        p.tg.nt = (c.co + 16 * g.nt - 1) / (16 * g.nt);
        for (int seg = 1; seg <= c.D; seg *= 2) {
            p.tg.zs = (c.D + seg - 1) / seg;
            p.tg.nz = (c.D + p.tg.zs - 1) / p.tg.zs;
            p.blocks = (int64_t)c.nb * p.tg.nx * p.tg.ny * p.tg.nz * p.tg.nt;
            if (p.blocks * 64 * g.wv >= (int64_t)1 << 32) continue;  // threads of a grid
            const double per_cu = std::min((double)res, ceil(p.blocks / 256.0));
            const double gens = ceil(p.blocks / (256.0 * per_cu));
            const int planes = std::min(p.tg.zs + 2, c.D);
            const double step = g.lat + 0.012 * (3 * g.yw * g.nt) * (g.wv / 4) * per_cu;
            p.us = gens * (2.5 + planes * (1.2 + 9.0 * nch * step));
            if (!found || p.us < best->us) *best = p;
            found = true;
        }
    }
    return found;
}

// 32-bit byte offsets within an image and the weights, 16-byte accesses
bool conv_march_plan(const ConvDims& c, const void* X, const void* Wk, const void* Y,
                     const void* Ybf, MarchPlan* p) {
    const int64_t lim = (int64_t)1 << 31;
    return c.ci % 32 == 0 &&
           (((uintptr_t)X | (uintptr_t)Wk | (uintptr_t)Y) & 15) == 0 &&
           ((uintptr_t)Ybf & 7) == 0 && (int64_t)c.D * c.H * c.W * c.ci * 2 < lim &&
           (int64_t)27 * c.ci * c.co * 2 < lim && march_plan(c, p);
}

template <int XT, int YW, int NT, int WV, int S>
static void launch_march(const MarchPlan& p, const ConvDims& c, const uint16_t* X,
                         const uint16_t* Wk, const float* bias, int relu, float* Y,
                         uint16_t* Ybf, hipStream_t s) {
    const auto k = k_conv_march<XT, YW, NT, WV, S>;
    if (p.lds > 64 * 1024)
        (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)kLds);
    hipLaunchKernelGGL(k, dim3((unsigned)p.blocks), dim3(64 * WV), p.lds, s, c, p.tg, X, Wk, bias,
                       relu, Y, Ybf);
}

void launch_conv_march(const MarchPlan& p, const ConvDims& c, const uint16_t* X,
                       const uint16_t* Wk, const float* bias, int relu, float* Y, uint16_t* Ybf,
                       hipStream_t s) {
    const MarchCfg& g = p.g;
#define GM_MARCH(XT, YW, NT, WV, S)                                                    \
    if (g.xt == XT && g.yw == YW && g.nt == NT && g.wv == WV && g.s == S)              \
        return launch_march<XT, YW, NT, WV, S>(p, c, X, Wk, bias, relu, Y, Ybf, s);
    GM_MARCH(16, 2, 2, 8, 9)
    GM_MARCH(16, 4, 1, 4, 9)
    GM_MARCH(16, 2, 1, 4, 9)
    GM_MARCH(8, 1, 2, 4, 9)
    GM_MARCH(8, 1, 1, 4, 9)
    GM_MARCH(16, 2, 2, 8, 3)
    GM_MARCH(16, 1, 4, 8, 1)
    GM_MARCH(16, 1, 2, 8, 3)
    GM_MARCH(16, 1, 2, 4, 3)
    GM_MARCH(16, 2, 1, 4, 3)
    GM_MARCH(8, 1, 2, 4, 3)
    GM_MARCH(8, 1, 1, 4, 3)
#undef GM_MARCH
}

}  // namespace gm
