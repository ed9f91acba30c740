// sl_raster_impl.h -- the parts of the raster below its walk: a fragment's
// shading, the attachments' texel access and blending, wave helpers, and the
// occupancy cap of its launches.  Included by sl_raster_wave.h.
//
// Reference routines reproduced: SL_FragmentProcessor::flush_tri_fragments
// (SL_FragmentProcessor.cpp:416-531).
#pragma once

#include <algorithm>

#include <hip/hip_fp16.h>

#include "sl_device.h"
#include "sl_stages.h"
#include "sl_kernels.h"

namespace slg {
namespace {

// Greatest value over the wave's 64 lanes (every lane active): pairs and
// quads with DPP quad permutes, the 16-lane row by rotating it 4 and 8 lanes,
// then the four rows' results read from lanes 0, 16, 32 and 48.  NaN inputs
// are ignored (fmaxf) unless every lane holds one.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}

__device__ __forceinline__ float wave_max_f32(float v)
{
    v = fmaxf(v, dpp_f32<0xB1>(v));    // quad_perm [1,0,3,2]: lane ^ 1
    v = fmaxf(v, dpp_f32<0x4E>(v));    // quad_perm [2,3,0,1]: lane ^ 2
    v = fmaxf(v, dpp_f32<0x124>(v));   // row_ror:4
    v = fmaxf(v, dpp_f32<0x128>(v));   // row_ror:8
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// Shading of one fragment from its record and its barycentric values s0..s2
// (perspective correction SL_FragmentProcessor.cpp:486-494, varyings :315-330,
// then the fragment program).  `wv` receives the visibility slot's varying.
// The destination a blend reads from a texel of n < 4 components
// (assign_alpha_pixel, SL_Framebuffer.cpp:296-311): (r, min, min, max),
// (r, g, min, max), and for three components (r, r, r, max).
__device__ __forceinline__ void blend_dst_read(int n, float one, float d[4])
{
    // selects, not conditional stores, so d stays in registers
    const float r = d[0];
    const float g = (n == 3) ? r : ((n == 1) ? 0.f : d[1]);
    const float b = (n == 4) ? d[2] : ((n == 3) ? r : 0.f);
    const float a = (n == 4) ? d[3] : one;
    d[1] = g;
    d[2] = b;
    d[3] = a;
}

// Output k (1..3) of a multiple-output program into colour attachment k at
// texel gi, written or blended as assign_pixel / assign_alpha_pixel do.
// These attachments are read and written in place: a texel is only ever
// touched by the lane that owns it.
__device__ __forceinline__ void write_extra_output(const RasterParams& P, int k, uint64_t gi, float4 o, int blendMode)
{
    const int n = P.colorXComps[k];
    if (P.colorXFloat[k])
    {
        float* px = reinterpret_cast<float*>(P.colorX[k]) + gi * (uint64_t)n;
        float d[4] = {o.x, o.y, o.z, o.w};
        if (blendMode != SL_BLEND_OFF)
        {
#pragma unroll
            for (int c = 0; c < 4; ++c) d[c] = (c < n) ? px[c] : 0.f;
            blend_dst_read(n, 1.f, d);
            blend(blendMode, o, d);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c < n) px[c] = d[c];
    }
    else if (P.colorXPacked[k] != 0)
    {
        const PackedFmt f = packed_format(P.colorXPacked[k]);
        uint8_t* px = P.colorX[k] + gi * (uint64_t)f.bytes;
        uint32_t w = 0;
        for (int b = 0; b < f.bytes; ++b) w |= (uint32_t)px[b] << (8 * b);
        float d[4] = {o.x, o.y, o.z, o.w};
        if (blendMode != SL_BLEND_OFF)
        {
            packed_decode(f, w, d);
            blend(blendMode, o, d);
        }
        w = packed_encode(f, d);
        for (int b = 0; b < f.bytes; ++b) px[b] = (uint8_t)(w >> (8 * b));
    }
    else
    {
        uint8_t* px = P.colorX[k] + gi * (uint64_t)n;
        float d[4] = {o.x, o.y, o.z, o.w};
        if (blendMode != SL_BLEND_OFF)
        {
#pragma unroll
            for (int c = 0; c < 4; ++c) d[c] = (c < n) ? (float)px[c] * 0.00392156862745f : 0.f;
            blend_dst_read(n, 255.f * 0.00392156862745f, d);
            blend(blendMode, o, d);
        }
        const uint32_t v = pack_rgba8(d);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c < n) px[c] = (uint8_t)(v >> (8 * c));
    }
}

// A point's varyings pass unchanged (SL_PointRasterizer.cpp:66-69); a line's
// are mixed by its position s0 (interpolate_line_varyings,
// SL_FragmentProcessor.cpp:119-145).  Outputs 1..3 of a multiple-output
// program go straight to their attachments at texel gi (attachments 3, 2, 1,
// as the reference's output switch falls through); output 0 is returned.
// Only the MRT raster variants carry that code.
template <bool MRT>
__device__ __forceinline__ bool shade(const RasterParams& P, const DrawDesc& D, const float hw[3], float bc3, uint32_t state,
                                      uint32_t rid, float s0, float s1, float s2, float4& out, float4& wv,
                                      uint64_t gi, int blendMode)
{
    const float t0 = s0 * hw[0], t1 = s1 * hw[1], t2 = s2 * hw[2];
    const float sinv = rcpf(((t0 + t1) + t2) + bc3);
    const float c0 = t0 * sinv, c1 = t1 * sinv, c2 = t2 * sinv;
    const float4* V = P.vars + (uint64_t)rid * P.varStride;
    const uint32_t nvMax = P.varStride / 3;
    const bool point = (state & kStatePoint) != 0u, line = (state & kStateLine) != 0u;
    Vary4 var;
#pragma unroll
    for (int i = 0; i < SL_SHADER_MAX_VARYING_VECTORS; ++i)
    {
        if (i < D.nvary)
        {
            const float4 a = V[i];
            if (point)
            {
                var.v[i] = a;
            }
            else if (line)
            {
                var.v[i] = mix4(a, V[nvMax + i], s0);
            }
            else
            {
                const float4 b = V[nvMax + i], e = V[2 * nvMax + i];
                var.v[i] = f4(((a.x * c0) + (b.x * c1)) + (e.x * c2), ((a.y * c0) + (b.y * c1)) + (e.y * c2),
                              ((a.z * c0) + (b.z * c1)) + (e.z * c2), ((a.w * c0) + (b.w * c1)) + (e.w * c2));
            }
        }
        else
        {
            var.v[i] = f4(0.f, 0.f, 0.f, 0.f);
        }
    }
    wv = f4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < SL_SHADER_MAX_VARYING_VECTORS; ++i)
        if ((uint32_t)i == D.visSlot) wv = var.v[i];
    if (!MRT || D.nout <= 1) return (D.nout > 0) && fragment_program(D, P.uniforms, var, out);
    float4 extra[3];
    const bool have = fragment_program(D, P.uniforms, var, out, extra);
    if (have)
        for (int k = (int)D.nout - 1; k >= 1; --k) write_extra_output(P, k - 1, gi, extra[k - 1], blendMode);
    return have;
}

// Attachment texels of P.colorComps components (8-bit: packed into the low
// bytes of a u32; float: the leading components of a float4), and the
// depth texel (R32F, or R16F read as float and written rounded to nearest).
__device__ __forceinline__ uint32_t load_color8(const RasterParams& P, uint64_t gi)
{
    const int n = P.colorComps;   // bytes per texel for a packed format
    if (n == 4) return reinterpret_cast<const uint32_t*>(P.color)[gi];
    const uint8_t* p = P.color + gi * (uint64_t)n;
    uint32_t v = 0;
    for (int k = 0; k < n; ++k) v |= (uint32_t)p[k] << (8 * k);
    return v;
}

__device__ __forceinline__ void store_color8(const RasterParams& P, uint64_t gi, uint32_t v)
{
    const int n = P.colorComps;
    if (n == 4) { reinterpret_cast<uint32_t*>(P.color)[gi] = v; return; }
    uint8_t* p = P.color + gi * (uint64_t)n;
    for (int k = 0; k < n; ++k) p[k] = (uint8_t)(v >> (8 * k));
}

__device__ __forceinline__ float4 load_colorF(const RasterParams& P, uint64_t gi)
{
    const int n = P.colorComps;
    if (n == 4) return reinterpret_cast<const float4*>(P.color)[gi];
    const float* p = reinterpret_cast<const float*>(P.color) + gi * (uint64_t)n;
    return make_float4(p[0], n > 1 ? p[1] : 0.f, n > 2 ? p[2] : 0.f, 0.f);
}

__device__ __forceinline__ void store_colorF(const RasterParams& P, uint64_t gi, float4 v)
{
    const int n = P.colorComps;
    if (n == 4) { reinterpret_cast<float4*>(P.color)[gi] = v; return; }
    float* p = reinterpret_cast<float*>(P.color) + gi * (uint64_t)n;
    p[0] = v.x;
    if (n > 1) p[1] = v.y;
    if (n > 2) p[2] = v.z;
}

__device__ __forceinline__ float load_depth(const RasterParams& P, uint64_t gi)
{
    return P.depthHalf ? __half2float(reinterpret_cast<const __half*>(P.depth)[gi]) : P.depth[gi];
}

__device__ __forceinline__ void store_depth(const RasterParams& P, uint64_t gi, float z)
{
    if (P.depthHalf) reinterpret_cast<__half*>(P.depth)[gi] = __float2half_rn(z);
    else P.depth[gi] = z;
}

template <int CF>
__device__ __forceinline__ void blend_into(uint32_t* col8, float4* colF, int blendMode, float4 out, int comps, int packed)
{
    if (CF == 1 && packed != 0)
    {
        // a packed texel: decoded whole, blended, clamped, encoded (SL_Framebuffer.cpp:370-560)
        const PackedFmt f = packed_format(packed);
        float o[4] = {out.x, out.y, out.z, out.w};
        if (blendMode != SL_BLEND_OFF)
        {
            packed_decode(f, *col8, o);
            blend(blendMode, out, o);
        }
        *col8 = packed_encode(f, o);
        return;
    }
    if (CF == 1)
    {
        if (blendMode == SL_BLEND_OFF)
        {
            const float o[4] = {out.x, out.y, out.z, out.w};
            *col8 = pack_rgba8(o);
        }
        else
        {
            float dcol[4];
            unpack_rgba8(*col8, dcol);
            blend_dst_read(comps, 255.f * 0.00392156862745f, dcol);   // max (255) cast to float
            blend(blendMode, out, dcol);
            *col8 = pack_rgba8(dcol);
        }
    }
    if (CF == 2)
    {
        if (blendMode == SL_BLEND_OFF)
        {
            *colF = out;
        }
        else
        {
            const float4 cur = *colF;
            float dcol[4] = {cur.x, cur.y, cur.z, cur.w};
            blend_dst_read(comps, 1.f, dcol);
            blend(blendMode, out, dcol);
            *colF = make_float4(dcol[0], dcol[1], dcol[2], dcol[3]);
        }
    }
}

constexpr uint32_t kNoPending = 0xFFFFFFFFu;

}  // namespace

// Dynamic LDS that caps the resident workgroups of a raster kernel at
// wgPerCU per CU (0: no cap): each workgroup then holds LDS / wgPerCU of the
// CU's LDS (its static arrays plus the rest as unused dynamic LDS), within
// the per-workgroup limit.
struct LdsLimits { size_t perCU, perBlock; };

static LdsLimits lds_limits()
{
    static const LdsLimits L = [] {
        int dev = 0, cu = 0, blk = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess) cu = 0;
        if (hipDeviceGetAttribute(&blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) blk = 0;
        return LdsLimits{(size_t)std::max(cu, 0), (size_t)std::max(blk, 0)};
    }();
    return L;
}

template <class Kernel>
static size_t occupancy_lds(Kernel kernel, uint32_t wgPerCU)
{
    if (wgPerCU == 0) return 0;
    hipFuncAttributes a{};
    if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(kernel)) != hipSuccess) return 0;
    const LdsLimits L = lds_limits();
    const size_t stat = a.sharedSizeBytes, want = std::min(L.perCU / wgPerCU, L.perBlock);
    return want > stat ? want - stat : 0;
}

}  // namespace slg
