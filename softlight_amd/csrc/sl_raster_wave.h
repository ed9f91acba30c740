// sl_raster_wave.h -- k_raster_wave, the fragment stage for batches of filled
// triangles: one wave per 8x8 pixel block, one pixel per lane.  Included by
// the sl_raster_wave*.hip translation units.
//
// Reference routines reproduced: SL_TriRasterizer::render_triangle_simd
// generic branch (SL_TriRasterizer.cpp:806-923),
// SL_FragmentProcessor::flush_tri_fragments (SL_FragmentProcessor.cpp:416-531).
#pragma once

#include "sl_raster_impl.h"

namespace slg {
namespace {

// Lanes of the wave below this one in `mask`.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ float readlane_f32(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// LDS traffic of one wave: its operations execute in order, so ordering them
// only needs the compiler kept from moving them.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// k_raster_wave: a wave owns an 8x8 block of its tile and walks the tile's
// record list; a pixel's depth, colour and pending fragment live in its
// lane's registers for the whole batch.
//
//   list     64 records at a time, one per lane: the lane works out its
//            record's coverage of the block, a 64-bit mask, with the
//            scanline rule itself (so the mask is exact), and the record's
//            depth plane with a bound on the float error of the depths the
//            walk computes.  A record whose plane lies behind every pixel of
//            the block leaves the list here.
//   filter   the records left, in order, each against the 64 pixels at once:
//            the pixels it covers whose depth test the plane's bound does not
//            already decide become queued fragments.  `bound` holds, per
//            pixel, a value no smaller than the depth after every fragment
//            queued so far.
//   flush    when 64 fragments wait: one fragment per lane, the exact
//            barycentrics (the reference's recurrence, stepped from the
//            span's first pixel) and depth; then each pixel takes its own
//            fragments in record order: depth test, counters, pending
//            fragment or blend.
//
// Why: a record's cost used to be the recurrence's steps (up to W / 4 dependent
// additions) for every lane it reached, although on overlapping triangles 98%
// of the depth tests fail by far more than rounding; and 512 pixels a wave
// left most of the chip's 1024 SIMDs idle on small targets.  Now the steps are
// taken only for fragments that can pass, 64 of them side by side.  Measured
// against a lane per (row, x mod 4, column segment) walking its own records
// with the tile in LDS (whole frames, read back): 4,096 overlapping triangles
// at 640x480 4,234 -> 381 us, 256 at 128x96 483 -> 185, 1,200 blended ones at
// 801x603 1,621 -> 458; the small triangles of a 1080p frame of 64 spheres
// (8.4 M) 579 -> 549, with four outputs at 1280x720 832 -> 588, 1,000 batched
// meshes 1,160 -> 1,024.
//
// The bound: with A_i = X |bx_i| + Y |by_i| + |bz_i| (X, Y the block's far
// corner) the walk's value is within sum |z_i| A_i 2^-24 (X / 4 + 8) of the
// plane's exact value (the start's three roundings, at most X / 4 + 1 steps,
// the depth sum's products and additions), the plane evaluated from its
// combined coefficients within 11 of the same units (block corners included);
// 2.125 (X / 4 + 13) units are allowed, and non-finite terms decide nothing.
//
// AUX: bit 0 debug buffers, bit 1 visibility, bit 3 several fragment outputs
// (as k_raster), bit 5 some draw of the batch blends.
template <int CF, int AUX>
__global__ __launch_bounds__(256) void k_raster_wave(RasterParams P, int tileShiftX, int tileShiftY, int wavesShift)
{
    constexpr bool DBG = (AUX & 1) != 0;
    constexpr bool VIS = (AUX & 2) != 0;
    constexpr bool MRT = (AUX & 8) != 0;
    constexpr bool BLEND = (AUX & 32) != 0;
    __shared__ uint32_t sIdW[4][64];
    __shared__ uint32_t sMetaW[4][64];
    __shared__ float4 sResW[4][64];

    // a frame whose setup outgrew the bin capacities leaves its targets untouched
    if (P.ctrl != nullptr && P.ctrl->overflow != 0u) return;

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    uint32_t* sId = sIdW[wave];
    uint32_t* sMeta = sMetaW[wave];
    float4* sRes = sResW[wave];

    // wave -> block of a tile; tiles in launch order (heaviest first)
    const int groupShift = tileShiftX + tileShiftY - 6 - wavesShift;    // log2 workgroups per tile
    const int slot = (int)(blockIdx.x >> groupShift);
    const int blk = (int)(((blockIdx.x & ((1u << groupShift) - 1u)) << wavesShift) + (uint32_t)wave);
    const int tile = (P.tileOrder != nullptr) ? (int)P.tileOrder[slot] : slot;
    const int tx = tile % P.tilesX, ty = tile / P.tilesX;
    const int bx0 = (tx << tileShiftX) + ((blk & ((1 << (tileShiftX - 3)) - 1)) << 3);
    const int by0 = (ty << tileShiftY) + ((blk >> (tileShiftX - 3)) << 3);
    if (bx0 >= P.W || by0 >= P.H) return;
    const uint2 range = P.tileRange[tile];
    const int x = bx0 + (lane & 7), y = by0 + (lane >> 3);
    const bool inb = x < P.W && y < P.H;
    const uint64_t gi = (uint64_t)y * P.W + x;

    // the pixel as it is before the batch, or cleared
    float depth = 0.f;
    uint32_t col8 = 0u;
    float4 colF = make_float4(0.f, 0.f, 0.f, 0.f), vis = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t dbgLast = 0u, dbgCount = 0u;
    if (P.clearDepth) depth = P.clearDepthValue;
    else if (inb) depth = load_depth(P, gi);
    if (CF == 1)
    {
        if (P.clearColor) col8 = P.clearRGBA8;
        else if (inb) col8 = load_color8(P, gi);
    }
    if (CF == 2)
    {
        if (P.clearColor) colF = make_float4(P.clearRGBAF[0], P.clearRGBAF[1], P.clearRGBAF[2], P.clearRGBAF[3]);
        else if (inb) colF = load_colorF(P, gi);
    }
    if (!P.clearDepth && inb)
    {
        if (DBG)
        {
            dbgLast = P.dbgLast[gi];
            dbgCount = P.dbgCount[gi];
        }
        if (VIS) vis = P.vis[gi];
    }
    uint32_t pend = kNoPending;                 // pending fragment: its record and barycentric values
    float ps0 = 0.f, ps1 = 0.f, ps2 = 0.f;

    // shades a fragment of this lane's pixel into its colour
    auto shade_into = [&](uint32_t rid, float s0, float s1, float s2, int blendMode) {
        const SetupRec& Q = P.recs[rid];
        const DrawDesc& QD = P.draws[Q.draw];
        const float qhw[3] = {Q.hw[0], Q.hw[1], Q.hw[2]};
        float4 out, wv;
        const bool have = shade<MRT>(P, QD, qhw, Q.bc3, Q.state, rid, s0, s1, s2, out, wv, gi, blendMode);
        if (have) blend_into<CF>(&col8, &colF, blendMode, out, P.colorComps, P.colorPacked);
        if (VIS) vis = make_float4(__uint_as_float(Q.seq), wv.x, wv.y, wv.z);
    };

    float bound = inb ? depth : -INFINITY;      // no smaller than the pixel's depth after the queued fragments
    uint64_t mine = 0;                          // queued fragments of this lane's pixel
    int queued = 0;
    uint32_t tested = 0, shaded = 0;

    // this lane's record of the current 64
    uint64_t mask = 0;
    uint32_t id = 0, state = 0;
    float zx = 0.f, zy = 0.f, zlo = 0.f, zwid = 0.f;
    uint64_t todo = 0;
    uint32_t base = range.x;
    bool more = true;
    while (more)
    {
        for (;;)
        {
            if (todo == 0)
            {
                if (base >= range.y)
                {
                    more = false;
                    break;
                }
                const int nb = (int)min(64u, range.y - base);
                const float top = wave_max_f32(bound);
                mask = 0;
                bool rej = false, raise = false;
                if (lane < nb)
                {
                    id = P.tileRecs[base + lane];
                    const SetupRec& R = P.recs[id];
                    const ScanEdges E = scan_edges(R);
                    state = R.state;
                    const int r0 = max(R.minY - by0, 0), r1 = min(min(R.maxY, P.H) - by0, 8);
                    const int xr = min(P.W - bx0, 8);
                    for (int r = r0; r < r1; ++r)
                    {
                        int32_t xMin, xMax;
                        scanline_step(E, (float)(by0 + r), xMin, xMax);
                        const int a = max(xMin, bx0) - bx0, b = max(min(xMax, bx0 + xr), bx0) - bx0;
                        if ((uint32_t)xMin < (uint32_t)xMax && a < b)
                            mask |= (uint64_t)((1u << b) - (1u << a)) << (8 * r);
                    }
                    if (mask != 0)
                    {
                        tested += (uint32_t)__popcll(mask);
                        const int dt = (int)(state & 7u);
                        const bool less = dt == SL_DEPTH_TEST_LESS_THAN || dt == SL_DEPTH_TEST_LESS_EQUAL;
                        raise = ((state >> 3) & 1u) != 0u && !less && dt != SL_DEPTH_TEST_EQUAL;
                        const float X = (float)(bx0 + 7), Y = (float)(by0 + 7);
                        float zc = R.bc3, mag = 0.f;
                        zx = 0.f;
                        zy = 0.f;
#pragma unroll
                        for (int i = 0; i < 3; ++i)
                        {
                            const float zi = R.z[i], bx = R.bx[i], by = R.by[i], bz = R.bz[i];
                            zx = fmaf(zi, bx, zx);
                            zy = fmaf(zi, by, zy);
                            zc = fmaf(zi, bz, zc);
                            mag = fmaf(fabsf(zi), fmaf(X, fabsf(bx), fmaf(Y, fabsf(by), fabsf(bz))), mag);
                        }
                        const float margin = fmaf(mag * (5.9604645e-8f * 2.125f), fmaf(0.25f, X, 13.f), 1e-37f);
                        zlo = zc - margin;
                        zwid = 2.125f * margin;
                        const float lo = (zlo + fminf(zx * (float)bx0, zx * X)) + fminf(zy * (float)by0, zy * Y);
                        rej = less && lo > top;
                    }
                }
                base += 64u;
                // records from the first one that can raise a depth on stay
                const uint64_t rb = __ballot(raise);
                const uint64_t before = (rb != 0) ? ((rb & (0ull - rb)) - 1ull) : ~0ull;
                todo = __ballot(mask != 0) & ~(__ballot(rej) & before);
                continue;
            }
            const int bi = __ffsll((unsigned long long)todo) - 1;
            const uint32_t st = (uint32_t)__builtin_amdgcn_readlane((int)state, bi);
            const uint64_t m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(mask >> 32), bi) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)mask, bi);
            const int dt = (int)(st & 7u);
            const bool less = dt == SL_DEPTH_TEST_LESS_THAN || dt == SL_DEPTH_TEST_LESS_EQUAL;
            const float zp = fmaf(readlane_f32(zx, bi), (float)x, fmaf(readlane_f32(zy, bi), (float)y, readlane_f32(zlo, bi)));
            const bool cand = ((m >> lane) & 1ull) != 0ull && !(less && zp > bound);
            const uint64_t cm = __ballot(cand);
            if (cm != 0)
            {
                const int n = __popcll(cm);
                if (queued + n > 64) break;
                if (cand)
                {
                    const uint32_t e = (uint32_t)queued + lanes_below(cm);
                    sId[e] = (uint32_t)__builtin_amdgcn_readlane((int)id, bi);
                    sMeta[e] = (uint32_t)lane | (st << 8);
                    mine |= 1ull << e;
                    if (((st >> 3) & 1u) != 0u)
                    {
                        // the depth it can leave; a half depth target rounds it
                        float hi = zp + readlane_f32(zwid, bi);
                        if (P.depthHalf) hi = hi + fmaf(fabsf(hi), 0.0009765625f, 1e-7f);
                        bound = less ? fminf(bound, hi) : (dt == SL_DEPTH_TEST_EQUAL ? bound : INFINITY);
                    }
                }
                queued += n;
            }
            todo &= todo - 1ull;
        }
        if (queued == 0) continue;

        // exact barycentrics and depth of the queued fragments, one per lane
        wave_lds_fence();
        if (lane < queued)
        {
            const SetupRec& R = P.recs[sId[lane]];
            const uint32_t px = sMeta[lane] & 63u;
            const int ex = bx0 + (int)(px & 7u);
            const float yf = (float)(by0 + (int)(px >> 3));
            int32_t xMin, xMax;
            scanline_step(scan_edges(R), yf, xMin, xMax);
            // bc(x) = fl(fl(x*dx) + fma(dy, y, c)) at the span's first pixel of
            // this one's class mod 4, then += 4*dx per group of 4 pixels
            const int g = (ex - xMin) >> 2;
            const float fx = (float)(ex - 4 * g);
            float s0 = (fx * R.bx[0]) + fmaf(R.by[0], yf, R.bz[0]);
            float s1 = (fx * R.bx[1]) + fmaf(R.by[1], yf, R.bz[1]);
            float s2 = (fx * R.bx[2]) + fmaf(R.by[2], yf, R.bz[2]);
            const float d0 = R.bx[0] * 4.f, d1 = R.bx[1] * 4.f, d2 = R.bx[2] * 4.f;
            if (g <= kStepLimit)
            {
                int k = 0;
                for (; k + 4 <= g; k += 4)
                {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        s0 = s0 + d0;
                        s1 = s1 + d1;
                        s2 = s2 + d2;
                    }
                }
                for (; k < g; ++k)
                {
                    s0 = s0 + d0;
                    s1 = s1 + d1;
                    s2 = s2 + d2;
                }
            }
            else
            {
                const float3 a = recur_advance3(make_float3(s0, s1, s2), make_float3(d0, d1, d2), g);
                s0 = a.x;
                s1 = a.y;
                s2 = a.z;
            }
            const float z = (((R.z[0] * s0) + (R.z[1] * s1)) + (R.z[2] * s2)) + R.bc3;
            sRes[lane] = make_float4(z, s0, s1, s2);
        }
        wave_lds_fence();
        // each pixel takes its fragments in record order
        while (mine != 0)
        {
            const int e = __ffsll((unsigned long long)mine) - 1;
            mine &= mine - 1ull;
            const float4 f = sRes[e];
            const uint32_t rid = sId[e], st = sMeta[e] >> 8;
            if (!depth_test((int)(st & 7u), f.x, depth)) continue;
            const int blendMode = (int)((st >> 4) & 7u);
            const bool hasOut = ((st >> 7) & 1u) != 0u;
            // an unblended fragment with outputs, and any whose visibility
            // record is wanted, waits until the pixel's colour is needed
            if ((hasOut && (!BLEND || blendMode == SL_BLEND_OFF)) || (VIS && !hasOut))
            {
                pend = rid;
                ps0 = f.y;
                ps1 = f.z;
                ps2 = f.w;
            }
            else if (BLEND && hasOut)
            {
                // a blended fragment reads the colour: the pending one first
                uint32_t r = (pend != kNoPending) ? pend : rid;
                bool own = pend == kNoPending;
                for (;;)
                {
                    shade_into(r, own ? f.y : ps0, own ? f.z : ps1, own ? f.w : ps2, own ? blendMode : SL_BLEND_OFF);
                    if (own) break;
                    r = rid;
                    own = true;
                }
                pend = kNoPending;
            }
            if (((st >> 3) & 1u) != 0u) depth = P.depthHalf ? __half2float(__float2half_rn(f.x)) : f.x;
            if (DBG)
            {
                dbgLast = P.recs[rid].seq;
                dbgCount += 1u;
            }
            ++shaded;
        }
        queued = 0;
        if (inb) bound = depth;
        wave_lds_fence();
    }

    if (pend != kNoPending) shade_into(pend, ps0, ps1, ps2, SL_BLEND_OFF);
    if (inb)
    {
        store_depth(P, gi, depth);
        if (CF == 1) store_color8(P, gi, col8);
        if (CF == 2) store_colorF(P, gi, colF);
        if (DBG)
        {
            P.dbgLast[gi] = dbgLast;
            P.dbgCount[gi] = dbgCount;
        }
        if (VIS) P.vis[gi] = vis;
    }

    // the block's counts (a lane's stay below 64 per record of its 64th of the list)
    unsigned long long t = tested, sh = shaded;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
    {
        t += __shfl_xor(t, off, 64);
        sh += __shfl_xor(sh, off, 64);
    }
    if (lane == 0 && t != 0)
    {
        FrameCtrl::CounterSlot& cs = P.ctrl->counters[blockIdx.x % kCounterSlots];
        atomicAdd(&cs.tested, t);
        if (sh != 0) atomicAdd(&cs.shaded, sh);
    }
}

}  // namespace

template <int CF, int AUX>
void launch_raster_wave_cfg(const RasterParams& p, int numTiles, int shx, int shy, hipStream_t s)
{
    const int blocksShift = shx + shy - 6, wavesShift = blocksShift < 2 ? blocksShift : 2;
    const auto kernel = k_raster_wave<CF, AUX>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)numTiles << (blocksShift - wavesShift)), dim3(64u << wavesShift),
                       occupancy_lds(kernel, p.wgPerCU), s, p, shx, shy, wavesShift);
}

}  // namespace slg
