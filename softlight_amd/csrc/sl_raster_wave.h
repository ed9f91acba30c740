// sl_raster_wave.h -- k_raster_wave, the fragment stage (filled and wireframe
// triangles, lines, points): one wave per 8x8 pixel block, one pixel per lane.
// Included by the sl_raster_*.hip translation units.
//
// Reference routines reproduced: SL_TriRasterizer::render_triangle_simd
// generic branch (SL_TriRasterizer.cpp:806-923), render_wireframe (:155-156),
// SL_LineRasterizer::render_line (SL_LineRasterizer.cpp:27-80),
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

// Inclusive prefix sum over the wave's 64 lanes (every lane active): within
// rows of 16 by shifts, then the last lanes of the rows before.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v)
{
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}

__device__ __forceinline__ uint32_t wave_prefix(uint32_t v)
{
    v = dpp_add<0x111, 0xF>(v);   // row_shr:1
    v = dpp_add<0x112, 0xF>(v);   // row_shr:2
    v = dpp_add<0x114, 0xF>(v);   // row_shr:4
    v = dpp_add<0x118, 0xF>(v);   // row_shr:8
    v = dpp_add<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
}

// LDS traffic of one wave: its operations execute in order, so ordering them
// only needs the compiler kept from moving them.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Depth and position along the line of its texel (vx, vy)
// (SL_LineRasterizer::render_line, SL_LineRasterizer.cpp:27-80).
__device__ __forceinline__ float line_depth(const SetupRec& R, int vx, int vy, float& interp)
{
    const float fx = (float)vx - R.x[0], fy = (float)vy - R.y[0];
    interp = sqrtf((fx * fx) + (fy * fy)) * R.bx[0];   // length(p - p0) * dist
    return R.z[0] + interp * (R.z[1] - R.z[0]);        // mix(z0, z1, interp)
}

// Row y's steps of a line's Bresenham walk, in closed form, into block row r
// of `mask`; with `wraps` (the block holds column 0) also the walk's texel
// (W, y - 1), which is texel 0 of row y, before or after them in walk order.
template <class Run>
__device__ __forceinline__ void line_row(const LineWalk& w, int W, int y, bool wraps, int r, const Run& run, uint64_t& mask,
                                         uint64_t& before, uint64_t& after)
{
    const int dyAbs = w.dErr >> 1;
    int xa = 1, xb = 0;
    if (!w.steep)
    {
        const int n = (y - w.Y1) * w.yErr;
        if (n >= 0 && n <= dyAbs)
        {
            xa = w.X1 + ((n == 0) ? 0 : (w.dx * (2 * n - 1)) / w.dErr + 1);
            xb = w.X1 + ((n == dyAbs) ? w.dx : (w.dx * (2 * n + 1)) / w.dErr);
        }
    }
    else
    {
        const int k = y - w.X1;
        if (k >= 0 && k <= w.dx) xa = xb = w.Y1 + w.yErr * line_minor_steps(w, k);
    }
    mask |= run(xa, xb + 1, r);
    if (wraps && y >= 1)
    {
        const int ka = w.steep ? (y - 1) - w.X1 : W - w.X1;
        if (ka >= 0 && ka <= w.dx)
        {
            const int m = w.Y1 + w.yErr * line_minor_steps(w, ka);
            if (w.steep ? (m == W) : (m == y - 1))
            {
                const int k0 = w.steep ? y - w.X1 : -w.X1;
                const bool first = !(xa <= 0 && 0 <= xb && k0 < ka);
                (first ? before : after) |= 1ull << (8 * r);
            }
        }
    }
}

// A list's 64 records queue their own fragments when they cover at most
// kDirectPixels pixels of the block each, on average, and none of those left
// reaches over more than kDirectColumns columns (whose fragments' exact values
// take many steps: the filter saves those of hidden ones).
constexpr uint32_t kDirectPixels = 8, kDirectColumns = 64;

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
//            Records that cover a few pixels each are not worth a step of
//            the wave: every lane queues its own record's fragments, at the
//            place a prefix sum over the 64 records gives it (raster kernel of
//            64 spheres at 1080p 65 -> 33 us, of 1,000 blended mesh draws 313
//            -> 251, of 16 views of 512x512 122 -> 71, of a frame of lines
//            290 -> 173).
//   flush    when 64 fragments wait: one fragment per lane, the exact
//            barycentrics (the reference's recurrence, stepped from the
//            span's first pixel) and depth, and a blended fragment's colour;
//            then each pixel takes its own fragments in record order: depth
//            test, counters, pending fragment or blend.  (Shading a blended
//            fragment when its turn came ran the programs for a lane or two
//            at a time: 330 -> 313 us of a 1,000-sphere blended scene's raster.
//            Those that fail their test are shaded for nothing: few where the
//            filter sees them first, all where hidden records queue their own,
//            16 hidden layers of 4-pixel triangles at 1080p 441 -> 480 us.)
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
// Wireframe triangles, lines and points go through the same three stages with
// masks and depths of their own: a wireframe row's second run can visit a
// pixel again and a line's texel (W, y - 1) is texel 0 of row y, before or
// after the row's own, so such a record has up to three masks, queued in the
// order the walk visits them.
//
// Heavy tiles (RasterParams::items): a workgroup takes a work item, a whole
// tile or one part of a split tile's record list (in batches of filled triangles
// alone the parts only: a launch of their own instance takes the whole tiles).  MODE 1 walks a part from +inf (-inf) and leaves the depth it
// ends with, the part's own result m; a MODE 0 part starts from
// fold(initial depth, m of the earlier parts) -- exactly the depth the
// sequential walk has there -- so it counts the fragments that pass exactly
// and ends with its last passing fragment pending; it leaves those per pixel
// and raises the pixel's entry in partWin to itself.  A last launch (merge)
// takes for every pixel the depth after all parts and the pending fragment of
// the last part that left one.  (The merge used to be done by the part that
// finished last, which searched up to 1,024 parts' results per pixel: the
// lines of a frame of 16 spheres, 1280x720, took 1,228 us in the two passes,
// now 290; the frame 1,363 -> 603.)
//
// AUX: bit 0 debug buffers, bit 1 visibility, bit 2 wireframe, line or point
// records in the batch, bit 3 several fragment outputs, bit 5 some draw of
// the batch blends, bit 6 (and bit 2) small records queue their own fragments.
template <int CF, int AUX, int MODE>
__global__ __launch_bounds__(256) void k_raster_wave(RasterParams P, int tileShiftX, int tileShiftY, int wavesShift, int merge)
{
    constexpr bool DBG = (AUX & 1) != 0;
    constexpr bool VIS = (AUX & 2) != 0;
    constexpr bool EXTRA = (AUX & 4) != 0;
    constexpr bool MRT = (AUX & 8) != 0;
    constexpr bool BLEND = (AUX & 32) != 0;
    constexpr bool DIRECT = (AUX & (64 | 4)) != 0;
    __shared__ uint32_t sIdW[4][64];
    __shared__ uint32_t sMetaW[4][64];
    __shared__ float4 sResW[4][64];
    __shared__ unsigned long long sMaskW[DIRECT ? 4 : 1][DIRECT ? 64 : 1];
    // blended fragments shaded one per lane in the flush; the outputs of a
    // several-output program go to their attachments, so those wait their turn
    constexpr bool EARLY = BLEND && !MRT && MODE == 0;
    __shared__ float4 sColW[EARLY ? 4 : 1][EARLY ? 64 : 1];
    __shared__ float4 sVisW[EARLY && VIS ? 4 : 1][EARLY && VIS ? 64 : 1];

    // a frame whose setup outgrew the bin capacities (or went wrong) leaves its
    // targets untouched: the host reads the flags after the whole frame
    if (P.ctrl != nullptr && (P.ctrl->overflow | P.ctrl->error) != 0u) return;

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    uint32_t* sId = sIdW[wave];
    uint32_t* sMeta = sMetaW[wave];
    float4* sRes = sResW[wave];
    unsigned long long* sMask = sMaskW[DIRECT ? wave : 0];
    float4* sCol = sColW[EARLY ? wave : 0];
    float4* sVis = sVisW[EARLY && VIS ? wave : 0];

    // wave -> block of a tile; tiles in launch order (heaviest first), or work items
    const int groupShift = tileShiftX + tileShiftY - 6 - wavesShift;    // log2 workgroups per tile
    const int slot = (int)(blockIdx.x >> groupShift);
    RasterItem item{};
    bool part = false;
    if (EXTRA && P.items != nullptr)
    {
        if ((uint32_t)slot >= P.itemCount[(MODE == 1 || merge) ? 1 : 0]) return;
        item = P.items[slot];
        if (item.parts == 0u || (merge && item.part != 0u)) return;    // a split tile's entry in launch order: its parts do the work
        part = item.parts > 1u && !merge;
    }
    else if (MODE == 1) return;
    const int blk = (int)(((blockIdx.x & ((1u << groupShift) - 1u)) << wavesShift) + (uint32_t)wave);
    const int tile = (EXTRA && P.items != nullptr) ? (int)item.tile : (P.tileOrder != nullptr) ? (int)P.tileOrder[slot] : slot;
    const int tx = tile % P.tilesX, ty = tile / P.tilesX;
    const int bx0 = (tx << tileShiftX) + ((blk & ((1 << (tileShiftX - 3)) - 1)) << 3);
    const int by0 = (ty << tileShiftY) + ((blk >> (tileShiftX - 3)) << 3);
    if (bx0 >= P.W || by0 >= P.H) return;
    uint2 range;
    if (EXTRA && P.items != nullptr) range = merge ? make_uint2(0u, 0u) : make_uint2(item.begin, item.end);
    else range = P.tileRange[tile];
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
    // a split tile's pixel in the part slots: slot s's entry at s * tilePix + tp
    const uint64_t tilePix = 1ull << (tileShiftX + tileShiftY);
    const uint64_t tp = (uint64_t)((y & ((1 << tileShiftY) - 1)) << tileShiftX) + (uint64_t)(x & ((1 << tileShiftX) - 1));
    if (MODE == 1) depth = (P.splitClass == kSplitMax) ? -INFINITY : INFINITY;
    if (EXTRA && MODE == 0 && (part || merge) && inb)
    {
        // the fold pass left fold(initial, m_0 .. m_j) in part j's slot
        const uint32_t upTo = merge ? item.parts : item.part;
        if (P.splitClass != kSplitConst && upTo > 0u) depth = P.partDepth[(uint64_t)(item.slot - item.part + upTo - 1u) * tilePix + tp];
        if (part && DBG) dbgLast = dbgCount = 0u;       // the merge adds the parts' counts
        if (merge)
        {
            const uint32_t win = P.partWin[(uint64_t)item.split * tilePix + tp];
            if (win != 0u)
            {
                const PartPixel q = P.partRes[(uint64_t)(item.slot + win - 1u) * tilePix + tp];
                pend = q.rid;
                ps0 = q.s0;
                ps1 = q.s1;
                ps2 = q.s2;
            }
            if (DBG)
            {
                for (uint32_t j = 0; j < item.parts; ++j)
                {
                    const PartPixel q = P.partRes[(uint64_t)(item.slot + j) * tilePix + tp];
                    if (q.count == 0u) continue;
                    dbgCount += q.count;
                    dbgLast = q.seq;
                }
            }
        }
    }

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
    uint64_t own = 0;                           // queued fragments of this lane's pixel (those the wave queued)
    int queued = 0;
    uint32_t tested = 0, shaded = 0;

    // this lane's record of the current 64
    uint64_t mask = 0, maskBefore = 0, maskAfter = 0;
    uint32_t id = 0, state = 0;
    float zx = 0.f, zy = 0.f, zlo = 0.f, zwid = 0.f;
    uint64_t todo = 0;
    uint32_t masks = 0;                         // masks left of the record at hand (EXTRA)
    bool viaLds = false;                        // some queued fragments were queued by their records
    bool direct = false;                        // the records at hand queue their own fragments
    uint32_t num = 0, upTo = 0, taken = 0;      // a record's fragments, theirs up to it, and those taken
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
                mask = maskBefore = maskAfter = 0;
                bool rej = false, raise = false, wide = false;
                if (lane < nb)
                {
                    id = P.tileRecs[base + lane];
                    const SetupRec& R = P.recs[id];
                    state = R.state;
                    const ScanEdges E = scan_edges(R);
                    const int r0 = max(R.minY - by0, 0), r1 = min(min(R.maxY, P.H) - by0, 8);
                    const int xr = min(P.W - bx0, 8);
                    // columns [from, to) of block row r
                    auto run = [&](int from, int to, int r) -> uint64_t {
                        const int a = max(from, bx0) - bx0, b = max(min(to, bx0 + xr), bx0) - bx0;
                        return a < b ? (uint64_t)((1u << b) - (1u << a)) << (8 * r) : 0ull;
                    };
                    const bool line = EXTRA && (state & kStateLine) != 0u, point = EXTRA && (state & kStatePoint) != 0u;
                    const bool wire = EXTRA && (state & kStateWire) != 0u;
                    if (!line && !point)
                    {
                        for (int r = r0; r < r1; ++r)
                        {
                            int32_t xMin, xMax;
                            scanline_step(E, (float)(by0 + r), xMin, xMax);
                            if ((uint32_t)xMin >= (uint32_t)xMax) continue;
                            if (!wire)
                            {
                                mask |= run(xMin, xMax, r);
                                continue;
                            }
                            // the run from the left end over the distance the left
                            // end moved since the row above, then the run up to the
                            // right end over the distance it moved; the second can
                            // start inside the first
                            int32_t xMin1, xMax1;
                            scanline_step(E, (float)(by0 + r) - 1.f, xMin1, xMax1);
                            const int32_t g0 = wire_gap(xMin, xMin1), g1 = wire_gap(xMax, xMax1);
                            const int64_t firstEnd = (int64_t)xMin + g0;
                            mask |= run(xMin, (firstEnd < (int64_t)xMax) ? (int)firstEnd : xMax, r);
                            if (firstEnd < (int64_t)xMax)
                            {
                                const int32_t t = (int32_t)((uint32_t)xMax - (uint32_t)g1 - 1u);
                                maskAfter |= run(max(xMin, t) + 1, xMax, r);
                            }
                        }
                    }
                    else if (point)
                    {
                        const int px = (int)R.x[0], py = (int)R.y[0];
                        if (py >= by0 + r0 && py < by0 + r1) mask = run(px, px + 1, py - by0);
                    }
                    else
                    {
                        const LineWalk w = line_walk_of(R);
                        const bool wraps = bx0 == 0 && (R.xbox & 0xFFFFu) == 0u;
                        for (int r = r0; r < r1; ++r) line_row(w, P.W, by0 + r, wraps, r, run, mask, maskBefore, maskAfter);
                    }
                    const uint32_t covers = (uint32_t)(__popcll(mask) + __popcll(maskBefore) + __popcll(maskAfter));
                    if (covers != 0u)
                    {
                        tested += covers;
                        const int dt = (int)(state & 7u);
                        const bool less = dt == SL_DEPTH_TEST_LESS_THAN || dt == SL_DEPTH_TEST_LESS_EQUAL;
                        raise = ((state >> 3) & 1u) != 0u && !less && dt != SL_DEPTH_TEST_EQUAL;
                        wide = (R.xbox >> 16) - (R.xbox & 0xFFFFu) > kDirectColumns;
                        const float X = (float)(bx0 + 7), Y = (float)(by0 + 7);
                        zx = 0.f;
                        zy = 0.f;
                        if (!line && !point)
                        {
                            float zc = R.bc3, mag = 0.f;
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
                        }
                        else if (covers == 1u)
                        {
                            // one texel (a point, a distant line): its depth itself
                            const uint64_t m = mask | maskBefore | maskAfter;
                            const int px = __ffsll((unsigned long long)m) - 1;
                            float interp;
                            zlo = point ? R.z[0] : line_depth(R, mask != 0 ? bx0 + (px & 7) : P.W, by0 + (px >> 3) - (mask != 0 ? 0 : 1), interp);
                            zwid = 0.f;
                            // a line of no length: NaN passes no ordered test
                            rej = zlo != zlo && dt != SL_DEPTH_TEST_OFF && dt != SL_DEPTH_TEST_NOT_EQUAL;
                        }
                        else
                        {
                            // depths between the first end's and the one at the
                            // greatest position a texel of the block can have
                            const float z0 = R.z[0], dz = R.z[1] - z0;
                            const float fx = fmaxf(fmaxf(fabsf((float)bx0 - R.x[0]), fabsf(X - R.x[0])), bx0 == 0 ? fabsf((float)P.W - R.x[0]) : 0.f);
                            const float fy = fmaxf(fabsf((float)(by0 - 1) - R.y[0]), fabsf(Y - R.y[0]));
                            const float far = sqrtf((fx * fx) + (fy * fy)) * fabsf(R.bx[0]) * 1.000001f;
                            const float margin = fmaf(1e-6f, fabsf(z0) + far * fabsf(dz), 1e-37f);
                            zlo = fminf(z0, z0 + far * dz) - margin;
                            zwid = far * fabsf(dz) + 2.125f * margin;
                            if (zlo != zlo || z0 + far * dz != z0 + far * dz) zlo = -INFINITY, zwid = INFINITY;
                        }
                        const float lo = (zlo + fminf(zx * (float)bx0, zx * X)) + fminf(zy * (float)by0, zy * Y);
                        rej = rej || (less && lo > top);
                        if (MODE == 1) tested = 0;
                    }
                }
                base += 64u;
                // records from the first one that can raise a depth on stay
                const uint64_t rb = __ballot(raise);
                const uint64_t before = (rb != 0) ? ((rb & (0ull - rb)) - 1ull) : ~0ull;
                todo = __ballot((mask | maskBefore | maskAfter) != 0) & ~(__ballot(rej) & before);
                direct = false;
                // records of a few pixels each queue their fragments themselves
                if (DIRECT && todo != 0 && ((rb | __ballot(wide)) & todo) == 0)
                {
                    num = (((todo >> lane) & 1ull) != 0ull) ? (uint32_t)(__popcll(mask) + __popcll(maskBefore) + __popcll(maskAfter)) : 0u;
                    upTo = wave_prefix(num);
                    taken = 0;
                    direct = (uint32_t)__builtin_amdgcn_readlane((int)upTo, 63) <= kDirectPixels * (uint32_t)__popcll(todo) &&
                             (!EXTRA || __ballot(num > 64u) == 0);
                }
                continue;
            }
            if (DIRECT && direct)
            {
                // as many of the records, in order, as the queue has room for
                const uint64_t fit = __ballot(num != 0u && upTo - taken <= 64u - (uint32_t)queued) & todo;
                if (fit == 0) break;
                if (((fit >> lane) & 1ull) != 0ull)
                {
                    uint32_t e = (uint32_t)queued + upTo - num - taken;
                    for (int q = EXTRA ? 0 : 1; q < (EXTRA ? 3 : 2); ++q)
                    {
                        for (uint64_t m = q == 0 ? maskBefore : (q == 1 ? mask : maskAfter); m != 0; m &= m - 1ull, ++e)
                        {
                            sId[e] = id;
                            sMeta[e] = (uint32_t)(__ffsll((unsigned long long)m) - 1) | (q != 1 ? 64u : 0u) | (state << 8);
                        }
                    }
                }
                const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)upTo, 63 - __clzll((long long)fit));
                queued += (int)(last - taken);
                taken = last;
                viaLds = true;
                todo &= ~fit;
                if (todo != 0) break;
                continue;
            }
            const int bi = __ffsll((unsigned long long)todo) - 1;
            // the record's masks in walk order
            if (EXTRA && masks == 0u)
                masks = (uint32_t)__builtin_amdgcn_readlane((maskBefore != 0 ? 1 : 0) | (mask != 0 ? 2 : 0) | (maskAfter != 0 ? 4 : 0), bi);
            const uint64_t mcur = !EXTRA || (masks & 3u) == 2u ? mask : ((masks & 1u) != 0u ? maskBefore : maskAfter);
            const uint32_t st = (uint32_t)__builtin_amdgcn_readlane((int)state, bi);
            const uint64_t m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(mcur >> 32), bi) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)mcur, bi);
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
                    // (a line's other masks hold its wrapped texels)
                    own |= 1ull << e;
                    sMeta[e] = (uint32_t)lane | (EXTRA && (masks & 3u) != 2u ? 64u : 0u) | (st << 8);
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
            if (EXTRA && (masks &= masks - 1u) != 0u) continue;
            todo &= todo - 1ull;
        }
        if (queued == 0) continue;

        // exact barycentrics and depth of the queued fragments, one per lane,
        // and each pixel's fragments as a mask
        if (DIRECT && viaLds) sMask[lane] = 0ull;
        wave_lds_fence();
        if (lane < queued)
        {
            const SetupRec& R = P.recs[sId[lane]];
            const uint32_t px = sMeta[lane] & 63u;
            const int ex = bx0 + (int)(px & 7u);
            const float yf = (float)(by0 + (int)(px >> 3));
            const uint32_t kind = EXTRA ? (sMeta[lane] >> 8) & (kStateWire | kStateLine | kStatePoint) : 0u;
            float z, s0 = 0.f, s1 = 0.f, s2 = 0.f;
            if (EXTRA && kind == kStatePoint)
            {
                z = R.z[0];
            }
            else if (EXTRA && kind == kStateLine)
            {
                const bool wrapped = (sMeta[lane] & 64u) != 0u;
                z = line_depth(R, wrapped ? P.W : ex, by0 + (int)(px >> 3) - (wrapped ? 1 : 0), s0);
            }
            else if (EXTRA && kind == kStateWire)
            {
                const float fx = (float)ex;
                s0 = fmaf(R.bx[0], fx, fmaf(R.by[0], yf, R.bz[0]));
                s1 = fmaf(R.bx[1], fx, fmaf(R.by[1], yf, R.bz[1]));
                s2 = fmaf(R.bx[2], fx, fmaf(R.by[2], yf, R.bz[2]));
                z = (((R.z[0] * s0) + (R.z[1] * s1)) + (R.z[2] * s2)) + R.bc3;
            }
            else
            {
                int32_t xMin, xMax;
                scanline_step(scan_edges(R), yf, xMin, xMax);
                // bc(x) = fl(fl(x*dx) + fma(dy, y, c)) at the span's first pixel of
                // this one's class mod 4, then += 4*dx per group of 4 pixels, all
                // of them stepped: the exact jump over whole binades
                // (sl_recurrence.h) costs a fragment as much as thousands of
                // steps (eight layers of two triangles each, back to front,
                // 2.1 M pixels a target, raster kernel with jumps above 256
                // steps and without: 1,920 columns 1,992 -> 308 us, 8,192
                // 13,016 -> 956, 65,535 106,704 -> 6,697)
                const int g = (ex - xMin) >> 2;
                const float fx = (float)(ex - 4 * g);
                s0 = (fx * R.bx[0]) + fmaf(R.by[0], yf, R.bz[0]);
                s1 = (fx * R.bx[1]) + fmaf(R.by[1], yf, R.bz[1]);
                s2 = (fx * R.bx[2]) + fmaf(R.by[2], yf, R.bz[2]);
                const float d0 = R.bx[0] * 4.f, d1 = R.bx[1] * 4.f, d2 = R.bx[2] * 4.f;
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
                z = (((R.z[0] * s0) + (R.z[1] * s1)) + (R.z[2] * s2)) + R.bc3;
            }
            sRes[lane] = make_float4(z, s0, s1, s2);
            if (DIRECT && viaLds) atomicOr(&sMask[px], 1ull << lane);
            const uint32_t st = sMeta[lane] >> 8;
            if (EARLY && ((st >> 7) & 1u) != 0u && ((st >> 4) & 7u) != SL_BLEND_OFF)
            {
                // a blended fragment's colour, before its depth test
                const DrawDesc& D = P.draws[R.draw];
                const float hw[3] = {R.hw[0], R.hw[1], R.hw[2]};
                float4 out, wv;
                (void)shade<false>(P, D, hw, R.bc3, R.state, sId[lane], s0, s1, s2, out, wv, 0, SL_BLEND_OFF);
                sCol[lane] = out;
                if (VIS) sVis[lane] = make_float4(__uint_as_float(R.seq), wv.x, wv.y, wv.z);
            }
        }
        wave_lds_fence();
        // each pixel takes its fragments in record order
        uint64_t mine = own;
        if (DIRECT && viaLds) mine |= sMask[lane];
        own = 0;
        viaLds = false;
        for (;;)
        {
            bool stall = false;
            while (mine != 0 && !stall)
            {
                const int e = __ffsll((unsigned long long)mine) - 1;
                const float4 f = sRes[e];
                const uint32_t rid = sId[e], st = sMeta[e] >> 8;
                if (!depth_test((int)(st & 7u), f.x, depth))
                {
                    mine &= mine - 1ull;
                    continue;
                }
                const int blendMode = (int)((st >> 4) & 7u);
                const bool hasOut = ((st >> 7) & 1u) != 0u;
                if (MODE == 1)
                {
                }
                else if ((hasOut && (!BLEND || blendMode == SL_BLEND_OFF)) || (VIS && !hasOut))
                {
                    // an unblended fragment with outputs, and any whose visibility
                    // record is wanted, waits until the pixel's colour is needed
                    pend = rid;
                    ps0 = f.y;
                    ps1 = f.z;
                    ps2 = f.w;
                }
                else if (BLEND && hasOut)
                {
                    // a blended fragment reads the colour: the pending one first,
                    // those of all pixels together
                    stall = pend != kNoPending;
                    if (stall) continue;
                    if (EARLY)
                    {
                        blend_into<CF>(&col8, &colF, blendMode, sCol[e], P.colorComps, P.colorPacked);
                        if (VIS) vis = sVis[e];
                    }
                    else
                    {
                        shade_into(rid, f.y, f.z, f.w, blendMode);
                    }
                }
                mine &= mine - 1ull;
                if (((st >> 3) & 1u) != 0u) depth = P.depthHalf ? __half2float(__float2half_rn(f.x)) : f.x;
                if (DBG)
                {
                    dbgLast = P.recs[rid].seq;
                    dbgCount += 1u;
                }
                ++shaded;
            }
            if (!BLEND || __ballot(stall) == 0) break;
            if (stall)
            {
                shade_into(pend, ps0, ps1, ps2, SL_BLEND_OFF);
                pend = kNoPending;
            }
        }
        queued = 0;
        if (inb) bound = depth;
        wave_lds_fence();
    }

    if (MODE == 1)
    {
        if (inb) P.partDepth[(uint64_t)item.slot * tilePix + tp] = depth;
        return;
    }
    if (EXTRA && part)
    {
        if (inb)
        {
            // the part's last passing fragment (and, with the debug buffers, its counts)
            if (pend != kNoPending || DBG) P.partRes[(uint64_t)item.slot * tilePix + tp] = PartPixel{pend, ps0, ps1, ps2, dbgCount, dbgLast};
            if (pend != kNoPending) atomicMax(&P.partWin[(uint64_t)item.split * tilePix + tp], item.part + 1u);
        }
    }
    else
    {
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
    }

    // the block's counts (a lane's 32 bits hold three masks of 64 for each
    // record of its 64th of the list)
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

// Between the passes over split tiles' parts: for every pixel of a split tile
// part j's slot gets fold(initial depth, m_0 .. m_j), the depth the sequential
// walk has after part j, and the pixel's entry in partWin is cleared.  One
// workgroup per split tile (the work item of its part 0).
static __global__ __launch_bounds__(256) void k_split_fold(RasterParams P, int tileShiftX, int tileShiftY)
{
    if (P.ctrl != nullptr && (P.ctrl->overflow | P.ctrl->error) != 0u) return;
    if (blockIdx.x >= P.itemCount[1]) return;
    const RasterItem item = P.items[blockIdx.x];
    if (item.part != 0u) return;
    const int tilePix = 1 << (tileShiftX + tileShiftY);
    const int tx = (int)item.tile % P.tilesX, ty = (int)item.tile / P.tilesX;
    for (int k = threadIdx.x; k < tilePix; k += 256)
    {
        P.partWin[(uint64_t)item.split * tilePix + k] = 0u;
        if (P.splitClass == kSplitConst) continue;
        const int gx = (tx << tileShiftX) + (k & ((1 << tileShiftX) - 1)), gy = (ty << tileShiftY) + (k >> tileShiftX);
        if (gx >= P.W || gy >= P.H) continue;
        float d = P.clearDepth ? P.clearDepthValue : load_depth(P, (uint64_t)gy * P.W + gx);
        float* m = P.partDepth + (uint64_t)item.slot * tilePix + k;
        for (uint32_t j = 0; j < item.parts; ++j)
        {
            const float mj = m[(uint64_t)j * tilePix];
            if (depth_test(P.splitDtest, mj, d)) d = mj;
            m[(uint64_t)j * tilePix] = d;
        }
    }
}

template <int CF, int AUX, int MODE>
static void launch_wave(const RasterParams& p, int units, int shx, int shy, int merge, hipStream_t s)
{
    const int blocksShift = shx + shy - 6, wavesShift = blocksShift < 2 ? blocksShift : 2;
    const auto kernel = k_raster_wave<CF, AUX, MODE>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)units << (blocksShift - wavesShift)), dim3(64u << wavesShift),
                       occupancy_lds(kernel, p.wgPerCU), s, p, shx, shy, wavesShift, merge);
}

// units: tiles, or (items) the most work items there can be; maxParts: the
// most parts of split tiles among them.
template <int CF, int AUX>
void launch_raster_wave_cfg(const RasterParams& p, int units, int maxParts, int shx, int shy, hipStream_t s)
{
    if constexpr ((AUX & 4) != 0)
    {
        if (p.items != nullptr)
        {
            if (p.splitClass != kSplitConst) launch_wave<0, 4, 1>(p, maxParts, shx, shy, 0, s);
            hipLaunchKernelGGL(k_split_fold, dim3((unsigned)maxParts), dim3(256), 0, s, p, shx, shy);
            launch_wave<CF, AUX, 0>(p, units, shx, shy, 0, s);
            launch_wave<CF, AUX, 0>(p, maxParts, shx, shy, 1, s);
            return;
        }
    }
    launch_wave<CF, AUX, 0>(p, units, shx, shy, 0, s);
}

}  // namespace slg
