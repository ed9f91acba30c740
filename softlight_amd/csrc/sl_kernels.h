// sl_kernels.h -- host-side launchers of the kernels in sl_kernels.hip.
#pragma once

#include "sl_device.h"

namespace slg {

hipError_t launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s);
hipError_t launch_vertex(const SetupParams& p, hipStream_t s);
// Clears the control block before a frame, keeping (and adding the last
// frame's overflow / error flags to) FrameCtrl::sticky, and na words of a.
hipError_t launch_frame_reset(FrameCtrl* ctrl, uint32_t* a, uint32_t na, hipStream_t s);
hipError_t launch_setup(const SetupParams& p, uint64_t chunks, hipStream_t s);
hipError_t launch_chunk_scan(const SetupParams& p, hipStream_t s);
// tris / prims: the batch holds triangle draws / point or line draws.
hipError_t launch_emit(const SetupParams& p, bool tris, bool prims, hipStream_t s);
// The clip jobs, and the bin entries of records that cover many tiles.
hipError_t launch_clip(const SetupParams& p, hipStream_t s);
// Binning splits the entries into at most `rows` (kMaxBinBlocks where the
// count matrix has room for them) blocks of `per` entries (a multiple of 64, at
// least kMinBinBlock).
constexpr uint32_t kMaxBinBlocks = 512;
constexpr uint32_t kMinBinBlock = 256;   // (1,024: a frame of 1,000 .. 3,000 entries spent 13 us in a few waves of the scatter, now 5)
// The kernels work out `per` from the device's entry count, so a launch needs
// only an upper bound of the entries (blocks past the count end at once).
__host__ __device__ inline uint32_t bin_per(uint32_t entries, uint32_t rows)
{
    const uint32_t per = (entries / rows + (entries % rows ? 1u : 0u) + 63u) / 64u * 64u;
    return per > kMinBinBlock ? per : kMinBinBlock;
}
// With items non-null the tile scan also writes the raster's work items of
// the heavy-tile split (see RasterItem): tiles of more than splitAbove
// records cut into parts of about partRecs records, at most maxParts parts;
// filled (a batch of filled triangles): the parts alone, split tiles' ranges
// left empty, and tiles with little of the frame not split (kFilledShare).
hipError_t launch_binning(const uint32_t* keys, const uint32_t* vals, FrameCtrl* ctrl, uint32_t cap,
                          uint32_t entries, uint32_t rows, uint32_t* counts, uint32_t* totals, uint2* range, uint32_t* out,
                          uint32_t* order, int numTiles, hipStream_t s, RasterItem* items = nullptr,
                          uint32_t* itemCount = nullptr, uint32_t partRecs = 1,
                          uint32_t splitAbove = 0, uint32_t maxParts = 0, bool filled = false);
// The raster of a batch: units workgroup shares, one per tile or (with
// p.items) the most work items there can be, maxParts of them parts.
hipError_t launch_raster(const RasterParams& p, int units, int maxParts, int cfg, bool debug, hipStream_t s);
// k_raster_wave of one colour format (CF: 0 none, 1 8-bit/packed, 2 float)
// and variant (AUX bits, see there) on tiles of 2^shx x 2^shy pixels; defined
// in sl_raster_wave.h and instantiated in the sl_raster_*.hip units.
template <int CF, int AUX>
void launch_raster_wave_cfg(const RasterParams& p, int units, int maxParts, int shx, int shy, hipStream_t s);

hipError_t launch_blit(const BlitParams& p, int srcType, int dstType, hipStream_t s);

}  // namespace slg
