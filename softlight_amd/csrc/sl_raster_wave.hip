// sl_raster_wave.hip -- k_raster_wave instances: filled triangles without debug buffers.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 0>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 0>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 0>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 32>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 32>(const RasterParams&, int, int, int, hipStream_t);
// visibility attachment (RGBA32F colour only)
template void launch_raster_wave_cfg<2, 2>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 34>(const RasterParams&, int, int, int, hipStream_t);
// several fragment outputs
template void launch_raster_wave_cfg<1, 8>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 8>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 40>(const RasterParams&, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 40>(const RasterParams&, int, int, int, hipStream_t);

}  // namespace slg
