// sl_raster_wave.hip -- k_raster_wave instances: filled triangles (plain, blended, visibility), no debug buffers.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 0>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 0>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 0>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 32>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 32>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 2>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 34>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
