// sl_raster_direct.hip -- k_raster_wave instances for batches of small triangles (records queue their own fragments).
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 64>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 64>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 64>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 96>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 96>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 66>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 98>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
