// sl_raster_mrt_direct.hip -- k_raster_wave instances for batches of small triangles with several fragment outputs.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<1, 72>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 72>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 104>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 104>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
