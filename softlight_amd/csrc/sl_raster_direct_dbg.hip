// sl_raster_direct_dbg.hip -- k_raster_wave instances for batches of small triangles, with the debug buffers.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 65>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 97>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 97>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 99>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 105>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 105>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
