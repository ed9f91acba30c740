// sl_raster_modes_dbg.hip -- k_raster_wave instances: batches with wireframe, line or point records and the debug buffers.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 5>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 37>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 37>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 45>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 45>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 39>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
