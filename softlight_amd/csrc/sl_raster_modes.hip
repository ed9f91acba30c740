// sl_raster_modes.hip -- k_raster_wave instances: batches with wireframe, line or point records.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 4>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 4>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 4>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 36>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 36>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 6>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
