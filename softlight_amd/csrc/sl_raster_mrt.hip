// sl_raster_mrt.hip -- k_raster_wave instances: several fragment outputs.
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<1, 8>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 8>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 40>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 40>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 44>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 44>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
