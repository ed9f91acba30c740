// sl_raster_wave_dbg.hip -- k_raster_wave instances with the debug buffers (blending compiled in: one instance serves both kinds of batch).
#include "sl_raster_wave.h"

namespace slg {

template void launch_raster_wave_cfg<0, 1>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 33>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 33>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 35>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<1, 41>(const RasterParams&, int, int, int, int, hipStream_t);
template void launch_raster_wave_cfg<2, 41>(const RasterParams&, int, int, int, int, hipStream_t);

}  // namespace slg
