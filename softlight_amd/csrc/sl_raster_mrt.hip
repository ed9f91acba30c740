// sl_raster_mrt.hip -- k_raster instances: batches with several fragment outputs and wireframe, line or point records.
#include "sl_raster_impl.h"

namespace slg {

template void launch_raster_cfg<1, 8>(const RasterParams&, int, int, hipStream_t);
template void launch_raster_cfg<2, 8>(const RasterParams&, int, int, hipStream_t);
template void launch_raster_cfg<1, 9>(const RasterParams&, int, int, hipStream_t);
template void launch_raster_cfg<2, 9>(const RasterParams&, int, int, hipStream_t);

}  // namespace slg
