// Instantiates the depthwise chain kernels on tiles of whole output rows for one element type.
#include "dw_tiles.h"

namespace ditto {

hipError_t DITTO_DWTILES_NAME(int mult, const DwTilesArgs& args, hipStream_t stream) {
  return launch_dw_tiles<DITTO_INST_T>(mult, args, stream);
}

}  // namespace ditto
