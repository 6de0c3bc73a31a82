// Instantiates the conv chain kernels on tiles of whole output rows for one element type.
#include "conv13_tiles.h"

namespace ditto {

hipError_t DITTO_CONVTILES_NAME(const ConvTilesArgs& args, hipStream_t stream) { return launch_conv_tiles<DITTO_INST_T>(args, stream); }
hipError_t DITTO_PACKTILES_NAME(const ConvTilesArgs& args, const void* w1, const void* w2, void* w1f, void* w2f, hipStream_t stream) {
  return launch_pack_conv_tiles<DITTO_INST_T>(args, w1, w2, w1f, w2f, stream);
}
hipError_t DITTO_CONV13TILES_NAME(const Conv13TilesArgs& args, hipStream_t stream) { return launch_conv13_tiles<DITTO_INST_T>(args, stream); }
hipError_t DITTO_PACK13TILES_NAME(const Conv13TilesArgs& args, const void* w1, const void* w2, void* w1f, void* w2f, hipStream_t stream) {
  return launch_pack_conv13_tiles<DITTO_INST_T>(args, w1, w2, w1f, w2f, stream);
}

}  // namespace ditto
