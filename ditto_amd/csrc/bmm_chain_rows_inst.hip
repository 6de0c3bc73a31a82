// Instantiates the chain kernel padded to 80 columns for one element type.
#include "bmm_chain_rows.h"

namespace ditto {

template <int NW>
static hipError_t launch(bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  typedef DITTO_INST_T T;
  if (softmax)
    return b_kl ? launch_bmm_chain_rows<T, 5, NW, kInterSoftmax, true>(args, stream)
                : launch_bmm_chain_rows<T, 5, NW, kInterSoftmax, false>(args, stream);
  return b_kl ? launch_bmm_chain_rows<T, 5, NW, kInterCast, true>(args, stream)
              : launch_bmm_chain_rows<T, 5, NW, kInterCast, false>(args, stream);
}

// nw: waves of a workgroup
hipError_t DITTO_ROWS_NAME(int nw, bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  return nw == 4 ? launch<4>(softmax, b_kl, args, stream) : nw == 8 ? launch<8>(softmax, b_kl, args, stream) : hipErrorInvalidValue;
}

}  // namespace ditto
