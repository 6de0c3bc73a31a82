// Instantiates the chain kernel of 32 rows per wave for one element type.
#include "bmm_chain_rows.h"

namespace ditto {

template <int DT, int NW>
static hipError_t launch(bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  typedef DITTO_INST_T T;
  if (softmax)
    return b_kl ? launch_bmm_chain_rows<T, DT, NW, kInterSoftmax, true>(args, stream)
                : launch_bmm_chain_rows<T, DT, NW, kInterSoftmax, false>(args, stream);
  return b_kl ? launch_bmm_chain_rows<T, DT, NW, kInterCast, true>(args, stream)
              : launch_bmm_chain_rows<T, DT, NW, kInterCast, false>(args, stream);
}

// dt: column tiles of 16; nw: waves of a workgroup
hipError_t DITTO_ROWS_NAME(int dt, int nw, bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  switch (10 * dt + nw) {
    case 44: return launch<4, 4>(softmax, b_kl, args, stream);
    case 48: return launch<4, 8>(softmax, b_kl, args, stream);
    case 54: return launch<5, 4>(softmax, b_kl, args, stream);
    case 58: return launch<5, 8>(softmax, b_kl, args, stream);
    case 88: return launch<8, 8>(softmax, b_kl, args, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace ditto
