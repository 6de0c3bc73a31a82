// Instantiates the key-splitting chain kernel for one element type.
#include "bmm_chain_split.h"

namespace ditto {

template <int DT, int RT>
static hipError_t launch(bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  typedef DITTO_INST_T T;
  if (softmax)
    return b_kl ? launch_bmm_chain_split<T, DT, RT, kInterSoftmax, true>(args, stream)
                : launch_bmm_chain_split<T, DT, RT, kInterSoftmax, false>(args, stream);
  return b_kl ? launch_bmm_chain_split<T, DT, RT, kInterCast, true>(args, stream)
              : launch_bmm_chain_split<T, DT, RT, kInterCast, false>(args, stream);
}

// dt: column tiles of 16 (4, 5, 8); rt: row tiles of a workgroup (1, 2)
hipError_t DITTO_SPLIT_NAME(int dt, int rt, bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  switch (10 * dt + rt) {
    case 41: return launch<4, 1>(softmax, b_kl, args, stream);
    case 42: return launch<4, 2>(softmax, b_kl, args, stream);
    case 51: return launch<5, 1>(softmax, b_kl, args, stream);
    case 52: return launch<5, 2>(softmax, b_kl, args, stream);
    case 81: return launch<8, 1>(softmax, b_kl, args, stream);
    case 82: return launch<8, 2>(softmax, b_kl, args, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace ditto
