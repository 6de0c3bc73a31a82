// Instantiates the key-splitting chain kernel whose workgroups own a few of the columns of F, for one element type.
#include "bmm_chain_split.h"

namespace ditto {

template <int DT, int CT>
static hipError_t launch(bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  typedef DITTO_INST_T T;
  if (softmax)
    return b_kl ? launch_bmm_chain_split<T, DT, 1, kInterSoftmax, true, CT>(args, stream)
                : launch_bmm_chain_split<T, DT, 1, kInterSoftmax, false, CT>(args, stream);
  return b_kl ? launch_bmm_chain_split<T, DT, 1, kInterCast, true, CT>(args, stream)
              : launch_bmm_chain_split<T, DT, 1, kInterCast, false, CT>(args, stream);
}

// dt: column tiles of 16 that K and N are padded to; ct: those a workgroup owns
hipError_t DITTO_SPLITCOLS_NAME(int dt, int ct, bool softmax, bool b_kl, const BmmChainArgs& args, hipStream_t stream) {
  switch (10 * dt + ct) {
    case 42: return launch<4, 2>(softmax, b_kl, args, stream);
    case 52: return launch<5, 2>(softmax, b_kl, args, stream);
    case 82: return launch<8, 2>(softmax, b_kl, args, stream);
    case 84: return launch<8, 4>(softmax, b_kl, args, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace ditto
