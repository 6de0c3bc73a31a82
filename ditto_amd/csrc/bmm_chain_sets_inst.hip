// Instantiates the chain kernels that take several chains of one shape in a launch (BmmSets) for one element type: softmax, B
// stored [L][K].
#include "bmm_chain_fp4m16.h"
#include "bmm_chain_rows.h"
#include "bmm_chain_split.h"

namespace ditto {

typedef DITTO_INST_T T;

template <int DT>
static hipError_t split(int rt, const BmmSetsArgs& args, hipStream_t stream) {
  return rt == 1 ? launch_bmm_chain_split<T, DT, 1, kInterSoftmax, false>(args, stream)
                 : launch_bmm_chain_split<T, DT, 2, kInterSoftmax, false>(args, stream);
}

template <int DT>
static hipError_t rows(int nw, const BmmSetsArgs& args, hipStream_t stream) {
  if constexpr (DT != 8)
    if (nw == 4) return launch_bmm_chain_rows<T, DT, 4, kInterSoftmax, false>(args, stream);
  return launch_bmm_chain_rows<T, DT, 8, kInterSoftmax, false>(args, stream);
}

hipError_t DITTO_SETS_NAME(BmmSetsKernel kernel, int dt, int q, const BmmSetsArgs& args, hipStream_t stream) {
  switch (kernel) {
    case BmmSetsKernel::split: return dt == 4 ? split<4>(q, args, stream) : dt == 5 ? split<5>(q, args, stream) : split<8>(q, args, stream);
    case BmmSetsKernel::rows: return dt == 4 ? rows<4>(q, args, stream) : dt == 5 ? rows<5>(q, args, stream) : rows<8>(q, args, stream);
    case BmmSetsKernel::rows64:
      return q == 4 ? launch_bmm_chain4m16<T, 64, kInterSoftmax, 1, false>(args, stream)
                    : launch_bmm_chain4m16<T, 64, kInterSoftmax, 2, false>(args, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace ditto
