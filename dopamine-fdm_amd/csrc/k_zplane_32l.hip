// k_zplane for the longer rows, FP32 form
#include "k_zplane_impl.h"

namespace dfp {
#define DFP_ZP_ONE(a, b, r) DFP_ZP_INSTANTIATE(float2, a, b, r)
DFP_ZP_LONG(DFP_ZP_ONE)
}  // namespace dfp
