// k_zplane for the rows up to 32 modes, FP64
#include "k_zplane_impl.h"

namespace dfp {
#define DFP_ZP_ONE(a, b, r) DFP_ZP_INSTANTIATE(double2, a, b, r)
DFP_ZP_SHORT(DFP_ZP_ONE)
}  // namespace dfp
