// exact_set_f16.hip -- the f16 exact-route kernels with the set frontier
// (instantiated here so that the sources build in parallel).
#include "exact_route.hpp"

namespace gofann {

GOFANN_EXACT_SET_LAUNCHES(, GOFANN_ELEM_F16)
GOFANN_EXACT_SET_LONG_LAUNCHES(, GOFANN_ELEM_F16)

}  // namespace gofann
