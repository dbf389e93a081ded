// exact_set_u8.hip -- the u8 exact-route kernels with the set frontier
// (instantiated here so that the sources build in parallel).
#include "exact_route.hpp"

namespace gofann {

GOFANN_EXACT_SET_LAUNCHES(, GOFANN_ELEM_U8)

}  // namespace gofann
