// exact_set_f32.hip -- the f32 exact-route kernels with the set frontier
// (instantiated here so that the sources build in parallel).
#include "exact_route.hpp"

namespace gofann {

GOFANN_EXACT_SET_LAUNCHES(, GOFANN_ELEM_F32)
GOFANN_EXACT_SET_LONG_LAUNCHES(, GOFANN_ELEM_F32)

}  // namespace gofann
