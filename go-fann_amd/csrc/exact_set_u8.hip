// exact_set_u8.hip -- the u8 exact-route kernels with the set frontier
// (instantiated here so that the sources build in parallel).
#include "exact_route.hpp"

namespace gofann {

template int launch_exact<0, GOFANN_ELEM_U8, 2>(GOFANN_EXACT_LAUNCH_ARGS);

}  // namespace gofann
