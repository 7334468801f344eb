// Pyramid operators with compile-time sizes.
#include "gen_fixed.hpp"

namespace nektar_amd {

hipError_t launch_fixed_pyr(const GenArgs &a) { return gen::launch_fixed_shape<gen::SH_PYR>(a); }

}  // namespace nektar_amd
