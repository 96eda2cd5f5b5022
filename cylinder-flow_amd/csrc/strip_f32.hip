// strip_f32.hip -- the large-domain D2Q9 kernel of strip_kernel.hpp for SF32 storage
#include "strip_kernel.hpp"

namespace lbm {

hipError_t strip_launch_f32(const StripLaunch &l, const FusedArgs &a, hipStream_t s) { return strip_launch_s<SF32>(l, a, s); }

}  // namespace lbm
