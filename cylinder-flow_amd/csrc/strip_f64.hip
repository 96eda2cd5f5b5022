// strip_f64.hip -- the large-domain D2Q9 kernel of strip_kernel.hpp for SF64 storage
#include "strip_kernel.hpp"

namespace lbm {

hipError_t strip_launch_f64(const StripLaunch &l, const FusedArgs &a, hipStream_t s) { return strip_launch_s<SF64>(l, a, s); }

}  // namespace lbm
