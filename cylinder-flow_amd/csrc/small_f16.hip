// small_f16.hip -- the several-steps-per-launch kernel of small_kernel.hpp for SF16 storage
#include "small_kernel.hpp"

namespace lbm {

hipError_t tb_launch_f16(const TbLaunch &l, const FusedArgs &a, hipStream_t s) { return tb_launch_s<SF16>(l, a, s); }

}  // namespace lbm
