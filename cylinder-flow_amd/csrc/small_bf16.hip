// small_bf16.hip -- the several-steps-per-launch kernel of small_kernel.hpp for SBF16 storage
#include "small_kernel.hpp"

namespace lbm {

hipError_t tb_launch_bf16(const TbLaunch &l, const FusedArgs &a, hipStream_t s) { return tb_launch_s<SBF16>(l, a, s); }

}  // namespace lbm
