// small_f32.hip -- the several-steps-per-launch kernel of small_kernel.hpp for SF32 storage
#include "small_kernel.hpp"

namespace lbm {

hipError_t tb_launch_f32(const TbLaunch &l, const FusedArgs &a, hipStream_t s) { return tb_launch_s<SF32>(l, a, s); }

}  // namespace lbm
