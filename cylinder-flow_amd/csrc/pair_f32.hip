// pair_f32.hip -- the two-step kernel of pair_kernel.hpp for SF32 storage
#include "pair_kernel.hpp"

namespace lbm {

PairOps pair_ops_f32() { return pair_ops<SF32>(); }

}  // namespace lbm
