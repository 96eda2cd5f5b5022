// pair_bf16.hip -- the two-step kernel of pair_kernel.hpp for SBF16 storage
#include "pair_kernel.hpp"

namespace lbm {

PairOps pair_ops_bf16() { return pair_ops<SBF16>(); }

}  // namespace lbm
