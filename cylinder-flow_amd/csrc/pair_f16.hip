// pair_f16.hip -- the two-step kernel of pair_kernel.hpp for SF16 storage
#include "pair_kernel.hpp"

namespace lbm {

PairOps pair_ops_f16() { return pair_ops<SF16>(); }

}  // namespace lbm
