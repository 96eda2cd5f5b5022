// pair_f64.hip -- the two-step kernel of pair_kernel.hpp for SF64 storage
#include "pair_kernel.hpp"

namespace lbm {

PairOps pair_ops_f64() { return pair_ops<SF64>(); }

}  // namespace lbm
