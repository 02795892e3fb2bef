// Small-grid MFMA conv: the bf16 instantiations with 4 row groups a unit.
#include "conv_split_kernel.hpp"

namespace tsp {

int split_launch_bf16_4(TSP_HALO_LAUNCH_ARGS, int) {
    return split_launch<true, 4, 1>(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad,
                                   ln, tr);
}

}  // namespace tsp
