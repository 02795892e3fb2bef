// Small-grid MFMA conv: the bf16 instantiations with 2 row groups a unit.
#include "conv_split_kernel.hpp"

namespace tsp {

int split_launch_bf16_2(TSP_HALO_LAUNCH_ARGS, int ncg) {
    if (ncg == 2)
        return split_launch<true, 2, 2>(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip,
                                       pad, ln, tr);
    return split_launch<true, 2, 1>(odt, planned, feats, n, ci, nbr, plan, weight, bias, co, out, s, osc, skip, pad,
                                   ln, tr);
}

}  // namespace tsp
