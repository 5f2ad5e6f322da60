// dop_rk4_f64.hip -- one-pass RK4 steps for f64 storage.
#include "dop_rk4_impl.hpp"

namespace dop {

hipError_t launch_pass_f64(const BGroup& g, const BProb* probs, const BItem* items, int parity,
                            int grid, hipStream_t s)
{
    return batch::launch_pass_group<double, kAccF64>(g, probs, items, parity, grid, s);
}

}  // namespace dop
