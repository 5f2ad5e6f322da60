// dop_rk4_f32.hip -- one-pass RK4 steps for f32 storage.
#include "dop_rk4_impl.hpp"

namespace dop {

hipError_t launch_pass_f32(const BGroup& g, const BProb* probs, const BItem* items, int parity,
                            int grid, hipStream_t s)
{
    if (g.acc == kAccF32Kahan)
        return batch::launch_pass_group<float, kAccF32Kahan>(g, probs, items, parity, grid, s);
    if (g.acc == kAccF32Wide)
        return batch::launch_pass_group<float, kAccF32Wide>(g, probs, items, parity, grid, s);
    return batch::launch_pass_group<float, kAccF32>(g, probs, items, parity, grid, s);
}

}  // namespace dop
