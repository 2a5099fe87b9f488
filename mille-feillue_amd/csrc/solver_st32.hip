// Resident CG / BiCGSTAB kernels on stencil planes of FP32 values (instantiated
// here so they compile in parallel).
#include "persistent.h"

namespace mf {

KernelChoice pick_stencil_f32(int L, int method, long long rows_per_wg, int G, bool sum64)
{
    return pick_stencil_class<1>(L, method, rows_per_wg, G, sum64);
}

}  // namespace mf
