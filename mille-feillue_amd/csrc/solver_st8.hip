// Resident CG / BiCGSTAB kernels on stencil planes of E4M3 values (instantiated
// here so they compile in parallel).
#include "persistent.h"

namespace mf {

KernelChoice pick_stencil_e4m3(int L, int method, long long rows_per_wg, int G, bool sum64)
{
    return pick_stencil_class<3>(L, method, rows_per_wg, G, sum64);
}

}  // namespace mf
