// The launch that does a decode step in order where the resident one gave up (step_kernel.h).  A file of its own: compiled beside it, the
// resident kernels spill more (two sequences 722 -> 730 us a step).
#include <hip/hip_runtime.h>

#include "step_kernel.h"

namespace terna {

void launch_step_ordered(const StepArgs& a, hipStream_t st)
{
    const dim3 grid(kStepOrderedGroups), threads(kStepThreads);
    if (a.M == 1) terna_decode_step_kernel<1, true><<<grid, threads, 0, st>>>(a);
    else if (a.M == 2) terna_decode_step_kernel<2, true><<<grid, threads, 0, st>>>(a);
    else terna_decode_step_kernel<4, true><<<grid, threads, 0, st>>>(a);
}

}  // namespace terna
