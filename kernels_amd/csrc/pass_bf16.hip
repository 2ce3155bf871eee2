// Pass kernels (several sweeps per pass) with BF16 storage.
#include "sweep_launch.hpp"

namespace prk {
int launch_pass_bf16(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s)
{
    return launch_pass_dtype<BF16>(p, sweeps, any, in, in_next, out, s);
}
}  // namespace prk
