// Pass kernels (several sweeps per pass) with F32 storage.
#include "sweep_launch.hpp"

namespace prk {
int launch_pass_f32(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *out, hipStream_t s)
{
    return launch_pass_dtype<F32>(p, sweeps, any, in, in_next, out, s);
}
}  // namespace prk
