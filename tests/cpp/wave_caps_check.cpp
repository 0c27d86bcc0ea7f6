// wave_check.cpp over the plans that the library launches (plan_wave_gather): its
// caps of a chunk's words (1,600 and 2,400 at P1) and its stages as launched.
#include "../../polyfem_amd/csrc/plans.hpp"

namespace pfgpu {
inline bool library_plan(const Pattern &pat, int n_local, const int32_t *elem_nodes, int rounds, int, int value_size, WavePlanHost &out)
{
    return plan_wave_gather(pat, n_local == 4 ? 1 : 2, rounds == 2 ? 1 : 4, elem_nodes, value_size, out);
}
} // namespace pfgpu

#define make_wave_plan library_plan
#include "wave_check.cpp"
