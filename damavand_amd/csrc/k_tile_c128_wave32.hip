// Fused tile passes, complex128, the one-wave shape of 32 amplitudes per thread.
#include "k_tile_impl.hpp"

namespace dmv {

int launch_tile_c128_wave32(int rlog, int tlog, bool nt, void *state, int n, StateLayout L, const DevPass *passes,
                            const DevPhase *phases, const DevOp *ops, uint32_t pass_idx)
{
    if (tlog == 6 && rlog == 5) return run_tile<double, double, 5, 6, false>(nt, state, n, L, passes, phases, ops, pass_idx);
    return kNotHandled;
}

}  // namespace dmv
