// Fused tile passes, complex64, 32 amplitudes per thread.  This shape computes in
// FP32: 32 complex128 amplitudes per thread do not fit the registers twice.
#include "k_tile_impl.hpp"

namespace dmv {

int launch_tile_c64_wide(int rlog, int tlog, bool nt, bool half, void *state, int n, StateLayout L,
                         const DevPass *passes, const DevPhase *phases, const DevOp *ops, uint32_t pass_idx)
{
    if (tlog != 8 || rlog != 5)
        return kNotHandled;
    return half ? run_tile<float, float, 5, 8, true>(nt, state, n, L, passes, phases, ops, pass_idx)
                : run_tile<float, float, 5, 8, false>(nt, state, n, L, passes, phases, ops, pass_idx);
}

}  // namespace dmv
