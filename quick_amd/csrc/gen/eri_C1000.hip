// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "C1000.h"

namespace qf {

// Direct-atomic launch; FP64 only.  The FP32 instantiation of the direct
// kernel is not built (it gave wrong Fock matrices on gfx950, cause not
// found): a request for it is refused with a nonzero return.
// os: 1 = the fused open-shell pass (second exchange density)
int launch_fock_C1000(const Task* t, int nt, const PairBlock* b, const MolDesc* m, int fp32, int os, int grid, LaunchTo& q)
{
    if (fp32) return 1;
    if (nt <= 0) return 0;
    if (grid <= 0 || grid > nt) grid = nt;
    if (os)
        q((fock_kernel<C1000, double, true>), dim3(grid), dim3(WAVE), 0, t, nt, b, m);
    else
        q((fock_kernel<C1000, double>), dim3(grid), dim3(WAVE), 0, t, nt, b, m);
    return 0;
}

// os & 3: 0 closed shell, 1 open shell with a second LDS tile, 2 open
// shell with the second exchange terms straight to G2; os & 4: the lean
// open-shell form (FP64; FP32 launches take the register form)
void launch_fock_tile_C1000(const TileGroup* g, int ng, const Task* t, const PairBlock* b, const MolDesc* m, int fp32, int os, int waves, size_t lds, int grid, LaunchTo& q)
{
    if (ng <= 0) return;
    if (grid <= 0 || grid > ng) grid = ng;
    const bool lean = (os & 4) != 0;
    os &= 3;
    const int k2 = os == 1;
    if (fp32 && os)
        q((fock_tile_kernel<C1000, float, true>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m, k2);
    else if (fp32)
        q((fock_tile_kernel<C1000, float>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m, 0);
    else if (os && lean)
        q((fock_tile_kernel<C1000, double, true, true>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m, k2);
    else if (os)
        q((fock_tile_kernel<C1000, double, true>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m, k2);
    else
        q((fock_tile_kernel<C1000, double>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m, 0);
}

}  // namespace qf
