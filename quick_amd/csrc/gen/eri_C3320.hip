// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "coop_C3320.h"

namespace qf {

// gscratch: COOP_GLOBAL_SLICES slices of LDS doubles when the class keeps its
// slots in global memory (the grid is then capped to that many workgroups)
void launch_fock_coop_C3320(const Task* t, int nt, const PairBlock* b, const MolDesc* m, int os, int grid, double* gscratch, LaunchTo& q)
{
    using D = C3320Coop;
    if (nt <= 0) return;
    if (grid <= 0 || grid > nt) grid = nt;
    if (D::GLOBAL_SLOTS && grid > COOP_GLOBAL_SLICES) grid = COOP_GLOBAL_SLICES;
    const size_t lds = D::GLOBAL_SLOTS ? 0 : D::LDS * sizeof(double);
    if (os)
        q((fock_coop_kernel<D, true>), dim3(grid), dim3(D::NT), lds, t, nt, b, m, gscratch);
    else
        q((fock_coop_kernel<D>), dim3(grid), dim3(D::NT), lds, t, nt, b, m, gscratch);
}

}  // namespace qf
