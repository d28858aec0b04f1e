// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "coop_C2220.h"
#include "md_C2220.h"

namespace qf {

// closed shell, FP64 only: an open-shell build runs the wave-per-quartet kernel
// instead, unless the class is asked for in two closed-shell passes
void launch_fock_tile_C2220(const TileGroup* g, int ng, const Task* t, const PairBlock* b, const MolDesc* m, int fp32, int os, int waves, size_t lds, int grid, LaunchTo& q)
{
    if (ng <= 0) return;
    if (grid <= 0 || grid > ng) grid = ng;
    (void)fp32;
    (void)os;
    q((fock_md_kernel<C2220Md>), dim3(grid), dim3(waves * WAVE), lds, g, ng, t, b, m);
}

// gscratch: COOP_GLOBAL_SLICES slices of LDS doubles when the class keeps its
// slots in global memory (the grid is then capped to that many workgroups)
void launch_fock_coop_C2220(const Task* t, int nt, const PairBlock* b, const MolDesc* m, int os, int grid, double* gscratch, LaunchTo& q)
{
    using D = C2220Coop;
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
