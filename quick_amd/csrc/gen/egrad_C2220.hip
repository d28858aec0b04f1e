// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "grad_C2220.h"

namespace qf {

// grad_tile: 3 natom doubles of LDS for the workgroup's gradient (0: atomics
// straight to md.grad); gscratch: COOP_GLOBAL_SLICES slices when the class
// keeps its slots in global memory
void launch_grad_C2220(const Task* t, int nt, const PairBlock* b, const MolDesc* m, int grid, size_t grad_tile, double* gscratch, int fp32, LaunchTo& q)
{
    using D = C2220Grad;
    if (nt <= 0) return;
    if (grid <= 0 || grid > nt) grid = nt;
    if (D::GLOBAL_SLOTS && grid > COOP_GLOBAL_SLICES) grid = COOP_GLOBAL_SLICES;
    const size_t lds = (D::GLOBAL_SLOTS ? 0 : D::LDS * sizeof(double)) + grad_tile;
    q((grad_coop_kernel<D>), dim3(grid), dim3(D::NT), lds, t, nt, b, m, gscratch, (int)(grad_tile / sizeof(double)), fp32);
}

}  // namespace qf
