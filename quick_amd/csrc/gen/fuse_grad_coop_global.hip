// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "../qf_gfuse.h"
#include "../qf_launch.h"
#include "grad_C2221.h"
#include "grad_C2222.h"

namespace qf {

// slots: doubles of LDS slots (wave-per-quartet classes); tile: doubles of the gradient
void launch_fuse_grad_coop_global(const FusedBlock* list, int n, const Task* t, const PairBlock* b, const MolDesc* m,
    int slots, int tile, double* gscratch, LaunchTo& q)
{
    const int grid = n > COOP_GLOBAL_SLICES ? COOP_GLOBAL_SLICES : n;
    q((fused_grad_coop_kernel<25290,
        FuseMember<84, C2221Grad>,
        FuseMember<85, C2222Grad>>),
      dim3(grid), dim3(WAVE), (slots + tile) * sizeof(double), list, n, t, b, m, gscratch, slots, tile);
}

}  // namespace qf
