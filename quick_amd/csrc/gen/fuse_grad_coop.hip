// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "../qf_gfuse.h"
#include "../qf_launch.h"
#include "grad_C2121.h"
#include "grad_C2211.h"
#include "grad_C2220.h"

namespace qf {

// slots: doubles of LDS slots (wave-per-quartet classes); tile: doubles of the gradient
void launch_fuse_grad_coop(const FusedBlock* list, int n, const Task* t, const PairBlock* b, const MolDesc* m,
    int slots, int tile, double* gscratch, LaunchTo& q)
{
    const int grid = n;
    q((fused_grad_coop_kernel<6582,
        FuseMember<68, C2121Grad>,
        FuseMember<82, C2211Grad>,
        FuseMember<83, C2220Grad>>),
      dim3(grid), dim3(WAVE), (slots + tile) * sizeof(double), list, n, t, b, m, gscratch, slots, tile);
}

}  // namespace qf
