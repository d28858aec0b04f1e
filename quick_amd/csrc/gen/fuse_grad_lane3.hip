// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "../qf_gfuse.h"
#include "../qf_launch.h"
#include "grad_C0000.h"
#include "grad_C1000.h"

namespace qf {

// slots: doubles of LDS slots (wave-per-quartet classes); tile: doubles of the gradient
void launch_fuse_grad_lane3(const FusedBlock* list, int n, const Task* t, const PairBlock* b, const MolDesc* m,
    int slots, int tile, double* gscratch, LaunchTo& q)
{
    (void)slots;
    (void)gscratch;
    q((fused_grad_md_kernel<3,
        FuseMember<0, C0000GradMd>,
        FuseMember<16, C1000GradMd>>),
      dim3(n), dim3(WAVE), tile * sizeof(double), list, t, b, m, tile);
}

}  // namespace qf
