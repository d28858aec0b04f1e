// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "../qf_gfuse.h"
#include "../qf_launch.h"
#include "grad_C1010.h"
#include "grad_C1100.h"
#include "grad_C2000.h"
#include "grad_C2100.h"

namespace qf {

// slots: doubles of LDS slots (wave-per-quartet classes); tile: doubles of the gradient
void launch_fuse_grad_lane2(const FusedBlock* list, int n, const Task* t, const PairBlock* b, const MolDesc* m,
    int slots, int tile, double* gscratch, LaunchTo& q)
{
    (void)slots;
    (void)gscratch;
    q((fused_grad_md_kernel<2,
        FuseMember<17, C1010GradMd>,
        FuseMember<32, C1100GradMd>,
        FuseMember<48, C2000GradMd>,
        FuseMember<64, C2100GradMd>>),
      dim3(n), dim3(WAVE), tile * sizeof(double), list, t, b, m, tile);
}

}  // namespace qf
