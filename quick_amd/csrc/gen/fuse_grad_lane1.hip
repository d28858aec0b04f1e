// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#include "../qf_gfuse.h"
#include "../qf_launch.h"
#include "grad_C1110.h"
#include "grad_C1111.h"
#include "grad_C2010.h"
#include "grad_C2011.h"
#include "grad_C2020.h"
#include "grad_C2110.h"
#include "grad_C2111.h"
#include "grad_C2120.h"
#include "grad_C2200.h"
#include "grad_C2210.h"

namespace qf {

// slots: doubles of LDS slots (wave-per-quartet classes); tile: doubles of the gradient
void launch_fuse_grad_lane1(const FusedBlock* list, int n, const Task* t, const PairBlock* b, const MolDesc* m,
    int slots, int tile, double* gscratch, LaunchTo& q)
{
    (void)slots;
    (void)gscratch;
    q((fused_grad_md_kernel<1,
        FuseMember<33, C1110GradMd>,
        FuseMember<34, C1111GradMd>,
        FuseMember<49, C2010GradMd>,
        FuseMember<50, C2011GradMd>,
        FuseMember<51, C2020GradMd>,
        FuseMember<65, C2110GradMd>,
        FuseMember<66, C2111GradMd>,
        FuseMember<67, C2120GradMd>,
        FuseMember<80, C2200GradMd>,
        FuseMember<81, C2210GradMd>>),
      dim3(n), dim3(WAVE), tile * sizeof(double), list, t, b, m, tile);
}

}  // namespace qf
