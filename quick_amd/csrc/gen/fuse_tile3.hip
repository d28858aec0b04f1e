// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "C0000.h"
#include "C1000.h"
#include "C1010.h"
#include "C1100.h"
#include "C2000.h"
#include "C2100.h"
#include "C3000.h"

namespace qf {

void launch_fuse_tile3(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)gscratch;
    if (os)
        q((fused_tile_kernel<3, true,
        FuseMember<0, C0000>,
        FuseMember<16, C1000>,
        FuseMember<17, C1010>,
        FuseMember<32, C1100>,
        FuseMember<48, C2000>,
        FuseMember<64, C2100>,
        FuseMember<96, C3000>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
    else
        q((fused_tile_kernel<3, false,
        FuseMember<0, C0000>,
        FuseMember<16, C1000>,
        FuseMember<17, C1010>,
        FuseMember<32, C1100>,
        FuseMember<48, C2000>,
        FuseMember<64, C2100>,
        FuseMember<96, C3000>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
}

}  // namespace qf
