// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "C1110.h"
#include "C2010.h"
#include "C2200.h"
#include "C3010.h"
#include "C3100.h"

namespace qf {

void launch_fuse_tile2(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)gscratch;
    if (os)
        q((fused_tile_kernel<2, true,
        FuseMember<33, C1110>,
        FuseMember<49, C2010>,
        FuseMember<80, C2200>,
        FuseMember<97, C3010>,
        FuseMember<112, C3100>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
    else
        q((fused_tile_kernel<2, false,
        FuseMember<33, C1110>,
        FuseMember<49, C2010>,
        FuseMember<80, C2200>,
        FuseMember<97, C3010>,
        FuseMember<112, C3100>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
}

}  // namespace qf
