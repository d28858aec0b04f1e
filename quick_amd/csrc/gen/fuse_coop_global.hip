// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "coop_C3232.h"
#include "coop_C3322.h"
#include "coop_C3331.h"
#include "coop_C3332.h"
#include "coop_C3333.h"

namespace qf {

void launch_fuse_coop_global(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)g;
    (void)waves;
    const int grid = n > COOP_GLOBAL_SLICES ? COOP_GLOBAL_SLICES : n;
    if (os)
        q((fused_coop_kernel<true, 35734,
        FuseMember<136, C3232Coop>,
        FuseMember<149, C3322Coop>,
        FuseMember<151, C3331Coop>,
        FuseMember<152, C3332Coop>,
        FuseMember<153, C3333Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
    else
        q((fused_coop_kernel<false, 35734,
        FuseMember<136, C3232Coop>,
        FuseMember<149, C3322Coop>,
        FuseMember<151, C3331Coop>,
        FuseMember<152, C3332Coop>,
        FuseMember<153, C3333Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
}

}  // namespace qf
