// Several quartet classes in one launch.
//
// A molecule of up to a few hundred functions has some hundred workgroups in
// each of its 21 to 55 classes, and one workgroup runs for 10-150 us: class by
// class, even on four hardware queues, the chip idles through the tail of
// every launch, and the smallest molecules pay a launch per class.  Here the
// classes that need the same registers (and therefore lose no occupancy to each
// other) share one kernel: the host lists the workgroups of all of them,
// longest first, and each looks up the class it runs.
#pragma once
#include "qf_coop.h"
#include "qf_device.h"

namespace qf {

template <int ID, class C>
struct FuseMember {
    static constexpr int id = ID;
    using type = C;
};

constexpr int kFuseTwoTiles = 256;   // FusedBlock::cls of a Fock launch: open shell with a second LDS tile
constexpr int kFuseFp32 = 256;       // ... of a gradient launch: the task is of the FP32 half of its class

// Tile classes; W: waves per SIMD the register budget of all of them targets.
template <int W, bool OS, class... M>
__global__ __attribute__((amdgpu_flat_work_group_size(WAVE, 4 * WAVE), amdgpu_waves_per_eu(W)))
void fused_tile_kernel(const FusedBlock* __restrict__ list, const TileGroup* __restrict__ groups,
                       const Task* __restrict__ tasks, const PairBlock* __restrict__ blocks,
                       const MolDesc* __restrict__ mols)
{
    extern __shared__ double qf_lds[];
    QF_BOYS_LDS_DECL;
    QF_BOYS_LDS_FILL();
    const FusedBlock f = cptr(list)[blockIdx.x];
    const TileGroup g = cptr(groups)[f.index];
    const int cls = f.cls & (kFuseTwoTiles - 1), k2 = f.cls & kFuseTwoTiles;
    (void)((cls == M::id && (fock_tile_group<typename M::type, double, OS, OS>(
                                 g, tasks, blocks, mols, k2, (QF_AS_LDS double*)qf_lds, QF_BOYS_LDS_PTR,
                                 (const QF_AS_LDS float*)nullptr),
                             true)) || ...);
}

// Wave-per-quartet classes; STRIDE: doubles of a workgroup's slice of the
// global slot buffer (classes with slots in LDS: unused).
template <bool OS, int STRIDE, class... M>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(4)))
void fused_coop_kernel(const FusedBlock* __restrict__ list, int n, const Task* __restrict__ tasks,
                       const PairBlock* __restrict__ blocks, const MolDesc* __restrict__ mols, double* gscratch)
{
    QF_BOYS_LDS_DECL;
    QF_BOYS_LDS_FILL();
    // (a loop over the list, which only the capped grids of the global slots
    // need, has the compiler hoist every class's invariants in front of it)
    int x = blockIdx.x;
    do {
        const FusedBlock f = cptr(list)[x];
        const Task t = cptr(tasks)[f.index];
        (void)((f.cls == M::id && (coop_task<typename M::type, OS>(
                                       t, blocks, mols, coop_slots<typename M::type, STRIDE>(gscratch),
                                       QF_BOYS_LDS_PTR),
                                   true)) || ...);
        x += gridDim.x;
    } while ((M::type::GLOBAL_SLOTS && ...) && x < n);
}

}  // namespace qf
