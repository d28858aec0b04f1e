// Gradient launches that hold several classes, as in qf_fuse.h.
#pragma once
#include "qf_fuse.h"
#include "qf_grad.h"

namespace qf {

// Per-lane classes; W: waves per SIMD the register budget of all of them targets.
template <int W, class... M>
__global__ __attribute__((amdgpu_flat_work_group_size(WAVE, WAVE), amdgpu_waves_per_eu(W)))
void fused_grad_md_kernel(const FusedBlock* __restrict__ list, const Task* __restrict__ tasks,
                          const PairBlock* __restrict__ blocks, const MolDesc* __restrict__ mols, int tile)
{
    QF_BOYS_LDS_DECL;
    QF_BOYS_LDS_FILL();
    constexpr int sizes[] = {kGradBra<typename M::type>...};
    constexpr auto largest = [](const int* v, int n) constexpr {
        int m = 0;
        for (int k = 0; k < n; ++k) m = v[k] > m ? v[k] : m;
        return m;
    };
    __shared__ double qf_bra[largest(sizes, sizeof...(M))];
    extern __shared__ double qf_lds[];
    QF_AS_LDS double* gt = (QF_AS_LDS double*)qf_lds;
    for (int x = threadIdx.x; x < tile; x += WAVE) gt[x] = 0.0;
    __syncthreads();
    const FusedBlock f = cptr(list)[blockIdx.x];
    const Task t = cptr(tasks)[f.index];
    const int cls = f.cls & (kFuseFp32 - 1), fp32 = f.cls & kFuseFp32;
    (void)((cls == M::id && (grad_md_task<typename M::type>(t, blocks, mols, (QF_AS_LDS double*)qf_bra, gt, tile,
                                                            fp32, QF_BOYS_LDS_PTR),
                             true)) || ...);
    grad_flush(mols + cptr(blocks)[t.bra_block].mol, gt, tile);
}

// Wave-per-quartet classes; the workgroup's gradient follows `slots` doubles of
// LDS slots, STRIDE: doubles of its slice of the global slot buffer.
template <int STRIDE, class... M>
__global__ __launch_bounds__(WAVE)
void fused_grad_coop_kernel(const FusedBlock* __restrict__ list, int n, const Task* __restrict__ tasks,
                            const PairBlock* __restrict__ blocks, const MolDesc* __restrict__ mols, double* gscratch,
                            int slots, int tile)
{
    QF_BOYS_LDS_DECL;
    QF_BOYS_LDS_FILL();
    extern __shared__ double qf_lds[];
    QF_AS_LDS double* gt = (QF_AS_LDS double*)qf_lds + slots;
    for (int x = threadIdx.x; x < tile; x += WAVE) gt[x] = 0.0;
    __syncthreads();
    const MolDesc* md_last = nullptr;
    int x = blockIdx.x;
    do {
        const FusedBlock f = cptr(list)[x];
        const Task t = cptr(tasks)[f.index];
        const int cls = f.cls & (kFuseFp32 - 1), fp32 = f.cls & kFuseFp32;
        md_last = mols + cptr(blocks)[t.bra_block].mol;
        (void)((cls == M::id &&
                (grad_coop_task<typename M::type>(t, blocks, mols, coop_slots<typename M::type, STRIDE>(gscratch), gt,
                                                  tile, fp32, QF_BOYS_LDS_PTR),
                 true)) || ...);
        x += gridDim.x;
    } while ((M::type::GLOBAL_SLOTS && ...) && x < n);
    grad_flush(md_last, gt, tile);
}

}  // namespace qf
