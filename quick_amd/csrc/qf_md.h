// Per-lane Fock kernel in Hermite Gaussians for the classes whose contracted
// integrals and recursion intermediates do not fit a lane's registers.
//
// Layout, screening, tile and flush are those of fock_tile_kernel: one quartet
// per lane, the wave's bras sharing their first Q-shell a, J_ab and the
// exchange terms in the workgroup's LDS tile.  What differs is the work per
// primitive quartet (gen_md.py, C::prim): the Hermite Coulomb integrals
// R_N, |N| <= La+Lb+Lc+Ld, stay in registers, and the integrals of one
// component pair (a, b) at a time go into J and K at once, with weights, so
// nothing is kept per contracted quartet but its exchange rows.  The bra's
// expansion products E_x E_y E_z are the same in every lane and come from a
// table in LDS that the wave fills once per bra primitive.
//
// Bound: FP64 VALU and its latency at one wave per SIMD (256 registers and as
// many accumulation registers, 0.3 KB of scratch per lane for (dp|pp), 1.3 to 2
// KB for the (dd| and (dp|dp) classes).  The exchange rows and J_ab leave the
// lane once per contracted quartet: added to the tile per primitive quartet,
// where lanes of one ket row meet at one address, (dp|pp) took 1.0 ms instead of
// 0.38.  Measured per class: gen_eri.py, MD_CLASSES.
#pragma once

#include "qf_device.h"

namespace qf {

// Orders the LDS accesses of one wave (which the LDS unit executes in order):
// the compiler moves none across.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class C>
__device__ __forceinline__ void fock_md_task(const Task& t, const PairBlock& bb, const PairBlock& kb,
                                             const MolDesc& md, QF_AS_GLOBAL double* G, const TileRef& tr,
                                             QF_AS_LDS double* bra)
{
    constexpr int na = ncart(C::La), nb = ncart(C::Lb), nc = ncart(C::Lc), nd = ncart(C::Ld);
    const int lane = threadIdx.x % WAVE;
    const bool in_range = lane < t.ket_count;
    const int j = in_range ? t.ket_start + lane : t.ket_start;
    const PairInfo ki = gptr(kb.info)[j];
    const int n = md.nbasis, ns = md.nshell;
    const auto cmc = cptr(md.cutmat);
    const auto cm = gptr(md.cutmat);
    const auto PJ = gptr(md.PJ);
    const auto PJu = cptr(md.PJ);
    const auto P = gptr(md.P);
    const auto bperm = cptr(bb.bperm);
    const auto index = gptr(C::index());
    const auto bp = cptr(bb.prim);     // bra data, the same in every lane: scalar loads
    const auto kp = gptr(kb.prim);
    const int bn = bb.n, bK = bb.K, kn = kb.n;
    const size_t kf = (size_t)kb.K * kn;

    const PairInfo b0 = cptr(bb.info)[bperm[t.kb]];
    const int sa = b0.sa, fa = b0.fa;
    const double cm_cd = 4.0 * cm[ki.sa * ns + ki.sb];
    const double cm_ac = cm[sa * ns + ki.sa];
    const double cm_ad = cm[sa * ns + ki.sb];
    double Dcd[nc * nd], Jcd[nc * nd];
#pragma unroll
    for (int x = 0; x < nc * nd; ++x) {
        Dcd[x] = PJ[(ki.fa + x / nd) * n + ki.fb + x % nd];
        Jcd[x] = 0.0;
    }
    bool touched = false;
    for (int kk0 = t.kb; kk0 < t.ke; ++kk0) {
        const int kk = wave_uniform(kk0);
        const int i = bperm[kk];
        const PairInfo bi = cptr(bb.info)[i];
        const double ytest = bi.ycut * ki.ycut;
        double dn = fmax(4.0 * cmc[bi.sa * ns + bi.sb], cm_cd);
        dn = fmax(dn, cm_ad);
        dn = fmax(dn, cm_ac);
        dn = fmax(dn, cm[bi.sb * ns + ki.sa]);
        dn = fmax(dn, cm[bi.sb * ns + ki.sb]);
        const bool valid = in_range && (ytest > md.cutoff) && (ytest * dn > md.cutoff) && (!t.same_block || j <= i) &&
                           (t.all_fp64 || ytest >= md.split);
        if (!__any(valid)) continue;
        touched = touched || valid;
        double Dbc[nb * nc], Dbd[nb * nd], Kbc[nb * nc], Kbd[nb * nd];
#pragma unroll
        for (int x = 0; x < nb * nc; ++x) {
            Dbc[x] = P[(bi.fb + x / nc) * n + ki.fa + x % nc] * kCons[C::Lb][x / nc];
            Kbc[x] = 0.0;
        }
#pragma unroll
        for (int x = 0; x < nb * nd; ++x) {
            Dbd[x] = P[(bi.fb + x / nd) * n + ki.fb + x % nd] * kCons[C::Lb][x / nd];
            Kbd[x] = 0.0;
        }
        const double s = 0.25 * (bi.qa != bi.qb ? 2.0 : 1.0) * (ki.qa != ki.qb ? 2.0 : 1.0) *
                         (bi.id != ki.id ? 2.0 : 1.0);
        const int maxm = bi.qfs + ki.qfs;
        double Jab[na * nb], Kac[na * nc], Kad[na * nd];
#pragma unroll
        for (int x = 0; x < na * nb; ++x) Jab[x] = 0.0;
#pragma unroll
        for (int x = 0; x < na * nc; ++x) Kac[x] = 0.0;
#pragma unroll
        for (int x = 0; x < na * nd; ++x) Kad[x] = 0.0;
        for (int ip0 = t.pb; ip0 < t.pe; ++ip0) {
            const int ip = wave_uniform(ip0);
            const double cb = dn * bp[(PF_CUT * bK + ip) * bn + i];
            if (!__any(valid && cb * kp[PF_CUT * kf + (size_t)t.qb * kn + j] > md.primlim)) break;
            const double zb = bp[(PF_ZETA * bK + ip) * bn + i];
            const double hb = bp[(PF_OOZ2 * bK + ip) * bn + i];
            const double Pb[3] = {bp[(PF_PX * bK + ip) * bn + i], bp[(PF_PY * bK + ip) * bn + i],
                                  bp[(PF_PZ * bK + ip) * bn + i]};
            const double Kb = bp[(PF_KC * bK + ip) * bn + i];
            wave_lds_fence();   // the previous primitive's table has been read
            const int dir = lane % 3;
            const double PA = dir == 0 ? Pb[0] - bi.A[0] : dir == 1 ? Pb[1] - bi.A[1] : Pb[2] - bi.A[2];
            const double AB = dir == 0 ? bi.AB[0] : dir == 1 ? bi.AB[1] : bi.AB[2];
            if (lane < 3) C::bra1d(PA, PA + AB, hb, bra + lane * C::N1);
            wave_lds_fence();
#pragma unroll
            for (int x0 = 0; x0 < C::NE; x0 += WAVE) {
                const int x = x0 + lane;
                const unsigned id = index[x < C::NE ? x : 0];
                const double v = bra[id & 255] * bra[C::N1 + ((id >> 8) & 255)] * bra[2 * C::N1 + (id >> 16)];
                if (x < C::NE) bra[3 * C::N1 + x] = v;
            }
            wave_lds_fence();
            for (int jp0 = t.qb; jp0 < t.qe; ++jp0) {
                const int jp = wave_uniform(jp0);
                const size_t ko = (size_t)jp * kn + j;
                const bool act = valid && cb * kp[PF_CUT * kf + ko] > md.primlim;
                if (!__any(act)) break;
                if (!act) continue;
                const double zk = kp[PF_ZETA * kf + ko], hk = kp[PF_OOZ2 * kf + ko], Kk = kp[PF_KC * kf + ko];
                const double Qk[3] = {kp[PF_PX * kf + ko], kp[PF_PY * kf + ko], kp[PF_PZ * kf + ko]};
                const double QC[3] = {Qk[0] - ki.A[0], Qk[1] - ki.A[1], Qk[2] - ki.A[2]};
                const double QD[3] = {QC[0] + ki.AB[0], QC[1] + ki.AB[1], QC[2] + ki.AB[2]};
                const double PQ[3] = {Pb[0] - Qk[0], Pb[1] - Qk[1], Pb[2] - Qk[2]};
                const double rs = qf_rsqrt(zb + zk);
                const double al = zb * zk * (rs * rs);
                const double rpq = PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2];
                double F[C::L + 1];
                boys_quick<C::L>(rpq * al, maxm, F, tr.boys);
                // the product table and the density blocks are the same for every primitive:
                // hoisted, they would be hundreds of registers
                int eo = 3 * C::N1, po = bi.fa * n + bi.fb;
                QF_OPAQUE(eo);
                QF_OPAQUE_S(po);
                C::prim(F, Kb * Kk * rs * s, -2.0 * al, PQ, QC, QD, hk, bra + eo, PJu + po, P, n,
                        fa * n + ki.fa, fa * n + ki.fb, Dcd, Dbc, Dbd, Jcd, Kbc, Kbd, Jab, Kac, Kad);
            }
        }
#pragma unroll
        for (int x = 0; x < na * nb; ++x) {
            const double v = wave_sum_all_active(Jab[x] * (kCons[C::La][x / nb] * kCons[C::Lb][x % nb]));
            if (lane == 0 && v != 0.0) lds_add(&tr.jab[(kk - tr.chunk_kb) * (na * nb) + x], v);
        }
        if (valid) {
#pragma unroll
            for (int a = 0; a < na; ++a) {
                QF_AS_LDS double* row = tr.k + a * tr.ncol;
#pragma unroll
                for (int c = 0; c < nc; ++c) lds_add(&row[ki.cola + c], Kac[a * nc + c] * kCons[C::La][a]);
#pragma unroll
                for (int d = 0; d < nd; ++d) lds_add(&row[ki.colb + d], Kad[a * nd + d] * kCons[C::La][a]);
            }
            const int r0 = na + (kk - tr.chunk_kb) * nb;
#pragma unroll
            for (int b = 0; b < nb; ++b) {
                QF_AS_LDS double* row = tr.k + (r0 + b) * tr.ncol;
#pragma unroll
                for (int c = 0; c < nc; ++c) lds_add(&row[ki.cola + c], Kbc[b * nc + c] * kCons[C::Lb][b]);
#pragma unroll
                for (int d = 0; d < nd; ++d) lds_add(&row[ki.colb + d], Kbd[b * nd + d] * kCons[C::Lb][b]);
            }
        }
    }
    if (!touched) return;
#pragma unroll
    for (int c = 0; c < nc; ++c)
#pragma unroll
        for (int d = 0; d < nd; ++d) atomic_add(&G[(ki.fa + c) * n + ki.fb + d], Jcd[c * nd + d]);
}

// One workgroup per TileGroup, as fock_tile_kernel (closed shell, FP64).
template <class C>
__global__ __attribute__((amdgpu_flat_work_group_size(WAVE, 4 * WAVE), amdgpu_waves_per_eu(1)))
void fock_md_kernel(const TileGroup* __restrict__ groups, int ngroups, const Task* __restrict__ tasks,
                    const PairBlock* __restrict__ blocks, const MolDesc* __restrict__ mols)
{
    constexpr int na = ncart(C::La), nb = ncart(C::Lb);
    constexpr int kBra = 3 * C::N1 + (C::NE > 0 ? C::NE : 1);
    extern __shared__ double qf_lds[];
    __shared__ double qf_bra[4 * kBra];
    QF_BOYS_LDS_DECL;
    QF_BOYS_LDS_FILL();
    QF_AS_LDS double* lds = (QF_AS_LDS double*)qf_lds;
    const int nw = blockDim.x / WAVE;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    QF_AS_LDS double* bra = (QF_AS_LDS double*)qf_bra + wave * kBra;
    for (int gi = blockIdx.x; gi < ngroups; gi += gridDim.x) {
        const TileGroup g = cptr(groups)[gi];
        const Task t0 = cptr(tasks)[g.task_begin];
        const PairBlock bb = cptr(blocks)[t0.bra_block];
        const PairBlock kb = cptr(blocks)[t0.ket_block];
        const MolDesc md = cptr(mols)[bb.mol];
        const int n = md.nbasis;
        const int ncol = kb.ncol;
        const int ntile = (na + g.nbra * nb) * ncol, njab = g.nbra * na * nb;
        for (int x = threadIdx.x; x < ntile + njab; x += blockDim.x) lds[x] = 0.0;
        __syncthreads();
        const auto G = gptr_rw(md.G + (size_t)(blockIdx.x % md.replicas) * n * n);
        const TileRef tr{lds, nullptr, lds + ntile, ncol, g.chunk_kb, QF_BOYS_LDS_PTR, nullptr};
        for (int ti = g.task_begin + wave; ti < g.task_end; ti += nw) {
            const Task t = cptr(tasks)[wave_uniform(ti)];
            fock_md_task<C>(t, bb, kb, md, G, tr, bra);
        }
        __syncthreads();
        tile_flush<na, nb>(lds, ntile, ntile, njab, ncol, g, bb, kb, md, G, G);
        __syncthreads();   // the next group reuses the tile
    }
}

}  // namespace qf
