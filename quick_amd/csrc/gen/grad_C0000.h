// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C0000Grad {
  static constexpr int La = 0, Lb = 0, Lc = 0, Ld = 0, L = 1;
  static constexpr int NACC = 10, NV = 6, NLV = 1, NX = 10, NH = 9, NLH = 1, NI = 1;
  static constexpr int ZS = 10, SINK = 11, CF = 29, DM = 69, LDS = 75;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 12, OAM = -1, OBP = 15, OBM = -1, OCP = 18, OCM = -1;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 100, QUARTET_FLOP = 52;
  static constexpr unsigned short FSLOT[2] = {21,22};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC0000Grad_vrr[6] = {{21,22,10,10,10,23,65535,2},{21,22,10,10,10,24,65535,1},{21,22,10,10,10,25,65535,0},{21,22,10,10,10,26,65535,5},{21,22,10,10,10,27,65535,4},{21,22,10,10,10,28,65535,3}};
__device__ const int kC0000Grad_vlev[2] = {0,6};
__device__ const GradAcc kC0000Grad_acc[10] = {{25,0,1},{24,1,1},{23,2,1},{21,3,2},{25,4,2},{24,5,2},{23,6,2},{28,7,3},{27,8,3},{26,9,3}};
__device__ const CoopHNode kC0000Grad_hrr[9] = {{17,6,3,5},{16,5,3,4},{15,4,3,3},{12,0,10,0},{13,1,10,0},{14,2,10,0},{18,7,10,0},{19,8,10,0},{20,9,10,0}};
__device__ const int kC0000Grad_hlev[2] = {0,9};
__device__ inline const CoopVNode* C0000Grad::vrr() { return kC0000Grad_vrr; }
__device__ inline const int* C0000Grad::vlev() { return kC0000Grad_vlev; }
__device__ inline const GradAcc* C0000Grad::acc() { return kC0000Grad_acc; }
__device__ inline const CoopHNode* C0000Grad::hrr() { return kC0000Grad_hrr; }
__device__ inline const int* C0000Grad::hlev() { return kC0000Grad_hlev; }
// (ss|ss): 4 Hermite Coulomb integrals, 0 bra products
struct C0000GradMd {
  static constexpr int La = 0, Lb = 0, Lc = 0, Ld = 0, L = 1;
  static constexpr int N1 = 1, NE = 0;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 3;      // waves per SIMD the register budget targets
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry, T out) {
    out[0] = 1.0;
  }
  // Dcd with 2 cons, Dbc and Dbd with hyb/2 cons; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[1], const double (&Dbc)[1], const double (&Dbd)[1], double& W, double (&gP)[3], double (&gR)[3], double (&gS)[3]) {
    double am = pref;
    const double r000_0 = F[0] * am;
    am *= m2a;
    const double r000_1 = F[1] * am;
    const double r100_0 = PQ[0] * r000_1;
    const double r010_0 = PQ[1] * r000_1;
    const double r001_0 = PQ[2] * r000_1;
    double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    {
      const double ac0 = P[oc + 0 * n + 0] * (kCons[0][0] * kCons[0][0]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[0][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[0][0] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        w = t000 + w;
        px = t100 + px;
        py = t010 + py;
        pz = t001 + pz;
      }
    }
    W = w;
    gP[0] = px; gP[1] = py; gP[2] = pz;
    gR[0] = sx; gR[1] = sy; gR[2] = sz;
    gS[0] = 0.0;
    gS[1] = 0.0;
    gS[2] = 0.0;
  }
};
__device__ const unsigned kC0000GradMd_index[1] = {0};
__device__ inline const unsigned* C0000GradMd::index() { return kC0000GradMd_index; }
}  // namespace qf
