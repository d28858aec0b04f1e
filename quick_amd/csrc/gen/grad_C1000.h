// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C1000Grad {
  static constexpr int La = 1, Lb = 0, Lc = 0, Ld = 0, L = 2;
  static constexpr int NACC = 25, NV = 21, NLV = 2, NX = 25, NH = 25, NLH = 1, NI = 3;
  static constexpr int ZS = 25, SINK = 26, CF = 75, DM = 115, LDS = 127;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 27, OAM = 33, OBP = 34, OBM = -1, OCP = 43, OCM = -1;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 194, QUARTET_FLOP = 156;
  static constexpr unsigned short FSLOT[3] = {52,53,54};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC1000Grad_vrr[21] = {{53,54,25,25,25,55,65535,2},{53,54,25,25,25,56,65535,1},{53,54,25,25,25,57,65535,0},{52,53,25,25,25,58,65535,2},{52,53,25,25,25,59,65535,1},{52,53,25,25,25,60,65535,0},{58,55,52,53,25,54,65535,18},{58,55,25,25,25,61,65535,1},{59,56,52,53,25,62,65535,17},{58,55,25,25,25,63,65535,0},{59,56,25,25,25,64,65535,0},{60,57,52,53,25,65,65535,16},{58,55,25,25,53,66,65535,261},{58,55,25,25,25,67,65535,4},{58,55,25,25,25,68,65535,3},{59,56,25,25,25,69,65535,5},{59,56,25,25,53,70,65535,260},{59,56,25,25,25,71,65535,3},{60,57,25,25,25,72,65535,5},{60,57,25,25,25,73,65535,4},{60,57,25,25,53,74,65535,259}};
__device__ const int kC1000Grad_vlev[3] = {0,6,21};
__device__ const GradAcc kC1000Grad_acc[25] = {{52,0,0},{65,1,1},{64,2,1},{62,3,1},{63,4,1},{61,5,1},{54,6,1},{60,7,2},{59,8,2},{58,9,2},{65,10,2},{64,11,2},{62,12,2},{63,13,2},{61,14,2},{54,15,2},{74,16,3},{73,17,3},{72,18,3},{71,19,3},{70,20,3},{69,21,3},{68,22,3},{67,23,3},{66,24,3}};
__device__ const CoopHNode kC1000Grad_hrr[25] = {{42,15,9,5},{41,14,9,4},{40,13,9,3},{39,14,8,5},{38,12,8,4},{37,11,8,3},{36,13,7,5},{35,11,7,4},{34,10,7,3},{33,0,25,0},{27,1,25,0},{28,2,25,0},{29,3,25,0},{30,4,25,0},{31,5,25,0},{32,6,25,0},{43,16,25,0},{44,17,25,0},{45,18,25,0},{46,19,25,0},{47,20,25,0},{48,21,25,0},{49,22,25,0},{50,23,25,0},{51,24,25,0}};
__device__ const int kC1000Grad_hlev[2] = {0,25};
__device__ inline const CoopVNode* C1000Grad::vrr() { return kC1000Grad_vrr; }
__device__ inline const int* C1000Grad::vlev() { return kC1000Grad_vlev; }
__device__ inline const GradAcc* C1000Grad::acc() { return kC1000Grad_acc; }
__device__ inline const CoopHNode* C1000Grad::hrr() { return kC1000Grad_hrr; }
__device__ inline const int* C1000Grad::hlev() { return kC1000Grad_hlev; }
// (ps|ss): 10 Hermite Coulomb integrals, 9 bra products
struct C1000GradMd {
  static constexpr int La = 1, Lb = 0, Lc = 0, Ld = 0, L = 2;
  static constexpr int N1 = 4, NE = 9;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 3;      // waves per SIMD the register budget targets
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry, T out) {
    const double be100 = X;
    const double be101 = h;
    const double bd100 = rx;
    out[0] = 1.0;
    out[1] = be100;
    out[2] = be101;
    out[3] = bd100;
  }
  // Dcd with 2 cons, Dbc and Dbd with hyb/2 cons; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[1], const double (&Dbc)[1], const double (&Dbd)[1], double& W, double (&gP)[3], double (&gR)[3], double (&gS)[3]) {
    double am = pref;
    const double r000_0 = F[0] * am;
    am *= m2a;
    const double r000_1 = F[1] * am;
    am *= m2a;
    const double r000_2 = F[2] * am;
    const double r100_1 = PQ[0] * r000_2;
    const double r010_1 = PQ[1] * r000_2;
    const double r001_1 = PQ[2] * r000_2;
    const double r100_0 = PQ[0] * r000_1;
    const double r010_0 = PQ[1] * r000_1;
    const double r001_0 = PQ[2] * r000_1;
    const double r200_0 = fma(1.0, r000_1, PQ[0] * r100_1);
    const double r110_0 = PQ[0] * r010_1;
    const double r101_0 = PQ[0] * r001_1;
    const double r020_0 = fma(1.0, r000_1, PQ[1] * r010_1);
    const double r011_0 = PQ[1] * r001_1;
    const double r002_0 = fma(1.0, r000_1, PQ[2] * r001_1);
    double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    {
      const double ac0 = P[oc + 0 * n + 0] * (kCons[1][0] * kCons[0][0]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[1][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[1][0] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t101 = y000 * r101_0;
        const double t110 = y000 * r110_0;
        const double t200 = y000 * r200_0;
        const double e0 = E[0];
        const double e1 = E[1];
        w = fma(e1, t100, fma(e0, t000, w));
        px = fma(e1, t200, fma(e0, t100, px));
        py = fma(e1, t110, fma(e0, t010, py));
        pz = fma(e1, t101, fma(e0, t001, pz));
        sx = fma(E[2], t000, sx);
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * (kCons[1][1] * kCons[0][0]);
      const double ad0 = P[od + 1 * n + 0] * (kCons[1][1] * kCons[0][0]);
      {
        const double ab = Pab[1 * n + 0] * (kCons[1][1] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t011 = y000 * r011_0;
        const double t020 = y000 * r020_0;
        const double t110 = y000 * r110_0;
        const double e0 = E[3];
        const double e1 = E[4];
        w = fma(e1, t010, fma(e0, t000, w));
        px = fma(e1, t110, fma(e0, t100, px));
        py = fma(e1, t020, fma(e0, t010, py));
        pz = fma(e1, t011, fma(e0, t001, pz));
        sy = fma(E[5], t000, sy);
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * (kCons[1][2] * kCons[0][0]);
      const double ad0 = P[od + 2 * n + 0] * (kCons[1][2] * kCons[0][0]);
      {
        const double ab = Pab[2 * n + 0] * (kCons[1][2] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t002 = y000 * r002_0;
        const double t011 = y000 * r011_0;
        const double t101 = y000 * r101_0;
        const double e0 = E[6];
        const double e1 = E[7];
        w = fma(e1, t001, fma(e0, t000, w));
        px = fma(e1, t101, fma(e0, t100, px));
        py = fma(e1, t011, fma(e0, t010, py));
        pz = fma(e1, t002, fma(e0, t001, pz));
        sz = fma(E[8], t000, sz);
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
__device__ const unsigned kC1000GradMd_index[9] = {1,2,3,256,512,768,65536,131072,196608};
__device__ inline const unsigned* C1000GradMd::index() { return kC1000GradMd_index; }
}  // namespace qf
