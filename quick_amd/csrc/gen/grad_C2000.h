// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C2000Grad {
  static constexpr int La = 2, Lb = 0, Lc = 0, Ld = 0, L = 3;
  static constexpr int NACC = 47, NV = 49, NLV = 3, NX = 47, NH = 49, NLH = 1, NI = 6;
  static constexpr int ZS = 47, SINK = 48, CF = 144, DM = 184, LDS = 205;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 49, OAM = 59, OBP = 62, OBM = -1, OCP = 80, OCM = -1;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 362, QUARTET_FLOP = 312;
  static constexpr unsigned short FSLOT[4] = {98,99,100,101};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC2000Grad_vrr[49] = {{100,101,47,47,47,102,65535,2},{100,101,47,47,47,103,65535,1},{100,101,47,47,47,104,65535,0},{99,100,47,47,47,105,65535,2},{99,100,47,47,47,106,65535,1},{99,100,47,47,47,107,65535,0},{98,99,47,47,47,108,65535,2},{98,99,47,47,47,109,65535,1},{98,99,47,47,47,110,65535,0},{105,102,99,100,47,101,65535,18},{105,102,47,47,47,111,65535,1},{106,103,99,100,47,112,65535,17},{105,102,47,47,47,113,65535,0},{106,103,47,47,47,114,65535,0},{107,104,99,100,47,115,65535,16},{108,105,98,99,47,116,65535,18},{108,105,47,47,47,117,65535,1},{109,106,98,99,47,118,65535,17},{108,105,47,47,47,119,65535,0},{109,106,47,47,47,120,65535,0},{110,107,98,99,47,121,65535,16},{116,101,108,105,47,98,65535,34},{116,101,47,47,47,99,65535,1},{118,112,47,47,47,100,65535,2},{118,112,109,106,47,102,65535,33},{116,101,47,47,47,103,65535,0},{117,111,47,47,47,104,65535,0},{118,112,47,47,47,122,65535,0},{121,115,47,47,47,123,65535,2},{121,115,47,47,47,124,65535,1},{121,115,110,107,47,125,65535,32},{116,101,47,47,105,126,65535,517},{116,101,47,47,47,127,65535,4},{116,101,47,47,47,128,65535,3},{117,111,47,47,106,129,65535,261},{117,111,47,47,105,130,65535,260},{117,111,47,47,47,131,65535,3},{118,112,47,47,47,132,65535,5},{118,112,47,47,106,133,65535,516},{118,112,47,47,47,134,65535,3},{119,113,47,47,107,135,65535,261},{119,113,47,47,47,136,65535,4},{119,113,47,47,105,137,65535,259},{120,114,47,47,47,138,65535,5},{120,114,47,47,107,139,65535,260},{120,114,47,47,106,140,65535,259},{121,115,47,47,47,141,65535,5},{121,115,47,47,47,142,65535,4},{121,115,47,47,107,143,65535,515}};
__device__ const int kC2000Grad_vlev[4] = {0,9,21,49};
__device__ const GradAcc kC2000Grad_acc[47] = {{110,0,0},{109,1,0},{108,2,0},{125,3,1},{124,4,1},{122,5,1},{102,6,1},{123,7,1},{104,8,1},{100,9,1},{103,10,1},{99,11,1},{98,12,1},{121,13,2},{120,14,2},{118,15,2},{119,16,2},{117,17,2},{116,18,2},{125,19,2},{124,20,2},{122,21,2},{102,22,2},{123,23,2},{104,24,2},{100,25,2},{103,26,2},{99,27,2},{98,28,2},{143,29,3},{142,30,3},{141,31,3},{140,32,3},{139,33,3},{138,34,3},{134,35,3},{133,36,3},{132,37,3},{137,38,3},{136,39,3},{135,40,3},{131,41,3},{130,42,3},{129,43,3},{128,44,3},{127,45,3},{126,46,3}};
__device__ const CoopHNode kC2000Grad_hrr[49] = {{79,28,18,5},{78,27,18,4},{77,26,18,3},{76,27,17,5},{75,25,17,4},{74,24,17,3},{70,25,15,5},{69,22,15,4},{68,21,15,3},{73,26,16,5},{72,24,16,4},{71,23,16,3},{67,24,14,5},{66,21,14,4},{65,20,14,3},{64,23,13,5},{63,20,13,4},{62,19,13,3},{59,0,47,0},{60,1,47,0},{61,2,47,0},{49,3,47,0},{50,4,47,0},{51,5,47,0},{52,6,47,0},{53,7,47,0},{54,8,47,0},{55,9,47,0},{56,10,47,0},{57,11,47,0},{58,12,47,0},{80,29,47,0},{81,30,47,0},{90,39,47,0},{91,40,47,0},{92,41,47,0},{93,42,47,0},{94,43,47,0},{95,44,47,0},{96,45,47,0},{97,46,47,0},{82,31,47,0},{83,32,47,0},{84,33,47,0},{85,34,47,0},{86,35,47,0},{87,36,47,0},{88,37,47,0},{89,38,47,0}};
__device__ const int kC2000Grad_hlev[2] = {0,49};
__device__ inline const CoopVNode* C2000Grad::vrr() { return kC2000Grad_vrr; }
__device__ inline const int* C2000Grad::vlev() { return kC2000Grad_vlev; }
__device__ inline const GradAcc* C2000Grad::acc() { return kC2000Grad_acc; }
__device__ inline const CoopHNode* C2000Grad::hrr() { return kC2000Grad_hrr; }
__device__ inline const int* C2000Grad::hlev() { return kC2000Grad_hlev; }
// (ds|ss): 20 Hermite Coulomb integrals, 39 bra products
struct C2000GradMd {
  static constexpr int La = 2, Lb = 0, Lc = 0, Ld = 0, L = 3;
  static constexpr int N1 = 9, NE = 39;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 2;      // waves per SIMD the register budget targets
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry, T out) {
    const double be100 = X;
    const double be101 = h;
    const double bd100 = rx;
    const double be200 = fma(1.0, be101, be100 * X);
    const double be201 = fma(be100, h, be101 * X);
    const double be202 = be101 * h;
    const double bd200 = fma(be100, rx, bd100 * X);
    const double bd201 = fma(be101, rx, bd100 * h);
    out[0] = 1.0;
    out[1] = be100;
    out[2] = be101;
    out[3] = bd100;
    out[4] = be200;
    out[5] = be201;
    out[6] = be202;
    out[7] = bd200;
    out[8] = bd201;
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
    am *= m2a;
    const double r000_3 = F[3] * am;
    const double r100_2 = PQ[0] * r000_3;
    const double r010_2 = PQ[1] * r000_3;
    const double r001_2 = PQ[2] * r000_3;
    const double r100_1 = PQ[0] * r000_2;
    const double r010_1 = PQ[1] * r000_2;
    const double r001_1 = PQ[2] * r000_2;
    const double r200_1 = fma(1.0, r000_2, PQ[0] * r100_2);
    const double r110_1 = PQ[0] * r010_2;
    const double r101_1 = PQ[0] * r001_2;
    const double r020_1 = fma(1.0, r000_2, PQ[1] * r010_2);
    const double r011_1 = PQ[1] * r001_2;
    const double r002_1 = fma(1.0, r000_2, PQ[2] * r001_2);
    const double r100_0 = PQ[0] * r000_1;
    const double r010_0 = PQ[1] * r000_1;
    const double r001_0 = PQ[2] * r000_1;
    const double r200_0 = fma(1.0, r000_1, PQ[0] * r100_1);
    const double r110_0 = PQ[0] * r010_1;
    const double r101_0 = PQ[0] * r001_1;
    const double r020_0 = fma(1.0, r000_1, PQ[1] * r010_1);
    const double r011_0 = PQ[1] * r001_1;
    const double r002_0 = fma(1.0, r000_1, PQ[2] * r001_1);
    const double r300_0 = fma(2.0, r100_1, PQ[0] * r200_1);
    const double r210_0 = PQ[1] * r200_1;
    const double r201_0 = PQ[2] * r200_1;
    const double r120_0 = PQ[0] * r020_1;
    const double r111_0 = PQ[0] * r011_1;
    const double r102_0 = PQ[0] * r002_1;
    const double r030_0 = fma(2.0, r010_1, PQ[1] * r020_1);
    const double r021_0 = PQ[2] * r020_1;
    const double r012_0 = PQ[1] * r002_1;
    const double r003_0 = fma(2.0, r001_1, PQ[2] * r002_1);
    double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    {
      const double ac0 = P[oc + 0 * n + 0] * (kCons[2][0] * kCons[0][0]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[2][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[2][0] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t101 = y000 * r101_0;
        const double t110 = y000 * r110_0;
        const double t200 = y000 * r200_0;
        const double t201 = y000 * r201_0;
        const double t210 = y000 * r210_0;
        const double t300 = y000 * r300_0;
        const double e0 = E[0];
        const double e1 = E[1];
        const double e2 = E[2];
        w = fma(e2, t200, fma(e1, t100, fma(e0, t000, w)));
        px = fma(e2, t300, fma(e1, t200, fma(e0, t100, px)));
        py = fma(e2, t210, fma(e1, t110, fma(e0, t010, py)));
        pz = fma(e2, t201, fma(e1, t101, fma(e0, t001, pz)));
        sx = fma(E[4], t100, fma(E[3], t000, sx));
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * (kCons[2][1] * kCons[0][0]);
      const double ad0 = P[od + 1 * n + 0] * (kCons[2][1] * kCons[0][0]);
      {
        const double ab = Pab[1 * n + 0] * (kCons[2][1] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t011 = y000 * r011_0;
        const double t020 = y000 * r020_0;
        const double t101 = y000 * r101_0;
        const double t110 = y000 * r110_0;
        const double t200 = y000 * r200_0;
        const double t111 = y000 * r111_0;
        const double t120 = y000 * r120_0;
        const double t210 = y000 * r210_0;
        const double e0 = E[5];
        const double e1 = E[6];
        const double e2 = E[7];
        const double e3 = E[8];
        w = fma(e3, t110, fma(e2, t100, fma(e1, t010, fma(e0, t000, w))));
        px = fma(e3, t210, fma(e2, t200, fma(e1, t110, fma(e0, t100, px))));
        py = fma(e3, t120, fma(e2, t110, fma(e1, t020, fma(e0, t010, py))));
        pz = fma(e3, t111, fma(e2, t101, fma(e1, t011, fma(e0, t001, pz))));
        sx = fma(E[10], t010, fma(E[9], t000, sx));
        sy = fma(E[12], t100, fma(E[11], t000, sy));
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * (kCons[2][2] * kCons[0][0]);
      const double ad0 = P[od + 2 * n + 0] * (kCons[2][2] * kCons[0][0]);
      {
        const double ab = Pab[2 * n + 0] * (kCons[2][2] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t011 = y000 * r011_0;
        const double t020 = y000 * r020_0;
        const double t110 = y000 * r110_0;
        const double t021 = y000 * r021_0;
        const double t030 = y000 * r030_0;
        const double t120 = y000 * r120_0;
        const double e0 = E[13];
        const double e1 = E[14];
        const double e2 = E[15];
        w = fma(e2, t020, fma(e1, t010, fma(e0, t000, w)));
        px = fma(e2, t120, fma(e1, t110, fma(e0, t100, px)));
        py = fma(e2, t030, fma(e1, t020, fma(e0, t010, py)));
        pz = fma(e2, t021, fma(e1, t011, fma(e0, t001, pz)));
        sy = fma(E[17], t010, fma(E[16], t000, sy));
      }
    }
    {
      const double ac0 = P[oc + 3 * n + 0] * (kCons[2][3] * kCons[0][0]);
      const double ad0 = P[od + 3 * n + 0] * (kCons[2][3] * kCons[0][0]);
      {
        const double ab = Pab[3 * n + 0] * (kCons[2][3] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t002 = y000 * r002_0;
        const double t011 = y000 * r011_0;
        const double t101 = y000 * r101_0;
        const double t110 = y000 * r110_0;
        const double t200 = y000 * r200_0;
        const double t102 = y000 * r102_0;
        const double t111 = y000 * r111_0;
        const double t201 = y000 * r201_0;
        const double e0 = E[18];
        const double e1 = E[19];
        const double e2 = E[20];
        const double e3 = E[21];
        w = fma(e3, t101, fma(e2, t100, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t201, fma(e2, t200, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t111, fma(e2, t110, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t102, fma(e2, t101, fma(e1, t002, fma(e0, t001, pz))));
        sx = fma(E[23], t001, fma(E[22], t000, sx));
        sz = fma(E[25], t100, fma(E[24], t000, sz));
      }
    }
    {
      const double ac0 = P[oc + 4 * n + 0] * (kCons[2][4] * kCons[0][0]);
      const double ad0 = P[od + 4 * n + 0] * (kCons[2][4] * kCons[0][0]);
      {
        const double ab = Pab[4 * n + 0] * (kCons[2][4] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t002 = y000 * r002_0;
        const double t011 = y000 * r011_0;
        const double t020 = y000 * r020_0;
        const double t101 = y000 * r101_0;
        const double t110 = y000 * r110_0;
        const double t012 = y000 * r012_0;
        const double t021 = y000 * r021_0;
        const double t111 = y000 * r111_0;
        const double e0 = E[26];
        const double e1 = E[27];
        const double e2 = E[28];
        const double e3 = E[29];
        w = fma(e3, t011, fma(e2, t010, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t111, fma(e2, t110, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t021, fma(e2, t020, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t012, fma(e2, t011, fma(e1, t002, fma(e0, t001, pz))));
        sy = fma(E[31], t001, fma(E[30], t000, sy));
        sz = fma(E[33], t010, fma(E[32], t000, sz));
      }
    }
    {
      const double ac0 = P[oc + 5 * n + 0] * (kCons[2][5] * kCons[0][0]);
      const double ad0 = P[od + 5 * n + 0] * (kCons[2][5] * kCons[0][0]);
      {
        const double ab = Pab[5 * n + 0] * (kCons[2][5] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double y000 = g0_0;
        const double t000 = y000 * r000_0;
        const double t001 = y000 * r001_0;
        const double t010 = y000 * r010_0;
        const double t100 = y000 * r100_0;
        const double t002 = y000 * r002_0;
        const double t011 = y000 * r011_0;
        const double t101 = y000 * r101_0;
        const double t003 = y000 * r003_0;
        const double t012 = y000 * r012_0;
        const double t102 = y000 * r102_0;
        const double e0 = E[34];
        const double e1 = E[35];
        const double e2 = E[36];
        w = fma(e2, t002, fma(e1, t001, fma(e0, t000, w)));
        px = fma(e2, t102, fma(e1, t101, fma(e0, t100, px)));
        py = fma(e2, t012, fma(e1, t011, fma(e0, t010, py)));
        pz = fma(e2, t003, fma(e1, t002, fma(e0, t001, pz)));
        sz = fma(E[38], t001, fma(E[37], t000, sz));
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
__device__ const unsigned kC2000GradMd_index[39] = {4,5,6,7,8,257,513,258,514,259,515,769,770,1024,1280,1536,1792,2048,65537,131073,65538,131074,65539,131075,196609,196610,65792,131328,66048,131584,66304,131840,196864,197120,262144,327680,393216,458752,524288};
__device__ inline const unsigned* C2000GradMd::index() { return kC2000GradMd_index; }
}  // namespace qf
