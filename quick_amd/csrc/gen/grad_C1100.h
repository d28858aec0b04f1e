// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C1100Grad {
  static constexpr int La = 1, Lb = 1, Lc = 0, Ld = 0, L = 3;
  static constexpr int NACC = 66, NV = 58, NLV = 3, NX = 66, NH = 92, NLH = 2, NI = 9;
  static constexpr int ZS = 66, SINK = 67, CF = 193, DM = 233, LDS = 255;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 68, OAM = 86, OBP = 89, OBM = 107, OCP = 110, OCM = -1;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 433, QUARTET_FLOP = 592;
  static constexpr unsigned short FSLOT[4] = {137,138,139,140};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC1100Grad_vrr[58] = {{139,140,66,66,66,141,65535,2},{139,140,66,66,66,142,65535,1},{139,140,66,66,66,143,65535,0},{138,139,66,66,66,144,65535,2},{138,139,66,66,66,145,65535,1},{138,139,66,66,66,146,65535,0},{137,138,66,66,66,147,65535,2},{137,138,66,66,66,148,65535,1},{137,138,66,66,66,149,65535,0},{144,141,138,139,66,140,65535,18},{144,141,66,66,66,150,65535,1},{145,142,138,139,66,151,65535,17},{144,141,66,66,66,152,65535,0},{145,142,66,66,66,153,65535,0},{146,143,138,139,66,154,65535,16},{147,144,137,138,66,155,65535,18},{147,144,66,66,66,156,65535,1},{148,145,137,138,66,157,65535,17},{147,144,66,66,66,158,65535,0},{148,145,66,66,66,159,65535,0},{149,146,137,138,66,160,65535,16},{147,144,66,66,138,161,65535,261},{147,144,66,66,66,162,65535,4},{147,144,66,66,66,163,65535,3},{148,145,66,66,66,164,65535,5},{148,145,66,66,138,165,65535,260},{148,145,66,66,66,166,65535,3},{149,146,66,66,66,167,65535,5},{149,146,66,66,66,168,65535,4},{149,146,66,66,138,169,65535,259},{155,140,147,144,66,138,65535,34},{155,140,66,66,66,139,65535,1},{157,151,66,66,66,141,65535,2},{157,151,148,145,66,142,65535,33},{155,140,66,66,66,143,65535,0},{156,150,66,66,66,170,65535,0},{157,151,66,66,66,171,65535,0},{160,154,66,66,66,172,65535,2},{160,154,66,66,66,173,65535,1},{160,154,149,146,66,174,65535,32},{155,140,66,66,144,175,65535,517},{155,140,66,66,66,176,65535,4},{155,140,66,66,66,177,65535,3},{156,150,66,66,145,178,65535,261},{156,150,66,66,144,179,65535,260},{156,150,66,66,66,180,65535,3},{157,151,66,66,66,181,65535,5},{157,151,66,66,145,182,65535,516},{157,151,66,66,66,183,65535,3},{158,152,66,66,146,184,65535,261},{158,152,66,66,66,185,65535,4},{158,152,66,66,144,186,65535,259},{159,153,66,66,66,187,65535,5},{159,153,66,66,146,188,65535,260},{159,153,66,66,145,189,65535,259},{160,154,66,66,66,190,65535,5},{160,154,66,66,66,191,65535,4},{160,154,66,66,146,192,65535,515}};
__device__ const int kC1100Grad_vlev[4] = {0,9,30,58};
__device__ const GradAcc kC1100Grad_acc[66] = {{137,0,0},{149,1,0},{148,2,0},{147,3,0},{160,4,1},{159,5,1},{157,6,1},{158,7,1},{156,8,1},{155,9,1},{174,10,1},{173,11,1},{171,12,1},{142,13,1},{172,14,1},{170,15,1},{141,16,1},{143,17,1},{139,18,1},{138,19,1},{149,20,2},{148,21,2},{147,22,2},{160,23,2},{159,24,2},{157,25,2},{158,26,2},{156,27,2},{155,28,2},{174,29,2},{173,30,2},{171,31,2},{142,32,2},{172,33,2},{170,34,2},{141,35,2},{143,36,2},{139,37,2},{138,38,2},{169,39,3},{168,40,3},{167,41,3},{166,42,3},{165,43,3},{164,44,3},{163,45,3},{162,46,3},{161,47,3},{192,48,3},{191,49,3},{190,50,3},{189,51,3},{188,52,3},{187,53,3},{183,54,3},{182,55,3},{181,56,3},{186,57,3},{185,58,3},{184,59,3},{180,60,3},{179,61,3},{178,62,3},{177,63,3},{176,64,3},{175,65,3}};
__device__ const CoopHNode kC1100Grad_hrr[92] = {{88,3,0,5},{87,2,0,4},{86,1,0,3},{85,19,9,5},{84,18,9,4},{83,17,9,3},{82,18,8,5},{81,16,8,4},{80,15,8,3},{76,16,6,5},{75,13,6,4},{74,12,6,3},{79,17,7,5},{78,15,7,4},{77,14,7,3},{73,15,5,5},{72,12,5,4},{71,11,5,3},{70,14,4,5},{69,11,4,4},{68,10,4,3},{137,28,22,5},{138,27,22,4},{139,26,22,3},{140,38,28,5},{141,27,21,5},{142,25,21,4},{143,24,21,3},{144,37,27,5},{145,35,27,4},{146,35,25,5},{147,32,25,4},{148,26,20,5},{149,24,20,4},{150,23,20,3},{151,36,26,5},{152,34,26,4},{153,33,26,3},{154,34,24,5},{155,31,24,4},{156,30,24,3},{157,33,23,5},{158,30,23,4},{159,29,23,3},{136,65,47,5},{135,64,46,5},{134,63,45,5},{133,62,47,4},{132,61,46,4},{131,60,45,4},{130,59,47,3},{129,58,46,3},{128,57,45,3},{127,62,44,5},{126,61,43,5},{125,60,42,5},{124,56,44,4},{123,55,43,4},{122,54,42,4},{121,53,44,3},{120,52,43,3},{119,51,42,3},{118,59,41,5},{117,58,40,5},{116,57,39,5},{115,53,41,4},{114,52,40,4},{113,51,39,4},{112,50,41,3},{111,49,40,3},{110,48,39,3},{107,1,66,0},{108,2,66,0},{109,3,66,0},{106,140,137,5},{105,144,137,4},{103,145,138,4},{104,151,137,3},{102,152,138,3},{101,153,139,3},{100,144,141,5},{99,146,141,4},{97,147,142,4},{98,154,141,3},{96,155,142,3},{95,156,143,3},{94,151,148,5},{93,154,148,4},{91,155,149,4},{92,157,148,3},{90,158,149,3},{89,159,150,3}};
__device__ const int kC1100Grad_hlev[3] = {0,74,92};
__device__ inline const CoopVNode* C1100Grad::vrr() { return kC1100Grad_vrr; }
__device__ inline const int* C1100Grad::vlev() { return kC1100Grad_vlev; }
__device__ inline const GradAcc* C1100Grad::acc() { return kC1100Grad_acc; }
__device__ inline const CoopHNode* C1100Grad::hrr() { return kC1100Grad_hrr; }
__device__ inline const int* C1100Grad::hlev() { return kC1100Grad_hlev; }
// (pp|ss): 20 Hermite Coulomb integrals, 63 bra products
struct C1100GradMd {
  static constexpr int La = 1, Lb = 1, Lc = 0, Ld = 0, L = 3;
  static constexpr int N1 = 12, NE = 63;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 2;      // waves per SIMD the register budget targets
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry, T out) {
    const double be010 = Y;
    const double be011 = h;
    const double bd010 = ry;
    const double be100 = X;
    const double be101 = h;
    const double bd100 = rx;
    const double be110 = fma(1.0, be101, be100 * Y);
    const double be111 = fma(be100, h, be101 * Y);
    const double be112 = be101 * h;
    const double bd110 = fma(be100, ry, bd100 * Y);
    const double bd111 = fma(be101, ry, bd100 * h);
    out[0] = 1.0;
    out[1] = be010;
    out[2] = be011;
    out[3] = bd010;
    out[4] = be100;
    out[5] = be101;
    out[6] = bd100;
    out[7] = be110;
    out[8] = be111;
    out[9] = be112;
    out[10] = bd110;
    out[11] = bd111;
  }
  // Dcd with 2 cons, Dbc and Dbd with hyb/2 cons; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[1], const double (&Dbc)[3], const double (&Dbd)[3], double& W, double (&gP)[3], double (&gR)[3], double (&gS)[3]) {
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
      const double ac0 = P[oc + 0 * n + 0] * (kCons[1][0] * kCons[0][0]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[1][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[1][0] * kCons[1][0]);
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
      {
        const double ab = Pab[0 * n + 1] * (kCons[1][0] * kCons[1][1]);
        const double g0_0 = fma(-ad0, Dbc[1], fma(-ac0, Dbd[1], ab * Dcd[0]));
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
      {
        const double ab = Pab[0 * n + 2] * (kCons[1][0] * kCons[1][2]);
        const double g0_0 = fma(-ad0, Dbc[2], fma(-ac0, Dbd[2], ab * Dcd[0]));
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
        const double e0 = E[13];
        const double e1 = E[14];
        const double e2 = E[15];
        const double e3 = E[16];
        w = fma(e3, t101, fma(e2, t100, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t201, fma(e2, t200, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t111, fma(e2, t110, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t102, fma(e2, t101, fma(e1, t002, fma(e0, t001, pz))));
        sx = fma(E[18], t001, fma(E[17], t000, sx));
        sz = fma(E[20], t100, fma(E[19], t000, sz));
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * (kCons[1][1] * kCons[0][0]);
      const double ad0 = P[od + 1 * n + 0] * (kCons[1][1] * kCons[0][0]);
      {
        const double ab = Pab[1 * n + 0] * (kCons[1][1] * kCons[1][0]);
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
        const double e0 = E[21];
        const double e1 = E[22];
        const double e2 = E[23];
        const double e3 = E[24];
        w = fma(e3, t110, fma(e2, t100, fma(e1, t010, fma(e0, t000, w))));
        px = fma(e3, t210, fma(e2, t200, fma(e1, t110, fma(e0, t100, px))));
        py = fma(e3, t120, fma(e2, t110, fma(e1, t020, fma(e0, t010, py))));
        pz = fma(e3, t111, fma(e2, t101, fma(e1, t011, fma(e0, t001, pz))));
        sx = fma(E[26], t010, fma(E[25], t000, sx));
        sy = fma(E[28], t100, fma(E[27], t000, sy));
      }
      {
        const double ab = Pab[1 * n + 1] * (kCons[1][1] * kCons[1][1]);
        const double g0_0 = fma(-ad0, Dbc[1], fma(-ac0, Dbd[1], ab * Dcd[0]));
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
        const double e0 = E[29];
        const double e1 = E[30];
        const double e2 = E[31];
        w = fma(e2, t020, fma(e1, t010, fma(e0, t000, w)));
        px = fma(e2, t120, fma(e1, t110, fma(e0, t100, px)));
        py = fma(e2, t030, fma(e1, t020, fma(e0, t010, py)));
        pz = fma(e2, t021, fma(e1, t011, fma(e0, t001, pz)));
        sy = fma(E[33], t010, fma(E[32], t000, sy));
      }
      {
        const double ab = Pab[1 * n + 2] * (kCons[1][1] * kCons[1][2]);
        const double g0_0 = fma(-ad0, Dbc[2], fma(-ac0, Dbd[2], ab * Dcd[0]));
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
        const double e0 = E[34];
        const double e1 = E[35];
        const double e2 = E[36];
        const double e3 = E[37];
        w = fma(e3, t011, fma(e2, t010, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t111, fma(e2, t110, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t021, fma(e2, t020, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t012, fma(e2, t011, fma(e1, t002, fma(e0, t001, pz))));
        sy = fma(E[39], t001, fma(E[38], t000, sy));
        sz = fma(E[41], t010, fma(E[40], t000, sz));
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * (kCons[1][2] * kCons[0][0]);
      const double ad0 = P[od + 2 * n + 0] * (kCons[1][2] * kCons[0][0]);
      {
        const double ab = Pab[2 * n + 0] * (kCons[1][2] * kCons[1][0]);
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
        const double e0 = E[42];
        const double e1 = E[43];
        const double e2 = E[44];
        const double e3 = E[45];
        w = fma(e3, t101, fma(e2, t100, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t201, fma(e2, t200, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t111, fma(e2, t110, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t102, fma(e2, t101, fma(e1, t002, fma(e0, t001, pz))));
        sx = fma(E[47], t001, fma(E[46], t000, sx));
        sz = fma(E[49], t100, fma(E[48], t000, sz));
      }
      {
        const double ab = Pab[2 * n + 1] * (kCons[1][2] * kCons[1][1]);
        const double g0_0 = fma(-ad0, Dbc[1], fma(-ac0, Dbd[1], ab * Dcd[0]));
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
        const double e0 = E[50];
        const double e1 = E[51];
        const double e2 = E[52];
        const double e3 = E[53];
        w = fma(e3, t011, fma(e2, t010, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t111, fma(e2, t110, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t021, fma(e2, t020, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t012, fma(e2, t011, fma(e1, t002, fma(e0, t001, pz))));
        sy = fma(E[55], t001, fma(E[54], t000, sy));
        sz = fma(E[57], t010, fma(E[56], t000, sz));
      }
      {
        const double ab = Pab[2 * n + 2] * (kCons[1][2] * kCons[1][2]);
        const double g0_0 = fma(-ad0, Dbc[2], fma(-ac0, Dbd[2], ab * Dcd[0]));
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
        const double e0 = E[58];
        const double e1 = E[59];
        const double e2 = E[60];
        w = fma(e2, t002, fma(e1, t001, fma(e0, t000, w)));
        px = fma(e2, t102, fma(e1, t101, fma(e0, t100, px)));
        py = fma(e2, t012, fma(e1, t011, fma(e0, t010, py)));
        pz = fma(e2, t003, fma(e1, t002, fma(e0, t001, pz)));
        sz = fma(E[62], t001, fma(E[61], t000, sz));
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
__device__ const unsigned kC1100GradMd_index[63] = {7,8,9,10,11,260,516,261,517,262,518,772,773,65540,131076,65541,131077,65542,131078,196612,196613,1025,1281,1026,1282,1027,1283,1537,1538,1792,2048,2304,2560,2816,66560,132096,66816,132352,67072,132608,197632,197888,262145,327681,262146,327682,262147,327683,393217,393218,262400,327936,262656,328192,262912,328448,393472,393728,458752,524288,589824,655360,720896};
__device__ inline const unsigned* C1100GradMd::index() { return kC1100GradMd_index; }
}  // namespace qf
