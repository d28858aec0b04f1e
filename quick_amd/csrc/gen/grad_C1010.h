// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C1010Grad {
  static constexpr int La = 1, Lb = 0, Lc = 1, Ld = 0, L = 3;
  static constexpr int NACC = 69, NV = 81, NLV = 3, NX = 69, NH = 69, NLH = 1, NI = 9;
  static constexpr int ZS = 69, SINK = 70, CF = 218, DM = 258, LDS = 280;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 71, OAM = 89, OBP = 92, OBM = -1, OCP = 119, OCM = 137;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 535, QUARTET_FLOP = 468;
  static constexpr unsigned short FSLOT[4] = {140,141,142,143};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC1010Grad_vrr[81] = {{142,143,69,69,69,144,65535,2},{142,143,69,69,69,145,65535,1},{142,143,69,69,69,146,65535,0},{141,142,69,69,69,147,65535,2},{141,142,69,69,69,148,65535,1},{141,142,69,69,69,149,65535,0},{140,141,69,69,69,150,65535,2},{140,141,69,69,69,151,65535,1},{140,141,69,69,69,152,65535,0},{141,142,69,69,69,153,65535,5},{141,142,69,69,69,154,65535,4},{141,142,69,69,69,155,65535,3},{140,141,69,69,69,156,65535,5},{140,141,69,69,69,157,65535,4},{140,141,69,69,69,158,65535,3},{147,144,141,142,69,143,65535,18},{147,144,69,69,69,159,65535,1},{148,145,141,142,69,160,65535,17},{147,144,69,69,69,161,65535,0},{148,145,69,69,69,162,65535,0},{149,146,141,142,69,163,65535,16},{150,147,140,141,69,164,65535,18},{150,147,69,69,69,165,65535,1},{151,148,140,141,69,166,65535,17},{150,147,69,69,69,167,65535,0},{151,148,69,69,69,168,65535,0},{152,149,140,141,69,169,65535,16},{147,144,69,69,142,170,65535,261},{147,144,69,69,69,171,65535,4},{147,144,69,69,69,172,65535,3},{148,145,69,69,69,173,65535,5},{148,145,69,69,142,174,65535,260},{148,145,69,69,69,175,65535,3},{149,146,69,69,69,176,65535,5},{149,146,69,69,69,177,65535,4},{149,146,69,69,142,178,65535,259},{150,147,69,69,141,179,65535,261},{150,147,69,69,69,180,65535,4},{150,147,69,69,69,181,65535,3},{151,148,69,69,69,182,65535,5},{151,148,69,69,141,183,65535,260},{151,148,69,69,69,184,65535,3},{152,149,69,69,69,185,65535,5},{152,149,69,69,69,186,65535,4},{152,149,69,69,141,187,65535,259},{164,143,69,69,147,140,65535,517},{164,143,69,69,69,141,65535,4},{164,143,69,69,69,142,65535,3},{165,159,69,69,148,144,65535,261},{165,159,69,69,147,145,65535,260},{165,159,69,69,69,146,65535,3},{166,160,69,69,69,188,65535,5},{166,160,69,69,148,189,65535,516},{166,160,69,69,69,190,65535,3},{167,161,69,69,149,191,65535,261},{167,161,69,69,69,192,65535,4},{167,161,69,69,147,193,65535,259},{168,162,69,69,69,194,65535,5},{168,162,69,69,149,195,65535,260},{168,162,69,69,148,196,65535,259},{169,163,69,69,69,197,65535,5},{169,163,69,69,69,198,65535,4},{169,163,69,69,149,199,65535,515},{179,170,150,147,153,200,65535,277},{179,170,69,69,69,201,65535,4},{180,171,150,147,69,202,65535,20},{179,170,69,69,69,203,65535,3},{180,171,69,69,69,204,65535,3},{181,172,150,147,69,205,65535,19},{182,173,151,148,69,206,65535,21},{183,174,69,69,69,207,65535,5},{183,174,151,148,154,208,65535,276},{182,173,69,69,69,209,65535,3},{183,174,69,69,69,210,65535,3},{184,175,151,148,69,211,65535,19},{185,176,152,149,69,212,65535,21},{185,176,69,69,69,213,65535,4},{186,177,152,149,69,214,65535,20},{187,178,69,69,69,215,65535,5},{187,178,69,69,69,216,65535,4},{187,178,152,149,155,217,65535,275}};
__device__ const int kC1010Grad_vlev[4] = {0,15,45,81};
__device__ const GradAcc kC1010Grad_acc[69] = {{158,0,0},{157,1,0},{156,2,0},{152,3,0},{151,4,0},{150,5,0},{199,6,1},{198,7,1},{197,8,1},{196,9,1},{195,10,1},{194,11,1},{190,12,1},{189,13,1},{188,14,1},{193,15,1},{192,16,1},{191,17,1},{146,18,1},{145,19,1},{144,20,1},{142,21,1},{141,22,1},{140,23,1},{187,24,2},{186,25,2},{185,26,2},{184,27,2},{183,28,2},{182,29,2},{181,30,2},{180,31,2},{179,32,2},{199,33,2},{198,34,2},{197,35,2},{196,36,2},{195,37,2},{194,38,2},{190,39,2},{189,40,2},{188,41,2},{193,42,2},{192,43,2},{191,44,2},{146,45,2},{145,46,2},{144,47,2},{142,48,2},{141,49,2},{140,50,2},{217,51,3},{216,52,3},{214,53,3},{215,54,3},{213,55,3},{212,56,3},{211,57,3},{210,58,3},{208,59,3},{209,60,3},{207,61,3},{206,62,3},{205,63,3},{204,64,3},{202,65,3},{203,66,3},{201,67,3},{200,68,3}};
__device__ const CoopHNode kC1010Grad_hrr[69] = {{118,50,32,5},{117,49,31,5},{116,48,30,5},{115,47,32,4},{114,46,31,4},{113,45,30,4},{112,44,32,3},{111,43,31,3},{110,42,30,3},{109,47,29,5},{108,46,28,5},{107,45,27,5},{106,41,29,4},{105,40,28,4},{104,39,27,4},{103,38,29,3},{102,37,28,3},{101,36,27,3},{100,44,26,5},{99,43,25,5},{98,42,24,5},{97,38,26,4},{96,37,25,4},{95,36,24,4},{94,35,26,3},{93,34,25,3},{92,33,24,3},{89,0,69,0},{90,1,69,0},{91,2,69,0},{71,6,69,0},{72,7,69,0},{81,16,69,0},{82,17,69,0},{83,18,69,0},{84,19,69,0},{85,20,69,0},{86,21,69,0},{87,22,69,0},{88,23,69,0},{73,8,69,0},{74,9,69,0},{75,10,69,0},{76,11,69,0},{77,12,69,0},{78,13,69,0},{79,14,69,0},{80,15,69,0},{137,3,69,0},{138,4,69,0},{139,5,69,0},{119,51,69,0},{120,52,69,0},{129,61,69,0},{130,62,69,0},{131,63,69,0},{132,64,69,0},{133,65,69,0},{134,66,69,0},{135,67,69,0},{136,68,69,0},{121,53,69,0},{122,54,69,0},{123,55,69,0},{124,56,69,0},{125,57,69,0},{126,58,69,0},{127,59,69,0},{128,60,69,0}};
__device__ const int kC1010Grad_hlev[2] = {0,69};
__device__ inline const CoopVNode* C1010Grad::vrr() { return kC1010Grad_vrr; }
__device__ inline const int* C1010Grad::vlev() { return kC1010Grad_vlev; }
__device__ inline const GradAcc* C1010Grad::acc() { return kC1010Grad_acc; }
__device__ inline const CoopHNode* C1010Grad::hrr() { return kC1010Grad_hrr; }
__device__ inline const int* C1010Grad::hlev() { return kC1010Grad_hlev; }
// (ps|ps): 20 Hermite Coulomb integrals, 9 bra products
struct C1010GradMd {
  static constexpr int La = 1, Lb = 0, Lc = 1, Ld = 0, L = 3;
  static constexpr int N1 = 4, NE = 9;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 2;      // waves per SIMD the register budget targets
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
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[3], const double (&Dbc)[3], const double (&Dbd)[1], double& W, double (&gP)[3], double (&gR)[3], double (&gS)[3]) {
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
    const double kxe100 = QC[0];
    const double kxe101 = (-hk);
    const double kxd100 = rc;
    const double kye100 = QC[1];
    const double kye101 = (-hk);
    const double kyd100 = rc;
    const double kze100 = QC[2];
    const double kze101 = (-hk);
    const double kzd100 = rc;
    const double k0_0_000 = kxe100;
    const double k0_0_100 = kxe101;
    const double k1_0_000 = kye100;
    const double k1_0_010 = kye101;
    const double k2_0_000 = kze100;
    const double k2_0_001 = kze101;
    double K0_0_000 = 0.0;
    double K1_0_000 = 0.0;
    double K2_0_000 = 0.0;
    double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    {
      const double ac0 = P[oc + 0 * n + 0] * (kCons[1][0] * kCons[1][0]);
      const double ac1 = P[oc + 0 * n + 1] * (kCons[1][0] * kCons[1][1]);
      const double ac2 = P[oc + 0 * n + 2] * (kCons[1][0] * kCons[1][2]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[1][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[1][0] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t200 = fma(y100, r300_0, fma(y010, r210_0, fma(y001, r201_0, y000 * r200_0)));
        const double e0 = E[0];
        const double e1 = E[1];
        w = fma(e1, t100, fma(e0, t000, w));
        px = fma(e1, t200, fma(e0, t100, px));
        py = fma(e1, t110, fma(e0, t010, py));
        pz = fma(e1, t101, fma(e0, t001, pz));
        sx = fma(E[2], t000, sx);
        const double z000 = fma(e1, r100_0, e0 * r000_0);
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * (kCons[1][1] * kCons[1][0]);
      const double ac1 = P[oc + 1 * n + 1] * (kCons[1][1] * kCons[1][1]);
      const double ac2 = P[oc + 1 * n + 2] * (kCons[1][1] * kCons[1][2]);
      const double ad0 = P[od + 1 * n + 0] * (kCons[1][1] * kCons[0][0]);
      {
        const double ab = Pab[1 * n + 0] * (kCons[1][1] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t020 = fma(y100, r120_0, fma(y010, r030_0, fma(y001, r021_0, y000 * r020_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double e0 = E[3];
        const double e1 = E[4];
        w = fma(e1, t010, fma(e0, t000, w));
        px = fma(e1, t110, fma(e0, t100, px));
        py = fma(e1, t020, fma(e0, t010, py));
        pz = fma(e1, t011, fma(e0, t001, pz));
        sy = fma(E[5], t000, sy);
        const double z000 = fma(e1, r010_0, e0 * r000_0);
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * (kCons[1][2] * kCons[1][0]);
      const double ac1 = P[oc + 2 * n + 1] * (kCons[1][2] * kCons[1][1]);
      const double ac2 = P[oc + 2 * n + 2] * (kCons[1][2] * kCons[1][2]);
      const double ad0 = P[od + 2 * n + 0] * (kCons[1][2] * kCons[0][0]);
      {
        const double ab = Pab[2 * n + 0] * (kCons[1][2] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t002 = fma(y100, r102_0, fma(y010, r012_0, fma(y001, r003_0, y000 * r002_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double e0 = E[6];
        const double e1 = E[7];
        w = fma(e1, t001, fma(e0, t000, w));
        px = fma(e1, t101, fma(e0, t100, px));
        py = fma(e1, t011, fma(e0, t010, py));
        pz = fma(e1, t002, fma(e0, t001, pz));
        sz = fma(E[8], t000, sz);
        const double z000 = fma(e1, r001_0, e0 * r000_0);
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    W = w;
    gP[0] = px; gP[1] = py; gP[2] = pz;
    gR[0] = sx; gR[1] = sy; gR[2] = sz;
    gS[0] = kxd100 * K0_0_000;
    gS[1] = kyd100 * K1_0_000;
    gS[2] = kzd100 * K2_0_000;
  }
};
__device__ const unsigned kC1010GradMd_index[9] = {1,2,3,256,512,768,65536,131072,196608};
__device__ inline const unsigned* C1010GradMd::index() { return kC1010GradMd_index; }
}  // namespace qf
