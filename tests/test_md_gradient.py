"""The Hermite-Gaussian gradient code of one primitive quartet (gen_md.py),
compiled for the CPU: its energy W against the integrals of
tests/md_reference.py and its gradient against finite differences of W, for
every class that has a per-lane gradient kernel.  Four-point differences of step 1e-3 carry an
error of about h^4 = 1e-12 of the function's scale plus 1e-13 of rounding."""
import os
import subprocess

import numpy as np
import pytest

from quick_amd.codegen import gen_grad as GG
from quick_amd.codegen import gen_md as GM
from quick_amd.codegen.gen_eri import comps
from tests import md_reference as MD

CLASSES = [c for c in GG.grad_classes() if GG.has_lane_grad(*c)]

HARNESS = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#define __host__
#define __device__
#define __forceinline__ inline
#define QF_OPAQUE(x)
static const double kCons[3][6] = {{1}, {1, 1, 1}, {1, CD, 1, CD, CD, 1}};
static double Pm[40 * 40];
static void boys(double T, int M, double* F)
{
    double term = 1.0 / (2 * M + 1), s = term;
    for (int k = 1; k < 400 && term > 1e-18; ++k) s += term *= 2 * T / (2 * M + 1 + 2 * k);
    F[M] = exp(-T) * s;
    for (int m = M - 1; m >= 0; --m) F[m] = (2 * T * F[m + 1] + exp(-T)) / (2 * m + 1);
}
template <class C>
double eval(const double (&X)[4][3], const double (&e)[4], double (&g)[12])
{
    const double p = e[0] + e[1], q = e[2] + e[3], mu = e[0] * e[1] / p, nu = e[2] * e[3] / q, al = p * q / (p + q);
    double P[3], Q[3], PQ[3], QC[3], QD[3], R[3], S[3], r2 = 0, R2 = 0, S2 = 0;
    for (int d = 0; d < 3; ++d) {
        P[d] = (e[0] * X[0][d] + e[1] * X[1][d]) / p;
        Q[d] = (e[2] * X[2][d] + e[3] * X[3][d]) / q;
        PQ[d] = P[d] - Q[d]; QC[d] = Q[d] - X[2][d]; QD[d] = Q[d] - X[3][d];
        R[d] = X[0][d] - X[1][d]; S[d] = X[2][d] - X[3][d];
        r2 += PQ[d] * PQ[d]; R2 += R[d] * R[d]; S2 += S[d] * S[d];
    }
    double F[C::L + 1];
    boys(al * r2, C::L, F);
    double tab[3 * C::N1 + C::NE + 1];
    for (int d = 0; d < 3; ++d)
        C::bra1d(P[d] - X[0][d], P[d] - X[1][d], 0.5 / p, -e[1] / p, e[0] / p, tab + d * C::N1);
    for (int x = 0; x < C::NE; ++x) {
        const unsigned id = C::index()[x];
        tab[3 * C::N1 + x] = tab[id & 255] * tab[C::N1 + ((id >> 8) & 255)] * tab[2 * C::N1 + (id >> 16)];
    }
    const int nb = (C::Lb + 1) * (C::Lb + 2) / 2, nc = (C::Lc + 1) * (C::Lc + 2) / 2, nd = (C::Ld + 1) * (C::Ld + 2) / 2;
    const int n = 40, fb = 10, fc = 20, fd = 30;
    double Dcd[nc * nd], Dbc[nb * nc], Dbd[nb * nd], W, gP[3], gR[3], gS[3];
    for (int c = 0; c < nc; ++c)
        for (int d = 0; d < nd; ++d) Dcd[c * nd + d] = 2 * Pm[(fc + c) * n + fd + d] * kCons[C::Lc][c] * kCons[C::Ld][d];
    for (int b = 0; b < nb; ++b) {
        for (int c = 0; c < nc; ++c) Dbc[b * nc + c] = 0.5 * Pm[(fb + b) * n + fc + c] * kCons[C::Lb][b] * kCons[C::Lc][c];
        for (int d = 0; d < nd; ++d) Dbd[b * nd + d] = 0.5 * Pm[(fb + b) * n + fd + d] * kCons[C::Lb][b] * kCons[C::Ld][d];
    }
    C::prim(F, 2 * pow(M_PI, 2.5) * exp(-mu * R2 - nu * S2) / (p * q * sqrt(p + q)), -2 * al, PQ, QC, QD, 0.5 / q,
            -e[3] / q, e[2] / q, (const double*)(tab + 3 * C::N1), (const double*)Pm + fb, (const double*)Pm, n, fc, fd,
            Dcd, Dbc, Dbd, W, gP, gR, gS);
    for (int d = 0; d < 3; ++d) {
        const double r = gR[d] - 2 * mu * R[d] * W, s = gS[d] - 2 * nu * S[d] * W;
        g[d] = e[0] / p * gP[d] + r;
        g[3 + d] = e[1] / p * gP[d] - r;
        g[6 + d] = -e[2] / q * gP[d] + s;
        g[9 + d] = -e[3] / q * gP[d] - s;
    }
    return W;
}
template <class C>
void show()
{
    double X[4][3], e[4], g[12], t[12];
    FILE* f = fopen(INPUT, "rb");
    if (!f || fread(X, 8, 12, f) != 12 || fread(e, 8, 4, f) != 4 || fread(Pm, 8, 1600, f) != 1600) exit(1);
    fclose(f);
    printf("%.17g", eval<C>(X, e, g));
    for (double v : g) printf(" %.17g", v);
    for (int k = 0; k < 12; ++k) {
        double d[2];
        for (int w = 1; w <= 2; ++w) {
            const double h = 1e-3 * w, x = X[k / 3][k % 3];
            X[k / 3][k % 3] = x + h;
            const double a = eval<C>(X, e, t);
            X[k / 3][k % 3] = x - h;
            d[w - 1] = (a - eval<C>(X, e, t)) / (2 * h);
            X[k / 3][k % 3] = x;
        }
        printf(" %.17g", (4 * d[0] - d[1]) / 3);
    }
    printf("\n");
}
"""


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("md")
    rng = np.random.default_rng(11)
    X, e, P = rng.uniform(0, 1.5, (4, 3)), rng.uniform(0.3, 1.3, 4), rng.uniform(-0.5, 0.5, (40, 40))
    inp = os.path.join(tmp, "in.bin")
    with open(inp, "wb") as fh:
        for a in (X, e, P):
            fh.write(np.ascontiguousarray(a).tobytes())
    src = HARNESS.replace("INPUT", '"%s"' % inp).replace("CD", "1.7320508075688772935")
    calls = ""
    for c in CLASSES:
        g, s = GM.md_grad_source("C%d%d%d%d" % c, *c)
        src += s
        calls += "show<%s>();" % g
    path = os.path.join(tmp, "md.cpp")
    with open(path, "w") as fh:
        fh.write(src + "int main() { %s }\n" % calls)
    exe = os.path.join(tmp, "md")
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-o", exe, path], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split("\n")
    return X, e, P, {c: np.array(list(map(float, line.split()))) for c, line in zip(CLASSES, out)}


def energy(cls, X, e, P):
    """sum Gamma (ab|cd) over unnormalised primitives with their cons factors (hyb = 1)."""
    shells = [(L, X[k], [e[k]], [1.0]) for k, L in enumerate(cls)]
    na, nb, nc, nd = (len(comps(L)) for L in cls)
    ab, cd = P[:na, 10:10 + nb], P[20:20 + nc, 30:30 + nd]
    ac, ad, bc, bd = P[:na, 20:20 + nc], P[:na, 30:30 + nd], P[10:10 + nb, 20:20 + nc], P[10:10 + nb, 30:30 + nd]
    gam = 2 * np.einsum("ab,cd->abcd", ab, cd) - 0.5 * (np.einsum("ac,bd->abcd", ac, bd) +
                                                       np.einsum("ad,bc->abcd", ad, bc))
    return float(np.sum(gam * MD.shell_block(shells, MD.boys_exact)))


@pytest.mark.parametrize("cls", CLASSES, ids=lambda c: "%d%d%d%d" % c)
def test_md_gradient_of_a_primitive_quartet(cls, results):
    X, e, P, out = results
    r = out[cls]
    W, g, num = r[0], r[1:13], r[13:25]
    scale = np.abs(g).max()
    assert np.abs(g - num).max() <= 1e-10 * max(1.0, scale)
    assert np.abs(g.reshape(4, 3).sum(0)).max() <= 1e-12 * max(1.0, scale)    # translational invariance
    assert abs(W - energy(cls, X, e, P)) <= 1e-12 * max(1.0, abs(W))
