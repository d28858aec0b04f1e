"""Per-lane kernels in Hermite Gaussians (McMurchie and Davidson, J. Comput.
Phys. 26, 218 (1978)): straight-line code of one primitive quartet, for the
gradient (md_grad_source) and for the Fock build (md_fock_source).

With Hermite expansions of the bra and ket pairs, E^{ab}_P and E^{cd}_Q, and
the Hermite Coulomb integrals R_N(P - Q), N = (t, u, v),

    (ab|cd) = sum_P E^{ab}_P sum_Q (-1)^|Q| E^{cd}_Q R_{P+Q},

and the gradient needs only W = sum_abcd Gamma_abcd (ab|cd) of the primitive
quartet as a function of the two pair centres and the two internuclear
vectors R = A - B and S = C - D:

    dW/dA = (alpha/p) dW/dP + dW/dR,   dW/dB = (beta/p) dW/dP - dW/dR,
    dW/dC = -(gamma/q) dW/dP + dW/dS   (W depends on P - Q only).

So a primitive quartet adds nine numbers and no set of contracted derivative
integrals is kept: what the lane holds is R_N up to La+Lb+Lc+Ld+1, the ket's
expansion coefficients and one component pair (a, b) at a time:

    Gamma_cd                       from the density blocks,
    Y_Q   = sum_cd Gamma_cd E^{cd}_Q,
    T_P   = sum_Q Y_Q R_{P+Q}      for P in the support of E^{ab} and its upper neighbours,
    W    += sum_P E_P T_P,  dW/dP_x += sum_P E_P T_{P+1x},  dW/dR_x += sum_P (dE_P/dR_x) T_P,
    Z_Q   = sum_P E_P R_{P+Q},     K_{cd,Q} += Gamma_cd Z_Q;

after all (a, b), dW/dS_x = sum_{cd,Q} (dE^{cd}_Q/dS_x) K_{cd,Q}.  E without
the factor exp(-mu R^2), which the primitive table holds; its derivative is
-2 mu R_x W.

The Fock build takes one component pair (a, b) at a time too: Z_Q as above,
(ab|cd) = sum_Q E^{cd}_Q Z_Q, and each integral goes into J and K at once, per
primitive quartet: no contracted integrals or recursion intermediates are
kept, which in the classes from (dp|pp) up fill more than the registers.

The bra pair is the same in every lane: its products
E_x E_y E_z and (dE_x) E_y E_z come from a table in LDS that the wave fills
once per bra primitive (bra1d and the index list).
"""
from __future__ import annotations

from .gen_eri import add, comps, ncart


def hermites(L):
    return [(t, u, v) for n in range(L + 1) for t in range(n, -1, -1) for u in range(n - t, -1, -1)
            for v in [n - t - u]]


def box(a, b):
    """Support of E^{ab}: t <= a_x + b_x and so on."""
    return [(t, u, v) for t in range(a[0] + b[0] + 1) for u in range(a[1] + b[1] + 1) for v in range(a[2] + b[2] + 1)]


def dbox(a, b, x):
    """Support of dE^{ab}/dR_x (the leading coefficient does not depend on R)."""
    if a[x] + b[x] == 0:
        return []
    return [P for P in box(a, b) if P[x] < a[x] + b[x]]


def sum_of(terms):
    """'+'-joined products as nested fma calls, first term plain."""
    out = None
    for x, y in terms:
        if out is None:
            out = y if x == "1" else "%s * %s" % (x, y)
        else:
            out = "(%s) + %s" % (out, y) if x == "1" else "fma(%s, %s, %s)" % (x, y, out)
    return out or "0.0"


class Table1D:
    """1D expansion coefficients e[i][j][t] and their derivatives d[i][j][t]
    by the internuclear component, i <= la, j <= lb.  sign = -1 carries the
    factor (-1)^t of the ket in the coefficients."""

    def __init__(self, la, lb, prefix, h, X, Y, rx, ry, sign=1):
        self.la, self.lb = la, lb
        self.lines = []
        self.names = {("e", 0, 0, 0): "1"}
        self.order = []
        for i in range(la + 1):
            for j in range(lb + 1):
                if i == j == 0:
                    continue
                src, Z, r = ((i - 1, j), X, rx) if j == 0 else ((i, j - 1), Y, ry)
                for kind in "ed":
                    top = i + j if kind == "e" else i + j - 1
                    for t in range(top + 1):
                        terms = []
                        n = self.names.get((kind,) + src + (t,))
                        if n:
                            terms.append((n, Z))
                        n = self.names.get((kind,) + src + (t - 1,))
                        if n:
                            terms.append((n, h if sign > 0 else "(-%s)" % h))
                        n = self.names.get((kind,) + src + (t + 1,))
                        if n:
                            terms.append(("%d.0" % (sign * (t + 1)), n))
                        if kind == "d":
                            n = self.names.get(("e",) + src + (t,))
                            if n:
                                terms.append((n, r))
                        name = "%s%s%d%d%d" % (prefix, kind, i, j, t)
                        self.lines.append("const double %s = %s;" % (name, sum_of(terms)))
                        self.names[(kind, i, j, t)] = name
                        self.order.append((kind, i, j, t))

    def get(self, kind, i, j, t):
        return self.names.get((kind, i, j, t))


def product(names):
    names = [n for n in names if n != "1"]
    return " * ".join(names) if names else "1"


def r_lines(L):
    """R_N^(0) for |N| <= L from R^(m) = (-2 alpha)^m F_m, as r<tuv>."""
    lines = []
    X = ("PQ[0]", "PQ[1]", "PQ[2]")

    def name(N, m):
        return "r%d%d%d_%d" % (N + (m,))

    lines.append("double am = pref;")
    for m in range(L + 1):
        lines.append("const double %s = F[%d] * am;" % (name((0, 0, 0), m), m))
        if m < L:
            lines.append("am *= m2a;")
    for m in range(L - 1, -1, -1):
        for N in hermites(L - m):
            if N == (0, 0, 0):
                continue
            d = min((k for k in range(3) if N[k]), key=lambda k: (N[k], k))   # a power of one has no second term
            lo = tuple(N[k] - (k == d) for k in range(3))
            terms = [(X[d], name(lo, m + 1))]
            if lo[d]:
                lo2 = tuple(lo[k] - (k == d) for k in range(3))
                terms.append(("%d.0" % lo[d], name(lo2, m + 1)))
            lines.append("const double %s = %s;" % (name(N, m), sum_of(terms)))
    return lines


def rn(N):
    return "r%d%d%d_0" % N


def plus(P, Q):
    return tuple(p + q for p, q in zip(P, Q))


def md_grad_source(name, La, Lb, Lc, Ld):
    ca, cb, cc, cd = comps(La), comps(Lb), comps(Lc), comps(Ld)
    na, nb, nc, nd = len(ca), len(cb), len(cc), len(cd)
    L = La + Lb + Lc + Ld + 1
    bra = Table1D(La, Lb, "b", "h", "X", "Y", "rx", "ry")
    index1 = {("e", 0, 0, 0): 0}
    for k in bra.order:
        index1[k] = len(index1)
    n1 = len(index1)
    prods = {}        # (ix, iy, iz) -> entry of the product table

    def bra_entry(a, b, P, dx=None):
        ids = []
        for x in range(3):
            k = ("d" if x == dx else "e", a[x], b[x], P[x])
            ids.append(index1[k])
        ids = tuple(ids)
        if ids == (0, 0, 0):
            return "1"
        if ids not in prods:
            prods[ids] = len(prods)
        return "E[%d]" % prods[ids]

    lines = list(r_lines(L))
    # ket coefficients of this lane, per direction
    ket = []
    for x in range(3):
        t = Table1D(Lc, Ld, "k%s" % "xyz"[x], "hk", "QC[%d]" % x, "QD[%d]" % x, "rc", "rd", sign=-1)
        lines += t.lines
        ket.append(t)
    kets = [(ic, id_, c, d) for ic, c in enumerate(cc) for id_, d in enumerate(cd)]
    for ic, id_, c, d in kets:
        for Q in box(c, d):
            p = product([ket[x].get("e", c[x], d[x], Q[x]) for x in range(3)])
            if p != "1":
                lines.append("const double k%d_%d_%d%d%d = %s;" % ((ic, id_) + Q + (p,)))

    def ke(ic, id_, c, d, Q):
        return "1" if product([ket[x].get("e", c[x], d[x], Q[x]) for x in range(3)]) == "1" else \
            "k%d_%d_%d%d%d" % ((ic, id_) + Q)

    Qall = sorted({Q for _, _, c, d in kets for Q in box(c, d)}, key=lambda q: (sum(q), q))
    KQ = {(ic, id_): sorted({Q for x in range(3) for Q in dbox(c, d, x)}, key=lambda q: (sum(q), q))
          for ic, id_, c, d in kets}
    Qz = sorted({Q for qs in KQ.values() for Q in qs}, key=lambda q: (sum(q), q))
    for (ic, id_), qs in KQ.items():
        for Q in qs:
            lines.append("double K%d_%d_%d%d%d = 0.0;" % ((ic, id_) + Q))
    lines.append("double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;")
    rows = na * (nc + nd) > 12       # many a rows: read again per quartet instead of kept in registers
    if rows:
        lines += ["QF_OPAQUE(oc);", "QF_OPAQUE(od);"]
    for ia, a in enumerate(ca):
        lines.append("{")
        for ic in range(nc):
            lines.append("  const double ac%d = P[oc + %d * n + %d] * (kCons[%d][%d] * kCons[%d][%d]);"
                         % (ic, ia, ic, La, ia, Lc, ic))
        for id_ in range(nd):
            lines.append("  const double ad%d = P[od + %d * n + %d] * (kCons[%d][%d] * kCons[%d][%d]);"
                         % (id_, ia, id_, La, ia, Ld, id_))
        for ib, b in enumerate(cb):
            lines.append("  {")
            o = "    "
            lines.append(o + "const double ab = Pab[%d * n + %d] * (kCons[%d][%d] * kCons[%d][%d]);"
                         % (ia, ib, La, ia, Lb, ib))
            for ic, id_, c, d in kets:
                lines.append(o + "const double g%d_%d = fma(-ad%d, Dbc[%d], fma(-ac%d, Dbd[%d], ab * Dcd[%d]));"
                             % (ic, id_, id_, ib * nc + ic, ic, ib * nd + id_, ic * nd + id_))
            for Q in Qall:
                lines.append(o + "const double y%d%d%d = %s;" % (Q + (sum_of(
                    [(ke(ic, id_, c, d, Q), "g%d_%d" % (ic, id_)) for ic, id_, c, d in kets if Q in box(c, d)]),)))
            B = box(a, b)
            ext = sorted(set(B) | {add(P, x) for P in B for x in range(3)}, key=lambda q: (sum(q), q))
            for P in ext:
                lines.append(o + "const double t%d%d%d = %s;" % (P + (sum_of(
                    [("y%d%d%d" % Q, rn(plus(P, Q))) for Q in Qall]),)))
            for k, P in enumerate(B):
                e = bra_entry(a, b, P)
                if e != "1":
                    lines.append(o + "const double e%d = %s;" % (k, e))
            for target, x in (("w", None), ("px", 0), ("py", 1), ("pz", 2)):
                s = target
                for k, P in enumerate(B):
                    T = "t%d%d%d" % (P if x is None else add(P, x))
                    s = "%s + %s" % (T, s) if bra_entry(a, b, P) == "1" else "fma(e%d, %s, %s)" % (k, T, s)
                lines.append(o + "%s = %s;" % (target, s))
            for x in range(3):
                D = dbox(a, b, x)
                if D:
                    s = "s" + "xyz"[x]
                    for P in D:
                        s = "fma(%s, t%d%d%d, %s)" % ((bra_entry(a, b, P, x),) + P + (s,))
                    lines.append(o + "s%s = %s;" % ("xyz"[x], s))
            for Q in Qz:
                lines.append(o + "const double z%d%d%d = %s;" % (Q + (sum_of(
                    [("1" if bra_entry(a, b, P) == "1" else "e%d" % k, rn(plus(P, Q))) for k, P in enumerate(B)]),)))
            for (ic, id_), qs in KQ.items():
                for Q in qs:
                    lines.append(o + "K%d_%d_%d%d%d = fma(g%d_%d, z%d%d%d, K%d_%d_%d%d%d);"
                                 % ((ic, id_) + Q + (ic, id_) + Q + (ic, id_) + Q))
            lines.append("  }")
        lines.append("}")
    lines += ["W = w;", "gP[0] = px; gP[1] = py; gP[2] = pz;", "gR[0] = sx; gR[1] = sy; gR[2] = sz;"]
    for x in range(3):
        terms = []
        for ic, id_, c, d in kets:
            for Q in dbox(c, d, x):
                p = product([ket[y].get("d" if y == x else "e", c[y], d[y], Q[y]) for y in range(3)])
                terms.append((p if "*" not in p else "(%s)" % p, "K%d_%d_%d%d%d" % ((ic, id_) + Q)))
        lines.append("gS[%d] = %s;" % (x, sum_of(terms)))
    nR, nK, nKQ = len(hermites(L)), sum(len(box(c, d)) for _, _, c, d in kets), sum(map(len, KQ.values()))
    regs = 2 * (nR + nK + nKQ + nc * nd + nb * (nc + nd) + 2 * len(Qall) + 45)
    waves = 1 if regs > 190 else 2 if regs > 130 else 3 if regs > 104 else 4
    g = name + "GradMd"
    src = ["// (%s%s|%s%s): %d Hermite Coulomb integrals, %d bra products"
           % ("spd"[La], "spd"[Lb], "spd"[Lc], "spd"[Ld], nR, len(prods)),
           "struct %s {" % g,
           "  static constexpr int La = %d, Lb = %d, Lc = %d, Ld = %d, L = %d;" % (La, Lb, Lc, Ld, L),
           "  static constexpr int N1 = %d, NE = %d;   // 1D entries per direction, product table" % (n1, len(prods)),
           "  static constexpr int MIN_WAVES = %d;      // waves per SIMD the register budget targets" % waves,
           "  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16",
           "  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p",
           "  template <class T>",
           "  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry,"
           " T out) {"]
    src += ["    " + l for l in bra.lines]
    src += ["    out[0] = 1.0;"] + ["    out[%d] = %s;" % (index1[k], bra.names[k]) for k in bra.order]
    src += ["  }",
            "  // Dcd with 2 cons, Dbc and Dbd with hyb/2 cons; oc, od: first elements of the a-c and a-d blocks of P",
            "  template <class ET, class PT, class PU>",
            "  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a,"
            " const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd,"
            " const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[%d],"
            " const double (&Dbc)[%d], const double (&Dbd)[%d], double& W, double (&gP)[3], double (&gR)[3],"
            " double (&gS)[3]) {" % (nc * nd, nb * nc, nb * nd)]
    src += ["    " + l for l in lines]
    src += ["  }", "};"]
    idx = sorted(prods, key=prods.get)
    src += ["__device__ const unsigned k%s_index[%d] = {%s};"
            % (g, max(1, len(idx)), ",".join(str(x | y << 8 | z << 16) for x, y, z in idx) or "0"),
            "__device__ inline const unsigned* %s::index() { return k%s_index; }" % (g, g)]
    return g, "\n".join(src) + "\n"


def md_fock_source(name, La, Lb, Lc, Ld):
    """Fock digestion of one primitive quartet.  ``out`` takes the sums that
    leave the lane: jab_add(k, v) for element k of J_ab, rows(ia, c, d) for row ia
    of the a-c and a-d exchange blocks."""
    ca, cb, cc, cd = comps(La), comps(Lb), comps(Lc), comps(Ld)
    nb, nc, nd = len(cb), len(cc), len(cd)
    L = La + Lb + Lc + Ld
    bra = Table1D(La, Lb, "b", "h", "X", "Y", "0.0", "0.0")
    order = [k for k in bra.order if k[0] == "e"]
    index1 = {("e", 0, 0, 0): 0}
    for k in order:
        index1[k] = len(index1)
    n1 = len(index1)
    prods = {}

    def bra_entry(a, b, P):
        ids = tuple(index1[("e", a[x], b[x], P[x])] for x in range(3))
        if ids == (0, 0, 0):
            return "1"
        if ids not in prods:
            prods[ids] = len(prods)
        return "E[%d]" % prods[ids]

    lines = list(r_lines(L))
    ket = []
    for x in range(3):
        t = Table1D(Lc, Ld, "k%s" % "xyz"[x], "hk", "QC[%d]" % x, "QD[%d]" % x, "0.0", "0.0", sign=-1)
        lines += [l for l in t.lines if l.startswith("const double k%se" % "xyz"[x])]
        ket.append(t)
    kets = [(ic, id_, c, d) for ic, c in enumerate(cc) for id_, d in enumerate(cd)]
    for ic, id_, c, d in kets:
        for Q in box(c, d):
            p = product([ket[x].get("e", c[x], d[x], Q[x]) for x in range(3)])
            lines.append("const double k%d_%d_%d%d%d = %s(kCons[%d][%d] * kCons[%d][%d]);"
                         % ((ic, id_) + Q + ("" if p == "1" else p + " * ", Lc, ic, Ld, id_)))
    Qall = sorted({Q for _, _, c, d in kets for Q in box(c, d)}, key=lambda q: (sum(q), q))
    lines += ["QF_OPAQUE(oc);", "QF_OPAQUE(od);"]
    for ia, a in enumerate(ca):
        lines.append("{")
        for ic in range(nc):
            lines.append("  const double ac%d = P[oc + %d * n + %d] * kCons[%d][%d];" % (ic, ia, ic, La, ia))
        for id_ in range(nd):
            lines.append("  const double ad%d = P[od + %d * n + %d] * kCons[%d][%d];" % (id_, ia, id_, La, ia))
        for ib, b in enumerate(cb):
            lines.append("  {")
            o = "    "
            lines.append(o + "const double ab = Pab[%d * n + %d] * (kCons[%d][%d] * kCons[%d][%d]);"
                         % (ia, ib, La, ia, Lb, ib))
            B = box(a, b)
            for k, P in enumerate(B):
                e = bra_entry(a, b, P)
                if e != "1":
                    lines.append(o + "const double e%d = %s;" % (k, e))
            for Q in Qall:
                lines.append(o + "const double z%d%d%d = %s;" % (Q + (sum_of(
                    [("1" if bra_entry(a, b, P) == "1" else "e%d" % k, rn(plus(P, Q))) for k, P in enumerate(B)]),)))
            lines.append(o + "double j = 0.0;")
            for ic, id_, c, d in kets:
                v = sum_of([("k%d_%d_%d%d%d" % ((ic, id_) + Q), "z%d%d%d" % Q) for Q in box(c, d)])
                lines.append(o + "{")
                lines.append(o + "  const double v = %s;" % v)
                lines.append(o + "  j = fma(Dcd[%d], v, j);" % (ic * nd + id_))
                lines.append(o + "  Jcd[%d] = fma(ab, v, Jcd[%d]);" % (ic * nd + id_, ic * nd + id_))
                lines.append(o + "  Kac[%d] = fma(Dbd[%d], v, Kac[%d]);" % (ia * nc + ic, ib * nd + id_, ia * nc + ic))
                lines.append(o + "  Kad[%d] = fma(Dbc[%d], v, Kad[%d]);" % (ia * nd + id_, ib * nc + ic, ia * nd + id_))
                lines.append(o + "  Kbc[%d] = fma(ad%d, v, Kbc[%d]);" % (ib * nc + ic, id_, ib * nc + ic))
                lines.append(o + "  Kbd[%d] = fma(ac%d, v, Kbd[%d]);" % (ib * nd + id_, ic, ib * nd + id_))
                lines.append(o + "}")
            lines.append(o + "Jab[%d] += j;" % (ia * nb + ib))
            lines.append("  }")
        lines.append("}")
    g = name + "Md"
    src = ["// (%s%s|%s%s): %d Hermite Coulomb integrals, %d bra products"
           % ("spd"[La], "spd"[Lb], "spd"[Lc], "spd"[Ld], len(hermites(L)), len(prods)),
           "struct %s {" % g,
           "  static constexpr int La = %d, Lb = %d, Lc = %d, Ld = %d, L = %d;" % (La, Lb, Lc, Ld, L),
           "  static constexpr int N1 = %d, NE = %d;   // 1D entries per direction, product table" % (n1, len(prods)),
           "  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16",
           "  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p",
           "  template <class T>",
           "  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, T out) {"]
    src += ["    " + l for l in bra.lines if l.startswith("const double be")]
    src += ["    out[0] = 1.0;"] + ["    out[%d] = %s;" % (index1[k], bra.names[k]) for k in order]
    src += ["  }",
            "  // Dbc and Dbd with the cons of b; oc, od: first elements of the a-c and a-d blocks of P",
            "  template <class ET, class PT, class PU>",
            "  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a,"
            " const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, const ET E,"
            " const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[%d], const double (&Dbc)[%d],"
            " const double (&Dbd)[%d], double (&Jcd)[%d], double (&Kbc)[%d], double (&Kbd)[%d], double (&Jab)[%d], double (&Kac)[%d],"
            " double (&Kad)[%d]) {"
            % (nc * nd, nb * nc, nb * nd, nc * nd, nb * nc, nb * nd, len(ca) * nb, len(ca) * nc, len(ca) * nd)]
    src += ["    " + l for l in lines]
    src += ["  }", "};"]
    idx = sorted(prods, key=prods.get)
    src += ["__device__ const unsigned k%s_index[%d] = {%s};"
            % (g, max(1, len(idx)), ",".join(str(x | y << 8 | z << 16) for x, y, z in idx) or "0"),
            "__device__ inline const unsigned* %s::index() { return k%s_index; }" % (g, g)]
    return g, "\n".join(src) + "\n"
