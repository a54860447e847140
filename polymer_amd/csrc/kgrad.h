// kgrad.h -- two-electron part of the nuclear gradient (the quantity
// FOURINDEX_ERI_GRADIENT accumulates, src/pfourindexgradient.f90:1334-1420):
//
//   dE2/dR = sum over shell quartets (ab|cd) of sum_{mu nu lam sig}
//            Gamma(mu nu lam sig) d(mu nu|lam sig)/dR,
//   Gamma  = f [4 D_mu,nu D_lam,sig - x (D_mu,lam D_nu,sig + D_mu,sig D_nu,lam)]
//
// over the symmetry-unique quartets (a >= b, c >= d, pair ab >= pair cd;
// f = 1/2 for each of a == b, c == d, ab == cd), with D the density in this
// library's contracted Cartesian basis and x the exchange scale.  That is
// E2 = 1/2 sum D D (mu nu|lam sig) - x/4 sum D D (mu lam|nu sig) over all
// function quadruples, differentiated at fixed D.  The derivative with
// respect to centre A of a primitive Cartesian Gaussian is
// 2 alpha [a + 1] - a_x [a - 1] (componentwise), taken on A, B and C; D's
// follows from translational invariance, -(dA + dB + dC).
//
// Integrals by Rys quadrature with the library's node tables (rys.h): for
// each primitive quartet and each of the n = (L + 1) / 2 + 1 roots, the
// one-dimensional factors G(i, k) of the two-electron recursion, then the
// horizontal transfers to I(i, j, k, l) for i + j <= La + Lb + 1 and
// k + l <= Lc + Ld + 1 -- one level above the quartet, for the derivatives --
// and from them, per axis, the factors v and their derivatives on A, B, C.
//
// The gradient is linear in the integrals, so the work of a quartet can be
// cut anywhere and each piece added to the per-atom sums by itself.  The unit
// is a primitive quartet, or one root of one for the classes of 36 integrals
// and more; S lanes share a quartet and take every S-th unit, S such that a
// lane has about `grain` units (GradChunks).  One lane per quartet left the
// launches at the length of their longest quartet (6561 primitive quartets
// of two oxygen 1s pairs of cc-pVDZ: 5 ms) and the d classes, few quartets of
// much work, on a fraction of the chip ((dp|dp) of (H2O)6 20 ms on 160
// wavefronts): 110 ms for (H2O)6 cc-pVDZ, now 5.7 (98 -> 0.6 for one water,
// 296 -> 114 for sixteen).  Primitive pairs come from the context's table (no exponentials
// or divisions here).  Quartets with Q_ab Q_cd, or Q_ab Q_cd times the
// largest |Gamma|, below the threshold are skipped; per-atom sums in LDS, one
// global atomic per atom coordinate per block.  The same code runs on the
// host (polyeri_grad_host) for the CPU tests.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "eri_kernels.h"
#include "rys.h"

namespace {

#define GRAD_LMAX 2                      // highest shell L of the library's basis (d)
#define GMAX (2 * GRAD_LMAX + 2)         // G(i, k): i, k <= 2 LMAX + 1
#define IMAX (GRAD_LMAX + 2)             // I(i, j, k, l): i, j, k <= LMAX + 1
#define LMAXD (GRAD_LMAX + 1)            //                l <= LMAX

struct RysTabs {
    const double* tab[RYS_NMAX + 1];
    const double* herm[RYS_NMAX + 1];
};

__device__ const double g_gtab1[] = RYS_TABLE_1;
__device__ const double g_gtab2[] = RYS_TABLE_2;
__device__ const double g_gtab3[] = RYS_TABLE_3;
__device__ const double g_gtab4[] = RYS_TABLE_4;
__device__ const double g_gtab5[] = RYS_TABLE_5;
__device__ const double g_gherm1[] = RYS_HERM_1;
__device__ const double g_gherm2[] = RYS_HERM_2;
__device__ const double g_gherm3[] = RYS_HERM_3;
__device__ const double g_gherm4[] = RYS_HERM_4;
__device__ const double g_gherm5[] = RYS_HERM_5;
static const double h_gtab1[] = RYS_TABLE_1, h_gtab2[] = RYS_TABLE_2, h_gtab3[] = RYS_TABLE_3,
                    h_gtab4[] = RYS_TABLE_4, h_gtab5[] = RYS_TABLE_5;
static const double h_gherm1[] = RYS_HERM_1, h_gherm2[] = RYS_HERM_2, h_gherm3[] = RYS_HERM_3,
                    h_gherm4[] = RYS_HERM_4, h_gherm5[] = RYS_HERM_5;

POLY_HD void rys_nodes_n(int n, double T, const RysTabs& rt, double* u, double* w) {
    switch (n) {
    case 1: rys_node<1>(T, 0, rt.tab[1], rt.herm[1], u[0], w[0]); break;
    case 2: for (int r = 0; r < 2; ++r) rys_node<2>(T, r, rt.tab[2], rt.herm[2], u[r], w[r]); break;
    case 3: for (int r = 0; r < 3; ++r) rys_node<3>(T, r, rt.tab[3], rt.herm[3], u[r], w[r]); break;
    case 4: for (int r = 0; r < 4; ++r) rys_node<4>(T, r, rt.tab[4], rt.herm[4], u[r], w[r]); break;
    default: for (int r = 0; r < 5; ++r) rys_node<5>(T, r, rt.tab[5], rt.herm[5], u[r], w[r]); break;
    }
}

POLY_HD void comp_of(int l, int q, int& lx, int& ly, int& lz) {
    // xx, xy, xz, yy, yz, zz order (x exponent descending, then y)
    int n = 0;
    for (int i = l; i >= 0; --i)
        for (int k = 0; k <= l - i; ++k) {
            if (n == q) { lx = i; ly = l - i - k; lz = k; return; }
            ++n;
        }
    lx = ly = lz = 0;
}

// binomial coefficients C(n, k), n <= 3 (the transfers go one level above d)
POLY_HD double binom(int n, int k) {
    return n == 3 ? (k == 0 || k == 3 ? 1.0 : 3.0) : n == 2 ? (k == 1 ? 2.0 : 1.0) : 1.0;
}

// One-dimensional factors of one axis for one root: I[i][j][k][l] for
// i <= ia, j <= jb, k <= kc, l <= ld with i + j <= na and k + l <= nc (the
// derivatives need one level above the quartet on one index at a time).
POLY_HD void axis_table(double PA, double QC, double PQ, double AB, double CD, double u, double ze, double et,
                        double rho, int na, int nc, int ia, int jb, int kc, int ld,
                        double (&I)[IMAX][IMAX][IMAX][LMAXD]) {
    double G[GMAX][GMAX];
    const double c00 = PA - rho / ze * PQ * u, d00 = QC + rho / et * PQ * u;
    const double b10 = 0.5 / ze * (1.0 - rho * u / ze), b01 = 0.5 / et * (1.0 - rho * u / et);
    const double b00 = 0.5 * u / (ze + et);
    G[0][0] = 1.0;
    for (int i = 0; i < na; ++i) G[i + 1][0] = c00 * G[i][0] + (i ? i * b10 * G[i - 1][0] : 0.0);
    for (int k = 0; k < nc; ++k)
        for (int i = 0; i <= na; ++i)
            G[i][k + 1] = d00 * G[i][k] + (k ? k * b01 * G[i][k - 1] : 0.0) + (i ? i * b00 * G[i - 1][k] : 0.0);
    // ket transfer: H[i][k][l] = sum_s C(l, s) CD^(l - s) G[i][k + s]
    double H[GMAX][IMAX][LMAXD];
    for (int i = 0; i <= na; ++i)
        for (int k = 0; k <= kc; ++k)
            for (int l = 0; l <= ld && k + l <= nc; ++l) {
                double s = 0.0, p = 1.0;
                for (int t = l; t >= 0; --t) {      // CD^(l - t) G[i][k + t]
                    s += binom(l, t) * p * G[i][k + t];
                    p *= CD;
                }
                H[i][k][l] = s;
            }
    for (int i = 0; i <= ia; ++i)
        for (int j = 0; j <= jb && i + j <= na; ++j)
            for (int k = 0; k <= kc; ++k)
                for (int l = 0; l <= ld && k + l <= nc; ++l) {
                    double s = 0.0, p = 1.0;
                    for (int t = j; t >= 0; --t) {
                        s += binom(j, t) * p * H[i + t][k][l];
                        p *= AB;
                    }
                    I[i][j][k][l] = s;
                }
}

// Shell data for the host's Schwarz bounds.
struct Sh {
    int L, p0, np;
    double x, y, z;
};

inline Sh shell_of(const GradShells& g, int s) {
    return Sh{g.L[s], g.p0[s], g.np[s], g.xyz[3 * s], g.xyz[3 * s + 1], g.xyz[3 * s + 2]};
}

// max over components of |(mu nu|mu nu)| for the Schwarz bound of pair (a, b)
inline double pair_bound(const GradShells& g, const RysTabs& rt, int a, int b) {
    const Sh A = shell_of(g, a), B = shell_of(g, b);
    const int na = A.L + B.L, n = (2 * na) / 2 + 1;
    const int ca = ncart(A.L), cb = ncart(B.L);
    double acc[36];
    for (int q = 0; q < ca * cb; ++q) acc[q] = 0.0;
    const double AB[3] = {A.x - B.x, A.y - B.y, A.z - B.z};
    const double ab2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
    double I3[3][IMAX][IMAX][IMAX][LMAXD];
    for (int i = 0; i < A.np; ++i)
        for (int j = 0; j < B.np; ++j) {
            const double al = g.alpha[A.p0 + i], be = g.alpha[B.p0 + j];
            const double ze = al + be, kab = std::exp(-al * be / ze * ab2);
            const double cab = g.coef[A.p0 + i] * g.coef[B.p0 + j] * kab;
            if (std::fabs(cab) < g.ptol) continue;
            const double P[3] = {(al * A.x + be * B.x) / ze, (al * A.y + be * B.y) / ze, (al * A.z + be * B.z) / ze};
            for (int k = 0; k < A.np; ++k)
                for (int l = 0; l < B.np; ++l) {
                    const double ga = g.alpha[A.p0 + k], de = g.alpha[B.p0 + l];
                    const double et = ga + de, kcd = std::exp(-ga * de / et * ab2);
                    const double ccd = g.coef[A.p0 + k] * g.coef[B.p0 + l] * kcd;
                    if (std::fabs(ccd) < g.ptol) continue;
                    const double Q[3] = {(ga * A.x + de * B.x) / et, (ga * A.y + de * B.y) / et,
                                         (ga * A.z + de * B.z) / et};
                    const double PQ[3] = {P[0] - Q[0], P[1] - Q[1], P[2] - Q[2]};
                    const double rho = ze * et / (ze + et);
                    const double T = rho * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
                    const double pref = 2.0 * POLY_PI * POLY_PI * POLY_SQRT_PI / (ze * et * std::sqrt(ze + et)) * cab * ccd;
                    double u[RYS_NMAX], w[RYS_NMAX];
                    rys_nodes_n(n, T, rt, u, w);
                    for (int r = 0; r < n; ++r) {
                        const double Pc[3] = {P[0], P[1], P[2]};
                        const double Ac[3] = {A.x, A.y, A.z};
                        for (int ax = 0; ax < 3; ++ax)
                            axis_table(Pc[ax] - Ac[ax], Q[ax] - Ac[ax], PQ[ax], AB[ax], AB[ax], u[r], ze, et, rho, na,
                                       na, A.L, B.L, A.L, B.L, I3[ax]);
                        for (int p = 0; p < ca; ++p)
                            for (int q = 0; q < cb; ++q) {
                                int x1, y1, z1, x2, y2, z2;
                                comp_of(A.L, p, x1, y1, z1);
                                comp_of(B.L, q, x2, y2, z2);
                                acc[p * cb + q] += w[r] * pref * I3[0][x1][x2][x1][x2] * I3[1][y1][y2][y1][y2] *
                                                   I3[2][z1][z2][z1][z2];
                            }
                    }
                }
        }
    double m = 0.0;
    for (int q = 0; q < ca * cb; ++q) m = std::fmax(m, std::fabs(acc[q]));
    return std::sqrt(m);
}

// One-dimensional factors of one axis for one root: v(i, j, k, l) and its
// derivatives on A, B and C, i <= LA, .., l <= LD.
template <int LA, int LB, int LC, int LD>
struct AxisFactors {
    double v[LA + 1][LB + 1][LC + 1][LD + 1], a[LA + 1][LB + 1][LC + 1][LD + 1], b[LA + 1][LB + 1][LC + 1][LD + 1],
        c[LA + 1][LB + 1][LC + 1][LD + 1];
};
template <int LA, int LB, int LC, int LD>
POLY_HD void axis_factors(double c00, double d00, double b10, double b01, double b00, double AB, double CD, double al2,
                          double be2, double ga2, AxisFactors<LA, LB, LC, LD>& f) {
    constexpr int NA = LA + LB + 1, NC = LC + LD + 1;
    double G[NA + 1][NC + 1];
    G[0][0] = 1.0;
#pragma unroll
    for (int i = 0; i < NA; ++i) G[i + 1][0] = c00 * G[i][0] + (i ? i * b10 * G[i - 1][0] : 0.0);
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int i = 0; i <= NA; ++i)
            G[i][k + 1] = d00 * G[i][k] + (k ? k * b01 * G[i][k - 1] : 0.0) + (i ? i * b00 * G[i - 1][k] : 0.0);
    // transfers: H(i, k, l) = sum_t C(l, t) CD^(l - t) G(i, k + t), then the same on the bra
    double H[NA + 1][LC + 2][LD + 1];
#pragma unroll
    for (int i = 0; i <= NA; ++i)
#pragma unroll
        for (int k = 0; k <= LC + 1; ++k)
#pragma unroll
            for (int l = 0; l <= LD; ++l) {
                if (k + l > NC) continue;
                double sum = 0.0, pw = 1.0;
#pragma unroll
                for (int t = l; t >= 0; --t) {
                    sum += binom(l, t) * pw * G[i][k + t];
                    pw *= CD;
                }
                H[i][k][l] = sum;
            }
    double I[LA + 2][LB + 2][LC + 2][LD + 1];
#pragma unroll
    for (int i = 0; i <= LA + 1; ++i)
#pragma unroll
        for (int j = 0; j <= LB + 1; ++j) {
            if (i + j > NA) continue;
#pragma unroll
            for (int k = 0; k <= LC + 1; ++k)
#pragma unroll
                for (int l = 0; l <= LD; ++l) {
                    if (k + l > NC) continue;
                    double sum = 0.0, pw = 1.0;
#pragma unroll
                    for (int t = j; t >= 0; --t) {
                        sum += binom(j, t) * pw * H[i + t][k][l];
                        pw *= AB;
                    }
                    I[i][j][k][l] = sum;
                }
        }
#pragma unroll
    for (int i = 0; i <= LA; ++i)
#pragma unroll
        for (int j = 0; j <= LB; ++j)
#pragma unroll
            for (int k = 0; k <= LC; ++k)
#pragma unroll
                for (int l = 0; l <= LD; ++l) {
                    f.v[i][j][k][l] = I[i][j][k][l];
                    f.a[i][j][k][l] = al2 * I[i + 1][j][k][l] - (i ? i * I[i - 1][j][k][l] : 0.0);
                    f.b[i][j][k][l] = be2 * I[i][j + 1][k][l] - (j ? j * I[i][j - 1][k][l] : 0.0);
                    f.c[i][j][k][l] = ga2 * I[i][j][k + 1][l] - (k ? k * I[i][j][k - 1][l] : 0.0);
                }
}

// The density of one quartet: Gamma of integral (p, q, s, t) without its
// degeneracy factor, from the six blocks of D (each a base address).
struct QuartetDensity {
    const double *ab, *cd, *ac, *ad, *bc, *bd;
    size_t n;
    double xfac;
    POLY_HD double gamma(int p, int q, int s, int t) const {
        return 4.0 * ab[p * n + q] * cd[s * n + t] -
               xfac * (ac[p * n + s] * bd[q * n + t] + ad[p * n + t] * bc[q * n + s]);
    }
};

// Lane `sub` of `lanes`: its units of the quartet of sorted pairs pij (class
// LA LB) and pkl (class LC LD), added to the sums on centres A, B, C.
template <int LA, int LB, int LC, int LD>
POLY_HD void grad_units(const GradArgs& g, const RysTabs& rt, int pij, int pkl, int sub, int lanes, double fdeg,
                        double (&gA)[3], double (&gB)[3], double (&gC)[3]) {
    constexpr int CA = ncart(LA), CB = ncart(LB), CC = ncart(LC), CD_ = ncart(LD), NI = CA * CB * CC * CD_;
    constexpr int NR = (LA + LB + LC + LD + 1) / 2 + 1;
    constexpr bool ROOTS = grad_root_units(NI);      // one root a unit
    const int a = g.pa[pij], b = g.pb[pij], c = g.pa[pkl], d = g.pb[pkl];
    const double* xa = g.xyz + 3 * a;
    const double* xb = g.xyz + 3 * b;
    const double* xc = g.xyz + 3 * c;
    const double* xd = g.xyz + 3 * d;
    const double AB[3] = {xa[0] - xb[0], xa[1] - xb[1], xa[2] - xb[2]};
    const double CD[3] = {xc[0] - xd[0], xc[1] - xd[1], xc[2] - xd[2]};
    const size_t n = (size_t)g.nbf;
    const int fa = g.f0[a], fb = g.f0[b], fc = g.f0[c], fd = g.f0[d];
    const QuartetDensity Q{g.D + fa * n + fb, g.D + fc * n + fd, g.D + fa * n + fc, g.D + fa * n + fd,
                           g.D + fb * n + fc, g.D + fb * n + fd, n, g.xfac};
    // the small classes keep Gamma in registers
    constexpr bool KEEP = NI <= 36;
    double gam[KEEP ? NI : 1];
    if constexpr (KEEP) {
#pragma unroll
        for (int p = 0; p < CA; ++p)
#pragma unroll
            for (int q = 0; q < CB; ++q)
#pragma unroll
                for (int s2 = 0; s2 < CC; ++s2)
#pragma unroll
                    for (int t = 0; t < CD_; ++t) gam[((p * CB + q) * CC + s2) * CD_ + t] = Q.gamma(p, q, s2, t);
    }
    const PrimPair* bra = g.prims + g.pp0[pij];
    const PrimPair* ket = g.prims + g.pp0[pkl];
    const int nk = g.pn[pkl], total = g.pn[pij] * nk * (ROOTS ? NR : 1);
    for (int e = 0; e < 3; ++e) gA[e] = gB[e] = gC[e] = 0.0;
    for (int w = sub; w < total; w += lanes) {
        const int pq = ROOTS ? w / NR : w;
        const int ip = pq / nk;
        const PrimPair bq = bra[ip], kq = ket[pq - ip * nk];
        const double ze = bq.zeta + kq.zeta;
        const double rs = rsqrt_fp64(ze), ize = rs * rs;
        const double roz = kq.zeta * ize, roe = bq.zeta * ize;
        const double PQ[3] = {bq.Px - kq.Px, bq.Py - kq.Py, bq.Pz - kq.Pz};
        const double PA[3] = {bq.PAx, bq.PAy, bq.PAz}, QC[3] = {kq.PAx, kq.PAy, kq.PAz};
        const double T = bq.zeta * roz * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
        const double pref = fdeg * bq.K * kq.K * rs;
        // 2 beta by difference: it rounds by 2^-53 zeta / beta of it, where the
        // pair's prefactor has fallen as fast (against the exponents themselves
        // 1e-14 of the largest component in cc-pVDZ, 1.5e-13 at zeta / beta = 1e8)
        const double be2 = 2.0 * bq.zeta - bq.a2;
        const int r0 = ROOTS ? w - pq * NR : 0, r1 = ROOTS ? r0 + 1 : NR;
#pragma unroll
        for (int r = r0; r < r1; ++r) {
            double u, wt;
            rys_node<NR>(T, r, rt.tab[NR], rt.herm[NR], u, wt);
            const double b10 = bq.h * (1.0 - roz * u), b01 = kq.h * (1.0 - roe * u), b00 = 0.5 * ize * u;
            AxisFactors<LA, LB, LC, LD> F[3];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax)
                axis_factors<LA, LB, LC, LD>(PA[ax] - roz * u * PQ[ax], QC[ax] + roe * u * PQ[ax], b10, b01, b00, AB[ax],
                                             CD[ax], bq.a2, be2, kq.a2, F[ax]);
            const double wr = wt * pref;
            auto block = [&](int p) {
                int a3[3];
                comp_of(LA, p, a3[0], a3[1], a3[2]);
#pragma unroll
                for (int q = 0; q < CB; ++q) {
                    int b3[3];
                    comp_of(LB, q, b3[0], b3[1], b3[2]);
#pragma unroll
                    for (int s2 = 0; s2 < CC; ++s2) {
                        int c3[3];
                        comp_of(LC, s2, c3[0], c3[1], c3[2]);
#pragma unroll
                        for (int t = 0; t < CD_; ++t) {
                            int d3[3];
                            comp_of(LD, t, d3[0], d3[1], d3[2]);
                            const double gm = KEEP ? gam[((p * CB + q) * CC + s2) * CD_ + t] : Q.gamma(p, q, s2, t);
                            const double f = wr * gm;
#define GV(e, x) F[e].x[a3[e]][b3[e]][c3[e]][d3[e]]
                            const double f0 = f * GV(1, v) * GV(2, v), f1 = f * GV(0, v) * GV(2, v),
                                         f2 = f * GV(0, v) * GV(1, v);
                            gA[0] += f0 * GV(0, a);
                            gA[1] += f1 * GV(1, a);
                            gA[2] += f2 * GV(2, a);
                            gB[0] += f0 * GV(0, b);
                            gB[1] += f1 * GV(1, b);
                            gB[2] += f2 * GV(2, b);
                            gC[0] += f0 * GV(0, c);
                            gC[1] += f1 * GV(1, c);
                            gC[2] += f2 * GV(2, c);
#undef GV
                        }
                    }
                }
            };
            if constexpr (NI <= 108) {
#pragma unroll
                for (int p = 0; p < CA; ++p) block(p);
            } else {
#pragma unroll 1
                for (int p = 0; p < CA; ++p) block(p);
            }
        }
    }
}

// Contribution of lane `sub` of `lanes` to the quartet of sorted pairs pij
// (class LA LB) and pkl (class LC LD): the atoms of its centres and the sums
// on A, B, C.  False where the quartet is below the threshold.
template <int LA, int LB, int LC, int LD>
POLY_HD bool quartet_cls(const GradArgs& g, const RysTabs& rt, int pij, int pkl, int sub, int lanes, int (&at)[4],
                         double (&gs)[3][3]) {
    const double qq = g.Qp[pij] * g.Qp[pkl];
    if (qq < g.tol) return false;
    const int a = g.pa[pij], b = g.pb[pij], c = g.pa[pkl], d = g.pb[pkl];
    // the density-weighted bound: Q_ab Q_cd max |Gamma| over the quartet
    const int ns = g.nsh;
    const double gmax = 4.0 * g.dsh[a * ns + b] * g.dsh[c * ns + d] +
                        std::fabs(g.xfac) * (g.dsh[a * ns + c] * g.dsh[b * ns + d] + g.dsh[a * ns + d] * g.dsh[b * ns + c]);
    if (qq * gmax < g.tol) return false;
    const double fdeg = (a == b ? 0.5 : 1.0) * (c == d ? 0.5 : 1.0) * (pij == pkl ? 0.5 : 1.0);
    grad_units<LA, LB, LC, LD>(g, rt, pij, pkl, sub, lanes, fdeg, gs[0], gs[1], gs[2]);
    at[0] = g.atom[a]; at[1] = g.atom[b]; at[2] = g.atom[c]; at[3] = g.atom[d];
    return true;
}
// add(atom, axis, value) of those sums; D's by translational invariance.
template <typename Add>
POLY_HD void add_centres(const int (&at)[4], const double (&gs)[3][3], Add add) {
    for (int e = 0; e < 3; ++e) {
        for (int x = 0; x < 3; ++x) add(at[x], e, gs[x][e]);
        add(at[3], e, -(gs[0][e] + gs[1][e] + gs[2][e]));
    }
}

__device__ RysTabs device_tabs() {
    RysTabs rt;
    rt.tab[0] = rt.herm[0] = nullptr;
    rt.tab[1] = g_gtab1; rt.tab[2] = g_gtab2; rt.tab[3] = g_gtab3; rt.tab[4] = g_gtab4; rt.tab[5] = g_gtab5;
    rt.herm[1] = g_gherm1; rt.herm[2] = g_gherm2; rt.herm[3] = g_gherm3; rt.herm[4] = g_gherm4; rt.herm[5] = g_gherm5;
    return rt;
}

RysTabs host_tabs() {
    RysTabs rt;
    rt.tab[0] = rt.herm[0] = nullptr;
    rt.tab[1] = h_gtab1; rt.tab[2] = h_gtab2; rt.tab[3] = h_gtab3; rt.tab[4] = h_gtab4; rt.tab[5] = h_gtab5;
    rt.herm[1] = h_gherm1; rt.herm[2] = h_gherm2; rt.herm[3] = h_gherm3; rt.herm[4] = h_gherm4; rt.herm[5] = h_gherm5;
    return rt;
}

// per-atom sums in LDS (3 natom doubles of dynamic shared memory), one
// global atomic per element per block.  Lane t of the launch: chunk c with
// coff[c] <= t < coff[c + 1] (found once per wavefront, then stepped), the
// item (t - coff[c]) / lanes of it.
template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(256) k_eri_grad(GradArgs g, int x0, int y0, double* __restrict__ grad) {
    extern __shared__ double sg[];
    for (int i = threadIdx.x; i < 3 * g.natom; i += blockDim.x) sg[i] = 0.0;
    __syncthreads();
    const RysTabs rt = device_tabs();
    const unsigned long long nt = g.coff[g.nchunk];
    for (unsigned long long t = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; t < nt;
         t += (unsigned long long)gridDim.x * blockDim.x) {
        const unsigned long long tw = t - (threadIdx.x & 63);
        int lo = 0, hi = g.nchunk - 1;             // largest c with coff[c] <= tw
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (g.coff[mid] <= tw) lo = mid;
            else hi = mid - 1;
        }
        while (g.coff[lo + 1] <= t) ++lo;          // t < coff[nchunk]
        const int r = (int)(t - g.coff[lo]), lanes = g.cij[3 * lo + 2], item = r / lanes;
        int at[4];
        double gs[3][3];
        const bool live = quartet_cls<LA, LB, LC, LD>(g, rt, x0 + g.cij[3 * lo], y0 + g.cij[3 * lo + 1] + item,
                                                      r - item * lanes, lanes, at, gs);
        const auto add = [&](int a, int e, double v) {
            if (v != 0.0) atomicAdd(&sg[3 * a + e], v);
        };
        // a wavefront inside one quartet adds once (64 lanes on one LDS
        // address would be added one after the other)
        const int c0 = __builtin_amdgcn_readfirstlane(lo), i0 = __builtin_amdgcn_readfirstlane(item);
        if (__all(lo == c0 && item == i0 && live) && __popcll(__ballot(1)) == 64) {
#pragma unroll
            for (int x = 0; x < 3; ++x)
#pragma unroll
                for (int e = 0; e < 3; ++e) gs[x][e] = wave_sum(gs[x][e]);
            if ((threadIdx.x & 63) == 0) add_centres(at, gs, add);
        } else if (live) {
            add_centres(at, gs, add);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 3 * g.natom; i += blockDim.x)
        if (sg[i] != 0.0) atomicAdd(&grad[i], sg[i]);
}

// one class pair's launch (device) or loop (host)
struct GradLaunch {
    const GradArgs& gq;
    int x0, y0;
    unsigned grid;
    size_t lds;
    double* d;
    hipStream_t s;
    template <int A, int B, int C, int D>
    void operator()() const {
        hipLaunchKernelGGL((k_eri_grad<A, B, C, D>), dim3(grid), dim3(256), lds, s, gq, x0, y0, d);
    }
};

struct GradHostRun {
    const GradArgs& gq;
    const RysTabs& rt;
    int x0, y0;
    double* grad;
    template <int A, int B, int C, int D>
    void operator()() const {
        for (int c = 0; c < gq.nchunk; ++c) {
            const int lanes = gq.cij[3 * c + 2];
            const int n = (int)(gq.coff[c + 1] - gq.coff[c]);
            for (int r = 0; r < n; ++r) {
                int at[4];
                double gs[3][3];
                if (quartet_cls<A, B, C, D>(gq, rt, x0 + gq.cij[3 * c], y0 + gq.cij[3 * c + 1] + r / lanes, r % lanes,
                                            lanes, at, gs))
                    add_centres(at, gs, [&](int a, int e, double v) { grad[3 * a + e] += v; });
            }
        }
    }
};

// Runs class pair (X, Y), Y <= X, of the pair classes
// ((ss) (ps) (pp) (ds) (dp) (dd) = 0 .. 5) through f.
constexpr int kGradPL[6][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}};
template <int X, typename F>
void grad_class_row(int Y, F&& f) {
    switch (Y) {
    case 0: f.template operator()<kGradPL[X][0], kGradPL[X][1], 0, 0>(); break;
    case 1: if constexpr (X >= 1) f.template operator()<kGradPL[X][0], kGradPL[X][1], 1, 0>(); break;
    case 2: if constexpr (X >= 2) f.template operator()<kGradPL[X][0], kGradPL[X][1], 1, 1>(); break;
    case 3: if constexpr (X >= 3) f.template operator()<kGradPL[X][0], kGradPL[X][1], 2, 0>(); break;
    case 4: if constexpr (X >= 4) f.template operator()<kGradPL[X][0], kGradPL[X][1], 2, 1>(); break;
    case 5: if constexpr (X >= 5) f.template operator()<kGradPL[X][0], kGradPL[X][1], 2, 2>(); break;
    default: break;
    }
}

}  // namespace

// the kernels of bra pair class X, one translation unit each (kgrad/kgrad_xX.hip)
#define GRAD_ROW_DECL(X)                                                                                       \
    void polyeri_grad_row_launch_##X(const GradArgs& gq, int Y, int x0, int y0, unsigned grid, size_t lds, double* d, \
                                     hipStream_t s);                                                           \
    void polyeri_grad_row_host_##X(const GradArgs& gq, int Y, int x0, int y0, double* grad);
GRAD_ROW_DECL(0) GRAD_ROW_DECL(1) GRAD_ROW_DECL(2) GRAD_ROW_DECL(3) GRAD_ROW_DECL(4) GRAD_ROW_DECL(5)
#undef GRAD_ROW_DECL
