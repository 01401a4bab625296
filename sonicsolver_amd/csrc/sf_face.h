// sf_face.h -- per-face FP64 arithmetic of the explicit Euler hot path for
// gfx950: characteristic WENO3 / WENO5-JS / TENO5 / WENO7 reconstruction on
// an axis-aligned face followed by a Rusanov, HLLC, Steger-Warming,
// Lax-Friedrichs, Roe or Lax-Wendroff flux.
//
// The operations are those of the reference functions cited at each
// definition (paths relative to the sonicSolver source tree).  On an
// axis-aligned face the unit normal and the tangent basis (l, m) are
// signed unit vectors, so every product with one of their zero components
// is dropped and every product with +-1 becomes a sign; for finite inputs
// this changes nothing but the sign of a zero.  FP64 division is a long
// instruction sequence on CDNA, so where the reference divides several
// times by one quantity the code takes one reciprocal, and the WENO
// weights are normalised with a single division (each definition says
// where).  With its fused multiply-adds, results differ from the
// reference in the last few bits only.
//
// Every fused multiply-add below is written out and the compiler fuses none
// of its own (which of two products a sum would be fused with depends on
// what else a kernel does with them), so a face has the same bits in every
// kernel that evaluates it.
#pragma once

#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace sfamd {

enum : unsigned {
    kFlagState = 1u, kFlagChar = 2u, kFlagTeno = 4u, kFlagFlux = 8u, kFlagDt = 16u
};

// Tangent basis of Riemann::buildCharacteristicMatrix for n = e_AXIS
// (SF_riemann.cpp:88-97):
//   x: l = (-0, 1, 0), m = (0, 0, 1)
//   y: l = (-1, 0, 0), m = (0, -0, 1)
//   z: l = (-1, 0, 0), m = (0, -1, 0)
template <int AXIS> struct Basis;
template <> struct Basis<0> {
    static constexpr int nd = 0, li = 1, mi = 2;
    static constexpr double sl = 1.0, sm = 1.0;
};
template <> struct Basis<1> {
    static constexpr int nd = 1, li = 0, mi = 2;
    static constexpr double sl = -1.0, sm = 1.0;
};
template <> struct Basis<2> {
    static constexpr int nd = 2, li = 0, mi = 1;
    static constexpr double sl = -1.0, sm = -1.0;
};

__device__ __forceinline__ double sq(double x) { return x * x; }

__device__ __forceinline__ double dot3(const double* a, const double* b) {
    return fma(a[2], b[2], fma(a[1], b[1], a[0] * b[0]));
}

// Reciprocal, quotient and reciprocal square root from the hardware
// estimate (good to about 5e-8 relative) refined by NR Newton steps: with
// two, within about one ulp of the correctly rounded value for the normal,
// finite, nonzero operands of this path; with one, within about 10 ulps
// (reciprocal) and 20 ulps (reciprocal square root).  A zero or non-finite
// operand yields NaN, which the flux and state checks report.  The IEEE
// sequences hipcc emits for '/' and sqrt are two to three times longer.
template <int NR = 2>
__device__ __forceinline__ double frcp(double b) {
    double r = __builtin_amdgcn_rcp(b);
#pragma unroll
    for (int i = 0; i < NR; ++i) r = fma(fma(-b, r, 1.0), r, r);
    return r;
}

template <int NR = 2>
__device__ __forceinline__ double fdiv(double a, double b) {
    const double r = frcp<NR>(b);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

template <int NR = 2>
__device__ __forceinline__ double frsqrt(double z) {
    double y = __builtin_amdgcn_rsq(z);
    const double h = 0.5 * z;
#pragma unroll
    for (int i = 0; i < NR; ++i) y = y * fma(-h * y, y, 1.5);
    return y;
}

// sqrt(z) as z * rsqrt(z) (z > 0)
template <int NR = 2>
__device__ __forceinline__ double fsqrt(double z) { return z * frsqrt<NR>(z); }

// The reference's cutoff test RN(g / gs) < CT (CT = 1e-5) without the
// division.  RN(x) < CT exactly when x < CT - d with d half the gap from CT
// down to the next double (2^-70 for CT = 1e-5), i.e. when
// g < CT*gs - d*gs.  CT*gs = P + E exactly (FMA), d*gs is exact, and near
// the boundary g - P is exact (Sterbenz), so the comparison below decides
// exactly as the division does (up to a tie at the midpoint).
__device__ __forceinline__ bool teno_cut(double g, double gs) {
    const double P = 1.0e-5 * gs;
    const double E = __builtin_fma(1.0e-5, gs, -P);
    return g - P < fma(-0x1p-70, gs, E);
}

// Reconstruction in differences.  Every candidate value is the upwind node
// plus a combination of the differences d_k = c_{k+1} - c_k of neighbouring
// nodes, and every smoothness indicator is a function of them alone, so the
// functions below take the NS - 1 projected differences of a stencil and
// return the increments to add to the upwind nodes: the left one to node
// NS/2 - 1, the right one to node NS/2 (left reads d_0.., the mirrored right
// side the same differences in reverse).  Against projecting the NS nodes
// and rebuilding the differences per field this takes a fifth of a WENO5
// face's FP64 instructions away (721 -> 597 with HLLC) and half of a WENO7
// face's, and it rounds less: what is rounded is the increment, not the
// node.  The faces are bound by FP64 issue, so the sweeps follow: a whole
// 512^3 WENO5/HLLC pass 86.4 -> 79.5 ms, 256^3 WENO7/Rusanov 23.5 -> 14.4,
// 2048^2 TENO5/HLLC 7.0 -> 6.3 (together with the HLLC flux below).
//
// WENO5 / TENO5 indicators, scaled by 4 (exactly) so that the squared first
// difference needs no factor: b = 13/3 s^2 + f^2 + eps with s the second
// difference and f the one-sided or central first difference
// (SF_WENO5.cpp:42-62).  Two of the three second differences of each side
// belong to the other side too.
struct PairTerms {
    double fL[3], fR[3];   // first-difference terms of the candidates
    double bL[3], bR[3];   // 4 (beta + eps)
};

__device__ __forceinline__ PairTerms pair_terms(const double (&d)[5], double eps4) {
    PairTerms t;
    constexpr double k = 13.0 / 3.0;
    double s[4], g[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        s[i] = d[i + 1] - d[i];
        g[i] = fma(k * s[i], s[i], eps4);
    }
    // 3 d1 - d0, d3 - 3 d2, ...: through s, so that the factor is 2, which
    // the instruction holds (a literal 3 would cost a register move each)
    t.fL[0] = fma(2.0, d[1], s[0]);
    t.fL[1] = d[1] + d[2];
    t.fL[2] = fma(-2.0, d[2], s[2]);
    t.fR[0] = fma(-2.0, d[3], s[3]);
    t.fR[1] = d[3] + d[2];
    t.fR[2] = fma(2.0, d[2], s[1]);
    t.bL[0] = fma(t.fL[0], t.fL[0], g[0]);
    t.bL[1] = fma(t.fL[1], t.fL[1], g[1]);
    t.bL[2] = fma(t.fL[2], t.fL[2], g[2]);
    t.bR[0] = fma(t.fR[0], t.fR[0], g[3]);
    t.bR[1] = fma(t.fR[1], t.fR[1], g[2]);
    t.bR[2] = fma(t.fR[2], t.fR[2], g[1]);
    return t;
}

// a/b and c/d with one reciprocal (both denominators are positive and far
// from the ends of the exponent range here).
template <int NR = 2>
__device__ __forceinline__ void div_pair(double a, double b, double c, double d, double& x,
                                         double& y) {
    const double r = frcp<NR>(b * d);
    x = a * d * r;
    y = c * b * r;
}

// WENO5::weno5_core (SF_WENO5.cpp:42-62).  With AL = e1 e2, BL = e0 e2,
// CL = e0 e1 (e = b^2) the weights are (AL, 6 BL, 3 CL) / (AL + 6 BL + 3 CL);
// the candidates' increments are (5 d1 - 2 d0)/6 = (2 fL0 - d1)/6,
// (d1 + 2 d2)/6 and (4 d2 - d3)/6, whose factors 6 and 3 cancel those of the
// weights.
template <int NR>
__device__ __forceinline__ void weno5_pair(const double (&d)[5], double& left, double& right) {
    const PairTerms t = pair_terms(d, 4e-6);
    const double AL = sq(t.bL[1] * t.bL[2]), BL = sq(t.bL[0] * t.bL[2]), CL = sq(t.bL[0] * t.bL[1]);
    const double AR = sq(t.bR[1] * t.bR[2]), BR = sq(t.bR[0] * t.bR[2]), CR = sq(t.bR[0] * t.bR[1]);
    constexpr double s6 = 1.0 / 6.0, s3 = 1.0 / 3.0;
    const double h2 = 0.5 * d[2];
    const double nL = fma(AL, fma(s3, t.fL[0], -s6 * d[1]),
                          fma(BL, t.fL[1] + d[2], CL * fma(-0.5, t.fL[2], h2)));
    const double nR = fma(AR, fma(s3, t.fR[0], s6 * d[3]),
                          -fma(BR, t.fR[1] + d[2], CR * fma(0.5, t.fR[2], h2)));
    const double dL = fma(3.0, CL, fma(6.0, BL, AL)), dR = fma(3.0, CR, fma(6.0, BR, AR));
    div_pair<NR>(nL, dL, nR, dR, left, right);
}

// TENO5's stencil selection (SF_TENO5.cpp:60-89): gamma_k = (1 + tau5 /
// (beta_k + 1e-40))^6 and the cutoff of gamma_k / sum gamma at 1e-5.  The
// gammas only decide which stencils are kept, so the last bits of the
// quotients change a result only where a ratio lies within rounding of the
// cutoff.  Returns false where the sum of the gammas is not finite, which
// the reference treats as fatal (requireFiniteGammaSum, SF_TENO5.cpp:33-40).
// b[k] = 4 (beta_k + 1e-40): the factor cancels in the quotients.
__device__ __forceinline__ bool teno5_weights(const double b[3], double& c0, double& c1,
                                              double& c2) {
    const double tau5 = fabs(b[0] - b[2]);
    // tau5 / b_k for the three k from one reciprocal of b0 b1 b2 (each
    // b_k >= 4e-40, so the product stays far above the subnormal range)
    const double e01 = b[0] * b[1];
    const double t = tau5 * frcp(e01 * b[2]);
    auto p6 = [](double x) {   // three products: within a few ulps of x^6
        const double x3 = x * x * x;
        return x3 * x3;
    };
    const double g0 = p6(fma(t, b[1] * b[2], 1.0));
    const double g1 = p6(fma(t, b[0] * b[2], 1.0));
    const double g2 = p6(fma(t, e01, 1.0));
    const double gs = g0 + g1 + g2;
    c0 = teno_cut(g0, gs) ? 0.0 : 1.0;
    c1 = teno_cut(g1, gs) ? 0.0 : 1.0;
    c2 = teno_cut(g2, gs) ? 0.0 : 1.0;
    return gs < INFINITY;
}

// The kept candidates' linear weights (0.1, 0.6, 0.3), scaled by 10, times
// the increments as in weno5_pair.
__device__ __forceinline__ void teno5_pair(const double (&d)[5], double& left, double& right,
                                           unsigned& flags) {
    const PairTerms t = pair_terms(d, 4e-40);
    double l0, l1, l2, r0, r1, r2;
    const bool fin = teno5_weights(t.bL, l0, l1, l2) & teno5_weights(t.bR, r0, r1, r2);
    const double aL = fma(3.0, l2, fma(6.0, l1, l0));
    const double aR = fma(3.0, r2, fma(6.0, r1, r0));
    if (!fin || !(aL > 0.0) || !(aR > 0.0)) flags |= kFlagTeno;
    constexpr double s6 = 1.0 / 6.0, s3 = 1.0 / 3.0;
    const double h2 = 0.5 * d[2];
    const double nL = fma(l0, fma(s3, t.fL[0], -s6 * d[1]),
                          fma(l1, t.fL[1] + d[2], l2 * fma(-0.5, t.fL[2], h2)));
    const double nR = fma(r0, fma(s3, t.fR[0], s6 * d[3]),
                          -fma(r1, t.fR[1] + d[2], r2 * fma(0.5, t.fR[2], h2)));
    div_pair(nL, aL, nR, aR, left, right);
}

// WENO3::weno3_core (SF_WENO3.cpp:42-57) on both sides of a face.  The two
// candidates and the two squared spreads serve both sides; the weights are
// normalised with one division per side (alpha_k = d_k / e_k multiplied
// through by 3 e_A e_B) and the two divisions share one reciprocal.
template <int NR>
__device__ __forceinline__ void weno3_pair(const double (&d)[3], double& left, double& right) {
    const double eps = 1e-6;
    const double fA = d[0] + d[1], fB = d[1] + d[2];
    const double eA = sq(fma(fA, fA, eps)), eB = sq(fma(fB, fB, eps));
    // 6 x increments: candidates A and B from node 1 (left), node 2 (right)
    const double AL = fma(2.0, d[1], d[0]), BL = fma(4.0, d[1], -d[2]);
    const double AR = fma(-4.0, d[1], d[0]), BR = fma(-2.0, d[1], -d[2]);
    const double e2A = 2.0 * eA, e2B = 2.0 * eB;
    const double nL = fma(eB, AL, e2A * BL), nR = fma(eA, BR, e2B * AR);
    div_pair<NR>(nL, 6.0 * (eB + e2A), nR, 6.0 * (eA + e2B), left, right);
}

// WENO7::weno7_core (SF_WENO7.cpp:43-98) on both sides of a face.  The
// indicator of a four-node candidate over its target cell (beta4: the
// integral of the squared first, second and third derivatives of the
// cubic), written about the cell's centre, is a sum of three squares,
//   beta = G^2 + 13/12 B^2 + 781/720 t^2,
// with t the candidate's third difference, B its second derivative at the
// centre (a second difference, or one extrapolated by t) and G its first
// derivative there plus t/24: for the target cell between differences d_l
// and d_r (d_l to its left),
//   d_l + s/2 + 3/8 t   outermost upwind candidate (s, t its last ones)
//   (d_l + d_r)/2 - t/8 the two candidates around the cell
//   d_r - s/2 + 3/8 t   outermost downwind candidate (s, t its first ones).
// This takes 52 operations for the eight indicators of a field against
// about 240 for the polynomial form.  The weights (1, 12, 18, 4) / e_k are
// multiplied through by the product of the four e and normalised with one
// division per side; the two divisions share one reciprocal.
__device__ __forceinline__ void weno7_side(const double b[4], double q0, double q1, double q2,
                                           double q3, double& num, double& den) {
    const double e0 = sq(b[0]), e1 = sq(b[1]), e2 = sq(b[2]), e3 = sq(b[3]);
    const double e01 = e0 * e1, e23 = e2 * e3;
    const double w1 = 12.0 * e0, w2 = 18.0 * e3, w3 = 4.0 * e2;
    num = fma(e23, fma(e1, q0, w1 * q1), e01 * fma(w2, q2, w3 * q3));
    den = fma(e23, e1 + w1, e01 * (w2 + w3));
}

__device__ __forceinline__ void weno7_pair(const double (&d)[7], double& left, double& right) {
    constexpr double k2 = 13.0 / 12.0, k3 = 781.0 / 720.0, eps = 1e-6;
    double s[6], t[5], T[5];
#pragma unroll
    for (int i = 0; i < 6; ++i) s[i] = d[i + 1] - d[i];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        t[i] = s[i + 1] - s[i];
        T[i] = fma(k3 * t[i], t[i], eps);
    }
    auto beta = [](double G, double B, double Tt) { return fma(G, G, fma(k2 * B, B, Tt)); };
    const double DL = 0.5 * (d[2] + d[3]), DR = 0.5 * (d[3] + d[4]);
    double bL[4], bR[4];   // beta + eps
    bL[0] = beta(fma(0.5, s[1], fma(0.375, t[0], d[2])), s[1] + t[0], T[0]);
    bL[1] = beta(fma(-0.125, t[1], DL), s[2], T[1]);
    bL[2] = beta(fma(-0.125, t[2], DL), s[2], T[2]);
    bL[3] = beta(fma(-0.5, s[3], fma(0.375, t[3], d[3])), s[3] - t[3], T[3]);
    bR[0] = beta(fma(-0.5, s[4], fma(0.375, t[4], d[4])), s[4] - t[4], T[4]);
    bR[1] = beta(fma(-0.125, t[3], DR), s[3], T[3]);
    bR[2] = beta(fma(-0.125, t[2], DR), s[3], T[2]);
    bR[3] = beta(fma(0.5, s[2], fma(0.375, t[1], d[3])), s[2] + t[1], T[1]);
    // 12 x increments of the candidates: the outermost ones, and the three
    // that both sides use, from node 3 (left) and node 4 (right)
    const double L0 = fma(13.0, d[2], fma(-10.0, d[1], 3.0 * d[0]));
    const double R0 = fma(-13.0, d[4], fma(10.0, d[5], -3.0 * d[6]));
    const double p1 = fma(4.0, d[2], -d[1]), p2 = d[2] - d[4], p3 = fma(-4.0, d[4], d[5]);
    double nL, nR, dL, dR;
    weno7_side(bL, L0, fma(3.0, d[3], p1), fma(6.0, d[3], p2), fma(9.0, d[3], p3), nL, dL);
    weno7_side(bR, R0, fma(-3.0, d[3], p3), fma(-6.0, d[3], p2), fma(-9.0, d[3], p1), nR, dR);
    div_pair(nL, 12.0 * dL, nR, 12.0 * dR, left, right);
}

// Scheme ids (SF_SCHEME_*) and their stencils (SF_stencil.h:12-17):
//   0 WENO5 and 1 TENO5 read 6 nodes, 2 WENO3 reads 4, 3 WENO7 reads 8.
// newton: the Newton steps of every reciprocal and reciprocal square root
// in a face of the scheme.  One for WENO5 and WENO3, whose weights are
// smooth functions of their inputs, so a last-bit difference stays a
// last-bit difference; two for TENO5, whose stencil cutoff turns one into
// a different stencil, and for WENO7, which is held to the reference's
// own frozen Sod output.
template <int SCHEME> struct Stencil { static constexpr int ns = 6, newton = 1; };
template <> struct Stencil<1> { static constexpr int ns = 6, newton = 2; };
template <> struct Stencil<2> { static constexpr int ns = 4, newton = 1; };
template <> struct Stencil<3> { static constexpr int ns = 8, newton = 2; };

template <int SCHEME, int NR>
__device__ __forceinline__ void recon_pair(const double (&d)[Stencil<SCHEME>::ns - 1], double& left,
                                           double& right, unsigned& flags) {
    if constexpr (SCHEME == 1) teno5_pair(d, left, right, flags);
    else if constexpr (SCHEME == 2) weno3_pair<NR>(d, left, right);
    else if constexpr (SCHEME == 3) weno7_pair(d, left, right);
    else weno5_pair<NR>(d, left, right);
}

// Closure of SingleFluidStateModel::close + PerfectGasEOS
// (SF_singleFluidStateModel.cpp:49-71, SF_perfectGasEOS.h:24-32).
// One reciprocal of the density replaces the five divisions by rho.
struct Closed {
    double u[3], p, inv_rho;
    double c2, rc;   // squared sound speed and its reciprocal root: c = c2 rc
    __device__ __forceinline__ double c() const { return c2 * rc; }
};

// close_state with the reciprocal of the density given.
template <int NR = 2>
__device__ __forceinline__ Closed close_state_r(const double q[5], double gamma, double inv_rho) {
    Closed s;
    s.inv_rho = inv_rho;
    s.u[0] = q[1] * s.inv_rho;
    s.u[1] = q[2] * s.inv_rho;
    s.u[2] = q[3] * s.inv_rho;
    const double mu = dot3(q + 1, s.u);
    s.p = (gamma - 1.0) * fma(-0.5, mu, q[4]);
    s.c2 = gamma * s.p * s.inv_rho;
    s.rc = frsqrt<NR>(s.c2);
    return s;
}

template <int NR = 2>
__device__ __forceinline__ Closed close_state(const double q[5], double gamma) {
    return close_state_r<NR>(q, gamma, frcp<NR>(q[0]));
}

// Whether x is positive and finite: one class test (positive subnormal or
// normal) instead of two comparisons.
__device__ __forceinline__ bool positive_finite(double x) {
    return __builtin_amdgcn_class(x, 0x180);
}

// The closure's validity test, as PerfectGasEOS::fromDensityEnergy makes
// it on each face state the Rusanov flux closes (SF_perfectGasEOS.h:26-33
// with requireDensity and checked: rho > 0, and p, T, c > 0 and finite;
// for a perfect gas with rho > 0, T and c are positive and finite exactly
// when p is): the reference stops on a face whose reconstructed state
// fails it.
__device__ __forceinline__ bool closed_ok(const double q[5], const Closed& s) {
    return positive_finite(q[0]) && positive_finite(s.p);
}

// RusanovEOS::faceFlux, SF_rusanovEOS.cpp:47-77.
template <int ND, int NR = 2>
__device__ __forceinline__ void rusanov(const double qL[5], const double qR[5],
                                        double gamma, double out[5], unsigned& flags) {
    const Closed l = close_state<NR>(qL, gamma), r = close_state<NR>(qR, gamma);
    if (!closed_ok(qL, l) || !closed_ok(qR, r)) flags |= kFlagFlux;
    // (F(qL) + F(qR) - lambda (qR - qL)) / 2 with F the physical flux
    // (physicalFlux, SF_rusanovEOS.cpp:14-32), whose mass component is the
    // normal momentum
    const double unL = l.u[ND], unR = r.u[ND];
    const double lambda = fmax(fma(l.c2, l.rc, fabs(unL)), fma(r.c2, r.rc, fabs(unR)));
    out[0] = 0.5 * fma(-lambda, qR[0] - qL[0], qL[1 + ND] + qR[1 + ND]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        double f = fma(qR[1 + d], unR, qL[1 + d] * unL);
        if (d == ND) f += l.p + r.p;
        out[1 + d] = 0.5 * fma(-lambda, qR[1 + d] - qL[1 + d], f);
    }
    out[4] = 0.5 * fma(-lambda, qR[4] - qL[4], fma(qR[4] + r.p, unR, (qL[4] + l.p) * unL));
}

// HLLC (no reference counterpart).  Toro, "Riemann Solvers and Numerical
// Methods for Fluid Dynamics", 3rd ed.: Einfeldt wave speeds from Roe
// averages, contact speed eq. (10.37), star states eq. (10.39) with the
// tangential velocity of each side carried unchanged, flux eq. (10.38).
//
// The flux of eq. (10.38) through the star region of side K is the physical
// flux of its star state moving with the contact: with a = S_K - u_K,
// g = S - u_K, S the contact speed,
//   rho* = rho_K a / (S_K - S),  p* = p_K + rho_K a g,
//   E* = (a E_K - p_K u_K + p* S) / (S_K - S),
//   F = (rho* S, rho* S u + p* n, (E* + p*) S).
// The same formulas at S = u_K give side K's own physical flux, which is
// what the two supersonic regions take, so one choice of S serves all four
// regions and only side K's values are selected.  There rho* S is the normal
// momentum, taken as it is: against 80-bit arithmetic the flux of smooth WENO5
// faces at Mach 1.3 - 4 is off by 0.9e-17 (mass), 9.9e-17 (normal momentum),
// 2.5e-17 (tangential) and 3.5e-16 (energy) of its largest component in the
// mean; 6.3e-17, 2.3e-16, 5.4e-17 and 3.5e-16 with the quotient there, too,
// and 6.4e-17, 1.4e-16, 3.1e-17 and 4.5e-16 with the physical flux and the
// star correction formed separately.
template <int ND, int NR = 2>
__device__ __forceinline__ void hllc(const double qL[5], const double qR[5],
                                     double gamma, double out[5], unsigned& flags) {
    // 1/rho = (rsqrt rho)^2 and sqrt rho = rho rsqrt rho from one refined
    // reciprocal square root per side
    const double yL = frsqrt<NR>(qL[0]), yR = frsqrt<NR>(qR[0]);
    const Closed l = close_state_r<NR>(qL, gamma, yL * yL), r = close_state_r<NR>(qR, gamma, yR * yR);
    if (!closed_ok(qL, l) || !closed_ok(qR, r)) flags |= kFlagFlux;
    const double unL = l.u[ND], unR = r.u[ND];
    // Roe weights sqrt(rho_K) / (sqrt(rho_L) + sqrt(rho_R))
    const double sL = qL[0] * yL, sR = qR[0] * yR;
    const double inv = frcp<NR>(sL + sR);
    const double wL = sL * inv, wR = sR * inv;
    double ut[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) ut[d] = fma(wL, l.u[d], wR * r.u[d]);
    const double HL = (qL[4] + l.p) * l.inv_rho, HR = (qR[4] + r.p) * r.inv_rho;
    const double Ht = fma(wL, HL, wR * HR);
    const double ct2 = (gamma - 1.0) * fma(-0.5, dot3(ut, ut), Ht), rct = frsqrt<NR>(ct2);
    const double SL = fmin(fma(-l.c2, l.rc, unL), fma(-ct2, rct, ut[ND]));
    const double SR = fmax(fma(r.c2, r.rc, unR), fma(ct2, rct, ut[ND]));
    const double mL = qL[0] * (SL - unL), mR = qR[0] * (SR - unR);
    const double Ss = fdiv<NR>(fma(-unR, mR, fma(unL, mL, r.p - l.p)), mL - mR);
    // The left side where the fan leaves the face to the right (0 <= S_L) or
    // the contact does (0 <= S*), the right side otherwise.
    const bool supL = 0.0 <= SL, supR = SR <= 0.0;
    const bool sup = supL || supR;
    const bool left = supL || (!supR && 0.0 <= Ss);
    constexpr int t1 = ND == 0 ? 1 : 0, t2 = ND == 2 ? 1 : 2;
    const double E = left ? qL[4] : qR[4];
    const double p = left ? l.p : r.p;
    const double un = left ? unL : unR;
    const double ut1 = left ? l.u[t1] : r.u[t1], ut2 = left ? l.u[t2] : r.u[t2];
    const double SK = left ? SL : SR;
    const double mK = left ? mL : mR;
    const double S = sup ? un : Ss;
    const double rs = frcp<NR>(SK - S);
    const double ps = fma(mK, S - un, p);
    const double Es = rs * fma(SK - un, E, fma(ps, S, -p * un));
    const double m = sup ? (left ? qL[1 + ND] : qR[1 + ND]) : mK * rs * S;
    out[0] = m;
    out[1 + ND] = fma(m, S, ps);
    out[1 + t1] = m * ut1;
    out[1 + t2] = m * ut2;
    out[4] = (Es + ps) * S;
}

// Pressure as Numerics::pressure forms it (SF_utility.h:24-29), the form
// the flux splittings, the Roe flux and the characteristic matrix use.
struct Legacy {
    double inv_rho, u[3], p;
    bool ok;
};

template <int NR = 2>
__device__ __forceinline__ Legacy legacy_state(const double q[5], double gamma) {
    Legacy s;
    s.inv_rho = frcp<NR>(q[0]);
    const double ke = 0.5 * dot3(q + 1, q + 1) * s.inv_rho;
    s.p = (gamma - 1.0) * (q[4] - ke);
    s.u[0] = q[1] * s.inv_rho;
    s.u[1] = q[2] * s.inv_rho;
    s.u[2] = q[3] * s.inv_rho;
    s.ok = q[0] > 0.0 && s.p > 0.0;
    return s;
}

// One half of the Steger-Warming splitting of a state (POS: F+, else F-)
// for n = e_ND, with the reference's smoothed split of eigenvalues below
// 2 eps_sw = 0.02 (Riemann::splitStegerWarming, SF_riemann.cpp:15-67).
// The three distinct eigenvalues u_n, u_n + a, u_n - a are split once each.
template <int ND, bool POS, int NR = 2>
__device__ __forceinline__ void steger_half(const double q[5], double gamma, double f[5],
                                            unsigned& flags) {
    const Legacy s = legacy_state<NR>(q, gamma);
    if (!s.ok) flags |= kFlagFlux;
    const double a = fsqrt<NR>(gamma * s.p * s.inv_rho);
    const double un = s.u[ND];
    const double q2 = dot3(s.u, s.u);
    auto split = [](double lam) {
        const double eps_sw = 0.01;
        double lp;
        if (fabs(lam) < 2.0 * eps_sw) lp = 0.5 * (fma(lam * (1.0 / (4.0 * eps_sw)), lam, lam) + eps_sw);
        else lp = 0.5 * (lam + fabs(lam));
        return POS ? lp : lam - lp;
    };
    const double l0 = split(un), l3 = split(un + a), l4 = split(un - a);
    const double W1 = fma(2.0 * (gamma - 1.0), l0, l3) + l4;
    const double W2 = l3 - l4;
    const double W3 = l3 + l4;
    const double common = q[0] * frcp<NR>(2.0 * gamma);
    f[0] = common * W1;
#pragma unroll
    for (int d = 0; d < 3; ++d) f[1 + d] = common * ((d == ND) ? fma(a, W2, s.u[d] * W1) : s.u[d] * W1);
    f[4] = common * fma((a * a) * frcp<NR>(gamma - 1.0), W3, fma(a * un, W2, 0.5 * q2 * W1));
}

// StegerWarmingFlux::flux (SF_sw.cpp:21-27): F+(qL) + F-(qR).
template <int ND, int NR = 2>
__device__ __forceinline__ void steger_warming(const double qL[5], const double qR[5],
                                               double gamma, double out[5], unsigned& flags) {
    double fp[5], fm[5];
    steger_half<ND, true, NR>(qL, gamma, fp, flags);
    steger_half<ND, false, NR>(qR, gamma, fm, flags);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[v] = fp[v] + fm[v];
}

// One half of the local Lax-Friedrichs splitting, (F(q) +- lambda q) / 2
// with lambda = |u_n| + a of the state (Riemann::splitLaxFriedrichs,
// SF_riemann.cpp:125-154).
template <int ND, bool POS, int NR = 2>
__device__ __forceinline__ void laxf_half(const double q[5], double gamma, double f[5],
                                          unsigned& flags) {
    const Legacy s = legacy_state<NR>(q, gamma);
    if (!s.ok) flags |= kFlagFlux;
    const double a = fsqrt<NR>(gamma * s.p * s.inv_rho);
    const double un = s.u[ND];
    const double lam = POS ? fabs(un) + a : -(fabs(un) + a);
    double F[5];
    F[0] = q[0] * un;
#pragma unroll
    for (int d = 0; d < 3; ++d) F[1 + d] = (d == ND) ? fma(q[1 + d], un, s.p) : q[1 + d] * un;
    F[4] = (q[4] + s.p) * un;
#pragma unroll
    for (int v = 0; v < 5; ++v) f[v] = 0.5 * fma(lam, q[v], F[v]);
}

// LaxFriedrichsFlux::flux (SF_lxF.cpp:21-27).
template <int ND, int NR = 2>
__device__ __forceinline__ void lax_friedrichs(const double qL[5], const double qR[5],
                                               double gamma, double out[5], unsigned& flags) {
    double fp[5], fm[5];
    laxf_half<ND, true, NR>(qL, gamma, fp, flags);
    laxf_half<ND, false, NR>(qR, gamma, fm, flags);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[v] = fp[v] + fm[v];
}

// physicalEulerFlux (SF_face.h:112-128) for n = e_ND.
template <int ND>
__device__ __forceinline__ void euler_flux(const double q[5], const Legacy& s, double f[5]) {
    const double un = s.u[ND];
    f[0] = q[0] * un;
#pragma unroll
    for (int d = 0; d < 3; ++d) f[1 + d] = (d == ND) ? fma(q[0] * s.u[d], un, s.p) : q[0] * s.u[d] * un;
    f[4] = (q[4] + s.p) * un;
}

// The eigenvector matrices of Riemann::buildCharacteristicMatrix
// (SF_riemann.cpp:69-123) at a state q for n = e_AXIS, in the factored
// form used by the projections below.
template <int AXIS, int NR = 2>
struct CharBasis {
    double u[3], hq2, c, H, un, ul, um, b2, x1, xn, cn;

    // q may carry any common factor: the basis depends on ratios only.
    __device__ __forceinline__ CharBasis(const double q[5], double gamma, unsigned& flags) {
        using B = Basis<AXIS>;
        const double invR = frcp<NR>(q[0]);
        u[0] = q[1] * invR;
        u[1] = q[2] * invR;
        u[2] = q[3] * invR;
        const double ke = 0.5 * dot3(q + 1, u);
        const double p = (gamma - 1.0) * (q[4] - ke);
        if (!(q[0] > 0.0) || !(p > 0.0)) flags |= kFlagChar;
        hq2 = ke * invR;
        const double cz = gamma * p * invR;
        const double rc = frsqrt<NR>(cz);
        c = cz * rc;
        H = (q[4] + p) * invR;
        un = u[B::nd];
        ul = B::sl * u[B::li];
        um = B::sm * u[B::mi];
        b2 = 0.5 * ((gamma - 1.0) * (rc * rc));
        x1 = 0.5 * rc;
        xn = x1 * un;
        cn = c * un;
    }

    // w = L q (gemv5, SF_riemann.h:33-37).  With P = b2 (q2/2 rho - u.m + E)
    // and X = x1 (un rho - m_n), the rows of L give w0 = rho - 2P (the
    // acoustic-free row), w3 = P + X, w4 = P - X, and the shear rows
    // w1 = sl (m_l - u_l rho), w2 = sm (m_m - u_m rho).
    __device__ __forceinline__ void project(const double q[5], double w[5]) const {
        using B = Basis<AXIS>;
        const double r = q[0];
        const double e = fma(-u[0], q[1], fma(-u[1], q[2], fma(-u[2], q[3], q[4])));
        const double P = b2 * fma(hq2, r, e);
        const double X = fma(xn, r, -x1 * q[1 + B::nd]);
        w[0] = fma(-2.0, P, r);
        w[1] = fma(-ul, r, B::sl * q[1 + B::li]);
        w[2] = fma(-um, r, B::sm * q[1 + B::mi]);
        w[3] = P + X;
        w[4] = P - X;
    }

    // q = base + R w.  Every column of R carries u in the momentum rows
    // except the acoustic -+c on the normal and the shear units, so
    // q_m = u q_rho + (the rest).
    __device__ __forceinline__ void back(const double base[5], const double w[5],
                                         double q[5]) const {
        using B = Basis<AXIS>;
        const double sw = w[3] + w[4];
        const double r = w[0] + sw;
        const double dw = w[4] - w[3];
        q[0] = base[0] + r;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d == B::nd) q[1 + d] = fma(u[d], r, fma(c, dw, base[1 + d]));
            else if (d == B::li) q[1 + d] = fma(u[d], r, fma(B::sl, w[1], base[1 + d]));
            else q[1 + d] = fma(u[d], r, fma(B::sm, w[2], base[1 + d]));
        }
        q[4] = fma(hq2, w[0], fma(ul, w[1], fma(um, w[2], fma(H, sw, fma(cn, dw, base[4])))));
    }
};

// RoeFlux::flux (SF_roe.cpp:20-111) for n = e_AXIS: Roe averages,
// Harten's fix with delta = a~/10 on every wave, and the dissipation
// R |Lambda| L (qR - qL) with R, L of the characteristic basis at the
// state (rho~, rho~ u~, rho~ h~) -- the reference's energy slot holds
// rho~ h~, so that basis has sound speed sqrt(gamma) a~ -- and the wave
// speeds taken in the reference's order (u_n, u_n, u_n, u_n + a~,
// u_n - a~) against the basis columns (the fourth is its u_n - c wave).
template <int AXIS, int NR = 2>
__device__ __forceinline__ void roe(const double qL[5], const double qR[5], double gamma,
                                    double out[5], unsigned& flags) {
    constexpr int ND = Basis<AXIS>::nd;
    const double gm1 = gamma - 1.0;
    const Legacy l = legacy_state<NR>(qL, gamma), r = legacy_state<NR>(qR, gamma);
    if (!l.ok || !r.ok) flags |= kFlagFlux;
    const double hL = (qL[4] + l.p) * l.inv_rho, hR = (qR[4] + r.p) * r.inv_rho;
    const double sL = fsqrt<NR>(qL[0]), sR = fsqrt<NR>(qR[0]);
    const double inv = frcp<NR>(sL + sR);
    double ut[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) ut[d] = fma(sL, l.u[d], sR * r.u[d]) * inv;
    const double ht = fma(sL, hL, sR * hR) * inv;
    const double q2t = dot3(ut, ut);
    const double a2 = gm1 * fma(-0.5, q2t, ht);
    if (!(a2 > 0.0)) flags |= kFlagFlux;
    const double at = fsqrt<NR>(a2);
    const double unt = ut[ND];
    const double delta = 0.1 * at;
    auto fix = [delta](double lam) {
        const double v = fabs(lam);
        return v < 2.0 * delta ? 0.5 * fma(v * v, frcp<NR>(2.0 * delta), delta) : v;
    };
    const double lam0 = fix(unt), lam3 = fix(unt + at), lam4 = fix(unt - at);
    const double rt = sL * sR;
    double qt[5];
    qt[0] = rt;
#pragma unroll
    for (int d = 0; d < 3; ++d) qt[1 + d] = rt * ut[d];
    qt[4] = rt * fma(a2, frcp<NR>(gm1), 0.5 * q2t);
    const CharBasis<AXIS, NR> cb(qt, gamma, flags);
    double dq[5], al[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) dq[v] = qR[v] - qL[v];
    cb.project(dq, al);
    al[0] *= lam0;
    al[1] *= lam0;
    al[2] *= lam0;
    al[3] *= lam3;
    al[4] *= lam4;
    const double zero[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double dis[5];
    cb.back(zero, al, dis);
    double fL[5], fR[5];
    euler_flux<ND>(qL, l, fL);
    euler_flux<ND>(qR, r, fR);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[v] = 0.5 * (fL[v] + fR[v] - dis[v]);
}

// LaxWendroffFlux::flux (SF_lw.cpp:17-40): the physical flux of the
// Richtmyer half state q* = (qL + qR)/2 - (lambda/2)(F(qR) - F(qL)),
// lambda = dt / spacing with the step's dt.
template <int ND, int NR = 2>
__device__ __forceinline__ void lax_wendroff(const double qL[5], const double qR[5],
                                             double gamma, double lambda, double out[5],
                                             unsigned& flags) {
    const Legacy l = legacy_state<NR>(qL, gamma), r = legacy_state<NR>(qR, gamma);
    if (!l.ok || !r.ok || !(lambda > 0.0)) flags |= kFlagFlux;
    double fL[5], fR[5];
    euler_flux<ND>(qL, l, fL);
    euler_flux<ND>(qR, r, fR);
    double qh[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) qh[v] = fma(-0.5 * lambda, fR[v] - fL[v], 0.5 * (qL[v] + qR[v]));
    const Legacy h = legacy_state<NR>(qh, gamma);
    if (!h.ok) flags |= kFlagFlux;
    euler_flux<ND>(qh, h, out);
}

// Flux ids (SF_FLUX_*): 0 Rusanov, 1 HLLC, 2 Steger-Warming,
// 3 Lax-Friedrichs, 4 Roe, 5 Lax-Wendroff (which reads lw = dt / spacing).
template <int AXIS, int FLUX, int NR = 2>
__device__ __forceinline__ void riemann_flux(const double qL[5], const double qR[5],
                                             double gamma, double lw, double out[5],
                                             unsigned& flags) {
    constexpr int nd = Basis<AXIS>::nd;
    if constexpr (FLUX == 1) hllc<nd, NR>(qL, qR, gamma, out, flags);
    else if constexpr (FLUX == 2) steger_warming<nd, NR>(qL, qR, gamma, out, flags);
    else if constexpr (FLUX == 3) lax_friedrichs<nd, NR>(qL, qR, gamma, out, flags);
    else if constexpr (FLUX == 4) roe<AXIS, NR>(qL, qR, gamma, out, flags);
    else if constexpr (FLUX == 5) lax_wendroff<nd, NR>(qL, qR, gamma, lw, out, flags);
    else rusanov<nd, NR>(qL, qR, gamma, out, flags);
}

// Flux::characteristicWENOFaceFlux<NS> (SF_WENO.h:185-245) on a face of
// axis AXIS whose cofactor is area * e_AXIS.  st[s][v] holds the stencil
// nodes at offsets 1-NS/2 .. NS/2 around the face; base(side, q) gives the
// node on the face's left (side 0, st[NS/2-1]) or right (side 1, st[NS/2])
// once more, after the reconstruction: a caller whose nodes lie in LDS reads
// them again there, so that no register holds them across the
// reconstruction.  Returns the area-weighted flux.
template <int AXIS, int SCHEME, int FLUX, class Base>
__device__ __forceinline__ void face_flux_from(const double (&st)[Stencil<SCHEME>::ns][5],
                                               Base base, double gamma, double area,
                                               double out[5], unsigned& flags, double lw = 0.0) {
    constexpr int NS = Stencil<SCHEME>::ns;
    constexpr int NR = Stencil<SCHEME>::newton;
    // the characteristic basis of the face average (SF_WENO.h:207-211), from
    // twice the average
    double qa[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) qa[v] = st[NS / 2 - 1][v] + st[NS / 2][v];
    const CharBasis<AXIS, NR> cb(qa, gamma, flags);
    double ch[5][NS - 1];
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) {
        double dq[5], w[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) dq[v] = st[s + 1][v] - st[s][v];
        cb.project(dq, w);
#pragma unroll
        for (int v = 0; v < 5; ++v) ch[v][s] = w[v];
    }
    double wL[5], wR[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) recon_pair<SCHEME, NR>(ch[v], wL[v], wR[v], flags);
    double qb[5], qL[5], qR[5];
    base(0, qb);
    cb.back(qb, wL, qL);
    base(1, qb);
    cb.back(qb, wR, qR);
    double f[5];
    riemann_flux<AXIS, FLUX, NR>(qL, qR, gamma, lw, f, flags);
#pragma unroll
    for (int v = 0; v < 5; ++v) out[v] = f[v] * area;
}

// face_flux_from with the two nodes taken from the stencil.
template <int AXIS, int SCHEME, int FLUX>
__device__ __forceinline__ void face_flux(const double (&st)[Stencil<SCHEME>::ns][5],
                                          double gamma, double area, double out[5],
                                          unsigned& flags, double lw = 0.0) {
    constexpr int NS = Stencil<SCHEME>::ns;
    face_flux_from<AXIS, SCHEME, FLUX>(
        st,
        [&st](int side, double (&q)[5]) {
#pragma unroll
            for (int v = 0; v < 5; ++v) q[v] = st[NS / 2 - 1 + side][v];
        },
        gamma, area, out, flags, lw);
}

}  // namespace sfamd
