// ws_device.h -- device-side building blocks of the inviscid RHS (FP64).
//
// Two forms of each scalar kernel live here:
//   *_ref   the reference's operation order with contraction disabled, so that a
//           kernel built from them reproduces the CPU restatement bit for bit;
//   *_fast  the form the tiled kernels use: WENO smoothness written through
//           forward differences, product weights through prefix/suffix
//           products, and the division deferred so that the positive and
//           negative reconstructions of a face share one.
#pragma once

#include <hip/hip_runtime.h>

#include "ws_internal.h"

namespace ws {

__device__ __forceinline__ size_t fidx(uint32_t pitch, int nyg, int x, int y, int z)
{
    return (size_t)x + (size_t)pitch * ((size_t)y + (size_t)nyg * (size_t)z);
}

__device__ __forceinline__ size_t sidx(uint32_t pitch, int ny, int nz, int x, int y, int z, int m)
{
    return (size_t)x + (size_t)pitch * ((size_t)y + (size_t)ny * ((size_t)z + (size_t)nz * (size_t)m));
}

// ---------------------------------------------------------------------------
// Reference-order forms (bitwise anchor)
// ---------------------------------------------------------------------------

// WENO7-SYMBO positive reconstruction, OCFD_Schemes.cpp:306-368; s[0..7] = f(i-4..i+3),
// result at face i-1/2.  `R` is an index map so that the negative rule reuses the text:
// the negative reconstruction (OCFD_Schemes.cpp:491-553) is the positive rule on the
// reversed window, which is exactly how the reference spells it index by index.
template <bool REV>
__device__ __forceinline__ double weno_ref(const double *w)
{
#pragma clang fp contract(off)
    auto s = [&](int k) -> double { return REV ? w[7 - k] : w[k]; };
    double S0 = 0.0, S1 = 0.0, S2 = 0.0, S3 = 0.0, S4 = 0.0, t, t1;
    t =  -2.0*s(0) +  9.0*s(1) - 18.0*s(2) + 11.0*s(3); S0 += 720.0*t*t;
    t =       s(1) -  6.0*s(2) +  3.0*s(3) +  2.0*s(4); S1 += 720.0*t*t;
    t =  -2.0*s(2) -  3.0*s(3) +  6.0*s(4) -      s(5); S2 += 720.0*t*t;
    t = -11.0*s(3) + 18.0*s(4) -  9.0*s(5) +  2.0*s(6); S3 += 720.0*t*t;
    t = -26.0*s(4) + 57.0*s(5) - 42.0*s(6) + 11.0*s(7); S4 += 720.0*t*t;

    t = -6.0*s(0) + 24.0*s(1) - 30.0*s(2) + 12.0*s(3); S0 += 780.0*t*t;
    t =                          6.0*s(2) - 12.0*s(3) +  6.0*s(4); S1 += 780.0*t*t;
    t =                          6.0*s(3) - 12.0*s(4) +  6.0*s(5); S2 += 780.0*t*t;
    t = 12.0*s(3) - 30.0*s(4) + 24.0*s(5) -  6.0*s(6); S3 += 780.0*t*t;
    t = 18.0*s(4) - 48.0*s(5) + 42.0*s(6) - 12.0*s(7); S4 += 780.0*t*t;

    t = -6.0*s(0) + 18.0*(s(1) - s(2)) + 6.0*s(3); S0 += 781.0*t*t;
    t = -6.0*s(1) + 18.0*(s(2) - s(3)) + 6.0*s(4); S1 += 781.0*t*t;
    t = -6.0*s(2) + 18.0*(s(3) - s(4)) + 6.0*s(5); S2 += 781.0*t*t;
    t = -6.0*s(3) + 18.0*(s(4) - s(5)) + 6.0*s(6); S3 += 781.0*t*t;
    t = -6.0*s(4) + 18.0*(s(5) - s(6)) + 6.0*s(7); S4 += 781.0*t*t;

    t  = fmax(S0, S1);
    t1 = fmax(S2, S3);
    t  = fmax(t, t1);
    S4 = fmax(t, S4);
    {
        double t2, t3;
        t  = (0.0401954833730)*(2.592e-6+S1)*(2.592e-6+S2)*(2.592e-6+S3)*(2.592e-6+S4);
        t1 = (0.2493800006710)*(2.592e-6+S0)*(2.592e-6+S2)*(2.592e-6+S3)*(2.592e-6+S4);
        t2 = (0.4802686256260)*(2.592e-6+S0)*(2.592e-6+S1)*(2.592e-6+S3)*(2.592e-6+S4);
        t3 = (0.2009775476730)*(2.592e-6+S0)*(2.592e-6+S1)*(2.592e-6+S2)*(2.592e-6+S4);
        S4 = (0.0291783426580)*(2.592e-6+S0)*(2.592e-6+S1)*(2.592e-6+S2)*(2.592e-6+S3);
        S3 = t3; S2 = t2; S1 = t1; S0 = t;
    }
    t1 = 0.0;
    t = -3.0*s(0) + 13.0*s(1) - 23.0*s(2) + 25.0*s(3); t1 += S0*t;
    t =      s(1) -  5.0*s(2) + 13.0*s(3) +  3.0*s(4); t1 += S1*t;
    t =     -s(2) +  7.0*s(3) +  7.0*s(4) -      s(5); t1 += S2*t;
    t =  3.0*s(3) + 13.0*s(4) -  5.0*s(5) +      s(6); t1 += S3*t;
    t = 25.0*s(4) - 23.0*s(5) + 13.0*s(6) -  3.0*s(7); t1 += S4*t;
    t1 /= (12.0*(S0+S1+S2+S3+S4));
    return t1;
}

// Steger-Warming split, canonical form (OCFD_NS_Jacobian3d.cpp:69-127), no contraction.
__device__ __forceinline__ void split_ref(const KParams &k, double d, double u, double v, double w,
                                          double cc, double A1, double A2, double A3,
                                          double fp[5], double fm[5])
{
#pragma clang fp contract(off)
    double ss = sqrt(A1*A1 + A2*A2 + A3*A3);
    double Ak1 = A1 / ss, Ak2 = A2 / ss, Ak3 = A3 / ss;
    double vs = A1*u + A2*v + A3*w;
    double E1 = vs, E2 = vs - cc*ss, E3 = vs + cc*ss;
    double eps2 = k.eps2;
    double E1P = (E1 + sqrt(E1*E1 + eps2)) * 0.50;
    double E2P = (E2 + sqrt(E2*E2 + eps2)) * 0.50;
    double E3P = (E3 + sqrt(E3*E3 + eps2)) * 0.50;
    double E1M = E1 - E1P, E2M = E2 - E2P, E3M = E3 - E3P;
    double tmp0 = d / (2.0*k.gamma);
    double uc1 = u - cc*Ak1, uc2 = u + cc*Ak1;
    double vc1 = v - cc*Ak2, vc2 = v + cc*Ak2;
    double wc1 = w - cc*Ak3, wc2 = w + cc*Ak3;
    double vvc1 = (uc1*uc1 + vc1*vc1 + wc1*wc1) * 0.50;
    double vvc2 = (uc2*uc2 + vc2*vc2 + wc2*wc2) * 0.50;
    double vv = (k.gamma - 1.0) * (u*u + v*v + w*w);
    double W2 = k.c3*cc*cc;
    const double C1 = k.c1;
    fp[0] = tmp0 * (C1*E1P + E2P + E3P);
    fp[1] = tmp0 * (C1*E1P*u + E2P*uc1 + E3P*uc2);
    fp[2] = tmp0 * (C1*E1P*v + E2P*vc1 + E3P*vc2);
    fp[3] = tmp0 * (C1*E1P*w + E2P*wc1 + E3P*wc2);
    fp[4] = tmp0 * (E1P*vv + E2P*vvc1 + E3P*vvc2 + W2*(E2P + E3P));
    fm[0] = tmp0 * (C1*E1M + E2M + E3M);
    fm[1] = tmp0 * (C1*E1M*u + E2M*uc1 + E3M*uc2);
    fm[2] = tmp0 * (C1*E1M*v + E2M*vc1 + E3M*vc2);
    fm[3] = tmp0 * (C1*E1M*w + E2M*wc1 + E3M*wc2);
    fm[4] = tmp0 * (E1M*vv + E2M*vvc1 + E3M*vvc2 + W2*(E2M + E3M));
}

// SSP-RK3 stage value of one conserved component (src/solver/OCFD_time.cpp:15-65) in the
// reference's order with contraction off: fnv the step's initial state, fv the stage's
// current f (unused in stage 1), duv the RHS.  Shared by the stage kernels and the RHS
// launch that applies the stage itself, so both give the same bits.
template <int KRK>
__device__ __forceinline__ double rk3_stage_value(double fnv, double fv, double duv, double dt)
{
#pragma clang fp contract(off)
    if (KRK == 1) return fnv + dt * duv;
    if (KRK == 2) {
        const double t1 = 3.0 / 4.0, t2 = 1.0 / 4.0;
        return t1 * fnv + t2 * (fv + dt * duv);
    }
    const double t1 = 1.0 / 3.0, t2 = 2.0 / 3.0;
    return t1 * fnv + t2 * (fv + dt * duv);
}

// du + this direction's flux difference, without contraction: a launch that adds to du and
// one that applies the RK3 stage to the sum then hold the same bits whatever the compiler
// fuses in either.
__device__ __forceinline__ double acc_sum(double duv, double val)
{
#pragma clang fp contract(off)
    return duv + val;
}

// Primitives of one cell's conserved values r (get_duvwT, src/kernels/commen_kernel.cpp:78-110)
// with contraction off: e is the internal energy per volume, T = e / (d Cv).  Shared by the
// stage kernel and the RHS launch that derives the primitives itself.
struct CellPrims {
    double d, u, v, w, e, T;
};

__device__ __forceinline__ CellPrims cell_primitives(const double r[5], double cv)
{
#pragma clang fp contract(off)
    CellPrims p;
    p.d = r[0];
    p.u = r[1] / p.d;
    p.v = r[2] / p.d;
    p.w = r[3] / p.d;
    p.e = r[4] - 0.5 * p.d * (p.u * p.u + p.v * p.v + p.w * p.w);
    p.T = p.e / (p.d * cv);
    return p;
}

// Conserved values re-derived from the primitives on a boundary plane (OCFD_bc,
// src/boundary/OCFD_boundary.cpp:18-92), contraction off.
__device__ __forceinline__ void plane_conserved(const CellPrims &p, double cv, double r[5])
{
#pragma clang fp contract(off)
    r[0] = p.d;
    r[1] = p.u * p.d;
    r[2] = p.v * p.d;
    r[3] = p.w * p.d;
    r[4] = p.d * ((p.u * p.u + p.v * p.v + p.w * p.w) * 0.5 + cv * p.T);
}

// ---------------------------------------------------------------------------
// Fast forms (tiled kernels)
// ---------------------------------------------------------------------------

// Nonlinear weights are homogeneous of degree four in (eps + S_k), so the indicators may be
// scaled freely.  The FP64 form scales them by 1/(781*36): the third-difference term
// (781*36 D3^2) becomes a plain square, the first-derivative term (720) takes
// sqrt(720/(781*36)) in its coefficients and the second-difference term (780*36)
// sqrt(780/781), and eps becomes 2.592e-6/(781*36).  The FP32 form keeps the 1/720 scale
// (eps 3.6e-9): at 1/(781*36) the product of four (eps + S) factors of a smooth window would
// fall below FP32's normal range.
constexpr double kD0 = 0.0401954833730;
constexpr double kD1 = 0.2493800006710;
constexpr double kD2 = 0.4802686256260;
constexpr double kD3 = 0.2009775476730;
constexpr double kD4 = 0.0291783426580;
constexpr double kEpsS = 2.592e-6 / (781.0 * 36.0);
constexpr double kAS = 0.160025606145638858;    // sqrt(720 / (781 * 36))
constexpr double kBS = 0.999359590072005084;    // sqrt(780 / 781)
// linear weights over the central one
constexpr double kR0 = kD0 / kD2, kR1 = kD1 / kD2, kR3 = kD3 / kD2, kR4 = kD4 / kD2;

// Reciprocal of a positive normal number: the hardware estimate (24 bits) and one
// third-order step, r (1 + e + e^2) with e = 1 - x r, whose remainder e^3 is below 2^-69:
// one instruction less than two Newton steps, error within an ulp.
__device__ __forceinline__ double recip_nr(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// Square root of a positive normal number: reciprocal-square-root estimate refined
// with one coupled Newton step on (sqrt, 1/(2 sqrt)) and a final residual correction.
__device__ __forceinline__ double sqrt_nr(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    const double d = fma(-g, g, x);
    return fma(d, h, g);
}

// Square root of a positive normal number and its reciprocal: the reciprocal-square-root
// estimate y (24 bits) and one third-order step, with e = 1 - x y^2: sqrt(x) = x y (1 + e/2 +
// 3/8 e^2), 1/sqrt(x) = y (1 + e/2 + 3/8 e^2); the remainder 5/16 e^3 is below 2^-70.  Two
// instructions fewer than sqrt_nr; error within an ulp.
__device__ __forceinline__ double sqrt_h(double x)
{
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rsq(x), g = x * y;
    const double e = fma(-g, y, 1.0);
    return fma(g * e, fma(0.375, e, 0.5), g);
}

__device__ __forceinline__ void sqrt_rsqrt_h(double x, double &root, double &rcp)
{
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rsq(x), g = x * y;
    const double e = fma(-g, y, 1.0), p = fma(0.375, e, 0.5);
    root = fma(g * e, p, g);
    rcp = fma(y * e, p, y);
}

// K consecutive faces from K+7 points s[0..K+6] (face j uses s[j..j+7]); face j's value is
// base[j] + kNum num[j] / den[j].  The forward differences and the squared third differences
// (eps added) are formed once per point and shared by the K faces.
//
// Candidate k covers the window's points k .. k+3.  Its first-derivative term a_k, its
// second-derivative term b_k and its value's distance from the base point w3, c_k = 12 (q_k -
// w3), are (unscaled, D1_i, D2_i, D3_i, D4_i the forward differences from point i)
//   a0 = 6 D1_2 + 3 D2_1 + 2 D3_0    b0 = D2_1 + D3_0    c0 = a0 + b0
//   a1 = 6 D1_2 + 3 D2_2 - D3_1      b1 = D2_2           c1 = a1 + b1
//   a2 = 6 D1_2 + 3 D2_2 - D3_2      b2 = D2_3           c2 = a2 + b1
//   a3 = 6 D1_3 - 3 D2_3 + 2 D3_3    b3 = D2_3 - D3_3    c3 = a3 + b3
//   a4 = a3 + 11 D4_3                b4 = b3 - 2 D4_3    c4 = c3 - 3 D4_3
// Each of candidates 0 to 3 is built from differences of its own four points only, so beside
// a jump the candidates that do not cross it hold no value of the jump's size, and the face
// keeps an error of an ulp of the smooth side whatever the jump.  Candidate 4 goes over
// candidate 3: a jump inside 3 and outside 4 lies between points 3 and 4, where the cap on
// e4 leaves candidate 4 no more weight than the one with the largest indicator.  (Building all
// candidates from the central one by D4_0 .. D4_3 takes six instructions fewer per face and
// side but cancels the jump: 3e-14 of the quiet side's value at a ratio of 1e2, 3e-12 at 1e4,
// 3e-4 at 1e12, against 1.2e-16 at any ratio.)
// With d_k the linear weights over the central one, e_k = eps + S_k and P = e0 e1 e2 e3 e4,
// D = sum d_k P / e_k and N = sum d_k c_k P / e_k are formed in pairs (0, 1) and (3, 4).
// Bound by FP64 VALU issue (one instruction per four cycles), so the count is what matters:
// 68 instructions per face and side with K = 2, against 86 with every candidate built by itself
// and 62 for the central form above (a whole RHS of 600x256x128 2.19 ms, by the central form
// 2.09; an RK3 step of 600x128x128 3.89 ms, 3.76).
constexpr double kRho = kAS / kBS;              // c_k from the scaled a_k and b_k
constexpr double kNum = 1.0 / (12.0 * kAS);     // c_k are formed kAS times

template <bool REV, int K, typename Load>
__device__ __forceinline__ void weno_k(Load ld, double (&num)[K], double (&den)[K], double (&base)[K])
{
    // Every fused multiply-add here is written out: implicit contraction could fuse a shared
    // difference differently at different positions j, and a face computed by two threads
    // (at a tile edge) must come out bit for bit the same in both.
#pragma clang fp contract(off)
    constexpr int NP = K + 7;
    constexpr double SD = REV ? -1.0 : 1.0;     // odd differences of the reversed window change sign
    double s[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) s[i] = ld(i);
    double D1[NP - 1], D2[NP - 2], D3[NP - 3], C3[NP - 3], G[K + 1], B[K + 2];
#pragma unroll
    for (int i = 0; i < NP - 1; ++i) D1[i] = s[i + 1] - s[i];
#pragma unroll
    for (int i = 0; i < NP - 2; ++i) D2[i] = D1[i + 1] - D1[i];
#pragma unroll
    for (int i = 0; i < NP - 3; ++i) { D3[i] = D2[i + 1] - D2[i]; C3[i] = fma(D3[i], D3[i], kEpsS); }
    // the scaled first differences before and after each base point, and the scaled second
    // differences of the window's inner points
    constexpr int G0 = REV ? 3 : 2, B0 = REV ? 2 : 1;
#pragma unroll
    for (int i = 0; i < K + 1; ++i) G[i] = (6.0 * SD * kAS) * D1[G0 + i];
#pragma unroll
    for (int i = 0; i < K + 2; ++i) B[i] = kBS * D2[B0 + i];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        // differences of the window as the rule sees it (odd ones without their sign)
        auto g1 = [&](int k) { return G[(REV ? j + 6 - k : j + k) - G0]; };
        auto d2 = [&](int k) { return D2[REV ? j + 5 - k : j + k]; };
        auto b = [&](int k) { return B[(REV ? j + 5 - k : j + k) - B0]; };
        auto d3 = [&](int k) { return D3[REV ? j + 4 - k : j + k]; };
        auto c3 = [&](int k) { return C3[REV ? j + 4 - k : j + k]; };
        const double d4 = REV ? D3[j + 1] - D3[j] : D3[j + 4] - D3[j + 3];
        const double g12 = fma(3.0 * kAS, d2(2), g1(2));
        const double a0 = fma(2.0 * SD * kAS, d3(0), fma(3.0 * kAS, d2(1), g1(2)));
        const double a1 = fma(-SD * kAS, d3(1), g12);
        const double a2 = fma(-SD * kAS, d3(2), g12);
        const double a3 = fma(2.0 * SD * kAS, d3(3), fma(-3.0 * kAS, d2(3), g1(3)));
        const double a4 = fma(11.0 * kAS, d4, a3);
        const double b1 = b(2), b2 = b(3);
        const double b0 = fma(SD * kBS, d3(0), b(1));
        const double b3 = fma(-SD * kBS, d3(3), b2);
        const double b4 = fma(-2.0 * kBS, d4, b3);
        // e_k = eps + S_k (eps rides in C3)
        const double e0 = fma(a0, a0, fma(b0, b0, c3(0)));
        const double e1 = fma(a1, a1, fma(b1, b1, c3(1)));
        const double e2 = fma(a2, a2, fma(b2, b2, c3(2)));
        const double e3 = fma(a3, a3, fma(b3, b3, c3(3)));
        double e4 = fma(a4, a4, fma(b4, b4, c3(4)));
        e4 = fmax(fmax(fmax(e0, e1), fmax(e2, e3)), e4);
        const double q0 = fma(kRho, b0, a0), q1 = fma(kRho, b1, a1), q2 = fma(kRho, b1, a2);
        const double q3 = fma(kRho, b3, a3), q4 = fma(-3.0 * kAS, d4, q3);
        base[j] = s[REV ? j + 4 : j + 3];
        const double t0 = kR0 * e1, t1 = kR1 * e0, t3 = kR3 * e4, t4 = kR4 * e3;
        const double N01 = fma(q0, t0, q1 * t1), N34 = fma(q3, t3, q4 * t4);
        const double p01 = e0 * e1, p34 = e3 * e4, q34 = e2 * p01;
        num[j] = fma(p34, fma(e2, N01, q2 * p01), q34 * N34);
        den[j] = fma(p34, fma(e2, t0 + t1, p01), q34 * (t3 + t4));
    }
}

// The value of a face from its two halves (weno_k<false> and weno_k<true>), merged over one
// reciprocal.
__device__ __forceinline__ double face_merge(double nP, double dP, double bP, double nM, double dM, double bM)
{
#pragma clang fp contract(off)
    return fma(fma(nP, dM, nM * dP), kNum * recip_nr(dP * dM), bP + bM);
}

// One face of weno_k from the 8-point window q[0..7]: base + kNum num / den is its value.
template <bool REV>
__device__ __forceinline__ void face64(const double *q, double &num, double &den, double &base)
{
    double n[1], d[1], b[1];
    weno_k<REV, 1>([&](int i) { return q[i]; }, n, d, b);
    num = n[0];
    den = d[0];
    base = b[0];
}

// Mixed-precision form of weno_k: the window stays FP64 in LDS; its first differences
// are formed in FP64 and rounded to FP32, and everything after that (second and third
// differences, smoothness, weights, candidates) runs in FP32 on values taken relative to
// the face's base point w3.  The face value is base[j] + corr[j]: base in FP64, the FP32
// correction carries an error relative to the local variation of the window, not to the
// size of the flux.
//
// Range check: the weights are products of four (eps + S_k) factors, homogeneous of degree
// eight in the window's differences, and the numerator of degree nine.  D is at least
// d_4 eps^4 (about 5e-36 with eps = 3.6e-9), so it never falls below FP32's normal range,
// but it overflows once the window's first differences reach a few hundred (a strong
// discontinuity of the split flux); N may overflow a little earlier.  Bit j of `bad` is set
// unless |N| + D <= 2^125 (so that D, 1/D and N are normal numbers): the caller then
// recomputes that face in FP64 (weno_k), so FP32 weights are used only where they are
// representable.  Below that limit the FP32 correction's error stays relative to the
// window's variation (no catastrophic cancellation: the indicators are sums of squares
// and the weights a convex combination), so no other check is needed.
template <bool REV, int K, typename Load>
__device__ __forceinline__ void weno_k_mixed(Load ld, double (&base)[K], float (&corr)[K], unsigned &bad)
{
    // explicit FMAs only, as in weno_k: the same face must round the same at every position j
#pragma clang fp contract(off)
    bad = 0;
    constexpr int NP = K + 7;
    constexpr float fD0 = (float)kD0, fD1 = (float)kD1, fD2 = (float)kD2, fD3 = (float)kD3, fD4 = (float)kD4;
    // second and third differences carry sqrt(39): the 780-term of the indicators (39 in units
    // of the 720-term) becomes a plain square, and the other terms take 1/sqrt(39) in their
    // constant coefficients
    constexpr float fR = 6.2449979983983983f;          // sqrt(39)
    constexpr float fIR = 0.16012815380508713f;        // 1/sqrt(39)
    constexpr float fC = 39.05f / 39.0f, fEps = 3.6e-9f;
    double s[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) s[i] = ld(i);
    float D1[NP - 1], D2[NP - 2], D3[NP - 3], G1[NP - 1], C3[NP - 3], B2[NP - 2];
#pragma unroll
    for (int i = 0; i < NP - 1; ++i) { D1[i] = (float)(s[i + 1] - s[i]); G1[i] = 6.0f * D1[i]; }
#pragma unroll
    for (int i = 0; i < NP - 2; ++i) { D2[i] = (D1[i + 1] - D1[i]) * fR; B2[i] = D2[i] * D2[i]; }
#pragma unroll
    for (int i = 0; i < NP - 3; ++i) { D3[i] = D2[i + 1] - D2[i]; C3[i] = fmaf(fC * D3[i], D3[i], fEps); }
#pragma unroll
    for (int j = 0; j < K; ++j) {
        auto i1 = [&](int k) { return REV ? j + 6 - k : j + k; };
        auto i2 = [&](int k) { return REV ? j + 5 - k : j + k; };
        auto i3 = [&](int k) { return REV ? j + 4 - k : j + k; };
        const float sb = REV ? -fIR : fIR;
        const float a0 = fmaf(11.0f * fIR, D3[i3(0)], fmaf(sb * 15.0f, D2[i2(0)], G1[i1(0)]));
        const float a1 = fmaf(2.0f * fIR, D3[i3(1)], fmaf(sb * 9.0f, D2[i2(1)], G1[i1(1)]));
        const float a2 = fmaf(-1.0f * fIR, D3[i3(2)], fmaf(sb * 3.0f, D2[i2(2)], G1[i1(2)]));
        const float a3 = fmaf(2.0f * fIR, D3[i3(3)], fmaf(sb * -3.0f, D2[i2(3)], G1[i1(3)]));
        const float a4 = fmaf(11.0f * fIR, D3[i3(4)], fmaf(sb * -9.0f, D2[i2(4)], G1[i1(4)]));
        const float b0 = REV ? fmaf(-2.0f, D3[j + 4], D2[j + 5]) : fmaf(2.0f, D3[j], D2[j]);
        const float b3 = REV ? D2[j + 2] + D3[j + 1] : D2[j + 3] - D3[j + 3];
        const float b4 = REV ? fmaf(2.0f, D3[j], D2[j + 1]) : fmaf(-2.0f, D3[j + 4], D2[j + 4]);
        const float bb1 = REV ? B2[j + 3] : B2[j + 2];
        const float bb2 = REV ? B2[j + 2] : B2[j + 3];
        // e_k = eps + S_k (eps rides in C3)
        const float e0 = fmaf(a0, a0, fmaf(b0, b0, C3[i3(0)]));
        const float e1 = fmaf(a1, a1, bb1 + C3[i3(1)]);
        const float e2 = fmaf(a2, a2, bb2 + C3[i3(2)]);
        const float e3 = fmaf(a3, a3, fmaf(b3, b3, C3[i3(3)]));
        float e4 = fmaf(a4, a4, fmaf(b4, b4, C3[i3(4)]));
        e4 = fmaxf(fmaxf(fmaxf(e0, e1), fmaxf(e2, e3)), e4);
        // candidates relative to the base point w3 in Newton form over the forward
        // differences at each candidate's first point (D2 and D3 carry sqrt(39)); linear
        // weights folded in
        const float sd = REV ? -1.0f : 1.0f;
        auto d1 = [&](int k) { return D1[REV ? j + 6 - k : j + k]; };
        auto d2 = [&](int k) { return D2[REV ? j + 5 - k : j + k]; };
        auto d3 = [&](int k) { return D3[REV ? j + 4 - k : j + k]; };
        const float c0 = fmaf(sd * fD0 * (13.0f / 12.0f) * fIR, d3(0), fmaf(fD0 * (4.0f / 3.0f) * fIR, d2(0), (sd * fD0 * 0.5f) * d1(0)));
        const float c1 = fmaf(sd * fD1 * (1.0f / 4.0f) * fIR, d3(1), fmaf(fD1 * (5.0f / 6.0f) * fIR, d2(1), (sd * fD1 * 0.5f) * d1(1)));
        const float c2 = fmaf(sd * fD2 * (-1.0f / 12.0f) * fIR, d3(2), fmaf(fD2 * (1.0f / 3.0f) * fIR, d2(2), (sd * fD2 * 0.5f) * d1(2)));
        const float c3 = fmaf(sd * fD3 * (1.0f / 12.0f) * fIR, d3(3), fmaf(fD3 * (-1.0f / 6.0f) * fIR, d2(3), (sd * fD3 * 0.5f) * d1(3)));
        const float c4 = fmaf(sd * fD4 * (-1.0f / 4.0f) * fIR, d3(4), fmaf(fD4 * (1.0f / 3.0f) * fIR, d2(4),
                              fmaf(sd * fD4 * -0.5f, d1(4), (sd * fD4) * d1(3))));
        const float p01 = e0 * e1;
        float N = fmaf(c0, e1, c1 * e0);
        float D = fmaf(fD0, e1, fD1 * e0);
        N = fmaf(N, e2, c2 * p01);
        D = fmaf(D, e2, fD2 * p01);
        const float p012 = p01 * e2;
        N = fmaf(N, e3, c3 * p012);
        D = fmaf(D, e3, fD3 * p012);
        const float p0123 = p012 * e3;
        N = fmaf(N, e4, c4 * p0123);
        D = fmaf(D, e4, fD4 * p0123);
        corr[j] = N * __builtin_amdgcn_rcpf(D);
        base[j] = REV ? s[j + 4] : s[j + 3];
        // D >= eps^4 > 2^-126 always, so D and 1/D are normal and N finite when |N| + D <=
        // 2^125 (false for NaN; a finite |N| above 2^125 is sent to FP64 as well)
        const bool ok = fabsf(N) + D <= 4.25352958e+37f;
        bad |= ok ? 0u : (1u << j);
    }
}

// ---- one-sided closures at non-periodic domain faces (the reference's D0_bound) ------
// Reduced WENO5 reconstructions on 5-point windows s0..s4 without linear weights
// (src/boundary/OCFD_bound_Scheme.cpp:540-719, src/kernels/OCFD_Schemes.cpp:1110-1201), in
// the reference's operation order with contraction off.  The full P variant builds its
// first two weights from S1 and S2 before they are assigned (both still 0); that is the
// reference's behaviour and is kept.
__device__ __forceinline__ double bs_sign1(double x) { return x >= 0 ? 1.0 : -1.0; }

__device__ __forceinline__ double bs_minmod2(double a, double b)
{
#pragma clang fp contract(off)
    return 0.5 * (bs_sign1(a) + bs_sign1(b)) * fmin(fabs(a), fabs(b));
}

__device__ __forceinline__ double w5_p(double s0, double s1, double s2, double s3, double s4)
{
#pragma clang fp contract(off)
    const double ep = 1e-6;
    double S0 = 0.0, S1 = 0.0, S2 = 0.0, tmp;
    tmp = s2 - 2.0 * s3 + s4; S0 += 13 * tmp * tmp;
    tmp = 3.0 * s2 - 4.0 * s3 + s4; S0 += 3 * tmp * tmp;
    const double a0 = ((12.0 * ep + S1) * (12.0 * ep + S1)) * ((12.0 * ep + S2) * (12.0 * ep + S2));
    const double q03 = (2.0 * s2 + 5.0 * s3 - s4);
    tmp = s1 - 2.0 * s2 + s3; S1 += 13 * tmp * tmp;
    tmp = s1 - s3; S1 += 3 * tmp * tmp;
    const double a1 = ((12.0 * ep + S0) * (12.0 * ep + S0)) * ((12.0 * ep + S2) * (12.0 * ep + S2));
    const double q13 = (-s1 + 5.0 * s2 + 2.0 * s3);
    tmp = s0 - 2.0 * s1 + s2; S2 += 13 * tmp * tmp;
    tmp = s0 - 4.0 * s1 + 3.0 * s2; S2 += 3 * tmp * tmp;
    const double a2 = ((12.0 * ep + S0) * (12.0 * ep + S0)) * ((12.0 * ep + S1) * (12.0 * ep + S1));
    const double q23 = (2.0 * s0 - 7.0 * s1 + 11.0 * s2);
    return (a0 * q03 + a1 * q13 + a2 * q23) / (6.0 * (a0 + a1 + a2));
}

__device__ __forceinline__ double w5_m(double s0, double s1, double s2, double s3, double s4)
{
#pragma clang fp contract(off)
    const double ep = 1e-6;
    double S0 = 0.0, S1 = 0.0, S2 = 0.0, tmp;
    tmp = s2 - 2.0 * s1 + s0; S0 += 13 * tmp * tmp;
    tmp = 3.0 * s2 - 4.0 * s1 + s0; S0 += 3 * tmp * tmp;
    const double a0 = 1.0 / ((12.0 * ep + S0) * (12.0 * ep + S0));
    const double q03 = (2.0 * s2 + 5.0 * s1 - s0);
    tmp = s3 - 2.0 * s2 + s1; S1 += 13 * tmp * tmp;
    tmp = s3 - s1; S1 += 3 * tmp * tmp;
    const double a1 = 1.0 / ((12.0 * ep + S1) * (12.0 * ep + S1));
    const double q13 = (-s3 + 5.0 * s2 + 2.0 * s1);
    tmp = s4 - 2.0 * s3 + s2; S2 += 13 * tmp * tmp;
    tmp = s4 - 4.0 * s3 + 3.0 * s2; S2 += 3 * tmp * tmp;
    const double a2 = 1.0 / ((12.0 * ep + S2) * (12.0 * ep + S2));
    const double q23 = (2.0 * s4 - 7.0 * s3 + 11.0 * s2);
    return (a0 * q03 + a1 * q13 + a2 * q23) / (6.0 * (a0 + a1 + a2));
}

// single candidate k (weight a_k = 1/(12 ep + S_k)^2 cancels); q is the candidate, S its smoothness
__device__ __forceinline__ double w5_one(double S, double q)
{
#pragma clang fp contract(off)
    const double ep = 1e-6;
    const double a = 1.0 / ((12.0 * ep + S) * (12.0 * ep + S));
    return a * q / (6.0 * a);
}

__device__ __forceinline__ double w5_two(double Sa, double qa, double Sb, double qb)
{
#pragma clang fp contract(off)
    const double ep = 1e-6;
    const double a = 1.0 / ((12.0 * ep + Sa) * (12.0 * ep + Sa));
    const double b = 1.0 / ((12.0 * ep + Sb) * (12.0 * ep + Sb));
    return (a * qa + b * qb) / (6.0 * (a + b));
}

// smoothness of the three WENO5 candidates, in the reference's expression order
__device__ __forceinline__ double w5_S0p(double s2, double s3, double s4)
{
#pragma clang fp contract(off)
    double S = 0.0, tmp;
    tmp = s2 - 2.0 * s3 + s4; S += 13 * tmp * tmp;
    tmp = 3.0 * s2 - 4.0 * s3 + s4; S += 3 * tmp * tmp;
    return S;
}
__device__ __forceinline__ double w5_S1p(double s1, double s2, double s3)
{
#pragma clang fp contract(off)
    double S = 0.0, tmp;
    tmp = s1 - 2.0 * s2 + s3; S += 13 * tmp * tmp;
    tmp = s1 - s3; S += 3 * tmp * tmp;
    return S;
}
__device__ __forceinline__ double w5_S2p(double s0, double s1, double s2)
{
#pragma clang fp contract(off)
    double S = 0.0, tmp;
    tmp = s0 - 2.0 * s1 + s2; S += 13 * tmp * tmp;
    tmp = s0 - 4.0 * s1 + 3.0 * s2; S += 3 * tmp * tmp;
    return S;
}

// P face f (between cells f-1 and f) of a line of n cells; cell(c) gives the split value
// of cell c.  Returns true and the face value when a closure covers the face
// (OCFD_bound_scheme_kernel_p, OCFD_bound_Scheme.cpp:722-807; 5-point windows on cells
// f-3 .. f+1).  hi: the high face's form, 0 none, 1 D0_bound, 2 the fused path's rim kernel
// (split_Jac3d_Stager_Warming_ker_boundary, src/solver/OCFD_NS_Jacobian3d.cpp:1063-1085),
// which extrapolates the last face linearly, 1.5 f(n-1) - 0.5 f(n-2), where D0_bound
// limits the slope with minmod (the same value in exact arithmetic, other roundings).
template <typename Cell>
__device__ __forceinline__ bool closure_p(Cell cell, int n, int f, bool lo, int hi, double &out)
{
#pragma clang fp contract(off)
    if (lo && f <= 3) {
        if (f == 0) {
            out = cell(0);
        } else if (f == 1) {            // lift: candidate 0 on cells f-1 .. f+1
            const double s2 = cell(f - 1), s3 = cell(f), s4 = cell(f + 1);
            out = w5_one(w5_S0p(s2, s3, s4), (2.0 * s2 + 5.0 * s3 - s4));
        } else if (f == 2) {            // lift_plus: candidates 0 and 1
            const double s1 = cell(f - 2), s2 = cell(f - 1), s3 = cell(f), s4 = cell(f + 1);
            out = w5_two(w5_S0p(s2, s3, s4), (2.0 * s2 + 5.0 * s3 - s4), w5_S1p(s1, s2, s3),
                         (-s1 + 5.0 * s2 + 2.0 * s3));
        } else {
            out = w5_p(cell(f - 3), cell(f - 2), cell(f - 1), cell(f), cell(f + 1));
        }
        return true;
    }
    if (hi && f >= n - 2) {
        if (f == n) {
            const double a = cell(n - 1), b = cell(n - 2);
            out = hi == 2 ? 1.5 * a - 0.5 * b : a + 0.5 * bs_minmod2(a - b, a - b);
        } else if (f == n - 1) {        // right_plus: candidates 1 and 2
            const double s0 = cell(f - 3), s1 = cell(f - 2), s2 = cell(f - 1), s3 = cell(f);
            out = w5_two(w5_S1p(s1, s2, s3), (-s1 + 5.0 * s2 + 2.0 * s3), w5_S2p(s0, s1, s2),
                         (2.0 * s0 - 7.0 * s1 + 11.0 * s2));
        } else {
            out = w5_p(cell(f - 3), cell(f - 2), cell(f - 1), cell(f), cell(f + 1));
        }
        return true;
    }
    return false;
}

// M face f (OCFD_bound_scheme_kernel_m, OCFD_bound_Scheme.cpp:808-893; windows on cells
// f-2 .. f+2, mirrored candidates).  With the rim kernel's form (hi == 2,
// OCFD_NS_Jacobian3d.cpp:1075-1085) the last two faces both take 0.5 f(n-1) + 0.5 f(n-2),
// so the last cell's M difference vanishes.
template <typename Cell>
__device__ __forceinline__ bool closure_m(Cell cell, int n, int f, bool lo, int hi, double &out)
{
#pragma clang fp contract(off)
    if (lo && f <= 3) {
        if (f == 0) {                   // lift: candidate 2 on cells f .. f+2
            const double s2 = cell(f), s3 = cell(f + 1), s4 = cell(f + 2);
            double S = 0.0, tmp;
            tmp = s4 - 2.0 * s3 + s2; S += 13 * tmp * tmp;
            tmp = s4 - 4.0 * s3 + 3.0 * s2; S += 3 * tmp * tmp;
            out = w5_one(S, (2.0 * s4 - 7.0 * s3 + 11.0 * s2));
        } else if (f == 1) {            // lift_plus: candidates 1 and 2
            const double s1 = cell(f - 1), s2 = cell(f), s3 = cell(f + 1), s4 = cell(f + 2);
            double S1 = 0.0, S2 = 0.0, tmp;
            tmp = s3 - 2.0 * s2 + s1; S1 += 13 * tmp * tmp;
            tmp = s3 - s1; S1 += 3 * tmp * tmp;
            tmp = s4 - 2.0 * s3 + s2; S2 += 13 * tmp * tmp;
            tmp = s4 - 4.0 * s3 + 3.0 * s2; S2 += 3 * tmp * tmp;
            out = w5_two(S1, (-s3 + 5.0 * s2 + 2.0 * s1), S2, (2.0 * s4 - 7.0 * s3 + 11.0 * s2));
        } else {
            out = w5_m(cell(f - 2), cell(f - 1), cell(f), cell(f + 1), cell(f + 2));
        }
        return true;
    }
    if (hi && f >= n - 3) {
        if (f == n) {
            out = hi == 2 ? 0.5 * cell(n - 1) + 0.5 * cell(n - 2) : cell(n - 1);
        } else if (f == n - 1) {
            const double a = cell(n - 1), b = cell(n - 2);
            out = hi == 2 ? 0.5 * a + 0.5 * b : a - 0.5 * bs_minmod2(a - b, a - b);
        } else if (f == n - 2) {        // right_plus: candidates 0 and 1
            const double s0 = cell(f - 2), s1 = cell(f - 1), s2 = cell(f), s3 = cell(f + 1);
            double S0 = 0.0, S1 = 0.0, tmp;
            tmp = s2 - 2.0 * s1 + s0; S0 += 13 * tmp * tmp;
            tmp = 3.0 * s2 - 4.0 * s1 + s0; S0 += 3 * tmp * tmp;
            tmp = s3 - 2.0 * s2 + s1; S1 += 13 * tmp * tmp;
            tmp = s3 - s1; S1 += 3 * tmp * tmp;
            out = w5_two(S0, (2.0 * s2 + 5.0 * s1 - s0), S1, (-s3 + 5.0 * s2 + 2.0 * s1));
        } else {
            out = w5_m(cell(f - 2), cell(f - 1), cell(f), cell(f + 1), cell(f + 2));
        }
        return true;
    }
    return false;
}

// Steger-Warming split in the form the tiled FP64 kernels use: A1..A3 the metric terms, sn = |A|
// and rsn = 1/|A| supplied by the caller (constants when metrics are uniform).  The smoothed
// eigenvalues of a half are (E_i +- S_i) / 2 with E_i = vs, vs - cs, vs + cs (vs = A.u, cs = c |A|)
// and S_i = sqrt(E_i^2 + eps^2).  Each half is half the physical flux plus or minus a term of the
// S_i: the mass flux d vs / 2 +- t (c1 S_1 + S_2 + S_3), the momentum flux f0 u_i + t c/|A| (2 cs +-
// (S_3 - S_2)) A_i, the energy flux t (vs vv + E_2 H_2 + E_3 H_3) +- t (S_1 vv + S_2 H_2 + S_3 H_3)
// with t = d/(4 gamma), H_2,3 = |u|^2/2 + c^2/2 + W2 -+ c vs/|A|.  71 FP64 instructions against the
// 108 of split_mixed (whose shifted velocities u -+ c k are spelled out); a tile splits 25-31 %
// more points than it owns.  What the two halves share rounds alike in both and leaves the sum of
// a face's two values: the RHS's error against 64-bit-mantissa arithmetic is 0.91, 0.90, 0.89 and
// 1.00 of that with split_mixed's form (a jump at rest, Mach 2 blobs, vortices, rough flow); with
// the eigenvalues of each half formed first 0.99, 0.98, 0.97 and 1.00, with the negative ones as
// 2 vs - P_1 and so on 0.97, 0.99, 1.06 and 1.03.
__device__ __forceinline__ void split_fast(const KParams &k, double d, double u, double v, double w,
                                           double cc, double A1, double A2, double A3, double sn,
                                           double rsn, double fp[5], double fm[5])
{
    // contraction off: a point split by two tiles must come out the same in both
#pragma clang fp contract(off)
    const double vs = fma(A3, w, fma(A2, v, A1 * u));
    const double cs = cc * sn;
    const double E2 = vs - cs, E3 = vs + cs;
    // eps2n keeps the radicands positive and normal (a point at rest without smoothing too)
    const double S1 = sqrt_h(fma(vs, vs, k.eps2n));
    const double S2 = sqrt_h(fma(E2, E2, k.eps2n));
    const double S3 = sqrt_h(fma(E3, E3, k.eps2n));
    const double t = d * k.quarter_rcp_gamma;
    const double cr = cc * rsn, cv = cr * vs, tc = t * cr;
    const double q = fma(w, w, fma(v, v, u * u));
    const double vv = k.gm1 * q, H = fma(0.5, q, k.c3h * (cc * cc));
    const double H2 = H - cv, H3 = H + cv;
    const double m = 0.5 * d * vs, ms = fma(k.c1, S1, S2 + S3);
    const double e = t * fma(E3, H3, fma(E2, H2, vs * vv)), es = fma(S3, H3, fma(S2, H2, S1 * vv));
    const double dS = S3 - S2;
    const double gp = tc * fma(2.0, cs, dS), gm = tc * fma(2.0, cs, -dS);
    fp[0] = fma(t, ms, m);
    fp[1] = fma(gp, A1, fp[0] * u);
    fp[2] = fma(gp, A2, fp[0] * v);
    fp[3] = fma(gp, A3, fp[0] * w);
    fp[4] = fma(t, es, e);
    fm[0] = fma(-t, ms, m);
    fm[1] = fma(gm, A1, fm[0] * u);
    fm[2] = fma(gm, A2, fm[0] * v);
    fm[3] = fma(gm, A3, fm[0] * w);
    fm[4] = fma(-t, es, e);
}

// Steger-Warming split of the mixed-precision kernels: k1..k3 = A/|A|.  The mixed
// reconstruction rounds first differences of these values to FP32, where a last-bit change
// of a value can flip a rounding a hundred million times its size, so this form keeps its
// arithmetic.
__device__ __forceinline__ void split_mixed(const KParams &k, double d, double u, double v, double w,
                                           double cc, double A1, double A2, double A3, double sn,
                                           double k1, double k2, double k3, double fp[5], double fm[5])
{
    const double vs = fma(A3, w, fma(A2, v, A1 * u));
    const double cs = cc * sn;
    const double E1 = vs, E2 = vs - cs, E3 = vs + cs;
    // eps2n keeps the radicands positive and normal (a point at rest without smoothing too)
    const double E1P = 0.5 * (E1 + sqrt_nr(fma(E1, E1, k.eps2n)));
    const double E2P = 0.5 * (E2 + sqrt_nr(fma(E2, E2, k.eps2n)));
    const double E3P = 0.5 * (E3 + sqrt_nr(fma(E3, E3, k.eps2n)));
    const double E1M = E1 - E1P, E2M = E2 - E2P, E3M = E3 - E3P;
    const double t0 = d * k.half_rcp_gamma;
    const double ck1 = cc * k1, ck2 = cc * k2, ck3 = cc * k3;
    const double uc1 = u - ck1, uc2 = u + ck1;
    const double vc1 = v - ck2, vc2 = v + ck2;
    const double wc1 = w - ck3, wc2 = w + ck3;
    const double h1 = 0.5 * fma(wc1, wc1, fma(vc1, vc1, uc1 * uc1));
    const double h2 = 0.5 * fma(wc2, wc2, fma(vc2, vc2, uc2 * uc2));
    const double vv = k.gm1 * fma(w, w, fma(v, v, u * u));
    const double W2 = k.c3 * cc * cc;
    // positive part
    {
        const double a = t0 * (k.c1 * E1P), b = t0 * E2P, c = t0 * E3P;
        fp[0] = a + b + c;
        fp[1] = fma(c, uc2, fma(b, uc1, a * u));
        fp[2] = fma(c, vc2, fma(b, vc1, a * v));
        fp[3] = fma(c, wc2, fma(b, wc1, a * w));
        fp[4] = t0 * fma(W2, E2P + E3P, fma(E3P, h2, fma(E2P, h1, E1P * vv)));
    }
    {
        const double a = t0 * (k.c1 * E1M), b = t0 * E2M, c = t0 * E3M;
        fm[0] = a + b + c;
        fm[1] = fma(c, uc2, fma(b, uc1, a * u));
        fm[2] = fma(c, vc2, fma(b, vc1, a * v));
        fm[3] = fma(c, wc2, fma(b, wc1, a * w));
        fm[4] = t0 * fma(W2, E2M + E3M, fma(E3M, h2, fma(E2M, h1, E1M * vv)));
    }
}

}  // namespace ws
