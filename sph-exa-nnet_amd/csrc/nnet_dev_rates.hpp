// Device-side reaction-rate parameterizations for net14 / net86 / net87, evaluated
// cooperatively by the lanes of one workgroup (one particle per workgroup):
//   * one lane per fitted rate (net14: 10, net86/87: 150) computes the forward rate, its
//     reverse from the partition-function ratio, and both T-derivatives;
//   * the six hand-fitted rates (3-alpha, 12C+12C, 12C+16O, 16O+16O, 12C(a,g), 16O(a,g)) with
//     reverses and derivatives: their pow values and those every lane needs (powers of T and of
//     the density) one per lane in one pass, their exp values one per lane in another, then
//     combined by the wavefront (net86 / net87: two groups on each of three wavefronts);
//   * one lane per species computes the Coulomb-corrected binding energy and the screening
//     chemical potential mu/kT.
// A second phase applies screening per rate and scatters into the reaction-list order.
//
// Every expression keeps the operand order and grouping of the reference so that, with FMA
// contraction disabled, the only differences from the reference CPU build are the last-ulp
// differences between the device exp/log/pow and glibc's.
//   net14: parameterization/net14/net14.cpp:40-660, net14_tables.hpp:47-101
//   net86: parameterization/net86/net86.cpp:41-686
//   net87: parameterization/net87/net87.hpp:117-175, net87.cpp:102-141
#pragma once
#include <hip/hip_runtime.h>

#include "nnet_layout.hpp"

namespace nnet_amd
{
namespace phys
{
constexpr double pi       = 3.14159265358979323846264338327950288;
constexpr double Kb       = 1.380658e-16;
constexpr double Na       = 6.022137e23;
constexpr double e2       = 2.306022645e-19;
constexpr double MevToErg = 9.648529392e17;
} // namespace phys

// std::min / std::max semantics (a NaN first operand is returned unchanged)
__device__ __forceinline__ double dmin(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double dmax(double a, double b) { return (a < b) ? b : a; }

// Rate-bin of the partition-function tables (net14_tables.hpp:71-101).
__device__ __forceinline__ int temperature_bin(double T)
{
    const double e[23] = {1.5e8, 2e8, 3e8, 4e8, 5e8, 6e8, 7e8, 8e8, 9e8, 1e9, 1.5e9, 2e9,
                          2.5e9, 3e9, 3.5e9, 4e9, 4.5e9, 5e9, 6e9, 7e9, 8e9, 9e9, 1e10};
    int k = 0;
#pragma unroll
    for (int q = 0; q < 23; ++q)
        k += (T < e[q]) ? 0 : 1;
    // bins are monotone, so the count of edges not above T is the bin (NaN -> 23 as well)
    return k;
}


// Powers of t9 used by the rate expressions (t9 clamped at 10), net14.cpp:196-213.
struct RatePow
{
    double t9r, t9, t92, t93, t95, t912, t913, t923, t932, t943, t953, t9i, t9i13, t9i23, t9i32, t9rm1, t9r32;
    __device__ RatePow(double T, double cbrt_t9) // cbrt_t9: pow(t9, 1/3)
    {
        t9r   = T * 1.0e-09;
        t9    = dmin(10., t9r);
        t92   = t9 * t9;
        t93   = t92 * t9;
        t95   = t92 * t93;
        t912  = sqrt(t9);
        t913  = cbrt_t9;
        t923  = t913 * t913;
        t932  = t9 * t912;
        t943  = t9 * t913;
        t953  = t9 * t923;
        t9i   = 1. / t9;
        t9i13 = 1. / t913;
        t9i23 = 1. / t923;
        t9i32 = 1. / t932;
        t9rm1 = 1. / t9r;
        t9r32 = t9 * sqrt(t9r);
    }
};

// Powers of t9 used by the derivative expressions (no clamp), net14.cpp:341-362.
struct DerivPow
{
    double t9, t92, t93, t94, t95, t912, t913, t923, t932, t943, t952, t953, t9i, t9i2, t9i13, t9i23, t9i32, t9i43,
        t9i52, t9i53;
    __device__ DerivPow(double T, double cbrt_t9) // cbrt_t9: pow(t9, 1/3)
    {
        t9    = T * 1.0e-09;
        t92   = t9 * t9;
        t93   = t92 * t9;
        t94   = t93 * t9;
        t95   = t94 * t9;
        t912  = sqrt(t9);
        t913  = cbrt_t9;
        t923  = t913 * t913;
        t932  = t9 * t912;
        t943  = t9 * t913;
        t952  = t9 * t932;
        t953  = t9 * t923;
        t9i   = 1. / t9;
        t9i2  = t9i * t9i;
        t9i13 = 1. / t913;
        t9i23 = 1. / t923;
        t9i32 = 1. / t932;
        t9i43 = 1. / t943;
        t9i52 = 1. / t952;
        t9i53 = 1. / t953;
    }
};

// ---------------------------------------------------------------------------------------------
// The pow / exp values of the rate phase, one per lane.  A device pow is a chain of about a
// microsecond whatever the number of active lanes, so the phase's time is its number of pow and
// exp passes, not of values: every pow that depends on T and the density alone is a lane of one
// pass, and the exps of the six hand-fitted groups are lanes of another.  Each value comes from
// the reference's argument expression through the same function.  Phase 1 of the rates in one full
// iteration (all groups of a particle alone on its CU): net14 ideal gas 17.0 -> 8.6 us, net86 Helmholtz
// 11.7 -> 7.9, against one pow / exp per use with groups of their own lanes.
// ---------------------------------------------------------------------------------------------
// Lane k of the pow pass: 0, 1: (T/1e9)^(1/3), (T/1e9)^(5/3) of the fitted rates; 2, 3: t9^(1/3) of
// RatePow and DerivPow; 4: the electron-sphere radius (3/4 / (pi ne))^(1/3); 5 + j, j < NP1: pow j
// of the groups 1 (12C + 12C, j < 6) and 2 (12C + 16O), of t9a = t9 / (1 + c t9) with RatePow's t9
// (j = 0, 1, 6, 7) or DerivPow's.
namespace spx
{
constexpr int PF13 = 0, PF53 = 1, PR13 = 2, PD13 = 3, PAE = 4, PL1 = 5;
static_assert(PL1 + NP1 <= 64, "one pow per lane");
} // namespace spx
__device__ __forceinline__ double pow_lane(int k, double T, double rho)
{
    const double tq = T * 1.0e-09, tp = dmin(10., tq);
    const int    j = k - spx::PL1;
    double       num = 1., den = 1.;
    if (k < 2)
        num = T, den = 1.e9;
    else if (k < 4)
        num = k == 2 ? tp : tq;
    else if (k == 4)
        num = 3. / 4., den = phys::pi * (rho * phys::Na / 2.);
    else if (j < spx::NP1)
    {
        num = (j % 6) < 2 && j < 8 ? tp : tq;
        den = 1. + (j < 6 ? 0.0396 : 0.055) * num;
    }
    // exponents in sixths, one byte per lane (the quotient is the rounded exponent: 2/6 is 1/3)
    const uint64_t n = k < 8 ? 0x0505020202020a02ull : k < 16 ? 0x04fe050502fff8feull : 0xfff8ull;
    return pow(num / den, (double)(int8_t)(n >> (8 * (k & 7))) / 6.);
}

// Lane k < NE1 + NE2 of the exp pass: its argument is c X, plus or minus the term of its kind.
//   groups 0 (k < 12), 3 (12, 13), 4 (14 .. 23), 5 (24 .. 33), 2 (34, 35); from pow values: group 1
//   (36, 37) and group 2 (38 .. 41).
// x: which factor X is (XP..: a RatePow power, XQ..: a DerivPow power, XV: the pow value of lane
// src, XV2: its square); kinds: C: c X; D: c X - w, w = t92 / d; S: c X - w^2, w = t9 / d;
// M: c X - t92 d; F: 16O + 16O's four terms; A: c w^2 and B: (c w) w, w = t9 / (1 + 0.055 t9);
// V: c / X; V3: c / X - 2.12e-3 t93; C3: c X - 2.12e-3 t93.
struct SpxArg
{
    double  c, d;
    uint8_t x, kind, src;
};
enum : uint8_t { XPI, XQI, XPI13, XQI13, XPM1, XV, XV2 };
enum : uint8_t { KC, KD, KS, KM, KF, KA, KB, KV, KV3, KC3 };
static __device__ const SpxArg spx_arg[64] = {
    // group 0, triple alpha: r2abe, rbeac, r, rev (RatePow), then the derivative exps (DerivPow)
    {-1.0663, 0, XPI, KC, 0}, {-13.49, 0.009604, XPI13, KD, 0}, {-3.3364, 0, XPI, KC, 0}, {-23.57, 0.055225, XPI13, KD, 0},
    {-24.811, 0, XPI, KC, 0}, {-84.419412e0, 0, XPI, KC, 0},
    {-1.0663, 0, XQI, KC, 0}, {-13.49, 104.123282, XQI13, KM, 0}, {-3.3364, 0, XQI, KC, 0}, {-23.57, 18.10774106, XQI13, KM, 0},
    {-24.811, 0, XQI, KC, 0}, {-84.419412, 0, XQI, KC, 0},
    // group 3, 16O + 16O
    {-135.93, 0, XPI13, KF, 0}, {-135.93e0, 0, XQI13, KF, 0},
    // group 4, 12C(a,g)
    {-32.120, 12.222016, XPI13, KD, 0}, {-32.120, 0, XPI13, KC, 0}, {-27.499, 0, XPI, KC, 0}, {-15.541, 0, XPI, KC, 0},
    {-83.108047, 0, XPM1, KC, 0},
    {-32.120, 3.496, XQI13, KS, 0}, {-32.120, 0, XQI13, KC, 0}, {-27.499, 0, XQI, KC, 0}, {-15.541, 0, XQI, KC, 0},
    {-83.108047, 0, XQI, KC, 0},
    // group 5, 16O(a,g)
    {-39.757, 2.515396, XPI13, KD, 0}, {-10.297, 0, XPI, KC, 0}, {-12.226, 0, XPI, KC, 0}, {-20.093, 0, XPI, KC, 0},
    {-54.93807, 0, XPM1, KC, 0},
    {-39.757, 1.586, XQI13, KS, 0}, {-10.297, 0, XQI, KC, 0}, {-12.226, 0, XQI, KC, 0}, {-20.093, 0, XQI, KC, 0},
    {-54.903255, 0, XQI, KC, 0},
    // group 2, 12C + 16O: the exps that need no pow
    {-0.18, 0, XPI, KA, 0}, {-.18, 0, XPI, KB, 0},
    // group 1: r (t9a^(1/3)), vB (vA^(-1/3))
    {-84.165, 0, XV, KV3, spx::PL1 + 0}, {-84.165, 0, XV, KC3, spx::PL1 + 3},
    // group 2: r (t9a^(1/3), then its square), vD (vA^(2/3)), vB (vA^(-1/3))
    {-106.594, 0, XV, KV, spx::PL1 + 6}, {2.562, 0, XV2, KC, spx::PL1 + 6}, {2.562, 0, XV, KC, spx::PL1 + 10},
    {-106.594, 0, XV, KC, spx::PL1 + 9},
};
static_assert(spx::NE1 + spx::NE2 == 42, "lanes of the exp pass");

// pv: the lane's value of the pow pass (all lanes of the wavefront active)
__device__ __forceinline__ double exp_arg(const SpxArg& e, const RatePow& p, const DerivPow& q, double pv)
{
    const double v = __shfl(pv, e.src);
    const double X = e.x == XPI     ? p.t9i
                     : e.x == XQI   ? q.t9i
                     : e.x == XPI13 ? p.t9i13
                     : e.x == XQI13 ? q.t9i13
                     : e.x == XPM1  ? p.t9rm1
                     : e.x == XV    ? v
                                    : v * v;
    const double num = e.kind == KD ? p.t92 : e.kind == KA ? p.t9 : e.kind == KV || e.kind == KV3 ? e.c : q.t9;
    const double den = e.kind == KA   ? 1. + 0.055 * p.t9
                       : e.kind == KB ? 1. + .055 * q.t9
                       : e.kind == KV || e.kind == KV3 ? v
                                                       : e.d;
    const double w = num / den;
    double       a = e.c * (e.kind == KA ? w * w : X);
    if (e.kind == KB) a = e.c * w * w;
    if (e.kind == KV || e.kind == KV3) a = w;
    if (e.kind == KD) a = a - w;
    if (e.kind == KS) a = a - w * w;
    if (e.kind == KM) a = a - q.t92 * e.d;
    if (e.kind == KV3) a = a - 2.12e-03 * p.t93;
    if (e.kind == KC3) a = a - 2.12e-3 * q.t93;
    if (e.kind == KF)
    {
        const bool r = e.x == XPI13;
        a            = a - .629 * (r ? p.t923 : q.t923) - .445 * (r ? p.t943 : q.t943) + .0103 * (r ? p.t92 : q.t92);
    }
    return a;
}

// The outputs of the groups in MASK from the pass values (the reference's expressions, each exp /
// pow replaced by its value; net14.cpp:196-566), handed to out(group, r, rl, dr, drl) group by
// group (rl, drl only for groups 0, 4, 5; zero otherwise): v1(k), k < NE1: exp k, NE1 + j: pow j of
// groups 1 and 2; v2(k): exp NE1 + k.
template<int MASK, class V1, class V2, class Out>
__device__ __forceinline__ void special_combine(double T, const RatePow& p, const DerivPow& q, const V1& v1,
                                                const V2& v2, const Out& out)
{
    // group 0: triple alpha
    if constexpr ((MASK >> 0) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        const double r2abe = (7.40e+05 * p.t9i32) * v1(0) +
                             4.164e+09 * p.t9i23 * v1(1) *
                                 (1. + 0.031 * p.t913 + 8.009 * p.t923 + 1.732 * p.t9 + 49.883 * p.t943 + 27.426 * p.t953);
        const double rbeac = (130. * p.t9i32) * v1(2) +
                             2.510e+07 * p.t9i23 * v1(3) *
                                 (1. + 0.018 * p.t913 + 5.249 * p.t923 + 0.650 * p.t9 + 19.176 * p.t943 + 6.034 * p.t953);
        double r;
        if (T > 8e7)
            r = 2.90e-16 * (r2abe * rbeac) + 0.1 * 1.35e-07 * p.t9i32 * v1(4);
        else
            r = 2.90e-16 * (r2abe * rbeac) *
                    (0.01 + 0.2 * (1. + 4. * exp(-pow(0.025 * p.t9i, 3.263))) /
                                (1. + 4. * exp(-pow(p.t9 / 0.025, 9.227)))) +
                0.1 * 1.35e-07 * p.t9i32 * v1(4);
        const double rev = 2.e20 * v1(5);
        gr           = r;
        grl          = r * rev * p.t93;
        const double vD  = 1. + .031 * q.t913 + 8.009 * q.t923 + 1.732 * q.t9 + 49.883 * q.t943 + 27.426 * q.t953;
        const double vG  = 1. + .018 * q.t913 + 5.249 * q.t923 + .650 * q.t9 + 19.176 * q.t943 + 6.034 * q.t953;
        const double dvA = 24.811 * q.t9i2;
        const double dvB = 1.0663 * q.t9i2;
        const double dvC = q.t9i43 * 13.49 / 3. - 208.246564 * q.t9;
        const double dvD = (q.t9i23 * .031 + q.t9i13 * 16.018 + 5.196 + q.t913 * 199.532 + q.t923 * 137.13) / 3.;
        const double dvE = 3.3364 * q.t9i2;
        const double dvF = q.t9i43 * 23.57 / 3. - 36.21548212 * q.t9;
        const double dvG = (q.t9i23 * .018 + q.t9i13 * 10.498 + 1.950 + q.t913 * 76.704 + q.t923 * 30.17) / 3.;
        const double eB = v1(6), eC = v1(7), eE = v1(8), eF = v1(9);
        const double r2abe_ = 7.4e5 * q.t9i32 * eB + 4.164e9 * q.t9i23 * vD * eC;
        const double rbeac_ = 130. * q.t9i32 * eE + 2.510e7 * q.t9i23 * vG * eF;
        const double dr2abe = eB * (-1.11e6 * q.t9i52 + 7.4e5 * q.t9i32 * dvB) +
                              4.164e9 * eC * (-q.t9i53 * vD * 2. / 3. + q.t9i23 * dvC * vD + q.t9i23 * dvD);
        const double drbeac = eE * (-195. * q.t9i52 + 130. * q.t9i32 * dvE) +
                              2.510e7 * eF * (-2. * q.t9i53 * vG / 3. + q.t9i23 * dvF * vG + q.t9i23 * dvG);
        const double dr = (2.90e-16 * (dr2abe * rbeac_ + r2abe_ * drbeac) + 1.35e-8 * v1(10) * (-1.5 * q.t9i52 + q.t9i32 * dvA)) *
                          1.e-9;
        gdr           = dr;
        const double dvA2 = 84.419412 * q.t9i2;
        gdrl          = 2.00e20 * v1(11) * q.t93 * (dvA2 * r + 3. * q.t9i * r + dr) * 1.e-9;
        out(0, gr, grl, gdr, gdrl);
    }
    // group 1: 12C + 12C
    if constexpr ((MASK >> 1) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        const double t9a56 = v1(37);
        gr             = 4.27e+26 * t9a56 * p.t9i32 * v2(0);
        const double vA    = q.t9 / (1. + .0396 * q.t9);
        const double vA56  = v1(38);
        const double dvA   = vA * vA * q.t9i2;
        const double dvB   = 28.055 * dvA * v1(40) - 6.36e-3 * q.t92;
        gdr = 4.27e26 * q.t9i32 * v2(1) * (v1(41) * dvA * 5. / 6. - 1.5 * vA56 * q.t9i + vA56 * dvB) * 1.e-9;
        out(1, gr, grl, gdr, gdrl);
    }
    // group 2: 12C + 16O
    if constexpr ((MASK >> 2) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        if (T >= 5e8)
        {
            const double t9a56ap = v1(43);
            gr = 1.72e+31 * t9a56ap * p.t9i32 * v2(2) / (v1(34) + 1.06e-03 * v2(3));
        }
        const double t9 = T * 1.0e-09;
        if (t9 > .5)
        {
            const double vA   = q.t9 / (1. + .055 * q.t9);
            const double vA56 = v1(44);
            const double eC = v1(35), eD = v2(4);
            const double val  = eC + 1.06e-3 * eD;
            const double dvA  = vA * vA * q.t9i2;
            const double dvB  = 106.594 * v1(47) * dvA / 3.;
            const double dvC  = -.36 * vA * dvA;
            const double dvD  = 1.708 * dvA * v1(45);
            const double dval = dvC * eC + 1.06e-3 * dvD * eD;
            gdr = 1.72e31 * q.t9i32 * (v1(48) * dvA * 5. / 6. - 1.5 * vA56 * q.t9i + vA56 * (dvB - dval / val)) *
                      v2(5) / val * 1.e-9;
        }
        out(2, gr, grl, gdr, gdrl);
    }
    // group 3: 16O + 16O
    if constexpr ((MASK >> 3) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        gr           = 7.10e+36 * p.t9i23 * v1(12);
        const double dvA = 45.31 * q.t9i43 - .629 * q.t9i13 * 2. / 3. - .445 * q.t913 * 4. / 3. + .0206 * q.t9;
        gdr          = 7.10e36 * v1(13) * q.t9i23 * (-q.t9i * 2. / 3. + dvA) * 1.e-9;
        out(3, gr, grl, gdr, gdrl);
    }
    // group 4: 12C(a,g)16O
    if constexpr ((MASK >> 4) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        const double b1 = 1. + 0.0489 * p.t9i23, b2 = 1. + 0.2654 * p.t9i23;
        const double r  = 1.04e+08 / (p.t92 * (b1 * b1)) * v1(14) + 1.76e+08 / (p.t92 * (b2 * b2)) * v1(15) +
                         1.25e+03 * p.t9i32 * v1(16) + 1.43e-02 * p.t95 * v1(17);
        gr           = r;
        grl          = r * 5.13e+10 * p.t9r32 * v1(18);
        const double qb1 = 1. + .0489 * q.t9i23;
        const double vB  = qb1 * qb1;
        const double qb2 = 1. + .2654 * q.t9i23;
        const double vD  = qb2 * qb2;
        const double dvB = -(2. + .0978 * q.t9i23) * (.0326 * q.t9i53);
        const double dvC = 32.120 * q.t9i43 / 3. - 2. * q.t9 / (3.496 * 3.496);
        const double dvD = -(2. + .5308 * q.t9i23) * (.5308 * q.t9i53 / 3.);
        const double dvE = 32.120 * q.t9i43 / 3.;
        const double dvF = 27.499 * q.t9i2;
        const double dvG = 15.541 * q.t9i2;
        const double dr  = (1.04e8 * v1(19) * q.t9i2 * (-2. * q.t9i + dvC - dvB / vB) / vB +
                           1.76e8 * v1(20) * q.t9i2 * (-2. * q.t9i + dvE - dvD / vD) / vD +
                           1.25e3 * v1(21) * (-1.5 * q.t9i52 + dvF * q.t9i32) + 1.43e-2 * v1(22) * (5. * q.t94 + dvG * q.t95)) *
                          1.e-9;
        gdr          = dr;
        const double dvA = 83.108047 * q.t9i2;
        gdrl         = 5.13e10 * v1(23) * (dr * q.t932 + r * 1.5 * q.t912 + r * q.t932 * dvA) * 1.e-9;
        out(4, gr, grl, gdr, gdrl);
    }
    // group 5: 16O(a,g)20Ne
    if constexpr ((MASK >> 5) & 1)
    {
        double gr = 0, grl = 0, gdr = 0, gdrl = 0;
        const double r = (9.37e+09 * p.t9i23 * v1(24) + 62.1 * p.t9i32 * v1(25) + 538. * p.t9i32 * v1(26) +
                          13. * p.t92 * v1(27));
        gr           = r;
        grl          = r * 5.65e+10 * p.t9r32 * v1(28);
        const double dvB = 39.757 * q.t9i43 / 3. - 2. * q.t9 / (1.586 * 1.586);
        const double dvC = 10.297 * q.t9i2;
        const double dvD = 12.226 * q.t9i2;
        const double dvE = 20.093 * q.t9i2;
        const double dr  = (9.37e9 * v1(29) * (-q.t9i53 * 2. / 3. + q.t9i23 * dvB) +
                           62.1 * v1(30) * (-1.5 * q.t9i52 + q.t9i32 * dvC) + 538. * v1(31) * (-1.5 * q.t9i52 + q.t9i32 * dvD) +
                           13. * v1(32) * (2. * q.t9 + q.t92 * dvE)) *
                          1.e-9;
        gdr          = dr;
        const double dvA = 54.903255 * q.t9i2;
        gdrl         = 5.65e10 * v1(33) * (dr * q.t932 + 1.5 * r * q.t912 + r * q.t932 * dvA) * 1.e-9;
        out(5, gr, grl, gdr, gdrl);
    }
}

// Coulomb-corrected binding energy (net14.cpp:49-75, net14_tables.hpp:47-67) and screening mu/kT
// (net14.cpp:577-600) of a species from ae = pow(3/4 / (pi ne), 1/3).  The reference forms ae and
// the plasma parameter once for each of the two, as 3/4 / (pi ne) and 3 / (4 pi ne) and with the
// factors of kT exchanged: the same values (the factor 4 is exact), so their roots, pow and
// quotient are formed once.
__device__ __forceinline__ void species_coulomb(double T, double ae, double Z53, double BE0, double& be, double& mu)
{
    const double kbt        = phys::Kb * T;
    const double nakbt      = phys::Na * kbt;
    const double correction = -1.5 * nakbt;
    const double gam        = phys::e2 / (kbt * ae);
    const double x          = gam * Z53;
    const double sq         = sqrt(x);
    double       fn;
    if (x > 1)
    {
        const double a1 = -.898004, b1 = .96786, c1 = .220703, d1 = -.86097, e1 = 2.520058332;
        const double sq2 = sqrt(sq), cs = c1 / sq2;
        fn               = a1 * x + b1 * sq2 + cs + d1;
        mu               = a1 * x + 4. * (b1 * sq2 - cs) + d1 * log(x) - e1;
    }
    else
    {
        const double a = -.5 * 1.7320508075688772 /* sqrt(3.), correctly rounded */;
        const double w = pow(x, 1.9885);
        fn             = a * x * sq + .29561 * w;
        mu             = -(1. / 1.7320508075688772) * x * sq + w * .29561 / 1.9885;
    }
    be = BE0 + correction;
    be -= nakbt * fn;
}

// The electron-capture table interpolation of net87 (net87.cpp:102-141), by the 64 lanes of one
// wavefront (k = lane).  The reference finds the grid positions by linear searches (the first
// point not below log T, resp. log(rho Ye)); both grids ascend strictly, so that position is the
// number of grid points below the value, counted here with one ballot per grid instead of up to
// 92 dependent loads.  Lane c < 12 then interpolates rate c with the reference's expression.
__device__ __forceinline__ void electron_interpolate_wave(const double* logT, const double* logR, const double* tab,
                                                          double temp, double rhoElec, double* rate, int k)
{
    constexpr int nT = 41, nR = 51, nC = 12;
    static_assert(nT <= 64 && nR <= 64 && nC <= 64, "one grid point per lane");
    const double lt = log10(temp);
    const double lr = log10(rhoElec);
    const double gT = logT[k < nT ? k : 0];
    const double gR = logR[k < nR ? k : 0];
    int          it = (int)__popcll(__ballot(k < nT && gT < lt));
    int          ir = (int)__popcll(__ballot(k < nR && gR < lr));
    if (k >= nC) return;
    const int it0 = (it - 1 > 0) ? it - 1 : 0, ir0 = (ir - 1 > 0) ? ir - 1 : 0;
    it            = (it < nT - 1) ? it : nT - 1;
    ir            = (ir < nR - 1) ? ir : nR - 1;
    const double x2x  = logT[it] - lt;
    const double xx1  = -logT[it0] + lt;
    const double y2y  = logR[ir] - lr;
    const double yy1  = -logR[ir0] + lr;
    double       x2x1 = logT[it] - logT[it0];
    x2x1              = x2x1 == 0 ? 2 : x2x1;
    double y2y1       = logR[ir] - logR[ir0];
    y2y1              = y2y1 == 0 ? 2 : y2y1;
    const int c       = k;
    rate[c] = (tab[(it0 * nR + ir0) * nC + c] * x2x * y2y + tab[(it * nR + ir0) * nC + c] * xx1 * y2y +
               tab[(it0 * nR + ir) * nC + c] * x2x * yy1 + tab[(it * nR + ir) * nC + c] * xx1 * yy1) /
              (x2x1 * y2y1);
}

} // namespace nnet_amd
