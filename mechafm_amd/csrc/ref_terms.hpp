// The reference's pair-term arithmetic in its own operation order, for the
// kernels built with -ffp-contract=off (plain scan, flexible scan): every
// operation rounds as the reference's -O3 x86-64 build rounds it, and the
// divisions and square roots are IEEE.
#pragma once

#include "device_common.hpp"

namespace mafm {

struct V3 {
    double x, y, z;
};

__device__ inline double sq(double a) { return a * a; }   // pow(a, 2): the exact square
__device__ inline double len3(V3 a) { return sqrt((sq(a.x) + sq(a.y)) + sq(a.z)); }   // vectors.hpp:99-101

// Quotients by one divisor: the reciprocal's two Newton steps are shared, and
// each quotient is rounded by the residual step IEEE division ends with (the
// operations, and so the bits, of the compiler's a / d where it does not
// rescale its operands, which it does below 2^-970 and near the exponent's
// ends; div_fixup covers zeros, infinities and NaN).  An angle term has
// fourteen divisions by two lengths: 11 instructions each become 4.
struct Divisor {
    double d, y;
    __device__ explicit Divisor(double d_) : d(d_) {
        y = __builtin_amdgcn_rcp(d);
        y = fma(y, fma(-d, y, 1.0), y);
        y = fma(y, fma(-d, y, 1.0), y);
    }
    __device__ double operator()(double a) const {
        const double q = a * y;
        return __builtin_amdgcn_div_fixup(fma(fma(-d, q, a), y, q), d, a);
    }
    __device__ V3 operator()(V3 v) const { return {(*this)(v.x), (*this)(v.y), (*this)(v.z)}; }
};

// LJInteraction / MorseInteraction::eval (interactions.cpp:15-40) with
// r = p1 - p2, returning the force on atom i1 and the pair energy.
__device__ inline void vdw(int kind, double p0, double p1, double p2, V3 r, V3& f, double& e) {
    if (kind == 0) {
        double r_sqr = (sq(r.x) + sq(r.y)) + sq(r.z);
        double r6 = r_sqr * r_sqr * r_sqr;
        double term_a = p1 / (r6 * r6);
        double term_b = p0 / r6;
        e = term_a - term_b;
        double s = (12 * term_a - 6 * term_b) / r_sqr;
        f.x = s * r.x; f.y = s * r.y; f.z = s * r.z;
    } else {
        double rl = len3(r);
        double d_exp = exp(-p1 * (rl - p2));
        e = p0 * (sq(d_exp) - 2 * d_exp + 1);
        double f_abs = 2 * p0 * p1 * (sq(d_exp) - d_exp);
        double s = f_abs / rl;
        f.x = s * r.x; f.y = s * r.y; f.z = s * r.z;
    }
}

// CoulombInteraction::eval (interactions.cpp:42-51).
__device__ inline void coulomb(double qq, V3 r, V3& f, double& e) {
    double rl = len3(r);
    e = qq / rl;
    double s = qq / (rl * rl * rl);
    f.x = s * r.x; f.y = s * r.y; f.z = s * r.z;
}

// A site's van der Waals term and, where it has one, its Coulomb term: vdw and
// coulomb above with the distance and its reciprocal found once.
struct SiteTerms {
    V3 f, fc;
    double e, ec;
};

__device__ inline SiteTerms site_terms(int kind, bool coul, double p0, double p1, double p2, double qq, V3 r) {
    SiteTerms t;
    const double r_sqr = (sq(r.x) + sq(r.y)) + sq(r.z);
    double rl = 0, e_c = 0;
    if (kind == 0) {
        const double r6 = r_sqr * r_sqr * r_sqr;
        const double term_a = p1 / (r6 * r6);
        const double term_b = p0 / r6;
        t.e = term_a - term_b;
        const double s = (12 * term_a - 6 * term_b) / r_sqr;
        t.f.x = s * r.x; t.f.y = s * r.y; t.f.z = s * r.z;
        if (coul) {
            rl = sqrt(r_sqr);
            e_c = qq / rl;
        }
    } else {
        rl = sqrt(r_sqr);
        const Divisor by_rl(rl);
        const double d_exp = exp(-p1 * (rl - p2));
        t.e = p0 * (sq(d_exp) - 2 * d_exp + 1);
        const double f_abs = 2 * p0 * p1 * (sq(d_exp) - d_exp);
        const double s = by_rl(f_abs);
        t.f.x = s * r.x; t.f.y = s * r.y; t.f.z = s * r.z;
        if (coul) e_c = by_rl(qq);
    }
    t.fc = {0, 0, 0};
    t.ec = 0;
    if (coul) {
        t.ec = e_c;
        const double s = qq / (rl * rl * rl);
        t.fc.x = s * r.x; t.fc.y = s * r.y; t.fc.z = s * r.z;
    }
    return t;
}

}  // namespace mafm
