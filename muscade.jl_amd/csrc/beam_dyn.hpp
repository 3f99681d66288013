// Requestables and strain gauges of EulerBeam3D on jets: the corotated kinematics with their time
// derivatives, the inertia, added-mass, damping and roll-inertia loads, and first and second derivatives of
// the gauges' strains. (The solver's residual and tangent are in closed form: beam_math.hpp, beam_dir.hpp.)
//
// Reference: toolbox/BeamElement.jl:28-64 (resultants), :151-208 (residual,
// kinematics, corotated), toolbox/Rotations.jl:13-182, src/Taylor.jl:24-65
// (motion / motion⁻¹), src/Output.jl:131-181 (getresult).
//
// getresult evaluates the element on plain values, so every formula, squares among them, is exact calculus
// on its time levels.
//
// `Jet<NT,E>` carries q(t,ε) truncated at order NT-1 in t and 1 in ε, at most second order in all:
// v[n] = ∂ⁿq/∂tⁿ and e[n] = ∂(∂ⁿq/∂tⁿ)/∂ε.  With E = false it is the plain time jet.
#pragma once
#include "beam_math.hpp"

namespace mh {

template <int NT, bool E> struct Jet {
    static_assert(NT + (E ? 1 : 0) <= 3, "second order in all");
    double v[NT];
    double e[E ? NT : 1];
};

template <int NT, bool E> MH_HD Jet<NT, E> jzero() {
    Jet<NT, E> r;
#pragma unroll
    for (int n = 0; n < NT; ++n) r.v[n] = 0.;
#pragma unroll
    for (int n = 0; n < (E ? NT : 1); ++n) r.e[n] = 0.;
    return r;
}
template <int NT, bool E> MH_HD Jet<NT, E> operator+(const Jet<NT, E>& a, const Jet<NT, E>& b) {
    Jet<NT, E> r;
#pragma unroll
    for (int n = 0; n < NT; ++n) r.v[n] = a.v[n] + b.v[n];
    if constexpr (E) {
#pragma unroll
        for (int n = 0; n < NT; ++n) r.e[n] = a.e[n] + b.e[n];
    } else r.e[0] = 0.;
    return r;
}
template <int NT, bool E> MH_HD Jet<NT, E> operator-(const Jet<NT, E>& a, const Jet<NT, E>& b) {
    Jet<NT, E> r;
#pragma unroll
    for (int n = 0; n < NT; ++n) r.v[n] = a.v[n] - b.v[n];
    if constexpr (E) {
#pragma unroll
        for (int n = 0; n < NT; ++n) r.e[n] = a.e[n] - b.e[n];
    } else r.e[0] = 0.;
    return r;
}
template <int NT, bool E> MH_HD Jet<NT, E> operator-(const Jet<NT, E>& a) {
    Jet<NT, E> r;
#pragma unroll
    for (int n = 0; n < NT; ++n) r.v[n] = -a.v[n];
    if constexpr (E) {
#pragma unroll
        for (int n = 0; n < NT; ++n) r.e[n] = -a.e[n];
    } else r.e[0] = 0.;
    return r;
}
template <int NT, bool E> MH_HD Jet<NT, E> operator*(double s, const Jet<NT, E>& a) {
    Jet<NT, E> r;
#pragma unroll
    for (int n = 0; n < NT; ++n) r.v[n] = s * a.v[n];
    if constexpr (E) {
#pragma unroll
        for (int n = 0; n < NT; ++n) r.e[n] = s * a.e[n];
    } else r.e[0] = 0.;
    return r;
}
template <int NT, bool E> MH_HD Jet<NT, E> operator+(const Jet<NT, E>& a, double c) { Jet<NT, E> r = a; r.v[0] = a.v[0] + c; return r; }
// Leibniz product of truncated jets.
template <int NT, bool E> MH_HD Jet<NT, E> operator*(const Jet<NT, E>& a, const Jet<NT, E>& b) {
    Jet<NT, E> r;
    r.v[0] = a.v[0] * b.v[0];
    if constexpr (NT > 1) r.v[1] = a.v[1] * b.v[0] + a.v[0] * b.v[1];
    if constexpr (NT > 2) r.v[2] = a.v[2] * b.v[0] + 2. * (a.v[1] * b.v[1]) + a.v[0] * b.v[2];
    if constexpr (E) {
        r.e[0] = a.e[0] * b.v[0] + a.v[0] * b.e[0];
        if constexpr (NT > 1) r.e[1] = (a.e[1] * b.v[0] + a.v[1] * b.e[0]) + (a.e[0] * b.v[1] + a.v[0] * b.e[1]);
    } else r.e[0] = 0.;
    return r;
}
// Composition with a scalar function given f, f', f'' at a.v[0].
template <int NT, bool E> MH_HD Jet<NT, E> jfun(const Jet<NT, E>& a, const double* f) {
    Jet<NT, E> r;
    r.v[0] = f[0];
    if constexpr (NT > 1) r.v[1] = f[1] * a.v[1];
    if constexpr (NT > 2) r.v[2] = f[2] * (a.v[1] * a.v[1]) + f[1] * a.v[2];
    if constexpr (E) {
        r.e[0] = f[1] * a.e[0];
        if constexpr (NT > 1) r.e[1] = f[2] * (a.e[0] * a.v[1]) + f[1] * a.e[1];
    } else r.e[0] = 0.;
    return r;
}
// ------------------------------------------------------------ scalar functions
// Derivatives of sinc1 with the branches of Rotations.jl:14-45.
MH_HD double sinc1_d1(double x) {
    if (fabs(x) > 1e-3) { double s = sin(x), c = cos(x); return c / x - s / (x * x); }
    double x2 = x * x;
    return x * (-1. / 3. + x2 / 30.);
}
MH_HD double sinc1_d2(double x) {
    if (fabs(x) > 1e-1) { double s = sin(x), c = cos(x); return -s / x - 2. * c / (x * x) + 2. * s / (x * x * x); }
    double x2 = x * x;
    return -1. / 3. + x2 * (1. / 10. + x2 * (-1. / 168. + x2 * (1. / 6480.)));
}
template <int NT, bool E> MH_HD Jet<NT, E> jsinc1(const Jet<NT, E>& a) {
    const double x = a.v[0];
    double f[3];
    f[0] = sinc1(x);
    f[1] = sinc1_d1(x);
    f[2] = (NT + (E ? 1 : 0) > 2) ? sinc1_d2(x) : 0.;
    return jfun(a, f);
}
template <int NT, bool E> MH_HD Jet<NT, E> jsqrt(const Jet<NT, E>& a) {
    const double x = a.v[0], s = sqrt(x);
    double f[3] = {s, 0.5 / s, -0.25 / (x * s)};
    return jfun(a, f);
}
template <int NT, bool E> MH_HD Jet<NT, E> jrecip(const Jet<NT, E>& a) {
    const double x = a.v[0], r = 1. / x;
    double f[3] = {r, -(r * r), 2. * (r * r * r)};
    return jfun(a, f);
}
template <int NT, bool E> MH_HD Jet<NT, E> jacos(const Jet<NT, E>& a) {
    const double x = a.v[0], q = 1. - x * x, sq = sqrt(q);
    double f[3] = {acos(x), -1. / sq, -x / (q * sq)};
    return jfun(a, f);
}
// scac(x) = sinc1(acos x); 5th-order series in x-1 for |x-1| <= 1e-3 (Rotations.jl:61-68)
template <int NT, bool E> MH_HD Jet<NT, E> jscac(const Jet<NT, E>& a) {
    const double d = a.v[0] - 1.;
    if (fabs(d) > 1e-3) return jsinc1(jacos(a));
    const double c1 = 1. / 3., c2 = -2. / 90., c3 = 0.0052911879917544626, c4 = -0.0016229317117234072, c5 = 0.0005625;
    double f[3];
    f[0] = 1. + d * (c1 + d * (c2 + d * (c3 + d * (c4 + d * c5))));
    f[1] = c1 + d * (2. * c2 + d * (3. * c3 + d * (4. * c4 + d * (5. * c5))));
    f[2] = 2. * c2 + d * (6. * c3 + d * (12. * c4 + d * (20. * c5)));
    return jfun(a, f);
}

// ------------------------------------------------------------ rotations on jets
template <int NT, bool E> struct JM3 { Jet<NT, E> a[9]; };   // column-major 3×3
template <int NT, bool E> struct JV3 { Jet<NT, E> a[3]; };

// Rodrigues(v) = I + sinc1(θ) S + (sinc1(θ/2)²/2) spin²(S), θ = norm3(v) (Rotations.jl:106-135):
// the coefficient jets a = sinc1(θ), b = sinc1(θ/2)²/2.
template <int NT, bool E>
MH_HD void jrodrigues_coef(const JV3<NT, E>& v, Jet<NT, E>& a, Jet<NT, E>& b) {
    using J = Jet<NT, E>;
    const J& x = v.a[0]; const J& y = v.a[1]; const J& z = v.a[2];
    J ss = (x * x + y * y) + z * z;
    J th;
    if (sqrt(ss.v[0]) < 1e-14) th = jzero<NT, E>();
    else th = jsqrt(ss);
    a = jsinc1(th);
    J s = jsinc1(0.5 * th);
    b = 0.5 * (s * s);
}
// Column k of Rodrigues(v) from its coefficients, spin²(S) entrywise (Rotations.jl:114-122).
template <int K, int NT, bool E>
MH_HD JV3<NT, E> jrodrigues_col(const JV3<NT, E>& v, const Jet<NT, E>& a, const Jet<NT, E>& b) {
    const Jet<NT, E>& x = v.a[0]; const Jet<NT, E>& y = v.a[1]; const Jet<NT, E>& z = v.a[2];
    JV3<NT, E> r;
    if constexpr (K == 0) {
        r.a[0] = b * (-(z * z) + -(y * y)) + 1.;
        r.a[1] = a * z + b * (x * y);
        r.a[2] = -(a * y) + b * (z * x);
    } else if constexpr (K == 1) {
        r.a[0] = -(a * z) + b * (x * y);
        r.a[1] = b * (-(x * x) + -(z * z)) + 1.;
        r.a[2] = a * x + b * (y * z);
    } else {
        r.a[0] = a * y + b * (z * x);
        r.a[1] = -(a * x) + b * (y * z);
        r.a[2] = b * (-(x * x) + -(y * y)) + 1.;
    }
    return r;
}
template <int NT, bool E> MH_HD JM3<NT, E> jrodrigues(const JV3<NT, E>& v) {
    Jet<NT, E> a, b;
    jrodrigues_coef<NT, E>(v, a, b);
    JV3<NT, E> c0 = jrodrigues_col<0>(v, a, b), c1 = jrodrigues_col<1>(v, a, b), c2 = jrodrigues_col<2>(v, a, b);
    JM3<NT, E> r;
#pragma unroll
    for (int i = 0; i < 3; ++i) { r.a[i] = c0.a[i]; r.a[3 + i] = c1.a[i]; r.a[6 + i] = c2.a[i]; }
    return r;
}
// A ∘₁ B with a constant B
template <int NT, bool E> MH_HD JM3<NT, E> jmul_const(const JM3<NT, E>& A, const m3& B) {
    JM3<NT, E> r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.a[i + 3 * j] = (at(B, 0, j) * A.a[i] + at(B, 1, j) * A.a[i + 3]) + at(B, 2, j) * A.a[i + 6];
    return r;
}
template <int NT, bool E> MH_HD JV3<NT, E> jmulT(const JM3<NT, E>& A, const JV3<NT, E>& v) {   // Aᵀ v
    JV3<NT, E> r;
#pragma unroll
    for (int j = 0; j < 3; ++j) r.a[j] = (A.a[3 * j] * v.a[0] + A.a[3 * j + 1] * v.a[1]) + A.a[3 * j + 2] * v.a[2];
    return r;
}
template <int NT, bool E> MH_HD JV3<NT, E> jmulv(const JM3<NT, E>& A, const JV3<NT, E>& v) {   // A v
    JV3<NT, E> r;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.a[i] = (A.a[i] * v.a[0] + A.a[i + 3] * v.a[1]) + A.a[i + 6] * v.a[2];
    return r;
}

// ------------------------------------------------------------ element dynamics
// Per element, what the loads need from the kinematics jets.
struct DynKin {
    double r0[9];             // rₛₘ
    double r1[9], r2[9];      // ṙₛₘ, r̈ₛₘ
    double xd[4][3];          // ẋ at the Gauss points
    double xdd[4][3];         // ẍ at the Gauss points
};
template <int NT> MH_HD double jlevel(const Jet<NT, false>& a, int n) { return n < NT ? a.v[n] : 0.; }

// The rotation chain (v₁,v₂) ↦ (rₛₘ, Δv) of BeamElement.jl:192-208 on time jets.
// Neither R₂ = Rodrigues(v₂) nor the relative rotation M = R₂R₁ᵀ is held whole: φ = Rodrigues⁻¹(M)
// reads only tr M = Σₖ R₁eₖ·R₂eₖ and the axial vector of M − Mᵀ, Σₖ R₁eₖ × R₂eₖ, so R₂ is
// formed a column at a time; rₛₘ = Rodrigues(Δv)·(R₁ rₘ) applies Rodrigues(Δv) to one column
// of R₁rₘ at a time, w ↦ w + a Δv×w + b (Δv (Δv·w) − |Δv|² w). This keeps the live jets
// of the chain to about 21 instead of the 27 of three whole matrices.
template <int NT, bool E>
MH_HD void dyn_rotation_chain(const BeamGeo& G, const JV3<NT, E>& v1, const JV3<NT, E>& v2, JM3<NT, E>& rsm,
                              JV3<NT, E>& dv) {
    using J = Jet<NT, E>;
    JM3<NT, E> R1 = jrodrigues<NT, E>(v1);
    J tr, ax[3];
    {
        J a2, b2;
        jrodrigues_coef<NT, E>(v2, a2, b2);
        auto add = [&](const JV3<NT, E>& c2, int k, bool first) {
            const J* c1 = &R1.a[3 * k];
            J d = (c1[0] * c2.a[0] + c1[1] * c2.a[1]) + c1[2] * c2.a[2];
            J x = c1[1] * c2.a[2] - c1[2] * c2.a[1];
            J y = c1[2] * c2.a[0] - c1[0] * c2.a[2];
            J z = c1[0] * c2.a[1] - c1[1] * c2.a[0];
            if (first) { tr = d; ax[0] = x; ax[1] = y; ax[2] = z; }
            else { tr = tr + d; ax[0] = ax[0] + x; ax[1] = ax[1] + y; ax[2] = ax[2] + z; }
        };
        add(jrodrigues_col<0>(v2, a2, b2), 0, true);
        add(jrodrigues_col<1>(v2, a2, b2), 1, false);
        add(jrodrigues_col<2>(v2, a2, b2), 2, false);
    }
    // Rodrigues⁻¹(M) = spin⁻¹(M)/scac((tr M - 1)/2) (Rotations.jl:101), Δv = φ/2
    J rs = jrecip(jscac(0.5 * (tr + (-1.))));
#pragma unroll
    for (int c = 0; c < 3; ++c) dv.a[c] = 0.5 * ((0.5 * ax[c]) * rs);
    JM3<NT, E> R1m = jmul_const(R1, G.rm);
    J ah, bh;
    jrodrigues_coef<NT, E>(dv, ah, bh);
    const J& x = dv.a[0]; const J& y = dv.a[1]; const J& z = dv.a[2];
    J n2 = (x * x + y * y) + z * z;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const J* w = &R1m.a[3 * j];
        J cx = y * w[2] - z * w[1], cy = z * w[0] - x * w[2], cz = x * w[1] - y * w[0];
        J s = (x * w[0] + y * w[1]) + z * w[2];
        rsm.a[3 * j] = (w[0] + ah * cx) + bh * (x * s - n2 * w[0]);
        rsm.a[3 * j + 1] = (w[1] + ah * cy) + bh * (y * s - n2 * w[1]);
        rsm.a[3 * j + 2] = (w[2] + ah * cz) + bh * (z * s - n2 * w[2]);
    }
}
// Kinematics (BeamElement.jl:176-208) on time jets. Xj: the 12 element dofs as jets.
template <int NT>
MH_HD void dyn_kinematics(const BeamGeo& G, const Jet<NT, false>* Xj, DynKin& k) {
    using J = Jet<NT, false>;
    const double L = G.L;
    JV3<NT, false> u1, u2;
#pragma unroll
    for (int c = 0; c < 3; ++c) { u1.a[c] = Xj[c]; u2.a[c] = Xj[6 + c]; }
    JM3<NT, false> rsm;
    JV3<NT, false> dv;
    JV3<NT, false> v1, v2;
#pragma unroll
    for (int c = 0; c < 3; ++c) { v1.a[c] = Xj[3 + c]; v2.a[c] = Xj[9 + c]; }
    dyn_rotation_chain<NT, false>(G, v1, v2, rsm, dv);
    // uₗ₂ = rₛₘᵀ(u₂ + tgₘ/2 - cₛ) - tgₑ/2,  vₗ₂ = rₛₘᵀ Δv
    JV3<NT, false> dd, cs;
    const double tg[3] = {G.tgm.x, G.tgm.y, G.tgm.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        cs.a[c] = 0.5 * (u1.a[c] + u2.a[c]);
        dd.a[c] = (u2.a[c] + tg[c] * 0.5) - cs.a[c];
    }
    JV3<NT, false> ul = jmulT(rsm, dd), vl = jmulT(rsm, dv);
    ul.a[0] = ul.a[0] + (-(L * 0.5));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const double z = G.zgp[g];
        const double ya = 2. * z, yu = -4. * (z * z * z) + 3. * z, yv = (z * z - 1. / 4.) * L;
        JV3<NT, false> p;
        p.a[0] = ya * ul.a[0] + L * z;
        p.a[1] = yu * ul.a[1] + yv * vl.a[2];
        p.a[2] = yu * ul.a[2] - yv * vl.a[1];
        JV3<NT, false> x = jmulv(rsm, p);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            J xc = x.a[c] + cs.a[c];
            k.xd[g][c] = jlevel(xc, 1);
            k.xdd[g][c] = jlevel(xc, 2);
        }
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) { k.r0[i] = jlevel(rsm.a[i], 0); k.r1[i] = jlevel(rsm.a[i], 1); k.r2[i] = jlevel(rsm.a[i], 2); }
}

struct BeamDynSection {
    double mu, iota1, w;
    double Ca[3], Cl[3], Cq[3];
};

// External loads of the resultants (BeamElement.jl:28-64): per Gauss point the force
// fₑ (fw, inertia, added mass, linear and quadratic damping, minus U) and the
// element's roll-inertia couple mₑ (the same at every Gauss point).
MH_HD void dyn_loads(const DynKin& k, const BeamDynSection& S, const double* U, double (*fe)[3], double* me) {
    const double* r0 = k.r0;
    for (int g = 0; g < 4; ++g) {
        double xl1[3], xl2[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {   // x ∘₁ r₀ = r₀ᵀx
            xl1[j] = (k.xd[g][0] * r0[3 * j] + k.xd[g][1] * r0[3 * j + 1]) + k.xd[g][2] * r0[3 * j + 2];
            xl2[j] = (k.xdd[g][0] * r0[3 * j] + k.xdd[g][1] * r0[3 * j + 1]) + k.xdd[g][2] * r0[3 * j + 2];
        }
        double fal[3], fll[3], fql[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            fal[j] = S.Ca[j] * xl2[j];
            fll[j] = S.Cl[j] * xl1[j];
            double q = S.Cq[j] * (xl1[j] * xl1[j]);
            fql[j] = xl1[j] < 0. ? -q : q;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            double fa = (r0[i] * fal[0] + r0[i + 3] * fal[1]) + r0[i + 6] * fal[2];
            double fl = (r0[i] * fll[0] + r0[i + 3] * fll[1]) + r0[i + 6] * fll[2];
            double fq = (r0[i] * fql[0] + r0[i + 3] * fql[1]) + r0[i + 6] * fql[2];
            double f = (((S.mu * k.xdd[g][i] + fa) + fl) + fq) + (i == 2 ? S.w : 0.);
            fe[g][i] = f + (-U[i]);
        }
    }
    // vᵢ₂ = spin⁻¹(ṙᵀṙ + r₀ᵀr̈) (Rotations.jl:177-182); only its first component is used
    double a21 = ((k.r1[6] * k.r1[3] + k.r1[7] * k.r1[4]) + k.r1[8] * k.r1[5]) +
            ((r0[6] * k.r2[3] + r0[7] * k.r2[4]) + r0[8] * k.r2[5]);
    double a12 = ((k.r1[3] * k.r1[6] + k.r1[4] * k.r1[7]) + k.r1[5] * k.r1[8]) +
            ((r0[3] * k.r2[6] + r0[4] * k.r2[7]) + r0[5] * k.r2[8]);
    double m1 = S.iota1 * (0.5 * (a21 - a12));
#pragma unroll
    for (int i = 0; i < 3; ++i) me[i] = r0[i] * m1;
}

// Rotation vector of a rotation matrix (value only).
MH_HD v3 rotvec(const m3& r) {
    double sc = scac((at(r, 0, 0) + at(r, 1, 1) + at(r, 2, 2) - 1.) / 2.);
    return mk((at(r, 2, 1) - at(r, 1, 2)) / 2. / sc, (at(r, 0, 2) - at(r, 2, 0)) / 2. / sc, (at(r, 1, 0) - at(r, 0, 1)) / 2. / sc);
}

// Requestables of the element (BeamElement.jl:28-64,151-174) at X (ND time levels), what
// getresult extracts (src/Output.jl:131-181). getresult evaluates the element on plain
// values. ☼ε and ♢κ = (vₗ₂[1], vₗ₂[3], −vₗ₂[2])·2/L
// with their ND time levels, then per Gauss point ☼x and ☼κgp (ND levels each) and the
// resultants' ☼fᵢ, ☼mᵢ, ☼fₑ (as returned by `resultants`, before the U-load is subtracted)
// and ☼mₑ. Layout: ε[ND], κ[ND][3], then per Gauss point x[ND][3], κgp[ND][3], fᵢ, mᵢ[3],
// fₑ[3], mₑ[3] (beam_nres(ND) numbers).
constexpr int beam_nres(int ND) { return 4 * ND + 4 * (6 * ND + 10); }
template <int ND> MH_HD void dyn_requestables(const BeamGeo& G, const BeamSection& S, const BeamDynSection& D,
                                              const double (*X)[12], double* __restrict__ out) {
    using J = Jet<ND, false>;
    J Xj[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        Xj[i] = jzero<ND, false>();
#pragma unroll
        for (int n = 0; n < ND; ++n) Xj[i].v[n] = X[n][i];
    }
    const double L = G.L;
    JV3<ND, false> u1, u2, v1, v2;
#pragma unroll
    for (int c = 0; c < 3; ++c) { u1.a[c] = Xj[c]; u2.a[c] = Xj[6 + c]; v1.a[c] = Xj[3 + c]; v2.a[c] = Xj[9 + c]; }
    JM3<ND, false> rsm;
    JV3<ND, false> dv;
    dyn_rotation_chain<ND, false>(G, v1, v2, rsm, dv);
    JV3<ND, false> dd, cs;
    const double tg[3] = {G.tgm.x, G.tgm.y, G.tgm.z};
    const double cm[3] = {G.cm.x, G.cm.y, G.cm.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        cs.a[c] = 0.5 * (u1.a[c] + u2.a[c]);
        dd.a[c] = (u2.a[c] + tg[c] * 0.5) - cs.a[c];
    }
    JV3<ND, false> ul = jmulT(rsm, dd), vl = jmulT(rsm, dv);
    ul.a[0] = ul.a[0] + (-(L * 0.5));
    // ε = √((uₗ₂[1]+L/2)² + uₗ₂[2]² + uₗ₂[3]²)·2/L − 1
    const J a0 = ul.a[0] + 0.5 * L;
    const J eps = (2. / L) * jsqrt((a0 * a0 + ul.a[1] * ul.a[1]) + ul.a[2] * ul.a[2]) + (-1.);
    int q = 0;
#pragma unroll
    for (int d = 0; d < ND; ++d) out[q++] = eps.v[d];
    const J km[3] = {(2. / L) * vl.a[0], (2. / L) * vl.a[2], (2. / L) * (-vl.a[1])};
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int c = 0; c < 3; ++c) out[q++] = km[c].v[d];
    // loads (values) from the time jets of the Gauss points
    DynKin k;
    dyn_kinematics<ND>(G, Xj, k);
    double fe[4][3], me[3];
    const double U0[3] = {0., 0., 0.};
    dyn_loads(k, D, U0, fe, me);
    const double ka = 2. / L, kv = 2. / L;
    for (int g = 0; g < 4; ++g) {
        const double z = G.zgp[g];
        const double ya = 2. * z, yu = -4. * (z * z * z) + 3. * z, yv = (z * z - 1. / 4.) * L;
        const double ku = (-24. * z) / (L * L);
        JV3<ND, false> p;
        p.a[0] = ya * ul.a[0] + L * z;
        p.a[1] = yu * ul.a[1] + yv * vl.a[2];
        p.a[2] = yu * ul.a[2] - yv * vl.a[1];
        JV3<ND, false> x = jmulv(rsm, p);
        J kg[3] = {ka * vl.a[0], ku * ul.a[1] + kv * vl.a[2], ku * ul.a[2] - kv * vl.a[1]};
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int c = 0; c < 3; ++c) out[q++] = d == 0 ? (x.a[c].v[0] + cs.a[c].v[0]) + cm[c] : x.a[c].v[d] + cs.a[c].v[d];
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int c = 0; c < 3; ++c) out[q++] = kg[c].v[d];
        out[q++] = S.EA * eps.v[0];
        out[q++] = S.GJ * kg[0].v[0];
        out[q++] = S.EI3 * kg[1].v[0];
        out[q++] = S.EI2 * kg[2].v[0];
#pragma unroll
        for (int c = 0; c < 3; ++c) out[q++] = fe[g][c];
#pragma unroll
        for (int c = 0; c < 3; ++c) out[q++] = me[c];
    }
}

// The strain-gauge requestables εₐₓ = ε and κ = ♢κ (BeamElement.jl:155,172;
// StrainGaugeOnBeamElement.jl:73) on jets whose "time" level carries ∂/∂X_i and whose ε
// level carries ∂/∂X_j: with the seeds X_k = X₀_k + t·δ_ki + ε·δ_kj, v[0] is the value,
// v[1] = ∂/∂X_i, e[0] = ∂/∂X_j and e[1] = ∂²/∂X_i∂X_j.
MH_HD void gauge_jets(const BeamGeo& G, const double* X0, int i, int j, Jet<2, true>* q) {
    using J = Jet<2, true>;
    J Xj[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        Xj[k].v[0] = X0[k]; Xj[k].v[1] = k == i ? 1. : 0.;
        Xj[k].e[0] = k == j ? 1. : 0.; Xj[k].e[1] = 0.;
    }
    const double L = G.L;
    JV3<2, true> u1, u2, v1, v2;
#pragma unroll
    for (int c = 0; c < 3; ++c) { u1.a[c] = Xj[c]; u2.a[c] = Xj[6 + c]; v1.a[c] = Xj[3 + c]; v2.a[c] = Xj[9 + c]; }
    JM3<2, true> rsm;
    JV3<2, true> dv;
    dyn_rotation_chain<2, true>(G, v1, v2, rsm, dv);
    JV3<2, true> dd;
    const double tg[3] = {G.tgm.x, G.tgm.y, G.tgm.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const J cs = 0.5 * (u1.a[c] + u2.a[c]);
        dd.a[c] = (u2.a[c] + tg[c] * 0.5) - cs;
    }
    JV3<2, true> ul = jmulT(rsm, dd), vl = jmulT(rsm, dv);
    ul.a[0] = ul.a[0] + (-(L * 0.5));
    const J a0 = ul.a[0] + 0.5 * L;
    q[0] = (2. / L) * jsqrt((a0 * a0 + ul.a[1] * ul.a[1]) + ul.a[2] * ul.a[2]) + (-1.);
    q[1] = (2. / L) * vl.a[0];
    q[2] = (2. / L) * vl.a[2];
    q[3] = (2. / L) * (-vl.a[1]);
}

}  // namespace mh
