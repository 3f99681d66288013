// Analytic FP64 residual and tangent of the static corotated EulerBeam3D.
//
// Reference: toolbox/BeamElement.jl:122-208 (constructor, residual, kinematics,
// corotated), toolbox/Rotations.jl:13-135 (sinc1, scac, Rodrigues, Rodrigues⁻¹).
// Muscade differentiates the element with nested forward-mode duals
// (src/Adiff.jl, src/Taylor.jl). This file computes the same R = ∂Π/∂X and
// K = ∂R/∂X in closed form instead:
//
//   * the static residual is the gradient of Π(X) = Σ_gp dL·(½EA ε² +
//     ½ mᵢ·κ + fₑ·x) (fₑ constant in the static case), so K is its Hessian;
//   * Π depends on the 12 element dofs through the corotated frame rₛₘ and the
//     translations and rotations seen from it (BeamSpin): first and second
//     derivatives along node spins are taken in the frame's own axes.
//
// Everything is `__host__ __device__` so the same code can be exercised on the
// host in unit harnesses; the product path runs it on the GPU only.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>

// A phase ends: what follows is neither scheduled nor loaded before it. Without phases the compiler
// reads a whole record into registers at once and spills (564 B a lane of the direction kernel).
#if defined(__HIP_DEVICE_COMPILE__)
#define MH_PHASE() do { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); } while (0)
#else
#define MH_PHASE() do {} while (0)
#endif

namespace mh {

#define MH_HD __host__ __device__ __forceinline__

struct v3 { double x, y, z; };
struct m3 { double a[9]; };   // column-major: a[i + 3*j] = M(i,j)

MH_HD v3 mk(double x, double y, double z) { v3 r; r.x = x; r.y = y; r.z = z; return r; }
MH_HD v3 operator+(v3 a, v3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
MH_HD v3 operator-(v3 a, v3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
MH_HD v3 operator*(double s, v3 a) { return mk(s * a.x, s * a.y, s * a.z); }
MH_HD double dot(v3 a, v3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
MH_HD v3 cross(v3 a, v3 b) { return mk(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x); }
MH_HD double& at(m3& m, int i, int j) { return m.a[i + 3 * j]; }
MH_HD double at(const m3& m, int i, int j) { return m.a[i + 3 * j]; }
MH_HD v3 col(const m3& m, int j) { return mk(m.a[3 * j], m.a[3 * j + 1], m.a[3 * j + 2]); }
MH_HD v3 mul(const m3& m, v3 v) {
    return mk(at(m, 0, 0) * v.x + at(m, 0, 1) * v.y + at(m, 0, 2) * v.z,
              at(m, 1, 0) * v.x + at(m, 1, 1) * v.y + at(m, 1, 2) * v.z,
              at(m, 2, 0) * v.x + at(m, 2, 1) * v.y + at(m, 2, 2) * v.z);
}
MH_HD v3 mulT(const m3& m, v3 v) {   // Mᵀ v
    return mk(at(m, 0, 0) * v.x + at(m, 1, 0) * v.y + at(m, 2, 0) * v.z,
              at(m, 0, 1) * v.x + at(m, 1, 1) * v.y + at(m, 2, 1) * v.z,
              at(m, 0, 2) * v.x + at(m, 1, 2) * v.y + at(m, 2, 2) * v.z);
}
MH_HD m3 mul(const m3& A, const m3& B) {
    m3 r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.a[i + 3 * j] = at(A, i, 0) * at(B, 0, j) + at(A, i, 1) * at(B, 1, j) + at(A, i, 2) * at(B, 2, j);
    return r;
}
MH_HD m3 mulABt(const m3& A, const m3& B) {   // A Bᵀ
    m3 r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.a[i + 3 * j] = at(A, i, 0) * at(B, j, 0) + at(A, i, 1) * at(B, j, 1) + at(A, i, 2) * at(B, j, 2);
    return r;
}

// ------------------------------------------------------------ scalar kernels
// sinc1(x) = sin(x)/x with the small-argument series that Base.sinc uses
// (Rotations.jl:13): |x/π| < 1e-3 → 1 - x²/6 + x⁴/120.
MH_HD double sinpi_red(double y) {
    double x = fabs(y);
    double n = rint(2. * x);
    double rx = -0.5 * n + x;
    long q = (long)n & 3;
    double res;
    const double pi = 3.141592653589793;
    if (q == 0) res = sin(pi * rx);
    else if (q == 1) res = cos(pi * rx);
    else if (q == 2) res = 0. - sin(pi * rx);
    else res = 0. - cos(pi * rx);
    return __builtin_signbit(y) ? -res : res;
}
MH_HD double sinc1(double x) {
    const double pi = 3.141592653589793;
    double y = x / pi;
    if (fabs(y) < 1e-3) { double y2 = y * y; return 1. + y2 * (-(pi * pi) / 6. + y2 * (pi * pi * pi * pi / 120.)); }
    return sinpi_red(y) / (pi * y);
}
// scac(x) = sinc1(acos x), 5th-order series for |x-1| <= 1e-3 (Rotations.jl:61-68)
MH_HD double scac(double x) {
    double dx = x - 1.;
    if (fabs(dx) > 1e-3) return sinc1(acos(x));
    return 1. + dx * (1. / 3. + dx * (-2. / 90. + dx * (0.0052911879917544626 + dx * (-0.0016229317117234072 + dx * (0.0005625)))));
}

// Coefficients of the rotation-vector exponential and its derivatives, for θ = |v|:
//   a = sinθ/θ, b = (1-cosθ)/θ², c = (θ-sinθ)/θ³, β = b'(θ)/θ, γ = c'(θ)/θ,
//   e = (1 - a/(2b))/θ²  (coefficient of spin² in T⁻¹).
// a and b are evaluated like Rodrigues (Rotations.jl:131-135): a = sinc1(θ),
// b = sinc1(θ/2)²/2, with θ reset to 0 below 1e-14 like norm3 (Rotations.jl:106-112).
struct ExpCoef { double a, b, c, beta, gamma, e; };
MH_HD ExpCoef exp_coef(double th) {
    ExpCoef k;
    if (th < 1e-14) th = 0.;
    k.a = sinc1(th);
    double s = sinc1(th / 2.);
    k.b = s * s / 2.;
    double t2 = th * th;
    if (th < 0.1) {
        k.c = 1. / 6. + t2 * (-1. / 120. + t2 * (1. / 5040. + t2 * (-1. / 362880.)));
        k.beta = -1. / 12. + t2 * (1. / 180. + t2 * (-1. / 6720. + t2 * (1. / 453600.)));
        k.gamma = -1. / 60. + t2 * (1. / 1260. + t2 * (-1. / 60480. + t2 * (1. / 4989600.)));
        k.e = 1. / 12. + t2 * (1. / 720. + t2 * (1. / 30240. + t2 * (1. / 1209600.)));
    } else {
        k.c = (1. - k.a) / t2;
        k.beta = (k.a - 2. * k.b) / t2;
        k.gamma = (k.b - 3. * k.c) / t2;
        k.e = (1. - k.a / (2. * k.b)) / t2;
    }
    return k;
}
MH_HD double norm3(v3 v) {
    double n = sqrt(v.x * v.x + v.y * v.y + v.z * v.z);
    return n < 1e-14 ? 0. : n;
}
// Rodrigues(v) = I + a S + b S² (Rotations.jl:131-135, spin² per :114-122)
MH_HD m3 rodrigues(v3 v, const ExpCoef& k) {
    m3 r;
    double x = v.x, y = v.y, z = v.z;
    // S = spin(v); S² = v vᵀ - |v|² I
    double ab = x * y, ca = z * x, bc = y * z;
    double a2 = -x * x, b2 = -y * y, c2 = -z * z;
    at(r, 0, 0) = 1. + k.b * (c2 + b2);
    at(r, 1, 0) = k.a * z + k.b * ab;
    at(r, 2, 0) = -k.a * y + k.b * ca;
    at(r, 0, 1) = -k.a * z + k.b * ab;
    at(r, 1, 1) = 1. + k.b * (a2 + c2);
    at(r, 2, 1) = k.a * x + k.b * bc;
    at(r, 0, 2) = k.a * y + k.b * ca;
    at(r, 1, 2) = -k.a * x + k.b * bc;
    at(r, 2, 2) = 1. + k.b * (a2 + b2);
    return r;
}
// T(v)⁻¹ = I - ½ S + e S²
MH_HD m3 tangent_inv(v3 v, const ExpCoef& k) {
    m3 r;
    double x = v.x, y = v.y, z = v.z;
    double xx = x * x, yy = y * y, zz = z * z;
    at(r, 0, 0) = 1. - k.e * (yy + zz);
    at(r, 1, 1) = 1. - k.e * (xx + zz);
    at(r, 2, 2) = 1. - k.e * (xx + yy);
    at(r, 0, 1) = 0.5 * z + k.e * x * y;
    at(r, 1, 0) = -0.5 * z + k.e * x * y;
    at(r, 0, 2) = -0.5 * y + k.e * x * z;
    at(r, 2, 0) = 0.5 * y + k.e * x * z;
    at(r, 1, 2) = 0.5 * x + k.e * y * z;
    at(r, 2, 1) = -0.5 * x + k.e * y * z;
    return r;
}
// Symmetric 3×3 stored as (xx,yy,zz,xy,xz,yz).
struct s3 { double xx, yy, zz, xy, xz, yz; };
// sym part of the bilinear form (x,y) ↦ g·∂T(v)[x]y:
//   β sym(v (g×v)ᵀ) + γ sym(v (S²g)ᵀ) + c[(g·v)I - sym(g vᵀ)],  S²g = v(v·g) - g|v|²
MH_HD s3 dT_form(v3 v, v3 g, const ExpCoef& k) {
    v3 gv = cross(g, v);
    double vg = dot(v, g), vv = dot(v, v);
    v3 s2g = vg * v - vv * g;
    v3 p = k.beta * gv + k.gamma * s2g;   // B = v pᵀ + c[(g·v)I - g vᵀ]...
    s3 r;
    r.xx = v.x * p.x + k.c * (vg - g.x * v.x);
    r.yy = v.y * p.y + k.c * (vg - g.y * v.y);
    r.zz = v.z * p.z + k.c * (vg - g.z * v.z);
    r.xy = 0.5 * (v.x * p.y + p.x * v.y) - 0.5 * k.c * (g.x * v.y + v.x * g.y);
    r.xz = 0.5 * (v.x * p.z + p.x * v.z) - 0.5 * k.c * (g.x * v.z + v.x * g.z);
    r.yz = 0.5 * (v.y * p.z + p.y * v.z) - 0.5 * k.c * (g.y * v.z + v.y * g.z);
    return r;
}
MH_HD v3 smul(const s3& s, v3 x) {
    return mk(s.xx * x.x + s.xy * x.y + s.xz * x.z, s.xy * x.x + s.yy * x.y + s.yz * x.z, s.xz * x.x + s.yz * x.y + s.zz * x.z);
}

// ---------------------------------------------------------- element geometry
struct BeamGeo {
    v3 cm, tgm;
    m3 rm;        // columns t, n, b
    double L;
    double zgp[4], dL[4];
    int bad;      // orient2 nearly parallel to the element (BeamElement.jl:135)
};
MH_HD BeamGeo beam_geometry(v3 c1, v3 c2, v3 o2) {   // BeamElement.jl:122-148
    BeamGeo g;
    g.cm = mk((c1.x + c2.x) / 2., (c1.y + c2.y) / 2., (c1.z + c2.z) / 2.);
    g.tgm = c2 - c1;
    double L = sqrt(dot(g.tgm, g.tgm));
    v3 t = mk(g.tgm.x / L, g.tgm.y / L, g.tgm.z / L);
    double no = sqrt(dot(o2, o2));
    o2 = mk(o2.x / no, o2.y / no, o2.z / no);
    double d = dot(o2, t);
    v3 n = o2 - d * t;
    double nn = sqrt(dot(n, n));
    g.bad = !(nn > 1e-3);
    n = mk(n.x / nn, n.y / nn, n.z / nn);
    v3 b = cross(t, n);
    g.rm.a[0] = t.x; g.rm.a[1] = t.y; g.rm.a[2] = t.z;
    g.rm.a[3] = n.x; g.rm.a[4] = n.y; g.rm.a[5] = n.z;
    g.rm.a[6] = b.x; g.rm.a[7] = b.y; g.rm.a[8] = b.z;
    g.L = L;
    const double s30 = 5.477225575051661;      // √30
    const double s65 = 1.0954451150103321;     // √(6/5)
    g.dL[0] = L / 2. * (18. - s30) / 36.; g.dL[1] = L / 2. * (18. + s30) / 36.;
    g.dL[2] = g.dL[1]; g.dL[3] = g.dL[0];
    double z1 = 0.5 * sqrt(3. / 7. + 2. / 7. * s65), z2 = 0.5 * sqrt(3. / 7. - 2. / 7. * s65);
    g.zgp[0] = -z1; g.zgp[1] = -z2; g.zgp[2] = z2; g.zgp[3] = z1;
    return g;
}



// ------------------------------------------------------------ compact tangent
// The static tangent of the 2-node beam has an exact block structure: the
// translations enter Π only through d = ½(u₂-u₁) (internal terms) and
// c = ½(u₁+u₂) (linearly, external load), so with A = ∂²Π/∂d² (global frame),
// T = ∂²Π/∂d∂v (3×6 over the rotation dofs v = (v₁,v₂)) and S = ∂²Π/∂v² (6×6):
//     K[u₁,u₁] = K[u₂,u₂] = ¼A,  K[u₁,u₂] = K[u₂,u₁] = -¼A,
//     K[u₁,v]  = -½T,            K[u₂,v]  = +½T,          K[v,v] = S,
// and K is symmetric. These 45 numbers are the element output; the scatter
// multiplies by the exact powers of two ±1, ±½, ±¼.
// Slots: A at 0..5 (xx,yy,zz,xy,xz,yz), T at 6..23 (T[a][r] = 6 + 6a + r),
// S at 24..44 (upper triangle, row-major: 24 + sym6(r,s)).
constexpr int kCompact = 45;
MH_HD int sym3(int a, int b) {   // (xx,yy,zz,xy,xz,yz)
    if (a > b) { int t = a; a = b; b = t; }
    return a == b ? a : (a == 0 ? 2 + b : 5);
}
MH_HD int sym6(int r, int s) {   // upper triangle of 6×6, row-major
    if (r > s) { int t = r; r = s; s = t; }
    return r * 6 - (r * (r - 1)) / 2 + (s - r);
}
// Compact slot and exact multiplier of element entry K[i][j] (i,j = 0..11,
// element dof order t1,t2,t3,r1,r2,r3 of node 1 then node 2).
MH_HD int compact_slot(int i, int j, double* mult) {
    int ni = i / 6, a = i % 6, nj = j / 6, b = j % 6;
    bool ri = a >= 3, rj = b >= 3;
    if (!ri && !rj) { *mult = (ni == nj) ? 0.25 : -0.25; return sym3(a, b); }
    if (!ri && rj) { *mult = ni == 0 ? -0.5 : 0.5; return 6 + 6 * a + (3 * nj + b - 3); }
    if (ri && !rj) { *mult = nj == 0 ? -0.5 : 0.5; return 6 + 6 * b + (3 * ni + a - 3); }
    *mult = 1.;
    return 24 + sym6(3 * ni + a - 3, 3 * nj + b - 3);
}

struct BeamSection { double EA, EI2, EI3, GJ, w; };
struct BeamOut { double R[12]; double Kc[kCompact]; int nan; };

// ------------------------------------------------ coefficient functions of t = θ²
// a = sinθ/θ, b = (1−cosθ)/θ², c = (θ−sinθ)/θ³, each with its first two derivatives in t
// (a′ = ½(c−b), b′ = (a−2b)/2t, c′ = (b−3c)/2t). Series for t < 1 (last term below 1e-18).
struct RotFun { double a, b, c, a1, b1, c1, a2, b2, c2; };
MH_HD RotFun rot_fun(double t) {
    RotFun f;
    if (t < 1.) {
        // 1/(2k+2)!, 1/(2k+3)!
        const double B[10] = {0.5, 1. / 24., 1. / 720., 1. / 40320., 1. / 3628800., 1. / 479001600., 1. / 87178291200.,
                              1. / 20922789888000., 1. / 6402373705728000., 1. / 2432902008176640000.};
        const double C[10] = {1. / 6., 1. / 120., 1. / 5040., 1. / 362880., 1. / 39916800., 1. / 6227020800.,
                              1. / 1307674368000., 1. / 355687428096000., 1. / 121645100408832000.,
                              1. / 51090942171709440000.};
        const double u = -t;
        double b = 0., b1 = 0., b2 = 0., c = 0., c1 = 0., c2 = 0.;
#pragma unroll
        for (int k = 9; k >= 0; --k) {
            b = b * u + B[k]; c = c * u + C[k];
            if (k > 0) { b1 = b1 * u - k * B[k]; c1 = c1 * u - k * C[k]; }
            if (k > 1) { b2 = b2 * u + k * (k - 1) * B[k]; c2 = c2 * u + k * (k - 1) * C[k]; }
        }
        f.b = b; f.b1 = b1; f.b2 = b2; f.c = c; f.c1 = c1; f.c2 = c2;
        f.a = 1. - t * c;
    } else {
        const double th = sqrt(t), h = 0.5 / t, sh = sin(0.5 * th);
        f.a = sin(th) / th;
        f.b = 2. * sh * sh / t;
        f.c = (1. - f.a) / t;
        f.b1 = (f.a - 2. * f.b) * h;
        f.c1 = (f.b - 3. * f.c) * h;
        const double a1 = 0.5 * (f.c - f.b);
        f.b2 = (a1 - 4. * f.b1) * h;
        f.c2 = (f.b1 - 5. * f.c1) * h;
    }
    f.a1 = 0.5 * (f.c - f.b);
    f.a2 = 0.5 * (f.c1 - f.b1);
    return f;
}
// τ = tan(φ/4)/φ and κ = ½e − ¼τ, e = (1 − (φ/2)cot(φ/2))/φ², with two derivatives in t = φ² = 4θ²,
// from the functions at θ = φ/2 (< π/2): τ = b/2a, κ = −c/8a.
struct HalfFun { double k, k1, k2, q, q1, q2; };   // τ, τ′, τ″, κ, κ′, κ″
MH_HD HalfFun half_fun(const RotFun& f) {
    const double h = 0.5 / f.a, g = f.a1 / f.a;
    HalfFun o;
    o.k = f.b * h;
    const double k1 = f.b1 * h - g * o.k;
    o.k1 = 0.25 * k1;
    o.k2 = 0.0625 * ((f.b2 - f.a2 / f.a * f.b) * h - 2. * g * k1);
    const double q = f.c * h, q1 = f.c1 * h - g * q;
    o.q = -0.25 * q;
    o.q1 = -0.0625 * q1;
    o.q2 = -0.015625 * ((f.c2 - f.a2 / f.a * f.c) * h - 2. * g * q1);
    return o;
}

// The corotated frame (BeamElement.jl:192-208): r = rₛₘ, d = uₗ₂ + (L/2, 0, 0), vl = vₗ₂.
struct BeamFrame { m3 r; v3 d, vl; RotFun f1, f2, fh; };   // coefficients at |v₁|², |v₂|², |vₗ|²
MH_HD void beam_frame(const BeamGeo& G, const double* X, BeamFrame& f) {
    const v3 v1 = mk(X[3], X[4], X[5]), v2 = mk(X[9], X[10], X[11]);
    ExpCoef k;
    f.f1 = rot_fun(dot(v1, v1)); f.f2 = rot_fun(dot(v2, v2));
    k.a = f.f1.a; k.b = f.f1.b;
    const m3 R1 = rodrigues(v1, k);
    k.a = f.f2.a; k.b = f.f2.b;
    const m3 M = mulABt(rodrigues(v2, k), R1);
    // Δv = ½ Rodrigues⁻¹(M), Rodrigues⁻¹(M) = spin⁻¹(M)/scac((tr M - 1)/2)
    const double h = 0.25 / scac((at(M, 0, 0) + at(M, 1, 1) + at(M, 2, 2) - 1.) / 2.);
    const v3 dv = mk((at(M, 2, 1) - at(M, 1, 2)) * h, (at(M, 0, 2) - at(M, 2, 0)) * h, (at(M, 1, 0) - at(M, 0, 1)) * h);
    f.fh = rot_fun(dot(dv, dv));
    k.a = f.fh.a; k.b = f.fh.b;
    f.r = mul(mul(rodrigues(dv, k), R1), G.rm);
    // (u₂ + ½tgₘ) − cₛₘ in the reference's order: its rounding is the axial strain's
    const v3 cs = mk(0.5 * (X[0] + X[6]), 0.5 * (X[1] + X[7]), 0.5 * (X[2] + X[8]));
    f.d = mulT(f.r, mk(X[6] + G.tgm.x * 0.5 - cs.x, X[7] + G.tgm.y * 0.5 - cs.y, X[8] + G.tgm.z * 0.5 - cs.z));
    f.vl = mulT(f.r, dv);
}

// The loads held fixed in the closed form: moments over the Gauss points of e_gp = dL_gp·fₑ with the
// shape factors 1, ya, yu, yv of x_gp (global), and the couple Σ dL·mₑ. For a constant load ya and yu
// sum to zero and yv to −L²/6.
struct BeamLoads { v3 e0, ea, eu, ev, m; };

// Residual and compact tangent of Π = Π_int + Σ_gp e_gp·x_gp + m·vₛₘ with the loads held fixed;
// GEN = false: a constant load (ea = eu = m = 0). vₛₘ = Rodrigues⁻¹(rₛₘ) (BeamElement.jl:203).
//
// In the corotated frame (components along r's axes), with the node spins t_n = rᵀT(v_n)δv_n,
// s = t₁+t₂, Δ = t₂−t₁, V = spin vₗ:
//   frame spin ω = ½s − τVΔ, δvₗ = CΔ, C = ½I + 4κV², δd = rᵀδ(½(u₂−u₁)) + d×ω
// (τ, κ: half_fun at |φ|² = 4|vₗ|²). The Gauss sums of the internal energy are exact:
// Π_int = ½EA·L·ε² + ½(k₃d_y² + k₂d_z²) + ½vₗ·D vₗ, k = 48EI/L³, D = 4/L·diag(GJ, EI₂, EI₃).
// Second derivatives: of ω and vₗ along constant node spins (the curvature of the rotations),
//   N·W₂ + F_v·V₂ = Δ·(kA I + sym(v hᵀ))Δ + ½τ(N·s v·Δ − N·v s·Δ) + ½s·(P×Δ),
// of body vectors b = rᵀB: ω×(ω×b). The axial force meets the rotations only through d×ω and drops
// out of Q (the ω-ω part) and of the coupling to translations.
//
// Bound: FP64 latency at two waves per SIMD, then HBM. Over six columns of global spins the same
// element took 6,299 counted operations and 462 registers (one wave per SIMD); here 2,794 and 256.
// 973,000 elements: 320 µs before, 142 now.
struct BeamSpin {
    v3 Fb, N, Fv, ve, a, u;          // forces and moment, body loads
    s3 Q, KD; m3 KS;                 // ω-ω, Δ-Δ, s-Δ
    double k2, k3, c2, c3, tau, al, be;   // bending springs, axial terms of D_uu, τ, C = αI + βvvᵀ
    v3 l1, l2;                       // node moments (global)
    RotFun f1, f2;                   // T(v_n)
};
template <bool GEN>
MH_HD void beam_spin(const BeamSection& S, double L, const BeamFrame& f, const double* X, const BeamLoads& ld, BeamSpin& o) {
    const m3& r = f.r;
    const v3 d = f.d, v = f.vl;
    const v3 v1 = mk(X[3], X[4], X[5]), v2 = mk(X[9], X[10], X[11]);
    const double k3 = 48. * S.EI3 / (L * L * L), k2 = 48. * S.EI2 / (L * L * L);
    const v3 D = mk(4. / L * S.GJ, 4. / L * S.EI2, 4. / L * S.EI3);
    const double ell = sqrt(dot(d, d)), de = 2. / (L * ell);
    const double eps = ell * 2. / L - 1., fa = S.EA * L * eps;
    const v3 ve = mulT(r, ld.ev);
    v3 a = mk(0., 0., 0.), u = a;
    // forces conjugate to d (Fb: without the axial force along d) and vₗ, moment conjugate to ω
    v3 Fb = mk(0., k3 * d.y, k2 * d.z), N;
    const v3 Fv = mk(D.x * v.x, D.y * v.y - ve.z, D.z * v.z + ve.y);
    if (GEN) {
        a = mulT(r, ld.ea); u = mulT(r, ld.eu);
        Fb = Fb + mk(a.x, u.y, u.z);
    }
    N = cross(Fb, d) + cross(mk(0., v.z, -v.y), ve);
    s3 Q;   // ω-ω
    {
        auto sy = [](s3& q, v3 x, v3 y, double w) {   // q += w·sym(x yᵀ)
            q.xx += w * x.x * y.x; q.yy += w * x.y * y.y; q.zz += w * x.z * y.z;
            q.xy += 0.5 * w * (x.x * y.y + x.y * y.x); q.xz += 0.5 * w * (x.x * y.z + x.z * y.x);
            q.yz += 0.5 * w * (x.y * y.z + x.z * y.y);
        };
        const v3 rv = mk(0., v.z, -v.y);
        double tr = dot(Fb, d) + dot(rv, ve);
        Q.xx = Q.yy = Q.zz = Q.xy = Q.xz = Q.yz = 0.;
        sy(Q, Fb, d, 1.);
        sy(Q, rv, ve, 1.);
        const v3 gy = mk(d.z, 0., -d.x), gz = mk(-d.y, d.x, 0.);
        sy(Q, gy, gy, k3);
        sy(Q, gz, gz, k2);
        if (GEN) {
            const v3 dx = mk(d.x, 0., 0.), dyz = mk(0., d.y, d.z);
            N = N + cross(dx, a) + cross(dyz, u);
            tr += d.x * a.x + (d.y * u.y + d.z * u.z);
            sy(Q, dx, a, 1.);
            sy(Q, dyz, u, 1.);
            sy(Q, mk(0., -a.z, a.y), mk(0., -d.z, d.y), 2.);
            sy(Q, mk(u.z, 0., -u.x), gy, 2.);
            sy(Q, mk(-u.y, u.x, 0.), gz, 2.);
            // couple: μ = T(ψ)⁻ᵀ rᵀm and −Jᵀ dT(ψ, μ) J, J = T(ψ)⁻¹ (r = Rodrigues(ψ) commutes with them)
            double sc = scac((at(r, 0, 0) + at(r, 1, 1) + at(r, 2, 2) - 1.) / 2.);
            const v3 psi = mk((at(r, 2, 1) - at(r, 1, 2)) / 2. / sc, (at(r, 0, 2) - at(r, 2, 0)) / 2. / sc,
                              (at(r, 1, 0) - at(r, 0, 1)) / 2. / sc);
            const ExpCoef kp = exp_coef(norm3(psi));
            const m3 J = tangent_inv(psi, kp);
            const v3 mu = mulT(J, mulT(r, ld.m));
            N = N + mu;
            const s3 B = dT_form(psi, mu, kp);
            const v3 J0 = col(J, 0), J1 = col(J, 1), J2 = col(J, 2), B0 = smul(B, J0), B1 = smul(B, J1), B2 = smul(B, J2);
            Q.xx -= dot(J0, B0); Q.yy -= dot(J1, B1); Q.zz -= dot(J2, B2);
            Q.xy -= dot(J0, B1); Q.xz -= dot(J0, B2); Q.yz -= dot(J1, B2);
        }
        Q.xx -= tr; Q.yy -= tr; Q.zz -= tr;
    }
    o.c2 = fa * de;
    o.c3 = S.EA * L * de * de - o.c2 / (ell * ell);
    // rotations: node moments and the spin blocks K₁₁, K₁₂, K₂₂
    const double vv = dot(v, v);
    const HalfFun hf = half_fun(f.fh);
    const double tau = hf.k, be = 4. * hf.q, al = 0.5 - be * vv;
    const v3 P = al * Fv + (be * dot(v, Fv)) * v, Nv = cross(N, v);
    o.f1 = f.f1; o.f2 = f.f2;
    const v3 pD = P - tau * Nv;
    o.l1 = mul(r, 0.5 * N - pD); o.l2 = mul(r, 0.5 * N + pD);
    m3 QV;   // Q V
    m3& KS = o.KS;   // K_sΔ = −½τQV + ½GᵀC + ¼τ(N vᵀ − N·v I) + ¼spin(P), G = spin(e₁) spin(ve)
    s3& KD = o.KD;   // K_ΔΔ = τ²VᵀQV + C D C + sym(C G W) + kA I + sym(v hᵀ)
    {
        const v3 q0 = mk(Q.xx, Q.xy, Q.xz), q1 = mk(Q.xy, Q.yy, Q.yz), q2 = mk(Q.xz, Q.yz, Q.zz);
        // rows of QV: q×v
        const v3 w0 = cross(q0, v), w1 = cross(q1, v), w2 = cross(q2, v);
        QV.a[0] = w0.x; QV.a[3] = w0.y; QV.a[6] = w0.z;
        QV.a[1] = w1.x; QV.a[4] = w1.y; QV.a[7] = w1.z;
        QV.a[2] = w2.x; QV.a[5] = w2.y; QV.a[8] = w2.z;
        // VᵀQV: columns QV_j → −v×(QV_j)
        const v3 c0 = cross(col(QV, 0), v), c1 = cross(col(QV, 1), v), c2 = cross(col(QV, 2), v);
        const double t2 = tau * tau;
        KD.xx = t2 * c0.x; KD.yy = t2 * c1.y; KD.zz = t2 * c2.z;
        KD.xy = t2 * c1.x; KD.xz = t2 * c2.x; KD.yz = t2 * c2.y;
        const double b2 = be * be * (D.x * v.x * v.x + D.y * v.y * v.y + D.z * v.z * v.z), ab = al * be;
        const double fv = dot(Fv, v);
        const double kA = fv * (-0.5 * tau + be * al);
        const double kB = 0.5 * tau - 16. * hf.q1 * vv + be * (al - 1. - tau * vv);
        const double kC = fv * (16. * hf.q1 + 2. * be * be + be * tau);
        const double c = tau * tau + 4. * hf.k1 + be * tau;
        const v3 h = kB * Fv + kC * v - c * Nv;
        KD.xx += al * al * D.x + (2. * ab * D.x + b2) * v.x * v.x + kA + v.x * h.x;
        KD.yy += al * al * D.y + (2. * ab * D.y + b2) * v.y * v.y + kA + v.y * h.y;
        KD.zz += al * al * D.z + (2. * ab * D.z + b2) * v.z * v.z + kA + v.z * h.z;
        KD.xy += (ab * (D.x + D.y) + b2) * v.x * v.y + 0.5 * (v.x * h.y + v.y * h.x);
        KD.xz += (ab * (D.x + D.z) + b2) * v.x * v.z + 0.5 * (v.x * h.z + v.z * h.x);
        KD.yz += (ab * (D.y + D.z) + b2) * v.y * v.z + 0.5 * (v.y * h.z + v.z * h.y);
        // G = ve e₁ᵀ − (ve·e₁) I; GᵀC = e₁ (C ve)ᵀ − veₓ C, CGW = −τ(C ve (e₁ᵀV) − veₓ C V); CV = αV
        const v3 Cve = al * ve + (be * dot(v, ve)) * v;
        const v3 eV = mk(0., -v.z, v.y);   // row e₁ᵀV
        // sym(αV) = 0, so only the dyad remains: CGW + (CGW)ᵀ = −τ(Cve eVᵀ + eV Cveᵀ)
        KD.yy -= 2. * tau * Cve.y * eV.y; KD.zz -= 2. * tau * Cve.z * eV.z;
        KD.xy -= tau * Cve.x * eV.y; KD.xz -= tau * Cve.x * eV.z; KD.yz -= tau * (Cve.y * eV.z + Cve.z * eV.y);
        const double nv = 0.25 * tau * dot(N, v), t4 = 0.25 * tau, ht = 0.5 * tau;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double vj = j == 0 ? v.x : (j == 1 ? v.y : v.z);
            KS.a[3 * j] = t4 * N.x * vj - ht * QV.a[3 * j];
            KS.a[3 * j + 1] = t4 * N.y * vj - ht * QV.a[3 * j + 1];
            KS.a[3 * j + 2] = t4 * N.z * vj - ht * QV.a[3 * j + 2];
        }
        KS.a[0] -= nv; KS.a[4] -= nv; KS.a[8] -= nv;
        KS.a[0] += 0.5 * Cve.x; KS.a[3] += 0.5 * Cve.y; KS.a[6] += 0.5 * Cve.z;   // ½e₁(C ve)ᵀ
        const double hx = 0.5 * ve.x;
        KS.a[0] -= hx * (al + be * v.x * v.x); KS.a[4] -= hx * (al + be * v.y * v.y); KS.a[8] -= hx * (al + be * v.z * v.z);
        const double sxy = hx * be * v.x * v.y, sxz = hx * be * v.x * v.z, syz = hx * be * v.y * v.z;
        KS.a[1] -= sxy; KS.a[3] -= sxy; KS.a[2] -= sxz; KS.a[6] -= sxz; KS.a[5] -= syz; KS.a[7] -= syz;
        KS.a[1] += 0.25 * P.z; KS.a[3] -= 0.25 * P.z;
        KS.a[2] -= 0.25 * P.y; KS.a[6] += 0.25 * P.y;
        KS.a[5] += 0.25 * P.x; KS.a[7] -= 0.25 * P.x;
    }
    o.Fb = Fb; o.N = N; o.Fv = Fv; o.ve = ve; o.a = a; o.u = u; o.Q = Q;
    o.k2 = k2; o.k3 = k3; o.tau = tau; o.al = al; o.be = be;
}

template <bool GEN>
MH_HD void beam_tangent(const BeamSection& S, double L, const BeamFrame& f, const double* X, const BeamLoads& ld,
                        BeamOut& out) {
    const m3& r = f.r;
    const v3 d = f.d, v = f.vl;
    const v3 v1 = mk(X[3], X[4], X[5]), v2 = mk(X[9], X[10], X[11]);
    BeamSpin o;
    beam_spin<GEN>(S, L, f, X, ld, o);
    const RotFun &f1 = o.f1, &f2 = o.f2;
    const v3 &Fb = o.Fb, &a = o.a, &u = o.u, &l1 = o.l1, &l2 = o.l2;
    const s3 &Q = o.Q, &KD = o.KD;
    const m3& KS = o.KS;
    const double k2 = o.k2, k3 = o.k3, tau = o.tau;
    // translations: residual and A = r D_uu rᵀ, D_uu = c₂I + c₃ d dᵀ + diag(0, k₃, k₂)
    {
        const v3 g = mul(r, Fb + o.c2 * d);
        out.R[0] = 0.5 * (ld.e0.x - g.x); out.R[1] = 0.5 * (ld.e0.y - g.y); out.R[2] = 0.5 * (ld.e0.z - g.z);
        out.R[6] = 0.5 * (ld.e0.x + g.x); out.R[7] = 0.5 * (ld.e0.y + g.y); out.R[8] = 0.5 * (ld.e0.z + g.z);
        const double c2 = o.c2, c3 = o.c3;
        const v3 dg = mul(r, d), ry = col(r, 1), rz = col(r, 2);
        out.Kc[0] = c2 + (c3 * dg.x * dg.x + k3 * ry.x * ry.x + k2 * rz.x * rz.x);
        out.Kc[1] = c2 + (c3 * dg.y * dg.y + k3 * ry.y * ry.y + k2 * rz.y * rz.y);
        out.Kc[2] = c2 + (c3 * dg.z * dg.z + k3 * ry.z * ry.z + k2 * rz.z * rz.z);
        out.Kc[3] = c3 * dg.x * dg.y + k3 * ry.x * ry.y + k2 * rz.x * rz.y;
        out.Kc[4] = c3 * dg.x * dg.z + k3 * ry.x * ry.z + k2 * rz.x * rz.z;
        out.Kc[5] = c3 * dg.y * dg.z + k3 * ry.y * ry.z + k2 * rz.y * rz.z;
    }
    auto Tt = [](v3 w, const RotFun& k, v3 q) { const v3 y = cross(w, q); return q - k.b * y + k.c * cross(w, y); };
    {
        const v3 q1 = Tt(v1, f1, l1), q2 = Tt(v2, f2, l2);
        out.R[3] = q1.x; out.R[4] = q1.y; out.R[5] = q1.z;
        out.R[9] = q2.x; out.R[10] = q2.y; out.R[11] = q2.z;
    }
    // L_n = rᵀT(v_n), column j: rᵀ(e_j + b v×e_j + c v×(v×e_j))
    auto Lcol = [&](v3 w, const RotFun& k, int j) {
        const v3 e = mk(j == 0 ? 1. : 0., j == 1 ? 1. : 0., j == 2 ? 1. : 0.), y = cross(w, e);
        return mulT(r, e + k.b * y + k.c * cross(w, y));
    };
    v3 L1[3], L2[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) { L1[j] = Lcol(v1, f1, j); L2[j] = Lcol(v2, f2, j); }
    auto dyt = [](v3 w, v3 g, const RotFun& k) {
        ExpCoef q;
        q.c = k.c; q.beta = 2. * k.b1; q.gamma = 2. * k.c1;
        return dT_form(w, g, q);
    };
    double* Sm = out.Kc + 24;
    {
        auto sm = [&](double sg) {   // ¼Q + K_ΔΔ + sg (K_sΔ + K_sΔᵀ)
            s3 k;
            k.xx = 0.25 * Q.xx + KD.xx + 2. * sg * KS.a[0]; k.yy = 0.25 * Q.yy + KD.yy + 2. * sg * KS.a[4];
            k.zz = 0.25 * Q.zz + KD.zz + 2. * sg * KS.a[8];
            k.xy = 0.25 * Q.xy + KD.xy + sg * (KS.a[1] + KS.a[3]);
            k.xz = 0.25 * Q.xz + KD.xz + sg * (KS.a[2] + KS.a[6]);
            k.yz = 0.25 * Q.yz + KD.yz + sg * (KS.a[5] + KS.a[7]);
            return k;
        };
        const s3 K1 = sm(-1.), B1 = dyt(v1, l1, f1);
        const v3 x0 = smul(K1, L1[0]), x1 = smul(K1, L1[1]), x2 = smul(K1, L1[2]);
        Sm[sym6(0, 0)] = dot(L1[0], x0) + B1.xx; Sm[sym6(0, 1)] = dot(L1[0], x1) + B1.xy;
        Sm[sym6(0, 2)] = dot(L1[0], x2) + B1.xz; Sm[sym6(1, 1)] = dot(L1[1], x1) + B1.yy;
        Sm[sym6(1, 2)] = dot(L1[1], x2) + B1.yz; Sm[sym6(2, 2)] = dot(L1[2], x2) + B1.zz;
        const s3 K2 = sm(1.), B2 = dyt(v2, l2, f2);
        const v3 y0 = smul(K2, L2[0]), y1 = smul(K2, L2[1]), y2 = smul(K2, L2[2]);
        Sm[sym6(3, 3)] = dot(L2[0], y0) + B2.xx; Sm[sym6(3, 4)] = dot(L2[0], y1) + B2.xy;
        Sm[sym6(3, 5)] = dot(L2[0], y2) + B2.xz; Sm[sym6(4, 4)] = dot(L2[1], y1) + B2.yy;
        Sm[sym6(4, 5)] = dot(L2[1], y2) + B2.yz; Sm[sym6(5, 5)] = dot(L2[2], y2) + B2.zz;
        // K₁₂ = ¼Q − K_ΔΔ + K_sΔ − K_sΔᵀ
        const double qxx = 0.25 * Q.xx - KD.xx, qyy = 0.25 * Q.yy - KD.yy, qzz = 0.25 * Q.zz - KD.zz;
        const double qxy = 0.25 * Q.xy - KD.xy, qxz = 0.25 * Q.xz - KD.xz, qyz = 0.25 * Q.yz - KD.yz;
        const double axy = KS.a[3] - KS.a[1], axz = KS.a[6] - KS.a[2], ayz = KS.a[7] - KS.a[5];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const v3 q = L2[j];
            const v3 z = mk(qxx * q.x + (qxy + axy) * q.y + (qxz + axz) * q.z,
                            (qxy - axy) * q.x + qyy * q.y + (qyz + ayz) * q.z,
                            (qxz - axz) * q.x + (qyz - ayz) * q.y + qzz * q.z);
#pragma unroll
            for (int i = 0; i < 3; ++i) Sm[sym6(i, 3 + j)] = dot(L1[i], z);
        }
    }
    // T = r T_ω [W₁L₁ | W₂L₂], W = ½I ± τV, T_ω ω = ω×Fb + (0, k₃, k₂)∘(d×ω) + ((a×ω)ₓ, (u×ω)_y, (u×ω)_z)
    auto Tcol = [&](v3 l, double sg) {
        const v3 w = 0.5 * l + (sg * tau) * cross(v, l);   // ω of this node's column
        const v3 dw = cross(d, w);
        v3 t = cross(w, Fb) + mk(0., k3 * dw.y, k2 * dw.z);
        if (GEN) { const v3 aw = cross(a, w), uw = cross(u, w); t = t + mk(aw.x, uw.y, uw.z); }
        return mul(r, t);
    };
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const v3 t1 = Tcol(L1[j], 1.), t2 = Tcol(L2[j], -1.);
        out.Kc[6 + j] = t1.x; out.Kc[12 + j] = t1.y; out.Kc[18 + j] = t1.z;
        out.Kc[9 + j] = t2.x; out.Kc[15 + j] = t2.y; out.Kc[21 + j] = t2.z;
    }
    int nan = 0;
    // Muscade's residual always contracts mₑ with ∂vₛₘ/∂X (BeamElement.jl:170), with
    // vₛₘ = Rodrigues⁻¹(rₛₘ) = spin⁻¹(rₛₘ)/scac((tr rₛₘ - 1)/2): for a corotated frame at
    // a half turn, scac and acos′ there make it NaN even where mₑ = 0.
    if (!GEN) nan |= !((at(r, 0, 0) + at(r, 1, 1) + at(r, 2, 2) - 1.) / 2. > -1.);
    for (int i = 0; i < 12; ++i) nan |= (out.R[i] != out.R[i]);
    for (int i = 0; i < kCompact; ++i) nan |= (out.Kc[i] != out.Kc[i]);
    out.nan = nan;
}
// The static element: fₑ constant along the beam.
MH_HD void beam_static(const BeamGeo& G, const BeamSection& S, v3 fe, const double* X, BeamOut& out) {
    BeamFrame f;
    beam_frame(G, X, f);
    BeamLoads ld;
    ld.e0 = G.L * fe;
    ld.ev = (-G.L * G.L / 6.) * fe;
    ld.ea = ld.eu = ld.m = mk(0., 0., 0.);
    beam_tangent<false>(S, G.L, f, X, ld, out);
}

// Λ·∂R/∂X (g, 12) and Λ·∂R/∂fₑ (gf) of the static element: the second derivative of Π along Λ, without
// forming the tangent. Returns whether a value is NaN (the element's own NaN included).
MH_HD int beam_static_vjp(const BeamGeo& G, const BeamSection& S, v3 fe, const double* X, const double* lam, double* g,
                          v3& gf) {
    const double L = G.L;
    BeamFrame f;
    beam_frame(G, X, f);
    BeamLoads ld;
    ld.e0 = L * fe;
    ld.ev = (-L * L / 6.) * fe;
    ld.ea = ld.eu = ld.m = mk(0., 0., 0.);
    BeamSpin o;
    beam_spin<false>(S, L, f, X, ld, o);
    const m3& r = f.r;
    const v3 d = f.d, v = f.vl, v1 = mk(X[3], X[4], X[5]), v2 = mk(X[9], X[10], X[11]);
    const v3 u1 = mk(lam[0], lam[1], lam[2]), r1 = mk(lam[3], lam[4], lam[5]), u2 = mk(lam[6], lam[7], lam[8]),
             r2 = mk(lam[9], lam[10], lam[11]);
    auto T = [](v3 w, const RotFun& k, v3 q, double sg) { const v3 y = cross(w, q); return q + (sg * k.b) * y + k.c * cross(w, y); };
    const v3 t1 = mulT(r, T(v1, o.f1, r1, 1.)), t2 = mulT(r, T(v2, o.f2, r2, 1.));
    const v3 s = t1 + t2, dl = t2 - t1, D = mulT(r, 0.5 * (u2 - u1));
    const v3 w = 0.5 * s - o.tau * cross(v, dl), dw = cross(d, w);
    // d: D_uu D + T_ω ω
    const v3 k = mk(0., o.k3, o.k2);
    auto had = [](v3 x, v3 y) { return mk(x.x * y.x, x.y * y.y, x.z * y.z); };
    const v3 gd = mul(r, o.c2 * D + (o.c3 * dot(d, D)) * d + had(k, D) + cross(w, o.Fb) + had(k, dw));
    // T_ωᵀD on both nodes' frame spins
    const v3 q = cross(o.Fb, D) + cross(had(k, D), d), qv = o.tau * cross(v, q);
    const v3 ys = 0.25 * smul(o.Q, s) + mul(o.KS, dl), yd = mulT(o.KS, s) + smul(o.KD, dl);
    const v3 y1 = ys - yd + 0.5 * q - qv, y2 = ys + yd + 0.5 * q + qv;
    ExpCoef kc;
    kc.c = o.f1.c; kc.beta = 2. * o.f1.b1; kc.gamma = 2. * o.f1.c1;
    const v3 g1 = T(v1, o.f1, mul(r, y1), -1.) + smul(dT_form(v1, o.l1, kc), r1);
    kc.c = o.f2.c; kc.beta = 2. * o.f2.b1; kc.gamma = 2. * o.f2.c1;
    const v3 g2 = T(v2, o.f2, mul(r, y2), -1.) + smul(dT_form(v2, o.l2, kc), r2);
    g[0] = -0.5 * gd.x; g[1] = -0.5 * gd.y; g[2] = -0.5 * gd.z; g[3] = g1.x; g[4] = g1.y; g[5] = g1.z;
    g[6] = 0.5 * gd.x; g[7] = 0.5 * gd.y; g[8] = 0.5 * gd.z; g[9] = g2.x; g[10] = g2.y; g[11] = g2.z;
    // Σ_gp dL x_gp = L cₛₘ − L²/6 r(vₗ×e₁)
    const v3 dvl = o.al * dl + (o.be * dot(v, dl)) * v;
    gf = (0.5 * L) * (u1 + u2) + (-L * L / 6.) * mul(r, cross(w, mk(0., v.z, -v.y)) + mk(0., dvl.z, -dvl.y));
    int nan = !((at(r, 0, 0) + at(r, 1, 1) + at(r, 2, 2) - 1.) / 2. > -1.);
    for (int i = 0; i < 12; ++i) nan |= g[i] != g[i];
    return nan;
}

}  // namespace mh
