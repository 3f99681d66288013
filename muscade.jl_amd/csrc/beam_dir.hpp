// Directions of the dynamic EulerBeam3D in closed form: the derivatives of its loads and of the
// Jacobians of x_gp and vₛₘ along a trial path X⁽ⁿ⁾ + ε·δX⁽ⁿ⁾ (n < 3 time levels), in the
// corotated frame.
//
// With r = rₛₘ, vectors in components along r's axes (body frame), the rotations as spins:
//   node spins      t_n = rᵀ T(v_n) δv_n  (T = I + bS + cS², the left Jacobian of Rodrigues)
//   frame spin      ω   = ½(s − τ φ×Δ),  s = t₁+t₂, Δ = t₂−t₁, τ = tan(|φ|/4)/|φ|
//   δvₗ             =  ½Δ + κ φ×(φ×Δ),   κ = ½e − ¼τ (e of T⁻¹),   φ = rᵀφ = 2vₗ
// (ω = Pᵀt₁ + Pt₂ with P = (I + Rodrigues(φ/2))⁻¹ = ½(I − τ spin φ), and a
// rigid spin moves vₗ not at all), all of them time jets. Along a rotation
//   δx_gp = r·((yu − ya) A + yv B),  A = (ω_y d_z − ω_z d_y, −d_x ω_z, d_x ω_y),
//   B = (−ω_y v_y − ω_z v_z, ω_x v_y + δv_z, ω_x v_z − δv_y),  d = uₗ + (L/2, 0, 0), v = vₗ,
// along translations δx_gp = r diag(ya, yu, yu) rᵀ δd + δc. The time derivatives of r·(…) in the
// body frame come from Ω = ṙ's spin and r₀ᵀr̈.
//
// These are exact calculus. Muscade's power rule (src/Adiff.jl:230) takes the second time
// derivative of the square in Rodrigues as 2ss̈: r̈ and vₗ's second derivative differ from
// calculus by −r Γ and by −(Γᵀvₗ + ½F), with Γ, F (RuleRec below) functions of v_n, v̇_n alone; what
// their derivatives share is in the record too (a direction takes 500 operations for them; carried on
// first-order jets they took 3,500).
#pragma once
#include "beam_dyn.hpp"

namespace mh {

// Time jets of vectors, level by level.
template <int ND> struct TV { v3 v[ND]; };
template <int ND> MH_HD TV<ND> tcross(const TV<ND>& a, const TV<ND>& b) {
    TV<ND> r;
    r.v[0] = cross(a.v[0], b.v[0]);
    if constexpr (ND > 1) r.v[1] = cross(a.v[1], b.v[0]) + cross(a.v[0], b.v[1]);
    if constexpr (ND > 2) r.v[2] = cross(a.v[2], b.v[0]) + 2. * cross(a.v[1], b.v[1]) + cross(a.v[0], b.v[2]);
    return r;
}
template <int ND> MH_HD TV<ND> tscale(const double* k, const TV<ND>& a) {   // scalar jet k
    TV<ND> r;
    r.v[0] = k[0] * a.v[0];
    if constexpr (ND > 1) r.v[1] = k[1] * a.v[0] + k[0] * a.v[1];
    if constexpr (ND > 2) r.v[2] = k[2] * a.v[0] + (2. * k[1]) * a.v[1] + k[0] * a.v[2];
    return r;
}
template <int ND> MH_HD TV<ND> tadd(const TV<ND>& a, double s, const TV<ND>& b) {
    TV<ND> r;
#pragma unroll
    for (int n = 0; n < ND; ++n) r.v[n] = a.v[n] + s * b.v[n];
    return r;
}
// f(t(time)) on the levels of t = v·v, from f, f′, f″.
template <int ND> MH_HD void tcompose(double f0, double f1, double f2, const double* t, double* o) {
    o[0] = f0;
    if constexpr (ND > 1) o[1] = f1 * t[1];
    if constexpr (ND > 2) o[2] = f2 * t[1] * t[1] + f1 * t[2];
}
template <int ND> MH_HD void tnorm2(const TV<ND>& v, double* t) {
    t[0] = dot(v.v[0], v.v[0]);
    if constexpr (ND > 1) t[1] = 2. * dot(v.v[0], v.v[1]);
    if constexpr (ND > 2) t[2] = 2. * (dot(v.v[1], v.v[1]) + dot(v.v[0], v.v[2]));
}

// ------------------------------------------------ the power rule's part (third level only)
// q = (d/dt sinc1(|v|/2))² of a rotation vector v, what the square's power rule leaves out of b″, times
// C = cos|v| and g = |v|sin|v|, and their derivatives: δ(qC) = c1 v·δv + c2 δ(v·v̇), likewise g1, g2.
struct LostSquare { double c, g, c1, c2, g1, g2; };
MH_HD LostSquare lost_square(v3 v, v3 vd, const RotFun& f) {   // f at |v|²
    const double t = dot(v, v), s = dot(v, vd), C = 1. - f.b * t, g = t * f.a;
    double f0, f1;   // derivatives of sinc1(|v|/2) in t; b is half its square
    if (t < 1.) {
        const double i = 1. / sqrt(2. * f.b);
        f0 = f.b1 * i;
        f1 = (f.b2 - f0 * f0) * i;
    } else {
        const RotFun h = rot_fun(0.25 * t);
        f0 = 0.25 * h.a1;
        f1 = 0.0625 * h.a2;
    }
    const double sd = (2. * f0) * s, q = sd * sd, qt = (4. * f1) * (sd * s), qs = (4. * f0) * sd;
    LostSquare o;
    o.c = q * C; o.c1 = 2. * (qt * C) - q * f.a; o.c2 = qs * C;
    o.g = q * g; o.g1 = 2. * (qt * g) + q * (f.a + C); o.g2 = qs * g;
    return o;
}
// A rotation vector v below norm3's 1e-14 (Rotations.jl:106-112) has its length's derivatives reset: the
// coefficient sinc1(θ) then keeps no second derivative, and Rodrigues″ differs from calculus by
// −spin z with z = 0, δz = −⅓(|v̇|² δv + 2(δv·v̇) v̇).
MH_HD v3 lost_length(v3 v, v3 d, v3 e) {
    return dot(v, v) < 1e-28 ? (-1. / 3.) * (dot(d, d) * e + (2. * dot(e, d)) * d) : mk(0., 0., 0.);
}
// Γ and F of the header, with a_n = rₘᵀv_n (node rotations in the reference axes) and v = vₗ:
//   Γ = spin g + q₁C₁ a₁a₁ᵀ + q_hC_h vvᵀ − (q₁C₁|a₁|² + q_hC_h|v|²) I
//   g = q₁g₁ a₁ + q_hg_h v + z₁ + z_h + ½T(v)F
//   F = A x − B z + k v,  k = k₁σ + k₂ v·x + k₃ v·z
//   x = q₂g₂ a₂ + z₂ − q₁g₁ a₁ − z₁,  z = Σ q_nC_n (a_n·v) a_n,  σ = Σ q_nC_n |a_n|²
// (z_i the lost lengths). With H = Rodrigues(v), M = H² and X = Σ q_n (C_n(a_na_nᵀ − |a_n|²I) ± g_n spin a_n)
// the power rule takes H X H off M's second derivative and F = (Hᵀax(MX) − sc′ tr(MX) v)/sc; ax(MX) =
// C H x − S H z + (…)v gives the form above: S = sin|v|/|v|, C = cos|v|, A = 1/S, B = 1/C, s = −2a′/a at
// |φ|² = 4|v|² (a = sinc), k₁ = 2sC/S − 1, k₂ = 4s − b(1+2C)/(SC), k₃ = (b − 2sS)/C.
struct RuleRec {
    m3 gam;              // Γ
    v3 F;
    m3 rm;               // reference axes: a_n = rₘᵀv_n
    LostSquare sq[3];    // of a₁, a₂, v
    double A, B, k1, k2, k3, k, b, c;   // b, c of T(v)
    v3 y, x, u;          // ∂F/∂|v|², x, ∂(½T(v)F)/∂|v|² at fixed F
};
MH_HD void rule_record(const m3& rm, const v3* a, const v3* ad, const RotFun* fn, const RotFun& f, v3 v, v3 vd, RuleRec& o) {
    const double th = dot(v, v);
#pragma unroll
    for (int n = 0; n < 2; ++n) o.sq[n] = lost_square(a[n], ad[n], fn[n]);
    o.rm = rm;
    o.sq[2] = lost_square(v, vd, f);
    // p = a(4|v|²) = SC and its derivatives in |v|²
    const double S = f.a, S1 = f.a1, C = 1. - f.b * th, C1 = -0.5 * S, ip = 1. / (S * C);
    const double pd = S1 * C + S * C1, pdd = f.a2 * C + 2. * S1 * C1 - 0.5 * S * S1;
    const double s = -0.5 * pd * ip, s1 = -0.5 * (pdd - pd * pd * ip) * ip;
    o.A = 1. / S; o.B = 1. / C; o.b = f.b; o.c = f.c;
    const double A1 = -S1 * o.A * o.A, B1 = -C1 * o.B * o.B;
    o.k1 = 2. * s * C * o.A - 1.;
    const double d1 = 2. * (s1 * C * o.A + s * (C1 * o.A + C * A1));
    const double e = f.b * (1. + 2. * C), e1 = f.b1 * (1. + 2. * C) + 2. * f.b * C1;
    o.k2 = 4. * s - e * o.A * o.B;
    const double d2 = 4. * s1 - (e1 * o.A * o.B + e * (A1 * o.B + o.A * B1));
    o.k3 = (f.b - 2. * s * S) * o.B;
    const double d3 = (f.b1 - 2. * (s1 * S + s * S1)) * o.B + (f.b - 2. * s * S) * B1;
    const double b0 = o.sq[0].c * dot(a[0], v), b1 = o.sq[1].c * dot(a[1], v), r1 = o.sq[0].c * dot(a[0], a[0]);
    const double sig = r1 + o.sq[1].c * dot(a[1], a[1]);
    const v3 z = b0 * a[0] + b1 * a[1], n1 = o.sq[0].g * a[0];
    o.x = o.sq[1].g * a[1] - n1;
    const double vx = dot(v, o.x), vz = dot(v, z);
    o.k = o.k1 * sig + o.k2 * vx + o.k3 * vz;
    o.F = o.A * o.x - o.B * z + o.k * v;
    o.y = A1 * o.x - B1 * z + (d1 * sig + d2 * vx + d3 * vz) * v;
    const v3 vF = cross(v, o.F), vvF = cross(v, vF);
    o.u = (0.5 * f.b1) * vF + (0.5 * f.c1) * vvF;
    const v3 g = n1 + o.sq[2].g * v + 0.5 * (o.F + f.b * vF + f.c * vvF);
    const double q1 = o.sq[0].c, qh = o.sq[2].c, rho = r1 + qh * th;
    const v3 p1 = q1 * a[0], ph = qh * v;
    const double xy = p1.x * a[0].y + ph.x * v.y, xz = p1.x * a[0].z + ph.x * v.z, yz = p1.y * a[0].z + ph.y * v.z;
    o.gam.a[0] = p1.x * a[0].x + ph.x * v.x - rho;
    o.gam.a[4] = p1.y * a[0].y + ph.y * v.y - rho;
    o.gam.a[8] = p1.z * a[0].z + ph.z * v.z - rho;
    o.gam.a[1] = xy + g.z; o.gam.a[3] = xy - g.z;
    o.gam.a[2] = xz - g.y; o.gam.a[6] = xz + g.y;
    o.gam.a[5] = yz + g.x; o.gam.a[7] = yz - g.x;
}
// The nodes' part of δΓ, δF: δz, δ(v·z), δσ and its share of node 1, δ(q₁g₁a₁ + z₁), δx, and a₁ and
// ½δ(q₁C₁)a₁ + q₁C₁δa₁ of the symmetric part.
struct NodesDelta { v3 z, n1, x, a, p; double vz, sig, r1; };
// Node n (0, then 1) along δa, δȧ (moves) and δv.
MH_HD void node_delta(const RuleRec& R, int n, bool moves, v3 v, v3 dv, v3 a, v3 ad, v3 da, v3 dad, NodesDelta& o) {
    const LostSquare& q = R.sq[n];
    double dc = 0., dg = 0., r = 0., ds = dot(a, dv);
    const double s = dot(a, v), qc = q.c;
    v3 g = mk(0., 0., 0.);
    if (moves) {
        const double aa = dot(a, da), as = dot(da, ad) + dot(a, dad);
        dc = q.c1 * aa + q.c2 * as;
        dg = q.g1 * aa + q.g2 * as;
        ds = ds + dot(da, v);
        r = dc * dot(a, a) + (2. * qc) * aa;
        g = dg * a + q.g * da + lost_length(a, ad, da);
    } else {
        da = g;
    }
    const double b = qc * s, db = dc * s + qc * ds;
    const v3 z = db * a + b * da;
    const double vz = db * s + b * ds;
    if (n == 0) {
        o.z = z; o.vz = vz; o.sig = o.r1 = r; o.n1 = g;
        o.a = a; o.p = (0.5 * dc) * a + qc * da;
    } else {
        o.z = o.z + z; o.vz = o.vz + vz; o.sig = o.sig + r; o.x = g - o.n1;
    }
}
// δΓ, and dF2 = ½δF, along the nodes' part and δv, δv̇ of vₗ.
MH_HD void rule_delta(const RuleRec& R, v3 v, v3 vd, const NodesDelta& o, v3 dv, v3 dvd, m3& dG, v3& dF2) {
    const double dth = 2. * dot(v, dv);
    const double dk = R.k1 * o.sig + R.k2 * (dot(dv, R.x) + dot(v, o.x)) + R.k3 * o.vz;
    const v3 dF = R.A * o.x - R.B * o.z + dth * R.y + dk * v + R.k * dv;
    const v3 vF = cross(v, R.F), w = cross(dv, R.F) + cross(v, dF);
    const LostSquare& h = R.sq[2];
    const double dd = dot(dv, vd) + dot(v, dvd), hc = (0.5 * h.c1) * dth + h.c2 * dd, hg = (0.5 * h.g1) * dth + h.g2 * dd;
    dF2 = 0.5 * dF;
    const v3 g = o.n1 + hg * v + h.g * dv + lost_length(v, vd, dv) + dth * R.u +
                 (dF2 + (0.5 * R.b) * w + (0.5 * R.c) * (cross(dv, vF) + cross(v, w)));
    const double rho = o.r1 + hc * dot(v, v) + h.c * dth;
    const v3 a = o.a, p = o.p, r = (0.5 * hc) * v + h.c * dv;
    const double xy = (a.x * p.y + p.x * a.y) + (v.x * r.y + r.x * v.y), xz = (a.x * p.z + p.x * a.z) + (v.x * r.z + r.x * v.z),
                 yz = (a.y * p.z + p.y * a.z) + (v.y * r.z + r.y * v.z);
    dG.a[0] = 2. * (a.x * p.x + v.x * r.x) - rho;
    dG.a[4] = 2. * (a.y * p.y + v.y * r.y) - rho;
    dG.a[8] = 2. * (a.z * p.z + v.z * r.z) - rho;
    dG.a[1] = xy + g.z; dG.a[3] = xy - g.z;
    dG.a[2] = xz - g.y; dG.a[6] = xz + g.y;
    dG.a[5] = yz + g.x; dG.a[7] = yz - g.x;
}

// ------------------------------------------------ the element's record
// What every direction of an element reads, written once per element by the value pass. All
// members are doubles: the record is also an array of kDynRec<ND> numbers in this order.
template <int ND> struct DynBase {
    double r0[9];          // rₛₘ
    v3 om, omd;            // Ω, Ω̇ (body)
    v3 d[ND], vl[ND];      // uₗ + (L/2,0,0), vₗ on time levels (exact calculus)
    double bc[2][2 * ND];  // per node: b and c of T(v_n) on time levels
    double tau[ND], kap[ND];
    double l1[4][3], l2[4][3];   // per Gauss point: r₀ᵀẋ, r₀ᵀẍ
    double m1;             // roll couple: mₑ = m₁ r₀ e₁
    v3 psi; double epsi;   // Rodrigues⁻¹(rₛₘ) and e of its T⁻¹: vₛₘ,ε·D = ω·(T(ψ)⁻ᵀD) for body D
    double L;
};
template <int ND> struct DynRec : DynBase<ND> {};
template <> struct DynRec<3> : DynBase<3> { RuleRec rule; };
template <int ND> constexpr int kRecBase = 45 + 12 * ND;
template <int ND> constexpr int kDynRec = kRecBase<ND> + (ND > 2 ? 56 : 0);
static_assert(sizeof(DynRec<2>) == sizeof(double) * kDynRec<2> && sizeof(DynRec<3>) == sizeof(double) * kDynRec<3> &&
              sizeof(DynRec<1>) == sizeof(double) * kDynRec<1>, "the record is an array of doubles");
template <int ND> MH_HD TV<ND> tlevels(const v3* a) {
    TV<ND> r;
#pragma unroll
    for (int n = 0; n < ND; ++n) r.v[n] = a[n];
    return r;
}
MH_HD m3 m3_of(const double* a) {
    m3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.a[i] = a[i];
    return r;
}
// r₀ᵀr̈ = spin(Ω̇) + spin(Ω)² − Γ.
MH_HD m3 dyn_q2(v3 w, v3 wd) {
    m3 Q;
    const double xy = w.x * w.y, xz = w.x * w.z, yz = w.y * w.z;
    Q.a[0] = -(w.y * w.y + w.z * w.z); Q.a[4] = -(w.x * w.x + w.z * w.z); Q.a[8] = -(w.x * w.x + w.y * w.y);
    Q.a[1] = xy + wd.z; Q.a[3] = xy - wd.z;
    Q.a[2] = xz - wd.y; Q.a[6] = xz + wd.y;
    Q.a[5] = yz + wd.x; Q.a[7] = yz - wd.x;
    return Q;
}
MH_HD m3 dyn_q2(v3 w, v3 wd, const m3& gam) {
    m3 Q = dyn_q2(w, wd);
#pragma unroll
    for (int i = 0; i < 9; ++i) Q.a[i] -= gam.a[i];
    return Q;
}
// The Gauss points (z in units of L, weight in units of L) and the shape factors ya, yu, yv of
// x_gp = r (L z e₁ + (ya uₗₓ, yu u_y + yv v_z, yu u_z − yv v_y)) + cₛₘ (BeamElement.jl:74-79,142-146).
struct GpShape { double w, z, ya, yu, yv; };
MH_HD GpShape gp_shape(int g, double L) {
    GpShape s;
    const double z = (g == 0 || g == 3) ? 0.43056815579702629 : 0.16999052179242813;
    s.w = ((g == 0 || g == 3) ? 0.17392742256872693 : 0.32607257743127307) * L;
    s.z = g < 2 ? -z : z;
    s.ya = 2. * s.z;
    s.yu = -4. * (s.z * s.z * s.z) + 3. * s.z;
    s.yv = (s.z * s.z - 0.25) * L;
    return s;
}

// The record of an element, number q handed to put(q, value), and the loads that the closed form of
// the static part takes (beam_tangent<true>), from its frame. X: ND rows of the 12 dofs. The spin Ω and
// vₗ's time derivatives are those of the header along the nodes' velocities, and their derivatives.
template <int ND, class Put>
MH_HD void dyn_record(const BeamGeo& G, const BeamDynSection& S, const double (*X)[12], const double* U,
                      const BeamFrame& f, Put put, BeamLoads& ld) {
    int q = 0;
    auto put3 = [&](v3 a) { put(q, a.x); put(q + 1, a.y); put(q + 2, a.z); q += 3; };
    const double L = G.L;
    const v3 c0 = col(f.r, 0), c1 = col(f.r, 1), c2 = col(f.r, 2), zero = mk(0., 0., 0.);
    put3(c0); put3(c1); put3(c2);
    auto body = [&](v3 a) { return mk(dot(c0, a), dot(c1, a), dot(c2, a)); };
    TV<ND> vn[2];
    double tn[2][3], th[3];
    const RotFun fn[2] = {f.f1, f.f2};
#pragma unroll
    for (int n = 0; n < ND; ++n) { vn[0].v[n] = mk(X[n][3], X[n][4], X[n][5]); vn[1].v[n] = mk(X[n][9], X[n][10], X[n][11]); }
    tnorm2(vn[0], tn[0]);
    tnorm2(vn[1], tn[1]);
    const HalfFun hf = half_fun(f.fh);
    v3 om = zero, omd = zero;
    TV<ND> vl;
    vl.v[0] = f.vl;
    if constexpr (ND > 1) {
        v3 t[2], td[2];   // rᵀT(v_n)v̇_n and rᵀ times its derivative
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const v3 v = vn[i].v[0], w = vn[i].v[1], y = cross(v, w), z = cross(v, y);
            t[i] = body(w + fn[i].b * y + fn[i].c * z);
            if constexpr (ND > 2) {
                const v3 a = vn[i].v[2], yd = cross(v, a), zd = cross(w, y) + cross(v, yd);
                td[i] = body(a + (fn[i].b1 * tn[i][1]) * y + fn[i].b * yd + (fn[i].c1 * tn[i][1]) * z + fn[i].c * zd);
            }
        }
        const v3 dl = t[1] - t[0], y = cross(f.vl, dl), z = cross(f.vl, y);
        om = 0.5 * (t[0] + t[1]) - hf.k * y;
        vl.v[1] = 0.5 * dl + (4. * hf.q) * z;
        if constexpr (ND > 2) {
            const v3 t1 = td[0] - cross(om, t[0]), t2 = td[1] - cross(om, t[1]), dd = t2 - t1;
            const v3 yd = cross(vl.v[1], dl) + cross(f.vl, dd), zd = cross(vl.v[1], y) + cross(f.vl, yd);
            const double s = 8. * dot(f.vl, vl.v[1]);
            omd = 0.5 * (t1 + t2) - (hf.k1 * s) * y - hf.k * yd;
            vl.v[2] = 0.5 * dd + 4. * ((hf.q1 * s) * z + hf.q * zd);
        }
    }
    put3(om); put3(omd);
    // d in body components: (rᵀa)′ = rᵀa′ − Ω×(rᵀa), …
    TV<ND> d;
    v3 cs[ND];
    d.v[0] = f.d;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        const v3 u1 = mk(X[n][0], X[n][1], X[n][2]), u2 = mk(X[n][6], X[n][7], X[n][8]);
        cs[n] = 0.5 * (u1 + u2);
        if (n == 1) d.v[n] = body(u2 - cs[n]) - cross(om, d.v[0]);
        if (n == 2) {
            const v3 a1 = d.v[n - 1] + cross(om, d.v[0]);
            d.v[n] = body(u2 - cs[n]) - cross(omd, d.v[0]) - cross(om, d.v[n - 1]) - cross(om, a1);
        }
    }
#pragma unroll
    for (int n = 0; n < ND; ++n) put3(d.v[n]);
#pragma unroll
    for (int n = 0; n < ND; ++n) put3(vl.v[n]);
    double k[ND];
    auto putn = [&]() {
#pragma unroll
        for (int n = 0; n < ND; ++n) put(q + n, k[n]);
        q += ND;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        tcompose<ND>(fn[i].b, fn[i].b1, fn[i].b2, tn[i], k); putn();
        tcompose<ND>(fn[i].c, fn[i].c1, fn[i].c2, tn[i], k); putn();
    }
    tnorm2(vl, th);
#pragma unroll
    for (int n = 0; n < ND; ++n) th[n] *= 4.;
    tcompose<ND>(hf.k, hf.k1, hf.k2, th, k); putn();
    tcompose<ND>(hf.q, hf.q1, hf.q2, th, k); putn();
    // the power rule
    v3 ddl = mk(0., 0., 0.), dvl = ddl;   // what it takes off d″, vₗ″
    m3 Q2;
    double gx = 0.;
    if constexpr (ND > 2) {
        auto ref = [&](v3 a) { return mulT(G.rm, a); };
        const v3 a[2] = {ref(vn[0].v[0]), ref(vn[1].v[0])}, ad[2] = {ref(vn[0].v[1]), ref(vn[1].v[1])};
        RuleRec ru;
        rule_record(G.rm, a, ad, fn, f.fh, vl.v[0], vl.v[1], ru);
        const double* p = reinterpret_cast<const double*>(&ru);
#pragma unroll
        for (int i = 0; i < 56; ++i) put(kRecBase<ND> + i, p[i]);
        Q2 = dyn_q2(om, omd, ru.gam);
        ddl = mulT(ru.gam, d.v[0]);
        dvl = mulT(ru.gam, vl.v[0]) + 0.5 * ru.F;
        gx = 0.5 * (ru.gam.a[5] - ru.gam.a[7]);
    }
    // loads at the Gauss points, body frame
    ld.e0 = ld.ea = ld.eu = ld.ev = mk(0., 0., 0.);
#pragma unroll
    for (int gp = 0; gp < 4; ++gp) {
        const GpShape h = gp_shape(gp, L);
        auto shape = [&](v3 dd, v3 vv) { return mk(h.ya * dd.x, h.yu * dd.y + h.yv * vv.z, h.yu * dd.z - h.yv * vv.y); };
        const v3 p0 = shape(d.v[0], vl.v[0]);
        v3 xd = mk(0., 0., 0.), xdd = xd;
        if constexpr (ND > 1) {
            const v3 p1 = shape(d.v[1], vl.v[1]);
            xd = p1 + cross(om, p0) + body(cs[1]);
            if constexpr (ND > 2)
                xdd = shape(d.v[2] - ddl, vl.v[2] - dvl) + 2. * cross(om, p1) + mul(Q2, p0) + body(cs[2]);
        }
        put(q + 3 * gp, xd.x); put(q + 3 * gp + 1, xd.y); put(q + 3 * gp + 2, xd.z);
        put(q + 12 + 3 * gp, xdd.x); put(q + 13 + 3 * gp, xdd.y); put(q + 14 + 3 * gp, xdd.z);
        auto bl = [&](int j, double x1, double x2) { return S.mu * x2 + (S.Ca[j] * x2 + S.Cl[j] * x1 + S.Cq[j] * (x1 * fabs(x1))); };
        const double f0 = bl(0, xd.x, xdd.x), f1 = bl(1, xd.y, xdd.y), f2 = bl(2, xd.z, xdd.z);
        const v3 e = h.w * (f0 * c0 + f1 * c1 + f2 * c2 + mk(-U[0], -U[1], S.w - U[2]));
        ld.e0 = ld.e0 + e; ld.ea = ld.ea + h.ya * e; ld.eu = ld.eu + h.yu * e; ld.ev = ld.ev + h.yv * e;
    }
    q += 24;
    const double m1 = ND > 2 ? S.iota1 * (omd.x - gx) : 0.;
    put(q++, m1);
    ld.m = (m1 * L) * c0;
    {
        const v3 psi = rotvec(f.r);
        put3(psi);
        put(q++, exp_coef(norm3(psi)).e);
    }
    put(q++, L);
}

// ------------------------------------------------ a direction
// Level-0 Jacobian data of a rotation direction (a row of the tangent's load part) and the load
// moments of a direction (a column): K_load(row, column) = A·(mu − ma) + B·mv + w·mw for a rotation
// row, r₀(½m0 ± ½(ma_x, mu_y, mu_z)) for the translation rows of node 2 / 1.
struct DirRow { v3 A, B, w; };
struct DirCol { v3 m0, ma, mu, mv, mw; };
// δx_gp⁽ⁿ⁾ = ya·a[n] + yu·u[n] + yv·v[n] + c[n], body components, n = 0..ND−1.
template <int ND> struct DirPath { v3 a[ND], u[ND], v[ND], c[ND]; };

// The load derivatives summed over the Gauss points. w0: the frame spin, dm1: δm₁.
template <int ND>
MH_HD void dir_moments(const BeamDynSection& S, const DynRec<ND>& R, const DirPath<ND>& p, v3 w0,
                       double dm1, DirCol& o) {
    o.m0 = o.ma = o.mu = o.mv = mk(0., 0., 0.);
    const v3 Ca = mk(S.Ca[0], S.Ca[1], S.Ca[2]), Cl = mk(S.Cl[0], S.Cl[1], S.Cl[2]), Cq = mk(S.Cq[0], S.Cq[1], S.Cq[2]);
    auto had = [](v3 a, v3 b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); };
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        MH_PHASE();
        const GpShape h = gp_shape(g, R.L);
        const double ya = h.ya, yu = h.yu, yv = h.yv;
        const v3 l1 = mk(R.l1[g][0], R.l1[g][1], R.l1[g][2]);
        const v3 s1 = had(Cq, mk(fabs(l1.x), fabs(l1.y), fabs(l1.z)));
        const v3 d1 = ND > 1 ? (ya * p.a[ND > 1 ? 1 : 0] + yu * p.u[ND > 1 ? 1 : 0]) +
                                   (yv * p.v[ND > 1 ? 1 : 0] + p.c[ND > 1 ? 1 : 0]) : mk(0., 0., 0.);
        v3 b = had(Cl + s1, l1);
        v3 f = had(Cl + 2. * s1, d1 - cross(w0, l1));   // the body load turns with the frame
        if constexpr (ND > 2) {
            const v3 l2 = mk(R.l2[g][0], R.l2[g][1], R.l2[g][2]);
            const v3 d2 = (ya * p.a[2] + yu * p.u[2]) + (yv * p.v[2] + p.c[2]);
            b = b + had(Ca, l2);
            f = f + had(Ca, d2 - cross(w0, l2)) + S.mu * d2;
        }
        f = h.w * (f + cross(w0, b));
        o.m0 = o.m0 + f;
        o.ma = o.ma + ya * f;
        o.mu = o.mu + yu * f;
        o.mv = o.mv + yv * f;
    }
    const v3 D = R.L * mk(dm1, w0.z * R.m1, -w0.y * R.m1);   // δ(m₁e₁) + ω×m₁e₁
    const v3 pD = cross(R.psi, D);
    o.mw = D + 0.5 * pD + R.epsi * cross(R.psi, pD);         // T(ψ)⁻ᵀ = I + ½S + eS²
}

// rᵀ T(v)δv of a node, v and δv on time levels (global), in body components.
template <int ND> MH_HD TV<ND> node_spin(const DynRec<ND>& R, const double* bc, const TV<ND>& v, const TV<ND>& dv) {
    const TV<ND> y = tcross(v, dv);
    const TV<ND> t = tadd(tadd(dv, 1., tscale(bc, y)), 1., tscale(bc + ND, tcross(v, y)));
    auto body = [&](v3 a) {
        return mk(R.r0[0] * a.x + R.r0[1] * a.y + R.r0[2] * a.z, R.r0[3] * a.x + R.r0[4] * a.y + R.r0[5] * a.z,
                  R.r0[6] * a.x + R.r0[7] * a.y + R.r0[8] * a.z);
    };
    TV<ND> o;
    o.v[0] = body(t.v[0]);
    if constexpr (ND > 1) {
        const v3 b1 = body(t.v[1]);
        o.v[1] = b1 - cross(R.om, o.v[0]);
        if constexpr (ND > 2) o.v[2] = body(t.v[2]) - cross(R.omd, o.v[0]) - cross(R.om, o.v[1]) - cross(R.om, b1);
    }
    return o;
}

// The power rule's part of a rotation direction: −r₀ c with c = Γp + Y(Γᵀd, Γᵀvₗ + ½F) on the shapes of p,
// its derivative along node spins s, Δ: c on the shapes ya, yu, yv, and ax(δΓ)ₓ. nodes: the nodes' part.
template <class Nodes>
MH_HD void rule_path(const DynRec<3>& R, const TV<3>& s, const TV<3>& dl, Nodes nodes, v3& ca, v3& cu, v3& cv, double& gx) {
    m3 dG;
    v3 dF2, w, dv;
    const v3 v = R.vl[0];
    {
        const v3 y = cross(v, dl.v[0]), z = cross(v, y);   // the first levels of rotation_path
        w = 0.5 * s.v[0] - R.tau[0] * y;
        dv = 0.5 * dl.v[0] + (4. * R.kap[0]) * z;
        const v3 dvd = 0.5 * dl.v[1] + 4. * (R.kap[1] * z + R.kap[0] * (cross(R.vl[1], y) +
                       cross(v, cross(R.vl[1], dl.v[0]) + cross(v, dl.v[1]))));
        NodesDelta o;
        nodes(v, dv, o);
        MH_PHASE();
        rule_delta(R.rule, v, R.vl[1], o, dv, dvd, dG, dF2);
    }
    MH_PHASE();
    const v3 d = R.d[0], dd = cross(d, w);
    const m3& G = R.rule.gam;
    gx = 0.5 * (dG.a[5] - dG.a[7]);
    auto col = [](const m3& m, int j) { return mk(m.a[3 * j], m.a[3 * j + 1], m.a[3 * j + 2]); };
    const v3 g = mulT(G, d), dg = mulT(dG, d) + mulT(G, dd);
    ca = cross(w, d.x * col(G, 0) + mk(g.x, 0., 0.)) + d.x * col(dG, 0) + dd.x * col(G, 0) + mk(dg.x, 0., 0.);
    cu = cross(w, d.y * col(G, 1) + d.z * col(G, 2) + mk(0., g.y, g.z)) + d.y * col(dG, 1) + dd.y * col(G, 1) +
         d.z * col(dG, 2) + dd.z * col(G, 2) + mk(0., dg.y, dg.z);
    const v3 f = mulT(G, v) + 0.5 * R.rule.F, df = mulT(dG, v) + mulT(G, dv) + dF2;
    cv = cross(w, v.z * col(G, 1) - v.y * col(G, 2) + mk(0., f.z, -f.y)) + v.z * col(dG, 1) + dv.z * col(G, 1) -
         v.y * col(dG, 2) - dv.y * col(G, 2) + mk(0., df.z, -df.y);
}
// Path of x_gp along the rotations with node spins sum s and difference Δ (body jets), the row data
// and δm₁. c: the power rule's part of δẍ on the shapes ya, yu, yv, gx: ax(δΓ)ₓ.
template <int ND>
MH_HD void rotation_path(const BeamDynSection& S, const DynRec<ND>& R, const TV<ND>& s, const TV<ND>& dl,
                         v3 ca, v3 cu, v3 cv, double gx, DirPath<ND>& p, DirRow& row, double& dm1) {
    const TV<ND> vl = tlevels<ND>(R.vl), y = tcross(vl, dl);   // φ×Δ = 2y
    TV<ND> w = tscale(R.tau, y), dv = tscale(R.kap, tcross(vl, y));
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        w.v[n] = 0.5 * s.v[n] - w.v[n];
        dv.v[n] = 0.5 * dl.v[n] + 4. * dv.v[n];
    }
    // m₁ = ι₁(Ω̇ₓ − ax(Γ)ₓ), δΩ̇ = ω̈ + Ω̇×ω + Ω×ω̇
    dm1 = 0.;
    if constexpr (ND > 2) dm1 = S.iota1 * ((w.v[2].x + cross(R.omd, w.v[0]).x + cross(R.om, w.v[1]).x) - gx);
    auto fA = [](v3 d, v3 o) { return mk(o.y * d.z - o.z * d.y, -d.x * o.z, d.x * o.y); };
    auto fB = [](v3 v, v3 o) { return mk(-(o.y * v.y + o.z * v.z), o.x * v.y, o.x * v.z); };
    auto rot = [](v3 v) { return mk(0., v.z, -v.y); };
    TV<ND> A, B;
    A.v[0] = fA(R.d[0], w.v[0]);
    B.v[0] = fB(R.vl[0], w.v[0]) + rot(dv.v[0]);
    p.u[0] = A.v[0]; p.v[0] = B.v[0];
    row.A = A.v[0]; row.B = B.v[0]; row.w = w.v[0];
    if constexpr (ND > 1) {
        A.v[1] = fA(R.d[1], w.v[0]) + fA(R.d[0], w.v[1]);
        B.v[1] = fB(R.vl[1], w.v[0]) + fB(R.vl[0], w.v[1]) + rot(dv.v[1]);
        p.u[1] = A.v[1] + cross(R.om, A.v[0]);
        p.v[1] = B.v[1] + cross(R.om, B.v[0]);
    }
    if constexpr (ND > 2) {
        A.v[2] = fA(R.d[2], w.v[0]) + 2. * fA(R.d[1], w.v[1]) + fA(R.d[0], w.v[2]);
        B.v[2] = fB(R.vl[2], w.v[0]) + 2. * fB(R.vl[1], w.v[1]) + fB(R.vl[0], w.v[2]) + rot(dv.v[2]);
        auto two = [&](v3 a0, v3 a1, v3 a2) {
            return a2 + cross(R.omd, a0) + cross(R.om, 2. * a1 + cross(R.om, a0));
        };
        p.u[2] = two(A.v[0], A.v[1], A.v[2]);
        p.v[2] = two(B.v[0], B.v[1], B.v[2]);
    }
#pragma unroll
    for (int n = 0; n < ND; ++n) { p.a[n] = mk(-p.u[n].x, -p.u[n].y, -p.u[n].z); p.c[n] = mk(0., 0., 0.); }
    if constexpr (ND > 2) { p.a[2] = p.a[2] - ca; p.u[2] = p.u[2] - cu; p.v[2] = p.v[2] - cv; }
}

// Path of x_gp along translations: δd = ½(δu₂ − δu₁), δc = ½(δu₁ + δu₂) on time levels (global).
template <int ND> MH_HD void translation_path(const DynRec<ND>& R, const TV<ND>& dd, const TV<ND>& dc, DirPath<ND>& p) {
    auto body = [&](v3 a) {
        return mk(R.r0[0] * a.x + R.r0[1] * a.y + R.r0[2] * a.z, R.r0[3] * a.x + R.r0[4] * a.y + R.r0[5] * a.z,
                  R.r0[6] * a.x + R.r0[7] * a.y + R.r0[8] * a.z);
    };
    auto ex = [](v3 q) { return mk(q.x, 0., 0.); };
    auto off = [](v3 q) { return mk(0., q.y, q.z); };
#pragma unroll
    for (int n = 0; n < ND; ++n) { p.c[n] = body(dc.v[n]); p.v[n] = mk(0., 0., 0.); }
    const v3 D0 = body(dd.v[0]);
    p.a[0] = ex(D0); p.u[0] = off(D0);
    if constexpr (ND > 1) {
        const v3 b1 = body(dd.v[1]), D1 = b1 - cross(R.om, D0);
        p.a[1] = ex(D1) + cross(R.om, ex(D0));
        p.u[1] = off(D1) + cross(R.om, off(D0));
        if constexpr (ND > 2) {
            const m3 Q = dyn_q2(R.om, R.omd, R.rule.gam);
            const v3 D2 = body(dd.v[2]) - 2. * cross(R.om, b1) + mulT(Q, D0);
            p.a[2] = ex(D2) + 2. * cross(R.om, ex(D1)) + mul(Q, ex(D0));
            p.u[2] = off(D2) + 2. * cross(R.om, off(D1)) + mul(Q, off(D0));
        }
    }
}

// The six translation rows' values of a column (unscaled): node 1 in t1, node 2 in t2.
template <int ND> MH_HD void translation_rows(const DynRec<ND>& R, const DirCol& c, v3& t1, v3& t2) {
    const m3 r = m3_of(R.r0);
    const v3 h = 0.5 * c.m0, y = mk(0.5 * c.ma.x, 0.5 * c.mu.y, 0.5 * c.mu.z);
    t1 = mul(r, h - y);
    t2 = mul(r, h + y);
}
MH_HD double rotation_row(const DirRow& r, const DirCol& c) {
    return (dot(r.A, c.mu - c.ma) + dot(r.B, c.mv)) + dot(r.w, c.mw);
}

// One rotation dof of node nd (0, 1), component k, with the seed σ on its time levels. V: ND rows of
// the six rotation dofs (node 1, node 2).
template <int ND>
MH_HD void rotation_direction(const BeamDynSection& S, const DynRec<ND>& R, const double (*V)[6], int nd, int k,
                              const double* sg, DirRow& row, DirCol& col) {
    TV<ND> v, dv;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        v.v[n] = nd ? mk(V[n][3], V[n][4], V[n][5]) : mk(V[n][0], V[n][1], V[n][2]);
        dv.v[n] = mk(k == 0 ? sg[n] : 0., k == 1 ? sg[n] : 0., k == 2 ? sg[n] : 0.);
    }
    double bc[2 * ND];
#pragma unroll
    for (int i = 0; i < 2 * ND; ++i) bc[i] = nd ? R.bc[1][i] : R.bc[0][i];
    const TV<ND> t = node_spin<ND>(R, bc, v, dv);
    TV<ND> dl;
#pragma unroll
    for (int n = 0; n < ND; ++n) dl.v[n] = (nd ? 1. : -1.) * t.v[n];
    v3 ca = mk(0., 0., 0.), cu = ca, cv = ca;
    double gx = 0.;
    if constexpr (ND > 2) {
        MH_PHASE();
        rule_path(R, t, dl, [&](v3 vl, v3 dvl, NodesDelta& o) {
            const m3& rm = R.rule.rm;
            const v3 ek = mk(rm.a[k], rm.a[3 + k], rm.a[6 + k]);   // rₘᵀeₖ
#pragma unroll
            for (int n = 0; n < 2; ++n)
                node_delta(R.rule, n, n == nd, vl, dvl, mulT(rm, mk(V[0][3 * n], V[0][3 * n + 1], V[0][3 * n + 2])),
                           mulT(rm, mk(V[1][3 * n], V[1][3 * n + 1], V[1][3 * n + 2])), sg[0] * ek, sg[1] * ek, o);
        }, ca, cu, cv, gx);
        MH_PHASE();
    }
    DirPath<ND> p;
    double dm1;
    rotation_path<ND>(S, R, t, dl, ca, cu, cv, gx, p, row, dm1);
    dir_moments<ND>(S, R, p, row.w, dm1, col);
}
// One translation dof of node nd, component k.
template <int ND>
MH_HD void translation_direction(const BeamDynSection& S, const DynRec<ND>& R, int nd, int k,
                                 const double* sg, DirCol& col) {
    TV<ND> dd, dc;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        const double h = 0.5 * sg[n];
        dc.v[n] = mk(k == 0 ? h : 0., k == 1 ? h : 0., k == 2 ? h : 0.);
        dd.v[n] = (nd ? 1. : -1.) * dc.v[n];
    }
    DirPath<ND> p;
    translation_path<ND>(R, dd, dc, p);
    dir_moments<ND>(S, R, p, mk(0., 0., 0.), 0., col);
}
// Every dof at once, seeds dX[n][dof] on the time levels (the δr direction of :step).
template <int ND>
MH_HD void full_direction(const BeamDynSection& S, const DynRec<ND>& R, const double (*V)[6],
                          const double (*dX)[12], DirRow& row, DirCol& col) {
    TV<ND> t[2];
#pragma unroll
    for (int nd = 0; nd < 2; ++nd) {
        TV<ND> v, dv;
#pragma unroll
        for (int n = 0; n < ND; ++n) {
            v.v[n] = mk(V[n][3 * nd], V[n][3 * nd + 1], V[n][3 * nd + 2]);
            dv.v[n] = mk(dX[n][6 * nd + 3], dX[n][6 * nd + 4], dX[n][6 * nd + 5]);
        }
        t[nd] = node_spin<ND>(R, R.bc[nd], v, dv);
    }
    const TV<ND> s = tadd(t[0], 1., t[1]), dl = tadd(t[1], -1., t[0]);
    v3 ca = mk(0., 0., 0.), cu = ca, cv = ca;
    double gx = 0.;
    if constexpr (ND > 2) {
        MH_PHASE();
        rule_path(R, s, dl, [&](v3 vl, v3 dvl, NodesDelta& o) {
            const m3& rm = R.rule.rm;
#pragma unroll
            for (int n = 0; n < 2; ++n)
                node_delta(R.rule, n, true, vl, dvl, mulT(rm, mk(V[0][3 * n], V[0][3 * n + 1], V[0][3 * n + 2])),
                           mulT(rm, mk(V[1][3 * n], V[1][3 * n + 1], V[1][3 * n + 2])),
                           mulT(rm, mk(dX[0][6 * n + 3], dX[0][6 * n + 4], dX[0][6 * n + 5])),
                           mulT(rm, mk(dX[1][6 * n + 3], dX[1][6 * n + 4], dX[1][6 * n + 5])), o);
        }, ca, cu, cv, gx);
        MH_PHASE();
    }
    {
        DirPath<ND> p;
        double dm1;
        rotation_path<ND>(S, R, s, dl, ca, cu, cv, gx, p, row, dm1);
        dir_moments<ND>(S, R, p, row.w, dm1, col);
    }
    MH_PHASE();
    TV<ND> dd, dc;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        const v3 u1 = mk(dX[n][0], dX[n][1], dX[n][2]), u2 = mk(dX[n][6], dX[n][7], dX[n][8]);
        dc.v[n] = 0.5 * (u1 + u2);
        dd.v[n] = 0.5 * (u2 - u1);
    }
    DirPath<ND> p;
    DirCol c;
    translation_path<ND>(R, dd, dc, p);
    dir_moments<ND>(S, R, p, mk(0., 0., 0.), 0., c);
    col.m0 = col.m0 + c.m0; col.ma = col.ma + c.ma; col.mu = col.mu + c.mu; col.mv = col.mv + c.mv; col.mw = col.mw + c.mw;
}

// ------------------------------------------------ the adjoint's contraction
// y = ∂x_gp/∂X₀·Λ and ∂vₛₘ/∂X₀·Λ, as a row of the load part (see DirRow): y_gp = (yu − ya) A + yv B +
// (ya, yu, yu)∘d + c in body components.
struct DirLam { DirRow r; v3 d, c; };
template <int ND>
MH_HD void lambda_row(const DynRec<ND>& R, const double (*V)[6], const double* lam, DirLam& o) {
    v3 t[2];
    const m3 r = m3_of(R.r0);
#pragma unroll
    for (int nd = 0; nd < 2; ++nd) {
        const v3 v = mk(V[0][3 * nd], V[0][3 * nd + 1], V[0][3 * nd + 2]);
        const v3 dv = mk(lam[6 * nd + 3], lam[6 * nd + 4], lam[6 * nd + 5]), y = cross(v, dv);
        t[nd] = mulT(r, dv + R.bc[nd][0] * y + R.bc[nd][ND] * cross(v, y));
    }
    const v3 dl = t[1] - t[0], d = R.d[0], vl = R.vl[0], y = cross(vl, dl);
    const v3 w = 0.5 * (t[0] + t[1]) - R.tau[0] * y, dv = 0.5 * dl + (4. * R.kap[0]) * cross(vl, y);
    o.r.A = mk(w.y * d.z - w.z * d.y, -d.x * w.z, d.x * w.y);
    o.r.B = mk(-(w.y * vl.y + w.z * vl.z), w.x * vl.y + dv.z, w.x * vl.z - dv.y);
    o.r.w = w;
    const v3 u1 = mk(lam[0], lam[1], lam[2]), u2 = mk(lam[6], lam[7], lam[8]);
    o.d = mulT(r, 0.5 * (u2 - u1));
    o.c = mulT(r, 0.5 * (u1 + u2));
}
MH_HD double lambda_contract(const DirLam& y, const DirCol& c) {
    return rotation_row(y.r, c) + ((y.d.x * c.ma.x + y.d.y * c.mu.y + y.d.z * c.mu.z) + dot(y.c, c.m0));
}
// Σ_gp dL·∂x_gp/∂X₀ along a rotation row's dof (or along Λ), global components.
template <int ND> MH_HD v3 row_load(const DynRec<ND>& R, const DirRow& w) {
    v3 s = mk(0., 0., 0.);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const GpShape h = gp_shape(g, R.L);
        s = s + h.w * ((h.yu - h.ya) * w.A + h.yv * w.B);
    }
    return mul(m3_of(R.r0), s);
}

}  // namespace mh
