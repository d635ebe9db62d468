// Quadrature of the elements that lie far from a collocation row (device code).
//
// The discretisation is the 6x6 collapsed Gauss-Legendre rule (mesh.cu:597-672):
// 36 kernel evaluations per (row, element) pair, exact for polynomials of
// degree 10 on the triangle.  Seen from a distance the integrand is smooth over
// the element, and a rule of lower degree gives the same sums: with rho the
// largest centroid-vertex distance, d the distance of the row from the centroid
// and kappa = k rho, the difference from the 36-point sums in FP64, relative to
// the sums of the magnitudes, over 1200 directions of the row and ten triangles
// (equilateral, thin, random, a 1 : 50 needle) is at most / root mean square
//      7 points (degree 5)   d >=  24 rho, kappa <= 0.22    3.3e-8 / 1.1e-8
//     12 points (degree 7)   d >=   8 rho, kappa <= 0.6     2.8e-8 / 5e-9
//     16 points (degree 8)   d >= 5.5 rho, kappa <= 0.6     1.8e-8 / 8e-9
// at those limits, falling as (rho / d)^(degree + 1) and kappa^(degree + 1)
// past them: half of one FP32 rounding (6e-8) at most, of the several that an
// entry takes.  The limits are where the error reaches that half.  The
// 36-point rule stays for closer pairs and for elements that the wavelength
// does not resolve (kappa = 0.6 is 6 elements per wavelength).
//
// The rules are the fully symmetric ones of degree 5 and 8 (Dunavant 1985, the
// 7- and 16-point rules) and the rotationally symmetric one of degree 7
// (Gatermann 1988), their points and weights found by solving the moment
// equations in FP64 (largest moment residual 1e-14).
//
// What bounds it: the vector ALU.  At 10242 nodes and 2 kHz the kernel issues
// 305 VALU instructions a pair (915 with 36 points for every pair), 0.195 per
// SIMD-cycle of the 0.25 that a SIMD of 16 lanes can, with 4 waves per SIMD.
// There it takes 2.08 ms (5.16 with 36 points everywhere), and for 40962 nodes
// at 12 kHz 36.4 ms alone, 38.5 to 40 within a solve (81).
#pragma once

#include <hip/hip_runtime.h>

namespace bem {

// A rule is a centroid weight wc (0: no such point), n3 orbits of three points
// with coordinates (b, a, a), (a, b, a), (a, a, b), b = 1 - 2 a, and ng points
// with general coordinates (g1, g2, 1 - g1 - g2); the weights sum to 1/2, as
// the collapsed rule's W do.
struct Far7 {
    static constexpr int n3 = 2, ng = 0;
    static constexpr double wc = 0.1125000000000008;
    static constexpr double a[] = {0.1012865073234565, 0.4701420641051153};
    static constexpr double wa[] = {0.06296959027241369, 0.06619707639425271};
    static constexpr double g1[1] = {0}, g2[1] = {0}, wg[1] = {0};
};
struct Far12 {
    static constexpr int n3 = 0, ng = 12;
    static constexpr double wc = 0;
    static constexpr double a[1] = {0}, wa[1] = {0};
    static constexpr double g1[] = {0.2064414986700104, 0.2777161669763746, 0.515842334353615,
        0.06751786707391888, 0.06238226509440399, 0.870099867831677, 0.05522545665691733, 0.6232720494910858,
        0.3215024938519968, 0.6609491961867425, 0.03432430294508175, 0.3047265008681757};
    static constexpr double g2[] = {0.2777161669763746, 0.515842334353615, 0.2064414986700104,
        0.06238226509440399, 0.870099867831677, 0.06751786707391888, 0.6232720494910858, 0.3215024938519968,
        0.05522545665691733, 0.03432430294508175, 0.3047265008681757, 0.6609491961867425};
    static constexpr double wg[] = {0.0674931870098144, 0.0674931870098144, 0.0674931870098144,
        0.02651702815743806, 0.02651702815743806, 0.02651702815743806, 0.04388140871444057,
        0.04388140871444057, 0.04388140871444057, 0.02877504278497367, 0.02877504278497367,
        0.02877504278497367};
};
struct Far16 {
    static constexpr int n3 = 3, ng = 6;
    static constexpr double wc = 0.07215780383890857;
    static constexpr double a[] = {0.05054722831703081, 0.4592925882927483, 0.1705693077517907};
    static constexpr double wa[] = {0.01622924881159761, 0.04754581713363121, 0.0516086852673578};
    static constexpr double g1[] = {0.2631128296345501, 0.008394777409992858, 0.2631128296345501,
        0.7284923929554571, 0.008394777409992858, 0.7284923929554571};
    static constexpr double g2[] = {0.008394777409992858, 0.2631128296345501, 0.7284923929554571,
        0.2631128296345501, 0.7284923929554571, 0.008394777409992858};
    static constexpr double wg[] = {0.01361515708722193, 0.01361515708722193, 0.01361515708722193,
        0.01361515708722193, 0.01361515708722193, 0.01361515708722193};
};

constexpr float kFar7D2 = 576.0f, kFar7K2 = 0.0484f;  // (d / rho)^2 from, kappa^2 up to
constexpr float kFar12D2 = 64.0f, kFar16D2 = 30.25f, kFarK2 = 0.36f;

// Element record of the far rules: the centroid in FP64, the vertices 1 and 2
// from it (times 2), the vertices' squared distances from it, and |y - c|^2 of
// the rules' general points.
struct alignas(64) FarRec {
    double c[3];
    float u1[3], u2[3];  // 2 (p1 - c), 2 (p2 - c)
    float uu[3];         // |p_j - c|^2
    float rho2;          // the largest of them
    float far7, far12, far16;  // squared distances from which the rules are used
    float n[3];          // unit normal
    float sJ;            // |e1 x e2| / (4 pi)
    int nodes[3];
    float beta[2], gamma[2];
    float d12[12], d16[6];
    int pad[2];
};
static_assert(sizeof(FarRec) == 256, "record size");

// The records are written by an earlier kernel and only read here, at an
// element index that is the same for the whole wave: read through the constant
// address space they are scalar loads into SGPRs.
typedef __attribute__((address_space(4))) const FarRec CFarRec;
typedef __attribute__((address_space(4))) const float CFloat;
typedef __attribute__((address_space(4))) const int CInt;

// The centroid from the row (point x), in FP64: the common phase k r0 is good
// to FP32 however many wavelengths the row is away.
struct FarDist {
    double x, y, z, r02;
    float r02f;
};
template <class C3>
__device__ __forceinline__ FarDist far_dist(const C3 &c, double xd, double yd, double zd) {
    FarDist d;
    d.x = c[0] - xd;
    d.y = c[1] - yd;
    d.z = c[2] - zd;
    d.r02 = fma(d.x, d.x, fma(d.y, d.y, d.z * d.z));
    d.r02f = (float)d.r02;
    return d;
}

// what the sums need of the pair (T_j = 2 (c - x).(p_j - c) / r0^2), and the
// phase and normal distance of its terms
struct FarGeom {
    float r02f, i0, i02, kr0, kr0rev, s0, c0, dn, T1, T2;
};
__device__ __forceinline__ FarGeom far_geom(CFarRec &fr, const FarDist &d, float k, float krev, double kf64) {
    FarGeom g;
    const float y = __builtin_amdgcn_rsqf(d.r02f);
    const double ra = d.r02 * (double)y;
    const double err = fma(-ra, ra, d.r02);  // r0^2 - ra^2
    const double r0 = fma(err, 0.5 * (double)y, ra);
    g.r02f = d.r02f;
    g.i0 = __builtin_fmaf(0.5f * y, (float)err * y * y, y);
    const float u0 = (float)__builtin_amdgcn_fract(r0 * kf64);
    g.s0 = __builtin_amdgcn_sinf(u0);
    g.c0 = __builtin_amdgcn_cosf(u0);
    const float r0f = (float)r0;
    g.kr0 = k * r0f;
    g.kr0rev = krev * r0f;
    const float ax = (float)d.x, ay = (float)d.y, az = (float)d.z;
    g.dn = fr.n[0] * ax + fr.n[1] * ay + fr.n[2] * az;
    g.i02 = g.i0 * g.i0;
    g.T1 = g.i02 * __builtin_fmaf(ax, fr.u1[0], __builtin_fmaf(ay, fr.u1[1], az * fr.u1[2]));
    g.T2 = g.i02 * __builtin_fmaf(ax, fr.u2[0], __builtin_fmaf(ay, fr.u2[1], az * fr.u2[2]));
    return g;
}
__device__ __forceinline__ FarGeom far_geom(CFarRec &fr, const float4 &x, float k, float krev, double kf64) {
    return far_geom(fr, far_dist(fr.c, (double)x.x, (double)x.y, (double)x.z), k, krev, kf64);
}

// Sums over a far element, relative to the centroid's distance r0: with
// i0 = 1 / r0, w = r0 / r and e^{-i phi}, phi = k (r - r0),
//   h_j = sum W N_j w^2 (w + i k r0) e^{-i phi},  g_j = sum W N_j w e^{-i phi},
//   c = sum W w^3
// (times i0^3 e^{-i k r0}, i0 e^{-i k r0} and i0^3 they are the sums of
// e^{-ikr} (1/r^3 + ik/r^2), e^{-ikr}/r and 1/r^3).
struct FarSums {
    float hr[3], hi[3], gr[3], gi[3], c;
};

// one point: t = (r / r0)^2 - 1, phi / (2 pi) = (k r0 / 2 pi) d, d = r / r0 - 1 =
// sqrt(1 + t) - 1.  d is first 1 + t times its reciprocal square root, less 1, which
// carries the rounding of both (6e-8 and a bias of about 8e-9, times k r0: at 40
// radians the phases were off by 4e-7, and the solution at 40962 nodes and 12 kHz
// by 7.7e-7 where 36 points a pair give 5.5e-7); one Newton step on
// (1 + d)^2 = 1 + t removes it (entries past 20 node spacings: 4.2e-7 -> 1.2e-7 of
// their size, 36 points 7.8e-7; the solution 4.8e-7) for 4 more instructions, 5 %
// of the assembly.  A division t / (1 + sqrt(1 + t)) took up to 8 %.
template <bool G>
__device__ __forceinline__ void far_point(float t, float kr0, float kr0rev, float &hr, float &hi, float &p, float &gr,
                                          float &gi) {
    const float op = t + 1.0f;
    const float w = __builtin_amdgcn_rsqf(op);
    float d = __builtin_fmaf(op, w, -1.0f);
    d = __builtin_fmaf(0.5f, __builtin_fmaf(-d, d, __builtin_fmaf(-2.0f, d, t)), d);
    const float u = kr0rev * d;
    const float sn = __builtin_amdgcn_sinf(u), cs = __builtin_amdgcn_cosf(u);
    const float w2 = w * w, q = w2 * kr0;
    p = w2 * w;
    hr = __builtin_fmaf(cs, p, sn * q);
    hi = __builtin_fmaf(cs, q, -sn * p);
    if (G) {
        gr = w * cs;
        gi = -w * sn;
    }
}

// IMP: g_1, g_2, g_3; SRC without IMP: their sum, in g[0].  T_j = 2 (c - x).(p_j - c) / r0^2.
template <class R, bool IMP, bool SRC>
__device__ __forceinline__ void far_sums(CFloat *uu, CFloat *dd, float T1, float T2, float i02, float kr0,
                                         float kr0rev, FarSums &s) {
    constexpr bool G = IMP || SRC;
    // the centroid: t = 0, w = 1, phi = 0
    const float h0i = (float)(R::wc / 3) * kr0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        s.hr[j] = (float)(R::wc / 3);
        s.hi[j] = h0i;
        s.gr[j] = IMP ? (float)(R::wc / 3) : 0.f;
        s.gi[j] = 0.f;
    }
    s.c = (float)R::wc;
    if (SRC && !IMP) s.gr[0] = (float)R::wc;
    if (R::n3 > 0) {
        // point j of an orbit is (b - a) (p_j - c) from the centroid; the sums
        // share the orbit's total: W [a (H1 + H2 + H3) + (b - a) H_j]
        const float D[3] = {uu[0] * i02, uu[1] * i02, uu[2] * i02};
        const float T[3] = {T1, T2, -T1 - T2};
        float tr = 0.f, ti = 0.f, tgr = 0.f, tgi = 0.f;
#pragma unroll
        for (int o = 0; o < R::n3; o++) {
            const double a = R::a[o], l = 1.0 - 3.0 * a, W = R::wa[o];
            float hr[3], hi[3], p[3], gr[3], gi[3];
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const float t = __builtin_fmaf((float)(l * l), D[j], (float)l * T[j]);
                far_point<G>(t, kr0, kr0rev, hr[j], hi[j], p[j], gr[j], gi[j]);
                s.hr[j] = __builtin_fmaf((float)(W * l), hr[j], s.hr[j]);
                s.hi[j] = __builtin_fmaf((float)(W * l), hi[j], s.hi[j]);
                if (IMP) {
                    s.gr[j] = __builtin_fmaf((float)(W * l), gr[j], s.gr[j]);
                    s.gi[j] = __builtin_fmaf((float)(W * l), gi[j], s.gi[j]);
                }
            }
            tr = __builtin_fmaf((float)(W * a), hr[0] + hr[1] + hr[2], tr);
            ti = __builtin_fmaf((float)(W * a), hi[0] + hi[1] + hi[2], ti);
            s.c = __builtin_fmaf((float)W, p[0] + p[1] + p[2], s.c);
            if (G) {
                const double wg = IMP ? W * a : W;
                tgr = __builtin_fmaf((float)wg, gr[0] + gr[1] + gr[2], tgr);
                tgi = __builtin_fmaf((float)wg, gi[0] + gi[1] + gi[2], tgi);
            }
        }
#pragma unroll
        for (int j = 0; j < 3; j++) {
            s.hr[j] += tr;
            s.hi[j] += ti;
            if (IMP || (SRC && j == 0)) {
                s.gr[j] += tgr;
                s.gi[j] += tgi;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < R::ng; q++) {
        const double N[3] = {R::g1[q], R::g2[q], 1.0 - R::g1[q] - R::g2[q]}, W = R::wg[q];
        const float t = __builtin_fmaf((float)(N[0] - N[2]), T1, __builtin_fmaf((float)(N[1] - N[2]), T2, dd[q] * i02));
        float hr, hi, p, gr, gi;
        far_point<G>(t, kr0, kr0rev, hr, hi, p, gr, gi);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            s.hr[j] = __builtin_fmaf((float)(W * N[j]), hr, s.hr[j]);
            s.hi[j] = __builtin_fmaf((float)(W * N[j]), hi, s.hi[j]);
            if (IMP) {
                s.gr[j] = __builtin_fmaf((float)(W * N[j]), gr, s.gr[j]);
                s.gi[j] = __builtin_fmaf((float)(W * N[j]), gi, s.gi[j]);
            }
        }
        s.c = __builtin_fmaf((float)W, p, s.c);
        if (SRC && !IMP) {
            s.gr[0] = __builtin_fmaf((float)W, gr, s.gr[0]);
            s.gi[0] = __builtin_fmaf((float)W, gi, s.gi[0]);
        }
    }
}

// The pair's terms from its sums: p_j = h_j - beta g_j with
// h_j = -dn sJ i0^3 e^{-i k r0} h_j', g_j = i rho omega sJ i0 e^{-i k r0} g_j',
// c = -dn sJ i0^3 c', and the boundary term gamma sum_j g_j.
template <bool IMP, bool SRC>
__device__ __forceinline__ void far_terms(CFarRec &fr, const FarGeom &g, const FarSums &s, float rw, float *pr,
                                          float *pi, float &cval, float &btr, float &bti) {
    const float m = -g.dn * fr.sJ * (g.i02 * g.i0);
    const float fx = m * g.c0, fy = -m * g.s0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        pr[j] = __builtin_fmaf(fx, s.hr[j], -fy * s.hi[j]);
        pi[j] = __builtin_fmaf(fx, s.hi[j], fy * s.hr[j]);
    }
    cval = m * s.c;
    if (IMP || SRC) {
        const float sg = rw * fr.sJ * g.i0;
        const float qx = sg * g.s0, qy = sg * g.c0;
        float gsr = 0, gsi = 0;
#pragma unroll
        for (int j = 0; j < (IMP ? 3 : 1); j++) {
            const float Gr = __builtin_fmaf(qx, s.gr[j], -qy * s.gi[j]);
            const float Gi = __builtin_fmaf(qx, s.gi[j], qy * s.gr[j]);
            if (IMP) {
                pr[j] -= fr.beta[0] * Gr - fr.beta[1] * Gi;
                pi[j] -= fr.beta[0] * Gi + fr.beta[1] * Gr;
            }
            gsr += Gr;
            gsi += Gi;
        }
        btr = fr.gamma[0] * gsr - fr.gamma[1] * gsi;
        bti = fr.gamma[0] * gsi + fr.gamma[1] * gsr;
    }
}

}  // namespace bem
