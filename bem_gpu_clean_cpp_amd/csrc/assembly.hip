// Collocation assembly on gfx950.
//
// The reference (atomicFuncs.cu:69-298) launches one thread per (collocation
// row, element) pair and scatters every result with float atomicAdd into A and
// B, so the summation order changes from run to run.  Here a wave owns a block
// of consecutive rows (one row per lane) and a column tile (a compact patch of
// nodes); it walks the tile's element list in a fixed order and accumulates
// straight into its own rows of A in HBM.  No other wave writes those entries,
// so there are no atomics and the result is bitwise repeatable.  Writes are
// coalesced: the 64 lanes of a wave write 64 consecutive rows of one column.
//
// Kernels:
//   prep_elems      one thread per element: p3, e1, e2, unit normal, J, ca/cb,
//                   cc/cb -- the element-uniform data the quadrature reads with
//                   scalar loads;
//   sing_elems      one thread per (element, vertex): the vertex-collapsed rule
//                   of the reference (mesh.cu:253-595) in FP64;
//   asm_tile        the regular 6x6 rule (mesh.cu:597-672) for every (row,
//                   element) pair of a tile, FP32 (or FP64), with the singular
//                   lanes taking the FP64 values; asm_tile_fast is its FP32
//                   form, with rules of 7, 12 or 16 points where every row of
//                   the wave is far enough from the element (far_rules.hpp);
//   asm_finalize    per row: 1 - sum c on the node diagonal
//                   (atomicFuncs.cu:227-235, 99-102), and the boundary-condition
//                   vector sum_e (cc/cb) sum_j g_j (atomicFuncs.cu:104-115);
//   rhs_fill        B[:, s] = incident_s - bterm.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "bem_internal.hpp"
#include "far_rules.hpp"
#include "xcd.hpp"

namespace bem {

// ------------------------------------------------------------ device math ---
// sin(2 pi t), cos(2 pi t) for t >= 0 in revolutions, FP32: the quadrant is
// removed exactly (u = t - j/4 with j = rint(4t) is exact in binary floating
// point), then near-minimax polynomials in u on [-1/8, 1/8] (coefficients fitted
// for this library; max abs error 9e-8 after FP32 rounding).
__device__ __forceinline__ void sincos_rev(float t, float &sn, float &cs) {
    const float j = __builtin_rintf(4.0f * t);
    const float u = __builtin_fmaf(j, -0.25f, t);
    const float u2 = u * u;
    float s = __builtin_fmaf(u2, -75.24006652832031f, 81.58812713623047f);
    s = __builtin_fmaf(u2, s, -41.34162902832031f);
    s = __builtin_fmaf(u2, s, 6.283185005187988f);
    s = u * s;
    float c = __builtin_fmaf(u2, 59.24602508544922f, -85.44374084472656f);
    c = __builtin_fmaf(u2, c, 64.93932342529297f);
    c = __builtin_fmaf(u2, c, -19.739208221435547f);
    c = __builtin_fmaf(u2, c, 1.0f);
    const int q = (int)j;
    const float ss = (q & 1) ? c : s;
    const float cc = (q & 1) ? s : c;
    sn = (q & 2) ? -ss : ss;
    cs = ((q + 1) & 2) ? -cc : cc;
}

__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq(double x) { return 1.0 / sqrt(x); }

// ------------------------------------------------------------- arguments ---
template <typename R>
struct QTab {
    R xi1[kNQ], xi2[kNQ], w[kNQ];
};

struct SingTab {
    double xi1[3][kNQ], xi2[3][kNQ], w[kNQ];
};

template <typename R>
struct AsmArgs {
    const float4 *__restrict__ pts;
    const ElemRec<R> *__restrict__ recs;
    const FarRec *__restrict__ far;  // FP32 fast kernel: the far rules' element records
    const R *__restrict__ sing;  // (e*3+v)*16: p[0..5], c[6], bterm[7..8]
    const int *__restrict__ tile_ptr;
    const int *__restrict__ tile_entries;
    const int *__restrict__ tile_slots;  // element-once plan: side column of each ghost vertex
    typename std::conditional<sizeof(R) == 4, float2, double2>::type *side;
    typename std::conditional<sizeof(R) == 4, float2, double2>::type *A;
    R *cpart;
    typename std::conditional<sizeof(R) == 4, float2, double2>::type *bpart;
    long ldA;
    long Mp;
    int M, N, nrbg, nwg;
    int r0;  // first row assembled (rows r0..M-1 land in A rows 0..M-r0-1)
    R k, kf, rw;  // k, k/(2 pi), rho*omega
    double kf64;  // k/(2 pi)
    int far_rho2, far7_rho2;  // (FP32 bits) rho^2 up to which the wavelength lets the far rules be used
    int impedance;  // any element with ca != 0
    QTab<R> q;
};

// (xcd_remap, xcd.hpp: consecutive logical ids, here the row blocks of one
// tile, which share the tile's element records, land on the same XCD)

// --------------------------------------------------------- element prep ---
// 6-point Gauss-Legendre nodes and weights on [-1, 1]
struct GL6 {
    static constexpr double eta[6] = {-0.9324695142031520278123016, -0.6612093864662645136613996,
                                      -0.2386191860831969086305017, 0.2386191860831969086305017,
                                      0.6612093864662645136613996,  0.9324695142031520278123016};
    static constexpr double w[6] = {0.1713244923791703450402961, 0.3607615730481386075698335,
                                    0.4679139345726910473898703, 0.4679139345726910473898703,
                                    0.3607615730481386075698335, 0.1713244923791703450402961};
};

template <typename R>
__global__ void prep_elems(const double *__restrict__ pts64, const int *__restrict__ elems,
                           const float2 *__restrict__ bc, int E, ElemRec<R> *__restrict__ out) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const int n0 = elems[3 * e], n1 = elems[3 * e + 1], n2 = elems[3 * e + 2];
    double p1[3], p2[3], p3[3], e1[3], e2[3];
    for (int d = 0; d < 3; d++) {
        p1[d] = pts64[3 * n0 + d];
        p2[d] = pts64[3 * n1 + d];
        p3[d] = pts64[3 * n2 + d];
        e1[d] = p1[d] - p3[d];
        e2[d] = p2[d] - p3[d];
    }
    // crossProd = (p1-p3) x (p2-p3), normal = crossProd / |crossProd| (mesh.cu:612-617)
    double cr[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    double J = sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    ElemRec<R> r;
    for (int d = 0; d < 3; d++) {
        r.p3[d] = (R)p3[d];
        r.e1[d] = (R)e1[d];
        r.e2[d] = (R)e2[d];
        r.n[d] = (R)(cr[d] / J);
    }
    r.J = (R)J;
    // bc = ca/cb and cc/cb (atomicFuncs.cu:87, 105), complex division
    const float2 ca = bc[3 * e], cb = bc[3 * e + 1], cc = bc[3 * e + 2];
    const double den = (double)cb.x * cb.x + (double)cb.y * cb.y;
    r.beta[0] = (R)(((double)ca.x * cb.x + (double)ca.y * cb.y) / den);
    r.beta[1] = (R)(((double)ca.y * cb.x - (double)ca.x * cb.y) / den);
    r.gamma[0] = (R)(((double)cc.x * cb.x + (double)cc.y * cb.y) / den);
    r.gamma[1] = (R)(((double)cc.y * cb.x - (double)cc.x * cb.y) / den);
    r.nodes[0] = n0;
    r.nodes[1] = n1;
    r.nodes[2] = n2;
    double f[3];
    for (int d = 0; d < 3; d++) {
        f[d] = e2[d] - e1[d];
        r.f[d] = (R)f[d];
    }
    for (int t = 0; t < 6; t++) {
        const double th = 0.5 + 0.5 * GL6::eta[t];
        double vv = 0;
        for (int d = 0; d < 3; d++) vv += (e1[d] + th * f[d]) * (e1[d] + th * f[d]);
        r.vv[t] = (R)vv;
    }
    for (int i = 0; i < (int)(sizeof(r.pad) / sizeof(int)); i++) r.pad[i] = 0;
    out[e] = r;
}

__global__ void prep_far(const double *__restrict__ pts64, const int *__restrict__ elems,
                         const ElemRec<double> *__restrict__ recs, int E, FarRec *__restrict__ out) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const ElemRec<double> &rec = recs[e];
    FarRec r;
    double u[3][3], uu[3] = {0, 0, 0};
    for (int d = 0; d < 3; d++) {
        double s = 0;
        for (int j = 0; j < 3; j++) s += pts64[3 * elems[3 * e + j] + d];
        r.c[d] = s / 3.0;
        for (int j = 0; j < 3; j++) {
            u[j][d] = pts64[3 * elems[3 * e + j] + d] - r.c[d];
            uu[j] += u[j][d] * u[j][d];
        }
        r.u1[d] = (float)(2.0 * u[0][d]);
        r.u2[d] = (float)(2.0 * u[1][d]);
        r.n[d] = (float)rec.n[d];
    }
    r.sJ = (float)(rec.J / (4.0 * kPi));
    for (int j = 0; j < 3; j++) r.uu[j] = (float)uu[j];
    const double rho2 = fmax(uu[0], fmax(uu[1], uu[2]));
    r.rho2 = (float)rho2;
    r.far7 = (float)(kFar7D2 * rho2);
    r.far12 = (float)(kFar12D2 * rho2);
    r.far16 = (float)(kFar16D2 * rho2);
    for (int j = 0; j < 3; j++) r.nodes[j] = rec.nodes[j];
    for (int j = 0; j < 2; j++) {
        r.beta[j] = (float)rec.beta[j];
        r.gamma[j] = (float)rec.gamma[j];
    }
    auto dist2 = [&](double n1, double n2) {
        double s = 0;
        for (int d = 0; d < 3; d++) {
            const double y = n1 * u[0][d] + n2 * u[1][d] + (1.0 - n1 - n2) * u[2][d];
            s += y * y;
        }
        return (float)s;
    };
#pragma unroll
    for (int q = 0; q < Far12::ng; q++) r.d12[q] = dist2(Far12::g1[q], Far12::g2[q]);
#pragma unroll
    for (int q = 0; q < Far16::ng; q++) r.d16[q] = dist2(Far16::g1[q], Far16::g2[q]);
    r.pad[0] = r.pad[1] = 0;
    out[e] = r;
}

// ------------------------------------------------------ singular, FP64 ---
// One thread per (element, vertex v): the reference's vertex rule for x = p_v,
// g_l_sgl{v+1}/h_l_sgl{v+1}/c_l_sgl{v+1} (mesh.cu:253-595), in FP64.  Stores
// the A contributions h_j - (ca/cb) g_j (j = 0..2), c, and (cc/cb) sum_j g_j.
template <typename Rout>
__global__ void sing_elems(const double *__restrict__ pts64, const int *__restrict__ elems,
                           const float2 *__restrict__ bc, int E, double k, double rw, SingTab tab,
                           Rout *__restrict__ out) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= 3 * E) return;
    const int e = id / 3, v = id % 3;
    double p[3][3];
    for (int j = 0; j < 3; j++)
        for (int d = 0; d < 3; d++) p[j][d] = pts64[3 * elems[3 * e + j] + d];
    double e1[3], e2[3];
    for (int d = 0; d < 3; d++) {
        e1[d] = p[0][d] - p[2][d];
        e2[d] = p[1][d] - p[2][d];
    }
    double cr[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    const double J = sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    const double nx = cr[0] / J, ny = cr[1] / J, nz = cr[2] / J;
    const double *x = p[v];
    const double inv4pi = 1.0 / (4.0 * kPi);
    double gr[3] = {0, 0, 0}, gi[3] = {0, 0, 0}, hr[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, c = 0;
    for (int q = 0; q < kNQ; q++) {
        const double xi1 = tab.xi1[v][q], xi2 = tab.xi2[v][q];
        const double N[3] = {xi1, xi2, 1.0 - xi1 - xi2};
        const double temp = tab.w[q] * J;  // 0.25 w_n w_m rho J
        double rv[3];
        for (int d = 0; d < 3; d++) rv[d] = N[0] * p[0][d] + N[1] * p[1][d] + N[2] * p[2][d] - x[d];
        const double r = sqrt(rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2]);
        const double prpn2 = (rv[0] * nx + rv[1] * ny + rv[2] * nz) / r;
        double sn, cs;
        sincos(k * r, &sn, &cs);
        const double Gr = cs * inv4pi / r, Gi = -sn * inv4pi / r;  // exp(-ikr)/(4 pi r)
        // dG/dn = G (-1/r - ik) dr/dn
        const double Hr = (Gr * (-1.0 / r) + Gi * k) * prpn2;
        const double Hi = (Gi * (-1.0 / r) - Gr * k) * prpn2;
        const double dG0 = -inv4pi / (r * r) * prpn2;
        for (int j = 0; j < 3; j++) {
            gr[j] += temp * N[j] * Gr;
            gi[j] += temp * N[j] * Gi;
            hr[j] += temp * N[j] * Hr;
            hi[j] += temp * N[j] * Hi;
        }
        c += temp * dG0;
    }
    // g_j *= i rho omega (mesh.cu:668-670)
    double Gjr[3], Gji[3];
    for (int j = 0; j < 3; j++) {
        Gjr[j] = -rw * gi[j];
        Gji[j] = rw * gr[j];
    }
    const float2 ca = bc[3 * e], cb = bc[3 * e + 1], cc = bc[3 * e + 2];
    const double den = (double)cb.x * cb.x + (double)cb.y * cb.y;
    const double br = ((double)ca.x * cb.x + (double)ca.y * cb.y) / den;
    const double bi = ((double)ca.y * cb.x - (double)ca.x * cb.y) / den;
    const double yr = ((double)cc.x * cb.x + (double)cc.y * cb.y) / den;
    const double yi = ((double)cc.y * cb.x - (double)cc.x * cb.y) / den;
    Rout *o = out + (size_t)id * 16;
    double sgr = 0, sgi = 0;
    for (int j = 0; j < 3; j++) {
        o[2 * j] = (Rout)(hr[j] - (br * Gjr[j] - bi * Gji[j]));
        o[2 * j + 1] = (Rout)(hi[j] - (br * Gji[j] + bi * Gjr[j]));
        sgr += Gjr[j];
        sgi += Gji[j];
    }
    o[6] = (Rout)c;
    o[7] = (Rout)(yr * sgr - yi * sgi);
    o[8] = (Rout)(yr * sgi + yi * sgr);
    for (int i = 9; i < 16; i++) o[i] = 0;
}

// ------------------------------------------------- regular quadrature ---
template <typename R>
__device__ __forceinline__ void sincos_phase(R r, R k, R kf, R &sn, R &cs);
template <>
__device__ __forceinline__ void sincos_phase<float>(float r, float, float kf, float &sn, float &cs) {
    sincos_rev(r * kf, sn, cs);
}
template <>
__device__ __forceinline__ void sincos_phase<double>(double r, double k, double, double &sn, double &cs) {
    sincos(k * r, &sn, &cs);
}

template <typename R>
__device__ __forceinline__ R shfl_xor(R v, int m) {
    return __shfl_xor(v, m, 64);
}

// One wave = RPW = 64/QG consecutive rows; QG lanes share a row and split the
// 36 quadrature points (QG = 1: a lane does all of them).  A workgroup is 4
// waves on 4 consecutive row blocks of the same tile.
template <typename R, int QG, bool IMP>
__global__ __launch_bounds__(256) void asm_tile(AsmArgs<R> a) {
    using C2 = typename std::conditional<sizeof(R) == 4, float2, double2>::type;
    constexpr int RPW = 64 / QG;
    constexpr int NQL = kNQ / QG;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int L = xcd_remap(blockIdx.x, a.nwg);
    const int tile = L / a.nrbg;
    const int rbg = L - tile * a.nrbg;
    const int row = a.r0 + (rbg * 4 + wave) * RPW + lane / QG;
    const int qg = (QG == 1) ? 0 : (lane % QG);
    const bool active = row < a.M;
    const float4 xp = a.pts[active ? row : 0];
    const R x0 = xp.x, x1 = xp.y, x2 = xp.z;

    R txi1[NQL], txi2[NQL], tw[NQL];
#pragma unroll
    for (int i = 0; i < NQL; i++) {
        const int q = qg + QG * i;
        txi1[i] = a.q.xi1[q];
        txi2[i] = a.q.xi2[q];
        tw[i] = a.q.w[q];
    }
    const R k = a.k, kf = a.kf;
    const R inv4pi = (R)(1.0 / (4.0 * kPi));
    R c_acc = 0, br_acc = 0, bi_acc = 0;

    const int it0 = a.tile_ptr[tile], it1 = a.tile_ptr[tile + 1];
    for (int it = it0; it < it1; ++it) {
        const int ent = a.tile_entries[it];
        const int e = ent >> 8;
        const ElemRec<R> &rec = a.recs[e];
        const R ax = rec.p3[0] - x0, ay = rec.p3[1] - x1, az = rec.p3[2] - x2;
        const R e10 = rec.e1[0], e11 = rec.e1[1], e12 = rec.e1[2];
        const R e20 = rec.e2[0], e21 = rec.e2[1], e22 = rec.e2[2];
        // (y - x).n is constant over a flat element: n.(p3 - x)
        const R dn = rec.n[0] * ax + rec.n[1] * ay + rec.n[2] * az;
        R h1r = 0, h1i = 0, h2r = 0, h2i = 0, htr = 0, hti = 0, gr = 0, gi = 0, cc = 0;
        R g1r = 0, g1i = 0, g2r = 0, g2i = 0;
#pragma unroll
        for (int i = 0; i < NQL; i++) {
            const R dx = fma(txi1[i], e10, fma(txi2[i], e20, ax));
            const R dy = fma(txi1[i], e11, fma(txi2[i], e21, ay));
            const R dz = fma(txi1[i], e12, fma(txi2[i], e22, az));
            const R r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            const R rinv = rsq(r2);
            const R r = r2 * rinv;
            R sn, cs;
            sincos_phase<R>(r, k, kf, sn, cs);
            // 4 pi G = (cos kr - i sin kr) / r
            const R Gr = cs * rinv, Gi = -sn * rinv;
            const R w2 = tw[i] * rinv;
            // 4 pi r G (1/r + ik), weighted; dG/dn = -(dn/4pi) rinv G~ (rinv + ik)
            const R Hr = (fma(Gr, rinv, -k * Gi)) * w2;
            const R Hi = (fma(Gi, rinv, k * Gr)) * w2;
            htr += Hr;
            hti += Hi;
            h1r = fma(txi1[i], Hr, h1r);
            h1i = fma(txi1[i], Hi, h1i);
            h2r = fma(txi2[i], Hr, h2r);
            h2i = fma(txi2[i], Hi, h2i);
            const R wGr = tw[i] * Gr, wGi = tw[i] * Gi;
            gr += wGr;
            gi += wGi;
            if (IMP) {
                g1r = fma(txi1[i], wGr, g1r);
                g1i = fma(txi1[i], wGi, g1i);
                g2r = fma(txi2[i], wGr, g2r);
                g2i = fma(txi2[i], wGi, g2i);
            }
            cc = fma(w2 * rinv, rinv, cc);
        }
        if (QG > 1) {
#pragma unroll
            for (int m = 1; m < QG; m <<= 1) {
                h1r += shfl_xor(h1r, m); h1i += shfl_xor(h1i, m);
                h2r += shfl_xor(h2r, m); h2i += shfl_xor(h2i, m);
                htr += shfl_xor(htr, m); hti += shfl_xor(hti, m);
                gr += shfl_xor(gr, m); gi += shfl_xor(gi, m);
                cc += shfl_xor(cc, m);
                if (IMP) {
                    g1r += shfl_xor(g1r, m); g1i += shfl_xor(g1i, m);
                    g2r += shfl_xor(g2r, m); g2i += shfl_xor(g2i, m);
                }
            }
        }
        const R sJ = rec.J * inv4pi;
        const R sh = -dn * sJ;
        // h_j (mesh.cu:661-663), N3 = 1 - N1 - N2
        R p0r = sh * h1r, p0i = sh * h1i;
        R p1r = sh * h2r, p1i = sh * h2i;
        R p2r = sh * (htr - h1r - h2r), p2i = sh * (hti - h1i - h2i);
        // sum_j g_j = i rho omega (J/4pi) sum w G~  (mesh.cu:657-659, 668-670)
        const R sg = a.rw * sJ;
        const R gsr = -sg * gi, gsi = sg * gr;
        if (IMP) {
            // p_j = h_j - beta g_j
            const R br = rec.beta[0], bi = rec.beta[1];
            const R G0r = -sg * g1i, G0i = sg * g1r;
            const R G1r = -sg * g2i, G1i = sg * g2r;
            const R G2r = gsr - G0r - G1r, G2i = gsi - G0i - G1i;
            p0r -= br * G0r - bi * G0i; p0i -= br * G0i + bi * G0r;
            p1r -= br * G1r - bi * G1i; p1i -= br * G1i + bi * G1r;
            p2r -= br * G2r - bi * G2i; p2i -= br * G2i + bi * G2r;
        }
        R cval = -dn * sJ * cc;  // c_l_nsgl (mesh.cu:645, 665)
        R btr = rec.gamma[0] * gsr - rec.gamma[1] * gsi;
        R bti = rec.gamma[0] * gsi + rec.gamma[1] * gsr;
        // singular rows: x is a vertex of e (atomicFuncs.cu:75-76): take the FP64 rule
        const int sv = (row == rec.nodes[0]) ? 0 : (row == rec.nodes[1]) ? 1 : (row == rec.nodes[2]) ? 2 : -1;
        if (sv >= 0) {
            const R *s = a.sing + ((size_t)e * 3 + sv) * 16;
            p0r = s[0]; p0i = s[1]; p1r = s[2]; p1i = s[3]; p2r = s[4]; p2i = s[5];
            cval = s[6];
            btr = s[7];
            bti = s[8];
        }
        // scatter into this wave's own rows of A (first touch writes)
        const bool writer = active && (QG == 1 || qg == 0);
        if (writer) {
            const R pr[3] = {p0r, p1r, p2r}, pi[3] = {p0i, p1i, p2i};
#pragma unroll
            for (int j = 0; j < 3; j++) {
                if ((ent >> j) & 1) {
                    C2 *dst = a.A + (size_t)rec.nodes[j] * a.ldA + (row - a.r0);
                    C2 v;
                    if ((ent >> (3 + j)) & 1) {
                        v.x = pr[j];
                        v.y = pi[j];
                    } else {
                        v = *dst;
                        v.x += pr[j];
                        v.y += pi[j];
                    }
                    *dst = v;
                }
            }
        }
        if ((ent >> 6) & 1) {
            c_acc += cval;
            br_acc += btr;
            bi_acc += bti;
        }
    }
    if (active && (QG == 1 || qg == 0)) {
        a.cpart[(size_t)tile * a.Mp + (row - a.r0)] = c_acc;
        C2 b;
        b.x = br_acc;
        b.y = bi_acc;
        a.bpart[(size_t)tile * a.Mp + (row - a.r0)] = b;
    }
}

// ------------------------------------------- FP32 fast path (one lane/row) ---
// The 6x6 collapsed rule is separable: with theta_n, rho_m the mapped
// Gauss-Legendre nodes, xi = rho_m ((1 - theta_n), theta_n) and
// W = 0.25 w_n w_m rho_m, so the point offset is y - x = a + rho_m v_n with
// v_n = e1 + theta_n (e2 - e1) (one vector per theta row), and the
// shape-function sums factor per theta row:
//   h_1 = sum_n (1 - theta_n) A_n,  h_2 = sum_n theta_n A_n,  h_tot = sum_n B_n,
//   A_n = sum_m W rho_m H~,  B_n = sum_m W H~.
// All rule constants are compile-time literals.  sin / cos of the phase come
// from v_sin_f32 / v_cos_f32, which take revolutions u = k r / (2 pi) and are
// specified for |u| <= 256 (measured on gfx950: max abs error 1.2e-7 against
// sin(2 pi u) of the FP32 u over that whole range).  RAW passes u = r k/(2 pi)
// as one rounded product; otherwise u is first reduced to |u| <= 1/2 with the
// round-to-nearest magic constant 1.5 * 2^23 (for geometries that reach past
// 256 revolutions).  The rounding of the product adds an error of the order of
// the one r already carries: at 8 kHz on icosphere s5 the relative Frobenius
// error of A against FP64 goes from 1.060e-7 to 1.063e-7, and the kernel
// runs 5 % faster (two fewer dependent instructions per point).
// The squared distance of a point is formed from its coordinates' differences
// a + rho_m v_n where a row is near the element (closer than the far rules
// allow).  For the other rows on 36 points, those of elements that the
// wavelength does not resolve, it is expanded per theta row,
//   r^2 = |a|^2 + rho_m (2 a.v_n + rho_m |v_n|^2),
// two FMAs per point instead of six.  Its rounding error grows as (|a| / r)^2,
// that of the differences as |a| / r: on a 2562-node body, the entries of the
// nearest nodes for rows 0.01 edge lengths off the surface were off by 1.2e-4
// (median; at most 2e-3), with the differences by 8e-7 (7e-6); FP64 2e-13
// (2e-12) and 1.5e-15 (1e-14).  It costs 0.08 of 2.0 ms at 10242 nodes, 5 of 43
// us at 642.
__device__ __forceinline__ constexpr float gl_theta(int n) { return (float)(0.5 + 0.5 * GL6::eta[n]); }
__device__ __forceinline__ constexpr float gl_rho(int m) { return (float)(0.5 + 0.5 * GL6::eta[m]); }
// theta_n - theta_{n+1} for n < 5, theta_5 for n = 5
__device__ __forceinline__ constexpr float gl_dtheta(int n) {
    return n < 5 ? (float)(0.5 * (GL6::eta[n] - GL6::eta[n < 5 ? n + 1 : n])) : (float)(0.5 + 0.5 * GL6::eta[5]);
}
__device__ __forceinline__ constexpr float gl_W(int n, int m) {
    return (float)(0.25 * GL6::w[n] * GL6::w[m] * (0.5 + 0.5 * GL6::eta[m]));
}
__device__ __forceinline__ constexpr float gl_Wrho(int n, int m) {
    return (float)(0.25 * GL6::w[n] * GL6::w[m] * (0.5 + 0.5 * GL6::eta[m]) * (0.5 + 0.5 * GL6::eta[m]));
}

typedef __attribute__((address_space(4))) const ElemRec<float> CElemRec;

__device__ __forceinline__ bool wave_all(bool p) { return __builtin_amdgcn_ballot_w64(!p) == 0; }

// sums over the 36 points: S = sum W rho H~ and ht = sum W H~; the theta moment
// h2 = sum_n theta_n A_n of the per-row sums A_n comes from the running totals
// S_n of S after each row,
//   h2 = sum_{n<5} (theta_n - theta_{n+1}) S_n + theta_5 S_5,
// and h1 = S - h2 (likewise g1, g2 from SC = sum W rho G~)
struct Sums36 {
    float Sr = 0, Si = 0, h2r = 0, h2i = 0, htr = 0, hti = 0, gr = 0, gi = 0, cc = 0;
    float SCr = 0, SCi = 0, g2r = 0, g2i = 0;
};
// one point: 4 pi r dG/dn / (-dn) = (cos kr - i sin kr)(1/r^3 + i k/r^2) and
// 4 pi G = (cos kr - i sin kr) / r
struct Point36 {
    float Hr, Hi, Gr, Gi, q3;
};
template <bool RAW>
__device__ __forceinline__ Point36 point36(float r2, float k, float krev) {
    const float MAGIC = 12582912.0f;  // 1.5 * 2^23
    const float rinv = __builtin_amdgcn_rsqf(r2);
    const float r = r2 * rinv;
    float u;
    if (RAW) {
        u = r * krev;
    } else {
        const float t2 = __builtin_fmaf(r, krev, MAGIC);
        const float jf = t2 - MAGIC;
        u = __builtin_fmaf(r, krev, -jf);
    }
    const float sn = __builtin_amdgcn_sinf(u), cs = __builtin_amdgcn_cosf(u);
    const float rinv2 = rinv * rinv;
    const float q2k = k * rinv2;  // k/r^2
    Point36 p;
    p.q3 = rinv2 * rinv;  // 1/r^3
    p.Hr = __builtin_fmaf(cs, p.q3, sn * q2k);
    p.Hi = __builtin_fmaf(cs, q2k, -sn * p.q3);
    p.Gr = cs * rinv;
    p.Gi = -sn * rinv;
    return p;
}
template <bool IMP, bool RAW, bool SRC>
__device__ __forceinline__ void sums36(CElemRec &rec, float ax, float ay, float az, float k, float krev, Sums36 &s) {
    const float aa = __builtin_fmaf(ax, ax, __builtin_fmaf(ay, ay, az * az));
    // 2 a.v_n = 2 a.e1 + 2 theta_n a.f
    const float ae1 = __builtin_fmaf(ax, rec.e1[0], __builtin_fmaf(ay, rec.e1[1], az * rec.e1[2]));
    const float af = __builtin_fmaf(ax, rec.f[0], __builtin_fmaf(ay, rec.f[1], az * rec.f[2]));
    const float ae1x2 = ae1 + ae1;
#pragma unroll
    for (int n = 0; n < 6; n++) {
        const float th = gl_theta(n);
        const float tav = __builtin_fmaf(2.0f * th, af, ae1x2);
        const float vv = rec.vv[n];
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const float rho = gl_rho(m), W = gl_W(n, m), Wr = gl_Wrho(n, m);
            const Point36 p = point36<RAW>(__builtin_fmaf(rho, __builtin_fmaf(rho, vv, tav), aa), k, krev);
            s.Sr = __builtin_fmaf(Wr, p.Hr, s.Sr);
            s.Si = __builtin_fmaf(Wr, p.Hi, s.Si);
            s.htr = __builtin_fmaf(W, p.Hr, s.htr);
            s.hti = __builtin_fmaf(W, p.Hi, s.hti);
            if (IMP || SRC) {
                s.gr = __builtin_fmaf(W, p.Gr, s.gr);
                s.gi = __builtin_fmaf(W, p.Gi, s.gi);
            }
            if (IMP) {
                s.SCr = __builtin_fmaf(Wr, p.Gr, s.SCr);
                s.SCi = __builtin_fmaf(Wr, p.Gi, s.SCi);
            }
            s.cc = __builtin_fmaf(W, p.q3, s.cc);
        }
        // theta moment of the rho-weighted sums from their running totals
        const float dth = gl_dtheta(n);
        s.h2r = __builtin_fmaf(dth, s.Sr, s.h2r);
        s.h2i = __builtin_fmaf(dth, s.Si, s.h2i);
        if (IMP) {
            s.g2r = __builtin_fmaf(dth, s.SCr, s.g2r);
            s.g2i = __builtin_fmaf(dth, s.SCi, s.g2i);
        }
    }
}
// theta and 0.25 w of a theta row
struct ThetaRow32 {
    float th, w;
};
__device__ constexpr ThetaRow32 kTheta32[6] = {
#define BEM_TH(n) {(float)(0.5 + 0.5 * GL6::eta[n]), (float)(0.25 * GL6::w[n])}
    BEM_TH(0), BEM_TH(1), BEM_TH(2), BEM_TH(3), BEM_TH(4), BEM_TH(5)
#undef BEM_TH
};
// the same for a row near the element.  (The theta rows are a loop: unrolled,
// both forms together take 111 to 185 registers instead of 72 to 91, and the
// assembly of 10242 nodes 2.3 ms instead of 2.0.)
template <bool IMP, bool RAW, bool SRC>
__device__ __forceinline__ void sums36_near(CElemRec &rec, float ax, float ay, float az, float k, float krev,
                                            Sums36 &s) {
#pragma unroll 1
    for (int n = 0; n < 6; n++) {
        const ThetaRow32 t = kTheta32[n];
        const float vx = __builtin_fmaf(t.th, rec.f[0], rec.e1[0]), vy = __builtin_fmaf(t.th, rec.f[1], rec.e1[1]),
                    vz = __builtin_fmaf(t.th, rec.f[2], rec.e1[2]);
        // sums over m with w_m rho_m and w_m rho_m^2
        float br = 0, bi = 0, ar = 0, ai = 0, gbr = 0, gbi = 0, gar = 0, gai = 0, c = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const float rho = gl_rho(m), wr = (float)(GL6::w[m] * (0.5 + 0.5 * GL6::eta[m])),
                        wr2 = (float)(GL6::w[m] * (0.5 + 0.5 * GL6::eta[m]) * (0.5 + 0.5 * GL6::eta[m]));
            const float dx = __builtin_fmaf(rho, vx, ax), dy = __builtin_fmaf(rho, vy, ay),
                        dz = __builtin_fmaf(rho, vz, az);
            const Point36 p =
                point36<RAW>(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)), k, krev);
            br = __builtin_fmaf(wr, p.Hr, br);
            bi = __builtin_fmaf(wr, p.Hi, bi);
            ar = __builtin_fmaf(wr2, p.Hr, ar);
            ai = __builtin_fmaf(wr2, p.Hi, ai);
            if (IMP || SRC) {
                gbr = __builtin_fmaf(wr, p.Gr, gbr);
                gbi = __builtin_fmaf(wr, p.Gi, gbi);
            }
            if (IMP) {
                gar = __builtin_fmaf(wr2, p.Gr, gar);
                gai = __builtin_fmaf(wr2, p.Gi, gai);
            }
            c = __builtin_fmaf(wr, p.q3, c);
        }
        const float w2 = t.w * t.th;
        s.htr = __builtin_fmaf(t.w, br, s.htr);
        s.hti = __builtin_fmaf(t.w, bi, s.hti);
        s.Sr = __builtin_fmaf(t.w, ar, s.Sr);
        s.Si = __builtin_fmaf(t.w, ai, s.Si);
        s.h2r = __builtin_fmaf(w2, ar, s.h2r);
        s.h2i = __builtin_fmaf(w2, ai, s.h2i);
        if (IMP || SRC) {
            s.gr = __builtin_fmaf(t.w, gbr, s.gr);
            s.gi = __builtin_fmaf(t.w, gbi, s.gi);
        }
        if (IMP) {
            s.SCr = __builtin_fmaf(t.w, gar, s.SCr);
            s.SCi = __builtin_fmaf(t.w, gai, s.SCi);
            s.g2r = __builtin_fmaf(w2, gar, s.g2r);
            s.g2i = __builtin_fmaf(w2, gai, s.g2i);
        }
        s.cc = __builtin_fmaf(t.w, c, s.cc);
    }
}

// The rule is chosen per (wave, element): the fewest points that every row of
// the wave may take.  Element records and tile lists are read as scalar loads
// (constant address space): as vector loads, which the compiler falls back to
// because it cannot see that A is never the record array, a pair took 19 vector
// memory instructions instead of 6 and a chain of waits (10242 nodes: 2.78 ms
// against 2.12).
// IMP: some element has ca != 0; SRC: some element has cc != 0 (without it
// the boundary term is zero and no g is summed).
template <bool IMP, bool RAW, bool GH, bool SRC>
__global__ __launch_bounds__(256) void asm_tile_fast(AsmArgs<float> a) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int L = xcd_remap(blockIdx.x, a.nwg);
    const int tile = L / a.nrbg;
    const int rbg = L - tile * a.nrbg;
    const int row = a.r0 + (rbg * 4 + wave) * 64 + lane;
    const bool active = row < a.M;
    if (wave_all(!active)) return;  // the workgroup's last waves may have no rows
    const unsigned lrow = (unsigned)(row - a.r0);
    const float4 xp = a.pts[active ? row : 0];
    const double xd = xp.x, yd = xp.y, zd = xp.z;
    const float k = a.k;
    const float krev = a.kf;  // k / (2 pi)
    const float inv4pi = (float)(1.0 / (4.0 * kPi));
    float c_acc = 0, br_acc = 0, bi_acc = 0;
    CInt *entries = (CInt *)a.tile_entries, *slots = (CInt *)a.tile_slots;
    const int it0 = ((CInt *)a.tile_ptr)[tile], it1 = ((CInt *)a.tile_ptr)[tile + 1];
    // what an entry's first loads and branches need, asked for while the entry
    // before is integrated: a wave that is alone on its SIMD (small meshes)
    // then waits for fewer loads in turn
    struct Next {
        int ent, rho2, node[3], slot[3];
        float far16;
        double c[3];
    } nx;
    auto fetch = [&](int it) {
        nx.ent = entries[it];
        CFarRec &f = ((CFarRec *)a.far)[nx.ent >> 8];
        nx.rho2 = __float_as_int(f.rho2);
        nx.far16 = f.far16;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            nx.node[j] = f.nodes[j];
            nx.slot[j] = GH ? slots[3 * it + j] : 0;
            nx.c[j] = f.c[j];
        }
    };
    if (it0 < it1) fetch(it0);
    for (int it = it0; it < it1; ++it) {
        const Next cur = nx;
        const int ent = cur.ent;
        const int e = ent >> 8;
        if (it + 1 < it1) fetch(it + 1);
        CFarRec &fr = ((CFarRec *)a.far)[e];
        // the three columns this pair adds to: A's, or a ghost vertex's side
        // column; their values so far are asked for before the quadrature
        float2 *col[3];
        float2 v[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            col[j] = nullptr;
            if ((ent >> j) & 1) col[j] = a.A + (size_t)cur.node[j] * a.ldA;
            else if (GH) col[j] = a.side + (size_t)cur.slot[j] * a.Mp;
            v[j] = make_float2(0.f, 0.f);
            if (col[j] && !((ent >> (3 + j)) & 1) && active) v[j] = col[j][lrow];
        }
        const FarDist fd = far_dist(cur.c, xd, yd, zd);
        const float r02f = fd.r02f;
        const int rho2 = cur.rho2;  // (positive floats compare as integers: scalar compares)
        float pr[3], pi[3], cval, btr = 0, bti = 0;
        const bool distant = wave_all(!active || r02f >= cur.far16);
        if (distant && rho2 <= a.far_rho2) {
            const FarGeom g = far_geom(fr, fd, k, krev, a.kf64);
            FarSums s;
            if (rho2 <= a.far7_rho2 && wave_all(!active || r02f >= fr.far7))
                far_sums<Far7, IMP, SRC>(fr.uu, nullptr, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            else if (wave_all(!active || r02f >= fr.far12))
                far_sums<Far12, IMP, SRC>(fr.uu, fr.d12, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            else
                far_sums<Far16, IMP, SRC>(fr.uu, fr.d16, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            far_terms<IMP, SRC>(fr, g, s, a.rw, pr, pi, cval, btr, bti);
        } else {
            CElemRec &rec = ((CElemRec *)a.recs)[e];
            const float ax = rec.p3[0] - xp.x, ay = rec.p3[1] - xp.y, az = rec.p3[2] - xp.z;
            const float dn = rec.n[0] * ax + rec.n[1] * ay + rec.n[2] * az;
            Sums36 q;
            if (distant) sums36<IMP, RAW, SRC>(rec, ax, ay, az, k, krev, q);
            else sums36_near<IMP, RAW, SRC>(rec, ax, ay, az, k, krev, q);
            const float h1r = q.Sr - q.h2r, h1i = q.Si - q.h2i;
            const float g1r = q.SCr - q.g2r, g1i = q.SCi - q.g2i;
            const float sJ = rec.J * inv4pi;
            const float sh = -dn * sJ;
            float p0r = sh * h1r, p0i = sh * h1i;
            float p1r = sh * q.h2r, p1i = sh * q.h2i;
            float p2r = sh * (q.htr - q.Sr), p2i = sh * (q.hti - q.Si);
            const float sg = a.rw * sJ;
            const float gsr = -sg * q.gi, gsi = sg * q.gr;
            if (IMP) {
                const float br = rec.beta[0], bi = rec.beta[1];
                const float G0r = -sg * g1i, G0i = sg * g1r;
                const float G1r = -sg * q.g2i, G1i = sg * q.g2r;
                const float G2r = gsr - G0r - G1r, G2i = gsi - G0i - G1i;
                p0r -= br * G0r - bi * G0i; p0i -= br * G0i + bi * G0r;
                p1r -= br * G1r - bi * G1i; p1i -= br * G1i + bi * G1r;
                p2r -= br * G2r - bi * G2i; p2i -= br * G2i + bi * G2r;
            }
            cval = -dn * sJ * q.cc;
            if (IMP || SRC) {
                btr = rec.gamma[0] * gsr - rec.gamma[1] * gsi;
                bti = rec.gamma[0] * gsi + rec.gamma[1] * gsr;
            }
            const int sv = (row == rec.nodes[0]) ? 0 : (row == rec.nodes[1]) ? 1 : (row == rec.nodes[2]) ? 2 : -1;
            if (sv >= 0) {
                const float *sg2 = a.sing + ((size_t)e * 3 + sv) * 16;
                p0r = sg2[0]; p0i = sg2[1]; p1r = sg2[2]; p1i = sg2[3]; p2r = sg2[4]; p2i = sg2[5];
                cval = sg2[6];
                btr = sg2[7];
                bti = sg2[8];
            }
            pr[0] = p0r; pr[1] = p1r; pr[2] = p2r;
            pi[0] = p0i; pi[1] = p1i; pi[2] = p2i;
        }
        if (active) {
#pragma unroll
            for (int j = 0; j < 3; j++)
                if (col[j]) col[j][lrow] = make_float2(v[j].x + pr[j], v[j].y + pi[j]);
        }
        if ((ent >> 6) & 1) {
            c_acc += cval;
            if (IMP || SRC) {
                br_acc += btr;
                bi_acc += bti;
            }
        }
    }
    if (active) {
        a.cpart[(size_t)tile * a.Mp + (row - a.r0)] = c_acc;
        if (IMP || SRC) a.bpart[(size_t)tile * a.Mp + (row - a.r0)] = make_float2(br_acc, bi_acc);
    }
}

// ------------------------------------------- FP64 fast path (one lane/row) ---
// sin and cos for |x| <= 0.8: near-minimax polynomials (coefficients fitted in
// 60 digits for this library; absolute error 1.5e-17 before rounding).
__device__ __forceinline__ void sincos_small(double x, double &sn, double &cs) {
    const double z = x * x;
    double p = fma(z, 1.5909586259665044e-10, -2.5051009657015125e-08);
    p = fma(z, p, 2.755731549825422e-06);
    p = fma(z, p, -0.00019841269835557402);
    p = fma(z, p, 0.00833333333333013);
    p = fma(z, p, -0.16666666666666663);
    sn = fma(z * x, p, x);
    double q = fma(z, -1.137728782340167e-11, 2.0876069826994487e-09);
    q = fma(z, q, -2.7557316893681153e-07);
    q = fma(z, q, 2.4801587298014246e-05);
    q = fma(z, q, -0.0013888888888886886);
    q = fma(z, q, 0.041666666666666664);
    cs = fma(z * z, q, fma(z, -0.5, 1.0));
}
// the same for |x| < 2^30: the quadrant is removed with pi/2 in three parts
// (Cody and Waite 1980)
__device__ __forceinline__ void sincos_wide(double x, double &sn, double &cs) {
    const double n = rint(x * 0.6366197723675814);
    double f = fma(-n, 1.5707963267948966, x);
    f = fma(-n, 6.123233995736766e-17, f);
    f = fma(-n, -1.4973849048591698e-33, f);
    double s, c;
    sincos_small(f, s, c);
    const int q = (int)n;
    const double a = (q & 1) ? c : s, b = (q & 1) ? s : c;
    sn = (q & 2) ? -a : a;
    cs = ((q + 1) & 2) ? -b : b;
}
// 1 / sqrt(x): v_rsq_f64 (relative error 2^-23) and one third-order step
__device__ __forceinline__ double rsq_f64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// kappa^2 up to which an element's phases from its centroid's stay within 0.8
constexpr float kSmallPhase64 = 0.63f;

// rule constants of a theta row: 2 theta, 0.25 w, and 0.25 w (1 - theta), 0.25 w theta
struct ThetaRow {
    double th2, w, w1, w2;
};
__device__ constexpr ThetaRow kTheta[6] = {
#define BEM_TH(n)                                                                            \
    {                                                                                        \
        1.0 + GL6::eta[n], 0.25 * GL6::w[n], 0.25 * GL6::w[n] * (0.5 - 0.5 * GL6::eta[n]),   \
            0.25 * GL6::w[n] * (0.5 + 0.5 * GL6::eta[n])                                     \
    }
    BEM_TH(0), BEM_TH(1), BEM_TH(2), BEM_TH(3), BEM_TH(4), BEM_TH(5)
#undef BEM_TH
};

typedef __attribute__((address_space(4))) const ElemRec<double> CElemRec64;

// Sums of the 36 points relative to the phase k r0 of the element's centroid;
// SMALL: |k (r - r0)| <= 0.8 on the element, so its sine and cosine need no
// quadrant.  NEAR: distances from the coordinates' differences, otherwise
// expanded per theta row (as sums36).
struct FastSums64 {
    double hr[3], hi[3], gr[3], gi[3], c;
};
template <bool IMP, bool SRC, bool SMALL, bool NEAR>
__device__ __forceinline__ void fast_sums64(CElemRec64 &rec, double ax, double ay, double az, double k, double kr0,
                                            FastSums64 &s) {
    const double aa = fma(ax, ax, fma(ay, ay, az * az));
    const double ae1 = fma(ax, rec.e1[0], fma(ay, rec.e1[1], az * rec.e1[2]));
    const double af = fma(ax, rec.f[0], fma(ay, rec.f[1], az * rec.f[2]));
    double htr = 0, hti = 0, gtr = 0, gti = 0;
    s.hr[0] = s.hr[1] = s.hi[0] = s.hi[1] = s.gr[0] = s.gr[1] = s.gi[0] = s.gi[1] = s.c = 0;
#pragma unroll 1
    for (int n = 0; n < 6; n++) {
        const ThetaRow th = kTheta[n];
        const double tav = fma(th.th2, af, ae1 + ae1), v = rec.vv[n], t = 0.5 * th.th2;
        const double vx = fma(t, rec.f[0], rec.e1[0]), vy = fma(t, rec.f[1], rec.e1[1]), vz = fma(t, rec.f[2], rec.e1[2]);
        // sums over m: B with w_m rho_m, A with w_m rho_m^2
        double ar = 0, ai = 0, br = 0, bi = 0, gbr = 0, gbi = 0, gar = 0, gai = 0, c = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const double rho = 0.5 + 0.5 * GL6::eta[m], wr = GL6::w[m] * rho, wr2 = wr * rho;
            double r2;
            if (NEAR) {
                const double dx = fma(rho, vx, ax), dy = fma(rho, vy, ay), dz = fma(rho, vz, az);
                r2 = fma(dx, dx, fma(dy, dy, dz * dz));
            } else {
                r2 = fma(rho, fma(rho, v, tav), aa);
            }
            const double y = rsq_f64(r2);
            const double d = fma(k, r2 * y, -kr0);
            double sn, cs;
            if (SMALL) sincos_small(d, sn, cs);
            else sincos_wide(d, sn, cs);
            const double y2 = y * y;
            const double q3 = y2 * y, q2k = k * y2;
            const double Hr = fma(cs, q3, sn * q2k), Hi = fma(cs, q2k, -sn * q3);
            br = fma(wr, Hr, br);
            bi = fma(wr, Hi, bi);
            ar = fma(wr2, Hr, ar);
            ai = fma(wr2, Hi, ai);
            c = fma(wr, q3, c);
            if (IMP || SRC) {
                const double Gr = cs * y, Gi = -sn * y;
                gbr = fma(wr, Gr, gbr);
                gbi = fma(wr, Gi, gbi);
                if (IMP) {
                    gar = fma(wr2, Gr, gar);
                    gai = fma(wr2, Gi, gai);
                }
            }
        }
        htr = fma(th.w, br, htr);
        hti = fma(th.w, bi, hti);
        s.hr[0] = fma(th.w1, ar, s.hr[0]);
        s.hi[0] = fma(th.w1, ai, s.hi[0]);
        s.hr[1] = fma(th.w2, ar, s.hr[1]);
        s.hi[1] = fma(th.w2, ai, s.hi[1]);
        s.c = fma(th.w, c, s.c);
        if (IMP || SRC) {
            gtr = fma(th.w, gbr, gtr);
            gti = fma(th.w, gbi, gti);
        }
        if (IMP) {
            s.gr[0] = fma(th.w1, gar, s.gr[0]);
            s.gi[0] = fma(th.w1, gai, s.gi[0]);
            s.gr[1] = fma(th.w2, gar, s.gr[1]);
            s.gi[1] = fma(th.w2, gai, s.gi[1]);
        }
    }
    s.hr[2] = htr - s.hr[0] - s.hr[1];
    s.hi[2] = hti - s.hi[0] - s.hi[1];
    s.gr[2] = gtr - s.gr[0] - s.gr[1];  // (without IMP: the whole sum)
    s.gi[2] = gti - s.gi[0] - s.gi[1];
}

// The FP64 form of asm_tile_fast: the separable 36-point rule on every pair, on
// the element-once plan.  Bound by the vector ALU: the generic kernel spent
// about 290 issue slots a point on the library's sincos, square root and
// division, at 396 registers (one wave per SIMD); here a point's phase is
// taken from the centroid's, whose sine and cosine are computed once per pair,
// so what is left is small and needs no reduction, and 1/r is one rsq step:
// about 45 slots.  5762 nodes: 21.4 ms before.
template <bool IMP, bool SRC>
__global__ __launch_bounds__(256) void asm_tile_fast64(AsmArgs<double> a) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int L = xcd_remap(blockIdx.x, a.nwg);
    const int tile = L / a.nrbg;
    const int rbg = L - tile * a.nrbg;
    const int row = a.r0 + (rbg * 4 + wave) * 64 + lane;
    const bool active = row < a.M;
    if (wave_all(!active)) return;  // the workgroup's last waves may have no rows
    const unsigned lrow = (unsigned)(row - a.r0);
    const float4 xp = a.pts[active ? row : 0];
    const double x0 = xp.x, x1 = xp.y, x2 = xp.z;
    const double k = a.k, inv4pi = 1.0 / (4.0 * kPi);
    double c_acc = 0, br_acc = 0, bi_acc = 0;
    CInt *entries = (CInt *)a.tile_entries, *slots = (CInt *)a.tile_slots;
    const int it0 = ((CInt *)a.tile_ptr)[tile], it1 = ((CInt *)a.tile_ptr)[tile + 1];
    for (int it = it0; it < it1; ++it) {
        const int ent = entries[it];
        const int e = ent >> 8;
        CFarRec &fr = ((CFarRec *)a.far)[e];
        CElemRec64 &rec = ((CElemRec64 *)a.recs)[e];
        const double cx = fr.c[0] - x0, cy = fr.c[1] - x1, cz = fr.c[2] - x2;
        const double r02 = fma(cx, cx, fma(cy, cy, cz * cz));
        // (a row on the centroid: rsq_f64(0) is NaN, the distance is zero)
        const double kr0 = r02 > 0 ? k * (r02 * rsq_f64(r02)) : 0.0;
        const double ax = rec.p3[0] - x0, ay = rec.p3[1] - x1, az = rec.p3[2] - x2;
        const double dn = rec.n[0] * ax + rec.n[1] * ay + rec.n[2] * az;
        FastSums64 s;
        const bool distant = wave_all(!active || r02 >= (double)fr.far12);
        // (positive floats compare as integers)
        if (__float_as_int(fr.rho2) > a.far_rho2)
            fast_sums64<IMP, SRC, false, true>(rec, ax, ay, az, k, kr0, s);
        else if (distant)
            fast_sums64<IMP, SRC, true, false>(rec, ax, ay, az, k, kr0, s);
        else
            fast_sums64<IMP, SRC, true, true>(rec, ax, ay, az, k, kr0, s);
        double s0, c0;
        sincos_wide(kr0, s0, c0);
        const double sJ = rec.J * inv4pi, m = -dn * sJ;
        const double fx = m * c0, fy = -m * s0;
        double pr[3], pi[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            pr[j] = fma(fx, s.hr[j], -fy * s.hi[j]);
            pi[j] = fma(fx, s.hi[j], fy * s.hr[j]);
        }
        double cval = m * s.c, btr = 0, bti = 0;
        if (IMP || SRC) {
            const double sg = a.rw * sJ, qx = sg * s0, qy = sg * c0;
            double gsr = 0, gsi = 0;
#pragma unroll
            for (int j = IMP ? 0 : 2; j < 3; j++) {
                const double Gr = fma(qx, s.gr[j], -qy * s.gi[j]), Gi = fma(qx, s.gi[j], qy * s.gr[j]);
                if (IMP) {
                    pr[j] -= rec.beta[0] * Gr - rec.beta[1] * Gi;
                    pi[j] -= rec.beta[0] * Gi + rec.beta[1] * Gr;
                }
                gsr += Gr;
                gsi += Gi;
            }
            btr = rec.gamma[0] * gsr - rec.gamma[1] * gsi;
            bti = rec.gamma[0] * gsi + rec.gamma[1] * gsr;
        }
        const int sv = (row == rec.nodes[0]) ? 0 : (row == rec.nodes[1]) ? 1 : (row == rec.nodes[2]) ? 2 : -1;
        if (sv >= 0) {
            const double *sg2 = a.sing + ((size_t)e * 3 + sv) * 16;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                pr[j] = sg2[2 * j];
                pi[j] = sg2[2 * j + 1];
            }
            cval = sg2[6];
            btr = sg2[7];
            bti = sg2[8];
        }
        if (active) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
                double2 *col = (ent >> j) & 1 ? a.A + (size_t)rec.nodes[j] * a.ldA
                                              : a.side + (size_t)slots[3 * it + j] * a.Mp;
                double2 v = make_double2(0.0, 0.0);
                if (!((ent >> (3 + j)) & 1)) v = col[lrow];
                col[lrow] = make_double2(v.x + pr[j], v.y + pi[j]);
            }
        }
        if ((ent >> 6) & 1) {
            c_acc += cval;
            if (IMP || SRC) {
                br_acc += btr;
                bi_acc += bti;
            }
        }
    }
    if (active) {
        a.cpart[(size_t)tile * a.Mp + lrow] = c_acc;
        if (IMP || SRC) a.bpart[(size_t)tile * a.Mp + lrow] = make_double2(br_acc, bi_acc);
    }
}

// Columns of nodes no element references: only the diagonal survives.
template <typename C2>
__global__ void zero_columns(C2 *A, long ldA, int M, const int *__restrict__ cols, int ncols) {
    const int c = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncols || i >= M) return;
    C2 z;
    z.x = 0;
    z.y = 0;
    A[(size_t)cols[c] * ldA + i] = z;
}

// Element-once plan: column of ghost node g += its side columns, in the order
// they were made (the column is set when the node's own tile wrote nothing).
// W rows per thread, 16-byte accesses: two adjacent rows in FP32 (ldA and Mp
// are even), one in FP64.
template <typename V4, int W>
__global__ void ghost_reduce(V4 *A, long ldA, int nrows, const V4 *__restrict__ side, long Mp,
                             const int *__restrict__ gptr, const int *__restrict__ gnode,
                             const int *__restrict__ gown, const int *__restrict__ gslot) {
    const int g = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (nrows + W - 1) / W) return;
    // (an odd last row of W = 2 takes the padding row with it: both are in bounds)
    V4 *col = A + (size_t)gnode[g] * (ldA / W);
    const int s0 = gptr[g], s1 = gptr[g + 1];
    V4 acc{};
    if (gown[g]) acc = col[i];
    for (int t = s0; t < s1; t++) {
        const V4 v = side[(size_t)gslot[t] * (Mp / W) + i];
        acc.x += v.x;
        acc.y += v.y;
        if constexpr (W == 2) {
            acc.z += v.z;
            acc.w += v.w;
        }
    }
    col[i] = acc;
}

// Per row: sum of the tile partials in FP64 in a fixed order (16 runs of
// consecutive tiles, one per wave of the workgroup, then the runs).  One wave
// per 64 rows walked all tiles in turn before: 45 us for 4002 rows in 500
// tiles, bound by the chain of loads.
// Rows r0..M-1 (local index i = row - r0 in A, the partials and bterm).
// src == 0: no element has a boundary term, its partials are not read.
constexpr int kFinRuns = 16;
template <typename R, typename C2>
__global__ __launch_bounds__(64 * kFinRuns) void asm_finalize(C2 *A, long ldA, int M, int N, int P, long Mp, int r0,
                                                              const R *__restrict__ cpart,
                                                              const C2 *__restrict__ bpart,
                                                              double2 *__restrict__ bterm, int src) {
    __shared__ double red[3][kFinRuns][64];
    const int lane = threadIdx.x & 63, run = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    const int row = r0 + i;
    double cs = 0, br = 0, bi = 0;
    if (row < M) {
        const int per = (P + kFinRuns - 1) / kFinRuns;
        const int t1 = min(P, (run + 1) * per);
        for (int t = run * per; t < t1; t++) {
            cs += (double)cpart[(size_t)t * Mp + i];
            if (src) {
                const C2 b = bpart[(size_t)t * Mp + i];
                br += (double)b.x;
                bi += (double)b.y;
            }
        }
    }
    red[0][run][lane] = cs;
    red[1][run][lane] = br;
    red[2][run][lane] = bi;
    __syncthreads();
    if (run > 0 || row >= M) return;
    for (int q = 1; q < kFinRuns; q++) {
        cs += red[0][q][lane];
        br += red[1][q][lane];
        bi += red[2][q][lane];
    }
    if (row < N) {
        C2 *d = A + (size_t)row * ldA + i;
        C2 v = *d;
        v.x = (R)((double)v.x + (1.0 - cs));
        *d = v;
    }
    bterm[i] = make_double2(br, bi);
}

// B[:, s] = inc_s(x) - bterm: point source q G(x, src) (atomicFuncs.cu:238-242)
// or plane wave amp exp(-i k d.x); computed in FP64.
template <typename C2>
__global__ void rhs_fill(const double *__restrict__ pts64, int M, double k, int kind, double amp,
                         const float *__restrict__ params, int nrhs, const double2 *__restrict__ bterm,
                         C2 *B, long ldB) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = blockIdx.y;
    if (i >= M || s >= nrhs) return;
    const double x = pts64[3 * i], y = pts64[3 * i + 1], z = pts64[3 * i + 2];
    const double px = params[3 * s], py = params[3 * s + 1], pz = params[3 * s + 2];
    double ir, ii;
    if (kind == BEM_RHS_PLANE) {
        double sn, cs;
        sincos(k * (px * x + py * y + pz * z), &sn, &cs);
        ir = amp * cs;
        ii = -amp * sn;
    } else {
        const double dx = x - px, dy = y - py, dz = z - pz;
        const double r = sqrt(dx * dx + dy * dy + dz * dz);
        double sn, cs;
        sincos(k * r, &sn, &cs);
        const double g = amp / (4.0 * kPi * r);
        ir = g * cs;
        ii = -g * sn;
        if (amp == 0.0) ir = ii = 0.0;
    }
    const double2 bt = bterm[i];
    C2 v;
    v.x = ir - bt.x;
    v.y = ii - bt.y;
    B[(size_t)s * ldB + i] = v;
}

// rho^2 (as FP32 bits) up to which kappa^2 = k^2 rho^2 allows a rule (a NaN k: none)
static void far_limits(double k, float kappa2, int &far_rho2, int &far7_rho2) {
    const float k2 = (float)(k * k), f = kappa2 / k2, f7 = kFar7K2 / k2;
    far_rho2 = far7_rho2 = -1;
    if (f >= 0.f) memcpy(&far_rho2, &f, sizeof f);
    if (f7 >= 0.f) memcpy(&far7_rho2, &f7, sizeof f7);
}

// ------------------------------------------------------------- field ---
// Exterior pressure (genExtPressure / pntElemOffset, mesh.cu:1008-1073) at P
// points for R nodal solutions.  Lane = field point; a workgroup of 16 waves
// walks a chunk of 64 elements, 4 per wave (element data and the solutions'
// nodal values uniform, read with scalar loads), with the far rules
// (far_rules.hpp) or the regular 6x6 rule as each point's distance asks, and
// accumulates sum_j (h_j - beta g_j) X[node_j] + gamma sum_j g_j; the waves'
// sums are added in LDS and the chunk partials by field_finalize, both in a
// fixed order that does not depend on P: a point's value is the same bit for
// bit alone and among others.
//
// What bounds it: with few points the chain of elements a wave walks alone,
// since most lanes idle (64 elements a wave took 312 us for one point of a
// 642-node body, and field_finalize's one thread per point 36 us for 8820
// elements); with many, the vector ALU.
constexpr int kFieldChunk = 64;
constexpr int kFieldWaves = 16;
constexpr int kFieldR = 16;

struct FieldArgs {
    const float4 *__restrict__ xs;  // w: the point's place in the result (int)
    const ElemRec<double> *__restrict__ recs;
    const FarRec *__restrict__ far;
    const float2 *__restrict__ X;  // N x R, ldx
    long ldx;
    float2 *part;                  // [chunk][r][P]
    int P, E, R, r0;
    float k, kf, rw;
    double kf64;
    int far_rho2, far7_rho2;
};

// p_j = h_j - beta g_j and the boundary term of one (point, element) pair by
// the 36-point rule, the distances in FP64: in FP32 the error of r grows as
// (size / distance)^2 next to the surface.
__device__ __forceinline__ void field_pair_near(const FieldArgs &a, CElemRec64 &rec, const float4 xp, float *pr,
                                                float *pi, float &btr, float &bti) {
    const double ax = rec.p3[0] - (double)xp.x, ay = rec.p3[1] - (double)xp.y, az = rec.p3[2] - (double)xp.z;
    const float dn = (float)(rec.n[0] * ax + rec.n[1] * ay + rec.n[2] * az);
    const double aa = fma(ax, ax, fma(ay, ay, az * az));
    const double ae1x2 = 2.0 * fma(ax, rec.e1[0], fma(ay, rec.e1[1], az * rec.e1[2]));
    const double af = fma(ax, rec.f[0], fma(ay, rec.f[1], az * rec.f[2]));
    float hr[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, gr[3] = {0, 0, 0}, gi[3] = {0, 0, 0};
#pragma unroll 1
    for (int n = 0; n < 6; n++) {
        const ThetaRow th = kTheta[n];
        const double tav = fma(th.th2, af, ae1x2), vv = rec.vv[n];
        // sums over m with w_m rho_m and w_m rho_m^2
        float br = 0, bi = 0, ar = 0, ai = 0, gbr = 0, gbi = 0, gar = 0, gai = 0;
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const double rho = 0.5 + 0.5 * GL6::eta[m];
            const float wr = (float)(GL6::w[m] * rho), wr2 = (float)(GL6::w[m] * rho * rho);
            const float r2 = (float)fma(rho, fma(rho, vv, tav), aa);
            const float rinv = rsq(r2);
            float sn, cs;
            sincos_rev(r2 * rinv * a.kf, sn, cs);
            const float rinv2 = rinv * rinv, q3 = rinv2 * rinv, q2k = a.k * rinv2;
            const float Hr = fmaf(cs, q3, sn * q2k), Hi = fmaf(cs, q2k, -sn * q3);
            const float Gr = cs * rinv, Gi = -sn * rinv;
            br = fmaf(wr, Hr, br);
            bi = fmaf(wr, Hi, bi);
            ar = fmaf(wr2, Hr, ar);
            ai = fmaf(wr2, Hi, ai);
            gbr = fmaf(wr, Gr, gbr);
            gbi = fmaf(wr, Gi, gbi);
            gar = fmaf(wr2, Gr, gar);
            gai = fmaf(wr2, Gi, gai);
        }
        const float w = (float)th.w, w1 = (float)th.w1, w2 = (float)th.w2;
        hr[0] = fmaf(w1, ar, hr[0]);
        hi[0] = fmaf(w1, ai, hi[0]);
        hr[1] = fmaf(w2, ar, hr[1]);
        hi[1] = fmaf(w2, ai, hi[1]);
        hr[2] = fmaf(w, br - ar, hr[2]);  // N_3 = 1 - rho
        hi[2] = fmaf(w, bi - ai, hi[2]);
        gr[0] = fmaf(w1, gar, gr[0]);
        gi[0] = fmaf(w1, gai, gi[0]);
        gr[1] = fmaf(w2, gar, gr[1]);
        gi[1] = fmaf(w2, gai, gi[1]);
        gr[2] = fmaf(w, gbr - gar, gr[2]);
        gi[2] = fmaf(w, gbi - gai, gi[2]);
    }
    const float sJ = (float)(rec.J * (1.0 / (4.0 * kPi))), sh = -dn * sJ, sg = a.rw * sJ;
    const float b0 = (float)rec.beta[0], b1 = (float)rec.beta[1];
    float gsr = 0, gsi = 0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const float Gr = -sg * gi[j], Gi = sg * gr[j];
        pr[j] = sh * hr[j] - (b0 * Gr - b1 * Gi);
        pi[j] = sh * hi[j] - (b0 * Gi + b1 * Gr);
        gsr += Gr;
        gsi += Gi;
    }
    btr = (float)rec.gamma[0] * gsr - (float)rec.gamma[1] * gsi;
    bti = (float)rec.gamma[0] * gsi + (float)rec.gamma[1] * gsr;
}

// RG: right-hand sides of a pass (the last ones of a.R may be fewer)
template <int RG>
__global__ __launch_bounds__(64 * kFieldWaves) void field_part(FieldArgs a) {
    constexpr int kShare = RG < 4 ? RG : 4;  // right-hand sides summed over the waves together
    __shared__ float2 red[kShare][kFieldWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const int chunk = blockIdx.y;
    const bool active = p < a.P;
    const float4 xp = a.xs[active ? p : 0];
    constexpr int per = kFieldChunk / kFieldWaves;
    const int e0 = __builtin_amdgcn_readfirstlane(chunk * kFieldChunk + wave * per), e1 = min(a.E, e0 + per);
    const int nr = min(RG, a.R - a.r0);
    float accr[RG], acci[RG];
#pragma unroll
    for (int r = 0; r < RG; r++) {
        accr[r] = 0;
        acci[r] = 0;
    }
    for (int e = e0; e < e1; e++) {
        CFarRec &fr = ((CFarRec *)a.far)[e];
        const FarGeom g = far_geom(fr, xp, a.k, a.kf, a.kf64);
        float pr[3], pi[3], btr, bti;
        const bool k16 = __float_as_int(fr.rho2) <= a.far_rho2, k7 = __float_as_int(fr.rho2) <= a.far7_rho2;
        if (k16 && g.r02f >= fr.far16) {
            FarSums s;
            if (k7 && g.r02f >= fr.far7)
                far_sums<Far7, true, true>(fr.uu, nullptr, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            else if (g.r02f >= fr.far12)
                far_sums<Far12, true, true>(fr.uu, fr.d12, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            else
                far_sums<Far16, true, true>(fr.uu, fr.d16, g.T1, g.T2, g.i02, g.kr0, g.kr0rev, s);
            float cval;
            far_terms<true, true>(fr, g, s, a.rw, pr, pi, cval, btr, bti);
        } else {
            field_pair_near(a, ((CElemRec64 *)a.recs)[e], xp, pr, pi, btr, bti);
        }
#pragma unroll
        for (int r = 0; r < RG; r++) {
            if (r < nr) {
                CFloat *xc = (CFloat *)(a.X + (size_t)(a.r0 + r) * a.ldx);
                float sr = btr, si = bti;
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    const float xr = xc[2 * (size_t)fr.nodes[j]], xi = xc[2 * (size_t)fr.nodes[j] + 1];
                    sr += pr[j] * xr - pi[j] * xi;
                    si += pr[j] * xi + pi[j] * xr;
                }
                accr[r] += sr;
                acci[r] += si;
            }
        }
    }
#pragma unroll
    for (int rb = 0; rb < RG; rb += kShare) {
        if (rb >= nr) break;
        if (rb > 0) __syncthreads();
#pragma unroll
        for (int r = 0; r < kShare; r++) red[r][wave][lane] = make_float2(accr[rb + r], acci[rb + r]);
        __syncthreads();
        if (wave < kShare && rb + wave < nr && active) {
            float sr = 0, si = 0;
#pragma unroll
            for (int w = 0; w < kFieldWaves; w++) {
                const float2 v = red[wave][w][lane];
                sr += v.x;
                si += v.y;
            }
            a.part[((size_t)chunk * a.R + a.r0 + rb + wave) * a.P + p] = make_float2(sr, si);
        }
    }
}

// out[w, r] = inc_r(x_p) - sum_chunks part, w the place that x_p names, in FP64: 16
// runs of every 16th chunk per point, then the runs in order
constexpr int kFieldRuns = 16;
__global__ __launch_bounds__(256) void field_finalize(const float4 *__restrict__ xs, int P, int R, int nchunks,
                                                      const float2 *__restrict__ part, double k, int kind, double amp,
                                                      const float *__restrict__ params, float2 *out, long ldo) {
    __shared__ double2 red[kFieldRuns][16];
    const int lp = threadIdx.x & 15, run = threadIdx.x >> 4;
    const int p = blockIdx.x * 16 + lp;
    const int r = blockIdx.y;
    double sr = 0, si = 0;
    if (p < P)
        for (int c = run; c < nchunks; c += kFieldRuns) {
            const float2 v = part[((size_t)c * R + r) * P + p];
            sr += v.x;
            si += v.y;
        }
    red[run][lp] = make_double2(sr, si);
    __syncthreads();
    if (run > 0 || p >= P) return;
    for (int q = 1; q < kFieldRuns; q++) {
        sr += red[q][lp].x;
        si += red[q][lp].y;
    }
    const float4 xp = xs[p];
    const double x = xp.x, y = xp.y, z = xp.z;
    double ir = 0, ii = 0;
    if (params) {
        const double px = params[3 * r], py = params[3 * r + 1], pz = params[3 * r + 2];
        double sn, cs;
        if (kind == BEM_RHS_PLANE) {
            sincos(k * (px * x + py * y + pz * z), &sn, &cs);
            ir = amp * cs;
            ii = -amp * sn;
        } else if (amp != 0.0) {
            const double dx = x - px, dy = y - py, dz = z - pz;
            const double rr = sqrt(dx * dx + dy * dy + dz * dz);
            sincos(k * rr, &sn, &cs);
            ir = amp * cs / (4.0 * kPi * rr);
            ii = -amp * sn / (4.0 * kPi * rr);
        }
    }
    out[(size_t)r * ldo + __float_as_int(xp.w)] = make_float2((float)(ir - sr), (float)(ii - si));
}

size_t field_part_bytes(int E, int P, int R) {
    return sizeof(float2) * (size_t)((E + kFieldChunk - 1) / kFieldChunk) * R * P;
}

// Queues the field on s: params (3 R, or null: no incident field) and part
// (field_part_bytes) on the device; nothing is allocated, no wait.
int field_run(const DeviceProblem &dp, float k, const float4 *xs, int P, const float2 *X, long ldx, int R, int kind,
              double amp, const float *params, float2 *part, float2 *out, long ldo, hipStream_t s) {
    const Config &cfg = config();
    const int nch = (dp.E + kFieldChunk - 1) / kFieldChunk;
    FieldArgs a;
    a.xs = xs;
    a.recs = dp.rec64;
    a.far = dp.far32;
    a.X = X;
    a.ldx = ldx;
    a.part = part;
    a.P = P;
    a.E = dp.E;
    a.R = R;
    a.k = k;
    a.kf = (float)((double)k / (2.0 * kPi));
    a.kf64 = (double)k / (2.0 * kPi);
    a.rw = (float)((double)cfg.density * (double)(k * cfg.speed));
    far_limits((double)k, kFarK2, a.far_rho2, a.far7_rho2);
    TimedRegion tr;
    timing_begin(tr, "field_part", s);
    for (int r0 = 0; r0 < R; r0 += kFieldR) {
        a.r0 = r0;
        const dim3 grid((P + 63) / 64, nch), block(64 * kFieldWaves);
        if (R - r0 == 1) field_part<1><<<grid, block, 0, s>>>(a);
        else if (R - r0 <= 4) field_part<4><<<grid, block, 0, s>>>(a);
        else field_part<kFieldR><<<grid, block, 0, s>>>(a);
        HIP_CALL(hipGetLastError());
    }
    timing_end(tr, s);
    field_finalize<<<dim3((P + 15) / 16, R), 256, 0, s>>>(xs, P, R, nch, part, (double)k, kind, amp, params, out, ldo);
    HIP_CALL(hipGetLastError());
    return EXIT_SUCCESS;
}

// Points in the order of a Z-curve through 32^3 cells of a box (lo, and cells per
// length inv); points outside go to its outer cells, and so does a NaN.  Each point
// takes the rule that its own distance to an element asks for, so a wave of points
// from all over the body runs every rule on most elements; a point's value is the
// same in any order.
constexpr int kCells = 1 << 15;
struct CellBox {
    float lo[3], inv[3];
};
__global__ void k_cell_count(const float4 *__restrict__ xs, int P, CellBox b, int *__restrict__ cell,
                             int *__restrict__ count) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const float x[3] = {xs[p].x, xs[p].y, xs[p].z};
    int z = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float t = (x[d] - b.lo[d]) * b.inv[d];
        const int c = t >= 31.f ? 31 : t > 0.f ? (int)t : 0;
#pragma unroll
        for (int q = 0; q < 5; q++) z |= ((c >> q) & 1) << (3 * q + d);
    }
    cell[p] = z;
    atomicAdd(&count[z], 1);
}
// counts to first places, one workgroup
__global__ __launch_bounds__(1024) void k_cell_scan(int *count) {
    __shared__ int s[1024];
    const int t = threadIdx.x;
    int c[kCells / 1024], sum = 0;
#pragma unroll
    for (int i = 0; i < kCells / 1024; i++) {
        c[i] = count[t * (kCells / 1024) + i];
        sum += c[i];
    }
    s[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d *= 2) {
        const int v = t >= d ? s[t - d] : 0;
        __syncthreads();
        s[t] += v;
        __syncthreads();
    }
    int at = s[t] - sum;
#pragma unroll
    for (int i = 0; i < kCells / 1024; i++) {
        count[t * (kCells / 1024) + i] = at;
        at += c[i];
    }
}
__global__ void k_cell_place(const float4 *__restrict__ xs, int P, const int *__restrict__ cell,
                             int *__restrict__ at, float4 *__restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < P) out[atomicAdd(&at[cell[p]], 1)] = xs[p];
}
__global__ void k_zero_int(int *v, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = 0;
}

// Whether the points are sorted: from 4e6 pairs on (30 us of launches) and 256
// elements (of fewer, most are near to most points in any order), with one point at
// least within the 12-point rule's distance (8 rho) of the body's box.  Points at
// 1.05 radii in random order, in the order given and sorted: 2562 nodes, 1030: 0.43 and
// 0.35 ms, 30000: 8.4 and 2.7 (6.6 with 36 points everywhere); 642 nodes, 3200: 0.40
// and 0.29; 162, 13000: 0.41 and 0.33; 42, 60000: 0.47 and 0.56.
static bool field_sorts(const DeviceProblem &dp, const bem_cart_coord *pts, int P) {
    if (dp.E < 256 || (double)dp.E * P < 4e6) return false;
    const double m = std::sqrt((double)kFar12D2) * dp.rho;
    float lo[3], hi[3];
    for (int d = 0; d < 3; d++) {
        lo[d] = (float)(dp.nlo[d] - m);
        hi[d] = (float)(dp.nhi[d] + m);
    }
    for (int p = 0; p < P; p++) {
        const float *x = pts[p].coords;
        if (x[0] > lo[0] && x[0] < hi[0] && x[1] > lo[1] && x[1] < hi[1] && x[2] > lo[2] && x[2] < hi[2]) return true;
    }
    return false;
}

int field_fp32(DeviceProblem &dp, float k, const float4 *xs, const bem_cart_coord *pts, int P, const float2 *X,
               long ldx, int R, const RhsSpec &rhs, float2 *out, long ldo, hipStream_t s) {
    if (P <= 0 || R <= 0) return EXIT_SUCCESS;
    // (one allocation: smaller ones beside it may be cut out of the block that its
    // last use left, which then has to be mapped anew, 1 ms for 77 MB)
    bool sort = field_sorts(dp, pts, P);
    const size_t pbytes = (field_part_bytes(dp.E, P, R) + 255) / 256 * 256;
    char *mem = nullptr;
    float *params = nullptr;
    if (sort && hipMallocAsync((void **)&mem, pbytes + sizeof(float4) * P + sizeof(int) * ((size_t)P + kCells), s) !=
                    hipSuccess) {
        (void)hipGetLastError();
        mem = nullptr;
        sort = false;  // (no room: the order given)
    }
    if (!mem) HOST_CALL(salloc(&mem, pbytes, s));
    float2 *part = (float2 *)mem;
    if (sort) {
        float4 *sorted = (float4 *)(mem + pbytes);
        int *cell = (int *)(sorted + P);
        CellBox b;
        for (int d = 0; d < 3; d++) {
            const double m = std::sqrt((double)kFar7D2) * dp.rho, w = dp.nhi[d] - dp.nlo[d] + 2 * m;
            b.lo[d] = (float)(dp.nlo[d] - m);
            b.inv[d] = w > 0 ? (float)(32.0 / w) : 0.f;
        }
        int *count = cell + P;
        k_zero_int<<<kCells / 1024, 1024, 0, s>>>(count, kCells);
        k_cell_count<<<(P + 255) / 256, 256, 0, s>>>(xs, P, b, cell, count);
        k_cell_scan<<<1, 1024, 0, s>>>(count);
        k_cell_place<<<(P + 255) / 256, 256, 0, s>>>(xs, P, cell, count, sorted);
        xs = sorted;
    }
    if (!rhs.params.empty()) {
        HOST_CALL(salloc(&params, rhs.params.size(), s));
        HIP_CALL(hipMemcpyAsync(params, rhs.params.data(), rhs.params.size() * sizeof(float), hipMemcpyHostToDevice, s));
    }
    const int rc = field_run(dp, k, xs, P, X, ldx, R, rhs.kind, (double)rhs.amp, rhs.nrhs >= R ? params : nullptr, part,
                             out, ldo, s);
    (void)hipStreamSynchronize(s);
    sfree(mem, s);
    sfree(params, s);
    return rc;
}

// ------------------------------------------- near-singular, FP64 ---
// The reference integrates every element that does not hold the collocation
// point with the 6x6 collapsed rule (g_h_c_l_nsgl, mesh.cu:597-672; the only
// exclusion is the vertex test, atomicFuncs.cu:75-76).  For a point closer to
// the element than about its size the integrand peaks inside the element and
// the rule's error grows to 1e-3 at a quarter of the element size.  With
// bem_set_near_field on, every (row, element) pair closer than a factor times
// the element's longest edge gets an FP64 correction
//     delta = (integral by adaptive subdivision) - (the 6x6 rule in FP64),
// added to the assembled entries after the row-owned assembly, in a fixed
// order per row.  The subdivision splits a triangle into four at its edge
// midpoints, depth first; a sub-triangle is integrated with the same 6x6
// collapsed rule once its distance from the point (centroid distance minus
// circumradius) is at least kNearEta times its longest edge, or at the depth
// limit.  The path through the quadtree is kept as two bits per level, so the
// walk needs no stack: each sub-triangle is rebuilt from the root.
constexpr double kNearEta = 1.5;
constexpr int kNearOut = 13;  // g (3 complex), h (3 complex), c

struct NearArgs {
    const double *__restrict__ pts64;  // 3 M: nodes then extra rows
    const int *__restrict__ elems;     // 3 E
    const int *__restrict__ row;       // per pair
    const int *__restrict__ elem;      // per pair
    int p0, p1;                        // pairs [p0, p1)
    int levels;
    double k, rw;                      // k, rho omega
    double qu[kNQ], qv[kNQ], qw[kNQ];  // 6x6 collapsed rule on the unit triangle: (u, v) and weight
    double *__restrict__ out;
};

struct NearAcc {
    double gr[3], gi[3], hr[3], hi[3], c;
};

// the collapsed rule over the sub-triangle (a, b, c) of the element's
// (xi1, xi2) plane, scaled by its area ratio `det`; y = p3 + xi1 e1 + xi2 e2
__device__ void near_leaf(const NearArgs &a, const double *x, const double *p3, const double *e1, const double *e2,
                          const double *n, double J, const double *va, const double *vb, const double *vc,
                          double det, NearAcc &acc) {
    const double inv4pi = 1.0 / (4.0 * kPi);
    for (int q = 0; q < kNQ; q++) {
        const double u = a.qu[q], v = a.qv[q];
        const double xi1 = vc[0] + u * (va[0] - vc[0]) + v * (vb[0] - vc[0]);
        const double xi2 = vc[1] + u * (va[1] - vc[1]) + v * (vb[1] - vc[1]);
        const double N[3] = {xi1, xi2, 1.0 - xi1 - xi2};
        double rv[3];
        for (int d = 0; d < 3; d++) rv[d] = p3[d] + xi1 * e1[d] + xi2 * e2[d] - x[d];
        const double r2 = rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2];
        const double r = sqrt(r2);
        const double prpn2 = (rv[0] * n[0] + rv[1] * n[1] + rv[2] * n[2]) / r;  // dr/dn_y
        double sn, cs;
        sincos(a.k * r, &sn, &cs);
        const double w = a.qw[q] * det * J;
        // G = exp(-ikr) / (4 pi r); dG/dn = G (-1/r - ik) dr/dn; dG0/dn = -dr/dn / (4 pi r^2)
        const double Gr = cs * inv4pi / r, Gi = -sn * inv4pi / r;
        const double Hr = (Gr * (-1.0 / r) + Gi * a.k) * prpn2;
        const double Hi = (Gi * (-1.0 / r) - Gr * a.k) * prpn2;
        for (int j = 0; j < 3; j++) {
            acc.gr[j] += w * N[j] * Gr;
            acc.gi[j] += w * N[j] * Gi;
            acc.hr[j] += w * N[j] * Hr;
            acc.hi[j] += w * N[j] * Hi;
        }
        acc.c += -w * prpn2 * inv4pi / r2;
    }
}

// One thread per pair: delta = adaptive - rule, with g scaled by i rho omega
// as the reference scales it (mesh.cu:668-670).
__global__ __launch_bounds__(64) void near_elems(NearArgs a) {
    const int id = a.p0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= a.p1) return;
    const int e = a.elem[id], row = a.row[id];
    double x[3], p[3][3];
    for (int d = 0; d < 3; d++) x[d] = a.pts64[3 * (size_t)row + d];
    for (int j = 0; j < 3; j++)
        for (int d = 0; d < 3; d++) p[j][d] = a.pts64[3 * (size_t)a.elems[3 * e + j] + d];
    double e1[3], e2[3];
    for (int d = 0; d < 3; d++) {
        e1[d] = p[0][d] - p[2][d];
        e2[d] = p[1][d] - p[2][d];
    }
    const double cr[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    const double J = sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    const double n[3] = {cr[0] / J, cr[1] / J, cr[2] / J};
    const double A0[2] = {1.0, 0.0}, B0[2] = {0.0, 1.0}, C0[2] = {0.0, 0.0};
    NearAcc rule = {}, ad = {};
    near_leaf(a, x, p[2], e1, e2, n, J, A0, B0, C0, 1.0, rule);
    // depth-first walk of the quadtree; digits of the path, 2 bits per level
    unsigned long long path = 0;
    int level = 0;
    for (;;) {
        double va[2] = {1.0, 0.0}, vb[2] = {0.0, 1.0}, vc[2] = {0.0, 0.0};
        for (int l = 1; l <= level; l++) {
            const int dgt = (int)((path >> (2 * (l - 1))) & 3);
            const double ab[2] = {0.5 * (va[0] + vb[0]), 0.5 * (va[1] + vb[1])};
            const double bc[2] = {0.5 * (vb[0] + vc[0]), 0.5 * (vb[1] + vc[1])};
            const double ca[2] = {0.5 * (vc[0] + va[0]), 0.5 * (vc[1] + va[1])};
            double na[2], nb[2], nc[2];
            if (dgt == 0) { na[0] = va[0]; na[1] = va[1]; nb[0] = ab[0]; nb[1] = ab[1]; nc[0] = ca[0]; nc[1] = ca[1]; }
            else if (dgt == 1) { na[0] = ab[0]; na[1] = ab[1]; nb[0] = vb[0]; nb[1] = vb[1]; nc[0] = bc[0]; nc[1] = bc[1]; }
            else if (dgt == 2) { na[0] = ca[0]; na[1] = ca[1]; nb[0] = bc[0]; nb[1] = bc[1]; nc[0] = vc[0]; nc[1] = vc[1]; }
            else { na[0] = bc[0]; na[1] = bc[1]; nb[0] = ca[0]; nb[1] = ca[1]; nc[0] = ab[0]; nc[1] = ab[1]; }
            va[0] = na[0]; va[1] = na[1]; vb[0] = nb[0]; vb[1] = nb[1]; vc[0] = nc[0]; vc[1] = nc[1];
        }
        // physical vertices, centroid distance, circumradius bound, longest edge
        double Y[3][3], cen[3] = {0, 0, 0};
        const double *vv[3] = {va, vb, vc};
        for (int t = 0; t < 3; t++)
            for (int d = 0; d < 3; d++) {
                Y[t][d] = p[2][d] + vv[t][0] * e1[d] + vv[t][1] * e2[d];
                cen[d] += Y[t][d] / 3.0;
            }
        double rad = 0, diam = 0;
        for (int t = 0; t < 3; t++) {
            double q = 0, s = 0;
            for (int d = 0; d < 3; d++) {
                q += (Y[t][d] - cen[d]) * (Y[t][d] - cen[d]);
                s += (Y[t][d] - Y[(t + 1) % 3][d]) * (Y[t][d] - Y[(t + 1) % 3][d]);
            }
            rad = fmax(rad, sqrt(q));
            diam = fmax(diam, sqrt(s));
        }
        const double dc = sqrt((x[0] - cen[0]) * (x[0] - cen[0]) + (x[1] - cen[1]) * (x[1] - cen[1]) +
                               (x[2] - cen[2]) * (x[2] - cen[2]));
        if (level >= a.levels || dc - rad >= kNearEta * diam) {
            near_leaf(a, x, p[2], e1, e2, n, J, va, vb, vc, ldexp(1.0, -2 * level), ad);
            // next sibling, climbing past last children
            while (level > 0 && ((path >> (2 * (level - 1))) & 3) == 3) {
                path &= ~(3ull << (2 * (level - 1)));
                level--;
            }
            if (level == 0) break;
            path += 1ull << (2 * (level - 1));
        } else {
            level++;  // first child: digit 0
        }
    }
    double *o = a.out + (size_t)id * kNearOut;
    // g_j = i rho omega int N_j G
    for (int j = 0; j < 3; j++) {
        const double dgr = ad.gr[j] - rule.gr[j], dgi = ad.gi[j] - rule.gi[j];
        o[2 * j] = -a.rw * dgi;
        o[2 * j + 1] = a.rw * dgr;
        o[6 + 2 * j] = ad.hr[j] - rule.hr[j];
        o[6 + 2 * j + 1] = ad.hi[j] - rule.hi[j];
    }
    o[12] = ad.c - rule.c;
}

// One thread per row r0 + i: the row's pair corrections in pair order,
// A[i, node_j] += dh_j - (ca/cb) dg_j, A[i, i] -= dc on node rows,
// bterm[i] += (cc/cb) sum_j dg_j (atomicFuncs.cu:86-115 for the corrections)
template <typename R, typename C2>
__global__ void near_apply(C2 *A, long ldA, int M, int N, int r0, const int *__restrict__ ptr,
                           const int *__restrict__ elem, const int *__restrict__ elems, const float2 *__restrict__ bc,
                           const double *__restrict__ d, double2 *__restrict__ bterm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = r0 + i;
    if (row >= M) return;
    double btr = 0, bti = 0, dc = 0;
    for (int q = ptr[row]; q < ptr[row + 1]; q++) {
        const int e = elem[q];
        const double *o = d + (size_t)q * kNearOut;
        const float2 ca = bc[3 * e], cb = bc[3 * e + 1], cc = bc[3 * e + 2];
        const double den = (double)cb.x * cb.x + (double)cb.y * cb.y;
        const double br = ((double)ca.x * cb.x + (double)ca.y * cb.y) / den;
        const double bi = ((double)ca.y * cb.x - (double)ca.x * cb.y) / den;
        const double gr = ((double)cc.x * cb.x + (double)cc.y * cb.y) / den;
        const double gi = ((double)cc.y * cb.x - (double)cc.x * cb.y) / den;
        double sgr = 0, sgi = 0;
        for (int j = 0; j < 3; j++) {
            const double dgr = o[2 * j], dgi = o[2 * j + 1];
            const double pr = o[6 + 2 * j] - (br * dgr - bi * dgi);
            const double pi = o[6 + 2 * j + 1] - (br * dgi + bi * dgr);
            C2 *a = A + (size_t)elems[3 * e + j] * ldA + i;
            C2 v = *a;
            v.x = (R)((double)v.x + pr);
            v.y = (R)((double)v.y + pi);
            *a = v;
            sgr += dgr;
            sgi += dgi;
        }
        btr += gr * sgr - gi * sgi;
        bti += gr * sgi + gi * sgr;
        dc += o[12];
    }
    if (row < N && dc != 0.0) {
        C2 *a = A + (size_t)row * ldA + i;
        C2 v = *a;
        v.x = (R)((double)v.x - dc);
        *a = v;
    }
    double2 b = bterm[i];
    b.x += btr;
    b.y += bti;
    bterm[i] = b;
}

namespace {
// distance from x to the triangle (a, b, c): closest point by the regions of
// the plane around the triangle (the vertex, edge and face regions of the
// barycentric test)
double point_triangle_distance(const double *x, const double *a, const double *b, const double *c) {
    auto sub = [](const double *u, const double *v, double *o) {
        for (int d = 0; d < 3; d++) o[d] = u[d] - v[d];
    };
    auto dot = [](const double *u, const double *v) { return u[0] * v[0] + u[1] * v[1] + u[2] * v[2]; };
    double ab[3], ac[3], ap[3], bp[3], cp[3], q[3];
    sub(b, a, ab);
    sub(c, a, ac);
    sub(x, a, ap);
    auto dist_to = [&](const double *y) {
        return std::sqrt((x[0] - y[0]) * (x[0] - y[0]) + (x[1] - y[1]) * (x[1] - y[1]) + (x[2] - y[2]) * (x[2] - y[2]));
    };
    auto on = [&](const double *o, const double *dir, double t) {
        for (int d = 0; d < 3; d++) q[d] = o[d] + t * dir[d];
        return dist_to(q);
    };
    const double d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0 && d2 <= 0) return dist_to(a);
    sub(x, b, bp);
    const double d3 = dot(ab, bp), d4 = dot(ac, bp);
    if (d3 >= 0 && d4 <= d3) return dist_to(b);
    const double vc = d1 * d4 - d3 * d2;
    if (vc <= 0 && d1 >= 0 && d3 <= 0) return on(a, ab, d1 / (d1 - d3));
    sub(x, c, cp);
    const double d5 = dot(ab, cp), d6 = dot(ac, cp);
    if (d6 >= 0 && d5 <= d6) return dist_to(c);
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0 && d2 >= 0 && d6 <= 0) return on(a, ac, d2 / (d2 - d6));
    const double va = d3 * d6 - d5 * d4;
    if (va <= 0 && (d4 - d3) >= 0 && (d5 - d6) >= 0) {
        double bc[3];
        sub(c, b, bc);
        return on(b, bc, (d4 - d3) / ((d4 - d3) + (d5 - d6)));
    }
    const double den = 1.0 / (va + vb + vc);
    const double v = vb * den, w = vc * den;
    for (int d = 0; d < 3; d++) q[d] = a[d] + ab[d] * v + ac[d] * w;
    return dist_to(q);
}
}  // namespace

// (row, element) pairs with dist(x_row, element) < factor * (longest edge),
// the element not holding the row's node; sorted by row, then element.  A
// uniform grid over the element centroids, cells as wide as the largest
// reach, bounds the search to the 27 cells around each row point.
void near_pairs(const std::vector<double> &pts, int M, int N, const std::vector<int> &elems, double factor,
                std::vector<int> &ptr, std::vector<int> &prow, std::vector<int> &pelem) {
    const int E = (int)(elems.size() / 3);
    std::vector<double> cen(3 * (size_t)E), reach(E), hmax(E);
    double cell = 0, lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int e = 0; e < E; e++) {
        const double *v[3] = {&pts[3 * (size_t)elems[3 * e]], &pts[3 * (size_t)elems[3 * e + 1]],
                              &pts[3 * (size_t)elems[3 * e + 2]]};
        double h = 0, r = 0;
        for (int d = 0; d < 3; d++) cen[3 * e + d] = (v[0][d] + v[1][d] + v[2][d]) / 3.0;
        for (int t = 0; t < 3; t++) {
            double s = 0, q = 0;
            for (int d = 0; d < 3; d++) {
                s += (v[t][d] - v[(t + 1) % 3][d]) * (v[t][d] - v[(t + 1) % 3][d]);
                q += (v[t][d] - cen[3 * e + d]) * (v[t][d] - cen[3 * e + d]);
            }
            h = std::max(h, std::sqrt(s));
            r = std::max(r, std::sqrt(q));
        }
        hmax[e] = h;
        reach[e] = r + factor * h;
        cell = std::max(cell, reach[e]);
        for (int d = 0; d < 3; d++) {
            lo[d] = std::min(lo[d], cen[3 * e + d]);
            hi[d] = std::max(hi[d], cen[3 * e + d]);
        }
    }
    cell = std::max(cell, 1e-30);
    int nc[3];
    for (int d = 0; d < 3; d++) nc[d] = std::max(1, std::min(1024, (int)((hi[d] - lo[d]) / cell) + 1));
    auto cell_of = [&](const double *y, int *c) {
        for (int d = 0; d < 3; d++) c[d] = std::max(0, std::min(nc[d] - 1, (int)((y[d] - lo[d]) / cell)));
    };
    std::vector<std::vector<int>> grid((size_t)nc[0] * nc[1] * nc[2]);
    for (int e = 0; e < E; e++) {
        int c[3];
        cell_of(&cen[3 * e], c);
        grid[((size_t)c[0] * nc[1] + c[1]) * nc[2] + c[2]].push_back(e);
    }
    ptr.assign((size_t)M + 1, 0);
    prow.clear();
    pelem.clear();
    std::vector<int> found;
    for (int i = 0; i < M; i++) {
        const double *x = &pts[3 * (size_t)i];
        int c[3];
        cell_of(x, c);
        found.clear();
        for (int a = std::max(0, c[0] - 1); a <= std::min(nc[0] - 1, c[0] + 1); a++)
            for (int b = std::max(0, c[1] - 1); b <= std::min(nc[1] - 1, c[1] + 1); b++)
                for (int z = std::max(0, c[2] - 1); z <= std::min(nc[2] - 1, c[2] + 1); z++)
                    for (int e : grid[((size_t)a * nc[1] + b) * nc[2] + z]) {
                        const int *n = &elems[3 * e];
                        if (i < N && (n[0] == i || n[1] == i || n[2] == i)) continue;  // singular rule
                        const double dc = std::sqrt((x[0] - cen[3 * e]) * (x[0] - cen[3 * e]) +
                                                    (x[1] - cen[3 * e + 1]) * (x[1] - cen[3 * e + 1]) +
                                                    (x[2] - cen[3 * e + 2]) * (x[2] - cen[3 * e + 2]));
                        if (dc >= reach[e]) continue;
                        const double d = point_triangle_distance(x, &pts[3 * (size_t)n[0]], &pts[3 * (size_t)n[1]],
                                                                 &pts[3 * (size_t)n[2]]);
                        if (d < factor * hmax[e]) found.push_back(e);
                    }
        std::sort(found.begin(), found.end());
        for (int e : found) {
            prow.push_back(i);
            pelem.push_back(e);
        }
        ptr[i + 1] = (int)prow.size();
    }
}

// the pairs of the device problem for the current bem_set_near_field setting
static int near_prepare(DeviceProblem &dp, hipStream_t s) {
    const Config &cfg = config();
    if (cfg.near_factor == dp.near_factor && cfg.near_levels == dp.near_levels) return EXIT_SUCCESS;
    sfree(dp.near_ptr, s);
    sfree(dp.near_row, s);
    sfree(dp.near_elem, s);
    sfree(dp.near_out, s);
    dp.near_npairs = 0;
    dp.hnear_ptr.clear();
    dp.near_factor = cfg.near_factor;
    dp.near_levels = cfg.near_levels;
    if (cfg.near_factor <= 0) return EXIT_SUCCESS;
    std::vector<int> prow, pelem;
    near_pairs(dp.hpts, dp.M, dp.N, dp.helems, cfg.near_factor, dp.hnear_ptr, prow, pelem);
    dp.near_npairs = (int)prow.size();
    HOST_CALL(salloc(&dp.near_ptr, dp.hnear_ptr.size(), s));
    HOST_CALL(salloc(&dp.near_row, std::max<size_t>(1, prow.size()), s));
    HOST_CALL(salloc(&dp.near_elem, std::max<size_t>(1, pelem.size()), s));
    HOST_CALL(salloc(&dp.near_out, std::max<size_t>(1, prow.size()) * kNearOut, s));
    HIP_CALL(hipMemcpyAsync(dp.near_ptr, dp.hnear_ptr.data(), dp.hnear_ptr.size() * sizeof(int), hipMemcpyHostToDevice,
                            s));
    if (!prow.empty()) {
        HIP_CALL(hipMemcpyAsync(dp.near_row, prow.data(), prow.size() * sizeof(int), hipMemcpyHostToDevice, s));
        HIP_CALL(hipMemcpyAsync(dp.near_elem, pelem.data(), pelem.size() * sizeof(int), hipMemcpyHostToDevice, s));
    }
    HIP_CALL(hipStreamSynchronize(s));  // the host vectors go out of scope
    return EXIT_SUCCESS;
}

// corrections of rows r0..M-1 of A (ld ldA, row r0 first) and their bterm
template <typename R, typename C2>
static int near_correct(DeviceProblem &dp, double k, double rw, C2 *A, long ldA, int r0, double2 *bterm,
                        hipStream_t s) {
    HOST_CALL(near_prepare(dp, s));
    if (dp.near_npairs == 0) return EXIT_SUCCESS;
    const int p0 = dp.hnear_ptr[r0], p1 = dp.hnear_ptr[dp.M];
    if (p1 > p0) {
        NearArgs a;
        a.pts64 = dp.pts64;
        a.elems = dp.elems;
        a.row = dp.near_row;
        a.elem = dp.near_elem;
        a.p0 = p0;
        a.p1 = p1;
        a.levels = dp.near_levels;
        a.k = k;
        a.rw = rw;
        const Config &cfg = config();
        for (int n = 0; n < kQOrder; n++) {
            const double theta = 0.5 + 0.5 * cfg.qp[n];
            for (int m = 0; m < kQOrder; m++) {
                const double rho = 0.5 + 0.5 * cfg.qp[m];
                const int q = n * kQOrder + m;
                a.qu[q] = rho * (1 - theta);  // xi1 = rho (1 - theta), xi2 = rho theta (mesh.cu:623-636)
                a.qv[q] = rho * theta;
                a.qw[q] = 0.25 * cfg.qw[n] * cfg.qw[m] * rho;
            }
        }
        a.out = dp.near_out;
        TimedRegion tr;
        timing_begin(tr, "near_elems", s);
        near_elems<<<(p1 - p0 + 63) / 64, 64, 0, s>>>(a);
        HIP_CALL(hipGetLastError());
        timing_end(tr, s);
    }
    const int nrows = dp.M - r0;
    near_apply<R, C2><<<(nrows + 255) / 256, 256, 0, s>>>(A, ldA, dp.M, dp.N, r0, dp.near_ptr, dp.near_elem, dp.elems,
                                                        dp.bc, dp.near_out, bterm);
    HIP_CALL(hipGetLastError());
    return EXIT_SUCCESS;
}

// ------------------------------------------- field without allocations ---
// The exterior field for callers that cannot allocate device memory (code
// under HIP graph capture, serving loops): the partial sums, the points in
// the kernels' float4 layout and the source point live in one file-scope
// device array of fixed size.  Each device holds its own copy of the array;
// host code reaches it only through the address hipGetSymbolAddress returns
// on that device, kept per device below.  Every call on a device shares that
// device's array, so calls that overlap on one device race.
constexpr size_t kNoAllocScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// the scratch array's device address on the current device (looked up once per device)
int scratch_address(void **out) {
    int dev = 0;
    HIP_CALL(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) BEM_FAIL("device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        HIP_CALL(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) BEM_FAIL("no device address for the scratch array");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return EXIT_SUCCESS;
}

size_t round256(size_t b) { return (b + 255) / 256 * 256; }
}  // namespace

// 12-byte points (cartCoord) to the kernels' float4 layout, and the
// incident point source's position next to them
__global__ void k_pack_field_points(const float *__restrict__ xs, int P, float4 *__restrict__ xs4, float sx, float sy,
                                    float sz, float *__restrict__ params) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < P) xs4[p] = make_float4(xs[3 * p], xs[3 * p + 1], xs[3 * p + 2], __int_as_float(p));
    if (p == 0) {
        params[0] = sx;
        params[1] = sy;
        params[2] = sz;
    }
}

size_t field_noalloc_bytes(int E, int P) {
    const size_t nch = (size_t)(E + kFieldChunk - 1) / kFieldChunk;
    return round256(sizeof(float4) * (size_t)P) + 256 + sizeof(float2) * nch * (size_t)P;
}

size_t field_noalloc_capacity() { return kNoAllocScratchBytes; }

int field_fp32_noalloc(const DeviceProblem &dp, float k, const float *xs, int P, const float2 *X, float strength,
                       const float *src, float2 *out, hipStream_t s) {
    if (P <= 0) return EXIT_SUCCESS;
    const size_t need = field_noalloc_bytes(dp.E, P);
    if (need > kNoAllocScratchBytes)
        BEM_FAIL("%d field points on %d elements need %zu bytes of scratch, more than its %zu", P, dp.E, need,
                 kNoAllocScratchBytes);
    void *base = nullptr;
    HOST_CALL(scratch_address(&base));
    unsigned char *b = (unsigned char *)base;
    float4 *xs4 = (float4 *)b;
    float *params = (float *)(b + round256(sizeof(float4) * (size_t)P));
    float2 *part = (float2 *)(b + round256(sizeof(float4) * (size_t)P) + 256);
    k_pack_field_points<<<(P + 255) / 256, 256, 0, s>>>(xs, P, xs4, src[0], src[1], src[2], params);
    HIP_CALL(hipGetLastError());
    return field_run(dp, k, xs4, P, X, dp.N, 1, BEM_RHS_POINT, (double)strength, params, part, out, P, s);
}

// --------------------------------------------------------------- host ---
// Launch shape of the assembly: qg lanes per row (1 or 4) and P column tiles,
// P x ceil(M / (64 / qg)) waves in all.  More tiles cost more halo elements
// (an element straddling tiles is integrated once per tile) but give more
// waves to balance over the 1024 SIMDs; the default aims at kDefaultWaves.
// bem_autotune_assembly times candidate shapes for a mesh on the device and
// records the fastest for its size class (M and E in half-octave buckets),
// which device problems of that class built afterwards use.
constexpr int kDefaultWaves = 16384;

namespace {
struct TileShape {
    int qg = 0, waves = 0;
};
std::mutex g_tune_mu;
std::map<std::pair<int, int>, TileShape> g_tune;
thread_local const TileShape *t_force = nullptr;  // candidate under test
thread_local bool t_untuned = false;              // no shape asked for, whatever the table holds

int half_octave(long v) { return (int)std::lround(2.0 * std::log2((double)std::max(1L, v))); }

bool tuned_shape(int M, int E, TileShape &out) {
    if (t_untuned) return false;
    if (t_force) {
        out = *t_force;
        return true;
    }
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find({half_octave(M), half_octave(E)});
    if (it == g_tune.end()) return false;
    out = it->second;
    return true;
}
}  // namespace

// halo share (elements integrated per element) from which the element-once
// plan is taken
constexpr double kGhostMinDup = 1.05;

// side columns the element-once plan may use: about the nodes on the tile
// boundaries (4 sqrt(N P) + P; 4190 for N = 10242 in 102 tiles, which need
// 3110), and never more than 2 N.  (A bound of N / 2 kept meshes of a few
// thousand nodes on fewer, longer tiles: 2562 nodes took 0.41 ms in 53 tiles,
// 0.27 ms in 320; 642 nodes 0.23 ms in 35, 0.064 ms in 160.)
static long ghost_slot_bound(int N, int P) {
    return std::min(2L * N, (long)(4.0 * std::sqrt((double)N * P)) + P);
}

// wave_factor: the element-once plan has no halo to pay for more tiles, and
// runs at twice the waves (10242 nodes: 2.16 ms with 102 tiles, 1.90 with
// 204).  A wave walks its tile's list alone, so on a small mesh the longest
// list is the assembly's time, and tiles go down to a few nodes.
static int choose_tiles(int M, int N, int E, int rows_per_wave, int wave_factor = 1) {
    const char *env = getenv("BEM_TILES");
    if (env && atoi(env) > 0) return std::min(atoi(env), N);
    TileShape t;
    const int target_waves = (tuned_shape(M, E, t) ? t.waves : kDefaultWaves) * wave_factor;
    const int nrb = (M + rows_per_wave - 1) / rows_per_wave;
    int P = (target_waves + nrb - 1) / nrb;
    // nodes per tile of the element-once plan: 4 below 1000 nodes, 8 up to 320
    // tiles, then 16 (4002 nodes: 0.536 ms in 320 tiles, 0.556 in 640, with
    // twice the side columns)
    const int most = wave_factor == 1 ? N / 8 : N < 1000 ? N / 4 : std::min(N / 8, std::max(320, N / 16));
    P = std::max(1, std::min(P, std::max(1, most)));
    return P;
}

// lanes per row asked for by the environment or the tuner; 0: none
static int asked_qg(int M, int E) {
    const char *env = getenv("BEM_QG");
    if (env) {
        int q = atoi(env);
        if (q == 1 || q == 4) return q;
    }
    TileShape t;
    return tuned_shape(M, E, t) ? t.qg : 0;
}

// lanes per row of the halo plan's kernels.  (FP32 runs the element-once plan
// with one lane a row at every size it can be built for: 642 nodes 0.064 ms
// against 0.122 ms with four lanes, 162 nodes 0.05 against 0.066 ms.)
static int choose_qg(int M, int E) {
    const int q = asked_qg(M, E);
    return q ? q : ((long)M * E < 4000000L) ? 4 : 1;
}

// Times the FP32 (or FP64) assembly of mesh m at wavenumber k for each
// candidate shape (2 warm + 3 timed launches each, HIP events on stream s)
// and records the fastest for the mesh's size class.
int autotune_assembly(const Mesh &m, double k, int precision, int *best_qg, int *best_waves, double *best_ms,
                      double *default_ms, hipStream_t s) {
    const int M = m.N() + m.C(), E = m.E();
    std::vector<TileShape> cand;
    for (int qg : {1, 4})
        for (int w : {4096, 8192, 16384, 32768}) cand.push_back(TileShape{qg, w});
    // the shape of an untuned build
    TileShape def{1, kDefaultWaves};
    {
        DeviceProblem dp;
        t_untuned = true;
        const int rc = device_problem_build(m, dp, s);
        t_untuned = false;
        if (!dp.use_ghost) def.qg = dp.qg;
        device_problem_free(dp);
        HOST_CALL(rc);
    }
    double bms = 1e300, dms = -1;
    TileShape best = def;
    hipEvent_t e0, e1;
    HIP_CALL(hipEventCreate(&e0));
    HIP_CALL(hipEventCreate(&e1));
    size_t n = ((size_t)M + 63) / 64 * 64 * (size_t)m.N();
    void *A = nullptr;
    HIP_CALL(hipMallocAsync(&A, n * (precision == BEM_PREC_FP64 ? sizeof(double2) : sizeof(float2)), s));
    int rc = EXIT_SUCCESS;
    for (const TileShape &c : cand) {
        DeviceProblem dp;
        t_force = &c;
        rc = device_problem_build(m, dp, s);
        t_force = nullptr;
        if (rc != EXIT_SUCCESS) break;
        float ms = 0;
        for (int rep = 0; rep < 5 && rc == EXIT_SUCCESS; rep++) {
            if (rep == 2) (void)hipEventRecord(e0, s);
            rc = precision == BEM_PREC_FP64 ? assemble_fp64(dp, k, (double2 *)A, s)
                                            : assemble_fp32(dp, (float)k, (float2 *)A, s);
        }
        (void)hipEventRecord(e1, s);
        (void)hipEventSynchronize(e1);
        (void)hipEventElapsedTime(&ms, e0, e1);
        device_problem_free(dp);
        if (rc != EXIT_SUCCESS) break;
        const double avg = ms / 3.0;
        if (c.qg == def.qg && c.waves == def.waves) dms = avg;
        if (avg < bms) {
            bms = avg;
            best = c;
        }
    }
    (void)hipFreeAsync(A, s);
    (void)hipStreamSynchronize(s);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    HOST_CALL(rc);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune[{half_octave(M), half_octave(E)}] = best;
    }
    if (best_qg) *best_qg = best.qg;
    if (best_waves) *best_waves = best.waves;
    if (best_ms) *best_ms = bms;
    if (default_ms) *default_ms = dms;
    return EXIT_SUCCESS;
}

// The tuned shapes as text lines: "M-bucket E-bucket qg waves" for the
// assembly, then the products' "p ..." lines (gemm.hip), and back.
int tune_save(const char *file) {
    FILE *f = fopen(file, "w");
    if (!f) BEM_FAIL("cannot write %s", file);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        for (const auto &kv : g_tune)
            fprintf(f, "%d %d %d %d\n", kv.first.first, kv.first.second, kv.second.qg, kv.second.waves);
    }
    product_tune_save(f);
    fclose(f);
    return EXIT_SUCCESS;
}

int tune_load(const char *file) {
    FILE *f = fopen(file, "r");
    if (!f) BEM_FAIL("cannot read %s", file);
    char line[256];
    while (fgets(line, sizeof line, f)) {
        int a, b, q, w;
        if (product_tune_parse(line)) continue;
        if (sscanf(line, "%d %d %d %d", &a, &b, &q, &w) == 4 && (q == 1 || q == 4) && w > 0) {
            std::lock_guard<std::mutex> lk(g_tune_mu);
            g_tune[{a, b}] = TileShape{q, w};
        }
    }
    fclose(f);
    return EXIT_SUCCESS;
}

void tune_clear() {
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune.clear();
    }
    product_tune_clear();
}

// Upper bound of the HBM bytes that the problem of a mesh of M rows (nodes +
// CHIEF), N nodes and E elements and its assemblies in one precision allocate.
size_t device_problem_bytes(int M, int N, int E, bool fp64) {
    const size_t Mp = ((size_t)M + 63) / 64 * 64, real = fp64 ? sizeof(double) : sizeof(float);
    const int qg = choose_qg(M, E);
    const size_t P = (size_t)choose_tiles(M, N, E, 64 / qg);
    size_t b = 0;
    b += sizeof(float4) * M + sizeof(double) * 3 * M + sizeof(double2) * M;        // points, bterm
    b += (sizeof(int) + sizeof(float2)) * 3 * (size_t)E;                            // elements, bc
    b += (sizeof(ElemRec<float>) + sizeof(ElemRec<double>) + sizeof(FarRec)) * (size_t)E;  // element records
    b += real * 48 * (size_t)E;                                                      // singular terms
    b += sizeof(int) * (P + 1 + 3 * (size_t)E + N);                                  // tile CSR, isolated
    b += 40 * 256;                                                                   // the packed arrays' alignment
    size_t tiles = P, sides = 0;
    if (asked_qg(M, E) != 4) {
        // element-once plan: its side columns and index arrays
        const int gP = choose_tiles(M, N, E, 64, 2);
        sides = (size_t)ghost_slot_bound(N, gP);
        tiles = std::max(P, (size_t)gP);
        b += sizeof(int) * (gP + 1 + 4 * (size_t)E + 2 * (size_t)N + 2 * sides);
    }
    return b + real * (3 * tiles + 2 * sides) * Mp;  // tile partials, side columns
}

namespace {
// Arrays packed into one device allocation and, for those with host data, one
// copy: 27 allocations and 14 pageable copies were most of the time it took
// to set a small mesh up.  Every array starts at a multiple of 256 bytes;
// the ones with host data come first.
struct Pack {
    struct Item {
        void **dst;
        const void *src;
        size_t bytes;
    };
    std::vector<Item> items;
    template <typename T>
    void add(T **dst, const T *src, size_t n) {
        items.push_back(Item{(void **)dst, src, n * sizeof(T)});
    }
    // (the stream is waited for: the packed copy and its sources may go)
    int place(char **mem, hipStream_t s) {
        std::stable_partition(items.begin(), items.end(), [](const Item &i) { return i.src != nullptr; });
        size_t total = 0, up = 0;
        for (const Item &i : items) {
            total += (i.bytes + 255) / 256 * 256;
            if (i.src) up = total;
        }
        HOST_CALL(salloc(mem, std::max<size_t>(total, 256), s));
        std::vector<char> host(up);
        size_t at = 0;
        for (const Item &i : items) {
            *i.dst = *mem + at;
            if (i.src && i.bytes) memcpy(host.data() + at, i.src, i.bytes);
            at += (i.bytes + 255) / 256 * 256;
        }
        if (up) {
            HIP_CALL(hipMemcpyAsync(*mem, host.data(), up, hipMemcpyHostToDevice, s));
            HIP_CALL(hipStreamSynchronize(s));
        }
        return EXIT_SUCCESS;
    }
};

double diagonal(const double *lo, const double *hi) {
    double s = 0;
    for (int d = 0; d < 3; d++) s += (hi[d] - lo[d]) * (hi[d] - lo[d]);
    return std::sqrt(s);
}

// the halo plan's tiles on the device (built when a kernel that walks them runs)
int halo_plan(DeviceProblem &dp, hipStream_t s) {
    if (dp.P > 0) return EXIT_SUCCESS;
    Mesh m;
    m.pnts.resize(3 * (size_t)dp.N);
    for (size_t i = 0; i < m.pnts.size(); i++) m.pnts[i] = (float)dp.hpts[i];
    m.elems.resize(dp.E);
    for (int e = 0; e < dp.E; e++)
        for (int j = 0; j < 3; j++) m.elems[e].nodes[j] = dp.helems[3 * e + j];
    TilePlan plan;
    build_tile_plan(m, dp.hP, plan);
    Pack pk;
    pk.add(&dp.tile_ptr, (const int *)plan.ptr.data(), plan.ptr.size());
    pk.add(&dp.tile_entries, (const int *)plan.entries.data(), plan.entries.size());
    HOST_CALL(pk.place(&dp.halo_mem, s));
    dp.P = plan.P;
    return EXIT_SUCCESS;
}

// The arrays an assembly in R writes besides the matrix, one allocation per
// precision, grown when a plan of more tiles asks for it: the singular terms,
// the tile partials of c and the BC sums (P tiles), the side columns, for Mp
// rows at a time.
template <typename R>
int asm_scratch(DeviceProblem &dp, int P, long nside, long Mp, R **sing, R **cpart, R **bpart, R **side,
                hipStream_t s) {
    const size_t pad = 256 / sizeof(R);
    auto up = [&](size_t n) { return (n + pad - 1) / pad * pad; };
    const size_t ns = up((size_t)dp.E * 48), nc = up((size_t)P * Mp), nb = up((size_t)2 * P * Mp);
    const size_t n = ns + nc + nb + (size_t)2 * nside * Mp;
    char *&mem = sizeof(R) == 4 ? dp.scratch32 : dp.scratch64;
    size_t &cap = sizeof(R) == 4 ? dp.cap32 : dp.cap64;
    if (cap < n * sizeof(R)) {
        sfree(mem, s);
        cap = 0;
        HOST_CALL(salloc(&mem, n * sizeof(R), s));
        cap = n * sizeof(R);
    }
    *sing = (R *)mem;
    *cpart = *sing + ns;
    *bpart = *cpart + nc;
    *side = *bpart + nb;
    return EXIT_SUCCESS;
}
}  // namespace

int device_problem_build(const Mesh &m, DeviceProblem &dp, hipStream_t s) {
    HOST_CALL(validate_mesh(m));
    HOST_CALL(ensure_quad());
    device_problem_free(dp);
    dp.st = s;
    dp.N = m.N();
    dp.C = m.C();
    dp.M = dp.N + dp.C;
    dp.E = m.E();
    dp.ldA = ((long)dp.M + 63) / 64 * 64;
    dp.Mp = dp.ldA;
    std::vector<float4> p4(dp.M);
    dp.hpts.resize(3 * (size_t)dp.M);
    for (int i = 0; i < dp.M; i++) {
        const float *src = i < dp.N ? &m.pnts[3 * i] : &m.chief[3 * (i - dp.N)];
        p4[i] = make_float4(src[0], src[1], src[2], 0.f);
        for (int d = 0; d < 3; d++) {
            dp.hpts[3 * i + d] = src[d];
            dp.lo[d] = i ? std::min(dp.lo[d], (double)src[d]) : src[d];
            dp.hi[d] = i ? std::max(dp.hi[d], (double)src[d]) : src[d];
        }
    }
    dp.diam = diagonal(dp.lo, dp.hi);
    for (int i = 0; i < dp.N; i++)
        for (int d = 0; d < 3; d++) {
            const double x = dp.hpts[3 * (size_t)i + d];
            dp.nlo[d] = i ? std::min(dp.nlo[d], x) : x;
            dp.nhi[d] = i ? std::max(dp.nhi[d], x) : x;
        }
    dp.rho = 0;
    dp.helems.resize(3 * (size_t)dp.E);
    std::vector<float2> bc(3 * (size_t)dp.E);
    std::vector<char> used(dp.N, 0);
    dp.impedance = dp.source = 0;
    for (int e = 0; e < dp.E; e++) {
        for (int j = 0; j < 3; j++) {
            dp.helems[3 * e + j] = m.elems[e].nodes[j];
            used[m.elems[e].nodes[j]] = 1;
            bc[3 * e + j] = make_float2(m.elems[e].bc[j].x, m.elems[e].bc[j].y);
        }
        double c[3], q = 0;
        for (int d = 0; d < 3; d++) {
            c[d] = 0;
            for (int j = 0; j < 3; j++) c[d] += dp.hpts[3 * (size_t)dp.helems[3 * e + j] + d] / 3.0;
        }
        for (int j = 0; j < 3; j++) {
            double r2 = 0;
            for (int d = 0; d < 3; d++) {
                const double y = dp.hpts[3 * (size_t)dp.helems[3 * e + j] + d] - c[d];
                r2 += y * y;
            }
            q = std::max(q, r2);
        }
        dp.rho = std::max(dp.rho, std::sqrt(q));
        // (a NaN counts as set)
        if (!(bc[3 * e].x == 0.f && bc[3 * e].y == 0.f)) dp.impedance = 1;
        if (!(bc[3 * e + 2].x == 0.f && bc[3 * e + 2].y == 0.f)) dp.source = 1;
    }
    std::vector<int> isolated;  // nodes no element references
    for (int i = 0; i < dp.N; i++)
        if (!used[i]) isolated.push_back(i);
    dp.n_isolated = (int)isolated.size();
    const int qg = choose_qg(dp.M, dp.E);
    dp.qg = qg;
    dp.hP = choose_tiles(dp.M, dp.N, dp.E, 64 / qg);
    // element-once plan for the FP32 fast kernel: taken when the halo plan
    // integrates at least 5 % of the elements twice and the side columns stay
    // within ghost_slot_bound (device_problem_bytes counts that bound).  It
    // runs at twice the waves as well, so it pays below 10 %: the 40962-node
    // ellipsoid (52 tiles, 7.9 % twice) assembled in 82.9 ms against 91.0 ms
    // (36 points everywhere).
    // Too many side columns for the bound: fewer tiles (two thirds each try).
    // A halo under 5 % is left as it is.
    dp.use_ghost = 0;
    GhostPlan gp;
    int gP = choose_tiles(dp.M, dp.N, dp.E, 64, 2);
    for (int tries = 0; asked_qg(dp.M, dp.E) != 4 && !getenv("BEM_NO_GHOST_PLAN") && tries < 8 && gP >= 4; tries++) {
        build_ghost_plan(m, gP, gp);
        if (gp.P != gP || gp.dup < kGhostMinDup || gp.nslots == 0) break;
        // (ghost_reduce puts the ghost nodes on grid.y: at most 65535)
        if (gp.nslots <= ghost_slot_bound(dp.N, gP) && gp.gnode.size() <= 65535) {
            dp.use_ghost = 1;
            break;
        }
        gP = gP * 2 / 3;
    }
    Pack pk;
    pk.add(&dp.pts, (const float4 *)p4.data(), p4.size());
    pk.add(&dp.pts64, (const double *)dp.hpts.data(), dp.hpts.size());
    pk.add(&dp.elems, (const int *)dp.helems.data(), dp.helems.size());
    pk.add(&dp.bc, (const float2 *)bc.data(), bc.size());
    pk.add(&dp.isolated, (const int *)isolated.data(), isolated.size());
    if (dp.use_ghost) {
        dp.gP = gP;
        dp.nslots = gp.nslots;
        dp.ngnodes = (int)gp.gnode.size();
        pk.add(&dp.gtile_ptr, (const int *)gp.ptr.data(), gp.ptr.size());
        pk.add(&dp.gtile_entries, (const int *)gp.entries.data(), gp.entries.size());
        pk.add(&dp.gtile_slots, (const int *)gp.slots.data(), gp.slots.size());
        pk.add(&dp.gred_ptr, (const int *)gp.gptr.data(), gp.gptr.size());
        pk.add(&dp.gred_node, (const int *)gp.gnode.data(), gp.gnode.size());
        pk.add(&dp.gred_own, (const int *)gp.gown.data(), gp.gown.size());
        pk.add(&dp.gred_slot, (const int *)gp.gslot.data(), gp.gslot.size());
    }
    pk.add(&dp.rec32, (const ElemRec<float> *)nullptr, dp.E);
    pk.add(&dp.rec64, (const ElemRec<double> *)nullptr, dp.E);
    pk.add(&dp.far32, (const FarRec *)nullptr, dp.E);
    pk.add(&dp.bterm, (const double2 *)nullptr, dp.M);
    HOST_CALL(pk.place(&dp.mem, s));
    const int bs = 256;
    prep_elems<float><<<(dp.E + bs - 1) / bs, bs, 0, s>>>(dp.pts64, dp.elems, dp.bc, dp.E, dp.rec32);
    HIP_CALL(hipGetLastError());
    prep_elems<double><<<(dp.E + bs - 1) / bs, bs, 0, s>>>(dp.pts64, dp.elems, dp.bc, dp.E, dp.rec64);
    HIP_CALL(hipGetLastError());
    prep_far<<<(dp.E + bs - 1) / bs, bs, 0, s>>>(dp.pts64, dp.elems, dp.rec64, dp.E, dp.far32);
    HIP_CALL(hipGetLastError());
    dp.mesh_version = m.version;
    return EXIT_SUCCESS;
}

// The problem of `base` with the P points `xs` in the place of its CHIEF
// points, for rows N..N+P-1 (r0 = N) of an assembly: the element records and
// the tiles are base's, which has to outlive dp; only the points, and the
// arrays that the assembly writes, are dp's own.  Building it as a mesh of its
// own took 2 ms of host time a call on 2562 nodes.
int device_problem_rows(const DeviceProblem &base, const float *xs, int P, DeviceProblem &dp, hipStream_t s) {
    device_problem_free(dp);
    if (base.M == 0) BEM_FAIL("device problem not built");
    dp = base;
    dp.borrowed = true;
    dp.mem = dp.halo_mem = dp.scratch32 = dp.scratch64 = nullptr;
    dp.cap32 = dp.cap64 = 0;
    dp.pts = nullptr;
    dp.pts64 = nullptr;
    dp.bterm = nullptr;
    dp.near_ptr = dp.near_row = dp.near_elem = nullptr;
    dp.near_out = nullptr;
    dp.near_factor = 0;
    dp.near_levels = dp.near_npairs = 0;
    dp.hnear_ptr.clear();
    dp.st = s;
    dp.C = P;
    dp.M = dp.N + P;
    dp.ldA = ((long)dp.M + 63) / 64 * 64;
    dp.Mp = ((long)P + 63) / 64 * 64;
    dp.hpts.resize(3 * (size_t)dp.N);
    dp.hpts.insert(dp.hpts.end(), xs, xs + 3 * (size_t)P);
    std::vector<float4> p4(dp.M);
    for (int i = 0; i < dp.M; i++) {
        const double *x = &dp.hpts[3 * (size_t)i];
        p4[i] = make_float4((float)x[0], (float)x[1], (float)x[2], 0.f);
        if (i >= dp.N)
            for (int d = 0; d < 3; d++) {
                dp.lo[d] = std::min(dp.lo[d], x[d]);
                dp.hi[d] = std::max(dp.hi[d], x[d]);
            }
    }
    dp.diam = diagonal(dp.lo, dp.hi);
    if (dp.P == 0) dp.hP = choose_tiles(dp.M, dp.N, dp.E, 64 / dp.qg);
    Pack pk;
    pk.add(&dp.pts, (const float4 *)p4.data(), p4.size());
    pk.add(&dp.pts64, (const double *)dp.hpts.data(), dp.hpts.size());
    pk.add(&dp.bterm, (const double2 *)nullptr, (size_t)P);
    return pk.place(&dp.mem, s);
}

void device_problem_free(DeviceProblem &dp) {
    hipStream_t st = dp.st;
    sfree(dp.mem, st);
    sfree(dp.halo_mem, st);
    sfree(dp.scratch32, st);
    sfree(dp.scratch64, st);
    sfree(dp.near_ptr, st);
    sfree(dp.near_row, st);
    sfree(dp.near_elem, st);
    sfree(dp.near_out, st);
    dp = DeviceProblem{};
    dp.st = st;
}

static void sing_tab(SingTab &t) {
    QuadTables q;
    quad_tables(q);
    const Config &c = config();
    for (int n = 0; n < kQOrder; n++) {
        const double theta = 0.5 + 0.5 * c.qp[n];
        for (int m = 0; m < kQOrder; m++) {
            const double rho = 0.5 + 0.5 * c.qp[m];
            const int qi = n * kQOrder + m;
            // vertex 1: (1-rho, rho(1-theta)); vertex 2: (rho theta, 1-rho);
            // vertex 3: (rho(1-theta), rho theta) (mesh.cu:272-273, 312-313, 352-353)
            t.xi1[0][qi] = 1 - rho;
            t.xi2[0][qi] = rho * (1 - theta);
            t.xi1[1][qi] = rho * theta;
            t.xi2[1][qi] = 1 - rho;
            t.xi1[2][qi] = rho * (1 - theta);
            t.xi2[2][qi] = rho * theta;
            t.w[qi] = q.dw[qi];
        }
    }
}

// Rows a.r0..a.M-1 into a.A and their boundary-condition sums into bterm.
template <typename R, typename C2>
static int assemble_rows(const DeviceProblem &dp, AsmArgs<R> a, bool ghost, int P, double2 *bterm, hipStream_t s) {
    const int nrows = a.M - a.r0, rpw = ghost ? 64 : 64 / dp.qg;
    a.nrbg = ((nrows + rpw - 1) / rpw + 3) / 4;
    a.nwg = a.nrbg * P;
    {
        TimedRegion tr;
        timing_begin(tr, sizeof(R) == 4 ? "asm_tile_f32" : "asm_tile_f64", s);
        const dim3 grid(a.nwg), block(256);
        if (sizeof(R) == 8 && ghost) {
            AsmArgs<double> &ad = *(AsmArgs<double> *)&a;
            if (dp.impedance) asm_tile_fast64<true, true><<<grid, block, 0, s>>>(ad);
            else if (dp.source) asm_tile_fast64<false, true><<<grid, block, 0, s>>>(ad);
            else asm_tile_fast64<false, false><<<grid, block, 0, s>>>(ad);
        } else if (dp.qg == 4 && !ghost) {
            if (dp.impedance) asm_tile<R, 4, true><<<grid, block, 0, s>>>(a);
            else asm_tile<R, 4, false><<<grid, block, 0, s>>>(a);
        } else if (sizeof(R) == 4 && !getenv("BEM_GENERIC_TILE")) {
            // v_sin_f32 / v_cos_f32 are specified for |x| <= 256 revolutions:
            // the phase k r / (2 pi) goes to them unreduced while every
            // distance (at most the bounding-box diagonal of the points) keeps
            // it below that
            const bool raw = a.kf64 * dp.diam < 250.0;
            AsmArgs<float> &af = *(AsmArgs<float> *)&a;
#define BEM_FAST(IMP_, SRC_)                                                                     \
    do {                                                                                         \
        if (ghost && raw) asm_tile_fast<IMP_, true, true, SRC_><<<grid, block, 0, s>>>(af);      \
        else if (ghost) asm_tile_fast<IMP_, false, true, SRC_><<<grid, block, 0, s>>>(af);       \
        else if (raw) asm_tile_fast<IMP_, true, false, SRC_><<<grid, block, 0, s>>>(af);         \
        else asm_tile_fast<IMP_, false, false, SRC_><<<grid, block, 0, s>>>(af);                 \
    } while (0)
            if (dp.impedance) BEM_FAST(true, true);
            else if (dp.source) BEM_FAST(false, true);
            else BEM_FAST(false, false);
#undef BEM_FAST
        } else {
            if (dp.impedance) asm_tile<R, 1, true><<<grid, block, 0, s>>>(a);
            else asm_tile<R, 1, false><<<grid, block, 0, s>>>(a);
        }
        HIP_CALL(hipGetLastError());
        timing_end(tr, s);
    }
    if (ghost && dp.ngnodes > 0) {
        if (a.ldA % 2 || a.Mp % 2) BEM_FAIL("ghost_reduce needs even leading dimensions (ldA %ld, Mp %ld)", a.ldA, a.Mp);
        TimedRegion tr;
        timing_begin(tr, "ghost_reduce", s);
        constexpr int W = sizeof(R) == 4 ? 2 : 1;
        using V4 = typename std::conditional<sizeof(R) == 4, float4, double2>::type;
        dim3 grid(((nrows + W - 1) / W + 255) / 256, dp.ngnodes);
        ghost_reduce<V4, W><<<grid, 256, 0, s>>>((V4 *)a.A, a.ldA, nrows, (const V4 *)a.side, a.Mp, dp.gred_ptr,
                                                 dp.gred_node, dp.gred_own, dp.gred_slot);
        HIP_CALL(hipGetLastError());
        timing_end(tr, s);
    }
    if (dp.n_isolated > 0) {
        dim3 grid((nrows + 255) / 256, dp.n_isolated);
        zero_columns<C2><<<grid, 256, 0, s>>>(a.A, a.ldA, nrows, dp.isolated, dp.n_isolated);
        HIP_CALL(hipGetLastError());
    }
    {
        TimedRegion tr;
        timing_begin(tr, "asm_finalize", s);
        asm_finalize<R, C2><<<(nrows + 63) / 64, 64 * kFinRuns, 0, s>>>(
            a.A, a.ldA, a.M, dp.N, P, a.Mp, a.r0, a.cpart, a.bpart, bterm, dp.impedance || dp.source);
        HIP_CALL(hipGetLastError());
        timing_end(tr, s);
    }
    return EXIT_SUCCESS;
}

// Rows of a radiation operator of n rows that are assembled at a time in P tiles:
// blocks of equal height (a multiple of a workgroup's 256 rows) of at most 8192
// workgroups.  The tiles are the mesh's, however many points there are, so the
// partials and side columns of all of them at once would take up to twice the
// operator's own bytes: 642 nodes, 200000 points: 2.0 GB beside 1.03 GB; in blocks
// 0.15.  (4096 workgroups leave the 6001 points of a 2562-node map in two blocks:
// 0.55 ms instead of 0.39.)
static int operator_rows(int n, int P) {
    const int most = 256 * ((8192 + P - 1) / P), blocks = (n + most - 1) / most;
    return ((n + blocks - 1) / blocks + 255) / 256 * 256;
}

// Rows r0..M-1 of the system into A (ld ldA, row r0 first) and their
// boundary-condition sums into bterm; r0 = 0 is the whole collocation system,
// r0 = N the operator of a field's points.
template <typename R, typename C2>
static int assemble_impl(DeviceProblem &dp, R k, C2 *A, long ldA, int r0, double2 *bterm, hipStream_t s) {
    HOST_CALL(ensure_quad());
    if (dp.M == 0) BEM_FAIL("device problem not built");
    const Config &cfg = config();
    const double kd = (double)k;
    const double rw = (double)cfg.density * (double)(k * (R)cfg.speed);  // rho * omega, omega = k c
    QuadTables qt;
    quad_tables(qt);
    SingTab st;
    sing_tab(st);
    // the plan this call walks, and the arrays it writes
    // (FP64: the fast kernel's phases hold up to 2^30 quadrants)
    const bool ghost = dp.use_ghost && !getenv("BEM_ASM_HALO") && !getenv("BEM_GENERIC_TILE") &&
                       (sizeof(R) == 4 || std::fabs(kd) * dp.diam < 1e8);
    if (!ghost) HOST_CALL(halo_plan(dp, s));
    const int P = ghost ? dp.gP : dp.P;
    R *sing = nullptr, *cpart = nullptr, *bpart = nullptr, *side = nullptr;
    const int block = r0 < dp.N ? dp.M - r0 : std::min(dp.M - r0, operator_rows(dp.M - r0, P));
    const long Mp = ((long)block + 63) / 64 * 64;
    HOST_CALL(asm_scratch<R>(dp, P, ghost ? dp.nslots : 0, Mp, &sing, &cpart, &bpart, &side, s));
    if (r0 < dp.N) {  // (rows that are no nodes meet no singular pair)
        TimedRegion tr;
        timing_begin(tr, "sing_elems", s);
        const int n = 3 * dp.E, bs = 128;
        sing_elems<R><<<(n + bs - 1) / bs, bs, 0, s>>>(dp.pts64, dp.elems, dp.bc, dp.E, kd, rw, st, sing);
        HIP_CALL(hipGetLastError());
        timing_end(tr, s);
    }
    AsmArgs<R> a;
    a.pts = dp.pts;
    a.recs = (const ElemRec<R> *)(sizeof(R) == 4 ? (void *)dp.rec32 : (void *)dp.rec64);
    a.far = dp.far32;
    a.sing = sing;
    a.tile_ptr = dp.tile_ptr;
    a.tile_entries = dp.tile_entries;
    a.cpart = cpart;
    a.bpart = (C2 *)bpart;
    a.ldA = ldA;
    a.Mp = Mp;
    a.N = dp.N;
    a.k = k;
    a.kf = (R)(kd / (2.0 * kPi));
    a.kf64 = kd / (2.0 * kPi);
    a.rw = (R)rw;
    far_limits(kd, sizeof(R) == 4 ? kFarK2 : kSmallPhase64, a.far_rho2, a.far7_rho2);
    a.impedance = dp.impedance;
    for (int q = 0; q < kNQ; q++) {
        a.q.xi1[q] = sizeof(R) == 4 ? (R)qt.xi1[q] : (R)qt.dxi1[q];
        a.q.xi2[q] = sizeof(R) == 4 ? (R)qt.xi2[q] : (R)qt.dxi2[q];
        a.q.w[q] = sizeof(R) == 4 ? (R)qt.w[q] : (R)qt.dw[q];
    }
    a.tile_slots = nullptr;
    a.side = nullptr;
    if (ghost) {
        a.tile_ptr = dp.gtile_ptr;
        a.tile_entries = dp.gtile_entries;
        a.tile_slots = dp.gtile_slots;
        a.side = (C2 *)side;
    }
    for (int b0 = r0; b0 < dp.M; b0 += block) {
        a.r0 = b0;
        a.M = std::min(dp.M, b0 + block);
        a.A = A + (b0 - r0);
        HOST_CALL((assemble_rows<R, C2>(dp, a, ghost, P, bterm + (b0 - r0), s)));
    }
    // opt-in FP64 near-singular corrections, after every row is complete
    if (cfg.near_factor > 0 || dp.near_factor > 0) HOST_CALL((near_correct<R, C2>(dp, kd, rw, A, ldA, r0, bterm, s)));
    return EXIT_SUCCESS;
}

int assemble_fp32(DeviceProblem &dp, float k, float2 *A, hipStream_t s) {
    return assemble_impl<float, float2>(dp, k, A, dp.ldA, 0, dp.bterm, s);
}
int assemble_fp64(DeviceProblem &dp, double k, double2 *A, hipStream_t s) {
    return assemble_impl<double, double2>(dp, k, A, dp.ldA, 0, dp.bterm, s);
}

template <typename C2>
static int rhs_impl(DeviceProblem &dp, double k, C2 *B, long ldB, const RhsSpec &rhs, hipStream_t s) {
    if (rhs.nrhs <= 0) return EXIT_SUCCESS;
    if (rhs.nrhs > kMaxRhs) BEM_FAIL("at most %d right-hand sides, got %d", kMaxRhs, rhs.nrhs);
    float *params = nullptr;
    HOST_CALL(salloc(&params, 3 * (size_t)rhs.nrhs, s));
    HIP_CALL(hipMemcpyAsync(params, rhs.params.data(), 3 * sizeof(float) * rhs.nrhs, hipMemcpyHostToDevice, s));
    dim3 grid((dp.M + 255) / 256, rhs.nrhs);
    rhs_fill<C2><<<grid, 256, 0, s>>>(dp.pts64, dp.M, k, rhs.kind, (double)rhs.amp, params, rhs.nrhs, dp.bterm, B, ldB);
    hipError_t e = hipGetLastError();
    (void)hipStreamSynchronize(s);
    sfree(params, s);
    HIP_CALL(e);
    return EXIT_SUCCESS;
}

// ------------------------------------------------- field as a GEMM ---
// fdp is the mesh with the P field points as its extra rows (the CHIEF
// position).  Rows N..N+P-1 of the collocation formula are the radiation
// operator: p(x) = inc(x) - bterm(x) - sum_j F[x, j] p_j (genExtPressure,
// mesh.cu:1038-1073, as a matrix).  F is P x N (ldF), fbterm P values.
int field_matrix_fp32(DeviceProblem &fdp, float k, float2 *F, long ldF, double2 *fbterm, hipStream_t s) {
    if (fdp.M <= fdp.N) BEM_FAIL("field problem has no field points");
    if (ldF < fdp.M - fdp.N) BEM_FAIL("ldF must be >= P");
    return assemble_impl<float, float2>(fdp, k, F, ldF, fdp.N, fbterm, s);
}

__global__ void k_sub_c(float2 *out, long ldo, const float2 *__restrict__ Y, long ldy, int P) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (i >= P) return;
    const float2 y = Y[(size_t)r * ldy + i];
    float2 o = out[(size_t)r * ldo + i];
    o.x -= y.x;
    o.y -= y.y;
    out[(size_t)r * ldo + i] = o;
}

// out (P x R, ldo) = inc_r(x_p) - bterm_p - (F X)_p for the FP32 solutions X
// (N x R, ldx): one GEMV (R = 1) or one MFMA product (R > 1) over F.
// ws >= max(ws_gemv_n(P, N, 1), ws_gemm(P, N, R)); Y: P x R scratch (ldF).
int field_apply_fp32(DeviceProblem &fdp, double k, const float2 *F, long ldF, const double2 *fbterm, const float2 *X,
                     long ldx, const RhsSpec &rhs, float2 *Y, float2 *out, long ldo, void *ws, hipStream_t s) {
    const int N = fdp.N, P = fdp.M - fdp.N, R = rhs.nrhs;
    if (R <= 0 || P <= 0) return EXIT_SUCCESS;
    {
        TimedRegion tr;
        timing_begin(tr, "field_gemm", s);
        if (R == 1) HOST_CALL(gemv_n_f32(F, ldF, P, N, X, 0, Y, 0, 1, ws, s));
        else HOST_CALL(gemm_n_f32(F, ldF, P, N, X, ldx, Y, ldF, R, ws, s));
        timing_end(tr, s);
    }
    float *params = nullptr;
    HOST_CALL(salloc(&params, 3 * (size_t)R, s));
    HIP_CALL(hipMemcpyAsync(params, rhs.params.data(), 3 * sizeof(float) * R, hipMemcpyHostToDevice, s));
    dim3 grid((P + 255) / 256, R);
    rhs_fill<float2><<<grid, 256, 0, s>>>(fdp.pts64 + 3 * (size_t)N, P, k, rhs.kind, (double)rhs.amp, params, R,
                                          fbterm, out, ldo);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        k_sub_c<<<grid, 256, 0, s>>>(out, ldo, Y, ldF, P);
        e = hipGetLastError();
    }
    (void)hipStreamSynchronize(s);  // params is a host-side copy source
    sfree(params, s);
    HIP_CALL(e);
    return EXIT_SUCCESS;
}

int rhs_fp32(DeviceProblem &dp, double k, float2 *B, long ldB, const RhsSpec &rhs, hipStream_t s) {
    return rhs_impl<float2>(dp, k, B, ldB, rhs, s);
}
int rhs_fp64(DeviceProblem &dp, double k, double2 *B, long ldB, const RhsSpec &rhs, hipStream_t s) {
    return rhs_impl<double2>(dp, k, B, ldB, rhs, s);
}

}  // namespace bem
