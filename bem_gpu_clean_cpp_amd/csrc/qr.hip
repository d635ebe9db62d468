// Blocked Householder least squares on the device: the job of qrSolver
// (numerical.cu:580-644: geqrf, unmqr with Q^H, trsm) and of the reference's
// own blocked WY QR (QR_thin, numerical.cu:246-504), without host round trips
// inside a panel.
//
//   qr_panel    one workgroup factors a panel of nb columns in place: for each
//               column a Householder reflector H = I - tau v v^H (v_0 = 1,
//               tau real, beta = -phase(alpha) ||x||), applied to the rest of
//               the panel; then the triangular factor T of the compact WY form
//               H_1 ... H_nb = I - V T V^H (Schreiber & Van Loan 1989).
//   qr_vhc      W = T^H (V^H C) for the trailing columns C (one workgroup per
//               column, the nb dot products in one pass over the column);
//   qr_update   C -= V W (the rank-nb trailing update, GEMM-shaped);
//   FP32 panels are formed from their Gram matrix instead (qr_gram, qr_recon,
//               qr_form_v), and FP32 trailing updates run on MFMA: V^H C as the
//               adjoint product (C^H V, gemm.hip) against an explicit copy of
//               the panel's V, then W = T^H (V^H C) and C -= V W in one launch;
//   trsv_upper  R x = (Q^H b)[0:N] by column-oriented back substitution.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <thread>
#include <vector>

#include "bem_internal.hpp"

namespace bem {

template <typename T>
struct QT;
template <>
struct QT<float> {
    using c2 = float2;
};
template <>
struct QT<double> {
    using c2 = double2;
};

constexpr int kNB = 32;  // panel width
constexpr int kCG = 8;   // panel columns updated together
constexpr int kColThreads = 256;  // rows per workgroup of the column launches

template <typename T>
__device__ __forceinline__ T wsum(T v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// V[i, l] of panel starting at column j0: unit at row j0+l, stored below it.
template <typename C2>
__device__ __forceinline__ C2 vget(const C2 *A, long lda, int j0, int l, int i) {
    C2 z;
    if (i == j0 + l) {
        z.x = 1;
        z.y = 0;
    } else if (i > j0 + l) {
        z = A[(size_t)(j0 + l) * lda + i];
    } else {
        z.x = 0;
        z.y = 0;
    }
    return z;
}

// (at most 1024 threads, all of the workgroup; shared arrays of the caller)
template <typename T>
__device__ __forceinline__ void panel_one_wg(typename QT<T>::c2 *A, long lda, int M, int j0, int nb,
                             typename QT<T>::c2 *Tout /* nb x nb, ld kNB */, int make_t,
                             typename QT<T>::c2 (*s_Y)[kNB] /* v_l^H v_m for l < m */,
                             typename QT<T>::c2 (*s_T)[kNB]) {
    using C2 = typename QT<T>::c2;
    __shared__ T red[2][16];
    __shared__ T s_tau[kNB];
    __shared__ T s_red[16][2 * kCG];
    __shared__ T s_d[2 * kCG];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nw = blockDim.x >> 6;
    for (int jj = 0; jj < nb; jj++) {
        const int j = j0 + jj;
        C2 *col = A + (size_t)j * lda;
        // s = sum_{i>j} |A[i,j]|^2
        T s = 0;
        for (int i = j + 1 + tid; i < M; i += blockDim.x) s += col[i].x * col[i].x + col[i].y * col[i].y;
        s = wsum(s);
        if (lane == 0) red[0][wid] = s;
        __syncthreads();
        T tot = 0;
        for (int q = 0; q < nw; q++) tot += red[0][q];
        const C2 alpha = col[j];
        const T aa = sqrt(alpha.x * alpha.x + alpha.y * alpha.y);
        const T xnorm = sqrt(aa * aa + tot);
        T tau = 0;
        C2 scale;
        scale.x = 0;
        scale.y = 0;
        C2 beta;
        beta = alpha;
        if (tot > 0 || (xnorm > 0 && alpha.y != 0)) {
            const T phr = aa > 0 ? alpha.x / aa : (T)1, phi = aa > 0 ? alpha.y / aa : (T)0;
            beta.x = -phr * xnorm;
            beta.y = -phi * xnorm;
            // scale = 1 / (alpha - beta)
            const T dr = alpha.x - beta.x, di = alpha.y - beta.y;
            const T dd = dr * dr + di * di;
            scale.x = dr / dd;
            scale.y = -di / dd;
            tau = (T)2 / ((T)1 + tot / dd);
        }
        __syncthreads();  // everyone read alpha / red
        for (int i = j + 1 + tid; i < M; i += blockDim.x) {
            const C2 v = col[i];
            C2 o;
            o.x = v.x * scale.x - v.y * scale.y;
            o.y = v.x * scale.y + v.y * scale.x;
            col[i] = o;
        }
        if (tid == 0) {
            col[j] = beta;
            s_tau[jj] = tau;
        }
        __syncthreads();
        // apply H^H = H (tau real) to the remaining panel columns, 8 at a time:
        // every thread takes rows i > j for all 8 columns, one block reduction
        // of the 8 dot products, then the rank-1 update of those rows
        for (int c0 = j + 1; c0 < j0 + nb; c0 += kCG) {
            const int ncg = min(kCG, j0 + nb - c0);
            T dr[kCG], di[kCG];
#pragma unroll
            for (int c = 0; c < kCG; c++) {
                dr[c] = 0;
                di[c] = 0;
            }
            for (int i = j + 1 + tid; i < M; i += blockDim.x) {
                const C2 v = col[i];
#pragma unroll
                for (int c = 0; c < kCG; c++) {
                    if (c < ncg) {
                        const C2 a = A[(size_t)(c0 + c) * lda + i];
                        dr[c] += v.x * a.x + v.y * a.y;
                        di[c] += v.x * a.y - v.y * a.x;
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < kCG; c++) {
                const T r = wsum(dr[c]), im = wsum(di[c]);
                if (lane == 0) {
                    s_red[wid][2 * c] = r;
                    s_red[wid][2 * c + 1] = im;
                }
            }
            __syncthreads();
            if (tid < 2 * ncg) {
                T t = 0;
                for (int q = 0; q < nw; q++) t += s_red[q][tid];
                const int c = tid >> 1;
                const C2 aj = A[(size_t)(c0 + c) * lda + j];  // row j: v_j = 1
                s_d[tid] = (t + ((tid & 1) ? aj.y : aj.x)) * tau;
            }
            __syncthreads();
            for (int i = j + 1 + tid; i < M; i += blockDim.x) {
                const C2 v = col[i];
#pragma unroll
                for (int c = 0; c < kCG; c++) {
                    if (c < ncg) {
                        const T er = s_d[2 * c], ei = s_d[2 * c + 1];
                        C2 *pa = A + (size_t)(c0 + c) * lda + i;
                        C2 a = *pa;
                        a.x -= er * v.x - ei * v.y;
                        a.y -= er * v.y + ei * v.x;
                        *pa = a;
                    }
                }
            }
            if (tid < ncg) {
                C2 *pa = A + (size_t)(c0 + tid) * lda + j;
                C2 a = *pa;
                a.x -= s_d[2 * tid];
                a.y -= s_d[2 * tid + 1];
                *pa = a;
            }
            __syncthreads();
        }
    }
    if (!make_t) {  // T is formed by qr_make_t from an MFMA V^H V: pass the taus on its diagonal
        for (int p = tid; p < kNB * kNB; p += blockDim.x) {
            const int l = p / kNB, m = p % kNB;
            C2 z;
            z.x = (l == m && l < nb) ? s_tau[l] : (T)0;
            z.y = 0;
            Tout[p] = z;
        }
        return;
    }
    // Y[l][m] = v_l^H v_m for l < m (dot over rows >= j0+m)
    for (int p = wid; p < nb * nb; p += nw) {
        const int l = p / nb, m = p % nb;
        if (l >= m) continue;
        T dr = 0, di = 0;
        for (int i = j0 + m + lane; i < M; i += 64) {
            const C2 vl = vget(A, lda, j0, l, i), vm = vget(A, lda, j0, m, i);
            dr += vl.x * vm.x + vl.y * vm.y;
            di += vl.x * vm.y - vl.y * vm.x;
        }
        dr = wsum(dr);
        di = wsum(di);
        if (lane == 0) {
            s_Y[l][m].x = dr;
            s_Y[l][m].y = di;
        }
    }
    __syncthreads();
    // T upper triangular (LAPACK larft, forward columnwise): T_mm = tau_m,
    // T[0:m, m] = -tau_m T[0:m, 0:m] Y[0:m, m]; column m in parallel over rows
    for (int p = tid; p < kNB * kNB; p += blockDim.x) {
        s_T[p / kNB][p % kNB].x = 0;
        s_T[p / kNB][p % kNB].y = 0;
    }
    __syncthreads();
    for (int m = 0; m < nb; m++) {
        if (tid < m) {
            T zr = 0, zi = 0;
            for (int q = tid; q < m; q++) {
                const C2 t = s_T[tid][q], y = s_Y[q][m];
                zr += t.x * y.x - t.y * y.y;
                zi += t.x * y.y + t.y * y.x;
            }
            s_T[tid][m].x = -s_tau[m] * zr;
            s_T[tid][m].y = -s_tau[m] * zi;
        } else if (tid == m) {
            s_T[m][m].x = s_tau[m];
        }
        __syncthreads();
    }
    for (int p = tid; p < kNB * kNB; p += blockDim.x) Tout[p] = s_T[p / kNB][p % kNB];
}

template <typename T>
__global__ __launch_bounds__(1024) void qr_panel(typename QT<T>::c2 *A, long lda, int M, int j0, int nb,
                                                 typename QT<T>::c2 *Tout, int make_t) {
    __shared__ typename QT<T>::c2 s_Y[kNB][kNB], s_T[kNB][kNB];
    panel_one_wg<T>(A, lda, M, j0, nb, Tout, make_t, s_Y, s_T);
}

// Sum of 2 kNB = 64 per-lane values over the wave, scattered: on return lane
// l holds the wave total of slot l in x[0].  Each halving step sends one half
// of the live slots to the partner lane and keeps the other half (the half
// picked by the lane's bit H), so 32 + 16 + ... + 1 = 63 shuffles replace the
// 64 x 6 of one butterfly sum per slot.
template <int H, typename T>
__device__ __forceinline__ void reduce_scatter_step(T (&x)[2 * kNB], int lane) {
    const bool up = (lane & H) != 0;
#pragma unroll
    for (int i = 0; i < H; i++) {
        const T send = up ? x[i] : x[i + H];
        const T keep = up ? x[i + H] : x[i];
        x[i] = keep + __shfl_xor(send, H, 64);
    }
}
template <typename T>
__device__ __forceinline__ void wave_reduce_scatter64(T (&x)[2 * kNB], int lane) {
    reduce_scatter_step<32>(x, lane);
    reduce_scatter_step<16>(x, lane);
    reduce_scatter_step<8>(x, lane);
    reduce_scatter_step<4>(x, lane);
    reduce_scatter_step<2>(x, lane);
    reduce_scatter_step<1>(x, lane);
}

// FP32: the two wide steps as lane-half swaps (v_permlane32_swap exchanges
// lanes 32-63 of its first operand with lanes 0-31 of its second,
// v_permlane16_swap the odd 16-lane rows of the first with the even rows of
// the second), so the lane whose bit H is clear ends with its own and its
// partner's x[i] and the other lane with both x[i + H]: one add, no select.
// The narrow steps read the partner through DPP: row_ror:8 pairs l with l ^ 8
// inside a row, row_half_mirror pairs l with 7 - l inside 8 lanes (opposite
// bit 2, same higher bits, which is all the scatter needs), quad_perm
// [2,3,0,1] and [1,0,3,2] pair across bits 1 and 0.
template <int H>
__device__ __forceinline__ void reduce_scatter_swap(float (&x)[2 * kNB]) {
#pragma unroll
    for (int i = 0; i < H; i++) {
        const unsigned a = __float_as_uint(x[i]), b = __float_as_uint(x[i + H]);
        if constexpr (H == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
            x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else {
            const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
            x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
    }
}
template <int H, int CTRL>
__device__ __forceinline__ void reduce_scatter_dpp(float (&x)[2 * kNB], int lane) {
    const bool up = (lane & H) != 0;
#pragma unroll
    for (int i = 0; i < H; i++) {
        const float send = up ? x[i] : x[i + H];
        const float keep = up ? x[i + H] : x[i];
        x[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), CTRL, 0xF, 0xF, false));
    }
}
template <>
__device__ __forceinline__ void wave_reduce_scatter64<float>(float (&x)[2 * kNB], int lane) {
    reduce_scatter_swap<32>(x);
    reduce_scatter_swap<16>(x);
    reduce_scatter_dpp<8, 0x128>(x, lane);  // row_ror:8
    reduce_scatter_dpp<4, 0x141>(x, lane);  // row_half_mirror
    reduce_scatter_dpp<2, 0x4E>(x, lane);   // quad_perm [2,3,0,1]
    reduce_scatter_dpp<1, 0xB1>(x, lane);   // quad_perm [1,0,3,2]
}

// FP32 panels in three launches instead of one step per column.  The panel P
// (rows j0..M-1, nb <= 32 columns) gets the same compact WY form as from
// reflectors, by way of its Gram matrix:
//   qr_gram    partials of G = P^H P in FP64 (exact products of FP32 numbers);
//   qr_recon   one workgroup: Cholesky G = R^H R, then the reflectors from R
//              and the top rows P_1 alone (Householder reconstruction: Ballard,
//              Demmel, Grigori, Jacquelin, Nguyen & Solomonik 2014): P_1 - S R =
//              L U with unit diagonal phases S chosen against cancellation as
//              the elimination goes, s_k = -phase(pivot), so |U_kk| >= R_kk and
//              no pivoting is needed.  Then V = [L; P_2 U^-1], R_h = S R and
//              T = -U R_h^-1 L^-H, with Q^H P = [R_h; 0] for
//              Q = I - V T V^H: the phases and tau of the column-wise algorithm;
//   qr_form_v  the rows P_2 U^-1 of V, and V with its unit diagonal and zeros.
// All in FP64, with V, R and T rounded to FP32 once.  The loss of orthogonality
// is about 1e-18 kappa^2 (kappa: condition number of the panel with columns
// scaled to norm 1), so panels of kappa^2 > 1e9, those whose Gram matrix is not
// numerically positive definite (dependent or zero columns, numbers that are
// not finite) and those with a column that needs no reflection take the
// column-wise algorithm inside qr_recon instead, in one workgroup; where the panels
// of a matrix do so again and again, PanelRoute sends the next ones to a launch per
// column.
//
// 5 + 32 + 5 us a panel of up to 2000 rows.  The column-wise panels that this
// replaces were bound by their 32 serial steps: 69 us (256 rows), 98 (512) and
// 135 (1024) with the panel in one workgroup's registers, 330 + 40 us with a
// launch per column above.  With qr_trail, a QR solve of 642 nodes went from
// 4.1 to 2.8 ms, 1962: 22.1 to 9.1, 10242: 317 to 150.
constexpr int kNN = kNB * kNB;
// rows up to which the trailing update sums the partials of C^H V itself (each
// 128 rows of it sum them again): QR solve of 4002 nodes 23.9-24.3 ms for 0 to
// 2048, 26.4 always; 10242 nodes 150 ms, 175 always; below 2000 nodes within 2 %
constexpr int kTrailRows = 1024;
constexpr int kGramChunk = 64;      // rows of a panel staged at a time
constexpr int kGramParts = 16;      // at most this many partials (one workgroup sums them)
constexpr double kPanelCond2 = 1e9;

// part[blk][i][j] = sum over the block's rpb rows (a multiple of kGramChunk) of
// conj(P_i) P_j, zero past nb, on FP64 MFMA in the three-product form; wave w
// takes the 16 x 16 tile (w % 2, w / 2).  Pc receives a copy of the panel
// (qr_form_v writes V over the panel while it reads P).
__global__ __launch_bounds__(256) void qr_gram(const float2 *__restrict__ A, long lda, int M, int j0, int nb, int rpb,
                                               double2 *__restrict__ part, float2 *__restrict__ Pc, long ldv) {
    typedef double v4d __attribute__((ext_vector_type(4)));
    __shared__ float2 s_p[kNB][kGramChunk + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kk = lane >> 4;
    const int a0 = 16 * (wave & 1), b0 = 16 * (wave >> 1);
    v4d acc[3];
#pragma unroll
    for (int q = 0; q < 3; q++) acc[q] = (v4d){0, 0, 0, 0};
    for (int r0 = 0; r0 < rpb; r0 += kGramChunk) {
        const int i = blockIdx.x * rpb + r0 + lane;  // row of the panel
        float2 v[kNB / 4];
#pragma unroll
        for (int u = 0; u < kNB / 4; u++) {
            const int c = wave + 4 * u;
            v[u] = make_float2(0.f, 0.f);
            if (j0 + i < M && c < nb) v[u] = A[(size_t)(j0 + c) * lda + j0 + i];
        }
        __syncthreads();  // the previous rows are read
#pragma unroll
        for (int u = 0; u < kNB / 4; u++) {
            const int c = wave + 4 * u;
            s_p[c][lane] = v[u];
            if (j0 + i < M) Pc[(size_t)c * ldv + i] = v[u];
        }
        __syncthreads();
#pragma unroll 4
        for (int r = 0; r < kGramChunk; r += 4) {
            const float2 x = s_p[a0 + m][r + kk], y = s_p[b0 + m][r + kk];
            const double ur = x.x, ui = -(double)x.y, vr = y.x, vi = y.y;
            acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ur, vr + vi, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ur + ui, vi, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(ui - ur, vr, acc[2], 0, 0, 0);
        }
    }
    double2 *pb = part + (size_t)blockIdx.x * kNN;
#pragma unroll
    for (int v = 0; v < 4; v++)
        pb[(a0 + kk + 4 * v) * kNB + b0 + m] = make_double2(acc[0][v] - acc[1][v], acc[0][v] + acc[2][v]);
}

// 1 / x and 1 / sqrt(x): the hardware's estimates (relative error 2^-23) and one
// third-order step
__device__ __forceinline__ double rcp_step(double x) {
    const double y = __builtin_amdgcn_rcp(x), e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}
__device__ __forceinline__ double rsq_step(double x) {
    const double y = __builtin_amdgcn_rsq(x), e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 zfms(double2 c, double2 a, double2 b) {  // c - a b
    return make_double2(fma(-a.x, b.x, fma(a.y, b.y, c.x)), fma(-a.x, b.y, fma(-a.y, b.x, c.y)));
}

// R_kk = d rd from the pivot d of G, and for the pivot p of the top rows
// s = -phase(p) and 1 / (p - s R_kk) = -conj(s) / (|p| + R_kk)
struct PanelPivot {
    double rd;
    double2 s, inv;
    __device__ __forceinline__ PanelPivot(double d, double2 p) {
        rd = rsq_step(d);
        const double aa = fma(p.x, p.x, p.y * p.y), y = rsq_step(aa);
        s = make_double2(aa > 0 ? -p.x * y : -1.0, aa > 0 ? -p.y * y : 0.0);
        const double q = rcp_step(fma(d, rd, aa > 0 ? aa * y : 0.0));
        inv = make_double2(-s.x * q, s.y * q);
    }
};

// The reflectors of a panel from the partials of its Gram matrix: R (above and
// on the diagonal) and L (below it) to the top rows of the panel, T to Tout,
// the top rows of V to Vd, U^-1 to Y (row-major), *bad = 0.  Panels that the
// reconstruction does not take (above) are factored column by column instead,
// with T, and *bad = 1.  The host learns it from seen (pinned memory, or null).
//
// One workgroup eliminates two matrices in place and in step: G and P_1 - S R.
// Step k needs row k of R only, which is row k of G's elimination scaled, so
// both take one barrier a step: the rows and columns k of both as they stand go
// through shared memory, and every thread finishes the pivots for itself.  Wave
// w holds the rows w + 8 e (e < 4), lanes 0..31 the columns of G, lanes 32..63
// those of P_1 - S R, so that what depends on the row is known to the wave.  The
// update is one multiply-add per entry: the pivot entry of a published row is 1
// and that of a column -1, and the publishing threads clear the entries that
// start anew (inverse of row and column k).  Afterwards G holds U0^-1 (j >= i),
// and P_1 - S R holds U^-1 (j >= i) and L^-1 (j < i); U0, U and L follow from the
// published rows and columns.
// 32 us, 21 of them the 32 steps (the FP64 chain of the pivots, a round through
// shared memory and a barrier each).  Both matrices in every thread, the row
// conditions per lane: 36 us; 256 or 1024 threads 37 to 41; the two eliminations
// one after the other 45.  (Entries are separate doubles: branches on whole
// entries, or a select of their addresses, put them in scratch memory: 93 us.)
constexpr int kRecThreads = 512, kRecWaves = kRecThreads / 64, kEnt = kNB / kRecWaves;
__global__ __launch_bounds__(kRecThreads) void qr_recon(const double2 *__restrict__ part, int nblk, float2 *A, long lda,
                                                        int M, int j0, int nb, float2 *__restrict__ Tout,
                                                        float2 *__restrict__ Vd, long ldv, double2 *__restrict__ Y,
                                                        int *__restrict__ bad, int *seen) {
    __shared__ double2 s_row[2][kNB][kNB];   // published rows of G and P_1 - S R
    __shared__ double2 s_cw[kNB][kNB + 1];   // published columns of P_1 - S R
    __shared__ double2 s_cg[2][kNB];         // and of G (two buffers)
    __shared__ double2 s_piv[2][kNB], s_sign[kNB], s_u[kNB], s_inv[kNB];
    __shared__ double s_g[kNB], s_w[kRecWaves];
    __shared__ int s_flat;
    const int tid = threadIdx.x, lane = tid & 63, j = tid & 31;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool top = lane >= kNB;  // this lane's matrix is P_1 - S R
    const int Mp = M - j0;
    double x[kEnt], y[kEnt];
    {
        // the lanes of either matrix sum half of the partials of G
        constexpr int kHalf = kGramParts / 2;
        double2 v[kEnt][kHalf];
        const int b0 = top ? kHalf : 0;
#pragma unroll
        for (int e = 0; e < kEnt; e++)
#pragma unroll
            for (int b = 0; b < kHalf; b++)
                v[e][b] = part[(size_t)min(b0 + b, nblk - 1) * kNN + (w + kRecWaves * e) * kNB + j];
#pragma unroll
        for (int e = 0; e < kEnt; e++) {
            const int i = w + kRecWaves * e;
            float2 t = make_float2(0.f, 0.f);
            if (i < Mp && j < nb) t = A[(size_t)(j0 + j) * lda + j0 + i];
            double gx = 0, gy = 0;
#pragma unroll
            for (int b = 0; b < kHalf; b++) {
                gx += b0 + b < nblk ? v[e][b].x : 0.0;
                gy += b0 + b < nblk ? v[e][b].y : 0.0;
            }
            gx += __shfl_xor(gx, 32, 64);
            gy += __shfl_xor(gy, 32, 64);
            const bool in = i < nb && j < nb;
            gx = in ? gx : i == j ? 1.0 : 0.0;
            gy = in ? gy : 0.0;
            if (i == j) s_g[i] = gx;  // |P_i|^2
            x[e] = top ? (double)t.x : gx;
            y[e] = top ? (double)t.y : gy;
        }
    }
    if (tid == 0) s_flat = 0;
    double2 *const myrow = &s_row[top][0][0];
#pragma unroll
    for (int ek = 0; ek < kEnt; ek++) {  // k = kRecWaves ek + kw: row k is entry ek of wave kw
        for (int kw = 0; kw < kRecWaves; kw++) {
            const int k = kRecWaves * ek + kw;
            const bool at = j == k;
            double2 *const col = top ? s_cw[k] : s_cg[k & 1];
            if (w == kw) {
                const bool none = !top && j < k;
                myrow[k * kNB + j] = make_double2(at ? 1.0 : none ? 0.0 : x[ek], at || none ? 0.0 : y[ek]);
                if (at) s_piv[top][k] = make_double2(x[ek], y[ek]);
                if (j >= k) {
                    x[ek] = at ? -1.0 : 0.0;
                    y[ek] = 0.0;
                }
            }
            if (at) {
#pragma unroll
                for (int e = 0; e < kEnt; e++) {
                    col[w + kRecWaves * e] = make_double2(x[e], y[e]);
                    x[e] = 0.0;
                    y[e] = 0.0;
                }
            }
            __syncthreads();
            const double2 ra = s_row[0][k][j], rw = s_row[1][k][j];
            double2 c[kEnt];
#pragma unroll
            for (int e = 0; e < kEnt; e++) c[e] = col[w + kRecWaves * e];
            const PanelPivot pv(s_piv[0][k].x, s_piv[1][k]);
            const double tx = j > k ? ra.x * pv.rd : 0.0, ty = j > k ? ra.y * pv.rd : 0.0;  // R_kj
            const double2 rb = zfms(rw, pv.s, make_double2(tx, ty));
            const double rx = top ? rb.x : ra.x, ry = top ? rb.y : ra.y;
            const double ix = top ? pv.inv.x : pv.rd * pv.rd, iy = top ? pv.inv.y : 0.0;
            // rows up to k keep their entries left of column k
            const double mx = j < k ? 0.0 : rx, my = j < k ? 0.0 : ry;
            const bool below = w > kw;
            const double ex = below ? rx : mx, ey = below ? ry : my;
#pragma unroll
            for (int e = 0; e < kEnt; e++) {
                const double fx = fma(c[e].x, ix, -c[e].y * iy), fy = fma(c[e].x, iy, c[e].y * ix);
                const double qx = e > ek ? rx : e < ek ? mx : ex, qy = e > ek ? ry : e < ek ? my : ey;
                x[e] = fma(-fx, qx, fma(fy, qy, x[e]));
                y[e] = fma(-fx, qy, fma(-fy, qx, y[e]));
            }
        }
    }
    __syncthreads();
    if (tid < kNB) {
        const double d = s_piv[0][tid].x;
        const double2 p = s_piv[1][tid];
        const PanelPivot pv(d, p);
        s_sign[tid] = pv.s;
        s_inv[tid] = pv.inv;
        s_u[tid] = make_double2(fma(-pv.s.x, d * pv.rd, p.x), fma(-pv.s.y, d * pv.rd, p.y));
        // a real pivot with no weight left below it needs no reflection
        if (tid < nb && p.y == 0 && d - p.x * p.x <= 1e-12 * (p.x * p.x)) s_flat = 1;
    }
    __syncthreads();
    // G = U0^H D^-1 U0, D = diag(U0): R = D^-1/2 U0, R^-1 = U0^-1 D^1/2; the
    // condition number of the panel with its columns scaled to norm 1.  The lanes
    // of G form Ri = R^-1 S^H and R_h = S R, those of P_1 - S R form -U and L.
    double2 first[kEnt], second[kEnt];
    double k2 = 0;
    {
        const double2 sgn = s_sign[j], inv = s_inv[j];
        const double dj = s_piv[0][j].x, rj = dj * rsq_step(dj);
#pragma unroll
        for (int e = 0; e < kEnt; e++) {
            const int i = w + kRecWaves * e;
            const bool up = j >= i, off = j > i;
            const double ri = rsq_step(s_piv[0][i].x);
            const double2 ra = s_row[0][i][j], si = s_sign[i], ui = s_u[i];
            const double2 r = make_double2(off ? ra.x * ri : 0.0, off ? ra.y * ri : 0.0);
            const double2 Rh = zmul(si, make_double2(j == i ? rj : r.x, r.y));
            const double2 Ri = make_double2(up ? x[e] * rj : 0.0, up ? y[e] * rj : 0.0);
            const double2 Ris = zmul(Ri, make_double2(sgn.x, -sgn.y));
            const double2 u = zfms(s_row[1][i][j], si, r), l = zmul(s_cw[j][i], inv);
            k2 = top ? 0.0 : fma(kNB * s_g[i], fma(Ri.x, Ri.x, Ri.y * Ri.y), k2);
            first[e].x = !top ? Ris.x : off ? -u.x : j == i ? -ui.x : 0.0;
            first[e].y = !top ? Ris.y : off ? -u.y : j == i ? -ui.y : 0.0;
            second[e].x = !top ? Rh.x : up ? (j == i ? 1.0 : 0.0) : l.x;
            second[e].y = !top ? Rh.y : up ? 0.0 : l.y;
        }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) k2 += __shfl_xor(k2, m, 64);
    if (lane == 0) s_w[w] = k2;
    __syncthreads();
    k2 = 0;
#pragma unroll
    for (int q = 0; q < kRecWaves; q++) k2 += s_w[q];
    const bool take = k2 <= kPanelCond2 && !s_flat;  // (not a NaN)
    if (tid == 0 && seen) __hip_atomic_store(seen, take ? 0 : 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (!take) {
        __syncthreads();
        panel_one_wg<float>(A, lda, M, j0, nb, Tout, 1, (float2(*)[kNB])&s_row[0][0][0],
                            (float2(*)[kNB])&s_row[1][0][0]);
        if (tid == 0) *bad = 1;
        return;
    }
    if (tid == 0) *bad = 0;
    // T = -U (R^-1 S^H) L^-H: rows of entries 2 top, 2 top + 1 of the wave
#pragma unroll
    for (int e = 0; e < kEnt; e++) {
        const int i = w + kRecWaves * e;
        s_row[top][i][j] = first[e];
        if (top) s_cw[j][i] = make_double2(i == j ? 1.0 : j > i ? 0.0 : x[e], j >= i ? 0.0 : -y[e]);  // L^-H
    }
    const int e0 = top ? kEnt / 2 : 0;
    double2 t[kEnt / 2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kEnt / 2; e++) t[e] = make_double2(0.0, 0.0);
#pragma unroll 4
        for (int k = 0; k < kNB; k++) {
            const double2 v = s_cw[k][j];
#pragma unroll
            for (int e = 0; e < kEnt / 2; e++) t[e] = zfms(t[e], s_row[h][w + kRecWaves * (e0 + e)][k], v);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kEnt / 2; e++) {
            const int i = w + kRecWaves * (e0 + e);
            if (h == 0) s_cw[i][j] = t[e];
            else {
                const bool iu = j >= i && j < nb;
                Tout[i * kNB + j] = make_float2(iu ? (float)t[e].x : 0.f, iu ? (float)t[e].y : 0.f);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kEnt; e++) {
        const int i = w + kRecWaves * e;
        const bool iu = j >= i && j < nb, low = j < nb && j < i;
        const float2 v = make_float2((float)second[e].x, (float)second[e].y);
        if (top) Y[i * kNB + j] = make_double2(iu ? x[e] : 0.0, iu ? y[e] : 0.0);
        if (i < Mp) {
            if (top ? low : iu) A[(size_t)(j0 + j) * lda + j0 + i] = v;
            if (top) Vd[(size_t)j * ldv + i] = j < nb ? v : make_float2(0.f, 0.f);
        }
    }
}

// Rows 32.. of V = P_2 U^-1 to the panel and to Vd, on FP64 MFMA in the
// three-product form: 64 rows a workgroup, 16 a wave; U^-1 is the operand of the
// result's rows, so that 16 lanes store 16 consecutive rows of a column.  With
// *bad, Vd from the panel's reflectors, all rows.
__global__ __launch_bounds__(256) void qr_form_v(const float2 *__restrict__ Pc, const double2 *__restrict__ Y,
                                                 const int *__restrict__ bad, float2 *__restrict__ A, long lda, int M,
                                                 int j0, int nb, float2 *__restrict__ Vd, long ldv) {
    typedef double v4d __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kk = lane >> 4;
    const int i = blockIdx.x * 64 + 16 * wave + m, ic = min(i, M - j0 - 1);
    float2 p[kNB / 4];
    double2 y[kNB / 4][2];
#pragma unroll
    for (int u = 0; u < kNB / 4; u++) {
        p[u] = Pc[(size_t)(4 * u + kk) * ldv + ic];
#pragma unroll
        for (int g = 0; g < 2; g++) y[u][g] = Y[(4 * u + kk) * kNB + 16 * g + m];
    }
    if (*bad) {
        if (j0 + i < M)
            for (int c = kk; c < kNB; c += 4)
                Vd[(size_t)c * ldv + i] =
                    c < nb ? vget((const float2 *)A, lda, j0, c, j0 + i) : make_float2(0.f, 0.f);
        return;
    }
    v4d acc[2][3];
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int q = 0; q < 3; q++) acc[g][q] = (v4d){0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < kNB / 4; u++) {
        const double pr = p[u].x, pi = p[u].y;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const double yr = y[u][g].x, yi = y[u][g].y;
            acc[g][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(yr, pr + pi, acc[g][0], 0, 0, 0);
            acc[g][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(yr + yi, pi, acc[g][1], 0, 0, 0);
            acc[g][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(yi - yr, pr, acc[g][2], 0, 0, 0);
        }
    }
    if (i < kNB || j0 + i >= M) return;
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int c = 16 * g + kk + 4 * q;
            const float2 v = make_float2((float)(acc[g][0][q] - acc[g][1][q]), (float)(acc[g][0][q] + acc[g][2][q]));
            if (c < nb) A[(size_t)(j0 + c) * lda + j0 + i] = v;
            Vd[(size_t)c * ldv + i] = v;  // (zero past nb)
        }
}

// FP32 panels of a matrix whose panels the Gram matrix does not take (PanelRoute):
// one launch per column, the rows split over workgroups (one row per thread).
// Launch jj applies the reflector of column jj to the workgroup's rows and then forms
// the partials of column jj + 1 from the updated rows: |x|^2 below its
// diagonal and sum conj(x_r) a_c(r) for the later columns c, x being the
// column below the diagonal before scaling.  With v = x / (alpha - beta) below
// the diagonal and v_j = 1,
//   v^H a_c = a_c(j) + conj(scale) sum_{r > j} conj(x_r) a_c(r),
// so the reflector's products need no pass of their own after its norm.  The
// partials are summed in a fixed order by every workgroup of the next launch.
// Row j of the panel (alpha and the a_c(j)) travels in its own buffer,
// written by the workgroup holding the row, because that workgroup overwrites
// the row during the launch that reads it.  jj = -1 only forms the partials of
// column 0.  Column indices are runtime values here, so the row is walked with
// compile-time column loops and compares, never by a runtime register index.
// Leaves the reflectors and R in place and tau_jj on Tout's diagonal.
template <int NT>
__global__ __launch_bounds__(NT) void qr_panel_col(float2 *A, long lda, int M, int j0, int jj, const float *zin,
                                                   const float2 *rin, float *zout, float2 *rout, int nblk,
                                                   float2 *Tout) {
    __shared__ float s_red[NT / 64][2 * kNB];
    __shared__ float s_z[2 * kNB];
    __shared__ float2 s_d[kNB];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int i = j0 + blockIdx.x * NT + tid;
    const bool live = i < M;
    const int ic = min(i, M - 1);
    float2 a[kNB];
#pragma unroll
    for (int c = 0; c < kNB; c++) a[c] = A[(size_t)(j0 + c) * lda + ic];
    if (jj >= 0) {
        const int j = j0 + jj;
        if (tid < 2 * kNB) {
            float t = 0.f;
            for (int q = 0; q < nblk; q++) t += zin[(size_t)q * 2 * kNB + tid];
            s_z[tid] = t;
        }
        __syncthreads();
        const float tot = s_z[2 * jj];
        const float2 alpha = rin[jj];
        const float aa = sqrtf(alpha.x * alpha.x + alpha.y * alpha.y);
        const float xnorm = sqrtf(aa * aa + tot);
        float tau = 0.f;
        float2 scale = make_float2(0.f, 0.f), beta = alpha;
        if (tot > 0 || (xnorm > 0 && alpha.y != 0)) {
            const float phr = aa > 0 ? alpha.x / aa : 1.f, phi = aa > 0 ? alpha.y / aa : 0.f;
            beta = make_float2(-phr * xnorm, -phi * xnorm);
            const float dr = alpha.x - beta.x, di = alpha.y - beta.y;
            const float dd = dr * dr + di * di;
            scale = make_float2(dr / dd, -di / dd);
            tau = 2.f / (1.f + tot / dd);
        }
        if (tid < kNB) {
            const int c = tid;
            float2 d = make_float2(0.f, 0.f);
            if (c > jj) {
                // tau (a_c(j) + conj(scale) S_c)
                const float sx = s_z[2 * c], sy = s_z[2 * c + 1];
                const float2 ac = rin[c];
                d.x = tau * (ac.x + scale.x * sx + scale.y * sy);
                d.y = tau * (ac.y + scale.x * sy - scale.y * sx);
            }
            s_d[c] = d;
        }
        if (blockIdx.x == 0 && tid == 0) Tout[jj * kNB + jj] = make_float2(tau, 0.f);
        __syncthreads();
        if (live && i >= j) {
            float2 x = make_float2(0.f, 0.f);
#pragma unroll
            for (int c = 0; c < kNB; c++)
                if (c == jj) x = a[c];
            const bool below = i > j;
            const float2 v = below ? make_float2(x.x * scale.x - x.y * scale.y, x.x * scale.y + x.y * scale.x)
                                   : make_float2(1.f, 0.f);
#pragma unroll
            for (int c = 0; c < kNB; c++) {
                if (c == jj) {
                    a[c] = below ? v : beta;
                } else if (c > jj) {
                    const float2 d = s_d[c];
                    a[c].x -= d.x * v.x - d.y * v.y;
                    a[c].y -= d.x * v.y + d.y * v.x;
                }
                if (c >= jj) A[(size_t)(j0 + c) * lda + i] = a[c];
            }
        }
    }
    if (jj + 1 < kNB) {
        const int k = jj + 1, j1 = j0 + k;
        float2 x = make_float2(0.f, 0.f);
#pragma unroll
        for (int c = 0; c < kNB; c++)
            if (c == k) x = a[c];
        const bool below = live && i > j1;
        float z[2 * kNB];
#pragma unroll
        for (int c = 0; c < kNB; c++) {
            float pr = 0.f, pi = 0.f;
            if (below) {
                if (c == k) {
                    pr = x.x * x.x + x.y * x.y;
                } else if (c > k) {
                    pr = x.x * a[c].x + x.y * a[c].y;
                    pi = x.x * a[c].y - x.y * a[c].x;
                }
            }
            z[2 * c] = pr;
            z[2 * c + 1] = pi;
        }
        if (live && i == j1) {
#pragma unroll
            for (int c = 0; c < kNB; c++)
                if (c >= k) rout[c] = a[c];
        }
        wave_reduce_scatter64(z, lane);
        s_red[wid][lane] = z[0];
        __syncthreads();
        if (tid < 2 * kNB) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < NT / 64; w++) t += s_red[w][tid];
            zout[(size_t)blockIdx.x * 2 * kNB + tid] = t;
        }
    }
}

// T of the compact WY form from the taus (on Tout's diagonal) and
// Y[m * ldy + l] = (V^H V)[l][m]: LAPACK larft, forward columnwise, as in qr_panel
template <typename T>
__global__ void qr_make_t(typename QT<T>::c2 *Tout, int nb, const typename QT<T>::c2 *Y, int ldy) {
    using C2 = typename QT<T>::c2;
    __shared__ C2 s_T[kNB][kNB];
    __shared__ C2 s_Y[kNB][kNB + 1];
    __shared__ T s_tau[kNB];
    const int tid = threadIdx.x;
    if (tid < kNB) s_tau[tid] = Tout[tid * kNB + tid].x;
    for (int p = tid; p < kNB * kNB; p += blockDim.x) {
        s_T[p / kNB][p % kNB].x = 0;
        s_T[p / kNB][p % kNB].y = 0;
        // the serial column loop below reads Y from shared memory only
        s_Y[p / kNB][p % kNB] = Y[(size_t)(p / kNB) * ldy + p % kNB];
    }
    __syncthreads();
    for (int m = 0; m < nb; m++) {
        if (tid < m) {
            T zr = 0, zi = 0;
            for (int q = tid; q < m; q++) {
                const C2 t = s_T[tid][q], y = s_Y[m][q];
                zr += t.x * y.x - t.y * y.y;
                zi += t.x * y.y + t.y * y.x;
            }
            s_T[tid][m].x = -s_tau[m] * zr;
            s_T[tid][m].y = -s_tau[m] * zi;
        } else if (tid == m) {
            s_T[m][m].x = s_tau[m];
        }
        __syncthreads();
    }
    for (int p = tid; p < kNB * kNB; p += blockDim.x) Tout[p] = s_T[p / kNB][p % kNB];
}

// W[:, c] = op(T) (V^H C[:, c]); op = conj-transpose (apply Q^H) or identity (apply Q)
template <typename T>
__global__ __launch_bounds__(256) void qr_vhc(const typename QT<T>::c2 *A, long lda, int M, int j0, int nb,
                                              const typename QT<T>::c2 *Tm, const typename QT<T>::c2 *C, long ldc,
                                              typename QT<T>::c2 *W, int conjT) {
    using C2 = typename QT<T>::c2;
    __shared__ T red[2][4][kNB];
    __shared__ C2 z[kNB];
    const int c = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const C2 *cc = C + (size_t)c * ldc;
    T zr[kNB], zi[kNB];
#pragma unroll
    for (int l = 0; l < kNB; l++) {
        zr[l] = 0;
        zi[l] = 0;
    }
    for (int i = j0 + tid; i < M; i += 256) {
        const C2 a = cc[i];
#pragma unroll
        for (int l = 0; l < kNB; l++) {
            if (l < nb) {
                const C2 v = vget(A, lda, j0, l, i);
                zr[l] += v.x * a.x + v.y * a.y;
                zi[l] += v.x * a.y - v.y * a.x;
            }
        }
    }
#pragma unroll
    for (int l = 0; l < kNB; l++) {
        const T r = wsum(zr[l]), im = wsum(zi[l]);
        if (lane == 0) {
            red[0][wid][l] = r;
            red[1][wid][l] = im;
        }
    }
    __syncthreads();
    if (tid < nb) {
        C2 s;
        s.x = red[0][0][tid] + red[0][1][tid] + red[0][2][tid] + red[0][3][tid];
        s.y = red[1][0][tid] + red[1][1][tid] + red[1][2][tid] + red[1][3][tid];
        z[tid] = s;
    }
    __syncthreads();
    if (tid < nb) {
        // w = T^H z (conjT) or T z
        T wr = 0, wi = 0;
        for (int q = 0; q < nb; q++) {
            C2 t = conjT ? Tm[q * kNB + tid] : Tm[tid * kNB + q];
            if (conjT) t.y = -t.y;
            wr += t.x * z[q].x - t.y * z[q].y;
            wi += t.x * z[q].y + t.y * z[q].x;
        }
        C2 o;
        o.x = wr;
        o.y = wi;
        W[(size_t)c * kNB + tid] = o;
    }
}

// C[i, c] -= sum_l V[i, l] W[l, c]
template <typename T>
__global__ __launch_bounds__(256) void qr_update(const typename QT<T>::c2 *A, long lda, int M, int j0, int nb,
                                                 const typename QT<T>::c2 *W, typename QT<T>::c2 *C, long ldc) {
    using C2 = typename QT<T>::c2;
    __shared__ C2 w[kNB];
    const int c = blockIdx.y;
    const int i = j0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (threadIdx.x < nb) w[threadIdx.x] = W[(size_t)c * kNB + threadIdx.x];
    __syncthreads();
    if (i >= M) return;
    T sr = 0, si = 0;
    for (int l = 0; l < nb; l++) {
        const C2 v = vget(A, lda, j0, l, i);
        sr += v.x * w[l].x - v.y * w[l].y;
        si += v.x * w[l].y + v.y * w[l].x;
    }
    C2 *p = C + (size_t)c * ldc + i;
    C2 o = *p;
    o.x -= sr;
    o.y -= si;
    *p = o;
}

// Vd[l][i - j0] = V[i, l] of the panel (explicit unit diagonal and zeros above
// it; columns l >= nb zero), rows j0..M-1, 32 columns, ld ldvd
template <typename T>
__global__ void k_build_v(const typename QT<T>::c2 *A, long lda, int M, int j0, int nb, typename QT<T>::c2 *Vd,
                          long ldvd) {
    using C2 = typename QT<T>::c2;
    const int i = j0 + blockIdx.x * blockDim.x + threadIdx.x;
    const int l = blockIdx.y;
    if (i >= M) return;
    C2 z;
    if (l < nb) {
        z = vget(A, lda, j0, l, i);
    } else {
        z.x = 0;
        z.y = 0;
    }
    Vd[(size_t)l * ldvd + (i - j0)] = z;
}

// R x = b (upper, non-unit), one workgroup per right-hand side, in place in B.
template <typename T>
__global__ __launch_bounds__(1024) void trsv_upper(const typename QT<T>::c2 *Rm, long ldr, int N,
                                                   typename QT<T>::c2 *B, long ldb) {
    using C2 = typename QT<T>::c2;
    __shared__ C2 xj;
    C2 *b = B + (size_t)blockIdx.x * ldb;
    for (int j = N - 1; j >= 0; j--) {
        if (threadIdx.x == 0) {
            const C2 r = Rm[(size_t)j * ldr + j], v = b[j];
            const T d = r.x * r.x + r.y * r.y;
            C2 x;
            x.x = (v.x * r.x + v.y * r.y) / d;
            x.y = (v.y * r.x - v.x * r.y) / d;
            b[j] = x;
            xj = x;
        }
        __syncthreads();
        const C2 x = xj;
        const C2 *rc = Rm + (size_t)j * ldr;
        for (int i = threadIdx.x; i < j; i += blockDim.x) {
            const C2 r = rc[i];
            C2 o = b[i];
            o.x -= r.x * x.x - r.y * x.y;
            o.y -= r.x * x.y + r.y * x.x;
            b[i] = o;
        }
        __syncthreads();
    }
}

// Whole least-squares solve of a small factored system in one workgroup per
// right-hand side, b held in shared memory (M entries, dynamic): Q^H b panel
// by panel (z = V^H b as one scattered reduction of the kNB products, w = T^H z,
// b -= V w), then R x = b[0:N] by blocks of kNB columns from the bottom: one
// wave solves the diagonal block with the block's rows of R in registers, then
// the whole workgroup removes the block's unknowns from the rows above.  The
// same arithmetic as qr_vhc + qr_update + trsv_upper without their 3 np + N
// launches and barrier steps.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void qr_solve_small(const typename QT<T>::c2 *A, long lda, int M, int N,
                                                     const typename QT<T>::c2 *Tb, typename QT<T>::c2 *B, long ldb) {
    using C2 = typename QT<T>::c2;
    extern __shared__ unsigned char qss_raw[];
    C2 *sb = (C2 *)qss_raw;
    __shared__ T s_red[NT / 64][2 * kNB];
    __shared__ C2 s_z[kNB], s_w[kNB];
    __shared__ C2 s_T[kNB * kNB];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    C2 *b = B + (size_t)blockIdx.x * ldb;
    for (int i = tid; i < M; i += NT) sb[i] = b[i];
    // Every load below is unconditional from a clamped, valid address, with
    // the unit diagonal, the zeros above it and columns past N selected
    // afterwards, so the loads of a thread are all in flight together.
    const int np = (N + kNB - 1) / kNB;
    for (int p = 0; p < np; p++) {
        const int j0 = p * kNB, nb = min(kNB, N - j0);
        for (int e = tid; e < kNB * kNB; e += NT) s_T[e] = Tb[(size_t)p * kNB * kNB + e];
        __syncthreads();  // sb (first panel) and s_T
        T x[2 * kNB];
#pragma unroll
        for (int l = 0; l < 2 * kNB; l++) x[l] = 0;
        for (int i = j0 + tid; i < M; i += NT) {
            const C2 bi = sb[i];
#pragma unroll
            for (int l0 = 0; l0 < kNB; l0 += kCG) {
                C2 raw[kCG];
#pragma unroll
                for (int u = 0; u < kCG; u++) raw[u] = A[(size_t)min(j0 + l0 + u, N - 1) * lda + i];
#pragma unroll
                for (int u = 0; u < kCG; u++) {
                    const int l = l0 + u;
                    const bool below = i > j0 + l && l < nb, diag = i == j0 + l && l < nb;
                    const T vx = below ? raw[u].x : (diag ? (T)1 : (T)0), vy = below ? raw[u].y : (T)0;
                    x[2 * l] += vx * bi.x + vy * bi.y;
                    x[2 * l + 1] += vx * bi.y - vy * bi.x;
                }
                __builtin_amdgcn_sched_barrier(0);  // one chunk's loads live at a time
            }
        }
        wave_reduce_scatter64(x, lane);
        s_red[wid][lane] = x[0];
        __syncthreads();
        if (tid < 2 * kNB) {
            T t = 0;
#pragma unroll
            for (int w = 0; w < NT / 64; w++) t += s_red[w][tid];
            ((T *)s_z)[tid] = t;
        }
        __syncthreads();
        if (tid < nb) {
            // w = T^H z; T upper triangular
            T wr = 0, wi = 0;
            for (int q = 0; q <= tid; q++) {
                const C2 t = s_T[q * kNB + tid];
                wr += t.x * s_z[q].x + t.y * s_z[q].y;
                wi += t.x * s_z[q].y - t.y * s_z[q].x;
            }
            s_w[tid].x = wr;
            s_w[tid].y = wi;
        } else if (tid < kNB) {
            // a narrow last panel: these meet zeros below, which shared
            // memory's old contents (infinities, NaNs) would not survive
            s_w[tid].x = 0;
            s_w[tid].y = 0;
        }
        __syncthreads();
        for (int i = j0 + tid; i < M; i += NT) {
            T sr = 0, si = 0;
#pragma unroll
            for (int l0 = 0; l0 < kNB; l0 += kCG) {
                C2 raw[kCG];
#pragma unroll
                for (int u = 0; u < kCG; u++) raw[u] = A[(size_t)min(j0 + l0 + u, N - 1) * lda + i];
#pragma unroll
                for (int u = 0; u < kCG; u++) {
                    const int l = l0 + u;
                    const bool below = i > j0 + l && l < nb, diag = i == j0 + l && l < nb;
                    const T vx = below ? raw[u].x : (diag ? (T)1 : (T)0), vy = below ? raw[u].y : (T)0;
                    sr += vx * s_w[l].x - vy * s_w[l].y;
                    si += vx * s_w[l].y + vy * s_w[l].x;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            sb[i].x -= sr;
            sb[i].y -= si;
        }
        __syncthreads();  // sb, and s_T / s_w before the next panel
    }
    for (int p = np - 1; p >= 0; p--) {
        const int c0 = p * kNB, nb = min(kNB, N - c0);
        if (wid == 0) {
            // lane l owns row c0 + l of the diagonal block
            const int r = c0 + lane, rc = min(r, N - 1);
            C2 rr[kNB];
#pragma unroll
            for (int m = 0; m < kNB; m++) rr[m] = A[(size_t)min(c0 + m, N - 1) * lda + rc];
#pragma unroll
            for (int m = 0; m < kNB; m++) {
                if (!(lane < nb && m < nb && m >= lane)) {
                    rr[m].x = 0;
                    rr[m].y = 0;
                }
            }
            C2 bl = sb[rc];
            if (lane >= nb) {
                bl.x = 0;
                bl.y = 0;
            }
#pragma unroll
            for (int m = kNB - 1; m >= 0; m--) {
                if (m < nb) {
                    // lane m divides by the diagonal; everyone takes x_m from it
                    C2 xm;
                    const T d = rr[m].x * rr[m].x + rr[m].y * rr[m].y;
                    xm.x = lane == m ? (bl.x * rr[m].x + bl.y * rr[m].y) / d : 0;
                    xm.y = lane == m ? (bl.y * rr[m].x - bl.x * rr[m].y) / d : 0;
                    xm.x = __shfl(xm.x, m, 64);
                    xm.y = __shfl(xm.y, m, 64);
                    if (lane < m) {
                        bl.x -= rr[m].x * xm.x - rr[m].y * xm.y;
                        bl.y -= rr[m].x * xm.y + rr[m].y * xm.x;
                    } else if (lane == m) {
                        bl = xm;
                    }
                }
            }
            if (lane < nb) sb[r] = bl;
        }
        __syncthreads();
        for (int i = tid; i < c0; i += NT) {
            T sr = 0, si = 0;
#pragma unroll
            for (int m0 = 0; m0 < kNB; m0 += kCG) {
                C2 raw[kCG];
#pragma unroll
                for (int u = 0; u < kCG; u++) raw[u] = A[(size_t)min(c0 + m0 + u, N - 1) * lda + i];
#pragma unroll
                for (int u = 0; u < kCG; u++) {
                    if (m0 + u < nb) {
                        const C2 xv = sb[c0 + m0 + u];
                        sr += raw[u].x * xv.x - raw[u].y * xv.y;
                        si += raw[u].x * xv.y + raw[u].y * xv.x;
                    }
                }
            }
            sb[i].x -= sr;
            sb[i].y -= si;
        }
        __syncthreads();
    }
    for (int i = tid; i < N; i += NT) b[i] = sb[i];
}

// Solves with a factored system, by groups of kGB panels (kGW columns).  A group's
// reflectors act as one block, I - V T V^H with V the kGB panels side by side,
// and its diagonal block of R is used through its inverse, so Q^H b takes one
// launch per group and the back substitution another, instead of one per
// panel; the launches are bound by latency (each a few loads deep), so their
// number is what counts.  The two kGW x kGW triangles of every group are formed
// once after the factorisation (qr_cross, qr_group, 70 us), in FP64.  A solve of
// 642 unknowns takes 13 launches of 7 to 12 us, where a launch per panel took 43
// of 8 to 10.  QR solve with refinement: 642 nodes 2.8 -> 2.3 ms, 1962: 9.1 ->
// 6.9, 10242: 150 -> 128.
constexpr int kGB = 4, kGW = kGB * kNB, kGG = kGW * kGW;
constexpr int kPairs = kGB * (kGB - 1) / 2;  // panels s < t of a group

__device__ __forceinline__ double2 to_d2(float2 v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ double2 to_d2(double2 v) { return v; }

// V's entry of row i and column c (unit diagonal, zero above it), from the
// matrix's
template <typename C2>
__device__ __forceinline__ C2 v_entry(C2 raw, int i, int c) {
    C2 z;
    z.x = i > c ? raw.x : i == c ? 1 : 0;
    z.y = i > c ? raw.y : 0;
    return z;
}

// Workgroups of the pairs: cross[((g kPairs + q) nsplit + split)][i][j] = the
// split's part of V_s^H V_t, q the pair (s, t) of group g, on FP64 MFMA (as
// qr_gram).  Workgroups past them (one per panel): Rinv[p], the inverse of the
// panel's diagonal block of R, lane j of one wave its column j by back
// substitution.  Both zero past N.
template <typename T>
__global__ __launch_bounds__(256) void qr_cross(const typename QT<T>::c2 *__restrict__ A, long lda, int M, int N,
                                                int npair, int nsplit, double2 *__restrict__ cross,
                                                double2 *__restrict__ Rinv) {
    using C2 = typename QT<T>::c2;
    typedef double v4d __attribute__((ext_vector_type(4)));
    constexpr int kRows = 32;
    __shared__ double2 s_v[2][kNB][kRows + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int np = (N + kNB - 1) / kNB;
    if ((int)blockIdx.x >= npair * nsplit) {
        const int c0 = (blockIdx.x - npair * nsplit) * kNB, nb = min(kNB, N - c0);
        double2(*s_r)[kRows + 1] = s_v[0];
        for (int e = tid; e < kNN; e += 256) {
            const int i = e % kNB, k = e / kNB;
            double2 v = make_double2(i == k ? 1.0 : 0.0, 0.0);
            if (i <= k && k < nb) v = to_d2(A[(size_t)(c0 + k) * lda + c0 + i]);
            s_r[i][k] = v;
        }
        __syncthreads();
        if (tid < kNB) {
            const int j = tid;
            double tx[kNB], ty[kNB];
#pragma unroll
            for (int i = kNB - 1; i >= 0; i--) {
                double sr = i == j ? 1.0 : 0.0, si = 0;
#pragma unroll
                for (int k = i + 1; k < kNB; k++) {
                    const double2 r = s_r[i][k];
                    sr = fma(-r.x, tx[k], fma(r.y, ty[k], sr));
                    si = fma(-r.x, ty[k], fma(-r.y, tx[k], si));
                }
                const double2 d = s_r[i][i];
                const double q = 1.0 / fma(d.x, d.x, d.y * d.y);
                tx[i] = fma(sr, d.x, si * d.y) * q;
                ty[i] = fma(si, d.x, -sr * d.y) * q;
            }
            double2 *out = Rinv + (size_t)(c0 / kNB) * kNN;
#pragma unroll
            for (int i = 0; i < kNB; i++) {
                const bool in = i <= j && j < nb;
                out[i * kNB + j] = make_double2(in ? tx[i] : 0.0, in ? ty[i] : 0.0);
            }
        }
        return;
    }
    const int pair = blockIdx.x / nsplit, split = blockIdx.x % nsplit;
    const int g = pair / kPairs, q = pair % kPairs;
    const int t = q >= 3 ? 3 : q >= 1 ? 2 : 1, sp = q - t * (t - 1) / 2;  // (0,1) (0,2) (1,2) (0,3) (1,3) (2,3)
    const int ps = g * kGB + sp, pt = g * kGB + t;
    const int m = lane & 15, kk = lane >> 4, a0 = 16 * (wave & 1), b0 = 16 * (wave >> 1);
    v4d acc[3];
#pragma unroll
    for (int c = 0; c < 3; c++) acc[c] = (v4d){0, 0, 0, 0};
    if (pt < np) {
        // rows from panel t's first on (V_t is zero above), in chunks
        const int r0 = pt * kNB, nch = (M - r0 + kRows - 1) / kRows;
        const int per = (nch + nsplit - 1) / nsplit, ch1 = min(nch, (split + 1) * per);
        for (int ch = split * per; ch < ch1; ch++) {
            const int i = r0 + ch * kRows + (tid & 31), ic = min(i, M - 1);
            double2 v[2][kNB / 8];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int u = 0; u < kNB / 8; u++) {
                    const int c = (h ? pt : ps) * kNB + (tid >> 5) + 8 * u;
                    const C2 raw = A[(size_t)min(c, N - 1) * lda + ic];
                    v[h][u] = i < M && c < N ? to_d2(v_entry(raw, i, c)) : make_double2(0.0, 0.0);
                }
            __syncthreads();  // the previous rows are read
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int u = 0; u < kNB / 8; u++) s_v[h][(tid >> 5) + 8 * u][tid & 31] = v[h][u];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kRows; r += 4) {
                const double2 x = s_v[0][a0 + m][r + kk], y = s_v[1][b0 + m][r + kk];
                const double ur = x.x, ui = -x.y, vr = y.x, vi = y.y;
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ur, vr + vi, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ur + ui, vi, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(ui - ur, vr, acc[2], 0, 0, 0);
            }
        }
    }
    double2 *out = cross + (size_t)blockIdx.x * kNN;
#pragma unroll
    for (int v = 0; v < 4; v++)
        out[(a0 + kk + 4 * v) * kNB + b0 + m] = make_double2(acc[0][v] - acc[1][v], acc[0][v] + acc[2][v]);
}

// The triangles of a group: G = T (GT[g][k kGW + l] = T_kl), whose inverse has
// the panels' T^-1 on its diagonal and V_s^H V_t above it, and G = R_gg^-1
// (GR[g][k kGW + l] = (R_gg^-1)_lk, so that both are read with l across the
// lanes).  Blocks of column t from the diagonal up,
//   G_tt = D_t,  G_st = -D_s sum_{u = s+1..t} O_su G_ut,
// D the panels' T or Rinv, O the cross products or R.  One workgroup per column
// t (blockIdx.y) and triangle (blockIdx.z), thread (i, j) one entry of a block,
// FP64; the finished blocks of the column stay in shared memory.
template <typename T>
__global__ __launch_bounds__(1024) void qr_group(const typename QT<T>::c2 *__restrict__ A, long lda, int N,
                                                 const typename QT<T>::c2 *__restrict__ Tb,
                                                 const double2 *__restrict__ cross, int nsplit,
                                                 const double2 *__restrict__ Rinv, double2 *__restrict__ GT,
                                                 double2 *__restrict__ GR) {
    __shared__ double2 s_o[kNB][kNB + 1], s_g[kNB][kNB];
    const int i = threadIdx.x >> 5, j = threadIdx.x & 31;
    const int g = blockIdx.x, t = blockIdx.y;
    const bool tri_r = blockIdx.z;
    const int np = (N + kNB - 1) / kNB;
    double2 *out = (tri_r ? GR : GT) + (size_t)g * kGG;
    auto diag = [&](int sp) {  // entry (i, j) of D_sp
        const int p = g * kGB + sp;
        if (p >= np) return make_double2(0.0, 0.0);
        return tri_r ? Rinv[(size_t)p * kNN + threadIdx.x] : to_d2(Tb[(size_t)p * kNN + threadIdx.x]);
    };
    auto off = [&](int sp, int u) {  // entry (i, j) of O_su, sp < u
        const int ps = g * kGB + sp, pu = g * kGB + u;
        double2 v = make_double2(0.0, 0.0);
        if (pu >= np) return v;
        if (tri_r) {
            const int c = pu * kNB + j;
            return c < N ? to_d2(A[(size_t)c * lda + ps * kNB + i]) : v;
        }
        const double2 *x = cross + (size_t)(g * kPairs + u * (u - 1) / 2 + sp) * nsplit * kNN + threadIdx.x;
        for (int k = 0; k < nsplit; k++) {
            const double2 w = x[(size_t)k * kNN];
            v.x += w.x;
            v.y += w.y;
        }
        return v;
    };
    auto store = [&](int sp, double2 v) {
        const int k = sp * kNB + i, l = t * kNB + j;
        out[tri_r ? l * kGW + k : k * kGW + l] = v;
    };
    double2 own[kGB];  // this thread's entries of G_tt, G_{t-1,t}, ..
    own[0] = diag(t);
    store(t, own[0]);
    for (int sp = t + 1; sp < kGB; sp++) store(sp, make_double2(0.0, 0.0));
#pragma unroll
    for (int d = 1; d < kGB; d++) {
        const int sp = t - d;
        if (sp < 0) break;
        double2 acc = make_double2(0.0, 0.0);
        const double2 dd = diag(sp);
#pragma unroll
        for (int e = 0; e < d; e++) {  // u = t - e
            const double2 o = off(sp, t - e);
            __syncthreads();
            s_o[i][j] = o;
            s_g[i][j] = own[e];
            __syncthreads();
#pragma unroll 8
            for (int k = 0; k < kNB; k++) acc = zfms(acc, s_o[i][k], s_g[k][j]);
        }
        __syncthreads();
        s_o[i][j] = dd;
        s_g[i][j] = make_double2(-acc.x, -acc.y);
        __syncthreads();
        acc = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int k = 0; k < kNB; k++) acc = zfms(acc, s_o[i][k], s_g[k][j]);
        own[d] = acc;
        store(sp, acc);
    }
}

// s_w[h][l] = part h of sum_k f(G[k][l], s_z[k]) over the kGW / 2 entries k of
// half h = tid / kGW, l = tid % kGW, f = conj(g) z (CONJ) or g z; the sum of the
// two parts is the product.  The first loads are independent of s_z: the
// caller's barrier that completes s_z is between them and the products.
template <bool CONJ>
struct TriProduct {
    static constexpr int kLoads = kGW / 8;  // in flight
    const double2 *Gl;
    double2 v[kLoads];
    __device__ __forceinline__ TriProduct(const double2 *G) {
        Gl = G + (size_t)(threadIdx.x / kGW) * (kGW / 2) * kGW + threadIdx.x % kGW;
#pragma unroll
        for (int k = 0; k < kLoads; k++) v[k] = Gl[(size_t)k * kGW];
    }
    __device__ __forceinline__ double2 apply(const double2 *s_z) {
        const double2 *z = s_z + (threadIdx.x / kGW) * (kGW / 2);
        double sr = 0, si = 0;
#pragma unroll
        for (int k0 = 0; k0 < kGW / 2; k0 += kLoads) {
            double2 n[kLoads];
            if (k0 + kLoads < kGW / 2) {
#pragma unroll
                for (int k = 0; k < kLoads; k++) n[k] = Gl[(size_t)(k0 + kLoads + k) * kGW];
            }
#pragma unroll
            for (int k = 0; k < kLoads; k++) {
                const double2 x = z[k0 + k];
                const double gy = CONJ ? -v[k].y : v[k].y;
                sr = fma(v[k].x, x.x, fma(-gy, x.y, sr));
                si = fma(v[k].x, x.y, fma(gy, x.x, si));
            }
            if (k0 + kLoads < kGW / 2) {
#pragma unroll
                for (int k = 0; k < kLoads; k++) v[k] = n[k];
            }
        }
        return make_double2(sr, si);
    }
};

// Launch g of Q^H B (g = -1, 0, ..): finishes group g on the workgroup's rows
// (z = sum of the partials of V_g^H b in a fixed order, w = T_g^H z, b -= V_g w),
// then forms their partial of V_{g+1}^H b, b being final for group g + 1.
// g = -1 only forms the partials of group 0.  A workgroup takes rpb rows (a
// multiple of 64), 64 at a time, wave w the panel w of either group, one
// right-hand side per blockIdx.y.  The partials (kGW values a workgroup)
// alternate between two buffers.  Triangles and sums are FP64 for either type:
// FP32 solves of 252 to 1962 unknowns are off by 1.8e-7, one panel at a time in
// FP32 by 4.5e-7, and by 5.1e-7 with FP32 triangles (which saved 1 to 2 us a
// launch).
template <typename T>
__global__ __launch_bounds__(256) void qr_apply_group(const typename QT<T>::c2 *__restrict__ A, long lda, int M, int N,
                                                      const double2 *__restrict__ GT, typename QT<T>::c2 *B, long ldb,
                                                      int g, int ng, int rpb, const double *__restrict__ zin,
                                                      double *__restrict__ zout, int nblk) {
    using C2 = typename QT<T>::c2;
    __shared__ double2 s_z[kGW], s_w[2][kGW], s_part[2][4][64];
    const int tid = threadIdx.x, lane = tid & 63, col = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ca = (g * kGB + wave) * kNB, cb = ca + kGW;  // first columns of the wave's panels
    const bool next = g + 1 < ng;
    C2 *b = B + (size_t)col * ldb;
    const int row0 = blockIdx.x * rpb;
    C2 va[kNB], vb[kNB], braw;
    // columns past N read the last one: they meet zeros of T
    auto load = [&](int i) {
        const int ic = min(i, M - 1);
        braw = b[ic];
        const C2 *pa = A + ic;
        if (g >= 0) {
#pragma unroll
            for (int l = 0; l < kNB; l++) va[l] = pa[(unsigned)min(ca + l, N - 1) * (size_t)lda];
        }
        if (next) {
#pragma unroll
            for (int l = 0; l < kNB; l++) vb[l] = pa[(unsigned)min(cb + l, N - 1) * (size_t)lda];
        }
    };
    if (sizeof(T) == 4) load(row0 + lane);
    if (g >= 0) {
        TriProduct<true> tp(GT + (size_t)g * kGG);
        double t = 0;
        const double *zp = zin + (size_t)col * nblk * 2 * kGW + tid;
        for (int q0 = 0; q0 < nblk; q0 += 8) {
            double z[8];
#pragma unroll
            for (int u = 0; u < 8; u++) z[u] = zp[(size_t)min(q0 + u, nblk - 1) * 2 * kGW];
#pragma unroll
            for (int u = 0; u < 8; u++) t += q0 + u < nblk ? z[u] : 0;
        }
        ((double *)s_z)[tid] = t;
        __syncthreads();
        s_w[tid / kGW][tid % kGW] = tp.apply(s_z);
        __syncthreads();
    }
    double x[2 * kNB];
#pragma unroll
    for (int l = 0; l < 2 * kNB; l++) x[l] = 0;
    for (int r = 0; r < rpb; r += 64) {
        const int i = row0 + r + lane;
        if (r || sizeof(T) != 4) load(i);
        const int il = i - ca, in = i - cb;  // rows of the panels
        double2 bi = to_d2(braw);
        if (g >= 0) {
            double2 sum = make_double2(0.0, 0.0);
#pragma unroll
            for (int l = 0; l < kNB; l++) {
                const double2 v = to_d2(v_entry(va[l], il, l));
                const double2 w0 = s_w[0][wave * kNB + l], w1 = s_w[1][wave * kNB + l];
                const double wx = w0.x + w1.x, wy = w0.y + w1.y;
                sum.x = fma(v.x, wx, fma(-v.y, wy, sum.x));
                sum.y = fma(v.x, wy, fma(v.y, wx, sum.y));
            }
            const int h = (r >> 6) & 1;
            s_part[h][wave][lane] = sum;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < 4; w++) {
                bi.x -= s_part[h][w][lane].x;
                bi.y -= s_part[h][w][lane].y;
            }
            C2 o;
            o.x = (T)bi.x;
            o.y = (T)bi.y;
            if (wave == 0 && i < M) b[i] = o;
            bi = to_d2(o);  // (what later launches read)
        }
        if (next) {
            if (i >= M) bi.x = bi.y = 0;
#pragma unroll
            for (int l = 0; l < kNB; l++) {
                const C2 v = v_entry(vb[l], in, l);
                x[2 * l] = fma((double)v.x, bi.x, fma((double)v.y, bi.y, x[2 * l]));
                x[2 * l + 1] = fma((double)v.x, bi.y, fma(-(double)v.y, bi.x, x[2 * l + 1]));
            }
        }
    }
    if (next) {
        wave_reduce_scatter64(x, lane);
        zout[((size_t)col * nblk + blockIdx.x) * 2 * kGW + wave * 2 * kNB + lane] = x[0];
    }
}

// One group of R x = b from the bottom: every workgroup forms the group's
// unknowns R_gg^-1 b_g (b_g is not written in this step), workgroup 0 stores
// them in X, and every workgroup removes them from its 64 rows above the group,
// wave w the columns of panel w.  Sums in FP64.
template <typename T>
__global__ __launch_bounds__(256) void trsv_group(const typename QT<T>::c2 *__restrict__ A, long lda, int N,
                                                  const double2 *__restrict__ GR, typename QT<T>::c2 *B, long ldb,
                                                  typename QT<T>::c2 *__restrict__ X, long ldx, int g) {
    using C2 = typename QT<T>::c2;
    __shared__ double2 s_b[kGW], s_x[2][kGW], s_part[4][64];
    const int tid = threadIdx.x, lane = tid & 63, col = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = g * kGW, i = blockIdx.x * 64 + lane, ic = min(i, c0 > 0 ? c0 - 1 : 0);
    C2 *b = B + (size_t)col * ldb;
    C2 v[kNB];
    const C2 braw = b[ic];
#pragma unroll
    for (int l = 0; l < kNB; l++) v[l] = A[(size_t)min(c0 + wave * kNB + l, N - 1) * lda + ic];
    TriProduct<false> tp(GR + (size_t)g * kGG);
    if (tid < kGW) s_b[tid] = c0 + tid < N ? to_d2(b[c0 + tid]) : make_double2(0.0, 0.0);
    __syncthreads();
    s_x[tid / kGW][tid % kGW] = tp.apply(s_b);
    __syncthreads();
    if (blockIdx.x == 0 && tid < kGW && c0 + tid < N) {
        C2 x;
        x.x = (T)(s_x[0][tid].x + s_x[1][tid].x);
        x.y = (T)(s_x[0][tid].y + s_x[1][tid].y);
        X[(size_t)col * ldx + c0 + tid] = x;
    }
    double2 sum = make_double2(0.0, 0.0);
#pragma unroll
    for (int l = 0; l < kNB; l++) {
        const double2 x0 = s_x[0][wave * kNB + l], x1 = s_x[1][wave * kNB + l], a = to_d2(v[l]);
        const bool in = c0 + wave * kNB + l < N;
        const double xx = in ? x0.x + x1.x : 0, xy = in ? x0.y + x1.y : 0;
        sum.x = fma(a.x, xx, fma(-a.y, xy, sum.x));
        sum.y = fma(a.x, xy, fma(a.y, xx, sum.y));
    }
    s_part[wave][lane] = sum;
    __syncthreads();
    if (wave == 0 && i < c0) {
        double2 bi = to_d2(braw);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            bi.x -= s_part[w][lane].x;
            bi.y -= s_part[w][lane].y;
        }
        C2 o;
        o.x = (T)bi.x;
        o.y = (T)bi.y;
        b[i] = o;
    }
}

// ------------------------------------------------------------------ host ---
template <typename T>
struct QRFactor {
    using C2 = typename QT<T>::c2;
    C2 *A = nullptr;  // factored copy (owned by caller)
    long lda = 0;
    int M = 0, N = 0;
    C2 *Tb = nullptr;  // per-panel T factors
    C2 *W = nullptr;   // workspace nb x max(ncols)
    int wcols = 0;
    C2 *Vd = nullptr;  // explicit panel V (FP32 MFMA trailing update)
    C2 *Yz = nullptr;  // V^H V of the panel (kNB x kNB)
    char *gws = nullptr;
    long ldv = 0;
    // panels by Householder reconstruction: copy of the panel, partials of its
    // Gram matrix, U^-1, and whether it took the column-wise algorithm
    float2 *Pc = nullptr;
    double2 *gram = nullptr, *Y = nullptr;
    int *bad = nullptr;
    double2 *pinned = nullptr;  // PinnedPool block: which panels took it
    // partials and panel rows of the column launches
    float *zcol = nullptr;
    long zcol_stride = 0;
    float2 *rcol = nullptr;
    // triangles of the groups of panels, for the solves
    double2 *GT = nullptr, *GR = nullptr;
    hipStream_t st = nullptr;
    ~QRFactor() {
        if (pinned) {
            (void)hipStreamSynchronize(st);  // (a panel may still write its flag)
            PinnedPool::release(pinned);
        }
        sfree(zcol, st);
        sfree(rcol, st);
        sfree(Tb, st);
        sfree(W, st);
        sfree(Vd, st);
        sfree(Yz, st);
        sfree(gws, st);
        sfree(Pc, st);
        sfree(gram, st);
        sfree(Y, st);
        sfree(bad, st);
        sfree(GT, st);
        sfree(GR, st);
    }
};

template <typename T>
static int qr_apply(const QRFactor<T> &f, typename QT<T>::c2 *C, long ldc, int nc, int conjT, hipStream_t s) {
    if (nc <= 0) return EXIT_SUCCESS;
    if (nc > f.wcols) BEM_FAIL("QR workspace too small");
    const int np = (f.N + kNB - 1) / kNB;
    for (int pi = 0; pi < np; pi++) {
        const int p = conjT ? pi : np - 1 - pi;  // Q^H: H_nb..H_1 order of panels 0..; Q: reverse
        const int j0 = p * kNB, nb = std::min(kNB, f.N - j0);
        qr_vhc<T><<<nc, 256, 0, s>>>(f.A, f.lda, f.M, j0, nb, f.Tb + (size_t)p * kNB * kNB, C, ldc, f.W, conjT);
        HIP_CALL(hipGetLastError());
        dim3 g((unsigned)((f.M - j0 + 255) / 256), (unsigned)nc);
        qr_update<T><<<g, 256, 0, s>>>(f.A, f.lda, f.M, j0, nb, f.W, C, ldc);
        HIP_CALL(hipGetLastError());
    }
    return EXIT_SUCCESS;
}

// A panel of kNB columns column by column, one launch each
template <typename T>
static int panel_columns(QRFactor<T> &f, int j0, float2 *Tp, hipStream_t s) {
    if (!f.zcol) {
        f.zcol_stride = (long)((f.M + kColThreads - 1) / kColThreads) * 2 * kNB;
        HOST_CALL(salloc(&f.rcol, (size_t)2 * kNB, s));
        HOST_CALL(salloc(&f.zcol, (size_t)2 * f.zcol_stride, s));
    }
    const int nblk = (f.M - j0 + kColThreads - 1) / kColThreads;
    for (int jj = -1; jj < kNB; jj++) {
        const int bi = jj & 1, bo = (jj + 1) & 1;
        qr_panel_col<kColThreads><<<nblk, kColThreads, 0, s>>>(
            (float2 *)f.A, f.lda, f.M, j0, jj, f.zcol + (size_t)bi * f.zcol_stride,
            (const float2 *)f.rcol + (size_t)bi * kNB, f.zcol + (size_t)bo * f.zcol_stride,
            (float2 *)f.rcol + (size_t)bo * kNB, nblk, Tp);
        HIP_CALL(hipGetLastError());
    }
    return EXIT_SUCCESS;
}

// Whether a panel is tried by way of its Gram matrix or goes column by column at
// once.  After one that was tried and not taken, the next 4 go column by column,
// then one is tried, and so on: with each one not taken the wait doubles, up to 64
// panels, and with each one taken it halves.  A panel's outcome is asked for two
// panels later, by when qr_recon has written it and the device has the panel
// between to work on.  The rule depends on the outcomes only, not on when they
// arrive.
//
// A panel that is not taken costs qr_recon's one workgroup 0.5 ms at 700 rows, 1.7
// at 4000, 5.7 at 10000; the column launches 0.3 to 0.6.  QR solves of matrices
// with no panel that is taken, all of them tried before: 700 x 642 14.1 -> 9.2 ms
// (3.2 with all taken), 4200 x 4000 228 -> 77 (22), 10300 x 2000 380 -> 78 (19).
class PanelRoute {
public:
    int start(int np, double2 **pinned) {
        if ((size_t)np * sizeof(int) > PinnedPool::kBytes) return EXIT_SUCCESS;  // (no flags: all are tried)
        HOST_CALL(PinnedPool::acquire(pinned));
        flag_ = (int *)*pinned;
        for (int p = 0; p < np; p++) flag_[p] = -1;
        return EXIT_SUCCESS;
    }
    int *seen(int p) const { return flag_ ? flag_ + p : nullptr; }
    int decide(int p, hipStream_t s, bool *gram) {
        if (flag_ && p >= 2 && tried_[p & 1]) {
            int bad = 0;
            HOST_CALL(outcome(flag_ + p - 2, s, &bad));
            hold_ = bad ? std::min(64, std::max(4, 2 * hold_)) : hold_ / 2;
            until_ = bad ? p + hold_ : std::min(until_, p + hold_);
        }
        // (one panel at a time while there is a wait)
        *gram = !hold_ || (p >= until_ && !tried_[(p + 1) & 1]);
        tried_[p & 1] = *gram;
        return EXIT_SUCCESS;
    }

private:
    // waits for a panel's outcome; an error of the stream, asked for every 20 ms
    // (a query itself goes through the stream: at every turn it took 3 us a panel),
    // ends the wait
    static int outcome(int *flag, hipStream_t s, int *bad) {
        using clock = std::chrono::steady_clock;
        auto next = clock::now() + std::chrono::milliseconds(20);
        for (;;) {
            for (int n = 0; n < 64; n++) {
                const int v = __atomic_load_n(flag, __ATOMIC_ACQUIRE);
                if (v >= 0) {
                    *bad = v;
                    return EXIT_SUCCESS;
                }
            }
            std::this_thread::yield();
            if (clock::now() < next) continue;
            const hipError_t e = hipStreamQuery(s);
            if (e != hipErrorNotReady && __atomic_load_n(flag, __ATOMIC_ACQUIRE) < 0)
                BEM_FAIL("a QR panel did not run: %s", hipGetErrorString(e));
            next = clock::now() + std::chrono::milliseconds(20);
        }
    }
    int *flag_ = nullptr;
    bool tried_[2] = {false, false};  // of the last two panels, by parity
    int hold_ = 0, until_ = 0;
};

template <typename T>
static int qr_factor(QRFactor<T> &f, int extra_cols, hipStream_t s) {
    using C2 = typename QT<T>::c2;
    const int np = (f.N + kNB - 1) / kNB;
    f.st = s;
    HOST_CALL(salloc(&f.Tb, (size_t)np * kNB * kNB, s));
    f.wcols = std::max(f.N, extra_cols);
    HOST_CALL(salloc(&f.W, (size_t)kNB * f.wcols, s));
    // FP32: trailing updates on MFMA (C^H V with the adjoint product, then
    // C -= V W with the rank-32 update, which also forms W); FP64 keeps the
    // VALU kernels
    const bool mfma = sizeof(T) == 4 && !getenv("BEM_QR_VALU");
    const bool global_panel = getenv("BEM_QR_GPANEL") != nullptr;
    if (mfma) {
        f.ldv = (f.lda + 63) / 64 * 64;
        HOST_CALL(salloc(&f.Vd, (size_t)f.ldv * kNB, s));
        HOST_CALL(salloc(&f.Yz, (size_t)kNB * kNB, s));
        size_t wsz = 0;
        for (int p = 0; p < np; p++) {
            const int j0 = p * kNB, nb = std::min(kNB, f.N - j0);
            wsz = std::max(wsz, ws_gemm_h_f32(f.M - j0, kNB, kNB));
            if (f.N - (j0 + nb) > 0) wsz = std::max(wsz, ws_gemm_h_f32(f.M - j0, f.N - (j0 + nb), kNB));
        }
        HOST_CALL(salloc(&f.gws, std::max<size_t>(wsz, 1), s));
        if (!global_panel) {
            HOST_CALL(salloc(&f.Pc, (size_t)f.ldv * kNB, s));
            HOST_CALL(salloc(&f.gram, (size_t)kGramParts * kNN, s));
            HOST_CALL(salloc(&f.Y, (size_t)kNN, s));
            HOST_CALL(salloc(&f.bad, 1, s));
        }
    }
    PanelRoute route;
    if (mfma && !global_panel) HOST_CALL(route.start(np, &f.pinned));
    for (int p = 0; p < np; p++) {
        const int j0 = p * kNB, nb = std::min(kNB, f.N - j0);
        TimedRegion tr;
        timing_begin(tr, sizeof(T) == 4 ? "qr_panel_f32" : "qr_panel_f64", s);
        C2 *Tp = f.Tb + (size_t)p * kNB * kNB;
        const int Mp = f.M - j0;
        bool gram = mfma && !global_panel;
        if (gram) HOST_CALL(route.decide(p, s, &gram));
        if (mfma && !global_panel && !gram && nb == kNB) {
            HOST_CALL(panel_columns(f, j0, (float2 *)Tp, s));
        } else if (mfma && !global_panel) {
            gram = true;  // (also a narrow last panel, which the column launches do not take)
            const int rpb = kGramChunk * ((Mp + kGramChunk * kGramParts - 1) / (kGramChunk * kGramParts));
            const int nblk = (Mp + rpb - 1) / rpb;
            float2 *Af = (float2 *)f.A, *Vf = (float2 *)f.Vd;
            qr_gram<<<nblk, 256, 0, s>>>(Af, f.lda, f.M, j0, nb, rpb, f.gram, f.Pc, f.ldv);
            qr_recon<<<1, kRecThreads, 0, s>>>(f.gram, nblk, Af, f.lda, f.M, j0, nb, (float2 *)Tp, Vf, f.ldv, f.Y, f.bad,
                                              route.seen(p));
            qr_form_v<<<(Mp + 63) / 64, 256, 0, s>>>(f.Pc, f.Y, f.bad, Af, f.lda, f.M, j0, nb, Vf, f.ldv);
        } else {
            qr_panel<T><<<1, 1024, 0, s>>>(f.A, f.lda, f.M, j0, nb, Tp, mfma ? 0 : 1);
        }
        HIP_CALL(hipGetLastError());
        if (mfma && !gram) {
            dim3 gv((unsigned)((Mp + 255) / 256), kNB);
            k_build_v<T><<<gv, 256, 0, s>>>(f.A, f.lda, f.M, j0, nb, f.Vd, f.ldv);
            HIP_CALL(hipGetLastError());
            HOST_CALL(gemm_h_f32((const float2 *)f.Vd, f.ldv, Mp, kNB, (const float2 *)f.Vd, f.ldv, (float2 *)f.Yz,
                                 kNB, kNB, f.gws, s));
            qr_make_t<T><<<1, 64, 0, s>>>(Tp, nb, f.Yz, kNB);
            HIP_CALL(hipGetLastError());
        }
        timing_end(tr, s);
        const int nc = f.N - (j0 + nb);
        if (nc > 0) {
            C2 *Ct = f.A + (size_t)(j0 + nb) * f.lda;
            TimedRegion tu;
            timing_begin(tu, sizeof(T) == 4 ? "qr_trailing_f32" : "qr_trailing_f64", s);
            if (mfma) {
                float2 *Cb = (float2 *)(Ct + j0);  // rows j0.., columns j0+nb..
                const bool direct = Mp <= kTrailRows;
                ProdParts zp;
                HOST_CALL(gemm_h_f32(Cb, f.lda, Mp, nc, (const float2 *)f.Vd, f.ldv, (float2 *)f.W, f.N, kNB, f.gws, s,
                                     false, direct ? &zp : nullptr));
                if (!direct) zp = {(const float2 *)f.W, f.N, 1};
                HOST_CALL(qr_trail_f32((const float2 *)f.Vd, f.ldv, Mp, (const float2 *)Tp, nb, zp, nc, Cb, f.lda, s));
            } else {
                qr_vhc<T><<<nc, 256, 0, s>>>(f.A, f.lda, f.M, j0, nb, f.Tb + (size_t)p * kNB * kNB, Ct, f.lda,
                                             f.W, 1);
                HIP_CALL(hipGetLastError());
                dim3 g((unsigned)((f.M - j0 + 255) / 256), (unsigned)nc);
                qr_update<T><<<g, 256, 0, s>>>(f.A, f.lda, f.M, j0, nb, f.W, Ct, f.lda);
                HIP_CALL(hipGetLastError());
            }
            timing_end(tu, s);
        }
    }
    return EXIT_SUCCESS;
}

static int group_splits(int npair) { return std::max(1, std::min(16, 1024 / npair)); }

// rows of a workgroup of a solve's launches: at most 64 workgroups
static int solve_rows(int M) { return 64 * ((M + 64 * 64 - 1) / (64 * 64)); }

// device bytes of a factorisation beyond the matrix and of its solves (FP64: R
// right-hand sides at once, FP32: one after the other)
size_t qr_work_bytes(int M, int N, int R, bool fp64) {
    const size_t np = ((size_t)N + kNB - 1) / kNB, ng = (np + kGB - 1) / kGB, ld = ((size_t)M + 63) / 64 * 64;
    const size_t splits = group_splits((int)(ng * kPairs));
    size_t b = (fp64 ? sizeof(double2) : sizeof(float2)) * kNB * (np * kNB + N);   // T factors, W
    b += sizeof(double2) * (2 * ng * kGG + (ng * kPairs * splits + np) * kNN);       // triangles and what forms them
    if (!fp64) b += sizeof(float2) * 2 * kNB * ld + sizeof(double2) * (kGramParts + 1) * kNN;  // V, panel, Gram
    if (!fp64) b += 2 * kNB * (sizeof(float2) + 2 * sizeof(float) * (((size_t)M + kColThreads - 1) / kColThreads));  // column launches
    const size_t nblk = ((size_t)M + solve_rows(M) - 1) / solve_rows(M);
    b += (fp64 ? (size_t)R : 1) * (2 * nblk * 2 * kGW * sizeof(double) + (fp64 ? sizeof(double2) : sizeof(float2)) * N);
    return b;
}

// The triangles of the groups of panels (qr_cross, qr_group), once per
// factorisation.  The cross products split their rows over up to 16 workgroups
// while there are few groups.
template <typename T>
static int qr_groups(QRFactor<T> &f, hipStream_t s) {
    if (f.GT) return EXIT_SUCCESS;
    const int np = (f.N + kNB - 1) / kNB, ng = (np + kGB - 1) / kGB;
    const int npair = ng * kPairs, nsplit = group_splits(npair);
    double2 *cross = nullptr, *rinv = nullptr;
    HOST_CALL(salloc(&f.GT, (size_t)ng * kGG, s));
    HOST_CALL(salloc(&f.GR, (size_t)ng * kGG, s));
    HOST_CALL(salloc(&cross, (size_t)npair * nsplit * kNN, s));
    int rc = salloc(&rinv, (size_t)np * kNN, s);
    if (rc == EXIT_SUCCESS) {
        qr_cross<T><<<npair * nsplit + np, 256, 0, s>>>(f.A, f.lda, f.M, f.N, npair, nsplit, cross, rinv);
        qr_group<T><<<dim3(ng, kGB, 2), 1024, 0, s>>>(f.A, f.lda, f.N, f.Tb, cross, nsplit, rinv, f.GT, f.GR);
        if (hipGetLastError() != hipSuccess) rc = EXIT_FAILURE;
    }
    sfree(cross, s);
    sfree(rinv, s);
    if (rc != EXIT_SUCCESS) BEM_FAIL("QR solve launches failed");
    return EXIT_SUCCESS;
}

// Least squares solve with a factored A: B (M x R, ldb) <- solution in B[0:N].
constexpr size_t kSmallSolveLds = 48 * 1024;  // b of up to 6144 FP32 / 3072 FP64 rows
constexpr int kSmallSolveRhs = 64;

template <typename T>
static int qr_solve_factored(QRFactor<T> &f, typename QT<T>::c2 *B, long ldb, int R, hipStream_t s) {
    using C2 = typename QT<T>::c2;
    if (R <= 0) return EXIT_SUCCESS;
    // the whole solve in one workgroup per right-hand side, b in shared memory: on
    // request, and for small FP64 systems, whose factorisation serves one solve, so
    // that the triangles of the row-split launches below (70 us) do not pay (14
    // unknowns: 0.33 against 0.45 ms for factorisation and solve; 194: 6.12 and 6.19;
    // 642: 21.96 and 21.57).  FP32 systems of that size are solved several times, or
    // with FP64 sums that this kernel does not have.
    const size_t lds = sizeof(C2) * (size_t)f.M;
    const bool small = sizeof(T) == 8 && f.N <= 256 && !getenv("BEM_QR_PER_COLUMN_SOLVE");
    if (lds <= kSmallSolveLds && R <= kSmallSolveRhs && (small || getenv("BEM_QR_ONE_WG_SOLVE"))) {
        // 2 kNB partial sums per thread plus a chunk of 8 loads: the register
        // room of 512 (FP32) or 256 (FP64) threads
        constexpr int nt = sizeof(T) == 4 ? 512 : 256;
        qr_solve_small<T, nt><<<R, nt, lds, s>>>(f.A, f.lda, f.M, f.N, f.Tb, B, ldb);
        HIP_CALL(hipGetLastError());
        return EXIT_SUCCESS;
    }
    if (getenv("BEM_QR_PER_COLUMN_SOLVE")) {
        HOST_CALL(qr_apply<T>(f, B, ldb, R, 1, s));
        trsv_upper<T><<<R, 1024, 0, s>>>(f.A, f.lda, f.N, B, ldb);
        HIP_CALL(hipGetLastError());
        return EXIT_SUCCESS;
    }
    // one launch per group of panels for Q^H B and one for the back
    // substitution, the rows spread over at most 64 workgroups
    HOST_CALL(qr_groups<T>(f, s));
    const int ng = ((f.N + kNB - 1) / kNB + kGB - 1) / kGB;
    const int rpb = solve_rows(f.M), nblk = (f.M + rpb - 1) / rpb;
    const size_t zn = (size_t)R * nblk * 2 * kGW;
    double *zb = nullptr;
    C2 *X = nullptr;
    HOST_CALL(salloc(&zb, 2 * zn, s));
    int rc = salloc(&X, (size_t)f.N * R, s);
    for (int g = -1; g < ng && rc == EXIT_SUCCESS; g++) {
        qr_apply_group<T><<<dim3(nblk, R), 256, 0, s>>>(f.A, f.lda, f.M, f.N, f.GT, B, ldb, g, ng, rpb,
                                                        zb + (g & 1) * zn, zb + ((g + 1) & 1) * zn, nblk);
        if (hipGetLastError() != hipSuccess) rc = EXIT_FAILURE;
    }
    for (int g = ng - 1; g >= 0 && rc == EXIT_SUCCESS; g--) {
        const unsigned rows = std::max(1, g * kGW / 64);
        trsv_group<T><<<dim3(rows, R), 256, 0, s>>>(f.A, f.lda, f.N, f.GR, B, ldb, X, f.N, g);
        if (hipGetLastError() != hipSuccess) rc = EXIT_FAILURE;
    }
    if (rc == EXIT_SUCCESS &&
        hipMemcpy2DAsync(B, sizeof(C2) * ldb, X, sizeof(C2) * f.N, sizeof(C2) * f.N, R, hipMemcpyDeviceToDevice,
                         s) != hipSuccess)
        rc = EXIT_FAILURE;
    sfree(zb, s);
    sfree(X, s);
    if (rc != EXIT_SUCCESS) BEM_FAIL("QR solve launches failed");
    return EXIT_SUCCESS;
}

// Plain least squares: A (overwritten with its factorisation), B -> solution.
template <typename T>
static int qr_lsq_impl(typename QT<T>::c2 *A, long lda, int M, int N, typename QT<T>::c2 *B, long ldb, int R,
                       hipStream_t s) {
    if (M < N || N <= 0) BEM_FAIL("least squares needs M >= N > 0 (got %d x %d)", M, N);
    QRFactor<T> f;
    f.A = A;
    f.lda = lda;
    f.M = M;
    f.N = N;
    HOST_CALL(qr_factor<T>(f, R, s));
    HOST_CALL(qr_solve_factored<T>(f, B, ldb, R, s));
    HIP_CALL(hipStreamSynchronize(s));
    return EXIT_SUCCESS;
}

int qr_lsq_f32(float2 *A, long lda, int M, int N, float2 *B, long ldb, int R, hipStream_t s) {
    return qr_lsq_impl<float>(A, lda, M, N, B, ldb, R, s);
}
int qr_lsq_f64(double2 *A, long lda, int M, int N, double2 *B, long ldb, int R, hipStream_t s) {
    return qr_lsq_impl<double>(A, lda, M, N, B, ldb, R, s);
}

__global__ void k_identity(float2 *Q, long ldq, int M) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i < M) Q[(size_t)j * ldq + i] = make_float2(i == j ? 1.f : 0.f, 0.f);
}

// Least squares plus explicit Q: A <- R (upper triangle, zero below), Q (M x M).
int qr_lsq_with_q_f32(float2 *A, long lda, int M, int N, float2 *B, long ldb, int R, float2 *Q, long ldq,
                      hipStream_t s) {
    if (M < N || N <= 0) BEM_FAIL("least squares needs M >= N > 0 (got %d x %d)", M, N);
    QRFactor<float> f;
    f.A = A;
    f.lda = lda;
    f.M = M;
    f.N = N;
    HOST_CALL(qr_factor<float>(f, std::max(R, M), s));
    if (Q) {
        dim3 g((unsigned)((M + 255) / 256), (unsigned)M);
        k_identity<<<g, 256, 0, s>>>(Q, ldq, M);
        HIP_CALL(hipGetLastError());
        HOST_CALL(qr_apply<float>(f, Q, ldq, M, 0, s));
    }
    HOST_CALL(qr_solve_factored<float>(f, B, ldb, R, s));
    HIP_CALL(hipStreamSynchronize(s));
    return EXIT_SUCCESS;
}

// ------------------------------------------------ refined LS (FP32 + FP64) ---
int resid_n_f32a(const float2 *A, long lda, long M, long N, const double2 *x, long ldx, const double2 *b, long ldb,
                 double2 *r, long ldr, int R, void *ws, hipStream_t s);

__global__ void k_z2c(const double2 *__restrict__ in, float2 *__restrict__ out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float2((float)in[i].x, (float)in[i].y);
}
__global__ void k_addc2z(const float2 *__restrict__ d, double2 *__restrict__ x, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x[i].x += d[i].x;
        x[i].y += d[i].y;
    }
}
__global__ void k_sumsq(const double2 *__restrict__ v, int n, double *out);
__global__ void k_sumsq_c(const float2 *__restrict__ v, int n, double *out);
__global__ void k_sumsq(const double2 *__restrict__ v, int n, double *out) {
    __shared__ double red[16];
    double s = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += v[i].x * v[i].x + v[i].y * v[i].y;
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) t += red[q];
        *out = t;
    }
}
__global__ void k_sumsq_c(const float2 *__restrict__ v, int n, double *out) {
    __shared__ double red[16];
    double s = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += (double)v[i].x * v[i].x + (double)v[i].y * v[i].y;
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) t += red[q];
        *out = t;
    }
}

// FP32 QR least squares wrapped in FP64 iterative refinement: the fixed-point
// iteration x <- x + QRsolve(b - A x) with the residual accumulated in FP64
// from the FP32 matrix.  A32 (kept), B64: M x R FP64 rhs, X64: N x R FP64
// solution (out).  Stops when ||correction|| <= refine_tol ||x|| or when the
// correction no longer shrinks (an inconsistent least-squares system keeps a
// nonzero residual, so the residual itself is not the test).
int qr_refined_f32(const float2 *A32, long lda, int M, int N, const double2 *B64, long ldb, double2 *X64, long ldx,
                   int R, double refine_tol, int max_refine, bem_solve_stats *st, hipStream_t s) {
    if (M < N || N <= 0) BEM_FAIL("least squares needs M >= N > 0 (got %d x %d)", M, N);
    QRFactor<float> f;
    HOST_CALL(salloc(&f.A, (size_t)lda * N, s));
    HIP_CALL(hipMemcpyAsync(f.A, A32, sizeof(float2) * lda * N, hipMemcpyDeviceToDevice, s));
    f.lda = lda;
    f.M = M;
    f.N = N;
    float2 *rb = nullptr;
    double2 *r64 = nullptr;
    double *dn = nullptr;
    char *gws = nullptr;
    int refinements = 0;
    double worst = 0;
    bool conv = true;
    int rc = EXIT_FAILURE;
    const int bs = 256;
    if (qr_factor<float>(f, 1, s) != EXIT_SUCCESS) goto out;
    if (salloc(&rb, (size_t)lda, s) || salloc(&r64, (size_t)lda, s) || salloc(&dn, 2, s)) goto out;
    if (salloc(&gws, ws_gemv_n(M, N, 1), s)) goto out;
    for (int r = 0; r < R; r++) {
        const double2 *b = B64 + (size_t)r * ldb;
        double2 *x = X64 + (size_t)r * ldx;
        if (hipMemsetAsync(x, 0, sizeof(double2) * N, s) != hipSuccess) goto out;
        double prev = 1e300, rel = 0;
        for (int it = 0; it <= max_refine; it++) {
            if (resid_n_f32a(A32, lda, M, N, x, 0, b, 0, r64, 0, 1, gws, s) != EXIT_SUCCESS) goto out;
            k_z2c<<<(M + bs - 1) / bs, bs, 0, s>>>(r64, rb, M);
            if (qr_solve_factored<float>(f, rb, lda, 1, s) != EXIT_SUCCESS) goto out;
            k_addc2z<<<(N + bs - 1) / bs, bs, 0, s>>>(rb, x, N);
            k_sumsq_c<<<1, 1024, 0, s>>>(rb, N, dn);
            k_sumsq<<<1, 1024, 0, s>>>(x, N, dn + 1);
            double h[2];
            if (hipMemcpyAsync(h, dn, 2 * sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess) goto out;
            if (hipStreamSynchronize(s) != hipSuccess) goto out;
            rel = std::sqrt(h[0] / std::max(h[1], 1e-300));
            refinements++;
            if (rel <= refine_tol || rel >= 0.5 * prev) break;
            prev = rel;
        }
        worst = std::max(worst, rel);
        conv = conv && rel <= std::max(refine_tol, 1e-5);
    }
    rc = EXIT_SUCCESS;
out:
    if (st) {
        st->refinements = refinements;
        st->iterations = 0;
        st->converged = conv ? 1 : 0;
        st->residual = worst;
    }
    sfree(f.A, s);
    sfree(rb, s);
    sfree(r64, s);
    sfree(dn, s);
    sfree(gws, s);
    (void)hipStreamSynchronize(s);
    if (rc != EXIT_SUCCESS) BEM_FAIL("refined QR least squares failed");
    return rc;
}

}  // namespace bem
