// Resolution-matrix mode of the QML engine (gfx950, FP64).
//
// With a resolution matrix R (N x M, banded: row i has rnb values at
// matrix-grid columns rcol0 + i*ros ...) the reference builds, per chunk,
//   Q_k = R Qhat_k R^T,  Qhat_k(v) = (dk/pi) cos(k_c v) sin(dk v/2)/(dk v/2)
//                                    (dk/pi at v = 0),
//   S   = R Shat R^T,    Shat = the 2D signal table at (z, v),
// with v, z taken on the matrix's grid (core/chunk_estimate.cpp:384-480,
// mathtools/matrix_helper.cpp:877-902,1075-1084), then applies the z-bin
// weights on the pixel grid.  Here S and every Q_k (k < KBIN_UPP) are
// materialised once per iteration in the chunk's FP64 matrix arena (qb_off),
// over the whole batch at a time.
//
// The band window is a difference of edge terms: with the band edges
// k_n, k_n+1 (k_c their mean, dk their difference),
//   Qhat_k(v) = P_n+1(v) - P_n(v),   P_e(v) = sin(k_e v) / (pi v)  (k_e/pi at 0),
// the same function as the reference's product form by the sum-to-product
// identity.  So Q_k = Z_k+1 - Z_k with Z_e = R P_e R^T: one sandwich per band
// edge, and each band is the difference of two consecutive ones, taken in
// registers.  With v = u_b - u_a (u = c ln lambda, relative to a point of the
// block's own range so that |u| stays small), sin(k v) = sin(k u_b) cos(k u_a)
// - cos(k u_b) sin(k u_a): sines and cosines are evaluated once per grid point
// and edge, not once per grid pair and band.
//
// That is the form for any band.  Where the band is narrow on the scale of the
// chunk's velocities v <= vmax (all practical ones), the window's definition
//   Qhat_k(v) = 1/pi int_{k_n}^{k_n+1} cos(k v) dk
// is summed over n Gauss-Legendre nodes instead, exact to 1e-17 of Qhat(0) at
// n = dk vmax / 4 + O(n^1/3) of them (rmat_nodes), and since v = u_b - u_a,
//   Q_k = sum_m w_m/pi (R c_m)(R c_m)^T + (R s_m)(R s_m)^T,
// with c_m, s_m the cosine and sine of k_m u on the fine grid: R is applied to
// 2 n vectors (k_rm_nodes), and Q_k is the product of an N x 2n matrix with its
// transpose (k_rm_bands).  The phases k_m u carry both operands' rounding, so
// that the nodes' errors stay at the rounding of a cosine.  An element of Q_k
// costs 2 n multiply-adds on the matrix cores (30 to 130 on 100 to 1200 pixels of
// 55 km/s), against about 800 by the edges, whose taps go through LDS.  160
// chunks of 100 to 1200 pixels oversampled three times, 29 bands: 37 -> 7 ms
// (k_rm_nodes 1.8, k_rm_bands 5.1 for 13 GB written), and the largest error
// against extended precision falls from 1.5e-12 to 2.5e-13 of Q_k's peak.
//
// The host lays every R row inside the grid (rcol0 >= 0; a diagonal-storage
// matrix gets nelem/2 extrapolated grid points on each side, whose weights
// are zero), so every tap loop below has the same trip count.
//
// S is formed by k_rm_signal, the Q_k of a chunk without groups by k_rm_sandwich:
// each chunk by its own shape, whatever the others of its batch.
//
// k_rm_sandwich<TJ>: one 16 x TJ output tile (I0.., J0..) per block, tiles
// touching the upper triangle only.  The fine rows of its 16 R rows (the a
// range, 15 ros + rnb) and the fine columns of its TJ R columns (the b range,
// (TJ-1) ros + rnb, in passes of 32) are fixed for the block.  Per edge e:
//   per pass:  Qh (a x 32, LDS) <- P_e(a, b)
//              T  (16 x b, LDS) <- R_I Qh                  (rnb taps, FP64 FMA)
//   Z[i][j] = sum_t T[i][j ros + t] R[j][t]                (rnb taps, registers)
//   Q_e-1 = Z_e - Z_e-1 written to the upper triangle and mirrored, as
//   Resolution::sandwich fills it.
#include "qml_common.hpp"
#include "qml_kernels.hpp"

#include <algorithm>
#include <cmath>

namespace qml {

namespace {
constexpr double RM_PI = 3.14159265358979323846;
constexpr int RM_BW = 32;    // fine columns per pass
constexpr int RM_QP = 33;    // row pitch of Qh (doubles)

}  // namespace

template <int TJ, int EM, int NPM>
__global__ __launch_bounds__(256) void k_rm_sandwich(const ChunkDev *cs, const double *rin, BinsDev bins, RmLayout lay,
                                                     double *mat) {
    constexpr int NO = TJ / 16;                   // outputs per thread
    // EM: Qh entries per thread (rows ar0 + 8 s, s < EM); 8 EM >= 15 ros + rnb.
    // NPM: passes at most ((TJ - 1) ros + rnb <= 32 NPM), their 1/(pi v) kept in registers
    const ChunkDev c = cs[blockIdx.z];
    if (!c.rm || c.ngrp) return;   // the bands of a chunk with groups come from k_rm_bands
    const int Np = c.Np, N = c.N, M = c.rM, nb = c.rnb, os = c.ros, kbu = c.kbu;
    const int I0 = blockIdx.y * 16, J0 = blockIdx.x * TJ;
    if (I0 >= Np || J0 >= Np || J0 + TJ - 1 < I0) return;
    const int tid = threadIdx.x, ti = tid >> 4, tj = tid & 15;
    const int i = I0 + ti;
    const size_t NN = (size_t)Np * Np;
    double *Qb = mat + c.qb_off;
    if (I0 >= N || J0 >= N) {                     // all padding
        for (int o = 0; o < NO; ++o) {
            const int j = J0 + tj + 16 * o;
            if (j < i) continue;
            for (int k = 0; k < kbu; ++k) {
                Qb[k * NN + (size_t)i * Np + j] = 0.0;
                Qb[k * NN + (size_t)j * Np + i] = 0.0;
            }
        }
        return;
    }
    const double *R = rin + c.rin_off;            // N x nb
    const double *grid = R + (size_t)N * nb;      // M wavelengths (units of lambda_Lya)
    const int amin = c.rcol0 + I0 * os, ra = 15 * os + nb;
    const int bmin = c.rcol0 + J0 * os, rb = (TJ - 1) * os + nb;
    const int npass = (rb + RM_BW - 1) / RM_BW;
    const int npts = ra + RM_BW * npass;          // the a points, then the b points
    const int ref = min(M - 1, (amin + bmin + rb) / 2);

    extern __shared__ double lds[];
    double *Qh = lds;                             // lay.qr x RM_QP
    double *Tb = Qh + lay.qr * RM_QP;             // 16 x lay.tw
    double *Ri = Tb + 16 * lay.tw;                // 16 x lay.nbm
    double *Rj = Ri + 16 * lay.nbm;               // TJ x lay.nbm
    double *ush = Rj + TJ * lay.nbm;              // lay.npts
    double2 *scs = reinterpret_cast<double2 *>(ush + lay.npts);

    for (int e = tid; e < 16 * nb; e += 256) {
        const int r = e / nb, tt = e - r * nb;
        Ri[r * lay.nbm + tt] = (I0 + r < N) ? R[(size_t)(I0 + r) * nb + tt] : 0.0;
    }
    for (int e = tid; e < TJ * nb; e += 256) {
        const int r = e / nb, tt = e - r * nb;
        Rj[r * lay.nbm + tt] = (J0 + r < N) ? R[(size_t)(J0 + r) * nb + tt] : 0.0;
    }
    const double gref = grid[ref];
    for (int p = tid; p < npts; p += 256) {
        const int g = min(M - 1, p < ra ? amin + p : bmin + (p - ra));
        ush[p] = SPEED_OF_LIGHT * log(grid[g] / gref);
    }
    __syncthreads();

    const int q0 = tid & 15;                      // T step: row ti, columns q0, q0 + 16
    const int bb = tid & 31, ar0 = tid >> 5;      // Qh entries: rows ar0 + 8 s, column bb
    const double *Rti = Ri + ti * lay.nbm;
    const double *Qti = Qh + ti * os * RM_QP;
    double zp[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) zp[o] = 0.0;

    // 1/(pi v) of this thread's entries in every pass (v = u_b - u_a does not
    // depend on the edge); the entry on the shared grid point (v = 0, at most
    // one per pass and column) gets 0 here and k_e/pi written after the rest.
    // Points past the grid, which stand on its last one, take no part
    double inv[NPM][EM];
    int dsel[NPM];
#pragma unroll
    for (int p = 0; p < NPM; ++p) {
        dsel[p] = -1;
        const double ub = (p < npass) ? ush[ra + p * RM_BW + bb] : 0.0;
#pragma unroll
        for (int s = 0; s < EM; ++s) {
            const double d = (ub - ush[ar0 + 8 * s]) * RM_PI;
            const bool live = p < npass && ar0 + 8 * s < ra && amin + ar0 + 8 * s < M && bmin + p * RM_BW + bb < M;
            inv[p][s] = (live && d != 0.0) ? 1.0 / d : 0.0;
            if (live && d == 0.0) dsel[p] = s;
        }
    }

    for (int e = 0; e <= kbu; ++e) {
        const double ke = bins.ke[e], kpi = ke / RM_PI;
        for (int p = tid; p < npts; p += 256) {
            double sv, cv;
            sincos(ke * ush[p], &sv, &cv);
            scs[p] = make_double2(sv, cv);
        }
        __syncthreads();
        // the a points' (sin, cos) at this edge: the same in every pass
        double2 sa[EM];
#pragma unroll
        for (int s = 0; s < EM; ++s) sa[s] = scs[ar0 + 8 * s];
#pragma unroll
        for (int p = 0; p < NPM; ++p) {
            if (p >= npass) break;
            const int pc = p * RM_BW + bb;
            // rows past the a range fill Qh rows that the T step never reads
            const double2 sb = scs[ra + pc];
#pragma unroll
            for (int s = 0; s < EM; ++s)
                Qh[(ar0 + 8 * s) * RM_QP + bb] = (sb.x * sa[s].y - sb.y * sa[s].x) * inv[p][s];
            if (dsel[p] >= 0) Qh[(ar0 + 8 * dsel[p]) * RM_QP + bb] = kpi;
            __syncthreads();
            double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
            int tt = 0;
            for (; tt + 3 < nb; tt += 4) {
                const double *q = Qti + tt * RM_QP + q0;
                const double w0 = Rti[tt], w1 = Rti[tt + 1], w2 = Rti[tt + 2], w3 = Rti[tt + 3];
                const double a0 = q[0], a1 = q[16], b0 = q[RM_QP], b1 = q[RM_QP + 16];
                const double c0 = q[2 * RM_QP], c1 = q[2 * RM_QP + 16], d0 = q[3 * RM_QP], d1 = q[3 * RM_QP + 16];
                t0 += w0 * a0;
                t1 += w0 * a1;
                t2 += w1 * b0;
                t3 += w1 * b1;
                t0 += w2 * c0;
                t1 += w2 * c1;
                t2 += w3 * d0;
                t3 += w3 * d1;
            }
            for (; tt + 1 < nb; tt += 2) {
                const double w0 = Rti[tt], w1 = Rti[tt + 1];
                const double *q = Qti + tt * RM_QP + q0;
                t0 += w0 * q[0];
                t1 += w0 * q[16];
                t2 += w1 * q[RM_QP];
                t3 += w1 * q[RM_QP + 16];
            }
            if (tt < nb) {
                const double w0 = Rti[tt];
                const double *q = Qti + tt * RM_QP + q0;
                t0 += w0 * q[0];
                t1 += w0 * q[16];
            }
            Tb[ti * lay.tw + p * RM_BW + q0] = t0 + t2;
            Tb[ti * lay.tw + p * RM_BW + q0 + 16] = t1 + t3;
            __syncthreads();
        }
        double z[NO];
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const double *tr = Tb + ti * lay.tw + (tj + 16 * o) * os;
            const double *rr = Rj + (tj + 16 * o) * lay.nbm;
            double s0 = 0.0, s1 = 0.0;
            int tt = 0;
            for (; tt + 3 < nb; tt += 4) {
                const double x0 = tr[tt], x1 = tr[tt + 1], x2 = tr[tt + 2], x3 = tr[tt + 3];
                const double y0 = rr[tt], y1 = rr[tt + 1], y2 = rr[tt + 2], y3 = rr[tt + 3];
                s0 += x0 * y0;
                s1 += x1 * y1;
                s0 += x2 * y2;
                s1 += x3 * y3;
            }
            for (; tt + 1 < nb; tt += 2) {
                s0 += tr[tt] * rr[tt];
                s1 += tr[tt + 1] * rr[tt + 1];
            }
            if (tt < nb) s0 += tr[tt] * rr[tt];
            z[o] = s0 + s1;
        }
        if (e > 0) {
            double *Q = Qb + (size_t)(e - 1) * NN;
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                const int j = J0 + tj + 16 * o;
                if (j >= i) {
                    const double val = z[o] - zp[o];
                    Q[(size_t)i * Np + j] = val;
                    Q[(size_t)j * Np + i] = val;
                }
            }
        }
#pragma unroll
        for (int o = 0; o < NO; ++o) zp[o] = z[o];
    }
}

namespace {
constexpr int RN_ROWS = 64, RN_NODES = 8;   // rows and nodes of a k_rm_nodes step
typedef double gd4 __attribute__((ext_vector_type(4)));
// k_rm_signal's row pitch of R in LDS: 16 rows read at columns os apart fall on distinct banks
__host__ __device__ inline int signal_pitch(int os, int nb) { return nb + ((nb - os) % 2 == 0); }
}  // namespace

// V[col + 2m][i] = a_m sum_t R[i][t] cos(k_m u(i, t)), V[col + 2m + 1][i] the
// sine's: 64 rows of R per workgroup, eight nodes at a time.  The phases of the
// rows' fine points are evaluated once per node in LDS (a row shares nb - os of
// its points with the next); a thread then sums the taps of its row for two
// nodes.  V is stored node by node, so that both sides of k_rm_bands read it
// along i.  Rows past N have no weights and give zeros.  Bound by the LDS reads
// of the taps.
__global__ __launch_bounds__(256) void k_rm_nodes(const ChunkDev *cs, const double *rin, const RmBand *bands,
                                                  const RmNode *nodes, int grp, double *mat) {
    const ChunkDev c = cs[blockIdx.z];
    const int I0 = blockIdx.x * RN_ROWS, k = blockIdx.y;
    if (!c.ngrp || k >= c.kbu || I0 >= c.Np) return;
    const RmBand b = bands[c.rmb_off + k];
    if (b.grp != grp) return;
    const int N = c.N, M = c.rM, nb = c.rnb, os = c.ros, ra = (RN_ROWS - 1) * os + nb;
    const int amin = c.rcol0 + I0 * os;
    const double *R = rin + c.rin_off, *grid = R + (size_t)N * nb;
    extern __shared__ double lds[];
    double2 *cs2 = reinterpret_cast<double2 *>(lds);   // RN_NODES x ra
    double *Ri = lds + 2 * RN_NODES * ra;              // RN_ROWS x nb
    double *ush = Ri + RN_ROWS * nb;                   // ra
    const int tid = threadIdx.x;
    for (int e = tid; e < RN_ROWS * nb; e += 256) {
        const int r = e / nb;
        Ri[e] = (I0 + r < N) ? R[(size_t)I0 * nb + e] : 0.0;
    }
    const double gref = grid[M / 2];
    // log1p of the difference: u to its own rounding, where a rounded ratio leaves c eps
    for (int p = tid; p < ra; p += 256)
        ush[p] = SPEED_OF_LIGHT * log1p((grid[min(M - 1, amin + p)] - gref) / gref);
    __syncthreads();
    const int row = tid & 63, q = tid >> 6;
    const double *w = Ri + row * nb;
    const double2 *x0 = cs2 + q * ra + row * os, *x1 = x0 + (RN_NODES / 2) * ra;
    double *V = mat + c.mat_off + (size_t)b.col * c.Np + I0 + row;
    const RmNode *nd = nodes + b.node;
    for (int m0 = 0; m0 < b.n; m0 += RN_NODES) {
        for (int e = tid; e < RN_NODES * ra; e += 256) {
            const int m = e / ra;
            const RmNode x = nd[m0 + m];
            const double u = ush[e - m * ra], p = x.kh * u, d = __builtin_fma(x.kh, u, -p) + x.kl * u;
            double sv, cv;
            sincos(p, &sv, &cv);
            cs2[e] = make_double2(cv - d * sv, sv + d * cv);
        }
        __syncthreads();
        double c0 = 0.0, s0 = 0.0, c1 = 0.0, s1 = 0.0;
        for (int t = 0; t < nb; ++t) {
            const double r = w[t];
            const double2 y0 = x0[t], y1 = x1[t];
            c0 += r * y0.x;
            s0 += r * y0.y;
            c1 += r * y1.x;
            s1 += r * y1.y;
        }
        const int m = m0 + q;
        const double a0 = nd[m].a, a1 = nd[m + RN_NODES / 2].a;
        V[(size_t)(2 * m) * c.Np] = a0 * c0;
        V[(size_t)(2 * m + 1) * c.Np] = a0 * s0;
        V[(size_t)(2 * m + RN_NODES) * c.Np] = a1 * c1;
        V[(size_t)(2 * m + RN_NODES + 1) * c.Np] = a1 * s1;
        __syncthreads();
    }
}

// Q_k = V^T V over the band's 2n rows of V: one upper 64 x 64 tile per
// workgroup, a 32 x 32 quarter per wave, written to both triangles.  A lane
// loads two neighbouring i of one row of V, which are the operands of two
// 16-row blocks (block x holds the rows i0 + 2 r + x), straight from L1 and L2:
// two 16-byte loads feed four MFMAs, so LDS would only add its barriers.  The
// loads of the next 16 rows are issued before the products of these.
__global__ __launch_bounds__(256) void k_rm_bands(const ChunkDev *cs, const RmBand *bands, int grp, double *mat) {
    const ChunkDev c = cs[blockIdx.z];
    const int k = blockIdx.y, x = blockIdx.x;
    if (!c.ngrp || k >= c.kbu || x >= c.ntu) return;
    const RmBand b = bands[c.rmb_off + k];
    if (b.grp != grp) return;
    // tile x of the upper triangle, column by column
    int J = (int)((sqrtf(8.0f * x + 1.0f) - 1.0f) * 0.5f);
    while (J * (J + 1) / 2 > x) --J;
    while ((J + 1) * (J + 2) / 2 <= x) ++J;
    const int I = x - J * (J + 1) / 2;
    const int Np = c.Np, tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64), wm = wv / 2, wn = wv % 2;
    if (I == J && wm > wn) return;   // the mirror image of quarter (0, 1)
    const int r0 = I * TILE + 32 * wm, c0 = J * TILE + 32 * wn;
    const double *V = mat + c.mat_off + (size_t)(b.col + lq) * Np + 2 * lr;
    const size_t step = (size_t)4 * Np;
    gd4 acc[2][2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int f = 0; f < 2; ++f) acc[e][f] = gd4{0.0, 0.0, 0.0, 0.0};
    dvec2 na[4], nb[4];
    auto fetch = [&](int s) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            na[h] = *(GlobalD2 *)(V + (4 * s + h) * step + r0);
            nb[h] = *(GlobalD2 *)(V + (4 * s + h) * step + c0);
        }
        asm volatile("" ::: "memory");   // issued here, not where the values are first needed
    };
    const int ns = b.n / 8;   // 16 rows of V each
    fetch(0);
    for (int s = 0; s < ns; ++s) {
        dvec2 a[4], d[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            a[h] = na[h];
            d[h] = nb[h];
        }
        if (s + 1 < ns) fetch(s + 1);
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    acc[e][f] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[h][e], d[h][f], acc[e][f], 0, 0, 0);
    }
    double *Q = mat + c.qb_off + (size_t)k * Np * Np;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *(dvec2 *)(Q + (size_t)(r0 + 8 * u + 2 * lq + e) * Np + c0 + 2 * lr) = dvec2{acc[e][0][u], acc[e][1][u]};
    if (r0 == c0) return;   // symmetric in itself
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *(dvec2 *)(Q + (size_t)(c0 + 2 * lr + f) * Np + r0 + 8 * u + 2 * lq) = dvec2{acc[0][f][u], acc[1][f][u]};
}

// S = R Shat R^T: one upper 64 x 64 tile per workgroup, a 32 x 32 quarter per
// wave, on the matrix cores without an intermediate in LDS.  For 16 fine columns
// b at a time, each lane evaluates the signal at the (b, a) it holds as the first
// operand of T^T = Shat^T R_I^T; the accumulator of T^T is laid out as the second
// operand of S^T += R_J T^T.  A quarter evaluates 31 ros + rnb points a side, 1.7
// times its own.  u and sqrt(lambda), in units of the table's steps, are formed
// once per point, so that v and z are a difference and a product.  Bound by the
// gathers of the table, two 16-byte rows a point.  160 chunks of 100 to 1200 pixels
// oversampled three times: 12.7 -> 1.7 ms (as a pass of k_rm_sandwich, whose
// registers leave two waves per SIMD to hide them), error against extended
// precision 4e-14 -> 1.3e-15 of S's peak.  More than 57 taps a row take over 64 KB
// of LDS, one workgroup a CU from 81 KB on, and are faster all the same: 64 chunks
// of 480 to 600 pixels with 81 taps, S and Q_k together 25.9 -> 3.2 ms (6.2 with
// S by the sandwich).
__global__ __launch_bounds__(256) void k_rm_signal(const ChunkDev *cs, const double *rin, const TableDev *tabs,
                                                   BinsDev bins, double *mat) {
    typedef const double __attribute__((ext_vector_type(2), aligned(8), address_space(1))) GlobalD2u;
    const ChunkDev c = cs[blockIdx.y];
    const int x = blockIdx.x;
    if (!c.rm || x >= c.ntu) return;
    int J = (int)((sqrtf(8.0f * x + 1.0f) - 1.0f) * 0.5f);
    while (J * (J + 1) / 2 > x) --J;
    while ((J + 1) * (J + 2) / 2 <= x) ++J;
    const int I = x - J * (J + 1) / 2;
    const int Np = c.Np, N = c.N, M = c.rM, nb = c.rnb, os = c.ros;
    const int pitch = signal_pitch(os, nb), npt = (TILE - 1) * os + nb + 16;
    const double *R = rin + c.rin_off, *grid = R + (size_t)N * nb;
    const TableDev t = tabs[c.table];
    const int amin = c.rcol0 + I * TILE * os, bmin = c.rcol0 + J * TILE * os;
    extern __shared__ double lds[];
    double2 *pa = reinterpret_cast<double2 *>(lds), *pb = pa + npt;   // (u / dv, sqrt(lambda / dz))
    double *Ri = lds + 4 * npt, *Rj = Ri + TILE * pitch;
    const int tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    for (int e = tid; e < TILE * nb; e += 256) {
        const int r = e / nb, o = r * pitch + (e - r * nb);
        Ri[o] = (I * TILE + r < N) ? R[(size_t)I * TILE * nb + e] : 0.0;
        Rj[o] = (J * TILE + r < N) ? R[(size_t)J * TILE * nb + e] : 0.0;
    }
    const double gref = grid[min(M - 1, (amin + bmin + npt) / 2)], rdz = sqrt(t.dz);
    for (int p = tid; p < 2 * npt; p += 256) {
        const double l = grid[min(M - 1, p < npt ? amin + p : bmin + p - npt)];
        pa[p] = make_double2(SPEED_OF_LIGHT * log1p((l - gref) / gref) / t.dv, sqrt(l) / rdz);
    }
    __syncthreads();
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64), wm = wv / 2, wn = wv % 2;
    if (I == J && wm > wn) return;   // the mirror image of quarter (0, 1)
    const int a0 = 32 * wm * os, b0 = 32 * wn * os, ra = 31 * os + nb;
    const int ns = bins.turn_off_sfid ? 0 : (ra + 3) / 4, nbb = bins.turn_off_sfid ? 0 : (ra + 15) / 16;
    const double v0 = t.v1 / t.dv, z0 = (1.0 + t.z1) / t.dz;
    const double *ri0 = Ri + (32 * wm + lr) * pitch, *ri1 = ri0 + 16 * pitch;
    const double *rj0 = Rj + (32 * wn + lr) * pitch, *rj1 = rj0 + 16 * pitch;
    auto tap = [&](const double *row, int p) {   // the row's weight at its point p, 0 past its ends
        const double w = row[min((unsigned)p, (unsigned)(nb - 1))];
        return (unsigned)p < (unsigned)nb ? w : 0.0;
    };
    gd4 z[2][2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int f = 0; f < 2; ++f) z[e][f] = gd4{0.0, 0.0, 0.0, 0.0};
    for (int q = 0; q < nbb; ++q) {
        const int bl = b0 + 16 * q + lr;
        const double2 wb = pb[bl];
        gd4 t0 = {0.0, 0.0, 0.0, 0.0}, t1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int s = 0; s < ns; ++s) {
            const int al = 4 * s + lq;
            const double2 wa = pa[a0 + al];
            const double yy = ((bmin + bl >= amin + a0 + al) ? wb.x - wa.x : wa.x - wb.x) - v0;
            const double xx = wa.y * wb.y - z0;
            const int nx = interp_index(xx, t.nz), ny = interp_index(yy, t.nv);
            const double *p = t.s + ((size_t)nx + (size_t)t.nz * ny);
            const dvec2 lo = *(GlobalD2u *)p, hi = *(GlobalD2u *)(p + t.nz);
            const double dx = xx - nx, dy = yy - ny;
            const double val = (lo.x * (1 - dx) + lo.y * dx) * (1 - dy) + (hi.x * (1 - dx) + hi.y * dx) * dy;
            t0 = __builtin_amdgcn_mfma_f64_16x16x4f64(val, tap(ri0, al - lr * os), t0, 0, 0, 0);
            t1 = __builtin_amdgcn_mfma_f64_16x16x4f64(val, tap(ri1, al - (16 + lr) * os), t1, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int b = 16 * q + 4 * u + lq;
            const double w0 = tap(rj0, b - lr * os), w1 = tap(rj1, b - (16 + lr) * os);
            z[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(w0, t0[u], z[0][0], 0, 0, 0);
            z[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(w1, t0[u], z[0][1], 0, 0, 0);
            z[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(w0, t1[u], z[1][0], 0, 0, 0);
            z[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(w1, t1[u], z[1][1], 0, 0, 0);
        }
    }
    double *S = mat + c.qb_off + (size_t)c.kbu * Np * Np;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = I * TILE + 32 * wm + 16 * e + lr, j = J * TILE + 32 * wn + 16 * f + 4 * u + lq;
                if (j < i) continue;
                S[(size_t)j * Np + i] = z[e][f][u];
                S[(size_t)i * Np + j] = z[e][f][u];
            }
}

size_t rmat_signal_lds(int os, int nb) {
    // at most 90 KB under 15 os + nb <= RM_ROWS (81 taps), of a CU's 160
    return 8 * (4 * ((size_t)(TILE - 1) * os + nb + 16) + 2 * TILE * signal_pitch(os, nb));
}

size_t rmat_node_lds(int os, int nb) {
    const size_t ra = (RN_ROWS - 1) * os + nb;
    return 8 * (2 * RN_NODES * ra + RN_ROWS * nb + ra);   // at most 61 KB under 15 os + nb <= RM_ROWS
}

int rmat_nodes(double dk, double vmax) {
    // n nodes integrate cos(x t) over [-1, 1] to 1e-17 up to x = 2 (n - 8.75 n^(1/3) + 9.6)
    // (found from n = 8 to 256); beyond 256 nodes the edges cost no more.  The
    // limits are formed once: a plan asks for every band of every chunk
    struct Limits {
        double x[32];
        Limits() {
            for (int k = 0; k < 32; ++k) x[k] = 2.0 * (8.0 * (k + 1) - 8.75 * std::cbrt(8.0 * (k + 1)) + 9.6);
        }
    };
    static const Limits lim;
    if (!(dk > 0 && vmax >= 0)) return 0;
    const int k = (int)(std::lower_bound(lim.x, lim.x + 32, 0.5 * dk * vmax) - lim.x);
    return k < 32 ? 8 * (k + 1) : 0;
}

RmLayout rmat_layout(int tj, int ra_max, int rb_max, int nb_max) {
    RmLayout l;
    const int npass = (rb_max + RM_BW - 1) / RM_BW;
    l.em = (ra_max <= 80) ? 10 : RM_ROWS / 8;
    l.npass = npass;
    l.qr = 8 * l.em;
    l.tw = RM_BW * npass + 1;
    l.nbm = nb_max;
    // every entry row 8 em - 1 reads a point inside the arrays; even count: (sin, cos) pairs follow
    l.npts = (std::max(ra_max + RM_BW * npass, 8 * l.em) + 1) / 2 * 2;
    l.tj = tj;
    l.bytes = 8 * (l.qr * RM_QP + 16 * l.tw + (16 + tj) * l.nbm + 3 * l.npts);
    return l;
}

bool rmat_layout_ok(const RmLayout &lay) {
    return lay.bytes <= 65536 && ((lay.tj == 32 && lay.em == 10 && lay.npass <= 4) ||
                                  (lay.tj == 16 && (lay.em == 10 || lay.em == RM_ROWS / 8) && lay.npass <= 3));
}

bool launch_rmat(const LaunchCtx &L) {
    if (L.rm_kbu < 0) return true;
    const RmLayout &lay = L.rm_lay;
    const int nt = L.np_max / TILE;
    k_rm_signal<<<dim3(nt * (nt + 1) / 2, L.nchunks), 256, L.rm_sig_lds, L.stream>>>(L.chunks, L.rin, L.tables, L.bins,
                                                                                     L.mat);
    if (L.rm_edges) {
        const dim3 g(L.np_max / lay.tj, L.np_max / 16, L.nchunks);
        if (lay.tj == 32 && lay.em == 10 && lay.npass <= 4)
            k_rm_sandwich<32, 10, 4><<<g, 256, lay.bytes, L.stream>>>(L.chunks, L.rin, L.bins, lay, L.mat);
        else if (lay.tj == 16 && lay.em == 10 && lay.npass <= 3)
            k_rm_sandwich<16, 10, 3><<<g, 256, lay.bytes, L.stream>>>(L.chunks, L.rin, L.bins, lay, L.mat);
        else if (lay.tj == 16 && lay.em == RM_ROWS / 8 && lay.npass <= 3)
            k_rm_sandwich<16, RM_ROWS / 8, 3><<<g, 256, lay.bytes, L.stream>>>(L.chunks, L.rin, L.bins, lay, L.mat);
        else
            return false;
    }
    for (int gr = 0; gr < L.rm_groups; ++gr) {
        k_rm_nodes<<<dim3(L.np_max / RN_ROWS, L.rm_kbu, L.nchunks), 256, L.rm_lds, L.stream>>>(
            L.chunks, L.rin, L.rm_bands, L.rm_nodes, gr, L.mat);
        k_rm_bands<<<dim3(nt * (nt + 1) / 2, L.rm_kbu, L.nchunks), 256, 0, L.stream>>>(L.chunks, L.rm_bands, gr,
                                                                                       L.mat);
    }
    return true;
}

}  // namespace qml
