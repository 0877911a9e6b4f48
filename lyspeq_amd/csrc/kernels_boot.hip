// Poisson bootstrap of the per-chunk results.  FastBootstrap form
// (core/bootstrapper.hpp:183-221,282-375; core/one_qso_estimate.cpp:200-239,
// core/one_qso_estimate.hpp:55-60):
//
//   k_boot_collapse   theta_q = sum over the spectrum's chunks, in chunk order,
//                     of (d - b) - t at the chunk's fisher_index_start
//                     (OneQSOEstimate::collapseBootstrap)
//   k_boot_realize    R[b][i] = sum over spectra q, in queue order, of
//                     p[q][b] theta_q[i] (addBootPowerOnly: one dger per spectrum)
//   k_boot_mean(_part) mean[i] = (sum over b of R[b][i]) / nboots, as sum * (1/n)
//   k_boot_cov(_part) cov[i][j] = sum over b of (R[b][i] - mean[i])(R[b][j] -
//                     mean[j]), times 1/(nboots - 1) (dsyr per realisation)
//
// The complete form (k_boot_collapse_fisher, k_boot_build, the chunk
// engine's batched Cholesky, k_boot_solve) follows below.
//
// All FP64.  The sums over chunks and spectra run in the reference's order, one
// thread per output element of a 64 x 64 tile, with the operands staged through
// LDS 16 terms at a time; those over realisations run in ranges whose partial
// sums are added in order.  HBM traffic is
// small next to the chunk step (nboots x nspectra ints, nboots x T doubles).
#include "qml_common.hpp"
#include "qml_kernels.hpp"

#include <algorithm>
#include <climits>
#include <mutex>

namespace qml {

namespace {
constexpr int BT = 64;   // output tile edge
constexpr int KT = 16;   // terms staged per step
}

// One block per spectrum; its chunks are qchunk[qptr[q] .. qptr[q+1]).
__global__ __launch_bounds__(256) void k_boot_collapse(const ChunkOut *outs, const double *dbt, const int *qptr,
                                                       const int *qchunk, int T, double *theta) {
    const int q = blockIdx.x;
    const int c0 = qptr[q], c1 = qptr[q + 1];
    for (int i = threadIdx.x; i < T; i += blockDim.x) {
        double acc = 0.0;
        for (int k = c0; k < c1; ++k) {
            const ChunkOut o = outs[qchunk[k]];
            const int r = i - o.fis;
            if (r < 0 || r >= o.nq) continue;
            const double *v = dbt + o.dbt_off;
            acc += (v[r] - v[o.nq + r]) - v[2 * o.nq + r];
        }
        theta[(size_t)q * T + i] = acc;
    }
}

// R (nboots x T) = P^T Theta with P nqso x nboots (ints) and Theta nqso x T.
__global__ __launch_bounds__(256) void k_boot_realize(const int *P, const double *theta, int nqso, int nboots,
                                                      int T, double *R) {
    __shared__ double sp[KT][BT + 1], st[KT][BT + 1];
    const int b0 = blockIdx.y * BT, i0 = blockIdx.x * BT;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;   // 4 x 4 outputs per thread
    double acc[4][4] = {};
    for (int q0 = 0; q0 < nqso; q0 += KT) {
        for (int e = threadIdx.x; e < KT * BT; e += 256) {
            const int k = e / BT, c = e % BT;
            const int q = q0 + k;
            sp[k][c] = (q < nqso && b0 + c < nboots) ? (double)P[(size_t)q * nboots + b0 + c] : 0.0;
            st[k][c] = (q < nqso && i0 + c < T) ? theta[(size_t)q * T + i0 + c] : 0.0;
        }
        __syncthreads();
        const int kn = min(KT, nqso - q0);
        for (int k = 0; k < kn; ++k) {
            double p[4], t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                p[u] = sp[k][ty + 16 * u];
                t[u] = st[k][tx + 16 * u];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[u][v] += p[u] * t[v];
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int b = b0 + ty + 16 * u, i = i0 + tx + 16 * v;
            if (b < nboots && i < T) R[(size_t)b * T + i] = acc[u][v];
        }
}

// Sums over a range of realisations, blockIdx.y of gridDim.y: part[y][i], or the
// mean itself where there is one range.  One thread per band ran down all
// realisations (968 us at 4000 x 455).
__global__ __launch_bounds__(256) void k_boot_mean_part(const double *R, int nboots, int T, double *part, double *mean) {
    __shared__ double red[4][64];
    const int l = threadIdx.x % 64, w = threadIdx.x / 64, i = blockIdx.x * 64 + l;
    const int b0 = (int)((long long)nboots * blockIdx.y / gridDim.y);
    const int b1 = (int)((long long)nboots * (blockIdx.y + 1) / gridDim.y);
    double s = 0.0;
    if (i < T)
#pragma unroll 4
        for (int b = b0 + w; b < b1; b += 4) s += R[(size_t)b * T + i];
    red[w][l] = s;
    __syncthreads();
    if (w != 0 || i >= T) return;
    s = (red[0][l] + red[1][l]) + (red[2][l] + red[3][l]);
    if (gridDim.y == 1) mean[i] = s * (1.0 / nboots);
    else part[(size_t)blockIdx.y * T + i] = s;
}
__global__ __launch_bounds__(256) void k_boot_mean(const double *part, int nparts, int nboots, int T, double *mean) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= T) return;
    double s = 0.0;
    for (int p = 0; p < nparts; ++p) s += part[(size_t)p * T + i];
    mean[i] = s * (1.0 / nboots);
}

// Upper 64 x 64 tiles of sum over b of (R - mean)(R - mean)^T on the matrix
// cores: a workgroup takes one tile and the range blockIdx.y of the
// realisations, a quarter of it per wave, whose 16 blocks of 16 x 16 stay in
// registers; a fragment is 16 consecutive bands of four realisations, loaded
// one step ahead.  36 tiles at T = 455 would leave the chip empty without the
// split over realisations (798 us at 4000 x 455 with one workgroup a tile).  Where
// there is one range (under 32 realisations) the covariance itself is written,
// here and by k_boot_mean_part: a call of two realisations is a few launches.
__device__ __forceinline__ void put_cov(double *cov, int T, int i, int j, double c) {
    if (i >= T || j >= T || j < i) return;
    cov[(size_t)i * T + j] = c;
    cov[(size_t)j * T + i] = c;
}
typedef double bd4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256, 2) void k_boot_cov_part(const double *R, const double *mean, int nboots, int T,
                                                          double *part, double *cov) {
    __shared__ double red[2][4][256];
    int t = blockIdx.x, J = 0;   // tile t of the upper triangle by columns: I <= J
    while (t > J) { t -= J + 1; ++J; }
    const int I = t, tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64);
    const long long s0 = 4LL * blockIdx.y + w, ns = 4LL * gridDim.y;
    const int b0 = (int)(nboots * s0 / ns), b1 = (int)(nboots * (s0 + 1) / ns);
    int ia[4], ja[4];
    double mi[4], mj[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        ia[x] = min(64 * I + 16 * x + lr, T - 1);
        ja[x] = min(64 * J + 16 * x + lr, T - 1);
        mi[x] = mean[ia[x]];
        mj[x] = mean[ja[x]];
    }
    bd4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = bd4{0.0, 0.0, 0.0, 0.0};
    double va[4], vb[4];
    auto fetch = [&](int b) {
        const double *row = R + (size_t)min(b + lq, nboots - 1) * T;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            va[x] = row[ia[x]];
            vb[x] = row[ja[x]];
        }
    };
    if (b0 < b1) fetch(b0);
    for (int b = b0; b < b1; b += 4) {
        double a[4], c[4];
        const bool in = b + lq < b1;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            a[x] = in ? va[x] - mi[x] : 0.0;
            c[x] = in ? vb[x] - mj[x] : 0.0;
        }
        fetch(b + 4);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], c[y], acc[x][y], 0, 0, 0);
    }
    double *C = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * BT * BT;
    int flip = 0;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
#pragma unroll
            for (int u = 0; u < 4; ++u) red[flip][w][64 * u + lane] = acc[x][y][u];
            __syncthreads();
            const double c = (red[flip][0][tid] + red[flip][1][tid]) + (red[flip][2][tid] + red[flip][3][tid]);
            const int i = 16 * x + tid / 16, j = 16 * y + tid % 16;
            if (gridDim.y > 1) C[i * BT + j] = c;
            else put_cov(cov, T, 64 * I + i, 64 * J + j, c * (1.0 / (nboots - 1)));
            flip ^= 1;
        }
}
// cov from the ranges' partial tiles, mirrored into the lower triangle.
__global__ __launch_bounds__(256) void k_boot_cov(const double *part, int nparts, int nboots, int T, double *cov) {
    int t = blockIdx.x, J = 0;
    while (t > J) { t -= J + 1; ++J; }
    const int I = t;
    const double scale = 1.0 / (nboots - 1);
    for (int e = blockIdx.y * 256 + threadIdx.x; e < BT * BT; e += 256 * gridDim.y) {
        const int i = I * BT + e / BT, j = J * BT + e % BT;
        double s = 0.0;
        for (int p = 0; p < nparts; ++p) s += part[((size_t)p * gridDim.x + blockIdx.x) * BT * BT + e];
        put_cov(cov, T, i, j, s * scale);
    }
}

// Ranges of realisations for the covariance: enough for about two workgroups
// per CU, at least 16 realisations each; for the mean, at least 64.
static int cov_parts(int nboots, int T) {
    const int nt = (T + BT - 1) / BT, tiles = nt * (nt + 1) / 2;
    return std::max(1, std::min((512 + tiles - 1) / tiles, nboots / 16));
}
static int mean_parts(int nboots) { return std::max(1, std::min(64, nboots / 64)); }

// ------------------------------------------------ complete bootstrap --
// The complete form (PoissonBootstrapper::_oneBoot, core/bootstrapper.hpp:
// 223-262; OneQSOEstimate::addBoot, core/one_qso_estimate.hpp:43-53): per
// realisation b, F_b = sum over spectra of p_qb F_q (upper) and x_b the
// solution of F_b x = sum p_qb theta_q (LAPACKE_safeSolveCho,
// mathtools/matrix_helper.cpp:385-396: empty diagonals set to 1, their x
// zeroed).

// Each spectrum's collapsed Fisher matrix (OneQSOEstimate::collapseBootstrap,
// core/one_qso_estimate.cpp:224-234): ndim x ndim at fq_off[q], summed over its
// chunks in chunk order, the lower triangle (element (r, c), c <= r, is the
// chunks' (c, r)), so that k_boot_build reads along c.  A block takes 32 rows r
// of one spectrum; each 32 x 32 tile is read along r and turned in LDS.
__global__ __launch_bounds__(256) void k_boot_collapse_fisher(const ChunkOut *outs, const double *fc,
                                                              const int *qptr, const int *qchunk,
                                                              const int *qstart, const int *qdim,
                                                              const long long *fq_off, double *fq) {
    __shared__ double tile[32][33];
    const int q = blockIdx.x, r0 = blockIdx.y * 32;
    const int c0 = qptr[q], c1 = qptr[q + 1], is = qstart[q], nd = qdim[q];
    if (r0 >= nd) return;
    double *F = fq + fq_off[q];
    const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
    for (int k0 = 0; k0 <= r0; k0 += 32) {
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int i = k0 + ty + 8 * s, j = r0 + tx;   // the chunks' row and column
            double acc = 0.0;
            if (i <= j && j < nd) {
                for (int k = c0; k < c1; ++k) {
                    const ChunkOut o = outs[qchunk[k]];
                    const int a = i + is - o.fis, b = j + is - o.fis;
                    if (a < 0 || b >= o.nq) continue;   // a <= b
                    acc += fc[o.fc_off + (size_t)a * o.nq + b];
                }
            }
            tile[ty + 8 * s][tx] = acc;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int r = r0 + ty + 8 * s, c = k0 + tx;
            if (r < nd && c <= r) F[(size_t)r * nd + c] = tile[tx][ty + 8 * s];
        }
    }
}

// The batch's weights as doubles, realisation contiguous: Wt[q][b], zero past nb.
__global__ __launch_bounds__(256) void k_boot_weights(const int *W, int nqso, int b0, int nb, double *Wt) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;   // nqso BOOT_BATCH may exceed 32 bits
    const int q = (int)(e / BOOT_BATCH), b = (int)(e % BOOT_BATCH);
    if (q < nqso) Wt[e] = (b < nb) ? (double)W[(size_t)(b0 + b) * nqso + q] : 0.0;
}

// F_b's lower triangle (identity past T, empty diagonals set to 1) in the L
// slot of realisation b's matrices.  A wave takes one row r, 64 columns and RB
// realisations: the spectra covering band r in queue order are the same for
// the whole wave, so their weights are scalars and each Fisher element is
// loaded once for RB realisations (read for every realisation by itself it
// was 82 GB a batch at 4096 spectra: 3.8 ms a batch of 128 at 200 spectra,
// 0.20 ms now).  The sums run in queue order; a spectrum of weight zero adds
// nothing, also where its element is not finite.
template <int RB>
__global__ __launch_bounds__(256) void k_boot_build(const double *__restrict__ Wt, int nb, int T, int Np,
                                                    const int *__restrict__ band_ptr,
                                                    const BandEntry *__restrict__ band, const double *__restrict__ fq,
                                                    double *mat) {
    const int r = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int cb = blockIdx.x * 64, c = cb + threadIdx.x % 64, g0 = blockIdx.z * RB;
    if (cb > r) return;
    double acc[RB];
#pragma unroll
    for (int u = 0; u < RB; ++u) acc[u] = 0.0;
    if (r < T) {
        const int k1 = band_ptr[r + 1];
        for (int k = band_ptr[r]; k < k1; ++k) {
            const BandEntry e = band[k];
            if (e.is > cb + 63) continue;
            const double f = (c >= e.is && c <= r) ? fq[e.off + (long long)(r - e.is) * e.nd + (c - e.is)] : 0.0;
            const double *w = Wt + (size_t)e.q * BOOT_BATCH + g0;
            if (__builtin_expect(__any(!(fabs(f) <= 1.79769313486231571e308)), 0)) {
#pragma unroll
                for (int u = 0; u < RB; ++u)
                    if (w[u] != 0.0) acc[u] = fma(w[u], f, acc[u]);
            } else {
#pragma unroll
                for (int u = 0; u < RB; ++u) acc[u] = fma(w[u], f, acc[u]);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < RB; ++u) {
        if (g0 + u >= nb) break;
        double v = acc[u];
        if (c == r && (r >= T || v == 0.0)) v = 1.0;
        mat[(size_t)(2 * (g0 + u) + 1) * Np * Np + (size_t)r * Np + c] = v;
    }
}

// The right-hand sides, one workgroup per band, a thread per realisation.
__global__ __launch_bounds__(BOOT_BATCH) void k_boot_rhs(const double *Wt, int nb, int T, int Np, const int *band_ptr,
                                                         const BandEntry *band, const double *theta, double *rhs) {
    const int i = blockIdx.x, b = threadIdx.x;
    double acc = 0.0;
    if (i < T)
        for (int k = band_ptr[i]; k < band_ptr[i + 1]; ++k) {
            const int q = band[k].q;
            const double w = Wt[(size_t)q * BOOT_BATCH + b];
            if (w != 0.0) acc = fma(w, theta[(size_t)q * T + i], acc);
        }
    if (b < nb) rhs[(size_t)b * Np + i] = acc;
}

// x of L L^T x = rhs per realisation (one block each) by block substitution
// with the inverted diagonal blocks, written to R[b0 + b] (T values): one
// right-hand side needs no more of the inverse, whose other blocks were two
// thirds of the factorisation's work.  A band no weighted spectrum covers has a
// zero row and a zero right-hand side with its diagonal set to 1, so its x is
// zero, as safeSolveCho leaves it.  Each block row is a matrix-vector product of
// all 512 threads: forward eight threads to a row, 128 bytes of it each time;
// backward a wave to every eighth row, 512 bytes of it.
__global__ __launch_bounds__(512) void k_boot_solve(const double *mat, const double *rhs, int b0, int T, int Np,
                                                    double *R) {
    const int b = blockIdx.x, tid = threadIdx.x, nt = Np / 64;
    const double *L = mat + (size_t)(2 * b + 1) * Np * Np, *Li = L + (size_t)Np * Np;
    extern __shared__ double sh[];
    double *y = sh, *t = sh + Np, *red = t + 64;   // Np, 64, 8 x 64
    const int row = tid / 8, o = tid % 8, w = tid / 64, l = tid % 64;
    for (int i = tid; i < Np; i += 512) y[i] = rhs[(size_t)b * Np + i];
    __syncthreads();
    auto row_sum = [&](double s) {
        for (int d = 4; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
        return s;
    };
    for (int p = 0; p < nt; ++p) {
        const double *Lr = L + (size_t)(64 * p + row) * Np;
        double s = 0.0;
#pragma unroll 4
        for (int k = 2 * o; k < 64 * p; k += 16) {
            const dvec2 v = *(const dvec2 *)(Lr + k);
            s += v.x * y[k] + v.y * y[k + 1];
        }
        s = row_sum(s);
        if (o == 0) t[row] = y[64 * p + row] - s;
        __syncthreads();
        const double *Ir = Li + (size_t)(64 * p + row) * Np + 64 * p;
        s = 0.0;
#pragma unroll
        for (int k = 2 * o; k < 64; k += 16) {
            const dvec2 v = *(const dvec2 *)(Ir + k);
            s += v.x * t[k] + v.y * t[k + 1];
        }
        s = row_sum(s);
        __syncthreads();
        if (o == 0) y[64 * p + row] = s;
        __syncthreads();
    }
    auto col_sum = [&](double s, double *dst, double sign, const double *add) {
        red[64 * w + l] = s;
        __syncthreads();
        if (w == 0) {
            double v = 0.0;
            for (int q = 0; q < 8; ++q) v += red[64 * q + l];
            dst[l] = (add ? add[l] : 0.0) + sign * v;
        }
        __syncthreads();
    };
    for (int p = nt - 1; p >= 0; --p) {
        double s = 0.0;
#pragma unroll 8
        for (int i = 64 * (p + 1) + w; i < Np; i += 8) s += L[(size_t)i * Np + 64 * p + l] * y[i];
        col_sum(s, t, -1.0, y + 64 * p);
        s = 0.0;
#pragma unroll
        for (int i = w; i < 64; i += 8) s += Li[(size_t)(64 * p + i) * Np + 64 * p + l] * t[i];
        col_sum(s, y + 64 * p, 1.0, nullptr);
    }
    for (int i = tid; i < T; i += 512) R[(size_t)(b0 + b) * T + i] = y[i];
}

void launch_boot_collapse_fisher(hipStream_t st, const ChunkOut *outs, const double *fc, const int *qptr,
                                 const int *qchunk, const int *qstart, const int *qdim, const long long *fq_off,
                                 int nqso, int dim_max, double *fq) {
    k_boot_collapse_fisher<<<dim3(nqso, (dim_max + 31) / 32), 256, 0, st>>>(outs, fc, qptr, qchunk, qstart, qdim,
                                                                           fq_off, fq);
}

void launch_boot_build(hipStream_t st, const int *W, int nqso, int b0, int nb, int T, int Np, const int *band_ptr,
                       const BandEntry *band, const double *fq, const double *theta, double *Wt, double *mat,
                       double *rhs) {
    constexpr int RB = 32;
    static_assert(BOOT_BATCH % RB == 0, "whole groups of realisations");
    k_boot_weights<<<((size_t)nqso * BOOT_BATCH + 255) / 256, 256, 0, st>>>(W, nqso, b0, nb, Wt);
    k_boot_build<RB><<<dim3(Np / 64, Np / 4, (nb + RB - 1) / RB), 256, 0, st>>>(Wt, nb, T, Np, band_ptr, band, fq, mat);
    k_boot_rhs<<<Np, BOOT_BATCH, 0, st>>>(Wt, nb, T, Np, band_ptr, band, theta, rhs);
}

void launch_boot_solve(hipStream_t st, const double *mat, const double *rhs, int b0, int nb, int T, int Np,
                       double *R) {
    k_boot_solve<<<nb, 512, ((size_t)Np + 64 + 512) * sizeof(double), st>>>(mat, rhs, b0, T, Np, R);
}

void launch_boot_collapse(hipStream_t st, const ChunkOut *outs, const double *dbt, const int *qptr,
                          const int *qchunk, int nqso, int T, double *theta) {
    k_boot_collapse<<<nqso, 256, 0, st>>>(outs, dbt, qptr, qchunk, T, theta);
}

size_t boot_meancov_scratch(int nboots, int T) {
    const size_t nt = (T + BT - 1) / BT;
    return std::max((size_t)mean_parts(nboots) * T, (size_t)cov_parts(nboots, T) * (nt * (nt + 1) / 2) * BT * BT);
}
void launch_boot_meancov(hipStream_t st, const double *R, int nboots, int T, double *scratch, double *mean,
                         double *cov) {
    const int nt = (T + BT - 1) / BT, tiles = nt * (nt + 1) / 2, mp = mean_parts(nboots), cp = cov_parts(nboots, T);
    k_boot_mean_part<<<dim3(nt, mp), 256, 0, st>>>(R, nboots, T, scratch, mean);
    if (mp > 1) k_boot_mean<<<(T + 255) / 256, 256, 0, st>>>(scratch, mp, nboots, T, mean);
    k_boot_cov_part<<<dim3(tiles, cp), 256, 0, st>>>(R, mean, nboots, T, scratch, cov);
    if (cp > 1) k_boot_cov<<<dim3(tiles, 4), 256, 0, st>>>(scratch, cp, nboots, T, cov);
}

void launch_bootstrap(hipStream_t st, const ChunkOut *outs, const double *dbt, const int *qptr, const int *qchunk,
                      int nqso, int T, const int *P, int nboots, double *theta, double *R, double *scratch,
                      double *mean, double *cov) {
    launch_boot_collapse(st, outs, dbt, qptr, qchunk, nqso, T, theta);
    const int tt = (T + BT - 1) / BT;
    k_boot_realize<<<dim3(tt, (nboots + BT - 1) / BT), 256, 0, st>>>(P, theta, nqso, nboots, T, R);
    launch_boot_meancov(st, R, nboots, T, scratch, mean, cov);
}

// ---------------------------------------------------------------------------
// Median bootstrap (PoissonBootstrapper::_medianBootstrap,
// core/bootstrapper.hpp:301-346,376-390, with stats::medianOfUnsortedVector,
// mathtools/stats.cpp:8-28): per band the median over the realisations, the
// deviations from it, and per band pair (i <= j) the median of the products
// of the deviations, mirrored to the lower triangle.  A median of n values is
// the value of rank n/2 for odd n and the half-sum of ranks n/2 - 1 and n/2
// for even n, the ranks of the ascending order.
//
// One workgroup per median.  Up to MED_REGS values per thread stay in registers
// and the rank is closed in by counting: 64 evenly spaced values, sorted in each
// wave, give the first pivots; a count is one compare and one population count
// per 64 values and one barrier, and the next pivot follows from it, first among
// the sorted sample, then by interpolation between the bracket's ends; what is
// left at 64 values or fewer is ranked exactly.  Eight counts are typical.  Where
// two pivots have nothing between them, the least value of the bracket and its
// copies are counted: a median with many equal values ends there.  The values are
// read once; the radix select below reads them three times and its waves queue on
// the few histogram bins that hold a band pair's exponents.  Bound by the barriers
// and compares of the counts.  455 bands x 8000 realisations: 4.65 -> 2.31 ms for
// the 103740 pairs.  Whole calls with the copies: 5.7 -> 3.3 ms, x 500 1.29 -> 1.04; 200 bands of whole numbers x 8000
// 2.3 -> 0.89, x 500 0.38 -> 0.23 (2.7 and 0.65 where counting gave up on equal
// values and the radix select followed).
//
// Few bands, longer columns (more than 8192 values), NaNs, and brackets with an
// end at infinity or whose copies part the two ranks of an even count take a radix
// select over order-preserving 64-bit keys of the FP64 values: eight passes of 8
// bits, most significant first, each a 256-bin LDS histogram of the values
// still matching the selected prefix and a block scan that picks the digit
// holding the rank; for even n one more pass counts the values at or below the
// selected one and finds the next larger value.  After the first two passes the
// keys of the selected bin (up to 4096) are copied to LDS and the rest of the
// select reads only them.  Either way the selected values are the sorted
// array's, bit for bit; products are formed the same way in every pass (one FP64
// multiply).  Realisations are transposed first so that a band's values are
// contiguous.

namespace {

// Ascending keys are ascending values; -0 sorts below +0 (the two are equal
// values, so the median does not depend on it).
__device__ __forceinline__ unsigned long long order_key(double x) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

__device__ __forceinline__ double key_value(unsigned long long k) {
    const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)u);
}

template <bool PROD>
__device__ __forceinline__ unsigned long long median_term(const double *a, const double *b, int i) {
    return order_key(PROD ? a[i] * b[i] : a[i]);
}

constexpr int MED_CAP = 4096;   // keys of the median's 16-bit bin kept in LDS
constexpr int MED_REGS = 32;    // values per thread held in registers, at most

struct SelectLds {
    unsigned int hist[256];
    unsigned int wave_tot[4];
    unsigned long long wave_min[4];
    unsigned int digit, rank, binsize, ncand;
    unsigned long long cand[MED_CAP];
};

// One radix pass: the 8-bit digit at `shift` of the keys key(i), i < count,
// that match prefix under mask; selects the digit whose bin holds rank r and
// leaves r as the rank within that bin and s.binsize as the bin's count.
template <class Key>
__device__ void radix_pass(Key key, int count, int shift, unsigned long long &prefix, unsigned long long &mask,
                           unsigned int &r, SelectLds &s) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    s.hist[tid] = 0;
    __syncthreads();
    for (int i = tid; i < count; i += 256) {
        const unsigned long long k = key(i);
        if ((k & mask) == prefix) atomicAdd(&s.hist[(k >> shift) & 255u], 1u);
    }
    __syncthreads();
    // inclusive scan of the 256 bins: within the wave, then across waves
    const unsigned int c = s.hist[tid];
    unsigned int incl = c;
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned int v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
    }
    if (lane == 63) s.wave_tot[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += s.wave_tot[w];
    const unsigned int excl = incl - c;
    if (excl <= r && r < incl) {   // exactly one bin holds the rank
        s.digit = (unsigned)tid;
        s.rank = r - excl;
        s.binsize = c;
    }
    __syncthreads();
    prefix |= (unsigned long long)s.digit << shift;
    mask |= 0xffull << shift;
    r = s.rank;
    __syncthreads();
}

// Block-wide sum of cnt and minimum of mn; every thread gets both.
__device__ void block_sum_min(unsigned int &cnt, unsigned long long &mn, SelectLds &s) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int d = 32; d >= 1; d >>= 1) {
        cnt += __shfl_xor(cnt, d, 64);
        const unsigned long long o = __shfl_xor(mn, d, 64);
        mn = o < mn ? o : mn;
    }
    if (lane == 0) {
        s.wave_tot[wave] = cnt;
        s.wave_min[wave] = mn;
    }
    __syncthreads();
    cnt = 0;
    mn = ~0ull;
    for (int w = 0; w < 4; ++w) {
        cnt += s.wave_tot[w];
        mn = s.wave_min[w] < mn ? s.wave_min[w] : mn;
    }
    __syncthreads();
}

// Among key(i), i < count: how many are <= sel, and the smallest above it.
template <class Key>
__device__ void count_le_min_gt(Key key, int count, unsigned long long sel, unsigned int &tot,
                                unsigned long long &gmin, SelectLds &s) {
    unsigned int cnt = 0;
    unsigned long long mn = ~0ull;
    for (int i = threadIdx.x; i < count; i += 256) {
        const unsigned long long k = key(i);
        if (k <= sel) ++cnt;
        else mn = k < mn ? k : mn;
    }
    block_sum_min(cnt, mn, s);
    tot = cnt;
    gmin = mn;
}

__device__ __forceinline__ double lane_value(double x, int lane) {   // lane is uniform
    const long long u = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// The next double above x < infinity.
__device__ __forceinline__ double value_above(double x) {
    const long long u = __double_as_longlong(x);
    return x == 0.0 ? __longlong_as_double(1) : __longlong_as_double(x > 0.0 ? u + 1 : u - 1);
}

// The median of the n <= 256 R values by counting (see above); false where it
// is left to the radix select.  Called by all 256 threads.
template <bool PROD, int R>
__device__ bool count_median(const double *a, const double *b, int n, SelectLds &s, double &median) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool two = n % 2 == 0;
    const int r0 = two ? n / 2 - 1 : n / 2, r1 = r0 + two;   // the ranks wanted
    double v[R];
    bool nan = false;
    constexpr int G = R < 8 ? R : 8;
#pragma unroll
    for (int g = 0; g < R; g += G) {   // eight loads in flight, none behind a test of its own
#pragma unroll
        for (int k = g; k < g + G; ++k) v[k] = __builtin_inf();   // never below a pivot
        if (R == G || 256 * g < n) {
#pragma unroll
            for (int k = g; k < g + G; ++k) {
                const int i = tid + 256 * k, e = min(i, n - 1);
                const double x = PROD ? a[e] * b[e] : a[e];
                nan |= x != x;
                v[k] = i < n ? x : __builtin_inf();
            }
        }
    }
    // the same sorted sample in every wave, one value a lane
    double smp;
    {
        const int i = (int)((long long)lane * n / 64);
        smp = PROD ? a[i] * b[i] : a[i];
#pragma unroll
        for (int k = 2; k <= 64; k *= 2)
#pragma unroll
            for (int j = k / 2; j >= 1; j /= 2) {
                const double o = __shfl_xor(smp, j, 64);
                smp = (((lane & k) == 0) == ((lane & j) == 0)) ? fmin(smp, o) : fmax(smp, o);
            }
    }
    if (tid == 0) s.ncand = 0;
    if (lane == 0) s.wave_min[wave] = 0;
    if (__any(nan) && lane == 0) s.wave_min[wave] = 1;
    int turn = 0;
    auto total = [&](int c) {   // over the waves
        unsigned int *tot = s.hist + 4 * (turn++ & 1);
        if (lane == 0) tot[wave] = (unsigned int)c;
        __syncthreads();
        return __builtin_amdgcn_readfirstlane((int)(tot[0] + tot[1] + tot[2] + tot[3]));
    };
    // values below pl: cl <= r0 of them; below ph: ch > r1
    int cl = 0, ch = n, L = -1, H = 64, m = (int)((long long)r0 * 64 / n);
    double pl = -__builtin_inf(), ph = __builtin_inf();
    bool open = true;   // no upper end yet
    // The least value t not below pl: 1 if both ranks lie among its copies, else 0
    // with the lower end past them, or 2 where the copies part the ranks.
    auto settle = [&]() -> int {
        double t = __builtin_inf();
#pragma unroll
        for (int k = 0; k < R; ++k) t = v[k] >= pl ? fmin(t, v[k]) : t;
        for (int d = 1; d < 64; d *= 2) t = fmin(t, __shfl_xor(t, d, 64));
        // past total's places: a wave may still be reading the NaN flags in wave_min
        double *mins = reinterpret_cast<double *>(s.hist + 8);
        if (lane == 0) mins[wave] = t;
        __syncthreads();
        t = fmin(fmin(mins[0], mins[1]), fmin(mins[2], mins[3]));
        t = lane_value(t, 0);   // uniform, and so the next pivots
        if (!(t < __builtin_inf())) return 2;
        int c = 0, z = 0;
#pragma unroll
        for (int k = 0; k < R; ++k) c += __popcll(__ballot(v[k] <= t));
        c = total(c);
        if (c <= r0) {
            cl = c;
            pl = value_above(t);
            return 0;
        }
        if (c <= r1) return 2;
        if (t == 0.0) {   // -0 sorts before +0
#pragma unroll 1
            for (int i = tid; i < (n + 255) / 256 * 256; i += 256) {
                const double x = i < n ? (PROD ? a[i] * b[i] : a[i]) : 0.0;
                z += __popcll(__ballot(__double_as_longlong(x) == LLONG_MIN));
            }
            z = total(z) + cl;
        }
        const double lo = t == 0.0 ? (r0 < z ? -0.0 : 0.0) : t, hi = t == 0.0 ? (r1 < z ? -0.0 : 0.0) : t;
        median = two ? (lo + hi) / 2 : lo;
        return 1;
    };
    for (int step = 0; ch - cl > 64; ++step) {
        if (step == 24) return false;
        double p;
        if (H - L > 1) {
            p = lane_value(smp, m);
        } else {   // between two finite ends
            p = pl + (ph - pl) * ((r0 + 0.5 - cl) / (ch - cl) + ((step & 1) ? 0.06 : -0.06));
            if (!(p > pl && p < ph)) return false;
        }
        int c = 0;
#pragma unroll
        for (int k = 0; k < R; ++k) c += __popcll(__ballot(v[k] < p));
        c = total(c);
        if (step == 0 && (s.wave_min[0] | s.wave_min[1] | s.wave_min[2] | s.wave_min[3])) return false;
        const bool below = c <= r0, above = c > r1;
        if (!below && !above) return false;   // the pivot parts the two ranks
        const bool still = c == (below ? cl : ch);
        if (below) {
            cl = c;
            pl = p;
        } else {
            ch = c;
            ph = p;
            open = false;
        }
        bool stuck = false;
        if (H - L > 1) {
            // the sample's own spacing to the rank, then one further, so that the
            // next count closes the bracket from the other side
            if (below) L = m;
            else H = m;
            const int d = (int)((long long)(r0 - c) * 64 / n);
            m = m + d + (below ? 1 : -1);
            m = max(L + 1, min(H - 1, m));
            stuck = (below && still) || (H - L <= 1 && (open || L < 0 || !(ph - pl < __builtin_inf())));
        } else {
            stuck = still;   // nothing between the last two pivots
        }
        if (stuck) {   // many equal values, or an end at infinity
            const int r = settle();
            if (r == 1) return true;
            if (r == 2 || (H - L <= 1 && (open || !(ph - pl < __builtin_inf())))) return false;
        }
    }
    __syncthreads();
    // at most 64 values in [pl, ph)
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const bool in = v[k] >= pl && (open ? tid + 256 * k < n : v[k] < ph);
        const unsigned long long mask = __ballot(in);
        if (mask) {
            unsigned int base = 0;
            if (lane == 0) base = atomicAdd(&s.ncand, (unsigned int)__popcll(mask));
            base = __shfl(base, 0, 64) + __popcll(mask & ((1ull << lane) - 1));
            if (in && base < 64) s.cand[base] = order_key(v[k]);
        }
    }
    __syncthreads();
    const int cnt = (int)s.ncand;
    if (cnt != ch - cl) return false;   // NaNs before any count
    // the rank of this lane's key among them; equal keys keep their places
    const unsigned long long key = s.cand[min(lane, cnt - 1)];
    int rank = 0;
    for (int j = 0; j < cnt; ++j) {
        const unsigned long long o = s.cand[j];
        rank += (o < key) || (o == key && j < lane);
    }
    if (lane < cnt && rank == r0 - cl) s.wave_min[0] = key;   // every wave writes the same
    if (lane < cnt && rank == r1 - cl) s.wave_min[1] = key;
    __syncthreads();
    const double lo = key_value(s.wave_min[0]), hi = key_value(s.wave_min[1]);
    median = two ? (lo + hi) / 2 : lo;
    return true;
}

// The median of the n values a[i] (PROD false) or a[i] * b[i] (PROD true).
// Called by all 256 threads of the block; every thread returns the median.  By
// counting if R > 0 values per thread hold the column, else by radix select.
// The first two passes read the values; when the selected 16-bit bin holds
// at most MED_CAP keys they are copied to LDS once and the remaining six
// passes (and the even-count step) read only those, else every pass reads
// the values again.
template <bool PROD, int R>
__device__ double block_median(const double *a, const double *b, int n, SelectLds &s) {
    if (R > 0 && n <= 256 * R) {
        double m;
        if (count_median<PROD, (R > 0 ? R : 1)>(a, b, n, s, m)) return m;
        __syncthreads();
    }
    const unsigned int r_lo = (n % 2 == 0) ? (unsigned)(n / 2 - 1) : (unsigned)(n / 2);
    auto gkey = [a, b](int i) { return median_term<PROD>(a, b, i); };
    auto lkey = [&s](int i) { return s.cand[i]; };
    unsigned long long prefix = 0, mask = 0;
    unsigned int r = r_lo;
    radix_pass(gkey, n, 56, prefix, mask, r, s);
    radix_pass(gkey, n, 48, prefix, mask, r, s);
    const unsigned int nbin = s.binsize, r_bin = r;
    const bool in_lds = nbin <= (unsigned)MED_CAP;
    unsigned long long above = ~0ull;   // smallest key above the bin
    if (in_lds) {
        if (threadIdx.x == 0) s.ncand = 0;
        __syncthreads();
        unsigned int unused = 0;
        for (int i = threadIdx.x; i < n; i += 256) {
            const unsigned long long k = gkey(i);
            if ((k & mask) == prefix) {
                const unsigned int at = atomicAdd(&s.ncand, 1u);
                if (at < (unsigned)MED_CAP) s.cand[at] = k;   // at < nbin always
            } else if (k > prefix) {
                above = k < above ? k : above;
            }
        }
        block_sum_min(unused, above, s);
        for (int shift = 40; shift >= 0; shift -= 8) radix_pass(lkey, (int)nbin, shift, prefix, mask, r, s);
    } else {
        for (int shift = 40; shift >= 0; shift -= 8) radix_pass(gkey, n, shift, prefix, mask, r, s);
    }
    const double lo = key_value(prefix);
    if (n % 2 != 0) return lo;
    // even n: the value of rank n/2 is lo itself when more than n/2 values
    // are at or below it, else the smallest value above it
    unsigned int tot;
    unsigned long long gmin;
    double hi;
    if (in_lds) {
        // (r_lo - r_bin) values lie below the bin
        count_le_min_gt(lkey, (int)nbin, prefix, tot, gmin, s);
        hi = (tot >= r_bin + 2) ? lo : key_value(gmin < above ? gmin : above);
    } else {
        count_le_min_gt(gkey, n, prefix, tot, gmin, s);
        hi = (tot >= (unsigned)(n / 2 + 1)) ? lo : key_value(gmin);
    }
    return (lo + hi) / 2;
}
}  // namespace

// R (nboots x T, one realisation per row) to X (T x nboots), 64 x 64 tiles.
__global__ __launch_bounds__(256) void k_boot_transpose(const double *R, int nboots, int T, double *X) {
    __shared__ double tile[64][65];
    const int b0 = blockIdx.y * 64, i0 = blockIdx.x * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int rr = ty; rr < 64; rr += 4) {
        const int b = b0 + rr, i = i0 + tx;
        tile[rr][tx] = (b < nboots && i < T) ? R[(size_t)b * T + i] : 0.0;
    }
    __syncthreads();
    for (int rr = ty; rr < 64; rr += 4) {
        const int i = i0 + rr, b = b0 + tx;
        if (i < T && b < nboots) X[(size_t)i * nboots + b] = tile[tx][rr];
    }
}

// One block per band: median[i], then X[i][:] -= median[i] (_calcuateMedian,
// and the subtraction at the start of _calcuateMadCovariance).
template <int R>
__global__ __launch_bounds__(256, 4) void k_boot_median(double *X, int nboots, double *median) {
    __shared__ SelectLds s;
    double *x = X + (size_t)blockIdx.x * nboots;
    const double m = block_median<false, R>(x, x, nboots, s);
    if (threadIdx.x == 0) median[blockIdx.x] = m;
    __syncthreads();
    for (int i = threadIdx.x; i < nboots; i += 256) x[i] -= m;
}

// One block per band pair j >= i: mad[i][j] = mad[j][i] = median over b of
// X[i][b] X[j][b].  The triangle is folded into a grid of W = T rounded up to 8
// by 8 (Q + 1), Q = ceil((W - 8) / 16): row y = 8 q + r holds the pairs of i = y
// and, left of them, those of i = W - 8 q + r, shifted by whole eights.  So column
// x always reads the bands j = x mod 8, an eighth of them per XCD, whose L2 then
// holds them.  455 bands, the whole call: 8000 realisations 3.85 -> 3.76 ms, 20000
// 12.8 -> 12.7; 200 bands of 20000 3.2 -> 2.8, 257 of 12000 3.0 -> 2.4 (folded
// with a width of T + 1, where a band is read on every XCD).
template <int R>
__global__ __launch_bounds__(256, 4) void k_boot_mad(const double *X, int nboots, int T, double *mad) {
    const int x = blockIdx.x, y = blockIdx.y, up = (int)gridDim.x - y / 8 * 8;
    const bool left = x < y / 8 * 8;
    const int i = left ? up + y % 8 : y, j = left ? x + up : x;
    if (j < i || j >= T || (left && i < (int)gridDim.y)) return;   // rows below gridDim.y are first ones
    __shared__ SelectLds s;
    const double m = block_median<true, R>(X + (size_t)i * nboots, X + (size_t)j * nboots, nboots, s);
    if (threadIdx.x == 0) {
        mad[(size_t)i * T + j] = m;
        mad[(size_t)j * T + i] = m;
    }
}

template <int R>
static void launch_medians(hipStream_t st, int nboots, int T, double *X, double *median, double *mad) {
    k_boot_median<R><<<T, 256, 0, st>>>(X, nboots, median);
    const int W = (T + 7) / 8 * 8, Q = (W - 8 + 15) / 16;
    k_boot_mad<R><<<dim3(W, 8 * (Q + 1)), 256, 0, st>>>(X, nboots, T, mad);
}

void launch_boot_median(hipStream_t st, const double *R, int nboots, int T, double *X, double *median,
                        double *mad) {
    k_boot_transpose<<<dim3((T + 63) / 64, (nboots + 63) / 64), 256, 0, st>>>(R, nboots, T, X);
    // Values per thread, by the registers they take (two each) and the loads and
    // compares past the column's end: 455 bands with the copies, 500 realisations
    // 1.04 ms with 2, 1.13 with 8 (radix select 1.29), 2048 1.50 with 8 (2.0), 8000
    // 3.3 with 32 (5.7).  With 80, two waves run on a SIMD and the counts' masks
    // spill: 8193 5.9 -> 8.0, 20000 13.9 -> 16.6, so longer columns take the radix
    // select (12.7 at 20000).  Where the pairs fit the chip at once (256 CUs, four
    // workgroups each), a pair's own latency counts, and the radix select's is the
    // shorter: 32 bands, 500 realisations 91 us (97 by counting), 8000 243 (253); 64
    // bands 111 (112) and 386 (351).
    if (T * (T + 1LL) / 2 <= 1024)
        launch_medians<0>(st, nboots, T, X, median, mad);
    else if (nboots <= 256 * 2)
        launch_medians<2>(st, nboots, T, X, median, mad);
    else if (nboots <= 256 * 8)
        launch_medians<8>(st, nboots, T, X, median, mad);
    else if (nboots <= 256 * MED_REGS)
        launch_medians<MED_REGS>(st, nboots, T, X, median, mad);
    else
        launch_medians<0>(st, nboots, T, X, median, mad);
}

// Scratch of the allocation-free median bootstrap: the realisations
// transposed to band-major, BOOT_NOALLOC_MAX doubles (64 MiB) per device,
// held from the library's load on a device until the process ends.  Its
// address on each device comes from hipGetSymbolAddress at qml_create (with
// that device current); host code never passes the array's own name.
static __device__ __align__(256) double scratch[BOOT_NOALLOC_MAX];

namespace {
std::mutex g_scratch_mu;
double *g_scratch_ptr[BOOT_NOALLOC_DEVICES] = {};
}

int boot_noalloc_setup(int device) {
    if (device < 0 || device >= BOOT_NOALLOC_DEVICES) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return (int)hipSuccess;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    g_scratch_ptr[device] = (double *)ptr;
    return (int)hipSuccess;
}

double *boot_noalloc_scratch(int device) {
    if (device < 0 || device >= BOOT_NOALLOC_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_ptr[device];
}

}  // namespace qml
