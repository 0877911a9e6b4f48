// The S/Q lookup tables on the device (SQLookupTable::computeTables,
// core/sq_table.cpp:201-323), for many (R, dv) pairs at once.
//
//   derivative: Q_kn(v) = (1/pi) int_{k1}^{k2} W(k)^2 cos(k v) dk, W(k) =
//               sinc(k dv/2) exp(-(k R)^2/2), R the 1-sigma resolution in
//               km/s (core/fiducial_cosmology.cpp:305-331).  The reference
//               integrates with QUADPACK's QAWO; here Filon's rule over 2M
//               panels, which integrates the cosine weight exactly and the
//               smooth W^2 to O(h^4).
//   signal:     the reference's real FFT of W^2 P_fid(k, z) on n = 2^(ceil(
//               log2(4 Nv)) + 1) points spaced dx = (Lv/(Nv-1))/2, divided by
//               the grid length, every second point kept (core/sq_table.cpp:
//               221-227,296-311; mathtools/real_field.cpp:40-92).  The kept
//               points are the inverse transform's cosine sums, evaluated here
//               directly: S(v_j) = (1/L) [F_0 + 2 sum_{0<m<n/2} F_m cos(k_m v_j)
//               + F_{n/2}], with the modes where W^2 < 1e-40 W^2(0) left out.
//
// Derivative: one workgroup per (pair, band, 256 velocities); the integrand at
// the Filon nodes sits in LDS and each thread sums one velocity with the cosine
// advanced by the three-term recurrence, re-seeded every 32 steps.
// Signal: a matrix product over the modes, cos(k_m v_j) x W^2(m) P(m, z), on the
// FP64 matrix cores (see k_signal_sum).
#include "qml_common.hpp"
#include "qml_kernels.hpp"

namespace qml {

namespace {

constexpr double TAB_PI = 3.14159265358979323846;

__device__ __forceinline__ double window_sq(double k, double dv, double R) {
    const double x = k * dv / 2.0;
    const double s = (x == 0.0) ? 1.0 : sin(x) / x;
    const double kr = k * R;
    const double w = s * exp(-kr * kr / 2.0);
    return w * w;
}

// Filon's alpha, beta, gamma at theta = t h (series below 0.02)
__device__ __forceinline__ void filon_coeffs(double th, double &a, double &b, double &g) {
    if (fabs(th) < 0.02) {
        const double t2 = th * th;
        a = 2.0 * th * t2 / 45.0 - 2.0 * th * t2 * t2 / 315.0 + 2.0 * th * t2 * t2 * t2 / 4725.0;
        b = 2.0 / 3.0 + 2.0 * t2 / 15.0 - 4.0 * t2 * t2 / 105.0 + 2.0 * t2 * t2 * t2 / 567.0;
        g = 4.0 / 3.0 - 2.0 * t2 / 15.0 + t2 * t2 / 210.0 - t2 * t2 * t2 / 11340.0;
        return;
    }
    double s, c;
    sincos(th, &s, &c);
    const double t3 = th * th * th;
    a = (th * th + th * s * c - 2.0 * s * s) / t3;
    b = 2.0 * (th * (1.0 + c * c) - 2.0 * s * c) / t3;
    g = 4.0 * (s - th * c) / t3;
}

constexpr int MAX_FILON_NODES = 2 * 128 + 1;

// pairs: (R_kms, dv) per table; out: npairs x nk x nv
__global__ __launch_bounds__(256) void k_deriv_table(const double *pairs, const double *kedges, int nk, int nv,
                                                     double dxv, int M, double *out) {
    const int kn = blockIdx.y, p = blockIdx.z;
    const double R = pairs[2 * p], dv = pairs[2 * p + 1];
    const double a = kedges[kn], b = kedges[kn + 1];
    const double h = (b - a) / (2 * M);
    __shared__ double f[MAX_FILON_NODES];
    for (int j = threadIdx.x; j <= 2 * M; j += 256) f[j] = window_sq(a + j * h, dv, R) / TAB_PI;
    __syncthreads();
    const int iv = blockIdx.x * 256 + threadIdx.x;
    if (iv >= nv) return;
    const double t = dxv * iv;
    double al, be, ga;
    filon_coeffs(t * h, al, be, ga);
    const double twoc = 2.0 * cos(t * h);
    double se = 0.0, so = 0.0, cprev = 0.0, c = 0.0;
    for (int j = 0; j <= 2 * M; ++j) {
        if (j % 32 == 0) {
            // re-seed: c = cos(t x_j), cprev = cos(t x_{j-1})
            c = cos(t * (a + j * h));
            cprev = cos(t * (a + (j - 1) * h));
        }
        const double term = f[j] * c;
        if (j & 1) so += term;
        else se += term;
        const double cn = twoc * c - cprev;
        cprev = c;
        c = cn;
    }
    // the end nodes carry half the even weight
    se -= 0.5 * (f[0] * cos(t * a) + f[2 * M] * cos(t * b));
    const double v = h * (al * (f[2 * M] * sin(t * b) - f[0] * sin(t * a)) + be * se + ga * so);
    out[((size_t)p * nk + kn) * nv + iv] = v;
}

// P_fid(k_m, z_i) (core/fiducial_cosmology.cpp:273-282) on the signal grid:
// pk[m * nzp + i], zero for i >= nz and past the last mode.  Eight modes and 32
// redshifts a workgroup: mpad nzp may exceed 32 bits (4097 velocities at 65535
// redshifts: 2.1e9)
__global__ __launch_bounds__(256) void k_pfid_grid(double dk, int nmode, int mpad, double z1, double dz, int nz, int nzp,
                                                   PD13 pd, double *pk) {
    const int m = blockIdx.x * 8 + threadIdx.x / 32, iz = blockIdx.y * 32 + threadIdx.x % 32;
    if (m >= mpad || iz >= nzp) return;
    double p = 0.0;
    if (m < nmode && iz < nz) {
        const double k = m * dk, z = z1 + dz * iz;
        const double K0 = 0.009, Z0 = 3.0;
        const double q0 = k / K0 + 1e-15;
        const double x0 = (1.0 + z) / (1.0 + Z0);
        const double lq = log(q0);
        p = pd.A * TAB_PI / K0 * pow(q0, 2.0 + pd.n + pd.alpha * lq + pd.beta * log(x0)) * pow(x0, pd.B) /
            (1.0 + pd.lambda * k * k);
    }
    pk[(size_t)m * nzp + iz] = p;
}

// W^2 of each pair's modes, doubled where the inverse transform counts a mode
// twice: w2[p * mpad + m], zero past the pair's last kept mode.
__global__ __launch_bounds__(256) void k_signal_window(const double *pairs, const int *mend, int nhalf, int mpad,
                                                       double dk, double *w2) {
    const int p = blockIdx.y, m = blockIdx.x * 256 + threadIdx.x;
    if (m >= mpad) return;
    double w = 0.0;
    if (m <= mend[p]) w = ((m == 0 || m == nhalf) ? 1.0 : 2.0) * window_sq(m * dk, pairs[2 * p + 1], pairs[2 * p]);
    w2[(size_t)p * mpad + m] = w;
}

// out[p][iv][iz] = inv_len times the sum over pair p's modes of
// cos(k_m v_iv) w2(m) pk(m, iz), z contiguous.  A workgroup takes 32 velocities
// and 16 Y redshifts, its eight waves an eighth of the modes each, four modes a
// step on v_mfma_f64_16x16x4f64: lane l's A values are the cosines of its two
// velocities at mode l / 16 of the step, advanced by rotation by four modes and
// re-seeded every 256 modes; its B values the weighted power at that mode.  The
// phase k_m v_iv = 2 pi m iv / nhalf, nhalf a power of two, is reduced exactly in
// integers.  The modes are split whatever the number of pairs, so that one pair
// fills the chip and its sums do not depend on the others; the eighths are added
// in LDS.  Bound by the matrix cores with many pairs, by the steps' latency with
// one.  Redshifts go 32 at a time, the rest with Y = 1 where it fits in 16: the
// matrix work is for whole blocks of 16.  Whole calls for 48 pairs of 4601
// velocities, 8000 to 20000 modes, with the copy out: 29 redshifts 28.3 -> 9.5
// ms, 9 redshifts 8.5 -> 3.0, 2 redshifts 2.38 -> 2.24; one pair of 1601, 9
// redshifts 187 -> 84 us (one thread per velocity and redshift before).  With
// 64 velocities a workgroup one pair at 29 redshifts takes 390 us, not 259, and
// 48 pairs 2 to 5 % less up to 16 redshifts; with 16, 48 pairs take 9 to 20 %
// more.  Partial tables in memory, 32 columns whatever N_Z, took 12.0, 4.8 and
// 3.3 ms and 233 us, and eight times the tables' memory.
constexpr int SIG_PARTS = 8, SIG_SEED = 256, SIG_X = 2;   // SIG_X: 16-velocity blocks of a workgroup
typedef double sd4 __attribute__((ext_vector_type(4)));
template <int Y>
__global__ __launch_bounds__(64 * SIG_PARTS, 4) void k_signal_sum(
    const int *mend, const double *__restrict__ w2, const double *__restrict__ pk, int nhalf, int mpad, int nzp,
    int nv, int nz, int z0, double inv_len, double *out) {
    constexpr int X = SIG_X, E = 4 * X * Y;   // accumulator elements of a lane
    __shared__ double red[SIG_PARTS / 2][E][64];
    const int p = blockIdx.z, zb = z0 + 16 * Y * blockIdx.y, v0 = blockIdx.x * 16 * X;
    const int tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    const int s = __builtin_amdgcn_readfirstlane(tid / 64);
    const int modes = mend[p] + 1;
    const int len = ((modes + SIG_PARTS - 1) / SIG_PARTS + 31) / 32 * 32;   // modes of a range
    const int m0 = s * len, m1 = min(m0 + len, (modes + 31) / 32 * 32);
    const unsigned mask = nhalf - 1;
    const double unit = 2.0 / nhalf;
    const double *w = w2 + (size_t)p * mpad, *pz = pk + zb + lr;
    unsigned iv[X];
    double rc[X], rs[X], cc[X], ss[X];
#pragma unroll
    for (int x = 0; x < X; ++x) {
        iv[x] = v0 + 16 * x + lr;
        sincospi(unit * ((4u * iv[x]) & mask), &rs[x], &rc[x]);   // the rotation by four modes
        cc[x] = ss[x] = 0.0;
    }
    sd4 acc[X][Y];
#pragma unroll
    for (int x = 0; x < X; ++x)
#pragma unroll
        for (int y = 0; y < Y; ++y) acc[x][y] = sd4{0.0, 0.0, 0.0, 0.0};
    for (int m = m0; m < m1; m += 32) {
        if ((m - m0) % SIG_SEED == 0) {
#pragma unroll
            for (int x = 0; x < X; ++x) sincospi(unit * (((unsigned)(m + lq) * iv[x]) & mask), &ss[x], &cc[x]);
        }
        double b[8][Y];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int mm = m + 4 * t + lq;
            const double wm = w[mm];
#pragma unroll
            for (int y = 0; y < Y; ++y) {
                // a mode that is left out adds nothing, also where its power overflowed
                const double pw = pz[(size_t)mm * nzp + 16 * y];
                b[t][y] = wm == 0.0 ? 0.0 : wm * pw;
            }
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int x = 0; x < X; ++x) {
#pragma unroll
                for (int y = 0; y < Y; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(cc[x], b[t][y], acc[x][y], 0, 0, 0);
                const double c = cc[x] * rc[x] - ss[x] * rs[x];
                ss[x] = ss[x] * rc[x] + cc[x] * rs[x];
                cc[x] = c;
            }
    }
    // the eighths in pairs: 4 + 4, 2 + 2, then the last two as they are written out
#pragma unroll
    for (int h = SIG_PARTS / 2; h >= 1; h /= 2) {
        if (s >= h && s < 2 * h) {
#pragma unroll
            for (int e = 0; e < E; ++e) red[s - h][e][lane] = acc[e / (4 * Y)][e / 4 % Y][e % 4];
        }
        __syncthreads();
        if (s < h) {
#pragma unroll
            for (int e = 0; e < E; ++e) acc[e / (4 * Y)][e / 4 % Y][e % 4] += red[s][e][lane];
        }
        __syncthreads();
    }
    if (s == 0) {
#pragma unroll
        for (int e = 0; e < E; ++e) red[0][e][lane] = acc[e / (4 * Y)][e / 4 % Y][e % 4];
    }
    __syncthreads();
    // element e = (x Y + y) 4 + u of a lane: velocity 16 x + 4 u + lane / 16, redshift 16 y + lane % 16
    for (int o = tid; o < 64 * E; o += 64 * SIG_PARTS) {
        const int iz = o % (16 * Y), i = o / (16 * Y), e = (i / 16 * Y + iz / 16) * 4 + i % 16 / 4;
        if (v0 + i < nv && zb + iz < nz)
            out[((size_t)p * nv + v0 + i) * nz + zb + iz] = inv_len * red[0][e][i % 4 * 16 + iz % 16];
    }
}

}  // namespace

void launch_deriv_tables(hipStream_t st, const double *pairs, int npairs, const double *kedges, int nk, int nv,
                         double dxv, int M, double *out) {
    if (npairs <= 0 || nk <= 0 || nv <= 0) return;
    dim3 grid((nv + 255) / 256, nk, npairs);
    k_deriv_table<<<grid, 256, 0, st>>>(pairs, kedges, nk, nv, dxv, M, out);
}

SignalGrid signal_grid(int nhalf, int nz) {
    SignalGrid g;
    g.nhalf = nhalf;
    g.mpad = (nhalf + 1 + 31) / 32 * 32;
    g.nzp = (nz + 15) / 16 * 16;
    return g;
}

void launch_pfid_grid(hipStream_t st, const SignalGrid &g, double dk, double z1, double dz, int nz, PD13 pd,
                      double *pk) {
    k_pfid_grid<<<dim3((g.mpad + 7) / 8, (g.nzp + 31) / 32), 256, 0, st>>>(dk, g.nhalf + 1, g.mpad, z1, dz, nz, g.nzp, pd, pk);
}

void launch_signal_tables(hipStream_t st, const SignalGrid &g, const double *pairs, const int *mend, int npairs,
                          const double *pk, double dk, double inv_len, int nv, int nz, double *w2, double *out) {
    if (npairs <= 0 || nv <= 0 || nz <= 0) return;
    k_signal_window<<<dim3((g.mpad + 255) / 256, npairs), 256, 0, st>>>(pairs, mend, g.nhalf, g.mpad, dk, w2);
    const int wide = g.nzp / 32, gx = (nv + 16 * SIG_X - 1) / (16 * SIG_X);
    if (wide > 0)
        k_signal_sum<2><<<dim3(gx, wide, npairs), 64 * SIG_PARTS, 0, st>>>(mend, w2, pk, g.nhalf, g.mpad, g.nzp, nv, nz, 0,
                                                                          inv_len, out);
    if (g.nzp % 32)
        k_signal_sum<1><<<dim3(gx, 1, npairs), 64 * SIG_PARTS, 0, st>>>(mend, w2, pk, g.nhalf, g.mpad, g.nzp, nv, nz,
                                                                       32 * wide, inv_len, out);
}

}  // namespace qml
