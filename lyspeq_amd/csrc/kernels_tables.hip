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

// part[s][p][iv][iz] = the sum over range s of pair p's modes of
// cos(k_m v_iv) w2(m) pk(m, iz).  A wave takes 64 velocities and 32 redshifts,
// four modes a step on v_mfma_f64_16x16x4f64: lane l's A values are the cosines
// of its four velocities at mode l / 16 of the step, advanced by rotation by
// four modes and re-seeded every 256 modes; its B values the weighted power at
// that mode.  A cosine thus serves 32 redshifts and a loaded power 64
// velocities; one thread per velocity and redshift advanced the same cosine for
// each redshift (26.4 ms for 48 pairs at 4601 x 29 and 8000 to 20000 modes,
// 3.8 ms here).  The phase k_m v_iv = 2 pi m iv / nhalf, nhalf a power of two, is
// reduced exactly in integers.  The modes are cut into SIG_PARTS ranges whatever
// the number of pairs, so that one pair fills the chip and its sums do not
// depend on the others.
constexpr int SIG_PARTS = 8, SIG_SEED = 256;
typedef double sd4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256, 2) void k_signal_sum(const int *mend, const double *__restrict__ w2,
                                                       const double *__restrict__ pk, int nhalf, int mpad, int nzp,
                                                       int nv, int nz, double *part) {
    const int p = blockIdx.z, s = blockIdx.y % SIG_PARTS, zb = 32 * (blockIdx.y / SIG_PARTS);
    const int lane = threadIdx.x % 64, lr = lane % 16, lq = lane / 16;
    const int v0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / 64)) * 64;
    if (v0 >= nv) return;
    const int modes = mend[p] + 1;
    const int len = ((modes + SIG_PARTS - 1) / SIG_PARTS + 31) / 32 * 32;   // modes of a range
    const int m0 = s * len, m1 = min(m0 + len, (modes + 31) / 32 * 32);
    const unsigned mask = nhalf - 1;
    const double unit = 2.0 / nhalf;
    const double *w = w2 + (size_t)p * mpad, *pz = pk + zb + lr;
    unsigned iv[4];
    double rc[4], rs[4], cc[4], ss[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        iv[x] = v0 + 16 * x + lr;
        sincospi(unit * ((4u * iv[x]) & mask), &rs[x], &rc[x]);   // the rotation by four modes
        cc[x] = ss[x] = 0.0;
    }
    sd4 acc[4][2];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = sd4{0.0, 0.0, 0.0, 0.0};
    for (int m = m0; m < m1; m += 32) {
        if ((m - m0) % SIG_SEED == 0) {
#pragma unroll
            for (int x = 0; x < 4; ++x) sincospi(unit * (((unsigned)(m + lq) * iv[x]) & mask), &ss[x], &cc[x]);
        }
        double b[8][2];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int mm = m + 4 * t + lq;
            const double wm = w[mm];
            // a mode that is left out adds nothing, also where its power overflowed
            b[t][0] = wm == 0.0 ? 0.0 : wm * pz[(size_t)mm * nzp];
            b[t][1] = wm == 0.0 ? 0.0 : wm * pz[(size_t)mm * nzp + 16];
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(cc[x], b[t][y], acc[x][y], 0, 0, 0);
                const double c = cc[x] * rc[x] - ss[x] * rs[x];
                ss[x] = ss[x] * rc[x] + cc[x] * rs[x];
                cc[x] = c;
            }
    }
    double *o = part + ((size_t)s * gridDim.z + p) * nv * nz;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = v0 + 16 * x + 4 * u + lq, iz = zb + 16 * y + lr;
                if (i < nv && iz < nz) o[(size_t)i * nz + iz] = acc[x][y][u];
            }
}

// out (npairs x nv x nz, z contiguous) = the ranges' sums times inv_len
__global__ __launch_bounds__(256) void k_signal_table(const double *part, size_t total, double inv_len, double *out) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < SIG_PARTS; ++k) s += part[(size_t)k * total + e];
    out[e] = s * inv_len;
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
    g.nzp = (nz + 31) / 32 * 32;
    g.parts = SIG_PARTS;
    return g;
}

void launch_pfid_grid(hipStream_t st, const SignalGrid &g, double dk, double z1, double dz, int nz, PD13 pd,
                      double *pk) {
    k_pfid_grid<<<dim3((g.mpad + 7) / 8, (g.nzp + 31) / 32), 256, 0, st>>>(dk, g.nhalf + 1, g.mpad, z1, dz, nz, g.nzp, pd, pk);
}

void launch_signal_tables(hipStream_t st, const SignalGrid &g, const double *pairs, const int *mend, int npairs,
                          const double *pk, double dk, double inv_len, int nv, int nz, double *w2, double *part,
                          double *out) {
    if (npairs <= 0 || nv <= 0 || nz <= 0) return;
    k_signal_window<<<dim3((g.mpad + 255) / 256, npairs), 256, 0, st>>>(pairs, mend, g.nhalf, g.mpad, dk, w2);
    k_signal_sum<<<dim3((nv + 255) / 256, SIG_PARTS * (g.nzp / 32), npairs), 256, 0, st>>>(mend, w2, pk, g.nhalf, g.mpad,
                                                                                          g.nzp, nv, nz, part);
    const size_t total = (size_t)npairs * nv * nz;
    k_signal_table<<<(total + 255) / 256, 256, 0, st>>>(part, total, inv_len, out);
}

}  // namespace qml
