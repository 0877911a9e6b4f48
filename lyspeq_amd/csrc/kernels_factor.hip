// Batched blocked Cholesky factorisation A = L L^T and triangular inverse
// Li = L^-1 of every chunk of a batch (gfx950, FP64).
//
// Right-looking with 64x64 blocks (Np is a multiple of 64).  The L slot of
// the matrix arena starts as a copy of A's lower blocks and is factorised in
// place.  Block
// column p takes three launches over the whole batch:
//   diag   : one workgroup per chunk factors the updated block (p,p) and
//            inverts it (Li[p,p] = L[p,p]^-1);
//   panel  : TRSM tiles L[i,p] = A[i,p] Li[p,p]^T for i > p, and the tiles of
//            block row p of the inverse, Li[p,j] = -Li[p,p] sum_{k=j}^{p-1}
//            L[p,k] Li[k,j] for j < p (rows k < p of Li are final by then);
//   update : trailing tiles A[i,j] -= L[i,p] L[j,p]^T for p < j <= i.
// The 64x64 tile products run on v_mfma_f64_16x16x4f64, four waves per
// workgroup, each owning a 32x32 quarter.  The panel and update kernels
// stage their operands in K slabs of 16 (17 KB of LDS, at most 128 VGPRs),
// so that they fit on a CU beside the whitening products of the other
// stream (two workgroups of 64 KB) instead of waiting for one to drain; the
// MFMAs still run over k in the same order, so the results are the same.  A non-positive pivot marks the
// chunk failed (status) and is replaced by 1, as in the reference's LAPACK
// error path the chunk's results are then discarded.
#include "qml_common.hpp"
#include "qml_kernels.hpp"

namespace qml {

typedef double fd4 __attribute__((ext_vector_type(4)));
constexpr int FB = 64, FLD = FB + 1;   // block size, LDS row pitch (doubles)

// Element (r, c) of the 64x64 tile held in acc by this lane: for u = 0..3,
// r = 32 wm + 16 x + 4 u + lane/16, c = 32 wn + 16 y + lane%16.
template <class F>
__device__ __forceinline__ void tile_each(const fd4 (&acc)[2][2], F f) {
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int wm = w / 2, wn = w % 2;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                f(wm * 32 + x * 16 + 4 * u + lane / 16, wn * 32 + y * 16 + lane % 16, acc[x][y][u]);
}

__device__ __forceinline__ void tile_zero(fd4 (&acc)[2][2]) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = fd4{0.0, 0.0, 0.0, 0.0};
}

// A 64x64 block in registers: thread t holds the column pairs 2 (e % 32)
// of rows e / 32, e = t + 256 q (16-byte global loads through a
// global-space pointer, so that they count in vmcnt only).
struct BlockRegs {
    dvec2 v[FB * FB / 512];
};
__device__ __forceinline__ void fetch_block(BlockRegs &R, const double *M, int Np, int r0, int c0) {
#pragma unroll
    for (int q = 0; q < FB * FB / 512; ++q) {
        const int e = threadIdx.x + 256 * q, r = e / 32, c2 = 2 * (e % 32);
        R.v[q] = *(GlobalD2 *)(M + (size_t)(r0 + r) * Np + c0 + c2);
    }
}
// s[r * FLD + c] = block(r, c), or s[c * FLD + r] transposed
__device__ __forceinline__ void put_block(double *s, const BlockRegs &R, bool transpose) {
#pragma unroll
    for (int q = 0; q < FB * FB / 512; ++q) {
        const int e = threadIdx.x + 256 * q, r = e / 32, c2 = 2 * (e % 32);
        if (transpose) {
            s[c2 * FLD + r] = R.v[q].x;
            s[(c2 + 1) * FLD + r] = R.v[q].y;
        } else {
            s[r * FLD + c2] = R.v[q].x;
            s[r * FLD + c2 + 1] = R.v[q].y;
        }
    }
}
// s[r * FLD + c] = M[(r0 + r) * Np + c0 + c] (or transposed) for a 64x64 block
__device__ __forceinline__ void load_block(double *s, const double *M, int Np, int r0, int c0, bool transpose) {
    BlockRegs R;
    fetch_block(R, M, Np, r0, c0);
    put_block(s, R, transpose);
}

// K slabs of 16: S[r * KLD + k] for r in [0, 64), k in [0, 16)
constexpr int KS = 16, KLD = KS + 1;

// acc += S_a S_b^T over one slab (k ascending, four MFMA steps)
__device__ __forceinline__ void tile_nt16(const double *sa, const double *sb, fd4 (&acc)[2][2]) {
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int wm = w / 2, wn = w % 2;
#pragma unroll
    for (int k = 0; k < KS; k += 4) {
        double a[2], b[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            a[q] = sa[(wm * 32 + q * 16 + lane % 16) * KLD + k + lane / 16];
            b[q] = sb[(wn * 32 + q * 16 + lane % 16) * KLD + k + lane / 16];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], b[y], acc[x][y], 0, 0, 0);
    }
}

// Slab s of a 64x64 block in registers: 64 rows x 16 columns (row slab,
// M[r0 + r][c0 + 16 s + k]) or 16 rows x 64 columns (column slab for a
// transposed operand, M[r0 + 16 s + k][c0 + c]); two 16-byte loads a thread.
struct SlabRegs {
    dvec2 v[2];
};
__device__ __forceinline__ void fetch_slab(SlabRegs &R, const double *M, int Np, int r0, int c0, int s, bool transpose) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = threadIdx.x + 256 * q;
        if (transpose) {
            const int k = e / 32, c2 = 2 * (e % 32);
            R.v[q] = *(GlobalD2 *)(M + (size_t)(r0 + KS * s + k) * Np + c0 + c2);
        } else {
            const int r = e / 8, k2 = 2 * (e % 8);
            R.v[q] = *(GlobalD2 *)(M + (size_t)(r0 + r) * Np + c0 + KS * s + k2);
        }
    }
}
__device__ __forceinline__ void put_slab(double *S, const SlabRegs &R, bool transpose) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = threadIdx.x + 256 * q;
        if (transpose) {
            const int k = e / 32, c2 = 2 * (e % 32);
            S[c2 * KLD + k] = R.v[q].x;
            S[(c2 + 1) * KLD + k] = R.v[q].y;
        } else {
            const int r = e / 8, k2 = 2 * (e % 8);
            S[r * KLD + k2] = R.v[q].x;
            S[r * KLD + k2 + 1] = R.v[q].y;
        }
    }
}

// acc += A B^T over the four slabs of 64x64 operand blocks A (rows ra0,
// columns ca0 of Ma) and B (rows rb0, columns cb0 of Mb, or the transpose
// of the block at (rb0, cb0) when tb); the next slab is loaded into
// registers while one is multiplied.
__device__ __forceinline__ void block_nt(double *sa, double *sb, const double *Ma, int ra0, int ca0, const double *Mb,
                                         int rb0, int cb0, bool tb, int Np, fd4 (&acc)[2][2]) {
    SlabRegs ra, rb;
    fetch_slab(ra, Ma, Np, ra0, ca0, 0, false);
    fetch_slab(rb, Mb, Np, rb0, cb0, 0, tb);
#pragma unroll 1
    for (int s = 0; s < FB / KS; ++s) {
        put_slab(sa, ra, false);
        put_slab(sb, rb, tb);
        __syncthreads();
        if (s + 1 < FB / KS) {
            fetch_slab(ra, Ma, Np, ra0, ca0, s + 1, false);
            fetch_slab(rb, Mb, Np, rb0, cb0, s + 1, tb);
        }
        tile_nt16(sa, sb, acc);
        __syncthreads();
    }
}

// The L slot starts as the lower block triangle of A (its blocks above the
// diagonal are never read) and the Li slot with zeros above its diagonal
// blocks, which the split products' conversion reads.
__global__ __launch_bounds__(256) void k_chol_init(const ChunkDev *cs, double *mat) {
    const ChunkDev c = cs[blockIdx.y];
    const int Np = c.Np, h = Np / 2;
    const size_t n = (size_t)Np * Np;
    const dvec2 *A = (const dvec2 *)(mat + c.mat_off);
    dvec2 *L = (dvec2 *)(mat + c.mat_off + n), *Li = (dvec2 *)(mat + c.mat_off + 2 * n);
    const size_t total = n / 2, step = (size_t)gridDim.x * 256;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total; e += step) {
        const int r = (int)(e / h), q = 2 * (int)(e % h);
        if (q / FB <= r / FB) L[e] = A[e];
        else Li[e] = dvec2{0.0, 0.0};
    }
}

__device__ __forceinline__ double lane_of(double x, int lane) {
    const long long u = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// x / s with rs ~ 1 / s: the quotient's residual folded back in once
__device__ __forceinline__ double quotient(double x, double s, double rs) {
    const double q = x * rs;
    return fma(fma(-q, s, x), rs, q);
}

// s = sqrt(d) and rs = 1 / s for d > 0: the hardware's reciprocal root and
// two Newton steps on it, then one on the root; out of the range where those
// neither overflow nor lose bits, sqrt and a division.
__device__ __forceinline__ void root_pair(double d, double &s, double &rs) {
    if (d > 1e-280 && d < 1e280) {
        double y = __builtin_amdgcn_rsq(d);
        y = fma(0.5 * y, fma(-d * y, y, 1.0), y);
        y = fma(0.5 * y, fma(-d * y, y, 1.0), y);
        s = d * y;
        s = fma(0.5 * y, fma(-s, s, d), s);
        rs = fma(y, fma(-s, y, 1.0), y);
    } else {
        s = sqrt(d);
        rs = 1.0 / s;
    }
}

// Factors the updated diagonal block, L[p,p], and inverts it, Li[p,p], in
// 16-column panels.  The 64 pivots are one dependent chain, so the kernel's
// time is that chain's latency: a panel is factored by one wave with a row
// per lane and the panel's 16 columns in registers, where a column costs a
// reciprocal root and register broadcasts instead of three barriers and two
// trips through LDS; the trailing 16 x 16 blocks are updated on the matrix
// cores, one block a wave.  The inverse takes the four 16 x 16 diagonal
// blocks by forward substitution, a wave each, then
// Li[i,j] = -Li[i,i] sum_k L[i,k] Li[k,j] by block subdiagonals.
// LDS: strictly below the diagonal L, from the diagonal up Li^T (33 KB).
// 25 us a launch at 1 to 128 chunks; column by column in LDS it took 141.
constexpr int PB = 16;   // panel width
__global__ __launch_bounds__(256) void k_chol_diag(const ChunkDev *cs, double *mat, int *status, int p) {
    const ChunkDev c = cs[blockIdx.x];
    const int Np = c.Np, tid = threadIdx.x, p0 = p * FB;
    if (p0 >= Np) return;
    double *L = mat + c.mat_off + (size_t)Np * Np;
    double *Li = mat + c.mat_off + 2 * (size_t)Np * Np;
    __shared__ double a[FB * FLD];
    __shared__ double sd[FB], sr[FB];   // L's diagonal and its reciprocals
    const int w = tid / 64, l = tid % 64, lr = l % 16, lq = l / 16;
    load_block(a, L, Np, p0, p0, false);
    __syncthreads();
    int fail = 0;
#pragma unroll 1
    for (int kb = 0; kb < FB; kb += PB) {
        if (w == 0) {
            const int row = kb + l;
            double x[PB];
#pragma unroll
            for (int j = 0; j < PB; ++j) x[j] = (row < FB) ? a[row * FLD + kb + j] : 0.0;
#pragma unroll
            for (int k = 0; k < PB; ++k) {
                const double d = lane_of(x[k], k);
                double s = 1.0, rs = 1.0;
                if (d > 0.0) root_pair(d, s, rs);
                else fail = 1;
                const double q = quotient(x[k], s, rs);
                if (l == k) { sd[row] = s; sr[row] = rs; }
                x[k] = (l > k) ? q : 0.0;
#pragma unroll
                for (int j = k + 1; j < PB; ++j) x[j] = fma(-x[k], lane_of(x[k], j), x[j]);
            }
            if (row < FB) {
#pragma unroll
                for (int j = 0; j < PB; ++j)
                    if (l > j) a[row * FLD + kb + j] = x[j];
            }
        }
        __syncthreads();
        // trailing blocks (i, j), kb/16 < j <= i < 4: A -= L[i,kb] L[j,kb]^T
        const int b0 = kb / PB + 1;
        int t = 0;
        for (int i = b0; i < FB / PB; ++i)
            for (int j = b0; j <= i; ++j, ++t) {
                if ((t & 3) != w) continue;
                fd4 acc;
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[u] = a[(PB * i + 4 * u + lq) * FLD + PB * j + lr];
#pragma unroll
                for (int k = 0; k < PB; k += 4)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[(PB * i + lr) * FLD + kb + k + lq],
                                                               a[(PB * j + lr) * FLD + kb + k + lq], acc, 0, 0, 0);
#pragma unroll
                for (int u = 0; u < 4; ++u) a[(PB * i + 4 * u + lq) * FLD + PB * j + lr] = acc[u];
            }
        __syncthreads();
    }
    for (int e = tid; e < FB * FB; e += 256) {
        const int i = e / FB, j = e % FB;
        L[(size_t)(p0 + i) * Np + p0 + j] = (j < i) ? a[i * FLD + j] : (j == i) ? sd[i] : 0.0;
    }
    __syncthreads();   // the upper part now takes Li^T
    // diagonal block w: lane lr solves column lr of its inverse
    if (l < PB) {
        double x[PB];
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            double s = (i == lr) ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < i; ++k) s = fma(-a[(PB * w + i) * FLD + PB * w + k], x[k], s);
            x[i] = (i >= lr) ? quotient(s, sd[PB * w + i], sr[PB * w + i]) : 0.0;
        }
#pragma unroll
        for (int i = 0; i < PB; ++i)
            if (i >= lr) a[(PB * w + lr) * FLD + PB * w + i] = x[i];
    }
    __syncthreads();
#pragma unroll 1
    for (int t = 1; t < FB / PB; ++t) {   // block subdiagonal t, block (i, i - t) by wave i - t
        const int j = w, i = w + t;
        if (i < FB / PB) {
            fd4 s = {0.0, 0.0, 0.0, 0.0}, x = {0.0, 0.0, 0.0, 0.0};
            for (int k = j; k < i; ++k)
#pragma unroll
                for (int q = 0; q < PB; q += 4) {
                    const int r = q + lq;   // Li[k,j](r, lr), zero above its diagonal
                    const double b = (k > j || r >= lr) ? a[(PB * j + lr) * FLD + PB * k + r] : 0.0;
                    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a[(PB * i + lr) * FLD + PB * k + r], b, s, 0, 0, 0);
                }
            // element u of s holds row 4 u + lane / 16: the B operand of step u
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = 4 * q + lq;
                const double v = (lr >= r) ? -a[(PB * i + r) * FLD + PB * i + lr] : 0.0;
                x = __builtin_amdgcn_mfma_f64_16x16x4f64(v, s[q], x, 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) a[(PB * j + lr) * FLD + PB * i + 4 * u + lq] = x[u];
        }
        __syncthreads();
    }
    for (int e = tid; e < FB * FB; e += 256) {
        const int i = e / FB, j = e % FB;
        Li[(size_t)(p0 + i) * Np + p0 + j] = (j <= i) ? a[j * FLD + i] : 0.0;
    }
    if (tid == 0) {   // wave 0 saw every pivot
        if (p == 0) status[c.gidx] = fail;
        else if (fail) status[c.gidx] = 1;
    }
}

__global__ __launch_bounds__(256, 4) void k_chol_panel(const ChunkDev *cs, double *mat, int p, int ntrsm) {
    const ChunkDev c = cs[blockIdx.y];
    const int Np = c.Np, nt = Np / FB, p0 = p * FB, bx = blockIdx.x;
    if (p >= nt) return;
    double *L = mat + c.mat_off + (size_t)Np * Np;
    double *Li = mat + c.mat_off + 2 * (size_t)Np * Np;
    __shared__ double sa[FB * KLD];
    __shared__ double sb[FB * KLD];
    fd4 acc[2][2];
    tile_zero(acc);
    if (bx < ntrsm) {
        // TRSM tile: L[i,p] = A[i,p] Li[p,p]^T
        const int i = p + 1 + bx;
        if (i >= nt) return;
        block_nt(sa, sb, L, i * FB, p0, Li, p0, p0, false, Np, acc);
        tile_each(acc, [&](int r, int q, double x) { L[(size_t)(i * FB + r) * Np + p0 + q] = x; });
        return;
    }
    // block row p of the inverse: T = sum_{k=j}^{p-1} L[p,k] Li[k,j]
    const int j = bx - ntrsm;
    if (j >= p) return;
#pragma unroll 1
    for (int k = j; k < p; ++k) block_nt(sa, sb, L, p0, k * FB, Li, k * FB, j * FB, true, Np, acc);
    // Li[p,j] = -Li[p,p] T: T^T as the B operand, slab s holding rows
    // [16 s, 16 s + 16) of T, which the waves of row half s / 2 hold in
    // acc[s % 2] (rows 32 wm + 16 x + 4 u + lane / 16)
    fd4 t[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) t[x][y] = acc[x][y];
    tile_zero(acc);
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64, wm = w / 2, wn = w % 2;
    SlabRegs ra;
    fetch_slab(ra, Li, Np, p0, p0, 0, false);
#pragma unroll 1
    for (int s = 0; s < FB / KS; ++s) {
        put_slab(sa, ra, false);
        if (wm == s / 2) {
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    sb[(wn * 32 + y * 16 + lane % 16) * KLD + 4 * u + lane / 16] = t[s % 2][y][u];
        }
        __syncthreads();
        if (s + 1 < FB / KS) fetch_slab(ra, Li, Np, p0, p0, s + 1, false);
        tile_nt16(sa, sb, acc);
        __syncthreads();
    }
    tile_each(acc, [&](int r, int q, double x) { Li[(size_t)(p0 + r) * Np + j * FB + q] = -x; });
}

__global__ __launch_bounds__(256, 4) void k_chol_update(const ChunkDev *cs, double *mat, int p) {
    const ChunkDev c = cs[blockIdx.y];
    const int Np = c.Np, nt = Np / FB, p0 = p * FB;
    const int m = nt - p - 1;                 // trailing block rows of this chunk
    int t = blockIdx.x;
    if (m <= 0 || t >= m * (m + 1) / 2) return;
    // t -> (i, j), p < j <= i < nt, row-major over the lower triangle
    int i = 0;
    while (t > i) { t -= i + 1; ++i; }
    const int bi = p + 1 + i, bj = p + 1 + t;
    double *L = mat + c.mat_off + (size_t)Np * Np;
    __shared__ double sa[FB * KLD];
    __shared__ double sb[FB * KLD];
    fd4 acc[2][2];
    tile_zero(acc);
    block_nt(sa, sb, L, bi * FB, p0, L, bj * FB, p0, false, Np, acc);
    tile_each(acc, [&](int r, int q, double x) { L[(size_t)(bi * FB + r) * Np + bj * FB + q] -= x; });
}

static void factor(const LaunchCtx &L, int *status, bool inverse) {
    const int ntmax = L.np_max / FB;
    for (int p = 0; p < ntmax; ++p) {
        const int m = ntmax - p - 1;
        k_chol_diag<<<L.nchunks, 256, 0, L.stream>>>(L.chunks, L.mat, status, p);
        // TRSM tiles (m of them), then the inverse's tiles j < p
        const int gx = m + (inverse ? p : 0);
        if (gx > 0) k_chol_panel<<<dim3(gx, L.nchunks), 256, 0, L.stream>>>(L.chunks, L.mat, p, m);
        if (m > 0) k_chol_update<<<dim3(m * (m + 1) / 2, L.nchunks), 256, 0, L.stream>>>(L.chunks, L.mat, p);
    }
}
void launch_cholesky(const LaunchCtx &L, int *status) {
    k_chol_init<<<dim3(64, L.nchunks), 256, 0, L.stream>>>(L.chunks, L.mat);
    factor(L, status, true);
}
void launch_cholesky_in_place(const LaunchCtx &L, int *status) { factor(L, status, false); }

// The inverse is formed inside the blocked factorisation.
void launch_trinv(const LaunchCtx &) {}

}  // namespace qml
