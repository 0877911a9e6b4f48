// The FP64 products of the QML engine (gfx950, v_mfma_f64_16x16x4f64).
//
// As the split products do, they write X_j = M + M^T (M the lower triangle of
// X_j with its diagonal halved, stored as T = M^T):
//   whiten_left :  P_j = Li M                (lower 64-tiles, J <= I, over k in
//                                             [64 J, 64 (I+1)))
//   whiten_right:  G_j = P_j Li^T + Li P_j^T (upper tiles, k < 64 (I+1))
//   gram        :  E_s = sum over G tile s of G_j G_j'
// which is N^3/2 multiply-adds a member; the dense form Y = Li X, G = Y Li^T on
// upper tiles took 5/6 N^3, with a stack and Y twice as large.  The matrix
// cores are the bound: a wave multiplies only the k where its operands are not
// exact zeros (Li and P are lower triangular, T is upper, and past the chunk's
// N pixels everything vanishes).
#include "qml_common.hpp"
#include "qml_kernels.hpp"

namespace qml {

typedef double gd4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int GK = 16, GLD = GK + 2;   // K of a stage, LDS row pitch (doubles)

__device__ __forceinline__ gd4 mma(double a, double b, gd4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int upper_index(int I, int J, int nt) { return I * nt - I * (I - 1) / 2 + (J - I); }

// consecutive work items stay on one XCD (blockIdx % 8), with its L2
__device__ __forceinline__ int xcd_item(int nwork) {
    const int per = (nwork + 7) / 8;
    return (blockIdx.x % 8) * per + blockIdx.x / 8;
}

}  // namespace

// One 64 x 64 tile per workgroup, a 32 x 32 quarter (2 x 2 blocks) per wave.
// Both operands are staged row by row with k contiguous; a lane reads two
// consecutive k as one 16-byte LDS load, and lanes l/16 = 0..3 hold k = 2 (l/16)
// and 2 (l/16) + 1 of each eight: A and B use the same order, so the sum runs
// over the same terms.  The pitch of 18 doubles puts any eight consecutive
// rows on distinct banks.  Two LDS stages (37 KB, four workgroups per CU), one
// barrier a stage, and two register sets, so that a load has two stages to
// arrive: with one, a memory latency was longer than a wave's 16 MFMAs.  The
// multiply is branch-free inside (a test per 16 x 16 block saved a tenth of the
// MFMAs but made the compiler copy the accumulators every stage).  The quarters
// rotate over the waves, so that the SIMDs share the corners' idle ones.
// Measured on 128 chunks of 150 to 700 pixels (13 300 members): left 39.5 ->
// 15.6 ms, right 29.0 -> 29.8 ms for twice the multiply-adds, matrix cores 66 %
// and 63 % busy (one register set: 60 %; a test per block: 53 %).
template <bool RIGHT>
__global__ __launch_bounds__(256, 4) void k_gemm64(const ChunkDev *cs, const Work *work, int nwork,
                                                   const double *Abase, const double *Bbase, double *Cbase, int jlo) {
    const int li = xcd_item(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    const int Np = c.Np, N = c.N, I0 = wk.I * TILE, J0 = wk.J * TILE;
    const size_t mem = (size_t)c.stk_off + (size_t)(wk.j - jlo) * Np * Np;
    // LEFT: A = Li, B = T; RIGHT: A = P, B = Li, then the two exchanged
    const double *A = Abase + (RIGHT ? mem : (size_t)c.lic_off), *B = Bbase + (RIGHT ? (size_t)c.lic_off : mem);
    __shared__ double sa[2][TILE * GLD], sb[2][TILE * GLD];
    const int tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    const int quarter = (__builtin_amdgcn_readfirstlane(tid / 64) + li) & 3;
    const int wm = quarter / 2, wn = quarter % 2;
    const int r0 = I0 + 32 * wm, c0 = J0 + 32 * wn;
    // on a diagonal tile P's upper quarter is zero (and never read), and G's
    // lower one is the upper one's mirror image
    const bool active = !(wk.I == wk.J && (RIGHT ? wm > wn : wm < wn));
    const int kbeg = RIGHT ? 0 : J0;
    const int kend = max(kbeg, min(I0 + TILE, (N + GK - 1) / GK * GK));
    const int ns = (kend - kbeg) / GK, total = RIGHT ? 2 * ns : ns;
    // the quarter multiplies k in [klo, khi), nothing where it lies past N
    const bool inside = active && r0 < N && c0 < N;
    const int klo = RIGHT ? 0 : c0, khi = inside ? r0 + 32 : 0;
    gd4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = gd4{0.0, 0.0, 0.0, 0.0};

    // thread t stages the 16 bytes t % 8 of rows t / 8 and t / 8 + 32
    const int gr = tid / 8, gk = 2 * (tid % 8);
    const size_t oa = (size_t)(I0 + gr) * Np + gk, ob = (size_t)(J0 + gr) * Np + gk, half = (size_t)32 * Np;
    struct Regs { dvec2 a[2], b[2]; } r0s, r1s;
    auto fetch = [&](int s, Regs &r) {
        const bool second = RIGHT && s >= ns;
        const double *x = second ? B : A, *y = second ? A : B;
        const int k = kbeg + (second ? s - ns : s) * GK;
        r.a[0] = *(GlobalD2 *)(x + oa + k);
        r.a[1] = *(GlobalD2 *)(x + oa + half + k);
        r.b[0] = *(GlobalD2 *)(y + ob + k);
        r.b[1] = *(GlobalD2 *)(y + ob + half + k);
        asm volatile("" ::: "memory");   // issued here, not where the values are first needed
    };
    auto put = [&](int buf, const Regs &r) {
        *(dvec2 *)(&sa[buf][gr * GLD + gk]) = r.a[0];
        *(dvec2 *)(&sa[buf][(gr + 32) * GLD + gk]) = r.a[1];
        *(dvec2 *)(&sb[buf][gr * GLD + gk]) = r.b[0];
        *(dvec2 *)(&sb[buf][(gr + 32) * GLD + gk]) = r.b[1];
    };
    auto multiply = [&](int s) {
        const int buf = s & 1, k = kbeg + ((RIGHT && s >= ns) ? s - ns : s) * GK;
        if (k < klo || k >= khi) return;
        dvec2 a[2][2], b[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                a[x][h] = *(const dvec2 *)(&sa[buf][(32 * wm + 16 * x + lr) * GLD + 8 * h + 2 * lq]);
                b[x][h] = *(const dvec2 *)(&sb[buf][(32 * wn + 16 * x + lr) * GLD + 8 * h + 2 * lq]);
            }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = mma(a[x][h].x, b[y][h].x, acc[x][y]);
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = mma(a[x][h].y, b[y][h].y, acc[x][y]);
        }
    };
    if (total > 0) {
        // stage s + 2 is loaded while s is multiplied and s + 1 waits in the
        // other register set; loads past the sweep repeat its last stage
        fetch(0, r0s);
        fetch(min(1, total - 1), r1s);
        put(0, r0s);
        __syncthreads();
        for (int s = 0; s < total; s += 2) {
            fetch(min(s + 2, total - 1), r0s);
            multiply(s);
            put(1, r1s);
            __syncthreads();
            if (s + 1 >= total) break;
            fetch(min(s + 3, total - 1), r1s);
            multiply(s + 1);
            put(0, r0s);
            __syncthreads();
        }
    }
    if (!active) return;
    // element u of a block: row 4 u + lane / 16, column lane % 16
    if (!RIGHT) {
        double *C = Cbase + mem;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    C[(size_t)(r0 + 16 * x + 4 * u + lq) * Np + c0 + 16 * y + lr] = acc[x][y][u];
    } else {
        double *C = Cbase + c.g_off + ((size_t)wk.j * c.ntu + upper_index(wk.I, wk.J, c.nt)) * TILE * TILE;
        const bool mirror = wk.I == wk.J && wm != wn;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = 32 * wm + 16 * x + 4 * u + lq, q = 32 * wn + 16 * y + lr;
                    C[r * TILE + q] = acc[x][y][u];
                    if (mirror) C[q * TILE + r] = acc[x][y][u];
                }
    }
}

// E over one G tile for members [64 I, 64 I + 64) x [64 J, 64 J + 64): the
// tile's 4096 terms are split over the workgroup's eight waves, and each wave
// holds the 16 x 16 blocks of the pair that lie inside the m members (on I = J
// the upper ones only) in registers, 10 or 16 at most.  No LDS in the loop: a
// lane loads 16 consecutive bytes of its member's row, so that four lanes
// cover 64 and the k order is the products' above; the next step's loads are in
// flight while this one is multiplied (32 terms a step where I = J, whose steps
// are short, 8 else).  The partial sums of the waves meet in LDS, block by
// block.  (64 x 64 tiles of padded members took 537 us for 64 chunks with
// m = 21, this 134 us; the survey sample with m up to 175 took 8.9 ms, now 5.8.)
constexpr int GW = 8;   // waves
__global__ __launch_bounds__(64 * GW, 2) void k_gram64(const ChunkDev *cs, const Work *work, int nwork, const double *G,
                                                    double *gram) {
    const int li = xcd_item(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    constexpr int KW = TILE * TILE / GW;   // terms per wave
    __shared__ double red[2][GW][256];
    const int tid = threadIdx.x, lane = tid % 64, lr = lane % 16, lq = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64);
    const int nb = (c.m + 15) / 16, na = min(4, nb - 4 * wk.I), nc = min(4, nb - 4 * wk.J);
    const size_t ktot = (size_t)c.ntu * TILE * TILE;
    const double *base = G + c.g_off + (size_t)wk.j * TILE * TILE + w * KW + 2 * lq;
    const double *pa[4], *pc[4];   // rows past the last member repeat it; their sums are not used
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        pa[x] = base + (size_t)min(64 * wk.I + 16 * x + lr, c.m - 1) * ktot;
        pc[x] = base + (size_t)min(64 * wk.J + 16 * x + lr, c.m - 1) * ktot;
    }
    const int ntile = c.mt * (c.mt + 1) / 2;
    int s = wk.j, I = 0;   // the G tile's row and column: off the diagonal it counts twice
    while (s >= c.nt - I) { s -= c.nt - I; ++I; }
    const double wgt = s == 0 ? 1.0 : 2.0;
    double *C = gram + c.gram_off + ((size_t)wk.j * ntile + upper_index(wk.I, wk.J, c.mt)) * TILE * TILE;
    int flip = 0;
    auto reduce = [&](const gd4 &v, int x, int y) {
        double (*r)[256] = red[flip];
#pragma unroll
        for (int u = 0; u < 4; ++u) r[w][64 * u + lane] = v[u];
        __syncthreads();
        if (tid < 256) {
            double t = r[0][tid];
#pragma unroll
            for (int q = 1; q < GW; ++q) t += r[q][tid];
            C[(16 * x + tid / 16) * TILE + 16 * y + tid % 16] = wgt * t;
        }
        flip ^= 1;
    };
    gd4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = gd4{0.0, 0.0, 0.0, 0.0};
    if (wk.I == wk.J) {
        constexpr int U = 4, ST = 8 * U;
        dvec2 f[2][4][U];
        auto fetch = [&](int b, int k) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (x < na)
#pragma unroll
                    for (int t = 0; t < U; ++t) f[b][x][t] = *(GlobalD2 *)(pa[x] + k + 8 * t);
        };
        auto step = [&](int b) {
#pragma unroll
            for (int t = 0; t < U; ++t)
#pragma unroll
                for (int y = 0; y < 4; ++y)
                    if (y < na) {
#pragma unroll
                        for (int x = 0; x <= y; ++x) acc[x][y] = mma(f[b][x][t].x, f[b][y][t].x, acc[x][y]);
#pragma unroll
                        for (int x = 0; x <= y; ++x) acc[x][y] = mma(f[b][x][t].y, f[b][y][t].y, acc[x][y]);
                    }
        };
        fetch(0, 0);
#pragma unroll 1
        for (int k = 0; k < KW; k += 2 * ST) {
            fetch(1, k + ST);
            step(0);
            if (k + 2 * ST < KW) fetch(0, k + 2 * ST);
            step(1);
        }
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x <= y; ++x)
                if (y < na) reduce(acc[x][y], x, y);
    } else {
        constexpr int ST = 8;
        dvec2 fa[2][4], fc[2][4];
        auto fetch = [&](int b, int k) {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                fa[b][x] = *(GlobalD2 *)(pa[x] + k);   // all four blocks of I lie inside when I < J
                if (x < nc) fc[b][x] = *(GlobalD2 *)(pc[x] + k);
            }
        };
        auto step = [&](int b) {
#pragma unroll
            for (int y = 0; y < 4; ++y)
                if (y < nc) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[x][y] = mma(fa[b][x].x, fc[b][y].x, acc[x][y]);
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[x][y] = mma(fa[b][x].y, fc[b][y].y, acc[x][y]);
                }
        };
        fetch(0, 0);
#pragma unroll 1
        for (int k = 0; k < KW; k += 2 * ST) {
            fetch(1, k + ST);
            step(0);
            if (k + 2 * ST < KW) fetch(0, k + 2 * ST);
            step(1);
        }
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (y < nc) reduce(acc[x][y], x, y);
    }
}

void launch_gemm64_left(hipStream_t st, const ChunkDev *chunks, const Work *work, int nwork, const double *li,
                        const double *X, double *Y, int jlo) {
    k_gemm64<false><<<8 * ((nwork + 7) / 8), 256, 0, st>>>(chunks, work, nwork, li, X, Y, jlo);
}
void launch_gemm64_right(hipStream_t st, const ChunkDev *chunks, const Work *work, int nwork, const double *li,
                         const double *Y, double *G, int jlo) {
    k_gemm64<true><<<8 * ((nwork + 7) / 8), 256, 0, st>>>(chunks, work, nwork, Y, li, G, jlo);
}
void launch_gram64(hipStream_t st, const ChunkDev *chunks, const Work *work, int nwork, const double *G,
                   double *gram) {
    k_gram64<<<8 * ((nwork + 7) / 8), 64 * GW, 0, st>>>(chunks, work, nwork, G, gram);
}

}  // namespace qml
