// Dense MFMA products of the QML engine in FP32 and split BF16 (gfx950); the
// FP64 ones are in kernels_gemm64.hip.
//
//   whiten_left :  Y_j = Li X_j              (Li lower triangular: K-range of
//                                             tile row I is [0, 64 (I+1)); X_j is
//                                             symmetric and read row-wise as B^T)
//   whiten_right:  G_j = Y_j Li^T            (upper tiles only, K-range
//                                             [0, 64 (J+1)), tile-packed out)
// The split-BF16x3 products instead write X_j = M + M^T (M the lower
// triangle of X_j with its diagonal halved, stored as T = M^T):
//   whiten_left :  P_j = Li M                (lower 128-tiles, K-range of tile
//                                             (I, J) is [128 J, 128 (I+1)))
//   whiten_right:  G_j = P_j Li^T + Li P_j^T (upper tiles, K-range [0, 128 (I+1)))
//   gram        :  E_s = sum_{k in G tile s} G_j[k] G_j'[k]   (split-K partials,
//                                             x2 for off-diagonal G tiles)
//
// FP32 (k_gemm): one 256-thread workgroup computes a 64x64 output tile; each
// of its four waves owns a 32x32 quarter made of 2x2 16x16 MFMA blocks on
// v_mfma_f32_16x16x4f32, FP32 operands and accumulation.
// Split BF16 (k_gemm_bf3): 128x128 output tiles on operands stored as two
// bf16 planes (hi, lo), v_mfma_f32_16x16x32_bf16 with FP32 accumulation:
//   BF16x3 a b ~ a_hi b_hi + a_hi b_lo + a_lo b_hi;
//   BF16x4 the same with a_lo b_lo added first (four MFMAs per block).
// The work list holds (chunk, member or split, I, J) per workgroup; work is
// assigned so that consecutive items stay on one XCD (blockIdx % 8 selects
// the XCD), keeping a chunk's operands in that XCD's L2.
#include "qml_common.hpp"
#include "qml_kernels.hpp"

#include <type_traits>

namespace qml {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

enum { MODE_LEFT = 0, MODE_RIGHT = 1, MODE_GRAM = 2 };

__device__ __forceinline__ int upper_tile_index(int I, int J, int nt) {
    return I * nt - I * (I - 1) / 2 + (J - I);
}

__device__ __forceinline__ bool packed_tile_is_diag(int s, int nt) {
    int I = 0;
    while (s >= nt - I) { s -= nt - I; ++I; }
    return s == 0;
}

__device__ __forceinline__ int xcd_logical(int nwork) {
    const int per = (nwork + 7) / 8;
    return (blockIdx.x % 8) * per + blockIdx.x / 8;
}

// Problem description of one work item.
struct Prob {
    const float *A;  // row-major, rows of the output tile, K contiguous (lda)
    const float *B;  // row-major N x K (ldb)
    int lda, ldb;
    int kbeg, kend;
    int arows, brows;   // valid rows of A / B^T (members for the Gram); others read as 0
};

// --------------------------------------------------------------- FP32 path --
__device__ __forceinline__ void mainloop_k4(const Prob &p, int I0, int J0, f4 (&acc)[2][2]) {
    constexpr int KB = 16, PAD = 4;
    __shared__ float As[KB][64 + PAD];
    __shared__ float Bs[KB][64 + PAD];
    const int tid = threadIdx.x, lane = tid % 64, w = tid / 64;
    const int wm = w / 2, wn = w % 2;
    // row tid/4, four consecutive k at (tid%4)*4
    const int ar = tid / 4, ak = (tid % 4) * 4;
    float ra[4], rb[4];
    auto gload = [&](int k0) {
        const bool aok = (I0 + ar) < p.arows, bok = (J0 + ar) < p.brows;
        const float *pa = p.A + (size_t)(I0 + ar) * p.lda + k0 + ak;
        const float *pb = p.B + (size_t)(J0 + ar) * p.ldb + k0 + ak;
#pragma unroll
        for (int u = 0; u < 4; ++u) ra[u] = aok ? pa[u] : 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) rb[u] = bok ? pb[u] : 0.0f;
    };
    auto sstore = [&]() {
#pragma unroll
        for (int u = 0; u < 4; ++u) As[ak + u][ar] = ra[u];
#pragma unroll
        for (int u = 0; u < 4; ++u) Bs[ak + u][ar] = rb[u];
    };
    if (p.kbeg >= p.kend) return;
    gload(p.kbeg);
    sstore();
    __syncthreads();
    for (int k0 = p.kbeg; k0 < p.kend; k0 += KB) {
        const bool more = k0 + KB < p.kend;
        if (more) gload(k0 + KB);
#pragma unroll
        for (int kk = 0; kk < KB; kk += 4) {
            float a[2], b[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                a[q] = As[kk + lane / 16][wm * 32 + q * 16 + lane % 16];
                b[q] = Bs[kk + lane / 16][wn * 32 + q * 16 + lane % 16];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], b[y], acc[x][y], 0, 0, 0);
        }
        __syncthreads();
        if (more) sstore();
        __syncthreads();
    }
}

// ------------------------------------------------------------------ kernel --
template <int MODE>
__global__ __launch_bounds__(256) void k_gemm(const ChunkDev *cs, const Work *work, int nwork,
                                              const void *Abase, const void *Bbase, void *Cbase, int jlo) {
    using T = float;
    const int li = xcd_logical(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    const int Np = c.Np;
    const size_t msz = (size_t)Np * Np;
    Prob p;
    int I0, J0;
    if (MODE == MODE_LEFT) {
        p.A = (const T *)Abase + c.lic_off;
        // X_j is symmetric, so its rows serve as the K-contiguous rows of B^T
        p.B = (const T *)Bbase + c.stk_off + (wk.j - jlo) * msz;
        p.lda = p.ldb = Np;
        p.kbeg = 0;
        p.kend = (wk.I + 1) * TILE;
        p.arows = p.brows = Np;
        I0 = wk.I * TILE;
        J0 = wk.J * TILE;
    } else if (MODE == MODE_RIGHT) {
        p.A = (const T *)Abase + c.stk_off + (wk.j - jlo) * msz;
        p.B = (const T *)Bbase + c.lic_off;
        p.lda = p.ldb = Np;
        p.kbeg = 0;
        p.kend = (wk.J + 1) * TILE;
        p.arows = p.brows = Np;
        I0 = wk.I * TILE;
        J0 = wk.J * TILE;
    } else {
        const int ktot = c.ntu * TILE * TILE;
        p.A = (const T *)Abase + c.g_off;
        p.B = p.A;
        p.lda = p.ldb = ktot;
        p.kbeg = wk.j * TILE * TILE;
        p.kend = p.kbeg + TILE * TILE;
        p.arows = p.brows = c.m;
        I0 = wk.I * TILE;
        J0 = wk.J * TILE;
    }
    f4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[x][y][u] = 0;
    mainloop_k4(p, I0, J0, acc);

    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int wm = w / 2, wn = w % 2;
    // row of accumulator element u inside a 16x16 block
    auto brow = [&](int u) { return 4 * (lane / 16) + u; };
    if (MODE == MODE_LEFT) {
        T *C = (T *)Cbase + c.stk_off + (wk.j - jlo) * msz;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = I0 + wm * 32 + x * 16 + brow(u);
                    const int q = J0 + wn * 32 + y * 16 + lane % 16;
                    C[(size_t)r * Np + q] = (T)acc[x][y][u];
                }
    } else if (MODE == MODE_RIGHT) {
        T *C = (T *)Cbase + c.g_off + (size_t)wk.j * c.ntu * TILE * TILE
             + (size_t)upper_tile_index(wk.I, wk.J, c.nt) * TILE * TILE;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = wm * 32 + x * 16 + brow(u);
                    const int q = wn * 32 + y * 16 + lane % 16;
                    C[r * TILE + q] = (T)acc[x][y][u];
                }
    } else {
        const int ntile = c.mt * (c.mt + 1) / 2;
        const double wgt = packed_tile_is_diag(wk.j, c.nt) ? 1.0 : 2.0;
        double *C = (double *)Cbase + c.gram_off
                  + ((size_t)wk.j * ntile + upper_tile_index(wk.I, wk.J, c.mt)) * TILE * TILE;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int r = wm * 32 + x * 16 + brow(u);
                    const int q = wn * 32 + y * 16 + lane % 16;
                    C[r * TILE + q] = wgt * (double)acc[x][y][u];
                }
    }
}

// offdiag: whether Gram items lie off the diagonal (more than 128 members)
void launch_bf3(hipStream_t st, int mode, int nprod, int nst, const ChunkDev *chunks, const Work *work, int nwork,
                const void *A, const void *B, void *C, int jlo, bool offdiag);

template <int MODE>
static void launch_mode(hipStream_t st, int prec, int nst, const ChunkDev *chunks, const Work *work, int nwork,
                        const void *A, const void *B, void *C, int jlo, bool offdiag = false) {
    if (nwork <= 0) return;
    if (prec >= 2) {   // split BF16: three products, or four with lo * lo
        launch_bf3(st, MODE, prec == 3 ? 4 : 3, nst, chunks, work, nwork, A, B, C, jlo, offdiag);
        return;
    }
    const int grid = 8 * ((nwork + 7) / 8);
    k_gemm<MODE><<<grid, 256, 0, st>>>(chunks, work, nwork, A, B, C, jlo);
}

void launch_gemm_whiten_left(hipStream_t st, int prec, int nst, const ChunkDev *chunks, const Work *work,
                             int nwork, const void *li, const void *X, void *Y, int jlo) {
    if (prec == 0) {
        if (nwork > 0) launch_gemm64_left(st, chunks, work, nwork, (const double *)li, (const double *)X, (double *)Y, jlo);
        return;
    }
    launch_mode<MODE_LEFT>(st, prec, nst, chunks, work, nwork, li, X, Y, jlo);
}
void launch_gemm_whiten_right(hipStream_t st, int prec, int nst, const ChunkDev *chunks, const Work *work,
                              int nwork, const void *li, const void *Y, void *G, int jlo) {
    if (prec == 0) {
        if (nwork > 0) launch_gemm64_right(st, chunks, work, nwork, (const double *)li, (const double *)Y, (double *)G, jlo);
        return;
    }
    launch_mode<MODE_RIGHT>(st, prec, nst, chunks, work, nwork, Y, li, G, jlo);
}
void launch_gemm_gram(hipStream_t st, int prec, int nst, const ChunkDev *chunks, const Work *work, int nwork,
                      bool offdiag, const void *G, double *gram) {
    if (prec == 0) {
        if (nwork > 0) launch_gram64(st, chunks, work, nwork, (const double *)G, gram);
        return;
    }
    launch_mode<MODE_GRAM>(st, prec, nst, chunks, work, nwork, G, G, gram, 0, offdiag);
}

}  // namespace qml

namespace qml {

// ------------------------------------------------- split-BF16x3 GEMMs --
// Operands are stored pre-split: element (r, k) of an operand is hi[o] +
// hi[lo_off + o] (two bf16 planes), so the main loop moves bytes and issues
// MFMAs only.  The whitening products' operands (Li, the stack, P) are in
// the blocked layout of bf3_tiled, o = bf3_tiled(r, k, Np), so that a
// staged 16 x 32 block is one contiguous kilobyte; the Gram's (the G store,
// one row per member) are row-major, o = r ld + k.  Every product is A B^T with both operands K-major
// (X_j is symmetric; Li^T and the Gram are NT by construction).
//
// A workgroup computes a 128x128 tile with one wave per 64x64 quarter
// (4x4 blocks of 16x16, three v_mfma_f32_16x16x32_bf16 per block and K step:
// lo*hi, hi*lo, hi*hi; NPROD = 4 adds lo*lo first).  The lo*lo term is as
// large as what the two-plane split leaves out of each operand (both about
// 2^-16 of the product); adding it about halves the error of the products.  Waves whose quarter lies outside the matrix, or
// strictly below the diagonal for the upper-only products, skip their MFMAs
// (a separate copy of the loop) but still stage their share of the operands.
// NST LDS stages: the whitening products use one (168 VGPRs and 36 KB of
// LDS, three workgroups per CU; the next stage waits in registers), the Gram
// two (two workgroups per CU, a second register set two stages ahead).
//
// LDS: per stage four planes (A hi, A lo, B hi, B lo) of rows x 32 bf16
// (64 bytes, unpadded).  The four 16-byte chunks of row r sit at slot
// c ^ (((r >> 1) ^ ((r >> 3) & 1)) & 3): any 16 consecutive rows (from a multiple
// of 16) read at one chunk, and the staging writes (four rows' four chunks
// per 16 lanes), then fall on 16 distinct 16-byte slots of a 256-byte span
// of the 64 banks, and any aligned 8 of them on 8 distinct slots of 128
// bytes.
//
// The MFMA is issued as B-fragment x A-fragment, so that each lane ends with
// four consecutive columns of one output row (8-byte bf16 / 32-byte FP64
// stores) instead of four rows of one column.
constexpr int BK = 32;

// the swizzle repeats every 16 rows, so fragment block x sits at a fixed
// offset x * 16 * BK from block 0
__device__ __forceinline__ int bf3_slot(int r, int c) { return r * BK + ((c ^ bf3_swz(r & 15)) << 3); }

// 128x128 output tiles of four waves (2 x 2), each a 64x64 quarter
constexpr int BF3_BM = 128, BF3_BN = 128;
constexpr int BF3_PL = BF3_BM * BK;   // elements per LDS plane
constexpr int BF3_STG = 4 * BF3_PL;   // elements per stage: A hi, A lo, B hi, B lo
constexpr int BF3_EP = 72;            // row pitch of the staged epilogue block, in bf16

// First row (column) of tile row (column) I of a whitening product.  Where Np
// is an odd number of 64-blocks the half tile comes first, not last: tile row 0
// then starts 64 rows before the matrix.  The sums of a row tile run to its
// last row, so a half tile costs the right product half its waves over 64 terms
// there and over all of Np at the end (13 % of the steps over N ~ U[150, 700]).
__device__ __forceinline__ int bf3_origin(int I, int Np) { return I * 128 - ((Np & 64) ? 64 : 0); }
// a byte in the global address space
typedef const char __attribute__((address_space(1))) GlobalB;

// Operands and K range of one work item (tile I, J of member or split j).
struct Bf3Item {
    const __bf16 *Ahi, *Bhi;   // hi planes; the lo planes follow at alo / blo elements
    long long lda, ldb, alo, blo;
    int arows, brows, kbeg, kend, Mv, Nv;
};

template <int MODE>
__device__ __forceinline__ Bf3Item bf3_item(const ChunkDev &c, const Work &wk, int jlo, const __bf16 *Abase,
                                            const __bf16 *Bbase) {
    Bf3Item t;
    const int Np = c.Np;
    const long long msz = (long long)Np * Np;
    const int I0 = bf3_origin(wk.I, Np), J0 = bf3_origin(wk.J, Np);
    t.kbeg = 0;
    if (MODE == MODE_LEFT) {
        // P = Li M, lower tiles (J <= I): Li[i,k] needs k <= i and the stored
        // T = M^T (upper triangle of X_j, diagonal halved) needs k >= n
        t.Ahi = Abase + c.lic_off;
        t.Bhi = Bbase + c.stk_off + 2 * (wk.j - jlo) * msz;
        t.lda = t.ldb = Np;
        t.alo = t.blo = msz;
        t.arows = t.brows = Np;
        t.kbeg = max(0, J0);
        t.kend = min(Np, I0 + BF3_BM);
        t.Mv = t.Nv = Np;
    } else if (MODE == MODE_RIGHT) {
        // G = P Li^T + Li P^T, upper tiles (I <= J): both terms need
        // k <= min(i, n) <= i, so k < I0 + BM; the second term swaps the
        // operand bases (same row offsets)
        t.Ahi = Abase + c.stk_off + 2 * (wk.j - jlo) * msz;
        t.Bhi = Bbase + c.lic_off;
        t.lda = t.ldb = Np;
        t.alo = t.blo = msz;
        t.arows = t.brows = Np;
        t.kend = min(Np, I0 + BF3_BM);
        t.Mv = t.Nv = Np;
    } else {
        const long long ktot = (long long)c.ntu * TILE * TILE;
        t.Ahi = t.Bhi = Abase + c.g_off;
        t.lda = t.ldb = 2 * ktot;
        t.alo = t.blo = ktot;
        t.arows = t.brows = c.m;
        t.kbeg = wk.j * TILE * TILE;
        t.kend = t.kbeg + TILE * TILE;
        t.Mv = t.Nv = c.m;
    }
    if (MODE != MODE_GRAM) {
        // past the chunk's N pixels every product is an exact zero (D = 0
        // there), so the sweep ends at N rounded up to a K step
        const int kn32 = (c.N + BK - 1) / BK * BK;
        t.kend = max(t.kbeg, min(t.kend, kn32));
    }
    return t;
}

// The K steps [tlo, thi) of a term that a wave multiplies: those whose products
// are not exact zeros.  Li[i][k] = 0 for k > i, the stored T[n][k] = 0 for k < n
// and P is lower triangular, so LEFT (rows i of Li, rows n of T) needs k in
// [c0, r0 + 64), and RIGHT (P or Li rows i in both terms) k < r0 + 64.  Past the
// chunk's N pixels (D = 0) T, P and G vanish, so k < N and a wave whose rows or
// columns all lie past N multiplies nothing.  The accumulators start at +0 and
// no sum of exact zeros changes them, so the results are those of the full
// sweep, bit for bit; and what is never multiplied need not be written: T's
// 64-blocks below the diagonal and P's above it are not.
template <int MODE>
__device__ __forceinline__ void bf3_steps(const ChunkDev &c, bool active, int r0, int c0, int kbeg, int kend, int &tlo,
                                          int &thi) {
    const int kn32 = (c.N + BK - 1) / BK * BK;
    const bool pad = MODE != MODE_GRAM && (r0 >= c.N || c0 >= c.N);
    tlo = (MODE == MODE_LEFT) ? max(0, (c0 - kbeg) / BK) : 0;
    thi = (!active || pad) ? 0 : (MODE == MODE_GRAM) ? (kend - kbeg) / BK : (min(r0 + 64, kn32) - kbeg) / BK;
}

// One BK step of a wave's 64x64 quarter out of LDS, the hi planes of A and B
// at sa and sb and their lo planes behind them: fragment row offsets aoff /
// boff (rows 16x + lane%16 of the wave's slab, chunk lane/16).
template <int NPROD>
__device__ __forceinline__ void bf3_mfma(const __bf16 *sa, const __bf16 *sb, int aoff, int boff, f4 (&acc)[4][4]) {
    bf8 bh[4], bl[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        bh[y] = *(const bf8 *)(sb + boff + y * 16 * BK);
        bl[y] = *(const bf8 *)(sb + BF3_PL + boff + y * 16 * BK);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const bf8 ah = *(const bf8 *)(sa + aoff + x * 16 * BK);
        const bf8 al = *(const bf8 *)(sa + BF3_PL + aoff + x * 16 * BK);
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            if constexpr (NPROD == 4)
                acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[y], al, acc[x][y], 0, 0, 0);
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[y], al, acc[x][y], 0, 0, 0);
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[y], ah, acc[x][y], 0, 0, 0);
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[y], ah, acc[x][y], 0, 0, 0);
        }
    }
}

// Output of a wave's 64x64 quarter at (r0, c0); ep is the wave's own LDS
// region of 64 rows x BF3_EP (the stage buffers are free: the caller passed
// a barrier after the last step).
//   Gram: FP64 partials, x2 for off-diagonal G tiles, into the split's block.
//   LEFT / RIGHT: the FP32 block split into bf16 hi and lo planes, written
//   through LDS: the wave stages one plane (64 rows of 128 bytes at a row
//   pitch of 144 bytes, against bank conflicts) in its region, then each
//   store instruction writes eight full 128-byte rows, 16 bytes per lane.
//   One wave's LDS operations complete in order, so no barrier is needed.
template <int MODE>
__device__ __forceinline__ void bf3_epilogue(f4 (&acc)[4][4], const ChunkDev &c, const Work &wk, int jlo, int r0,
                                             int c0, void *Cbase, __bf16 *ep, int lane) {
    // lane holds C[16x + lane%16][16y + 4(lane/16) + u], u = 0..3
    const int orow = lane % 16, ocol = 4 * (lane / 16);
    if (MODE == MODE_GRAM) {
        const int ntile = c.mt * (c.mt + 1) / 2;
        const double wgt = packed_tile_is_diag(wk.j, c.nt) ? 1.0 : 2.0;
        double *C = (double *)Cbase + c.gram_off
                  + ((size_t)wk.j * ntile + upper_tile_index(r0 / TILE, c0 / TILE, c.mt)) * TILE * TILE;
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                d4 v;
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = wgt * (double)acc[x][y][u];
                double *o = C + (16 * x + orow) * TILE + 16 * y + ocol;
                *(double2 *)o = double2{v[0], v[1]};
                *(double2 *)(o + 2) = double2{v[2], v[3]};
            }
        return;
    }
    const int Np = c.Np;
    const long long msz = (long long)Np * Np;
    __bf16 *C = (__bf16 *)Cbase;
    long long base, ldc, lo;
    if (MODE == MODE_LEFT) {
        // P in the blocked layout: the quarter's eight 1 KB blocks
        base = c.stk_off + 2 * (wk.j - jlo) * msz;
        ldc = Np;
        lo = msz;
    } else {
        const long long ktot = (long long)c.ntu * TILE * TILE;
        base = c.g_off + 2 * wk.j * ktot + (long long)upper_tile_index(r0 / TILE, c0 / TILE, c.nt) * TILE * TILE;
        ldc = TILE;
        lo = ktot;
    }
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    // hi plane first; acc then keeps the residual v - hi for the lo plane
#pragma unroll 1
    for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                bf4 h;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    h[u] = (__bf16)acc[x][y][u];
                    acc[x][y][u] -= (float)h[u];
                }
                *(bf4 *)(ep + (16 * x + orow) * BF3_EP + 16 * y + ocol) = h;
            }
        __bf16 *Cp = C + base + plane * lo;
        typedef unsigned int u4 __attribute__((ext_vector_type(4)));
        if (MODE == MODE_LEFT) {
            // store s8 writes block (r0/16 + s8/2, c0/32 + s8%2) whole: lane i
            // fills slot i, row i/4 of the block, chunk (i%4) ^ bf3_swz(i/4)
            const int rr = lane / 4, ch = (lane % 4) ^ bf3_swz(rr);
#pragma unroll
            for (int s8 = 0; s8 < 8; ++s8) {
                const int rb = s8 / 2, kb = s8 % 2;
                __builtin_nontemporal_store(*(const u4 *)(ep + (16 * rb + rr) * BF3_EP + 32 * kb + 8 * ch),
                                            (u4 *)(Cp + bf3_tiled(r0 + 16 * rb, c0 + 32 * kb, Np) + 8 * lane));
            }
        } else {
#pragma unroll
            for (int s8 = 0; s8 < 8; ++s8) {
                const int r = 8 * s8 + lane / 8, ch = lane % 8;
                __builtin_nontemporal_store(*(const u4 *)(ep + r * BF3_EP + 8 * ch),
                                            (u4 *)(Cp + (long long)r * ldc + 8 * ch));
            }
        }
    }
}

template <int MODE, int NST, int NPROD>
__global__ __launch_bounds__(256, NST == 1 ? 3 : 2)
void k_gemm_bf3(const ChunkDev *cs, const Work *work, int nwork, const __bf16 *Abase, const __bf16 *Bbase,
                void *Cbase, int jlo) {
    constexpr int BM = BF3_BM, BN = BF3_BN;
    constexpr int RP = 256 / 4;                 // rows staged per pass
    constexpr int PA = BM / RP, PB = BN / RP;   // staging passes per plane
    constexpr int PLA = BF3_PL, PLB = BF3_PL;   // elements per LDS plane
    constexpr int STG = BF3_STG;                // elements per stage
    const int li = xcd_logical(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    const int I0 = (MODE == MODE_GRAM) ? wk.I * BM : bf3_origin(wk.I, c.Np);
    const int J0 = (MODE == MODE_GRAM) ? wk.J * BN : bf3_origin(wk.J, c.Np);
    const Bf3Item it = bf3_item<MODE>(c, wk, jlo, Abase, Bbase);
    const __bf16 *Ahi = it.Ahi, *Bhi = it.Bhi;
    const long long lda = it.lda, ldb = it.ldb, alo = it.alo, blo = it.blo;
    const int arows = it.arows, brows = it.brows, kbeg = it.kbeg, kend = it.kend, Mv = it.Mv, Nv = it.Nv;
    constexpr int SMEM = (NST * STG > 4 * 64 * BF3_EP) ? NST * STG : 4 * 64 * BF3_EP;
    __shared__ __attribute__((aligned(16))) __bf16 smem[SMEM];
    const int tid = threadIdx.x, lane = tid % 64, w = tid / 64;
    const int wm = w / 2, wn = w % 2;
    const int r0 = I0 + 64 * wm, c0 = J0 + 64 * wn;
    bool active = r0 >= 0 && c0 >= 0 && r0 < Mv && c0 < Nv;
    active = active && (MODE == MODE_LEFT ? c0 <= r0 : c0 >= r0);
    // steps of a term that the wave multiplies (bf3_steps)
    int tlo, thi;
    bf3_steps<MODE>(c, active, r0, c0, kbeg, kend, tlo, thi);
    const auto on = [&](int st) { return st >= tlo && st < thi; };
    f4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = f4{0.f, 0.f, 0.f, 0.f};
    // Staging: thread t loads the 16-byte chunk t%4 of rows t/4 + RP*q, so
    // four consecutive lanes read one contiguous 64-byte row segment.  Rows
    // past the operand read row 0 instead: for the whitening products Np is
    // a multiple of 64, so such rows only feed inactive waves; for the Gram
    // they feed output rows >= m that are never read.  The loads are
    // therefore unconditional (no exec branches).
    static_assert(PA >= 1 && PA <= 2 && PB >= 1 && PB <= 2, "staging passes");
    const int lr = tid / 4, lc = tid % 4;
    const auto arow = [&](int q) { const int r = I0 + lr + RP * q; return r >= 0 && r < arows ? r : 0; };
    const auto brow = [&](int q) { const int r = J0 + lr + RP * q; return r >= 0 && r < brows ? r : 0; };
    // per-thread element offsets of the staged rows; the operand bases are
    // workgroup-uniform.  The whitening products' offsets stay below Np^2
    // (32 bits); the Gram's rows are whole members of 2 ntu TILE^2 elements,
    // so m ntu >= 2^18 (e.g. N ~ 2900 with 250 stored Q) needs 64 bits.
    // In the blocked layout chunk lc of row r at K step 0 is bf3_tiled(r,
    // 8 lc, Np), and K step k0 (a multiple of 32) adds 16 k0.
    using off_t = typename std::conditional<MODE == MODE_GRAM, long long, int>::type;
    const auto roff = [&](int r, long long ld) -> off_t {
        if constexpr (MODE == MODE_GRAM) return (off_t)r * (off_t)ld + 8 * lc;
        else return (off_t)bf3_tiled(r, 8 * lc, (int)ld);
    };
    const off_t oa0 = roff(arow(0), lda), oa1 = roff(arow(PA - 1), lda);
    const off_t ob0 = roff(brow(0), ldb), ob1 = roff(brow(PB - 1), ldb);
    constexpr int KSC = (MODE == MODE_GRAM) ? 1 : 16;   // element offset per unit of k
    const int wa0 = bf3_slot(lr, lc), wa1 = bf3_slot(lr + RP * (PA - 1), lc);
    const int wb0 = bf3_slot(lr, lc), wb1 = bf3_slot(lr + RP * (PB - 1), lc);
    // two staging register sets (P, Q): stage k+2 is in flight while k+1 waits
    // to be stored and k is multiplied
    uint4 Prah0, Pral0, Prah1, Pral1, Prbh0, Prbl0, Prbh1, Prbl1;
    [[maybe_unused]] uint4 Qrah0, Qral0, Qrah1, Qral1, Qrbh0, Qrbl0, Qrbh1, Qrbl1;
    // fragment reads: row 16x + lane%16 of the wave's 64-row slab, chunk lane/16
    const int rr = lane % 16, cq = lane / 16;
    const int aoff = bf3_slot(64 * wm + rr, cq), boff = bf3_slot(64 * wn + rr, cq);
#define QML_BF3_GLOADX(R, XA, XB, k0)                                            \
    R##rah0 = *(const uint4 *)((XA) + oa0 + KSC * (k0));                         \
    R##ral0 = *(const uint4 *)((XA) + alo + oa0 + KSC * (k0));                   \
    R##rbh0 = *(const uint4 *)((XB) + ob0 + KSC * (k0));                         \
    R##rbl0 = *(const uint4 *)((XB) + blo + ob0 + KSC * (k0));                   \
    if constexpr (PA > 1) {                                                      \
        R##rah1 = *(const uint4 *)((XA) + oa1 + KSC * (k0));                     \
        R##ral1 = *(const uint4 *)((XA) + alo + oa1 + KSC * (k0));               \
    }                                                                            \
    if constexpr (PB > 1) {                                                      \
        R##rbh1 = *(const uint4 *)((XB) + ob1 + KSC * (k0));                     \
        R##rbl1 = *(const uint4 *)((XB) + blo + ob1 + KSC * (k0));               \
    }
#define QML_BF3_GLOAD(R, k0) QML_BF3_GLOADX(R, Ahi, Bhi, k0)
#define QML_BF3_SSTORE(R, st)                                                    \
    {                                                                            \
        __bf16 *s0 = smem + (st) * STG;                                          \
        *(uint4 *)(s0 + wa0) = R##rah0;                                          \
        *(uint4 *)(s0 + PLA + wa0) = R##ral0;                                    \
        *(uint4 *)(s0 + 2 * PLA + wb0) = R##rbh0;                                \
        *(uint4 *)(s0 + 2 * PLA + PLB + wb0) = R##rbl0;                          \
        if constexpr (PA > 1) {                                                  \
            *(uint4 *)(s0 + wa1) = R##rah1;                                      \
            *(uint4 *)(s0 + PLA + wa1) = R##ral1;                                \
        }                                                                        \
        if constexpr (PB > 1) {                                                  \
            *(uint4 *)(s0 + 2 * PLA + wb1) = R##rbh1;                            \
            *(uint4 *)(s0 + 2 * PLA + PLB + wb1) = R##rbl1;                      \
        }                                                                        \
    }
#define QML_BF3_MFMA(st) bf3_mfma<NPROD>(smem + (st) * STG, smem + (st) * STG + 2 * BF3_PL, aoff, boff, acc);
// One K sweep over n = (kend - kbeg)/BK stages, two steps per pass: the
// loads of stage s+2 are issued (into the register set just stored), stage
// s is multiplied out of LDS, and stage s+1 (loaded a whole step earlier)
// goes into the other LDS buffer.  Loads past the sweep repeat the last
// stage (unconditional, so the wait counts stay exact) and are not stored.
#define QML_BF3_SWEEP(DO_MFMA)                                                \
    {                                                                         \
        const int ns = (kend - kbeg) / BK;                                    \
        const int klast = kend - BK;                                          \
        QML_BF3_GLOAD(P, kbeg)                                                \
        QML_BF3_GLOAD(Q, min(kbeg + BK, klast))                               \
        QML_BF3_SSTORE(P, 0)                                                  \
        __syncthreads();                                                      \
        int s = 0;                                                            \
        for (; s + 1 < ns; s += 2) {                                          \
            const int k0 = kbeg + s * BK;                                     \
            QML_BF3_GLOAD(P, min(k0 + 2 * BK, klast))                         \
            if (DO_MFMA && on(s)) QML_BF3_MFMA(0)                             \
            QML_BF3_SSTORE(Q, 1)                                              \
            __syncthreads();                                                  \
            QML_BF3_GLOAD(Q, min(k0 + 3 * BK, klast))                         \
            if (DO_MFMA && on(s + 1)) QML_BF3_MFMA(1)                         \
            if (s + 2 < ns) QML_BF3_SSTORE(P, 0)                              \
            __syncthreads();                                                  \
        }                                                                     \
        if (s < ns) {                                                         \
            if (DO_MFMA && on(s)) QML_BF3_MFMA(0)                             \
            __syncthreads();                                                  \
        }                                                                     \
    }
// Single LDS stage: stage s+1 is loaded into registers while stage s is
// multiplied, then stored once every wave has read stage s.  The last stage
// is multiplied outside the loop, so no load is left in flight into the
// epilogue.
#define QML_BF3_SWEEP1(DO_MFMA)                                               \
    {                                                                         \
        const int ns = (kend - kbeg) / BK;                                    \
        QML_BF3_GLOAD(P, kbeg)                                                \
        QML_BF3_SSTORE(P, 0)                                                  \
        __syncthreads();                                                      \
        for (int s = 0; s + 1 < ns; ++s) {                                    \
            QML_BF3_GLOAD(P, kbeg + (s + 1) * BK)                             \
            if (DO_MFMA && on(s)) QML_BF3_MFMA(0)                             \
            __syncthreads();                                                  \
            QML_BF3_SSTORE(P, 0)                                              \
            __syncthreads();                                                  \
        }                                                                     \
        if (DO_MFMA && on(ns - 1)) QML_BF3_MFMA(0)                            \
        __syncthreads();                                                      \
    }
#define QML_BF3_RUN                                                           \
    if constexpr (NST == 1) {                                                 \
        if (active) QML_BF3_SWEEP1(true)                                      \
        else QML_BF3_SWEEP1(false)                                            \
    } else {                                                                  \
        if (active) QML_BF3_SWEEP(true)                                       \
        else QML_BF3_SWEEP(false)                                             \
    }
// The right product's two terms as one sweep of 2n stages: P rows I
// against Li rows J, then Li rows I against P rows J (the same staged row
// offsets with the operand bases swapped), so the second term's first stage
// is in flight while the first term's last one is multiplied.
#define QML_BF3_SWEEP1_2T(DO_MFMA)                                            \
    {                                                                         \
        const int ns = (kend - kbeg) / BK;                                    \
        QML_BF3_GLOAD(P, kbeg)                                                \
        QML_BF3_SSTORE(P, 0)                                                  \
        __syncthreads();                                                      \
        for (int s = 0; s + 1 < 2 * ns; ++s) {                                \
            const int sn = s + 1;                                             \
            const bool second = sn >= ns;                                     \
            const __bf16 *xa = second ? Bhi : Ahi, *xb = second ? Ahi : Bhi;  \
            QML_BF3_GLOADX(P, xa, xb, kbeg + (second ? sn - ns : sn) * BK)    \
            if (DO_MFMA && on(s < ns ? s : s - ns)) QML_BF3_MFMA(0)           \
            __syncthreads();                                                  \
            QML_BF3_SSTORE(P, 0)                                              \
            __syncthreads();                                                  \
        }                                                                     \
        if (DO_MFMA && on(ns - 1)) QML_BF3_MFMA(0)                            \
        __syncthreads();                                                      \
    }
    if (kbeg < kend) {
        if constexpr (MODE == MODE_RIGHT && NST == 1) {
            if (active) QML_BF3_SWEEP1_2T(true)
            else QML_BF3_SWEEP1_2T(false)
        } else {
            QML_BF3_RUN
            static_assert(MODE != MODE_RIGHT || NST == 1, "the right product's two terms need one stage");
        }
    }
#undef QML_BF3_GLOAD
#undef QML_BF3_SSTORE
#undef QML_BF3_MFMA
#undef QML_BF3_SWEEP
#undef QML_BF3_SWEEP1
#undef QML_BF3_RUN
#undef QML_BF3_SWEEP1_2T
#undef QML_BF3_GLOADX
    if (!active) return;
    bf3_epilogue<MODE>(acc, c, wk, jlo, r0, c0, Cbase, smem + w * 64 * BF3_EP, lane);
}

// ------------------------------------------ split BF16, direct-to-LDS loads --
// The same products, tiles, LDS layout and MFMA order as k_gemm_bf3 (so the
// same results, bit for bit), with the operands staged by
// global_load_lds_dwordx4: each load moves 16 bytes per lane from global
// memory straight into LDS at (M0 base) + 16 x lane, with no register
// round trip, so several steps can be in flight at once without registers
// held for them.  Each operand has its own ring of slots (16 KB: its hi and lo
// planes, 128 rows of 32): NM for the member's (the stack T, or P; the Gram's
// rows I), NL for Li (the Gram's rows J).  Each wave loads four 1 KB blocks of
// 16 rows of either operand per step.  For the whitening products a block is
// stored in slot order (bf3_tiled), so lane i loads the block's 16 bytes at
// 16 i; for the Gram lane i loads row i/4 of the block at the chunk that the
// swizzle places in slot i, (i%4) ^ bf3_swz(i/4).  Rows outside the operand
// read row 0, as in k_gemm_bf3.
//
// Step s waits for its own blocks (s_waitcnt vmcnt counting what was issued
// after them), passes one barrier, issues Li's step s + NL - 1 and the
// member's s + NM - 1 into the slots that step s - 1 read (every wave is past
// that step), then multiplies step s.  The barrier is the bare s_barrier (no
// memory fence, which would wait for every load in flight), with compiler-level
// memory clobbers so that no LDS access moves across it.
//
// The whitening products take (NM, NL) = (3, 2): the member's panels come from
// HBM and have two steps to arrive, Li's from L2 one, and two workgroups of
// 80 KB fill a CU.  (2, 2) took 6 % longer for the left product and 3 % for the
// right; the Gram, whose operands are the same rows, is 4 % faster with (2, 2).
// What bounds the products is the traffic past L2, not the steps' structure:
// on 640 chunks of 150-700 pixels the left moves 86 GB at 4.4 TB/s (a copy runs
// at 4.4 to 5.3), the right 109 GB at 3.5, P about 1.7 times over.  Reading
// the next step's fragments a step ahead, or running a workgroup through up to
// eight items without a break, changed nothing (the latter cost locality: 24
// echelle chunks 18.6 -> 22.9 ms).  (3, 3): one workgroup of 96 KB, 1.7 x
// slower.
template <int PENDING>
__device__ __forceinline__ void bf3_wait_step(bool last) {
    // s_waitcnt: vmcnt <= PENDING, or 0 on the last step; lgkmcnt 0; expcnt not
    // waited on.  Encoding: vmcnt[3:0] and [15:14], expcnt[6:4], lgkmcnt[11:8].
    constexpr int ENC = (PENDING & 15) | (7 << 4) | ((PENDING >> 4) << 14);
    if (PENDING == 0 || last) __builtin_amdgcn_s_waitcnt(7 << 4);
    else __builtin_amdgcn_s_waitcnt(ENC);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int MODE, int NM, int NL, int NPROD>
__global__ __launch_bounds__(256, NM + NL < 6 ? 2 : 1)
void k_gemm_bf3d(const ChunkDev *cs, const Work *work, int nwork, const __bf16 *Abase, const __bf16 *Bbase,
                 void *Cbase, int jlo) {
    static_assert(NM >= NL && NL >= 2 && NM <= 3, "two or three slots");
    const int li = xcd_logical(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    const int I0 = (MODE == MODE_GRAM) ? wk.I * BF3_BM : bf3_origin(wk.I, c.Np);
    const int J0 = (MODE == MODE_GRAM) ? wk.J * BF3_BN : bf3_origin(wk.J, c.Np);
    const Bf3Item it = bf3_item<MODE>(c, wk, jlo, Abase, Bbase);
    constexpr int SLOT = 2 * BF3_PL;   // elements
    constexpr int SMEM = ((NM + NL) * SLOT > 4 * 64 * BF3_EP) ? (NM + NL) * SLOT : 4 * 64 * BF3_EP;
    __shared__ __attribute__((aligned(1024))) __bf16 smem[SMEM];
    const int tid = threadIdx.x, lane = tid % 64;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wm = w / 2, wn = w % 2;
    const int r0 = I0 + 64 * wm, c0 = J0 + 64 * wn;
    const bool active = r0 >= 0 && c0 >= 0 && r0 < it.Mv && c0 < it.Nv && (MODE == MODE_LEFT ? c0 <= r0 : c0 >= r0);
    f4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = f4{0.f, 0.f, 0.f, 0.f};
    // the member's operand is B of the left product and A of the others; the
    // right product's second term exchanges the roles
    constexpr bool mb = MODE == MODE_LEFT;
    const __bf16 *Mhi = mb ? it.Bhi : it.Ahi, *Lhi = mb ? it.Ahi : it.Bhi;
    // byte offsets of the lanes from a uniform base: the whitening products'
    // planes fit 32 bits (Np <= 16384), the Gram's rows do not
    using off_t = typename std::conditional<MODE == MODE_GRAM, long long, unsigned>::type;
    const int rl = lane / 4;
    const int ch = (lane % 4) ^ bf3_swz(rl);
    // this wave's blocks of a slot: plane w / 2 (hi, lo), rows 64 (w % 2) + 16 b;
    // blocked layout: the 16 rows of a block lie all inside the operand or all
    // outside it (Np is a multiple of 64), and lane i reads slot i of the block
    const auto offset = [&](int row0, int b, int rows, long long ld, long long lo) -> off_t {
        const int rb = row0 + 64 * (w % 2) + 16 * b, r = rb + rl;
        const bool in = r >= 0 && r < rows;
        const off_t plane = (off_t)((w / 2) ? lo : 0);
        if constexpr (MODE == MODE_GRAM) return 2 * ((off_t)(in ? r : 0) * (off_t)ld + plane + 8 * ch);
        else return 2 * ((off_t)bf3_tiled(in ? rb : 0, 0, (int)ld) + plane + 8 * lane);
    };
    // by row panel (I0 or J0); the right product stages both panels of both
    // operands, which share their layout
    off_t oi[4], oj[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        oi[b] = offset(I0, b, it.arows, it.lda, it.alo);
        oj[b] = offset(J0, b, it.brows, it.ldb, it.blo);
    }
    constexpr int STEP = 2 * BK * (MODE == MODE_GRAM ? 1 : 16);   // bytes from step to step
    const int kbeg = it.kbeg;
    const int ns = (it.kend - kbeg) / BK;
    const int total = (MODE == MODE_RIGHT) ? 2 * ns : ns;
    GlobalB *const m0 = (GlobalB *)Mhi + (size_t)kbeg * (STEP / BK), *const l0 = (GlobalB *)Lhi + (size_t)kbeg * (STEP / BK);
    const int dst0 = (w / 2) * BF3_PL + (w % 2) * 64 * BK;
    const auto issue = [&](GlobalB *x, bool rows_i, int s, int slot) {
        x += (size_t)((MODE == MODE_RIGHT && s >= ns) ? s - ns : s) * STEP;
        __bf16 *dst = smem + slot * SLOT + dst0;
#pragma unroll
        for (int b = 0; b < 4; ++b)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(x + (rows_i ? oi[b] : oj[b])),
                (__attribute__((address_space(3))) void *)(dst + b * 16 * BK), 16, 0, 0);
    };
    const auto issue_m = [&](int s, int slot) { issue(m0, mb ? false : !(MODE == MODE_RIGHT && s >= ns), s, slot); };
    const auto issue_l = [&](int s, int slot) { issue(l0, mb ? true : (MODE == MODE_RIGHT && s >= ns), s, NM + slot); };
    const int rr = lane % 16, cq = lane / 16;
    const int aoff = bf3_slot(64 * wm + rr, cq), boff = bf3_slot(64 * wn + rr, cq);
    int tlo, thi;
    bf3_steps<MODE>(c, active, r0, c0, kbeg, it.kend, tlo, thi);
    if (total > 0) {
        issue_m(0, 0);
        issue_l(0, 0);
        if (NL == 3 && total > 1) issue_l(1, 1);
        if (NM == 3 && total > 1) issue_m(1, 1);
        int sm = 0, sl = 0;   // the slots of step s
        for (int s = 0; s < total; ++s) {
            bf3_wait_step<4 * (NM + NL - 4)>(s + 1 >= total);
            const int pm = sm == 0 ? NM - 1 : sm - 1, pl = sl == 0 ? NL - 1 : sl - 1;   // step s - 1's
            if (s + NL - 1 < total) issue_l(s + NL - 1, pl);
            if (s + NM - 1 < total) issue_m(s + NM - 1, pm);
            const bool second = MODE == MODE_RIGHT && s >= ns;
            const int k = second ? s - ns : s;
            if (k >= tlo && k < thi) {
                const __bf16 *m = smem + sm * SLOT, *l = smem + (NM + sl) * SLOT;
                bf3_mfma<NPROD>((mb || second) ? l : m, (mb || second) ? m : l, aoff, boff, acc);
            }
            sm = sm + 1 == NM ? 0 : sm + 1;
            sl = sl + 1 == NL ? 0 : sl + 1;
        }
        // every wave is done with the slots before the epilogue reuses LDS
        bf3_wait_step<0>(true);
    }
    if (!active) return;
    bf3_epilogue<MODE>(acc, c, wk, jlo, r0, c0, Cbase, smem + w * 64 * BF3_EP, lane);
}

// The Gram where no chunk of the batch has more than 128 members (every work item
// on the diagonal): all pairs of the members over one G tile, each member's row
// staged once.  Wave W sums the upper 16 x 16 blocks of row
// blocks W and 7 - W (nine; with 64 members or fewer row block W alone), so that
// the waves carry equal parts, and blocks past the members are left out.  A block
// sums its 4096 terms in the same order as k_gemm_bf3, so the same results, bit
// for bit.  Three slots of 16 KB, two steps in flight, three workgroups per CU.
// Bound by reading the G store, 64 bytes a row and plane at a time, or on small
// batches by the latency of the 128 steps: 64 chunks of 256 pixels, 23 members, 190
// -> 62 us against k_gemm_bf3d (whose 640 items take two turns on the chip), 640
// chunks of 150 to 700 pixels 8.8 -> 8.6 ms.  With items off the diagonal that
// kernel takes all: in a launch of their own they read the G tiles once more (160
// chunks of up to 190 members 5.1 -> 6.3 ms).
template <int NPROD, int MB, int W, class Issue>
__device__ __forceinline__ void gram_sweep(const Issue &issue, const __bf16 *smem, int mb, const ChunkDev &c,
                                           const Work &wk, double *gram) {
    constexpr int X1 = (MB == 8) ? 7 - W : MB, N1 = (MB == 8) ? W + 1 : 1, ns = TILE * TILE / BK;
    const int lane = threadIdx.x % 64, off = bf3_slot(lane % 16, lane / 16);
    f4 acc0[MB - W], acc1[N1];
#pragma unroll
    for (int y = 0; y < MB - W; ++y) acc0[y] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int y = 0; y < N1; ++y) acc1[y] = f4{0.f, 0.f, 0.f, 0.f};
    const auto mul = [](bf8 xh, bf8 xl, bf8 yh, bf8 yl, f4 acc) {
        if constexpr (NPROD == 4) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yl, xl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yh, xl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yl, xh, acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(yh, xh, acc, 0, 0, 0);
    };
    issue(0, 0);
    issue(1, 1);
    int sl = 0;
    for (int s = 0; s < ns; ++s) {
        bf3_wait_step<MB / 2>(s + 1 >= ns);
        if (s + 2 < ns) issue(s + 2, sl == 0 ? 2 : sl - 1);
        const __bf16 *st = smem + sl * 2 * BF3_PL + off;
        const auto part = [&](int y, int pl) { return *(const bf8 *)(st + pl * BF3_PL + y * 16 * BK); };
        if (W < mb) {
            const bf8 ah = part(W, 0), al = part(W, 1);
            bf8 bh = {}, bl = {};
            if constexpr (MB == 8) {
                bh = part(X1, 0);
                bl = part(X1, 1);
            }
#pragma unroll
            for (int y = W; y < MB; ++y) {
                if (y >= mb) break;
                const bf8 yh = (y == W) ? ah : part(y, 0), yl = (y == W) ? al : part(y, 1);
                acc0[y - W] = mul(ah, al, yh, yl, acc0[y - W]);
                if (y >= X1) acc1[y - X1] = mul(bh, bl, yh, yl, acc1[y - X1]);
            }
        }
        sl = sl == 2 ? 0 : sl + 1;
    }
    // lane holds C[16x + lane%16][16y + 4(lane/16) + u], u = 0..3
    const double wgt = packed_tile_is_diag(wk.j, c.nt) ? 1.0 : 2.0;
    const int base = wk.I * (BF3_BM / TILE);
    double *E = gram + c.gram_off + (size_t)wk.j * (c.mt * (c.mt + 1) / 2) * TILE * TILE;
    const auto put = [&](int x, int y, f4 acc) {
        double *o = E + (size_t)upper_tile_index(base + x / 4, base + y / 4, c.mt) * TILE * TILE
                  + (16 * (x % 4) + lane % 16) * TILE + 16 * (y % 4) + 4 * (lane / 16);
        *(double2 *)o = double2{wgt * (double)acc[0], wgt * (double)acc[1]};
        *(double2 *)(o + 2) = double2{wgt * (double)acc[2], wgt * (double)acc[3]};
    };
#pragma unroll
    for (int y = W; y < MB; ++y) {
        if (y >= mb) break;
        put(W, y, acc0[y - W]);
        if (y >= X1) put(X1, y, acc1[y - X1]);
    }
}

template <int NPROD>
__global__ __launch_bounds__(256, 3) void k_gram_bf3(const ChunkDev *cs, const Work *work, int nwork,
                                                     const __bf16 *G, double *gram) {
    const int li = xcd_logical(nwork);
    if (li >= nwork) return;
    const Work wk = work[li];
    if (wk.c < 0) return;
    const ChunkDev c = cs[wk.c];
    __shared__ __attribute__((aligned(1024))) __bf16 smem[3 * 2 * BF3_PL];
    const int lane = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int I0 = wk.I * BF3_BM, mb = (min(BF3_BM, c.m - I0) + 15) / 16;
    const long long ktot = (long long)c.ntu * TILE * TILE;
    const int rl = lane / 4, ch = (lane % 4) ^ bf3_swz(rl);
    const auto sweep = [&](auto size) {
        constexpr int MB = decltype(size)::value, NB = MB / 2;   // NB blocks of 16 rows a wave and step
        const int row0 = 16 * NB * (w % 2);
        GlobalB *src[NB];   // plane w / 2 (hi, lo); rows past the members read the first
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int row = I0 + row0 + 16 * b + rl;
            src[b] = (GlobalB *)(G + c.g_off + (row < c.m ? row : I0) * 2 * ktot + (w / 2) * ktot
                                 + (long long)wk.j * TILE * TILE + 8 * ch);
        }
        __bf16 *const dst0 = smem + (w / 2) * BF3_PL + row0 * BK;
        const auto issue = [&](int s, int slot) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void *)(src[b] + (size_t)s * (2 * BK)),
                    (__attribute__((address_space(3))) void *)(dst0 + slot * 2 * BF3_PL + b * 16 * BK), 16, 0, 0);
        };
        if (w == 0) gram_sweep<NPROD, MB, 0>(issue, smem, mb, c, wk, gram);
        else if (w == 1) gram_sweep<NPROD, MB, 1>(issue, smem, mb, c, wk, gram);
        else if (w == 2) gram_sweep<NPROD, MB, 2>(issue, smem, mb, c, wk, gram);
        else gram_sweep<NPROD, MB, 3>(issue, smem, mb, c, wk, gram);
    };
    if (mb <= 4) sweep(std::integral_constant<int, 4>{});
    else sweep(std::integral_constant<int, 8>{});
}

template <int NPROD>
static void launch_bf3_np(hipStream_t st, int mode, int nst, const ChunkDev *chunks, const Work *work, int nwork,
                          const __bf16 *a, const __bf16 *b, void *C, int jlo, bool offdiag) {
    const int grid = 8 * ((nwork + 7) / 8);
    // nst, the staging of the operands: 1 one LDS stage (three workgroups
    // per CU, the next stage in registers); 2 two LDS stages (two workgroups
    // per CU, a second register set two stages ahead; not for the right
    // product, whose two-term sweep uses 1 instead); 3 and 4 direct-to-LDS
    // loads with two stages (three of the member's operand in the whitening
    // products; two workgroups per CU) and three (one).  Each
    // output sums its K steps in the same order either way, so the results
    // are identical.
#define QML_BF3_LAUNCH(M, N) k_gemm_bf3<M, N, NPROD><<<grid, 256, 0, st>>>(chunks, work, nwork, a, b, C, jlo)
#define QML_BF3D_LAUNCH(M, N, K) k_gemm_bf3d<M, N, K, NPROD><<<grid, 256, 0, st>>>(chunks, work, nwork, a, b, C, jlo)
    if (mode == MODE_LEFT) {
        if (nst == 4) QML_BF3D_LAUNCH(MODE_LEFT, 3, 3);
        else if (nst == 3) QML_BF3D_LAUNCH(MODE_LEFT, 3, 2);
        else if (nst == 2) QML_BF3_LAUNCH(MODE_LEFT, 2);
        else QML_BF3_LAUNCH(MODE_LEFT, 1);
    } else if (mode == MODE_RIGHT) {
        if (nst == 4) QML_BF3D_LAUNCH(MODE_RIGHT, 3, 3);
        else if (nst == 3) QML_BF3D_LAUNCH(MODE_RIGHT, 3, 2);
        else QML_BF3_LAUNCH(MODE_RIGHT, 1);
    } else {
        if (nst == 4) QML_BF3D_LAUNCH(MODE_GRAM, 3, 3);
        else if (nst == 3 && !offdiag) k_gram_bf3<NPROD><<<grid, 256, 0, st>>>(chunks, work, nwork, a, (double *)C);
        else if (nst == 3) QML_BF3D_LAUNCH(MODE_GRAM, 2, 2);
        else if (nst == 1) QML_BF3_LAUNCH(MODE_GRAM, 1);
        else QML_BF3_LAUNCH(MODE_GRAM, 2);
    }
#undef QML_BF3_LAUNCH
#undef QML_BF3D_LAUNCH
}

void launch_bf3(hipStream_t st, int mode, int nprod, int nst, const ChunkDev *chunks, const Work *work, int nwork,
                const void *A, const void *B, void *C, int jlo, bool offdiag) {
    if (nwork <= 0) return;
    const __bf16 *a = (const __bf16 *)A, *b = (const __bf16 *)B;
    if (nprod == 4)
        launch_bf3_np<4>(st, mode, nst, chunks, work, nwork, a, b, C, jlo, offdiag);
    else
        launch_bf3_np<3>(st, mode, nst, chunks, work, nwork, a, b, C, jlo, offdiag);
}

}  // namespace qml
