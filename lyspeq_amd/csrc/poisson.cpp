// Unit-mean Poisson draws of the reference's PoissonRNG (core/bootstrapper.hpp:
// 19-37): std::mt19937_64 seeded once, std::poisson_distribution<int>(1.0).
// The distribution multiplies uniforms until the product is at most exp(-1) and
// returns one less than their number (Knuth); a uniform is one 64-bit output
// rounded to double and scaled by 2^-64, at most 1 - 2^-53.  The draws here are
// the same, number for number.
//
// Drawn through the library they took 70 ns each on the GPU's host (102 on an
// AVX-512 Xeon), most of it in the uniform's generic scaling and in one
// mispredicted branch per draw; 6 ns this way on the Xeon.  Here a block of
// generator outputs is twisted, tempered and scaled in vector loops; for every
// position the count of uniforms that a draw starting there takes is formed
// without branches, from products of up to eight (1 + the partial products above
// exp(-1), which never rise); the draws then hop from start to start.
#include "poisson.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace qml {

namespace {

// MT19937-64 (Nishimura 2000; the C++ standard's mersenne_twister_engine)
constexpr int MT_N = 312, MT_M = 156;
constexpr uint64_t MT_A = 0xB5026F5AA96619E9ull, MT_UP = 0xFFFFFFFF80000000ull, MT_LOW = 0x7FFFFFFFull;

constexpr int BLOCKS = 16, LEN = BLOCKS * MT_N;   // uniforms made at a time
constexpr int LOOK = 8;                           // factors looked at without a branch

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define QML_CLONES __attribute__((target_clones("avx512dq", "avx2", "default")))
#else
#define QML_CLONES
#endif

inline uint64_t twist(uint64_t cur, uint64_t next, uint64_t far) {
    const uint64_t x = (cur & MT_UP) | (next & MT_LOW);
    return far ^ (x >> 1) ^ ((0 - (x & 1)) & MT_A);
}

// `blocks` regenerations of the state into uniforms u[0 .. blocks MT_N).
QML_CLONES void uniforms(uint64_t *mt, double *u, int blocks) {
    for (int b = 0; b < blocks; ++b) {
        for (int i = 0; i < MT_M; ++i) mt[i] = twist(mt[i], mt[i + 1], mt[i + MT_M]);
        for (int i = MT_M; i < MT_N - 1; ++i) mt[i] = twist(mt[i], mt[i + 1], mt[i - MT_M]);
        mt[MT_N - 1] = twist(mt[MT_N - 1], mt[0], mt[MT_M - 1]);
        double *o = u + b * MT_N;
        for (int i = 0; i < MT_N; ++i) {
            uint64_t y = mt[i];
            y ^= (y >> 29) & 0x5555555555555555ull;
            y ^= (y << 17) & 0x71D67FFFEDA60000ull;
            y ^= (y << 37) & 0xFFF7EEE000000000ull;
            y ^= y >> 43;
            const double v = (double)y * 0x1p-64;
            o[i] = v < 1.0 ? v : 1.0 - 0x1p-53;
        }
    }
}

// n[i] = uniforms taken by a draw that starts at u[i], LOOK + 1 if the first
// LOOK do not end it.
QML_CLONES void counts(const double *u, double stop, int len, int *n) {
    for (int i = 0; i < len; ++i) {
        double p = u[i];
        int k = 1;
        for (int f = 1; f <= LOOK; ++f) {
            k += p > stop;
            p *= u[i + f];
        }
        n[i] = k;
    }
}

}  // namespace

void poisson_draws(uint64_t seed, long long count, int *out) {
    uint64_t mt[MT_N];
    mt[0] = seed;
    for (int i = 1; i < MT_N; ++i) mt[i] = 6364136223846793005ull * (mt[i - 1] ^ (mt[i - 1] >> 62)) + (uint64_t)i;
    const double stop = std::exp(-1.0);
    // a window of uniforms: up to TAIL left over from the one before, then LEN;
    // a draw is made from it only while LOOK + 1 uniforms remain past its start
    constexpr int TAIL = LOOK + 1;
    double u[TAIL + LEN];   // on the stack (60 KB): a C entry allocates nothing here
    int n[TAIL + LEN];
    int have = 0, at = 0, ready = 0;   // uniforms in the window, the next one, starts with a count
    // left: draws still to make, two uniforms each on average.  The few of a short
    // call come from one block: one draw through Python takes 6.9 us on a Xeon
    // host, 13.0 with all 16 blocks (the library's generator 6.9).
    const auto refill = [&](long long left) {
        const int keep = have - at;   // at most TAIL
        for (int i = 0; i < keep; ++i) u[i] = u[at + i];
        const int blocks = left > LEN / 2 ? BLOCKS : (int)(2 * left + TAIL) / MT_N + 1;
        uniforms(mt, u + keep, std::min(blocks, BLOCKS));
        have = keep + std::min(blocks, BLOCKS) * MT_N;
        at = 0;
        ready = have - LOOK;
        counts(u, stop, ready, n);
    };
    for (long long i = 0; i < count; ++i) {
        if (at >= ready) refill(count - i);
        int k = n[at];
        if (k <= LOOK) {
            at += k;
        } else {   // one draw in 10^5: a product of more factors
            double p = 1.0;
            k = 0;
            do {
                if (at == have) refill(count - i);
                p *= u[at++];
                ++k;
            } while (p > stop);
        }
        out[i] = k - 1;
    }
}

}  // namespace qml
