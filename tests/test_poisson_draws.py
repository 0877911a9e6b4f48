"""The engine's Poisson draws are the C++ standard library's, number for number
(std::poisson_distribution<int>(1.0) over std::mt19937_64, the reference's
PoissonRNG)."""
import subprocess

import numpy as np
import pytest

from lyspeq_amd.qml import poisson_draws

SRC = """
#include <cstdio>
#include <cstdlib>
#include <random>
int main(int, char **v) {
    std::mt19937_64 rng(std::strtoull(v[1], nullptr, 10));
    std::poisson_distribution<int> pd;
    for (long long i = 0, n = std::atoll(v[2]); i < n; ++i) std::printf("%d\\n", pd(rng));
}
"""


@pytest.fixture(scope="module")
def std_draws(tmp_path_factory):
    d = tmp_path_factory.mktemp("poisson")
    (d / "p.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", str(d / "p.cpp"), "-o", str(d / "p")], check=True)
    return lambda seed, n: np.array(subprocess.run([str(d / "p"), str(seed), str(n)], check=True,
                                                   capture_output=True, text=True).stdout.split(), dtype=np.int64)


# counts below, at and past a window of 16 x 312 uniforms; at 2e6 draws some
# take more uniforms than are looked at without a branch
@pytest.mark.parametrize("seed,n", [(0, 1), (1, 9), (2, 311), (3, 2496), (4, 5000), (7, 20000), (2**64 - 1, 2000000)])
def test_draws_are_the_standard_librarys(std_draws, seed, n):
    want = std_draws(seed, n)
    assert np.array_equal(poisson_draws(seed, n), want)
    if n == 2000000:
        assert want.max() >= 8


def test_short_calls_are_prefixes(std_draws):
    """A call makes as many blocks of uniforms as its count needs: every count
    up to three blocks and some around the full window gives the same draws."""
    want = std_draws(11, 6000)
    for n in list(range(1, 480)) + [2480, 2481, 2495, 2496, 2497, 2500, 2501, 4991, 4992, 5999]:
        assert np.array_equal(poisson_draws(11, n), want[:n]), n
