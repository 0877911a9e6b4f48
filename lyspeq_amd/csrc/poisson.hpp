// The draws behind qml_poisson_draws (host code).
#pragma once

#include <cstdint>

namespace qml {
// out[0 .. count): the first draws of std::poisson_distribution<int>(1.0) over
// std::mt19937_64(seed).
void poisson_draws(uint64_t seed, long long count, int *out);
}  // namespace qml
