// Plain C++ of the library, shared by kernels and host code and compiled alone
// by the tests: index arithmetic of the mesh, bounds.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#define PUFF_BOTH __host__ __device__ __forceinline__
#else
#define PUFF_BOTH inline
#endif

namespace puff {

// Component (0: real, 1: imaginary) of a node in an interleaved mesh, counted
// in components.  Meshes hold up to 2^31 - 1 nodes: twice that is past an int.
PUFF_BOTH uint32_t node_component(int node, int part) { return 2u * (uint32_t)node + (uint32_t)part; }

// Largest (kx^2 + ky^2) / |2 kz| over the wavenumbers with kz != 0 (0 if none).
template <typename V>
double largest_phase_rate(const V& kx, const V& ky, const V& kz) {
    auto largest = [](const V& k) {
        double m = 0.0;
        for (double v : k) m = std::max(m, v * v);
        return m;
    };
    const double k2 = largest(kx) + largest(ky);
    double rate = 0.0;
    for (double v : kz)
        if (v != 0.0) rate = std::max(rate, k2 * std::fabs(1.0 / (2.0 * v)));
    return rate;
}

}  // namespace puff
