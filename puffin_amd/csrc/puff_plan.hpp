// Plain C++ of the library, shared by kernels and host code and compiled alone
// by the tests: index arithmetic of the mesh.
#pragma once

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

}  // namespace puff
