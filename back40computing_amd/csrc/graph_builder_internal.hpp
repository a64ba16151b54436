// graph_builder_internal.hpp -- host helpers of graph_builder.cpp shared
// with the device CSR builder (b40c_csr_build.hip).  Not installed.
#pragma once

#include <stdint.h>

#include <vector>

// The seeded vertex permutation that scrambles R-MAT ids (b40c_graph_rmat).
void b40c_rmat_permutation(int32_t scale, uint64_t seed, std::vector<int32_t> *perm);

namespace b40c_hip {
// A device CSR built by b40c_csr_build.hip leaves its owner's hands: freed, or
// its arrays taken over (the builder gives its kept memory back with the last).
void device_csr_gone(int device);
}  // namespace b40c_hip
