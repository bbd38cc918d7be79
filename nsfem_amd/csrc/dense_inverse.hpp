// Dense inverse of a symmetric positive definite matrix on the GPU, for the
// V-cycle's coarsest level.
#pragma once

#include <vector>

#include "common.hpp"

namespace nsfem
{
    // Inverse of m (n x n, row-major, host) into out (ld x ld, row-major,
    // device; rows and columns past n are zero), symmetrised.  Returns false,
    // with out unspecified, when a pivot has lost all but rounding noise of its
    // diagonal (not positive definite).  Blocking.
    template <typename T>
    bool denseInverseGpu(int n, const std::vector<double> & m, int ld, T * out, hipStream_t s);
} // namespace nsfem
