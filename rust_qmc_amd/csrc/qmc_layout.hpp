// qmc_layout.hpp -- positions between the ensemble's layout ([3N][ld] in the
// state type, walker fastest) and the caller's ([W][N][3] doubles).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qmc {

// the first n walkers of pos; out holds [n][n3]
template <class T>
hipError_t positions_out(const T* pos, int64_t ld, int64_t n, int n3, double* out, hipStream_t st);
// likewise; the columns n .. nz of pos (nz >= n) are set to zero
template <class T>
hipError_t positions_in(const double* in, int64_t ld, int64_t n, int64_t nz, int n3, T* pos, hipStream_t st);

}  // namespace qmc
