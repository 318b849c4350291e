// qmc_layout.hpp -- positions between the ensemble's layout ([3N][ld] in the
// state type, walker fastest) and the caller's ([W][N][3] doubles).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace qmc {

template <class T>
hipError_t positions_out(const T* pos, int64_t ld, int64_t W, int n3, double* out, hipStream_t st);
// columns W .. ld of pos are set to zero
template <class T>
hipError_t positions_in(const double* in, int64_t ld, int64_t W, int n3, T* pos, hipStream_t st);

}  // namespace qmc
