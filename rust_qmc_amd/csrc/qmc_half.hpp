// qmc_half.hpp -- the half-wave engine: FP64 sweeps of 21 + 21-electron
// systems (benzene), one walker per 32 lanes, nothing shared between
// wavefronts but read-only tables.
#pragma once

#include "qmc_kernels.hpp"
#include "qmc_terms.hpp"

namespace qmc {

constexpr int HALF_W = 2;  // walkers per wavefront, which is one partial-sum row

constexpr int HALF_ROWS = 72;  // MO rows of the LDS table

// the engine runs a system that the packed parameter table holds with at
// most one shell per lane
inline bool half_fits(const TermTab& T) {
  const int n = T.sh0[T.n_nuc];
  return n <= 32 && T.sh[n - 1].row + (T.sh[n - 1].sp ? 4 : 1) <= HALF_ROWS;
}

inline int64_t half_blocks(int64_t W) { return (W + HALF_W - 1) / HALF_W; }

// single-electron Metropolis and drift-diffusion sweeps, as tile_sweep and
// tile_dd (partial sums of half_blocks(E.W) rows)
hipError_t half_sweep(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                      hipStream_t st);
hipError_t half_dd(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                   hipStream_t st);

}  // namespace qmc
