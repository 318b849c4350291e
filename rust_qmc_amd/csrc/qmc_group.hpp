// qmc_group.hpp -- the lane-group engine: a walker is owned by a group of
// G = 2, 4, 8 or 16 lanes (the smallest that holds its electrons), one
// electron per lane.
#pragma once

#include "qmc_derivs.hpp"
#include "qmc_kernels.hpp"

namespace qmc {

struct GroupOps {
  int nu, nd;
  int wpb;                               // walkers per block (partial-sum row)
  // largest walker counts of the sweeps, derivatives and evaluations (see
  // make_group)
  int64_t w_sweep, w_deriv, w_eval;
  bool (*match)(const DevSys<double>&);  // null for the run-time shell loops
  // all-electron Metropolis; _ns: compiled for a Jastrow without Pade series terms
  hipError_t (*ae64)(const void*, EnsView<double>, SweepArgs, double*, double*, hipStream_t);
  hipError_t (*ae32)(const void*, EnsView<float>, SweepArgs, double*, double*, hipStream_t);
  hipError_t (*ae64_ns)(const void*, EnsView<double>, SweepArgs, double*, double*, hipStream_t);
  hipError_t (*ae32_ns)(const void*, EnsView<float>, SweepArgs, double*, double*, hipStream_t);
  // single-electron Metropolis and drift-diffusion sweeps in FP64 for a
  // Jastrow without series terms; null for the run-time shell loops
  hipError_t (*sweep64_ns)(const void*, EnsView<double>, SweepArgs, double*, double*, hipStream_t);
  hipError_t (*dd64_ns)(const void*, EnsView<double>, SweepArgs, double*, double*, hipStream_t);
  // the derivative matrix Y in FP64 (both precisions) for such a Jastrow;
  // null for the run-time shell loops
  hipError_t (*derivs_ns)(const void*, DerivArgs, hipStream_t);
  // qmc_evaluate's outputs from [W][N][3] positions, likewise
  hipError_t (*eval_ns)(const void*, int64_t, const double*, EvalOut, int*, hipStream_t);
};

// the lane-group kernels of a system, chosen as find_engine chooses the
// register engine's (the same electron counts and shell structures)
const GroupOps* find_group(const DevSys<double>& D, bool generic_only);

}  // namespace qmc
