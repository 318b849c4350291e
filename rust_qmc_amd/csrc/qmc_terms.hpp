// qmc_terms.hpp -- per-configuration terms (ln|psi|, gradients, Laplacians,
// E_L, parameter and nuclear derivatives) of 21 + 21-electron systems such
// as benzene: one electron per lane, a spin sector of three walkers per
// wavefront.
#pragma once

#include "qmc_derivs.hpp"
#include "qmc_kernels.hpp"
#include "qmc_sys.hpp"

namespace qmc {

constexpr int TERMS_N = 21;      // electrons per spin
constexpr int TERMS_W = 3;       // walkers per workgroup (63 of 64 lanes)
constexpr int TERMS_MAXSH = 40;  // shells
constexpr int TERMS_MAXP = 6;    // primitives per shell
constexpr int TERMS_ROWS = 80;   // MO coefficient rows (AOs, and an s row for every p-only shell)
constexpr int TERMS_PRIM = 160;  // primitive slots
constexpr int TERMS_MO = 6;      // distinct MOs whose coefficients follow the geometry
constexpr int TERMS_GRP = 32;    // MO-derivative groups per spin

// Shell patterns of a nucleus that are compiled: the 6-31G ones of a
// first-row atom (s of 6 primitives, sp of 3, sp of 1) and of hydrogen (s of
// 3, s of 1), whose shells then form one block of straight-line code; any
// other nucleus runs shell by shell.
enum : int { TERMS_PAT_ANY = 0, TERMS_PAT_631G = 1, TERMS_PAT_631G_H = 2 };

// The system as the kernel reads it, all with wave-uniform addresses and
// packed, so that benzene's table (13.6 KB) stays in the 16 KB scalar cache:
// the shells sorted by centre, their primitives zero-padded to 1, 3 or 6,
// the MO rows in the same order.
struct TermShell {
  int sp, np, row, p0;  // 1: s and p parts (4 MO rows), 0: s only (1 row); padded primitive count; first row, slot
};
struct TermPrim {
  double ex, cs, cp;
};
// d ln D / d R_{I,c} += sum_q d[q][c] (A^-1)_{m,k} chi_q(r_k), q the shell's s, px, py, pz
struct TermMoGrp {
  int sh, mi, I, pad;  // shell record, index into mo_list, the shell's centre
  double d[4][3];
};
struct TermTab {
  int n_nuc, n_mo, same;   // same: both spins' MO rows are equal
  int sh0[MAXN + 1];       // shells of nucleus I: [sh0[I], sh0[I + 1])
  int pat[MAXN];           // their pattern (TERMS_PAT_*)
  int g0[2][MAXN + 1];     // MO-derivative groups of (spin, nucleus)
  int mo_list[TERMS_MO];
  double nuc[MAXN][3];
  TermShell sh[TERMS_MAXSH];
  TermPrim pr[TERMS_PRIM];
  double mo[2][TERMS_ROWS][TERMS_N];
  TermMoGrp grp[2][TERMS_GRP];
};

// fills T from the system and its MO-derivative tables; false when the
// kernels do not fit it (21 + 21 electrons, s / p / sp Gaussian shells of at
// most 6 primitives, a Pade or no Jastrow without series terms)
bool terms_table(const DevSys<double>& D, const MoDerivPair* pairs, const MoDerivEntry* ents, const int p0[3],
                 TermTab& T);

// the derivative matrix Y as wave_derivs, in FP64
hipError_t terms_derivs(const void* Sd, const TermTab* T, DerivArgs A, hipStream_t st);
// qmc_evaluate's outputs from [W][N][3] positions, in FP64
hipError_t terms_eval(const void* Sd, const TermTab* T, int64_t W, const double* pos, EvalOut O, int* sing,
                      hipStream_t st);
// E_L of an ensemble's walkers (its eloc) from their positions
hipError_t terms_eloc(const void* Sd, const TermTab* T, EnsView<double> E, hipStream_t st);

}  // namespace qmc
