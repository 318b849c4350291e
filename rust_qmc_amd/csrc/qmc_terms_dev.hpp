// qmc_terms_dev.hpp -- radial sums of the packed shell records (TermTab).
#pragma once

#include <type_traits>

#include "qmc_device.hpp"
#include "qmc_terms.hpp"

namespace qmc {

// radial sums of a shell: R = sum c e, and with DER R_a = sum c a e and
// R_aa = sum c a^2 e
template <int NP, bool P, bool DER>
__device__ __forceinline__ void radial(const TermPrim* q, double r2, double s[3], double p[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) s[k] = p[k] = 0.0;
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const double a = q[k].ex, e = M<double>::exn(-a * r2);
    const double cs = q[k].cs * e;
    s[0] += cs;
    if constexpr (DER) {
      s[1] += cs * a;
      s[2] += cs * a * a;
    }
    if constexpr (P) {
      const double cp = q[k].cp * e;
      p[0] += cp;
      if constexpr (DER) {
        p[1] += cp * a;
        p[2] += cp * a * a;
      }
    }
  }
}

// f(integral_constant NP) for the shell's padded primitive count
template <class F>
__device__ __forceinline__ void by_count(int np, F f) {
  if (np == 1)
    f(std::integral_constant<int, 1>{});
  else if (np == 3)
    f(std::integral_constant<int, 3>{});
  else
    f(std::integral_constant<int, 6>{});
}

// body(NP, SP, primitives, first MO row) for every shell of nucleus I, NP
// and SP integral constants (padded primitive count, sp shell or s shell)
template <class Body>
__device__ __forceinline__ void nucleus_shells(const TermTab& T, int I, Body body) {
  using std::integral_constant;
  const int pat = T.pat[I];
  const TermShell h = T.sh[T.sh0[I]];
  const TermPrim* pr = T.pr + h.p0;
  if (pat == TERMS_PAT_631G) {
    body(integral_constant<int, 6>{}, integral_constant<bool, false>{}, pr, h.row);
    body(integral_constant<int, 3>{}, integral_constant<bool, true>{}, pr + 6, h.row + 1);
    body(integral_constant<int, 1>{}, integral_constant<bool, true>{}, pr + 9, h.row + 5);
  } else if (pat == TERMS_PAT_631G_H) {
    body(integral_constant<int, 3>{}, integral_constant<bool, false>{}, pr, h.row);
    body(integral_constant<int, 1>{}, integral_constant<bool, false>{}, pr + 3, h.row + 1);
  } else {
    for (int t = T.sh0[I]; t < T.sh0[I + 1]; ++t) {
      const TermShell q = T.sh[t];
      by_count(q.np, [&](auto np) {
        if (q.sp)
          body(np, integral_constant<bool, true>{}, T.pr + q.p0, q.row);
        else
          body(np, integral_constant<bool, false>{}, T.pr + q.p0, q.row);
      });
    }
  }
}

}  // namespace qmc
