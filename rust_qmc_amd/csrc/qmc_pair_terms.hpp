// qmc_pair_terms.hpp -- the feature columns of the derivative matrix Y and
// the Jastrow-parameter terms of one particle pair, shared by the
// derivative kernels.
#pragma once

#include "qmc_device.hpp"

namespace qmc {

struct DerivLayout {
  int P, M, N, Qp;
  __device__ __forceinline__ int o(int k) const { return k; }
  __device__ __forceinline__ int om(int I, int c) const { return P + 3 * I + c; }
  __device__ __forceinline__ int e() const { return P + 3 * M; }
  __device__ __forceinline__ int one() const { return P + 3 * M + 1; }
  __device__ __forceinline__ int de(int k) const { return P + 3 * M + 2 + k; }
  __device__ __forceinline__ int f(int I, int c) const { return 2 * P + 3 * M + 2 + 3 * I + c; }
  __device__ __forceinline__ int g(int q, int c) const { return Qp + 3 * q + c; }
};

// O_k and d E_L / d p_k terms of one electron pair (Pade Jastrow only),
// handed to addO(slot, v) and addE(slot, v) by parameter slot: 0 = b_ee,
// 1 = a (a_para for same spins, a_anti otherwise), 2 + k = series term k.
// (dx, dy, dz) = r_i - r_j and gd(c) = G_i[c] - G_j[c], the difference of
// the two electrons' d ln psi / d r (read only when the pair is apart).
template <class T, class GD, class AO, class AE>
__device__ __forceinline__ void ee_pair_terms(const DevSys<T>& S, T dx, T dy, T dz, bool same, GD gd, AO addO,
                                              AE addE) {
  const int K = S.k_ee;
  T r, ir;
  M<T>::dist_inv(dx * dx + dy * dy + dz * dz, r, ir);
  const T a = same ? S.a_para : S.a_anti;
  const T* c = same ? S.c_para : S.c_anti;
  PairDerivs<T> pd;
  pd.init(r, S.b_ee, a, K, c);
  // O: d u / d b_ee = -(a + s') x^2, d u / d a = x, d u / d c_k = x^(k+2)
  addO(0, -pd.A1 * pd.x * pd.x);
  addO(1, pd.x);
  if (r < T(1e-10)) return;
  // Delta = (G_i - G_j) . rhat_ij
  const T dlt = gd(0) * (dx * ir) + gd(1) * (dy * ir) + gd(2) * (dz * ir);
  T du1, dl;
  pd.d_b(r, ir, S.b_ee, du1, dl);
  addE(0, -(dl + dlt * du1));
  pd.d_a(ir, S.b_ee, du1, dl);
  addE(1, -(dl + dlt * du1));
  T xk = T(1);
#pragma unroll
  for (int k = 0; k < MAXK; ++k) {  // unrolled, so the slot is a constant
    if (k >= K) break;
    addO(2 + k, xk * pd.x * pd.x);
    pd.d_c(k, ir, S.b_ee, xk, du1, dl);
    addE(2 + k, -(dl + dlt * du1));
    xk *= pd.x;
  }
}

// The same for electron i and nucleus I (slot 0 = b_en, 2 + k = the term k
// of the nucleus' species); (dx, dy, dz) = r_i - R_I and g(c) = G_i[c].
template <class T, class GI, class AO, class AE>
__device__ __forceinline__ void en_pair_terms(const DevSys<T>& S, int I, T dx, T dy, T dz, GI g, AO addO, AE addE) {
  const int Ke = S.k_en;
  T r, ir;
  M<T>::dist_inv(dx * dx + dy * dy + dz * dz, r, ir);
  const T* c = S.d_en[S.species[I]];
  PairDerivs<T> pd;
  pd.init(r, S.b_en, -S.Z[I], Ke, c);
  // d u_en / d b_en = (Z - s') y^2 = -A1 y^2
  addO(0, -pd.A1 * pd.x * pd.x);
  if (r < T(1e-10)) {
    T xk = T(1);
#pragma unroll
    for (int k = 0; k < MAXK; ++k) {
      if (k >= Ke) break;
      addO(2 + k, xk * pd.x * pd.x);
      xk *= pd.x;
    }
    return;
  }
  const T dlt = g(0) * (dx * ir) + g(1) * (dy * ir) + g(2) * (dz * ir);
  T du1, dl;
  pd.d_b(r, ir, S.b_en, du1, dl);
  addE(0, -(T(0.5) * dl + dlt * du1));
  T xk = T(1);
#pragma unroll
  for (int k = 0; k < MAXK; ++k) {
    if (k >= Ke) break;
    addO(2 + k, xk * pd.x * pd.x);
    pd.d_c(k, ir, S.b_en, xk, du1, dl);
    addE(2 + k, -(T(0.5) * dl + dlt * du1));
    xk *= pd.x;
  }
}

// feature columns of a pair slot: e-e (class 0 anti, 1 para) and e-n
// (species sp) Jastrow parameters in the order [b_ee, b_en, a_anti,
// a_para, c_anti[K], c_para[K], d_en[species][Ke]]
template <class T>
__device__ __forceinline__ int ee_slot_col(const DevSys<T>& S, int cls, int slot) {
  return slot == 0 ? 0 : (slot == 1 ? 2 + cls : 4 + cls * S.k_ee + slot - 2);
}
template <class T>
__device__ __forceinline__ int en_slot_col(const DevSys<T>& S, int sp, int slot) {
  return slot == 0 ? 1 : 4 + 2 * S.k_ee + sp * S.k_en + slot - 2;
}

}  // namespace qmc
