// qmc_group_dev.hpp -- device pieces of the lane-group engine: sums over a
// group of G lanes, the LDS tables of a wavefront's walkers, and a Slater
// inverse spread over the group with one matrix row per lane.
#pragma once

#include "qmc_wave_dev.hpp"

namespace qmc {

// sum over the G lanes of a group (aligned groups within a DPP row); every
// lane of the group gets the bit-identical sum
template <int G>
__device__ __forceinline__ double gsum(double v) {
  if constexpr (G >= 2) v += dpp_mov<0xB1>(v);
  if constexpr (G >= 4) v += dpp_mov<0x4E>(v);
  if constexpr (G >= 8) v += dpp_mov<0x141>(v);
  if constexpr (G >= 16) v += dpp_mov<0x140>(v);
  return v;
}

constexpr int group_lanes(int n) { return n <= 2 ? 2 : n <= 4 ? 4 : n <= 8 ? 8 : 16; }

// AO capacity of the LDS coefficient table: the compiled structure's count,
// or the largest system's
template <class Bs>
struct GroupAo {
  static constexpr int v = MAXAO;
};
template <class Bd>
struct GroupAo<CtBasis<Bd>> {
  static constexpr int v = bd_a0<Bd>(Bd::n_shell);
};

// Shapes and LDS of one wavefront: WPB walkers of N electrons.  A lane's
// electron is slot `slot` of sector `sp`; lanes past the electrons shadow
// electron 0 and are left out of every sum and store.
template <int NU, int ND, class Bs>
struct GroupShape {
  static constexpr int N = NU + ND, NS = NU > ND ? NU : ND, G = group_lanes(N), WPB = 64 / G;
  static constexpr int NSP = NS + (NS & 1);  // coefficient rows padded to 16 bytes
  struct Lds {
    double mo[GroupAo<Bs>::v][2][NSP];  // MO coefficients [ao][spin][m], zero past the sector's size
    double xyz[WPB][N][3];
    double prop[WPB][N][4];  // sweeps: each electron's proposal (or normals) and acceptance uniform
    double row[64][NS + 1];  // inverse rows in transit (odd stride: 64 lanes over all banks)
  };
};

template <int NU, int ND, class Bs, class Lds>
__device__ __forceinline__ void group_fill_mo(const DevSys<double>& S, Lds& L) {
  using Sh = GroupShape<NU, ND, Bs>;
  for (int q = threadIdx.x; q < S.n_ao * 2 * Sh::NSP; q += blockDim.x) {
    const int m = q % Sh::NSP, sp = (q / Sh::NSP) % 2, ao = q / (2 * Sh::NSP);
    L.mo[ao][sp][m] = m < (sp ? ND : NU) ? S.moT[sp][ao][m] : 0.0;
  }
  __syncthreads();
}

// add(ao, chi_ao(x, y, z)) for every AO; the functions of mo_values
template <class Bs, class Add>
__device__ __forceinline__ void ao_values(const DevSys<double>& S, double x, double y, double z, Add add) {
  Bs::shells(S, [&](auto sh) {
    const int c = sh.center(), kind = sh.kind(), p0 = sh.p0(), np = sh.nprim(), a0 = sh.a0();
    const double dx = x - S.nuc[c][0], dy = y - S.nuc[c][1], dz = z - S.nuc[c][2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (kind <= SH_P1) {
      double rs = 0.0, rp = 0.0;
      for (int k = 0; k < np; ++k) {
        const double e = prim_e(S, p0 + k, r2);
        if (kind == SH_S || kind == SH_SP) rs += S.coef_s[p0 + k] * e;
        if (kind != SH_S) rp += S.coef_p[p0 + k] * e;
      }
      if (kind == SH_S || kind == SH_SP) add(a0, rs);
      if (kind == SH_P1) {
        const int m = sh.m();
        add(a0, (m == 0 ? dx : (m == 1 ? dy : dz)) * rp);
      } else if (kind != SH_S) {
        const int b = kind == SH_SP ? a0 + 1 : a0;
        add(b, dx * rp);
        add(b + 1, dy * rp);
        add(b + 2, dz * rp);
      }
    } else {
      const double s = M<double>::dist(r2);
      double v = 0.0;
      for (int k = 0; k < np; ++k) {
        double sp = 1.0;
        for (int q = 0; q < sh.pw(k); ++q) sp *= s;
        v += S.coef_s[p0 + k] * sp * prim_e(S, p0 + k, s);
      }
      add(a0, v);
    }
  });
}

// One electron's Jastrow sums over the other electrons of its walker and
// the nuclei, and its share of the potential.
struct PairSums {
  double u_ee, u_en;        // ln J terms (e-e: both ends of a pair count it)
  double gx, gy, gz, lap;   // grad and sum of u'' + 2u'/r
  double sq;                // sum of u'^2 over e-e pairs
  double v;                 // 1/2 sum 1/r_ij - sum Z/r
};

template <int NU, int ND, class Bs, class Js, class Lds>
__device__ __forceinline__ PairSums group_pairs(const DevSys<double>& S, const Lds& L, int grp, int g, int sp, double x,
                                                double y, double z) {
  constexpr int N = NU + ND;
  PairSums P{};
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const double dx = x - L.xyz[grp][j][0], dy = y - L.xyz[grp][j][1], dz = z - L.xyz[grp][j][2];
    double r, ir, u1, lp;
    M<double>::dist_inv(dx * dx + dy * dy + dz * dz, r, ir);
    const bool same = (j < NU) == (sp == 0);
    uee_d<double, Js>(S, r, ir, same, u1, lp);
    const double u = uee_val<double, Js>(S, r, same) + S.cst_ee;
    const bool other = j != g, ok = other && r >= 1e-10;
    const double f = ok ? u1 * ir : 0.0;
    P.u_ee += other ? u : 0.0;
    P.gx += f * dx;
    P.gy += f * dy;
    P.gz += f * dz;
    P.lap += ok ? lp : 0.0;
    P.sq += ok ? u1 * u1 : 0.0;
    P.v += other ? 0.5 * ir : 0.0;
  }
  const bool en_on = S.en_on;
  Bs::nuclei(S, [&](int I) {
    const double dx = x - S.nuc[I][0], dy = y - S.nuc[I][1], dz = z - S.nuc[I][2];
    double r, ir;
    M<double>::dist_inv(dx * dx + dy * dy + dz * dz, r, ir);
    P.v -= S.Z[I] * ir;
    if (en_on) {
      double u1, lp;
      uen_d<double, Js>(S, r, ir, I, u1, lp);
      P.u_en += uen_val<double, Js>(S, r, I);
      const bool ok = r >= 1e-10;
      const double f = ok ? u1 * ir : 0.0;
      P.gx += f * dx;
      P.gy += f * dy;
      P.gz += f * dz;
      P.lap += ok ? lp : 0.0;
    }
  });
  return P;
}

// -1/2 lap psi / psi of one electron plus its potential share, from the
// determinant terms of its weights and its pair sums (electron_terms);
// on_shell as det_terms_w, gd receives grad D / D and lap the Laplacian
template <class Bs, class Wgt, class OnShell>
__device__ __forceinline__ double group_energy(const DevSys<double>& S, double x, double y, double z, Wgt wgt,
                                               const PairSums& P, OnShell on_shell, double gd[3], double& lap) {
  double ld;
  det_terms_w<double, Wgt, OnShell, Bs>(S, x, y, z, wgt, gd[0], gd[1], gd[2], ld, on_shell);
  const double gs = S.grad_scale;
  const double lj = (S.flags & F_J2_LAP_QUIRK) ? P.lap + P.sq : P.lap + P.gx * P.gx + P.gy * P.gy + P.gz * P.gz;
  lap = ld + lj + 2.0 * gs * (gd[0] * P.gx + gd[1] * P.gy + gd[2] * P.gz);
  return -0.5 * lap + P.v;
}
template <class Bs, class Wgt>
__device__ __forceinline__ double group_energy(const DevSys<double>& S, double x, double y, double z, Wgt wgt,
                                               const PairSums& P) {
  double gd[3], lap;
  return group_energy<Bs>(S, x, y, z, wgt, P, NoShell{}, gd, lap);
}

// Both sectors' Slater matrices inverted at once, one row (electron) per
// lane: a[m] = phi_m(r_slot) in, Gauss-Jordan in place without row
// interchanges (each column's pivot is its largest |a| over the rows not
// used yet), rows passed between lanes by permutes.  Out: col[m] =
// (A^-1)_{m, slot}, ln|det| and sign of the lane's sector (ln 0 = -inf and
// sign 0 when a pivot is exactly zero; col is then not finite).
template <int NU, int ND, class Lds>
__device__ __forceinline__ void group_invert(Lds& L, int lane, int base, int slot, int ns, double* a, double* col,
                                             double& la, double& sg) {
  constexpr int NS = NU > ND ? NU : ND;
  constexpr bool even = NU == ND;  // every lane's sector has NS rows
  int piv[NS], mine = 0;
  bool used = false, sing = false;
  LogAcc<double> det;
  double dummy = 0.0;
  sg = 1.0;
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    const bool act = even || c < ns;
    const double v = used ? -1.0 : pivot_mag(a[c]);
    double best = -2.0;
    int p = 0;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const double w = __shfl(v, (base + i) & 63, 64);
      if ((even || i < ns) && w > best) {
        best = w;
        p = i;
      }
    }
    double pr[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) pr[j] = __shfl(a[j], base + p, 64);
    piv[c] = p;
    if (act) {
      const double pv = pr[c];
      if (best == 0.0) sing = true;
      const double ip = 1.0 / pv;
      const bool me = slot == p;
      const double f = me ? 0.0 : a[c];
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const double q = pr[j] * ip;
        if (j != c) a[j] = me ? q : a[j] - f * q;
      }
      a[c] = me ? ip : -f * ip;
      if (me) {
        used = true;
        mine = c;
      }
      det.add(dummy, pv);
      if (pv < 0.0) sg = -sg;
    }
  }
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = i + 1; j < NS; ++j)
      if ((even || j < ns) && piv[i] > piv[j]) sg = -sg;
  la = 0.0;
  det.fold(la);
  if (sing) {
    la = -INFINITY;
    sg = 0.0;
  }
  // (A^-1)_{m, slot} = a of lane piv[m], entry `mine`
#pragma unroll
  for (int j = 0; j < NS; ++j) L.row[lane][j] = a[j];
  wave_sync();
#pragma unroll
  for (int m = 0; m < NS; ++m) col[m] = (even || m < ns) ? L.row[base + piv[m]][mine] : 0.0;
  wave_sync();
}

}  // namespace qmc
