// qmc_group.hip -- the lane-group engine's kernels.
#include "qmc_group.hpp"

#include "qmc_group_dev.hpp"
#include "qmc_pair_terms.hpp"

namespace qmc {

// ---------------------------------------------------------------------------
// All-electron Metropolis (MCMCSimulation::metropolis_step, vmc.rs:95-119):
// every electron moved at once, ln|psi| recomputed, E_L recomputed on
// acceptance and cached otherwise.  Positions are kept in T; everything
// after the proposal runs in FP64 (the state's own ln|psi| always did).
//
// A step is one long serial chain, so with one walker per lane it was the
// latency of that chain that counted, and the whole walker (both inverses,
// all positions) had to fit one lane: 256 + 256 registers with spills.
// With one electron per lane the proposal, the orbitals, the Slater rows
// and the Jastrow sums of a walker run side by side, a lane holds one row of
// its sector's inverse, and a launch has G times the wavefronts.  Measured in
// FP64, us per step, before / now: H2 7.6 / 3.1 at 20 walkers and 8.7 / 5.3
// at 65,536; Li 22 / 5.0 at 16,384; CH4 STO-3G 137 / 18 at 8,192, 148 / 129
// at 65,536; CH4 6-31G 203 / 145 at 65,536.  Up to one
// wavefront per SIMD a step takes the time of one wavefront's own
// instructions: 66 % of its cycles issue vector instructions (970 a step for
// H2 at 4,096 walkers, 3,270 for CH4 6-31G at 20), 20 to 22 % wait for LDS,
// scalar loads and permutes, the rest are dependences.  The compiled CH4
// instances take 256 vector registers and 63 to 186 accumulator ones as
// overflow, and keep 260 to 380 scalar values in vector lanes (6-31G most);
// no instance uses scratch.
// ---------------------------------------------------------------------------
template <int NU, int ND, class Bs, class Js, class T>
__global__ void __launch_bounds__(64) group_ae_kernel(const DevSys<double>* __restrict__ Sp, EnsView<T> E,
                                                      SweepArgs A, double* __restrict__ partial,
                                                      double* __restrict__ el_trace) {
  using Sh = GroupShape<NU, ND, Bs>;
  constexpr int N = Sh::N, NS = Sh::NS, G = Sh::G, WPB = Sh::WPB;
  __shared__ typename Sh::Lds L;
  const DevSys<double>& S = *Sp;
  const int64_t blk = (int64_t)blockIdx.y * gridDim.x + blockIdx.x, nblk = (E.W + WPB - 1) / WPB;
  if (blk >= nblk) return;
  group_fill_mo<NU, ND, Bs>(S, L);
  const int lane = threadIdx.x, grp = lane / G, g = lane % G;
  const bool elec = g < N;
  const int sp = elec && g >= NU ? 1 : 0, slot = elec ? g - (sp ? NU : 0) : 0, ns = sp ? ND : NU;
  const int base = grp * G + (sp ? NU : 0);  // first lane of this lane's sector
  const int e = S.sector_elec[sp][slot];
  const int64_t w = blk * WPB + grp;
  const bool live = w < E.W;
  const int64_t wl = live ? w : E.W - 1;  // walkers past the end shadow the last one and write nothing
  T r[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = E.pos[(e * 3 + c) * E.ld + wl];
  double ldet = E.logdet[wl], ju = E.ju[wl], sgn = E.sign[wl], el = E.eloc[wl];
  const uint32_t k0 = (uint32_t)A.seed, k1 = (uint32_t)(A.seed >> 32);
  const uint32_t wid = (uint32_t)(A.walker0 + wl);
  const T sigma = (T)A.step_size;
  const double* mo = &L.mo[0][sp][0];
  for (int s = 0; s < A.n_steps; ++s) {
    const uint32_t step = A.step0 + (uint32_t)s;
    T z[3], q[3];
    Rng<T>::normals3(philox(wid, step, (uint32_t)e, RNG_ALL, k0, k1), z);
#pragma unroll
    for (int c = 0; c < 3; ++c) q[c] = r[c] + sigma * z[c];
    const double x = (double)q[0], y = (double)q[1], zz = (double)q[2];
    if (elec) {
      L.xyz[grp][g][0] = x;
      L.xyz[grp][g][1] = y;
      L.xyz[grp][g][2] = zz;
    }
    wave_sync();
    double a[NS], col[NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) a[m] = 0.0;
    ao_values<Bs>(S, x, y, zz, [&](int ao, double v) {
#pragma unroll
      for (int m = 0; m < NS; ++m) a[m] += mo[ao * 2 * Sh::NSP + m] * v;
    });
    const PairSums P = group_pairs<NU, ND, Bs, Js>(S, L, grp, g, sp, x, y, zz);
    double la, sg;
    group_invert<NU, ND>(L, lane, base, slot, ns, a, col, la, sg);
    if constexpr (ND > 0) {
      la = __shfl(la, grp * G, 64) + __shfl(la, grp * G + NU, 64);
      sg = __shfl(sg, grp * G, 64) * __shfl(sg, grp * G + NU, 64);
    }
    const double jun = gsum<G>(elec ? 0.5 * P.u_ee + P.u_en : 0.0);
    const double U = u01d(philox(wid, step, (uint32_t)N, RNG_ALL, k0, k1).x);
    const bool acc = U < M<double>::ex(2.0 * ((la + jun) - (ldet + ju)));
    if (__any(acc)) {
      auto wgt = [&](int ao) {
        double v = 0.0;
#pragma unroll
        for (int m = 0; m < NS; ++m) v += mo[ao * 2 * Sh::NSP + m] * col[m];
        return v;
      };
      const double ei = group_energy<Bs>(S, x, y, zz, wgt, P);
      const double en = gsum<G>(elec ? ei : 0.0) + S.vnn;
      if (acc) {
#pragma unroll
        for (int c = 0; c < 3; ++c) r[c] = q[c];
        ldet = la;
        ju = jun;
        sgn = sg;
        el = en;
      }
    }
    const bool head = live && g == 0;
    if (el_trace && head) el_trace[(int64_t)s * A.trace_ld + w] = el;
    const double e1 = wsum(head ? el : 0.0), e2 = wsum(head ? el * el : 0.0), na = wsum(head && acc ? 1.0 : 0.0);
    if (lane == 0) {
      double* p = partial + ((int64_t)s * nblk + blk) * 3;
      p[0] = e1;
      p[1] = e2;
      p[2] = na;
    }
  }
  if (live && elec) {
#pragma unroll
    for (int c = 0; c < 3; ++c) E.pos[(e * 3 + c) * E.ld + w] = r[c];
  }
  if (live && g == 0) {
    E.logdet[w] = ldet;
    E.ju[w] = ju;
    E.sign[w] = sgn;
    E.eloc[w] = el;
  }
}

// ---------------------------------------------------------------------------
// Single-electron Metropolis (sector_moves) and drift-diffusion
// (sector_moves_dd) sweeps in FP64.  Lane g owns electron g and its column of
// the inverse; within a move the lanes take
//   the primitives g, g + G, ... of the basis, whose coefficients against the
//     sector's MOs they hold in registers: MO values (and, weighted by the
//     mover's column, the quantum force) from one sum over the group
//   the mover's partners: electron g, or a nucleus on the lanes past the
//     electrons
//   the Sherman-Morrison update of their own column.
// The random numbers of a sweep are drawn by all electrons' lanes at once.
// ---------------------------------------------------------------------------
template <class Bd>
struct GroupBasis {
  static constexpr int np = bd_p0<Bd>(Bd::n_shell);
  static constexpr bool gauss = Bd::kind[0] <= SH_P1;
  static constexpr bool any_p() {
    for (int i = 0; i < Bd::n_shell; ++i)
      if (Bd::kind[i] == SH_SP) return true;
    return false;
  }
  static constexpr bool supported() {  // s / sp Gaussians, or Slater functions of power up to 3
    for (int i = 0; i < Bd::n_shell; ++i) {
      const bool g = Bd::kind[i] <= SH_P1;
      if (g != gauss || (g && Bd::kind[i] != SH_S && Bd::kind[i] != SH_SP)) return false;
    }
    for (int i = 0; i < np; ++i)
      if (Bd::pw[i] > 3) return false;
    return true;
  }
};

template <class Bd, bool DD>
__global__ void __launch_bounds__(64) group_sweep_kernel(const DevSys<double>* __restrict__ Sp, EnsView<double> E,
                                                         SweepArgs A, double* __restrict__ partial,
                                                         double* __restrict__ el_trace) {
  constexpr int NU = Bd::nu, ND = Bd::nd;
  using Bs = CtBasis<Bd>;
  using Sh = GroupShape<NU, ND, Bs>;
  using GB = GroupBasis<Bd>;
  static_assert(GB::supported(), "primitive kinds of the lane-group sweeps");
  constexpr int N = Sh::N, NS = Sh::NS, G = Sh::G, WPB = Sh::WPB, MN = Bd::n_nuc;
  constexpr int RN = (GB::np + G - 1) / G;  // primitives per lane
  constexpr int PT = (N + MN + G - 1) / G;  // partners per lane
  constexpr bool HP = GB::any_p();
  __shared__ typename Sh::Lds L;
  const DevSys<double>& S = *Sp;
  const int lane = threadIdx.x, grp = lane / G, g = lane % G;
  const int64_t Wn = E.n_live ? *E.n_live : E.W;
  if ((int64_t)blockIdx.x * WPB >= Wn) {  // past a branching population's live walkers: zero partial sums only
    if (lane == 0)
      for (int s = 0; s < A.n_steps; ++s)
        for (int q = 0; q < 3; ++q) partial[((int64_t)s * gridDim.x + blockIdx.x) * 3 + q] = 0.0;
    return;
  }
  group_fill_mo<NU, ND, Bs>(S, L);
  const bool elec = g < N;
  const int sp = elec && g >= NU ? 1 : 0, slot = elec ? g - (sp ? NU : 0) : 0, ns = sp ? ND : NU;
  const int e = S.sector_elec[sp][slot];
  const int64_t w = (int64_t)blockIdx.x * WPB + grp;
  const bool live = w < Wn;
  const int64_t wl = live ? w : Wn - 1;  // walkers past the end shadow the last one and write nothing
  // this lane's electron and inverse column
  double r[3], col[NS];
#pragma unroll
  for (int c = 0; c < 3; ++c) r[c] = E.pos[(e * 3 + c) * E.ld + wl];
#pragma unroll
  for (int m = 0; m < NS; ++m)
    col[m] = elec && m < ns ? E.ainv[((sp ? NU * NU : 0) + m * ns + slot) * E.ld + wl] : 0.0;
  double ldet = E.logdet[wl], ju = E.ju[wl], sgn = E.sign[wl], el = 0.0;
  // this lane's primitives
  double pex[RN], pc[RN][3], pcs[RN], pcp[RN];
  int pa0[RN], ppw[RN];
  bool psp[RN];
#pragma unroll
  for (int t = 0; t < RN; ++t) {
    const int idx = t * G + g;
    pex[t] = pcs[t] = pcp[t] = 0.0;
    pc[t][0] = pc[t][1] = pc[t][2] = 0.0;
    pa0[t] = ppw[t] = 0;
    psp[t] = false;
    if (idx < GB::np) {
      pex[t] = S.prim_exp[idx];
      pcs[t] = S.coef_s[idx];
      if (HP) pcp[t] = S.coef_p[idx];
      ppw[t] = S.prim_pow[idx];
      static_for<0, Bd::n_shell>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if (idx >= bd_p0<Bd>(i) && idx < bd_p0<Bd>(i) + Bd::nprim[i]) {
          pa0[t] = bd_a0<Bd>(i);
          psp[t] = Bd::kind[i] == SH_SP;
#pragma unroll
          for (int c = 0; c < 3; ++c) pc[t][c] = S.nuc[Bd::center[i]][c];
        }
      });
    }
  }
  // this lane's partners: its own electron, then nuclei
  double px[PT][3], pa[PT], pb[PT];
  bool pn[PT];  // a nucleus with an e-n Jastrow term
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    const int i = t * G + g - N;
    pn[t] = i >= 0 && i < MN && S.en_on;
    const int I = i >= 0 && i < MN ? i : 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) px[t][c] = S.nuc[I][c];
    pa[t] = pn[t] ? -S.Z[I] : 0.0;
    pb[t] = S.b_en;
  }
  const double b_ee = S.b_ee, a_para = S.a_para, a_anti = S.a_anti, gs = S.grad_scale;
  const uint32_t k0 = (uint32_t)A.seed, k1 = (uint32_t)(A.seed >> 32);
  const uint32_t wid = (uint32_t)(A.walker0 + wl);
  const uint32_t step0 = DD && A.step0_dev ? *A.step0_dev : A.step0;
  const double sigma = A.step_size;
  const double s2t = sqrt(2.0 * sigma), i4t = 0.25 / sigma;  // drift-diffusion: step_size is the time step
  if (elec) {
#pragma unroll
    for (int c = 0; c < 3; ++c) L.xyz[grp][g][c] = r[c];
  }
  const double* mo = &L.mo[0][sp][0];
  for (int s = 0; s < A.n_steps; ++s) {
    const uint32_t step = step0 + (uint32_t)s;
    {
      double z[3], U;
      Rng<double>::move(philox(wid, step, (uint32_t)e, DD ? RNG_DRIFT : RNG_SINGLE, k0, k1), z, U);
      if (elec) {
#pragma unroll
        for (int c = 0; c < 3; ++c) L.prop[grp][g][c] = DD ? z[c] : r[c] + sigma * z[c];
        L.prop[grp][g][3] = U;
      }
      wave_sync();
    }
    int acc = 0;
    LogAcc<double> lacc;
    auto sector = [&](auto na_tag, int msp) {
      constexpr int NA = decltype(na_tag)::value;
      // the lane's primitives against the sector's MOs
      double ks[RN][NS], kx[HP ? RN : 1][NS][3];
#pragma unroll
      for (int t = 0; t < RN; ++t)
#pragma unroll
        for (int m = 0; m < NA; ++m) {
          const double* c = &L.mo[pa0[t]][msp][m];
          ks[t][m] = pcs[t] * c[0];
          if constexpr (HP) {
#pragma unroll
            for (int q = 0; q < 3; ++q) kx[t][m][q] = psp[t] ? pcp[t] * c[psp[t] ? (q + 1) * 2 * Sh::NSP : 0] : 0.0;
          }
        }
      const double ape = sp == msp ? a_para : a_anti;  // the lane's electron with the mover
#pragma unroll 1
      for (int k = 0; k < NA; ++k) {
        const int ml = k + (msp ? NU : 0);  // the mover's lane in its group
        const bool mover = g == ml;
        double ak[NA];
#pragma unroll
        for (int m = 0; m < NA; ++m) ak[m] = __shfl(col[m], grp * G + ml, 64);
        const double ox = L.xyz[grp][ml][0], oy = L.xyz[grp][ml][1], oz = L.xyz[grp][ml][2];
        const double U = L.prop[grp][ml][3];
        double nx = L.prop[grp][ml][0], ny = L.prop[grp][ml][1], nz = L.prop[grp][ml][2];
        double phi[NA];
        // one primitive at d: e (its radial factor without the coefficient)
        auto prim = [&](int t, double x, double y, double zz, double& dx, double& dy, double& dz, double& sr) {
          dx = x - pc[t][0];
          dy = y - pc[t][1];
          dz = zz - pc[t][2];
          const double r2 = dx * dx + dy * dy + dz * dz;
          if constexpr (GB::gauss) {
            return M<double>::exn(-pex[t] * r2);
          } else {
            sr = M<double>::dist(r2);
            const double q = ppw[t] == 0 ? 1.0 : (ppw[t] == 1 ? sr : (ppw[t] == 2 ? sr * sr : sr * sr * sr));
            return q * M<double>::exn(-pex[t] * sr);
          }
        };
        // force weights: the value R and gradient of sum_m phi_m ak_m at a point
        auto force = [&](double x, double y, double zz, double v[4], bool values) {
          v[0] = v[1] = v[2] = v[3] = 0.0;
#pragma unroll
          for (int t = 0; t < RN; ++t) {
            double dx, dy, dz, sr = 0.0;
            const double ee = prim(t, x, y, zz, dx, dy, dz, sr);
            double ws = 0.0, wx = 0.0, wy = 0.0, wz = 0.0;
#pragma unroll
            for (int m = 0; m < NA; ++m) {
              ws += ks[t][m] * ak[m];
              if constexpr (HP) {
                wx += kx[t][m][0] * ak[m];
                wy += kx[t][m][1] * ak[m];
                wz += kx[t][m][2] * ak[m];
              }
            }
            if (values) {
#pragma unroll
              for (int m = 0; m < NA; ++m) {
                double c = ks[t][m];
                if constexpr (HP) c += kx[t][m][0] * dx + kx[t][m][1] * dy + kx[t][m][2] * dz;
                phi[m] += ee * c;
              }
            }
            const double val = ee * (ws + (wx * dx + wy * dy + wz * dz));
            double q;
            if constexpr (GB::gauss)
              q = -2.0 * pex[t] * val;
            else  // s^p e^{-zeta s}: (p / s - zeta) / s, zero at the centre
              q = sr > 0.0 ? val * ((double)ppw[t] / sr - pex[t]) / sr : 0.0;
            v[0] += val;
            v[1] += q * dx + ee * wx;
            v[2] += q * dy + ee * wy;
            v[3] += q * dz + ee * wz;
          }
        };
        // the lane's Jastrow partners at a point: value and, for the force, gradient
        auto partners = [&](double x, double y, double zz, double u[4]) {
          u[0] = u[1] = u[2] = u[3] = 0.0;
#pragma unroll
          for (int t = 0; t < PT; ++t) {
            const bool pe = t == 0 && elec, on = pe ? !mover : pn[t];
            const double qx = pe ? r[0] : px[t][0], qy = pe ? r[1] : px[t][1], qz = pe ? r[2] : px[t][2];
            const double ca = pe ? ape : pa[t], cb = pe ? b_ee : pb[t];
            const double dx = x - qx, dy = y - qy, dz = zz - qz;
            double rr, ir;
            M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
            const double iD = M<double>::rcp(1.0 + cb * rr);
            u[0] += on ? ca * rr * iD : 0.0;
            if constexpr (DD) {
              const double f = on && rr >= 1e-10 ? gs * ca * iD * iD * ir : 0.0;
              u[1] += f * dx;
              u[2] += f * dy;
              u[3] += f * dz;
            }
          }
        };
        double R, du, gg = 0.0, uo[4], un[4];
#pragma unroll
        for (int m = 0; m < NA; ++m) phi[m] = 0.0;
        partners(ox, oy, oz, uo);
        if constexpr (DD) {
          double fo[4], fn[4], d0[3], d1[3];
          force(ox, oy, oz, fo, false);
          const double fx = gsum<G>(fo[1] + uo[1]), fy = gsum<G>(fo[2] + uo[2]), fz = gsum<G>(fo[3] + uo[3]);
          cap_drift(2.0 * fx, 2.0 * fy, 2.0 * fz, sigma, A.max_drift, d0);
          nx = ox + d0[0] + s2t * nx;
          ny = oy + d0[1] + s2t * ny;
          nz = oz + d0[2] + s2t * nz;
          force(nx, ny, nz, fn, true);
          partners(nx, ny, nz, un);
          R = gsum<G>(fn[0]);
          const double iR = M<double>::rcp(R);
          const double hx = gsum<G>(fn[1] * iR + un[1]), hy = gsum<G>(fn[2] * iR + un[2]),
                       hz = gsum<G>(fn[3] * iR + un[3]);
          cap_drift(2.0 * hx, 2.0 * hy, 2.0 * hz, sigma, A.max_drift, d1);
          const double a0 = nx - ox - d0[0], a1 = ny - oy - d0[1], a2 = nz - oz - d0[2];
          const double b0 = ox - nx - d1[0], b1 = oy - ny - d1[1], b2 = oz - nz - d1[2];
          gg = ((a0 * a0 + a1 * a1 + a2 * a2) - (b0 * b0 + b1 * b1 + b2 * b2)) * i4t;
#pragma unroll
          for (int m = 0; m < NA; ++m) phi[m] = gsum<G>(phi[m]);
        } else {
#pragma unroll
          for (int t = 0; t < RN; ++t) {
            double dx, dy, dz, sr = 0.0;
            const double ee = prim(t, nx, ny, nz, dx, dy, dz, sr);
#pragma unroll
            for (int m = 0; m < NA; ++m) {
              double c = ks[t][m];
              if constexpr (HP) c += kx[t][m][0] * dx + kx[t][m][1] * dy + kx[t][m][2] * dz;
              phi[m] += ee * c;
            }
          }
          partners(nx, ny, nz, un);
          R = 0.0;
#pragma unroll
          for (int m = 0; m < NA; ++m) {
            phi[m] = gsum<G>(phi[m]);
            R += phi[m] * ak[m];
          }
        }
        du = gsum<G>(un[0] - uo[0]);
        const double p = R * R * M<double>::ex(2.0 * du + gg);
        if (U < p) {
          const double iR = M<double>::rcp(R);
          if (elec && sp == msp) {
            double wj = 0.0;
#pragma unroll
            for (int m = 0; m < NA; ++m) wj += phi[m] * col[m];
            const double f = wj * iR;
#pragma unroll
            for (int m = 0; m < NA; ++m) col[m] = mover ? ak[m] * iR : col[m] - ak[m] * f;
          }
          if (mover) {
            r[0] = nx;
            r[1] = ny;
            r[2] = nz;
            L.xyz[grp][ml][0] = nx;
            L.xyz[grp][ml][1] = ny;
            L.xyz[grp][ml][2] = nz;
          }
          lacc.add(ldet, R);
          if (R < 0.0) sgn = -sgn;
          ju += du;
          ++acc;
        }
      }
    };
    sector(std::integral_constant<int, NU>{}, 0);
    if constexpr (ND > 0) sector(std::integral_constant<int, ND>{}, 1);
    lacc.fold(ldet);
    wave_sync();
    const PairSums P = group_pairs<NU, ND, Bs, JsNone>(S, L, grp, g, sp, r[0], r[1], r[2]);
    auto wgt = [&](int ao) {
      double v = 0.0;
#pragma unroll
      for (int m = 0; m < NS; ++m) v += mo[ao * 2 * Sh::NSP + m] * col[m];
      return v;
    };
    const double ei = group_energy<Bs>(S, r[0], r[1], r[2], wgt, P);
    el = gsum<G>(elec ? ei : 0.0) + S.vnn;
    const bool head = live && g == 0;
    if (el_trace && head) el_trace[(int64_t)s * A.trace_ld + w] = el;
    const double e1 = wsum(head ? el : 0.0), e2 = wsum(head ? el * el : 0.0), na = wsum(head ? (double)acc : 0.0);
    if (lane == 0) {
      double* q = partial + ((int64_t)s * gridDim.x + blockIdx.x) * 3;
      q[0] = e1;
      q[1] = e2;
      q[2] = na;
    }
  }
  if (live && elec) {
#pragma unroll
    for (int c = 0; c < 3; ++c) E.pos[(e * 3 + c) * E.ld + w] = r[c];
#pragma unroll
    for (int m = 0; m < NS; ++m)
      if (m < ns) E.ainv[((sp ? NU * NU : 0) + m * ns + slot) * E.ld + w] = col[m];
  }
  if (live && g == 0) {
    E.logdet[w] = ldet;
    E.ju[w] = ju;
    E.sign[w] = sgn;
    E.eloc[w] = el;
  }
}

// ---------------------------------------------------------------------------
// The derivative matrix (derivs_kernel's columns) with one electron per
// lane: E_L, O, dE_L/dp, Omega and the electron part of the HF force in
// FP64.  Omega and the force are summed per nucleus in registers, then over
// the group.
// ---------------------------------------------------------------------------
template <class Bd>
__global__ void __launch_bounds__(64) group_derivs_kernel(const DevSys<double>* __restrict__ Sp, DerivArgs A) {
  constexpr int NU = Bd::nu, ND = Bd::nd;
  using Bs = CtBasis<Bd>;
  using Sh = GroupShape<NU, ND, Bs>;
  constexpr int N = Sh::N, NS = Sh::NS, G = Sh::G, WPB = Sh::WPB, MN = Bd::n_nuc, QM = 2 * 4 + 6 * MN + 2;
  __shared__ typename Sh::Lds L;
  __shared__ double grad[WPB][N][3];      // d ln psi / d r
  __shared__ double feat[WPB][QM];
  const DevSys<double>& S = *Sp;
  group_fill_mo<NU, ND, Bs>(S, L);
  const int lane = threadIdx.x, grp = lane / G, g = lane % G;
  const bool elec = g < N;
  const int sp = elec && g >= NU ? 1 : 0, slot = elec ? g - (sp ? NU : 0) : 0, ns = sp ? ND : NU;
  const int base = grp * G + (sp ? NU : 0), e = S.sector_elec[sp][slot];
  const int64_t w = (int64_t)blockIdx.x * WPB + grp;
  const int64_t wl = w < A.W ? w : A.W - 1;  // walkers past the end shadow the last one and write nothing
  double r[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int q = 3 * e + c;
    r[c] = A.pos_aos ? A.pos_aos[wl * 3 * N + q] : (A.pos64 ? A.pos64[q * A.ld + wl] : (double)A.pos32[q * A.ld + wl]);
    if (elec) L.xyz[grp][g][c] = r[c];
  }
  wave_sync();
  const double x = r[0], y = r[1], z = r[2];
  const double* mo = &L.mo[0][sp][0];
  double a[NS], col[NS], la, sg;
#pragma unroll
  for (int m = 0; m < NS; ++m) a[m] = 0.0;
  ao_values<Bs>(S, x, y, z, [&](int ao, double v) {
#pragma unroll
    for (int m = 0; m < NS; ++m) a[m] += mo[ao * 2 * Sh::NSP + m] * v;
  });
  group_invert<NU, ND>(L, lane, base, slot, ns, a, col, la, sg);
#pragma unroll
  for (int m = 0; m < NS; ++m) col[m] = sg == 0.0 ? (m == slot ? 1.0 : 0.0) : col[m];  // singular: identity
  double om[MN][3], f[MN][3];
#pragma unroll
  for (int I = 0; I < MN; ++I)
#pragma unroll
    for (int c = 0; c < 3; ++c) om[I][c] = f[I][c] = 0.0;
  const PairSums P = group_pairs<NU, ND, Bs, JsNone>(S, L, grp, g, sp, x, y, z);
  auto wgt = [&](int ao) {
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < NS; ++m) v += mo[ao * 2 * Sh::NSP + m] * col[m];
    return v;
  };
  auto on_shell = [&](int c, double sx, double sy, double sz) {
    om[c][0] -= sx;
    om[c][1] -= sy;
    om[c][2] -= sz;
  };
  double gd[3], lap;
  const double ei = group_energy<Bs>(S, x, y, z, wgt, P, on_shell, gd, lap);
  Bs::nuclei(S, [&](int I) {
    const double dx = x - S.nuc[I][0], dy = y - S.nuc[I][1], dz = z - S.nuc[I][2];
    double rr, ir;
    M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
    const double f3 = rr > 1e-10 ? S.Z[I] * ir * ir * ir : 0.0;  // methane.rs:1253
    f[I][0] += f3 * dx;
    f[I][1] += f3 * dy;
    f[I][2] += f3 * dz;
    if (S.en_on) {  // d u_en / d R_I = -u1 (r_i - R_I) / r (methane.rs:1071-1090)
      double u1, lp;
      uen_d<double, JsNone>(S, rr, ir, I, u1, lp);
      const double q = rr >= 1e-10 ? u1 * ir : 0.0;
      om[I][0] -= q * dx;
      om[I][1] -= q * dy;
      om[I][2] -= q * dz;
    }
  });
  double O[4] = {0.0, 0.0, 0.0, 0.0}, dE[4] = {0.0, 0.0, 0.0, 0.0};
  if (A.P > 0) {  // Pade: [b_ee, b_en, a_anti, a_para], every pair once (offset d around the walker's electrons)
    const double gi[3] = {gd[0] + P.gx, gd[1] + P.gy, gd[2] + P.gz};
    if (elec) {
#pragma unroll
      for (int c = 0; c < 3; ++c) grad[grp][g][c] = gi[c];
    }
    wave_sync();
    for (int d = 1; 2 * d <= N; ++d) {
      const int j = g + d < N ? g + d : g + d - N, jc = j < N ? j : 0;  // lanes past the electrons read slot 0
      const bool on = elec && (2 * d < N || g < d);
      const bool same = (jc >= NU) == (sp == 1);
      const double dx = x - L.xyz[grp][jc][0], dy = y - L.xyz[grp][jc][1], dz = z - L.xyz[grp][jc][2];
      double rr, ir;
      M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
      PairDerivs<double> pd;
      pd.init(rr, S.b_ee, same ? S.a_para : S.a_anti, 0, nullptr);
      const bool far = on && rr >= 1e-10;
      const double dlt = (gi[0] - grad[grp][jc][0]) * (dx * ir) + (gi[1] - grad[grp][jc][1]) * (dy * ir) +
                         (gi[2] - grad[grp][jc][2]) * (dz * ir);
      double du1, dl;
      pd.d_b(rr, ir, S.b_ee, du1, dl);
      O[0] -= on ? pd.A1 * pd.x * pd.x : 0.0;
      dE[0] -= far ? dl + dlt * du1 : 0.0;
      pd.d_a(ir, S.b_ee, du1, dl);
      const double oa = on ? pd.x : 0.0, da = far ? dl + dlt * du1 : 0.0;
      O[2] += same ? 0.0 : oa;
      O[3] += same ? oa : 0.0;
      dE[2] -= same ? 0.0 : da;
      dE[3] -= same ? da : 0.0;
    }
    Bs::nuclei(S, [&](int I) {
      en_pair_terms(S, I, x - S.nuc[I][0], y - S.nuc[I][1], z - S.nuc[I][2], [&](int c) { return gi[c]; },
                    [&](int sl, double v) { O[1] += sl == 0 ? v : 0.0; },
                    [&](int sl, double v) { dE[1] += sl == 0 ? v : 0.0; });
    });
  }
  const DerivLayout Ly{A.P, A.M, N, A.Qp};
  const bool head = g == 0;
  auto put = [&](int q, double v) {
    v = gsum<G>(elec ? v : 0.0);
    if (head) feat[grp][q] = v;
  };
  if (A.P > 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      put(Ly.o(k), O[k]);
      put(Ly.de(k), dE[k]);
    }
  }
#pragma unroll
  for (int I = 0; I < MN; ++I)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      put(Ly.om(I, c), om[I][c]);
      put(Ly.f(I, c), f[I][c]);
    }
  put(Ly.e(), ei);
  if (head) {
    feat[grp][Ly.e()] += S.vnn;
    feat[grp][Ly.one()] = 1.0;
  }
  wave_sync();
  const int nq = Ly.f(MN, 0);
  for (int t = lane; t < A.Qp * WPB; t += 64) {  // the block's walkers in consecutive lanes
    const int q = t / WPB, k = t % WPB;
    const int64_t wk = (int64_t)blockIdx.x * WPB + k;
    if (wk < A.W) A.Y[(int64_t)q * A.ldy + wk] = q < nq ? feat[k][q] : 0.0;
  }
}

// ---------------------------------------------------------------------------
// qmc_evaluate with one electron per lane, in FP64 (eval_kernel's outputs).
// ---------------------------------------------------------------------------
template <class Bd>
__global__ void __launch_bounds__(64) group_eval_kernel(const DevSys<double>* __restrict__ Sp, int64_t W,
                                                        const double* __restrict__ pos, EvalOut O, int* singular_count) {
  constexpr int NU = Bd::nu, ND = Bd::nd;
  using Bs = CtBasis<Bd>;
  using Sh = GroupShape<NU, ND, Bs>;
  constexpr int N = Sh::N, NS = Sh::NS, G = Sh::G, WPB = Sh::WPB;
  __shared__ typename Sh::Lds L;
  const DevSys<double>& S = *Sp;
  group_fill_mo<NU, ND, Bs>(S, L);
  const int lane = threadIdx.x, grp = lane / G, g = lane % G;
  const bool elec = g < N;
  const int sp = elec && g >= NU ? 1 : 0, slot = elec ? g - (sp ? NU : 0) : 0, ns = sp ? ND : NU;
  const int base = grp * G + (sp ? NU : 0), e = S.sector_elec[sp][slot];
  const int64_t w = (int64_t)blockIdx.x * WPB + grp;
  const bool live = w < W;
  const int64_t wl = live ? w : W - 1;  // walkers past the end shadow the last one and write nothing
  const double x = pos[(wl * N + e) * 3], y = pos[(wl * N + e) * 3 + 1], z = pos[(wl * N + e) * 3 + 2];
  if (elec) {
    L.xyz[grp][g][0] = x;
    L.xyz[grp][g][1] = y;
    L.xyz[grp][g][2] = z;
  }
  wave_sync();
  const double* mo = &L.mo[0][sp][0];
  double a[NS], col[NS], la, sg;
#pragma unroll
  for (int m = 0; m < NS; ++m) a[m] = 0.0;
  ao_values<Bs>(S, x, y, z, [&](int ao, double v) {
#pragma unroll
    for (int m = 0; m < NS; ++m) a[m] += mo[ao * 2 * Sh::NSP + m] * v;
  });
  const PairSums P = group_pairs<NU, ND, Bs, JsNone>(S, L, grp, g, sp, x, y, z);
  group_invert<NU, ND>(L, lane, base, slot, ns, a, col, la, sg);
#pragma unroll
  for (int m = 0; m < NS; ++m) col[m] = sg == 0.0 ? (m == slot ? 1.0 : 0.0) : col[m];  // singular: identity
  if constexpr (ND > 0) {
    la = __shfl(la, grp * G, 64) + __shfl(la, grp * G + NU, 64);
    sg = __shfl(sg, grp * G, 64) * __shfl(sg, grp * G + NU, 64);
  }
  const double ju = gsum<G>(elec ? 0.5 * P.u_ee + P.u_en : 0.0);
  if (live && g == 0) {
    if (O.logabs) O.logabs[w] = la + ju;
    if (O.sign) O.sign[w] = sg;
    if (sg == 0.0 && singular_count) atomicAdd(singular_count, 1);
  }
  if (!O.eloc && !O.grad && !O.lap) return;
  auto wgt = [&](int ao) {
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < NS; ++m) v += mo[ao * 2 * Sh::NSP + m] * col[m];
    return v;
  };
  double gd[3], lap;
  const double ei = group_energy<Bs>(S, x, y, z, wgt, P, NoShell{}, gd, lap);
  const double el = gsum<G>(elec ? ei : 0.0) + S.vnn, gs = S.grad_scale;
  if (live && g == 0 && O.eloc) O.eloc[w] = el;
  if (live && elec) {
    if (O.grad) {
      double* q = O.grad + (w * N + e) * 3;
      q[0] = gd[0] + gs * P.gx;
      q[1] = gd[1] + gs * P.gy;
      q[2] = gd[2] + gs * P.gz;
    }
    if (O.lap) O.lap[w * N + e] = lap;
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int NU, int ND, class Bs, class Js, class T>
static hipError_t launch_ae(const void* Sd, EnsView<T> E, SweepArgs A, double* partial, double* trace, hipStream_t st) {
  // rows of at most 65,536 workgroups: a walker takes up to 16 lanes, and a
  // grid dimension holds fewer than 2^32 of them
  constexpr int wpb = GroupShape<NU, ND, Bs>::WPB;
  const int64_t nblk = (E.W + wpb - 1) / wpb, x = nblk < 65536 ? nblk : 65536;
  const dim3 grid((unsigned)x, (unsigned)((nblk + x - 1) / x));
  group_ae_kernel<NU, ND, Bs, Js, T><<<grid, 64, 0, st>>>((const DevSys<double>*)Sd, E, A, partial, trace);
  return hipGetLastError();
}

template <class Bd, bool DD>
static hipError_t launch_sweep(const void* Sd, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                               hipStream_t st) {
  constexpr int wpb = GroupShape<Bd::nu, Bd::nd, CtBasis<Bd>>::WPB;
  group_sweep_kernel<Bd, DD><<<(unsigned)((E.W + wpb - 1) / wpb), 64, 0, st>>>((const DevSys<double>*)Sd, E, A, partial,
                                                                             trace);
  return hipGetLastError();
}

template <class Bd>
static hipError_t launch_group_derivs(const void* Sd, DerivArgs A, hipStream_t st) {
  constexpr int wpb = GroupShape<Bd::nu, Bd::nd, CtBasis<Bd>>::WPB;
  if (A.M != Bd::n_nuc || (A.P != 0 && A.P != 4)) return hipErrorInvalidValue;
  group_derivs_kernel<Bd><<<(unsigned)((A.W + wpb - 1) / wpb), 64, 0, st>>>((const DevSys<double>*)Sd, A);
  return hipGetLastError();
}

template <class Bd>
static hipError_t launch_group_eval(const void* Sd, int64_t W, const double* pos, EvalOut O, int* sing,
                                    hipStream_t st) {
  constexpr int wpb = GroupShape<Bd::nu, Bd::nd, CtBasis<Bd>>::WPB;
  group_eval_kernel<Bd><<<(unsigned)((W + wpb - 1) / wpb), 64, 0, st>>>((const DevSys<double>*)Sd, W, pos, O, sing);
  return hipGetLastError();
}

template <int NU, int ND, class Bs, class JsFast>
static GroupOps make_group(bool (*match)(const DevSys<double>&)) {
  GroupOps o;
  o.nu = NU;
  o.nd = ND;
  o.wpb = GroupShape<NU, ND, Bs>::WPB;
  o.match = match;
  o.ae64 = &launch_ae<NU, ND, Bs, JsRt, double>;
  o.ae32 = &launch_ae<NU, ND, Bs, JsRt, float>;
  o.ae64_ns = &launch_ae<NU, ND, Bs, JsFast, double>;
  o.ae32_ns = &launch_ae<NU, ND, Bs, JsFast, float>;
  o.sweep64_ns = o.dd64_ns = nullptr;
  o.derivs_ns = nullptr;
  o.eval_ns = nullptr;
  o.w_sweep = o.w_deriv = o.w_eval = 0;
  return o;
}
template <class Bd>
static GroupOps compiled_group() {
  GroupOps o = make_group<Bd::nu, Bd::nd, CtBasis<Bd>, JsNone>(&basis_matches<Bd, double>);
  o.sweep64_ns = &launch_sweep<Bd, false>;
  o.dd64_ns = &launch_sweep<Bd, true>;
  o.derivs_ns = &launch_group_derivs<Bd>;
  o.eval_ns = &launch_group_eval<Bd>;
  // Walkers of one round, a wavefront on each of the 1,024 SIMDs: up to
  // there a launch takes the time of one walker's chain, which the lanes
  // shorten; past it the lanes that a group leaves idle (6 of 16 for CH4) and
  // the sums over it cost throughput, and one walker per lane overtakes.
  // Measured in FP64, us per sweep, lane groups against one walker per lane
  // (CH4: 6-31G): Metropolis H2 4.0 / 4.6 at 32,768 and 6.2 / 4.9 at 65,536
  // walkers, Li 6.4 / 8.7 at 16,384 and 9.7 / 9.0 at 32,768, CH4 16.7 / 83 at
  // 4,096, 64 / 85 at 16,384 and 128 / 85 at 32,768; drift-diffusion H2
  // 5.6 / 6.3 at 32,768, Li 12.0 / 13.4 at 16,384, CH4 25.6 / 120 at 4,096 and
  // 98 / 122 at 16,384.  Per derivative call: CH4 54 / 116 at 4,096, 71 / 118
  // at 8,192 and, mixed, 105 / 93 at 16,384; Li 34 / 36 at 16,384; H2 no
  // gain.  Per evaluation: CH4 37 / 117 at 4,096, 115 / 124 at 32,768 and
  // 202 / 147 at 65,536; H2 29 / 31 and Li 36 / 39 at 65,536.
  constexpr int G = GroupShape<Bd::nu, Bd::nd, CtBasis<Bd>>::G;
  const int64_t round = 1024 * o.wpb;
  o.w_sweep = (G == 16 ? 4 : 1) * round;
  o.w_deriv = (G == 16 ? 2 : G == 4 ? 1 : 0) * round;
  o.w_eval = G == 16 ? 8 * round : 65536;
  return o;
}
template <int NU, int ND>
static GroupOps generic_group() {
  return make_group<NU, ND, RtBasis, JsRt>(nullptr);
}

static const GroupOps kGroups[] = {
    compiled_group<BdH2>(),       compiled_group<BdLiSeeded>(), compiled_group<BdLiRef>(),
    compiled_group<BdCH4Sto3g>(), compiled_group<BdCH4631g>(),  generic_group<1, 0>(),
    generic_group<1, 1>(),        generic_group<2, 1>(),        generic_group<2, 2>(),
    generic_group<3, 2>(),        generic_group<3, 3>(),        generic_group<4, 4>(),
    generic_group<5, 5>(),
};

const GroupOps* find_group(const DevSys<double>& D, bool generic_only) {
  for (const auto& o : kGroups) {
    if (o.nu != D.n_up || o.nd != D.n_dn) continue;
    if (o.match && (generic_only || !o.match(D))) continue;
    return &o;
  }
  return nullptr;
}

}  // namespace qmc
