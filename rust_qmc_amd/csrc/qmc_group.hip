// qmc_group.hip -- the lane-group engine's kernels.
#include "qmc_group.hpp"

#include "qmc_group_dev.hpp"

namespace qmc {

// ---------------------------------------------------------------------------
// All-electron Metropolis (MCMCSimulation::metropolis_step, vmc.rs:95-119):
// every electron moved at once, ln|psi| recomputed, E_L recomputed on
// acceptance and cached otherwise.  Positions are kept in T; everything
// after the proposal runs in FP64 (the state's own ln|psi| always did).
//
// A step is one long serial chain, so with one walker per lane it is the
// latency of that chain that counts, and the whole walker (both inverses,
// all positions) has to fit one lane: 256 + 256 registers with spills.
// With one electron per lane the proposal, the orbitals, the Slater rows
// and the Jastrow sums of a walker run side by side, a lane holds one row of
// each inverse, and a launch has G times the wavefronts.
// ---------------------------------------------------------------------------
template <int NU, int ND, class Bs, class Js, class T>
__global__ void __launch_bounds__(64) group_ae_kernel(const DevSys<double>* __restrict__ Sp, EnsView<T> E,
                                                      SweepArgs A, double* __restrict__ partial,
                                                      double* __restrict__ el_trace) {
  using Sh = GroupShape<NU, ND, Bs>;
  constexpr int N = Sh::N, NS = Sh::NS, G = Sh::G, WPB = Sh::WPB;
  __shared__ typename Sh::Lds L;
  const DevSys<double>& S = *Sp;
  group_fill_mo<NU, ND, Bs>(S, L);
  const int lane = threadIdx.x, grp = lane / G, g = lane % G;
  const bool elec = g < N;
  const int sp = elec && g >= NU ? 1 : 0, slot = elec ? g - (sp ? NU : 0) : 0, ns = sp ? ND : NU;
  const int base = grp * G + (sp ? NU : 0);  // first lane of this lane's sector
  const int e = S.sector_elec[sp][slot];
  const int64_t w = (int64_t)blockIdx.x * WPB + grp;
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
      double* p = partial + ((int64_t)s * gridDim.x + blockIdx.x) * 3;
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
// launchers
// ---------------------------------------------------------------------------
template <int NU, int ND, class Bs, class Js, class T>
static hipError_t launch_ae(const void* Sd, EnsView<T> E, SweepArgs A, double* partial, double* trace, hipStream_t st) {
  constexpr int wpb = GroupShape<NU, ND, Bs>::WPB;
  group_ae_kernel<NU, ND, Bs, Js, T><<<(unsigned)((E.W + wpb - 1) / wpb), 64, 0, st>>>((const DevSys<double>*)Sd, E, A,
                                                                                     partial, trace);
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
  return o;
}
template <class Bd>
static GroupOps compiled_group() {
  return make_group<Bd::nu, Bd::nd, CtBasis<Bd>, JsNone>(&basis_matches<Bd, double>);
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
