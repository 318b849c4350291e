// qmc_terms.hip -- evaluation and derivatives of 21 + 21-electron systems.
//
// A workgroup of two wavefronts takes three walkers; wavefront s owns spin
// sector s of all three, lane 21 g + k electron k of walker g.  Every lane
// then does the same work on its own electron with the same (scalar) shell,
// coefficient and Jastrow parameters: its Slater row, one row of the
// Gauss-Jordan inversion, its AO derivatives against its inverse column and
// its Jastrow partners, with 63 of 64 lanes busy and nothing but the rows
// in transit, the positions and the sums over electrons in LDS.
//
// Measured for 8,192 benzene walkers, E_L with every derivative: 7,670 us
// with a wavefront per walker, about 350 here; 1,003 evaluations 458 -> 105
// us a call.  Cycles per wavefront: Slater rows 50 k, inversion 41 k,
// determinant and nuclear terms 80 k, partners 11 k, parameters 20 k, for
// about 20 k vector and 1 k scalar-load instructions: a wavefront waits 39 %
// of its cycles (coefficient rows from the scalar cache, rows in transit) and
// issues vector instructions for 33 %, at two wavefronts per SIMD (1,003
// evaluations, under one per SIMD: 51 % and 32 %).  The rows from LDS were
// slower (500 us a measure call against 402: the wider loads spill).  The
// evaluation spills 24 registers (100 bytes of scratch), the derivatives none.
#include "qmc_terms.hpp"

#include <cstring>

#include "qmc_pair_terms.hpp"
#include "qmc_terms_dev.hpp"
#include "qmc_wave_dev.hpp"

namespace qmc {
namespace {

constexpr int NS = TERMS_N, GW = TERMS_W, RS = NS;  // row stride in transit: odd, so 64 lanes use all banks

struct TermLds {
  double row[2][GW * NS * RS];     // per wavefront: inverse rows in transit, then the rows of a sum
  double colv[2][GW][NS + 1];      // |a| of a pivot search
  double prow[2][GW][NS + 1];      // pivot row
  int piv[2][GW][NS + 1];
  double xyz[GW][2 * NS][3];
  double g[GW][2 * NS][3];         // d ln psi / d r
  double cm[2][TERMS_MO][GW * NS]; // inverse entries of the MOs that follow the geometry
  double part[2][6 * MAXN][GW];    // per wavefront: Omega and F sums of its electrons
  double sums[2][9][GW];
};

// sums over the 21 electrons of each walker of the NR (at most 20) values
// per lane that this wavefront stored at buf[r * 64 + lane]: out[r][g]
template <int NR>
__device__ __forceinline__ void lane_sums(const double* buf, int lane, double (*out)[GW]) {
  wave_sync();
  for (int t = lane; t < NR * GW; t += 64) {
    const int r = t / GW, g = t % GW;
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NS; ++i) s += buf[r * 64 + g * NS + i];
    out[r][g] = s;
  }
  wave_sync();
}
template <int NR>
__device__ __forceinline__ void lane_sums(double* buf, int lane, const double* v, double (*out)[GW]) {
#pragma unroll
  for (int r = 0; r < NR; ++r) buf[r * 64 + lane] = v[r];
  lane_sums<NR>(buf, lane, out);
}

struct TermArgs {
  DerivArgs D;  // W, positions and, for the derivatives, the feature matrix
  EvalOut O;
  int* sing;
};

template <bool DERIV>
__global__ void __launch_bounds__(128, 2) terms_kernel(const DevSys<double>* __restrict__ Sp,
                                                    const TermTab* __restrict__ Tp, TermArgs A) {
  __shared__ TermLds L;
  const DevSys<double>& S = *Sp;
  const TermTab& T = *Tp;
  const int sp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int l = lane < GW * NS ? lane : GW * NS - 1;  // the last lane shadows its neighbour
  const bool mine_ok = lane < GW * NS;
  const int grp = l / NS, slot = l % NS;
  const int64_t w = (int64_t)blockIdx.x * GW + grp;
  const bool live = w < A.D.W;
  const int64_t wl = live ? w : A.D.W - 1;  // walkers past the end shadow the last one and write nothing
  const int e = S.sector_elec[sp][slot];
  double r[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int q = 3 * e + c;
    r[c] = A.D.pos_aos ? A.D.pos_aos[wl * 6 * NS + q]
                       : (A.D.pos64 ? A.D.pos64[q * A.D.ld + wl] : (double)A.D.pos32[q * A.D.ld + wl]);
    L.xyz[grp][sp * NS + slot][c] = r[c];
  }
  __syncthreads();
  const double x = r[0], y = r[1], z = r[2];
  const double* mo = &T.mo[T.same ? 0 : sp][0][0];
  const int M = T.n_nuc;

  // ---- Slater row a[m] = phi_m(r) ----
  double a[NS];
#pragma unroll
  for (int m = 0; m < NS; ++m) a[m] = 0.0;
  for (int I = 0; I < M; ++I) {
    const double dx = x - T.nuc[I][0], dy = y - T.nuc[I][1], dz = z - T.nuc[I][2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    nucleus_shells(T, I, [&](auto np, auto is_sp, const TermPrim* pr, int row) {
      constexpr int NP = decltype(np)::value;
      constexpr bool SP = decltype(is_sp)::value;
      const double* C = mo + row * NS;
      double s[3], p[3];
      radial<NP, SP, false>(pr, r2, s, p);
#pragma unroll
      for (int m = 0; m < NS; ++m) a[m] += C[m] * s[0];
      if constexpr (SP) {
        const double px = dx * p[0], py = dy * p[0], pz = dz * p[0];
#pragma unroll
        for (int m = 0; m < NS; ++m) a[m] += C[NS + m] * px;
#pragma unroll
        for (int m = 0; m < NS; ++m) a[m] += C[2 * NS + m] * py;
#pragma unroll
        for (int m = 0; m < NS; ++m) a[m] += C[3 * NS + m] * pz;
      }
    });
  }

  // ---- inverse, one row per lane: Gauss-Jordan in place without row
  // interchanges; column c's pivot is its largest |a| over the unused rows
  // (ties to the lowest row) ----
  LogAcc<double> det;
  double dummy = 0.0, sg = 1.0;
  bool used = false, sing = false;
  int mine = 0;
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    L.colv[sp][grp][slot] = used ? -1.0 : pivot_mag(a[c]);
    wave_sync();
    double best = -2.0;
    int p = 0;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const double v = L.colv[sp][grp][i];
      if (v > best) {
        best = v;
        p = i;
      }
    }
    const bool me = slot == p;
    if (me) {
#pragma unroll
      for (int j = 0; j < NS; ++j) L.prow[sp][grp][j] = a[j];
      L.piv[sp][grp][c] = p;
      used = true;
      mine = c;
    }
    wave_sync();
    double pr[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) pr[j] = L.prow[sp][grp][j];
    const double pv = pr[c], ip = 1.0 / pv;
    if (pv == 0.0) sing = true;
    det.add(dummy, pv);
    if (pv < 0.0) sg = -sg;
    const double f = me ? 0.0 : a[c];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const double q = pr[j] * ip;
      if (j != c) a[j] = me ? q : a[j] - f * q;
    }
    a[c] = me ? ip : -f * ip;
  }
  double* row = L.row[sp];
#pragma unroll
  for (int j = 0; j < NS; ++j) row[l * RS + j] = a[j];
  wave_sync();
  // col[m] = (A^-1)_{m, slot}: entry `mine` of the row that was column m's pivot
  double col[NS];
  int inversions = 0;
#pragma unroll
  for (int m = 0; m < NS; ++m) {
    const int p = L.piv[sp][grp][m];
    col[m] = sing ? (m == slot ? 1.0 : 0.0) : row[(grp * NS + p) * RS + mine];
    if (m > mine && p < slot) ++inversions;
  }
  if constexpr (DERIV) {
    for (int i = 0; i < T.n_mo; ++i) {
      const int m = T.mo_list[i];
      L.cm[sp][i][l] = sing ? (m == slot ? 1.0 : 0.0) : row[(grp * NS + L.piv[sp][grp][m]) * RS + mine];
    }
  }
  wave_sync();

  // ---- determinant and electron-nucleus terms, nucleus by nucleus ----
  double gdx = 0.0, gdy = 0.0, gdz = 0.0, ld = 0.0;
  double gux = 0.0, guy = 0.0, guz = 0.0, lu = 0.0, u = 0.0, pot = 0.0;
  auto one_nucleus = [&](int I, double* o) {  // o: the six rows of this nucleus at a stride of 64
    double ox = 0.0, oy = 0.0, oz = 0.0;
    const double dx = x - T.nuc[I][0], dy = y - T.nuc[I][1], dz = z - T.nuc[I][2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    nucleus_shells(T, I, [&](auto np, auto is_sp, const TermPrim* pr, int row) {
      constexpr int NP = decltype(np)::value;
      constexpr bool SP = decltype(is_sp)::value;
      const double* C = mo + row * NS;
      double ws = 0.0, wx = 0.0, wy = 0.0, wz = 0.0, s[3], p[3];
      radial<NP, SP, true>(pr, r2, s, p);
#pragma unroll
      for (int m = 0; m < NS; ++m) ws += C[m] * col[m];
      if constexpr (SP) {
#pragma unroll
        for (int m = 0; m < NS; ++m) wx += C[NS + m] * col[m];
#pragma unroll
        for (int m = 0; m < NS; ++m) wy += C[2 * NS + m] * col[m];
#pragma unroll
        for (int m = 0; m < NS; ++m) wz += C[3 * NS + m] * col[m];
      }
      // s: grad = -2 R_a d, lap = -6 R_a + 4 r^2 R_aa; p_m = d_m R: grad_j =
      // delta_jm R - 2 d_m R_a d_j, lap = d_m (-10 R_a + 4 r^2 R_aa)
      const double wd = wx * dx + wy * dy + wz * dz;
      const double gf = -2.0 * (s[1] * ws + p[1] * wd);
      const double sx = gf * dx + wx * p[0], sy = gf * dy + wy * p[0], sz = gf * dz + wz * p[0];
      ld += ws * (-6.0 * s[1] + 4.0 * r2 * s[2]) + wd * (-10.0 * p[1] + 4.0 * r2 * p[2]);
      gdx += sx;
      gdy += sy;
      gdz += sz;
      ox -= sx;
      oy -= sy;
      oz -= sz;
    });
    double rr, ir;
    qmc::M<double>::dist_inv(r2, rr, ir);
    pot -= S.Z[I] * ir;
    if (S.en_on) {
      double u1, lp;
      uen_d<double, JsNone>(S, rr, ir, I, u1, lp);
      if constexpr (!DERIV) u += uen_val<double, JsNone>(S, rr, I);
      const bool ok = rr >= 1e-10;
      const double f = ok ? u1 * ir : 0.0;
      gux += f * dx;
      guy += f * dy;
      guz += f * dz;
      lu += ok ? lp : 0.0;
      ox -= f * dx;
      oy -= f * dy;
      oz -= f * dz;
    }
    if constexpr (DERIV) {
      for (int i = T.g0[sp][I]; i < T.g0[sp][I + 1]; ++i) {  // MO coefficients that follow R_I
        const TermMoGrp& G = T.grp[sp][i];
        const TermShell q = T.sh[G.sh];
        const double ex = x - T.nuc[G.I][0], ey = y - T.nuc[G.I][1], ez = z - T.nuc[G.I][2];
        double s[3], p[3];
        by_count(q.np, [&](auto np) {
          radial<decltype(np)::value, true, false>(T.pr + q.p0, ex * ex + ey * ey + ez * ez, s, p);
        });
        const double cv = L.cm[sp][G.mi][l];
        const double c0 = cv * s[0], c1 = cv * ex * p[0], c2 = cv * ey * p[0], c3 = cv * ez * p[0];
        ox += G.d[0][0] * c0 + G.d[1][0] * c1 + G.d[2][0] * c2 + G.d[3][0] * c3;
        oy += G.d[0][1] * c0 + G.d[1][1] * c1 + G.d[2][1] * c2 + G.d[3][1] * c3;
        oz += G.d[0][2] * c0 + G.d[1][2] * c1 + G.d[2][2] * c2 + G.d[3][2] * c3;
      }
      const double f3 = rr > 1e-10 ? S.Z[I] * ir * ir * ir : 0.0;  // methane.rs:1253
      o[0] = ox;
      o[1 * 64] = oy;
      o[2 * 64] = oz;
      o[3 * 64] = f3 * dx;
      o[4 * 64] = f3 * dy;
      o[5 * 64] = f3 * dz;
    }
  };
  if constexpr (DERIV) {
    double* o = row + lane;
    int I = 0;
    for (; I + 3 <= M; I += 3) {
#pragma unroll 1
      for (int k = 0; k < 3; ++k) one_nucleus(I + k, o + 6 * 64 * k);
      lane_sums<18>(row, lane, &L.part[sp][6 * I]);
    }
    for (; I < M; ++I) {
      one_nucleus(I, o);
      lane_sums<6>(row, lane, &L.part[sp][6 * I]);
    }
  } else {
    for (int I = 0; I < M; ++I) one_nucleus(I, nullptr);
  }

  // ---- Jastrow partners and 1/r of the other electrons ----
  double pairsq = 0.0, pee = 0.0;
  auto partner = [&](int j, bool same, bool other) {
    const double* rj = L.xyz[grp][j];
    const double dx = x - rj[0], dy = y - rj[1], dz = z - rj[2];
    double rr, ir, u1, lp;
    qmc::M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
    uee_d<double, JsNone>(S, rr, ir, same, u1, lp);
    if constexpr (!DERIV) u += other ? 0.5 * (uee_val<double, JsNone>(S, rr, same) + S.cst_ee) : 0.0;
    const bool ok = other && rr >= 1e-10;
    const double f = ok ? u1 * ir : 0.0;
    gux += f * dx;
    guy += f * dy;
    guz += f * dz;
    lu += ok ? lp : 0.0;
    pairsq += ok ? u1 * u1 : 0.0;
    pee += other ? ir : 0.0;
  };
#pragma unroll 3
  for (int j = 0; j < NS; ++j) partner(sp * NS + j, true, j != slot);
#pragma unroll 3
  for (int j = 0; j < NS; ++j) partner((1 - sp) * NS + j, false, true);
  const double gs = S.grad_scale;
  const double lj = (S.flags & F_J2_LAP_QUIRK) ? lu + pairsq : lu + gux * gux + guy * guy + guz * guz;
  const double lap = ld + lj + 2.0 * gs * (gdx * gux + gdy * guy + gdz * guz);
  const double ei = -0.5 * lap + 0.5 * pee + pot;

  if constexpr (!DERIV) {
    double la = 0.0;
    det.fold(la);
    if (sing) {
      la = -INFINITY;
      sg = 0.0;
    }
    const double v[3] = {ei, u, (double)inversions};
    lane_sums<3>(row, lane, v, L.sums[sp]);
    if (slot == 0) {
      L.sums[sp][3][grp] = la;
      L.sums[sp][4][grp] = sg;
    }
    if (live && mine_ok) {
      if (A.O.grad) {
        double* g = A.O.grad + w * 6 * NS + 3 * e;
        g[0] = gdx + gs * gux;
        g[1] = gdy + gs * guy;
        g[2] = gdz + gs * guz;
      }
      if (A.O.lap) A.O.lap[w * 2 * NS + e] = lap;
    }
    __syncthreads();
    if (threadIdx.x < GW) {
      const int g = threadIdx.x;
      const int64_t wg = (int64_t)blockIdx.x * GW + g;
      if (wg < A.D.W) {
        const int inv = (int)(L.sums[0][2][g] + L.sums[1][2][g]);
        const double s = L.sums[0][4][g] * L.sums[1][4][g];
        if (A.O.eloc) A.O.eloc[wg] = L.sums[0][0][g] + L.sums[1][0][g] + S.vnn;
        if (A.O.logabs)
          A.O.logabs[wg] = L.sums[0][3][g] + L.sums[1][3][g] + (L.sums[0][1][g] + L.sums[1][1][g]);
        if (A.O.sign) A.O.sign[wg] = inv & 1 ? -s : s;
        if (s == 0.0 && A.sing) atomicAdd(A.sing, 1);
      }
    }
  } else {
    double* gl = L.g[grp][sp * NS + slot];
    gl[0] = gdx + gux;
    gl[1] = gdy + guy;
    gl[2] = gdz + guz;
    __syncthreads();
    // ---- Jastrow parameters [b_ee, b_en, a_anti, a_para]: every e-e pair
    // once (same spin: offsets 1..10 around the sector; opposite spin: (k,
    // k + d) by the up lane for d <= 10, by the down lane for d > 10) ----
    double v[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, ei};
    if (S.jas_kind == JAS_PADE) {
      auto pair = [&](int j, bool same) {
        const double* rj = L.xyz[grp][j];
        const double* gj = L.g[grp][j];
        const double gi[3] = {gdx + gux, gdy + guy, gdz + guz};
        const int ca = same ? 3 : 2;
        double dr, dx = x - rj[0], dy = y - rj[1], dz = z - rj[2], ir;
        qmc::M<double>::dist_inv(dx * dx + dy * dy + dz * dz, dr, ir);
        PairDerivs<double> pd;
        pd.init(dr, S.b_ee, same ? S.a_para : S.a_anti, 0, nullptr);
        v[0] -= pd.A1 * pd.x * pd.x;
        v[ca] += pd.x;
        const bool ok = dr >= 1e-10;
        const double dlt = (gi[0] - gj[0]) * (dx * ir) + (gi[1] - gj[1]) * (dy * ir) + (gi[2] - gj[2]) * (dz * ir);
        double du1, dl;
        pd.d_b(dr, ir, S.b_ee, du1, dl);
        v[4] -= ok ? dl + dlt * du1 : 0.0;
        pd.d_a(ir, S.b_ee, du1, dl);
        v[4 + ca] -= ok ? dl + dlt * du1 : 0.0;
      };
      for (int d = 1; d <= NS / 2; ++d) {
        const int j = slot + d;
        pair(sp * NS + (j < NS ? j : j - NS), true);
      }
      for (int d = sp ? NS / 2 + 1 : 0; d < (sp ? NS : NS / 2 + 1); ++d) {
        const int j = sp ? (slot >= d ? slot - d : slot - d + NS) : (slot + d < NS ? slot + d : slot + d - NS);
        pair((1 - sp) * NS + j, false);
      }
      const double gi[3] = {gdx + gux, gdy + guy, gdz + guz};
      for (int I = 0; I < M; ++I)
        en_pair_terms(S, I, x - S.nuc[I][0], y - S.nuc[I][1], z - S.nuc[I][2], [&](int c) { return gi[c]; },
                      [&](int sl, double q) { v[1] += sl == 0 ? q : 0.0; },
                      [&](int sl, double q) { v[5] += sl == 0 ? q : 0.0; });
    }
    lane_sums<9>(row, lane, v, L.sums[sp]);
    __syncthreads();
    const DerivLayout Ly{A.D.P, M, 2 * NS, A.D.Qp};
    for (int t = threadIdx.x; t < A.D.Qp * GW; t += 128) {
      const int q = t / GW, g = t % GW;
      const int64_t wg = (int64_t)blockIdx.x * GW + g;
      if (wg >= A.D.W) continue;
      double o = 0.0;
      if (q < A.D.P) {
        o = L.sums[0][q][g] + L.sums[1][q][g];
      } else if (q < Ly.e()) {
        const int k = q - A.D.P, i = 6 * (k / 3) + k % 3;
        o = L.part[0][i][g] + L.part[1][i][g];
      } else if (q == Ly.e()) {
        o = L.sums[0][8][g] + L.sums[1][8][g] + S.vnn;
      } else if (q == Ly.one()) {
        o = 1.0;
      } else if (q < Ly.f(0, 0)) {
        const int k = q - Ly.de(0);
        o = L.sums[0][4 + k][g] + L.sums[1][4 + k][g];
      } else if (q < Ly.f(M, 0)) {
        const int k = q - Ly.f(0, 0), i = 6 * (k / 3) + 3 + k % 3;
        o = L.part[0][i][g] + L.part[1][i][g];
      }
      A.D.Y[(int64_t)q * A.D.ldy + wg] = o;
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool terms_table(const DevSys<double>& D, const MoDerivPair* pairs, const MoDerivEntry* ents, const int p0[3],
                 TermTab& T) {
  if (D.n_up != NS || D.n_dn != NS || D.k_ee != 0 || D.k_en != 0 || D.n_shell > TERMS_MAXSH || D.n_nuc > MAXN)
    return false;
  if (D.jas_kind != JAS_PADE && D.jas_kind != JAS_NONE) return false;
  std::memset(&T, 0, sizeof T);
  T.n_nuc = D.n_nuc;
  int rec_of[MAXSH], n = 0, row = 0, prim = 0;
  for (int I = 0; I < D.n_nuc; ++I) {
    T.sh0[I] = n;
    for (int c = 0; c < 3; ++c) T.nuc[I][c] = D.nuc[I][c];
    for (int i = 0; i < D.n_shell; ++i) {
      if (D.sh_center[i] != I) continue;
      const int kind = D.sh_kind[i], np = D.sh_nprim[i];
      if ((kind != SH_S && kind != SH_SP && kind != SH_P) || np < 1 || np > TERMS_MAXP) return false;
      const int rows = kind == SH_S ? 1 : 4;
      if (row + rows > TERMS_ROWS) return false;
      TermShell& q = T.sh[n];
      q.sp = kind != SH_S;
      q.np = np == 1 ? 1 : np <= 3 ? 3 : 6;
      q.row = row;
      q.p0 = prim;
      if (prim + q.np > TERMS_PRIM) return false;
      for (int k = 0; k < np; ++k)
        T.pr[prim + k] = TermPrim{D.prim_exp[D.sh_prim0[i] + k], kind == SH_P ? 0.0 : D.coef_s[D.sh_prim0[i] + k],
                                  kind == SH_S ? 0.0 : D.coef_p[D.sh_prim0[i] + k]};
      prim += q.np;
      for (int r = kind == SH_P ? 1 : 0; r < rows; ++r)
        for (int s = 0; s < 2; ++s)
          for (int m = 0; m < NS; ++m) T.mo[s][row + r][m] = D.moT[s][D.sh_ao0[i] + r - (kind == SH_P ? 1 : 0)][m];
      rec_of[i] = n++;
      row += rows;
    }
  }
  T.sh0[D.n_nuc] = n;
  if (n != D.n_shell) return false;
  for (int I = 0; I < D.n_nuc; ++I) {
    const TermShell* q = T.sh + T.sh0[I];
    const int k = T.sh0[I + 1] - T.sh0[I];
    auto is = [&](int i, int np, int sp) { return q[i].np == np && q[i].sp == sp; };
    T.pat[I] = k == 3 && is(0, 6, 0) && is(1, 3, 1) && is(2, 1, 1) ? TERMS_PAT_631G
               : k == 2 && is(0, 3, 0) && is(1, 1, 0)             ? TERMS_PAT_631G_H
                                                                  : TERMS_PAT_ANY;
  }
  T.same = std::memcmp(T.mo[0], T.mo[1], sizeof T.mo[0]) == 0;
  // MO-derivative groups: (spin, nucleus, shell, MO) with its 4 x 3 matrix
  for (int s = 0; s < 2; ++s) {
    int ng = 0;
    for (int I = 0; I < D.n_nuc; ++I) {
      T.g0[s][I] = ng;
      for (int p = p0[s]; p < p0[s + 1]; ++p)
        for (int k = pairs[p].e0; k < pairs[p].e1; ++k) {
          if (ents[k].I != I) continue;
          int mi = 0;
          while (mi < T.n_mo && T.mo_list[mi] != pairs[p].m) ++mi;
          if (mi == T.n_mo) {
            if (T.n_mo == TERMS_MO) return false;
            T.mo_list[T.n_mo++] = pairs[p].m;
          }
          const int sh = pairs[p].sh, rec = rec_of[sh];
          const int q = D.sh_kind[sh] == SH_P ? pairs[p].q + 1 : pairs[p].q;
          int g = T.g0[s][I];
          while (g < ng && !(T.grp[s][g].sh == rec && T.grp[s][g].mi == mi)) ++g;
          if (g == ng) {
            if (ng == TERMS_GRP) return false;
            ++ng;
            T.grp[s][g].sh = rec;
            T.grp[s][g].mi = mi;
            T.grp[s][g].I = D.sh_center[sh];
          }
          T.grp[s][g].d[q][ents[k].c] += ents[k].d;
        }
    }
    T.g0[s][D.n_nuc] = ng;
  }
  return true;
}

hipError_t terms_derivs(const void* Sd, const TermTab* T, DerivArgs D, hipStream_t st) {
  TermArgs A{D, {}, nullptr};
  terms_kernel<true><<<(unsigned)((D.W + GW - 1) / GW), 128, 0, st>>>((const DevSys<double>*)Sd, T, A);
  return hipGetLastError();
}

hipError_t terms_eval(const void* Sd, const TermTab* T, int64_t W, const double* pos, EvalOut O, int* sing,
                      hipStream_t st) {
  TermArgs A{};
  A.D.W = W;
  A.D.pos_aos = pos;
  A.O = O;
  A.sing = sing;
  terms_kernel<false><<<(unsigned)((W + GW - 1) / GW), 128, 0, st>>>((const DevSys<double>*)Sd, T, A);
  return hipGetLastError();
}

hipError_t terms_eloc(const void* Sd, const TermTab* T, EnsView<double> E, hipStream_t st) {
  TermArgs A{};
  A.D.W = E.W;
  A.D.pos64 = E.pos;
  A.D.ld = E.ld;
  A.O.eloc = E.eloc;
  terms_kernel<false><<<(unsigned)((E.W + GW - 1) / GW), 128, 0, st>>>((const DevSys<double>*)Sd, T, A);
  return hipGetLastError();
}

}  // namespace qmc
