// qmc_half.hip -- the half-wave engine: a walker of 21 + 21 electrons on 32
// lanes of one wavefront, in FP64.
//
// Lane g of a walker holds shell g of the basis (its exponents and
// coefficients in registers), columns g of both sectors' inverses (g < 21)
// and, in two rounds, the Jastrow partners g, g + 32 of the 42 electrons and
// the nuclei.  A move is then
//   the mover's inverse column through LDS to all lanes; for drift-diffusion
//     the shell's AO weights against it, from the MO table in LDS
//   the shell at the proposal (drift-diffusion: at both ends), one primitive
//     loop of six without branches
//   the MO values, lane m summing the walker's AO values (in LDS) against
//     column m of the MO table
//   the partners, sums over the 32 lanes by DPP and row swaps, the test, and
//     the Sherman-Morrison update of the lane's own column.
// Wavefronts never wait for each other: the MFMA tile that this replaces
// spent two workgroup barriers per move and held one wavefront per SIMD.
// In drift-diffusion sweeps of 2,048 walkers, one wavefront per SIMD, a
// wavefront waits 46 % of its cycles (LDS reads above all) and issues vector
// instructions for 40 %; in Metropolis sweeps of 8,192, two per SIMD, 49 % and
// 27 %.  A drift-diffusion sweep is 64,900 vector and 9,000 LDS instructions,
// whose bank conflicts hold the LDS for 13 % of the time.
#include "qmc_half.hpp"

#include "qmc_terms_dev.hpp"
#include "qmc_wave_dev.hpp"

namespace qmc {
namespace {

constexpr int NS = TERMS_N, N2 = 2 * NS;
constexpr int MS = NS + 1;                // row stride: even, so rows are read 16 bytes at a time
constexpr int PR = 24;                    // rows per unrolled step of the MO sums
constexpr int XR = HALF_ROWS;             // MO rows, padded with zeros to whole steps
static_assert(XR % PR == 0, "whole steps");
constexpr int ZR = XR;                    // a zero row, for the p parts that s shells do not have

struct HalfWave {  // one wavefront's two walkers
  double pos[HALF_W][N2][3];              // sector slots: up 0..20, down 21..41
  double rng[HALF_W][NS][4];              // a sector's normals and acceptance uniforms
  double col[HALF_W][MS];                 // the mover's inverse column
  double x[HALF_W][XR + 2];              // AO values of the proposal, by MO-table row
  double phi[HALF_W][MS];
  double park[NS][64];                    // the resting sector's columns
};
template <int NW>
struct HalfLds {
  double mo[2][XR + 1][MS];
  HalfWave w[NW];
};
static_assert(sizeof(HalfLds<8>) <= 160 * 1024, "eight wavefronts share a CU's LDS");

// sum over the 32 lanes of a walker: DPP within each row of 16, then the two
// rows swapped (v_permlane16_swap); the same value in every lane
__device__ __forceinline__ double hsum(double v) {
  v = rsum(v);
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
  const u2 a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const u2 b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __hiloint2double((int)b.x, (int)a.x) + __hiloint2double((int)b.y, (int)a.y);
}

template <bool DD, int NW>
__global__ void __launch_bounds__(64 * NW, NW / 4) half_kernel(const DevSys<double>* __restrict__ Sp,
                                                     const TermTab* __restrict__ Tp, EnsView<double> E, SweepArgs A,
                                                     double* __restrict__ partial, double* __restrict__ el_trace,
                                                     int64_t nrow) {
  extern __shared__ double lds_raw[];
  HalfLds<NW>& L = *(HalfLds<NW>*)lds_raw;
  const DevSys<double>& S = *Sp;
  const TermTab& T = *Tp;
  const int n_nuc = T.n_nuc, nsh = T.sh0[n_nuc], rows = T.sh[nsh - 1].row + (T.sh[nsh - 1].sp ? 4 : 1);
  for (int q = threadIdx.x; q < 2 * (XR + 1) * MS; q += 64 * NW) {
    const int m = q % MS, r = (q / MS) % (XR + 1), s = q / (MS * (XR + 1));
    L.mo[s][r][m] = r < rows && m < NS ? T.mo[s][r][m] : 0.0;
  }
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = threadIdx.x & 63;
  const int ww = l >> 5, g = l & 31;
  const int64_t prow = (int64_t)blockIdx.x * NW + wv;
  const int64_t Wn = E.n_live ? *E.n_live : E.W;
  if (prow >= nrow) return;
  if (prow * HALF_W >= Wn) {  // past a branching population's live walkers: zero partial sums only
    if (l == 0)
      for (int s = 0; s < A.n_steps; ++s)
        for (int q = 0; q < 3; ++q) partial[((int64_t)s * nrow + prow) * 3 + q] = 0.0;
    return;
  }
  HalfWave& H = L.w[wv];
  const int64_t w = prow * HALF_W + ww;
  const bool live = w < Wn;
  const int64_t wl = live ? w : Wn - 1;  // a walker past the end shadows the last one and writes nothing
  const bool own = g < NS;
  const int k0c = own ? g : 0;
  double cur[NS];  // the moving sector's column; the other rests in the park
#pragma unroll
  for (int m = 0; m < NS; ++m) {
    cur[m] = own ? E.ainv[(int64_t)(m * NS + k0c) * E.ld + wl] : 0.0;
    H.park[m][l] = own ? E.ainv[(int64_t)(NS * NS + m * NS + k0c) * E.ld + wl] : 0.0;
  }
  auto swap_sector = [&] {
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      const double v = H.park[m][l];
      H.park[m][l] = cur[m];
      cur[m] = v;
    }
  };
  if (own) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int e = S.sector_elec[s][g];
#pragma unroll
      for (int c = 0; c < 3; ++c) H.pos[ww][s * NS + g][c] = E.pos[(int64_t)(3 * e + c) * E.ld + wl];
    }
  }
  for (int r = l; r < HALF_W * (XR + 2); r += 64) (&H.x[0][0])[r] = 0.0;
  double ldet = E.logdet[wl], ju = E.ju[wl], sgn = E.sign[wl], el = 0.0;
  // the lane's shell, zero coefficients past the shells
  double ex[TERMS_MAXP], cs[TERMS_MAXP], cp[TERMS_MAXP], ctr[3] = {0.0, 0.0, 0.0};
  const bool has = g < nsh;
  const TermShell q = T.sh[has ? g : 0];
  const bool psh = has && q.sp;
  const int r0 = has ? q.row : ZR, r1 = psh ? q.row + 1 : ZR, rst = psh ? 1 : 0;  // MO rows r0, r1 + j rst
#pragma unroll
  for (int k = 0; k < TERMS_MAXP; ++k) {
    const bool on = has && k < q.np;
    const TermPrim p = T.pr[q.p0 + (on ? k : 0)];
    ex[k] = on ? p.ex : 0.0;
    cs[k] = on ? p.cs : 0.0;
    cp[k] = on ? p.cp : 0.0;
  }
  for (int I = 0; I < n_nuc; ++I)
    if (g >= T.sh0[I] && g < T.sh0[I + 1]) {
#pragma unroll
      for (int c = 0; c < 3; ++c) ctr[c] = T.nuc[I][c];
    }
  // the lane's partners: electron slot g; electron slot g + 32 or nucleus g - 10
  constexpr int E2 = N2 - 32;
  const bool el2 = g < E2, nuc2 = g >= E2 && g - E2 < n_nuc && S.en_on;
  double np[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) np[c] = T.nuc[nuc2 ? g - E2 : 0][c];
  const double a_para = S.a_para, a_anti = S.a_anti, b_ee = S.b_ee, gs = S.grad_scale;
  const double b2 = el2 ? b_ee : S.b_en, a2 = nuc2 ? -S.Z[g - E2] : 0.0;
  const uint32_t k0 = (uint32_t)A.seed, k1 = (uint32_t)(A.seed >> 32);
  const uint32_t wid = (uint32_t)(A.walker0 + wl);
  const uint32_t step0 = DD && A.step0_dev ? *A.step0_dev : A.step0;
  const double sigma = A.step_size, s2t = sqrt(2.0 * sigma), i4t = 0.25 / sigma;
  const double* xw = H.x[ww];

  for (int st = 0; st < A.n_steps; ++st) {
    const uint32_t step = step0 + (uint32_t)st;
    int acc = 0;
    LogAcc<double> lacc;
#pragma unroll 1
    for (int sp = 0; sp < 2; ++sp) {
      const double(*mo)[MS] = L.mo[T.same ? 0 : sp];
      if (own) {
        double z[3], U;
        Rng<double>::move(philox(wid, step, (uint32_t)S.sector_elec[sp][g], DD ? RNG_DRIFT : RNG_SINGLE, k0, k1), z, U);
        H.rng[ww][g][0] = z[0];
        H.rng[ww][g][1] = z[1];
        H.rng[ww][g][2] = z[2];
        H.rng[ww][g][3] = U;
      }
      const double ap1 = (g < NS) == (sp == 0) ? a_para : a_anti;
      const double ap2 = el2 ? (sp == 1 ? a_para : a_anti) : a2;  // slots past 31 are spin-down
#pragma unroll 1
      for (int k = 0; k < NS; ++k) {
        const int ms = sp * NS + k;
        if (g == k) {
#pragma unroll
          for (int m = 0; m < NS; ++m) H.col[ww][m] = cur[m];
        }
        wave_sync();
        const double ox = H.pos[ww][ms][0], oy = H.pos[ww][ms][1], oz = H.pos[ww][ms][2];
        const double z0 = H.rng[ww][k][0], z1 = H.rng[ww][k][1], z2 = H.rng[ww][k][2], U = H.rng[ww][k][3];
        // the lane's shell at a point: s and p radial sums (with their
        // exponent-weighted ones for gradients)
        auto shell = [&](double x, double y, double z, double d[3], double& rs, double& rp, double& rsa, double& rpa) {
          d[0] = x - ctr[0];
          d[1] = y - ctr[1];
          d[2] = z - ctr[2];
          const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
          rs = rp = rsa = rpa = 0.0;
#pragma unroll
          for (int i = 0; i < TERMS_MAXP; ++i) {
            const double ee = M<double>::exn(-ex[i] * r2);
            const double s = cs[i] * ee, p = cp[i] * ee;
            rs += s;
            rp += p;
            if constexpr (DD) {
              rsa += s * ex[i];
              rpa += p * ex[i];
            }
          }
        };
        // the lane's two partners at a point: value and scaled gradient
        auto partners = [&](double x, double y, double z, double u[4]) {
          u[0] = u[1] = u[2] = u[3] = 0.0;
          auto one = [&](bool on, const double* r, double a, double b) {
            const double dx = x - r[0], dy = y - r[1], dz = z - r[2];
            double rr, ir;
            M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
            const double iD = M<double>::rcp(1.0 + b * rr);
            u[0] += on ? a * rr * iD : 0.0;
            if constexpr (DD) {
              const double f = on && rr >= 1e-10 ? gs * a * iD * iD * ir : 0.0;
              u[1] += f * dx;
              u[2] += f * dy;
              u[3] += f * dz;
            }
          };
          one(g != ms, H.pos[ww][g], ap1, b_ee);
          const double* p2 = H.pos[ww][el2 ? 32 + g : 0];
          const double r2[3] = {el2 ? p2[0] : np[0], el2 ? p2[1] : np[1], el2 ? p2[2] : np[2]};
          one(el2 ? 32 + g != ms : nuc2, r2, ap2, b2);
        };
        // AO values to LDS, then lane m's MO value phi_m = sum_r x[r] C[r][m]
        auto mo_values = [&](const double d[3], double rs, double rp) {
          double* xr = H.x[ww];
          xr[r0] = rs;
          xr[r1] = d[0] * rp;
          xr[r1 + rst] = d[1] * rp;
          xr[r1 + 2 * rst] = d[2] * rp;
          wave_sync();
          double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
          for (int r = 0; r < rows; r += PR) {
#pragma unroll
            for (int i = 0; i < PR; i += 4) {
              p0 += xw[r + i] * mo[r + i][k0c];
              p1 += xw[r + i + 1] * mo[r + i + 1][k0c];
              p2 += xw[r + i + 2] * mo[r + i + 2][k0c];
              p3 += xw[r + i + 3] * mo[r + i + 3][k0c];
            }
          }
          if (own) H.phi[ww][g] = (p0 + p1) + (p2 + p3);
          wave_sync();
        };
        double nx, ny, nz, R, du, p, dn[3], rs, rp, rsa, rpa, uo[4], un[4];
        partners(ox, oy, oz, uo);
        if constexpr (DD) {
          double ws = 0.0, wx = 0.0, wy = 0.0, wz = 0.0;
#pragma unroll
          for (int m = 0; m < NS; ++m) {
            const double c = H.col[ww][m];
            ws += mo[r0][m] * c;
            wx += mo[r1][m] * c;
            wy += mo[r1 + rst][m] * c;
            wz += mo[r1 + 2 * rst][m] * c;
          }
          auto force = [&](const double d[3], double v[4]) {
            const double wd = wx * d[0] + wy * d[1] + wz * d[2], t = -2.0 * (ws * rsa + wd * rpa);
            v[0] = ws * rs + wd * rp;
            v[1] = t * d[0] + wx * rp;
            v[2] = t * d[1] + wy * rp;
            v[3] = t * d[2] + wz * rp;
          };
          double d[3], fo[4], fn[4], c0[3], c1[3];
          shell(ox, oy, oz, d, rs, rp, rsa, rpa);
          force(d, fo);
          cap_drift(2.0 * hsum(fo[1] + uo[1]), 2.0 * hsum(fo[2] + uo[2]), 2.0 * hsum(fo[3] + uo[3]), sigma, A.max_drift,
                    c0);
          nx = ox + c0[0] + s2t * z0;
          ny = oy + c0[1] + s2t * z1;
          nz = oz + c0[2] + s2t * z2;
          shell(nx, ny, nz, dn, rs, rp, rsa, rpa);
          force(dn, fn);
          partners(nx, ny, nz, un);
          R = hsum(fn[0]);
          du = hsum(un[0] - uo[0]);
          const double iR = M<double>::rcp(R);
          cap_drift(2.0 * hsum(fn[1] * iR + un[1]), 2.0 * hsum(fn[2] * iR + un[2]), 2.0 * hsum(fn[3] * iR + un[3]), sigma,
                    A.max_drift, c1);
          const double f0 = nx - ox - c0[0], f1 = ny - oy - c0[1], f2 = nz - oz - c0[2];
          const double h0 = ox - nx - c1[0], h1 = oy - ny - c1[1], h2 = oz - nz - c1[2];
          const double gg = ((f0 * f0 + f1 * f1 + f2 * f2) - (h0 * h0 + h1 * h1 + h2 * h2)) * i4t;
          p = R * R * M<double>::ex(2.0 * du + gg);
          mo_values(dn, rs, rp);
        } else {
          nx = ox + sigma * z0;
          ny = oy + sigma * z1;
          nz = oz + sigma * z2;
          shell(nx, ny, nz, dn, rs, rp, rsa, rpa);
          partners(nx, ny, nz, un);
          mo_values(dn, rs, rp);
          R = 0.0;
        }
        double v = 0.0;
#pragma unroll
        for (int m = 0; m < NS; ++m) v += H.phi[ww][m] * cur[m];
        if constexpr (!DD) {
          R = __shfl(v, (l & 32) | k, 64);
          du = hsum(un[0] - uo[0]);
          p = R * R * M<double>::ex(2.0 * du);
        }
        if (U < p) {  // uniform within the walker's lanes
          const double iR = M<double>::rcp(R);
          // column j takes A_j - c v_j / R; the mover's own becomes c / R
          const double sk = g == k ? 0.0 : 1.0, f = g == k ? -iR : v * iR;
#pragma unroll
          for (int m = 0; m < NS; ++m) cur[m] = fma(-H.col[ww][m], f, cur[m] * sk);
          if (g == k) {
            H.pos[ww][ms][0] = nx;
            H.pos[ww][ms][1] = ny;
            H.pos[ww][ms][2] = nz;
          }
          lacc.add(ldet, R);
          if (R < 0.0) sgn = -sgn;
          ju += du;
          ++acc;
        }
        wave_sync();
      }
      if (sp == 0) swap_sector();
    }
    lacc.fold(ldet);

    // local energy: the 21 electrons of a sector on the lanes that hold their
    // inverse columns, one sector after the other
    double es = 0.0;
#pragma unroll 1
    for (int sp = 1; sp >= 0; --sp) {
      const double(*mo)[MS] = L.mo[T.same ? 0 : sp];
      const double* ri = H.pos[ww][sp * NS + k0c];
      const double x = ri[0], y = ri[1], z = ri[2];
      double gdx = 0.0, gdy = 0.0, gdz = 0.0, ld = 0.0, gux = 0.0, guy = 0.0, guz = 0.0, lu = 0.0, pot = 0.0;
      for (int I = 0; I < n_nuc; ++I) {
        const double dx = x - T.nuc[I][0], dy = y - T.nuc[I][1], dz = z - T.nuc[I][2];
        const double d2 = dx * dx + dy * dy + dz * dz;
        nucleus_shells(T, I, [&](auto np, auto is_sp, const TermPrim* pr, int row) {
          constexpr int NP = decltype(np)::value;
          constexpr bool SP = decltype(is_sp)::value;
          const double* C = mo[row];
          double ws = 0.0, wx = 0.0, wy = 0.0, wz = 0.0, s[3], p[3];
          radial<NP, SP, true>(pr, d2, s, p);
#pragma unroll
          for (int m = 0; m < NS; ++m) ws += C[m] * cur[m];
          if constexpr (SP) {
#pragma unroll
            for (int m = 0; m < NS; ++m) {
              wx += C[MS + m] * cur[m];
              wy += C[2 * MS + m] * cur[m];
              wz += C[3 * MS + m] * cur[m];
            }
          }
          const double wd = wx * dx + wy * dy + wz * dz;
          const double gf = -2.0 * (s[1] * ws + p[1] * wd);
          gdx += gf * dx + wx * p[0];
          gdy += gf * dy + wy * p[0];
          gdz += gf * dz + wz * p[0];
          ld += ws * (-6.0 * s[1] + 4.0 * d2 * s[2]) + wd * (-10.0 * p[1] + 4.0 * d2 * p[2]);
        });
        double rr, ir;
        M<double>::dist_inv(d2, rr, ir);
        pot -= S.Z[I] * ir;
        if (S.en_on) {
          double u1, lp;
          uen_d<double, JsNone>(S, rr, ir, I, u1, lp);
          const bool ok = rr >= 1e-10;
          const double f = ok ? u1 * ir : 0.0;
          gux += f * dx;
          guy += f * dy;
          guz += f * dz;
          lu += ok ? lp : 0.0;
        }
      }
      double pairsq = 0.0;
      auto partner = [&](int j, bool same, bool other) {
        const double* rj = H.pos[ww][j];
        const double dx = x - rj[0], dy = y - rj[1], dz = z - rj[2];
        double rr, ir, u1, lp;
        M<double>::dist_inv(dx * dx + dy * dy + dz * dz, rr, ir);
        uee_d<double, JsNone>(S, rr, ir, same, u1, lp);
        const bool ok = other && rr >= 1e-10;
        const double f = ok ? u1 * ir : 0.0;
        gux += f * dx;
        guy += f * dy;
        guz += f * dz;
        lu += ok ? lp : 0.0;
        pairsq += ok ? u1 * u1 : 0.0;
        pot += other ? 0.5 * ir : 0.0;
      };
#pragma unroll 3
      for (int j = 0; j < NS; ++j) partner(sp * NS + j, true, j != k0c);
#pragma unroll 3
      for (int j = 0; j < NS; ++j) partner((1 - sp) * NS + j, false, true);
      const double lj = (S.flags & F_J2_LAP_QUIRK) ? lu + pairsq : lu + gux * gux + guy * guy + guz * guz;
      const double lap = ld + lj + 2.0 * gs * (gdx * gux + gdy * guy + gdz * guz);
      es += own ? -0.5 * lap + pot : 0.0;
      if (sp == 1) swap_sector();
    }
    el = hsum(es) + S.vnn;
    const bool head = live && g == 0;
    if (el_trace && head) el_trace[(int64_t)st * A.trace_ld + w] = el;
    if (g == 0) {
      H.phi[ww][0] = live ? el : 0.0;
      H.phi[ww][1] = live ? el * el : 0.0;
      H.phi[ww][2] = live ? (double)acc : 0.0;
    }
    wave_sync();
    if (l < 3) partial[((int64_t)st * nrow + prow) * 3 + l] = H.phi[0][l] + H.phi[1][l];
    wave_sync();
  }
  if (live && own) {
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      E.ainv[(int64_t)(m * NS + g) * E.ld + w] = cur[m];
      E.ainv[(int64_t)(NS * NS + m * NS + g) * E.ld + w] = H.park[m][l];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int e = S.sector_elec[s][g];
#pragma unroll
      for (int c = 0; c < 3; ++c) E.pos[(int64_t)(3 * e + c) * E.ld + w] = H.pos[ww][s * NS + g][c];
    }
  }
  if (live && g == 0) {
    E.logdet[w] = ldet;
    E.ju[w] = ju;
    E.sign[w] = sgn;
    E.eloc[w] = el;
  }
}

template <bool DD, int NW>
hipError_t launch_half(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                       hipStream_t st) {
  const int64_t nrow = half_blocks(E.W);
  constexpr int lds = (int)sizeof(HalfLds<NW>);
  hipError_t e = hipFuncSetAttribute((const void*)half_kernel<DD, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  half_kernel<DD, NW><<<(unsigned)((nrow + NW - 1) / NW), 64 * NW, lds, st>>>((const DevSys<double>*)Sd, T, E, A, partial,
                                                                           trace, nrow);
  return hipGetLastError();
}
template <bool DD>
hipError_t launch_by_count(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial,
                           double* trace, hipStream_t st) {
  // Up to 2,048 walkers one wavefront per SIMD covers the chip, with 512
  // registers each; past that two per SIMD share a CU's tables, at 256
  // registers (53 and 77 of them spilled to scratch).  us per sweep, four / eight wavefronts per
  // workgroup / the tile engine: Metropolis 202 / 275 / 371 at 2,048 walkers,
  // 393 / 277 / 373 at 4,096, 782 / 550 / 742 at 8,192; drift-diffusion 290 /
  // 445 / 569, 576 / 448 / 570, 1,146 / 894 / 1,137.
  if (E.W <= 2048) return launch_half<DD, 4>(Sd, T, E, A, partial, trace, st);
  return launch_half<DD, 8>(Sd, T, E, A, partial, trace, st);
}

}  // namespace

hipError_t half_sweep(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                      hipStream_t st) {
  return launch_by_count<false>(Sd, T, E, A, partial, trace, st);
}
hipError_t half_dd(const void* Sd, const TermTab* T, EnsView<double> E, SweepArgs A, double* partial, double* trace,
                   hipStream_t st) {
  return launch_by_count<true>(Sd, T, E, A, partial, trace, st);
}

}  // namespace qmc
