// Hydrostatic equilibrium for batches of temperature columns: pyrh's hse()
// (pyrh.pyx:427-487, rh/rhf1d/pyrh_hse.c:67-399).  Per layer, from the top
// down, the reference repeats until n_Htot settles: rho from n_Htot, n_e from
// LTE ionisation of every element (get_ne, rh/rhf1d/pyrh_background.c:459-549),
// LTE populations and chemical equilibrium, the continuum opacity at the
// evaluation wavelength (pyrh_Background, pyrh_background.c:144-457), p_g from
// the layer above, and n_Htot = (p_g/kT - n_e)/totalAbund.
//
// The layers are a serial chain, so what bounds the builder is the length of
// that chain, not the chip's rate.  Everything that a layer's temperature
// alone fixes (about 320 numbers: every exponential, power and table look-up)
// is formed first by k_hse_tables, in parallel over columns and depths;
// k_hse then runs the chain with a group of lanes per column that share the
// elements of the electron-density step and the molecules of the chemical
// equilibrium, on the layer's numbers staged in LDS.
#include "rhg_equil.hpp"
#include "rhg_hse.hpp"

namespace rhg {

namespace {

constexpr int HSE_N_MAX_ELECTRON_ITER = 10;  // rh/rhf1d/pyrh_background.h:1-2
constexpr double HSE_MAX_ELECTRON_ERROR = 1.0E-2;

// What the layer's temperature fixes in the Saha factors: pow(C1/T, 1.5),
// exp(E_ION_HMIN/kT) (these two in this order, as chem_eq takes them),
// pow(C1/T, -1.5) and exp(Uk0 + chi_H/kT).
struct HseT {
  double p15, eHmin, pm15, eH;
};

__device__ __forceinline__ HseT hse_tcache(const DevHse &H, double T, double Uk0) {
  const double C1 = (HPLANCK / (2.0 * PI * M_ELECTRON)) * (HPLANCK / KBOLTZMANN);
  const double kT = KBOLTZMANN * T;
  HseT t;
  t.p15 = pow(C1 / T, 1.5);
  t.eHmin = exp(0.754 * EV / kT);
  t.pm15 = pow(C1 / T, -1.5);
  t.eH = exp(Uk0 + H.el_ionpot[0] / kT);
  return t;
}

// 1 / x and a / b by the hardware reciprocal estimate refined by two Newton
// steps (relative error ~1e-16, not correctly rounded): the quotients inside
// the sums over elements and molecules, where the IEEE division sequence is a
// long dependent chain.  The few of a pressure iteration itself are IEEE: a
// rounded reciprocal would bias every layer alike
__device__ __forceinline__ double hrcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ double hdiv(double a, double b) { return a * hrcp(b); }

// Cross-lane moves within a row of 16 lanes
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sums over the `lanes` (a power of two) consecutive lanes of an
// aligned group; every lane ends with the same bits, so control flow on the
// result is uniform in the group.  Up to 16 lanes the partners are in the
// same row (quad permutations xor 1 and xor 2, half-row and row mirror).
template <int N>
__device__ __forceinline__ void group_sum(double (&x)[N], int lanes) {
  if (lanes >= 2) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += dpp_move<0xb1>(x[i]);   // quad_perm [1,0,3,2]
  }
  if (lanes >= 4) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += dpp_move<0x4e>(x[i]);   // quad_perm [2,3,0,1]
  }
  if (lanes >= 8) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += dpp_move<0x141>(x[i]);  // row_half_mirror
  }
  if (lanes >= 16) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += dpp_move<0x140>(x[i]);  // row_mirror
  }
  for (int o = 16; o < lanes; o <<= 1) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += __shfl_xor(x[i], o);
  }
}

// LDS written by some lanes of the wavefront is read by others after this
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// Saha-Boltzmann level sums of one model atom at temperature T, grouped by
// the ionisation difference dZ to the ground level: g[d] = sum over levels
// i >= 1 with dZ_i = d of g_i/g_0 exp(-(E_i - E_0)/kT) (rh/ltepops.c:87-100),
// d < HSE_NDZ, and g[HSE_NDZ] the same sum over the neutral levels before
// the first ionised one (the neutral fraction of rh/chemequil.c:222-236).
// The LTE normalisation is then 1 + sum_d g[d] / (cNe_T)^d for any n_e.
__device__ void hse_level_groups(const DevModel &M, int ia, double T, double *g, int gs) {
  const int l0 = ldc(M.atom_level_ptr)[ia], nl = ldc(M.atom_level_ptr)[ia + 1] - l0;
  double acc[HSE_NDZ + 1];
#pragma unroll
  for (int d = 0; d <= HSE_NDZ; d++) acc[d] = 0.0;
  bool neutral = ldc(M.level_stage)[l0] == 0;
  for (int i = 1; i < nl; i++) {
    const double dE = ldc(M.level_E)[l0 + i] - ldc(M.level_E)[l0];
    const double r = (ldc(M.level_g)[l0 + i] / ldc(M.level_g)[l0]) * exp(-(dE / (KBOLTZMANN * T)));
    const int dZ = ldc(M.level_stage)[l0 + i] - ldc(M.level_stage)[l0];
    if (ldc(M.level_stage)[l0 + i] > 0) neutral = false;
#pragma unroll
    for (int d = 0; d < HSE_NDZ; d++)
      if (dZ == d) acc[d] += r;
    if (neutral) acc[HSE_NDZ] += r;
  }
#pragma unroll
  for (int d = 0; d <= HSE_NDZ; d++) g[d * gs] = acc[d];
}

// sum_d g[d] ci^d (ci = 1 / cNe_T)
__device__ __forceinline__ double hse_group_sum(const double *g, double ci) {
  double sum = 0.0, p = 1.0;
#pragma unroll
  for (int d = 0; d < HSE_NDZ; d++) {
    sum += g[d] * p;
    p *= ci;
  }
  return sum;
}

// What a layer's temperature fixes of the continuum opacity at wavelength ls
// (pyrh_Background, pyrh_background.c:256-400; no metal bound-free): the
// factors that multiply the densities of each absorber, to a[HSE_A_*] with
// stride as.  The H- terms carry the H- fudge factor.
__device__ void hse_opacity_factors(const DevModel &M, const DevHse &H, int ls, double T, double *a,
                                    int as) {
  const double *lc = M.lamconst + (int64_t) ls * RHG_LC_NCONST;
  const double C0 = Q_ELECTRON * Q_ELECTRON / (4.0 * PI * EPSILON_0) / sqrt(M_ELECTRON);
  const double sigma_ff = 4.0 / 3.0 * sqrt(2.0 * PI / (3.0 * KBOLTZMANN)) * (C0 * C0 * C0) /
                          (HPLANCK * CLIGHT);
  const double kT = KBOLTZMANN * T, stim = 1.0 - exp(-lc[RHG_LC_HC_KLA] / T);
  // H- bound-free, times n_H-
  a[HSE_A_HMBF * as] = lc[RHG_LC_HMIN_BF_ON] != 0.0
                           ? stim * lc[RHG_LC_HMIN_BF_ALPHA] * H.hmin_fudge : 0.0;
  // H- free-free, times n_H0 n_e
  double x;
  if (lc[RHG_LC_HMIN_FF_LIDX] >= 0.0) {
    const double ti = clamp_index(NTHETA, M.hminff_theta, THETA0 / T);
    x = 1.0E-29 * kT * bilinear(NTHETA, NFF, M.hminff_kappa, ti, lc[RHG_LC_HMIN_FF_LIDX]);
  } else {
    const double Ck = (KBOLTZMANN * THETA0 * 1.0E-32), sqrt_theta = sqrt(THETA0 / T);
    double theta_n = 1.0;
    x = 0.0;
    for (int n = 1; n < 6; n++) {
      theta_n *= sqrt_theta;
      x += theta_n * lc[RHG_LC_HFF_LONG0 + n - 1];
    }
    x *= Ck;
  }
  a[HSE_A_HMFF * as] = x * H.hmin_fudge;
  // OH and CH bound-free, times n_OH, n_CH
  auto molecule = [&](const double *Tt, const double *cross, int nT, int nE, double eidx) -> double {
    if (!(eidx >= 0.0) || T < ldc(Tt)[0] || T > ldc(Tt)[nT - 1]) return 0.0;
    const int i2 = locate_asc(nT, Tt, T);
    const double ti = (i2 == nT - 1) ? (double) i2
                                     : (double) i2 + (T - Tt[i2]) / (Tt[i2 + 1] - Tt[i2]);
    return stim * (exp(LG10 * bilinear(nT, nE, cross, ti, eidx)) * (CM_TO_M * CM_TO_M));
  };
  a[HSE_A_OH * as] = molecule(M.oh_T, M.oh_cross, NTOH, NEOH, lc[RHG_LC_OH_EIDX]);
  a[HSE_A_CH * as] = molecule(M.ch_T, M.ch_cross, NTCH, NECH, lc[RHG_LC_CH_EIDX]);
  // H free-free, times n_e n_p
  const double y = (lc[RHG_LC_GFF_CY] * T) / (HPLANCK * CLIGHT), x3 = lc[RHG_LC_GFF_X3];
  const double gIII = 1.0 + 0.1728 * x3 * (1.0 + y) - 0.0496 * (x3 * x3) * (1.0 + (1.0 + y) * 0.33333333 * y);
  a[HSE_A_HFF * as] = sigma_ff / sqrt(T) * lc[RHG_LC_HFF_NU3] * stim * ((gIII > 1.0) ? gIII : 1.0);
  // H2+ free-free, times n_H0 n_p
  x = 0.0;
  if (lc[RHG_LC_H2P_LIDX] >= 0.0) {
    const double ti = clamp_index(NTEMP_H2P, M.h2pff_temp, T);
    x = (1.0E-29 * 1.0E-20) * bilinear(NTEMP_H2P, NFF_H2P, M.h2pff_kappa, ti, lc[RHG_LC_H2P_LIDX]);
  }
  a[HSE_A_H2P * as] = x;
  // H2- free-free, times n_H2 n_e
  x = 0.0;
  if (lc[RHG_LC_H2M_LIDX] >= 0.0) {
    const double ti = clamp_index(NTHETA_H2, M.h2mff_theta, THETA0 / T);
    x = 1.0E-29 * kT * bilinear(NTHETA_H2, NFF_H2, M.h2mff_kappa, ti, lc[RHG_LC_H2M_LIDX]);
  }
  a[HSE_A_H2M * as] = x;
  // H bound-free (rh/hydrogen.c:150-208, active-layer branch), times the
  // ground-level density and 1 / cNe_T^d of the level's ionisation difference
  const int lH = ldc(M.atom_level_ptr)[0], cp0 = ldc(M.lam_cont_ptr)[ls], cp1 = ldc(M.lam_cont_ptr)[ls + 1];
  double g[HSE_NDZ];
#pragma unroll
  for (int d = 0; d < HSE_NDZ; d++) g[d] = 0.0;
  const double expla = exp(-lc[RHG_LC_BF_HC_KLA] / T);
  for (int e = cp0; e < cp1; e++) {
    const int ci = ldc(M.lam_cont_idx)[e];
    if (ldc(M.cont_atom)[ci] != 0) continue;
    const int i = ldc(M.cont_i)[ci], dZ = ldc(M.level_stage)[lH + i] - ldc(M.level_stage)[lH];
    const double dE = ldc(M.level_E)[lH + i] - ldc(M.level_E)[lH];
    const double r = i == 0 ? 1.0
                            : (ldc(M.level_g)[lH + i] / ldc(M.level_g)[lH]) * exp(-(dE / kT));
    const double t = ldc(M.lam_cont_alpha)[e] * (1.0 - expla) * r;
#pragma unroll
    for (int d = 0; d < HSE_NDZ; d++)
      if (dZ == d) g[d] += t;
  }
#pragma unroll
  for (int d = 0; d < HSE_NDZ; d++) a[(HSE_A_HBF + d) * as] = g[d];
}

// get_ne(fromscratch = TRUE) with hydrogen in LTE at one point: the starting
// value from hydrogen ionisation (pyrh_background.c:489-502; its partition
// function is that of neutral hydrogen, Solve_ne, rh/solvene.c:78-88), then
// Newton steps on charge conservation over every element's LTE ionisation
// fractions (getfjk, rh/solvene.c:145-197) and H-.  The quotients by sum1 and
// n_e are products with their reciprocals (a last-place difference).
__device__ double hse_get_ne(const DevModel &M, const DevHse &H, double T, double nHtot,
                             const HseT &tc) {
  const double kT = KBOLTZMANN * T;
  const Linear1At pf(M.npf, M.Tpf, T);
  const double PhiH = 0.5 * tc.p15 * tc.eH;
  double ne_old = (sqrt(1.0 + 4.0 * nHtot * PhiH) - 1.0) / (2.0 * PhiH), ne = ne_old;
  const double PhiHmin = 0.25 * tc.p15 * tc.eHmin;
  const double CTp = tc.pm15;
  for (int niter = 0; niter < HSE_N_MAX_ELECTRON_ITER; niter++) {
    const double CT_ne = 2.0 * CTp / ne_old, inv_ne = 1.0 / ne_old;
    double err = ne_old / nHtot, sum = 0.0;
    for (int e = 0; e < H.nel; e++) {
      const int ns = H.el_nstage[e];
      double u[NSTAGE_MAX], du[NSTAGE_MAX];
      u[0] = 1.0;
      du[0] = 0.0;
      double sum1 = 1.0, sum2 = 0.0;
      const double *lp = H.el_logpf + H.el_pf_ptr[e], *ip = H.el_ionpot + H.el_pf_ptr[e] / M.npf;
      double Uk = pf(lp);
#pragma unroll
      for (int j = 1; j < NSTAGE_MAX; j++) {
        u[j] = du[j] = 0.0;
        if (j < ns) {
          const double Ukp1 = pf(lp + j * M.npf);
          const double r = exp(Ukp1 - Uk - ip[j - 1] / kT);
          Uk = Ukp1;
          u[j] = u[j - 1] * CT_ne * r;
          du[j] = (double) (-j) * u[j] * inv_ne;
          sum1 += u[j];
          sum2 += du[j];
        }
      }
      const double inv1 = 1.0 / sum1;
      if (e == 0) {
        const double f0 = u[0] * inv1, df0 = (du[0] - f0 * sum2) * inv1;
        err += ne_old * f0 * PhiHmin;
        sum -= (f0 + ne_old * df0) * PhiHmin;
      }
      const double ab = H.el_abund[e];
#pragma unroll
      for (int j = 1; j < NSTAGE_MAX; j++) {
        if (j < ns) {
          const double f = u[j] * inv1, df = (du[j] - f * sum2) * inv1, akj = ab * j;
          err -= akj * f;
          sum += akj * df;
        }
      }
    }
    ne = ne_old - nHtot * err / (1.0 - nHtot * sum);
    const double dne = fabs((ne - ne_old) / ne_old);
    ne_old = ne;
    if (dne <= HSE_MAX_ELECTRON_ERROR) break;
  }
  return ne;
}

// The chain's view of one column: its lane group and the group's LDS.
struct HseGroup {
  int sub, lpc;              // lane in the group, lanes of the group
  uint64_t mask;             // the group's lanes in the wavefront
  double *rec;               // [H.nrec] what the layer's temperature fixes
  double *nm;                // [nmol] molecule densities
  const double *eab;         // [nel] abundances (shared by the workgroup)
  const int32_t *ecode;      // [nel] HSE_CODE_H | first stage slot << 4 | stages
  const uint32_t *mcnt;      // [nmol] count of nucleus i in bits 4 i
  const int32_t *mchg;       // [nmol] charge
};

__device__ __forceinline__ bool group_any(bool x, const HseGroup &G) {
  return (__ballot(x) & G.mask) != 0;
}

// hse_get_ne on the group's lanes: lane sub takes elements sub, sub + lpc, ...
// two at a time, with the stage factors of the layer's record (the elements
// are in order of their stage counts, so that lanes end their stages
// together).  With u_j = prod CT_ne r_j, s = sum u_j, A = sum j u_j and
// B = sum j^2 u_j, an element adds -ab A / s to the error and
// -ab (B - A^2 / s) / (s n_e) to its derivative (getfjk's sums over its
// stages, collected).
__device__ __forceinline__ double hse_group_ne(const DevHse &H, const HseGroup &G, double nHtot) {
  const double p15 = G.rec[HSE_T_P15];
  const double PhiH = 0.5 * p15 * G.rec[HSE_T_EH];
  double ne_old = (sqrt(1.0 + 4.0 * nHtot * PhiH) - 1.0) / (2.0 * PhiH), ne = ne_old;
  const double PhiHmin = 0.25 * p15 * G.rec[HSE_T_EHMIN];
  const double CT2 = 2.0 * G.rec[HSE_T_PM15], inv_nH = hrcp(nHtot);
  for (int niter = 0; niter < HSE_N_MAX_ELECTRON_ITER; niter++) {
    const double inv_ne = hrcp(ne_old), CT_ne = CT2 * inv_ne;
    double acc[2] = {(G.sub == 0) ? ne_old * inv_nH : 0.0, 0.0};
    for (int e0 = G.sub; e0 < H.nel; e0 += 2 * G.lpc) {
      const int e1 = e0 + G.lpc;
      const int c0 = G.ecode[e0], c1 = e1 < H.nel ? G.ecode[e1] : 1;
      const double ab0 = G.eab[e0], ab1 = e1 < H.nel ? G.eab[e1] : 0.0;
      const int n0 = c0 & 15, n1 = c1 & 15;
      const double *r0 = G.rec + ((c0 >> 4) & 0xffff) - 1, *r1 = G.rec + ((c1 >> 4) & 0xffff) - 1;
      double u0 = 1.0, s0 = 1.0, A0 = 0.0, B0 = 0.0, u1 = 1.0, s1 = 1.0, A1 = 0.0, B1 = 0.0;
      double fj = 0.0;
      for (int j = 1; j < n0; j++) {   // n1 <= n0
        fj += 1.0;
        const double fj2 = fj * fj;
        u0 *= CT_ne * r0[j];
        s0 += u0;
        A0 = fma(fj, u0, A0);
        B0 = fma(fj2, u0, B0);
        u1 *= j < n1 ? CT_ne * r1[j] : 0.0;
        s1 += u1;
        A1 = fma(fj, u1, A1);
        B1 = fma(fj2, u1, B1);
      }
      const double i0 = hrcp(s0), i1 = hrcp(s1), f0 = A0 * i0, f1 = A1 * i1;
      acc[0] -= ab0 * f0 + ab1 * f1;
      acc[1] -= (ab0 * (fma(-A0, f0, B0) * i0) + ab1 * (fma(-A1, f1, B1) * i1)) * inv_ne;
      // H-, from hydrogen's neutral fraction 1 / s and its derivative
      const double hi = (c0 & HSE_CODE_H) ? i0 : i1, hf = (c0 & HSE_CODE_H) ? f0 : f1;
      if ((c0 | c1) & HSE_CODE_H) {
        acc[0] += ne_old * hi * PhiHmin;
        acc[1] -= fma(hf, hi, hi) * PhiHmin;
      }
    }
    group_sum(acc, G.lpc);
    ne = ne_old - nHtot * acc[0] / (1.0 - nHtot * acc[1]);
    const bool done = fabs(ne - ne_old) <= HSE_MAX_ELECTRON_ERROR * fabs(ne_old);
    ne_old = ne;
    if (done) break;
  }
  return ne;
}

// Chemical equilibrium of one layer (rh/chemequil.c:107-393, the Newton
// iteration of chem_eq) with the molecules shared by the group's lanes.  The
// reduced system takes two sums over the molecules, with s_m the Saha product
// and c the counts: Q_i = sum c_i s_m, which completes the right-hand side
// (f1 - B f2 collapses to n_i - a_i + Q_i), and P_ij = sum c_i c_j s_m.  In
// y_i = x_i / n_i the system is (diag(n) + P) y = r, symmetric and for
// positive densities positive definite, so it takes an L D L^T factorisation
// without pivoting, which serves the solution and its refinement.
template <int NN>
__device__ __forceinline__ void hse_group_chem(const DevModel &M, const HseGroup &G, double ne,
                                               double nHtot, const double (&fn0)[NN],
                                               const double *phi, double fHmin,
                                               double (&nnuc)[NN]) {
  constexpr int NP = NN * (NN + 1) / 2;
  const int Nm = M.nmol;
  // up to 16 lanes share the molecules (the rows of a larger group alike)
  const int ml = G.lpc < 16 ? G.lpc : 16, ms = G.sub & (ml - 1);
  double a[NN];
#pragma unroll
  for (int i = 0; i < NN; i++) {
    a[i] = ldc(M.nucl_abund)[i] * nHtot;
    nnuc[i] = a[i];
  }
  for (int m = ms; m < Nm; m += ml) G.nm[m] = 0.0;
  const double inv_e = hrcp(ne);
  for (int niter = 1; niter <= N_MAX_CHEM_ITER; niter++) {
    double fn[NN], acc[NN + NP];
#pragma unroll
    for (int i = 0; i < NN; i++) fn[i] = fn0[i] * nnuc[i];
#pragma unroll
    for (int i = 0; i < NN + NP; i++) acc[i] = 0.0;
    auto saha = [&](int m, uint32_t cnt) {
      double sv = phi[m];
#pragma unroll
      for (int i = 0; i < NN; i++)
        for (int q = (cnt >> (4 * i)) & 15; q > 0; q--) sv *= fn[i];
      const int chg = G.mchg[m];
      for (int q = 0; q < chg; q++) sv *= inv_e;
      for (int q = 0; q < -chg; q++) sv *= ne;
      return sv;
    };
    for (int m = ms; m < Nm; m += ml) {
      const uint32_t cnt = G.mcnt[m];
      const double sv = saha(m, cnt);
      int p = NN;
#pragma unroll
      for (int i = 0; i < NN; i++) {
        const double cs = (double) ((cnt >> (4 * i)) & 15) * sv;
        acc[i] += cs;
#pragma unroll
        for (int j = i; j < NN; j++, p++) acc[p] = fma((double) ((cnt >> (4 * j)) & 15), cs, acc[p]);
      }
    }
    group_sum(acc, ml);
    // K = diag(n) + P, upper triangle; L D L^T with the factors U = L^T
    double K[NN][NN], U[NN][NN], inv[NN], r[NN], y[NN];
    {
      int p = NN;
#pragma unroll
      for (int i = 0; i < NN; i++)
#pragma unroll
        for (int j = i; j < NN; j++, p++) K[i][j] = i == j ? acc[p] + nnuc[i] : acc[p];
    }
    K[0][0] += fHmin * nnuc[0];
#pragma unroll
    for (int i = 0; i < NN; i++) {
      r[i] = nnuc[i] - a[i] + acc[i];
      if (i == 0) r[0] += fHmin * nnuc[0];
    }
    {
      double W[NN][NN];
#pragma unroll
      for (int i = 0; i < NN; i++)
#pragma unroll
        for (int j = i; j < NN; j++) W[i][j] = K[i][j];
#pragma unroll
      for (int j = 0; j < NN; j++) {
        inv[j] = hrcp(W[j][j]);
#pragma unroll
        for (int i = j + 1; i < NN; i++) {
          U[j][i] = W[j][i] * inv[j];
#pragma unroll
          for (int k = i; k < NN; k++) W[i][k] = fma(-U[j][i], W[j][k], W[i][k]);
        }
      }
    }
    auto solve = [&](double (&b)[NN]) {
#pragma unroll
      for (int j = 0; j < NN; j++)
#pragma unroll
        for (int i = j + 1; i < NN; i++) b[i] = fma(-U[j][i], b[j], b[i]);
#pragma unroll
      for (int i = NN - 1; i >= 0; i--) {
        b[i] *= inv[i];
#pragma unroll
        for (int k = i + 1; k < NN; k++) b[i] = fma(-U[i][k], b[k], b[i]);
      }
    };
#pragma unroll
    for (int i = 0; i < NN; i++) y[i] = r[i];
    solve(y);
    {
      double res[NN];
#pragma unroll
      for (int i = 0; i < NN; i++) {
        res[i] = r[i];
#pragma unroll
        for (int j = 0; j < NN; j++) res[i] = fma(j < i ? -K[j][i] : -K[i][j], y[j], res[i]);
      }
      solve(res);
#pragma unroll
      for (int i = 0; i < NN; i++) y[i] += res[i];
    }
    // back substitution for the molecules; another iteration while a density
    // changes by more than the limit (rh/maxchange.c:32-50 over the last two
    // solutions)
    bool more = false;
    for (int m = ms; m < Nm; m += ml) {
      const uint32_t cnt = G.mcnt[m];
      const double sv = saha(m, cnt), nold = G.nm[m];
      double t = 0.0;
#pragma unroll
      for (int j = 0; j < NN; j++) t = fma((double) ((cnt >> (4 * j)) & 15), y[j], t);
      const double nnew = nold - ((nold - sv) + sv * t);
      G.nm[m] = nnew;
      if (nnew != 0.0 && fabs(nnew - nold) > CHEM_ITER_LIMIT * fabs(nnew)) more = true;
    }
#pragma unroll
    for (int i = 0; i < NN; i++) {
      const double nold = nnuc[i];
      nnuc[i] -= y[i] * nold;
      if (nnuc[i] != 0.0 && fabs(nnuc[i] - nold) > CHEM_ITER_LIMIT * fabs(nnuc[i])) more = true;
    }
    if (!group_any(more, G)) break;
  }
  wave_sync();
}

// One pass of the layer loop body (pyrh_hse.c:226-238, :295-307): n_e, and
// when the pressure step needs it (tau500 scale) the LTE populations
// (SetLTEQuantities, rh/ltepops.c:33-113 for the atoms that matter here:
// the molecule nuclei, hydrogen, helium), chemical equilibrium and the
// continuum opacity with the scattering (Thomson, Rayleigh on H, He, H2).
template <int NN>
__device__ __forceinline__ void hse_layer(const DevModel &M, const DevHse &H, const HseGroup &G,
                                          double nHtot, bool opacity, double &ne_out,
                                          double &opac_out) {
  const double ne = hse_group_ne(H, G, nHtot);
  ne_out = ne;
  if (!opacity) return;
  const double *rec = G.rec, *lg = rec + HSE_NMISC, *phi = lg + (NN + 1) * (HSE_NDZ + 1);
  const double p15 = rec[HSE_T_P15], ci = hrcp(0.5 * ne * p15);
  double nstar0n[NN], fn0[NN], nnuc[NN], fracn[NN];
#pragma unroll
  for (int i = 0; i < NN; i++) {
    const double *g = lg + i * (HSE_NDZ + 1);
    const double ntot = ldc(M.atom_abund)[ldc(M.nucl_atom)[i]] * nHtot;
    const double inv = hrcp(1.0 + hse_group_sum(g, ci));
    nstar0n[i] = ntot * inv;
    fn0[i] = inv + g[HSE_NDZ] * inv;
  }
  const double PhiHmin = 0.25 * p15 * rec[HSE_T_EHMIN];
  hse_group_chem<NN>(M, G, ne, nHtot, fn0, phi, ne * fn0[0] * PhiHmin, nnuc);
#pragma unroll
  for (int i = 0; i < NN; i++) fracn[i] = nnuc[i] / (ldc(M.atom_abund)[ldc(M.nucl_atom)[i]] * nHtot);
  const double nH0 = nstar0n[0] * fracn[0];
  double np = rec[HSE_T_NP];
  for (int m = 0; m < H.np_dz; m++) np *= ci;
  np *= nH0;
  const double nHmin = ne * (nnuc[0] * PhiHmin);
  const double nH2 = M.mol_h2 >= 0 ? G.nm[M.mol_h2] : 0.0;
  const double nOH = M.mol_oh >= 0 ? G.nm[M.mol_oh] : 0.0;
  const double nCH = M.mol_ch >= 0 ? G.nm[M.mol_ch] : 0.0;
  double sca = ne * H.sigma_thomson;
  if (H.ray_H > 0.0) sca += H.ray_H * nH0;
  if (H.he_atom >= 0 && H.ray_He > 0.0) {
    double nHe0 = (ldc(M.atom_abund)[H.he_atom] * nHtot) *
                  hrcp(1.0 + hse_group_sum(lg + NN * (HSE_NDZ + 1), ci));
#pragma unroll
    for (int i = 0; i < NN; i++)
      if (ldc(M.nucl_atom)[i] == H.he_atom) nHe0 = nstar0n[i] * fracn[i];
    sca += H.ray_He * nHe0;
  }
  if (H.ray_H2 > 0.0) sca += H.ray_H2 * nH2;
  const double *a = rec + HSE_A0;
  double total = nHmin * a[HSE_A_HMBF] + (nH0 * ne) * a[HSE_A_HMFF];
  total += nOH * a[HSE_A_OH] + nCH * a[HSE_A_CH];
  total += nH0 * hse_group_sum(a + HSE_A_HBF, ci);
  total += (ne * np) * a[HSE_A_HFF] + (nH0 * np) * a[HSE_A_H2P];
  if (nH2 > 0.0) total += (nH2 * ne) * a[HSE_A_H2M];
  opac_out = total + sca * H.scatt_fudge;
  // the molecule densities are read before the next pass rewrites them
  wave_sync();
}

}  // namespace

// What each (column, depth)'s temperature fixes, to tab[point * H.nrec + slot]
// (point = column of the chunk * Nmax + depth): 64 points x one segment of at
// most HSE_SEG slots per workgroup, so that a single column's 82 depths still
// make some 60 workgroups.  A segment is one of
//   stages     r = exp(U_j - U_{j-1} - chi_{j-1}/kT) of HSE_SEG (element,
//              stage) pairs (getfjk, rh/solvene.c:180-190; U from
//              getKuruczpf = Linear on Tpf, rh/solvene.c:202-211)
//   groups     hse_level_groups of one atom
//   molecules  equilibrium constants
//   misc       HSE_T_* and the opacity factors
// Lanes are points, so all lanes take the same branch; the slots go through
// LDS so that the record is written in runs.
__global__ void __launch_bounds__(HSE_BLOCK)
k_hse_tables(const DevModel *__restrict__ Mp, DevHse H, int npts, int Nmax,
             const int32_t *__restrict__ ndep, const double *__restrict__ temp,
             double *__restrict__ tab) {
  const DevModel &M = *Mp;
  __shared__ double buf[HSE_SEG][HSE_BLOCK + 1];
  const int lane = threadIdx.x, p0 = blockIdx.x * HSE_BLOCK, p = p0 + lane;
  const CInt *sg = ldc(H.seg) + 4 * blockIdx.y;
  const int kind = sg[0], first = sg[1], n = sg[2], slot0 = sg[3];
  if (p < npts && p % Nmax < ndep[p / Nmax]) {
    const double T = temp[p];
    double *b = &buf[0][lane];
    constexpr int bs = HSE_BLOCK + 1;
    if (kind == HSE_SEG_STAGES) {
      const Linear1At pf(M.npf, M.Tpf, T);
      const double kT = KBOLTZMANN * T;
      for (int s = 0; s < n; s++) {
        const int o = ldc(H.sl_pf)[first + s];
        const double *lp = H.el_logpf + o;
        b[s * bs] = exp(pf(lp + M.npf) - pf(lp) - ldc(H.sl_ip)[first + s] / kT);
      }
    } else if (kind == HSE_SEG_GROUPS) {
      hse_level_groups(M, first, T, b, bs);
    } else if (kind == HSE_SEG_MOLECULES) {
      for (int s = 0; s < n; s++) b[s * bs] = equilconstant(M, first + s, T);
    } else {
      const HseT t = hse_tcache(H, T, 0.0);
      b[HSE_T_P15 * bs] = t.p15;
      b[HSE_T_EHMIN * bs] = t.eHmin;
      b[HSE_T_PM15 * bs] = t.pm15;
      b[HSE_T_EH * bs] = t.eH;
      const int l0 = ldc(M.atom_level_ptr)[0], l1 = ldc(M.atom_level_ptr)[1] - 1;
      b[HSE_T_NP * bs] = l1 == l0 ? 1.0 : (ldc(M.level_g)[l1] / ldc(M.level_g)[l0]) *
                             exp(-((ldc(M.level_E)[l1] - ldc(M.level_E)[l0]) / (KBOLTZMANN * T)));
      hse_opacity_factors(M, H, H.lam_index, T, b + HSE_A0 * bs, bs);
    }
  }
  __syncthreads();
  for (int i = lane; i < n * HSE_BLOCK; i += HSE_BLOCK) {
    const int q = i / n, s = i % n;
    if (p0 + q < npts) tab[(int64_t) (p0 + q) * H.nrec + slot0 + s] = buf[s][q];
  }
}

// The layer chain: bound by its length for few columns (one of 82 layers:
// 2.0 ms, 15.3 with every exponential inside the chain and 16 lanes) and by
// instruction issue for many (16384: 7.0 ms and 2.7 for the tables, 31.4
// before).  185 VGPRs: two waves per SIMD; a bound of three spills.
template <int NN>
__global__ void __launch_bounds__(HSE_BLOCK, 2)
k_hse(const DevModel *__restrict__ Mp, DevHse H, int lpc, int cpb, int ncol, int Nmax,
      const int32_t *__restrict__ ndep, int atm_scale, const double *__restrict__ scale,
      const double *__restrict__ temp, const double *__restrict__ pg_top,
      const double *__restrict__ tab, double *__restrict__ ne_out, double *__restrict__ nH_out,
      double *__restrict__ rho_out, double *__restrict__ pg_out, int32_t *__restrict__ niter_out) {
  const DevModel &M = *Mp;
  // LDS: abundances [nel], element codes [nel], molecule counts and charges
  // [nmol], then per column its record and molecule densities
  extern __shared__ double lds[];
  double *eab = lds;
  int32_t *ecode = (int32_t *) (eab + H.nel);
  uint32_t *mcnt = (uint32_t *) (ecode + H.nel);
  int32_t *mchg = (int32_t *) (mcnt + M.nmol);
  for (int e = threadIdx.x; e < H.nel; e += HSE_BLOCK) {
    ecode[e] = H.el_code[e];
    eab[e] = H.el_ab[e];
  }
  for (int m = threadIdx.x; m < M.nmol; m += HSE_BLOCK) {
    uint32_t c = 0;
    for (int i = 0; i < NN; i++) c |= (uint32_t) M.mol_cnt[m * NNUC_MAX + i] << (4 * i);
    mcnt[m] = c;
    mchg[m] = M.mol_charge[m];
  }
  __syncthreads();
  const int grp = threadIdx.x / lpc, sub = threadIdx.x % lpc;
  const int ic = blockIdx.x * cpb + grp;
  if (grp >= cpb || ic >= ncol) return;
  HseGroup G;
  G.sub = sub;
  G.lpc = lpc;
  G.mask = (lpc == 64 ? ~0ull : (1ull << lpc) - 1) << (grp * lpc);
  G.rec = lds + H.lds_col0 + grp * H.lds_col;
  G.nm = G.rec + H.nrec;
  G.eab = eab;
  G.ecode = ecode;
  G.mcnt = mcnt;
  G.mchg = mchg;
  const int N = ndep[ic];
  const int64_t o = (int64_t) ic * Nmax;
  const double *sc = scale + o, *Tc = temp + o, *rc = tab + o * H.nrec;
  const bool store = (sub == 0);
  const bool tau = (atm_scale == 0);
  const double g = M.gravity, LOG10 = log(10.0), wH = AMU * M.wght_per_H;
  const double tA = M.totalAbund;
  auto load = [&](int k) {
    wave_sync();
    const double *r = rc + (int64_t) k * H.nrec;
#pragma unroll 8
    for (int s = sub; s < H.nrec; s += lpc) G.rec[s] = r[s];
    wave_sync();
  };

  // the top layer (pyrh_hse.c:210-273; p_g is given) and the layers below
  // (pyrh_hse.c:278-351)
  double pg = pg_top[ic], ne = 0.0, opac = 0.0, rho = 0.0, z_prev = 0.0;
  for (int k = 0; k < N; k++) {
    const double z = tau ? pow10d(sc[k]) : sc[k] * KM_TO_M;
    const double T = Tc[k];
    load(k);
    const double pg_prev = pg, rho_prev = rho, ne_prev = ne;
    double dlogtau = 0.0, beta1 = 0.0;
    if (k > 0) {
      if (tau) {
        const double q = rho / opac;
        pg += g * rho / opac * (z - z_prev);
        beta1 = q * z_prev;
        dlogtau = log10(z) - log10(z_prev);
      } else {
        pg += g * rho * (z_prev - z);
      }
    }
    double nH = (pg / KBOLTZMANN / T - ne_prev) / tA;
    int iter = 0;
    while (iter < H.nmax_iter) {
      rho = wH * nH;
      hse_layer<NN>(M, H, G, nH, tau, ne, opac);
      if (k > 0) {
        if (tau) pg = pg_prev + LOG10 * g * (rho / opac * z + beta1) / 2 * dlogtau;
        else pg = pg_prev + g * (z_prev - z) * sqrt(rho * rho_prev);
      }
      const double old = nH;
      nH = (pg / KBOLTZMANN / T - ne) / tA;
      iter++;
      if (fabs(hdiv(nH - old, nH)) <= H.iter_limit) break;
    }
    if (store) {
      ne_out[o + k] = ne;
      nH_out[o + k] = nH;
      rho_out[o + k] = rho;
      pg_out[o + k] = pg;
      if (niter_out) niter_out[o + k] = iter;
    }
    z_prev = z;
  }
  if (store) {
    for (int k = N; k < Nmax; k++) {
      ne_out[o + k] = 0.0;
      nH_out[o + k] = 0.0;
      rho_out[o + k] = 0.0;
      pg_out[o + k] = 0.0;
      if (niter_out) niter_out[o + k] = 0;
    }
  }
}

// get_ne_from_nH (rh/rhf1d/pyrh_hse.c:555-678): n_e at every (column,
// depth) point from T and n_Htot in cm^-3 (Solve_ne from scratch,
// rh/solvene.c:53-135), one point per lane; n_e returned in cm^-3 as the
// entry point converts back (and zero past ndep).
__global__ void __launch_bounds__(HSE_BLOCK)
k_ne_from_nh(const DevModel *__restrict__ Mp, DevHse H, int ncol, int Nmax,
             const int32_t *__restrict__ ndep, const double *__restrict__ temp,
             const double *__restrict__ nH, double *__restrict__ ne_out) {
  const DevModel &M = *Mp;
  const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (int64_t) ncol * Nmax) return;
  const int ic = (int) (gid / Nmax), k = (int) (gid % Nmax);
  if (k >= ndep[ic]) {
    ne_out[gid] = 0.0;
    return;
  }
  const double CUBE_CM = CM_TO_M * CM_TO_M * CM_TO_M;
  const double T = temp[gid], nHtot = nH[gid] / CUBE_CM;
  const double Uk = linear1(M.npf, M.Tpf, H.el_logpf, T);
  ne_out[gid] = hse_get_ne(M, H, T, nHtot, hse_tcache(H, T, Uk)) * CUBE_CM;
}

#define RHG_INST_HSE(NN)                                                                         \
  template __global__ void k_hse<NN>(const DevModel *, DevHse, int, int, int, int,               \
                                     const int32_t *, int, const double *, const double *,       \
                                     const double *, const double *, double *, double *,         \
                                     double *, double *, int32_t *);
RHG_INST_HSE(1)
RHG_INST_HSE(2)
RHG_INST_HSE(3)
RHG_INST_HSE(4)
RHG_INST_HSE(5)
RHG_INST_HSE(6)
RHG_INST_HSE(7)
RHG_INST_HSE(8)
#undef RHG_INST_HSE

}  // namespace rhg
