// NLTE populations of one active atom per column: the accelerated lambda
// iteration of rhf1d() (rh/iterate.c:48-143) as a sequence of batched
// kernels over all columns at once.
//
// The iteration's arrays are depth-fastest and its kernels put a column's
// depths on consecutive lanes.  One column is then hundreds of wavefronts
// rather than one lane of each (the iteration of a single column used to be
// as long as that of 1500), and the only serial chains left are a wavefront
// scan (the short-characteristic recursion is affine in I) and the Feautrier
// elimination.
//
// Set-up (once per batch, after k_state of the background model)
//   k_nlte_pre      (column, depth): scattering opacity at the reference
//                   wavelength (the depth scale), LTE populations, Doppler
//                   widths, damping and the collision matrix.
//   k_nlte_bg       depth-fastest copies of the column state's fields and of
//                   the LTE continuum, with the scattering opacity added.
//   k_nlte_profile  (column, depth, line, wavelength): absorption profiles
//                   for every ray and direction; k_nlte_wphi: their
//                   normalisation.
// Iteration (per pass, over the columns still iterating)
//   k_nlte_bezier   (column, wavelength with a line): the rays of the
//   k_nlte_feautrier (column, continuum-only wavelength)
//                   wavelength with the diagonal operator; new mean
//                   intensity and, with the operator, the radiative rate
//                   terms of every transition active there.
//   k_nlte_stateq   (column, depth): rate matrix = collisions + the rate
//                   terms summed over the transitions' wavelengths; the
//                   statistical-equilibrium solve.
//   k_nlte_ng       (column): Ng acceleration and the maximum relative
//                   change.
#include "rhg_nlte.hpp"

namespace rhg {

namespace {

// rh/planck.c:38-63 for a wavelength in nm
__device__ __forceinline__ double planck_lam(double T, double lambda) {
  const double hc_kla = (HPLANCK * CLIGHT) / (KBOLTZMANN * NM_TO_M * lambda);
  const double twohnu3_c2 = (2.0 * HPLANCK * CLIGHT) / ((NM_TO_M * lambda) * (NM_TO_M * lambda) *
                                                         (NM_TO_M * lambda));
  const double hc_Tkla = hc_kla / T;
  return (hc_Tkla <= MAX_EXPONENT) ? twohnu3_c2 / (exp(hc_Tkla) - 1.0) : 0.0;
}

// 1 / b and a / b by the hardware reciprocal estimate refined by two Newton
// steps (relative error ~1e-16, not correctly rounded): the quotients of the
// rays, where the IEEE division sequence is a long dependent chain per use
__device__ __forceinline__ double nrcp(double b) {
  double r = __builtin_amdgcn_rcp(b);
  double e = fma(-b, r, 1.0);
  r = fma(r, e, r);
  e = fma(-b, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ double ndiv(double a, double b) { return a * nrcp(b); }

// Fritsch & Butland monotone derivative, rh/bezier_aux.c:34-51, from the
// slopes of the two intervals and alpha = (1 + dn / (up + dn)) / 3
__device__ __forceinline__ double monotone(double f_up, double f_dn, double alpha) {
  const double p = f_up * f_dn;
  return p > 0.0 ? p * nrcp(fma(alpha, f_dn, (1.0 - alpha) * f_up)) : 0.0;
}

// x of the lane `ctrl` names, or `old` where there is none
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp(double old, double x) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(x), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(x), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}
// x of the previous / the next lane (0 where there is none)
template <int CTRL>
__device__ __forceinline__ double shift(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_prev(double x) { return shift<0x138>(x); }   // wave_shr:1
__device__ __forceinline__ double from_next(double x) { return shift<0x130>(x); }   // wave_shl:1

// LDS written by some lanes of the wavefront is read by others after this
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double max0(double x) { return x > 0.0 ? x : 0.0; }

// RH's splineEval with precomputed second derivatives, rh/spline.c:70-97
__device__ double spline_eval_M(int n, const double *x, const double *y, const double *Mv,
                                double xv) {
  if (xv <= x[0]) return y[0];
  if (xv >= x[n - 1]) return y[n - 1];
  const int j = locate_asc(n, x, xv);
  const double hj = x[j + 1] - x[j];
  const double fx = (xv - x[j]) / hj;
  const double fx1 = 1 - fx;
  return fx1 * y[j] + fx * y[j + 1] +
         (fx1 * (fx1 * fx1 - 1) * Mv[j] + fx * (fx * fx - 1) * Mv[j + 1]) * (hj * hj) / 6.0;
}

constexpr double HC = HPLANCK * CLIGHT;
constexpr double FOURPI = 4.0 * PI;
constexpr double HC_4PI = HC / FOURPI;

}  // namespace

// ---------------------------------------------------------------------------
// Set-up per (column, depth).  Scattering opacity at the reference
// wavelength joins chi_ref before convertScales (rh/background.c:461-463);
// LTE populations of the active atom (rh/ltepops.c:33-113), its total and
// Doppler width (rh/readatom.c:213-220); damping of each line
// (rh/broad.c:273-316); collision rates (rh/collision.c:450-760).
__global__ void k_nlte_pre(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap,
                           NlteBufs B) {
  const DevModel &M = *Mp;
  const DevNlte &A = *Ap;
  const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  const int ncol = B.ncol, Nmax = B.Nmax;
  if (p >= (int64_t) ncol * Nmax) return;
  const int k = (int) (p % Nmax), ic = (int) (p / Nmax);
  if (k >= B.ndep[ic]) return;
  const int64_t ss = (int64_t) Nmax * ncol, fs = B.fs;
  double *st = B.state + (int64_t) k * ncol + ic;
  const double T = st[RHG_CF_T * ss], ne = st[RHG_CF_NE * ss], nHtot = st[RHG_CF_NHTOT * ss];
  const double nH0 = st[RHG_CF_NH0 * ss], np = st[RHG_CF_NP * ss], nH2 = st[RHG_CF_NH2 * ss];
  const double vturb = st[RHG_CF_VTURB * ss];
  const double c1 = (HPLANCK / (2.0 * PI * M_ELECTRON)) * (HPLANCK / KBOLTZMANN);
  const double cNe_T = 0.5 * ne * pow(c1 / T, 1.5);
  const int64_t pk = (int64_t) ic * B.Kp + k;

  double nHe = 0.0;
  if (A.he_atom >= 0) {
    const int l0 = ldc(M.atom_level_ptr)[A.he_atom], nl = ldc(M.atom_level_ptr)[A.he_atom + 1] - l0;
    nHe = (ldc(M.atom_abund)[A.he_atom] * nHtot) / atom_sum(M, l0, nl, T, cNe_T);
  }
  B.nHe[pk] = nHe;
  {
    const int lr = M.ref_index;
    double sca = ne * A.sigma_thomson;
    sca += A.ray_H[lr] * nH0;
    if (A.he_atom >= 0) sca += A.ray_He[lr] * nHe;
    sca += A.ray_H2[lr] * nH2;
    sca *= ldc(M.lamconst)[(int64_t) lr * RHG_LC_NCONST + RHG_LC_SCATT_FUDGE];
    st[RHG_CF_HEIGHT * ss] += sca;
  }

  const int nl = A.nl, a = A.atom_index, l0 = ldc(M.atom_level_ptr)[a];
  const double ntotal = ldc(M.atom_abund)[a] * nHtot;
  const double n0 = ntotal / atom_sum(M, l0, nl, T, cNe_T);
  for (int i = 0; i < nl; i++) {
    const double ns = (i == 0) ? n0 : level_ratio(M, l0, i, T, cNe_T) * n0;
    B.nstar[(int64_t) i * fs + pk] = ns;
    B.pops[(int64_t) i * fs + pk] = ns;
  }
  B.ntot[pk] = ntotal;
  const double vtherm = 2.0 * KBOLTZMANN / (AMU * A.weight);
  const double vbroad = sqrt(vtherm * T + vturb * vturb);
  B.vbroad[pk] = vbroad;

  for (int l = 0; l < A.nline; l++) {
    const double cDop = (NM_TO_M * A.ln_lambda0[l]) / (4.0 * PI);
    double Qelast = 0.0;
    if (A.ln_vdw[l]) {
      // rh/broad.c:87-100 (Unsold), 125-136 (Barklem), 145
      double G = A.ln_vdw[l] == 2
                     ? A.ln_vdw_cross[l] * pow(T, (1.0 - A.ln_vdw_alpha[l]) / 2.0) +
                           A.ln_vdw_cross_he[l] * pow(T, 0.3)
                     : A.ln_vdw_cross[l] * pow(T, 0.3);
      G *= nH0;
      Qelast += G;
    }
    if (A.ln_stark[l] == 1) {
      Qelast += A.ln_stark_c[l] * ne;
    } else if (A.ln_stark[l] == 2) {
      const double vrel = pow(A.ln_stark_C[l] * T, 0.16666667) * A.ln_stark_Cm[l];
      Qelast += A.ln_stark_c[l] * vrel * ne;
    }
    B.adamp[(int64_t) l * fs + pk] = (A.ln_Grad[l] + Qelast) * cDop / vbroad;
  }

  for (int q = 0; q < nl * nl; q++) B.Cmat[(int64_t) q * fs + pk] = 0.0;
  const double C0 = ((E_RYDBERG / sqrt(M_ELECTRON)) * PI * (RBOHR * RBOHR)) *
                    sqrt(8.0 / (PI * KBOLTZMANN));
  for (int r = 0; r < A.ncoll; r++) {
    const int i1 = A.coll_i[r], j1 = A.coll_j[r], c0 = A.coll_ptr[r], nT = A.coll_ptr[r + 1] - c0;
    const double Cv = nT > 2 ? spline_eval_M(nT, A.coll_T + c0, A.coll_c + c0, A.coll_M + c0, T)
                             : linear1(nT, A.coll_T + c0, A.coll_c + c0, T);
    double *Cij = B.Cmat + (int64_t) (i1 * nl + j1) * fs + pk;
    double *Cji = B.Cmat + (int64_t) (j1 * nl + i1) * fs + pk;
    const double nsi = B.nstar[(int64_t) i1 * fs + pk], nsj = B.nstar[(int64_t) j1 * fs + pk];
    double Cdown, Cup;
    switch (A.coll_type[r]) {
      case 0:   // OMEGA
        Cdown = C0 * ne * Cv / (A.g[j1] * sqrt(T));
        *Cij += Cdown;
        *Cji += Cdown * nsj / nsi;
        break;
      case 1:   // CE
        Cdown = Cv * ne * (A.g[i1] / A.g[j1]) * sqrt(T);
        *Cij += Cdown;
        *Cji += Cdown * nsj / nsi;
        break;
      case 2:   // CI
        Cup = Cv * ne * exp(-(A.E[j1] - A.E[i1]) / (KBOLTZMANN * T)) * sqrt(T);
        *Cji += Cup;
        *Cij += Cup * nsi / nsj;
        break;
      case 3:   // CP
        Cdown = np * Cv;
        *Cij += Cdown;
        *Cji += Cdown * nsj / nsi;
        break;
      case 4:   // CH
        Cup = nH0 * Cv;
        *Cji += Cup;
        *Cij += Cup * nsi / nsj;
        break;
      case 5:   // CH0
        *Cij += nH0 * Cv;
        break;
      case 6:   // CH+
        *Cji += np * Cv;
        break;
    }
  }
}

// Depth-fastest copies: row io < nout is the output wavelength's LTE
// continuum with the scattering opacity (Thomson and Rayleigh on H, He and
// H2, rh/background.c:342-465), its emissivity and the scattering opacity;
// rows nout .. nout + NG_N - 1 are the column state's fields of NG_*.  One
// 32 x 32 tile (columns x depths) of a row per workgroup of 256 threads,
// turned in LDS, so that the column-fastest reads and the depth-fastest
// writes are both in runs.
__global__ void __launch_bounds__(256)
k_nlte_bg(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap, NlteBufs B,
          const int32_t *__restrict__ out_ls) {
  const DevNlte &A = *Ap;
  const DevModel &M = *Mp;
  const int ncol = B.ncol, Nmax = B.Nmax, nrow = B.nout + NG_N;
  const int row = (int) (blockIdx.x % nrow), tile = (int) (blockIdx.x / nrow);
  const int nkt = (Nmax + 31) / 32, c0 = tile / nkt * 32, k0 = tile % nkt * 32;
  const int64_t ss = (int64_t) Nmax * ncol;
  __shared__ double t[3][32][33];
  const bool wave = row < B.nout;
  const int ls = wave ? out_ls[row] : 0;
  for (int i = threadIdx.x; i < 1024; i += 256) {
    const int c = i % 32, k = i / 32, ic = c0 + c, kk = k0 + k;
    if (ic >= ncol || kk >= Nmax || kk >= B.ndep[ic]) continue;
    const double *st = B.state + (int64_t) kk * ncol + ic;
    if (wave) {
      double sca = st[RHG_CF_NE * ss] * A.sigma_thomson;
      sca += A.ray_H[ls] * st[RHG_CF_NH0 * ss];
      if (A.he_atom >= 0) sca += A.ray_He[ls] * B.nHe[(int64_t) ic * B.Kp + kk];
      sca += A.ray_H2[ls] * st[RHG_CF_NH2 * ss];
      // the scattering fudge factor, rh/background.c:453-462
      sca *= ldc(M.lamconst)[(int64_t) ls * RHG_LC_NCONST + RHG_LC_SCATT_FUDGE];
      const int64_t q = (int64_t) row * ss + (int64_t) kk * ncol + ic;
      t[0][k][c] = B.lte_chi[q] + sca;
      t[1][k][c] = B.lte_eta[q];
      t[2][k][c] = sca;
    } else {
      const int f = row - B.nout;
      t[0][k][c] = st[(f == NG_T ? RHG_CF_T : f == NG_VLOS ? RHG_CF_VLOS
                       : f == NG_DZ ? RHG_CF_DZ : RHG_CF_HEIGHT) * ss];
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 1024; i += 256) {
    const int k = i % 32, c = i / 32, ic = c0 + c, kk = k0 + k;
    if (ic >= ncol || kk >= Nmax || kk >= B.ndep[ic]) continue;
    const int64_t pk = (int64_t) ic * B.Kp + kk;
    if (wave) {
      const int64_t q = (int64_t) row * B.fs + pk;
      B.cchi[q] = t[0][k][c];
      B.ceta[q] = t[1][k][c];
      B.csca[q] = t[2][k][c];
    } else {
      B.geo[(int64_t) (row - B.nout) * B.fs + pk] = t[0][k][c];
    }
  }
}

// Field-free absorption profiles of the atom's lines for every ray and
// direction, rh/profile.c:67-371 (Voigt function of Armstrong,
// rh/voigt.c:126-243), one (column, depth) x (line, wavelength) per thread,
// and into the rate accumulators (unused until the first iteration) the
// wavelength's part of the normalisation integral.  Row
// blockIdx.x % nphi of the lines' wavelengths is grid point la of line l.
__global__ void k_nlte_profile(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap,
                               NlteBufs B) {
  const DevModel &M = *Mp;
  const DevNlte &A = *Ap;
  const int ncol = B.ncol, Nmax = B.Nmax, row = (int) (blockIdx.x % A.nphi);
  const int64_t p = (int64_t) (blockIdx.x / A.nphi) * blockDim.x + threadIdx.x;
  if (p >= (int64_t) ncol * Nmax) return;
  const int k = (int) (p % Nmax), ic = (int) (p / Nmax);
  if (k >= B.ndep[ic]) return;
  int l = 0;
  while (l + 1 < A.nline && row >= A.ln_phi[l + 1]) l++;
  const int la = row - A.ln_phi[l];
  const int64_t fs = B.fs, pk = (int64_t) ic * B.Kp + k;
  const double vb = B.vbroad[pk], vz = B.geo[NG_VLOS * fs + pk];
  const double adamp = B.adamp[(int64_t) l * fs + pk];
  const int t = A.ln_tr[l], nrays = A.nrays;
  const double lambda0 = A.ln_lambda0[l];
  const int ls = A.tr_nblue[t] + la;
  const double lamla = ldc(M.lamconst)[(int64_t) ls * RHG_LC_NCONST + RHG_LC_LAMBDA];
  const double wl = A.tr_wlam[A.tr_ptr[t] + la];
  const double v = (lamla - lambda0 - 0.0) * CLIGHT / (vb * lambda0);
  double wphi = 0.0;
  for (int mu = 0; mu < nrays; mu++) {
    const double wlamu = wl * 0.5 * A.wmu[mu];
    const double vlos = A.muz[mu] * vz / vb;
    for (int to_obs = 0; to_obs <= 1; to_obs++) {
      const double sign = to_obs ? 1.0 : -1.0;
      const double vk = v + sign * vlos;
      const double ph = voigt_armstrong(adamp, vk) * 1.0 / (SQRTPI * vb);
      B.phi[((int64_t) (row * nrays + mu) * 2 + to_obs) * fs + pk] = ph;
      wphi += ph * wlamu;
    }
  }
  B.acc[(int64_t) row * fs + pk] = wphi;
}

// 1 / the profile's integral over its quadrature, one (column, depth, line)
// per thread
__global__ void k_nlte_wphi(const DevNlte *__restrict__ Ap, NlteBufs B) {
  const DevNlte &A = *Ap;
  const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  const int Nmax = B.Nmax, l = blockIdx.y;
  if (p >= (int64_t) B.ncol * Nmax) return;
  const int k = (int) (p % Nmax), ic = (int) (p / Nmax);
  if (k >= B.ndep[ic]) return;
  const int64_t pk = (int64_t) ic * B.Kp + k;
  const int n = A.tr_nlam[A.ln_tr[l]];
  const double *w = B.acc + (int64_t) A.ln_phi[l] * B.fs + pk;
  double sum = 0.0;
#pragma unroll 8
  for (int la = 0; la < n; la++) sum += w[(int64_t) la * B.fs];
  B.wphi[(int64_t) l * B.fs + pk] = 1.0 / sum;
}

// ---------------------------------------------------------------------------
// Radiative rate terms at one depth for the rays of one direction
// (addtoCoupling and addtoGamma, rh/fillgamma.c:82-332), summed over the
// rays.  The members of the active set are described per wavelength by
// SetInfo; per depth the kernel passes the members' populations, gij and
// quadrature weights, and per ray the absorption V of each member.
template <int MS>
struct SetInfo {
  int n;                                  // members
  int ti[MS], tj[MS], ent[MS], line[MS], prow[MS];
  double tw[MS], gline[MS], cV[MS], alpha[MS], wlam[MS];
  // per member: members with the same lower level / upper level / whose
  // upper level is this member's lower level (with 2hnu^3/c^2 != 0 for the
  // sums, rh/fillgamma.c:251-332), and the count of the last without that
  // condition (rh/fillgamma.c:204-214)
  uint32_t m_up[MS], m_jj[MS], m_ji[MS];
  int ncross[MS];
};

// per-depth member data: populations' difference x = n_i - gij n_j, emission
// e = tw gij n_j, gij and the quadrature weight
template <int MS>
struct SetDepth {
  double x[MS], e[MS], gij[MS], wla[MS];
};

// member data of the set at one depth (offset pk of a row, temperature T)
template <int MS>
__device__ __forceinline__ void set_depth(const NlteBufs &B, const SetInfo<MS> &si, int64_t pk,
                                          double T, double lam, SetDepth<MS> &sd) {
#pragma clang fp contract(fast)
  const double hc_k = HC / (KBOLTZMANN * NM_TO_M);
  const int64_t fs = B.fs;
  const double bf = exp(-hc_k / (lam * T));
#pragma unroll
  for (int n = 0; n < MS; n++) {
    sd.x[n] = sd.e[n] = sd.gij[n] = sd.wla[n] = 0.0;
    if (n < si.n) {
      const double ni = B.pops[(int64_t) si.ti[n] * fs + pk], nj = B.pops[(int64_t) si.tj[n] * fs + pk];
      if (si.line[n] >= 0) {
        sd.gij[n] = si.gline[n];
        sd.wla[n] = si.wlam[n] * B.wphi[(int64_t) si.line[n] * fs + pk] * (1.0 / HC_4PI);
      } else {
        sd.gij[n] = B.nstar[(int64_t) si.ti[n] * fs + pk] / B.nstar[(int64_t) si.tj[n] * fs + pk] * bf;
        sd.wla[n] = FOURPI / HPLANCK * (si.wlam[n] / lam);
      }
      sd.x[n] = ni - sd.gij[n] * nj;
      sd.e[n] = si.tw[n] * sd.gij[n] * nj;
    }
  }
}

// accumulate the rate terms of one ray (intensity I, operator Psi / chi in
// PsiC, direction weight wmu, absorption V of each member) into sIJ, sJI
template <int MS>
__device__ __forceinline__ void rate_terms(const SetInfo<MS> &si, const SetDepth<MS> &sd,
                                           const double (&V)[MS], double I, double PsiC,
                                           double wmu, double (&sIJ)[MS], double (&sJI)[MS]) {
#pragma clang fp contract(fast)
  double eta = 0.0;
#pragma unroll
  for (int n = 0; n < MS; n++)
    if (n < si.n) eta += V[n] * sd.e[n];
  const double Ieff = I - PsiC * eta, pw = PsiC * wmu;
  double chicc[MS], U[MS];
#pragma unroll
  for (int n = 0; n < MS; n++) {
    chicc[n] = V[n] * sd.wla[n] * sd.x[n];
    U[n] = si.tw[n] * sd.gij[n] * V[n];
  }
#pragma unroll
  for (int n = 0; n < MS; n++) {
    if (n < si.n) {
      double chi_up = 0.0, Uj = 0.0, chi_dn = 0.0, Ui = 0.0;
#pragma unroll
      for (int m = 0; m < MS; m++) {
        if ((si.m_up[n] >> m) & 1u) chi_up += chicc[m];
        if ((si.m_jj[n] >> m) & 1u) { Uj += U[m]; chi_dn += chicc[m]; }
        if ((si.m_ji[n] >> m) & 1u) Ui += U[m];
      }
      const double wlamu = V[n] * sd.wla[n] * wmu;
      sJI[n] += Ieff * wlamu;
      sIJ[n] += (si.tw[n] + Ieff) * sd.gij[n] * wlamu;
      sIJ[n] -= chi_up * Uj * pw;
      for (int c = 0; c < si.ncross[n]; c++) sJI[n] += chi_dn * Ui * pw;
    }
  }
}

// The active set of wavelength ls: members, their constants and coupling
// masks.
template <int MS>
__device__ __forceinline__ void set_info(const DevNlte &A, int ls, double lam, SetInfo<MS> &si) {
  const int p0 = A.as_ptr[ls];
  si.n = A.as_ptr[ls + 1] - p0;
  const double twohc = 2.0 * HC / (NM_TO_M * NM_TO_M * NM_TO_M);
#pragma unroll
  for (int n = 0; n < MS; n++) {
    si.ti[n] = si.tj[n] = si.ent[n] = si.line[n] = si.prow[n] = 0;
    si.tw[n] = si.gline[n] = si.cV[n] = si.alpha[n] = si.wlam[n] = 0.0;
    if (n < si.n) {
      const int t = A.as_tr[p0 + n], la = ls - A.tr_nblue[t];
      si.ti[n] = A.tr_i[t];
      si.tj[n] = A.tr_j[t];
      si.ent[n] = A.tr_ptr[t] + la;
      si.wlam[n] = A.tr_wlam[A.tr_ptr[t] + la];
      if (A.tr_type[t] == 0) {
        const int l = A.tr_line[t];
        si.line[n] = l;
        si.prow[n] = (A.ln_phi[l] + la) * A.nrays;
        si.gline[n] = A.ln_Bji[l] / A.ln_Bij[l];
        si.cV[n] = HC_4PI * A.ln_Bij[l] * 1.0;
        si.tw[n] = A.ln_Aji[l] / A.ln_Bji[l];
      } else {
        si.line[n] = -1;
        si.tw[n] = twohc / (lam * lam * lam);
        si.alpha[n] = A.tr_alpha[A.tr_ptr[t] + la];
      }
    }
  }
#pragma unroll
  for (int n = 0; n < MS; n++) {
    uint32_t up = 0, jj = 0, ji = 0;
    int nc = 0;
#pragma unroll
    for (int m = 0; m < MS; m++) {
      if (m < si.n) {
        if (si.tw[m] != 0.0) {
          if (si.ti[m] == si.ti[n]) up |= 1u << m;
          if (si.tj[m] == si.tj[n]) jj |= 1u << m;
          if (si.tj[m] == si.ti[n]) ji |= 1u << m;
        }
        if (si.tj[m] == si.ti[n]) nc++;
      }
    }
    si.m_up[n] = up;
    si.m_jj[n] = jj;
    si.m_ji[n] = ji;
    si.ncross[n] = nc;
  }
}

// ---------------------------------------------------------------------------
// Short-characteristic rays with the scalar cubic Bezier method and its
// diagonal operator (rh/rhf1d/bezier_1D.c:306-541).  L lanes per ray
// direction (32: half a wavefront each, 64: a wavefront each; the first L
// threads inward, the others outward), lane l holding the sweep's points
// t = l P .. l P + P - 1 (depth t inward, N-1-t outward), so both directions
// run the same code at the same time.  Everything but the intensity is local
// to a point and its neighbours; the recursion I[t] = E[t] I[t-1] + b[t] is a
// scan over the L lanes.

// What the points fix for every ray: path |z[t] - z[t-1]|, its reciprocal and
// the derivative's interval weight.
template <int P>
struct RayPath {
  double dz[P], idz[P], al[P];
};

// The neighbouring lanes of a ray direction.  With L = 128 a direction's lanes
// are two wavefronts (first half and second half), which meet in `edge`
// (RAY_EDGE doubles of LDS per direction, one slot per exchange of a sweep):
// a slot is written again only after the barriers of the exchanges that
// follow its reading.
constexpr int RAY_EDGE = 15;
template <int L>
struct RayLanes {
  double *edge;   // of this direction (L > 64)
  bool second;    // the lane is in the direction's second wavefront

  // up: replaced by the previous lane's values, dn: by the next lane's (the
  // first and the last lane of a direction get values that are never used)
  template <int SLOT, int NU, int ND>
  __device__ __forceinline__ void exchange(double (&up)[NU], double (&dn)[ND]) const {
    if constexpr (L > 64) {
      const int lane = threadIdx.x & 63;
      if (!second && lane == 63)
#pragma unroll
        for (int i = 0; i < NU; i++) edge[SLOT + i] = up[i];
      if (second && lane == 0)
#pragma unroll
        for (int i = 0; i < ND; i++) edge[SLOT + NU + i] = dn[i];
    }
#pragma unroll
    for (int i = 0; i < NU; i++) up[i] = from_prev(up[i]);
#pragma unroll
    for (int i = 0; i < ND; i++) dn[i] = from_next(dn[i]);
    if constexpr (L > 64) {
      __syncthreads();
      const int lane = threadIdx.x & 63;
      if (second && lane == 0)
#pragma unroll
        for (int i = 0; i < NU; i++) up[i] = edge[SLOT + i];
      if (!second && lane == 63)
#pragma unroll
        for (int i = 0; i < ND; i++) dn[i] = edge[SLOT + NU + i];
    }
  }
  template <int SLOT>
  __device__ __forceinline__ double prev(double x) const {
    double up[1] = {x}, dn[1] = {0.0};
    if constexpr (L > 64) exchange<SLOT>(up, dn);
    else up[0] = from_prev(x);
    return up[0];
  }
  template <int SLOT>
  __device__ __forceinline__ double next(double x) const {
    double up[1] = {0.0}, dn[1] = {x};
    if constexpr (L > 64) exchange<SLOT>(up, dn);
    else dn[0] = from_next(x);
    return dn[0];
  }
};

// one ray's intensity and operator at the points from the opacities C (with
// reciprocals iC), source functions S, 1 / mu and the boundary's Planck
// function (outward: B at the two deepest points)
template <int L, int P>
__device__ __forceinline__ void ray_sweep(const RayLanes<L> &lanes, const RayPath<P> &g, int t0,
                                          int N, bool outward, double zmu, double B2_0, double B2_1,
                                          const double (&C)[P], const double (&S)[P],
                                          double (&I)[P], double (&Psi)[P]) {
#pragma clang fp contract(fast)
  double f[P], dchi[P], dtau[P], idt[P], sl[P], dS[P], E[P], b[P];
  double CS_prev[2] = {C[P - 1], S[P - 1]}, C0_next[1] = {C[0]};
  lanes.template exchange<0>(CS_prev, C0_next);
  const double C_prev = CS_prev[0], S_prev = CS_prev[1], C_next = C0_next[0];
#pragma unroll
  for (int s = 0; s < P; s++) f[s] = (C[s] - (s ? C[s > 0 ? s - 1 : 0] : C_prev)) * g.idz[s];
  const double f_next = lanes.template next<3>(f[0]);
#pragma unroll
  for (int s = 0; s < P; s++) {
    const int t = t0 + s;
    const double fn = s < P - 1 ? f[s < P - 1 ? s + 1 : s] : f_next;
    dchi[s] = monotone(f[s], fn, g.al[s]);
    if (t == 0) dchi[s] = fn;
    if (t == N - 1) dchi[s] = f[s];
  }
  const double dchi_prev = lanes.template prev<5>(dchi[P - 1]);
#pragma unroll
  for (int s = 0; s < P; s++) {
    const double Cm = s ? C[s > 0 ? s - 1 : 0] : C_prev, dm = s ? dchi[s > 0 ? s - 1 : 0] : dchi_prev;
    const double z3 = g.dz[s] * (1.0 / 3.0);
    const double c1 = max0(C[s] - z3 * dchi[s]), c2 = max0(Cm + z3 * dm);
    dtau[s] = g.dz[s] * zmu * (C[s] + Cm + c1 + c2) * 0.25;
    idt[s] = nrcp(dtau[s]);
    sl[s] = (S[s] - (s ? S[s > 0 ? s - 1 : 0] : S_prev)) * idt[s];
  }
  double none[1] = {0.0}, ts_next[2] = {dtau[0], sl[0]};
  lanes.template exchange<7>(none, ts_next);
  const double dtau_next = ts_next[0], sl_next = ts_next[1];
#pragma unroll
  for (int s = 0; s < P; s++) {
    const double tn = s < P - 1 ? dtau[s < P - 1 ? s + 1 : s] : dtau_next;
    const double sn = s < P - 1 ? sl[s < P - 1 ? s + 1 : s] : sl_next;
    // monotone() with alpha = (2 tn + dtau) / (3 (tn + dtau)), one reciprocal
    const double ts = tn + dtau[s], p = sl[s] * sn;
    dS[s] = p > 0.0 ? 3.0 * p * ts * nrcp((ts + dtau[s]) * sl[s] + (ts + tn) * sn) : 0.0;
    if (t0 + s == 0) dS[s] = sn;
  }
  const double dS_prev = lanes.template prev<10>(dS[P - 1]);
#pragma unroll
  for (int s = 0; s < P; s++) {
    const int t = t0 + s;
    const double Cm = s ? C[s > 0 ? s - 1 : 0] : C_prev, Sm = s ? S[s > 0 ? s - 1 : 0] : S_prev;
    const double dSm = s ? dS[s > 0 ? s - 1 : 0] : dS_prev;
    // the last interval is linear, on its own (trapezoidal) path
    const bool last = t == N - 1;
    const double dt = last ? 0.5 * zmu * (C[s] + Cm) * g.dz[s] : dtau[s];
    const double eps = exp(-dt), dt2 = dt * dt, dt3 = dt2 * dt;
    double alpha, beta, gamma, theta, e;
    if (dt >= 5.e-2) {   // bezier3_coeffs, rh/bezier_aux.c:333-359
      const double i3 = idt[s] * idt[s] * idt[s];
      e = eps;
      alpha = (-6.0 + 6.0 * dt - 3.0 * dt2 + dt3 + 6.0 * eps) * i3;
      beta = (6.0 + (-6.0 - dt * (6.0 + dt * (3.0 + dt))) * eps) * i3;
      gamma = 3.0 * (6.0 + (-4.0 + dt) * dt - 2.0 * (3.0 + dt) * eps) * i3;
      theta = 3.0 * (eps * (6.0 + dt2 + 4.0 * dt) + 2.0 * dt - 6.0) * i3;
    } else {
      const double dt4 = dt2 * dt2;
      e = 1.0 - dt + 0.5 * dt2 - dt3 * (1.0 / 6.0) + dt4 * (1.0 / 24.0);
      alpha = 0.25 * dt - 0.05 * dt2 + dt3 * (1.0 / 120.0) - dt4 * (1.0 / 840.0);
      beta = 0.25 * dt - 0.20 * dt2 + dt3 * (1.0 / 12.0) - dt4 * (1.0 / 42.0);
      gamma = 0.25 * dt - 0.10 * dt2 + dt3 * 0.025 - dt4 * (1.0 / 210.0);
      theta = 0.25 * dt - 0.15 * dt2 + dt3 * 0.05 - dt4 * (1.0 / 84.0);
    }
    const double d3 = dt * (1.0 / 3.0);
    E[s] = e;
    b[s] = alpha * S[s] + beta * Sm + gamma * max0(S[s] - d3 * dS[s]) + theta * max0(Sm + d3 * dSm);
    Psi[s] = alpha + gamma;
    if (last) {
      // w3, rh/w3.c:44-63
      const bool thin = dt < 5.0E-4, thick = dt > 50.0;
      const double w0 = thin ? dt * (1.0 - 0.5 * dt) : thick ? 1.0 : 1.0 - eps;
      const double w1 = thin ? dt2 * (0.5 - dt / 3.0) : thick ? 1.0 : w0 - dt * eps;
      const double w1t = ndiv(w1, dt);
      E[s] = 1.0 - w0;
      b[s] = w0 * S[s] - w1t * (S[s] - Sm);
      Psi[s] = w0 - w1t;
    }
    if (t == 0) {
      const double C1 = P > 1 ? C[P > 1 ? 1 : 0] : C_next;
      const double d0 = 0.5 * zmu * (C[s] + C1) * g.dz[s];   // dz[0] holds the first interval
      E[s] = 0.0;
      b[s] = outward ? B2_1 - ndiv(B2_0 - B2_1, d0) : 0.0;
      Psi[s] = 0.0;
    }
  }
  // the lane's points composed, an inclusive scan over the lanes, then the
  // points from the previous lane's intensity (E = 0 at t = 0, so the
  // composed offset is the intensity itself)
  double LE = E[0], Lb = b[0];
#pragma unroll
  for (int s = 1; s < P; s++) {
    Lb = fma(E[s], Lb, b[s]);
    LE *= E[s];
  }
#define RAY_SCAN(CTRL, ROWS)                                                              \
  {                                                                                       \
    const double pe = dpp<CTRL, ROWS>(1.0, LE), pb = dpp<CTRL, ROWS>(0.0, Lb);            \
    Lb = fma(LE, pb, Lb);                                                                 \
    LE *= pe;                                                                             \
  }
  RAY_SCAN(0x111, 0xf)   // row_shr:1
  RAY_SCAN(0x112, 0xf)   // row_shr:2
  RAY_SCAN(0x114, 0xf)   // row_shr:4
  RAY_SCAN(0x118, 0xf)   // row_shr:8
  RAY_SCAN(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
  if constexpr (L >= 64) RAY_SCAN(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef RAY_SCAN
  double Iu = from_prev(Lb);
  if constexpr (L > 64) {
    // the first wavefront's last intensity enters the second (moves between
    // lanes stay outside of the branches: every lane has to take part)
    const double Eu = from_prev(LE);
    if (!lanes.second && (threadIdx.x & 63) == 63) lanes.edge[12] = Lb;
    __syncthreads();
    const double I1 = lanes.edge[12];
    if (lanes.second) Iu = (threadIdx.x & 63) == 0 ? I1 : fma(Eu, I1, Iu);
  }
#pragma unroll
  for (int s = 0; s < P; s++) {
    Iu = t0 + s == 0 ? b[s] : fma(E[s], Iu, b[s]);
    I[s] = Iu;
  }
}

// the lane's points: depths, paths and interval weights (points
// past the last stand at the last depth and are never read)
template <int L, int P>
__device__ __forceinline__ void ray_points(const RayLanes<L> &lanes, const NlteBufs &B, int64_t col,
                                           int t0, int N, bool outward, int (&k)[P],
                                           RayPath<P> &g) {
#pragma clang fp contract(fast)
#pragma unroll
  for (int s = 0; s < P; s++) {
    const int t = t0 + s < N ? t0 + s : N - 1, tu = t > 0 ? t : 1;
    k[s] = outward ? N - 1 - t : t;
    // the interval between t - 1 and t (at t = 0: between 0 and 1)
    g.dz[s] = B.geo[NG_DZ * B.fs + col + (outward ? N - tu : tu)];
    g.idz[s] = nrcp(g.dz[s]);
  }
  const double dz_next = lanes.template next<13>(g.dz[0]);
#pragma unroll
  for (int s = 0; s < P; s++) {
    const double dn = s < P - 1 ? g.dz[s < P - 1 ? s + 1 : s] : dz_next;
    g.al[s] = 0.333333333333333333333333 * (1.0 + dn * nrcp(dn + g.dz[s]));
  }
}

// Wavelengths with an active line, one (column, wavelength) per workgroup of
// 2 L threads:
// the rays in both directions, the new mean intensity and with eval_op the
// radiative rate terms (rh/rhf1d/formal.c:44-346, rh/fillgamma.c:82-332),
// summed over the rays in registers; the outward lanes' sums are turned to
// the inward lanes' depths through LDS at the end.  J is
// double-buffered per column (jpar): the previous J enters the source
// function, the new one is built.
// Measured on a pass over 465 such wavelengths: one column 26 us (5.3 ms with
// a lane per column: all its wavefronts on one XCD, one lane of each), 1500
// columns of 82 depths 8.0 ms (16.5), bound by the issue of 3.8e9 vector
// instructions and the waits of the two wavefronts per SIMD that the registers
// allow: 9.9 ms with the member data in registers and a ray's profiles loaded
// as it begins.  P = 3 at 32 lanes per direction covers 82 depths with 85% of
// the lanes.  Deeper columns take more lanes, not more points: above 256 depths
// two wavefronts per direction with three or four points (up to 10 registers
// spilled), where one with eight spilled 167 to 813 and fell behind a lane per
// column.  Solves of three Ca II iterations, a lane per column / one wavefront /
// these: 2000 columns of 256 depths 501 / 310 / 310 ms, 1500 of 384
// 620 / 673 / 283, 1200 of 512 804 / 587 / 428.
template <int L, int P, int MS>
__global__ void __launch_bounds__(2 * L, (P <= 3 && MS <= 2 ? 2 : 1))
k_nlte_bezier(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap, NlteBufs B,
              const int32_t *__restrict__ act, int nact, const int32_t *__restrict__ out_ls,
              const int32_t *__restrict__ io_list, int nlist, int il_off, int nlist_all,
              int eval_op) {
#pragma clang fp contract(fast)
  extern __shared__ double turn[];
  const DevModel &M = *Mp;
  const DevNlte &A = *Ap;
  int slot, il;
  xcd_tile(blockIdx.x, nact, nlist, slot, il);
  if (slot >= nact) return;
  const int ic = act[slot], io = io_list[il], ls = out_ls[io];
  const int N = B.ndep[ic], nrays = A.nrays;
  const int64_t fs = B.fs, col = (int64_t) ic * B.Kp;
  const int64_t wo = (int64_t) io * fs + col, jb = (int64_t) B.nout * fs;
  const int par = B.jpar[ic];
  const double *Jold = B.J + par * jb + wo;
  double *Jnew = B.J + (1 - par) * jb + wo;
  const double lam = ldc(M.lamconst)[(int64_t) ls * RHG_LC_NCONST + RHG_LC_LAMBDA];
  SetInfo<MS> si;
  set_info<MS>(A, ls, lam, si);
  const bool outward = threadIdx.x >= L;
  const int t0 = (int) (threadIdx.x & (L - 1)) * P;
  const double *Tc = B.geo + NG_T * fs + col;
  const double B2_0 = planck_lam(Tc[N - 2], lam), B2_1 = planck_lam(Tc[N - 1], lam);
  int k[P];
  RayPath<P> g;
  __shared__ double edge[L > 64 ? 2 * RAY_EDGE : 1];
  const RayLanes<L> lanes{L > 64 && outward ? edge + RAY_EDGE : edge, L > 64 && (threadIdx.x & 64)};
  ray_points<L, P>(lanes, B, col, t0, N, outward, k, g);
  // member data of the lane's points: in LDS, column threadIdx.x of each row,
  // where it fits (the registers then hold the next ray's profiles)
  constexpr bool STASH = nlte_stash(L, P, MS);
  double *stash = turn + L * P + threadIdx.x;
  SetDepth<MS> sd_r[STASH ? 1 : P];
  auto put_depth = [&](int s, const SetDepth<MS> &d) {
    if constexpr (STASH) {
#pragma unroll
      for (int n = 0; n < MS; n++) {
        double *q = stash + (s * MS + n) * 4 * 2 * L;
        q[0] = d.x[n];
        q[2 * L] = d.e[n];
        q[4 * L] = d.gij[n];
        q[6 * L] = d.wla[n];
      }
    } else {
      sd_r[s] = d;
    }
  };
  auto get_depth = [&](int s) -> SetDepth<MS> {
    if constexpr (STASH) {
      SetDepth<MS> d;
#pragma unroll
      for (int n = 0; n < MS; n++) {
        const double *q = stash + (s * MS + n) * 4 * 2 * L;
        d.x[n] = q[0];
        d.e[n] = q[2 * L];
        d.gij[n] = q[4 * L];
        d.wla[n] = q[6 * L];
      }
      return d;
    } else {
      return sd_r[s];
    }
  };
  double cc[P], s0[P], js[P], sIJ[P][MS], sJI[P][MS];
#pragma unroll
  for (int s = 0; s < P; s++) {
    SetDepth<MS> d;
    set_depth<MS>(B, si, col + k[s], Tc[k[s]], lam, d);
    put_depth(s, d);
    cc[s] = B.cchi[wo + k[s]];
    s0[s] = fma(B.csca[wo + k[s]], Jold[k[s]], B.ceta[wo + k[s]]);
    js[s] = 0.0;
#pragma unroll
    for (int n = 0; n < MS; n++) sIJ[s][n] = sJI[s][n] = 0.0;
  }
  const int dir = outward ? 1 : 0;
  // a ray's profiles are loaded one ray ahead
  double ph[P][MS];
  auto fetch = [&](int mu) {
#pragma unroll
    for (int s = 0; s < P; s++)
#pragma unroll
      for (int n = 0; n < MS; n++)
        ph[s][n] = n < si.n && si.line[n] >= 0
                       ? B.phi[((int64_t) (si.prow[n] + mu) * 2 + dir) * fs + col + k[s]] : 0.0;
  };
  fetch(0);
  for (int mu = 0; mu < nrays; mu++) {
    const double zmu = 1.0 / A.muz[mu], wmu = 0.5 * A.wmu[mu];
    double V[P][MS], C[P], S[P], iC[P], I[P], Psi[P];
#pragma unroll
    for (int s = 0; s < P; s++) {
      const SetDepth<MS> d = get_depth(s);
      double chi = 0.0, eta = 0.0;
#pragma unroll
      for (int n = 0; n < MS; n++) {
        V[s][n] = 0.0;
        if (n < si.n) {
          V[s][n] = si.line[n] >= 0 ? si.cV[n] * ph[s][n] : si.alpha[n];
          chi += V[s][n] * d.x[n];
          eta += V[s][n] * d.e[n];
        }
      }
      C[s] = chi + cc[s];
      iC[s] = nrcp(C[s]);
      S[s] = (eta + s0[s]) * iC[s];
    }
    if (mu + 1 < nrays) fetch(mu + 1);
    ray_sweep<L, P>(lanes, g, t0, N, outward, zmu, B2_0, B2_1, C, S, I, Psi);
#pragma unroll
    for (int s = 0; s < P; s++) {
      js[s] += wmu * I[s];
      if (eval_op)
        rate_terms<MS>(si, get_depth(s), V[s], I[s], Psi[s] * iC[s], wmu, sIJ[s], sJI[s]);
    }
  }
  // the inward lanes add the outward lanes' sum at each of their depths
  auto both = [&](int s, double x) -> double { return x + turn[k[s]]; };
  auto put = [&](auto &&value) {
    __syncthreads();
#pragma unroll
    for (int s = 0; s < P; s++)
      if (outward && t0 + s < N) turn[k[s]] = value(s);
    __syncthreads();
  };
  put([&](int s) { return js[s]; });
  double dJmax = 0.0;
#pragma unroll
  for (int s = 0; s < P; s++) {
    if (!outward && t0 + s < N) {
      const double jn = both(s, js[s]), dJ = fabs(1.0 - Jold[k[s]] / jn);
      Jnew[k[s]] = jn;
      dJmax = dJmax > dJ ? dJmax : dJ;
    }
  }
  for (int o = L < 64 ? L / 2 : 32; o >= 1; o >>= 1) {
    const double x = __shfl_xor(dJmax, o);
    dJmax = dJmax > x ? dJmax : x;
  }
  if constexpr (L > 64) {
    if (threadIdx.x == 64) edge[0] = dJmax;
    __syncthreads();
    if (threadIdx.x == 0) dJmax = dJmax > edge[0] ? dJmax : edge[0];
  }
  if (threadIdx.x == 0) B.dJ[(int64_t) ic * nlist_all + il_off + il] = dJmax;
  if (!eval_op) return;
#pragma unroll
  for (int n = 0; n < MS; n++) {
    if (n < si.n) {
      double *aij = B.acc + ((int64_t) si.ent[n] * 2) * fs + col;
      put([&](int s) { return sIJ[s][n]; });
#pragma unroll
      for (int s = 0; s < P; s++)
        if (!outward && t0 + s < N) aij[k[s]] = both(s, sIJ[s][n]);
      put([&](int s) { return sJI[s][n]; });
#pragma unroll
      for (int s = 0; s < P; s++)
        if (!outward && t0 + s < N) aij[fs + k[s]] = both(s, sJI[s][n]);
    }
  }
}

#define RHG_INST_BEZ(L, P, MS)                                                                  \
  template __global__ void k_nlte_bezier<L, P, MS>(const DevModel *, const DevNlte *, NlteBufs,  \
                                                   const int32_t *, int, const int32_t *,        \
                                                   const int32_t *, int, int, int, int);
#define RHG_INST_BEZ_MS(L, P) RHG_INST_BEZ(L, P, 2) RHG_INST_BEZ(L, P, 4)
RHG_INST_BEZ_MS(32, 1)
RHG_INST_BEZ_MS(32, 2)
RHG_INST_BEZ_MS(32, 3)
RHG_INST_BEZ_MS(64, 2)
RHG_INST_BEZ_MS(64, 3)
RHG_INST_BEZ_MS(64, 4)
RHG_INST_BEZ_MS(128, 3)
RHG_INST_BEZ_MS(128, 4)
RHG_INST_BEZ(32, 1, 8)
RHG_INST_BEZ(32, 2, 8)
RHG_INST_BEZ(64, 2, 8)
RHG_INST_BEZ(128, 2, 8)
RHG_INST_BEZ(128, 3, 8)
RHG_INST_BEZ(128, 4, 8)
#undef RHG_INST_BEZ_MS
#undef RHG_INST_BEZ

// The member data of one depth at mu of the final ray: opacity and emission
// of the active set (Armstrong profiles as the set-up's).
__device__ __forceinline__ void emergent_set(const NlteBufs &B, const DevNlte &A,
                                             const SetInfo<NLTE_MAXSET> &si, int64_t pk, double lam,
                                             double mu, double &chi, double &eta) {
  const int64_t fs = B.fs;
  const double T = B.geo[NG_T * fs + pk], vb = B.vbroad[pk], vz = B.geo[NG_VLOS * fs + pk];
  SetDepth<NLTE_MAXSET> sd;
  set_depth<NLTE_MAXSET>(B, si, pk, T, lam, sd);
  chi = eta = 0.0;
#pragma unroll
  for (int n = 0; n < NLTE_MAXSET; n++) {
    if (n < si.n) {
      double V = si.alpha[n];
      if (si.line[n] >= 0) {
        const int l = si.line[n];
        const double lambda0 = A.ln_lambda0[l];
        const double v = (lam - lambda0 - 0.0) * CLIGHT / (vb * lambda0);
        const double vlos = mu * vz / vb;
        V = si.cV[n] * (voigt_armstrong(B.adamp[(int64_t) l * fs + pk], v + 1.0 * vlos) * 1.0 /
                        (SQRTPI * vb));
      }
      chi += V * sd.x[n];
      eta += V * sd.e[n];
    }
  }
}

// The emergent spectrum after convergence, pyrh's final ray
// (rh/rhf1d/pyrh_solveray.c:82-107), at the wavelengths with a line: one ray
// at the caller's mu with the converged populations, background scattering
// from the last J, no update of J.  One (column, wavelength) per wavefront,
// as k_nlte_bezier (every lane group carries the one outward ray).  I goes to
// stokes[(column * 4) * nout + io]; Q, U, V are zero (field-free).
template <int L, int P>
__global__ void __launch_bounds__(64)
k_nlte_emergent(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap, NlteBufs B,
                const int32_t *__restrict__ act, int nact, const int32_t *__restrict__ out_ls,
                const int32_t *__restrict__ io_list, int nlist, double mu,
                double *__restrict__ stokes) {
  const DevModel &M = *Mp;
  const DevNlte &A = *Ap;
  int slot, il;
  xcd_tile(blockIdx.x, nact, nlist, slot, il);
  if (slot >= nact) return;
  const int ic = act[slot];
  const int io = io_list[il], ls = out_ls[io], N = B.ndep[ic];
  const int64_t fs = B.fs, col = (int64_t) ic * B.Kp, wo = (int64_t) io * fs + col;
  const double *Jl = B.J + B.jpar[ic] * (int64_t) B.nout * fs + wo;
  const double lam = ldc(M.lamconst)[(int64_t) ls * RHG_LC_NCONST + RHG_LC_LAMBDA];
  SetInfo<NLTE_MAXSET> si;
  set_info<NLTE_MAXSET>(A, ls, lam, si);
  const int t0 = (int) (threadIdx.x & (L - 1)) * P;
  const double *Tc = B.geo + NG_T * fs + col;
  const double B2_0 = planck_lam(Tc[N - 2], lam), B2_1 = planck_lam(Tc[N - 1], lam);
  int k[P];
  RayPath<P> g;
  const RayLanes<L> lanes{nullptr, false};
  ray_points<L, P>(lanes, B, col, t0, N, true, k, g);
  double C[P], S[P], I[P], Psi[P];
#pragma unroll
  for (int s = 0; s < P; s++) {
    double chi, eta;
    emergent_set(B, A, si, col + k[s], lam, mu, chi, eta);
    C[s] = chi + B.cchi[wo + k[s]];
    S[s] = fma(B.csca[wo + k[s]], Jl[k[s]], eta + B.ceta[wo + k[s]]) / C[s];
  }
  ray_sweep<L, P>(lanes, g, t0, N, true, 1.0 / mu, B2_0, B2_1, C, S, I, Psi);
#pragma unroll
  for (int s = 0; s < P; s++) {
    if (threadIdx.x < L && t0 + s == N - 1) {
      double *o = stokes + (int64_t) ic * 4 * B.nout + io;
      o[0] = I[s];
      o[B.nout] = 0.0;
      o[2 * (int64_t) B.nout] = 0.0;
      o[3 * (int64_t) B.nout] = 0.0;
    }
  }
}
#define RHG_INST_EM(L, P)                                                                       \
  template __global__ void k_nlte_emergent<L, P>(const DevModel *, const DevNlte *, NlteBufs,   \
                                                 const int32_t *, int, const int32_t *,         \
                                                 const int32_t *, int, double, double *);
RHG_INST_EM(32, 1)
RHG_INST_EM(32, 2)
RHG_INST_EM(32, 3)
RHG_INST_EM(64, 2)
RHG_INST_EM(64, 3)
RHG_INST_EM(64, 4)
RHG_INST_EM(64, 6)
RHG_INST_EM(64, 8)
#undef RHG_INST_EM

// ---------------------------------------------------------------------------
// Wavelengths with continua only: one opacity for all rays, and per ray the
// Feautrier solution with its two-sided diagonal operator
// (rh/rhf1d/feautrier.c:56-202, dark top, thermalised bottom, STANDARD order;
// P is the mean of the two directions, weighted by the full ray weight).
// One wavefront per wavelength and group of up to `per` active columns:
//   1  depths on the lanes: opacity, source function and the rays' common
//      path factor (chi_k + chi_{k+1}) (z_k - z_{k+1}) into LDS;
//   2  (column, ray) on the lanes: elimination and back substitution, the
//      only serial part, with F and z in LDS, overwritten by Psi and P;
//   3  depths on the lanes: J and the rate terms summed over the rays.
// More rays than NLTE_FE_RAYS run phases 2 and 3 in chunks.  MS is the
// largest active set among the wavelengths of io_list (the member loops are
// unrolled to it).  EM: the final ray at mu instead (k_nlte_emergent's
// counterpart): one ray, its emergent intensity to stokes.
// The elimination is written in F and q = F / (1 + F): with r = dtau_k /
// dtau_{k-1} and d the mean of the two, F_k = d dtau_k + r q_{k-1} and
// z_k = (d dtau_k S_k + r z_{k-1}) / (1 + F_k), one reciprocal in the chain.
template <int MS, bool EM>
__global__ void __launch_bounds__(64)
k_nlte_feautrier(const DevModel *__restrict__ Mp, const DevNlte *__restrict__ Ap, NlteBufs B,
                 const int32_t *__restrict__ act, int nact, int per, int Nd,
                 const int32_t *__restrict__ out_ls, const int32_t *__restrict__ io_list, int nlist,
                 int il_off, int nlist_all, int eval_op, double mu_em, double *__restrict__ stokes) {
#pragma clang fp contract(fast)
  extern __shared__ double lds[];
  const DevModel &M = *Mp;
  const DevNlte &A = *Ap;
  int grp, il;
  xcd_tile(blockIdx.x, (nact + per - 1) / per, nlist, grp, il);
  if (grp >= (nact + per - 1) / per) return;
  const int io = io_list[il], ls = out_ls[io], nrays = EM ? 1 : A.nrays;
  const int first = grp * per, n_it = nact - first < per ? nact - first : per;
  const int64_t fs = B.fs, jb = (int64_t) B.nout * fs;
  const double lam = ldc(M.lamconst)[(int64_t) ls * RHG_LC_NCONST + RHG_LC_LAMBDA];
  SetInfo<MS> si;
  set_info<MS>(A, ls, lam, si);
  const int lane = threadIdx.x;
  constexpr int RF = EM ? 1 : NLTE_FE_RAYS;
  const int FS = per * RF;   // F and z: [Nd][per * RF]
  double *Xs = lds, *Ss = Xs + per * Nd, *Cs = Ss + per * Nd, *Fs = Cs + per * Nd,
         *Zs = Fs + Nd * FS;
  auto column = [&](int it) { return act[first + it]; };

  for (int it = 0; it < n_it; it++) {
    const int ic = column(it), N = B.ndep[ic];
    const int64_t col = (int64_t) ic * B.Kp, wo = (int64_t) io * fs + col;
    const double *Jo = B.J + B.jpar[ic] * jb + wo, *Tc = B.geo + NG_T * fs + col;
    for (int k = lane; k < N; k += 64) {
      double chi = 0.0, eta = 0.0;
      if constexpr (EM) {
        SetInfo<NLTE_MAXSET> s8;
        set_info<NLTE_MAXSET>(A, ls, lam, s8);
        emergent_set(B, A, s8, col + k, lam, mu_em, chi, eta);
      } else {
        SetDepth<MS> sd;
        set_depth<MS>(B, si, col + k, Tc[k], lam, sd);
#pragma unroll
        for (int n = 0; n < MS; n++) {
          if (n < si.n) {
            // a line at a Feautrier wavelength (not produced by the set-up):
            // its profile of the first ray
            const double V = si.line[n] >= 0
                                 ? si.cV[n] * B.phi[((int64_t) si.prow[n] * 2) * fs + col + k]
                                 : si.alpha[n];
            chi += V * sd.x[n];
            eta += V * sd.e[n];
          }
        }
      }
      const double C = chi + B.cchi[wo + k];
      Cs[it * Nd + k] = C;
      Ss[it * Nd + k] = fma(B.csca[wo + k], Jo[k], eta + B.ceta[wo + k]) / C;
    }
    wave_sync();
    const double *z = B.geo + NG_HEIGHT * fs + col;
    for (int k = lane; k < N - 1; k += 64)
      Xs[it * Nd + k] = (Cs[it * Nd + k] + Cs[it * Nd + k + 1]) * (z[k] - z[k + 1]);
  }
  wave_sync();

  for (int c0 = 0; c0 < nrays; c0 += RF) {
    const int nrc = nrays - c0 < RF ? nrays - c0 : RF;
    const int it_s = lane / RF, r_s = lane % RF;
    if (it_s < n_it && r_s < nrc) {
      const int ic = column(it_s), N = B.ndep[ic];
      const double *Tc = B.geo + NG_T * fs + (int64_t) ic * B.Kp;
      const double B2_0 = planck_lam(Tc[N - 2], lam), B2_1 = planck_lam(Tc[N - 1], lam);
      const double zmu = 0.5 / (EM ? mu_em : A.muz[c0 + r_s]);
      const double *X = Xs + it_s * Nd, *Sv = Ss + it_s * Nd;
      double *F = Fs + lane, *Z = Zs + lane;
      const double dt0 = zmu * X[0], abc0 = 1.0 + 2.0 / dt0, C1_0 = 2.0 / (dt0 * dt0);
      double Fk = abc0 / C1_0, zk = Sv[0] / (abc0 + C1_0), q = ndiv(Fk, 1.0 + Fk);
      F[0] = Fk;
      Z[0] = zk;
      double dtm = dt0, idtm = nrcp(dt0);
#pragma unroll 2
      for (int k = 1; k < N - 1; k++) {
        const double dt = zmu * X[k], d = 0.5 * (dt + dtm) * dt, r = dt * idtm;
        Fk = fma(r, q, d);
        const double i1 = nrcp(1.0 + Fk);
        zk = fma(d, Sv[k], r * zk) * i1;
        q = Fk * i1;
        F[k * FS] = Fk;
        Z[k * FS] = zk;
        dtm = dt;
        idtm = nrcp(dt);
      }
      // back substitution with the two-sided operator
      const double hN = B2_1 - (B2_0 - B2_1) / dtm;
      const double abcN = 1.0 + 2.0 / dtm, A1N = 2.0 / (dtm * dtm);
      const double SN = Sv[N - 1] + 2.0 * hN / dtm;
      double P = (SN + A1N * zk) / (abcN + A1N * q);
      double h = abcN / (A1N + abcN);   // G / (1 + G), G = abcN / A1N
      Z[(N - 1) * FS] = P;
      F[(N - 1) * FS] = 1.0 / (abcN + A1N * q);
      double dtk = dtm, idtk = idtm, Fc = Fk;
#pragma unroll 2
      for (int k = N - 2; k >= 1; k--) {
        const double Fm = F[(k - 1) * FS], dm = zmu * X[k - 1], idm = nrcp(dm);
        P = fma(P, nrcp(1.0 + Fc), Z[k * FS]);
        const double id = nrcp(0.5 * (dtk + dm));
        const double qm = ndiv(Fm, 1.0 + Fm);
        const double Psi = nrcp(1.0 + id * (idm * qm + idtk * h));
        const double G = fma(dm * idtk, h, 0.5 * (dtk + dm) * dm);
        h = ndiv(G, 1.0 + G);
        Z[k * FS] = P;
        F[k * FS] = Psi;
        dtk = dm;
        idtk = idm;
        Fc = Fm;
      }
      P = fma(P, nrcp(1.0 + Fc), Z[0]);
      if constexpr (EM) {
        // (1 + f0) P[0] - h0 / (1 + r0) with r0 = h0 = 0
        double *o = stokes + (int64_t) ic * 4 * B.nout + io;
        o[0] = (1.0 + 1.0) * P;
        o[B.nout] = 0.0;
        o[2 * (int64_t) B.nout] = 0.0;
        o[3 * (int64_t) B.nout] = 0.0;
      } else {
        Z[0] = P;
        F[0] = 1.0 / (abc0 + C1_0 * h);
      }
    }
    if constexpr (EM) return;
    wave_sync();
    for (int it = 0; it < n_it; it++) {
      const int ic = column(it), N = B.ndep[ic];
      const int64_t col = (int64_t) ic * B.Kp, wo = (int64_t) io * fs + col;
      const int par = B.jpar[ic];
      const double *Jo = B.J + par * jb + wo, *Tc = B.geo + NG_T * fs + col;
      double *Jn = B.J + (1 - par) * jb + wo;
      double dJ_it = 0.0;
      for (int k = lane; k < N; k += 64) {
        const double *F = Fs + k * FS + it * RF, *Z = Zs + k * FS + it * RF;
        double j = c0 ? Jn[k] : 0.0;
        for (int r = 0; r < nrc; r++) j += Z[r] * A.wmu[c0 + r];
        Jn[k] = j;
        if (c0 + RF >= nrays) {
          const double dJ = fabs(1.0 - Jo[k] / j);
          dJ_it = dJ_it > dJ ? dJ_it : dJ;
        }
        if (!eval_op) continue;
        SetDepth<MS> sd;
        set_depth<MS>(B, si, col + k, Tc[k], lam, sd);
        double V[MS], aIJ[MS], aJI[MS];
#pragma unroll
        for (int n = 0; n < MS; n++) {
          V[n] = aIJ[n] = aJI[n] = 0.0;
          if (n < si.n) {
            V[n] = si.line[n] >= 0 ? si.cV[n] * B.phi[((int64_t) si.prow[n] * 2) * fs + col + k]
                                   : si.alpha[n];
            if (c0 > 0) {
              const double *aij = B.acc + ((int64_t) si.ent[n] * 2) * fs + col + k;
              aIJ[n] = aij[0];
              aJI[n] = aij[fs];
            }
          }
        }
        const double iC = 1.0 / Cs[it * Nd + k];
        for (int r = 0; r < nrc; r++)
          rate_terms<MS>(si, sd, V, Z[r], F[r] * iC, A.wmu[c0 + r], aIJ, aJI);
#pragma unroll
        for (int n = 0; n < MS; n++) {
          if (n < si.n) {
            double *aij = B.acc + ((int64_t) si.ent[n] * 2) * fs + col + k;
            aij[0] = aIJ[n];
            aij[fs] = aJI[n];
          }
        }
      }
      if (c0 + RF >= nrays) {
        for (int o = 32; o >= 1; o >>= 1) {
          const double x = __shfl_xor(dJ_it, o);
          dJ_it = dJ_it > x ? dJ_it : x;
        }
        if (lane == 0) B.dJ[(int64_t) ic * nlist_all + il_off + il] = dJ_it;
      }
    }
    wave_sync();
  }
}
#define RHG_INST_FE(MS, EM)                                                                      \
  template __global__ void k_nlte_feautrier<MS, EM>(const DevModel *, const DevNlte *, NlteBufs, \
                                                    const int32_t *, int, int, int,              \
                                                    const int32_t *, const int32_t *, int, int,  \
                                                    int, int, double,                            \
                                                    double *);
RHG_INST_FE(2, false)
RHG_INST_FE(4, false)
RHG_INST_FE(6, false)
RHG_INST_FE(8, false)
RHG_INST_FE(2, true)
#undef RHG_INST_FE

// the new J becomes the previous one for the columns just solved
__global__ void k_nlte_flip(NlteBufs B, const int32_t *__restrict__ act, int nact) {
  const int slot = blockIdx.x * blockDim.x + threadIdx.x;
  if (slot >= nact) return;
  const int ic = act[slot];
  B.jpar[ic] = 1 - B.jpar[ic];
}

// max over the list wavelengths of the per-wavelength dJ, a wavefront per
// column
__global__ void __launch_bounds__(64)
k_nlte_djmax(NlteBufs B, const int32_t *__restrict__ act, int nact, int nlist,
             double *__restrict__ djmax) {
  const int ic = act[blockIdx.x];
  double d = 0.0;
  for (int il = threadIdx.x; il < nlist; il += 64) {
    const double x = B.dJ[(int64_t) ic * nlist + il];
    d = d > x ? d : x;
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const double x = __shfl_xor(d, o);
    d = d > x ? d : x;
  }
  if (threadIdx.x == 0) djmax[ic] = d;
}

// ---------------------------------------------------------------------------
// Crout LU decomposition with implicit pivoting, back substitution and one
// step of iterative improvement, rh/ludcmp.c:36-177, on an NLP x NLP system
// held in registers (compile-time indices; the dynamic pivot row is
// selected by comparison).  A system of n < NLP equations is padded with
// identity rows and zero right-hand sides, which leaves every operation on
// the first n rows and columns unchanged.
template <int NLP>
__device__ __forceinline__ void lu_decomp_r(double (&a)[NLP][NLP], int (&index)[NLP]) {
  double vv[NLP];
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    double big = 0.0;
#pragma unroll
    for (int j = 0; j < NLP; j++) {
      const double temp = fabs(a[i][j]);
      if (temp > big) big = temp;
    }
    vv[i] = 1.0 / big;
  }
#pragma unroll
  for (int j = 0; j < NLP; j++) {
#pragma unroll
    for (int i = 0; i < j; i++) {
      double sum = a[i][j];
#pragma unroll
      for (int k = 0; k < i; k++) sum -= a[i][k] * a[k][j];
      a[i][j] = sum;
    }
    double big = 0.0;
    int imax = 0;
#pragma unroll
    for (int i = j; i < NLP; i++) {
      double sum = a[i][j];
#pragma unroll
      for (int k = 0; k < j; k++) sum -= a[i][k] * a[k][j];
      a[i][j] = sum;
      const double dum = vv[i] * fabs(sum);
      if (dum >= big) {
        big = dum;
        imax = i;
      }
    }
#pragma unroll
    for (int i = j + 1; i < NLP; i++) {
      if (i == imax) {
#pragma unroll
        for (int k = 0; k < NLP; k++) {
          const double d = a[i][k];
          a[i][k] = a[j][k];
          a[j][k] = d;
        }
        vv[i] = vv[j];
      }
    }
    index[j] = imax;
    if (a[j][j] == 0.0) a[j][j] = 1.0e-20;
    const double dum = 1.0 / a[j][j];
#pragma unroll
    for (int i = j + 1; i < NLP; i++) a[i][j] *= dum;
  }
}

template <int NLP>
__device__ __forceinline__ void lu_backsubst_r(const double (&a)[NLP][NLP],
                                               const int (&index)[NLP], double (&b)[NLP]) {
  int ii = -1;
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    const int ip = index[i];
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < NLP; q++)
      if (q == ip) sum = b[q];
#pragma unroll
    for (int q = 0; q < NLP; q++)
      if (q == ip) b[q] = b[i];
    if (ii >= 0) {
#pragma unroll
      for (int j = 0; j < i; j++)
        if (j >= ii) sum -= a[i][j] * b[j];
    } else if (sum) {
      ii = i;
    }
    b[i] = sum;
  }
#pragma unroll
  for (int i = NLP - 1; i >= 0; i--) {
    double sum = b[i];
#pragma unroll
    for (int j = i + 1; j < NLP; j++) sum -= a[i][j] * b[j];
    b[i] = sum / a[i][i];
  }
}

template <int NLP>
__device__ __forceinline__ void solve_improve_r(double (&a)[NLP][NLP], double (&b)[NLP]) {
  double ac[NLP][NLP], bc[NLP], res[NLP];
  int index[NLP];
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    bc[i] = b[i];
#pragma unroll
    for (int j = 0; j < NLP; j++) ac[i][j] = a[i][j];
  }
  lu_decomp_r<NLP>(a, index);
  lu_backsubst_r<NLP>(a, index, b);
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    res[i] = bc[i];
#pragma unroll
    for (int j = 0; j < NLP; j++) res[i] -= ac[i][j] * b[j];
  }
  lu_backsubst_r<NLP>(a, index, res);
#pragma unroll
  for (int i = 0; i < NLP; i++) b[i] += res[i];
}

// Rate matrix and statistical equilibrium at D depths of one column,
// rh/statequil.c:36-216: Gamma = C + the rate terms of each transition
// summed over its wavelengths; the diagonal is minus the column sums; the
// equation of the most populated level (isum = -1, else level isum) is
// replaced by particle conservation.  The workgroup's wavefronts share
// the sums (a transition's two directions are a task, the depths on the
// lanes), the first one solves.  A task alone adds to its matrix element, as
// long as no two transitions join the same levels; where some do (share = 0),
// the first wavefront takes all tasks, in the transitions' order.  Launch
// (columns, ceil(Nmax / D)) workgroups with D nl^2 doubles of LDS, D =
// stateq_depths.
template <int NLP>
__global__ void __launch_bounds__(64 * stateq_waves(NLP))
k_nlte_stateq(const DevNlte *__restrict__ Ap, NlteBufs B, const int32_t *__restrict__ act,
              int nact, int isum, int share) {
  constexpr int D = stateq_depths(NLP), NT = 64 * stateq_waves(NLP) / D;
  const DevNlte &A = *Ap;
  extern __shared__ double gam[];   // [nl * nl][D]
  const int nl = A.nl, lane = threadIdx.x % D, w = threadIdx.x / D;
  const int ic = act[blockIdx.x], k = blockIdx.y * D + lane, N = B.ndep[ic];
  if ((int) blockIdx.y * D >= N) return;
  const int64_t fs = B.fs, pk = (int64_t) ic * B.Kp + (k < N ? k : N - 1);
  for (int q = w; q < nl * nl; q += NT) gam[q * D + lane] = B.Cmat[(int64_t) q * fs + pk];
  __syncthreads();
  const int nt = share ? 2 * A.ntrans : (w ? 0 : 2 * A.ntrans);
  for (int t = w; t < nt; t += share ? NT : 1) {
    const int tr = t >> 1, i = A.tr_i[tr], j = A.tr_j[tr], ne = A.tr_nlam[tr];
    const double *x = B.acc + ((int64_t) A.tr_ptr[tr] * 2 + (t & 1)) * fs + pk;
    double sum = 0.0;
#pragma unroll 16
    for (int e = 0; e < ne; e++) sum += x[(int64_t) (2 * e) * fs];
    gam[((t & 1) ? j * nl + i : i * nl + j) * D + lane] += sum;
  }
  __syncthreads();
  if (w != 0 || k >= N) return;
  double a[NLP][NLP], nk[NLP];
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    nk[i] = (i < nl) ? B.pops[(int64_t) i * fs + pk] : 0.0;
#pragma unroll
    for (int j = 0; j < NLP; j++)
      a[i][j] = (i < nl && j < nl) ? gam[(i * nl + j) * D + lane] : (i == j ? 1.0 : 0.0);
  }
  int ie = 0;
  if (isum == -1) {
    double nmax = 0.0;
#pragma unroll
    for (int i = 0; i < NLP; i++)
      if (i < nl && nk[i] > nmax) {
        nmax = nk[i];
        ie = i;
      }
  } else {
    ie = isum;
  }
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    if (i < nl) {
      a[i][i] = 0.0;
      nk[i] = 0.0;
      double GamDiag = 0.0;
#pragma unroll
      for (int j = 0; j < NLP; j++)
        if (j < nl) GamDiag += a[j][i];
      a[i][i] = -GamDiag;
    }
  }
  const double ntotal = B.ntot[pk];
#pragma unroll
  for (int i = 0; i < NLP; i++) {
    if (i == ie) {
      nk[i] = ntotal;
#pragma unroll
      for (int j = 0; j < NLP; j++)
        if (j < nl) a[i][j] = 1.0;
    }
  }
  solve_improve_r<NLP>(a, nk);
#pragma unroll
  for (int i = 0; i < NLP; i++)
    if (i < nl) B.pops[(int64_t) i * fs + pk] = nk[i];
}

template __global__ void k_nlte_stateq<4>(const DevNlte *, NlteBufs, const int32_t *, int, int, int);
template __global__ void k_nlte_stateq<6>(const DevNlte *, NlteBufs, const int32_t *, int, int, int);
template __global__ void k_nlte_stateq<8>(const DevNlte *, NlteBufs, const int32_t *, int, int, int);
template __global__ void k_nlte_stateq<16>(const DevNlte *, NlteBufs, const int32_t *, int, int, int);

// ---------------------------------------------------------------------------
// Ng acceleration of one column's populations and the maximum relative
// change, rh/accelerate.c:34-146 and rh/maxchange.c:32-50, over the
// populations flattened level by level (index i * N + k).  The history
// holds norder + 2 solutions; ng_init stored the starting solution in slot
// 0, so before iteration niter (1-based) the count is niter.
// A workgroup per column, the flattened populations over its threads.
__global__ void __launch_bounds__(NG_BLOCK)
k_nlte_ng(const DevNlte *__restrict__ Ap, NlteBufs B, const int32_t *__restrict__ act, int nact,
          int niter, int norder, int ndelay, int nperiod, double *__restrict__ dpops) {
  const DevNlte &A = *Ap;
  constexpr int NSUM = NLTE_MAXNG * (NLTE_MAXNG + 1), NW = NG_BLOCK / 64;
  __shared__ double part[NW][NSUM], coef[NLTE_MAXNG];
  const int ic = act[blockIdx.x], N = B.ndep[ic], nl = A.nl, tid = threadIdx.x, w = tid >> 6;
  const int NS = norder + 2, np = nl * N;
  const int64_t fs = B.fs, hs = (int64_t) nl * fs, o = (int64_t) ic * B.Kp;
  auto at = [&](int p) { return (int64_t) (p / N) * fs + o + p % N; };
  auto H = [&](int s, int64_t q) -> double & { return B.hist[(int64_t) s * hs + q]; };
  const int cur = niter % NS;
  for (int p = tid; p < np; p += NG_BLOCK) {
    const int64_t q = at(p);
    H(cur, q) = B.pops[q];
  }
  const int count = niter + 1;
  if (norder > 0 && count >= ndelay && !((count - ndelay) % nperiod)) {
    double Am[NLTE_MAXNG][NLTE_MAXNG], bv[NLTE_MAXNG];
#pragma unroll
    for (int i = 0; i < NLTE_MAXNG; i++) {
      bv[i] = 0.0;
#pragma unroll
      for (int j = 0; j < NLTE_MAXNG; j++) Am[i][j] = 0.0;
    }
    // (each thread reads the history entries that it writes)
    for (int p = tid; p < np; p += NG_BLOCK) {
      const int64_t q = at(p);
      double D[NLTE_MAXNG + 1];
#pragma unroll
      for (int r = 0; r <= NLTE_MAXNG; r++) {
        D[r] = 0.0;
        // count >= ndelay >= norder + 2, so both slots are >= 0
        if (r <= norder) D[r] = H((count - 1 - r) % NS, q) - H((count - 2 - r) % NS, q);
      }
      const double wt = 1.0 / fabs(B.pops[q]);
#pragma unroll
      for (int j = 0; j < NLTE_MAXNG; j++) {
        if (j < norder) {
          bv[j] += wt * D[0] * (D[0] - D[j + 1]);
#pragma unroll
          for (int ii = 0; ii < NLTE_MAXNG; ii++)
            if (ii < norder) Am[ii][j] += wt * (D[j + 1] - D[0]) * (D[ii + 1] - D[0]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NLTE_MAXNG; i++) {
      for (int s = 32; s >= 1; s >>= 1) bv[i] += __shfl_xor(bv[i], s);
      if ((tid & 63) == 0) part[w][i] = bv[i];
#pragma unroll
      for (int j = 0; j < NLTE_MAXNG; j++) {
        for (int s = 32; s >= 1; s >>= 1) Am[i][j] += __shfl_xor(Am[i][j], s);
        if ((tid & 63) == 0) part[w][NLTE_MAXNG * (i + 1) + j] = Am[i][j];
      }
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
      for (int i = 0; i < NLTE_MAXNG; i++) {
        bv[i] = 0.0;
        for (int v = 0; v < NW; v++) bv[i] += part[v][i];
#pragma unroll
        for (int j = 0; j < NLTE_MAXNG; j++) {
          Am[i][j] = (i < norder && j < norder) ? 0.0 : (i == j ? 1.0 : 0.0);
          for (int v = 0; v < NW; v++) Am[i][j] += part[v][NLTE_MAXNG * (i + 1) + j];
        }
      }
      solve_improve_r<NLTE_MAXNG>(Am, bv);
#pragma unroll
      for (int i = 0; i < NLTE_MAXNG; i++) coef[i] = bv[i];
    }
    __syncthreads();
    const int i0 = (count - 1) % NS;
    for (int p = tid; p < np; p += NG_BLOCK) {
      const int64_t q = at(p);
      double s = B.pops[q];
      const double h0 = H(i0, q);
#pragma unroll
      for (int r = 0; r < NLTE_MAXNG; r++)
        if (r < norder) s += coef[r] * (H((count - 2 - r) % NS, q) - h0);
      B.pops[q] = s;
      H(i0, q) = s;
    }
  }
  double dmax = 0.0;
  {
    const int so = (count - 2) % NS, sc = (count - 1) % NS;
    for (int p = tid; p < np; p += NG_BLOCK) {
      const int64_t q = at(p);
      const double c = H(sc, q);
      if (c) {
        const double d = fabs((c - H(so, q)) / c);
        dmax = dmax > d ? dmax : d;
      }
    }
  }
  for (int s = 32; s >= 1; s >>= 1) {
    const double x = __shfl_xor(dmax, s);
    dmax = dmax > x ? dmax : x;
  }
  __syncthreads();
  if ((tid & 63) == 0) part[w][0] = dmax;
  __syncthreads();
  if (tid == 0) {
    for (int v = 1; v < NW; v++) dmax = dmax > part[v][0] ? dmax : part[v][0];
    dpops[ic] = dmax;
  }
}

// populations (src: current or LTE) to the caller's layout
// [ncol][nl][Nmax], zero past ndep
__global__ void k_nlte_out(const DevNlte *__restrict__ Ap, NlteBufs B, const double *__restrict__ src,
                           double *__restrict__ out) {
  const DevNlte &A = *Ap;
  const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  const int ncol = B.ncol, Nmax = B.Nmax, nl = A.nl;
  if (p >= (int64_t) ncol * nl * Nmax) return;
  const int k = (int) (p % Nmax);
  const int64_t q = p / Nmax;
  const int i = (int) (q % nl), ic = (int) (q / nl);
  out[p] = k < B.ndep[ic] ? src[(int64_t) i * B.fs + (int64_t) ic * B.Kp + k] : 0.0;
}

}  // namespace rhg
