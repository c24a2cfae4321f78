// Hydrostatic-equilibrium builder (pyrh's hse(), rh/rhf1d/pyrh_hse.c:67-399)
// on the GPU: the device tables and the kernel.
#pragma once

#include "rhg_kernels.hpp"

namespace rhg {

// Device mirror of rhg_hse_t (element tables in device memory).
struct DevHse {
  int nel;
  const int32_t *el_nstage, *el_pf_ptr;
  const double *el_logpf, *el_ionpot, *el_abund;
  int lam_index, he_atom;
  double ray_H, ray_He, ray_H2, sigma_thomson, hmin_fudge, scatt_fudge;
  int nmax_iter;
  double iter_limit;
  // the record of what a layer's temperature fixes (nrec doubles: HSE_NMISC
  // numbers, HSE_NDZ + 1 level groups per molecule nucleus and He, a constant
  // per molecule, a factor per ionisation stage) and the segments
  // k_hse_tables forms it in: per segment kind, first item, slots, first
  // slot; per stage factor the partition-function row of the lower stage and
  // the ionisation potential [J]; the elements by stage count, most first:
  // first slot << 4 | stages (HSE_CODE_H: hydrogen), and the abundance
  int nrec, np_dz;
  const int32_t *seg, *sl_pf, *el_code;
  const double *sl_ip, *el_ab;
  // LDS of k_hse in doubles: first column, per column
  int lds_col0, lds_col;
};

constexpr int HSE_BLOCK = 64;
constexpr int32_t HSE_CODE_H = 1 << 30;
// ionisation differences to the ground level the level groups distinguish
constexpr int HSE_NDZ = 4;
// the record's first numbers: pow(C1/T, +-1.5), exp(E_ION_HMIN/kT),
// exp(Uk0 + chi_H/kT), the proton's level ratio times cNe_T^np_dz, and from
// HSE_A0 on the opacity factors
enum { HSE_T_P15 = 0, HSE_T_EHMIN, HSE_T_PM15, HSE_T_EH, HSE_T_NP, HSE_A0 };
enum { HSE_A_HMBF = 0, HSE_A_HMFF, HSE_A_OH, HSE_A_CH, HSE_A_HFF, HSE_A_H2P, HSE_A_H2M, HSE_A_HBF };
constexpr int HSE_NMISC = HSE_A0 + HSE_A_HBF + HSE_NDZ;
// segments of k_hse_tables
enum { HSE_SEG_STAGES = 0, HSE_SEG_GROUPS, HSE_SEG_MOLECULES, HSE_SEG_MISC };
constexpr int HSE_SEG = 16;
static_assert(HSE_NMISC <= HSE_SEG && HSE_NDZ + 1 <= HSE_SEG, "a segment holds them");

// Launch (ceil(npts / HSE_BLOCK), segments) workgroups of HSE_BLOCK threads.
__global__ void k_hse_tables(const DevModel *Mp, DevHse H, int npts, int Nmax, const int32_t *ndep,
                             const double *temp, double *tab);

// One column per group of `lpc` consecutive lanes (lpc a power of two up to
// 64), cpb <= 64 / lpc columns per workgroup, serial over depth from the top.
// The lanes of a group split the elements of each electron-density Newton
// step and the molecules of the chemical equilibrium; everything else they
// compute alike, and lane 0 of the group stores.  Launch ceil(ncol / cpb)
// workgroups of HSE_BLOCK threads with lds_col0 + cpb lds_col doubles of LDS.
template <int NN>
__global__ void k_hse(const DevModel *Mp, DevHse H, int lpc, int cpb, int ncol, int Nmax,
                      const int32_t *ndep, int atm_scale, const double *scale, const double *temp,
                      const double *pg_top, const double *tab, double *ne_out, double *nH_out,
                      double *rho_out, double *pg_out, int32_t *niter_out);

__global__ void k_ne_from_nh(const DevModel *Mp, DevHse H, int ncol, int Nmax,
                             const int32_t *ndep, const double *temp, const double *nH,
                             double *ne_out);

}  // namespace rhg
