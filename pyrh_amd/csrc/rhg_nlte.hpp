// NLTE solution of one active atom per column: device copy of the atom,
// the batch's device arrays and the kernels of the accelerated lambda
// iteration (rh/iterate.c:48-143 as rhf1d() runs it).
#pragma once

#include "rhg_kernels.hpp"

namespace rhg {

constexpr double RBOHR = 5.29177349E-11;       // rh/constant.h
constexpr double E_RYDBERG = 2.1798741E-18;

// transitions active at one wavelength, and levels of the active atom
constexpr int NLTE_MAXSET = 8;
constexpr int NLTE_MAXLEV = 16;
constexpr int NLTE_MAXNG = 4;                  // Ng order
// rays of k_nlte_feautrier solved together (more rays in chunks of this many)
constexpr int NLTE_FE_RAYS = 5;
// LDS of a k_nlte_feautrier workgroup for `per` columns of at most Nd depths,
// in doubles
constexpr int nlte_fe_lds(int Nd, int per, int rays) { return per * Nd * (3 + 2 * rays); }
// threads of k_nlte_ng; wavefronts of k_nlte_stateq for up to nlp levels
constexpr int NG_BLOCK = 256;
constexpr int stateq_waves(int nlp) { return nlp <= 6 ? 8 : 4; }
constexpr int stateq_depths(int nlp) { return nlp <= 8 ? 64 : 16; }   // of a workgroup: at most 32 KB of LDS
// depth-fastest copies of column-state fields (rows of NlteBufs::geo)
enum { NG_T = 0, NG_VLOS, NG_DZ, NG_HEIGHT, NG_N };
// k_nlte_bezier: whether the member data of a thread's P points lies in LDS
// (48 KB at most), and a workgroup's LDS in doubles
constexpr bool nlte_stash(int L, int P, int MS) { return MS <= 2 && L * P <= 384; }
constexpr int nlte_bez_lds(int L, int P, int MS) {
  return L * P + (nlte_stash(L, P, MS) ? P * MS * 4 * 2 * L : 0);
}
// rows of depths are padded to whole 64-byte lines
constexpr int nlte_pitch(int Nmax) { return (Nmax + 7) & ~7; }

// Device mirror of rhg_nlte_t, plus two derived tables: the transition of
// each line (ln_tr) and each line's first row in the profile array
// (ln_phi).  Entry e of the quadrature of transition t at grid point
// nblue + la is tr_ptr[t] + la; it also numbers the rate accumulators.
struct DevNlte {
  int nl, atom_index, he_atom, ntrans, nline, ncoll, nrays, nentry, nphi;
  double weight, sigma_thomson;
  const double *E, *g;
  const int32_t *stage;
  const int32_t *tr_type, *tr_i, *tr_j, *tr_nblue, *tr_nlam, *tr_ptr, *tr_line;
  const double *tr_wlam, *tr_alpha;
  const double *ln_lambda0, *ln_Aji, *ln_Bji, *ln_Bij, *ln_Grad, *ln_vdw_cross, *ln_vdw_alpha,
      *ln_vdw_cross_he, *ln_stark_c, *ln_stark_C, *ln_stark_Cm;
  const int32_t *ln_vdw, *ln_stark, *ln_tr, *ln_phi;
  const int32_t *as_ptr, *as_tr, *as_bezier;
  const int32_t *coll_type, *coll_i, *coll_j, *coll_ptr;
  const double *coll_T, *coll_c, *coll_M;
  const double *muz, *wmu, *ray_H, *ray_He, *ray_H2;
};

// Device arrays of one batch of ncol columns.  Except for the LTE inputs
// (state, lte_chi, lte_eta: column-fastest) every per-depth array is
// depth-fastest: x[row * fs + column * Kp + k], fs = ncol * Kp, row being a
// level, a line, a level pair (i * nl + j), an output wavelength, ...
struct NlteBufs {
  int ncol, Nmax, Kp, nfield, nout;
  int64_t fs;
  const int32_t *ndep;
  double *state;                  // LTE column state, fields RHG_CF_*
  const double *lte_chi, *lte_eta;  // [nout]: LTE continuum
  double *geo;                    // [NG_N]: T, vlos, path, height
  double *nstar, *pops;           // [nl]: LTE and current populations
  double *ntot, *vbroad, *nHe;    // [1]: atom total, Doppler width, He I ground
  double *adamp, *wphi;           // [nline]: damping, 1 / profile normalisation
  double *Cmat;                   // [nl * nl]: collision matrix
  double *phi;                    // [(nphi * nrays + mu) * 2 + to_obs]: profiles
  double *cchi, *ceta, *csca;     // [nout]: background opacity (with scattering),
                                  //         emissivity and scattering opacity
  double *J;                      // [2 * nout]: mean intensity, previous and new
  int32_t *jpar;                  // per column: which half of J is the previous
  double *acc;                    // [nentry * 2 + s]: rate terms per quadrature point
  double *dJ;                     // column x [nlist]: max |1 - J_old / J| per wavelength
  double *hist;                   // [(ng_order + 2) * nl]: Ng history
};

__global__ void k_nlte_pre(const DevModel *Mp, const DevNlte *Ap, NlteBufs B);
// (tiles of 32 columns x 32 depths) (nout + NG_N) workgroups of 256 threads
__global__ void k_nlte_bg(const DevModel *Mp, const DevNlte *Ap, NlteBufs B,
                          const int32_t *out_ls);
// nphi ceil(ncol Nmax / 64) workgroups of 64 threads
__global__ void k_nlte_profile(const DevModel *Mp, const DevNlte *Ap, NlteBufs B);
__global__ void k_nlte_wphi(const DevNlte *Ap, NlteBufs B);
template <int L, int P, int MS>
__global__ void k_nlte_bezier(const DevModel *Mp, const DevNlte *Ap, NlteBufs B,
                              const int32_t *act, int nact, const int32_t *out_ls,
                              const int32_t *io_list, int nlist, int il_off, int nlist_all,
                              int eval_op);
template <int MS, bool EM>
__global__ void k_nlte_feautrier(const DevModel *Mp, const DevNlte *Ap, NlteBufs B,
                                 const int32_t *act, int nact, int per, int Nd,
                                 const int32_t *out_ls, const int32_t *io_list, int nlist,
                                 int il_off, int nlist_all, int eval_op, double mu_em,
                                 double *stokes);
__global__ void k_nlte_flip(NlteBufs B, const int32_t *act, int nact);
template <int L, int P>
__global__ void k_nlte_emergent(const DevModel *Mp, const DevNlte *Ap, NlteBufs B,
                                const int32_t *act, int nact, const int32_t *out_ls,
                                const int32_t *io_list, int nlist, double mu, double *stokes);
__global__ void k_nlte_djmax(NlteBufs B, const int32_t *act, int nact, int nlist,
                             double *djmax);
template <int NLP>
__global__ void k_nlte_stateq(const DevNlte *Ap, NlteBufs B, const int32_t *act, int nact,
                              int isum, int share);
__global__ void k_nlte_ng(const DevNlte *Ap, NlteBufs B, const int32_t *act, int nact,
                          int niter, int norder, int ndelay, int nperiod, double *dpops);
__global__ void k_nlte_out(const DevNlte *Ap, NlteBufs B, const double *src, double *out);

}  // namespace rhg
