// Response functions of the emergent Stokes vector to the atmosphere,
// dStokes(lambda)/d p(k) for p in {T, v_LOS, B, gamma, chi, v_mic} at every
// depth k, for the polarized (DELO-Bezier) wavelengths.
//
// Four parts:
//  1. Tangents of the column state.  The equilibria of one depth depend
//     only on that depth's inputs, so one central difference with every
//     depth perturbed at once gives d(field)/d p(k) at all depths
//     (k_rf_perturb + k_state twice, FP64); the same for the continuum and
//     for chi at the reference wavelength.
//  2. k_rf_points: the points (opacity, source functions, reduced
//     propagation matrix) of every ray and depth, in parallel over depths;
//     k_rf_forward: the recursion of k_formal_stokes on them, which also
//     keeps, per ray, the 13 carried scalars entering each depth step
//     (Stokes vector, derivatives of S and q, optical-depth interval, chi
//     derivative).
//  3. k_rf_reverse: one reverse depth sweep per ray for the four outputs
//     I, Q, U, V at once, with the hand-written vector-Jacobian product of
//     each step (delo_step_vjp, rhg_adjoint.hpp), reading the same points.
//     Each point's adjoint is stored once, when the last step reading it is
//     done, with those of the path lengths |dz| and of the lower boundary's
//     Planck values.
//  4. k_rf_chain: per (ray, depth), the point adjoints pulled back through
//     the point's formation (line opacity, Zeeman-split Voigt profiles,
//     continuum) to the column state and contracted with each parameter's
//     state tangent, plus the path-length terms (tau500 scale: dz(j)
//     depends on chi_ref at j-1 and j) and the boundary terms.
// The recursion, its adjoint and the points are FP64 in both forms; the FP32
// form evaluates the Voigt functions (and their derivatives) in float.
#pragma once

#include "rhg_adjoint.hpp"

namespace rhg {

template <typename T>
__device__ __forceinline__ T &point_ref(Point<T> &p, int m) {
  switch (m) {
    case 0: return p.chi;
    case 1: return p.S[0];
    case 2: return p.S[1];
    case 3: return p.S[2];
    case 4: return p.S[3];
    case 5: return p.q[0];
    case 6: return p.q[1];
    default: return p.q[2];
  }
}

template <typename T>
__device__ __forceinline__ T point_get(const Point<T> &p, int m) {
  switch (m) {
    case 0: return p.chi;
    case 1: return p.S[0];
    case 2: return p.S[1];
    case 3: return p.S[2];
    case 4: return p.S[3];
    case 5: return p.q[0];
    case 6: return p.q[1];
    case 7: return p.q[2];
    default: return p.r[m - 8];
  }
}

// ---------------------------------------------------------------------------
// 2. forward pass storing the carried recursion state

// carry[((t * Nmax + k) * NCARRY_STEP + c) * ncol + column] (t = entry of the
// wavelength list): the carried state entering the step at depth k
// (k = 1 .. N-2); k = 0 holds the state entering the last interval.
// pts[((t * Nmax + k) * 8 + m) * ncol + column]: the points (point_get order).
#define RF_SETUP()                                                                       \
  const DevModel &M = *Mp;                                                               \
  int cb, t;                                                                             \
  xcd_tile(blockIdx.x, (ncol + 63) / 64, nlist, cb, t);                                  \
  const int ic = cb * 64 + threadIdx.x;                                                  \
  if (ic >= ncol) return;                                                                \
  const int io = io_list[t];                                                             \
  const int N = ndep[ic];                                                                \
  const int ls = out_ls[io];                                                             \
  const int64_t fs = (int64_t) Nmax * ncol;                                              \
  const double *st0 = state + ic;                                                        \
  const double *dzc = st0 + (int64_t) RHG_CF_DZ * fs;                                    \
  const double *Tc = st0 + (int64_t) RHG_CF_T * fs;                                      \
  const double *lc = M.lamconst + (int64_t) ls * RHG_LC_NCONST;                          \
  (void) lc; (void) Tc; (void) dzc;
// the wavelength's line table (before RF_SETUP: every lane of the wavefront
// takes part in staging it)
#define RF_LINE_TABLE()                                                                  \
  int cb0, t0;                                                                           \
  xcd_tile(blockIdx.x, (ncol + 63) / 64, nlist, cb0, t0);                                \
  if (cb0 * 64 >= ncol) return;                                                          \
  auto tab = [&]() {                                                                     \
    const int ls0 = out_ls[io_list[t0]];                                                 \
    if constexpr (LT) {                                                                  \
      extern __shared__ __align__(8) char lds_tab[];                                     \
      return stage_lines(*Mp, ls0, lds_tab, tab_maxl, tab_maxc);                         \
    } else {                                                                             \
      const int p0 = ldc(Mp->lam_line_ptr)[ls0];                                         \
      return LineTabG(*Mp, p0, ldc(Mp->lam_line_ptr)[ls0 + 1] - p0);                     \
    }                                                                                    \
  }()
#define DZ(kk) dzc[(int64_t) (kk) * ncol]
#define CAR(kk, c) car[((((int64_t) t * Nmax + (kk)) * NCARRY_STEP + (c)) * ncol) + ic]
// the point at depth jj
#define RF_POINT(jj, P)                                                                  \
  do {                                                                                   \
    const double *pp_ = pts + ((int64_t) t * Nmax + (jj)) * 8 * ncol + ic;               \
    P.chi = pp_[0];                                                                      \
    _Pragma("unroll") for (int n_ = 0; n_ < 4; n_++) P.S[n_] = pp_[(1 + n_) * (int64_t) ncol]; \
    _Pragma("unroll") for (int n_ = 0; n_ < 3; n_++) P.q[n_] = pp_[(5 + n_) * (int64_t) ncol]; \
  } while (0)

// The points of depths blockIdx.y * kd .. + kd - 1 of every ray: FP64, with
// the Voigt functions in R, the wavelength's line list staged in LDS (LT) or
// read from the model.  A ray's sweeps are a serial chain over depth and a
// small batch has few rays, so forming the points inside the sweeps (twice,
// and again in every wave's chain) left the chip idle: the points are formed
// here with every depth at once and read back, 64 bytes each.
//   90 columns of 64-256 depths, 350 wavelengths of the 400-line list, FP64:
//   forward 23.0 -> 2.3 + 9.9 for the points, reverse 75.8 -> 25.3 ms (5.0 for
//   points and forward and 9.0 since lists are dealt out in pieces, xcd_tile);
//   the 512-column 112-wavelength batch (FP32 form) 0.85 -> 0.20 + 0.25 and
//   1.87 -> 1.17 ms
// The synthesis of a batch of few rays takes the same two steps (MO: with the
// magneto-optical terms, three more numbers per point).
template <typename R, bool LT, bool MO>
__global__ void __launch_bounds__(64, 3)
k_rf_points(const DevModel *__restrict__ Mp, const int32_t *__restrict__ ndep,
            const int32_t *__restrict__ moving_arr, int ncol, int Nmax,
            const double *__restrict__ state, const int32_t *__restrict__ out_ls,
            const int32_t *__restrict__ io_list, int nlist, const R *__restrict__ cchi,
            const R *__restrict__ ceta, double mu_d, int kd, double *__restrict__ pts,
            int tab_maxl, int tab_maxc) {
  RF_LINE_TABLE();
  RF_SETUP();
  const int moving = moving_arr[ic];
  const R *cc = cchi + (int64_t) io * Nmax * ncol + ic;
  const R *ce = ceta + (int64_t) io * Nmax * ncol + ic;
  const int has_line = ldc(M.lam_line_ptr)[ls + 1] > ldc(M.lam_line_ptr)[ls];
  const int k0 = (int) blockIdx.y * kd, k1 = N < k0 + kd ? N : k0 + kd;
  for (int k = k0; k < k1; k++) {
    Point<double> P;
    form_point_vt<R, R, MO>(tab, M.ncont, has_line, st0 + (int64_t) k * ncol, fs, mu_d, moving,
                            cc[(int64_t) k * ncol], ce[(int64_t) k * ncol], P);
    constexpr int NC = point_ncomp(MO);
    double *pp = pts + ((int64_t) t * Nmax + k) * NC * ncol + ic;
#pragma unroll
    for (int m = 0; m < NC; m++) pp[m * (int64_t) ncol] = point_get(P, m);
  }
}

// TAPE: with the carried state for the reverse sweep; without, the synthesis
// of few rays, to column perm[ic] of the caller where there is a permutation.
template <int FORM, bool TAPE, bool MO>
__global__ void __launch_bounds__(64)
k_rf_forward(const DevModel *__restrict__ Mp, const int32_t *__restrict__ ndep,
             int ncol, int Nmax,
             const double *__restrict__ state, const int32_t *__restrict__ out_ls,
             const int32_t *__restrict__ io_list, int nlist, int nout,
             const double *__restrict__ pts, double mu_d,
             double *__restrict__ stokes, double *__restrict__ car,
             const int32_t *__restrict__ perm) {
  RF_SETUP();
  const double imu = 1.0 / mu_d;
  const double B2a = planck(Tc[(int64_t) (N - 2) * ncol], lc[RHG_LC_HC_KLA], lc[RHG_LC_TWOHNU3_C2]);
  const double B2b = planck(Tc[(int64_t) (N - 1) * ncol], lc[RHG_LC_HC_KLA], lc[RHG_LC_TWOHNU3_C2]);
  DeloState<double> s;
  Point<double> Pn, Pa;
  auto point = [&](int k, Point<double> &P) {
    constexpr int NC = point_ncomp(MO);
    const double *pp = pts + ((int64_t) t * Nmax + k) * NC * ncol + ic;
    P.chi = pp[0];
#pragma unroll
    for (int n = 0; n < 4; n++) P.S[n] = pp[(1 + n) * (int64_t) ncol];
#pragma unroll
    for (int n = 0; n < 3; n++) {
      P.q[n] = pp[(5 + n) * (int64_t) ncol];
      P.r[n] = MO ? pp[(8 + n) % NC * (int64_t) ncol] : 0.0;
    }
  };
  point(N - 1, Pa);
  auto tape = [&](int k) {
    if constexpr (TAPE) {
      double cv[NCARRY_STEP];
      carry_to_array(s, cv);
#pragma unroll
      for (int c = 0; c < NCARRY_STEP; c++) CAR(k, c) = cv[c];
    }
  };
  for (int j = N - 1; j >= -1; j--) {
    // the next point's loads are in flight while this step runs
    Pn = Pa;
    if (j > 0) point(j - 1, Pa);
    if (j == N - 1) {
      s.Pu = Pn;
    } else if (j == N - 2) {
      s.P0 = Pn;
    } else if (j == N - 3) {
      delo_prologue<double>(s, Pn, DZ(N - 1), DZ(N - 2), imu, B2a, B2b);
    } else {
      const int k = j + 2;
      tape(k);
      if constexpr (MO) delo_step_mo<double>(s, Pn, j >= 0, DZ(k), j >= 0 ? DZ(k - 1) : 0.0, imu);
      else delo_step<double>(s, Pn, j >= 0, DZ(k), j >= 0 ? DZ(k - 1) : 0.0, imu);
    }
  }
  tape(0);
  double x[4];
  if constexpr (MO) delo_final_mo<double>(s, DZ(1), imu, x);
  else delo_final<double>(s, DZ(1), imu, x);
  const int oc = perm ? perm[ic] : ic;
  double *out = stokes + (int64_t) oc * 4 * nout + io;
#pragma unroll
  for (int i = 0; i < 4; i++) out[(int64_t) i * nout] = x[i];
}

// ---------------------------------------------------------------------------
// 3. reverse sweep

// adjoint layout (t = list entry, o = output I, Q, U, V):
//   aP[(((t * 4 + o) * Nmax + k) * 8 + m) * ncol + column]   point k (chi, S, q)
//   aZ[((t * 4 + o) * Nmax + k) * ncol + column]     (k = 1 .. N-1: |dz(k)|)
//   aB[((t * 4 + o) * 2 + i) * ncol + column]          (i = 0: B(N-2), 1: B(N-1))
#define AP(o, kk, m) aP[(((((int64_t) t * 4 + (o)) * Nmax + (kk)) * 8 + (m)) * ncol) + ic]
#define AZ(o, kk) aZ[((((int64_t) t * 4 + (o)) * Nmax + (kk)) * ncol) + ic]
#define AB(o, i) aB[((((int64_t) t * 4 + (o)) * 2 + (i)) * ncol) + ic]

__device__ __forceinline__ void carry_from_array(const double *c, StepCarry &s) {
#pragma unroll
  for (int i = 0; i < 4; i++) s.Iv[i] = c[i];
#pragma unroll
  for (int i = 0; i < 4; i++) s.dSu[i] = c[4 + i];
#pragma unroll
  for (int i = 0; i < 3; i++) s.dqu[i] = c[8 + i];
  s.dtau_uw = c[11];
  s.dchi_c = c[12];
}

// The point adjoints of a sweep live in LDS, in a ring of four depth slots
// (depth j in slot j & 3) per output and component: [slot][o][m][lane].
// Each lane touches only its own entries.  add() takes the slots of the
// VJP routines (0 = Pu, 1 = P0, 2 = Pd, 3 = Pn) relative to the depth kp1 of
// Pu.
template <typename A>
struct PbarRing {
  A *base;
  int lane, kp1;
  __device__ __forceinline__ A &at(int depth, int o, int m) const {
    return base[((((depth & 3) * 4 + o) * 8) + m) * 64 + lane];
  }
  __device__ __forceinline__ void add(int slot, int o, int m, double v) const {
    at(kp1 - slot, o, m) += A(v);
  }
};

// One reverse sweep per (column, wavelength) for the four outputs at once:
// the last interval, each depth step and the prologue by their hand-written
// vector-Jacobian products (rhg_adjoint.hpp), on k_rf_points's points (one
// read per step, the point k+1 entering the window of step k); the carried
// state entering each step comes from the forward pass.  A point's adjoint
// is complete after the step at which it is the second point downwind
// (k = j + 2) and is stored then, once; a path length's after the step
// downwind of it.
template <typename R>
__global__ void __launch_bounds__(64)
k_rf_reverse(const DevModel *__restrict__ Mp, const int32_t *__restrict__ ndep,
             int ncol, int Nmax,
             const double *__restrict__ state, const int32_t *__restrict__ out_ls,
             const int32_t *__restrict__ io_list, int nlist, const double *__restrict__ pts,
             double mu_d, const double *__restrict__ car,
             R *__restrict__ aP, R *__restrict__ aZ, R *__restrict__ aB) {
  __shared__ R ring_lds[4 * 4 * 8 * 64];
  RF_SETUP();
  const double imu = 1.0 / mu_d;
  PbarRing<R> ring{ring_lds, (int) threadIdx.x, 1};
  for (int d = 0; d < 4; d++)
#pragma unroll
    for (int o = 0; o < 4; o++)
#pragma unroll
      for (int m = 0; m < 8; m++) ring.at(d, o, m) = R(0);

  // window of points: Pw[0..3] = depths k+1, k, k-1, k-2 at step k (shifted
  // before each step); path-length adjoints |dz(k)|, |dz(k-1)|
  Point<double> Pw[4];
  R zb[4][2];
  StepCarry Cb[4];
#pragma unroll
  for (int o = 0; o < 4; o++) zb[o][0] = zb[o][1] = R(0);

  // --- last interval: Pu = depth 1, P0 = depth 0
  RF_POINT(1, Pw[0]);
  RF_POINT(0, Pw[1]);
  {
    double cv[NCARRY_STEP];
#pragma unroll
    for (int c = 0; c < NCARRY_STEP; c++) cv[c] = CAR(0, c);
    StepCarry C0;
    carry_from_array(cv, C0);
    const double xb[4][4] = {{1, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 1, 0}, {0, 0, 0, 1}};
    R dzb[4] = {R(0), R(0), R(0), R(0)};
    ring.kp1 = 1;
    delo_final_vjp<4>(C0, Pw[0], Pw[1], DZ(1), imu, xb, Cb, ring, dzb);
#pragma unroll
    for (int o = 0; o < 4; o++) zb[o][0] = dzb[o];
  }
#pragma unroll
  for (int o = 0; o < 4; o++) AZ(o, 0) = R(0);

  // --- steps k = 1 .. N-2, the reverse of the forward order
  for (int k = 1; k <= N - 2; k++) {
    Pw[3] = Pw[2];
    Pw[2] = Pw[1];
    Pw[1] = Pw[0];
    RF_POINT(k + 1, Pw[0]);
    double cv[NCARRY_STEP];
#pragma unroll
    for (int c = 0; c < NCARRY_STEP; c++) cv[c] = CAR(k, c);
    StepCarry C;
    carry_from_array(cv, C);
    const bool has_pn = k >= 2;
    R dzb[4], dz1b[4];
#pragma unroll
    for (int o = 0; o < 4; o++) { dzb[o] = zb[o][0]; dz1b[o] = zb[o][1]; }
    ring.kp1 = k + 1;
    delo_step_vjp<4>(C, Pw[0], Pw[1], Pw[2], Pw[3], has_pn, DZ(k), has_pn ? DZ(k - 1) : 0.0,
                     imu, Cb, ring, dzb, dz1b);
    // point k-2 and |dz(k-1)| are complete; the slot of k-2 is k+2's next
    if (has_pn) {
#pragma unroll
      for (int o = 0; o < 4; o++) {
#pragma unroll
        for (int m = 0; m < 8; m++) {
          AP(o, k - 2, m) = ring.at(k - 2, o, m);
          ring.at(k - 2, o, m) = R(0);
        }
        AZ(o, k - 1) = dz1b[o];
      }
    }
#pragma unroll
    for (int o = 0; o < 4; o++) {
      zb[o][1] = dzb[o];
      zb[o][0] = R(0);
    }
  }
  // Pw[0..2] = depths N-1, N-2, N-3; zb = |dz(N-1)|, |dz(N-2)|

  // --- prologue
  {
    const double B2a = planck(Tc[(int64_t) (N - 2) * ncol], lc[RHG_LC_HC_KLA], lc[RHG_LC_TWOHNU3_C2]);
    const double B2b = planck(Tc[(int64_t) (N - 1) * ncol], lc[RHG_LC_HC_KLA], lc[RHG_LC_TWOHNU3_C2]);
    R dz1b[4], dz2b[4], bab[4], bbb[4];
#pragma unroll
    for (int o = 0; o < 4; o++) {
      dz1b[o] = zb[o][0];
      dz2b[o] = zb[o][1];
      bab[o] = bbb[o] = R(0);
    }
    ring.kp1 = N - 1;
    delo_prologue_vjp<4>(Pw[0], Pw[1], Pw[2], DZ(N - 1), DZ(N - 2), imu, B2a, B2b, Cb, ring,
                         dz1b, dz2b, bab, bbb);
#pragma unroll
    for (int o = 0; o < 4; o++) {
      AZ(o, N - 1) = dz1b[o];
      AZ(o, N - 2) = dz2b[o];
      AB(o, 0) = bab[o];
      AB(o, 1) = bbb[o];
#pragma unroll
      for (int m = 0; m < 8; m++) {
        AP(o, N - 1, m) = ring.at(N - 1, o, m);
        AP(o, N - 2, m) = ring.at(N - 2, o, m);
        AP(o, N - 3, m) = ring.at(N - 3, o, m);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// 4. chain to the atmosphere parameters

// rf[((((i * Nmax + k) * 4 + o) * nout + io) * ldr + column] for the i-th
// requested parameter pl.p[i]; chiref and dchiref are [column][depth] (as
// k_geometry writes chi_ref).  Per (ray, depth) the four outputs' point
// adjoints are pulled back through the point's formation: to the opacities
// and emissivities (reading the point itself from k_rf_points), per line to
// chi_l, eta_l, the damping, the Doppler width, v_LOS, B and the angles, and
// those are contracted with the parameters' state tangents.  What a parameter
// moves is known: T the line constants, the continuum, the path lengths and
// the boundary; v_mic the Doppler width and damping; v_LOS, B and the angles
// their own fields (the tangents of all other fields are zero).
//
// The depths are independent: workgroup (ray block, y) takes depths y * kd ..
// + kd - 1.  A Zeeman component costs one Voigt function with its derivative
// and four sums whatever the number of parameters: u = v - shift vB, so a
// Delta M group needs S(H), S(H_a), S(H_v), S(shift H_v) only.  (Evaluating
// the point on dual numbers, one tangent per parameter, was bound by the
// registers of those tangents: 1 wave per SIMD, 53.1 ms for 90 columns of
// 64-256 depths x 350 wavelengths of the 400-line list, FP64, T, v_LOS and
// B, and 2.49 ms for 512 columns x 112 wavelengths, FP32 form, all six.  This
// form: 33.4 and 1.59 ms at two waves per SIMD; 10.2 and 1.56 since lists are
// dealt out in pieces, xcd_tile.)
template <typename R, bool LT>
__global__ void __launch_bounds__(64, 2)
k_rf_chain(const DevModel *__restrict__ Mp, const int32_t *__restrict__ ndep,
           const int32_t *__restrict__ moving_arr, int ncol, int Nmax,
           const double *__restrict__ state, const double *__restrict__ dstate,
           const double *__restrict__ chiref, const double *__restrict__ dchiref,
           const double *__restrict__ pts, const R *__restrict__ dcchi,
           const R *__restrict__ dceta, const int32_t *__restrict__ out_ls,
           const int32_t *__restrict__ io_list, int nlist, int nout, double mu, int atm_scale,
           RfParamList pl, const R *__restrict__ aP, const R *__restrict__ aZ,
           const R *__restrict__ aB, R *__restrict__ rf, int64_t ldr, int kd, int tab_maxl,
           int tab_maxc) {
  RF_LINE_TABLE();
  RF_SETUP();
  const int moving = moving_arr[ic];
  const int lb = line_field_base(M.ncont);
  const int64_t tan_stride = (int64_t) state_nfield(M.ncont, M.nline) * fs;
  bool wants[RHG_RF_NPARAM];
#pragma unroll
  for (int q = 0; q < RHG_RF_NPARAM; q++) {
    wants[q] = false;
#pragma unroll
    for (int i = 0; i < RHG_RF_NPARAM; i++) wants[q] |= i < pl.npar && pl.p[i] == q;
  }
  const bool want_T = wants[RHG_RF_T], want_vm = wants[RHG_RF_VMIC];
  const int k0 = (int) blockIdx.y * kd, k1 = N < k0 + kd ? N : k0 + kd;
  for (int k = k0; k < k1; k++) {
    const double *stk = st0 + (int64_t) k * ncol;
    // tangent of field f along parameter q at this depth
    auto tangent = [&](int q, int f) { return dstate[q * tan_stride + f * fs + (int64_t) k * ncol + ic]; };
    Point<double> P;
    RF_POINT(k, P);
    // adjoints of chi_I,Q,U,V (ac) and eta_I,Q,U,V (ae): S_n = eta_n / chi_I,
    // q_n = chi_n / chi_I
    double ac[4][4], ae[4][4];
    const double ichi = rrcp(P.chi);
#pragma unroll
    for (int o = 0; o < 4; o++) {
      ac[o][0] = (double) AP(o, k, 0);
#pragma unroll
      for (int n = 0; n < 4; n++) {
        ae[o][n] = (double) AP(o, k, 1 + n) * ichi;
        ac[o][0] -= ae[o][n] * P.S[n];
      }
#pragma unroll
      for (int n = 0; n < 3; n++) {
        ac[o][1 + n] = (double) AP(o, k, 5 + n) * ichi;
        ac[o][0] -= ac[o][1 + n] * P.q[n];
      }
    }
    const double vz = stk[RHG_CF_VLOS * fs], Bf = stk[RHG_CF_B * fs], cosg = stk[RHG_CF_COSG * fs],
                 cos2x = stk[RHG_CF_COS2X * fs], sin2x = stk[RHG_CF_SIN2X * fs];
    const double sin2 = 1.0 - cosg * cosg;
    // adjoints of v_LOS, B, cos gamma, cos 2chi, sin 2chi; responses to T, v_mic
    double a_vz[4], a_B[4], a_g[4], a_c[4], a_s[4], r_T[4], r_vm[4];
#pragma unroll
    for (int o = 0; o < 4; o++) a_vz[o] = a_B[o] = a_g[o] = a_c[o] = a_s[o] = r_T[o] = r_vm[o] = 0.0;
    for (int i = 0; i < tab.n; i++) {
      const int l = tab.line(i);
      const double chi_l = stk[(lb + 4 * l) * fs], eta_l = stk[(lb + 4 * l + 1) * fs];
      const double adamp = stk[(lb + 4 * l + 2) * fs], ivb = stk[(lb + 4 * l + 3) * fs];
      double t_chi = 0.0, t_eta = 0.0, t_a = 0.0, t_ivb = 0.0, m_a = 0.0, m_ivb = 0.0;
      if (want_T) {
        t_chi = tangent(RHG_RF_T, lb + 4 * l);
        t_eta = tangent(RHG_RF_T, lb + 4 * l + 1);
        t_a = tangent(RHG_RF_T, lb + 4 * l + 2);
        t_ivb = tangent(RHG_RF_T, lb + 4 * l + 3);
      }
      if (want_vm) {
        m_a = tangent(RHG_RF_VMIC, lb + 4 * l + 2);
        m_ivb = tangent(RHG_RF_VMIC, lb + 4 * l + 3);
      }
      double dv = tab.dv(i);
      if (moving) dv += mu * vz;
      const double v = dv * ivb, sv = ivb * INV_SQRTPI;
      if (tab.damped(i) && tab.polar(i)) {
        const double vB1 = tab.larmor(i) * ivb, vB = vB1 * Bf;
        auto add = [&](int nz, double (&s)[4]) {
          const double sh = tab.shift(nz), sg = tab.strength(nz), u = v - sh * vB;
          R Ha, Hv;
          const R H0 = voigt_humlicek_d<R>((R) adamp, (R) u, humlicek_region(adamp, u), &Ha, &Hv);
          const double sHv = sg * (double) Hv;
          s[0] += sg * (double) H0;
          s[1] += sg * (double) Ha;
          s[2] += sHv;
          s[3] += sh * sHv;
        };
        double s[3][4] = {};
        const int c0 = tab.c0(i), c1 = tab.c1(i);
        if constexpr (LT) {
          const int cpi = tab.cpi(i), csp = tab.csp(i);
          for (int nz = c0; nz < cpi; nz++) add(nz, s[0]);
          for (int nz = cpi; nz < csp; nz++) add(nz, s[1]);
          for (int nz = csp; nz < c1; nz++) add(nz, s[2]);
        } else {
          for (int nz = c0; nz < c1; nz++) {
            const int q = tab.q(nz);
            if (q == -1) add(nz, s[0]);
            else if (q == 0) add(nz, s[1]);
            else add(nz, s[2]);
          }
        }
        const double sigma = s[2][0] + s[0][0], diff = s[2][0] - s[0][0];
        const double delta = 0.5 * s[1][0] - 0.25 * sigma;
        const double f0 = (delta * sin2 + 0.5 * sigma) * sv, fq = delta * sin2 * sv,
                     f3 = 0.5 * diff * cosg * sv;
#pragma unroll
        for (int o = 0; o < 4; o++) {
          const double w_chi = ac[o][0] * f0 + (ac[o][1] * cos2x + ac[o][2] * sin2x) * fq + ac[o][3] * f3;
          const double w_eta = ae[o][0] * f0 + (ae[o][1] * cos2x + ae[o][2] * sin2x) * fq + ae[o][3] * f3;
          double w[4];
#pragma unroll
          for (int n = 0; n < 4; n++) w[n] = ac[o][n] * chi_l + ae[o][n] * eta_l;
          // coefficients of delta sin^2 sv, sigma sv / 2 and diff cos g sv / 2
          const double X = w[0] + w[1] * cos2x + w[2] * sin2x;
          const double A_d = X * sin2 * sv, A_s = 0.5 * w[0] * sv, A_f = 0.5 * w[3] * cosg * sv;
          const double W0 = A_s - A_f - 0.25 * A_d, W1 = 0.5 * A_d, W2 = A_s + A_f - 0.25 * A_d;
          const double C_a = W0 * s[0][1] + W1 * s[1][1] + W2 * s[2][1];
          const double C_v = W0 * s[0][2] + W1 * s[1][2] + W2 * s[2][2];
          const double C_vB = -(W0 * s[0][3] + W1 * s[1][3] + W2 * s[2][3]);
          const double C_sv = X * delta * sin2 + w[0] * 0.5 * sigma + w[3] * 0.5 * diff * cosg;
          const double C_ivb = C_v * dv + C_vB * (tab.larmor(i) * Bf) + C_sv * INV_SQRTPI;
          if (moving) a_vz[o] += C_v * mu * ivb;
          a_B[o] += C_vB * vB1;
          a_g[o] += (0.5 * w[3] * diff - 2.0 * cosg * X * delta) * sv;
          a_c[o] += w[1] * fq;
          a_s[o] += w[2] * fq;
          r_T[o] += w_chi * t_chi + w_eta * t_eta + C_a * t_a + C_ivb * t_ivb;
          r_vm[o] += C_a * m_a + C_ivb * m_ivb;
        }
      } else {
        // an unpolarized profile: phi_I only
        double H, Ha = 0.0, Hv;
        if (tab.damped(i)) {
          // Armstrong's function is analytic: central differences
          const double h = 1.0e-6;
          H = voigt_armstrong(adamp, v);
          Ha = (voigt_armstrong(adamp + h, v) - voigt_armstrong(adamp > h ? adamp - h : adamp, v)) /
               (adamp > h ? 2.0 * h : h);
          Hv = (voigt_armstrong(adamp, v + h) - voigt_armstrong(adamp, v - h)) / (2.0 * h);
        } else {
          H = fabs(v) <= MAX_GAUSS_DOPPLER ? exp(-v * v) : 0.0;
          Hv = -2.0 * v * H;
        }
#pragma unroll
        for (int o = 0; o < 4; o++) {
          const double w0 = (ac[o][0] * chi_l + ae[o][0] * eta_l) * sv, f0 = H * sv;
          const double C_ivb = w0 * Hv * dv + w0 * H * rrcp(ivb);
          if (moving) a_vz[o] += w0 * Hv * mu * ivb;
          r_T[o] += (ac[o][0] * t_chi + ae[o][0] * t_eta) * f0 + w0 * Ha * t_a + C_ivb * t_ivb;
          r_vm[o] += w0 * Ha * m_a + C_ivb * m_ivb;
        }
      }
    }
    if (want_T) {
      const int64_t ck = ((int64_t) io * Nmax + k) * ncol + ic;
      const double dcc = (double) dcchi[ck], dce = (double) dceta[ck];
#pragma unroll
      for (int o = 0; o < 4; o++) r_T[o] += ac[o][0] * dcc + ae[o][0] * dce;
      // path lengths on the tau500 scale: |dz(j)| = 2 (tau_j - tau_{j-1}) /
      // (chi_ref(j-1) + chi_ref(j)), j = k and k + 1
      if (atm_scale == 0) {
        const double dchi = dchiref[(int64_t) ic * Nmax + k];
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
          const int j = k + jj;
          if (j >= 1 && j <= N - 1) {
            const double den = chiref[(int64_t) ic * Nmax + j - 1] + chiref[(int64_t) ic * Nmax + j];
            const double dzdT = -DZ(j) / den * dchi;
#pragma unroll
            for (int o = 0; o < 4; o++) r_T[o] += (double) AZ(o, j) * dzdT;
          }
        }
      }
      // the thermalised lower boundary's Planck values
      if (k >= N - 2) {
        const double T = Tc[(int64_t) k * ncol], x = lc[RHG_LC_HC_KLA] / T;
        double dB = 0.0;
        if (x <= MAX_EXPONENT) {
          const double e = exp(x), B = lc[RHG_LC_TWOHNU3_C2] / (e - 1.0);
          dB = B * x * e / (e - 1.0) / T;
        }
        const double dTdp = tangent(RHG_RF_T, RHG_CF_T);
#pragma unroll
        for (int o = 0; o < 4; o++) r_T[o] += (double) AB(o, k - (N - 2)) * (dB * dTdp);
      }
    }
    auto store = [&](int i, const double (&r)[4]) {
#pragma unroll
      for (int o = 0; o < 4; o++)
        rf[((((int64_t) i * Nmax + k) * 4 + o) * nout + io) * ldr + ic] = (R) r[o];
    };
    for (int i = 0; i < pl.npar; i++) {
      const int q = pl.p[i];
      double r[4];
      if (q == RHG_RF_T) {
        store(i, r_T);
      } else if (q == RHG_RF_VMIC) {
        store(i, r_vm);
      } else if (q == RHG_RF_VLOS) {
        const double t = tangent(q, RHG_CF_VLOS);
#pragma unroll
        for (int o = 0; o < 4; o++) r[o] = a_vz[o] * t;
        store(i, r);
      } else if (q == RHG_RF_B) {
        const double t = tangent(q, RHG_CF_B);
#pragma unroll
        for (int o = 0; o < 4; o++) r[o] = a_B[o] * t;
        store(i, r);
      } else {
        const double tg = tangent(q, RHG_CF_COSG), tc = tangent(q, RHG_CF_COS2X),
                     ts = tangent(q, RHG_CF_SIN2X);
#pragma unroll
        for (int o = 0; o < 4; o++) r[o] = a_g[o] * tg + a_c[o] * tc + a_s[o] * ts;
        store(i, r);
      }
    }
  }
}

#undef RF_SETUP
#undef RF_LINE_TABLE
#undef RF_POINT
#undef DZ
#undef CAR
#undef AP
#undef AZ
#undef AB

#define RHG_RF_INST(R)                                                                          \
  RHG_RF_PTS(R, false, false) RHG_RF_PTS(R, true, false) RHG_RF_FWD(R, true, false)             \
  template __global__ void k_rf_reverse<R>(const DevModel *, const int32_t *,                  \
                                           int, int, const double *, const int32_t *,          \
                                           const int32_t *, int, const double *, double,       \
                                           const double *, R *, R *, R *);                     \
  RHG_RF_CHAIN(R, false)                                                                        \
  RHG_RF_CHAIN(R, true)
#define RHG_RF_PTS(R, LT, MO)                                                                   \
  template __global__ void k_rf_points<R, LT, MO>(                                              \
      const DevModel *, const int32_t *, const int32_t *, int, int, const double *,             \
      const int32_t *, const int32_t *, int, const R *, const R *, double, int, double *, int, int);
#define RHG_RF_FWD(R, TAPE, MO)                                                                 \
  template __global__ void k_rf_forward<sizeof(R) == 4, TAPE, MO>(                              \
      const DevModel *, const int32_t *, int, int, const double *, const int32_t *,             \
      const int32_t *, int, int, const double *, double, double *, double *, const int32_t *);
#define RHG_RF_CHAIN(R, LT)                                                                     \
  template __global__ void k_rf_chain<R, LT>(const DevModel *, const int32_t *, const int32_t *, \
                                             int, int, const double *, const double *,          \
                                             const double *, const double *, const double *,    \
                                             const R *, const R *, const int32_t *,             \
                                             const int32_t *, int, int, double, int,            \
                                             RfParamList, const R *, const R *, const R *, R *, \
                                             int64_t, int, int, int);

}  // namespace rhg
