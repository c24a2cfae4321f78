// Response functions: the state-tangent kernels and the FP64 instantiations
// of the adjoint kernels of rhg_rf.hpp (the FP32 form's are in
// rhg_rf32.hip, compiled with FMA contraction and the FP32 form's FP64
// reciprocal).
#include "rhg_rf.hpp"

namespace rhg {

// ---------------------------------------------------------------------------
// 1. state tangents

// The perturbed copies of a batch's atmospheres [ncol][9][Nmax] (n values),
// side by side: copy s = blockIdx.y is the batch with row shift.row[s]
// moved by shift.h[s] at every column and depth.
__global__ void k_rf_perturb(const double *__restrict__ atmos, double *__restrict__ out,
                             int64_t n, int Nmax, RfShiftList shift) {
  const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int s = (int) blockIdx.y;
  const int r = (int) ((i / Nmax) % 9);
  out[(int64_t) s * n + i] = atmos[i] + (r == shift.row[s] ? shift.h[s] : 0.0);
}

// out[s * ncol + i] = ndep[i]: the depth counts of the copies side by side
__global__ void k_rf_rep_ndep(const int32_t *__restrict__ ndep, int ncol, int32_t *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncol) return;
  out[(int64_t) blockIdx.y * ncol + i] = ndep[i];
}

// Central difference of two copies in a batch of row width W (a column
// state [row][W], a continuum [row][W]): out[r][c] = (S[r][off_p + c] -
// S[r][off_m + c]) * scale for nrows rows and ncol columns, in the output
// type.
template <typename O>
__global__ void k_rf_diff(const double *__restrict__ S, int64_t W, int64_t off_p, int64_t off_m,
                          int ncol, int64_t nrows, double scale, O *__restrict__ out) {
  const int64_t g = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nrows * ncol) return;
  const int64_t r = g / ncol, c = g - r * ncol;
  const double *row = S + r * W;
  out[g] = (O) ((row[off_p + c] - row[off_m + c]) * scale);
}
template __global__ void k_rf_diff<double>(const double *, int64_t, int64_t, int64_t, int, int64_t,
                                           double, double *);
template __global__ void k_rf_diff<float>(const double *, int64_t, int64_t, int64_t, int, int64_t,
                                          double, float *);

// ---------------------------------------------------------------------------
// 5. the response functions contracted with a loss gradient

// out[m * ncol + c] = in[c * nm + m], a 32 x 32 tile per workgroup of 256
__global__ void __launch_bounds__(256)
k_rf_turn(const double *__restrict__ in, int ncol, int nm, double *__restrict__ out) {
  __shared__ double t[32][33];
  const int c0 = (int) blockIdx.x * 32, m0 = (int) blockIdx.y * 32, a = threadIdx.x & 31;
  for (int b = threadIdx.x >> 5; b < 32; b += 8)
    if (c0 + b < ncol && m0 + a < nm) t[b][a] = in[(int64_t) (c0 + b) * nm + m0 + a];
  __syncthreads();
  for (int b = threadIdx.x >> 5; b < 32; b += 8)
    if (c0 + a < ncol && m0 + b < nm) out[(int64_t) (m0 + b) * ncol + c0 + a] = t[a][b];
}

// out[c][row(i)][k] = sum over m = (Stokes parameter, wavelength) of
// gT[m][c] rf[i][k][m][c], columns on the lanes, two depths per thread (the
// gradient's row is read once for both).  Reads rf once: 451 MB for six
// parameters, 82 depths, 112 wavelengths and 512 columns in float, where the
// tensor library widened it to double and reordered it first (the whole
// gradient step 8.0 -> 5.4 ms).
template <typename R>
__global__ void __launch_bounds__(64)
k_rf_contract(const R *__restrict__ rf, const double *__restrict__ gT, int ncol, int nd, int nm,
              RfRowList rows, double *__restrict__ out) {
  const int c = (int) blockIdx.x * 64 + threadIdx.x, i = (int) blockIdx.z, k0 = 2 * (int) blockIdx.y;
  if (c >= ncol) return;
  const bool two = k0 + 1 < nd;
  const R *a = rf + ((int64_t) i * nd + k0) * nm * ncol + c, *b = two ? a + (int64_t) nm * ncol : a;
  double sa = 0.0, sb = 0.0;
#pragma unroll 8
  for (int m = 0; m < nm; m++) {
    const double g = gT[(int64_t) m * ncol + c];
    sa += g * (double) a[(int64_t) m * ncol];
    sb += g * (double) b[(int64_t) m * ncol];
  }
  double *o = out + ((int64_t) c * 9 + rows.row[i]) * nd + k0;
  o[0] = sa;
  if (two) o[1] = sb;
}
template __global__ void k_rf_contract<double>(const double *, const double *, int, int, int, RfRowList,
                                               double *);
template __global__ void k_rf_contract<float>(const float *, const double *, int, int, int, RfRowList,
                                              double *);

RHG_RF_INST(double)
// the synthesis of few rays
RHG_RF_PTS(double, false, true)
RHG_RF_PTS(double, true, true)
RHG_RF_FWD(double, false, false)
RHG_RF_FWD(double, false, true)

}  // namespace rhg
