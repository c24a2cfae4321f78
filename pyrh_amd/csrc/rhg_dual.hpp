// Functions of the formal solution and the line profiles with their
// derivatives, for the response functions.
#pragma once

#include "rhg_device.hpp"

namespace rhg {

// a value and its derivative
struct Dual {
  double v, d;
};

// Cubic Bezier weights with their derivatives in dt: the derivative of
// exactly the branch bezier3() evaluates.  Closed forms N(t)/t^3 give
// (N'(t) - 3 N(t)/t) / t^3 with
//   N_alpha' = 6 - 6t + 3t^2 - 6e,     N_beta'  = t^3 e,
//   N_gamma' = 3 (-4 + 2t + (4 + 2t) e),  N_theta' = 3 (2 - (2 + 2t + t^2) e),  e = exp(-t);
// the series (the reference's 4th-order branch, rh/bezier_aux.c:350-357) is
// differentiated term by term.
__device__ __forceinline__ Bezier3<Dual> bezier3_d(double t) {
  const Bezier3<double> b = bezier3(t);
  double da, db, dg, dth, de;
  if (t < 5.e-2) {
    const double t2 = t * t, t3 = t2 * t;
    da = 0.25 - 0.10 * t + t2 / 40.0 - t3 / 210.0;
    db = 0.25 - 0.40 * t + t2 / 4.0 - t3 * (4.0 / 42.0);
    dg = 0.25 - 0.20 * t + t2 * 0.075 - t3 * (4.0 / 210.0);
    dth = 0.25 - 0.30 * t + t2 * 0.15 - t3 * (4.0 / 84.0);
    de = -1.0 + t - 0.5 * t2 + t3 / 6.0;
  } else {
    const double e = b.eps, it = 1.0 / t, it3 = it * it * it;
    da = (6.0 - 6.0 * t + 3.0 * t * t - 6.0 * e) * it3 - 3.0 * b.alpha * it;
    db = e - 3.0 * b.beta * it;
    dg = 3.0 * (-4.0 + 2.0 * t + (4.0 + 2.0 * t) * e) * it3 - 3.0 * b.gamma * it;
    dth = 3.0 * (2.0 - (2.0 + 2.0 * t + t * t) * e) * it3 - 3.0 * b.theta * it;
    de = -e;
  }
  return {{b.alpha, da}, {b.beta, db}, {b.gamma, dg}, {b.theta, dth}, {b.eps, de}};
}

// w3 weights (rh/w3.c:44-63) with derivatives in dtau: w0' = e, w1' = dtau e
// (e = exp(-dtau)); the small-dtau series and the large-dtau limits are
// differentiated as written.
__device__ __forceinline__ void w3d(double dtau, double *w, double *dw) {
  w3(dtau, w);
  if (dtau < 5.0E-4) {
    dw[0] = 1.0 - dtau;
    dw[1] = dtau * (1.0 - dtau);
  } else if (dtau > 50.0) {
    dw[0] = dw[1] = 0.0;
  } else {
    const double e = exp(-dtau);
    dw[0] = e;
    dw[1] = dtau * e;
  }
}

// H and its partial derivatives in a and v.  w = H + iF is an analytic
// function of z = a - iv inside each region (a quotient N/D, region IV with
// exp(z^2)), so w' = (N' - w D') / D in closed form gives H_a = Re w' and
// H_v = Im w' (Cauchy-Riemann).  A dual-number evaluation of the same
// quotients costs three times the plain function; this about twice.
template <typename R>
__device__ __forceinline__ R voigt_humlicek_d(R a, R v, int region, R *Ha, R *Hv) {
  const cpx<R> z = {a, -v};
  cpx<R> n, d, dn, dd, e = {R(0), R(0)};
  if (region == 0) {
    n = {R(0.5641896) * z.r, R(0.5641896) * z.i};
    d = cmul(z, z);
    d.r = d.r + R(0.5);
    dn = {R(0.5641896), R(0)};
    dd = {R(2) * z.r, R(2) * z.i};
  } else if (region == 1) {
    const cpx<R> u = cmul(z, z);
    cpx<R> t = {R(0.5641896) * u.r + R(1.410474), R(0.5641896) * u.i};
    n = cmul(z, t);
    dn = {R(3.0 * 0.5641896) * u.r + R(1.410474), R(3.0 * 0.5641896) * u.i};
    d = cmul(u, {u.r + R(3), u.i});
    d.r = d.r + R(0.75);
    dd = cmul(z, {R(4) * u.r + R(6), R(4) * u.i});
  } else if (region == 2) {
    const R a3[5] = {R(0.5642236), R(3.778987), R(11.96482), R(20.20933), R(16.4955)};
    const R b3[5] = {R(6.699398), R(21.69274), R(39.27121), R(38.82363), R(16.4955)};
    n = {a3[0], R(0)};
    d = {z.r + b3[0], z.i};
    dn = {R(0), R(0)};
    dd = {R(1), R(0)};
#pragma unroll
    for (int k = 1; k < 5; k++) {
      dn = cmul(dn, z); dn.r = dn.r + n.r; dn.i = dn.i + n.i;
      dd = cmul(dd, z); dd.r = dd.r + d.r; dd.i = dd.i + d.i;
      n = cmul(n, z); n.r = n.r + a3[k];
      d = cmul(d, z); d.r = d.r + b3[k];
    }
  } else {
    const R a4[7] = {R(0.56419), R(1.320522), R(35.7668), R(219.031), R(1540.787), R(3321.99),
                     R(36183.31)};
    const R b4[7] = {R(1.841439), R(61.57037), R(364.2191), R(2186.181), R(9022.228), R(24322.84),
                     R(32066.6)};
    const cpx<R> zz = cmul(z, z), u = {-zz.r, -zz.i};
    cpx<R> p = {a4[0], R(0)}, pu = {R(0), R(0)}, du = {R(1), R(0)};
    d = {u.r + b4[0], u.i};
#pragma unroll
    for (int k = 1; k < 7; k++) {
      pu = cmul(u, pu); pu.r = pu.r + p.r; pu.i = pu.i + p.i;
      du = cmul(u, du); du.r = du.r + d.r; du.i = du.i + d.i;
      p = cmul(u, p); p.r = p.r + a4[k];
      d = cmul(u, d); d.r = d.r + b4[k];
    }
    const R ex = rexp(zz.r);
    R sn, cs;
    rsincos(zz.i, &sn, &cs);
    e = {ex * cs, ex * sn};
    n = cmul(z, p);
    // d/dz = -2z d/du: n' = p - 2 z^2 p_u = p + 2 u p_u, d' = -2 z d_u
    const cpx<R> upu = cmul(u, pu);
    dn = {p.r + R(2) * upu.r, p.i + R(2) * upu.i};
    dd = cmul({R(-2) * z.r, R(-2) * z.i}, du);
  }
  const R id = rrcp(d.r * d.r + d.i * d.i);
  auto over_d = [&](cpx<R> x) {
    return cpx<R>{(x.r * d.r + x.i * d.i) * id, (x.i * d.r - x.r * d.i) * id};
  };
  const cpx<R> w = over_d(n), wd = cmul(w, dd);
  const cpx<R> dw = over_d({dn.r - wd.r, dn.i - wd.i});
  if (region == 3) {
    const cpx<R> ze = cmul(z, e);
    *Ha = R(2) * ze.r - dw.r;
    *Hv = R(2) * ze.i - dw.i;
    return e.r - w.r;
  }
  *Ha = dw.r;
  *Hv = dw.i;
  return w.r;
}

}  // namespace rhg
