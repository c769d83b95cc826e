// Scalar pieces of the shared search space (multik.hip): plain functions of doubles, the same
// on the host and on the device.
#pragma once
#include <cmath>

#if defined(__HIPCC__)
#define OMX_HD __host__ __device__ inline
#else
#define OMX_HD inline
#endif

namespace omx {

// Position of d[a] among d[0 .. n) in ascending order, equal values by index and NaN last: over
// a = 0 .. n - 1 the positions are a permutation whatever d holds.  (Ranked by < alone, values
// that are not numbers all get position 0 and leave other positions without an owner.)
OMX_HD int mk_position(const double* d, int n, int a) {
  const double da = d[a];
  const bool na = da != da;
  int r = 0;
  for (int l = 0; l < n; ++l) {
    const double dl = d[l];
    const bool nl = dl != dl;
    const bool before = nl != na ? na : (!na && dl != da ? dl < da : l < a);
    r += before ? 1 : 0;
  }
  return r;
}

constexpr int MK_NODES = 8;  // interpolation nodes of the norm's Gram matrix

// The norm's entries 1 / (rho^2 + k^2) are interpolated in x = ln k, at Chebyshev nodes over the
// columns' range of x (widened to 2% where it is narrower).  In x every entry is analytic for
// |Im x| < pi / 2 whatever its rho, and the one at rho = 0 everywhere, where in k the nearest
// pole is k = 0 at rho = 0.  Worst relative error over rho and k, by the ratio of the largest
// to the smallest k of the range: 2e-12 at 1.2, 1e-9 at 1.5, 9e-8 at 2, 5e-6 at 3, 1.3e-4 at 5 (at
// nodes in k itself 4e-10, 2e-7, 2e-5, 8e-4, 2e-2).
struct MkRange {
  double c, h;  // centre and half-width in x
};
OMX_HD MkRange mk_range(double lo, double hi) {  // of |k|
  const double a = log(lo), b = log(hi);
  return MkRange{0.5 * (a + b), fmax(0.5 * (b - a), 0.01)};
}
OMX_HD void mk_extent(const double* k, int n, double& lo, double& hi) {
  lo = hi = fabs(k[0]);
  for (int j = 1; j < n; ++j) {
    const double a = fabs(k[j]);
    lo = fmin(lo, a);
    hi = fmax(hi, a);
  }
}
OMX_HD double mk_node(const MkRange& r, int t) {  // in x
  return r.c + r.h * cos(M_PI / MK_NODES * (t + 0.5));
}
// Lagrange weight of node t at k and its k-derivative
OMX_HD void mk_weight(const double* node, int t, double k, double& w, double& dw) {
  const double x = log(fabs(k));
  w = 1;
  dw = 0;
  for (int u = 0; u < MK_NODES; ++u) {
    if (u == t) continue;
    const double q = 1.0 / (node[t] - node[u]);
    dw = dw * (x - node[u]) * q + w * q;
    w *= (x - node[u]) * q;
  }
  dw /= k;
}

}  // namespace omx
