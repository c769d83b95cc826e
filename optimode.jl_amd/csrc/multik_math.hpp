// Scalar pieces of the shared search space (multik.hip): plain functions of doubles, the same
// on the host and on the device.
#pragma once

#if defined(__HIPCC__)
#define OMX_HD __host__ __device__ __forceinline__
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

}  // namespace omx
