// Scalar pieces of the shared search space (multik.hip): plain functions of doubles, the same
// on the host and on the device.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

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

constexpr int MK_MAXM = 18;   // columns per problem: nev (16) + guard (2)
constexpr int MK_MAXN = 54;   // search space [X W P]
constexpr int MK_GUARD = 2;
constexpr int MK_PLANES = 7;  // planes of a stored column
constexpr int MK_SWEEPS = 10;  // Jacobi sweeps whose rotations are kept (4 to 7 are made)
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

// columns of the widest block handed over for nev bands on a grid of K unknowns: the space's
// columns past the bands too
inline int multik_block(int nev, long K) {
  return int(std::max<long>(nev, std::min<long>(nev + MK_GUARD, K / 3)));
}

// Shapes and device bytes of the phase's large buffers, for P problems of at most mmax columns on
// N pixels.
struct MkSizes {
  long cs, slots, vecs;  // plane size; complex values of a problem's columns; columns in all
  int NT, pm;            // 16-column tiles, their columns
  long rpc;              // rows per Gram chunk
  int nch;               // Gram chunks
  long rotn;             // rotations kept per column
  size_t cols, dm, part, red, cblk, rot;
  size_t total() const { return cols + dm + part + red + cblk + rot; }
};
inline MkSizes multik_sizes(long N, long P, int mmax) {
  constexpr size_t C32 = 8, C64 = 16, ROT = 32;
  constexpr int NGRAM = 3 + MK_NODES + 1;
  MkSizes z;
  z.cs = (N + 63) / 64 * 64;
  z.slots = 5L * mmax * MK_PLANES * z.cs;
  z.vecs = P * mmax;
  const int nmax = 3 * mmax;
  z.NT = (nmax + 15) / 16;
  z.pm = 16 * z.NT;
  // about 128 Gram chunks over the problems, of whole 64-row steps, a stage of every wave or more
  // (32 / 64 / 128 / 256 chunks, us a launch: 128 / 111 / 103 / 103 at 256^2 and 30 columns, 554 /
  // 406 / 383 / 383 at 384^2 and 42, 1022 / 601 / 591 / 608 at 512 x 256 and 54)
  const long nchunk = std::max<long>(1, std::min<long>((N + 255) / 256, std::max<long>(8, 128 / P)));
  z.rpc = ((N + nchunk - 1) / nchunk + 63) / 64 * 64;
  z.nch = int((N + z.rpc - 1) / z.rpc);
  z.rotn = long(MK_SWEEPS) * nmax * ((nmax + 1) / 2);
  z.cols = C32 * size_t(P) * z.slots;
  z.dm = C32 * size_t(z.vecs) * 3 * z.cs;
  z.part = C32 * size_t(P) * z.nch * NGRAM * z.pm * z.pm;
  z.red = C64 * size_t(P) * NGRAM * z.pm * z.pm;
  z.cblk = C64 * size_t(z.vecs) * MK_MAXN * MK_MAXM;
  z.rot = ROT * size_t(z.vecs) * z.rotn;
  return z;
}

// Device bytes of a launch group of the batched solve: P problems, ninst bands in all, at most M
// a problem, on N pixels (vectors of K = 2 N in columns of ld).  Whichever is larger: one
// LOBPCG block per band (both precisions' batches), or the shared search space with the FP64
// blocks it hands over and their FP32 copy and residuals (a group of few modes a problem: its
// spaces are three columns per band and guard wide).  With both the refinement's and the
// correction solves' vectors and the problems' stacked fields.
inline size_t group_bytes(long N, long K, long ld, long P, long ninst, long M) {
  M = std::max(1L, std::min(M, 16L));  // mode counts outside are refused later
  const size_t lob = size_t(ninst) * M * (11 * size_t(ld) + 3 * size_t(N));
  const size_t both = size_t(ninst) * (16 * 16 * size_t(ld) + 16 * 3 * size_t(N)) + size_t(P) * 144 * size_t(N);
  const int mb = multik_block(int(M), K);
  const size_t blocks = size_t(ninst) * mb * (16 * (2 * size_t(ld) + 3 * size_t(N)) + 2 * 8 * size_t(ld));
  return both + std::max((16 + 8) * lob, blocks + multik_sizes(N, P, mb).total());
}

}  // namespace omx
