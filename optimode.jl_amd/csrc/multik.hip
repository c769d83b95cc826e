// Shared-subspace eigensolve of all bands at once (see multik.hpp).
//
// Storage per problem, FP32: column slots of 7 planes of cs complex values (cs = N rounded up
// to 64, the pads stay zero): planes 0-2 F0, 3-4 F1 (x, y), pixels column-major (iy fastest,
// the order of eps6c); planes 5-6 g1, g2, plane waves row-major (ix fastest).  Slots: X and P
// in two buffers each (an iteration reads one and writes the other), W in one.
//
// One iteration t (launches over all problems; a problem that is done returns at once):
//   gram    three eps^-1-weighted Gram matrices of [F0 F1] and the norm's at its nodes (MFMA)
//   reduce  sum of the chunk partials
//   dense   per band: its pencil at k_j, Ritz pair j, Newton step of k_j
//   combine X <- S C, P <- [W P] C, one pass over all planes (F0 and F1 stay consistent with g)
//   colE    eps^-1 (F0 + k F1), inverse FFT along y
//   rowR    inverse FFT along x, residual r = M x - lam x and its norm, P-map, FFT along x
//   control norms, convergence, the columns that still iterate, k
//   colP    FFT along y, eps_ave, FFT back
//   rowW    FFT along x, w = P r -> g, D0 and D1, FFT along x
//   colF    FFT along y of the five planes
#include "multik.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "fft_lds.hpp"
#include "multik_math.hpp"
#include "omx_errors.hpp"
#include "rng.hpp"
#include "solver.hpp"

namespace omx {

namespace {

constexpr int PLANES = MK_PLANES;
constexpr double MK_CLUSTER = 3e-5;  // bands whose k agree to this take their vectors at one k
// A problem is left to the per-band form when nothing has come nearer to its thresholds for
// MK_IDLE iterations (solves that converge pause for a few), or when its bands' k spread over
// more than MK_WIDEST, where the norm's interpolation (multik_math.hpp) is past the thresholds:
// bands that do not propagate at omega, tolerances below single precision.
constexpr int MK_IDLE = 40;
constexpr double MK_WIDEST = 12;
constexpr int FT = 512;   // threads of the transform kernels
constexpr int NGRAM = 3 + MK_NODES + 1;  // G00, G01, G11, the nodes, the k-independent part

struct MkState {
  int m, nev;              // columns, bands
  int na, np;              // W columns and P columns of the current search space
  int iter, done, par;     // done: 1 converged, 2 not finite, 3 given up; par: X / P buffer of the last space
  int ahead;               // most bands converged at once so far
  int idle;                // iterations since that or `worst` got better
  double worst;            // smallest over the iterations of the largest distance from the thresholds
  int moves;               // iterations whose Newton step moved a band's k by more than ftol
  int wcol[MK_MAXM];       // column of W slot s
  int pslot[MK_MAXM];      // P slots in use
  int its[MK_MAXM];        // iteration a band first met its thresholds (0: not yet)
  double omega2, tol, ftol;
  double k[MK_MAXM];       // current k per column
  double kold[MK_MAXM];    // k per column in the last iteration made
  double keval[MK_MAXM];   // k the column's Ritz pair was taken at
  double knew[MK_MAXM];    // after the Newton step
  double lam[MK_MAXM], slope[MK_MAXM], rnorm[MK_MAXM];
  double node[MK_NODES];   // interpolation nodes (in ln k) of the iteration under way
  float kap2[MK_NODES];    // their k^2
};

OMX_HD void set_node(MkState& s, const MkRange& r, int t) {
  s.node[t] = mk_node(r, t);
  s.kap2[t] = float(exp(2.0 * s.node[t]));
}

struct MkGeo {
  int nx, ny, mmax;
  long N, cs, slots;       // slots: complex values per problem in the column store
  double invdx, invdy;
  FFTFactors fx, fy;
  const c32 *twx, *twy;
  const float* eps6c;
  long eps_stride;
};

__device__ __forceinline__ long col_off(const MkGeo& g, int slot) { return long(slot) * PLANES * g.cs; }
// slots: X buffer b, P buffer b, W
__device__ __forceinline__ int slot_x(const MkGeo& g, int b, int c) { return b * g.mmax + c; }
__device__ __forceinline__ int slot_p(const MkGeo& g, int b, int c) { return (2 + b) * g.mmax + c; }
__device__ __forceinline__ int slot_w(const MkGeo& g, int c) { return 4 * g.mmax + c; }

// slot of search-space column q = [X (m) | W (na) | P (np)] with X, P in buffer b
__device__ __forceinline__ int space_slot(const MkGeo& g, const MkState& s, int b, int q) {
  if (q < s.m) return slot_x(g, b, q);
  if (q < s.m + s.na) return slot_w(g, q - s.m);
  return slot_p(g, b, s.pslot[q - s.m - s.na]);
}

// in-plane part of a plane wave: n = z x w / rho (y at rho = 0)
struct Wave {
  float n0, n1, rho2, rho;
};
__device__ __forceinline__ Wave wave_at(int ix, int iy, const MkGeo& g) {
  const float wx = -float(double(fft_index(ix, g.nx)) * g.invdx), wy = -float(double(fft_index(iy, g.ny)) * g.invdy);
  Wave v;
  v.rho2 = wx * wx + wy * wy;
  v.rho = sqrtf(v.rho2);
  const float ir = v.rho2 > 0.f ? 1.f / v.rho : 0.f;
  v.n0 = -wy * ir;
  v.n1 = v.rho2 > 0.f ? wx * ir : 1.f;
  return v;
}

// ---------------------------------------------------------------------------------------
// Start block: g of the X columns (buffer 0)
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_mk_start(MkGeo geo, c32* cols, const MkState* st, int p, const c64* src,
                                                  long lds, int nsrc, int hw, uint64_t seed) {
  const int c = blockIdx.y;
  const MkState& s = st[p];
  c32* g1 = cols + p * geo.slots + col_off(geo, slot_x(geo, 0, c)) + 5 * geo.cs;
  const double k = s.k[c];
  for (long e = long(blockIdx.x) * 256 + threadIdx.x; e < geo.N; e += long(gridDim.x) * 256) {
    const int iy = int(e / geo.nx), ix = int(e - long(iy) * geo.nx);
    const double wx = double(fft_index(ix, geo.nx)) * geo.invdx, wy = double(fft_index(iy, geo.ny)) * geo.invdy;
    const double w2 = wx * wx + wy * wy + k * k;
    c64 h1, h2;
    if (c >= nsrc) {
      // random, weighted like the operator's inverse so that the low plane waves lead
      const double f = 1.0 / w2;
      h1 = randn_at(seed, p, c, 2 * e);
      h2 = randn_at(seed, p, c, 2 * e + 1);
      h1 = c64{h1.x * f, h1.y * f};
      h2 = c64{h2.x * f, h2.y * f};
    } else if (hw > 0) {
      const int gx = ix < hw / 2 ? ix : ix - (geo.nx - hw), gy = iy < hw / 2 ? iy : iy - (geo.ny - hw);
      const bool in = (ix < hw / 2 || ix >= geo.nx - hw / 2) && (iy < hw / 2 || iy >= geo.ny - hw / 2);
      h1 = h2 = c64{0, 0};
      if (in) {
        const c64* v = src + long(c) * lds + 2 * (gx + long(hw) * gy);
        h1 = v[0];
        h2 = v[1];
      }
    } else {
      const c64* v = src + long(c) * lds + 2 * e;
      h1 = v[0];
      h2 = v[1];
    }
    const double w = sqrt(w2);
    g1[e] = c32{float(w * h1.x), float(w * h1.y)};
    g1[geo.cs + e] = c32{float(h2.x), float(h2.y)};
  }
}

// ---------------------------------------------------------------------------------------
// Gram matrices on the matrix cores.  As in block.hip: the four k slots of one
// v_mfma_f32_16x16x4 are four rows, lane (i = l % 16, g = l / 16) holds S consecutive rows of
// column i of each 16-column tile, loaded straight from HBM with 16-byte loads, and the
// waves of a block take interleaved stages.  KIND 0: F0^H e F0, 1: F0^H e F1, 2: F1^H e F1
// (e = eps^-1 per pixel, three components contracted per row), 3: the norm's matrices
// g^H psi g for NB of the nodes (psi = 1 / (rho^2 + kappa^2) on g1; the last one g2^H g2).
// Hermitian kinds compute the tiles on and above the diagonal only.
// ---------------------------------------------------------------------------------------
typedef float fx4 __attribute__((ext_vector_type(4)));
constexpr int GW = 8;  // waves per Gram block

__device__ __forceinline__ fx4 mfma(float a, float b, fx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int S> __device__ __forceinline__ void load_col(const c32* col, long row, c32 (&v)[S]) {
  if (col != nullptr) {
    const fx4* q = reinterpret_cast<const fx4*>(col + row);
#pragma unroll
    for (int j = 0; j < S / 2; ++j) {
      const fx4 w = q[j];
      v[2 * j] = c32{w.x, w.y};
      v[2 * j + 1] = c32{w.z, w.w};
    }
  } else {
#pragma unroll
    for (int j = 0; j < S; ++j) v[j] = c32{0.f, 0.f};
  }
}

template <int NT, int KIND, int NB, int S>
__device__ __forceinline__ void gram_body(const MkGeo& geo, const c32* const* cp, const float* kap2,
                                          float (*red)[8][64], int p, int q0, int nt, long rpc, c32* part) {
  constexpr int PM = 16 * NT, NQ = KIND == 3 ? NB : 1;
  const int chunk = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, g = lane >> 4;
  const c32* col[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) col[t] = cp[t * 16 + i16];
  fx4 ar[NQ][NT][NT], ai[NQ][NT][NT];
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) ar[q][a][b] = ai[q][a][b] = fx4{0.f, 0.f, 0.f, 0.f};
  // += conj(x) y over the rows of a stage, every tile pair
  auto product = [&](int q, const c32(&x)[NT][S], const c32(&y)[NT][S]) {
#pragma unroll
    for (int r = 0; r < S; ++r)
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) {
          if ((KIND != 1 && a > b) || a >= nt || b >= nt) continue;
          ar[q][a][b] = mfma(x[a][r].x, y[b][r].x, ar[q][a][b]);
          ai[q][a][b] = mfma(x[a][r].x, y[b][r].y, ai[q][a][b]);
          ar[q][a][b] = mfma(x[a][r].y, y[b][r].y, ar[q][a][b]);
          ai[q][a][b] = mfma(x[a][r].y, -y[b][r].x, ai[q][a][b]);
        }
  };
  const long r0 = chunk * rpc, r1 = r0 + rpc < geo.N ? r0 + rpc : geo.N;
  const float* eps = geo.eps6c + p * geo.eps_stride;
  for (long row = r0 + (wave * 4 + g) * S; row - g * S < r1; row += 4 * GW * S) {
    const bool in = row < r1;  // rows past r1 belong to the next chunk (or are pads)
    const c32* no = nullptr;
    if (KIND < 3) {
      float e[S][6];
#pragma unroll
      for (int r = 0; r < S; ++r)
#pragma unroll
        for (int c = 0; c < 6; ++c) e[r][c] = 0.f;
      if (in && row + S <= geo.N) {
        const fx4* q = reinterpret_cast<const fx4*>(eps + 6 * row);
#pragma unroll
        for (int j = 0; j < 6 * S / 4; ++j) {
          const fx4 w = q[j];
#pragma unroll
          for (int u = 0; u < 4; ++u) e[(4 * j + u) / 6][(4 * j + u) % 6] = w[u];
        }
      } else if (in) {
#pragma unroll
        for (int r = 0; r < S; ++r)
          if (row + r < geo.N)
#pragma unroll
            for (int c = 0; c < 6; ++c) e[r][c] = eps[6 * (row + r) + c];
      }
      c32 x[3][NT][S], y[3][NT][S];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const c32* c = in ? col[t] : no;
        if (KIND != 2)
#pragma unroll
          for (int a = 0; a < 3; ++a) load_col<S>(c ? c + a * geo.cs : no, row, x[a][t]);
        if (KIND != 0) {
          c32 f[2][S];
#pragma unroll
          for (int a = 0; a < 2; ++a) load_col<S>(c ? c + (3 + a) * geo.cs : no, row, f[a]);
#pragma unroll
          for (int r = 0; r < S; ++r) {
            y[0][t][r] = f[0][r] * e[r][0] + f[1][r] * e[r][3];
            y[1][t][r] = f[0][r] * e[r][3] + f[1][r] * e[r][1];
            if (KIND == 1) y[2][t][r] = f[0][r] * e[r][4] + f[1][r] * e[r][5];
            if (KIND == 2) {
              x[0][t][r] = f[0][r];
              x[1][t][r] = f[1][r];
            }
          }
        } else {
#pragma unroll
          for (int r = 0; r < S; ++r) {
            const c32 f0 = x[0][t][r], f1 = x[1][t][r], f2 = x[2][t][r];
            y[0][t][r] = f0 * e[r][0] + f1 * e[r][3] + f2 * e[r][4];
            y[1][t][r] = f0 * e[r][3] + f1 * e[r][1] + f2 * e[r][5];
            y[2][t][r] = f0 * e[r][4] + f1 * e[r][5] + f2 * e[r][2];
          }
        }
      }
#pragma unroll
      for (int a = 0; a < (KIND == 2 ? 2 : 3); ++a) product(0, x[a], y[a]);
    } else {
      c32 x[NT][S], x2[NT][S], y[NT][S];
      float rho2[S];
#pragma unroll
      for (int r = 0; r < S; ++r) {
        const long e = row + r;
        const int iy = int(e / geo.nx), ix = int(e - long(iy) * geo.nx);
        const float wx = float(double(fft_index(ix, geo.nx)) * geo.invdx);
        const float wy = float(double(fft_index(iy, geo.ny)) * geo.invdy);
        rho2[r] = wx * wx + wy * wy;
      }
      const bool last = q0 + NB > MK_NODES;  // this group holds the k-independent matrix
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const c32* c = in ? col[t] : no;
        if (q0 < MK_NODES) load_col<S>(c ? c + 5 * geo.cs : no, row, x[t]);
        if (last) load_col<S>(c ? c + 6 * geo.cs : no, row, x2[t]);
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        if (q0 + q < MK_NODES) {
          const float kk = kap2[q0 + q];
          float ps[S];
#pragma unroll
          for (int r = 0; r < S; ++r) ps[r] = 1.f / (rho2[r] + kk);
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < S; ++r) y[t][r] = x[t][r] * ps[r];
          product(q, x, y);
        } else if (q0 + q == MK_NODES) {
          product(q, x2, x2);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int gram = KIND == 3 ? 3 + q0 + q : KIND;
    if (gram >= NGRAM) break;
    c32* out = part + ((long(p) * gridDim.x + chunk) * NGRAM + gram) * PM * PM;
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        if ((KIND != 1 && a > b) || a >= nt || b >= nt) continue;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          red[wave][r][lane] = ar[q][a][b][r];
          red[wave][4 + r][lane] = ai[q][a][b][r];
        }
        __syncthreads();
        // wave w < 4 finishes accumulator register w: rows 4 g + w
        if (wave < 4) {
          float sr = 0.f, si = 0.f;
#pragma unroll
          for (int u = 0; u < GW; ++u) {
            sr += red[u][wave][lane];
            si += red[u][4 + wave][lane];
          }
          out[(a * 16 + 4 * g + wave) * PM + b * 16 + i16] = c32{sr, si};
        }
      }
  }
}

// One launch: blockIdx.z 0-2 the three eps^-1 kinds, then the node groups.  Eight waves per
// block: 128 chunks of four waves in a launch per kind left half the SIMDs without a wave
// (256^2, 30 columns: 155 us in four launches).
template <int NT, int NB, int S>
__global__ __launch_bounds__(64 * GW) void k_mk_gram(MkGeo geo, const c32* cols, const MkState* st, int buf, long rpc,
                                                     c32* part) {
  __shared__ const c32* cp[16 * NT];
  __shared__ float kap2[MK_NODES];
  __shared__ float red[GW][8][64];
  const int p = blockIdx.y, kind = blockIdx.z;
  const MkState& s = st[p];
  if (s.done) return;
  const int n = s.m + s.na + s.np, nt = (n + 15) / 16;
  if (threadIdx.x < 16 * NT)
    cp[threadIdx.x] =
        int(threadIdx.x) < n ? cols + p * geo.slots + col_off(geo, space_slot(geo, s, buf, threadIdx.x)) : nullptr;
  if (threadIdx.x < MK_NODES) kap2[threadIdx.x] = s.kap2[threadIdx.x];
  __syncthreads();
  if (kind == 0)
    gram_body<NT, 0, 1, S>(geo, cp, kap2, red, p, 0, nt, rpc, part);
  else if (kind == 1)
    gram_body<NT, 1, 1, S>(geo, cp, kap2, red, p, 0, nt, rpc, part);
  else if (kind == 2)
    gram_body<NT, 2, 1, S>(geo, cp, kap2, red, p, 0, nt, rpc, part);
  else
    gram_body<NT, 3, NB, S>(geo, cp, kap2, red, p, (kind - 3) * NB, nt, rpc, part);
}

// red[p][gram][e] = sum over the chunks, FP64, fixed order (16 elements x 16 chunk groups)
__global__ __launch_bounds__(256) void k_mk_reduce(const c32* part, int nchunk, int pm, const MkState* st, c64* red) {
  __shared__ double sx[16][17], sy[16][17];
  const int p = blockIdx.z, gram = blockIdx.y;
  const MkState& s = st[p];
  if (s.done) return;
  const int e = blockIdx.x * 16 + (threadIdx.x & 15), grp = threadIdx.x >> 4, el = threadIdx.x & 15;
  const int a = e / pm, b0 = (blockIdx.x * 16) % pm, n = s.m + s.na + s.np;
  // a block covers one row's 16-column tile: skip those not computed or not used
  if (a >= n || b0 >= n || (gram != 1 && (a >> 4) > (b0 >> 4))) return;
  const long esz = long(pm) * pm;
  const c32* q = part + (long(p) * nchunk * NGRAM + gram) * esz + e;
  double ax = 0, ay = 0;
#pragma unroll 8
  for (int c = grp; c < nchunk; c += 16) {
    const c32 v = q[long(c) * NGRAM * esz];
    ax += v.x;
    ay += v.y;
  }
  sx[grp][el] = ax;
  sy[grp][el] = ay;
  __syncthreads();
  if (grp == 0) {
    double tx = 0, ty = 0;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      tx += sx[u][el];
      ty += sy[u][el];
    }
    red[(long(p) * NGRAM + gram) * esz + e] = c64{tx, ty};
  }
}

// ---------------------------------------------------------------------------------------
// Dense step: one workgroup per band.
// ---------------------------------------------------------------------------------------
struct MkRot {
  double c;
  c64 s;
};

__device__ __forceinline__ void mk_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 1 / sqrt(x) for x in FP32's range: the FP32 estimate and two Newton steps (about 1e-15)
__device__ __forceinline__ double rsqrt_fast(double x) {
  double r = double(__builtin_amdgcn_rsqf(float(x)));
  const double h = 0.5 * x;
  r = r * (1.5 - h * r * r);
  r = r * (1.5 - h * r * r);
  return r;
}

// a value of lane l + 1 (UP false) or l - 1 (UP true) of the wavefront, lanes past the ends 0
template <bool UP> __device__ __forceinline__ double lane_shift(double v) {
  union {
    double d;
    int i[2];
  } u{v};
  u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], UP ? 0x138 : 0x130, 0xf, 0xf, true);
  u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], UP ? 0x138 : 0x130, 0xf, 0xf, true);
  return u.d;
}

// Parallel cyclic Jacobi (dense.hip's round-robin ordering and rotations) for Hermitian A
// (n x n, leading dimension ld) using A's symmetry: of the 2 x 2 blocks only those on and above
// the diagonal are computed and their mirrors stored.  Stops after a sweep whose rotations
// all have |sin| <= stop.  The eigenvectors are not accumulated (two thirds of a round's
// arithmetic): the rotations of round q go to rot[q npair + t], and a caller applies them in
// reverse to the few unit vectors it wants.  Returns the rounds made; A0 / A1 by parity hold
// the final matrix (rounds even: A0).
__device__ int mk_jacobi(c64* A0, c64* A1, int ld, int n, double stop, MkRot* rot) {
  __shared__ int big[3];
  __shared__ int rp[MK_MAXN / 2], rq[MK_MAXN / 2];
  __shared__ double rc[MK_MAXN / 2];
  __shared__ c64 rs[MK_MAXN / 2];
  __shared__ unsigned short tri[(MK_MAXN / 2) * (MK_MAXN / 2 + 1) / 2];
  const int m = n + (n & 1), npair = m / 2, nblk = npair * (npair + 1) / 2;
  if (n & 1)  // an odd size is padded by a zero row and column, which never rotate
    for (int e = threadIdx.x; e < m; e += blockDim.x) A0[n * ld + e] = A0[e * ld + n] = c64{0.0, 0.0};
  for (int e = threadIdx.x; e < npair * npair; e += blockDim.x) {
    const int a = e / npair, b = e - a * npair;
    if (a <= b) tri[a * npair - a * (a - 1) / 2 + (b - a)] = (unsigned short)(a * 64 + b);
  }
  if (threadIdx.x < 3) big[threadIdx.x] = 0;
  __syncthreads();
  c64 *Ac = A0, *An = A1;
  int rounds = 0, ua = (int(threadIdx.x) + m - 2) % (m - 1), ub = max(0, m - 2 - int(threadIdx.x));  // (t - 1), (m - 2 - t)
  for (int sweep = 0; sweep < MK_SWEEPS; ++sweep) {
    const int sl = sweep % 3;
    if (threadIdx.x == 0) big[(sweep + 1) % 3] = 0;
    for (int r = 0; r < m - 1; ++r) {
      if (int(threadIdx.x) < npair) {
        const int t = threadIdx.x;
        const int ia = t == 0 ? 0 : 1 + ua, ib = 1 + ub;
        ua = ua + 1 == m - 1 ? 0 : ua + 1;
        ub = ub + 1 == m - 1 ? 0 : ub + 1;
        const bool fwd = ia < ib;
        const int p = fwd ? ia : ib, q = fwd ? ib : ia;
        const double app = Ac[p * ld + p].x, aqq = Ac[q * ld + q].x;
        const c64 apq = Ac[p * ld + q];
        const double a2 = apq.x * apq.x + apq.y * apq.y;
        double c = 1.0;
        c64 sv{0.0, 0.0};
        // The angle is taken to FP32 accuracy (what is left of A_pq falls by 1e-7, a sweep's
        // other fill is larger), the rotation itself is unitary to FP64: three FP64 square
        // roots in a chain were half of a round's latency.
        if (a2 > 1e-30) {
          const double ia2 = rsqrt_fast(a2), z = 0.5 * (aqq - app) * ia2;
          const float az = fabsf(float(z));
          const float tf = az > 1e15f ? 0.f : 1.f / (az + sqrtf(1.f + az * az));
          c = rsqrt_fast(1.0 + double(tf) * tf);
          const double sn = double(tf) * c, f = (z >= 0 ? sn : -sn) * ia2;
          sv = c64{f * apq.x, f * apq.y};
          if (sn > stop) big[sl] = 1;
        }
        rp[t] = p;
        rq[t] = q;
        rc[t] = c;
        rs[t] = sv;
        // kept relative to (ia, ib), the order the reverse pass meets the pair in
        rot[long(rounds) * npair + t] = MkRot{c, fwd ? sv : c64{-sv.x, sv.y}};
      }
      __syncthreads();
      for (int idx = threadIdx.x; idx < nblk; idx += blockDim.x) {
        const int t1 = tri[idx] >> 6, t2 = tri[idx] & 63;
        const int p1 = rp[t1], q1 = rq[t1], p2 = rp[t2], q2 = rq[t2];
        const double c1 = rc[t1], c2 = rc[t2];
        const c64 s1 = rs[t1], s2 = rs[t2];
        const c64 x00 = Ac[p1 * ld + p2], x01 = Ac[p1 * ld + q2], x10 = Ac[q1 * ld + p2], x11 = Ac[q1 * ld + q2];
        const c64 y00 = x00 * c1 - s1 * x10, y01 = x01 * c1 - s1 * x11;
        const c64 y10 = cmulc(s1, x00) + x10 * c1, y11 = cmulc(s1, x01) + x11 * c1;
        const c64 z00 = y00 * c2 - cmulc(s2, y01), z01 = s2 * y00 + y01 * c2;
        const c64 z10 = y10 * c2 - cmulc(s2, y11), z11 = s2 * y10 + y11 * c2;
        An[p1 * ld + p2] = z00;
        An[p1 * ld + q2] = z01;
        An[q1 * ld + p2] = z10;
        An[q1 * ld + q2] = z11;
        if (t1 != t2) {
          An[p2 * ld + p1] = conj(z00);
          An[q2 * ld + p1] = conj(z01);
          An[p2 * ld + q1] = conj(z10);
          An[q2 * ld + q1] = conj(z11);
        }
      }
      __syncthreads();
      c64* tmp = Ac;
      Ac = An;
      An = tmp;
      ++rounds;
    }
    if (big[sl] == 0) break;
  }
  return rounds;
}

__device__ __forceinline__ double read_lane(double v, int l) {  // l uniform
  union {
    double d;
    int i[2];
  } u{v};
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
  return u.d;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
// 1 / x for normal x (estimate and two Newton steps)
__device__ __forceinline__ double rcp_fast(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = r * (2.0 - x * r);
  return r * (2.0 - x * r);
}

// c = D U^-1 v for a wavefront's vector (lane a holds entry a); dropped columns get 0
__device__ __forceinline__ c64 mk_backsub(c64 v, const c64* U, int ld, int n, const int* drop, const double* dsc,
                                          int lane) {
  for (int a = n - 1; a >= 0; --a) {
    const double ua = drop[a] ? 0.0 : rcp_fast(U[a * ld + a].x);
    const c64 ca{read_lane(v.x, a) * ua, read_lane(v.y, a) * ua};
    if (lane == a) v = ca;
    if (lane < a) v = v - U[lane * ld + a] * ca;
  }
  return lane < n ? v * dsc[lane] : c64{0.0, 0.0};
}

// Eigenpair j (0-based, ascending) of Hermitian A (n x n, all in LDS, destroyed): Householder
// tridiagonalisation with the congruence's layout (lane = column, rows dealt to the
// wavefronts; two barriers per step), then on the first wavefront multisection for the
// eigenvalue (64 Sturm counts per pass), the eigenvector of the tridiagonal matrix by its
// twisted factorisation, and the reflectors back.  Returns false, leaving the pair to the
// Jacobi, when another eigenvalue lies within 1e-4 of it: vectors of a cluster have to come
// from one decomposition.  lam and c = D U^-1 vector (into out) for every wavefront's use after
// the next barrier.  A full Jacobi (5 to 8 sweeps of n - 1 rounds at 0.8 us) finds n pairs
// where a band takes one.
template <int NW>
__device__ bool tridiag_pair(c64* A, int ld, int n, int j, c64 (*pr)[64], c64* part, double* lam, c64* out,
                             const c64* U, const int* drop, const double* dsc) {
  __shared__ double d[MK_MAXN], e[MK_MAXN], e2[MK_MAXN], dp[MK_MAXN], dm[MK_MAXN];
  __shared__ c64 tau[MK_MAXN];
  __shared__ int single;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const c64 zero{0.0, 0.0};
  if (wv == 0) pr[0][lane] = lane < n ? A[lane] : zero;
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    const c64 rowk = pr[k & 1][lane];
    if (k == n - 1) {
      if (threadIdx.x == 0) d[k] = pr[k & 1][k].x;
      break;
    }
    const c64 x = lane > k && lane < n ? conj(rowk) : zero;  // column k below the diagonal
    const double sg = wave_sum(lane > k + 1 ? abs2(x) : 0.0);
    const double ar = read_lane(x.x, k + 1), ai = read_lane(x.y, k + 1);
    c64 t = zero, v = lane == k + 1 ? c64{1.0, 0.0} : zero;
    double ek = ar;
    if (sg > 0.0 || ai != 0.0) {
      const double nrm = sqrt(ar * ar + ai * ai + sg);
      ek = ar >= 0 ? -nrm : nrm;
      const double ib = 1.0 / ek, dr = ar - ek, q = 1.0 / (dr * dr + ai * ai);
      t = c64{(ek - ar) * ib, -ai * ib};
      if (lane > k + 1) v = x * c64{dr * q, -ai * q};
    }
    // p = tau A v from the owned rows (A[a][b] v_b = conj(A[b][a]) v_b)
    c64 acc = zero;
    for (int b = wv; b < n; b += NW) {
      if (b <= k) continue;
      const c64 vb{read_lane(v.x, b), read_lane(v.y, b)};
      if (lane > k && lane < n) acc = acc + cmulc(A[b * ld + lane], vb);
    }
    part[wv * 64 + lane] = acc;
    if (wv == k % NW) {
      if (lane < n) A[k * ld + lane] = v;  // the reflector, for the way back
      if (lane == 0) {
        d[k] = pr[k & 1][k].x;
        e[k] = ek;
        e2[k] = ek * ek;
        tau[k] = t;
      }
    }
    __syncthreads();
    c64 pv = zero;
#pragma unroll
    for (int q = 0; q < NW; ++q) pv = pv + part[q * 64 + lane];
    pv = t * pv;
    const c64 pd = cmulc(pv, v);  // p^H v
    const c64 al = t * c64{-0.5 * wave_sum(pd.x), -0.5 * wave_sum(pd.y)};
    const c64 w = pv + al * v;
    for (int a = wv; a < n; a += NW) {
      if (a <= k) continue;
      const c64 va{read_lane(v.x, a), read_lane(v.y, a)}, wa{read_lane(w.x, a), read_lane(w.y, a)};
      if (lane > k && lane < n) {
        // v_a conj(w) + w_a conj(v)
        c64 u = A[a * ld + lane] - cmulc(w, va) - cmulc(v, wa);
        if (lane == a) u.y = 0.0;
        A[a * ld + lane] = u;
        if (a == k + 1) pr[(k + 1) & 1][lane] = u;
      }
    }
    __syncthreads();
  }
  __syncthreads();
  if (wv == 0) {
    const double di = lane < n ? d[lane] : 0.0;
    const double rad = (lane < n && lane > 0 ? fabs(e[lane - 1]) : 0.0) + (lane < n - 1 ? fabs(e[lane]) : 0.0);
    double lo = lane < n ? di - rad : 1e300, hi = lane < n ? di + rad : -1e300;
    for (int off = 32; off > 0; off >>= 1) {
      lo = fmin(lo, __shfl_xor(lo, off, 64));
      hi = fmax(hi, __shfl_xor(hi, off, 64));
    }
    const double scale = fmax(fabs(lo), fabs(hi)), tiny = 1e-30 * scale + 1e-300;
    lo -= 1e-12 * scale;
    hi += 1e-12 * scale;
    auto count = [&](double sig) {  // eigenvalues below sig
      double q = d[0] - sig;
      int c = q < 0;
      for (int i = 1; i < n; ++i) {
        if (fabs(q) < tiny) q = -tiny;
        q = (d[i] - sig) - e2[i - 1] * rcp_fast(q);
        c += q < 0;
      }
      return c;
    };
    for (int pass = 0; pass < 10 && hi - lo > 1e-13 * scale; ++pass) {
      const double sig = lo + (hi - lo) * ((lane + 1) * (1.0 / 65.0));
      const unsigned long long above = __ballot(count(sig) > j);
      const int f = above ? __ffsll((long long)above) - 1 : 64;
      const double nh = f < 64 ? __shfl(sig, f & 63, 64) : hi, nl = f > 0 ? __shfl(sig, (f - 1) & 63, 64) : lo;
      hi = nh;
      lo = nl;
    }
    const double l = 0.5 * (lo + hi), del = fmax(1e-4 * fabs(l), 1e-9 * scale);
    const int cc = count(lane == 0 ? l - del : l + del);
    const bool one = __shfl(cc, 1, 64) - __shfl(cc, 0, 64) == 1;
    if (lane == 0) {
      single = one ? 1 : 0;
      *lam = l;
    }
    if (one) {
      // LDL^H from the top (lane 0) and UDU^H from the bottom (lane 1), met at the index where
      // the twisted pivot is smallest
      if (lane < 2) {
        double q = 0;
        for (int i = 0; i < n; ++i) {
          const int r = lane == 0 ? i : n - 1 - i;
          q = (d[r] - l) - (i > 0 ? e2[lane == 0 ? r - 1 : r] * rcp_fast(q) : 0.0);
          if (fabs(q) < tiny) q = q < 0 ? -tiny : tiny;
          (lane == 0 ? dp : dm)[r] = q;
        }
      }
      mk_wave_sync();
      double g = lane < n ? fabs(dp[lane] + dm[lane] - (di - l)) : 1e300;
      int r = lane;
      for (int off = 32; off > 0; off >>= 1) {
        const double og = __shfl_xor(g, off, 64);
        const int orr = __shfl_xor(r, off, 64);
        if (og < g || (og == g && orr < r)) {
          g = og;
          r = orr;
        }
      }
      const double up = lane < n - 1 ? -e[lane] * rcp_fast(dp[lane]) : 0.0;
      const double dn = lane > 0 && lane < n ? -e[lane - 1] * rcp_fast(dm[lane]) : 0.0;
      // z_i = up_i z_{i+1} above the twist, dn_i z_{i-1} below it
      double z = lane == r ? 1.0 : 0.0, zc = 1.0;
      for (int i = r - 1; i >= 0; --i) {
        zc *= read_lane(up, i);
        if (lane == i) z = zc;
      }
      zc = 1.0;
      for (int i = r + 1; i < n; ++i) {
        zc *= read_lane(dn, i);
        if (lane == i) z = zc;
      }
      const double iz = 1.0 / sqrt(wave_sum(z * z));
      c64 yv{z * iz, 0.0};
      for (int k = n - 2; k >= 0; --k) {  // reflectors: y -= tau v (v^H y)
        const c64 v = lane > k && lane < n ? A[k * ld + lane] : zero;
        const c64 dt = cmulc(v, yv);
        const c64 sm = tau[k] * c64{wave_sum(dt.x), wave_sum(dt.y)};
        yv = yv - v * sm;
      }
      yv = mk_backsub(yv, U, ld, n, drop, dsc, lane);
      if (lane < n) out[lane] = yv;
    }
  }
  __syncthreads();
  return single != 0;
}

// Ritz pair j of the pencil (A(k), B(k)) of the search space at column j's k.  The pencil is
// scaled to unit B diagonal and reduced by the congruence that turns B into the identity
// (one elimination step per column, applied to A as well); columns whose pivot falls below
// 1e-5 (dependent to FP32 accuracy) are taken out of the space.  Bands whose k agree to 3e-5
// share one k, so that near-degenerate bands take different vectors of one decomposition.
// Latency-bound on one CU per band.
// FINAL false: Cx column j, lam, slope and the Newton step.  FINAL true (after the last
// iteration, at the k and on the Gram matrices of that iteration): the coefficients Cblk
// [column][vector] of the lowest msz vectors of each band's block.
template <int DT, bool FINAL>
__global__ __launch_bounds__(DT) void k_mk_dense(MkGeo geo, MkState* st, const c64* red, int pm, int ld, double stop,
                                                 const int* msz, c32* Cx, c64* Cblk, MkRot* rotg, long rotn) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int j = blockIdx.x, p = blockIdx.y;
  MkState& s = st[p];
  if (FINAL ? s.done != 1 || j >= s.nev : s.done || j >= s.m) return;
  const int n = s.m + s.na + s.np;
  c64* A = reinterpret_cast<c64*>(smem_raw);
  const int rows = (n + 1) & ~1;  // an odd size is padded to an even one in the Jacobi
  c64* A1 = A + rows * ld;
  c64* B = A1 + rows * ld;  // U of B = U^H U after the congruence
  __shared__ double node[MK_NODES], lw[MK_NODES], dlw[MK_NODES], dsc[MK_MAXN], diagv[MK_MAXN];
  __shared__ double kk_s, red_s[DT / 64];
  __shared__ int drop[MK_MAXN], rank[MK_MAXN];
  __shared__ c64 y[MK_MAXN];
  __shared__ c64 xs[DT / 64][64];
  __shared__ c64 prA[2][64], prB[2][64];
  __shared__ double lam_s;
  if (threadIdx.x == 0) {
    const double* kv = FINAL ? s.kold : s.k;
    int a = j, b = j;
    while (a > 0 && fabs(kv[a - 1] - kv[a]) < MK_CLUSTER * fabs(kv[a])) --a;
    while (b + 1 < s.m && fabs(kv[b + 1] - kv[b]) < MK_CLUSTER * fabs(kv[b])) ++b;
    double kk = 0;
    for (int i = a; i <= b; ++i) kk += kv[i];
    kk /= double(b - a + 1);
    kk_s = kk;
  }
  if (threadIdx.x < MK_NODES) node[threadIdx.x] = s.node[threadIdx.x];
  __syncthreads();
  const double kk = kk_s;
  if (threadIdx.x < MK_NODES) mk_weight(node, threadIdx.x, kk, lw[threadIdx.x], dlw[threadIdx.x]);
  __syncthreads();
  const long esz = long(pm) * pm;
  const c64* G = red + long(p) * NGRAM * esz;
  for (int e = threadIdx.x; e < n * n; e += DT) {
    const int a = e / n, b = e - a * n;
    if (a > b) continue;
    const long o = long(a) * pm + b;
    const c64 g00 = G[o], g01 = G[esz + o], g10 = G[esz + long(b) * pm + a], g11 = G[2 * esz + o];
    c64 va{g00.x + kk * (g01.x + g10.x) + kk * kk * g11.x, g00.y + kk * (g01.y - g10.y) + kk * kk * g11.y};
    c64 vb = G[(NGRAM - 1) * esz + o];
#pragma unroll
    for (int t = 0; t < MK_NODES; ++t) {
      const c64 w = G[(3 + t) * esz + o];
      vb.x += lw[t] * w.x;
      vb.y += lw[t] * w.y;
    }
    if (a == b) va.y = vb.y = 0;
    A[a * ld + b] = va;
    A[b * ld + a] = conj(va);
    B[a * ld + b] = vb;
  }
  __syncthreads();
  for (int a = threadIdx.x; a < n; a += DT) {
    const double d = B[a * ld + a].x;
    dsc[a] = d > 0 ? 1.0 / sqrt(d) : 0.0;
    drop[a] = 0;
  }
  __syncthreads();
  const double iN = 1.0 / double(geo.N);  // the transforms are unnormalised
  for (int e = threadIdx.x; e < n * n; e += DT) {
    const int a = e / n, b = e - a * n;
    const double f = dsc[a] * dsc[b];
    A[a * ld + b] = A[a * ld + b] * (f * iN);
    if (a <= b) B[a * ld + b] = B[a * ld + b] * f;
  }
  __syncthreads();
  // Congruence: after step k, rows and columns <= k of B are the identity's.  Lane b holds
  // column b, each wavefront the rows congruent to its number, and the pivot row comes from a
  // double buffer its owner filled one step earlier: one barrier per step (in three phases
  // with three barriers a step took 1.8 us).
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int NW = DT / 64;
  const c64 zero{0.0, 0.0};
  if (wv == 0) {
    prA[0][lane] = lane < n ? A[lane] : zero;
    prB[0][lane] = lane < n ? B[lane] : zero;
  }
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    const c64(*pa) = prA[k & 1];
    const c64(*pb) = prB[k & 1];
    const double d = pb[k].x;
    const bool bad = !(d > 1e-5);
    const double f = bad ? 0.0 : rsqrt_fast(d);
    const c64 ub = lane > k ? pb[lane] * f : zero;
    const c64 ak = lane != k ? pa[lane] * f : zero;
    const double akk = pa[k].x * f * f;
    const c64 fin = ak - ub * akk;  // row k after its own column operation
    for (int a = wv; a < n; a += NW) {
      if (a == k) {
        if (lane < n) A[k * ld + lane] = lane == k ? c64{akk, 0.0} : fin;
        if (lane > k && lane < n) B[k * ld + lane] = ub;
        if (lane == k) {
          B[k * ld + k] = c64{bad ? 0.0 : d * f, 0.0};  // U[k][k]
          drop[k] = bad ? 1 : 0;
        }
        continue;
      }
      const c64 ua{read_lane(ub.x, a), read_lane(ub.y, a)}, aka{read_lane(ak.x, a), read_lane(ak.y, a)};
      const c64 fa{read_lane(fin.x, a), read_lane(fin.y, a)};
      if (lane < n) {
        c64 v = A[a * ld + lane] - cmulc(ua, ak) - cmulc(aka, ub) + cmulc(ua, ub) * akk;
        if (lane == k) v = conj(fa);
        if (lane == a) v.y = 0.0;
        A[a * ld + lane] = v;
        c64 vb = zero;
        if (a > k && lane >= a) {
          vb = B[a * ld + lane] - cmulc(ua, ub);
          B[a * ld + lane] = vb;
        }
        if (a == k + 1) {
          prA[(k + 1) & 1][lane] = v;
          prB[(k + 1) & 1][lane] = vb;
        }
      }
    }
    __syncthreads();
  }
  // dropped columns: decoupled, at the end of the spectrum
  {
    double mx = 0;
    int any = 0;
    for (int a = 0; a < n; ++a) {
      mx = fmax(mx, fabs(A[a * ld + a].x));
      any |= drop[a];
    }
    __syncthreads();
    if (any)
      for (int e = threadIdx.x; e < n * n; e += DT) {
        const int a = e / n, b = e - a * n;
        if (drop[a] || drop[b]) A[a * ld + b] = a == b ? c64{16.0 * mx + 1.0, 0.0} : c64{0.0, 0.0};
      }
  }
  __syncthreads();
  bool jac = FINAL;
  if (!FINAL) {
    // keep the reduced matrix: the tridiagonal form overwrites it
    for (int a = wv; a < n; a += NW)
      if (lane < n) A1[a * ld + lane] = A[a * ld + lane];
    jac = !tridiag_pair<NW>(A, ld, n, j, prA, &xs[0][0], &lam_s, y, B, drop, dsc);
  }
  MkRot* rot = rotg + (long(p) * geo.mmax + j) * rotn;
  if (jac) {  // block-uniform
  const int rounds = mk_jacobi(FINAL ? A : A1, FINAL ? A1 : A, ld, n, stop, rot);
  const c64* Ad = ((rounds & 1) != 0) == FINAL ? A1 : A;
  for (int a = threadIdx.x; a < n; a += DT) diagv[a] = Ad[a * ld + a].x;
  __syncthreads();
  for (int a = threadIdx.x; a < n; a += DT) rank[mk_position(diagv, n, a)] = a;
  __threadfence_block();  // the block's rotations, read back below
  __syncthreads();
  if (!FINAL && threadIdx.x == 0) lam_s = diagv[rank[j]];
  // the wanted vectors: V e = (rotations in reverse) e, then c = D U^-1 V e; one wavefront per
  // vector, lane t the pair t of a round, the rotations staged in LDS
  const int m = n + (n & 1), npair = m / 2;
  const int v0 = FINAL ? 0 : j, nv = FINAL ? msz[p * MK_MAXM + j] : 1;
  // The vector stays in registers: lane t holds the pair's elements (xl, xr), and from a round to
  // the one before it all elements but the first move one place round the ring of pairs, i.e.
  // xl comes from lane t - 1 and xr from lane t + 1.
  MkRot* rl = reinterpret_cast<MkRot*>(A);  // both matrix buffers are free
  const int chunk = max(1, int(2L * rows * ld * sizeof(c64) / (sizeof(MkRot) * npair)));
  c64* Cb = Cblk + (long(p) * geo.mmax + j) * MK_MAXN * MK_MAXM;
  for (int base = 0; base < nv; base += DT / 64) {
    const bool mine = base + wv < nv;
    const int q = v0 + base + wv;
    // the pairs of the last round (rounds is a multiple of m - 1: its index within a sweep is m - 2)
    const int el = lane == 0 ? 0 : 1 + (lane - 1 + m - 2) % (m - 1), er = 1 + (m - 2 - min(lane, m - 2) + m - 2) % (m - 1);
    const int hot = mine ? rank[q] : -1;
    c64 xl{lane < npair && el == hot ? 1.0 : 0.0, 0.0}, xr{lane < npair && er == hot ? 1.0 : 0.0, 0.0};
    for (int r1 = rounds; r1 > 0; r1 -= chunk) {
      const int r0 = max(0, r1 - chunk), cnt = (r1 - r0) * npair;
      __syncthreads();
      for (int e = threadIdx.x; e < cnt; e += DT) rl[e] = rot[long(r0) * npair + e];
      __syncthreads();
      if (mine) {
        const int t = min(lane, npair - 1);
        MkRot R = rl[(r1 - 1 - r0) * npair + t];
        for (int r = r1 - 1; r >= r0; --r) {
          const MkRot Rn = rl[(max(r - 1, r0) - r0) * npair + t];
          const c64 yl = xl * R.c + R.s * xr, yr = xr * R.c - cmulc(R.s, xl);
          if (r == 0) {
            xl = yl;
            xr = yr;
          } else {
            // to round r - 1: L_t <- L_{t-1} (t >= 2), L_1 <- R_0, R_t <- R_{t+1}, R_last <- L_last
            const c64 sl{lane_shift<true>(lane == 0 ? yr.x : yl.x), lane_shift<true>(lane == 0 ? yr.y : yl.y)};
            const c64 sr{lane_shift<false>(yr.x), lane_shift<false>(yr.y)};
            xl = lane == 0 ? yl : sl;
            xr = lane == npair - 1 ? (npair == 1 ? yr : yl) : sr;
          }
          R = Rn;
        }
      }
    }
    if (mine && lane < npair) {  // pairs of round 0
      xs[wv][lane == 0 ? 0 : lane] = xl;
      xs[wv][1 + (m - 2 - lane)] = xr;
    }
    if (mine) {
      mk_wave_sync();
      c64 v = lane < n ? xs[wv][lane] : c64{0.0, 0.0};
      v = mk_backsub(v, B, ld, n, drop, dsc, lane);
      if (lane < n) {
        if (FINAL)
          Cb[lane * MK_MAXM + q] = v;
        else
          y[lane] = v;
      }
    }
  }
  }
  if (FINAL) return;
  __syncthreads();
  if (int(threadIdx.x) < n)
    Cx[(long(p) * MK_MAXN + threadIdx.x) * MK_MAXM + j] = c32{float(y[threadIdx.x].x), float(y[threadIdx.x].y)};
  // slope = y^H (dA/dk - lam dB/dk) y (y^H B y = 1)
  const double lam = lam_s;
  double acc = 0;
  for (int e = threadIdx.x; e < n * n; e += DT) {
    const int a = e / n, b = e - a * n;
    if (a > b) continue;
    const long o = long(a) * pm + b;
    const c64 g01 = G[esz + o], g10 = G[esz + long(b) * pm + a], g11 = G[2 * esz + o];
    c64 d{(g01.x + g10.x + 2 * kk * g11.x) * iN, (g01.y - g10.y + 2 * kk * g11.y) * iN};
#pragma unroll
    for (int t = 0; t < MK_NODES; ++t) {
      const c64 w = G[(3 + t) * esz + o];
      d.x -= lam * dlw[t] * w.x;
      d.y -= lam * dlw[t] * w.y;
    }
    if (a == b) d.y = 0;
    const c64 z = d * y[b];
    acc += (a == b ? 1.0 : 2.0) * (y[a].x * z.x + y[a].y * z.y);
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) red_s[wv] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double slope = 0;
    for (int w = 0; w < DT / 64; ++w) slope += red_s[w];
    // early Ritz values are far above the band's: the first steps move k by at most a tenth
    const double lim = (s.iter < 4 ? 0.1 : 0.25) * fabs(kk);
    double dk = -(lam - s.omega2) / slope;
    if (!isfinite(dk)) dk = 0;
    dk = fmin(fmax(dk, -lim), lim);
    s.keval[j] = kk;
    s.lam[j] = lam;
    s.slope[j] = slope;
    s.knew[j] = kk + dk;
  }
}

// ---------------------------------------------------------------------------------------
// Block update: X' = S Cx, P' = the W and P part of it, over the flat 7-plane columns.
// ---------------------------------------------------------------------------------------
template <int QM>
__global__ __launch_bounds__(256) void k_mk_combine(MkGeo geo, c32* cols, const MkState* st, const c32* Cx, int buf) {
  __shared__ const c32* in[MK_MAXN];
  __shared__ c32* outx[QM];
  __shared__ c32* outp[QM];
  __shared__ c32 Cs[MK_MAXN][QM];
  const int p = blockIdx.y;
  const MkState& s = st[p];
  if (s.done) return;
  const int m = s.m, n = m + s.na + s.np;
  c32* base = cols + p * geo.slots;
  // W and P first: their sum is P', then X's part completes X'
  for (int a = threadIdx.x; a < n; a += 256) {
    const int q = a < n - m ? a + m : a - (n - m);
    in[a] = base + col_off(geo, space_slot(geo, s, buf, q));
  }
  for (int e = threadIdx.x; e < n * QM; e += 256) {
    const int a = e / QM, j = e - a * QM, q = a < n - m ? a + m : a - (n - m);
    Cs[a][j] = j < m ? Cx[(long(p) * MK_MAXN + q) * MK_MAXM + j] : c32{0.f, 0.f};
  }
  if (threadIdx.x < QM) {
    const int j = threadIdx.x;
    outx[j] = j < m ? base + col_off(geo, slot_x(geo, buf ^ 1, j)) : nullptr;
    c32* q = nullptr;
    for (int w = 0; w < s.na; ++w)
      if (s.wcol[w] == j) q = base + col_off(geo, slot_p(geo, buf ^ 1, w));
    outp[j] = q;
  }
  __syncthreads();
  const int nwp = n - m;
  const long L = PLANES * geo.cs / 2;  // pairs of values
  for (long e = long(blockIdx.x) * 256 + threadIdx.x; e < L; e += long(gridDim.x) * 256) {
    c32 a0[QM], a1[QM];
#pragma unroll
    for (int j = 0; j < QM; ++j) a0[j] = a1[j] = c32{0.f, 0.f};
    auto add = [&](int from, int to) {
      int a = from;
      for (; a + 4 <= to; a += 4) {  // four columns' loads in flight together
        fx4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const fx4*>(in[a + u])[e];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < QM; ++j) {
            const c32 c = Cs[a + u][j];
            a0[j] = a0[j] + c32{v[u].x, v[u].y} * c;
            a1[j] = a1[j] + c32{v[u].z, v[u].w} * c;
          }
      }
      for (; a < to; ++a) {
        const fx4 v = reinterpret_cast<const fx4*>(in[a])[e];
#pragma unroll
        for (int j = 0; j < QM; ++j) {
          const c32 c = Cs[a][j];
          a0[j] = a0[j] + c32{v.x, v.y} * c;
          a1[j] = a1[j] + c32{v.z, v.w} * c;
        }
      }
    };
    add(0, nwp);
#pragma unroll
    for (int j = 0; j < QM; ++j)
      if (outp[j]) reinterpret_cast<fx4*>(outp[j])[e] = fx4{a0[j].x, a0[j].y, a1[j].x, a1[j].y};
    add(nwp, n);
#pragma unroll
    for (int j = 0; j < QM; ++j)
      if (outx[j]) reinterpret_cast<fx4*>(outx[j])[e] = fx4{a0[j].x, a0[j].y, a1[j].x, a1[j].y};
  }
}

// ---------------------------------------------------------------------------------------
// Transforms.  Column kernels hold TX columns (fixed ix, all iy) of each plane in LDS, row
// kernels RB rows; the intermediate field Dm is [problem column][plane][ix][iy].
// ---------------------------------------------------------------------------------------
// eps^-1 (F0 + k F1) of X (buffer buf), inverse FFT along y
template <int VPT>
__global__ __launch_bounds__(FT) void k_mk_colE(MkGeo geo, const c32* cols, const MkState* st, int buf, c32* Dm,
                                                int TX) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int p = blockIdx.y / geo.mmax, c = blockIdx.y - p * geo.mmax;
  const MkState& s = st[p];
  if (s.done || c >= s.m) return;
  const int ny = geo.ny;
  c32* tw = reinterpret_cast<c32*>(smem_raw);
  c32* sm = tw + ny;
  for (int t = threadIdx.x; t < ny; t += FT) tw[t] = geo.twy[t];
  const int ix0 = blockIdx.x * TX, tx = min(TX, geo.nx - ix0), nv = tx * ny;
  const float k = float(s.keval[c]);
  const c32* x = cols + p * geo.slots + col_off(geo, slot_x(geo, buf, c)) + long(ix0) * ny;
  const float* ep = geo.eps6c + p * geo.eps_stride + 6L * ix0 * ny;
  for (int e = threadIdx.x; e < TX * ny; e += FT) {
    c32 y0{0.f, 0.f}, y1 = y0, y2 = y0;
    if (e < nv) {
      const c32 d0 = x[e] + x[3 * geo.cs + e] * k, d1 = x[geo.cs + e] + x[4 * geo.cs + e] * k, d2 = x[2 * geo.cs + e];
      const float2* q = reinterpret_cast<const float2*>(ep + 6L * e);
      const float2 ea = q[0], eb = q[1], ec = q[2];  // xx yy, zz xy, xz yz
      y0 = d0 * ea.x + d1 * eb.y + d2 * ec.x;
      y1 = d0 * eb.y + d1 * ea.y + d2 * ec.y;
      y2 = d0 * ec.x + d1 * ec.y + d2 * eb.x;
    }
    sm[e] = y0;
    sm[TX * ny + e] = y1;
    sm[2 * TX * ny + e] = y2;
  }
  __syncthreads();
  fft_lds<float, +1, VPT>(sm, 3 * TX, ny, 1, geo.fy, tw);
  c32* d = Dm + long(blockIdx.y) * 3 * geo.cs + long(ix0) * ny;
  for (int e = threadIdx.x; e < nv; e += FT) {
    d[e] = sm[e];
    d[geo.cs + e] = sm[TX * ny + e];
    d[2 * geo.cs + e] = sm[2 * TX * ny + e];
  }
}

// rows of Dm into LDS, [plane][row][ix] with row stride nx + 1
__device__ __forceinline__ void rows_in(const MkGeo& geo, const c32* d, int iy0, int rb, int RB, int nplane, c32* sm) {
  const int nx = geo.nx, ny = geo.ny, sb = nx + 1;
  for (int e = threadIdx.x; e < nplane * RB * nx; e += FT) {
    const int q = e / RB, r = e - q * RB, a = q / nx, ix = q - a * nx;
    sm[(a * RB + r) * sb + ix] = r < rb ? d[a * geo.cs + long(ix) * ny + iy0 + r] : c32{0.f, 0.f};
  }
}
__device__ __forceinline__ void rows_out(const MkGeo& geo, c32* d, int iy0, int rb, int RB, int nplane, const c32* sm) {
  const int nx = geo.nx, ny = geo.ny, sb = nx + 1;
  for (int e = threadIdx.x; e < nplane * RB * nx; e += FT) {
    const int q = e / RB, r = e - q * RB, a = q / nx, ix = q - a * nx;
    if (r < rb) d[a * geo.cs + long(ix) * ny + iy0 + r] = sm[(a * RB + r) * sb + ix];
  }
}

// inverse FFT along x, M x, residual and its norm, the preconditioner's map, FFT along x
template <int VPT>
__global__ __launch_bounds__(FT) void k_mk_rowR(MkGeo geo, const c32* cols, const MkState* st, int buf, c32* Dm,
                                                int RB, double* normp) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int p = blockIdx.y / geo.mmax, c = blockIdx.y - p * geo.mmax;
  const MkState& s = st[p];
  if (s.done || c >= s.m) return;
  const int nx = geo.nx, sb = nx + 1;
  c32* tw = reinterpret_cast<c32*>(smem_raw);
  c32* sm = tw + nx;
  for (int t = threadIdx.x; t < nx; t += FT) tw[t] = geo.twx[t];
  const int iy0 = blockIdx.x * RB, rb = min(RB, geo.ny - iy0);
  c32* d = Dm + long(blockIdx.y) * 3 * geo.cs;
  rows_in(geo, d, iy0, rb, RB, 3, sm);
  __syncthreads();
  fft_lds<float, +1, VPT>(sm, 3 * RB, sb, 1, geo.fx, tw);
  const c32* g1 = cols + p * geo.slots + col_off(geo, slot_x(geo, buf, c)) + 5 * geo.cs + long(iy0) * nx;
  const float k = float(s.keval[c]), lam = float(s.lam[c]), scale = 1.f / float(geo.N);
  double acc = 0;
  for (int e = threadIdx.x; e < rb * nx; e += FT) {
    const int r = e / nx, ix = e - r * nx;
    const Wave w = wave_at(ix, iy0 + r, geo);
    const float mag2 = w.rho2 + k * k, mag = sqrtf(mag2), im = 1.f / mag;
    c32 *s0 = sm + r * sb + ix, *s1 = s0 + RB * sb, *s2 = s1 + RB * sb;
    const c32 e0 = *s0, e1 = *s1, e2 = *s2, x1 = g1[e], x2 = g1[geo.cs + e];
    const c32 en = e0 * w.n0 + e1 * w.n1, em = (e0 * w.n1 - e1 * w.n0) * k - e2 * w.rho;
    const c32 r1 = en * (-mag * scale) - x1 * (lam * im), r2 = em * scale - x2 * lam;
    acc += double(r1.x) * r1.x + double(r1.y) * r1.y + double(r2.x) * r2.x + double(r2.y) * r2.y;
    const c32 t = r2 * (k * im);
    *s0 = (r1 * w.n0 - t * w.n1) * im;
    *s1 = (r1 * w.n1 + t * w.n0) * im;
    *s2 = r2 * (w.rho * im * im);
  }
  __syncthreads();
  fft_lds<float, +1, VPT>(sm, 3 * RB, sb, 1, geo.fx, tw);
  rows_out(geo, d, iy0, rb, RB, 3, sm);
  __shared__ double red[FT / 64];
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0;
    for (int q = 0; q < FT / 64; ++q) t += red[q];
    normp[long(blockIdx.y) * gridDim.x + blockIdx.x] = t;
  }
}

// A problem's next state from its residual norms (one thread): thresholds, k, the columns that go
// on; ext: the extent of |k| over the columns
__device__ void control_step(MkState& s, const double* nr, int cur, double* ext) {
  bool all = true, bad = false, moved = false;
  int nconv = 0;
  double worst = 0;
  int act[MK_MAXM];
  for (int c = 0; c < s.m; ++c) {
    // w^2's distance at the column's own k (bands of a cluster are taken at a shared one)
    const double rn = nr[c], f = fabs(s.lam[c] + s.slope[c] * (s.k[c] - s.keval[c]) - s.omega2);
    bad = bad || !isfinite(rn) || !isfinite(s.lam[c]);
    act[c] = rn > s.tol;
    // by the distance itself, not the step made of it: a band that does not propagate at
    // omega shrinks its k, and with it the limited step times the slope, at any distance
    const bool still = f <= s.ftol, conv = !act[c] && still;
    if (c < s.nev) {
      moved = moved || !still;
      if (conv && !s.its[c]) s.its[c] = s.iter + 1;
      if (!conv) s.its[c] = 0;
      all = all && conv;
      nconv += conv;
      worst = fmax(worst, fmax(rn / s.tol, f / s.ftol));
    }
    s.rnorm[c] = rn;
    s.kold[c] = s.k[c];
    s.k[c] = s.knew[c];
  }
  bool wide = false;
  {  // the guard columns' k no further than a fifth below the bands' range
    double lo, hi;
    mk_extent(s.k, s.nev, lo, hi);
    wide = hi > MK_WIDEST * lo;
    for (int c = s.nev; c < s.m; ++c) s.k[c] = fmin(fmax(s.k[c], 0.8 * lo), hi);
    mk_extent(s.k, s.m, ext[0], ext[1]);
  }
  s.iter += 1;
  s.moves += moved;
  s.par = cur;
  if (bad) {
    s.done = 2;
    return;
  }
  if (all) {  // the current space and its coefficients are the result
    // bands close enough to have shared a k (k_mk_dense) are handed over at one k too: their
    // vectors are orthogonal there
    for (int a = 0; a < s.nev;) {
      int b = a;
      double sum = s.k[a];
      while (b + 1 < s.nev && fabs(s.k[b + 1] - s.k[b]) < MK_CLUSTER * fabs(s.k[b])) sum += s.k[++b];
      for (int i = a; i <= b; ++i) s.knew[i] = sum / (b - a + 1);
      a = b + 1;
    }
    for (int i = 0; i < s.nev; ++i) s.k[i] = s.knew[i];
    s.done = 1;
    return;
  }
  if (nconv > s.ahead || worst < 0.9 * s.worst) {
    s.ahead = max(s.ahead, nconv);
    s.worst = fmin(s.worst, worst);
    s.idle = 0;
  } else {
    s.idle += 1;
  }
  if (wide || s.idle >= MK_IDLE) {
    s.done = 3;
    return;
  }
  int np = 0;
  for (int w = 0; w < s.na; ++w)
    if (act[s.wcol[w]]) s.pslot[np++] = w;
  s.np = np;
  int na = 0;
  for (int c = 0; c < s.m; ++c)
    if (act[c]) s.wcol[na++] = c;
  s.na = na;
}

// Residual norms, convergence, the next search space.  One block per problem; the state is worked
// on in LDS (its fields are a serial chain for one thread: 9.6 us in global memory, 8.1 here).
__global__ __launch_bounds__(256) void k_mk_control(MkGeo geo, MkState* st, const double* normp, int nrb, int cur) {
  static_assert(sizeof(MkState) % sizeof(int) == 0, "copied by words");
  constexpr int WORDS = sizeof(MkState) / sizeof(int);
  const int p = blockIdx.x;
  __shared__ MkState s;
  __shared__ double nr[MK_MAXM], ext[2];
  int* const sw = reinterpret_cast<int*>(&s);
  int* const gw = reinterpret_cast<int*>(st + p);
  for (int w = threadIdx.x; w < WORDS; w += 256) sw[w] = gw[w];
  __syncthreads();
  if (s.done) return;
  const int lane = threadIdx.x & 63;
  for (int c = threadIdx.x >> 6; c < s.m; c += 4) {
    double a = 0;
    for (int b = lane; b < nrb; b += 64) a += normp[(long(p) * geo.mmax + c) * nrb + b];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (lane == 0) nr[c] = sqrt(a);
  }
  __syncthreads();
  if (threadIdx.x == 0) control_step(s, nr, cur, ext);
  __syncthreads();
  // the next iteration's nodes; those of the last one made stay for the handover
  if (!s.done && threadIdx.x < MK_NODES) set_node(s, mk_range(ext[0], ext[1]), threadIdx.x);
  __syncthreads();
  for (int w = threadIdx.x; w < WORDS; w += 256) gw[w] = sw[w];
}

// FFT along y, eps_ave, FFT back, for the columns that go on
template <int VPT>
__global__ __launch_bounds__(FT) void k_mk_colP(MkGeo geo, const MkState* st, c32* Dm, int TX) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int p = blockIdx.y / geo.mmax, w = blockIdx.y - p * geo.mmax;
  const MkState& s = st[p];
  if (s.done || w >= s.na) return;
  const int ny = geo.ny;
  c32* tw = reinterpret_cast<c32*>(smem_raw);
  c32* sm = tw + ny;
  for (int t = threadIdx.x; t < ny; t += FT) tw[t] = geo.twy[t];
  const int ix0 = blockIdx.x * TX, tx = min(TX, geo.nx - ix0), nv = tx * ny;
  c32* d = Dm + (long(p) * geo.mmax + s.wcol[w]) * 3 * geo.cs + long(ix0) * ny;
  for (int e = threadIdx.x; e < TX * ny; e += FT)
#pragma unroll
    for (int a = 0; a < 3; ++a) sm[a * TX * ny + e] = e < nv ? d[a * geo.cs + e] : c32{0.f, 0.f};
  __syncthreads();
  fft_lds<float, +1, VPT>(sm, 3 * TX, ny, 1, geo.fy, tw);
  const float* ep = geo.eps6c + p * geo.eps_stride + 6L * ix0 * ny;
  for (int e = threadIdx.x; e < nv; e += FT) {
    const float ea = 3.f / (ep[6L * e] + ep[6L * e + 1] + ep[6L * e + 2]);
#pragma unroll
    for (int a = 0; a < 3; ++a) sm[a * TX * ny + e] = sm[a * TX * ny + e] * ea;
  }
  __syncthreads();
  fft_lds<float, -1, VPT>(sm, 3 * TX, ny, 1, geo.fy, tw);
  for (int e = threadIdx.x; e < nv; e += FT)
#pragma unroll
    for (int a = 0; a < 3; ++a) d[a * geo.cs + e] = sm[a * TX * ny + e];
}

// START false: FFT along x, w = P r, its g into W.  START true: g of X (buffer 0) as it is.
// Then D0 and D1 of g, FFT along x (three planes, then two).
template <int VPT, bool START>
__global__ __launch_bounds__(FT) void k_mk_rowW(MkGeo geo, c32* cols, const MkState* st, const c32* Dm, int RB) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int p = blockIdx.y / geo.mmax, w = blockIdx.y - p * geo.mmax;
  const MkState& s = st[p];
  if (s.done || w >= (START ? s.m : s.na)) return;
  const int nx = geo.nx, sb = nx + 1, c = START ? w : s.wcol[w];
  c32* tw = reinterpret_cast<c32*>(smem_raw);
  c32* sm = tw + nx;
  for (int t = threadIdx.x; t < nx; t += FT) tw[t] = geo.twx[t];
  const int iy0 = blockIdx.x * RB, rb = min(RB, geo.ny - iy0);
  c32* out = cols + p * geo.slots + col_off(geo, START ? slot_x(geo, 0, w) : slot_w(geo, w));
  c32* g1 = out + 5 * geo.cs + long(iy0) * nx;
  if (!START) {
    rows_in(geo, Dm + (long(p) * geo.mmax + c) * 3 * geo.cs, iy0, rb, RB, 3, sm);
    __syncthreads();
    fft_lds<float, -1, VPT>(sm, 3 * RB, sb, 1, geo.fx, tw);
  } else {
    __syncthreads();
  }
  const float k = START ? 0.f : float(s.keval[c]), scale = 1.f / float(geo.N);
  for (int e = threadIdx.x; e < RB * nx; e += FT) {
    const int r = e / nx, ix = e - r * nx;
    c32 *s0 = sm + r * sb + ix, *s1 = s0 + RB * sb, *s2 = s1 + RB * sb;
    c32 a1{0.f, 0.f}, a2{0.f, 0.f};
    Wave v{0.f, 0.f, 0.f, 0.f};
    if (r < rb) {
      v = wave_at(ix, iy0 + r, geo);
      if (START) {
        a1 = g1[e];
        a2 = g1[geo.cs + e];
      } else {
        const c32 e0 = *s0, e1 = *s1, e2 = *s2;
        a1 = (e0 * v.n0 + e1 * v.n1) * scale;
        a2 = ((e0 * v.n1 - e1 * v.n0) * k - e2 * v.rho) * (-scale / (v.rho2 + k * k));
        g1[e] = a1;
        g1[geo.cs + e] = a2;
      }
    }
    *s0 = a1 * -v.n0;
    *s1 = a1 * -v.n1;
    *s2 = a2 * -v.rho;
  }
  __syncthreads();
  fft_lds<float, -1, VPT>(sm, 3 * RB, sb, 1, geo.fx, tw);
  rows_out(geo, out, iy0, rb, RB, 3, sm);
  __syncthreads();
  for (int e = threadIdx.x; e < RB * nx; e += FT) {  // this thread's own g2 of the loop above
    const int r = e / nx, ix = e - r * nx;
    c32 *s0 = sm + r * sb + ix, *s1 = s0 + RB * sb;
    c32 a2{0.f, 0.f};
    Wave v{0.f, 0.f, 0.f, 0.f};
    if (r < rb) {
      v = wave_at(ix, iy0 + r, geo);
      a2 = g1[geo.cs + e];
    }
    *s0 = a2 * v.n1;
    *s1 = a2 * -v.n0;
  }
  __syncthreads();
  fft_lds<float, -1, VPT>(sm, 2 * RB, sb, 1, geo.fx, tw);
  rows_out(geo, out + 3 * geo.cs, iy0, rb, RB, 2, sm);
}

// FFT along y of the five planes of W (START: of X, buffer 0); blockIdx.z: planes 0-2 or 3-4
template <int VPT, bool START>
__global__ __launch_bounds__(FT) void k_mk_colF(MkGeo geo, c32* cols, const MkState* st, int TX) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int p = blockIdx.y / geo.mmax, w = blockIdx.y - p * geo.mmax;
  const MkState& s = st[p];
  if (s.done || w >= (START ? s.m : s.na)) return;
  const int ny = geo.ny, a0 = blockIdx.z ? 3 : 0, na = blockIdx.z ? 2 : 3;
  c32* tw = reinterpret_cast<c32*>(smem_raw);
  c32* sm = tw + ny;
  for (int t = threadIdx.x; t < ny; t += FT) tw[t] = geo.twy[t];
  const int ix0 = blockIdx.x * TX, tx = min(TX, geo.nx - ix0), nv = tx * ny;
  c32* d = cols + p * geo.slots + col_off(geo, START ? slot_x(geo, 0, w) : slot_w(geo, w)) + a0 * geo.cs +
           long(ix0) * ny;
  for (int e = threadIdx.x; e < TX * ny; e += FT)
    for (int a = 0; a < na; ++a) sm[a * TX * ny + e] = e < nv ? d[a * geo.cs + e] : c32{0.f, 0.f};
  __syncthreads();
  fft_lds<float, -1, VPT>(sm, na * TX, ny, 1, geo.fy, tw);
  for (int e = threadIdx.x; e < nv; e += FT)
    for (int a = 0; a < na; ++a) d[a * geo.cs + e] = sm[a * TX * ny + e];
}

// Each band's block for the FP64 refinement: its lowest Ritz vectors at its k as transverse
// coefficients (h1 = g1 / |w|, h2 = g2), sums in FP64.  The space's G planes are read once per
// instance; blockIdx.z: groups of HQ vectors.
constexpr int HQ = 4;
__global__ __launch_bounds__(256) void k_mk_handover(MkGeo geo, const c32* cols, const MkState* st, const int2* inst,
                                                     const int* msz, const c64* Cblk, c64* X64, long ld, long istride) {
  __shared__ const c32* in[MK_MAXN];
  __shared__ c64 Cs[MK_MAXN][HQ];
  const int i = blockIdx.y, p = inst[i].x, j = inst[i].y, q0 = blockIdx.z * HQ;
  const MkState& s = st[p];
  if (s.done != 1) return;
  const int nq = min(HQ, msz[p * MK_MAXM + j] - q0);
  if (nq <= 0) return;
  const int n = s.m + s.na + s.np;
  const c64* Cb = Cblk + (long(p) * geo.mmax + j) * MK_MAXN * MK_MAXM;
  for (int a = threadIdx.x; a < n; a += 256)
    in[a] = cols + p * geo.slots + col_off(geo, space_slot(geo, s, s.par, a)) + 5 * geo.cs;
  for (int e = threadIdx.x; e < n * HQ; e += 256) {
    const int a = e / HQ, q = e - a * HQ;
    Cs[a][q] = q < nq ? Cb[a * MK_MAXM + q0 + q] : c64{0.0, 0.0};
  }
  __syncthreads();
  const double k = s.k[j];
  for (long e = long(blockIdx.x) * 256 + threadIdx.x; e < geo.N; e += long(gridDim.x) * 256) {
    const int iy = int(e / geo.nx), ix = int(e - long(iy) * geo.nx);
    const double wx = double(fft_index(ix, geo.nx)) * geo.invdx, wy = double(fft_index(iy, geo.ny)) * geo.invdy;
    const double im = 1.0 / sqrt(wx * wx + wy * wy + k * k);
    c64 a1[HQ], a2[HQ];
#pragma unroll
    for (int q = 0; q < HQ; ++q) a1[q] = a2[q] = c64{0.0, 0.0};
    for (int a = 0; a < n; ++a) {
      const c32 f1 = in[a][e], f2 = in[a][geo.cs + e];
      const c64 v1{f1.x, f1.y}, v2{f2.x, f2.y};
#pragma unroll
      for (int q = 0; q < HQ; ++q) {
        a1[q] = a1[q] + v1 * Cs[a][q];
        a2[q] = a2[q] + v2 * Cs[a][q];
      }
    }
#pragma unroll
    for (int q = 0; q < HQ; ++q)
      if (q < nq) {
        c64* o = X64 + i * istride + long(q0 + q) * ld + 2 * e;
        o[0] = a1[q] * im;
        o[1] = a2[q];
      }
  }
}

// every radix pass of nb sequences fits FT threads of vpt values
bool fits(int nb, const FFTFactors& f, int vpt) {
  for (int p = 0; p < f.n; ++p) {
    const int R = f.r[p];
    if ((long(nb) * (f.L / R) + FT - 1) / FT > (vpt + R - 1) / R) return false;
  }
  return true;
}

constexpr size_t MK_LDS = 64 * 1024;

// sequences of length L per block for three planes: at most 16, within MK_LDS and the bound of
// 16 values per thread; fewer while the launch would leave CUs idle.  The line at 512 blocks, two
// per CU: at 256^2 with 10 columns an iteration's transforms take 149 us with 4 sequences a
// block and 172 us with 8 (a line at 256); a line at 1024 changes nothing from 128^2 to 512 x 256.
int pick_rows(int L, int other, long vecs, const FFTFactors& f) {
  int r = 16;
  while (r > 1 && (sizeof(c32) * (L + 3 * size_t(r) * (L + 1)) > MK_LDS || !fits(3 * r, f, 16))) r /= 2;
  if (sizeof(c32) * (L + 3 * size_t(r) * (L + 1)) > 160 * 1024 || !fits(3 * r, f, 16)) return 0;
  while (r > 4 && long((other + r - 1) / r) * vecs < 512) r /= 2;
  return r;
}

}  // namespace

bool multik_fits(const Solver& S) {
  return S.nz == 1 && pick_rows(S.nx, S.ny, 1 << 20, S.p32.plan.fx) > 0 &&
         pick_rows(S.ny, S.nx, 1 << 20, S.p32.plan.fy) > 0;
}

std::vector<char> multik_solve(Solver& S, const std::vector<MkProblem>& probs, const float* eps6c, long eps_stride,
                               int maxit, const std::vector<int>& msize, c64* X64, long ld, long istride,
                               std::vector<double>& kout, std::vector<int>& iters, std::vector<int>& moves,
                               SolveStats& stats) {
  const int P = int(probs.size());
  std::vector<char> ok(P, 0);
  hipStream_t sm = S.stream;
  MkGeo g{};
  g.nx = S.nx;
  g.ny = S.ny;
  g.N = S.N;
  g.invdx = 1.0 / S.Dx;
  g.invdy = 1.0 / S.Dy;
  g.fx = S.p32.plan.fx;
  g.fy = S.p32.plan.fy;
  g.twx = S.p32.plan.twx;
  g.twy = S.p32.plan.twy;
  g.eps6c = eps6c;
  g.eps_stride = eps_stride;
  g.mmax = 1;
  int ninst = 0;
  const int most = int(std::min<long>(MK_MAXM, S.K / 3));
  std::vector<MkState> hs(P);
  for (int p = 0; p < P; ++p) {
    const MkProblem& q = probs[p];
    MkState& s = hs[p];
    std::memset(&s, 0, sizeof(s));
    s.nev = q.nev;
    s.m = std::max(q.nev, std::min(q.nev + MK_GUARD, most));
    s.omega2 = q.omega * q.omega;
    s.tol = q.tol;
    s.ftol = q.ftol;
    s.worst = 1e300;
    for (int j = 0; j < s.m; ++j) s.k[j] = s.knew[j] = s.keval[j] = q.k[std::min<size_t>(j, q.k.size() - 1)];
    double lo, hi;
    mk_extent(s.k, s.m, lo, hi);
    for (int t = 0; t < MK_NODES; ++t) set_node(s, mk_range(lo, hi), t);
    g.mmax = std::max(g.mmax, s.m);
    ninst += q.nev;
  }
  const MkSizes z = multik_sizes(S.N, P, g.mmax);
  g.cs = z.cs;
  g.slots = z.slots;
  const int nmax = 3 * g.mmax, NT = z.NT, pm = z.pm, nch = z.nch;
  const long vecs = z.vecs, rpc = z.rpc, rotn = z.rotn;
  const int RB = pick_rows(S.nx, S.ny, vecs, g.fx), TX = pick_rows(S.ny, S.nx, vecs, g.fy);
  if (RB == 0 || TX == 0) return ok;
  const int nrb = (S.ny + RB - 1) / RB, ncb = (S.nx + TX - 1) / TX;
  // the widest space's three matrices and the kernel's own arrays share a CU's 160 KB
  {
    hipFuncAttributes fa{}, fb{};
    OMX_HIP_CHECK(hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(&k_mk_dense<512, false>)));
    OMX_HIP_CHECK(hipFuncGetAttributes(&fb, reinterpret_cast<const void*>(&k_mk_dense<512, true>)));
    const size_t dyn = sizeof(c64) * 3 * size_t((nmax + 1) & ~1) * ((nmax + 1) | 1);
    if (std::max(fa.sharedSizeBytes, fb.sharedSizeBytes) + dyn > 160 * 1024) return ok;
  }
  MultiKWorkspace& W = S.multik_ws;
  // The pads past N of every plane are read as zeros.  The block update runs over them, so
  // coefficients that are not finite leave NaN there: they count as clear only after a call that
  // ended without.
  const long geom = g.cs * 64 + g.mmax;
  if (W.cols.size() < z.cols || W.geom != geom) {
    W.cols.ensure(z.cols);
    OMX_HIP_CHECK(hipMemsetAsync(W.cols.as<void>(), 0, W.cols.size(), sm));
  }
  W.geom = 0;
  W.dm.ensure(z.dm);
  W.part.ensure(z.part);
  W.red.ensure(z.red);
  W.cx.ensure(sizeof(c32) * size_t(P) * MK_MAXN * MK_MAXM);
  W.cblk.ensure(z.cblk);
  static_assert(sizeof(MkRot) == 32 && NGRAM == 3 + MK_NODES + 1, "multik_sizes");
  W.rot.ensure(z.rot);
  W.normp.ensure(sizeof(double) * size_t(vecs) * nrb);
  W.state.ensure(sizeof(MkState) * P);
  W.ints.ensure(sizeof(int) * size_t(P) * MK_MAXM + sizeof(int2) * ninst);
  if (W.snap_bytes < sizeof(MkState) * P) {
    for (int b = 0; b < 2; ++b) W.snap[b].alloc(sizeof(MkState) * P);
    W.snap_bytes = sizeof(MkState) * P;
  }
  for (int b = 0; b < 2; ++b)
    if (!W.ev[b]) OMX_HIP_CHECK(hipEventCreateWithFlags(&W.ev[b], hipEventDisableTiming));
  c32* cols = W.cols.as<c32>();
  c32* dm = W.dm.as<c32>();
  c32* part = W.part.as<c32>();
  c64* red = W.red.as<c64>();
  c32* cx = W.cx.as<c32>();
  c64* cblk = W.cblk.as<c64>();
  double* normp = W.normp.as<double>();
  MkState* st = W.state.as<MkState>();
  int2* instd = W.ints.as<int2>();
  int* mszd = reinterpret_cast<int*>(instd + ninst);
  std::vector<int> hmsz(size_t(P) * MK_MAXM, 0);
  std::vector<int2> hinst;
  for (int p = 0; p < P; ++p)
    for (int j = 0; j < probs[p].nev; ++j) {
      hmsz[size_t(p) * MK_MAXM + j] = msize[hinst.size()];
      hinst.push_back(int2{p, j});
    }
  OMX_HIP_CHECK(hipMemcpyAsync(st, hs.data(), sizeof(MkState) * P, hipMemcpyHostToDevice, sm));
  OMX_HIP_CHECK(hipMemcpyAsync(instd, hinst.data(), sizeof(int2) * ninst, hipMemcpyHostToDevice, sm));
  OMX_HIP_CHECK(hipMemcpyAsync(mszd, hmsz.data(), sizeof(int) * hmsz.size(), hipMemcpyHostToDevice, sm));
  const size_t ldsr = sizeof(c32) * (S.nx + 3 * size_t(RB) * (S.nx + 1));
  const size_t ldsc = sizeof(c32) * (S.ny + 3 * size_t(TX) * S.ny);
  const dim3 gr(nrb, unsigned(vecs)), gc(ncb, unsigned(vecs)), gc2(ncb, unsigned(vecs), 2);
  const int vpt = fits(3 * RB, g.fx, 8) && fits(3 * TX, g.fy, 8) ? 8 : 16;
  for (int p = 0; p < P; ++p)
    hipLaunchKernelGGL(k_mk_start, dim3(unsigned(std::min<long>((S.N + 255) / 256, 256)), hs[p].m), dim3(256), 0, sm, g,
                       cols, st, p, probs[p].src, probs[p].lds, probs[p].src ? probs[p].nsrc : 0, probs[p].lowres,
                       S.opt.seed);
  auto transforms = [&](auto V, auto START) {
    constexpr int v = decltype(V)::value;
    constexpr bool start = decltype(START)::value;
    hipLaunchKernelGGL((k_mk_rowW<v, start>), gr, dim3(FT), ldsr, sm, g, cols, st, dm, RB);
    hipLaunchKernelGGL((k_mk_colF<v, start>), gc2, dim3(FT), ldsc, sm, g, cols, st, TX);
  };
  using v8 = std::integral_constant<int, 8>;
  using v16 = std::integral_constant<int, 16>;
  if (vpt == 8)
    transforms(v8{}, std::true_type{});
  else
    transforms(v16{}, std::true_type{});
  // Rows per stage and lane, and norm matrices per block, by column tiles (us a launch, rows 2 /
  // 4 at the chosen matrices, then matrices 1 / 2 / 3 at the chosen rows): 18 columns at 128^2
  // 34.4 / 32.2, 32.5 / 28.6 / 32.2; 30 at 256^2 109 / 103, 106 / 95 / 103; 42 at 384^2 383 / 356,
  // 424 / 383 / 783; 54 at 512 x 256 591 / 753, 591 / 961 / 2459.  Above two tiles more of either
  // spills the accumulators; at two tiles 2 matrices and at three 4 rows are up to 8% faster than
  // what is launched.
  auto gram = [&](auto T, int buf) {
    constexpr int nt = decltype(T)::value;
    constexpr int S_ = nt <= 2 ? 4 : 2, NB = nt <= 2 ? 3 : (nt == 3 ? 2 : 1);
    hipLaunchKernelGGL((k_mk_gram<nt, NB, S_>), dim3(nch, P, 3 + (MK_NODES + NB) / NB), dim3(64 * GW), 0, sm, g, cols,
                       st, buf, rpc, part);
  };
  const int ldd = (nmax + 1) | 1;
  const size_t ldsd = sizeof(c64) * 3 * size_t((nmax + 1) & ~1) * ldd;
  auto dense = [&](auto F) {
    hipLaunchKernelGGL((k_mk_dense<512, decltype(F)::value>), dim3(g.mmax, P), dim3(512), ldsd, sm, g, st, red, pm, ldd,
                       S.opt.jac_stop32, mszd, cx, cblk, W.rot.as<MkRot>(), rotn);
  };
  const dim3 gcomb(unsigned(std::min<long>((PLANES * g.cs / 2 + 255) / 256, std::max(1, 2048 / P))), P);
  const bool prof = S.prof.enabled;
  // operator intervals (omx_get_kernel_stats): M x of every column of the problems that still
  // ran, P r of those that went on; counted once the iteration's state is known
  hipEvent_t mark[2][2] = {};
  auto count = [&](int at, const MkState* h) {
    double b = 0;
    for (int p = 0; p < P; ++p)
      if (h[p].iter == at + 1)
        b += 32.0 * S.N * h[p].m + 24.0 * S.N + (h[p].done ? 0.0 : 32.0 * S.N * h[p].na + 24.0 * S.N);
    if (b > 0)
      S.prof.commit(mark[at & 1][0], mark[at & 1][1], &S.prof.op32, b);
    else
      S.prof.recycle(mark[at & 1][0], mark[at & 1][1]);
  };
  int cur = 0, it = 0;
  bool fin = false;
  for (; it < maxit && !fin; ++it) {
    switch (NT) {
      case 1: gram(std::integral_constant<int, 1>{}, cur); break;
      case 2: gram(std::integral_constant<int, 2>{}, cur); break;
      case 3: gram(std::integral_constant<int, 3>{}, cur); break;
      default: gram(std::integral_constant<int, 4>{}, cur); break;
    }
    hipLaunchKernelGGL(k_mk_reduce, dim3(pm * pm / 16, NGRAM, P), dim3(256), 0, sm, part, nch, pm, st, red);
    dense(std::false_type{});
    if (g.mmax <= 4)
      hipLaunchKernelGGL((k_mk_combine<4>), gcomb, dim3(256), 0, sm, g, cols, st, cx, cur);
    else if (g.mmax <= 8)
      hipLaunchKernelGGL((k_mk_combine<8>), gcomb, dim3(256), 0, sm, g, cols, st, cx, cur);
    else if (g.mmax <= 12)
      hipLaunchKernelGGL((k_mk_combine<12>), gcomb, dim3(256), 0, sm, g, cols, st, cx, cur);
    else
      hipLaunchKernelGGL((k_mk_combine<MK_MAXM>), gcomb, dim3(256), 0, sm, g, cols, st, cx, cur);
    const hipEvent_t ea = prof ? S.prof.begin(sm) : nullptr;
    auto chain = [&](auto V) {
      constexpr int v = decltype(V)::value;
      hipLaunchKernelGGL((k_mk_colE<v>), gc, dim3(FT), ldsc, sm, g, cols, st, cur ^ 1, dm, TX);
      hipLaunchKernelGGL((k_mk_rowR<v>), gr, dim3(FT), ldsr, sm, g, cols, st, cur ^ 1, dm, RB, normp);
      hipLaunchKernelGGL(k_mk_control, dim3(P), dim3(256), 0, sm, g, st, normp, nrb, cur);
      hipLaunchKernelGGL((k_mk_colP<v>), gc, dim3(FT), ldsc, sm, g, st, dm, TX);
      transforms(V, std::false_type{});
    };
    if (vpt == 8)
      chain(v8{});
    else
      chain(v16{});
    OMX_HIP_CHECK(hipGetLastError());
    if (prof) {
      mark[it & 1][0] = ea;
      mark[it & 1][1] = S.prof.begin(sm);
    }
    OMX_HIP_CHECK(hipMemcpyAsync(W.snap[it & 1].as<void>(), st, sizeof(MkState) * P, hipMemcpyDeviceToHost, sm));
    OMX_HIP_CHECK(hipEventRecord(W.ev[it & 1], sm));
    cur ^= 1;
    if (it == 0) continue;
    // the state after the iteration before (an iteration enqueued after the end does nothing)
    OMX_HIP_CHECK(hipEventSynchronize(W.ev[(it - 1) & 1]));
    const MkState* h = W.snap[(it - 1) & 1].as<MkState>();
    if (prof) count(it - 1, h);
    fin = true;
    for (int p = 0; p < P; ++p) fin = fin && h[p].done;
    if (S.trace) {
      std::fprintf(stderr, "[omx] multik it %d:", it - 1);
      for (int p = 0; p < P; ++p) {
        double rm = 0;
        for (int j = 0; j < h[p].nev; ++j) rm = std::max(rm, h[p].rnorm[j]);
        std::fprintf(stderr, " [na %d np %d res %.1e k1 %.6f%s]", h[p].na, h[p].np, rm / h[p].omega2, h[p].k[0],
                     h[p].done == 1 ? " done" : (h[p].done ? " FAILED" : ""));
      }
      std::fprintf(stderr, "\n");
    }
  }
  OMX_HIP_CHECK(hipStreamSynchronize(sm));
  OMX_HIP_CHECK(hipMemcpy(hs.data(), st, sizeof(MkState) * P, hipMemcpyDeviceToHost));
  if (prof && it > 0) count(it - 1, hs.data());
  bool finite = true;
  for (int p = 0; p < P; ++p) {
    ok[p] = hs[p].done == 1;
    finite = finite && hs[p].done != 2;
  }
  if (finite) W.geom = geom;
  if (std::count(ok.begin(), ok.end(), 1) == 0) return ok;
  kout.clear();
  iters.clear();
  moves.clear();
  for (const MkState& h : hs) moves.push_back(h.moves);
  int mmax = 1;
  for (int p = 0, i = 0; p < P; ++p)
    for (int j = 0; j < probs[p].nev; ++j, ++i) {
      kout.push_back(hs[p].k[j]);
      iters.push_back(ok[p] ? hs[p].its[j] : 0);
      mmax = std::max(mmax, msize[i]);
      stats.matvec += iters.back();
      stats.precon += iters.back();
    }
  dense(std::true_type{});
  hipLaunchKernelGGL(k_mk_handover, dim3(unsigned(std::min<long>((S.N + 255) / 256, 512)), ninst, (mmax + HQ - 1) / HQ),
                     dim3(256), 0, sm, g, cols, st, instd, mszd, cblk, X64, ld, istride);
  OMX_HIP_CHECK(hipGetLastError());
  return ok;
}

}  // namespace omx
