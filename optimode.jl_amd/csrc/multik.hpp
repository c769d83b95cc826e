// Shared-subspace eigensolve of all bands at once (FP32 phase of solve_k on 2D cells).
//
// Every band j needs its own eigenpair: the j-th of M(k_j), at the k_j where it equals w^2.
// Instead of one LOBPCG block per band, all bands iterate in ONE search space
// S = [X W P] (m = nev + guard columns each), because the operator is quadratic in k once the
// transverse coefficients are scaled: with g = (|w| h_n-component, h_m-component),
// w = (0, 0, k) - G, rho = |(wx, wy)|,
//   D(k) = kx_tc(h) = D0 + k D1,  D0 = (-g1 n0, -g1 n1, -rho g2),  D1 = (g2 n1, -g2 n0, 0)
//   <h, M(k) h> = <F0 + k F1, eps^-1 (F0 + k F1)>,  F0 = fft(D0), F1 = fft(D1)
//   <h, h>      = sum |g1|^2 / (rho^2 + k^2) + |g2|^2
// so three Gram matrices of the transformed columns give S^H M(k) S for every k, and the
// norm's Gram matrix is interpolated in ln k from MK_NODES Chebyshev nodes over the columns' k
// range (multik_math.hpp, with the error by the range's width).  Per iteration each band
// solves its small pencil at its own k_j on its own workgroup, moves k_j by a Newton step of its
// Ritz value, and contributes one residual, one preconditioned direction W and one previous
// direction P.  The guard columns are there for the bands below them: their k stays at most a
// fifth below the bands' range (left to themselves, those that do not propagate at omega shrink
// their k without end and widen the interpolation's range with it: ten bands with such guards
// took 82 ms on 40 x 45, by way of the per-band form, and take 7).
#pragma once
#include <algorithm>
#include <vector>

#include "multik_math.hpp"
#include "omx_common.hpp"

namespace omx {

class Solver;
struct NewtonState;
struct SolveStats;

struct MkProblem {
  double omega = 0;
  int nev = 0;
  double tol = 0;                // residual a band stops at (absolute)
  double ftol = 0;               // |change of w^2| a band's k stops at
  std::vector<double> k;         // start k per band (size nev), or one value for all
  // start vectors (FP64, device): nsrc vectors with stride lds, entry c + 2 (ix + nx iy), or
  // with lowres = hw > 0 their hw x hw lowest plane waves; null: random
  const c64* src = nullptr;
  long lds = 0;
  int nsrc = 0;
  int lowres = 0;
};

// Runs the FP32 phase for the problems (all on S's grid; problem p reads the eps^-1 field
// eps6c + p * eps_stride).  Returns per problem whether all its bands converged within maxit
// iterations; the others are given up without holding those back.  Writes each band's block of
// FP64 Ritz vectors at its k for the problems that did: band j of problem p is instance
// i = off + j (off: bands of the problems before), columns 0 .. msize[i]-1 at X64 + i istride +
// c ld; kout[i] its k.  Iterations per band into iters, per problem those that moved a band's k
// into moves.  (Of a problem given up: nothing at X64, kout its last k, iters 0.)
std::vector<char> multik_solve(Solver& S, const std::vector<MkProblem>& probs, const float* eps6c, long eps_stride,
                               int maxit, const std::vector<int>& msize, c64* X64, long ld, long istride,
                               std::vector<double>& kout, std::vector<int>& iters, std::vector<int>& moves,
                               SolveStats& stats);

// whether the grid fits the phase's transforms
bool multik_fits(const Solver& S);

}  // namespace omx
