// Counter-based normal numbers (splitmix64, Box-Muller), the same for every kernel that
// draws start vectors.
#pragma once
#include "omx_common.hpp"

namespace omx {

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// complex normal of row `row` of column c of instance inst (unit variance)
__device__ __forceinline__ c64 randn_at(uint64_t seed, int inst, int c, long row) {
  const uint64_t key = mix64(seed ^ mix64(uint64_t(inst) * 0x100000001b3ull + uint64_t(c))) + uint64_t(row) * 2;
  const uint64_t h1 = mix64(key), h2 = mix64(key + 1);
  const double u1 = (double(h1 >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  const double u2 = double(h2 >> 11) * (1.0 / 9007199254740992.0);
  const double rad = sqrt(-2.0 * log(u1)) * 0.70710678118654752;
  double s, co;
  sincospi(2.0 * u2, &s, &co);
  return c64{rad * co, rad * s};
}

}  // namespace omx
