// How the constant-viscosity apply (k_visc_apply) lays its vertices over
// wavefronts and their LDS: plain host and device code, so that the sizes the
// host reserves can be checked without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>

#ifdef __HIPCC__
#define SFV_HD __host__ __device__ inline
#else
#define SFV_HD inline
#endif

namespace sfv {

// consecutive vertices per wavefront: kDiffHalf, kDiffWave
constexpr int kDiffApplyVerts[2] = {4, 2};

// doubles of LDS for a vertex of ni stored faces and nf faces: block products (or
// one-sided fluxes), right-hand side, area vectors, types; even: rows of four are
// read and written in pairs
template <bool GLOBAL>
SFV_HD int apply_lds(int ni, int nf) {
  const int part = GLOBAL ? 8 * ni : (ni > 2 ? 4 * ni * ni : 8 * ni);
  return (part + 4 * ni + 3 * nf + (ni + 1) / 2 + 1) & ~1;
}

// The vertex of lane group g in wavefront w, per groups to a wavefront: past the
// last one its groups mirror it; -1 where the whole wavefront is past it (the
// launch rounds up to whole workgroups): such a wavefront has no LDS of its own
// and returns.
SFV_HD long apply_vertex(long w, int per, int g, long V) {
  if (w * per >= V) return -1;
  const long v = w * per + g;
  return v < V ? v : V - 1;
}

// doubles of LDS of the fullest wavefront; size(v): apply_lds of vertex v
template <class Size>
int apply_lds_wave(long V, int per, Size size) {
  int most = 0;
  for (long w = 0; w * per < V; w++) {
    int sum = 0;
    for (int g = 0; g < per; g++) sum += size(apply_vertex(w, per, g, V));
    most = std::max(most, sum);
  }
  return most;
}

}  // namespace sfv
