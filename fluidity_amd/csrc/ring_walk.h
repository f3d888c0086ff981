// The walk of the nearest-particle search (field.hip) over the sub-cells around a sample. Apart from the
// kernel, and without its types, so that the same code compiles for the host.
#pragma once
#include <math.h>
#include <stdint.h>

#ifdef __HIPCC__
#define FL_WALK __device__ __forceinline__
#else
#define FL_WALK inline
#endif

namespace fl {

// Calls visit(ux, uy, uz) for sub-cells of the box blo .. bhi (sub-cell u covers the lattice coordinates
// [u + 1.5, u + 2.5)) around the sample at L, in rings of growing radius rho (cells). visit lowers best, the
// least squared distance so far (infinite at first). Within a ring the sub-cells touching the sample come
// first (they hold the nearest particle of a liquid sample, and lie in the first ring), then the rest; a
// plane, row or sub-cell whose box is farther than the least distance so far is skipped, and so is the run of
// a row that the previous ring visited. The walk ends when every unvisited sub-cell lies beyond the least
// distance, or the box is done.
template <class Visit>
FL_WALK void ring_walk(const double (&L)[3], const int32_t (&blo)[3], const int32_t (&bhi)[3], double h,
                       const double& best, Visit visit) {
  const double h2 = h * h;
  // Lattice gap between the sample and sub-cell u on one axis, less a slack for particles whose computed
  // sub-cell rounding moved across a face.
  const auto gap = [&](int a, int32_t u) {
    const double g = fmax(fmax((u + 1.5) - L[a], L[a] - (u + 2.5)), 0.0);
    return fmax(g - 1e-6, 0.0);
  };
  int32_t plo[3] = {0, 0, 0}, phi[3] = {-1, -1, -1};  // the previous ring's cube (empty at first)
  for (double rho = 1;;) {
    int32_t lo[3], hi[3];
    bool all = true;
    for (int a = 0; a < 3; ++a) {
      const double l = floor(L[a] - rho - 1.5), u = floor(L[a] + rho - 1.5);
      lo[a] = l <= blo[a] ? blo[a] : static_cast<int32_t>(fmin(l, double(bhi[a]) + 1));
      hi[a] = u >= bhi[a] ? bhi[a] : static_cast<int32_t>(fmax(u, double(blo[a]) - 1));
      all = all && l <= blo[a] && u >= bhi[a];
    }
    for (int pass = rho == 1 ? 0 : 1; pass < 2; ++pass)
      for (int32_t uz = lo[2]; uz <= hi[2]; ++uz) {
        const double gz = gap(2, uz), gz2 = gz * gz;
        if (pass == 0 ? gz != 0 : gz2 * h2 > best * (1 + 1e-9)) continue;
        for (int32_t uy = lo[1]; uy <= hi[1]; ++uy) {
          const double gy = gap(1, uy), gyz = gy * gy + gz2;
          if (pass == 0 ? gy != 0 : gyz * h2 > best * (1 + 1e-9)) continue;
          const bool inner = uy >= plo[1] && uy <= phi[1] && uz >= plo[2] && uz <= phi[2];
          for (int32_t ux = lo[0]; ux <= hi[0]; ++ux) {
            if (inner && ux == plo[0]) {
              ux = phi[0];
              continue;
            }
            const double gx = gap(0, ux);
            const double g2 = gx * gx + gyz;
            if ((g2 == 0) != (pass == 0)) continue;
            if (g2 * h2 > best * (1 + 1e-9)) continue;
            visit(ux, uy, uz);
          }
        }
      }
    for (int a = 0; a < 3; ++a) {
      plo[a] = lo[a];
      phi[a] = hi[a];
    }
    // The cube is empty in x where the sample lies farther than rho beside the box: no run to skip then (a skip
    // to phi = plo - 1 would come back to plo for ever).
    if (lo[0] > hi[0]) plo[0] = INT32_MAX;
    // Every unvisited particle lies at least (rho - rounding) cells from the sample.
    const double reach = sqrt(best) * (1 + 1e-12);
    if (__builtin_isfinite(best) && reach < (rho - 1e-6) * h) break;
    if (all) break;
    // The next ring: twice as far, or just beyond the least distance once there is one.
    rho = __builtin_isfinite(best) ? fmin(2 * rho, reach / h * (1 + 1e-9) + 1e-5) : 2 * rho;
  }
}

}  // namespace fl
