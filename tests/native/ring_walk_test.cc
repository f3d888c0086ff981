// The nearest-particle walk (fluidity_amd/csrc/ring_walk.h) compiled for the host, against a scan over all
// particles: every walk ends, visits no sub-cell twice and none outside the box, and finds the least squared
// distance. Clouds whose first particle lies 0 to 4 cells (and a fraction) from a bin boundary, moved along one
// axis at a time, with a sixth of the samples (drawn) that fields of radius 0.9, 1, 1.5 and 3 cells may take
// around them: among the particles and up to radius + 2 cells beyond them on every side.
#include <unistd.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "ring_walk.h"

namespace {

struct Point {
  double x[3];
};

int floor_div4(int v) { return v >= 0 ? v / 4 : -1 - (-(v + 1)) / 4; }

struct Cloud {
  std::vector<Point> points;
  int32_t blo[3], bhi[3];
  std::vector<std::vector<Point>> cells;  // by sub-cell of the box

  size_t index(int x, int y, int z) const {
    const size_t nx = bhi[0] - blo[0] + 1, ny = bhi[1] - blo[1] + 1;
    return (size_t(z - blo[2]) * ny + size_t(y - blo[1])) * nx + size_t(x - blo[0]);
  }
  // The box of the particles' bins (bin B holds lattice coordinates [4B + 1.5, 4B + 5.5)).
  void build(double h) {
    for (int a = 0; a < 3; ++a) {
      blo[a] = 1 << 30;
      bhi[a] = -(1 << 30);
      for (const Point& p : points) {
        const int b = floor_div4(static_cast<int>(std::floor(p.x[a] / h - 1.5)));
        blo[a] = std::min(blo[a], 4 * b);
        bhi[a] = std::max(bhi[a], 4 * b + 3);
      }
    }
    cells.assign(index(bhi[0], bhi[1], bhi[2]) + 1, {});
    for (const Point& p : points) {
      int u[3];
      for (int a = 0; a < 3; ++a) u[a] = static_cast<int>(std::floor(p.x[a] / h - 1.5));
      cells[index(u[0], u[1], u[2])].push_back(p);
    }
  }
};

long samples = 0, visits = 0;

// The walk's least squared distance at lattice L against the scan's.
bool sample(const Cloud& c, const double (&L)[3], double h, std::vector<long>& seen) {
  const double w[3] = {L[0] * h, L[1] * h, L[2] * h};
  const auto d2 = [&](const Point& p) {
    const double dx = w[0] - p.x[0], dy = w[1] - p.x[1], dz = w[2] - p.x[2];
    return dx * dx + dy * dy + dz * dz;
  };
  const double none = __builtin_inf();
  double want = none, best = none;
  for (const Point& p : c.points) want = std::min(want, d2(p));
  ++samples;
  bool ok = true;
  fl::ring_walk(L, c.blo, c.bhi, h, best, [&](int32_t x, int32_t y, int32_t z) {
    const int32_t u[3] = {x, y, z};
    for (int a = 0; a < 3; ++a)
      if (u[a] < c.blo[a] || u[a] > c.bhi[a]) {
        ok = false;
        return;
      }
    const size_t i = c.index(x, y, z);
    ok = ok && seen[i] != samples;
    seen[i] = samples;
    ++visits;
    for (const Point& p : c.cells[i]) best = std::min(best, d2(p));
  });
  if (!ok || best != want)
    std::printf("sample (%g, %g, %g): found %g, scan %g%s\n", L[0], L[1], L[2], best, want,
                ok ? "" : ", a sub-cell twice or outside the box");
  return ok && best == want;
}

bool check(Cloud& c, double h, double radius) {
  c.build(h);
  std::vector<long> seen(c.cells.size(), 0);
  int lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    double first = __builtin_inf(), last = -first;
    for (const Point& p : c.points) {
      first = std::min(first, p.x[a] / h);
      last = std::max(last, p.x[a] / h);
    }
    lo[a] = static_cast<int>(std::floor(first - radius)) - 2;
    hi[a] = static_cast<int>(std::floor(last + radius)) + 2;
  }
  bool ok = true;
  for (int z = lo[2]; z <= hi[2]; ++z)
    for (int y = lo[1]; y <= hi[1]; ++y)
      for (int x = lo[0]; x <= hi[0]; ++x)
        for (const double half : {0.0, 0.5}) {
          if (std::rand() % 6 != 0) continue;
          const double L[3] = {x + half, y + half, z + half};
          ok = sample(c, L, h, seen) && ok;
        }
  return ok;
}

}  // namespace

int main() {
  alarm(100);  // a walk that does not end ends the program
  std::srand(7);
  const auto uniform = [] { return (std::rand() + 0.5) / (RAND_MAX + 1.0); };
  bool ok = true;
  for (const double h : {1.0, 0.07})
    for (const double radius : {0.9, 1.0, 1.5, 3.0})
      for (int axis = 0; axis < 3; ++axis)
        for (int k = 0; k <= 40; ++k) {
          const auto place = [&](double x, double y, double z) {
            Point p{{x, y, z}};
            p.x[axis] += 0.1 * k;
            for (double& v : p.x) v *= h;
            return p;
          };
          Cloud one, cube, two;
          one.points = {place(0.0, 0.3, 0.3)};
          for (int q = 0; q < 27; ++q)
            cube.points.push_back(place((q % 3) * (0.9 + 0.1 * uniform()), (q / 3 % 3) * (0.9 + 0.1 * uniform()),
                                        (q / 9) * (0.9 + 0.1 * uniform())));
          two.points = {place(0.0, 0.0, 0.0), place(5.7, 4.1, 6.9)};
          for (Cloud* c : {&one, &cube, &two})
            if (!check(*c, h, radius)) {
              std::printf("h %g radius %g axis %d first particle at %g\n", h, radius, axis, 0.1 * k);
              ok = false;
            }
        }
  std::printf("%ld samples, %ld sub-cells visited\n", samples, visits);
  return ok ? 0 : 1;
}
