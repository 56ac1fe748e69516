"""The z-chunk of the several-level sweep, on the CPU: the choice among all numbers of chunks, at a cost
that does not grow with the number of slices (it is made for every call)."""
import hostrt

SOURCE = r"""
#include "pfdtd_internal.h"
#include <algorithm>
#include <chrono>
#include <cstdio>
using namespace pfdtd;

// a launch's time as the planner models it
double model(const SweepRate &r, int64_t blocks, int c, int levels) {
  const int64_t round = 256 * r.cap, rest = blocks % round;
  const double per = r.a + r.b * r.cap;
  double slice = (double)(blocks / round) * per;
  if (rest) slice += r.a + r.b * (double)((rest + 255) / 256);
  if (blocks > 4 * round) slice = std::min(slice, ((double)blocks / (double)round + 0.4) * per);
  return r.t0 + slice * (c + 2 * (levels - 1) + 2);
}

int among_all(int n, const int64_t *bxy, const int *zi, int levels, const SweepRate &rate) {
  int top = 1, best_c = 1;
  for (int i = 0; i < n; ++i) top = std::max(top, zi[i]);
  double best = 0;
  for (int nz = 1; nz <= top; ++nz) {
    const int c = (top + nz - 1) / nz;
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) blocks += bxy[i] * ((zi[i] + c - 1) / c);
    const double us = model(rate, blocks, c, levels);
    if (nz == 1 || us < best) best = us, best_c = c;
  }
  return best_c;
}

int main() {
  int fails = 0;
  const SweepRate rates[] = {{8, 4, 0, 1}, {3, 1.1, 0.5, 3}, {0, 1, 0, 1}};
  for (const SweepRate &r : rates)
    for (int levels : {3, 4, 5})
      for (int64_t b : {1, 7, 30, 200, 3000})
        for (int z = 1; z <= 800; z += z < 90 ? 1 : 37) {
          const int64_t bxy[2] = {b, b / 3 + 1};
          const int zi[2] = {z, z / 2 + 1};
          for (int n : {1, 2})
            if (sweep_zchunk(n, bxy, zi, levels, r) != among_all(n, bxy, zi, levels, r)) ++fails;
        }
  const auto t0 = std::chrono::steady_clock::now();
  int64_t one = 1;
  const int deep = 1 << 30;
  sweep_zchunk(1, &one, &deep, 5);
  const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  std::printf("fails %d, %.3f s for 2^30 slices\n", fails, s);
  return fails || s > 0.5;
}
"""


def test_chunks(tmp_path):
    out = hostrt.run_program(SOURCE, ["pfdtd_sweep.hip"], tmp_path)
    assert out.returncode == 0, out.stdout
