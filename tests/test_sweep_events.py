"""The event lists of the several-level sweep, on the CPU: for every wave tile, slice and row the walk of
the kernel finds the events of that row, receivers before sources and each in index order, and looks at
little else however many events the tile has."""
import hostrt

SOURCE = r"""
#include "pfdtd_internal.h"
#include <algorithm>
#include <cstdio>
#include <map>
#include <random>
using namespace pfdtd;

int fails = 0;

void check(int precision, int X, int Y, int Z, int slots, int n_rec, int n_src, int patch) {
  const SweepPlan p = plan_sweep(precision, X, Y, Z, 0, slots);
  std::mt19937 g(n_rec + 7 * n_src);
  auto pick = [&](int n) { return (int)(g() % (unsigned)n); };
  std::vector<SweepPoint> rec, src;
  for (int r = 0; r < n_rec; ++r)
    rec.push_back(patch ? SweepPoint{3 + r % patch, 5 + r / patch % patch, Z / 2, 0, (int32_t)((uint32_t)r | 0x80000000u)}
                        : SweepPoint{pick(X), pick(Y), pick(Z), pick(slots), (int32_t)((uint32_t)r | 0x80000000u)});
  for (int s = 0; s < n_src; ++s) src.push_back(SweepPoint{pick(X), pick(Y), pick(Z), pick(slots), s});
  std::vector<int32_t> ptr, data;
  sweep_events(p, slots, rec, src, ptr, data);
  const int ntile = p.nby * p.wy * p.nbx;
  if (ptr.size() != (size_t)slots * ntile + 1 || data.size() != kEvInts * (size_t)ptr.back()) ++fails;
  size_t found_rec = 0;
  for (int slot = 0; slot < slots; ++slot)
    for (int t = 0; t < ntile; ++t) {
      const int bx = t % p.nbx, w = t / p.nbx % p.wy, by = t / p.nbx / p.wy;
      const int first = ptr[slot * ntile + t], end = ptr[slot * ntile + t + 1];
      if (first == end) continue;
      for (int z = 0; z < Z; ++z)
        for (int row = 0; row < p.ty; ++row) {
          const int y = by * p.oy - p.lm + w * p.ty + row;
          std::vector<std::pair<int, int>> want, got;  // (x, id)
          for (const SweepPoint &q : rec)
            if (q.slot == slot && q.z == z && q.y == y && q.y / p.oy == by && q.x / p.ox == bx) want.push_back({q.x, q.id});
          for (const SweepPoint &q : src)
            if (q.slot == slot && q.z == z && q.y == y && q.x >= bx * p.ox - p.hx && q.x < bx * p.ox - p.hx + p.w)
              want.push_back({q.x, q.id});
          int looked = 0;
          for (int n = first; n < end;) {
            const int32_t *e = &data[kEvInts * n];
            ++looked;
            if (e[kEvZ] != z) {
              if (e[kEvZ] > z) break;
              n = e[kEvNextZ];
              continue;
            }
            if (e[kEvRow] != row) {
              if (e[kEvRow] > row) break;
              n = e[kEvNextRow];
              continue;
            }
            ++n;
            got.push_back({e[kEvX], e[kEvId]});
          }
          found_rec += std::count_if(got.begin(), got.end(), [](auto &v) { return v.second < 0; });
          std::map<int, int> slices;
          for (int n = first; n < end; ++n) ++slices[data[kEvInts * n + kEvZ]];
          if (got != want || looked > (int)(got.size() + slices.size()) + p.ty + 1) ++fails;
        }
    }
  if (found_rec != rec.size()) ++fails;
  std::printf("%d: %dx%dx%d slots %d tile %d: %d events, fails %d\n", precision, X, Y, Z, slots, p.tile, (int)ptr.back(), fails);
}

int main() {
  for (int precision : {0, 1, 2}) {
    check(precision, 40, 30, 9, 1, 64, 3, 8);
    check(precision, 40, 30, 9, 1, 400, 40, 4);  // several to a voxel
    check(precision, 120, 60, 7, 1, 300, 60, 0);
    check(precision, 130, 50, 8, 4, 200, 50, 0);
    check(precision, 70, 44, 6, 1, 0, 5, 0);
    check(precision, 70, 44, 6, 1, 5, 0, 0);
    check(precision, 3, 3, 3, 1, 2, 1, 0);
  }
  return fails ? 1 : 0;
}
"""


def test_event_lists(tmp_path):
    out = hostrt.run_program(SOURCE, ["pfdtd_sweep.hip"], tmp_path)
    assert out.returncode == 0, out.stdout + out.stderr
