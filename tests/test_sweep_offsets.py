"""The byte offsets at which the lanes of the several-level sweep store, on the CPU: a lane that owns its
columns and row stores at their place in the slice, every other one past the slice, also on grids whose
rows are a large part of 2^31 bytes."""
import hostrt

SOURCE = r"""
#include "pfdtd_sweep_kernel.h"
#include <cstdio>
#include <cstdlib>
using namespace pfdtd;

template <typename S, int V>
long check(int X, int Y) {
  typedef SweepTile<S, V> T;
  constexpr int NC = T::NC, OX = 64 * NC - 2 * T::HX, OY = T::TY * T::WY - 2 * T::LM;
  const int es = sizeof(S), nbx = (X - 1) / OX + 1, nby = (Y - 1) / OY + 1;
  const uint64_t slice = (uint64_t)X * Y * es;
  long bad = 0;
  for (int bx : {0, 1, nbx / 2, nbx - 2, nbx - 1})
    for (int by : {0, 1, nby - 2, nby - 1}) {
      if (bx < 0 || by < 0 || bx >= nbx || by >= nby) continue;
      for (int wave = 0; wave < T::WY; ++wave)
        for (int lane = 0; lane < 64; ++lane) {
          const int x0 = bx * OX - T::HX + NC * lane, yw = by * OY - T::LM + wave * T::TY;
          const SweepLane l = sweep_lane<NC, T::HX>(X, x0, yw, lane, es);
          const bool own_x = x0 >= bx * OX && x0 < bx * OX + OX && x0 < X, both = NC == 1 || x0 + 1 < X;
          for (int r = 0; r < T::TY; ++r) {
            const int y = yw + r;
            const bool own_y = y >= by * OY && y < by * OY + OY && y < Y;
            const uint32_t step = (uint32_t)X * (uint32_t)es, drop = own_y ? 0u : kDrop;
            const uint64_t place = own_x && own_y ? ((uint64_t)y * X + x0) * es : 0;
            const uint32_t a = l.at(r * step, drop), a1 = l.at1(r * step, drop);
            if (own_x && own_y && both ? a != place || a + (uint64_t)NC * es > slice : a < slice) ++bad;
            if (own_x && own_y && !both ? a1 != place : a1 < slice) ++bad;
          }
        }
    }
  if (bad) std::printf("%d x %d, %d bytes, tile %d: %ld wrong\n", X, Y, es, V, bad);
  return bad;
}

template <typename S>
long sizes() {
  const int es = sizeof(S);
  const int64_t cells = ((int64_t)1 << 31) / es - 1;
  long bad = 0;
  for (int Y : {3, 4, 5, 7, 8, 40, 60, 1000})
    for (int64_t X : {cells / Y, cells / Y - 1, cells / Y / 2, (int64_t)1000, (int64_t)113, (int64_t)3})
      bad += check<S, 0>((int)X, Y) + check<S, 1>((int)X, Y);
  return bad;
}

int main() { return sizes<float>() + sizes<double>() + sizes<h16>() ? 1 : 0; }
"""


def test_store_offsets(tmp_path):
    out = hostrt.run_program(SOURCE, [], tmp_path)
    assert out.returncode == 0, out.stdout
