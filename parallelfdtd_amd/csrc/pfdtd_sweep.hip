// pfdtd_sweep.hip -- plans, planes and event lists of the several-level sweep (pfdtd_sweep_kernel.h).
#include "pfdtd_sweep_kernel.h"

#include <algorithm>

namespace pfdtd {

// After a bundle of `rounds` rounds: the step and buffers of every job of the launch.
__global__ __launch_bounds__(kPoolMaxJobs) void pool_rotate_kernel(
    const PoolJobDev *__restrict__ jobs, PoolState *__restrict__ state, PoolLaunch pl, int rounds,
    int levels) {
  if ((int)threadIdx.x >= pl.n) return;
  const int job = pl.slot[threadIdx.x];
  const PoolState st = state[job];
  const int left = (jobs[job].n_steps - st.step + levels - 1) / levels;
  const int n = min(rounds, max(left, 0));
  int o1, o2;
  pool_spare(st.cur, st.past, o1, o2);
  state[job] = (n & 1) ? PoolState{st.step + n * levels, o2, o1}
                       : PoolState{st.step + n * levels, st.cur, st.past};
}

// Coefficient entry per voxel: row min(K, 6) of ncol material columns, or kStageRows * ncol outside;
// the centred scheme's entries are the position byte | material << 8.
__global__ __launch_bounds__(256) void pack_entry_kernel(const uint8_t *__restrict__ pos,
                                                         const uint8_t *__restrict__ mat,
                                                         uint16_t *__restrict__ pm, int X,
                                                         int pitch, int64_t rows, unsigned ncol,
                                                         int centred) {
  const int64_t n = rows * pitch;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / pitch;
    const int x = (int)(i - row * pitch);
    unsigned v = centred ? 0u : kStageRows * ncol;
    if (x < X) {
      const unsigned p = pos[row * X + x], m = mat[row * X + x];
      if (centred)
        v = p | min(m, ncol - 1) << 8;
      else if (p & 0x80u) v = min(p & 0x7Fu, 6u) * ncol + min(m, ncol - 1);
    }
    pm[i] = (uint16_t)v;
  }
}

hipError_t launch_pack_entry(const uint8_t *pos, const uint8_t *mat, uint16_t *pm, int X, int Y,
                             int Z, int pitch, int ncol, int scheme, hipStream_t stream) {
  const int64_t rows = (int64_t)Y * Z, n = rows * pitch;
  const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(pack_entry_kernel, dim3(grid), dim3(256), 0, stream, pos, mat, pm, X, pitch,
                     rows, (unsigned)ncol, scheme == 2);
  return hipGetLastError();
}

// A word per (wave tile, slice): bit r of the first byte is set when the tile's row r is plain air over
// its whole window (and inside the grid), of the second when it is never updated (rows 0 and Y-1, past
// the grid, slices 0 and Z-1), of the third when its entries are those of the slice below (never on
// slices 0, 1 and Z-1). Bits past the tile's rows are set in all. A wave per tile and run of slices, each
// lane's columns of the slice below kept in registers, so every entry is loaded once per tile. On
// 2048x1536x768 3.16 ms, a wave per slice with its slice below loaded again 9.26.
constexpr int kRowRun = 32;
template <int NC>
__global__ __launch_bounds__(64) void row_bits_kernel(const uint16_t *__restrict__ pm, int pitch,
                                                      uint32_t *__restrict__ out, int X, int Y,
                                                      int Z, int nbx, int ox, int hx, int oy,
                                                      int lm, int wy, int ty, unsigned ncol,
                                                      int centred) {
  const int lane = threadIdx.x;
  const int bx = blockIdx.x, tw = blockIdx.y;
  const int xs = bx * ox - hx, ys = (tw / wy) * oy - lm + (tw % wy) * ty, x = xs + NC * lane;
  const bool x_in = xs >= 0 && xs + 64 * NC <= X;
  const bool in0 = x >= 0 && x < X, in1 = NC == 2 && x + 1 >= 0 && x + 1 < X;
  const uint32_t past = (0xFFu << ty) & 0xFFu;
  const uint32_t use = (in0 ? 0xFFFFu : 0u) | (in1 ? 0xFFFF0000u : 0u);
  auto entry = [&](int z, int y) -> uint32_t {
    if (!use || y < 0 || y >= Y) return 0;
    const uint16_t *q = pm + ((size_t)z * Y + y) * pitch + x;  // x and pitch even with two columns
    return (NC == 2 ? *(const uint32_t *)q : (uint32_t)*q) & use;
  };
  auto is_air = [&](unsigned v) {
    return centred ? (v & 0xFFu) == 0x80u : v >= 6u * ncol && v < kStageRows * ncol;
  };
  for (int z0 = blockIdx.z * kRowRun; z0 < Z; z0 += gridDim.z * kRowRun) {
    uint32_t below[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) below[r] = r < ty && z0 > 0 ? entry(z0 - 1, ys + r) : 0;
    for (int z = z0; z < min(z0 + kRowRun, Z); ++z) {
      const bool shell = z == 0 || z == Z - 1;
      uint32_t ma = past, ms = shell ? 0xFFu : past, mu = past;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        if (r >= ty) break;
        const int y = ys + r;
        const uint32_t v = entry(z, y);
        const bool not_air = !x_in || y < 0 || y >= Y || !is_air(v & 0xFFFFu) || (NC == 2 && !is_air(v >> 16));
        const bool changed = z < 2 || v != below[r];
        below[r] = v;
        if (!shell) {
          if (__ballot(not_air) == 0) ma |= 1u << r;
          if (y <= 0 || y >= Y - 1) ms |= 1u << r;
          if (__ballot(changed) == 0) mu |= 1u << r;
        }
      }
      if (lane == 0) out[((size_t)tw * nbx + bx) * Z + z] = ma | ms << 8 | mu << 16;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void interleave_kernel(const T *__restrict__ f, int64_t N, int slots,
                                                         T *__restrict__ out) {
  const int64_t total = N * slots;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256)
    out[i] = f[(i % slots) * N + i / slots];
}

hipError_t launch_interleave(int elem_bytes, const void *field, int64_t N, int slots, void *out,
                             hipStream_t stream) {
  const dim3 grid((unsigned)std::min<int64_t>((N * slots + 255) / 256, 65536));
  if (elem_bytes == 2)
    hipLaunchKernelGGL(interleave_kernel<uint16_t>, grid, dim3(256), 0, stream,
                       (const uint16_t *)field, N, slots, (uint16_t *)out);
  else if (elem_bytes == 4)
    hipLaunchKernelGGL(interleave_kernel<uint32_t>, grid, dim3(256), 0, stream,
                       (const uint32_t *)field, N, slots, (uint32_t *)out);
  else
    hipLaunchKernelGGL(interleave_kernel<uint64_t>, grid, dim3(256), 0, stream,
                       (const uint64_t *)field, N, slots, (uint64_t *)out);
  return hipGetLastError();
}

// Time of a launch of `blocks` blocks marching chunks of c slices, in us: CUs hold up to `cap` blocks at
// a time; beyond four such rounds the last one is taken as partly overlapped.
static double sweep_us(const SweepRate &r, int64_t blocks, int c, int levels) {
  const int64_t round = 256 * r.cap, rest = blocks % round;
  const double per = r.a + r.b * r.cap;
  double slice = (double)(blocks / round) * per;
  if (rest) slice += r.a + r.b * (double)((rest + 255) / 256);
  if (blocks > 4 * round) slice = std::min(slice, ((double)blocks / (double)round + 0.4) * per);
  return r.t0 + slice * (c + 2 * (levels - 1) + 2);
}

// Slices per z-chunk for a launch over n grids of bxy[i] blocks per chunk and zi[i] slices: a launch
// takes as many rounds as the CUs' blocks go into its blocks, and a round the chunk's slices plus the 2
// (levels - 1) of its neighbours' and about two more to start. The chunk length with the least of both:
// on 256x256x256 FP32 24 slices (231 blocks) take 34 us per step, 16 slices (two rounds) 50 and 32
// slices 42; on 1024x768x384 48-64 slices 345, 32 and 96 slices 354 and 371.
int sweep_zchunk(int n, const int64_t *bxy, const int *zi, int levels, const SweepRate &rate) {
  int top = 1, best_c = 1;
  for (int i = 0; i < n; ++i) top = std::max(top, zi[i]);
  double best = 0;
  // every chunk length that a number of chunks gives, once: some 2 sqrt(top) of them
  for (int64_t nz = 1, c = top;; nz = ((int64_t)top + c - 2) / (c - 1), c = (top + nz - 1) / nz) {
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) blocks += bxy[i] * ((zi[i] + c - 1) / c);
    const double us = sweep_us(rate, blocks, (int)c, levels);
    if (nz == 1 || us < best) {
      best = us;
      best_c = (int)c;
    }
    if (c == 1) break;
  }
  return best_c;
}

namespace {

template <typename S, int V>
SweepPlan plan_of(int X, int Y, int Z, int zc, int slots) {
  typedef SweepTile<S, V> T;
  SweepPlan p;
  p.tile = V;
  p.nc = T::NC;
  p.ty = T::TY;
  p.wy = T::WY;
  p.lm = T::LM;
  p.w = 64 * T::NC;
  p.hx = T::HX;
  p.ox = p.w - 2 * p.hx;
  p.oy = T::TY * T::WY - 2 * T::LM;
  p.nbx = (int)(((int64_t)X + p.ox - 1) / p.ox);
  p.nby = (int)(((int64_t)Y + p.oy - 1) / p.oy);
  p.pitch = (int)((int64_t)X + (X & 1));
  p.band = 2;
  const int zi = std::max(Z - 2, 1);  // a size query may ask for a room without an inner slice
  const int64_t bxy = (int64_t)p.nbx * p.nby * slots;
  const SweepRate rate{T::T0, T::A, T::B, T::CAP};
  if (zc < 1) zc = sweep_zchunk(1, &bxy, &zi, T::LM, rate);
  p.zc = std::min(zc, zi);
  p.blocks = bxy * ((zi + p.zc - 1) / p.zc);
  p.us = sweep_us(rate, p.blocks, p.zc, T::LM);
  return p;
}

// The tile whose launch takes the least time per step. The small one moves the fields once per three
// steps, so it is only for runs whose four buffers fit the 256 MB Infinity Cache (256x256x256 FP64, 537
// MB: 49 us per step against 41; 200x150x120 FP64, 115 MB: 12.7 against 15.3). A serving pool's jobs
// share one launch and take the large one.
template <typename S>
SweepPlan plan_best(int X, int Y, int Z, int zc, int slots, bool pool) {
  const SweepPlan large = plan_of<S, 0>(X, Y, Z, zc, slots);
  if (pool || 4 * (int64_t)sizeof(S) * X * Y * Z * slots > (int64_t)256 << 20) return large;
  const SweepPlan small = plan_of<S, 1>(X, Y, Z, zc, slots);
  return small.us * large.lm < large.us * small.lm ? small : large;
}

static_assert(SweepTile<float, 0>::LM == kPoolLevels && SweepTile<h16, 0>::LM == kPoolLevels, "");

}  // namespace

hipError_t launch_sweep_pool(int precision, int tiles, const void *args, const PoolJobDev *jobs,
                             const PoolState *st, const PoolLaunch &pl, int zc, int round,
                             hipStream_t stream) {
  switch (precision) {
  case PFDTD_F32: return launch_pool_f32(tiles, args, jobs, st, pl, zc, round, stream);
  case PFDTD_F16: return launch_pool_f16(tiles, args, jobs, st, pl, zc, round, stream);
  case PFDTD_BF16: return launch_pool_bf16(tiles, args, jobs, st, pl, zc, round, stream);
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_pool_rotate(const PoolJobDev *jobs, PoolState *st, const PoolLaunch &pl,
                              int rounds, int levels, hipStream_t stream) {
  hipLaunchKernelGGL(pool_rotate_kernel, dim3(1), dim3(kPoolMaxJobs), 0, stream, jobs, st, pl,
                     rounds, levels);
  return hipGetLastError();
}

SweepPlan plan_sweep(int precision, int X, int Y, int Z, int zc, int slots, bool pool) {
  switch (precision) {
  case PFDTD_F64: return plan_best<double>(X, Y, Z, zc, slots, pool);
  case PFDTD_F16_DIFF:
  case PFDTD_F16: return plan_best<h16>(X, Y, Z, zc, slots, pool);
  case PFDTD_BF16: return plan_best<b16>(X, Y, Z, zc, slots, pool);
  default: return plan_best<float>(X, Y, Z, zc, slots, pool);
  }
}

void sweep_events(const SweepPlan &p, int slots, const std::vector<SweepPoint> &rec,
                  const std::vector<SweepPoint> &src, std::vector<int32_t> &ptr,
                  std::vector<int32_t> &data) {
  const int ntile = p.nby * p.wy * p.nbx;
  struct Ev {
    int tile, row;
    const SweepPoint *q;
  };
  std::vector<Ev> ev;
  auto add = [&](const SweepPoint &q, int bx, int by, int row) {
    ev.push_back(Ev{q.slot * ntile + (by * p.wy + row / p.ty) * p.nbx + bx, row % p.ty, &q});
  };
  for (const SweepPoint &q : rec)
    add(q, q.x / p.ox, q.y / p.oy, q.y % p.oy + p.lm);
  for (const SweepPoint &q : src)
    for (int by = std::max(0, (q.y - p.lm) / p.oy - 1); by < p.nby; ++by) {
      const int row = q.y - by * p.oy + p.lm;
      if (row < 0) break;
      if (row >= p.wy * p.ty) continue;
      for (int bx = std::max(0, (q.x - p.hx) / p.ox - 1); bx < p.nbx; ++bx) {
        const int col = q.x - bx * p.ox + p.hx;
        if (col < 0) break;
        if (col < p.w) add(q, bx, by, row);
      }
    }
  std::stable_sort(ev.begin(), ev.end(), [](const Ev &a, const Ev &b) {
    if (a.tile != b.tile) return a.tile < b.tile;
    return a.q->z != b.q->z ? a.q->z < b.q->z : a.row < b.row;
  });
  ptr.assign((size_t)slots * ntile + 1, 0);
  data.assign(kEvInts * ev.size(), 0);
  for (size_t i = ev.size(); i-- > 0;) {
    ++ptr[(size_t)ev[i].tile + 1];
    int32_t *d = &data[kEvInts * i];
    d[kEvZ] = ev[i].q->z;
    d[kEvX] = ev[i].q->x;
    d[kEvRow] = ev[i].row;
    d[kEvId] = ev[i].q->id;
    const bool z_goes_on = i + 1 < ev.size() && ev[i + 1].tile == ev[i].tile && ev[i + 1].q->z == ev[i].q->z;
    d[kEvNextZ] = z_goes_on ? d[kEvInts + kEvNextZ] : (int32_t)(i + 1);
    d[kEvNextRow] = z_goes_on && ev[i + 1].row == ev[i].row ? d[kEvInts + kEvNextRow] : (int32_t)(i + 1);
  }
  for (size_t i = 1; i < ptr.size(); ++i) ptr[i] += ptr[i - 1];
}

hipError_t launch_row_bits(const SweepPlan &p, const uint16_t *pm, uint32_t *out, int X, int Y,
                           int Z, int ncol, int scheme, hipStream_t stream) {
  const dim3 grid((unsigned)p.nbx, (unsigned)(p.nby * p.wy), (unsigned)((Z + kRowRun - 1) / kRowRun));
  if (p.nc == 2)
    hipLaunchKernelGGL(row_bits_kernel<2>, grid, dim3(64), 0, stream, pm, p.pitch, out, X, Y, Z, p.nbx,
                       p.ox, p.hx, p.oy, p.lm, p.wy, p.ty, (unsigned)ncol, scheme == 2);
  else
    hipLaunchKernelGGL(row_bits_kernel<1>, grid, dim3(64), 0, stream, pm, p.pitch, out, X, Y, Z, p.nbx,
                       p.ox, p.hx, p.oy, p.lm, p.wy, p.ty, (unsigned)ncol, scheme == 2);
  return hipGetLastError();
}

}  // namespace pfdtd
