// pfdtd_sweep_kernel.h -- several time levels of the forward update per sweep of the field.
//
// One launch reads P^n (A) and P^{n-1} (B) once and writes P^{n+L-1} (Cn) and P^{n+L} (Dn); the L-1
// levels between never leave the chip. Sources are injected and receivers gathered at every level,
// the last included, in the reference's order (a level's gather before the next step's injection),
// and the node arithmetic, sum order and storage rounding are the single step's, so the results are
// L single steps bit for bit.
//
// Tiling. A block of WY waves marches a z-chunk. A wave holds TY rows of a window of 64 NC columns,
// two slices of every level's rows in registers: at iteration k the rows of level i advance to slice
// k-i+1 from level i-1's slices k-i, k-i+1 and (just computed) k-i+2, row by row through all levels,
// and each new row takes the place of the oldest one. x-neighbours come from the lane's other column
// or a DPP shift; y-neighbours from the wave's other rows or, at its first and last row, from the
// neighbouring wave's through LDS: every wave publishes the edge rows of its new slices, one barrier
// per slice, double-buffered. So a block recomputes a halo only at its own border (L rows and HX
// columns on either side), where a sweep of independent waves recomputes one around every wave: the
// three-level sweep computes 1.8 nodes and loads 4.5 rows per node-update it keeps, this one 1.5 (L =
// 5) and 2.2.
//
// What bounds it (2048x1536x768 FP32, L = 5): 2.04-2.33 ms per step against 3.73-3.83 for the
// three-level sweep of independent waves, 19.4 GB written and 30.2 read per launch at 4.85 TB/s of a
// copy's 5.5: the traffic. FP64 (L = 4): 1024x768x384 0.64 ms against 1.03. Rooms in the Infinity Cache
// are bound by issue (below). Tiles measured before the last steps (ms per step, 2048x1536x768 FP32, same card): L = 4
// 8 rows 2.95, 6 rows 2.96; L = 5 6 rows 2.52, 7 rows (spills) 2.55; L = 6 does not fit LDS. Windows: stores of
// whole 64-byte lines matter (112 owned columns 2.99, 120 columns 3.26 with L = 4), so HX is 8
// although five columns would do; 16 (96 owned columns) 3.07.
//
// Rows of plain air at every level of an iteration take the air entry as an immediate (nine VALU
// operations per node); rows never updated at any level (the outer layer, past the grid) are zeros. Of
// the others, those whose entries are the same on the iteration's slices -- along walls, pillars and the
// sides of boxes, and inside solids -- gather one entry per node for all levels; the rest gather every
// node's entry at every level from LDS, the gathers of the next level in flight during the last. The
// choice is made by three bits per row and slice built once per domain. Made once for all rows of an
// iteration instead, it keeps both the old and the new queue entries live (75 registers more). Entries
// the slice above shares stay in their registers and are not loaded again.
//
// Solid voxels inside the room are computed: 0 times what surrounds them, which is NaN beside an infinity
// or NaN. Rows of them taken as zeros would stop those at a wall, unlike single steps. On a 1024x768x384
// hall, a quarter of it solid, that costs 292 -> 300 us per step in FP32, 282 -> 307 in FP16, 279 -> 294
// in BF16, nothing in FP64; zeros only while all that the rows read is finite, looked at on the way,
// costs every room 2 to 6 %.
//
// Within a CU the sweep is bound by issue: two waves of a SIMD issue some 1200 instructions each per
// slice, about 3.5 ns for two dependent FP32 additions and 1.3 for independent ones, so a lane's
// two columns are written side by side. us per step, one entry per node and level -> one per node ->
// columns side by side, and accesses behind the choice of the row: 1024x768x384 hall FP32 355 -> 320 ->
// 309, 256x256x256 FP32 33.4 -> 29.5 -> 27.3, 701x523x307 BF16 158 -> 142 -> 123, 130x98x66 FP32
// 12.2 -> 11.5 -> 10.8, 1024x768x384 FP64 750 -> 712 -> 725, 2048x1536x768 FP16 2004 -> 1962 -> 1955.
// Sixteen waves of 3 rows each (four waves per SIMD, 4 levels to fit 128 registers) take 371 on the
// hall and 28.6 on 256x256x256.
//
// The difference form (A holds P^n, B holds D^n = P^n - P^{n-1}; P^{n+L} to Dn and D^{n+L} to Cn, both
// from the last level) also keeps every level's rounded differences of one slice; the past value of a
// node is P - D in FP32, and a sample keeps it. 256 VGPRs, two spilled. 640x480x320 hall, 400 steps: 66.7 ms
// with the two-level sweep of independent waves -> 49.
//
// The centred boundaries take the same tiles: the entry plane holds position and material bytes, and the
// DIR and SIGN bits pick the neighbour that stands in for a missing one (15 VALU operations per air node,
// about 35 otherwise). 448x264x135 FP32, 300 steps in segments of 25: the sweeps 73 us per step with two
// levels of independent waves, 49 with five here.
//
// Loads, stores and masks. Slices are accessed through buffer descriptors: rows and columns past
// the grid read 0, stores that a lane or row does not own are given an offset past the slice and
// dropped, so the body has no masked branches. The loads of the next slice are issued as soon as a
// row has consumed its own, a whole iteration ahead of their use.
#pragma once

#include "../../include/pfdtd.h"
#include "pfdtd_device.h"

#include <type_traits>
#include <utility>

namespace pfdtd {

namespace {

__device__ __forceinline__ float sw_next(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xF, 0xF, true));
}
__device__ __forceinline__ float sw_prev(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ double sw_next(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x130, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x130, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sw_prev(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// Slice access through a buffer descriptor: out-of-range offsets read 0 and drop stores, so
// rows and columns past the grid need no clamps and masked stores no branches.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sw_rsrc(const void *p, uint32_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)nbytes,
                                           0x00020000);
}

template <int... R, typename F>
__device__ __forceinline__ void sw_inner_rows(std::integer_sequence<int, R...>, F &f) {
  (f(R + 1), ...);
}

// Keeps a value's computation ahead of the select that masks it (a select between it and 0 would
// otherwise become a lane-masked branch around the computation).
__device__ __forceinline__ void sw_keep(float &v) { asm("" : "+v"(v)); }
__device__ __forceinline__ void sw_keep(double &v) { asm("" : "+v"(v)); }

// Field stores are non-temporal (aux bit 1): a launch reads what the one before stored, a whole field ago,
// so a stored line only takes the place of rows that neighbouring tiles still read. us per step, plain ->
// non-temporal: 1024x768x384 FP64 719 -> 642, FP32 305 -> 294; rooms within the Infinity Cache and 16-bit
// fields within 1 %. Non-temporal loads of P^{n-1} lose the reuse between tiles: 1024x768x384 FP64 790.
constexpr int kStream = 2;

// NC columns of one row held by a lane, and their raw form in the storage type.
template <typename C, int NC>
struct Cols {
  C v[NC];
};
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <typename S, int NC>
struct Raw;
template <>
struct Raw<float, 2> {
  typedef u32x2 T;
  static __device__ __forceinline__ T ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
  }
  static __device__ __forceinline__ Cols<float, 2> up(T t) {
    return Cols<float, 2>{{__uint_as_float(t.x), __uint_as_float(t.y)}};
  }
  static __device__ __forceinline__ T pack(const Cols<float, 2> &c) {
    u32x2 t;
    t.x = __float_as_uint(c.v[0]);
    t.y = __float_as_uint(c.v[1]);
    return t;
  }
  static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t off, T t) {
    __builtin_amdgcn_raw_buffer_store_b64(t, r, (int)off, 0, kStream);
  }
  static __device__ __forceinline__ void st1(__amdgpu_buffer_rsrc_t r, uint32_t off, T t, int c) {
    __builtin_amdgcn_raw_buffer_store_b32(c ? t.y : t.x, r, (int)off, 0, kStream);
  }
};
template <>
struct Raw<float, 1> {
  typedef uint32_t T;
  static __device__ __forceinline__ T ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
  }
  static __device__ __forceinline__ Cols<float, 1> up(T t) { return Cols<float, 1>{{__uint_as_float(t)}}; }
  static __device__ __forceinline__ T pack(const Cols<float, 1> &c) { return __float_as_uint(c.v[0]); }
  static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t off, T t) {
    __builtin_amdgcn_raw_buffer_store_b32(t, r, (int)off, 0, kStream);
  }
  static __device__ __forceinline__ void st1(__amdgpu_buffer_rsrc_t r, uint32_t off, T t, int) {
    st(r, off, t);
  }
};
template <>
struct Raw<double, 1> {
  typedef u32x2 T;
  static __device__ __forceinline__ T ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
  }
  static __device__ __forceinline__ Cols<double, 1> up(T t) {
    return Cols<double, 1>{{__hiloint2double((int)t.y, (int)t.x)}};
  }
  static __device__ __forceinline__ T pack(const Cols<double, 1> &c) {
    return __builtin_bit_cast(u32x2, c.v[0]);
  }
  static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t off, T t) {
    __builtin_amdgcn_raw_buffer_store_b64(t, r, (int)off, 0, kStream);
  }
  static __device__ __forceinline__ void st1(__amdgpu_buffer_rsrc_t r, uint32_t off, T t, int) {
    st(r, off, t);
  }
};
template <typename S>
struct Raw<S, 1> {
  static_assert(sizeof(S) == 2, "16-bit storage");
  typedef uint16_t T;
  static __device__ __forceinline__ T ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
  }
  static __device__ __forceinline__ Cols<float, 1> up(T t) { return Cols<float, 1>{{Fmt<S>::val(S{t})}}; }
  static __device__ __forceinline__ T pack(const Cols<float, 1> &c) { return Fmt<S>::bits(c.v[0]); }
  static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t off, T t) {
    __builtin_amdgcn_raw_buffer_store_b16(t, r, (int)off, 0, kStream);
  }
  static __device__ __forceinline__ void st1(__amdgpu_buffer_rsrc_t r, uint32_t off, T t, int) {
    st(r, off, t);
  }
};
template <typename S>
struct Raw<S, 2> {
  static_assert(sizeof(S) == 2, "16-bit storage");
  typedef uint32_t T;
  static __device__ __forceinline__ T ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
  }
  static __device__ __forceinline__ Cols<float, 2> up(T t) {
    return Cols<float, 2>{{Fmt<S>::val(S{(uint16_t)(t & 0xFFFFu)}), Fmt<S>::val(S{(uint16_t)(t >> 16)})}};
  }
  static __device__ __forceinline__ T pack(const Cols<float, 2> &c) {
    return Fmt<S>::bits2(c.v[0], c.v[1]);
  }
  static __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, uint32_t off, T t) {
    __builtin_amdgcn_raw_buffer_store_b32(t, r, (int)off, 0, kStream);
  }
  static __device__ __forceinline__ void st1(__amdgpu_buffer_rsrc_t r, uint32_t off, T t, int c) {
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(c ? t >> 16 : t & 0xFFFFu), r, (int)off, 0, kStream);
  }
};

// x+1 and x-1 neighbours of column c of a lane's NC columns.
template <typename C, int NC>
__device__ __forceinline__ C x_next(const Cols<C, NC> &q, int c) {
  return c + 1 < NC ? q.v[c + 1 < NC ? c + 1 : 0] : sw_next(q.v[0]);
}
template <typename C, int NC>
__device__ __forceinline__ C x_prev(const Cols<C, NC> &q, int c) {
  return c > 0 ? q.v[c > 0 ? c - 1 : 0] : sw_prev(q.v[NC - 1]);
}

typedef const __attribute__((address_space(4))) int32_t *ConstI32;
typedef const __attribute__((address_space(4))) uint32_t *ConstU32;

// Slices of packed rows a wave keeps in LDS: the L - 1 slices above the first level's, rounded up
// to a power of two.
constexpr int sweep_ring(int L) { return L <= 2 ? 1 : L == 3 ? 2 : 4; }

constexpr int kForward = 0, kDiff = 1, kCentred = 2;  // modes of the sweep

constexpr uint32_t kDrop = 0x80000000u;  // offset bit that puts a store out of range (slices are below 2^31 bytes)

// A lane's offsets in a slice of X columns, from its first column x0 in the first row yw of its wave, and
// whether it drops the stores of its columns as a whole and of the first one alone (the last column of
// an odd width). The drop bits are kept apart from the offsets: a row of a very wide grid added to a
// dropped offset would carry it past 2^32 and back into the slice.
struct SweepLane {
  uint32_t off, drop, drop1;
  __host__ __device__ uint32_t at(uint32_t row_off, uint32_t row_drop) const {
    return (off + row_off) | drop | row_drop;
  }
  __host__ __device__ uint32_t at1(uint32_t row_off, uint32_t row_drop) const {
    return (off + row_off) | drop1 | row_drop;
  }
};
template <int NC, int HX>
__host__ __device__ __forceinline__ SweepLane sweep_lane(int X, int x0, int yw, int lane, int elem) {
  const bool own_x = NC * lane >= HX && NC * lane < 64 * NC - HX && x0 < X;
  const bool pair = NC == 1 || x0 + 1 < X;  // the lane's columns both lie in the grid
  return SweepLane{((uint32_t)yw * (uint32_t)X + (uint32_t)x0) * (uint32_t)elem,
                   own_x && pair ? 0u : kDrop, own_x && !pair ? 0u : kDrop};
}

}  // namespace

template <typename S>
using SweepArgsOf = SweepArgs<S, typename CoefOf<typename Fmt<S>::C>::T, typename Fmt<S>::C>;
// Arguments of a sweep in constant memory: the kernel's own, or a pool job's.
template <typename S>
using ConstSweepArgs = const __attribute__((address_space(4))) SweepArgsOf<S> *;

// One block of a sweep: tile `tile` of nbx x nby x (z-chunks of zc slices), fields fA, fB to fC, fD,
// first step `step`.
template <typename S, int L, int LM, int TY, int WY, int NC, int HX, int MODE>
__device__ __forceinline__ void sweep_block(ConstSweepArgs<S> args, unsigned tile, int slot, int zc,
                                            const S *__restrict__ gA, const S *__restrict__ gB,
                                            S *__restrict__ gC, S *__restrict__ gD, int step) {
#pragma clang fp contract(off)
  typedef typename Fmt<S>::C C;
  typedef typename CoefOf<C>::T CE;
  typedef ConstSweepArgs<S> ConstArgs;
  constexpr bool DIFF = MODE == kDiff, CENTRED = MODE == kCentred;
  const auto &a = *args;
  typedef Cols<C, NC> V;
  typedef Raw<S, NC> R;
  typedef typename std::conditional<NC == 2, uint32_t, uint16_t>::type PM;
  static_assert(TY >= 2 && TY <= 8 && L >= 1 && L <= LM && LM <= 5 && HX >= LM && HX % NC == 0, "");
  constexpr int W = 64 * NC, OX = W - 2 * HX;
  constexpr int H = WY * TY, OY = H - 2 * LM;
  constexpr int RING = sweep_ring(L);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int X = a.X, Y = a.Y, Z = a.Z;
  const unsigned ncol = (unsigned)a.ncol;
  const unsigned nxy = (unsigned)(a.nbx * a.nby);
  const unsigned tl = tile % nxy;
  const int bzi = (int)(tile / nxy);
  const unsigned bg = (unsigned)a.band;
  const unsigned band = tl / (bg * a.nbx), in_band = tl % (bg * a.nbx);
  const unsigned band_rows = min(bg, (unsigned)a.nby - band * bg);
  const int byi = (int)(band * bg + in_band % band_rows);
  const int bxi = (int)(in_band / band_rows);
  const int x0 = bxi * OX - HX + NC * lane;           // this lane's first column
  const int yw = byi * OY - LM + wave * TY;           // this wave's first row
  const int z0 = 1 + bzi * zc, z1 = min(z0 + zc, Z - 1);

  // LDS: coefficient rows | halo rows [2][L][WY][2][64] | packed rows [WY][RING][TY][64]
  extern __shared__ __align__(16) unsigned char s_dyn[];
  CE *s_coef = reinterpret_cast<CE *>(s_dyn);
  V *s_halo = reinterpret_cast<V *>(s_dyn + sizeof(CE) * (kStageRows * ncol + 1));
  PM *s_pm = reinterpret_cast<PM *>(s_halo + 2 * L * WY * 2 * 64) + wave * (RING * TY * 64) + lane;
  for (unsigned i = threadIdx.x; i < kStageRows * ncol; i += 64 * WY)
    s_coef[i] = a.coef[(i / ncol) * 256u + i % ncol];
  if (threadIdx.x == 0) {  // outside voxels: the result is 0
    CE e = a.coef[0];
    e.inv = 0;
    s_coef[kStageRows * ncol] = e;
  }

  const size_t XY = (size_t)X * (size_t)Y;
  const uint32_t sbytes = (uint32_t)(XY * sizeof(S));
  const size_t XYP = (size_t)a.pitch * (size_t)Y;
  const SweepLane sl = sweep_lane<NC, HX>(X, x0, yw, lane, (int)sizeof(S));
  const uint32_t vcol = sl.off;
  const uint32_t pcol = ((uint32_t)yw * (uint32_t)a.pitch + (uint32_t)x0) * 2u;
  // owned columns of this lane, owned rows of this wave
  const bool own_x = NC * lane >= HX && NC * lane < HX + OX && x0 < X;
  uint32_t own_rows = 0;
#pragma unroll
  for (int r = 0; r < TY; ++r) {
    const int br = wave * TY + r, y = yw + r;
    if (br >= LM && br < LM + OY && y < Y) own_rows |= 1u << r;
  }
  uint32_t upd_rows = 0;  // rows of 1..Y-2 (the difference form)
#pragma unroll
  for (int r = 0; r < TY; ++r)
    if (yw + r > 0 && yw + r < Y - 1) upd_rows |= 1u << r;
  bool col_ok[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) col_ok[c] = x0 + c > 0 && x0 + c < X - 1;
  // the tile with the last column of an odd width, which is stored on its own
  const bool odd_edge = NC == 2 && (X & 1) && bxi == a.nbx - 1;
  const C air_tk = a.air.tk, lam2 = a.lam2;
  CE air_e{};
  air_e.inv = a.air.inv;
  air_e.omb = a.air.omb;
  air_e.tk = air_tk;
  const uint32_t air_pm = a.air_pm, air_mask = a.air_mask, out_pm = CENTRED ? 0u : kStageRows * ncol * 0x10001u;

  // air, never updated and unchanged rows of this wave's tile (a byte each, a word per slice), and its events
  // by z
  const int wt = (byi * WY + wave) * a.nbx + bxi;
  const ConstU32 grows = (ConstU32)(a.row_bits + (size_t)wt * Z);
  int ev = 0, ev_end = 0;
  {
    const int et = slot * (a.nby * WY * a.nbx) + wt;
    ev = ((ConstI32)a.ev_ptr)[et];
    ev_end = ((ConstI32)a.ev_ptr)[et + 1];
  }
  struct EvHead {
    int z, row, next_row, next_z;
  };
  auto ev_head = [&](int n) -> EvHead {  // one load of four words
    ConstArgs ka = args;
    asm volatile("" : "+s"(ka));
    const ConstI32 g = (ConstI32)ka->events + kEvInts * (int64_t)n;
    return EvHead{g[kEvZ], g[kEvRow], g[kEvNextRow], g[kEvNextZ]};
  };

  V q[L][2][TY];  // level 0: P^n, level i: P^{n+i}; two slices each
  typename R::T pl[TY], pq[TY];  // raw P^n[k+1] and P^{n-1}[k] (the difference form: D^n[k])
  typename R::T qd[L][TY];       // the difference form: raw D of level i's slice k-i (i > 0)
  uint32_t pmr[TY];              // packed entries of slice k where it is not all air
#pragma unroll
  for (int i = 0; i < L; ++i)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < TY; ++r)
#pragma unroll
        for (int c = 0; c < NC; ++c) q[i][b][r].v[c] = (C)0;
#pragma unroll
  for (int r = 0; r < TY; ++r) {
    pmr[r] = 0;
#pragma unroll
    for (int i = 0; i < L; ++i) qd[i][r] = typename R::T{};
  }

  auto a_rsrc = [&](int k) {
    const bool in = k >= 0 && k < Z;
    return sw_rsrc(gA + (in ? (size_t)k * XY : 0), in ? sbytes : 0u);
  };
  auto b_rsrc = [&](int k) {
    const bool in = k >= 1 && k < Z - 1;
    return sw_rsrc(gB + (in ? (size_t)k * XY : 0), in ? sbytes : 0u);
  };
  auto load_pm = [&](int k) __attribute__((always_inline)) {
    const bool in = k >= 1 && k < Z - 1;
    const auto rp = sw_rsrc(a.pm + (in ? (size_t)k * XYP : 0), in ? (uint32_t)(XYP * 2) : 0u);
    uint32_t off = pcol, step = (uint32_t)a.pitch * 2u;
#pragma unroll
    for (int r = 0; r < TY; ++r, off += step)
      pmr[r] = NC == 2 ? __builtin_amdgcn_raw_buffer_load_b32(rp, (int)off, 0, 0)
                       : (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rp, (int)off, 0, 0);
  };
  auto halo_at = [&](int buf, int lev, int w, int side) -> V * {
    return s_halo + (((buf * L + lev) * WY + w) * 2 + side) * 64 + lane;
  };
  const int wu = wave > 0 ? wave - 1 : 0, wd = wave < WY - 1 ? wave + 1 : WY - 1;

  // row bytes of a slice: plain air, never updated, and the entries of the slice below; no row of a slice
  // outside 1..Z-2 is updated (the words of slices 0 and Z-1 say so)
  struct RowBits {
    uint32_t air, fixed, same;
  };
  auto row_word = [&](int k) -> uint32_t { return grows[k < 0 ? 0 : k > Z - 1 ? Z - 1 : k]; };
  auto row_bits = [&](uint32_t w) -> RowBits {
    return RowBits{w & air_mask, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu};
  };
  // the rows set in each of the n newest bytes of a history
  auto all_of = [](uint64_t h, int n) -> uint32_t {
    uint32_t v = 0xFFu;
#pragma unroll
    for (int j = 0; j < n; ++j) v &= (uint32_t)(h >> (8 * j));
    return v;
  };

  const int kb = z0 - (L - 1), ke = z1 - 1 + (L - 1);
  {
    const uint32_t rstep = (uint32_t)X * (uint32_t)sizeof(S);
    const auto r0 = a_rsrc(kb - 1), r1 = a_rsrc(kb), r2 = a_rsrc(kb + 1), rq = b_rsrc(kb);
#pragma unroll
    for (int r = 0; r < TY; ++r) {
      q[0][0][r] = R::up(R::ld(r0, vcol + r * rstep));
      q[0][1][r] = R::up(R::ld(r1, vcol + r * rstep));
    }
#pragma unroll
    for (int r = 0; r < TY; ++r) {
      pl[r] = R::ld(r2, vcol + r * rstep);
      pq[r] = R::ld(rq, vcol + r * rstep);
    }
    *halo_at((kb - 1) & 1, 0, wave, 0) = q[0][1][0];
    *halo_at((kb - 1) & 1, 0, wave, 1) = q[0][1][TY - 1];
  }
  // first event at or above the first slice of this chunk
  for (int hi = ev_end; ev < hi;) {
    const int mid = (ev + hi) >> 1;
    if (ev_head(mid).z < kb)
      ev = mid + 1;
    else
      hi = mid;
  }
  // row bytes of slices k, k-1, ...: those below the chunk count as air, fixed and unchanged (their
  // levels are not used)
  uint64_t hist = ~0ull, hist_f = ~0ull;
  uint32_t hist_u = ~0u;
  RowBits rows_k = row_bits(row_word(kb));
  uint32_t row_next = row_word(kb + 1);  // the words are loaded a slice ahead
  if ((rows_k.air | rows_k.fixed) != 0xFFu) load_pm(kb);
  // vmcnt(0): nothing may be in flight when the loop is entered. The compiler's wait for a row's
  // loads counts the accesses issued after them on whichever way into the loop has fewest, so the
  // few behind the first slice's loads would otherwise be the count on every iteration.
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();

  auto body = [&](auto cur_c, int k) __attribute__((always_inline)) {
    constexpr int cur = decltype(cur_c)::value;
    // slices prev = cur ^ 1 hold k-1 (level i: k-1-i), cur hold k (k-i)
    hist = (hist << 8) | rows_k.air;
    hist_f = (hist_f << 8) | rows_k.fixed;
    hist_u = (hist_u << 8) | rows_k.same;
    const int hb = (k - 1) & 1;
    uint32_t ev_rows = 0;  // rows with an event on one of the slices k-L+1 .. k
    if (ev < ev_end) {
      for (int n = ev; n < ev_end;) {
        const EvHead h = ev_head(n);
        if (h.z > k) break;
        if (h.z < k - (L - 1)) {
          ev = n = h.next_z;
        } else {
          ev_rows |= 1u << h.row;
          n = h.next_row;
        }
      }
    }
    // the rows that are air, fixed, of unchanged entries at every level, or have events: a byte each
    const uint32_t kinds = all_of(hist, L) | (all_of(hist_f, L) << 8) |
                           (all_of(hist_u, L - 1) << 16) | (ev_rows << 24);
    const RowBits rows_next = row_bits(row_next);
    row_next = row_word(k + 2);
    const auto ra = a_rsrc(k + 2), rb = b_rsrc(k + 1);
    const int sC = k - (L - 2), sD = k - (L - 1);
    const bool inD = sD >= z0 && sD < z1, inC = DIFF ? inD : L >= 2 && sC >= z0 && sC < z1;
    const auto rC = sw_rsrc(gC + (inC ? (size_t)(DIFF ? sD : sC) * XY : 0), inC ? sbytes : 0u);
    const auto rD = sw_rsrc(gD + (inD ? (size_t)sD * XY : 0), inD ? sbytes : 0u);
    // row offsets are formed where used: kept across the sweep they would hold 2 TY registers
    uint32_t rstep = (uint32_t)X * (uint32_t)sizeof(S);
    asm volatile("" : "+s"(rstep));
    V hu[L], hd[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
      hu[i] = *halo_at(hb, i, wu, 1);
      hd[i] = *halo_at(hb, i, wd, 0);
    }

    // One row of every level. KIND 0: plain air at all of them; 1: the table; 2: the table and
    // this row's events; 3: fixed at all of them; 4: the table, each node with one entry at all of
    // them.
    typename R::T raw_c{}, raw_d{};
    auto row = [&](auto kind, int r) __attribute__((always_inline)) {
      constexpr int KIND = decltype(kind)::value;
      constexpr bool TABLE = KIND == 1 || KIND == 2;
      // every level's entries first: the gathers then overlap the arithmetic
      uint32_t pm[L + 1];
      CE e[2][NC];
      CentredNode<C> cn[2][NC];
      auto entry_of = [&](uint32_t v, int c) { return c == 0 ? v & 0xFFFFu : v >> 16; };
      auto centred_of = [&](uint32_t v, int c) {
        const uint32_t w = entry_of(v, c);
        return centred_entry<C>(w & 0xFFu, w >> 8, s_coef, ncol, air_e);
      };
      V t[L + 1];
      t[0] = R::up(pl[r]);
      const V past0 = R::up(pq[r]);
      typename R::T d_in = pq[r], d_out{};
      auto gather = [&](int i) __attribute__((always_inline)) {
        if ((hist >> (8 * (i - 1) + r)) & 1ull)
          pm[i] = air_pm;
        else if ((hist_f >> (8 * (i - 1) + r)) & 1ull)
          pm[i] = out_pm;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if constexpr (CENTRED)
            cn[i & 1][c] = centred_of(pm[i], c);
          else
            e[i & 1][c] = s_coef[entry_of(pm[i], c)];
        }
      };
      if constexpr (TABLE) {
#pragma unroll
        for (int i = 2; i <= L; ++i)
          pm[i] = (uint32_t)s_pm[(((k - (i - 1)) & (RING - 1)) * TY + r) * 64];
        pm[1] = pmr[r];
        gather(1);
        __builtin_amdgcn_sched_barrier(0);
      }
      CE one[NC];
      if constexpr (KIND == 4) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if constexpr (CENTRED)
            cn[0][c] = centred_of(pmr[r], c);
          else
            one[c] = s_coef[entry_of(pmr[r], c)];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 1; i <= L; ++i) {
        const V zn = t[i - 1];
        const V zp = q[i - 1][cur ^ 1][r];
        const V ce = q[i - 1][cur][r];
        const V yn = r + 1 < TY ? q[i - 1][cur][r + 1 < TY ? r + 1 : r] : hd[i - 1];
        const V yp = r > 0 ? q[i - 1][cur][r > 0 ? r - 1 : r] : hu[i - 1];
        V past = i == 1 ? past0 : q[i >= 2 ? i - 2 : 0][cur ^ 1][r];
        V e_new;  // the level's difference, before rounding
        if constexpr (DIFF) {
          const V d = R::up(d_in);
#pragma unroll
          for (int c = 0; c < NC; ++c) past.v[c] = ce.v[c] - d.v[c];
        }
        const int s = k - (i - 1);
        if constexpr (TABLE) {
          if (i < L) {  // the next level's entries are in flight during this level
            gather(i + 1 <= L ? i + 1 : L);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        const bool row_ok = !((hist_f >> (8 * (i - 1) + r)) & 1ull);
        // both columns' chains side by side: one alone leaves its wave waiting on every result
        if constexpr (KIND == 3) {
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            t[i].v[c] = (C)0;
            e_new.v[c] = col_ok[c] && ((upd_rows >> r) & 1u) ? (C)0 - ce.v[c] : (C)0;
          }
        } else if constexpr (CENTRED) {
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const C xn = x_next(ce, c), xp = x_prev(ce, c);
            C v;
            if constexpr (KIND == 0) {
              v = centred_air<C>(ce.v[c], zn.v[c], zp.v[c], yn.v[c], yp.v[c], xn, xp, past.v[c], air_e,
                                 lam2);
            } else {
              v = centred_eval<C>(cn[KIND == 4 ? 0 : i & 1][c], ce.v[c], zn.v[c], zp.v[c], yn.v[c],
                                  yp.v[c], xn, xp, past.v[c], lam2);
              sw_keep(v);
              v = ((KIND == 4 || row_ok) && col_ok[c]) ? v : (C)0;
            }
            t[i].v[c] = v;
          }
        } else {
          C u[NC], m[NC], o[NC];
          auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < NC; ++c) f(c);
            if constexpr (NC > 1) __builtin_amdgcn_sched_barrier(0);
          };
          each([&](int c) { u[c] = zn.v[c] + zp.v[c]; });
          each([&](int c) { u[c] = u[c] + yn.v[c]; });
          each([&](int c) { u[c] = u[c] + yp.v[c]; });
          each([&](int c) { u[c] = u[c] + x_next(ce, c); });
          each([&](int c) { u[c] = u[c] + x_prev(ce, c); });
          if constexpr (KIND == 0) {
            each([&](int c) { m[c] = air_tk * ce.v[c]; });
            each([&](int c) { u[c] = lam2 * u[c]; });
            each([&](int c) { u[c] = m[c] + u[c]; });
            each([&](int c) { t[i].v[c] = u[c] - past.v[c]; });
            if constexpr (DIFF) each([&](int c) { e_new.v[c] = t[i].v[c] - ce.v[c]; });
          } else {
            auto entry = [&](int c) -> const CE & { return KIND == 4 ? one[c] : e[i & 1][c]; };
            each([&](int c) { m[c] = entry(c).tk * ce.v[c]; });
            each([&](int c) { u[c] = lam2 * u[c]; });
            each([&](int c) { o[c] = entry(c).omb * past.v[c]; });
            each([&](int c) { u[c] = m[c] + u[c]; });
            each([&](int c) { u[c] = u[c] - o[c]; });
            each([&](int c) {
              C v = entry(c).inv * u[c];
              sw_keep(v);
              t[i].v[c] = ((KIND == 4 || row_ok) && col_ok[c]) ? v : (C)0;
            });
            if constexpr (DIFF)
              each([&](int c) {
                C d = t[i].v[c] - ce.v[c];
                sw_keep(d);
                e_new.v[c] = col_ok[c] && (KIND == 4 || ((upd_rows >> r) & 1u)) ? d : (C)0;
              });
          }
        }
        // rounded to the storage type once: the stored bits and the value the next level reads
        typename R::T raw = R::pack(t[i]);
        if (i < L || KIND == 2) t[i] = R::up(raw);
        if constexpr (DIFF) d_out = R::pack(e_new);
        if constexpr (KIND == 2) {
          // the event arguments are re-read here, so that they hold no scalar registers across
          // the sweep
          ConstArgs ka = args;
          asm volatile("" : "+s"(ka));
          const ConstI32 gev = (ConstI32)ka->events;
          for (int n = ev; n < ev_end;) {
            const ConstI32 g = gev + kEvInts * (int64_t)n;
            const EvHead h{g[kEvZ], g[kEvRow], g[kEvNextRow], g[kEvNextZ]};
            if (h.z > s || (h.z == s && h.row > r)) break;
            if (h.z < s || h.row < r) {
              n = h.z < s ? h.next_z : h.next_row;
              continue;
            }
            ++n;
            const int xe = g[kEvX], id = g[kEvId];
            if (id < 0) {  // receiver
              const bool owned = own_x && ((own_rows >> r) & 1u) && s >= z0 && s < z1;
              const auto rr = sw_rsrc(ka->resp + (int64_t)(id & 0x7FFFFFFF) * ka->resp_steps,
                                      (uint32_t)ka->resp_steps * 8u);
#pragma unroll
              for (int c = 0; c < NC; ++c) {
                const double v = (double)t[i].v[c] * ka->inv_scale;
                __builtin_amdgcn_raw_buffer_store_b64(
                    __builtin_bit_cast(u32x2, v), rr,
                    (int)((uint32_t)(step + i - 1) * 8u | (owned && xe == x0 + c ? 0u : kDrop)), 0, 0);
              }
            } else if (step + i < ka->inject_end) {
              C smp = (C)0;
              if (step + i < ka->n_samples)
                smp = ((const __attribute__((address_space(4))) C *)ka->sig)[(int64_t)id * ka->n_samples + step + i];
              smp = smp * ka->scale;
              const bool hard = ((ConstI32)ka->src_kind)[id] == 0 || ka->soft_overwrite;
#pragma unroll
              for (int c = 0; c < NC; ++c) {
                const C v = Fmt<S>::round(hard ? smp : t[i].v[c] + smp);
                if constexpr (DIFF) {  // the difference keeps the past value
                  V d = R::up(d_out);
                  const C e = v - (t[i].v[c] - d.v[c]);
                  d.v[c] = xe == x0 + c ? e : d.v[c];
                  d_out = R::pack(d);
                }
                t[i].v[c] = xe == x0 + c ? v : t[i].v[c];
              }
            }
          }
        }
        if constexpr (KIND == 2) raw = R::pack(t[i]);
        if constexpr (DIFF) {
          if (i < L) {  // the next level's difference gives way to this one's
            d_in = qd[i < L ? i : 0][r];
            qd[i < L ? i : 0][r] = d_out;
          } else {
            raw_c = d_out;
          }
        } else {
          if (i == L - 1) raw_c = raw;
        }
        if (i == L) raw_d = raw;
      }
      if constexpr ((TABLE || KIND == 4) && L > 1) s_pm[((k & (RING - 1)) * TY + r) * 64] = (PM)pmr[r];
#pragma unroll
      for (int i = 0; i < L; ++i) q[i][cur ^ 1][r] = t[i];
    };
    // the choice is made row by row: one choice for all rows would keep every queue entry of
    // the iteration live beside its replacement
    auto rows = [&](int r) __attribute__((always_inline)) {
      if ((kinds >> (24 + r)) & 1u)
        row(std::integral_constant<int, 2>(), r);
      else if ((kinds >> r) & 1u)
        row(std::integral_constant<int, 0>(), r);
      else if ((kinds >> (8 + r)) & 1u)
        row(std::integral_constant<int, 3>(), r);
      else if ((kinds >> (16 + r)) & 1u)
        row(std::integral_constant<int, 4>(), r);
      else
        row(std::integral_constant<int, 1>(), r);
      // The accesses are the same on every way here: a wait for a row's loads counts the accesses
      // issued since on the way with fewest, and the compiler makes ways past all of the kinds.
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t drop = ((own_rows >> r) & 1u) ? 0u : kDrop;
      if (L >= 2 || DIFF) R::st(rC, sl.at(r * rstep, drop), raw_c);
      R::st(rD, sl.at(r * rstep, drop), raw_d);
      if (odd_edge) {
        if (L >= 2 || DIFF) R::st1(rC, sl.at1(r * rstep, drop), raw_c, 0);
        R::st1(rD, sl.at1(r * rstep, drop), raw_d, 0);
      }
      pl[r] = R::ld(ra, vcol + r * rstep);
      pq[r] = R::ld(rb, vcol + r * rstep);
    };
    // not a loop: its body is beyond what the compiler unrolls, and the queue would go to memory
    sw_inner_rows(std::make_integer_sequence<int, TY - 2>(), rows);
    rows(0);
    rows(TY - 1);
    // publish the edge rows of the new slices
#pragma unroll
    for (int i = 0; i < L; ++i) {
      *halo_at(hb ^ 1, i, wave, 0) = q[i][cur ^ 1][0];
      *halo_at(hb ^ 1, i, wave, 1) = q[i][cur ^ 1][TY - 1];
    }
    rows_k = rows_next;
    // entries of the slice below stay in their registers
    if ((rows_k.air | rows_k.fixed | rows_k.same) != 0xFFu) load_pm(k + 1);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  for (int k = kb;;) {
    body(std::integral_constant<int, 1>(), k);
    if (++k > ke) break;
    body(std::integral_constant<int, 0>(), k);
    if (++k > ke) break;
  }
}

// XCD-aware order: consecutive block ids are dealt round-robin to the 8 XCDs; every XCD walks a
// contiguous run of tiles.
__device__ __forceinline__ unsigned xcd_tile() {
  const unsigned total = gridDim.x, lin = blockIdx.x, full = total & ~7u;
  return lin < full ? (lin & 7u) * (full >> 3) + (lin >> 3) : lin;
}

// A context's sweep: the slots of a batch innermost, so that one XCD's L2 serves a tile's entries
// to all of them.
template <typename S, int L, int LM, int TY, int WY, int NC, int HX, int MODE>
__global__ __launch_bounds__(64 * WY, (WY + 3) / 4) void srl_sweep_kernel(SweepArgsOf<S> a) {
  const unsigned tile = xcd_tile();
  const int slot = (int)(tile % (unsigned)a.n_slots);
  const int64_t off = (int64_t)slot * a.slot_elems;
  sweep_block<S, L, LM, TY, WY, NC, HX, MODE>(
      (ConstSweepArgs<S>)__builtin_amdgcn_kernarg_segment_ptr(), tile / (unsigned)a.n_slots, slot,
      a.zc, a.A + off, a.B + off, a.Cn + off, a.Dn + off, a.step);
}

// Round `round` of a bundle for every job of a pool launch: L steps per job. A block finds its job by
// a binary search over the launch table. The state holds the step and buffers at the start of the
// bundle; rounds alternate between the two pairs of buffers.
template <typename S, int L, int LM, int TY, int WY, int NC, int HX>
__global__ __launch_bounds__(64 * WY, (WY + 3) / 4) void srl_sweep_pool_kernel(
    const SweepArgsOf<S> *__restrict__ args, const PoolJobDev *__restrict__ jobs,
    const PoolState *__restrict__ state, PoolLaunch pl, int zc, int round) {
  const int tile = (int)xcd_tile();
  int lo = 0, hi = pl.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pl.tile_end[mid] > tile)
      hi = mid;
    else
      lo = mid + 1;
  }
  const int job = pl.slot[lo];
  const PoolState st = state[job];
  const PoolJobDev &J = jobs[job];
  const int step = st.step + round * L;
  if (step >= J.n_steps) return;  // the whole block: no barrier has been reached
  int o1, o2;
  pool_spare(st.cur, st.past, o1, o2);
  const bool odd = round & 1;
  sweep_block<S, L, LM, TY, WY, NC, HX, kForward>(
      (ConstSweepArgs<S>)(args + job), (unsigned)(tile - (lo ? pl.tile_end[lo - 1] : 0)), 0, zc,
      (const S *)J.F[odd ? o2 : st.cur], (const S *)J.F[odd ? o1 : st.past],
      (S *)J.F[odd ? st.past : o1], (S *)J.F[odd ? st.cur : o2], step);
}

// Tiles of the sweep per storage type: columns per lane, rows per wave, waves, most levels, halo
// columns; and the cost model of a launch in us: T0 + slices marched (chunk + 2 (levels - 1) + 2) times
// A + B n, n <= CAP the blocks that share a CU.
//
// V = 0: eight waves at 238 (FP32) and 236 (FP64) VGPRs, two waves per SIMD and one block per CU (160 KB
// of LDS with 255 materials). V = 1: for rooms that give the large tile too few blocks or too short
// chunks. It computes 1.5 times the nodes and launches more often per step, but fills the chip with a
// third of the rows and half the columns per block, three blocks (FP64 two) to a CU. us per step, large ->
// small: 130x98x66 FP32 11.3 -> 6.9, FP16 12.1 -> 6.9, FP64 10.5 -> 8.1; 157x111x75 FP32 11.2 -> 7.9, FP64
// 11.4 -> 8.9; 200x150x120 FP32 13.2 -> 11.3, FP64 15.0 -> 12.8; 256x256x256 FP32 26.9 -> 32.9, FP64 41.5
// -> 50.0. Other small tiles, FP32 on 130x98x66: two columns and 2 rows 7.5, 3 rows 7.7.
//
// The rates are those of forward runs in FP32 and FP64. 16-bit storage, the difference form and the centred
// boundaries take them too, without rates of their own. Large -> small, us per step: FP16 256x256x256 27.5 ->
// 29.3, 448x264x135 21.6 -> 26.0, 200x150x120 12.4 -> 10.6, BF16 256x256x256 26.3 -> 29.5; difference form
// 256x256x256 34.2 -> 30.2, 320x240x200 29.0 -> 25.5, 640x480x320 124 -> 136; centred FP32 256x256x256 54.7
// -> 45.6, 448x264x135 46.4 -> 41.8, 640x480x320 201 -> 240, centred FP64 256x200x160 33.7 -> 37.6,
// 256x256x256 51.9 -> 63.4: for the last two modes the line lies up to 17 % off in the rooms between.
template <typename S, int V>
struct SweepTile {
  static constexpr int NC = 2, TY = 6, WY = 8, LM = 5, HX = 8, CAP = 1;
  static constexpr double T0 = 8, A = 4, B = 0;
};
template <>
struct SweepTile<double, 0> {
  static constexpr int NC = 1, TY = 8, WY = 8, LM = 4, HX = 4, CAP = 1;
  static constexpr double T0 = 2, A = 4.2, B = 0;
};
template <typename S>
struct SweepTile<S, 1> {
  static constexpr int NC = 1, TY = 3, WY = 8, LM = 3, HX = 4, CAP = 3;
  static constexpr double T0 = 3, A = 1.1, B = 0.5;
};
template <>
struct SweepTile<double, 1> {
  static constexpr int NC = 1, TY = 4, WY = 8, LM = 3, HX = 4, CAP = 2;
  static constexpr double T0 = 2, A = 1.6, B = 0.65;
};

template <typename S, int V, int L>
size_t sweep_lds(int ncol) {
  typedef SweepTile<S, V> T;
  typedef typename Fmt<S>::C C;
  return sizeof(typename CoefOf<C>::T) * (kStageRows * (size_t)ncol + 1) +
         sizeof(Cols<C, T::NC>) * 2 * L * T::WY * 2 * 64 +
         2 * T::NC * (size_t)T::WY * sweep_ring(L) * T::TY * 64;
}

template <typename S, int V, int L, int MODE>
hipError_t launch_levels(const SweepPlan &p, const SweepArgsOf<S> &a, hipStream_t stream) {
  typedef SweepTile<S, V> T;
  const size_t lds = sweep_lds<S, V, L>(a.ncol);
  hipLaunchKernelGGL((srl_sweep_kernel<S, L, T::LM, T::TY, T::WY, T::NC, T::HX, MODE>),
                     dim3((unsigned)p.blocks), dim3(64 * T::WY), lds, stream, a);
  return hipGetLastError();
}

template <typename S, int V, int MODE>
hipError_t launch_tile(const SweepPlan &p, const SweepArgsOf<S> &a, int levels, hipStream_t stream) {
  constexpr int LM = SweepTile<S, V>::LM;
  switch (levels) {
  case 1: return launch_levels<S, V, 1, MODE>(p, a, stream);
  case 2: return launch_levels<S, V, 2, MODE>(p, a, stream);
  case 3: return launch_levels<S, V, 3, MODE>(p, a, stream);
  case 4:
    if constexpr (LM >= 4) return launch_levels<S, V, 4, MODE>(p, a, stream);
    break;
  case 5:
    if constexpr (LM >= 5) return launch_levels<S, V, 5, MODE>(p, a, stream);
    break;
  }
  return hipErrorInvalidValue;
}

template <typename S, int MODE = kForward>
hipError_t launch_any(const SweepPlan &p, const SweepArgsOf<S> &a, int levels, hipStream_t stream) {
  return p.tile ? launch_tile<S, 1, MODE>(p, a, levels, stream)
                : launch_tile<S, 0, MODE>(p, a, levels, stream);
}

template <typename S>
hipError_t launch_pool(int tiles, const void *args, const PoolJobDev *jobs, const PoolState *st,
                       const PoolLaunch &pl, int zc, int round, hipStream_t stream) {
  typedef SweepTile<S, 0> T;
  const size_t lds = sweep_lds<S, 0, T::LM>(pl.ncol_max);
  hipLaunchKernelGGL((srl_sweep_pool_kernel<S, T::LM, T::LM, T::TY, T::WY, T::NC, T::HX>),
                     dim3((unsigned)tiles), dim3(64 * T::WY), lds, stream, (const SweepArgsOf<S> *)args, jobs, st, pl, zc, round);
  return hipGetLastError();
}

}  // namespace pfdtd
