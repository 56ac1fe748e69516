// fake_hip.cpp -- a stand-in for the HIP runtime, for tests of the library's host code without a GPU.
//
// Device memory is host memory with accounting (a budget, and the n-th allocation from now made to
// fail); copies and fills happen at once; kernels do not run. Every launch is logged with its kernel's
// name and grid; the launches of the several-level sweep also with the buffers they name, and whether
// those are live and long enough.
#include "pfdtd_internal.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

using namespace pfdtd;

namespace {

struct State {
  std::map<const void *, std::string> kernels;
  std::map<uintptr_t, size_t> live;  // allocations: address, bytes
  std::map<uintptr_t, std::string> built;  // row-bit buffers: the tile they were last built for
  size_t used = 0, budget = (size_t)1 << 40;
  int fail_in = -1;
  std::vector<std::string> log;
};
State &st() {
  static State s;
  return s;
}

struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
thread_local std::vector<Call> g_calls;

// Bytes from p to the end of its allocation, 0 when p is in none.
size_t room(const void *p) {
  auto it = st().live.upper_bound((uintptr_t)p);
  if (it == st().live.begin()) return 0;
  --it;
  const uintptr_t end = it->first + it->second;
  return (uintptr_t)p < end ? end - (uintptr_t)p : 0;
}

std::string num(long long v) { return std::to_string(v); }

// The text between `<` and `>` of a demangled-like kernel name is not at hand: the mangled one carries
// the template's integers as Li<n>E in order.
std::vector<int> ints_of(const std::string &mangled) {
  std::vector<int> v;
  for (size_t i = 0; (i = mangled.find("Li", i)) != std::string::npos; i += 2)
    v.push_back(std::atoi(mangled.c_str() + i + 2));
  return v;
}

template <typename A>
std::string sweep_line(const A &a, const std::vector<int> &t, unsigned blocks) {
  // t: L, LM, TY, WY, NC, HX, MODE
  const int TY = t[2], WY = t[3], NC = t[4], HX = t[5], LM = t[1];
  const int W = 64 * NC, OX = W - 2 * HX, OY = WY * TY - 2 * LM;
  const size_t tiles = (size_t)a.nbx * a.nby * WY;
  std::string bad;
  auto need = [&](const char *what, const void *p, size_t bytes) {
    if (room(p) < bytes) bad += std::string(" ") + what;
  };
  need("entries", a.pm, 2 * (size_t)a.pitch * a.Y * a.Z);
  need("row_bits", a.row_bits, 4 * tiles * a.Z);
  need("ev_ptr", a.ev_ptr, 4 * (tiles * a.n_slots + 1));
  if (room(a.ev_ptr) >= 4 * (tiles * a.n_slots + 1))
    need("events", a.events, sizeof(int32_t) * kEvInts * (size_t)a.ev_ptr[tiles * a.n_slots]);
  const size_t field = (size_t)a.slot_elems * a.n_slots * sizeof(*a.A);
  for (const void *f : {(const void *)a.A, (const void *)a.B, (const void *)a.Cn, (const void *)a.Dn})
    need("field", f, field);
  if (a.nbx != (a.X + OX - 1) / OX || a.nby != (a.Y + OY - 1) / OY) bad += " tiles";
  if ((long long)blocks != (long long)a.nbx * a.nby * ((a.Z - 2 + a.zc - 1) / a.zc) * a.n_slots) bad += " grid";
  auto it = st().built.find((uintptr_t)a.row_bits);
  const std::string key = num(OX) + "," + num(HX) + "," + num(OY) + "," + num(TY);
  if (it == st().built.end() || it->second != key) bad += " row_bits_of_another_tile";
  return " levels=" + num(t[0]) + " tile=" + key + " slots=" + num(a.n_slots) +
         " bad=" + (bad.empty() ? "none" : bad.substr(1));
}

void log_launch(const std::string &name, dim3 g, void **args) {
  std::string line = name;
  if (name.find("16srl_sweep_kernelI") != std::string::npos) {
    const auto t = ints_of(name);
    if (name.find("kernelId") != std::string::npos)
      line = "sweep f64" + sweep_line(*(const SweepArgs<double, CoefD, double> *)args[0], t, g.x);
    else if (name.find("kernelIf") != std::string::npos)
      line = "sweep f32" + sweep_line(*(const SweepArgs<float, CoefF, float> *)args[0], t, g.x);
    else
      line = "sweep 16bit" + sweep_line(*(const SweepArgs<h16, CoefF, float> *)args[0], t, g.x);
  } else if (name.find("15row_bits_kernel") != std::string::npos) {
    // (pm, pitch, out, X, Y, Z, nbx, ox, hx, oy, lm, wy, ty, ncol, centred)
    auto i = [&](int k) { return *(const int *)args[k]; };
    uint32_t *out = *(uint32_t **)args[2];
    st().built[(uintptr_t)out] = num(i(7)) + "," + num(i(8)) + "," + num(i(9)) + "," + num(i(12));
    line = "row_bits bad=" + std::string(room(out) < 4 * (size_t)g.x * i(11) * ((i(4) + i(9) - 1) / i(9)) * i(5)
                                             ? "out" : "none");
  } else if (name.find("21srl_sweep_pool_kernel") != std::string::npos) {
    // (args, jobs, state, launch, zc, round): blocks per job against the rooms they are for
    const auto *a = *(const SweepArgs<float, CoefF, float> **)args[0];
    const PoolLaunch &pl = *(const PoolLaunch *)args[3];
    const int zc = *(const int *)args[4];
    line = "pool_sweep jobs=" + num(pl.n);
    std::string bad;
    for (int k = 0; k < pl.n; ++k) {
      const auto &j = a[pl.slot[k]];
      const int got = pl.tile_end[k] - (k ? pl.tile_end[k - 1] : 0);
      if (got != j.nbx * j.nby * ((j.Z - 2 + zc - 1) / zc)) bad += " " + num(j.X) + "x" + num(j.Y) + "x" + num(j.Z);
    }
    line += " bad=" + (bad.empty() ? "none" : bad.substr(1));
  }
  st().log.push_back(line);
}

}  // namespace

extern "C" {

// ---- the test's controls
void fake_fail_malloc(int n) { st().fail_in = n; }  // the n-th allocation from now (0: the next), -1: none
void fake_budget(size_t bytes) { st().budget = bytes; }
size_t fake_used() { return st().used; }
void fake_clear_log() { st().log.clear(); }
int fake_log_lines() { return (int)st().log.size(); }
const char *fake_log_line(int i) { return st().log[(size_t)i].c_str(); }

// ---- the runtime
void **__hipRegisterFatBinary(const void *) {
  static void *h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  st().kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  g_calls.push_back(Call{g, b, lds, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  const Call c = g_calls.back();
  g_calls.pop_back();
  *g = c.grid;
  *b = c.block;
  *lds = c.lds;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, hipStream_t) {
  log_launch(st().kernels[f], g, args);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  *p = nullptr;
  if (st().fail_in == 0 || st().used + n > st().budget) {
    if (st().fail_in == 0) st().fail_in = -1;
    return hipErrorOutOfMemory;
  }
  if (st().fail_in > 0) --st().fail_in;
  *p = std::calloc(n ? n : 1, 1);
  st().live[(uintptr_t)*p] = n;
  st().used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = st().live.find((uintptr_t)p);
  if (it == st().live.end()) return hipSuccess;
  st().used -= it->second;
  st().live.erase(it);
  st().built.erase((uintptr_t)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = st().budget - st().used;
  *t = st().budget;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error of the stand-in runtime"; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char symbol[256];
  *p = symbol;
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) {
  *s = (hipStream_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free((void *)s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free((void *)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  std::free((void *)g);
  return hipSuccess;
}
hipError_t hipGraphInstantiateWithFlags(hipGraphExec_t *e, hipGraph_t, unsigned long long) {
  *e = (hipGraphExec_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  std::free((void *)e);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

}  // extern "C"
