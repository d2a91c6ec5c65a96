// A stand-in for the HIP runtime and for the kernel launchers (kernels.hpp,
// harmonic.hpp), so that the host code of a handle, a batch and a server runs
// on the CPU: device memory is address space with a limit, launches count
// themselves and check the buffers they are given, and an allocation inside a
// stream capture is refused and counted, as the runtime refuses it.
#pragma once

#include "harmonic.hpp"
#include "kernels.hpp"

#include <sys/mman.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>

namespace fake {

struct State {
  std::map<const char *, size_t> mem;  // allocations
  size_t used = 0, peak = 0, limit = SIZE_MAX;
  int capturing = 0;
  long refused_in_capture = 0, failures = 0, allocations = 0;
  // launches since reset(): expanded and direct far fields, shell sums by path
  long harm = 0, direct = 0, global = 0, steps = 0;
  size_t filled = 0;  // doubles of the largest fill
  void reset() { harm = direct = global = steps = filled = 0; }
};
inline State st;

inline void require(const void *p, size_t bytes, const char *what) {
  const char *c = static_cast<const char *>(p);
  auto it = st.mem.upper_bound(c);
  if (it != st.mem.begin()) {
    --it;
    if (c + bytes <= it->first + it->second) return;
  }
  std::printf("FAIL %s: %zu bytes at %p are not in one allocation\n", what,
              bytes, p);
  ++st.failures;
}

}  // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  using fake::st;
  if (st.capturing) {
    ++st.refused_in_capture;
    return hipErrorStreamCaptureUnsupported;
  }
  if (n > st.limit || st.used > st.limit - n) return hipErrorOutOfMemory;
  void *a = mmap(nullptr, n, PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (a == MAP_FAILED) return hipErrorOutOfMemory;
  st.mem[static_cast<const char *>(a)] = n;
  st.used += n;
  ++st.allocations;
  st.peak = st.used > st.peak ? st.used : st.peak;
  *p = a;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  using fake::st;
  auto it = st.mem.find(static_cast<const char *>(p));
  if (it == st.mem.end()) {
    ++st.failures;
    return hipErrorInvalidValue;
  }
  munmap(p, it->second);
  st.used -= it->second;
  st.mem.erase(it);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  fake::require(d, n, "hipMemcpy");
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k,
                          hipStream_t) {
  return k == hipMemcpyHostToDevice ? hipMemcpy(d, s, n, k) : hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 160 * 1024;  // LDS of a workgroup
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new char);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete reinterpret_cast<char *>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(new char);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<char *>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  ++fake::st.capturing;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  --fake::st.capturing;
  *g = reinterpret_cast<hipGraph_t>(new char);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *,
                               char *, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(new char);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<char *>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete reinterpret_cast<char *>(e);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = ::operator new(n);
  std::memset(*p, 0, n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  ::operator delete(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return hipSuccess;
}
}

namespace glst {
namespace dev {
void prepare_kernels(size_t) {}
void fill_u32(uint32_t *, uint32_t, size_t, hipStream_t) {}
void fill_f64(double *p, double, size_t n, hipStream_t) {
  if (n) fake::require(p, n * 8, "fill_f64");
  fake::st.filled = std::max(fake::st.filled, n);
}
void bin_chunks(bool, const double *, const double *, const double *, uint32_t,
                double, const GridShape &, uint32_t *, uint32_t *, uint32_t *,
                hipStream_t) { ++fake::st.steps; }
void hist_offsets(uint32_t *, uint32_t, uint32_t, uint32_t *, hipStream_t) {}
void cell_scan(const uint32_t *, uint32_t, uint32_t *, uint32_t *, hipStream_t,
               uint32_t *, uint2 *, uint32_t) {}
void bin_scatter(bool, const double *, const double *, const double *,
                 const double *, uint32_t, const uint32_t *, const uint32_t *,
                 const uint32_t *, const uint32_t *, const GridShape &,
                 uint32_t *, uint32_t *, double4 *, float4 *, float,
                 hipStream_t, const uint32_t *, uint2 *) {}
void sf(bool, const void *, const uint32_t *, const uint32_t *,
        const double4 *, const LrTaskArgs &, const SfGroup *, size_t, uint32_t,
        const GridShape &, void *, hipStream_t, const float *) {
  ++fake::st.direct;
}
bool rmt_lds(bool, uint32_t tmax, const void *, const double4 *,
             const uint32_t *, const uint32_t *, const uint32_t *, uint32_t,
             const GridShape &g, size_t lds, void *, hipStream_t, uint32_t,
             uint32_t, bool) {
  return rmt_nodes_per_group(g.nx, g.ny, g.nz, lds, tmax) > 0;
}
bool rmt_mfma(const void *, const double4 *, const uint32_t *,
              const uint32_t *, const uint32_t *, uint32_t, const GridShape &g,
              size_t lds, void *, hipStream_t, uint32_t, uint32_t, bool nm) {
  return rmt_mfma_nodes(g, lds, nm) > 0;
}
bool rmt_wave(const void *, const double4 *, const uint32_t *,
              const uint32_t *, const uint32_t *, uint32_t, const GridShape &g,
              void *, hipStream_t, uint32_t, uint32_t, bool) {
  return rmt_wave_fits(g);
}
void rmt_global(bool, const void *, double2 *G, const double4 *,
                const uint32_t *, const uint32_t *, const uint32_t *,
                uint32_t Kp, const GridShape &g, void *, hipStream_t, bool) {
  fake::require(G, static_cast<size_t>(g.ncell) * Kp * 16, "rmt_global");
  ++fake::st.global;
}
void lr(bool, const void *, const uint32_t *, const LrTaskArgs &,
        const LrGroup *, size_t, const void *, uint32_t, uint32_t n,
        uint32_t nsplit, double4 *partial, hipStream_t, const uint2 *,
        uint32_t) {
  fake::require(partial, static_cast<size_t>(n) * nsplit * 32, "lr");
}
uint32_t atom_groups_max(uint32_t n, uint32_t ncell) {
  return (n / 32 + ncell + 255) / 256 * 256;
}
void lr_reduce(const double4 *, uint32_t, uint32_t, const double4 *, double *,
               double *, double *, double *, hipStream_t) {}
void sr(bool, const double4 *, const uint32_t *, const GridShape &, double *,
        double *, double *, double *, double4 *, hipStream_t) {}
void unpermute(const uint32_t *, uint32_t, const double *, const double *,
               const double *, const double *, double *, double *, double *,
               double *, hipStream_t) {}
void bin_chunks_batch(bool, const double *, const double *, const double *,
                      const SysDev *, const BatchLaunch &, uint32_t *,
                      uint32_t *, uint32_t *, hipStream_t) { ++fake::st.steps; }
void hist_offsets_batch(uint32_t *, const SysDev *, const BatchLaunch &,
                        uint32_t *, hipStream_t) {}
void cell_scan_batch(const uint32_t *, const SysDev *, uint32_t, uint32_t *,
                     uint32_t *, hipStream_t, uint32_t *, uint2 *) {}
void bin_scatter_batch(bool, const double *, const double *, const double *,
                       const double *, const SysDev *, const BatchLaunch &,
                       const uint32_t *, const uint32_t *, const uint32_t *,
                       const uint32_t *, uint32_t *, uint32_t *, double4 *,
                       float4 *, hipStream_t, const uint32_t *, uint2 *) {}
void sf_batch(bool, const void *, const uint32_t *, const uint32_t *,
              const double4 *, const LrTaskArgs &, const SysDev *,
              const std::vector<BatchLaunch> &L, void *, hipStream_t,
              const float *, const uint32_t *) {
  for (const BatchLaunch &l : L) fake::st.direct += l.nblk > 0;
}
void rmt_batch(bool, const void *, const double4 *, const uint32_t *,
               const uint32_t *, const uint32_t *, const SysDev *,
               const BatchLaunch &, size_t, void *, hipStream_t) {}
void rmt_wave_batch(const void *, const double4 *, const uint32_t *,
                    const uint32_t *, const uint32_t *, const SysDev *,
                    const BatchLaunch &, void *, hipStream_t) {}
void lr_batch(bool, const void *, const uint32_t *, const LrTaskArgs &,
              const SysDev *, const std::vector<BatchLaunch> &, const void *,
              double4 *, hipStream_t, const uint2 *) {}
void lr_reduce_batch(const double4 *, const SysDev *, const BatchLaunch &,
                     const double4 *, double *, double *, double *, double *,
                     hipStream_t) {}
void sr_batch(bool, const double4 *, const uint32_t *, const SysDev *,
              const BatchLaunch &, double *, double *, double *, double *,
              double4 *, hipStream_t) {}
void sf_all_batch(const void *, const uint32_t *, const uint32_t *,
                  const LrTaskArgs &, const SysDev *, const BatchLaunch &,
                  void *, hipStream_t) { ++fake::st.direct; }
void lr_all_batch(const void *, const uint32_t *, const LrTaskArgs &,
                  const SysDev *, const BatchLaunch &, const void *, double4 *,
                  hipStream_t, const uint2 *) {}
size_t fused_lds_bytes(size_t n) { return n; }
uint32_t fused_workgroups(size_t, int) { return 256; }
long long wall_clock_rate() { return 100000; }
void step_fused(const FusedStep &, uint32_t, size_t, hipStream_t, int) {
  ++fake::st.direct;
}
void copy_runs(const CopyRun *, uint32_t, uint32_t, hipStream_t) {}
CoulombPlan coulomb_plan(uint32_t, size_t) { return {}; }
double4 *coulomb_scratch() { return nullptr; }
void coulomb_direct(const double *, const double *, const double *,
                    const double *, uint32_t, const CoulombPlan &, double4 *,
                    double *, double *, double *, double *, hipStream_t) {}

template <typename T>
size_t harm_lds_moments(uint32_t, uint32_t) { return 0; }
template <typename T>
size_t harm_lds_sf(uint32_t, uint32_t) { return 0; }
template <typename T>
size_t harm_lds_lr(uint32_t, uint32_t, uint32_t) { return 0; }
inline size_t tiles(const GridShape &g) {
  return (g.ncell + kHarmCells - 1) / kHarmCells;
}
template <typename T>
void harm_moments(const HarmPlanDev &, const HarmDev<T> &H, const void *,
                  const uint32_t *, const GridShape &g, T *mom, T *coef,
                  uint32_t *outside, hipStream_t) {
  ++fake::st.harm;
  fake::require(coef, tiles(g) * kHarmCells * H.stride * sizeof(T), "coef");
  fake::require(mom, static_cast<size_t>(g.ncell) *
                         std::max(H.rows * 16, H.ustride) * sizeof(T), "mom");
  fake::require(outside, g.ncell * 4, "outside");
}
template <typename T>
void harm_sf(const HarmPlanDev &P, const HarmDev<T> &, const void *,
             const uint32_t *, const double4 *, const GridShape &, const T *,
             const uint32_t *, T *, hipStream_t) {
  fake::require(P.unit, P.nunit * sizeof(uint2), "unit");
}
template <typename T>
void harm_lr(const HarmPlanDev &, const HarmDev<T> &, const GridShape &,
             const T *, T *, T *, hipStream_t) {}
template <typename T>
void harm_eval(const HarmPlanDev &, const HarmDev<T> &, const void *,
               const uint32_t *, const double4 *k64, uint32_t K,
               const GridShape &g, const T *, const T *R, const uint32_t *,
               T *, double4 *, hipStream_t) {
  fake::require(k64, K * sizeof(double4), "k64");
  fake::require(R, static_cast<size_t>(harm_row(g.ncell)) * K * 2 * sizeof(T),
                "R");
}
#define FAKE_HARM(T)                                                          \
  template size_t harm_lds_moments<T>(uint32_t, uint32_t);                    \
  template size_t harm_lds_sf<T>(uint32_t, uint32_t);                         \
  template size_t harm_lds_lr<T>(uint32_t, uint32_t, uint32_t);               \
  template void harm_moments<T>(const HarmPlanDev &, const HarmDev<T> &,      \
                                const void *, const uint32_t *,               \
                                const GridShape &, T *, T *, uint32_t *,      \
                                hipStream_t);                                 \
  template void harm_sf<T>(const HarmPlanDev &, const HarmDev<T> &,           \
                           const void *, const uint32_t *, const double4 *,   \
                           const GridShape &, const T *, const uint32_t *,    \
                           T *, hipStream_t);                                 \
  template void harm_lr<T>(const HarmPlanDev &, const HarmDev<T> &,           \
                           const GridShape &, const T *, T *, T *,            \
                           hipStream_t);                                      \
  template void harm_eval<T>(const HarmPlanDev &, const HarmDev<T> &,         \
                             const void *, const uint32_t *, const double4 *, \
                             uint32_t, const GridShape &, const T *,          \
                             const T *, const uint32_t *, T *, double4 *,     \
                             hipStream_t);
FAKE_HARM(float)
FAKE_HARM(double)
#undef FAKE_HARM
}  // namespace dev
}  // namespace glst
