// Fields and results of many small systems between the host and their own
// arenas in one copy each way: a batch of 512 1-gradient systems has a few KB
// per system, and a copy with its synchronisation costs 10-20 us whatever its
// size (512 systems: three copies each, 30 ms around 3 ms of solving).
// Bound by the one pageable copy; the kernels move a few MB.
#include <hip/hip_runtime.h>

#include "scf_device.h"
#include "scf_kernels.h"

namespace nscf {
namespace {

constexpr int kIoThreads = 256;

// one workgroup per system: its fields from / to packed[offset[i] ...]
__global__ void __launch_bounds__(kIoThreads) k_scatter_fields(DevSys *const *list, const size_t *offset,
                                                               const double *packed) {
  const DevSys &S = *list[blockIdx.x];
  const double *src = packed + offset[blockIdx.x];
  const int nvar = S.nit * S.M;
  for (int v = threadIdx.x; v < nvar; v += kIoThreads) S.x[v] = src[v];
}

__global__ void __launch_bounds__(kIoThreads) k_gather_fields(DevSys *const *list, const size_t *offset,
                                                              double *packed) {
  const DevSys &S = *list[blockIdx.x];
  double *dst = packed + offset[blockIdx.x];
  const int nvar = S.nit * S.M;
  for (int v = threadIdx.x; v < nvar; v += kIoThreads) dst[v] = S.x[v];
}

__global__ void __launch_bounds__(kIoThreads) k_gather_records(DevSys *const *list, int n, SolveRecord *rec) {
  const int i = blockIdx.x * kIoThreads + threadIdx.x;
  if (i >= n) return;
  const DevScalars &sc = *list[i]->sc;
  SolveRecord r;
  r.iterations = sc.iterations;
  r.status = sc.status;
  r.converged = sc.converged;
  r.fp32_iterations = sc.fp32_iterations;
  r.residual = sc.residual;
  r.t_begin = sc.t_begin;
  r.t_end = sc.t_end;
  rec[i] = r;
}

}  // namespace

hipError_t launch_scatter_fields(DevSys *const *list, int n, const size_t *offset, const double *packed,
                                 hipStream_t st) {
  hipLaunchKernelGGL(k_scatter_fields, dim3(n), dim3(kIoThreads), 0, st, list, offset, packed);
  return hipGetLastError();
}
hipError_t launch_gather_fields(DevSys *const *list, int n, const size_t *offset, double *packed, hipStream_t st) {
  hipLaunchKernelGGL(k_gather_fields, dim3(n), dim3(kIoThreads), 0, st, list, offset, packed);
  return hipGetLastError();
}
hipError_t launch_gather_records(DevSys *const *list, int n, SolveRecord *rec, hipStream_t st) {
  hipLaunchKernelGGL(k_gather_records, dim3((n + kIoThreads - 1) / kIoThreads), dim3(kIoThreads), 0, st, list, n,
                     rec);
  return hipGetLastError();
}

}  // namespace nscf
