// A HIP runtime without a device, preloaded into a CPU test's process: memory
// is host memory, kernels do not run (but for the columns' domains, which the
// host path waits for, and the packing of a real operator's slices), launches
// are recorded, allocations can be made to fail.  For the host code of the
// library: what it launches, and what a plan
// holds after an error.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
struct Launch {
  char name[96];
  uint64_t arg0[64];      // the first argument's bytes
  uint64_t arg1, arg2;    // the next two (8 bytes each), k_blk_operators only
};
std::vector<Launch> launches;
int fail_in = 0;
size_t limit = 0;
dim3 call_grid, call_block;

void domains(void** a, dim3 grid) {   // k_col_domain(n, ld, psi, label, clo, chi, dom)
  const int64_t n = *(int64_t*)a[0], ld = *(int64_t*)a[1];
  const double* psi = *(const double**)a[2];
  const int32_t *label = *(const int32_t**)a[3], *clo = *(const int32_t**)a[4], *chi = *(const int32_t**)a[5];
  int32_t* dom = *(int32_t**)a[6];
  for (unsigned b = 0; b < grid.y; ++b) {
    dom[2 * b] = (int32_t)n;
    dom[2 * b + 1] = 0;
    for (int64_t i = 0; i < n; ++i)
      if (psi[2 * (b * ld + i)] != 0.0 || psi[2 * (b * ld + i) + 1] != 0.0) {
        dom[2 * b] = std::min(dom[2 * b], clo[label[i]]);
        dom[2 * b + 1] = std::max(dom[2 * b + 1], chi[label[i]]);
      }
  }
}
void pack(void** a, dim3 grid) {   // k_slice_pack(sslice, soff, rp, ccol, cval, nnz, nf, np, real, scol, sval, sval32)
  const int32_t* sl = *(const int32_t**)a[0];
  const int64_t *soff = *(const int64_t**)a[1], *rp = *(const int64_t**)a[2];
  const int32_t* ccol = *(const int32_t**)a[3];
  const double* cval = *(const double**)a[4];
  const int64_t nnz = *(int64_t*)a[5], np = *(int64_t*)a[7];
  const int32_t nf = *(int32_t*)a[6];
  uint32_t* scol = *(uint32_t**)a[9];
  double* sval = *(double**)a[10];
  if (!*(int32_t*)a[8]) abort();
  for (unsigned i = 0; i < grid.x; ++i, sl += 4)
    for (int32_t l = 0; l < sl[1]; ++l)
      for (int32_t j = 0; j < 2 * sl[2]; ++j) {
        const int64_t e = rp[sl[0] + l] + j, at = soff[i] + 64 * (int64_t)(j / 2) + l;
        const bool in = e < rp[sl[0] + l + 1];
        scol[at] |= (uint32_t)(((in ? ccol[e] : sl[0] + l) - sl[3]) * 16) << (16 * (j & 1));
        for (int32_t s = 0; s < nf; ++s) sval[2 * (s * np + at) + (j & 1)] = in ? cval[2 * (s * nnz + e)] : 0.0;
      }
}
hipError_t launch(const void* f, dim3 grid, void** args) {
  const std::string& nm = names()[f];
  Launch l;
  memset(&l, 0, sizeof(l));
  strncpy(l.name, nm.c_str(), sizeof(l.name) - 1);
  memcpy(l.arg0, args[0], sizeof(l.arg0));
  if (nm.find("k_blk_operators") != std::string::npos) {
    l.arg1 = *(uint64_t*)args[1];
    l.arg2 = *(uint64_t*)args[2];
  }
  launches.push_back(l);
  if (nm.find("k_col_domain") != std::string::npos) domains(args, grid);
  if (nm.find("k_slice_pack") != std::string::npos) pack(args, grid);
  return hipSuccess;
}
}  // namespace

extern "C" {
void stub_fail_in(int n) { fail_in = n; }          // the n-th device allocation from now fails (0: none)
void stub_limit(size_t bytes) { limit = bytes; }   // larger device allocations fail (0: none)
void stub_clear() { launches.clear(); }
int stub_count() { return (int)launches.size(); }
const Launch* stub_launch(int i) { return &launches[(size_t)i]; }

void** __hipRegisterFatBinary(const void*) {
  static void* p;
  return &p;
}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
  call_grid = g;
  call_block = b;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = call_grid;
  *b = call_block;
  *lds = 0;
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t, hipStream_t) { return launch(f, g, args); }
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3, void** args, unsigned, hipStream_t) {
  return launch(f, g, args);
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if ((fail_in > 0 && --fail_in == 0) || (limit && n > limit)) return hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n ? n : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
  memset(a, 0, sizeof(*a));
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* v = calloc(1, (size_t)64 << 20);
  *p = v;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  free((void*)s);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)calloc(1, 8);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
  free((void*)e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}
