// A stand-in for the HIP runtime in host memory (test infrastructure): "device" blocks are host blocks
// whose sizes are known, copies happen at once, and an allocation of a chosen size or total can be
// made to fail.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

namespace host_runtime {
inline std::map<const char*, size_t> blocks;  // live blocks by address
inline size_t live = 0, limit = ~size_t(0), fail_size = 0;
inline long mallocs = 0, frees = 0, syncs = 0;
inline long allowed = -1;  // allocations that still succeed (-1: all)
inline hipError_t last = hipSuccess;
// bytes from p to the end of its block, 0 if p lies in none
inline size_t room(const void* p) {
  auto it = blocks.upper_bound(static_cast<const char*>(p));
  if (!p || it == blocks.begin()) return 0;
  --it;
  const size_t off = static_cast<const char*>(p) - it->first;
  return off < it->second ? it->second - off : 0;
}
}  // namespace host_runtime

#define CHECK(cond)                                                    \
  do {                                                                 \
    if (!(cond)) {                                                     \
      std::printf("line %d: %s does not hold\n", __LINE__, #cond);     \
      std::exit(1);                                                    \
    }                                                                  \
  } while (0)

extern "C" {
inline __attribute__((used)) hipError_t stand_in_malloc(void** p, size_t n) {
  using namespace host_runtime;
  if (n == fail_size || live + n > limit || allowed == 0) return last = hipErrorOutOfMemory;
  if (allowed > 0) --allowed;
  *p = std::calloc(1, n);
  blocks[static_cast<char*>(*p)] = n;
  live += n;
  ++mallocs;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return stand_in_malloc(p, n); }
hipError_t hipFree(void* p) {
  using namespace host_runtime;
  if (!p) return hipSuccess;
  auto it = blocks.find(static_cast<char*>(p));
  CHECK(it != blocks.end());
  live -= it->second;
  blocks.erase(it);
  std::free(p);
  ++frees;
  ++syncs;  // waits for the device
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  ++host_runtime::syncs;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = host_runtime::last;
  host_runtime::last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "stand-in error"; }
}
