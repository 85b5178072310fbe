// How blocking calls end, on a machine without a GPU. This program stands in for the HIP runtime: device
// memory is the heap, copies are made at once, and of the kernels only those run that tell the host that
// a call has ended. It checks what the library asks of the runtime:
//   - a call that handed pageable memory of the caller's to an asynchronous copy synchronises with its stream
//     after it, whatever it waits for besides (the runtime may hold on to those pages until then).
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "kraken_hip.h"

// ---- the stand-in ------------------------------------------------------------------------------
struct Block {
  size_t bytes;
  bool host;
  unsigned flags;
};
// Function-local: the library registers its kernels before this file's own variables are constructed.
struct Runtime {
  std::map<const void*, std::string> kernels;
  std::map<uintptr_t, Block> blocks;
  std::map<hipStream_t, bool> pageable;             // an asynchronous copy of pageable memory since the last wait
  dim3 grid, block;
  size_t shmem = 0;
  hipStream_t stream = nullptr;
};
static Runtime& rt() {
  static Runtime r;
  return r;
}
static const Block* block_of(const void* p) {
  auto it = rt().blocks.upper_bound((uintptr_t)p);
  if (it == rt().blocks.begin()) return nullptr;
  --it;
  return (uintptr_t)p < it->first + it->second.bytes ? &it->second : nullptr;
}
static hipError_t take(void** p, size_t bytes, bool host, unsigned flags) {
  *p = aligned_alloc(4096, (bytes + 4095) & ~(size_t)4095);
  if (!*p) return hipErrorOutOfMemory;
  rt().blocks[(uintptr_t)*p] = Block{bytes, host, flags};
  return hipSuccess;
}
static hipError_t give(void* p) {
  rt().blocks.erase((uintptr_t)p);
  free(p);
  return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return take(p, bytes, false, 0); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags) { return take(p, bytes, true, flags); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { *d = p; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  const Block* b = block_of(p);
  if (!b) return hipErrorInvalidValue;
  std::memset(a, 0, sizeof(*a));
  a->type = b->host ? hipMemoryTypeHost : hipMemoryTypeDevice;
  a->devicePointer = const_cast<void*>(p);
  a->allocationFlags = b->flags;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t bytes, hipMemcpyKind) { std::memcpy(d, s, bytes); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t bytes, hipMemcpyKind, hipStream_t stream) {
  if (!block_of(d) || !block_of(s)) rt().pageable[stream] = true;
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t bytes) { std::memset(d, v, bytes); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t bytes, hipStream_t) { std::memset(d, v, bytes); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t stream) {
  rt().pageable[stream] = false;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  static uintptr_t next = 0x1000;
  *s = reinterpret_cast<hipStream_t>(next += 16);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipErrorNotSupported; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "no such thing here"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPeekAtLastError() { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)1 << 33; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return take(p, (size_t)64 << 20, false, 0); }

void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  rt().kernels[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
  rt().grid = grid;
  rt().block = block;
  rt().shmem = shmem;
  rt().stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream) {
  *grid = rt().grid;
  *block = rt().block;
  *shmem = rt().shmem;
  *stream = rt().stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  const std::string& name = rt().kernels[f];
  if (name.find("signal_kernel") != std::string::npos) {
    __atomic_store_n(*static_cast<uint32_t**>(args[0]), *static_cast<uint32_t*>(args[1]), __ATOMIC_RELEASE);
  }
  return hipSuccess;
}
}  // extern "C"

// ---- the checks --------------------------------------------------------------------------------
static int failures = 0;
#define CHECK(cond)                                                    \
  do {                                                                 \
    if (!(cond)) {                                                     \
      std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond);    \
      ++failures;                                                      \
    }                                                                  \
  } while (0)

// A blocking call that succeeds and leaves no copy of pageable memory unwaited for.
static void whole(const char* what, int32_t rc) {
  if (rc != KRK_SUCCESS) {
    std::printf("FAILED %s: %d, %s\n", what, rc, krk_last_error_string());
    ++failures;
  }
  for (const auto& s : rt().pageable) {
    if (!s.second) continue;
    std::printf("FAILED %s: returned without synchronising after a copy of the caller's pages\n", what);
    ++failures;
  }
  rt().pageable.clear();
}

// Host arrays of megabytes, which are staged by the runtime's copies, and of kilobytes, which are not.
static void dense_pages(int64_t cells) {
  krk_optim sgd;
  CHECK(krk_optim_defaults(KRK_SGD, &sgd) == 0);
  std::vector<float> vals(cells);
  std::vector<int64_t> index(cells);
  for (int64_t i = 0; i < cells; ++i) index[i] = i;
  krk_dense* d = nullptr;
  CHECK(krk_dense_create(vals.data(), cells, 0, &d) == 0);
  whole("dense push", krk_dense_push(d, &sgd, vals.data(), cells, 0.1f, 0));
  whole("dense push_coo", krk_dense_push_coo(d, &sgd, index.data(), vals.data(), cells, 0.1f, 0));
  whole("dense push_coo of a few", krk_dense_push_coo(d, &sgd, index.data(), vals.data(), cells / 10, 0.1f, 0));
  whole("dense pull", krk_dense_pull(d, vals.data(), 0));
  CHECK(krk_dense_destroy(d) == 0);
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  CHECK(krk_runtime_init(0) == 0);
  if (which == "dense") {
    dense_pages((int64_t)5 << 20);
    dense_pages(2048);
  } else {
    return 2;
  }
  if (failures == 0) std::printf("%s ok\n", which.c_str());
  return failures != 0;
}
