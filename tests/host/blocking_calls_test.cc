// How blocking calls end, on a machine without a GPU. This program stands in for the HIP runtime: device
// memory is the heap, copies are made at once, and of the kernels only those run that tell the host that
// a call has ended. It checks what the library asks of the runtime:
//   - a call that handed pageable memory of the caller's to an asynchronous copy synchronises with its stream
//     after it, whatever it waits for besides (the runtime may hold on to those pages until then);
//   - a word that a launch under way will still write belongs to the call that waits for it until that launch has
//     ended, so that no other call waits on the same word; where all words are taken calls synchronise;
//   - a thread that waits lets others of its core run, on whom the end of its work may depend;
//   - a sparse gradient in host memory of a small dense table is scattered, which reads its indices once;
//   - sparse gradients of a small dense table go tile by tile from the push on that follows one whose indices were
//     seen to ascend, and are scattered for a while after one whose indices do not;
//   - a table's first sparse gradient in pageable memory takes at most seven of the runtime's commands;
//   - a decode gives large work space back;
//   - what a launch says behind its word is believed by the call that waits on the word only if it is that call's.
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "kraken_hip.h"

// ---- the stand-in ------------------------------------------------------------------------------
struct Block {
  size_t bytes;
  bool host;
  unsigned flags;
};
struct Late {
  uint32_t* word;
  uint32_t ticket;
};
// Function-local: the library registers its kernels before this file's own variables are constructed.
struct Runtime {
  std::map<const void*, std::string> kernels;
  std::map<uintptr_t, Block> blocks;
  std::map<hipStream_t, bool> pageable;             // an asynchronous copy of pageable memory since the last wait
  std::map<hipStream_t, std::vector<Late>> late;    // words that a stream's launches will write
  std::vector<uint32_t*> words;                     // of every launch that tells the host, null where it has none
  bool signals_late = false;
  int yields_until_told = 0;                        // > 0: late words are written at the last of so many sched_yields
  int synchronised = 0;
  int commands = 0;                                 // asynchronous copies and fills, and launches
  std::vector<std::string> launched;                // names, mangled
  int fail_after = 0;                               // > 0: that many launches from here an error is reported
  uint32_t* old_word = nullptr;                     // a word that a launch of a failed call writes over the next one's
  uint32_t old_ticket = 0;
  bool unordered = false;                           // what launches find out about a sparse gradient's indices
  uint32_t rows = 0;                                // what the tables' counters say
  std::function<void()> on_synchronise;
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
static void tell(hipStream_t stream, uint32_t* word, uint32_t ticket) {
  rt().words.push_back(word);
  if (!word) return;
  if (rt().signals_late) rt().late[stream].push_back(Late{word, ticket});
  else __atomic_store_n(word, ticket, __ATOMIC_RELEASE);
}

static void write_late() {
  for (auto& s : rt().late) {
    for (const Late& l : s.second) __atomic_store_n(l.word, l.ticket, __ATOMIC_RELEASE);
    s.second.clear();
  }
}

extern "C" {
int sched_yield() {
  if (rt().yields_until_told > 0 && --rt().yields_until_told == 0) write_late();
  return 0;
}
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
  rt().commands++;
  if (!block_of(d) || !block_of(s)) rt().pageable[stream] = true;
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t bytes) { std::memset(d, v, bytes); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t bytes, hipStream_t) {
  rt().commands++;
  std::memset(d, v, bytes);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t stream) {
  rt().synchronised++;
  if (rt().on_synchronise) rt().on_synchronise();
  for (const Late& l : rt().late[stream]) __atomic_store_n(l.word, l.ticket, __ATOMIC_RELEASE);
  rt().late[stream].clear();
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
hipError_t hipGetLastError() { return rt().fail_after > 0 && --rt().fail_after == 0 ? hipErrorUnknown : hipSuccess; }
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
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t stream) {
  const std::string& name = rt().kernels[f];
  rt().launched.push_back(name);
  rt().commands++;
  if (name.find("signal_unordered_kernel") != std::string::npos) {
    uint32_t* word = *static_cast<uint32_t**>(args[0]);
    const uint32_t ticket = *static_cast<uint32_t*>(args[1]);
    if (rt().fail_after > 0) {                        // a launch of a call that will fail: it ends during the next one
      rt().old_word = word;
      rt().old_ticket = ticket;
    } else {
      word[1] = rt().unordered ? 0u : ticket;
      tell(stream, word, ticket);
      if (rt().old_word) {
        if (rt().old_word != word) std::abort();
        word[1] = word[0] = rt().old_ticket;          // (that push's indices ascended)
        rt().old_word = nullptr;
      }
    }
  } else if (name.find("coo_update_kernel") != std::string::npos || name.find("coo_bits_update_kernel") != std::string::npos) {
    struct Tiles {   // CooTiles of krk_internal.h
      void *starts, *unordered;
      uint32_t tag, tiles;
      void* bits;
      uint32_t *told, ticket;
    };
    const Tiles& a = *static_cast<const Tiles*>(args[name.find("coo_bits") != std::string::npos ? 2 : 3]);
    if (a.told) *a.told = rt().unordered ? 0u : a.ticket;
  } else if (name.find("signal_kernel") != std::string::npos) {
    tell(stream, *static_cast<uint32_t**>(args[0]), *static_cast<uint32_t*>(args[1]));
  } else if (name.find("counters_kernel") != std::string::npos) {
    struct Counters {   // CountersArgs of sparse_table.hip
      int32_t n;
      uint32_t* word;
      uint32_t ticket;
      const uint32_t* counters[32];
      uint32_t* host[32];
    };
    const Counters& a = *static_cast<const Counters*>(args[0]);
    for (int i = 0; i < a.n; ++i) {
      std::memset(a.host[i], 0, 16);
      a.host[i][0] = rt().rows;
    }
    tell(stream, a.word, a.ticket);
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

static krk_sparse* make_table(int64_t dim) {
  krk_init init;
  krk_sparse* t = nullptr;
  CHECK(krk_init_defaults(KRK_INIT_CONSTANT, &init) == 0);
  CHECK(krk_sparse_create(dim, &init, 1000, &t) == 0);
  return t;
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

static void sparse_pages(int64_t n) {
  const int64_t dim = 8;
  krk_optim sgd;
  CHECK(krk_optim_defaults(KRK_SGD, &sgd) == 0);
  sgd.has_momentum = 1;
  sgd.momentum = 0.9f;
  std::vector<uint64_t> ids(n);
  std::vector<float> rows(n * dim), state(n * dim);
  std::vector<int32_t> at(n);
  std::vector<int64_t> steps(n), offsets(n + 1);
  std::vector<uint8_t> found(n);
  std::vector<float> wire(2 * (size_t)krk_wire_rows_bytes(n, dim) / 4 + 16);
  for (int64_t i = 0; i < n; ++i) ids[i] = 3 * (uint64_t)i + 1, offsets[i + 1] = i + 1;

  void* locked = nullptr;
  CHECK(krk_host_malloc(&locked, n * 8) == 0);
  std::memcpy(locked, ids.data(), n * 8);

  krk_sparse* t = make_table(dim);
  whole("pull", krk_sparse_pull(t, ids.data(), n, rows.data(), 0));
  whole("push", krk_sparse_push(t, &sgd, ids.data(), n, rows.data(), dim, 0.1f, 0));
  whole("push_raw", krk_sparse_push_raw(t, &sgd, ids.data(), n, rows.data(), dim, 0.1f, 0));
  whole("pull_pooled", krk_sparse_pull_pooled(t, ids.data(), n, offsets.data(), n, nullptr, KRK_POOL_SUM, 0.0f,
                                              rows.data(), 0));
  whole("pull_wire", krk_sparse_pull_wire(t, ids.data(), n, wire.data()));
  whole("lookup", krk_sparse_lookup(t, ids.data(), n, at.data(), 0));
  whole("lookup of page-locked ids", krk_sparse_lookup(t, static_cast<uint64_t*>(locked), n, at.data(), 0));
  whole("fetch by page-locked ids", krk_sparse_fetch(t, static_cast<uint64_t*>(locked), n, nullptr, rows.data(), 1, nullptr,
                                                     nullptr, 0));
  whole("import", krk_sparse_import(t, ids.data(), n, rows.data(), 0));
  whole("import_state", krk_sparse_import_state(t, ids.data(), n, KRK_ST_MOMENTUM_BUFFER, state.data(), steps.data(), 0));
  whole("fetch", krk_sparse_fetch(t, ids.data(), n, found.data(), rows.data(), KRK_ST_MOMENTUM_BUFFER, state.data(),
                                  steps.data(), 0));
  whole("fetch of what is there", krk_sparse_fetch(t, ids.data(), n, found.data(), nullptr, 1, nullptr, nullptr, 0));
  int64_t exported = 0;
  rt().rows = (uint32_t)n;
  whole("export", krk_sparse_export(t, ids.data(), rows.data(), KRK_ST_MOMENTUM_BUFFER, state.data(), steps.data(), n,
                                    &exported, 0));
  CHECK(exported == n);
  whole("export of ids", krk_sparse_export(t, ids.data(), nullptr, 1, nullptr, nullptr, n, &exported, 0));
  whole("export of values", krk_sparse_export(t, nullptr, rows.data(), 1, nullptr, nullptr, n, &exported, 0));
  rt().rows = 0;
  CHECK(krk_sparse_destroy(t) == 0);
  CHECK(krk_host_free(locked) == 0);

  krk_sparse* members[2] = {make_table(dim), make_table(dim)};
  krk_group* g = nullptr;
  CHECK(krk_group_create(members, 2, &g) == 0);
  const int64_t parts[3] = {0, n / 3, n};
  whole("group pull", krk_group_pull(g, ids.data(), parts, rows.data(), 0));
  whole("group push", krk_group_push(g, &sgd, ids.data(), parts, rows.data(), dim, 0.1f, 0));
  CHECK(krk_group_destroy(g) == 0);
  for (krk_sparse* m : members) CHECK(krk_sparse_destroy(m) == 0);

}

// After a call that had to synchronise the next ones wait for their word again.
static void words_after_pages() {
  const int64_t n = 50000;
  std::vector<uint64_t> ids(n);
  std::vector<float> rows(n * 8);
  krk_sparse* t = make_table(8);
  whole("pull", krk_sparse_pull(t, ids.data(), n, rows.data(), 0));
  rt().words.clear();
  rt().synchronised = 0;
  whole("pull", krk_sparse_pull(t, ids.data(), 10, rows.data(), 0));
  CHECK(rt().synchronised == 0 && rt().words.size() == 1 && rt().words[0] != nullptr);
  // page-locked memory that is not known to be coherent is read after a synchronise, memory that is is not
  for (const unsigned flags : {(unsigned)hipHostMallocDefault, (unsigned)hipHostMallocCoherent}) {
    void* out = nullptr;
    CHECK(hipHostMalloc(&out, 10 * 8 * 4, flags) == hipSuccess);
    rt().synchronised = 0;
    whole("pull", krk_sparse_pull(t, ids.data(), 10, static_cast<float*>(out), 0));
    CHECK((rt().synchronised != 0) == (flags == hipHostMallocDefault));
    CHECK(hipHostFree(out) == hipSuccess);
  }
  CHECK(krk_sparse_destroy(t) == 0);
}

// Calls whose launches end late, each begun while the one before it synchronises: 64 words, then none.
static void late_words() {
  constexpr int kWords = 64, kCalls = kWords + 2;
  std::vector<krk_sparse*> tables;
  for (int i = 0; i < kCalls; ++i) tables.push_back(make_table(8));
  uint64_t id = 7;
  std::vector<float> row(8);
  rt().words.clear();
  rt().signals_late = true;
  int depth = 0;
  rt().on_synchronise = [&]() {
    if (depth + 1 >= kCalls) return;
    ++depth;
    CHECK(krk_sparse_pull(tables[depth], &id, 1, row.data(), 0) == KRK_SUCCESS);
  };
  CHECK(krk_sparse_pull(tables[0], &id, 1, row.data(), 0) == KRK_SUCCESS);
  rt().on_synchronise = nullptr;
  rt().signals_late = false;
  CHECK((int)rt().words.size() == kCalls);
  std::set<uint32_t*> different(rt().words.begin(), rt().words.end());
  CHECK((int)different.size() == kWords + 1 && different.count(nullptr) == 1);
  // all of them are free again
  rt().words.clear();
  rt().synchronised = 0;
  for (krk_sparse* t : tables) CHECK(krk_sparse_pull(t, &id, 1, row.data(), 0) == KRK_SUCCESS);
  CHECK(rt().synchronised == 0);
  for (krk_sparse* t : tables) CHECK(krk_sparse_destroy(t) == 0);
}

// The word is written once the waiting thread has let others of its core run a few times.
static void one_core() {
  krk_sparse* t = make_table(8);
  uint64_t id = 7;
  std::vector<float> row(8);
  rt().signals_late = true;
  rt().synchronised = 0;
  constexpr int kCalls = 40;
  for (int i = 0; i < kCalls; ++i) {
    rt().yields_until_told = 5;
    CHECK(krk_sparse_pull(t, &id, 1, row.data(), 0) == KRK_SUCCESS);
  }
  rt().signals_late = false;
  rt().yields_until_told = 0;
  if (rt().synchronised > kCalls / 4) {
    std::printf("FAILED: %d of %d calls looked for as long as they may\n", rt().synchronised, kCalls);
    ++failures;
  }
  CHECK(krk_sparse_destroy(t) == 0);
}

// How many of the launches since the last look were of kernels of this name.
static int launches(const char* name) {
  int n = 0;
  for (const std::string& l : rt().launched) n += l.find(name) != std::string::npos;
  return n;
}

// Sparse gradients of tables below 2^22 elements: page-locked arrays of any size and pageable ones that pass through
// page-locked buffers (up to 1 MB) are filled and scattered, each of many pushes.
static void sparse_gradients_in_host_memory() {
  krk_optim sgd;
  CHECK(krk_optim_defaults(KRK_SGD, &sgd) == 0);
  for (const int64_t cells : {(int64_t)300, (int64_t)300000, ((int64_t)1 << 22) - 1}) {
    for (const bool locked : {true, false}) {
      const int64_t nnz = locked ? cells / 2 : std::min<int64_t>(cells / 2, 1 << 17);
      std::vector<float> vals(cells);
      std::vector<int64_t> index(nnz);
      for (int64_t i = 0; i < nnz; ++i) index[i] = i;
      void *l_index = nullptr, *l_vals = nullptr;
      CHECK(krk_host_malloc(&l_index, nnz * 8) == 0 && krk_host_malloc(&l_vals, nnz * 4) == 0);
      std::memcpy(l_index, index.data(), nnz * 8);
      krk_dense* d = nullptr;
      CHECK(krk_dense_create(vals.data(), cells, 0, &d) == 0);
      rt().launched.clear();
      for (int push = 0; push < 3; ++push)
        whole("push_coo", krk_dense_push_coo(d, &sgd, locked ? static_cast<int64_t*>(l_index) : index.data(),
                                             locked ? static_cast<float*>(l_vals) : vals.data(), nnz, 0.1f, 0));
      CHECK(launches("coo_add_kernel") == 3 && launches("dense_update_kernel") == 3);
      CHECK(launches("coo_tiles_bounds_kernel") == 0 && launches("coo_bits_kernel") == 0);
      CHECK(krk_dense_destroy(d) == 0);
      CHECK(krk_host_free(l_index) == 0 && krk_host_free(l_vals) == 0);
    }
  }
}

// Sparse gradients in pageable memory that is staged by copies. unordered: large ones are scattered behind the tiles.
static void first_sparse_gradient() {
  krk_optim adam;
  CHECK(krk_optim_defaults(KRK_ADAM, &adam) == 0);
  for (const int64_t cells : {(int64_t)2000000, (int64_t)5000000}) {
    std::vector<float> vals(cells);
    std::vector<int64_t> index(cells / 2);
    for (int64_t i = 0; i < cells / 2; ++i) index[i] = i;
    for (const bool unordered : {false, true}) {
      rt().unordered = unordered;
      krk_dense* d = nullptr;
      CHECK(krk_dense_create(vals.data(), cells, 0, &d) == 0);
      rt().launched.clear();
      rt().commands = 0;
      whole("push_coo", krk_dense_push_coo(d, &adam, index.data(), vals.data(), cells / 2, 0.1f, 0));
      CHECK(rt().commands <= (unordered && cells > 4200000 ? 10 : 7));
      CHECK(launches("coo_add_kernel") == (cells < 4200000 || unordered));
      CHECK(krk_dense_destroy(d) == 0);
    }
  }
}

// How many of n pushes of a gradient in device memory went tile by tile, and how many were scattered.
struct Ways {
  int tiles, scattered;
  bool operator==(const Ways& o) const { return tiles == o.tiles && scattered == o.scattered; }
};
static Ways push_in_device_memory(krk_dense* d, bool unordered, int n, int64_t nnz = 100) {
  static void *index = nullptr, *vals = nullptr;
  if (!index) CHECK(krk_malloc(&index, 8 * 100000) == 0 && krk_malloc(&vals, 4 * 100000) == 0);
  krk_optim sgd;
  CHECK(krk_optim_defaults(KRK_SGD, &sgd) == 0);
  rt().launched.clear();
  rt().unordered = unordered;
  for (int push = 0; push < n; ++push)
    whole("push_coo", krk_dense_push_coo(d, &sgd, static_cast<int64_t*>(index), static_cast<float*>(vals), nnz, 0.1f,
                                         KRK_DEVICE_PTRS));
  CHECK(launches("coo_tiles_bounds_kernel") == launches("coo_update_kernel"));
  return Ways{launches("coo_tiles_bounds_kernel"), launches("coo_add_kernel")};
}

static void order_of_sparse_gradients() {
  std::vector<float> vals(50000);
  krk_dense* d = nullptr;
  CHECK(krk_dense_create(vals.data(), (int64_t)vals.size(), 0, &d) == 0);
  rt().commands = 0;
  CHECK((push_in_device_memory(d, true, 1) == Ways{0, 1}));
  CHECK(rt().commands == 4);                        // fill, scatter, update, word
  CHECK((push_in_device_memory(d, true, 257) == Ways{0, 257}));   // never a look at the tiles
  CHECK((push_in_device_memory(d, false, 257) == Ways{0, 257}));  // some of them spared, then one that is looked at
  CHECK((push_in_device_memory(d, false, 300) == Ways{300, 0}));
  CHECK((push_in_device_memory(d, false, 1, 60000) == Ways{0, 1}));   // more entries than elements
  CHECK((push_in_device_memory(d, false, 3) == Ways{3, 0}));
  CHECK((push_in_device_memory(d, true, 1) == Ways{1, 1}));       // seen too late
  CHECK((push_in_device_memory(d, true, 300) == Ways{0, 300}));
  CHECK(krk_dense_destroy(d) == 0);
  CHECK(krk_dense_create(vals.data(), (int64_t)vals.size(), 0, &d) == 0);
  CHECK((push_in_device_memory(d, false, 5) == Ways{4, 1}));
  CHECK(krk_dense_destroy(d) == 0);
}

// A push that fails behind its last launch, and one of a shuffled gradient that gets the same word: the launch of the
// first ends behind that of the second.
static void word_of_a_failed_push() {
  const int64_t cells = (int64_t)1 << 22;
  std::vector<float> vals(cells);
  krk_dense* d[2] = {};
  for (krk_dense*& t : d) CHECK(krk_dense_create(vals.data(), cells, 0, &t) == 0);
  CHECK((push_in_device_memory(d[1], false, 1) == Ways{1, 0}));
  void *index = nullptr, *values = nullptr;
  CHECK(krk_malloc(&index, 800) == 0 && krk_malloc(&values, 400) == 0);
  krk_optim sgd;
  CHECK(krk_optim_defaults(KRK_SGD, &sgd) == 0);
  rt().fail_after = 3;                              // behind the launches of the tiles, the update and the word
  CHECK(krk_dense_push_coo(d[0], &sgd, static_cast<int64_t*>(index), static_cast<float*>(values), 100, 0.1f,
                           KRK_DEVICE_PTRS) != KRK_SUCCESS);
  CHECK(rt().fail_after == 0 && rt().old_word != nullptr);
  CHECK((push_in_device_memory(d[1], true, 1) == Ways{1, 1}));
  CHECK(rt().old_word == nullptr);
  for (krk_dense* t : d) CHECK(krk_dense_destroy(t) == 0);
}

// Decodes of few entries read the indices twice, whatever the tensor's size. A decode belongs to no object: what it
// keeps on the device afterwards is bounded.
static void work_space_of_decodes() {
  void* place = nullptr;                            // (no kernel runs: an address is enough)
  CHECK(krk_malloc(&place, 4096) == 0);
  const auto held = []() {
    size_t bytes = 0;
    for (const auto& b : rt().blocks) bytes += b.second.bytes;
    return bytes;
  };
  const size_t before = held();
  for (const int64_t n : {(int64_t)1 << 22, (int64_t)12 << 20, (int64_t)1 << 26}) {
    CHECK(krk_coo_to_dense(static_cast<int64_t*>(place), static_cast<float*>(place), (int64_t)3 << 19,
                           static_cast<float*>(place), n, KRK_DEVICE_PTRS) == KRK_SUCCESS);
    CHECK(launches("coo_bits_kernel") == 0 && launches("coo_tiles_write_kernel") == 1);
    rt().launched.clear();
  }
  for (const int64_t n : {(int64_t)1 << 23, (int64_t)1 << 31, (int64_t)5 << 30, (int64_t)1 << 23}) {
    CHECK(krk_coo_to_dense(static_cast<int64_t*>(place), static_cast<float*>(place), n / 4, static_cast<float*>(place), n,
                           KRK_DEVICE_PTRS) == KRK_SUCCESS);
    CHECK(launches("coo_bits_write_kernel") == 1 && launches("coo_tiles_write_kernel") == 0);
    rt().launched.clear();
    CHECK(held() - before <= ((size_t)256 << 20) + ((size_t)16 << 20));
  }
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  CHECK(krk_runtime_init(0) == 0);
  if (which == "dense") {
    dense_pages((int64_t)5 << 20);
    dense_pages(2048);
  } else if (which == "sparse") {
    sparse_pages(300000);
    sparse_pages(512);
    words_after_pages();
  } else if (which == "words") {
    late_words();
  } else if (which == "core") {
    one_core();
  } else if (which == "host_gradients") {
    sparse_gradients_in_host_memory();
  } else if (which == "gradients_order") {
    order_of_sparse_gradients();
  } else if (which == "old_words") {
    word_of_a_failed_push();
  } else if (which == "first_gradient") {
    first_sparse_gradient();
  } else if (which == "decodes") {
    work_space_of_decodes();
  } else {
    return 2;
  }
  if (failures == 0) std::printf("%s ok\n", which.c_str());
  return failures != 0;
}
