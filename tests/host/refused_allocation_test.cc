// A push of up to 2^20 ids takes work space for the sums of rows that many positions share, and is sorted
// where that cannot be had. This program stands between the library and hipMalloc and refuses what
// is larger than a limit: the push has the same result, and the next one, with the room, too. A decode of
// many entries keeps a bit an element, and reads the indices twice where it has no room for them.
#include <dlfcn.h>

#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "kraken_hip.h"

static size_t limit = SIZE_MAX;
static int refused = 0;

extern "C" int hipMalloc(void** p, size_t bytes) {
  using Malloc = int (*)(void**, size_t);
  static const Malloc real = reinterpret_cast<Malloc>(dlsym(RTLD_NEXT, "hipMalloc"));
  if (bytes > limit) {
    ++refused;
    return 2;   // hipErrorOutOfMemory
  }
  return real(p, bytes);
}

#define CHECK(cond)                                                    \
  do {                                                                 \
    if (!(cond)) {                                                     \
      std::printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #cond);    \
      return 1;                                                        \
    }                                                                  \
  } while (0)

int main() {
  const int64_t n = 70000, rows = 9000, dim = 64;
  std::vector<uint64_t> ids(n), names(rows);
  std::vector<float> grads(n * dim), got(rows * dim);
  std::vector<double> sums(rows * dim, 0.0);
  for (int64_t r = 0; r < rows; ++r) names[r] = 1000003ull * (uint64_t)r + 7;
  uint32_t x = 1;
  for (int64_t p = 0; p < n; ++p) {
    x = x * 1664525u + 1013904223u;
    const int64_t r = p % 3 == 0 ? 5 : (int64_t)(x >> 8) % rows;   // a third of the positions are one row's
    ids[p] = names[r];
    for (int64_t c = 0; c < dim; ++c) {
      const float g = (float)((int)((p * 7 + c * 3) % 129) - 64) / 4096.0f;   // every sum is exact
      grads[p * dim + c] = g;
      sums[r * dim + c] += g;
    }
  }
  krk_init init;
  krk_optim sgd;
  CHECK(krk_init_defaults(KRK_INIT_CONSTANT, &init) == 0 && krk_optim_defaults(KRK_SGD, &sgd) == 0);
  krk_sparse* t = nullptr;
  CHECK(krk_sparse_create(dim, &init, 20000, &t) == 0);
  void *d_ids = nullptr, *d_grads = nullptr;
  CHECK(krk_malloc(&d_ids, n * 8) == 0 && krk_malloc(&d_grads, n * dim * 4) == 0);
  CHECK(krk_memcpy_h2d(d_ids, ids.data(), n * 8) == 0 && krk_memcpy_h2d(d_grads, grads.data(), n * dim * 4) == 0);
  CHECK(krk_sparse_pull(t, names.data(), rows, got.data(), 0) == 0);
  const std::vector<float> before = got;
  for (int pass = 1; pass <= 3; ++pass) {
    // the sums' room is n / 4 rows, 4.5 MB; nothing else of the push is larger than 1.1 MB
    limit = pass == 3 ? SIZE_MAX : (size_t)2 << 20;
    refused = 0;
    CHECK(krk_sparse_push_raw(t, &sgd, static_cast<uint64_t*>(d_ids), n, static_cast<float*>(d_grads), dim, 0.5f,
                              KRK_DEVICE_PTRS) == 0);
    CHECK(refused == (pass == 3 ? 0 : 1));
    limit = SIZE_MAX;
    CHECK(krk_sparse_pull(t, names.data(), rows, got.data(), 0) == 0);
    for (int64_t i = 0; i < rows * dim; ++i) CHECK(got[i] == before[i] - (float)(0.5 * sums[i] * pass));
  }
  CHECK(krk_sparse_destroy(t) == 0);

  const int64_t len = (int64_t)1 << 23, nnz = len / 2;   // a megabyte of bits, 16 KB of everything else
  std::vector<int64_t> idx(nnz);
  std::vector<float> val(nnz), dense(len), want(len, 0.0f);
  for (int64_t j = 0; j < nnz; ++j) {
    idx[j] = 2 * j + (j * 7 % 5 == 0);
    val[j] = want[idx[j]] = (float)(j % 1000 + 1);
  }
  void *d_idx = nullptr, *d_val = nullptr, *d_dense = nullptr;
  CHECK(krk_malloc(&d_idx, nnz * 8) == 0 && krk_malloc(&d_val, nnz * 4) == 0 && krk_malloc(&d_dense, len * 4) == 0);
  CHECK(krk_memcpy_h2d(d_idx, idx.data(), nnz * 8) == 0 && krk_memcpy_h2d(d_val, val.data(), nnz * 4) == 0);
  for (int pass = 1; pass <= 2; ++pass) {
    limit = pass == 2 ? SIZE_MAX : (size_t)512 << 10;
    refused = 0;
    CHECK(krk_coo_to_dense(static_cast<int64_t*>(d_idx), static_cast<float*>(d_val), nnz, static_cast<float*>(d_dense),
                           len, KRK_DEVICE_PTRS) == 0);
    CHECK(refused == (pass == 2 ? 0 : 1));
    limit = SIZE_MAX;
    CHECK(krk_memcpy_d2h(dense.data(), d_dense, len * 4) == 0);
    CHECK(dense == want);
  }
  std::printf("refused allocation ok\n");
  return 0;
}
