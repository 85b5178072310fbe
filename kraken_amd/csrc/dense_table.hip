// Dense table: one parameter vector in HBM with its optimizer state, updated by a single fused
// pass per push. Replaces DenseTable::Pull / ::Push (ps/dense_table.cc:31-43), the whole-tensor
// Optim::Update chains (ps/optim/*.cc) and COO densification (t/coo_tensor_impl.cc:250-260,
// t/math.cc:1006-1046).
#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>
#include <vector>

#include "krk_internal.h"

struct krk_dense_group;

struct krk_dense : krk::ObjBase {
  int64_t n = 0;
  float* w = nullptr;
  float* state[KRK_ST_COUNT] = {};   // created on first use, zero filled
  float* coo_grad = nullptr;         // densified COO gradient
  krk::CooWork coo_work;             // work space of the tiled densify
  bool coo_ascends = false;          // small tables: the last blocking sparse push that was looked at had ascending indices
  int coo_plain = 0;                 // and how many will be scattered without a look (kCooPlainPushes)
  int64_t steps = 0;                 // Adam's kSteps (one counter for the whole tensor)
  bool sgd_started = false;          // momentum buffer exists (first update copies the gradient)
  hipStream_t own_stream = nullptr;  // the stream created with the table (a group lends its own)
  krk_dense_group* member_of = nullptr;
  float** group_state = nullptr;     // where the group's descriptor of this table keeps `state` (device)
};

namespace krk {
struct DenseDesc;
struct DenseBlock;
}

// The dense tables of one combined request: they share one stream, and one launch serves all.
struct krk_dense_group : krk::ObjBase {
  std::vector<krk_dense*> tables;
  std::vector<int64_t> start;        // where each member begins in the concatenated arrays
  std::vector<uint32_t> block_start; // the members' workgroups of a launch over all of them, and their number
  krk::DenseDesc* descs = nullptr;   // device: a descriptor per member
  const krk::DenseBlock* blocks = nullptr;   // behind them: one per workgroup
  int64_t total = 0;
  hipStream_t own_stream = nullptr;
};

namespace krk {

constexpr int kDenseBlock = 256;

// The gradient passes once: it is read with a non-temporal load. Parameters and moments keep
// ordinary accesses, so a small table stays in L2 from step to step (for a large one the hint was
// measured to change nothing).
typedef float dfloat4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ dfloat4 dense_load(const float* p, int64_t i) {
  return reinterpret_cast<const dfloat4*>(p)[i];
}
__device__ __forceinline__ void dense_store(float* p, int64_t i, dfloat4 v) {
  reinterpret_cast<dfloat4*>(p)[i] = v;
}

template <int OPT>
__global__ __launch_bounds__(kDenseBlock) void dense_update_kernel(
    float* __restrict__ w, float* __restrict__ s0, float* __restrict__ s1, float* __restrict__ s2,
    const float* __restrict__ grad, int64_t n, float lr, OptimK k, bool first, float bc1, float bc2, CooTiles unless) {
  if (unless.unordered && !coo_unordered(unless)) return;   // the gradient was applied tile by tile
  const int64_t n4 = n >> 2;
  const int64_t stride = (int64_t)gridDim.x * kDenseBlock;
  const dfloat4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t i = (int64_t)blockIdx.x * kDenseBlock + threadIdx.x; i < n4; i += stride) {
    const dfloat4 g4 = __builtin_nontemporal_load(reinterpret_cast<const dfloat4*>(grad) + i);
    const dfloat4 w4 = dense_load(w, i);
    const dfloat4 a4 = s0 ? dense_load(s0, i) : zero;
    const dfloat4 b4 = s1 ? dense_load(s1, i) : zero;
    const dfloat4 c4 = s2 ? dense_load(s2, i) : zero;
    float ww[4], a[4], b[4], c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ww[j] = w4[j]; a[j] = a4[j]; b[j] = b4[j]; c[j] = c4[j];
      optim_element<OPT>(k, lr, g4[j], ww[j], a[j], b[j], c[j], first, bc1, bc2);
    }
    dense_store(w, i, (dfloat4){ww[0], ww[1], ww[2], ww[3]});
    if (s0) dense_store(s0, i, (dfloat4){a[0], a[1], a[2], a[3]});
    if (s1) dense_store(s1, i, (dfloat4){b[0], b[1], b[2], b[3]});
    if (s2) dense_store(s2, i, (dfloat4){c[0], c[1], c[2], c[3]});
  }
  // tail (n not a multiple of 4)
  for (int64_t i = (n4 << 2) + (int64_t)blockIdx.x * kDenseBlock + threadIdx.x; i < n; i += stride) {
    float g = grad[i], ww = w[i];
    float a = s0 ? s0[i] : 0.0f, b = s1 ? s1[i] : 0.0f, c = s2 ? s2[i] : 0.0f;
    optim_element<OPT>(k, lr, g, ww, a, b, c, first, bc1, bc2);
    w[i] = ww;
    if (s0) s0[i] = a;
    if (s1) s1[i] = b;
    if (s2) s2[i] = c;
  }
}

static CooTiles no_tiles() { return CooTiles{}; }

static unsigned dense_grid(int64_t n) {
  int64_t blocks = (n / 4 + kDenseBlock - 1) / kDenseBlock;
  if (blocks < 1) blocks = 1;
  // Two workgroups per compute unit, grid-stride beyond that: seven streams (four read, three
  // written) through 512 workgroups run at 5.4 TB/s, through 256 or 4096 at 4.7-4.9.
  if (blocks > 512) blocks = 512;
  return (unsigned)blocks;
}

// State columns that were created, to be entered in the descriptors of a group (in the order of its stream).
// A launch takes many: the first push of 40 tables under Adam creates 80.
constexpr int kEntries = 200;
struct StateEntries {
  float** at[kEntries];
  float* value[kEntries];
};
static_assert(sizeof(StateEntries) + 16 <= 4096, "the arguments of one launch");
__global__ void enter_states_kernel(StateEntries e, int n) {
  const int i = threadIdx.x;
  if (i < n && e.at[i]) *e.at[i] = e.value[i];
}
// Columns on their way: a table has one when it is zeroed and, for a member of a group, entered.
struct StateList {
  hipStream_t stream = nullptr;
  int n = 0;
  bool grouped = false;
  krk_dense* table[kEntries];
  int state[kEntries];
  StateEntries e;
  ~StateList() {
    for (int i = 0; i < n; ++i) (void)hipFree(e.value[i]);   // given up on the way
  }
  int32_t add(krk_dense* t, int st) {
    if (n == kEntries) KRK_TRY(flush());
    DeviceGuard guard;
    KRK_HIP(hipMalloc(&guard.p, (size_t)t->n * sizeof(float)));
    KRK_HIP(hipMemsetAsync(guard.p, 0, (size_t)t->n * sizeof(float), t->stream));
    table[n] = t;
    state[n] = st;
    e.at[n] = t->group_state ? t->group_state + st : nullptr;
    e.value[n++] = guard.release<float>();
    grouped = grouped || t->group_state;
    return KRK_SUCCESS;
  }
  int32_t flush() {
    if (grouped) {   // (the members' stream is the group's)
      hipLaunchKernelGGL(enter_states_kernel, dim3(1), dim3(256), 0, stream, e, n);
      KRK_HIP(hipGetLastError());
    }
    for (int i = 0; i < n; ++i) table[i]->state[state[i]] = e.value[i];
    n = 0;
    grouped = false;
    return KRK_SUCCESS;
  }
};

// The states an optimizer's three slots stand for (krk_internal.h), -1 = unused.
static void dense_slots(const krk_optim& o, int32_t st[3]) {
  st[0] = st[1] = st[2] = -1;
  switch (o.type) {
    case KRK_SGD:
      if (o.has_momentum) st[0] = KRK_ST_MOMENTUM_BUFFER;
      break;
    case KRK_ADAGRAD:
      st[0] = KRK_ST_STATE_SUM;
      break;
    case KRK_ADAM:
      st[0] = KRK_ST_FIRST_MOMENT;
      st[1] = KRK_ST_SECOND_MOMENT;
      if (o.amsgrad) st[2] = KRK_ST_SECOND_MOMENT_MAX;
      break;
    default:
      st[0] = KRK_ST_SQUARE_AVERAGE;
      if (o.centered) st[1] = KRK_ST_G_AVE;
      if (o.has_momentum) st[2] = KRK_ST_MOMENTUM_BUFFER;
      break;
  }
}

// Creates the columns of the states st (-1: none) that n tables of one stream, those with elements, lack.
static int32_t ensure_states(krk_dense* const* tables, size_t n, const int32_t* st, int n_st, hipStream_t stream) {
  StateList list;
  list.stream = stream;
  for (size_t i = 0; i < n; ++i)
    for (int k = 0; k < n_st; ++k)
      if (st[k] >= 0 && tables[i]->n > 0 && !tables[i]->state[st[k]]) KRK_TRY(list.add(tables[i], st[k]));
  return list.n > 0 ? list.flush() : KRK_SUCCESS;
}

// Adam's bias corrections of a step (ps/optim/adam.cc:61-64) and SGD's first momentum update.
struct DenseStep {
  float bc1, bc2;
  bool first;        // SGD with momentum: the buffer does not exist yet
};

// The host's bookkeeping of one Optim::Update of table t: Adam's counter advanced, SGD's first momentum
// step noted. last: the step of a table before, whose powers serve this one if the counts are the same.
struct StepMemo {
  int64_t steps = -1;
  float bc1 = 1.0f, bc2 = 1.0f;
};
static DenseStep dense_step(krk_dense* t, const krk_optim& o, StepMemo* last) {
  DenseStep s{1.0f, 1.0f, false};
  if (o.type == KRK_SGD && o.has_momentum) {
    s.first = !t->sgd_started;
    t->sgd_started = true;
  } else if (o.type == KRK_ADAM) {
    const int64_t steps = ++t->steps;
    if (steps != last->steps) {
      last->steps = steps;
      last->bc1 = (float)(1.0 - (double)std::pow(o.beta1, (float)steps));
      last->bc2 = (float)(1.0 - (double)std::pow(o.beta2, (float)steps));
    }
    s.bc1 = last->bc1;
    s.bc2 = last->bc2;
  }
  return s;
}

// What an update of one table reads and writes.
struct DenseMember {
  float* w;
  float* s0;
  float* s1;
  float* s2;
  int64_t n;
  DenseStep step;
};

static int32_t dense_member(krk_dense* t, const krk_optim& o, DenseMember* m) {
  int32_t st[3];
  dense_slots(o, st);
  KRK_TRY(ensure_states(&t, 1, st, 3, t->stream));
  StepMemo none;
  const auto column = [&](int i) { return st[i] >= 0 ? t->state[st[i]] : nullptr; };
  *m = DenseMember{t->w, column(0), column(1), column(2), t->n, dense_step(t, o, &none)};
  return KRK_SUCCESS;
}

// launch(std::integral_constant<int, OPT>) with the optimizer's type as a constant
template <typename Launch>
static void with_optim(int32_t type, Launch launch) {
  switch (type) {
    case KRK_SGD: launch(std::integral_constant<int, KRK_SGD>()); break;
    case KRK_ADAGRAD: launch(std::integral_constant<int, KRK_ADAGRAD>()); break;
    case KRK_ADAM: launch(std::integral_constant<int, KRK_ADAM>()); break;
    default: launch(std::integral_constant<int, KRK_RMSPROP>()); break;
  }
}

// One Optim::Update on the whole tensor with a device-resident gradient.
static int32_t dense_apply(krk_dense* t, const krk_optim& o, const float* d_grad, float lr) {
  DenseMember m;
  KRK_TRY(dense_member(t, o, &m));
  const OptimK k = make_optim_k(o);
  with_optim(o.type, [&](auto opt) {
    hipLaunchKernelGGL((dense_update_kernel<opt.value>), dim3(dense_grid(t->n)), dim3(kDenseBlock), 0, t->stream, m.w,
                       m.s0, m.s1, m.s2, d_grad, t->n, lr, k, m.step.first, m.step.bc1, m.step.bc2, no_tiles());
  });
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

// ---- a sparse gradient applied tile by tile --------------------------------------------------
// The gradient of a tile is put together in LDS and applied from there, so it never exists in memory
// (a densified copy costs a write and a read of n floats: 107 of 430 us for 67 million elements).
// The tile's parameters and moments do not depend on the entries: they are requested first.
constexpr int kCooPer = kCooTile / 4 / kDenseBlock;   // 16-byte pieces of a tile a lane updates

__device__ __forceinline__ bool tiles_no_help(const CooTiles& tiles) {
  const bool unordered = coo_unordered(tiles);
  if (tiles.told && blockIdx.x == 0 && threadIdx.x == 0) *tiles.told = unordered ? 0u : tiles.ticket;
  return unordered;
}

template <int OPT>
__global__ __launch_bounds__(kDenseBlock) void coo_update_kernel(DenseMember m, const long long* __restrict__ idx,
                                                                 const float* __restrict__ val, CooTiles tiles,
                                                                 float lr, OptimK k) {
  if (tiles_no_help(tiles)) return;              // the launches that follow do the work
  __shared__ __align__(16) float grad[kCooTile];
  const dfloat4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t tile = blockIdx.x; tile < tiles.tiles; tile += gridDim.x) {
    const int64_t base = (int64_t)tile * kCooTile;
    const int64_t start = tiles.starts[tile], end = tiles.starts[tile + 1];
    const bool whole = base + kCooTile <= m.n;   // uniform
    dfloat4 w4[kCooPer], a4[kCooPer], b4[kCooPer], c4[kCooPer];
    if (whole) {
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) {
        const int64_t q = base / 4 + i * kDenseBlock + threadIdx.x;
        w4[i] = dense_load(m.w, q);
        a4[i] = m.s0 ? dense_load(m.s0, q) : zero;
        b4[i] = m.s1 ? dense_load(m.s1, q) : zero;
        c4[i] = m.s2 ? dense_load(m.s2, q) : zero;
      }
    }
#pragma unroll
    for (int i = 0; i < kCooPer; ++i) reinterpret_cast<dfloat4*>(grad)[i * kDenseBlock + threadIdx.x] = zero;
    __syncthreads();
    for (int64_t j0 = start + threadIdx.x; j0 < end; j0 += 4 * kDenseBlock) {
      long long at[4];
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t j = j0 + u * kDenseBlock;
        if (j < end) {
          at[u] = __builtin_nontemporal_load(idx + j);
          v[u] = __builtin_nontemporal_load(val + j);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j0 + u * kDenseBlock < end) grad[at[u] - base] = v[u];
    }
    __syncthreads();
    if (whole) {
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) {
        const int64_t q = base / 4 + i * kDenseBlock + threadIdx.x;
        const dfloat4 g4 = reinterpret_cast<const dfloat4*>(grad)[i * kDenseBlock + threadIdx.x];
        float ww[4], a[4], b[4], c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ww[j] = w4[i][j]; a[j] = a4[i][j]; b[j] = b4[i][j]; c[j] = c4[i][j];
          optim_element<OPT>(k, lr, g4[j], ww[j], a[j], b[j], c[j], m.step.first, m.step.bc1, m.step.bc2);
        }
        dense_store(m.w, q, (dfloat4){ww[0], ww[1], ww[2], ww[3]});
        if (m.s0) dense_store(m.s0, q, (dfloat4){a[0], a[1], a[2], a[3]});
        if (m.s1) dense_store(m.s1, q, (dfloat4){b[0], b[1], b[2], b[3]});
        if (m.s2) dense_store(m.s2, q, (dfloat4){c[0], c[1], c[2], c[3]});
      }
    } else {
      for (int64_t i = base + threadIdx.x; i < m.n; i += kDenseBlock) {
        float ww = m.w[i];
        float a = m.s0 ? m.s0[i] : 0.0f, b = m.s1 ? m.s1[i] : 0.0f, c = m.s2 ? m.s2[i] : 0.0f;
        optim_element<OPT>(k, lr, grad[i - base], ww, a, b, c, m.step.first, m.step.bc1, m.step.bc2);
        m.w[i] = ww;
        if (m.s0) m.s0[i] = a;
        if (m.s1) m.s1[i] = b;
        if (m.s2) m.s2[i] = c;
      }
    }
    __syncthreads();                             // the next tile clears the gradient
  }
}

// The same from the tile's bits: a wavefront's lanes see for themselves which entries are theirs, so nothing passes
// through LDS, no wavefront waits for another, and the indices are not read again: 1.75 GB in place of 2.0 for 67
// million elements under Adam with 33 million entries, 317 us (5.5 TB/s) in place of 365. Values that are read past
// the caches, as the other kernel does, are asked for several times by neighbours: 329.
template <int OPT>
__global__ __launch_bounds__(kDenseBlock) void coo_bits_update_kernel(DenseMember m, const float* __restrict__ val,
                                                                      CooTiles tiles, float lr, OptimK k) {
  if (tiles_no_help(tiles)) return;              // the launches that follow do the work
  const dfloat4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int lane = threadIdx.x & 63;
  uint32_t start = tiles.starts[blockIdx.x], end = tiles.starts[blockIdx.x + 1];   // (no workgroup without a tile)
  uint32_t word = tiles.bits[(size_t)blockIdx.x * (kCooTile / 32) + lane];
  for (uint32_t t = blockIdx.x; t < tiles.tiles; t += gridDim.x) {
    const int64_t base = (int64_t)t * kCooTile;
    const bool whole = base + kCooTile <= m.n;   // uniform
    dfloat4 w4[kCooPer], a4[kCooPer], b4[kCooPer], c4[kCooPer];
    if (whole) {
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) {
        const int64_t q = base / 4 + i * kDenseBlock + threadIdx.x;
        w4[i] = dense_load(m.w, q);
        a4[i] = m.s0 ? dense_load(m.s0, q) : zero;
        b4[i] = m.s1 ? dense_load(m.s1, q) : zero;
        c4[i] = m.s2 ? dense_load(m.s2, q) : zero;
      }
    }
    const CooTileBits tile(word);
    float g[kCooPer][4] = {};
    if (end > start) {                           // uniform
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) tile.quad(i * kDenseBlock + threadIdx.x, val, start, end, g[i]);
    }
    // the next tile's bits are there when its turn comes
    const uint32_t next = min(t + gridDim.x, tiles.tiles - 1u);
    start = tiles.starts[next];
    end = tiles.starts[next + 1];
    word = tiles.bits[(size_t)next * (kCooTile / 32) + lane];
    if (whole) {
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) {
        const int64_t q = base / 4 + i * kDenseBlock + threadIdx.x;
        float ww[4], a[4], b[4], c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ww[j] = w4[i][j]; a[j] = a4[i][j]; b[j] = b4[i][j]; c[j] = c4[i][j];
          optim_element<OPT>(k, lr, g[i][j], ww[j], a[j], b[j], c[j], m.step.first, m.step.bc1, m.step.bc2);
        }
        dense_store(m.w, q, (dfloat4){ww[0], ww[1], ww[2], ww[3]});
        if (m.s0) dense_store(m.s0, q, (dfloat4){a[0], a[1], a[2], a[3]});
        if (m.s1) dense_store(m.s1, q, (dfloat4){b[0], b[1], b[2], b[3]});
        if (m.s2) dense_store(m.s2, q, (dfloat4){c[0], c[1], c[2], c[3]});
      }
    } else {
#pragma unroll
      for (int i = 0; i < kCooPer; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t at = base + 4 * (i * kDenseBlock + threadIdx.x) + j;
          if (at >= m.n) continue;
          float ww = m.w[at];
          float a = m.s0 ? m.s0[at] : 0.0f, b = m.s1 ? m.s1[at] : 0.0f, c = m.s2 ? m.s2[at] : 0.0f;
          optim_element<OPT>(k, lr, g[i][j], ww, a, b, c, m.step.first, m.step.bc1, m.step.bc2);
          m.w[at] = ww;
          if (m.s0) m.s0[at] = a;
          if (m.s1) m.s1[at] = b;
          if (m.s2) m.s2[at] = c;
        }
      }
    }
  }
}

// End of an API call. Host arrays may have been staged by copies of pageable memory, whose pages the runtime may
// hold on to until it is asked to synchronise: only calls on device memory wait for a word.
static int32_t dense_finish(krk_dense* t, uint32_t flags) {
  if (flags & KRK_ASYNC) return KRK_SUCCESS;
  if (flags & KRK_DEVICE_PTRS) return wait_stream(t->stream);
  KRK_HIP(hipStreamSynchronize(t->stream));
  return KRK_SUCCESS;
}

constexpr unsigned kCooGrid = 512;

// Whether a push's indices were not found to be unordered, as its launches tell the host behind a word: by the word's
// number. (Not by a plain yes: that may be one that an earlier call's launch, which failed in between and gave its
// word back, has written meanwhile. What is no yes to this call is taken for a no, which is right for ordered ones too.)
// The last launch of a push of device arrays that waits writes both.
__global__ void signal_unordered_kernel(uint32_t* word, uint32_t ticket, CooTiles tiles) {
  word[1] = coo_unordered(tiles) ? 0u : ticket;
  signal_host(word, ticket);
}

// Waits for what a push enqueued. *unordered: what its launches found out. end is not open where there was no word to be
// had: neither is known then.
static int32_t dense_finish_coo(krk_dense* t, StreamWait* end, const CooTiles& tiles, uint32_t flags, bool* unordered,
                                bool* waited) {
  *waited = false;
  if (!end->word) return KRK_SUCCESS;
  uint32_t told = 0;
  if (flags & KRK_DEVICE_PTRS) {
    hipLaunchKernelGGL(signal_unordered_kernel, dim3(1), dim3(1), 0, t->stream, end->word, end->ticket, tiles);
    KRK_HIP(hipGetLastError());
    KRK_TRY(wait_for(end, t->stream, &told));
  } else {
    KRK_HIP(hipStreamSynchronize(t->stream));   // (see dense_finish)
    told = __atomic_load_n(end->told(), __ATOMIC_RELAXED);
    end->close();
  }
  *unordered = told != end->ticket;
  *waited = true;
  return KRK_SUCCESS;
}

// A small tensor's pushes that are zeroed and scattered into, with no look at their order, after one whose indices did
// not ascend.
constexpr int kCooPlainPushes = 256;

// One Optim::Update with a sparse gradient of nnz > 0 entries (device addresses); entries whose
// index lies outside [0, n) are skipped. A blocking call waits for the update anyway, so it is
// waited for here, and the launches for unordered indices follow only where there are any (three
// launches that look at a flag and leave: 13 us). So blocking calls go tile by tile whatever the size, once a
// push has been seen to ascend: 300 / 20,000 / 300,000 / 2 million elements, an entry in four, Adam, device
// arrays, 15.1 / 16.2 / 17.0 / 30.0 us by fill, scatter and update, 12.9 / 15.8 / 15.7 / 22.4 in tiles. A push that
// goes tile by tile and whose indices do not ascend is scattered after all, behind a second wait (shuffled, 36 / 63 us for
// 300,000 / 2 million elements, 19 / 48 where it is scattered at once), so the push before it decides: a small table's first
// one is scattered, and the scatter looks at the order in passing (28 to 31 us for 27 of 2 million elements); after one that does
// not ascend the next ones are scattered as they are.
// That is for device arrays. Indices that the kernels read in host memory cross PCIe twice in tiles and once in the
// scatter (page-locked, 300,000 / 2 million elements, an entry in four, 51 / 227 us and 37 / 132; pageable 64 and 52
// for 300,000). And from eight commands on between two synchronises the runtime gives back pinned pages and freed
// memory in a way that slows the copies and allocations which follow: a new table's first push of 2 million elements
// from pageable arrays takes 250 us with seven (two copies, Adam's columns, fill, scatter, update) and with nine mostly
// 3000, as does creating the next table. So a push of host arrays enqueues no launch
// that it can do without: a small one is always scattered, and of a large one the update itself says whether
// the tiles were of help. *waited: nothing is left to wait for.
static int32_t dense_apply_coo(krk_dense* t, const krk_optim& o, const long long* d_idx, const float* d_val,
                               int64_t nnz, float lr, uint32_t flags, bool* waited) {
  *waited = false;
  if (!t->coo_grad) {
    // (one allocation: a table's first sparse push pays for it)
    const size_t grad = ((size_t)t->n * sizeof(float) + 16 + 255) & ~(size_t)255;
    KRK_HIP(hipMalloc((void**)&t->coo_grad, grad + coo_tile_words(t->n) * sizeof(uint32_t)));
    t->coo_work.lent = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(t->coo_grad) + grad);
  }
  const bool small = t->n < kCooTiledFrom, waits = !(flags & KRK_ASYNC);
  bool tiled = coo_tiled(t->n, nnz), look = false, unordered = false;
  if (small && (flags & KRK_DEVICE_PTRS) && waits && nnz <= t->n) {   // (more entries than elements do not ascend)
    tiled = t->coo_ascends;
    look = !tiled && t->coo_plain == 0;
    if (t->coo_plain) --t->coo_plain;
  }
  CooTiles tiles;
  StreamWait end;
  if (!tiled) {
    if (look) KRK_TRY(coo_new_tag(&t->coo_work, t->n, &tiles));
    KRK_TRY(coo_densify(&t->coo_work, d_idx, d_val, nnz, t->coo_grad, t->n, t->stream, look ? &tiles : nullptr));
    KRK_TRY(dense_apply(t, o, t->coo_grad, lr));
    if (!look || !end.open()) return KRK_SUCCESS;
    KRK_TRY(dense_finish_coo(t, &end, tiles, flags, &unordered, waited));
    if (*waited) {
      t->coo_ascends = !unordered;
      t->coo_plain = unordered ? kCooPlainPushes : 0;
    }
    return KRK_SUCCESS;
  }
  DenseMember m;
  KRK_TRY(dense_member(t, o, &m));
  const OptimK k = make_optim_k(o);
  KRK_TRY(coo_find_tiles(&t->coo_work, d_idx, nnz, t->n, true, &tiles, t->stream));
  if (waits && end.open() && !(flags & KRK_DEVICE_PTRS)) {
    tiles.told = end.told();
    tiles.ticket = end.ticket;
  }
  const dim3 block(kDenseBlock);
  with_optim(o.type, [&](auto opt) {
    const dim3 grid(std::min(tiles.tiles, kCooGrid));
    if (tiles.bits) {
      hipLaunchKernelGGL((coo_bits_update_kernel<opt.value>), grid, block, 0, t->stream, m, d_val, tiles, lr, k);
    } else {
      hipLaunchKernelGGL((coo_update_kernel<opt.value>), grid, block, 0, t->stream, m, d_idx, d_val, tiles, lr, k);
    }
  });
  KRK_HIP(hipGetLastError());
  if (waits) {
    KRK_TRY(dense_finish_coo(t, &end, tiles, flags, &unordered, waited));
    if (*waited && !unordered) return KRK_SUCCESS;
    if (*waited && small) {
      t->coo_ascends = false;
      t->coo_plain = kCooPlainPushes;
    }
    *waited = false;
  }
  KRK_TRY(coo_scatter_if_unordered(tiles, d_idx, d_val, nnz, t->coo_grad, t->n, t->stream));
  with_optim(o.type, [&](auto opt) {
    hipLaunchKernelGGL((dense_update_kernel<opt.value>), dim3(dense_grid(t->n)), block, 0, t->stream, m.w, m.s0, m.s1,
                       m.s2, t->coo_grad, t->n, lr, k, m.step.first, m.step.bc1, m.step.bc2, tiles);
  });
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

// A pull into device memory: one workgroup per compute unit with four non-temporal 16-byte accesses
// in flight a lane is what copies fastest here (5.8 TB/s for 4 GiB; the runtime's own copy 4.4).
constexpr unsigned kCopyGrid = 256;
constexpr int kCopyAhead = 4;
__global__ __launch_bounds__(kDenseBlock) void dense_copy_kernel(const float* __restrict__ src, float* __restrict__ dst,
                                                                 int64_t n) {
  const int64_t n4 = n >> 2;
  const int64_t stride = (int64_t)gridDim.x * kDenseBlock;
  const dfloat4* s = reinterpret_cast<const dfloat4*>(src);
  dfloat4* d = reinterpret_cast<dfloat4*>(dst);
  int64_t i = (int64_t)blockIdx.x * kDenseBlock + threadIdx.x;
  for (; i + (kCopyAhead - 1) * stride < n4; i += kCopyAhead * stride) {
    dfloat4 v[kCopyAhead];
#pragma unroll
    for (int u = 0; u < kCopyAhead; ++u) v[u] = __builtin_nontemporal_load(s + i + u * stride);
#pragma unroll
    for (int u = 0; u < kCopyAhead; ++u) __builtin_nontemporal_store(v[u], d + i + u * stride);
  }
  for (; i < n4; i += stride) d[i] = s[i];
  const int64_t tail = (n4 << 2) + (int64_t)blockIdx.x * kDenseBlock + threadIdx.x;
  if (tail < n) dst[tail] = src[tail];
}

// ---- several dense tables in one launch ------------------------------------------------------
// Ps::CombinePullDenseTable (ps/ps_op.cc:177-252) pulls every dense parameter of the model in one
// request, and the worker does that after every step (pytorch/optimizer.py:151-173); one table per
// launch makes a model with dozens of small tensors pay a launch per tensor. Here the members'
// values (and, for the push, gradients) are one concatenated array in member order, and a launch
// serves all members that have elements.
//
// A request of dozens of small tensors is bound by the host's calls and by the trips to memory before a
// workgroup knows what to load. What does not change from call to call lies on the device with the
// group: a record per workgroup, which names its member, and a descriptor per member, in which a state
// column is entered when it is created. As arguments of the launch (3.8 KB, put together and copied on
// every call) they made a push and a pull of 40 tensors of 434k parameters take 11 us of the host, 6.2 and
// 5.0, and take 8.6 now, 4.9 and 3.9 (a pull also takes its members' locks no longer, a push computes the
// powers of equal step counts once).
struct DenseDesc {
  float* w;
  float* state[KRK_ST_COUNT];
  int64_t n;
  int64_t start;     // first element in the concatenated arrays of a combined request
};
struct DenseBlock {
  uint32_t member;
  uint32_t at, of;   // which of the member's workgroups this is
  uint32_t unused;
};

// What changes with every push: the members' steps, for the members of one launch.
constexpr int kDenseGroupChunk = 64;
struct DenseSteps {
  float bc1[kDenseGroupChunk], bc2[kDenseGroupChunk];
  unsigned long long first;
};

__global__ __launch_bounds__(kDenseBlock) void dense_group_pull_kernel(const DenseBlock* __restrict__ blocks,
                                                                       const DenseDesc* __restrict__ descs,
                                                                       float* __restrict__ out) {
  const DenseBlock b = blocks[blockIdx.x];
  const DenseDesc& m = descs[b.member];
  const int64_t lane = (int64_t)b.at * kDenseBlock + threadIdx.x;
  const int64_t stride = (int64_t)b.of * kDenseBlock;
  float* dst = out + m.start;
  const float* w = m.w;
  const int64_t n = m.n;
  // 16-byte accesses where the member begins on a 16-byte boundary of the output
  const int64_t n4 = (m.start & 3) == 0 ? n >> 2 : 0;
  for (int64_t i = lane; i < n4; i += stride)
    __builtin_nontemporal_store(dense_load(w, i), reinterpret_cast<dfloat4*>(dst) + i);
  for (int64_t i = (n4 << 2) + lane; i < n; i += stride) dst[i] = w[i];
}

// member0: the launch's first member
template <int OPT>
__global__ __launch_bounds__(kDenseBlock) void dense_group_update_kernel(const DenseBlock* __restrict__ blocks,
                                                                         const DenseDesc* __restrict__ descs,
                                                                         uint32_t member0, DenseSteps steps, int st0,
                                                                         int st1, int st2,
                                                                         const float* __restrict__ grads, float lr,
                                                                         OptimK k) {
  const DenseBlock b = blocks[blockIdx.x];
  const DenseDesc& m = descs[b.member];
  const uint32_t mi = b.member - member0;
  const int64_t lane = (int64_t)b.at * kDenseBlock + threadIdx.x;
  const int64_t stride = (int64_t)b.of * kDenseBlock;
  const float* grad = grads + m.start;
  float* w = m.w;
  float* s0 = st0 >= 0 ? m.state[st0] : nullptr;
  float* s1 = st1 >= 0 ? m.state[st1] : nullptr;
  float* s2 = st2 >= 0 ? m.state[st2] : nullptr;
  const bool first = (steps.first >> mi) & 1u;
  const float bc1 = steps.bc1[mi], bc2 = steps.bc2[mi];
  const dfloat4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int64_t n = m.n;
  const int64_t n4 = (m.start & 3) == 0 ? n >> 2 : 0;
  for (int64_t i = lane; i < n4; i += stride) {
    const dfloat4 g4 = __builtin_nontemporal_load(reinterpret_cast<const dfloat4*>(grad) + i);
    const dfloat4 w4 = dense_load(w, i);
    const dfloat4 a4 = s0 ? dense_load(s0, i) : zero;
    const dfloat4 b4 = s1 ? dense_load(s1, i) : zero;
    const dfloat4 c4 = s2 ? dense_load(s2, i) : zero;
    float ww[4], sa[4], sb[4], sc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ww[j] = w4[j]; sa[j] = a4[j]; sb[j] = b4[j]; sc[j] = c4[j];
      optim_element<OPT>(k, lr, g4[j], ww[j], sa[j], sb[j], sc[j], first, bc1, bc2);
    }
    dense_store(w, i, (dfloat4){ww[0], ww[1], ww[2], ww[3]});
    if (s0) dense_store(s0, i, (dfloat4){sa[0], sa[1], sa[2], sa[3]});
    if (s1) dense_store(s1, i, (dfloat4){sb[0], sb[1], sb[2], sb[3]});
    if (s2) dense_store(s2, i, (dfloat4){sc[0], sc[1], sc[2], sc[3]});
  }
  for (int64_t i = (n4 << 2) + lane; i < n; i += stride) {
    float g = grad[i], ww = w[i];
    float sa = s0 ? s0[i] : 0.0f, sb = s1 ? s1[i] : 0.0f, sc = s2 ? s2[i] : 0.0f;
    optim_element<OPT>(k, lr, g, ww, sa, sb, sc, first, bc1, bc2);
    w[i] = ww;
    if (s0) s0[i] = sa;
    if (s1) s1[i] = sb;
    if (s2) s2[i] = sc;
  }
}

// Workgroups a member of n elements gets in a combined launch.
static unsigned dense_member_blocks(int64_t n) { return n > 0 ? dense_grid(n) : 0u; }

// Puts the group's records and descriptors on the device. The members' streams have been waited for.
static int32_t dense_group_describe(krk_dense_group* g) {
  std::vector<DenseDesc> descs(g->tables.size());
  std::vector<DenseBlock> blocks;
  g->block_start.assign(1, 0u);
  for (size_t i = 0; i < g->tables.size(); ++i) {
    const krk_dense* t = g->tables[i];
    DenseDesc& d = descs[i];
    d.w = t->w;
    for (int st = 0; st < KRK_ST_COUNT; ++st) d.state[st] = t->state[st];
    d.n = t->n;
    d.start = g->start[i];
    const uint32_t of = dense_member_blocks(t->n);
    for (uint32_t b = 0; b < of; ++b) blocks.push_back(DenseBlock{(uint32_t)i, b, of, 0u});
    g->block_start.push_back((uint32_t)blocks.size());
  }
  const size_t desc_bytes = (descs.size() * sizeof(DenseDesc) + 255) & ~(size_t)255;
  std::vector<char> both(desc_bytes + blocks.size() * sizeof(DenseBlock));
  memcpy(both.data(), descs.data(), descs.size() * sizeof(DenseDesc));
  if (!blocks.empty()) memcpy(both.data() + desc_bytes, blocks.data(), blocks.size() * sizeof(DenseBlock));
  KRK_HIP(hipMalloc((void**)&g->descs, both.size()));
  g->blocks = reinterpret_cast<const DenseBlock*>(reinterpret_cast<const char*>(g->descs) + desc_bytes);
  KRK_HIP(hipMemcpyAsync(g->descs, both.data(), both.size(), hipMemcpyHostToDevice, g->stream));
  KRK_HIP(hipStreamSynchronize(g->stream));
  return KRK_SUCCESS;
}

// Takes the group's lock and then every member's, in member order.
struct DenseGroupLock {
  krk_dense_group* g;
  explicit DenseGroupLock(krk_dense_group* gg) : g(gg) {
    g->mu.lock();
    for (krk_dense* t : g->tables) t->mu.lock();
  }
  ~DenseGroupLock() {
    for (auto it = g->tables.rbegin(); it != g->tables.rend(); ++it) (*it)->mu.unlock();
    g->mu.unlock();
  }
  DenseGroupLock(const DenseGroupLock&) = delete;
  DenseGroupLock& operator=(const DenseGroupLock&) = delete;
};

}  // namespace krk

using namespace krk;

static int32_t check_dense(krk_dense* t) {
  if (!t) {
    set_error("null dense table handle");
    return KRK_E_ARGUMENT;
  }
  return ensure_runtime();
}

extern "C" {

int32_t krk_dense_create(const float* val, int64_t n, uint32_t flags, krk_dense** out) {
  if (!out || n < 0 || (n > 0 && !val)) return KRK_E_ARGUMENT;
  KRK_TRY(check_flags(flags & ~KRK_ASYNC));
  KRK_TRY(ensure_runtime());
  krk_dense* t = new (std::nothrow) krk_dense();
  if (!t) return KRK_E_DEVICE;
  t->n = n;
  int32_t rc = t->open_stream();
  t->own_stream = t->stream;
  if (rc == KRK_SUCCESS) {
    hipError_t e = hipMalloc((void**)&t->w, (size_t)(n ? n : 1) * sizeof(float));
    if (e == hipSuccess && n)
      e = hipMemcpyAsync(t->w, val, (size_t)n * sizeof(float),
                         (flags & KRK_DEVICE_PTRS) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                         t->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    if (e != hipSuccess) rc = hip_fail(e, "krk_dense_create", __FILE__, __LINE__);
  }
  if (rc != KRK_SUCCESS) {
    krk_dense_destroy(t);
    return rc;
  }
  *out = t;
  return KRK_SUCCESS;
}

int32_t krk_dense_destroy(krk_dense* t) {
  if (!t) return KRK_SUCCESS;
  if (t->member_of) {
    set_error("the dense table is still a member of a group: destroy the group first");
    return KRK_E_ARGUMENT;
  }
  if (t->stream) (void)hipStreamSynchronize(t->stream);
  if (t->w) (void)hipFree(t->w);
  if (t->coo_grad) (void)hipFree(t->coo_grad);
  t->coo_work.release();
  for (auto& s : t->state)
    if (s) (void)hipFree(s);
  t->close_stream();
  delete t;
  return KRK_SUCCESS;
}

int32_t krk_dense_sync(krk_dense* t) {
  KRK_TRY(check_dense(t));
  std::lock_guard<std::mutex> lk(t->mu);
  return dense_finish(t, 0);
}

int32_t krk_dense_pull(krk_dense* t, float* out, uint32_t flags) {
  KRK_TRY(check_dense(t));
  KRK_TRY(check_flags(flags));
  if (t->n > 0 && !out) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  if (t->n == 0) return dense_finish(t, flags);
  if ((flags & KRK_DEVICE_PTRS) && ((uintptr_t)out & 15) == 0) {
    const int64_t blocks = (t->n / 4 + kDenseBlock - 1) / kDenseBlock;
    hipLaunchKernelGGL(dense_copy_kernel, dim3((unsigned)std::min<int64_t>(std::max<int64_t>(blocks, 1), kCopyGrid)),
                       dim3(kDenseBlock), 0, t->stream, t->w, out, t->n);
    KRK_HIP(hipGetLastError());
  } else {
    KRK_HIP(hipMemcpyAsync(out, t->w, (size_t)t->n * sizeof(float),
                           (flags & KRK_DEVICE_PTRS) ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost,
                           t->stream));
  }
  return dense_finish(t, flags);
}

int32_t krk_dense_push(krk_dense* t, const krk_optim* o, const float* grad, int64_t n, float lr,
                       uint32_t flags) {
  KRK_TRY(check_dense(t));
  KRK_TRY(check_flags(flags));
  if (!o || o->type < KRK_ADAGRAD || o->type > KRK_SGD) return KRK_UNSUPPORTED_OPTIM;
  if (n < 0 || (n > 0 && !grad)) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  if (n != t->n) {   // ps/optim/sgd.cc:36-39: the reference's answer, whatever else is wrong with the request
    set_error("gradient has %lld elements, table has %lld", (long long)n, (long long)t->n);
    return KRK_GRADIENT_UNCOMPATIBLE;
  }
  if ((flags & KRK_DEVICE_PTRS) && ((uintptr_t)grad & 15)) {   // the update moves 16 bytes per lane
    set_error("device gradient must be 16-byte aligned");
    return KRK_E_ARGUMENT;
  }
  if (n == 0) return KRK_SUCCESS;
  const float* d_grad;
  KRK_TRY(t->input(grad, (size_t)n, flags, 0, &d_grad));
  KRK_TRY(dense_apply(t, *o, d_grad, lr));
  return dense_finish(t, flags);
}

int32_t krk_dense_push_coo(krk_dense* t, const krk_optim* o, const int64_t* idx, const float* val,
                           int64_t nnz, float lr, uint32_t flags) {
  KRK_TRY(check_dense(t));
  KRK_TRY(check_flags(flags));
  if (!o || o->type < KRK_ADAGRAD || o->type > KRK_SGD) return KRK_UNSUPPORTED_OPTIM;
  if (nnz < 0 || (nnz > 0 && (!idx || !val))) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  if (nnz == 0) return KRK_SUCCESS;   // ps/optim/adam.cc:26-29 : nothing is touched, not even kSteps
  if (t->n == 0) return KRK_GRADIENT_UNCOMPATIBLE;
  const int64_t* d_idx;
  const float* d_val;
  KRK_TRY(t->input(idx, (size_t)nnz, flags, 0, &d_idx));
  KRK_TRY(t->input(val, (size_t)nnz, flags, 1, &d_val));
  bool waited = false;
  KRK_TRY(dense_apply_coo(t, *o, reinterpret_cast<const long long*>(d_idx), d_val, nnz, lr, flags, &waited));
  return waited ? KRK_SUCCESS : dense_finish(t, flags);
}

int32_t krk_dense_state(krk_dense* t, int32_t state_type, float* out, uint32_t flags) {
  KRK_TRY(check_dense(t));
  KRK_TRY(check_flags(flags));
  if (state_type < 1 || state_type >= KRK_ST_COUNT || (t->n > 0 && !out)) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  if (t->n == 0) return KRK_SUCCESS;
  const size_t bytes = (size_t)t->n * sizeof(float);
  if (t->state[state_type]) {
    KRK_HIP(hipMemcpyAsync(out, t->state[state_type], bytes,
                           (flags & KRK_DEVICE_PTRS) ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost,
                           t->stream));
  } else if (flags & KRK_DEVICE_PTRS) {
    KRK_HIP(hipMemsetAsync(out, 0, bytes, t->stream));
  } else {
    memset(out, 0, bytes);
  }
  return dense_finish(t, flags);
}

int32_t krk_dense_size(krk_dense* t, int64_t* n) {
  if (!t || !n) return KRK_E_ARGUMENT;
  *n = t->n;
  return KRK_SUCCESS;
}

int32_t krk_dense_states(krk_dense* t, uint32_t* mask) {
  if (!t || !mask) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  uint32_t m = t->steps > 0 ? 1u : 0u;
  for (int st = 1; st < KRK_ST_COUNT; ++st) {
    if (t->state[st]) m |= 1u << st;   // states are created by the first update that needs them
  }
  *mask = m;
  return KRK_SUCCESS;
}

int32_t krk_dense_import_state(krk_dense* t, int32_t state_type, const float* state, int64_t steps,
                               uint32_t flags) {
  KRK_TRY(check_dense(t));
  KRK_TRY(check_flags(flags));
  if (state && (state_type < 1 || state_type >= KRK_ST_COUNT)) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  if (state && t->n > 0) {
    KRK_TRY(ensure_states(&t, 1, &state_type, 1, t->stream));
    KRK_HIP(hipMemcpyAsync(t->state[state_type], state, (size_t)t->n * sizeof(float),
                           (flags & KRK_DEVICE_PTRS) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                           t->stream));
    if (state_type == KRK_ST_MOMENTUM_BUFFER) t->sgd_started = true;
  }
  if (steps >= 0) t->steps = steps;
  // a host source buffer may be reused by the caller as soon as this returns
  return dense_finish(t, (flags & KRK_DEVICE_PTRS) ? flags : (flags & ~KRK_ASYNC));
}

int32_t krk_dense_group_create(krk_dense** tables, int32_t n, krk_dense_group** out) {
  if (!tables || !out || n <= 0) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  for (int i = 0; i < n; ++i) {
    if (!tables[i] || tables[i]->member_of) {
      set_error("group members must be dense tables that are in no other group");
      return KRK_E_ARGUMENT;
    }
    for (int j = 0; j < i; ++j)
      if (tables[j] == tables[i]) return KRK_E_ARGUMENT;
  }
  krk_dense_group* g = new (std::nothrow) krk_dense_group();
  if (!g) return KRK_E_DEVICE;
  const int32_t rc = g->open_stream();
  if (rc != KRK_SUCCESS) {
    delete g;
    return rc;
  }
  g->own_stream = g->stream;
  for (int i = 0; i < n; ++i) {
    krk_dense* t = tables[i];
    std::lock_guard<std::mutex> lk(t->mu);
    (void)hipStreamSynchronize(t->stream);
    t->stream = g->stream;   // from now on the table's own calls are ordered with the group's
    t->member_of = g;
    g->tables.push_back(t);
    g->start.push_back(g->total);
    g->total += t->n;
  }
  // (from here on the members' own calls may be creating columns: they are described under their locks)
  int32_t described;
  {
    DenseGroupLock lk(g);
    (void)hipStreamSynchronize(g->stream);
    described = dense_group_describe(g);
    for (size_t i = 0; i < g->tables.size() && described == KRK_SUCCESS; ++i)
      g->tables[i]->group_state = g->descs[i].state;
  }
  if (described != KRK_SUCCESS) {
    krk_dense_group_destroy(g);
    return described;
  }
  *out = g;
  return KRK_SUCCESS;
}

int32_t krk_dense_group_destroy(krk_dense_group* g) {
  if (!g) return KRK_SUCCESS;
  (void)hipStreamSynchronize(g->stream);
  for (krk_dense* t : g->tables) {
    std::lock_guard<std::mutex> lk(t->mu);
    t->stream = t->own_stream;
    t->member_of = nullptr;
    t->group_state = nullptr;
  }
  g->stream = g->own_stream;
  if (g->descs) (void)hipFree(g->descs);
  g->close_stream();
  delete g;
  return KRK_SUCCESS;
}

int32_t krk_dense_group_sync(krk_dense_group* g) {
  if (!g) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  DenseGroupLock lk(g);
  KRK_HIP(hipStreamSynchronize(g->stream));
  return KRK_SUCCESS;
}

int32_t krk_dense_group_size(krk_dense_group* g, int64_t* total) {
  if (!g || !total) return KRK_E_ARGUMENT;
  *total = g->total;
  return KRK_SUCCESS;
}

int32_t krk_dense_group_pull(krk_dense_group* g, float* out, uint32_t flags) {
  if (!g) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  KRK_TRY(check_flags(flags));
  if (g->total > 0 && !out) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(g->mu);   // nothing of the members' host side is looked at
  if (g->total == 0) return KRK_SUCCESS;
  float* d_out;
  KRK_TRY(g->output(out, (size_t)g->total, flags, 0, &d_out));
  hipLaunchKernelGGL(dense_group_pull_kernel, dim3(g->block_start.back()), dim3(kDenseBlock), 0, g->stream, g->blocks,
                     g->descs, d_out);
  KRK_HIP(hipGetLastError());
  KRK_TRY(g->output_back(out, (size_t)g->total, flags, 0));
  if ((flags & KRK_DEVICE_PTRS) && !(flags & KRK_ASYNC)) return wait_stream(g->stream);
  if (!(flags & KRK_ASYNC)) KRK_HIP(hipStreamSynchronize(g->stream));
  return KRK_SUCCESS;
}

int32_t krk_dense_group_push(krk_dense_group* g, const krk_optim* o, const float* grads, int64_t n, float lr,
                             uint32_t flags) {
  if (!g) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  KRK_TRY(check_flags(flags));
  if (!o || o->type < KRK_ADAGRAD || o->type > KRK_SGD) return KRK_UNSUPPORTED_OPTIM;
  if (n < 0 || (n > 0 && !grads)) return KRK_E_ARGUMENT;
  DenseGroupLock lk(g);
  if (n != g->total) {   // every member's ps/optim/sgd.cc:36-39 at once
    set_error("gradients hold %lld elements, the group's tables %lld", (long long)n, (long long)g->total);
    return KRK_GRADIENT_UNCOMPATIBLE;
  }
  if (n == 0) return KRK_SUCCESS;
  if ((flags & KRK_DEVICE_PTRS) && ((uintptr_t)grads & 15)) {
    set_error("device gradients must be 16-byte aligned");
    return KRK_E_ARGUMENT;
  }
  const float* d_grads;
  KRK_TRY(g->input(grads, (size_t)n, flags, 0, &d_grads));
  const OptimK k = make_optim_k(*o);
  int32_t st[3];
  dense_slots(*o, st);
  KRK_TRY(ensure_states(g->tables.data(), g->tables.size(), st, 3, g->stream));
  StepMemo memo;
  for (size_t i = 0; i < g->tables.size();) {
    const size_t member0 = i;
    DenseSteps steps;
    steps.first = 0;
    for (; i < g->tables.size() && i < member0 + kDenseGroupChunk; ++i) {
      krk_dense* t = g->tables[i];
      if (t->n == 0) continue;
      const DenseStep s = dense_step(t, *o, &memo);
      steps.bc1[i - member0] = s.bc1;
      steps.bc2[i - member0] = s.bc2;
      if (s.first) steps.first |= 1ull << (i - member0);
    }
    const uint32_t block0 = g->block_start[member0], blocks = g->block_start[i] - block0;
    if (blocks == 0) continue;
    with_optim(o->type, [&](auto opt) {
      hipLaunchKernelGGL((dense_group_update_kernel<opt.value>), dim3(blocks), dim3(kDenseBlock), 0, g->stream,
                         g->blocks + block0, g->descs, (uint32_t)member0, steps, st[0], st[1], st[2], d_grads, lr, k);
    });
    KRK_HIP(hipGetLastError());
  }
  if (flags & KRK_ASYNC) return KRK_SUCCESS;
  if (flags & KRK_DEVICE_PTRS) return wait_stream(g->stream);
  KRK_HIP(hipStreamSynchronize(g->stream));
  return KRK_SUCCESS;
}

int32_t krk_dense_steps(krk_dense* t, int64_t* steps) {
  if (!t || !steps) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(t->mu);
  *steps = t->steps;
  return KRK_SUCCESS;
}

}  // extern "C"
