// Shared internals of the HIP table engine (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "kraken_hip.h"

namespace krk {

// ---- error plumbing -------------------------------------------------------
void set_error(const char* fmt, ...);
int32_t hip_fail(hipError_t e, const char* what, const char* file, int line);

#define KRK_HIP(expr)                                                     \
  do {                                                                    \
    hipError_t krk_e_ = (expr);                                           \
    if (krk_e_ != hipSuccess) return ::krk::hip_fail(krk_e_, #expr, __FILE__, __LINE__); \
  } while (0)

#define KRK_TRY(expr)                    \
  do {                                   \
    int32_t krk_rc_ = (expr);            \
    if (krk_rc_ != KRK_SUCCESS) return krk_rc_; \
  } while (0)

int32_t ensure_runtime();
int current_device();
// Resolves, for the current device, the address of the fixed work space krk_dedup_noalloc uses.
int32_t noalloc_prepare();

// A device buffer that only ever grows; used for staging and scratch.
struct DeviceBuffer {
  void* ptr = nullptr;
  size_t bytes = 0;
  int32_t reserve(size_t want);
  void release();
  template <typename T>
  T* as() const {
    return reinterpret_cast<T*>(ptr);
  }
};

// Owns a fresh device allocation until it is handed over: error paths between hipMalloc and the
// hand-over free it.
struct DeviceGuard {
  void* p = nullptr;
  DeviceGuard() = default;
  DeviceGuard(const DeviceGuard&) = delete;
  DeviceGuard& operator=(const DeviceGuard&) = delete;
  ~DeviceGuard() {
    if (p) (void)hipFree(p);
  }
  template <typename T>
  T* release() {
    T* q = reinterpret_cast<T*>(p);
    p = nullptr;
    return q;
  }
};

// A host pointer that HIP knows as page-locked (hipHostMalloc, krk_host_malloc, a framework's
// pinned tensors) can be handed to kernels as it is: they read and write it across PCIe, which
// saves the staging copy and its launch. Returns the address kernels use, or null when the
// memory is pageable or not aligned to `align` bytes. coherent: whether the host is sure to see what
// kernels write there as soon as they have ended (allocated as coherent, which krk_host_malloc does; a framework's
// pinned tensors seldom say so, and calls that write to them synchronise).
void* direct_host_pointer(const void* p, size_t align, bool* coherent = nullptr);

// Page-locked host memory that grows and is kept.
struct HostBuffer {
  void* ptr = nullptr;
  size_t bytes = 0;
  int32_t reserve(size_t want);
  void release();
};

// Host arguments of up to this size pass through page-locked memory that the kernels read and write
// themselves; beyond it they are staged on the device by copies. A call's copies cost more than
// the kernel as long as the data is small: 4001 ids and rows of 16 floats (256 KB), push and
// pull, 101 us with copies, 61 us this way; 20,000 of them 216 and 187 us. Data that the kernels
// read at 40 GB/s in place of 8 TB/s, and what an object may keep locked (four such buffers of up
// to 1.5 MB), set the limit.
constexpr size_t kBounceMax = (size_t)1 << 20;

// That holds for what is read once, front to back. An argument that the kernels read several times
// over, or row by row in an order of their own, crosses PCIe again with each read, and in pieces of
// at least kHostPiece bytes: a pooled push reads a bag's gradient row once for every id of the bag.
// Where the reads come to kReadAgainMin bytes more than the argument has, it is copied to the device
// by a kernel first. Blocking calls on pageable memory, us, everything copied to the device by the
// runtime / everything read in place / by this rule: pooled pushes of 10,000 bags of 16 floats, ten
// ids each, 164 / 233 / 144, 2048 bags of 64 floats, 40 weighted ids each, 186 / 260 / 151, 256
// bags of 16 floats, four ids each (read in place) 91 / 41 / 41; push_raw of 16,000 ids of 8 floats
// 110 / 117 / 96; a codec step that selects over 260,000 values 168 / 228 / 145.
constexpr size_t kHostPiece = 128;
constexpr size_t kReadAgainMin = (size_t)128 << 10;
// bytes that `reads` reads of `bytes` each take across PCIe
inline size_t host_reads(int64_t reads, int64_t bytes) {
  return (size_t)reads * (bytes < (int64_t)kHostPiece ? kHostPiece : (size_t)bytes);
}
// Waiting for the end of a call. hipStreamSynchronize puts a packet of its own into the queue and waits for its
// signal: the host goes on 9.4 us after the launch of an empty kernel and 15 after those of a short kernel and one that
// writes a word. A host that looks at that word itself goes on after 6.0 and 10.0. So the last launch of a blocking
// call writes a number into a page-locked word and the host waits for the number to appear. What lies ahead
// of that launch in its stream has ended by then, and its writes are where kernels that start later, and
// the host in coherent memory, find them. To the runtime the stream is not synchronised then: a program that calls
// hipDeviceSynchronize all the same pays for the packet there, 9 us after up to three such calls and 22 to 30 after
// more, where it took 0.2 (a pull and the synchronise 15.8 -> 19.5 us, four and one 62.8 -> 72, sixteen 251 -> 223).
struct StreamWait {
  uint32_t* word = nullptr;   // null: not open
  uint32_t ticket = 0;
  StreamWait() = default;
  StreamWait(const StreamWait&) = delete;
  StreamWait& operator=(const StreamWait&) = delete;
  ~StreamWait() { close(); }
  static void prepare();   // the memory of the words, with the runtime
  bool open();    // takes a free word; false where there is none: the call then synchronises with the stream
  uint32_t* told() const { return word + 1; }
  void close();   // gives it back
};
// Waits until the word of an open wait holds its number, and closes it. A stream that takes longer than five
// milliseconds, has failed or is being captured is left to hipStreamSynchronize. The core is busy meanwhile, as it is in
// hipStreamSynchronize; after 50 us other threads may have it between two looks. told: what lies behind the word
// in its cache line (StreamWait::told), as the launch that wrote the word left it.
int32_t wait_for(StreamWait* w, hipStream_t stream, uint32_t* told = nullptr);
// The same for a stream whose last launch writes no word: puts a launch behind it that does.
int32_t wait_stream(hipStream_t stream);
// Called by the one wavefront of that launch.
__device__ __forceinline__ void signal_host(uint32_t* word, uint32_t ticket) {
  __threadfence_system();
  if (threadIdx.x == 0) __hip_atomic_store(word, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Copies host memory that kernels can address to device memory (both on 16 bytes; whole words).
int32_t copy_from_host(void* dst, const void* src, size_t bytes, hipStream_t stream);

// Every API object starts with this: its own stream, the host lock that serialises
// calls on it, and the staging buffers used when the caller hands over host pointers.
struct ObjBase {
  hipStream_t stream = nullptr;
  std::mutex mu;
  DeviceBuffer stage[4];
  HostBuffer bounce[4];
  bool bounced[4] = {false, false, false, false};  // output slot lies in `bounce`
  bool direct[4] = {false, false, false, false};   // output slot is the caller's own page-locked buffer
  // The end of a blocking call whose last launch writes `waiting`'s word (sparse_finish_begin): whether it has been
  // waited for, and whether the call has to synchronise instead: the caller's pageable memory takes part in an
  // asynchronous copy (the runtime may hold on to its pages until then), or an output lies in memory of the
  // caller's that is not known to be coherent.
  StreamWait waiting;
  bool waited = false, must_synchronise = false;
  int32_t finish_wait() {
    if (waiting.word && !must_synchronise) {
      KRK_TRY(wait_for(&waiting, stream));
    } else {
      KRK_HIP(hipStreamSynchronize(stream));
      waiting.close();
      must_synchronise = false;
    }
    waited = true;
    return KRK_SUCCESS;
  }
  // An asynchronous copy to or from pageable memory of the caller's.
  int32_t copy_pages(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    must_synchronise = true;
    waited = false;   // also where another output of the call has been waited for
    KRK_HIP(hipMemcpyAsync(dst, src, bytes, kind, stream));
    return KRK_SUCCESS;
  }
  int32_t open_stream();
  void close_stream();
  // Where kernels find a host array: the caller's page-locked memory, page-locked buffer `slot` or
  // staging buffer `slot` (a device pointer is passed through). read: the bytes the call's kernels
  // read of it, if that is not each byte once in order (host_reads).
  template <typename T>
  int32_t input(const T* p, size_t count, uint32_t flags, int slot, const T** dev, size_t read = 0) {
    if (flags & KRK_DEVICE_PTRS) {
      *dev = p;
      return KRK_SUCCESS;
    }
    const size_t bytes = count * sizeof(T);
    if (void* d = direct_host_pointer(p, 16)) {
      *dev = reinterpret_cast<const T*>(d);
      return KRK_SUCCESS;
    }
    if (bytes <= kBounceMax) {
      // host pointers make a call blocking: what an earlier call put here has been read
      KRK_TRY(bounce[slot].reserve(bytes + 16));
      std::memcpy(bounce[slot].ptr, p, bytes);
      *dev = reinterpret_cast<const T*>(bounce[slot].ptr);
      if (read < bytes + kReadAgainMin) return KRK_SUCCESS;
      KRK_TRY(stage[slot].reserve(bytes + 16));
      KRK_TRY(copy_from_host(stage[slot].ptr, bounce[slot].ptr, bytes, stream));
      *dev = stage[slot].as<T>();
      return KRK_SUCCESS;
    }
    KRK_TRY(stage[slot].reserve(bytes + 16));
    KRK_TRY(copy_pages(stage[slot].ptr, p, bytes, hipMemcpyHostToDevice));
    *dev = stage[slot].as<T>();
    return KRK_SUCCESS;
  }
  // Device destination for an output: the caller's pointer, or staging buffer `slot`.
  template <typename T>
  int32_t output(T* p, size_t count, uint32_t flags, int slot, T** dev) {
    if (flags & KRK_DEVICE_PTRS) {
      *dev = p;
      return KRK_SUCCESS;
    }
    direct[slot] = bounced[slot] = false;
    bool coherent = false;
    if (void* d = direct_host_pointer(p, 16, &coherent)) {
      direct[slot] = true;
      if (!coherent) must_synchronise = true;
      *dev = reinterpret_cast<T*>(d);
      return KRK_SUCCESS;
    }
    if (count * sizeof(T) <= kBounceMax) {
      KRK_TRY(bounce[slot].reserve(count * sizeof(T) + 16));
      bounced[slot] = true;
      *dev = reinterpret_cast<T*>(bounce[slot].ptr);
      return KRK_SUCCESS;
    }
    KRK_TRY(stage[slot].reserve(count * sizeof(T) + 16));
    *dev = stage[slot].as<T>();
    return KRK_SUCCESS;
  }
  // Brings an output to the caller's host memory; what the call enqueues for the host besides (its
  // counters) goes into the stream before, so that one wait covers both.
  template <typename T>
  int32_t output_back(T* p, size_t count, uint32_t flags, int slot) {
    if ((flags & KRK_DEVICE_PTRS) || !count || direct[slot]) return KRK_SUCCESS;
    if (bounced[slot]) {
      KRK_TRY(finish_wait());
      std::memcpy(p, bounce[slot].ptr, count * sizeof(T));
      return KRK_SUCCESS;
    }
    return copy_pages(p, stage[slot].ptr, count * sizeof(T), hipMemcpyDeviceToHost);
  }
};

inline int32_t check_flags(uint32_t flags) {
  if (flags & ~(KRK_DEVICE_PTRS | KRK_ASYNC | KRK_NOTE_ROWS | KRK_IDS_AS_PULLED)) {
    set_error("unknown flag bits 0x%x", flags);
    return KRK_E_ARGUMENT;
  }
  if ((flags & KRK_ASYNC) && !(flags & KRK_DEVICE_PTRS)) {
    set_error("KRK_ASYNC needs KRK_DEVICE_PTRS");
    return KRK_E_ARGUMENT;
  }
  return KRK_SUCCESS;
}

constexpr int kWave = 64;

// Workgroup b of a launch of n runs on XCD b mod 8, and the XCDs' L2 caches are separate. Tiles that write
// next to each other are therefore given to one XCD: it takes a stretch of consecutive tiles.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t n) {
  const uint32_t xcd = b % kXcds, each = n / kXcds, more = n % kXcds;
  return xcd * each + (xcd < more ? xcd : more) + b / kXcds;
}

// Inclusive prefix sum over a wavefront, all of whose lanes call it. Data-parallel moves inside rows of
// 16 lanes, then the rows' last lanes broadcast to the rows behind them: a tenth of the cycles of
// six shuffles through LDS, each of which waits for the one before.
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
#define KRK_DPP_ADD(ctrl, rows) \
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false)
  KRK_DPP_ADD(0x111, 0xf);   // row_shr:1
  KRK_DPP_ADD(0x112, 0xf);   // row_shr:2
  KRK_DPP_ADD(0x114, 0xf);   // row_shr:4
  KRK_DPP_ADD(0x118, 0xf);   // row_shr:8
  KRK_DPP_ADD(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
  KRK_DPP_ADD(0x143, 0xc);   // row_bcast:31 into rows 2 and 3
#undef KRK_DPP_ADD
  return v;
}
// Between LDS accesses of one wavefront's lanes and those of its other lanes to the same words. The hardware keeps
// one wavefront's LDS accesses in the order they are issued in; this keeps the compiler from issuing them in
// another one, which the barrier alone, no access to memory to it, need not. No instruction of its own.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Narrows the lanes of a wavefront (both halves of a mask) to those whose value has bit b as this lane's has it: four
// vector instructions, one vote and, for either half, a bitwise operation of three operands. All lanes call it.
__device__ __forceinline__ void match_bit(uint32_t v, int b, uint32_t& lo, uint32_t& hi) {
  const int32_t bit = (int32_t)(v << (31 - b)) >> 31;   // all ones or none
  const unsigned long long votes = __ballot(bit != 0);
  lo &= ~((uint32_t)votes ^ (uint32_t)bit);
  hi &= ~((uint32_t)(votes >> 32) ^ (uint32_t)bit);
}
// the lanes of `among` whose lowest `bits` bits equal this lane's (at most MAX; bits is uniform)
template <int MAX>
__device__ __forceinline__ unsigned long long same_value(uint32_t v, unsigned long long among, int bits = MAX) {
  uint32_t lo = (uint32_t)among, hi = (uint32_t)(among >> 32);
#pragma unroll
  for (int b = 0; b < MAX; ++b)
    if (b < bits) match_bit(v, b, lo, hi);
  return (unsigned long long)lo | ((unsigned long long)hi << 32);
}
constexpr uint64_t kEmptyKey = 0xFFFFFFFFFFFFFFFFull;
constexpr uint32_t kEmptyRow = 0xFFFFFFFFu;

// 64-bit finaliser used to place ids in the open-addressing table.
__host__ __device__ inline uint64_t mix64(uint64_t x) {
  x ^= x >> 33;
  x *= 0xFF51AFD7ED558CCDull;
  x ^= x >> 33;
  x *= 0xC4CEB9FE1A85EC53ull;
  x ^= x >> 33;
  return x;
}

__host__ __device__ inline uint64_t splitmix64(uint64_t x) {
  uint64_t z = x + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// ---- row initialiser, evaluated per element on the device ------------------
// kind 0: constant p0; kind 1: uniform [p0, p1); kind 2: normal(mean p0, std p1).
struct InitK {
  int32_t kind;
  float p0;
  float p1;
  uint64_t seed_mix;  // splitmix64(seed)
};

// Normal draws come in pairs: elements 2q and 2q + 1 of a row are the two values of one
// Box-Muller step on the bits drawn for q: k = upper 24 bits + 1 gives the radius
// sqrt(-2 log(k / 2^24)), j = the next 24 bits the angle 2 pi j / 2^24; the values are
// radius * cos(angle) and radius * sin(angle), independent standard normals.
//
// The logarithm and the sine / cosine are written out here, in double-precision +, -, *, /
// only (no library call, no fused multiply-add: the build contracts nothing), so that this file
// and the CPU oracle evaluate the same sequence of IEEE operations and agree to the bit, and so
// that the rare branch of a pull that creates rows stays small: the general-purpose library
// routines handle every argument there is and take several times the instructions and registers.
// Their arguments here are 24-bit fractions, which makes the argument reductions exact.

// log(k / 2^24) for k in [1, 2^24]: k = m 2^e with m in (1/sqrt 2, sqrt 2], log m by the atanh
// series in f = (m - 1) / (m + 1), |f| <= 0.1716 (eight terms: below 1e-14).
__device__ inline double log_u24(uint32_t k) {
  int e = 31 - __clz((int)k);
  double m = (double)k * (1.0 / (double)(1u << e));   // exact, in [1, 2)
  if (m > 1.4142135623730951) {
    m = m * 0.5;
    e = e + 1;
  }
  const double f = (m - 1.0) / (m + 1.0);
  const double z = f * f;
  double p = 0.066666666666666666;                    // 1/15
  p = p * z + 0.076923076923076927;                   // 1/13
  p = p * z + 0.090909090909090912;                   // 1/11
  p = p * z + 0.11111111111111111;                    // 1/9
  p = p * z + 0.14285714285714285;                    // 1/7
  p = p * z + 0.2;                                    // 1/5
  p = p * z + 0.33333333333333331;                    // 1/3
  p = p * z + 1.0;
  return 2.0 * f * p + (double)(e - 24) * 0.69314718055994529;
}

// sin and cos of 2 pi j / 2^24 for j in [0, 2^24): the nearest quarter turn is taken off in
// integers (exact), the rest, at most pi/4 either way, goes through the Taylor polynomials
// (degree 13 and 14: below 3e-14), and the quarter turns are put back by swapping and negating.
__device__ inline void sincos_u24(uint32_t j, double& sn, double& cs) {
  const int32_t quarter = (int32_t)((j + (1u << 21)) >> 22);
  const int32_t rest = (int32_t)j - (quarter << 22);          // in [-2^21, 2^21)
  const double t = (double)rest * 3.7450702829239286e-07;      // 2 pi / 2^24
  const double z = t * t;
  double s = 1.6059043836821613e-10;                  // 1/13!
  s = s * z - 2.505210838544172e-08;                  // 1/11!
  s = s * z + 2.7557319223985893e-06;                 // 1/9!
  s = s * z - 0.00019841269841269841;                 // 1/7!
  s = s * z + 0.0083333333333333332;                  // 1/5!
  s = s * z - 0.16666666666666666;                    // 1/3!
  s = s * z + 1.0;
  s = s * t;
  double c = -1.1470745597729725e-11;                 // 1/14!
  c = c * z + 2.08767569878681e-09;                   // 1/12!
  c = c * z - 2.7557319223985888e-07;                 // 1/10!
  c = c * z + 2.4801587301587302e-05;                 // 1/8!
  c = c * z - 0.0013888888888888889;                  // 1/6!
  c = c * z + 0.041666666666666664;                   // 1/4!
  c = c * z - 0.5;
  c = c * z + 1.0;
  switch (quarter & 3) {
    case 0: sn = s; cs = c; break;
    case 1: sn = c; cs = -s; break;
    case 2: sn = -s; cs = -c; break;
    default: sn = -c; cs = s; break;
  }
}

// both values of pair q of the row whose bits start at `key`
__device__ inline void init_normal_pair(const InitK& k, uint64_t key, int64_t q, float& even, float& odd) {
  const uint64_t r = splitmix64(key + (uint64_t)q * 0x9E3779B97F4A7C15ull);
  const double radius = sqrt(-2.0 * log_u24((uint32_t)(r >> 40) + 1u));
  double sn, cs;
  sincos_u24((uint32_t)(r >> 16) & 0xFFFFFFu, sn, cs);
  even = (float)((double)k.p0 + (double)k.p1 * (radius * cs));
  odd = (float)((double)k.p0 + (double)k.p1 * (radius * sn));
}

__device__ inline float init_element(const InitK& k, uint64_t id, int64_t j) {
  if (k.kind == 0) return k.p0;
  uint64_t key = splitmix64(id ^ k.seed_mix);
  if (k.kind == 1) {
    uint64_t r = splitmix64(key + (uint64_t)j * 0x9E3779B97F4A7C15ull);
    double u = (double)(r >> 40) * (1.0 / 16777216.0);
    return (float)((double)k.p0 + ((double)k.p1 - (double)k.p0) * u);
  }
  float even, odd;
  init_normal_pair(k, key, j >> 1, even, odd);
  return (j & 1) ? odd : even;
}

// ---- optimizer arithmetic, one element at a time ---------------------------
// Pre-narrowed scalars: the reference evaluates (1.0 - beta) in double and
// narrows to float at the Tensor operator (ps/optim/adam.cc:57-58 etc.).
struct OptimK {
  int32_t type;
  int32_t has_wd;
  int32_t has_momentum;
  int32_t nesterov;
  int32_t amsgrad;
  int32_t centered;
  float wd;
  float momentum;
  float one_minus_damp;
  float beta1;
  float beta2;
  float one_minus_b1;
  float one_minus_b2;
  float eps;
  float alpha;
  float one_minus_alpha;
  float acc0;
};
// The same for rows that count their own steps.
struct RowOptimK : OptimK {
  double log2_beta1;       // base-two logarithms of |beta1| and |beta2|, for one_minus_power (Adam)
  double log2_beta2;
};

// Adam's bias correction (float)(1.0 - (double)powf(beta, t)) (ps/optim/adam.cc:61-64) of a step count t >= 1,
// with log2_beta = log2(|beta|) in double. beta^t = 2^n * e^r, n the integer nearest to t * log2_beta,
// |r| <= ln(2) / 2; e^r is its Taylor series through r^10, in double, off by less than 2.2e-13, and the
// power is then rounded to float once (it is the correctly rounded one for 12 betas from 0.1 to 1 - 1e-7
// and all t to 200,000). A wavefront's rows close one after the other, each with two powf for all of its
// lanes: the reduction of 8.5 million pooled ids of 32 floats took 436 us with powf and takes 406.
__device__ __forceinline__ float one_minus_power(double log2_beta, float beta, uint64_t t) {
  // beyond +-1100 the power is 0 or infinite in float whatever it is; a beta of 0 comes as -infinity
  const double x = fmin(fmax(log2_beta * (double)t, -1100.0), 1100.0);
  const double n = rint(x);
  const double r = (x - n) * 0.69314718055994530942;
  double p = 1.0 / 3628800.0;
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  p = ldexp(p, (int)n);
  if (beta < 0.0f && (t & 1)) p = -p;
  return (float)(1.0 - (double)(float)p);
}

OptimK make_optim_k(const krk_optim& o);
RowOptimK make_row_optim_k(const krk_optim& o);
// Which state columns (bit per KRK_ST_*) and whether a step counter this optimizer touches.
uint32_t optim_state_mask(const krk_optim& o);

// State slots s0/s1/s2 per optimizer:
//   SGD      s0 = momentum buffer
//   Adagrad  s0 = state sum
//   Adam     s0 = first moment, s1 = second moment, s2 = second moment max
//   RMSprop  s0 = square average, s1 = g ave, s2 = momentum buffer
// `first` = this row has never been updated (SGD momentum copies the gradient then,
// ps/optim/sgd.cc:46-47). c1/c2 are Adam's bias corrections.
template <int OPT>
__device__ __forceinline__ void optim_element(const OptimK& k, float lr, float g, float& w,
                                              float& s0, float& s1, float& s2, bool first,
                                              float c1, float c2) {
  if (k.has_wd) g = g + k.wd * w;
  if (OPT == KRK_SGD) {
    // ps/optim/sgd.cc:41-60
    if (k.has_momentum) {
      if (first) {
        s0 = g;
      } else {
        s0 = k.momentum * s0 + k.one_minus_damp * g;
      }
      if (k.nesterov) {
        g = g + k.momentum * s0;
      } else {
        g = s0;
      }
    }
    w = w - g * lr;
  } else if (OPT == KRK_ADAGRAD) {
    // ps/optim/adagrad.cc:42-45
    s0 = s0 + g * g;
    float den = sqrtf(s0 + k.acc0) + k.eps;
    w = w - lr * (g / den);
  } else if (OPT == KRK_ADAM) {
    // ps/optim/adam.cc:57-78
    s0 = k.beta1 * s0 + k.one_minus_b1 * g;
    s1 = k.beta2 * s1 + k.one_minus_b2 * (g * g);
    float mt = s0 / c1;
    float vt = s1 / c2;
    float den;
    if (k.amsgrad) {
      s2 = fmaxf(s2, vt);
      den = sqrtf(s2) + k.eps;
    } else {
      den = sqrtf(vt) + k.eps;
    }
    w = w - (lr * mt) / den;
  } else {
    // ps/optim/rmsprop.cc:39-75
    s0 = k.alpha * s0 + k.one_minus_alpha * (g * g);
    float d = s0;
    if (k.centered) {
      s1 = s1 * k.alpha + k.one_minus_alpha * g;
      d = s0 - s1 * s1;
    }
    float den = sqrtf(d) + k.eps;
    if (k.has_momentum) {
      s2 = s2 * k.momentum + g / den;
      w = w - lr * s2;
    } else {
      w = w - (lr * g) / den;
    }
  }
}

// CooTensorImpl::ToDense (t/coo_tensor_impl.cc:250-260, t/math.cc:1006-1096) on the device: dense[0, n) = 0, then
// dense[idx[j]] += val[j]. Large tensors whose indices ascend strictly and lie in range (what ToCoo produces) are
// taken tile by tile: one launch over the indices finds where each tile's entries begin (coo_find_tiles), and
// whoever walks the tiles puts one together in LDS, or, where there are many entries, from a bit an element that
// the first launch leaves. Any other input is zeroed and scattered into; which of the two it is is decided on the
// device, and the launches of the other way look at the flag and leave.
constexpr int kCooTile = 2048;                   // floats of one tile: 8 KB of LDS
// Smaller tensors: zero + scatter, two launches are quicker than two and those of the other way, unless the call
// waits and learns which of the ways it was, and calls before it let it expect that (dense_apply_coo).
constexpr int64_t kCooTiledFrom = 1 << 22;
struct CooTiles {
  uint32_t* starts;       // [tiles + 1]: tile t owns entries [starts[t], starts[t + 1])
  uint32_t* unordered;    // == tag: the indices do not ascend strictly or leave [0, n)
  uint32_t tag;
  uint32_t tiles;
  uint32_t* bits;         // null, or a bit an element, 64 words a tile: whether an entry names it
  uint32_t* told;         // null, or page-locked: who walks the tiles puts `ticket` there, 0 if they are no help
  uint32_t ticket;
};
__device__ __forceinline__ bool coo_unordered(const CooTiles& t) { return *t.unordered == t.tag; }
struct CooWork {          // work space of one caller, kept between calls
  DeviceBuffer buffer, bits;
  uint32_t* lent = nullptr;   // room for coo_tile_words of the caller's tensor behind something else of the caller's
  void release() {
    buffer.release();
    bits.release();
  }
};
inline size_t coo_tile_words(int64_t n) { return (size_t)((n + kCooTile - 1) / kCooTile) + 2; }
// Which of a tile's elements have an entry, and how many entries of the tile lie before each of its 64 words: a lane
// holds the word of its number. All lanes of a wavefront.
struct CooTileBits {
  uint32_t word, before;
  __device__ __forceinline__ explicit CooTileBits(uint32_t w) : word(w) {
    const uint32_t own = (uint32_t)__popc(w);
    before = wave_inclusive_sum(own) - own;
  }
  // The gradient of the four elements of quad q of the tile, whose entries are [start, end) (end > start, or all bits are
  // clear): the values of those that have an entry, zero for the others.
  __device__ __forceinline__ void quad(int q, const float* __restrict__ val, uint32_t start, uint32_t end,
                                       float (&g)[4]) const {
    const uint32_t w = (uint32_t)__shfl((int)word, q >> 3);
    const int shift = (q & 7) * 4;
    const uint32_t mine = (w >> shift) & 15u;
    uint32_t at = start + (uint32_t)__shfl((int)before, q >> 3) + (uint32_t)__popc(w & ((1u << shift) - 1u));
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      // (read whether the element has an entry or not: four loads that wait for one another in no way)
      const float v = val[min(at, end - 1u)];
      g[c] = (mine >> c) & 1u ? v : 0.0f;
      at += (mine >> c) & 1u;
    }
  }
};
inline bool coo_tiled(int64_t n, int64_t nnz) { return n >= kCooTiledFrom && nnz < ((int64_t)1 << 31); }
// A call's tag, which its flag is not raised to yet: out without starts and bits.
int32_t coo_new_tag(CooWork* work, int64_t n, CooTiles* out);
// update: for an optimizer's update, which has more to wait for than a decode (bits pay earlier).
int32_t coo_find_tiles(CooWork* work, const long long* d_idx, int64_t nnz, int64_t n, bool update, CooTiles* out,
                       hipStream_t stream);
// What is left to do where the indices are unordered, and nothing otherwise: dense = the entries' sums.
int32_t coo_scatter_if_unordered(const CooTiles& tiles, const long long* d_idx, const float* d_val, int64_t nnz,
                                 float* d_dense, int64_t n, hipStream_t stream);
// look (smaller tensors): raised if the indices are not such as could be taken tile by tile.
int32_t coo_densify(CooWork* work, const long long* d_idx, const float* d_val, int64_t nnz, float* d_dense, int64_t n,
                    hipStream_t stream, const CooTiles* look = nullptr);

// Stable radix sort of n (key, payload) pairs by the low `bits` bits of the key (radix_sort.hip).
// keys / vals are overwritten; keys_alt / vals_alt hold n entries each; work holds
// radix_sort_work_bytes(n). *keys_sorted / *vals_sorted say which of the two pairs of arrays the
// result is in.
size_t radix_sort_work_bytes(int64_t n);
int32_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n,
                         int bits, void* work, hipStream_t stream, uint32_t** keys_sorted,
                         uint32_t** vals_sorted);

// ---- device-wide exclusive scan of int32 (three plain launches, no spinning) ----
// out[i] = sum(in[0..i)), total written to *total_out (device). in/out may alias. scratch must hold
// scan_scratch_bytes(n).
size_t scan_scratch_bytes(int64_t n);
int32_t exclusive_scan_i32(const int32_t* in, int32_t* out, int64_t n, int32_t* total_out,
                           void* scratch, hipStream_t stream);

}  // namespace krk
