// Threshold gradient codec ("DCT" = dynamic communication thresholding in the reference):
// DCTEmitter::DenseBag::MaybeToCoo (worker/dct_emitter.cc:16-43) and its decode,
// CooTensorImpl::ToDense (t/coo_tensor_impl.cc:250-260).
//
//   f = grad + e                                   error feedback
//   every life_span steps: tau = k-th largest |f|, k = (int64)(n * (1.0 - eta))
//   emit (idx, f[idx]) for |f| >= tau, idx ascending; e = |f| < tau ? f : 0
//
// tau comes from a three-pass radix select over the bit patterns of |f| (non-negative floats
// order like their bit patterns): 11 + 11 + 10 bits, each pass one LDS histogram per workgroup.
// The emit step writes the pairs in input order. Where the caller's buffers hold whatever comes it is
// one pass (emit_single_kernel); where the count decides whether anything may be written at all it is
// a count pass, a scan of the per-tile counts and a write pass that recomputes f.
#include <algorithm>
#include <atomic>
#include <new>

#include "krk_internal.h"

struct krk_dct : krk::ObjBase {
  int64_t n = 0;
  float* e = nullptr;            // residual
  float* e_next = nullptr;       // written by the emit pass, swapped in on success
  uint32_t* sel = nullptr;       // device: [0] prefix bits, [1] k remaining (lo), [2] tau bits, [3] nnz
  uint32_t* hist = nullptr;      // 2048 bins
  int32_t* tile_counts = nullptr;
  int32_t* tile_offsets = nullptr;
  void* scan_tmp = nullptr;
  unsigned long long* tile_state = nullptr;   // single-pass emit: what each tile announced
  uint32_t* tickets = nullptr;   // single-pass emit: [0] next tile, [1] workgroups that are done
  uint32_t emit_calls = 0;       // tags the announcements of one call
  uint32_t* host_sel = nullptr;  // pinned
  float tau = 0.0f;
  uint64_t step = 0;
  int64_t tiles = 0;
};

namespace krk {

constexpr int kCodecBlock = 256;
constexpr int kCodecItems = 8;
constexpr int kCodecTile = kCodecBlock * kCodecItems;
constexpr int kBins = 2048;

__device__ __forceinline__ uint32_t abs_bits(float f) { return __float_as_uint(f) & 0x7FFFFFFFu; }

struct Quad {
  float v[4];
};
typedef float vfloat4 __attribute__((ext_vector_type(4)));   // what the non-temporal builtins accept

__device__ __forceinline__ Quad whole_quad(const float* __restrict__ p, int64_t j) {
  const vfloat4 x = __builtin_nontemporal_load(reinterpret_cast<const vfloat4*>(p + j));
  return Quad{{x[0], x[1], x[2], x[3]}};
}
// four consecutive elements from j on; elements at or behind n read as zero
__device__ __forceinline__ Quad load_quad(const float* __restrict__ p, int64_t j, int64_t n, bool vec) {
  if (vec && j + 3 < n) return whole_quad(p, j);
  Quad q;
#pragma unroll
  for (int c = 0; c < 4; ++c) q.v[c] = j + c < n ? p[j + c] : 0.0f;
  return q;
}

// Histogram of `bits` bits of |g+e| at `shift`, over the elements whose higher bits equal the
// prefix chosen by the earlier passes. sel[0] = prefix (already shifted down to those bits).
__global__ __launch_bounds__(kCodecBlock) void select_hist_kernel(const float* __restrict__ g,
                                                                  const float* __restrict__ e, int64_t n,
                                                                  int shift, int bits, int prefix_shift,
                                                                  const uint32_t* __restrict__ sel,
                                                                  uint32_t* __restrict__ hist) {
  __shared__ uint32_t lh[kBins];
  for (int i = threadIdx.x; i < kBins; i += kCodecBlock) lh[i] = 0;
  __syncthreads();
  const uint32_t prefix = sel[0];
  const uint32_t mask = (1u << bits) - 1u;
  const int64_t stride = (int64_t)gridDim.x * kCodecBlock;
  const bool vec = ((uintptr_t)g & 15) == 0;
  // four consecutive elements a lane and trip, two trips in flight
  const int64_t quads = (n + 3) / 4;
  for (int64_t q = (int64_t)blockIdx.x * kCodecBlock + threadIdx.x; q < quads; q += 2 * stride) {
    Quad a[2], b[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t j = (q + u * stride) * 4;
      a[u] = load_quad(g, j, n, vec);
      b[u] = load_quad(e, j, n, true);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t j = (q + u * stride) * 4;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (j + c >= n) continue;
        const uint32_t v = abs_bits(a[u].v[c] + b[u].v[c]);
        if (prefix_shift >= 32 || (v >> prefix_shift) == prefix) atomicAdd(&lh[(v >> shift) & mask], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kBins; i += kCodecBlock) {
    const uint32_t c = lh[i];
    if (c) atomicAdd(&hist[i], c);
  }
}

// Finds the bin that holds the k-th largest element, counting from the top bin down; extends the
// prefix by that bin and leaves the rank still to be found inside it. One workgroup; clears the
// histogram. Every thread owns kBins / kCodecBlock consecutive bins: the bins above a thread's
// own are summed with a scan over the threads' totals, and the one thread whose bins straddle k
// walks them. Bin 0 takes whatever no higher bin covers (k larger than the histogram's total).
__global__ __launch_bounds__(kCodecBlock) void select_pick_kernel(uint32_t* __restrict__ hist, int bits,
                                                                  uint32_t* __restrict__ sel, int last) {
  constexpr int kPer = kBins / kCodecBlock;
  __shared__ uint32_t lh[kBins];
  __shared__ uint32_t above[kCodecBlock];      // inclusive suffix sums of the threads' totals
  const int nb = 1 << bits;
  const uint32_t k = sel[1];                   // read by all before the barriers, written by one after
  for (int i = threadIdx.x; i < kBins; i += kCodecBlock) {
    lh[i] = i < nb ? hist[i] : 0;
    hist[i] = 0;
  }
  __syncthreads();
  const int t = threadIdx.x;
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) mine += lh[t * kPer + j];
  above[t] = mine;
  __syncthreads();
  for (int d = 1; d < kCodecBlock; d <<= 1) {
    const uint32_t add = t + d < kCodecBlock ? above[t + d] : 0u;
    __syncthreads();
    above[t] += add;
    __syncthreads();
  }
  const uint32_t higher = above[t] - mine;     // elements in the bins of the threads above this one
  const bool owner = t == 0 ? higher < k : (higher < k && k <= higher + mine);
  if (owner) {
    uint32_t rem = k - higher;                 // rank inside this thread's bins, from the top
    int b = t * kPer + kPer - 1;
    for (; b > t * kPer; --b) {
      const uint32_t c = lh[b];
      if (c >= rem) break;
      rem -= c;
    }
    // b stopped on the bin, or on the thread's lowest bin: for thread 0 that is bin 0, the
    // catch-all; for the others the rank is known to lie inside it
    const uint32_t prefix = (sel[0] << bits) | (uint32_t)b;
    sel[0] = prefix;
    sel[1] = rem;
    if (last) sel[2] = prefix;   // the full bit pattern of tau
  }
}

__global__ void select_begin_kernel(uint32_t* sel, uint32_t k) {
  sel[0] = 0;
  sel[1] = k;
}

// A tile is kCodecTile consecutive elements; inside it each wavefront owns 512 consecutive
// elements and reads them as two rows of 256, a lane four consecutive floats of each (one
// 16-byte access), so every load and store is fully coalesced and the output order is still the
// input order: within a row an element's rank is the number of kept elements in lower lanes (four
// ballots, one per component, and population counts) plus those of the lane's own lower
// components; rows and waves are offset by running totals. A workgroup walks several tiles: a
// few hundred workgroups with many wide accesses in flight stream faster on this memory system
// than one workgroup per tile (6.5-7 TB/s against 4.5 TB/s for plain reads).
constexpr int kCodecRows = kCodecItems / 4;      // rows of 256 elements per wavefront and tile
constexpr int kCodecGrid = 1024;                 // workgroups of the two emit passes

// Per tile: how many elements have |g+e| >= tau. vec: g is 16-byte aligned (e always is).
__global__ __launch_bounds__(kCodecBlock) void emit_count_kernel(const float* __restrict__ g,
                                                                 const float* __restrict__ e, int64_t n,
                                                                 int64_t tiles, bool vec,
                                                                 const uint32_t* __restrict__ sel,
                                                                 int32_t* __restrict__ tile_counts) {
  __shared__ int wave_sum[kCodecBlock / 64];
  const uint32_t tau_bits = sel[2];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int64_t base = tile * kCodecTile + (int64_t)wave * (64 * kCodecItems) + lane * 4;
    Quad a[kCodecRows], b[kCodecRows];
#pragma unroll
    for (int r = 0; r < kCodecRows; ++r) {
      a[r] = load_quad(g, base + r * 256, n, vec);
      b[r] = load_quad(e, base + r * 256, n, true);
    }
    int c = 0;
#pragma unroll
    for (int r = 0; r < kCodecRows; ++r) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        c += (base + r * 256 + k < n && abs_bits(a[r].v[k] + b[r].v[k]) >= tau_bits) ? 1 : 0;
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) c += __shfl_down(c, d, 64);
    if (lane == 0) wave_sum[wave] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
      int s = 0;
#pragma unroll
      for (int w = 0; w < kCodecBlock / 64; ++w) s += wave_sum[w];
      tile_counts[tile] = s;
    }
    __syncthreads();                               // the next tile reuses wave_sum
  }
}

// A lane's elements of a tile of `ROWS` rows of 256 elements per wavefront.
template <int BLOCK, int ROWS>
__device__ __forceinline__ void load_tile(const float* __restrict__ g, const float* __restrict__ e, int64_t n,
                                          int64_t tile, bool vec, Quad (&a)[ROWS], Quad (&b)[ROWS]) {
  constexpr int64_t kTile = BLOCK / 64 * 256 * ROWS;
  const int64_t base = tile * kTile + (threadIdx.x >> 6) * (256 * ROWS) + (threadIdx.x & 63) * 4;
  if (vec && (tile + 1) * kTile <= n) {            // uniform
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      a[r] = whole_quad(g, base + r * 256);
      b[r] = whole_quad(e, base + r * 256);
    }
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      a[r] = load_quad(g, base + r * 256, n, vec);
      b[r] = load_quad(e, base + r * 256, n, true);
    }
  }
}

// One tile, of which a and b are what load_tile loaded: the kept (index, value) pairs in input order
// and the new residual. announce(kept) is called once the tile's count is known, by every thread;
// resolve() yields where the tile's pairs go, to every thread, and is asked for last, when everything
// that does not depend on it is done. A tile's pairs are first gathered in LDS in output order
// and then written out by consecutive lanes, so that the index and value arrays are written in whole
// lines (a lane writing its own few kept elements leaves partly written lines behind).
template <int BLOCK, int ROWS, typename Announce, typename Ahead, typename Resolve>
__device__ __forceinline__ void emit_tile(const Quad (&a)[ROWS], const Quad (&b)[ROWS], int64_t n, int64_t tile,
                                          uint32_t tau_bits, long long* __restrict__ idx, float* __restrict__ val,
                                          float* __restrict__ e_next, Announce announce, Ahead ahead, Resolve resolve) {
  constexpr int kWaveElems = 256 * ROWS;
  constexpr int kWaves = BLOCK / 64;
  constexpr int kTile = kWaves * kWaveElems;
  static_assert(kTile <= 65536, "a place inside the tile is kept in 16 bits");
  __shared__ int wave_sum[kWaves];
  __shared__ uint16_t kept_at[kTile];              // element's place inside the tile
  __shared__ float kept_val[kTile];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int local = wave * kWaveElems + lane * 4;
  const int64_t base = tile * kTile + local;
  Quad f[ROWS];
  unsigned long long masks[ROWS][4];
  int wave_total = 0;
  const bool whole = (tile + 1) * kTile <= n;      // uniform
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f[r].v[k] = a[r].v[k] + b[r].v[k];
      masks[r][k] = __ballot((whole || base + r * 256 + k < n) && abs_bits(f[r].v[k]) >= tau_bits);
      wave_total += __popcll(masks[r][k]);
    }
  }
  if (lane == 0) wave_sum[wave] = wave_total;
  __syncthreads();
  int off = 0, count = 0;                          // inside the tile's stretch of the output
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) off += wave_sum[w];
    count += wave_sum[w];
  }
  announce(count);
  ahead();
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int64_t j = base + r * 256;
    // kept elements of lower lanes, all four components of each
    int at = off;
    int row_total = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      at += __popcll(masks[r][k] & below);
      row_total += __popcll(masks[r][k]);
    }
    float rest[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool keep = (masks[r][k] >> lane) & 1ull;
      if (keep) {
        kept_at[at] = (uint16_t)(local + r * 256 + k);
        kept_val[at] = f[r].v[k];
        ++at;
      }
      rest[k] = keep ? 0.0f : f[r].v[k];           // t/math.cc:1098-1123 : |x| < th keeps x
    }
    if (whole || j + 3 < n) {
      const vfloat4 out = {rest[0], rest[1], rest[2], rest[3]};
      __builtin_nontemporal_store(out, reinterpret_cast<vfloat4*>(e_next + j));
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (j + k < n) e_next[j + k] = rest[k];
    }
    off += row_total;
  }
  const int64_t out0 = resolve(count);             // has a barrier: the pairs are in LDS
  const int64_t tile_base = tile * kTile;
  // (counted from a multiple of 64 of the output, so that a wavefront's stores are whole lines)
  for (int i = (int)threadIdx.x - (int)(out0 & 63); i < count; i += BLOCK) {
    if (i < 0) continue;
    __builtin_nontemporal_store((long long)(tile_base + kept_at[i]), idx + out0 + i);
    __builtin_nontemporal_store(kept_val[i], val + out0 + i);
  }
  __syncthreads();                                 // the next tile reuses the LDS arrays
}

__global__ __launch_bounds__(kCodecBlock) void emit_write_kernel(
    const float* __restrict__ g, const float* __restrict__ e, int64_t n, int64_t tiles, bool vec,
    const uint32_t* __restrict__ sel, const int32_t* __restrict__ tile_offsets, long long* __restrict__ idx,
    float* __restrict__ val, float* __restrict__ e_next) {
  const uint32_t tau_bits = sel[2];
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    Quad a[kCodecRows], b[kCodecRows];
    load_tile<kCodecBlock>(g, e, n, tile, vec, a, b);
    emit_tile<kCodecBlock>(a, b, n, tile, tau_bits, idx, val, e_next, [](int) {}, [] {},
                           [&](int) -> int64_t {
                             __syncthreads();
                             return tile_offsets[tile];
                           });
  }
}

// The whole emit step in one pass: gradient and residual are read once (a count pass ahead of the write pass read
// them twice: 536 MB more for 67 million elements, 95 of 333 us with the scan). Where a tile's pairs go is the number
// of pairs in the tiles before it, which the workgroups tell one another: tile_state[t] holds what tile t keeps as
// soon as that is known, and what tiles 0..t keep together once that is. A tile looks back over its predecessors, 64
// at a time, as far as the nearest whose total is known. Tiles are handed out by a counter in ascending order, so
// every predecessor of a tile is held by a workgroup that already runs, and it announces its count before it waits
// for anything: every wait ends. An announcement carries the number of the call, so the array is never cleared; the
// last workgroup to leave puts the counter back to zero.
// A workgroup takes its next tile's number, and asks for its elements, ahead of writing the one it has: a tile that
// is held but not announced is waited for by later tiles only, and its workgroup waits for earlier ones, so the
// lowest such tile's turn always comes.
// What bounds it is the rate of a copy: 67 million elements, of which 33 million are kept, 1.27 GB, 217 us (5.8
// TB/s). 243 us with each tile's loads behind the tile before it, two workgroups a compute unit, 8192 elements a
// tile; with the loads ahead, tiles of 8192 / 16,384 elements and 192, 256, 320, 384 workgroups 255, 222, 250, 248 /
// 230, 217, 216, 217: the fewer tiles are on their way, the less far a tile has to look back. The counter serves one
// workgroup after the other, some 15 ns each, which is what smaller tiles wait for (573 and 331 us in tiles of 2048
// and 4096); tensors that give few workgroups a tile are better off with them. A blocking step, us, as before / in
// tiles of 4096 / 8192 / 16,384: 300,000 elements 15.6 / 14.2 / 16.2 / 19.2, a million 17.6 / 19.1 / 17.4 / 19.9, 4
// million 31.9 / 31.6 / 29.2 / 32.6, 16 million 74 / 89 / 67 / 70, 33 million 132 / 170 / 119 / 119, 67 million 252 /
// 331 / 229 / 224. Above: compress, push and pull of 33 / 40 / 50 / 67 / 100 / 134 / 200 million elements in tiles of
// 8192 380 / 446 / 547 / 722 / 1073 / 1432 / 2139 us, of 16,384 373 / 442 / 547 / 710 / 1062 / 1422 / 2146: one in a
// hundred or nothing.
constexpr int64_t kSingleShort = (int64_t)1 << 19;
constexpr int64_t kSingleLong = (int64_t)1 << 25;
constexpr int kSingleBlock = 512;
constexpr int single_tile(int rows) { return (kSingleBlock / 64) * 256 * rows; }
constexpr int kSingleGrid = 256;
constexpr uint32_t kTileCount = 1u, kTileTotal = 2u;   // what the low word is: the tile's own count, or all up to it
constexpr uint32_t kMaxEmitCalls = 1u << 30;

__device__ __forceinline__ void tell(unsigned long long* state, uint32_t call, uint32_t what, uint32_t value) {
  __hip_atomic_store(state, ((unsigned long long)(call << 2 | what) << 32) | value, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

template <int ROWS>
__global__ __launch_bounds__(kSingleBlock) void emit_single_kernel(
    const float* __restrict__ g, const float* __restrict__ e, int64_t n, uint32_t tiles, bool vec,
    uint32_t* __restrict__ sel, unsigned long long* tile_state, uint32_t* tickets, uint32_t call,
    long long* __restrict__ idx, float* __restrict__ val, float* __restrict__ e_next,
    uint32_t* __restrict__ host_sel) {
  __shared__ uint32_t s_tile, s_before;
  const uint32_t tau_bits = sel[2];
  const int lane = threadIdx.x & 63;
  const bool once = tiles <= gridDim.x;            // a tile a workgroup: the counter is spared the second round
  if (threadIdx.x == 0) s_tile = atomicAdd(&tickets[0], 1u);
  __syncthreads();
  uint32_t tile = s_tile;
  __syncthreads();
  Quad a[ROWS], b[ROWS];
  if (tile < tiles) load_tile<kSingleBlock>(g, e, n, tile, vec, a, b);
  while (tile < tiles) {                           // the whole workgroup
    if (threadIdx.x == 0) s_tile = once ? tiles : atomicAdd(&tickets[0], 1u);
    uint32_t next = tiles;
    emit_tile<kSingleBlock>(
        a, b, n, tile, tau_bits, idx, val, e_next,
        [&](int count) {
          if (threadIdx.x == 0) tell(&tile_state[tile], call, tile == 0 ? kTileTotal : kTileCount, (uint32_t)count);
        },
        [&] {
          next = s_tile;                           // (a barrier behind its store)
          if (next < tiles) load_tile<kSingleBlock>(g, e, n, next, vec, a, b);
        },
        [&](int count) -> int64_t {
          if (threadIdx.x < 64) {
            uint32_t before = 0;
            int64_t base = (int64_t)tile - 1;      // lane l looks at tile base - l
            bool more = tile > 0;
            while (more) {
              const int64_t j = base - lane;
              unsigned long long word = (unsigned long long)(call << 2 | kTileTotal) << 32;   // before the first tile: nothing
              if (j >= 0) word = __hip_atomic_load(&tile_state[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              const uint32_t tag = (uint32_t)(word >> 32);
              const unsigned long long known = __ballot(tag == (call << 2 | kTileTotal));
              const unsigned long long open = __ballot((tag >> 2) != call);
              const int last = known ? __ffsll(known) - 1 : 63;   // the farthest tile that counts
              const unsigned long long need = last == 63 ? ~0ull : ((1ull << (last + 1)) - 1ull);
              if (open & need) {                   // one of them has not announced yet
                __builtin_amdgcn_s_sleep(1);
                continue;
              }
              uint32_t v = lane <= last ? (uint32_t)word : 0u;
#pragma unroll
              for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
              before += __shfl(v, 0);
              more = known == 0ull;
              base -= 64;
            }
            if (threadIdx.x == 0) {
              if (tile > 0) tell(&tile_state[tile], call, kTileTotal, before + (uint32_t)count);
              s_before = before;
              if (tile == tiles - 1) {             // the count and the threshold, where the host reads them
                sel[3] = before + (uint32_t)count;
                host_sel[2] = tau_bits;
                host_sel[3] = before + (uint32_t)count;
              }
            }
          }
          __syncthreads();
          return s_before;
        });
    tile = next;
  }
  if (threadIdx.x == 0 && atomicAdd(&tickets[1], 1u) == gridDim.x - 1) {
    __hip_atomic_store(&tickets[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&tickets[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---- densify in one pass over the output ------------------------------------------------------
// starts[from..to] = value for every lane's own range (empty: from > to); the whole wavefront calls.
// A lane writes a few tiles itself. Long ranges, the empty tiles of a tensor with few or clustered
// entries, are written by all lanes together, one range after the other: 100 entries at the front
// of 67 million elements leave 32,767 tiles behind the last one, a push of them 1196 us when
// one lane wrote them all, 226 us this way.
__device__ __forceinline__ void coo_start_tiles(uint32_t* __restrict__ starts, int from, int to, uint32_t value) {
  constexpr int kAlone = 8;
  const int lane = threadIdx.x & 63;
  const bool together = to - from >= kAlone;
  if (!together)
    for (int t = from; t <= to; ++t) starts[t] = value;
  for (unsigned long long left = __ballot(together); left != 0ull; left &= left - 1) {
    const int l = __ffsll(left) - 1;
    const int a = __shfl(from, l), b = __shfl(to, l);
    const uint32_t v = (uint32_t)__shfl((int)value, l);
    for (int t = a + lane; t <= b; t += 64) starts[t] = v;
  }
}

// Says that the indices are unordered. Stores to one word are served one after the other, some 30 ns each, and where
// the entries come in no order everyone has one: whoever finds the word written spares its own.
__device__ __forceinline__ void coo_raise(const CooTiles& out) {
  if (!coo_unordered(out)) __hip_atomic_store(out.unordered, out.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where each tile's entries begin: the first entry of a tile, and the first one behind the empty
// tiles before it, name themselves. A wavefront takes chunks of 256 entries in two rows of 128, a lane two
// neighbours of each in one 16-byte load (whole lines an access); the entry before a lane's two is
// its neighbour's second.
constexpr int kCooRows = 2;
constexpr int kCooChunk = kCooRows * 128;
typedef long long coo_pair __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void coo_load_chunk(const long long* __restrict__ idx, int64_t base, int64_t nnz, bool vec,
                                               coo_pair (&cur)[kCooRows]) {
  const int lane = threadIdx.x & 63;
  const bool whole = vec && base + kCooChunk <= nnz;   // uniform
#pragma unroll
  for (int r = 0; r < kCooRows; ++r) {
    const int64_t j = base + r * 128 + lane * 2;
    if (whole) {
      cur[r] = __builtin_nontemporal_load(reinterpret_cast<const coo_pair*>(idx + j));
    } else {
      cur[r][0] = idx[j < nnz ? j : nnz - 1];
      cur[r][1] = idx[j + 1 < nnz ? j + 1 : nnz - 1];
    }
  }
}

// The starts that a row of 128 entries from entry j of a lane on names; `last`: the entry before the row, then its
// last one. False where an entry does not ascend or lies outside [0, n).
__device__ __forceinline__ bool coo_row_starts(const coo_pair& cur, int64_t j, int64_t nnz, int64_t n, long long& last,
                                               const CooTiles& out) {
  const int lane = threadIdx.x & 63;
  long long prev = __shfl_up(cur[1], 1);
  if (lane == 0) prev = last;
  last = __shfl(cur[1], 63);
  // nearly every lane: two more entries of the tile the one before is in
  const bool quick = j + 2 < nnz && prev >= 0 && prev < cur[0] && cur[0] < cur[1] && cur[1] < n &&
                     (prev ^ cur[1]) < kCooTile;
  if (__ballot(!quick) == 0ull) return true;
  // A row that holds a wrong entry names no starts, which nobody will look at: where the entries come in no order,
  // every second one would write those of hundreds of tiles (half a million shuffled entries of 2 million
  // elements: 119 us with those, 9 without).
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const long long c = cur[i], before = i ? cur[0] : prev;
    bad = bad || (!quick && j + i < nnz && (c < 0 || c <= before || c >= n));   // before may be negative, and wrong, itself
  }
  if (__ballot(bad) != 0ull) return false;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool mine = !quick && j + i < nnz;
    const long long c = cur[i];
    int from = 1, to = 0, tile = 0;
    if (mine) {
      tile = (int)(c / kCooTile);
      from = prev < 0 ? 0 : (int)(prev / kCooTile) + 1;
      to = tile;
    }
    coo_start_tiles(out.starts, from, to, (uint32_t)(j + i));
    const bool end = mine && j + i == nnz - 1;
    if (__ballot(end) != 0ull)
      coo_start_tiles(out.starts, end ? tile + 1 : 1, end ? (int)out.tiles : 0, (uint32_t)nnz);
    prev = c;
  }
  return true;
}

__global__ __launch_bounds__(kCodecBlock) void coo_tiles_bounds_kernel(const long long* __restrict__ idx,
                                                                       int64_t nnz, int64_t n, bool vec, CooTiles out) {
  const int64_t step = (int64_t)gridDim.x * (kCodecBlock / 64) * kCooChunk;
  for (int64_t base = ((int64_t)blockIdx.x * (kCodecBlock / 64) + threadIdx.x / 64) * kCooChunk; base < nnz;
       base += step) {                               // a wavefront's lanes stay together
    coo_pair cur[kCooRows];
    coo_load_chunk(idx, base, nnz, vec, cur);
    long long last = base ? idx[base - 1] : -1;      // the entry before the row
    bool fine = true;
#pragma unroll
    for (int r = 0; r < kCooRows; ++r)
      fine &= coo_row_starts(cur[r], base + r * 128 + (threadIdx.x & 63) * 2, nnz, n, last, out);
    if (!fine) coo_raise(out);
  }
}

// The same, and a bit for every element that an entry names, so that who walks the tiles need not read the indices
// again. A wavefront takes a run of consecutive chunks and carries the words that later entries may share along:
// every word is written once, by the wavefront that holds the first of the entries behind the word before it, and
// nothing has to be cleared ahead. Words of tiles without entries are not written. The bits meet in LDS, in a window
// of up to two tiles' words that moves on by 64 of them, a line of memory; chunks wider than that take several
// windows. What bounds it is the read of the indices, and next to it instruction issue: nearly every chunk of a
// gradient that keeps a quarter of its elements is an easy one (no gap of a tile or more, all of it in the window,
// not the run's last), and those take a third of the general path's 200 vector instructions. 33 million entries among
// 67 million elements: the general path alone 58 us, with the easy one 55, with lines instead of each chunk's words
// 52 in runs of 4 (2, 8, 16: 55, 53, 55); without bits 44.6. The update that follows takes 317 us for 365.
constexpr int kCooRun = 4;                           // chunks of a wavefront
constexpr int kCooWindow = 128;

__global__ __launch_bounds__(kCodecBlock) void coo_bits_kernel(const long long* __restrict__ idx, int64_t nnz, int64_t n,
                                                               bool vec, CooTiles out) {
  static_assert(kCooTile == 64 * 32, "a tile's bits are a word a lane");
  __shared__ uint32_t wave_words[(kCodecBlock / 64) * kCooWindow];
  const int lane = threadIdx.x & 63;
  uint32_t* words = &wave_words[(threadIdx.x >> 6) * kCooWindow];
  words[lane] = 0u;
  words[lane + 64] = 0u;
  wave_lds_order();
  const int64_t run = ((int64_t)blockIdx.x * (kCodecBlock / 64) + threadIdx.x / 64) * (kCooRun * kCooChunk);
  if (run >= nnz) return;
  const int64_t stop = run + kCooRun * kCooChunk < nnz ? run + kCooRun * kCooChunk : nnz;
  coo_pair cur[kCooRows], ahead[kCooRows];
  coo_load_chunk(idx, run, nnz, vec, cur);
  long long last = run ? idx[run - 1] : -1;          // the entry before the chunk
  // entries of the run behind this one may lie in this one's last word
  const long long after = lane < 32 && stop + lane < nnz ? idx[stop + lane] : -1;
  bool fine = true;
  const bool small = n <= (int64_t)0xFFFFFFFF;
  // the first word that is not written yet; words[i]: what is known of word from + i, of at most 64 between two chunks
  uint32_t from = last < 0 ? 0u : (uint32_t)(last >> 5) + 1u;
  for (int64_t base = run; base < stop; base += kCooChunk) {
    if (base + kCooChunk < stop) coo_load_chunk(idx, base + kCooChunk, nnz, vec, ahead);
    const int64_t j = base + lane * 2;
    const bool ends = base + kCooChunk >= stop;
    if (small && !ends && last >= 0) {               // uniform: indices are their low halves, if in range
      uint32_t prev[kCooRows], most = 0u, high = 0u, before = (uint32_t)last;
#pragma unroll
      for (int r = 0; r < kCooRows; ++r) {
        const uint32_t c0 = (uint32_t)cur[r][0], c1 = (uint32_t)cur[r][1];
        // the entry before a lane's two: its lower neighbour's second (wave_shr:1), the lowest lane's the row before's last
        prev[r] = (uint32_t)__builtin_amdgcn_update_dpp((int)before, (int)c1, 0x138, 0xf, 0xf, false);
        before = (uint32_t)__builtin_amdgcn_readlane((int)c1, 63);
        high |= (uint32_t)(cur[r][0] >> 32) | (uint32_t)(cur[r][1] >> 32);
        most = max(most, max(c0 - prev[r] - 1u, c1 - c0 - 1u));
      }
      const uint32_t top = before >> 5;
      const bool easy = __ballot(high != 0u || most >= (uint32_t)kCooTile - 1u) == 0ull && before < (uint32_t)n &&
                        top - from < (uint32_t)kCooWindow;
      if (easy) {
#pragma unroll
        for (int r = 0; r < kCooRows; ++r) {
          const uint32_t c0 = (uint32_t)cur[r][0], c1 = (uint32_t)cur[r][1];
          const uint32_t t = prev[r] >> 11, t0 = c0 >> 11, t1 = c1 >> 11;
          if (t != t1) {                             // a lane in a tile's length: no gap passes over a whole tile
            if (t != t0) out.starts[t0] = (uint32_t)(j + r * 128);
            if (t0 != t1) out.starts[t1] = (uint32_t)(j + r * 128 + 1);
          }
          const uint32_t w0 = c0 >> 5, w1 = c1 >> 5, b0 = 1u << (c0 & 31u), b1 = 1u << (c1 & 31u);
          // (the first chunk's first entries may lie in the word before, which another wavefront writes)
          if (w0 != w1 && w0 - from < (uint32_t)kCooWindow) atomicOr(&words[w0 - from], b0);
          if (w1 - from < (uint32_t)kCooWindow) atomicOr(&words[w1 - from], w0 == w1 ? b0 | b1 : b1);
        }
        wave_lds_order();
        if (top - from >= 64u) {                     // a line of complete words, and the window moves on by it
          out.bits[from + lane] = words[lane];
          words[lane] = words[lane + 64];
          words[lane + 64] = 0u;
          from += 64u;
          wave_lds_order();
        }
        last = (long long)before;
#pragma unroll
        for (int r = 0; r < kCooRows; ++r) cur[r] = ahead[r];
        continue;
      }
    }
#pragma unroll
    for (int r = 0; r < kCooRows; ++r) fine &= coo_row_starts(cur[r], j + r * 128, nnz, n, last, out);
    if (!fine) break;                                // the bits will not be looked at
    const uint32_t top = (uint32_t)(last >> 5);
    const bool closes = base + kCooChunk >= nnz;     // behind the very last entry: the rest of its tile
    const uint32_t to = closes ? (top | 63u) + 1u : ends ? top + 1u : top;   // words [from, to) are complete
    uint32_t w[2 * kCooRows], bit[2 * kCooRows];
    bool on[2 * kCooRows];
#pragma unroll
    for (int r = 0; r < kCooRows; ++r) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t c = (uint32_t)cur[r][i];      // (n / 32 words: the low half says which bit, both which word)
        w[2 * r + i] = (uint32_t)(cur[r][i] >> 5);
        bit[2 * r + i] = 1u << (c & 31u);
        on[2 * r + i] = j + r * 128 + i < nnz;
      }
      if (on[2 * r + 1] && w[2 * r] == w[2 * r + 1]) {
        bit[2 * r + 1] |= bit[2 * r];
        on[2 * r] = false;
      }
    }
    const bool shares = ends && after > last && (after >> 5) == (long long)top;
    for (uint32_t at = from;;) {                     // the window: words from `at` to the end of the next tile
      const uint32_t behind = (at & ~63u) + kCooWindow, wide = behind - at;
#pragma unroll
      for (int i = 0; i < 2 * kCooRows; ++i)
        if (on[i] && w[i] - at < wide) atomicOr(&words[w[i] - at], bit[i]);
      if (shares && top - at < wide) atomicOr(&words[top - at], 1u << (after & 31));
      wave_lds_order();
      const uint32_t v0 = words[lane], v1 = words[lane + 64];
      if ((uint32_t)lane < wide && at + lane < to) out.bits[at + lane] = v0;
      if ((uint32_t)lane + 64u < wide && at + lane + 64u < to) out.bits[at + lane + 64u] = v1;
      words[lane] = 0u;
      words[lane + 64] = 0u;
      wave_lds_order();
      if (to <= behind && top < behind) {
        if (!ends) {                                 // the open word goes on as the next chunk's first
          const uint32_t open = (uint32_t)__shfl((int)(top - at < 64u ? v0 : v1), (int)((top - at) & 63u));
          if (lane == 0) words[0] = open;
          wave_lds_order();
        }
        break;
      }
      uint32_t next = top;                           // the nearest tile that has an entry (or is to be ended)
#pragma unroll
      for (int i = 0; i < 2 * kCooRows; ++i)
        if (on[i] && w[i] >= behind && w[i] < next) next = w[i];
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) next = min(next, (uint32_t)__shfl_xor((int)next, d));
      next &= ~63u;
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)(next < behind ? behind : next));
    }
    from = from > top ? from : top;
#pragma unroll
    for (int r = 0; r < kCooRows; ++r) cur[r] = ahead[r];
  }
  if (!fine) coo_raise(out);
}

// One workgroup per output tile: the tile is put together in LDS (zeros, then the tile's entries,
// whose range is known, so their loads do not wait for one another) and leaves in whole lines,
// past the caches.
__global__ __launch_bounds__(kCodecBlock) void coo_tiles_write_kernel(const long long* __restrict__ idx,
                                                                      const float* __restrict__ val,
                                                                      float* __restrict__ dense, int64_t n,
                                                                      CooTiles tiles) {
  if (coo_unordered(tiles)) return;              // the scatter launches that follow do the work
  __shared__ __align__(16) float tile[kCooTile];
  const int64_t base = (int64_t)blockIdx.x * kCooTile;
  const uint32_t start = tiles.starts[blockIdx.x];
  const uint32_t end = tiles.starts[blockIdx.x + 1];
  for (int i = threadIdx.x; i < kCooTile / 4; i += kCodecBlock)
    reinterpret_cast<float4*>(tile)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  __syncthreads();
  for (int64_t j0 = (int64_t)start + threadIdx.x; j0 < (int64_t)end; j0 += 4 * kCodecBlock) {
    long long at[4];
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t j = j0 + u * kCodecBlock;
      if (j < (int64_t)end) {
        at[u] = __builtin_nontemporal_load(idx + j);
        v[u] = __builtin_nontemporal_load(val + j);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j0 + u * kCodecBlock < (int64_t)end) tile[at[u] - base] = v[u];
  }
  __syncthreads();
  const int64_t left = n - base;
  const int cnt = left < kCooTile ? (int)left : kCooTile;
  if (cnt == kCooTile && (((uintptr_t)dense) & 15) == 0) {
    typedef float tile4 __attribute__((ext_vector_type(4)));
    for (int i = threadIdx.x; i < kCooTile / 4; i += kCodecBlock)
      __builtin_nontemporal_store(reinterpret_cast<const tile4*>(tile)[i], reinterpret_cast<tile4*>(dense + base) + i);
  } else {
    for (int i = threadIdx.x; i < cnt; i += kCodecBlock) dense[base + i] = tile[i];
  }
}

// The same from the bits: a wavefront's lanes see for themselves which entries are theirs, nothing passes through LDS.
__global__ __launch_bounds__(kCodecBlock) void coo_bits_write_kernel(const float* __restrict__ val,
                                                                     float* __restrict__ dense, int64_t n,
                                                                     CooTiles tiles) {
  if (coo_unordered(tiles)) return;
  const int64_t base = (int64_t)blockIdx.x * kCooTile;
  const uint32_t start = tiles.starts[blockIdx.x];
  const uint32_t end = tiles.starts[blockIdx.x + 1];
  const CooTileBits tile(tiles.bits[(size_t)blockIdx.x * (kCooTile / 32) + (threadIdx.x & 63)]);
  const bool whole = base + kCooTile <= n && (((uintptr_t)dense) & 15) == 0;
#pragma unroll
  for (int i = 0; i < kCooTile / 4 / kCodecBlock; ++i) {
    const int q = i * kCodecBlock + threadIdx.x;
    float g[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (end > start) tile.quad(q, val, start, end, g);   // uniform
    const int64_t at = base + 4 * q;
    if (whole) {
      __builtin_nontemporal_store((vfloat4){g[0], g[1], g[2], g[3]}, reinterpret_cast<vfloat4*>(dense + at));
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (at + c < n) dense[at + c] = g[c];
    }
  }
}

__global__ __launch_bounds__(kCodecBlock) void coo_zero_if_kernel(float* __restrict__ dense, int64_t n,
                                                                  CooTiles tiles) {
  if (!coo_unordered(tiles)) return;
  const int64_t step = (int64_t)gridDim.x * kCodecBlock;
  for (int64_t i = (int64_t)blockIdx.x * kCodecBlock + threadIdx.x; i < n; i += step) dense[i] = 0.0f;
}

// dense[idx[j]] += val[j]; repeated indices add up (t/math.cc:1043), indices outside [0, n) are
// skipped. kAddIf: only where the tiles were found to be unordered. kAddLook: and says whether tiles would be.
constexpr int kAddAll = 0, kAddIf = 1, kAddLook = 2;
template <int WHAT>
__global__ __launch_bounds__(kCodecBlock) void coo_add_kernel(const long long* __restrict__ idx,
                                                              const float* __restrict__ val, int64_t nnz,
                                                              float* __restrict__ dense, int64_t n, CooTiles tiles) {
  if (WHAT == kAddIf && !coo_unordered(tiles)) return;
  const int64_t step = (int64_t)gridDim.x * kCodecBlock, first = (int64_t)blockIdx.x * kCodecBlock + threadIdx.x;
  if (WHAT == kAddLook) {              // (ahead of the additions: behind them all workgroups would raise the flag at once)
    bool wrong = false;
    for (int64_t j = first; j < nnz; j += step) {
      const long long i = idx[j];
      wrong = wrong || i < 0 || i >= n || (j > 0 && idx[j - 1] >= i);
    }
    if (__syncthreads_or(wrong) && threadIdx.x == 0) coo_raise(tiles);
  }
  for (int64_t j = first; j < nnz; j += step) {
    const long long i = idx[j];
    if (i < 0 || i >= n) continue;
    unsafeAtomicAdd(&dense[i], val[j]);   // hardware fp32 add, no CAS loop
  }
}

// From an entry in this many elements on an entry's place is kept as a bit: 1/64 of the indices' bytes at an entry an
// element, an eighth at one in eight, and who walks the tiles reads that. 67 million elements, an entry in 1 / 2 / 4
// / 8 / 12 of them, blocking, us, by the indices and by bits: Adam push 560 / 452 / 382 / 356 / 343 and 468 / 404 /
// 369 / 355 / 349, decode 276 / 163 / 114 / 91 / 82 and 192 / 121 / 91 / 77 / 71. In small tensors the indices lie in
// the caches when they are read again, and the bits' launch is the longer one: an Adam push of 20,000 / 300,000 / 2
// million / 4 million elements, an entry in four, 18.1 / 17.3 / 23.7 / 34.0 us by bits and 15.1 / 15.2 / 21.7 / 34.5
// by the indices; four in five 17.9 / 16.9 / 24.7 / 36.7 and 15.4 / 15.5 / 24.6 / 39.9. Around the line, 2.5 / 3 /
// 3.5 / 4 / 5 million elements: an entry in eight 27.9 / 31.4 / 34.1 / 36.3 / 39.9 by bits and 25.2 / 29.4 / 33.6 /
// 35.6 / 40.0, in four 27.4 / 31.2 / 33.2 / 35.7 / 40.2 and 25.8 / 30.2 / 33.9 / 35.9 / 40.6, four in five 29.1 /
// 32.6 / 35.0 / 38.0 / 42.5 and 31.0 / 34.9 / 40.2 / 42.0 / 48.4.
constexpr int64_t kCooBitsFrom = 8;
constexpr int64_t kCooBitsLarge = (int64_t)3 << 20;
// A decode is two short launches, of which the bits make the first one 3 us longer whatever the tensor's size: what they
// spare has to be more entries than that. By the indices / by bits, us: an entry in eight of 4.2 / 8 / 12 / 16 / 24 million
// elements 23.3 / 27.2 / 31.5 / 35.5 / 43.3 and 26.6 / 28.8 / 31.6 / 34.6 / 40.6, in four of 4.2 / 6 / 8 / 12 million 24.4 /
// 27.4 / 29.7 / 35.4 and 26.1 / 27.6 / 28.9 / 32.1, in two of 4.2 / 6 million 27.1 / 30.9 and 26.1 / 28.4; 512 elements in a
// row of each 4096, of 8 / 12 / 16 / 24 million, 28.1 / 32.3 / 36.3 / 44.3 and 30.2 / 33.7 / 36.5 / 43.8.
constexpr int64_t kCooBitsDecode = (int64_t)7 << 18;

static unsigned stream_grid(int64_t n) {
  int64_t blocks = (n + kCodecBlock - 1) / kCodecBlock;
  if (blocks > 256 * 8) blocks = 256 * 8;
  if (blocks < 1) blocks = 1;
  return (unsigned)blocks;
}

// Every call of the process has another tag, so nothing lowers the flag, in new memory neither: what happens to be
// there is some other call's, or, should it be this one's, says 'unordered', which is slow and right for any indices.
static std::atomic<uint32_t> g_coo_tag{0};

int32_t coo_new_tag(CooWork* work, int64_t n, CooTiles* out) {
  uint32_t* room = work->lent;
  if (!room) {
    KRK_TRY(work->buffer.reserve(coo_tile_words(n) * sizeof(uint32_t)));
    room = work->buffer.as<uint32_t>();
  }
  out->unordered = room;
  out->starts = room + 1;
  out->tiles = (uint32_t)((n + kCooTile - 1) / kCooTile);
  out->bits = nullptr;
  out->told = nullptr;
  out->tag = g_coo_tag.fetch_add(1, std::memory_order_relaxed) + 1;
  return KRK_SUCCESS;
}

int32_t coo_find_tiles(CooWork* work, const long long* d_idx, int64_t nnz, int64_t n, bool update, CooTiles* out,
                       hipStream_t stream) {
  KRK_TRY(coo_new_tag(work, n, out));
  bool with_bits = nnz * kCooBitsFrom >= n && (update ? n >= kCooBitsLarge : nnz >= kCooBitsDecode);
  if (with_bits && work->bits.reserve((size_t)out->tiles * (kCooTile / 8)) != KRK_SUCCESS) {
    (void)hipGetLastError();                         // no failure of a later launch
    with_bits = false;                               // the indices are read again, then
  }
  if (with_bits) out->bits = work->bits.as<uint32_t>();
  const bool vec = ((uintptr_t)d_idx & 15) == 0;
  const dim3 block(kCodecBlock);
  if (with_bits) {
    constexpr int64_t per = (int64_t)(kCodecBlock / 64) * kCooRun * kCooChunk;
    hipLaunchKernelGGL(coo_bits_kernel, dim3((unsigned)((nnz + per - 1) / per)), block, 0, stream, d_idx, nnz, n, vec,
                       *out);
  } else {
    hipLaunchKernelGGL(coo_tiles_bounds_kernel, dim3(stream_grid((nnz + 3) / 4)), block, 0, stream, d_idx, nnz, n, vec,
                       *out);
  }
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

// A few workgroups that stride over the entries: when the tiles did the work they only look at the
// flag and leave (2048 of them took 4.7 us a launch for that).
static dim3 rare_grid(int64_t n) { return dim3(std::min(stream_grid(n), 512u)); }

int32_t coo_scatter_if_unordered(const CooTiles& tiles, const long long* d_idx, const float* d_val, int64_t nnz,
                                 float* d_dense, int64_t n, hipStream_t stream) {
  const dim3 block(kCodecBlock);
  hipLaunchKernelGGL(coo_zero_if_kernel, rare_grid(n), block, 0, stream, d_dense, n, tiles);
  hipLaunchKernelGGL(coo_add_kernel<kAddIf>, rare_grid(nnz), block, 0, stream, d_idx, d_val, nnz, d_dense, n, tiles);
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

int32_t coo_densify(CooWork* work, const long long* d_idx, const float* d_val, int64_t nnz, float* d_dense, int64_t n,
                    hipStream_t stream, const CooTiles* look) {
  if (n <= 0) return KRK_SUCCESS;
  const dim3 block(kCodecBlock);
  if (!coo_tiled(n, nnz) || nnz == 0) {
    KRK_HIP(hipMemsetAsync(d_dense, 0, (size_t)n * sizeof(float), stream));   // t/math.cc:1066 dense.Zero()
    const dim3 grid((unsigned)((nnz + kCodecBlock - 1) / kCodecBlock));
    if (nnz && look)
      hipLaunchKernelGGL(coo_add_kernel<kAddLook>, grid, block, 0, stream, d_idx, d_val, nnz, d_dense, n, *look);
    else if (nnz)
      hipLaunchKernelGGL(coo_add_kernel<kAddAll>, grid, block, 0, stream, d_idx, d_val, nnz, d_dense, n, CooTiles{});
    KRK_HIP(hipGetLastError());
    return KRK_SUCCESS;
  }
  CooTiles tiles;
  KRK_TRY(coo_find_tiles(work, d_idx, nnz, n, false, &tiles, stream));
  if (tiles.bits) {
    hipLaunchKernelGGL(coo_bits_write_kernel, dim3(tiles.tiles), block, 0, stream, d_val, d_dense, n, tiles);
  } else {
    hipLaunchKernelGGL(coo_tiles_write_kernel, dim3(tiles.tiles), block, 0, stream, d_idx, d_val, d_dense, n, tiles);
  }
  KRK_HIP(hipGetLastError());
  return coo_scatter_if_unordered(tiles, d_idx, d_val, nnz, d_dense, n, stream);
}

}  // namespace krk

using namespace krk;

static std::mutex g_densify_mu;          // krk_coo_to_dense owns no object: one shared work buffer
static CooWork g_densify_work;
// The bits of up to 2^31 elements are kept between calls. Giving them back and asking for them again takes 350 us, a
// tenth of a call on more elements than that.
constexpr size_t kDensifyBitsKept = (size_t)256 << 20;

extern "C" {

int32_t krk_dct_create(int64_t n, krk_dct** out) {
  if (!out || n < 0 || n >= (int64_t)0x7FFFFFFF) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  krk_dct* s = new (std::nothrow) krk_dct();
  if (!s) return KRK_E_DEVICE;
  s->n = n;
  s->tiles = (n + kCodecTile - 1) / kCodecTile;
  if (s->tiles < 1) s->tiles = 1;
  int32_t rc = s->open_stream();
  if (rc == KRK_SUCCESS) {
    const size_t nb = (size_t)(n ? n : 1) * sizeof(float);
    hipError_t e = hipMalloc((void**)&s->e, nb);
    if (e == hipSuccess) e = hipMalloc((void**)&s->e_next, nb);
    if (e == hipSuccess) e = hipMalloc((void**)&s->sel, 64);
    if (e == hipSuccess) e = hipMalloc((void**)&s->hist, kBins * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc((void**)&s->tile_counts, (size_t)s->tiles * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc((void**)&s->tile_offsets, (size_t)s->tiles * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&s->scan_tmp, scan_scratch_bytes(s->tiles));
    const size_t state_b = (size_t)((n + single_tile(2) - 1) / single_tile(2) + 1) * sizeof(unsigned long long);
    if (e == hipSuccess) e = hipMalloc((void**)&s->tile_state, state_b);
    if (e == hipSuccess) e = hipMalloc((void**)&s->tickets, 64);
    if (e == hipSuccess) e = hipMemsetAsync(s->tile_state, 0, state_b, s->stream);
    if (e == hipSuccess) e = hipMemsetAsync(s->tickets, 0, 64, s->stream);
    if (e == hipSuccess) e = hipHostMalloc((void**)&s->host_sel, 64, hipHostMallocCoherent);
    if (e == hipSuccess) e = hipMemsetAsync(s->e, 0, nb, s->stream);   // dct_emitter.cc:54 : val.Clone().Zero()
    if (e == hipSuccess) e = hipMemsetAsync(s->sel, 0, 64, s->stream);
    if (e == hipSuccess) e = hipMemsetAsync(s->hist, 0, kBins * sizeof(uint32_t), s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
    if (e != hipSuccess) rc = hip_fail(e, "krk_dct_create", __FILE__, __LINE__);
  }
  if (rc != KRK_SUCCESS) {
    krk_dct_destroy(s);
    return rc;
  }
  *out = s;
  return KRK_SUCCESS;
}

int32_t krk_dct_destroy(krk_dct* s) {
  if (!s) return KRK_SUCCESS;
  if (s->stream) (void)hipStreamSynchronize(s->stream);
  if (s->e) (void)hipFree(s->e);
  if (s->e_next) (void)hipFree(s->e_next);
  if (s->sel) (void)hipFree(s->sel);
  if (s->hist) (void)hipFree(s->hist);
  if (s->tile_counts) (void)hipFree(s->tile_counts);
  if (s->tile_offsets) (void)hipFree(s->tile_offsets);
  if (s->scan_tmp) (void)hipFree(s->scan_tmp);
  if (s->tile_state) (void)hipFree(s->tile_state);
  if (s->tickets) (void)hipFree(s->tickets);
  if (s->host_sel) (void)hipHostFree(s->host_sel);
  s->close_stream();
  delete s;
  return KRK_SUCCESS;
}

int32_t krk_dct_compress(krk_dct* s, const float* grad, uint64_t life_span, float eta, int64_t* idx,
                         float* val, int64_t capacity, int64_t* nnz, uint32_t flags) {
  if (!s || !nnz) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  KRK_TRY(check_flags(flags));
  if (flags & KRK_ASYNC) return KRK_E_ARGUMENT;   // the count comes back by value
  if (life_span == 0 || capacity < 0) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(s->mu);
  const int64_t n = s->n;
  if (n < 256) {   // worker/dct_emitter.cc:18-20
    *nnz = -1;
    return KRK_SUCCESS;
  }
  if (!grad || (capacity > 0 && (!idx || !val))) return KRK_E_ARGUMENT;
  const bool reselect = s->step % life_span == 0;   // :25
  const float* d_g;
  // the gradient of a call on host memory is counted, then written; a selection reads it three times before
  KRK_TRY(s->input(grad, (size_t)n, flags, 0, &d_g, host_reads(reselect ? 5 : 2, n * 4)));
  if (reselect) {
    const int64_t k = (int64_t)((double)n * (1.0 - (double)eta));   // :27
    if (k < 1 || k > n) {
      set_error("eta %g keeps %lld of %lld elements; TopK needs 1..n", (double)eta, (long long)k,
                (long long)n);
      return KRK_E_ARGUMENT;   // t/math.cc:628-633 rejects k == 0
    }
    hipLaunchKernelGGL(select_begin_kernel, dim3(1), dim3(1), 0, s->stream, s->sel, (uint32_t)k);
    const int pass_bits[3] = {11, 11, 10};
    int shift = 32;
    for (int p = 0; p < 3; ++p) {
      const int prefix_shift = shift;        // bits above this pass are already fixed
      shift -= pass_bits[p];
      hipLaunchKernelGGL(select_hist_kernel, dim3(stream_grid(n)), dim3(kCodecBlock), 0, s->stream, d_g,
                         s->e, n, shift, pass_bits[p], prefix_shift, s->sel, s->hist);
      hipLaunchKernelGGL(select_pick_kernel, dim3(1), dim3(kCodecBlock), 0, s->stream, s->hist,
                         pass_bits[p], s->sel, p == 2 ? 1 : 0);
    }
    KRK_HIP(hipGetLastError());
  }
  const bool vec = ((uintptr_t)d_g & 15) == 0;
  // Room for every element and device buffers: nothing can overflow and nothing is staged, so one
  // pass emits and the count comes with it.
  if ((flags & KRK_DEVICE_PTRS) && capacity >= n) {
    const int rows = n <= kSingleShort ? 2 : n <= kSingleLong ? 4 : 8;
    const int64_t tiles = (n + single_tile(rows) - 1) / single_tile(rows);
    if (++s->emit_calls == kMaxEmitCalls) {
      KRK_HIP(hipMemsetAsync(s->tile_state, 0, (size_t)tiles * sizeof(unsigned long long), s->stream));
      s->emit_calls = 1;
    }
    uint32_t* d_host_sel = nullptr;
    KRK_HIP(hipHostGetDevicePointer((void**)&d_host_sel, s->host_sel, 0));
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles < kSingleGrid ? tiles : kSingleGrid)), dim3(kSingleBlock), 0,
                         s->stream, d_g, s->e, n, (uint32_t)tiles, vec, s->sel, s->tile_state, s->tickets,
                         s->emit_calls, reinterpret_cast<long long*>(idx), val, s->e_next, d_host_sel);
    };
    if (rows == 8) launch(emit_single_kernel<8>);
    else if (rows == 4) launch(emit_single_kernel<4>);
    else launch(emit_single_kernel<2>);
    KRK_HIP(hipGetLastError());
    KRK_TRY(wait_stream(s->stream));
    *nnz = (int64_t)s->host_sel[3];
  } else {
    const dim3 emit_grid((unsigned)(s->tiles < kCodecGrid ? s->tiles : kCodecGrid));
    hipLaunchKernelGGL(emit_count_kernel, emit_grid, dim3(kCodecBlock), 0, s->stream, d_g, s->e, n, s->tiles, vec,
                       s->sel, s->tile_counts);
    KRK_HIP(hipGetLastError());
    KRK_TRY(exclusive_scan_i32(s->tile_counts, s->tile_offsets, s->tiles,
                               reinterpret_cast<int32_t*>(s->sel + 3), s->scan_tmp, s->stream));
    KRK_HIP(hipMemcpyAsync(s->host_sel, s->sel, 16, hipMemcpyDeviceToHost, s->stream));
    KRK_HIP(hipStreamSynchronize(s->stream));
    const int64_t count = (int64_t)s->host_sel[3];
    *nnz = count;
    if (count > capacity) {
      // nothing was committed: restore the threshold the next call will see
      if (reselect) {
        const uint32_t old_bits = __builtin_bit_cast(uint32_t, s->tau);
        KRK_HIP(hipMemcpyAsync(s->sel + 2, &old_bits, 4, hipMemcpyHostToDevice, s->stream));
        KRK_HIP(hipStreamSynchronize(s->stream));
      }
      set_error("compress needs room for %lld entries, caller offered %lld", (long long)count,
                (long long)capacity);
      return KRK_E_CAPACITY;
    }
    long long* d_idx;
    float* d_val;
    KRK_TRY(s->output(reinterpret_cast<long long*>(idx), (size_t)count, flags, 1, &d_idx));
    KRK_TRY(s->output(val, (size_t)count, flags, 2, &d_val));
    hipLaunchKernelGGL(emit_write_kernel, emit_grid, dim3(kCodecBlock), 0, s->stream, d_g, s->e, n,
                       s->tiles, vec, s->sel, s->tile_offsets, d_idx, d_val, s->e_next);
    KRK_HIP(hipGetLastError());
    KRK_TRY(s->output_back(reinterpret_cast<long long*>(idx), (size_t)count, flags, 1));
    KRK_TRY(s->output_back(val, (size_t)count, flags, 2));
    KRK_HIP(hipStreamSynchronize(s->stream));
  }
  const float new_tau = __builtin_bit_cast(float, s->host_sel[2]);
  float* tmp = s->e;
  s->e = s->e_next;
  s->e_next = tmp;
  s->tau = new_tau;
  s->step += 1;   // :40
  return KRK_SUCCESS;
}

int32_t krk_dct_tau(krk_dct* s, float* tau) {
  if (!s || !tau) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(s->mu);
  *tau = s->tau;
  return KRK_SUCCESS;
}

int32_t krk_dct_step(krk_dct* s, uint64_t* step) {
  if (!s || !step) return KRK_E_ARGUMENT;
  std::lock_guard<std::mutex> lk(s->mu);
  *step = s->step;
  return KRK_SUCCESS;
}

int32_t krk_dct_residual(krk_dct* s, float* out, uint32_t flags) {
  if (!s || (s->n > 0 && !out)) return KRK_E_ARGUMENT;
  KRK_TRY(ensure_runtime());
  KRK_TRY(check_flags(flags));
  std::lock_guard<std::mutex> lk(s->mu);
  if (s->n)
    KRK_HIP(hipMemcpyAsync(out, s->e, (size_t)s->n * sizeof(float),
                           (flags & KRK_DEVICE_PTRS) ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost,
                           s->stream));
  if (!(flags & KRK_ASYNC)) KRK_HIP(hipStreamSynchronize(s->stream));
  return KRK_SUCCESS;
}

int32_t krk_coo_to_dense(const int64_t* idx, const float* val, int64_t nnz, float* dense, int64_t n,
                         uint32_t flags) {
  KRK_TRY(ensure_runtime());
  KRK_TRY(check_flags(flags));
  if (n < 0 || nnz < 0 || (n > 0 && !dense) || (nnz > 0 && (!idx || !val))) return KRK_E_ARGUMENT;
  if (n == 0) return KRK_SUCCESS;
  hipStream_t st = nullptr;   // owns no object: runs on the null stream
  const bool host = !(flags & KRK_DEVICE_PTRS);
  float* d_dense = dense;
  const long long* d_idx = reinterpret_cast<const long long*>(idx);
  const float* d_val = val;
  char* tmp = nullptr;
  if (host) {
    const size_t nb = ((size_t)n * 4 + 255) & ~(size_t)255;
    const size_t ib = ((size_t)nnz * 8 + 255) & ~(size_t)255;
    KRK_HIP(hipMalloc((void**)&tmp, nb + ib + (size_t)nnz * 4 + 256));
    d_dense = reinterpret_cast<float*>(tmp);
    long long* si = reinterpret_cast<long long*>(tmp + nb);
    float* sv = reinterpret_cast<float*>(tmp + nb + ib);
    if (nnz) {
      hipError_t e = hipMemcpy(si, idx, (size_t)nnz * 8, hipMemcpyHostToDevice);
      if (e == hipSuccess) e = hipMemcpy(sv, val, (size_t)nnz * 4, hipMemcpyHostToDevice);
      if (e != hipSuccess) {
        (void)hipFree(tmp);
        return hip_fail(e, "krk_coo_to_dense staging", __FILE__, __LINE__);
      }
    }
    d_idx = si;
    d_val = sv;
  }
  hipError_t e = hipSuccess;
  {
    std::lock_guard<std::mutex> lk(g_densify_mu);
    const int32_t rc = coo_densify(&g_densify_work, d_idx, d_val, nnz, d_dense, n, st);
    // the shared work buffer is free for the next caller once this call's launches are done
    if (rc == KRK_SUCCESS && n >= kCooTiledFrom) e = hipStreamSynchronize(st);
    if (g_densify_work.bits.bytes > kDensifyBitsKept) g_densify_work.bits.release();
    if (rc != KRK_SUCCESS) {
      if (tmp) (void)hipFree(tmp);
      return rc;
    }
  }
  if (e == hipSuccess && host) e = hipMemcpy(dense, d_dense, (size_t)n * sizeof(float), hipMemcpyDeviceToHost);
  if (e == hipSuccess && !(flags & KRK_ASYNC)) e = hipStreamSynchronize(st);
  if (tmp) (void)hipFree(tmp);
  if (e != hipSuccess) return hip_fail(e, "krk_coo_to_dense", __FILE__, __LINE__);
  return KRK_SUCCESS;
}

}  // extern "C"
