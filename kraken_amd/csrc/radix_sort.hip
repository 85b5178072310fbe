// Stable least-significant-digit radix sort of (32-bit key, 32-bit payload) pairs on the device:
// what orders a large push's (row, position) pairs so that the gradient rows of one id are added
// up in position order (worker/emitter.cc:516-531 walks the request in order).
//
// A pass takes one digit of up to nine bits and is three launches with no waiting between workgroups:
//   1. radix_hist_kernel: every workgroup counts the digits of its tile of 3072 keys in LDS and
//      writes the counts digit-major, hist[digit][tile];
//   2. radix_scan_kernel: one workgroup per digit turns its row of counts into the number of
//      equal digits in earlier tiles, and notes the digit's total;
//   3. radix_scatter_kernel: a workgroup scans the 512 totals in LDS (where each digit's output
//      begins), ranks its tile's keys among equal digits in tile order (every wavefront finds the
//      lanes that hold the same digit with one ballot per digit bit, a per-wavefront histogram in
//      LDS turns into offsets by one scan over (digit, wavefront)), puts the tile into digit
//      order in LDS and writes it out from there, so that a digit's keys of the tile leave as one
//      piece: pair p of the ordered tile goes to begin[digit] + earlier[digit][tile] +
//      (p - where the digit starts in the tile).
// Equal digits keep their order in every pass, so the sort is stable.
//
// An XCD takes a stretch of consecutive tiles (xcd_tile): neighbouring tiles write neighbouring counts and, for
// every digit, neighbouring pieces of some 48 bytes, which meet in its L2 and leave as whole lines (the scatter
// of 8.5 million pairs 36.6 -> 32.4 us a pass; it moves 136 MB, 24 us at the rate of a copy).
#include "reduce_internal.h"

namespace krk {

namespace {

// 512 lanes of six keys and 16-bit counts: four workgroups fit a compute unit, and their phases (keys on their way,
// votes, scans, the tile's way through LDS) overlap. 8.5 million pairs by 24 bits, us: 1024 lanes of four 186, 512 of
// eight 153, of six 140; of twelve or sixteen 163 and 176.
constexpr int kRsBlock = 512;
constexpr int kRsItems = 6;
constexpr int kRsTile = kRsBlock * kRsItems;     // keys a workgroup takes
constexpr int kRsWaves = kRsBlock / kWave;
constexpr int kRsMaxBits = 9;
constexpr int kRsDigits = 1 << kRsMaxBits;

// ---- a pooled push's pairs, from the pull's notes and the bags' offsets ----
// The first pass puts them together as it reads them: its histogram takes the notes, the scan's launch
// finds the bags in which tiles begin, and the scatter works every position's bag out. A launch that wrote the pairs
// out in advance (a lane group a bag, as for requests short enough for buckets) moved 117 MB for 8.5 million positions,
// 32 us; without it the first histogram takes 15.5 us for 11 (the notes come from further away than pairs just
// written) and the first scatter 38 for 30: a pooled step of 891 us 872, of 2.4 million positions 264 and 257, of 1.3
// million 320 and 312 (rows of 32, 8 and 64 floats). Requests of up to 2^20
// positions keep that launch: in the partition's launches the same cost what it saved.

// The bag that the offsets step over p with, offsets[bag] <= p < offsets[bag + 1]: searched by a whole
// wavefront, 64 offsets a step. offsets[0] <= p < offsets[bags], which every step keeps true of what is left,
// also where offsets in between descend (they are not checked).
__device__ __forceinline__ int64_t bag_at(const long long* __restrict__ offsets, int64_t bags, long long p) {
  const int lane = threadIdx.x & (kWave - 1);
  int64_t lo = 0, hi = bags;
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t at = lo + (lane + 1) * step;
    const unsigned long long before = __ballot(at < hi && offsets[at] <= p);
    const int64_t steps = kWave - __clzll((long long)before);   // the last lane whose offset is not above p; none: 0
    lo += steps * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

// The bags in which the tiles of `tile` positions begin, starts[0..tiles], a wavefront each: work for a launch
// ahead of the one that needs them, whose workgroups waited 5 us for them with a search of their own
// (8.5 million positions, three rounds of workgroups: 43 us in place of 30).
__device__ __forceinline__ void find_tile_starts(const NotedBags& in, int64_t wave, int64_t tiles, int tile,
                                                 uint32_t* __restrict__ starts) {
  if (wave > tiles) return;
  const long long first = in.offsets[0], past = in.offsets[in.bags];
  long long p = wave * tile;
  if (p < first) p = first;
  if (p >= past) p = past - 1;
  const int64_t b = first < past ? bag_at(in.offsets, in.bags, p) : 0;   // (no position lies in a bag)
  if ((threadIdx.x & (kWave - 1)) == 0) starts[wave] = (uint32_t)b;
}

// The words of a tile's positions, element i of a lane being position wave * (64 * ITEMS) + i * 64 + lane
// of the tile: the lanes leave every bag's word where it begins (mark), and a position takes the nearest one at
// or before it (word), which votes find inside a wavefront's stretch, and a note per wavefront before that. Positions of
// no bag get kNoBag. Whatever the offsets hold, a position of the tile between the first and the last offset
// finds a word, that of the tile's first such position if no other. All lanes call all three in turn, with a
// barrier between mark and word; word_at (a word a position) and notes are LDS, free again after the next barrier.
template <int ITEMS, int LANES>
struct TileWords {
  static constexpr int kTile = LANES * ITEMS, kWaves = LANES / kWave;
  // A tile of more bags, nearly all of them empty, has its positions search for theirs: a batch may end in a
  // million empty bags, which the lanes of one workgroup would walk for milliseconds.
  static constexpr int64_t kWalked = 16 * LANES;
  const NotedBags& in;
  int64_t base, b, b0, b1;
  long long lo, hi, begin, end;
  int at[ITEMS];

  // (requests the first bags' ends; what the caller can request without waiting comes before it)
  __device__ __forceinline__ TileWords(const NotedBags& bags, const uint32_t* __restrict__ starts, int64_t tile,
                                       int64_t n)
      : in(bags), base(tile * kTile), begin(0), end(0) {
    b0 = starts[tile];
    b1 = starts[tile + 1];
    b1 = b1 < b0 ? b0 : b1;                            // (offsets that descend)
    b = b0 + threadIdx.x;
    if (b <= b1) {
      begin = in.offsets[b];
      end = in.offsets[b + 1];
    }
    const int64_t end_of_tile = base + kTile < n ? base + kTile : n;
    const long long first = in.offsets[0], past = in.offsets[in.bags];
    lo = first > base ? first : base;
    hi = past < end_of_tile ? past : end_of_tile;
  }

  __device__ __forceinline__ void mark(uint32_t* word_at, int* notes) {
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) word_at[i * LANES + t] = kNoBag;
    __syncthreads();
    if (lo < hi && b1 - b0 > kWalked) {
      for (long long p = lo + t; p < hi; p += LANES) {
        int64_t in_bag = b0, behind = b1 + 1;          // offsets[in_bag] <= p < offsets[behind]
        while (behind - in_bag > 1) {
          const int64_t middle = (in_bag + behind) / 2;
          if (in.offsets[middle] <= p) in_bag = middle; else behind = middle;
        }
        word_at[p - base] = in.words.pack((uint32_t)in_bag, in.offsets[in_bag + 1] - in.offsets[in_bag]);
      }
    } else if (lo < hi) {
      while (b <= b1) {
        const long long p = (b == b0 ? lo : begin) - base;
        if (b == b0 || (end > begin && p > lo - base && p < hi - base)) word_at[p] = in.words.pack((uint32_t)b, end - begin);
        b += LANES;
        if (b <= b1) {
          begin = in.offsets[b];
          end = in.offsets[b + 1];
        }
      }
    }
    __syncthreads();
    int nearest = -1;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int from = wave * (kWave * ITEMS) + i * kWave;
      const unsigned long long marked = __ballot(word_at[from + lane] != kNoBag);
      const unsigned long long here = marked & (~0ull >> (kWave - 1 - lane));
      at[i] = here ? from + kWave - 1 - __clzll((long long)here) : nearest;
      if (marked) nearest = from + kWave - 1 - __clzll((long long)marked);
    }
    if (lane == 0) notes[wave] = nearest;
  }

  __device__ __forceinline__ void word(const uint32_t* word_at, const int* notes, uint32_t (&out)[ITEMS]) const {
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    int earlier = -1;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int m = notes[w];
      if (w < wave && m >= 0) earlier = m;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int64_t j = base + wave * (kWave * ITEMS) + i * kWave + lane;
      const int from = at[i] >= 0 ? at[i] : earlier;
      out[i] = j >= lo && j < hi && from >= 0 ? word_at[from] : kNoBag;
    }
  }
};

struct NotedInput {
  NotedBags bags;
  TableView tv;
  uint32_t miss_key;
  uint32_t* starts;              // the bags in which tiles begin
};
__device__ __forceinline__ uint32_t noted_key(const NotedInput& in, uint32_t row, int64_t j) {
  return krk::noted_key(in.tv, row, in.bags.ids + j, 0u, in.miss_key);
}

struct NoWords {                 // pairs that are there
  __device__ __forceinline__ NoWords(const NotedBags&, const uint32_t*, int64_t, int64_t) {}
};

// The lanes that hold the digit of the wavefront's first lane are counted with one LDS add, the others
// with one each: a digit that many keys share (the hottest row of a skewed request) is likely
// that one, and adds to one counter are served one after the other. Finding all equal digits by
// votes, one per bit, kept the vector units busy for longer than the keys take to arrive (8.5
// million keys, nine bits: 24 us a pass for 34 MB). 1024 lanes with four keys each took 14.4 us, 256
// with twelve in three loads, and counts that leave through one XCD's L2, take 10.9.
constexpr int kHistLanes = 256;
typedef uint32_t keys4_t __attribute__((ext_vector_type(4), aligned(4)));

template <bool BAGS>
__global__ __launch_bounds__(kHistLanes) void radix_hist_kernel(const uint32_t* __restrict__ keys, int64_t n,
                                                              int shift, int bits, int64_t pitch,
                                                              uint32_t* __restrict__ hist, NotedInput in) {
  constexpr int kPer = kRsTile / kHistLanes;
  static_assert(kPer % 4 == 0, "four keys a load");
  __shared__ uint32_t count[kRsDigits];
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const uint32_t mask = (1u << bits) - 1u;
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t base = (int64_t)tile * kRsTile;
  uint32_t key[kPer];
  const bool whole = base + kRsTile <= n;
  if (whole) {
#pragma unroll
    for (int i = 0; i < kPer / 4; ++i) {
      const keys4_t x = *reinterpret_cast<const keys4_t*>(keys + base + (int64_t)(i * kHistLanes + t) * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) key[4 * i + q] = x[q];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int64_t j = base + i * kHistLanes + t;
      key[i] = j < n ? keys[j] : 0u;
    }
  }
  for (int d = t; d <= (int)mask; d += kHistLanes) count[d] = 0u;
  if constexpr (BAGS) {
    const long long first = in.bags.offsets[0], past = in.bags.offsets[in.bags.bags];
    bool plain = whole && base >= first && base + kRsTile <= past;
#pragma unroll
    for (int i = 0; i < kPer; ++i) plain = plain && key[i] != kEmptyRow;
    if (!plain) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int64_t j = whole ? base + (int64_t)(i / 4 * kHistLanes + t) * 4 + i % 4 : base + i * kHistLanes + t;
        if (j < n) key[i] = j >= first && j < past ? noted_key(in, key[i], j) : in.miss_key;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool live = whole || base + i * kHistLanes + t < n;
    const uint32_t digit = (key[i] >> shift) & mask;
    const unsigned long long on = __ballot(live);
    if (on == 0ull) break;                             // uniform: the tile's tail
    const int leader = __ffsll(on) - 1;
    const uint32_t shared = __builtin_amdgcn_readlane(digit, leader);
    const unsigned long long same = __ballot(live && digit == shared);
    if (lane == leader) {
      atomicAdd(&count[digit], (uint32_t)__popcll(same));
    } else if (live && digit != shared) {
      atomicAdd(&count[digit], 1u);
    }
  }
  __syncthreads();
  for (int d = t; d <= (int)mask; d += kHistLanes) {
    uint32_t* row = hist + (int64_t)d * pitch;
    row[tile] = count[d];
    if (tile == gridDim.x - 1)
      for (int64_t c = (int64_t)gridDim.x; c < pitch; ++c) row[c] = 0u;   // at most seven
  }
}

// One workgroup per digit: hist[digit][0..tiles) -> exclusive prefix sums in place, total[digit].
// A row is a dependent chain of trips to memory, so a trip takes 2048 tiles, eight a lane in two
// 16-byte loads (rows are `pitch` counts apart, a multiple of eight, and zero behind the last tile);
// one wavefront taking 64 tiles a trip walked the rows of 8.5 million keys for 20 us.
constexpr int kScanLanes = 256;
constexpr int kScanPer = 8;
__global__ __launch_bounds__(kScanLanes) void radix_scan_kernel(uint32_t* __restrict__ hist, int64_t pitch,
                                                                uint32_t* __restrict__ total, int digits, int64_t tiles,
                                                                NotedBags bags, uint32_t* __restrict__ starts) {
  if (blockIdx.x >= (uint32_t)digits) {
    find_tile_starts(bags, (int64_t)(blockIdx.x - digits) * (kScanLanes / kWave) + threadIdx.x / kWave, tiles, kRsTile,
                     starts);
    return;
  }
  __shared__ uint32_t wave_total[kScanLanes / kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  uint4* row = reinterpret_cast<uint4*>(hist + (int64_t)blockIdx.x * pitch);
  uint32_t carry = 0;
  for (int64_t c0 = 0; c0 < pitch; c0 += kScanLanes * kScanPer) {
    const int64_t c = c0 + threadIdx.x * kScanPer;
    const bool on = c < pitch;
    uint32_t v[kScanPer] = {};
    if (on) {
      const uint4 x = row[c / 4], y = row[c / 4 + 1];
      v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
      v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
    }
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kScanPer; ++i) sum += v[i];
    const uint32_t incl = wave_inclusive_sum(sum);
    if (lane == kWave - 1) wave_total[wave] = incl;
    __syncthreads();
    uint32_t at = carry + incl - sum;
#pragma unroll
    for (int w = 0; w < kScanLanes / kWave; ++w) {
      const uint32_t x = wave_total[w];
      if (w < wave) at += x;
      carry += x;
    }
    __syncthreads();                                   // the next trip writes wave_total
    uint32_t r[kScanPer];
#pragma unroll
    for (int i = 0; i < kScanPer; ++i) {
      r[i] = at;
      at += v[i];
    }
    if (on) {
      row[c / 4] = uint4{r[0], r[1], r[2], r[3]};
      row[c / 4 + 1] = uint4{r[4], r[5], r[6], r[7]};
    }
  }
  if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

template <int BITS, bool BAGS>
__global__ __launch_bounds__(kRsBlock, BITS == 9 ? 6 : 8) void radix_scatter_kernel(const uint32_t* __restrict__ keys,
                                                                 const uint32_t* __restrict__ vals, int64_t n,
                                                                 int shift, int64_t pitch,
                                                                 const uint32_t* __restrict__ hist,
                                                                 const uint32_t* __restrict__ total,
                                                                 uint32_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ vals_out, NotedInput in) {
  constexpr int kDigits = 1 << BITS;
  constexpr uint32_t kMask = kDigits - 1;
  __shared__ uint32_t gbase[kDigits];                  // where this tile's keys of the digit go in the output
  __shared__ uint32_t lstart[kDigits];                 // where they begin in the tile's own digit order
  __shared__ alignas(4) uint16_t wave_hist[kRsWaves * kDigits];   // [wave][digit]
  __shared__ uint32_t wave_total[kRsWaves];
  __shared__ uint32_t skey[kRsTile], sval[kRsTile];    // the tile in digit order
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  // element i of lane l in wavefront w is key w * (64 * kRsItems) + i * 64 + l of the tile: a wavefront's
  // keys are consecutive, and taking i in ascending order visits them in tile order
  const int64_t tile_base = (int64_t)tile * kRsTile;
  const int64_t base = tile_base + wave * (kWave * kRsItems) + lane;
  uint32_t key[kRsItems], val[kRsItems], rank[kRsItems];
#pragma unroll
  for (int i = 0; i < kRsItems; ++i) {
    const int64_t j = base + i * kWave;
    key[i] = j < n ? keys[j] : 0xFFFFFFFFu;
    val[i] = !BAGS && j < n ? vals[j] : 0u;
  }
  uint32_t all = 0, earlier = 0;
  if (t < kDigits) {
    all = total[t];
    earlier = hist[(int64_t)t * pitch + tile];
  }
  std::conditional_t<BAGS, TileWords<kRsItems, kRsBlock>, NoWords> words(in.bags, in.starts, tile, n);
  __shared__ int notes[kRsWaves];
  for (int i = t; i < kRsWaves * kDigits / 2; i += kRsBlock) reinterpret_cast<uint32_t*>(wave_hist)[i] = 0u;
  // an exclusive scan over the workgroup's first kDigits lanes (one value each), through wave_total
  auto scan_digits = [&](uint32_t v) -> uint32_t {
    const uint32_t incl = wave_inclusive_sum(v);
    if (lane == kWave - 1) wave_total[wave] = incl;
    __syncthreads();
    uint32_t offset = incl - v;
    for (int w = 0; w < wave; ++w) offset += wave_total[w];
    return offset;
  };
  // where each digit's output begins (scan of the totals), plus what earlier tiles hold of it
  {
    if constexpr (BAGS) words.mark(skey, notes);
    const uint32_t offset = scan_digits(all);            // its barrier: wave_hist is clear, too
    if (t < kDigits) gbase[t] = offset + earlier;
  }
  if constexpr (BAGS) {
    words.word(skey, notes, val);
#pragma unroll
    for (int i = 0; i < kRsItems; ++i) {
      const int64_t j = base + i * kWave;
      if (j >= n) continue;
      key[i] = val[i] != kNoBag ? noted_key(in, key[i], j) : in.miss_key;
      if (in.bags.bag_of) {
        in.bags.bag_of[j] = val[i];
        val[i] = (uint32_t)j;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kRsItems; ++i) {
    const bool live = base + i * kWave < n;            // the tile's tail holds no keys
    const uint32_t digit = (key[i] >> shift) & kMask;
    const unsigned long long same = same_value<BITS>(digit, __ballot(live));
    const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
    uint16_t* cell = &wave_hist[wave * kDigits + digit];
    const uint32_t old = *cell;                        // read by all lanes of the digit ...
    if (live && before == 0) *cell = (uint16_t)(old + (uint32_t)__popcll(same));   // ... then advanced by their first
    rank[i] = old + before;
  }
  __syncthreads();
  // per digit: what each wavefront holds of it becomes the count of the wavefronts before it,
  // and the digit's count in the tile goes on to the scan over digits (lane t owns digit t)
  uint32_t mine = 0;
  if (t < kDigits) {
#pragma unroll
    for (int w = 0; w < kRsWaves; ++w) {
      const uint32_t c = wave_hist[w * kDigits + t];
      wave_hist[w * kDigits + t] = (uint16_t)mine;
      mine += c;
    }
  }
  {
    const uint32_t offset = scan_digits(mine);
    if (t < kDigits) lstart[t] = offset;
  }
  __syncthreads();
  // the tile in digit order, in LDS: equal digits keep their order
#pragma unroll
  for (int i = 0; i < kRsItems; ++i) {
    if (base + i * kWave < n) {
      const uint32_t digit = (key[i] >> shift) & kMask;
      const uint32_t at = lstart[digit] + wave_hist[wave * kDigits + digit] + rank[i];
      skey[at] = key[i];
      sval[at] = val[i];
    }
  }
  __syncthreads();
  // out: consecutive lanes hold consecutive keys of a digit, which go to consecutive addresses
  // (a digit's eight or so keys of a tile leave as one piece, not as eight)
  const int64_t left = n - tile_base;
  const int here = left < kRsTile ? (int)left : kRsTile;
#pragma unroll
  for (int i = 0; i < kRsItems; ++i) {
    const int p = i * kRsBlock + t;
    if (p < here) {
      const uint32_t k = skey[p];
      const uint32_t digit = (k >> shift) & kMask;
      const uint32_t dest = gbase[digit] + (uint32_t)p - lstart[digit];
      keys_out[dest] = k;
      vals_out[dest] = sval[p];
    }
  }
}

template <int BITS>
void launch_scatter(const uint32_t* keys, const uint32_t* vals, int64_t n, int shift, int64_t tiles, int64_t pitch,
                    const uint32_t* hist, const uint32_t* total, uint32_t* keys_out, uint32_t* vals_out,
                    hipStream_t stream, const NotedInput* in) {
  if (in)
    hipLaunchKernelGGL((radix_scatter_kernel<BITS, true>), dim3((unsigned)tiles), dim3(kRsBlock), 0, stream, keys, vals,
                       n, shift, pitch, hist, total, keys_out, vals_out, *in);
  else
    hipLaunchKernelGGL((radix_scatter_kernel<BITS, false>), dim3((unsigned)tiles), dim3(kRsBlock), 0, stream, keys, vals,
                       n, shift, pitch, hist, total, keys_out, vals_out, NotedInput{});
}

// counts between two digits' rows of the histogram
int64_t hist_pitch(int64_t tiles) { return (tiles + kScanPer - 1) / kScanPer * kScanPer; }

}  // namespace

size_t radix_sort_work_bytes(int64_t n) {
  const int64_t tiles = (n + kRsTile - 1) / kRsTile;
  // the tiles' counts, the digits' totals, and the bags in which tiles begin
  return ((size_t)(hist_pitch(tiles) + 1) * kRsDigits + (size_t)tiles + 1) * sizeof(uint32_t);
}

static int32_t sort_pairs(const NotedInput* in, uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt,
                          int64_t n, int bits, void* work, hipStream_t stream, uint32_t** keys_sorted,
                          uint32_t** vals_sorted) {
  if (bits < 1) bits = 1;
  if (bits > 32) bits = 32;
  const int64_t tiles = (n + kRsTile - 1) / kRsTile;
  if (tiles * (int64_t)kRsBlock >= ((int64_t)1 << 31)) {
    set_error("radix_sort_pairs: too many pairs for one launch");
    return KRK_E_CAPACITY;
  }
  uint32_t* hist = reinterpret_cast<uint32_t*>(work);
  const int64_t pitch = hist_pitch(tiles);
  uint32_t* total = hist + pitch * kRsDigits;
  const int passes = (bits + kRsMaxBits - 1) / kRsMaxBits;
  const int width = (bits + passes - 1) / passes;      // 8 or 9 bits where that saves nothing else
  uint32_t* src_k = keys;
  uint32_t* src_v = vals;
  uint32_t* dst_k = keys_alt;
  uint32_t* dst_v = vals_alt;
  for (int pass = 0; pass < passes && n > 0; ++pass) {
    const int shift = pass * width;
    const int w = bits - shift < width ? bits - shift : width;
    const int digits = 1 << w;
    const NotedInput* from = pass == 0 ? in : nullptr;
    const uint32_t* read_k = from ? from->bags.rows : src_k;
    if (from)
      hipLaunchKernelGGL(radix_hist_kernel<true>, dim3((unsigned)tiles), dim3(kHistLanes), 0, stream, read_k, n, shift, w,
                         pitch, hist, *from);
    else
      hipLaunchKernelGGL(radix_hist_kernel<false>, dim3((unsigned)tiles), dim3(kHistLanes), 0, stream, read_k, n, shift,
                         w, pitch, hist, NotedInput{});
    // (one wavefront for each tile's first bag, and one more)
    const int64_t finders = from ? (tiles + 1 + kScanLanes / kWave - 1) / (kScanLanes / kWave) : 0;
    hipLaunchKernelGGL(radix_scan_kernel, dim3((unsigned)(digits + finders)), dim3(kScanLanes), 0, stream, hist, pitch,
                       total, digits, tiles, from ? from->bags : NotedBags{}, from ? from->starts : nullptr);
    switch (w) {
      case 1: launch_scatter<1>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 2: launch_scatter<2>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 3: launch_scatter<3>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 4: launch_scatter<4>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 5: launch_scatter<5>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 6: launch_scatter<6>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 7: launch_scatter<7>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      case 8: launch_scatter<8>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
      default: launch_scatter<9>(read_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream, from); break;
    }
    KRK_HIP(hipGetLastError());
    uint32_t* tk = src_k;
    uint32_t* tv = src_v;
    src_k = dst_k;
    src_v = dst_v;
    dst_k = tk;
    dst_v = tv;
  }
  *keys_sorted = src_k;
  *vals_sorted = src_v;
  return KRK_SUCCESS;
}

int32_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n,
                         int bits, void* work, hipStream_t stream, uint32_t** keys_sorted,
                         uint32_t** vals_sorted) {
  return sort_pairs(nullptr, keys, vals, keys_alt, vals_alt, n, bits, work, stream, keys_sorted, vals_sorted);
}

int32_t radix_sort_noted_bags(const NotedBags& bags, const TableView& tv, uint32_t miss_key, uint32_t* keys,
                              uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n, int bits, void* work,
                              hipStream_t stream, uint32_t** keys_sorted, uint32_t** vals_sorted) {
  const int64_t tiles = (n + kRsTile - 1) / kRsTile;
  uint32_t* starts = reinterpret_cast<uint32_t*>(work) + (hist_pitch(tiles) + 1) * kRsDigits;
  const NotedInput in{bags, tv, miss_key, starts};
  return sort_pairs(&in, keys, vals, keys_alt, vals_alt, n, bits, work, stream, keys_sorted, vals_sorted);
}

}  // namespace krk
