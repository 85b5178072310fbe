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
#include "krk_internal.h"

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

// The lanes that hold the digit of the wavefront's first lane are counted with one LDS add, the others
// with one each: a digit that many keys share (the hottest row of a skewed request) is likely
// that one, and adds to one counter are served one after the other. Finding all equal digits by
// votes, one per bit, kept the vector units busy for longer than the keys take to arrive (8.5
// million keys, nine bits: 24 us a pass for 34 MB). 1024 lanes with four keys each took 14.4 us, 256
// with twelve in three loads, and counts that leave through one XCD's L2, take 10.9.
constexpr int kHistLanes = 256;
typedef uint32_t keys4_t __attribute__((ext_vector_type(4), aligned(4)));
__global__ __launch_bounds__(kHistLanes) void radix_hist_kernel(const uint32_t* __restrict__ keys, int64_t n,
                                                              int shift, int bits, int64_t pitch,
                                                              uint32_t* __restrict__ hist) {
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
                                                                uint32_t* __restrict__ total) {
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

template <int BITS>
__global__ __launch_bounds__(kRsBlock, BITS == 9 ? 6 : 8) void radix_scatter_kernel(const uint32_t* __restrict__ keys,
                                                                 const uint32_t* __restrict__ vals, int64_t n,
                                                                 int shift, int64_t pitch,
                                                                 const uint32_t* __restrict__ hist,
                                                                 const uint32_t* __restrict__ total,
                                                                 uint32_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ vals_out) {
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
    val[i] = j < n ? vals[j] : 0u;
  }
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
    uint32_t all = 0, earlier = 0;
    if (t < kDigits) {
      all = total[t];
      earlier = hist[(int64_t)t * pitch + tile];
    }
    const uint32_t offset = scan_digits(all);            // its barrier: wave_hist is clear, too
    if (t < kDigits) gbase[t] = offset + earlier;
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
                    hipStream_t stream) {
  hipLaunchKernelGGL((radix_scatter_kernel<BITS>), dim3((unsigned)tiles), dim3(kRsBlock), 0, stream, keys, vals, n,
                     shift, pitch, hist, total, keys_out, vals_out);
}

// counts between two digits' rows of the histogram
int64_t hist_pitch(int64_t tiles) { return (tiles + kScanPer - 1) / kScanPer * kScanPer; }

}  // namespace

size_t radix_sort_work_bytes(int64_t n) {
  const int64_t tiles = (n + kRsTile - 1) / kRsTile;
  return (size_t)(hist_pitch(tiles) + 1) * kRsDigits * sizeof(uint32_t);
}

int32_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n,
                         int bits, void* work, hipStream_t stream, uint32_t** keys_sorted,
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
    hipLaunchKernelGGL(radix_hist_kernel, dim3((unsigned)tiles), dim3(kHistLanes), 0, stream, src_k, n, shift, w,
                       pitch, hist);
    hipLaunchKernelGGL(radix_scan_kernel, dim3((unsigned)digits), dim3(kScanLanes), 0, stream, hist, pitch, total);
    switch (w) {
      case 1: launch_scatter<1>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 2: launch_scatter<2>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 3: launch_scatter<3>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 4: launch_scatter<4>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 5: launch_scatter<5>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 6: launch_scatter<6>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 7: launch_scatter<7>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      case 8: launch_scatter<8>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
      default: launch_scatter<9>(src_k, src_v, n, shift, tiles, pitch, hist, total, dst_k, dst_v, stream); break;
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

}  // namespace krk
