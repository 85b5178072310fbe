// Groups a request's (key, payload) pairs by bucket: the first of the two steps in which a push of up to
// 2^20 ids brings the gradient rows of one id together (run_reduce.hip is the second). A bucket is a
// range of hashed keys, so all pairs of a key are in one, and pairs keep their order inside it
// (worker/emitter.cc:516-531 walks the request in order).
//
// Two launches, three where the second is much work, and no waiting between workgroups:
//   1. count_kernel: every workgroup counts its tile's buckets in LDS, hist[tile][bucket];
//   2. scan_kernel (above 64 tiles) turns a bucket's counts into the number of its pairs in earlier
//      tiles, and notes its total;
//   3. scatter_kernel: a workgroup scans the totals in LDS (where each bucket begins), ranks its
//      tile's pairs among those of the same bucket in tile order (every wavefront finds the lanes that
//      hold the same bucket with one ballot per bit, a per-wavefront histogram in LDS turns into
//      offsets by one scan over (bucket, wavefront)), puts the tile into bucket order in LDS and
//      writes it out from there, so that a bucket's pairs of the tile leave as one piece. Its first
//      workgroup also writes the plan of the reduction.
// Bound by latencies: kernels of 12 us for 50,000 pairs, 22 us for a million (24 MB), against 36 and 53 us for
// the three passes of a sort by whole row numbers.
#include "reduce_internal.h"

namespace krk {

namespace {

constexpr int kItems = 4;                        // pairs a lane takes
constexpr int kSmallLanes = 256;
constexpr int kLargeLanes = 1024;
constexpr int kMinBits = 8;
constexpr int kMaxBits = 10;                     // of a bucket
constexpr int kMaxBuckets = 1 << kMaxBits;
// Up to this many tiles the scatter adds a bucket's counts up by itself (neighbouring lanes read
// neighbouring counts) and the scan's launch, 4-5 us, is left out.
constexpr int kScatterScans = 64;

struct Input {
  const uint32_t *keys, *refs;   // pairs, or
  NotedRows noted;               // the rows of their positions
  TableView tv;
  int64_t n;
  uint32_t miss_key;
  RunHash hash;
};

// Pair j: its place, and whether it takes part.
template <bool NOTED>
__device__ __forceinline__ bool place(const Input& in, int64_t j, uint32_t key, uint32_t& h) {
  if (j >= in.n) return false;
  if (NOTED) key = noted_key(in.tv, key, in.noted.ids + j, 0u, in.miss_key);
  h = (key * in.hash.mult) & in.hash.mask;
  return key < in.miss_key;
}

// The lanes that hold the bucket of the wavefront's first pair are counted with one LDS add, the others
// with one each: a bucket that many pairs share (the hottest row's) is likely that one, and adds
// to one counter are served one after the other.
template <bool NOTED>
__global__ __launch_bounds__(kLargeLanes) void count_kernel(Input in, uint32_t* __restrict__ hist) {
  __shared__ uint32_t count[kMaxBuckets];
  const int t = threadIdx.x, lanes = blockDim.x;
  const int lane = t & (kWave - 1);
  const int buckets = 1 << in.hash.bucket_bits;
  const int shift = in.hash.bits - in.hash.bucket_bits;
  const uint32_t* __restrict__ keys = NOTED ? in.noted.rows : in.keys;
  const int64_t base = (int64_t)blockIdx.x * (lanes * kItems);
  uint32_t key[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t j = base + i * lanes + t;
    key[i] = j < in.n ? keys[j] : 0u;
  }
  for (int i = t; i < buckets; i += lanes) count[i] = 0u;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    uint32_t h = 0u;
    const bool live = place<NOTED>(in, base + i * lanes + t, key[i], h);
    const uint32_t bucket = h >> shift;
    const unsigned long long on = __ballot(live);
    if (on == 0ull) continue;                          // uniform
    const int leader = __ffsll(on) - 1;
    const uint32_t shared = __shfl(bucket, leader);
    const unsigned long long same = __ballot(live && bucket == shared);
    if (lane == leader) {
      atomicAdd(&count[bucket], (uint32_t)__popcll(same));
    } else if (live && bucket != shared) {
      atomicAdd(&count[bucket], 1u);
    }
  }
  __syncthreads();
  uint32_t* row = hist + (int64_t)blockIdx.x * buckets;
  for (int i = t; i < buckets; i += lanes) row[i] = count[i];
}

// hist[0..tiles)[bucket] -> exclusive prefix sums in place, total[bucket]. A workgroup takes 16 buckets
// (64 bytes of a tile's row); 64 lanes share a bucket's tiles, a stretch each.
constexpr int kScanBuckets = 16;
constexpr int kScanParts = kLargeLanes / kScanBuckets;
constexpr int kScanTiles = (int)(kRunsMax / (kSmallLanes * kItems) / kScanParts);   // of a stretch, at most
__global__ __launch_bounds__(kLargeLanes) void scan_kernel(uint32_t* __restrict__ hist, int tiles, int buckets,
                                                           uint32_t* __restrict__ total) {
  __shared__ uint32_t part[kScanParts][kScanBuckets];
  const int b = threadIdx.x & (kScanBuckets - 1), p = threadIdx.x / kScanBuckets;
  const int per = (tiles + kScanParts - 1) / kScanParts;
  uint32_t* col = hist + blockIdx.x * kScanBuckets + b;
  uint32_t v[kScanTiles], sum = 0;
#pragma unroll
  for (int i = 0; i < kScanTiles; ++i) {
    const int c = p * per + i;
    v[i] = i < per && c < tiles ? col[(int64_t)c * buckets] : 0u;
    sum += v[i];
  }
  part[p][b] = sum;
  __syncthreads();
  uint32_t at = 0, all = 0;
  for (int q = 0; q < kScanParts; ++q) {
    const uint32_t x = part[q][b];
    if (q < p) at += x;
    all += x;
  }
#pragma unroll
  for (int i = 0; i < kScanTiles; ++i) {
    const int c = p * per + i;
    if (i < per && c < tiles) col[(int64_t)c * buckets] = at;
    at += v[i];
  }
  if (p == 0) total[blockIdx.x * kScanBuckets + b] = all;
}

// exclusive prefix sum of one value per lane over the workgroup; total to all
template <int LANES>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* wave_total, uint32_t& total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const uint32_t incl = wave_inclusive_sum(v);
  __syncthreads();                                     // wave_total may still be read from a previous scan
  if (lane == kWave - 1) wave_total[wave] = incl;
  __syncthreads();
  uint32_t offset = incl - v;
  total = 0;
#pragma unroll
  for (int w = 0; w < LANES / kWave; ++w) {
    const uint32_t x = wave_total[w];
    if (w < wave) offset += x;
    total += x;
  }
  return offset;
}

template <int BITS, int LANES, bool NOTED>
__global__ __launch_bounds__(LANES) void scatter_kernel(Input in, const uint32_t* __restrict__ hist,
                                                        const uint32_t* __restrict__ total, int tiles,
                                                        uint32_t* __restrict__ out_h, uint32_t* __restrict__ out_refs,
                                                        RunCut cut, RunPlan plan) {
  constexpr int kBuckets = 1 << BITS;
  constexpr int kWaves = LANES / kWave;
  constexpr int kTile = LANES * kItems;
  constexpr int kPer = kBuckets > LANES ? kBuckets / LANES : 1;   // buckets a lane owns, side by side
  __shared__ uint32_t gbase[kBuckets];                 // where this tile's pairs of the bucket go in the output
  __shared__ uint32_t lstart[kBuckets];                // where they begin in the tile's own bucket order
  __shared__ uint32_t wave_hist[kWaves * kBuckets];    // [wave][bucket]
  __shared__ uint32_t wave_total[kWaves];
  __shared__ uint32_t skey[kTile], sval[kTile];        // the tile in bucket order
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const int shift = in.hash.bits - BITS;
  const uint32_t* __restrict__ keys = NOTED ? in.noted.rows : in.keys;
  // element i of lane l in wavefront w is pair w * 256 + i * 64 + l of the tile: a wavefront's
  // pairs are consecutive, and taking i in ascending order visits them in tile order
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);   // neighbours' pieces of a bucket meet in one L2
  const int64_t base = (int64_t)tile * kTile + wave * (kWave * kItems) + lane;
  uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int64_t j = base + i * kWave;
    key[i] = j < in.n ? keys[j] : 0u;
    val[i] = NOTED ? (uint32_t)j : j < in.n ? in.refs[j] : 0u;
  }
  for (int i = t; i < kWaves * kBuckets; i += LANES) wave_hist[i] = 0u;
  // where each bucket begins (scan of the totals), plus what earlier tiles hold of it (tiles > 0: hist
  // holds the counts themselves)
  const int first = t * kPer;
  {
    uint32_t all[kPer] = {}, earlier[kPer] = {}, mine = 0;
    if (first < kBuckets) {
      if (tiles > 0) {
#pragma unroll 8
        for (int c = 0; c < tiles; ++c) {
#pragma unroll
          for (int k = 0; k < kPer; ++k) {
            const uint32_t x = hist[c * kBuckets + first + k];
            all[k] += x;
            if (c < (int)tile) earlier[k] += x;
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          all[k] = total[first + k];
          earlier[k] = hist[(int64_t)tile * kBuckets + first + k];
        }
      }
#pragma unroll
      for (int k = 0; k < kPer; ++k) mine += all[k];
    }
    uint32_t live;
    const uint32_t begin = block_scan<LANES>(mine, wave_total, live);   // its barriers: wave_hist is clear, too
    uint32_t at = begin;
    if (first < kBuckets) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        gbase[first + k] = at + earlier[k];
        at += all[k];
      }
    }
    if (blockIdx.x == 0) {                             // the plan
      uint32_t sum = 0;                                // chunks of cut buckets, and above them how many are cut
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        if (all[k] > cut.whole) sum += cut.pieces(all[k]) + (1u << 16);
      uint32_t whole;
      uint32_t before = block_scan<LANES>(sum, wave_total, whole);
      at = begin;
      if (first < kBuckets) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
          plan.begin[first + k] = at;
          if (all[k] > cut.whole) {
            const uint32_t c = before >> 16;
            plan.cut[c] = CutBucket{(uint32_t)(first + k), before & 0xFFFFu, at, all[k]};
            plan.done[c] = 0u;
            before += cut.pieces(all[k]) + (1u << 16);
          }
          at += all[k];
        }
      }
      if (t == 0) {
        plan.begin[kBuckets] = live;
        plan.head[0] = whole >> 16;
        plan.head[1] = whole & 0xFFFFu;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    uint32_t h = 0u;
    const bool live = place<NOTED>(in, base + i * kWave, key[i], h);
    key[i] = h;
    const uint32_t bucket = h >> shift;
    const unsigned long long same = same_value<BITS>(bucket, __ballot(live));
    const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
    uint32_t* cell = &wave_hist[wave * kBuckets + bucket];
    const uint32_t old = *cell;                        // read by all lanes of the bucket ...
    if (live && before == 0) *cell = old + (uint32_t)__popcll(same);   // ... then advanced by their first
    rank[i] = live ? old + before : 0xFFFFFFFFu;
  }
  __syncthreads();
  // per bucket: what each wavefront holds of it becomes the count of the wavefronts before it,
  // and the bucket's count in the tile goes on to the scan over buckets
  uint32_t mine[kPer] = {}, sum = 0;
  if (first < kBuckets) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = wave_hist[w * kBuckets + first + k];
        wave_hist[w * kBuckets + first + k] = mine[k];
        mine[k] += c;
      }
      sum += mine[k];
    }
  }
  uint32_t here;
  {
    uint32_t offset = block_scan<LANES>(sum, wave_total, here);
    if (first < kBuckets) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        lstart[first + k] = offset;
        offset += mine[k];
      }
    }
  }
  __syncthreads();
  // the tile in bucket order, in LDS: equal buckets keep their order
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    if (rank[i] != 0xFFFFFFFFu) {
      const uint32_t bucket = key[i] >> shift;
      const uint32_t at = lstart[bucket] + wave_hist[wave * kBuckets + bucket] + rank[i];
      skey[at] = key[i];
      sval[at] = val[i];
    }
  }
  __syncthreads();
  // out: consecutive lanes hold consecutive pairs of a bucket, which go to consecutive addresses
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    const int p = i * LANES + t;
    if (p < (int)here) {
      const uint32_t k = skey[p];
      const uint32_t bucket = k >> shift;
      const uint32_t dest = gbase[bucket] + (uint32_t)p - lstart[bucket];
      out_h[dest] = k;
      out_refs[dest] = sval[p];
    }
  }
}

// Tiles of 256 lanes (1024 pairs) for short requests, of 1024 lanes beyond: 50,000 pairs are 13 tiles
// of 4096 on 256 compute units. From where the scatter would need the scan (64 tiles) larger tiles are as
// fast: 131,072 pairs, scatter and scan, 12.2 us with 32 tiles, 7.5 + 4.2 with 128.
int lanes_for(int64_t n) { return n <= (int64_t)kScatterScans * kSmallLanes * kItems ? kSmallLanes : kLargeLanes; }
int64_t tiles_for(int64_t n) { return (n + lanes_for(n) * kItems - 1) / (lanes_for(n) * kItems); }

struct Launch {
  Input in;
  int tiles;
  uint32_t *hist, *total, *out_h, *out_refs;
  RunCut cut;
  RunPlan plan;
  hipStream_t stream;
};

template <int BITS, int LANES, bool NOTED>
void launch_scatter(const Launch& l) {
  hipLaunchKernelGGL((scatter_kernel<BITS, LANES, NOTED>), dim3((unsigned)l.tiles), dim3(LANES), 0, l.stream, l.in,
                     l.hist, l.total, l.tiles <= kScatterScans ? l.tiles : 0, l.out_h, l.out_refs, l.cut, l.plan);
}

template <int LANES, bool NOTED>
int32_t run(const Launch& l) {
  const int bits = l.in.hash.bucket_bits;
  hipLaunchKernelGGL((count_kernel<NOTED>), dim3((unsigned)l.tiles), dim3(LANES), 0, l.stream, l.in, l.hist);
  if (l.tiles > kScatterScans)
    hipLaunchKernelGGL(scan_kernel, dim3((1u << bits) / kScanBuckets), dim3(kLargeLanes), 0, l.stream, l.hist, l.tiles,
                       1 << bits, l.total);
  switch (bits) {
    case 8: launch_scatter<8, LANES, NOTED>(l); break;
    case 9: launch_scatter<9, LANES, NOTED>(l); break;
    default: launch_scatter<10, LANES, NOTED>(l); break;
  }
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

}  // namespace

size_t partition_work_bytes(int64_t n, int bucket_bits) {
  return ((size_t)(tiles_for(n) + 1) << bucket_bits) * sizeof(uint32_t);
}

int32_t partition_pairs(const uint32_t* keys, const uint32_t* refs, const NotedRows& noted, const TableView& tv,
                        int64_t n, uint32_t miss_key, const RunHash& hash, uint32_t* out_h, uint32_t* out_refs,
                        const RunCut& cut, const RunPlan& plan, void* work, hipStream_t stream) {
  if (n > kRunsMax || hash.bucket_bits < kMinBits || hash.bucket_bits > kMaxBits) {
    set_error("partition_pairs: %lld pairs into 2^%d buckets", (long long)n, hash.bucket_bits);
    return KRK_E_CAPACITY;
  }
  Launch l;
  l.in = Input{keys, refs, noted, tv, n, miss_key, hash};
  l.tiles = (int)tiles_for(n);
  l.hist = reinterpret_cast<uint32_t*>(work);
  l.total = l.hist + ((size_t)l.tiles << hash.bucket_bits);
  l.out_h = out_h;
  l.out_refs = out_refs;
  l.cut = cut;
  l.plan = plan;
  l.stream = stream;
  if (lanes_for(n) == kSmallLanes) return noted.rows ? run<kSmallLanes, true>(l) : run<kSmallLanes, false>(l);
  return noted.rows ? run<kLargeLanes, true>(l) : run<kLargeLanes, false>(l);
}

}  // namespace krk
