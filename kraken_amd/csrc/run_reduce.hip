// The second step of a push of up to 2^20 ids (partition.hip is the first): the pairs of a bucket are
// sorted by key in LDS, every run of equal keys is added up in payload order, and each sum is
// handed to the optimizer once. One launch, one workgroup of 256 lanes per bucket, or per chunk of a
// bucket that holds more pairs than a chunk may (a row that many positions share brings that about).
//
// A whole bucket's rows are updated at once. A chunk of a cut bucket cannot do that, since its rows may
// go on in the next chunk: it adds its runs up and leaves a list, one entry for a run's sum, the pairs
// themselves for the shortest runs. The workgroup that is through last with a cut bucket
// merges: the chunks' lists, in order, are what the bucket's pairs were before, with few entries.
// Lists that do not fit into LDS at once (buckets of many cold rows) are sorted in memory, over the pairs,
// and taken a window at a time. No workgroup waits for another.
//
// Who adds a run up depends on its length: a lane group (up to 16 entries, the reference's order
// exactly), a wavefront, or the whole workgroup, whose lane groups add a stretch each and the
// stretches' sums are added in order. The order of additions does not depend on who is through
// last, so results do not change from run to run.
//
// What bounds it: a few dependent trips to memory (the plan, the pairs, records and gradient rows, for cut
// buckets the lists) and the LDS phases between them, 3-4 us of a small bucket's 12; for wide rows the
// gradients (a million rows of 128 floats, Zipf 1.3, 150 us = 3.9 TB/s of them and the records; 145 and
// four carry launches, 26, for the tiled reduction of a full sort). Of that request's 1785 workgroups 1000 run at
// first, four a compute unit (102 registers), and nine tenths of the gradients are read by 88 us; the last ones,
// of many cold rows, take 45 us from the 80th to 98th on. Six a compute unit, by launch bounds (18 to 22 registers in
// scratch memory), left it at 150 and slowed the passes of 131,072 to a million ids down by 3 to 10 %, as did
// the buckets' workgroups ahead of the chunks' or between them. An embedding layer's forward,
// backward and forward, us, with that sort and with buckets: 20,000 ids of 16 floats 72 / 50-59,
// 50,000 of 32 88 / 54, 131,072 of 16 102 / 62, 300,000 of 32 121 / 83, a million of 16 227 / 160,
// of 128 519 / 462; 10,000 bags of ten ids of 16 126 / 88.
#include "reduce_internal.h"

namespace krk {

namespace {

constexpr int kWaves = 4;
constexpr int kLanes = kWaves * kWave;
constexpr int kListItems = 8;                          // entries a lane takes
constexpr int kListMax = kLanes * kListItems;
constexpr int kRunBits = 8;                            // of a digit of the sort in LDS, at most
constexpr int kShortest = 16;                          // runs up to this length: one lane group each
// What a chunk of a cut bucket adds up before the merge: runs of this many entries on. A row that is not
// the hottest of its bucket may have a few entries in each of hundreds of chunks; passed on one by
// one, a row with 16 of them in 256 chunks did not fit into the merge's LDS, which made a
// reduction of 155 us one of 674. Fewer than four cost little to pass on,
// and every one of them less would take more room for sums (a row for this many pairs).
constexpr int kCutSum = 4;
constexpr int kPerGroup = 16;                          // a wavefront takes runs of up to this many entries per lane group
constexpr uint32_t kSummed = 0x80000000u;              // list entry: ref names a sum, not a payload

// Where entries come from and what becomes of the sums.
constexpr int kRows = 1;                               // gradient rows
constexpr int kBags = 2;                               // bags' gradient rows, scaled as they are read

struct RunLds {
  static constexpr int kLong = kListMax / (kShortest + 1) + 1;
  alignas(16) uint32_t key[kListMax];
  uint32_t ref[kListMax];
  // the sort's histogram [wave][digit], then a long run's partial sums [wave][up to 256 floats]
  alignas(16) uint32_t work[kWaves << kRunBits];
  alignas(4) uint16_t start[kListMax + 2];             // first entry of every run
  uint16_t long_run[kLong], wave_run[kLong];
  uint32_t wave_total[kWaves];
  uint32_t n_long, n_wave, last;
};

// What the entries of a key need to know: the record's table and the gradient rows.
struct Member {
  float* recs;
  int64_t stride;
  int c0, c1, c2, meta_off;
  const float* rows;
  const float* weights;
  const long long* offsets;
  int64_t row_start;
  uint32_t row_stride;
  uint32_t mean;
};

struct RunArgs {
  uint32_t* h;                   // pairs in bucket order
  uint32_t* refs;
  uint32_t* list_h;              // the lists of cut buckets' chunks, each where its pairs lie
  uint32_t* list_refs;
  float* sums;                   // sums of long runs of cut buckets
  RunPlan plan;
  RunHash hash;
  uint32_t max_chunks;           // workgroups for chunks of cut buckets, in front of the buckets'
  RunCut cut;
  int dim, elems, group;
};

// exclusive prefix sum of one value per lane over the workgroup; total to all
__device__ __forceinline__ uint32_t run_scan(uint32_t v, uint32_t* wave_total, uint32_t& total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const uint32_t incl = wave_inclusive_sum(v);
  lds_barrier();                                          // wave_total may still be read from a previous scan
  if (lane == kWave - 1) wave_total[wave] = incl;
  lds_barrier();
  uint32_t offset = incl - v;
  total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t x = wave_total[w];
    if (w < wave) offset += x;
    total += x;
  }
  return offset;
}

// Stable sort of the first len pairs by `bits` bits of the key from bit `from` on. (All lanes; the pairs
// need not be visible yet.)
__device__ __forceinline__ void sort_list(RunLds& s, int len, int bits, int from = 0) {
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const uint32_t key_mask = ((1u << bits) - 1u) << from;   // (from + bits: fewer than 32)
  const int per_lane = (len + kLanes - 1) / kLanes;    // 1..kListItems
  for (int j = len + t; j < per_lane * kLanes; j += kLanes) {
    s.key[j] = 0xFFFFFFFFu;                            // padding: the largest digit of every pass, behind its equals
    s.ref[j] = 0u;
  }
  lds_barrier();
  if (len <= kRankMax) {
    rank_list(s.key, s.ref, len, key_mask);
    return;
  }
  const int passes = (bits + kRunBits - 1) / kRunBits;
  const int width = (bits + passes - 1) / passes;
  const int digits = 1 << width;
  const int cells = kWaves << width;
  const int own = cells > kLanes ? cells / kLanes : 1; // counters a lane scans
  uint32_t* hist = s.work;                             // [kWaves][digits]
  const int wbase = wave * kWave * per_lane + lane;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = from + pass * width;
    uint32_t key[kListItems], ref[kListItems], rank[kListItems];
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      if (i < per_lane) {
        key[i] = s.key[wbase + i * kWave];
        ref[i] = s.ref[wbase + i * kWave];
      }
    }
    for (int i = t; i < cells; i += kLanes) hist[i] = 0u;
    lds_barrier();                                        // everyone holds its pairs; the histogram is clear
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      if (i < per_lane) {                              // uniform
        const uint32_t digit = ((key[i] & key_mask) >> shift) & (uint32_t)(digits - 1);
        const unsigned long long same = same_value<kRunBits>(digit, ~0ull, width);
        const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        uint32_t* cell = &hist[wave * digits + digit];
        const uint32_t old = *cell;                    // read by all lanes of the digit ...
        if (before == 0) *cell = old + (uint32_t)__popcll(same);   // ... then advanced by their first
        rank[i] = old + before;
      }
    }
    lds_barrier();
    // exclusive scan over (digit, wavefront)
    {
      uint32_t c[4], sum = 0, whole;
      const int at = t * own;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        c[k] = 0u;
        if (k < own && at < cells) c[k] = hist[((at + k) & (kWaves - 1)) * digits + (at + k) / kWaves];
        sum += c[k];
      }
      uint32_t offset = run_scan(sum, s.wave_total, whole);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k < own && at < cells) hist[((at + k) & (kWaves - 1)) * digits + (at + k) / kWaves] = offset;
        offset += c[k];
      }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      if (i < per_lane) {
        const uint32_t digit = ((key[i] & key_mask) >> shift) & (uint32_t)(digits - 1);
        const uint32_t dest = hist[wave * digits + digit] + rank[i];
        s.key[dest] = key[i];
        s.ref[dest] = ref[i];
      }
    }
    lds_barrier();
  }
}

// What one workgroup writes and another one reads within the launch: the lists, their lengths and the
// sums of cut buckets. These go past the L2 of the writer's and the reader's XCD (agent scope); the
// writer waits for its stores before it counts itself through. Fences in their place write back
// and drop the whole L2 each time: a million ids of 16 floats, 250 chunks of cut buckets among
// them, 135 us against 76.
__device__ __forceinline__ void share(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t shared_word(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int VEC>
__device__ __forceinline__ void share_row(float* p, const float (&v)[VEC]) {
#pragma unroll
  for (int c = 0; c < VEC; ++c) share(reinterpret_cast<uint32_t*>(p) + c, __float_as_uint(v[c]));
}
template <int VEC>
__device__ __forceinline__ void load_shared_row(const float* p, float (&v)[VEC]) {
#pragma unroll
  for (int c = 0; c < VEC; ++c) v[c] = __uint_as_float(shared_word(reinterpret_cast<const uint32_t*>(p) + c));
}

template <bool GROUPED>
using Source = std::conditional_t<GROUPED, GroupPooledSrc, PooledSrc>;

// The sums of a sorted list's runs. MERGE: of cut buckets' lists, whose entries may be sums themselves.
template <int OPT, int VEC, int FROM, bool GROUPED, bool MERGE>
struct Reducer {
  static constexpr bool kPooled = FROM == kBags;
  // gradient rows requested ahead of the sums, and short runs a lane group takes at a time
  static constexpr int kAhead = MERGE ? 4 : 8;
  static constexpr int kPair = MERGE ? 1 : 2;
  RunLds& s;
  const RunArgs& a;
  const Member* members;         // LDS (GROUPED) or the only one
  const ApplyArgs& args;
  const float* w;                // LDS: entries' weights
  BagWord words;
  bool weighted;
  int row_bits;
  uint32_t bucket;
  int low;                       // bits of a key's place inside its bucket
  uint32_t low_mask;
  uint32_t member_key;           // what the hash does not cover of a key: the workgroup's member

  // the key of entry j: row, and above it the member
  __device__ __forceinline__ uint32_t key_of(int j) const {
    const uint32_t h = (bucket << low) | (s.key[j] & low_mask);
    return ((h * a.hash.inverse) & a.hash.mask) | member_key;
  }
  __device__ __forceinline__ uint32_t row_of(uint32_t key) const {
    return GROUPED ? key & ((1u << row_bits) - 1u) : key;
  }
  // (read where it is used, out of LDS or scalar registers: copies would take vector registers)
  __device__ __forceinline__ const Member& member(uint32_t key) const {
    return GROUPED ? members[key >> row_bits] : *members;
  }
  __device__ __forceinline__ bool summed(int j) const { return MERGE && (s.key[j] & kSummed); }
  __device__ __forceinline__ void fetch(uint32_t of, int j, int e, float (&v)[VEC]) const {
    const uint32_t ref = s.ref[j];
    const Member& m = member(of);
    if (summed(j)) {
      load_shared_row<VEC>(a.sums + (int64_t)ref * a.dim + e * VEC, v);
    } else if constexpr (kPooled) {
      // a bag's row is read once for every id of the bag
      gload<VEC>(m.rows + (int64_t)words.bag(ref) * m.row_stride + e * VEC, v);
    } else {
      gload_once<VEC>((const KRK_GLOBAL float*)(m.rows + (int64_t)ref * m.row_stride) + e * VEC, v);
    }
  }
  __device__ __forceinline__ void scale(uint32_t of, int j, float (&v)[VEC]) const {
    if constexpr (kPooled) {
      if (summed(j)) return;
      const Member& m = member(of);
      if (m.mean) {
        const float r = mean_ratio(words, s.ref[j], m.offsets);
#pragma unroll
        for (int c = 0; c < VEC; ++c) v[c] = v[c] * r;
      }
      if (weighted) {
        const float x = w[j];
#pragma unroll
        for (int c = 0; c < VEC; ++c) v[c] = v[c] * x;
      }
    }
  }
  // adds entries [lo, hi) of a long run: kAhead of them pairwise, these sums alternately to two more (a
  // stretch of 128 then rounds a sum a dozen times, not 128 times)
  __device__ __forceinline__ void sum_entries(uint32_t of, int lo, int hi, int e, bool on, float (&acc)[VEC]) const {
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[c] = 0.0f;
    float odd[VEC] = {};
    for (int j0 = lo; j0 < hi; j0 += kAhead) {
      float v[kAhead][VEC];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (j0 + u < hi && on) {
          fetch(of, j0 + u, e, v[u]);
        } else {
#pragma unroll
          for (int c = 0; c < VEC; ++c) v[u][c] = 0.0f;
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (j0 + u < hi) scale(of, j0 + u, v[u]);
#pragma unroll
      for (int d = 1; d < kAhead; d <<= 1) {
#pragma unroll
        for (int u = 0; u < kAhead; u += 2 * d) {
#pragma unroll
          for (int c = 0; c < VEC; ++c) v[u][c] = v[u][c] + v[u + d][c];
        }
      }
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const float x = odd[c];
        odd[c] = acc[c] + v[0][c];
        acc[c] = x;
      }
    }
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[c] = acc[c] + odd[c];
  }
  // adds the lane groups' sums up inside the wavefront, neighbours first; the first group has the result
  __device__ __forceinline__ void fold_wave(float (&acc)[VEC]) const {
    const int sub = (threadIdx.x & (kWave - 1)) / a.group;
    for (int d = a.group; d < kWave; d <<= 1) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const float other = __shfl_down(acc[c], d);
        if ((sub & ((2 * d / a.group) - 1)) == 0) acc[c] = acc[c] + other;
      }
    }
  }
  // adds entries [lo, lo + count) with the whole workgroup; the first lane group has the result.
  // All lanes; ends with a barrier still to come before `work` may be written again.
  __device__ __forceinline__ void sum_block(uint32_t of, int first, int count, int e, bool on, int gl,
                                            float (&acc)[VEC]) const {
    const int lt = threadIdx.x / a.group;
    const int groups = kLanes / a.group;
    const int stretch = (count + groups - 1) / groups;
    const int end = first + count;
    const int lo = min(first + lt * stretch, end), hi = min(lo + stretch, end);
    sum_entries(of, lo, hi, e, on, acc);
    fold_wave(acc);
    const int lane_floats = a.group * VEC;
    const int lane = threadIdx.x & (kWave - 1);
    float* part = reinterpret_cast<float*>(s.work);    // [wave][lane_floats]
    lds_barrier();                                        // the last run's partial sums have been read
    if (lane < a.group) vstore<VEC>(part + (threadIdx.x / kWave) * lane_floats + gl * VEC, acc);
    lds_barrier();
    if (lt == 0) {
      static_assert(kWaves == 4, "(0 + 1) + (2 + 3)");
      float x[VEC], y[VEC], z[VEC];
      vload<VEC>(part + lane_floats + gl * VEC, x);
      vload<VEC>(part + 2 * lane_floats + gl * VEC, y);
      vload<VEC>(part + 3 * lane_floats + gl * VEC, z);
#pragma unroll
      for (int c = 0; c < VEC; ++c) acc[c] = (acc[c] + x[c]) + (y[c] + z[c]);
    }
  }
  __device__ __forceinline__ void locate(uint32_t of, TableView& tv, ApplyArgs& x) const {
    const Member& m = member(of);
    tv.recs = m.recs;
    tv.stride = m.stride;
    x = args;
    if constexpr (GROUPED) {
      x.c0 = m.c0;
      x.c1 = m.c1;
      x.c2 = m.c2;
      x.meta_off = m.meta_off;
    }
  }
  __device__ __forceinline__ void load(uint32_t of, int e, bool on, RowRegs<VEC>& r) const {
    TableView tv{};
    ApplyArgs x;
    locate(of, tv, x);
    load_row<OPT, VEC>(tv, row_of(of), e, on, x, r);
  }
  __device__ __forceinline__ void finish(uint32_t of, const float (&sum)[VEC], int e, bool on, int gl, bool last,
                                         RowRegs<VEC>& r) const {
    TableView tv{};
    ApplyArgs x;
    locate(of, tv, x);
    finish_row<OPT, VEC>(tv, row_of(of), sum, e, on, gl, last, a.dim, x, r);
  }

  // Where do the runs of the sorted list begin? Returns how many there are.
  __device__ __forceinline__ uint32_t find_runs(int len) const {
    const int t = threadIdx.x;
    const int per_lane = (len + kLanes - 1) / kLanes;
    const int j0 = t * per_lane;
    uint32_t heads = 0, runs;
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      const int j = j0 + i;
      if (i < per_lane && j < len && (j == 0 || ((s.key[j - 1] ^ s.key[j]) & low_mask))) heads |= 1u << i;
    }
    if (t == 0) s.n_long = s.n_wave = 0u;
    uint32_t r = run_scan((uint32_t)__popc(heads), s.wave_total, runs);
#pragma unroll
    for (int i = 0; i < kListItems; ++i)
      if (heads & (1u << i)) s.start[r++] = (uint16_t)(j0 + i);
    if (t == 0) s.start[runs] = (uint16_t)len;
    lds_barrier();
    const int wave_max = kPerGroup * (kWave / a.group);
    for (uint32_t q = (uint32_t)t; q < runs; q += kLanes) {
      const int count = (int)s.start[q + 1] - (int)s.start[q];
      if (count > wave_max) {
        s.long_run[atomicAdd(&s.n_long, 1u)] = (uint16_t)q;
      } else if (count > kShortest) {
        s.wave_run[atomicAdd(&s.n_wave, 1u)] = (uint16_t)q;
      }
    }
    lds_barrier();
    return runs;
  }

  // Adds the runs up. cut: all but the shortest ones, and the sums go to a.sums (the list's first entry
  // is entry `lo` of the pairs); otherwise every row is updated.
  __device__ __forceinline__ void reduce(uint32_t runs, bool cut, uint32_t lo) const {
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1);
    const int wave = t / kWave;
    const int gl = t & (a.group - 1);
    const int lt = t / a.group;
    const int groups = kLanes / a.group;
    const int per_wave = kWave / a.group;
    const int sub = lane / a.group;
    const uint32_t waves_runs = s.n_wave, longs = s.n_long;
    for (int e0 = 0; e0 < a.elems; e0 += a.group) {
      const int e = e0 + gl;
      const bool on = e < a.elems;
      const bool last = e0 + a.group >= a.elems;
      // runs for one wavefront each: its lane groups add a stretch each
      for (uint32_t k = (uint32_t)wave; k < waves_runs; k += kWaves) {
        const uint32_t q = s.wave_run[k];              // in any order: the runs are different rows
        const int first = s.start[q], end = s.start[q + 1];
        const int stretch = (end - first + per_wave - 1) / per_wave;
        const int from = min(first + sub * stretch, end), to = min(from + stretch, end);
        const uint32_t of = key_of(first);
        RowRegs<VEC> rec{};
        if (sub == 0 && !cut) load(of, e, on, rec);
        float acc[VEC];
        sum_entries(of, from, to, e, on, acc);
        fold_wave(acc);
        if (sub == 0) {
          if (cut) {
            if (on) share_row<VEC>(a.sums + (int64_t)((lo + (uint32_t)first) / kCutSum) * a.dim + e * VEC, acc);
          } else {
            finish(of, acc, e, on, gl, last, rec);
          }
        }
      }
      if (cut) {
        for (uint32_t q = (uint32_t)lt; q < runs; q += (uint32_t)groups) {
          const int first = s.start[q], end = s.start[q + 1];
          if (end - first < kCutSum || end - first > kShortest) continue;
          float acc[VEC];
          sum_entries(key_of(first), first, end, e, on, acc);
          if (on) share_row<VEC>(a.sums + (int64_t)((lo + (uint32_t)first) / kCutSum) * a.dim + e * VEC, acc);
        }
      }
      // short runs: one lane group each, two at a time, so that a round costs one trip to memory for
      // two records and their first gradient rows
      if (!cut) {
        constexpr int kHead = 2, kTail = 4;
        for (uint32_t q0 = (uint32_t)lt; q0 < runs; q0 += (uint32_t)(kPair * groups)) {
          int from[kPair], to[kPair];
          bool have[kPair];
          uint32_t of[kPair] = {};
          RowRegs<VEC> rec[kPair] = {};
          float head[kPair][kHead][VEC] = {};
#pragma unroll
          for (int x = 0; x < kPair; ++x) {
            const uint32_t q = q0 + (uint32_t)x * (uint32_t)groups;
            have[x] = q < runs;
            from[x] = have[x] ? (int)s.start[q] : 0;
            to[x] = have[x] ? (int)s.start[q + 1] : 0;
            if (to[x] - from[x] > kShortest) have[x] = false;   // a wavefront's or the workgroup's
            if (have[x]) {
              of[x] = key_of(from[x]);
              load(of[x], e, on, rec[x]);
#pragma unroll
              for (int u = 0; u < kHead; ++u)
                if (from[x] + u < to[x] && on) fetch(of[x], from[x] + u, e, head[x][u]);
            }
          }
#pragma unroll
          for (int x = 0; x < kPair; ++x) {
            if (!have[x]) continue;
            float acc[VEC] = {};
#pragma unroll
            for (int u = 0; u < kHead; ++u) {
              if (from[x] + u < to[x]) {
                if (on) scale(of[x], from[x] + u, head[x][u]);
#pragma unroll
                for (int c = 0; c < VEC; ++c) acc[c] = u == 0 ? head[x][u][c] : acc[c] + head[x][u][c];
              }
            }
            for (int j0 = from[x] + kHead; j0 < to[x]; j0 += kTail) {
              float v[kTail][VEC] = {};
#pragma unroll
              for (int u = 0; u < kTail; ++u)
                if (j0 + u < to[x] && on) fetch(of[x], j0 + u, e, v[u]);
#pragma unroll
              for (int u = 0; u < kTail; ++u) {
                if (j0 + u >= to[x]) break;
                if (on) scale(of[x], j0 + u, v[u]);
#pragma unroll
                for (int c = 0; c < VEC; ++c) acc[c] = acc[c] + v[u][c];
              }
            }
            finish(of[x], acc, e, on, gl, last, rec[x]);
          }
        }
      }
      // runs for the whole workgroup
      for (uint32_t k = 0; k < longs; ++k) {
        const uint32_t q = s.long_run[k];
        const int first = s.start[q], count = (int)s.start[q + 1] - first;
        const uint32_t of = key_of(first);
        RowRegs<VEC> rec{};
        if (lt == 0 && !cut) load(of, e, on, rec);   // on its way while the stretches are added
        float acc[VEC];
        sum_block(of, first, count, e, on, gl, acc);
        if (lt == 0) {
          if (cut) {
            if (on) share_row<VEC>(a.sums + (int64_t)((lo + (uint32_t)first) / kCutSum) * a.dim + e * VEC, acc);
          } else {
            finish(of, acc, e, on, gl, last, rec);
          }
        }
      }
    }
  }

  // Pooled requests: what the sums read of an entry besides its gradient row, once for all lanes of
  // its group. Weighted members' payloads are positions: they name the weight and the bag.
  __device__ __forceinline__ void resolve_weights(int len, float* weights, const uint32_t* bag_of) const {
    if constexpr (kPooled) {
      if (!weighted) return;
      for (int j = threadIdx.x; j < len; j += kLanes) {
        float x = 1.0f;
        if (!summed(j)) {
          const Member& m = member(key_of(j));
          if (m.weights) {
            const uint32_t p = s.ref[j];
            x = m.weights[p];
            const uint32_t word = bag_of[m.row_start + p];
            s.ref[j] = word == kNoBag ? 0u : word;
          }
        }
        weights[j] = x;
      }
      lds_barrier();
    }
  }
};

// Members of the request: one in registers, or all of them in LDS.
template <bool GROUPED>
__device__ __forceinline__ void load_members(Member* lds, const RunArgs& a, const TableView& tv,
                                             const ApplyArgs& args, const float* vals, const Source<GROUPED>& ps,
                                             const GroupSrc& gs) {
  if constexpr (GROUPED) {
    const int m = threadIdx.x;
    if (m < ps.call.n_tables) {
      const TableDesc& d = gs.descs[m];
      Member x;
      x.recs = d.tv.recs;
      x.stride = d.tv.stride;
      x.c0 = gs.st0 >= 0 ? d.col_off[gs.st0] : -1;
      x.c1 = gs.st1 >= 0 ? d.col_off[gs.st1] : -1;
      x.c2 = gs.st2 >= 0 ? d.col_off[gs.st2] : -1;
      x.meta_off = gs.use_meta ? d.meta_off : -1;
      x.rows = ps.call.rows[m];
      x.row_stride = ps.call.stride[m];
      x.weights = ps.pooled ? ps.call.weights[m] : nullptr;
      x.offsets = ps.pooled ? ps.call.offsets[m] : nullptr;
      x.mean = ps.pooled ? (ps.call.mean_bits >> m) & 1u : 0u;
      x.row_start = ps.pooled ? ps.call.row_start[m] : 0;
      lds[m] = x;
    }
  } else {
    Member& x = *lds;
    x.recs = tv.recs;
    x.stride = tv.stride;
    x.c0 = args.c0;
    x.c1 = args.c1;
    x.c2 = args.c2;
    x.meta_off = args.meta_off;
    x.rows = vals;
    x.row_stride = (uint32_t)a.dim;
    x.weights = ps.weight;
    x.offsets = ps.offsets;
    x.mean = ps.mean ? 1u : 0u;
    x.row_start = 0;
  }
}

constexpr int kOffsets = kWaves << kRunBits;           // lists whose offsets are held at a time, in `work`

// Sorts `n` entries by the low `bits` bits of their keys, where they do not fit into LDS: a digit at a time,
// from (h, refs) to (list_h, list_refs) and back, stable. Tiles of kListMax entries are sorted by the
// digit in LDS and appended to their digits' stretches. One workgroup, which is the only one that
// touches these entries by now. Returns whether the result lies in (list_h, list_refs).
__device__ __forceinline__ bool sort_far(RunLds& s, const RunArgs& a, uint32_t begin, uint32_t n, int bits) {
  const int t = threadIdx.x;
  const int passes = (bits + kRunBits - 1) / kRunBits;
  const int width = (bits + passes - 1) / passes;
  const uint32_t digit_mask = (1u << width) - 1u;
  static_assert((1 << kRunBits) == kLanes && sizeof(s.start) >= 2 * kLanes * sizeof(uint32_t), "a digit a lane");
  uint32_t* next = reinterpret_cast<uint32_t*>(s.start);   // where a digit's next entry goes
  uint32_t* first = next + kLanes;                         // where its entries begin in the tile
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = pass * width;
    const bool back = pass & 1;
    const uint32_t* src_h = (back ? a.list_h : a.h) + begin;
    const uint32_t* src_refs = (back ? a.list_refs : a.refs) + begin;
    uint32_t* dst_h = (back ? a.h : a.list_h) + begin;
    uint32_t* dst_refs = (back ? a.refs : a.list_refs) + begin;
    s.work[t] = 0u;
    lds_barrier();
    for (uint32_t j = (uint32_t)t; j < n; j += kLanes) atomicAdd(&s.work[(src_h[j] >> shift) & digit_mask], 1u);
    lds_barrier();
    uint32_t all;
    const uint32_t at = run_scan(s.work[t], s.wave_total, all);
    next[t] = at;
    for (uint32_t j0 = 0; j0 < n; j0 += kListMax) {
      const int len = (int)min((uint32_t)kListMax, n - j0);
      for (int j = t; j < len; j += kLanes) {
        s.key[j] = src_h[j0 + j];
        s.ref[j] = src_refs[j0 + j];
      }
      sort_list(s, len, width, shift);
      for (int j = t; j < len; j += kLanes) {
        const uint32_t d = (s.key[j] >> shift) & digit_mask;
        if (j == 0 || ((s.key[j - 1] >> shift) & digit_mask) != d) first[d] = (uint32_t)j;
      }
      lds_barrier();
      for (int j = t; j < len; j += kLanes) {
        const uint32_t d = (s.key[j] >> shift) & digit_mask;
        const uint32_t to = next[d] + (uint32_t)j - first[d];
        dst_h[to] = s.key[j];
        dst_refs[to] = s.ref[j];
      }
      lds_barrier();
      for (int j = t; j < len; j += kLanes) {
        const uint32_t d = (s.key[j] >> shift) & digit_mask;
        if (j == len - 1 || ((s.key[j + 1] >> shift) & digit_mask) != d) next[d] += (uint32_t)j + 1u - first[d];
      }
      lds_barrier();                                      // the next tile overwrites the entries
    }
    __syncthreads();                                      // the entries are where the next pass reads them
  }
  return passes & 1;
}

// Merges the lists of a cut bucket. weights: LDS for the entries' weights (pooled requests).
// Entries that do not fit into LDS are sorted in memory and taken a window at a time; every step is linear
// in the entries, whatever rows they are of. Gathering the lists again for every range of keys that fits
// walked all of them each time: pushes of 16,384 and of 65,536 pairs, all of one bucket's 16,384 rows of
// four floats, took 1.4 and 18 ms and take 0.53 and 1.5; of 2^20 pairs 24-34. The sort of such a
// request takes 0.05 to 0.16, but only rows as far apart as the multiplier's inverse share a bucket like
// this: of rows 1 to 4096 apart, in tables of 2^16 to 2^25 rows, none holds more than 2.1 times the average.
template <int OPT, int VEC, int FROM, bool GROUPED>
__device__ __forceinline__ void merge_lists(const Reducer<OPT, VEC, FROM, GROUPED, true>& r, const RunArgs& a,
                                            const CutBucket& cut, float* weights, const uint32_t* bag_of) {
  RunLds& s = r.s;
  const int t = threadIdx.x;
  const uint32_t pieces = a.cut.pieces(cut.len);
  uint32_t* offs = s.work;
  constexpr int kOwn = kOffsets / kLanes;

  // Where lists [c0, c0 + kOffsets) begin among these lists' entries, into offs; how many entries they are.
  auto offsets = [&](uint32_t c0) -> uint32_t {
    const uint32_t here = min((uint32_t)kOffsets, pieces - c0);
    const int own = (int)((here + kLanes - 1) / kLanes);   // 1..kOwn
    uint32_t n[kOwn], sum = 0, total;
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const uint32_t c = (uint32_t)(t * own + k);
      n[k] = k < own && c < here ? shared_word(a.plan.count + cut.base + c0 + c) : 0u;
      sum += n[k];
    }
    uint32_t at = run_scan(sum, s.wave_total, total);
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      if (k < own) offs[t * own + k] = at;
      at += n[k];
    }
    lds_barrier();
    return total;
  };
  uint32_t entries = 0;
  for (uint32_t c0 = 0; c0 < pieces; c0 += kOffsets) {
    entries += offsets(c0);
    lds_barrier();
  }
  const bool fits = entries <= (uint32_t)kListMax;     // uniform
  // the lists' entries, in list order, into LDS or over the bucket's pairs, which have been read
  for (uint32_t c0 = 0, before = 0; c0 < pieces; c0 += kOffsets) {
    const uint32_t here = min((uint32_t)kOffsets, pieces - c0);
    const uint32_t total = offsets(c0);
    constexpr int kTake = 4;                           // entries a lane takes a trip
    for (uint32_t e0 = 0; e0 < total; e0 += kLanes * kTake) {
      uint32_t key[kTake], ref[kTake];
#pragma unroll
      for (int k = 0; k < kTake; ++k) {
        const uint32_t e = e0 + (uint32_t)(k * kLanes + t);
        if (e < total) {
          uint32_t c = 0, hi = here;                   // the last list that begins at or before e
          while (hi - c > 1) {
            const uint32_t mid = (c + hi) / 2;
            if (offs[mid] <= e) c = mid; else hi = mid;
          }
          const uint32_t idx = cut.begin + (c0 + c) * a.cut.chunk + (e - offs[c]);
          key[k] = shared_word(a.list_h + idx);
          ref[k] = shared_word(a.list_refs + idx);
        }
      }
#pragma unroll
      for (int k = 0; k < kTake; ++k) {
        const uint32_t e = e0 + (uint32_t)(k * kLanes + t);
        if (e < total) {
          if (fits) {
            s.key[before + e] = key[k];
            s.ref[before + e] = ref[k];
          } else {
            a.h[cut.begin + before + e] = key[k];
            a.refs[cut.begin + before + e] = ref[k];
          }
        }
      }
    }
    before += total;
    lds_barrier();                                        // the offsets have been read
  }
  if (fits) {
    sort_list(s, (int)entries, r.low);
    const uint32_t runs = r.find_runs((int)entries);
    r.resolve_weights((int)entries, weights, bag_of);
    r.reduce(runs, false, 0u);
    return;
  }
  __syncthreads();                                        // the entries are in memory
  const bool in_lists = sort_far(s, a, cut.begin, entries, r.low);
  const uint32_t* sorted_h = (in_lists ? a.list_h : a.h) + cut.begin;
  const uint32_t* sorted_refs = (in_lists ? a.list_refs : a.refs) + cut.begin;
  auto window = [&](uint32_t from) -> int {
    const int len = (int)min((uint32_t)kListMax, entries - from);
    for (int j = t; j < len; j += kLanes) {
      s.key[j] = sorted_h[from + j];
      s.ref[j] = sorted_refs[from + j];
    }
    lds_barrier();
    return len;
  };
  for (uint32_t from = 0; from < entries;) {           // uniform
    int len = window(from);
    uint32_t runs = r.find_runs(len);
    bool whole_window = false;                         // of one row, which may go on behind it
    if (from + (uint32_t)len < entries) {
      if (runs > 1u) {                                 // the last row may go on: the next window's first
        len = s.start[runs - 1u];
        lds_barrier();
        runs = r.find_runs(len);
      } else {
        whole_window = true;
      }
    }
    if (!whole_window) {
      r.resolve_weights(len, weights, bag_of);
      r.reduce(runs, false, 0u);
      lds_barrier();                                      // the next window overwrites the entries
      from += (uint32_t)len;
      continue;
    }
    const uint32_t of_place = s.key[0] & r.low_mask;
    uint32_t end = from + (uint32_t)len;               // of the row's entries
    while (end < entries) {
      lds_barrier();
      len = window(end);
      runs = r.find_runs(len);
      const uint32_t more = (s.key[0] & r.low_mask) != of_place ? 0u : runs > 1u ? (uint32_t)s.start[1] : (uint32_t)len;
      end += more;
      if (more < (uint32_t)len) break;                 // uniform
    }
    // window by window, the first lane group keeps the sum
    const int gl = t & (a.group - 1);
    for (int e0 = 0; e0 < a.elems; e0 += a.group) {
      const int e = e0 + gl;
      const bool on = e < a.elems;
      float sum[VEC] = {};
      uint32_t of = 0;
      for (uint32_t at = from; at < end; at += kListMax) {
        lds_barrier();                                    // the last window has been read
        len = min(window(at), (int)(end - at));
        r.resolve_weights(len, weights, bag_of);
        of = r.key_of(0);
        float acc[VEC];
        r.sum_block(of, 0, len, e, on, gl, acc);
#pragma unroll
        for (int c = 0; c < VEC; ++c) sum[c] = at == from ? acc[c] : sum[c] + acc[c];
      }
      if (t < a.group) {
        RowRegs<VEC> rec{};
        r.load(of, e, on, rec);
        r.finish(of, sum, e, on, gl, e0 + a.group >= a.elems, rec);
      }
    }
    lds_barrier();
    from = end;
  }
}

template <int OPT, int VEC, int FROM, bool GROUPED>
__global__ __launch_bounds__(kLanes) void reduce_kernel(RunArgs a, TableView tv, ApplyArgs args,
                                                        const float* __restrict__ vals, Source<GROUPED> ps,
                                                        GroupSrc gs) {
  __shared__ RunLds s;
  __shared__ Member lds_members[GROUPED ? kMaxGroupTables : 1];
  __shared__ float weights[FROM == kBags ? kListMax : 1];
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int low = a.hash.bits - a.hash.bucket_bits;
  const uint32_t low_mask = (1u << low) - 1u;
  CutBucket cut;
  uint32_t piece = 0, which = 0, lo;
  int len;
  const bool is_cut = blockIdx.x < a.max_chunks;
  if (is_cut) {
    const uint32_t n_cut = a.plan.head[0];
    if (blockIdx.x >= a.plan.head[1]) return;
    // the last cut bucket whose chunks begin at or before this one
    for (uint32_t c0 = 0; c0 < n_cut; c0 += kWave) {
      const uint32_t c = c0 + (uint32_t)lane;
      const bool before = c < n_cut && a.plan.cut[c].base <= blockIdx.x;
      which += (uint32_t)__popcll(__ballot(before));
    }
    cut = a.plan.cut[--which];
    piece = blockIdx.x - cut.base;
    lo = cut.begin + piece * a.cut.chunk;
    len = (int)min(a.cut.chunk, cut.len - piece * a.cut.chunk);
  } else {
    cut.bucket = blockIdx.x - a.max_chunks;
    lo = a.plan.begin[cut.bucket];
    const uint32_t n = a.plan.begin[cut.bucket + 1] - lo;
    if (n == 0u || n > a.cut.whole) return;      // uniform for the workgroup, as the returns above
    len = (int)n;
  }
  for (int j = t; j < len; j += kLanes) {
    s.key[j] = a.h[lo + j] & low_mask;
    s.ref[j] = a.refs[lo + j];
  }
  Member one;
  load_members<GROUPED>(GROUPED ? lds_members : &one, a, tv, args, vals, ps, gs);
  bool weighted = false;
  const uint32_t* bag_of = nullptr;
  if constexpr (FROM == kBags) {
    if constexpr (GROUPED) weighted = ps.weighted; else weighted = ps.weight != nullptr;
    bag_of = ps.bag_of;
  }
  sort_list(s, len, low);
  const Reducer<OPT, VEC, FROM, GROUPED, false> r{
      s, a, GROUPED ? lds_members : &one, args, weights, ps.words, weighted, gs.row_bits, cut.bucket, low, low_mask, 0u};
  const uint32_t runs = r.find_runs(len);
  if (is_cut) {
    // the list: the shortest runs as they are, one entry for any other
    const int per_lane = (len + kLanes - 1) / kLanes;
    uint32_t keep = 0, is_long = 0, kept;
    {
      // the run of the lane's first entry: the last one that starts at or before it
      int q = 0;
      if (t * per_lane < len) {
        int hi = (int)runs;
        while (hi - q > 1) {
          const int mid = (q + hi) / 2;
          if ((int)s.start[mid] <= t * per_lane) q = mid; else hi = mid;
        }
      }
#pragma unroll
      for (int i = 0; i < kListItems; ++i) {
        const int j = t * per_lane + i;
        if (i < per_lane && j < len) {
          if (j >= (int)s.start[q + 1]) ++q;
          const bool lng = (int)s.start[q + 1] - (int)s.start[q] >= kCutSum;
          if (!lng || j == (int)s.start[q]) keep |= 1u << i;
          if (lng) is_long |= 1u << i;
        }
      }
    }
    uint32_t at = lo + run_scan((uint32_t)__popc(keep), s.wave_total, kept);
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      if (keep & (1u << i)) {
        const int j = t * per_lane + i;
        const bool lng = (is_long >> i) & 1u;
        share(a.list_h + at, s.key[j] | (lng ? kSummed : 0u));
        share(a.list_refs + at, lng ? (lo + (uint32_t)j) / kCutSum : s.ref[j]);
        ++at;
      }
    }
    if (t == 0) share(a.plan.count + blockIdx.x, kept);
    lds_barrier();
  }
  r.resolve_weights(len, weights, bag_of);
  r.reduce(runs, is_cut, lo);
  if (!is_cut) return;
  // the workgroup that is through last merges
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this wavefront's part of the list and sums is out
  __syncthreads();
  if (t == 0) {
    const uint32_t pieces = a.cut.pieces(cut.len);
    const uint32_t before = __hip_atomic_fetch_add(a.plan.done + which, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s.last = before + 1u == pieces ? 1u : 0u;
  }
  __syncthreads();
  if (!s.last) return;
  const Reducer<OPT, VEC, FROM, GROUPED, true> m{
      s, a, GROUPED ? lds_members : &one, args, weights, ps.words, weighted, gs.row_bits, cut.bucket, low, low_mask, 0u};
  merge_lists<OPT, VEC, FROM, GROUPED>(m, a, cut, weights, bag_of);
}

// ---- requests of at most kPickMax ids a table: no partition ------------------------------------
// One launch, a workgroup per (member, bucket), that reads the member's keys (at most eight a lane) and
// keeps those of its bucket. What bounds it are latencies: the keys, then records and gradient rows,
// and some 3 us of LDS phases, which is why the workgroup has four wavefronts: a barrier among
// sixteen, of which a few dozen entries need one, is 0.2 us (bucket_push_kernel on 100 ids of 8
// floats, keys 1.1, picking 2.1, sort 0.4, runs 1.8, updates 1.6 us).
struct PickArgs {
  const uint32_t* keys;          // rows, members' numbers above them, or noted rows
  uint32_t miss_key, row_mask;
  bool noted;                    // (kEmptyRow: look the id up, see NotedRows)
  const uint64_t* ids;           // of a single table
  int n;
};

template <int OPT, int VEC, int FROM, bool GROUPED>
__global__ __launch_bounds__(kLanes) void pick_kernel(RunArgs a, PickArgs p, TableView tv, ApplyArgs args,
                                                      const float* __restrict__ vals, Source<GROUPED> ps, GroupSrc gs) {
  __shared__ RunLds s;
  __shared__ Member lds_members[GROUPED ? kMaxGroupTables : 1];
  __shared__ float weights[FROM == kBags ? kListMax : 1];
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  const int low = a.hash.bits - a.hash.bucket_bits;
  const uint32_t low_mask = (1u << low) - 1u;
  const int m = GROUPED ? (int)(blockIdx.x >> a.hash.bucket_bits) : 0;
  const uint32_t bucket = blockIdx.x & ((1u << a.hash.bucket_bits) - 1u);
  int64_t first = 0;
  int all = p.n;
  const uint64_t* ids = p.ids;
  bool weighted = false, positions = false;            // positions: payloads of this member are positions
  const uint32_t* bag_of = nullptr;
  if constexpr (GROUPED) {
    first = ps.call.row_start[m];
    all = (int)(ps.call.row_start[m + 1] - first);
    ids = ps.call.ids[m];
    tv = gs.descs[m].tv;
    if constexpr (FROM == kBags) positions = weighted = ps.call.weights[m] != nullptr;
  } else if constexpr (FROM == kBags) {
    positions = weighted = ps.weight != nullptr;
  }
  if constexpr (FROM == kBags) bag_of = ps.bag_of;
  if (all <= 0) return;                                // uniform for the workgroup
  // item i of lane l in wavefront w is position (w * own + i) * 64 + l: taking i in ascending order visits
  // a wavefront's positions in order
  const int own = (all + kLanes - 1) / kLanes;         // 1..kListItems
  const int base = wave * own * kWave + lane;
  uint32_t key[kListItems], ref[kListItems];
#pragma unroll
  for (int i = 0; i < kListItems; ++i) {
    const int j = base + i * kWave;
    key[i] = i < own && j < all ? p.keys[first + j] : 0xFFFFFFFFu;
    ref[i] = (uint32_t)j;
    if constexpr (FROM == kBags) {
      if (!positions && i < own && j < all) ref[i] = bag_of[first + j];
    }
  }
  Member one;
  load_members<GROUPED>(GROUPED ? lds_members : &one, a, tv, args, vals, ps, gs);
  if (p.noted) {
#pragma unroll
    for (int i = 0; i < kListItems; ++i) {
      const int j = base + i * kWave;
      if (i < own && j < all && key[i] == kEmptyRow) key[i] = probe_find_alone(tv, ids[j]);
    }
  }
  // the bucket's positions, in order
  unsigned long long take[kListItems];
  uint32_t mine = 0;
#pragma unroll
  for (int i = 0; i < kListItems; ++i) {
    const bool live = i < own && key[i] < p.miss_key;
    key[i] = ((key[i] & p.row_mask) * a.hash.mult) & a.hash.mask;
    take[i] = __ballot(live && key[i] >> low == bucket);
    mine += (uint32_t)__popcll(take[i]);
  }
  if (lane == 0) s.wave_total[wave] = mine;
  lds_barrier();
  uint32_t at = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t x = s.wave_total[w];
    if (w < wave) at += x;
    total += x;
  }
  const int len = (int)total;
  if (len == 0) return;                                // uniform
#pragma unroll
  for (int i = 0; i < kListItems; ++i) {
    if (take[i] & (1ull << lane)) {
      const uint32_t to = at + (uint32_t)__popcll(take[i] & ((1ull << lane) - 1ull));
      s.key[to] = key[i] & low_mask;
      s.ref[to] = ref[i];
    }
    at += (uint32_t)__popcll(take[i]);
  }
  sort_list(s, len, low);
  const Reducer<OPT, VEC, FROM, GROUPED, false> r{
      s, a, GROUPED ? lds_members : &one, args, weights, ps.words, weighted, gs.row_bits, bucket, low, low_mask,
      GROUPED ? (uint32_t)m << gs.row_bits : 0u};
  const uint32_t runs = r.find_runs(len);
  r.resolve_weights(len, weights, bag_of);
  r.reduce(runs, false, 0u);
}

template <int OPT, int VEC, int FROM, bool GROUPED>
int32_t launch_reduce(const RunArgs& a, const PickArgs* pick, const TableView& tv, const ApplyArgs& args,
                      const float* vals, const Source<GROUPED>& ps, const GroupSrc& gs, hipStream_t stream) {
  if (pick) {
    unsigned members = 1;
    if constexpr (GROUPED) members = (unsigned)ps.call.n_tables;
    hipLaunchKernelGGL((pick_kernel<OPT, VEC, FROM, GROUPED>), dim3(members << a.hash.bucket_bits), dim3(kLanes), 0,
                       stream, a, *pick, tv, args, vals, ps, gs);
    KRK_HIP(hipGetLastError());
    return KRK_SUCCESS;
  }
  hipLaunchKernelGGL((reduce_kernel<OPT, VEC, FROM, GROUPED>), dim3(a.max_chunks + (1u << a.hash.bucket_bits)),
                     dim3(kLanes), 0, stream, a, tv, args, vals, ps, gs);
  KRK_HIP(hipGetLastError());
  return KRK_SUCCESS;
}

template <int OPT, int VEC>
int32_t launch_source(const RunArgs& a, const PickArgs* pick, const TableView& tv, const ApplyArgs& args, const float* vals,
                      const PooledSrc& ps, const GroupSrc* gs, const GroupPooledSrc* gps, hipStream_t stream) {
  const GroupSrc plain{nullptr, 0, -1, -1, -1, 0};
  if constexpr (OPT != kOptStore) {
    if (gs) {
      return gps->pooled ? launch_reduce<OPT, VEC, kBags, true>(a, pick, tv, args, vals, *gps, *gs, stream)
                         : launch_reduce<OPT, VEC, kRows, true>(a, pick, tv, args, vals, *gps, *gs, stream);
    }
    if (ps.pooled) return launch_reduce<OPT, VEC, kBags, false>(a, pick, tv, args, vals, ps, plain, stream);
  }
  return launch_reduce<OPT, VEC, kRows, false>(a, pick, tv, args, vals, ps, plain, stream);
}

template <int VEC>
int32_t launch_opt(int opt, const RunArgs& a, const PickArgs* pick, const TableView& tv, const ApplyArgs& args, const float* vals,
                   const PooledSrc& ps, const GroupSrc* gs, const GroupPooledSrc* gps, hipStream_t stream) {
  switch (opt) {
    case kOptStore: return launch_source<kOptStore, VEC>(a, pick, tv, args, vals, ps, gs, gps, stream);
    case KRK_SGD: return launch_source<KRK_SGD, VEC>(a, pick, tv, args, vals, ps, gs, gps, stream);
    case KRK_ADAGRAD: return launch_source<KRK_ADAGRAD, VEC>(a, pick, tv, args, vals, ps, gs, gps, stream);
    case KRK_ADAM: return launch_source<KRK_ADAM, VEC>(a, pick, tv, args, vals, ps, gs, gps, stream);
    default: return launch_source<KRK_RMSPROP, VEC>(a, pick, tv, args, vals, ps, gs, gps, stream);
  }
}

// Buckets of a request of n pairs: a hundred pairs each, as long as a tile's counts of them are little
// work for the partition (64 or 256 a bucket are within 3 % of it from 20,000 to 300,000 ids).
int bucket_bits_for(int64_t n) {
  int bits = 8;
  while (bits < 10 && ((int64_t)128 << bits) < n) ++bits;
  return bits;
}
// A chunk is what one workgroup walks, and what it walks longest is one row's gradients; with chunks
// shorter than a bucket commonly is, though, most buckets are cut. Reduction with chunks of 512 / 1024 /
// 2048 pairs, us: 50,000 ids of 100 floats 39 / 49 / 69, 300,000 of 32 38 / 38 / 47, a million of 16
// 107 / 74 / 76, of 128 (Zipf 1.3) 186 / 150 / 170.
uint32_t chunk_for(int64_t n) { return n > ((int64_t)1 << 18) ? kListMax / 2 : kListMax / 4; }
// Nor may buckets be cut because they hold many pairs on average: a bucket stays whole up to a quarter more
// than that (distinct rows vary by a twentieth, rows at even distances by up to a third). A push of 2^20
// ids, us, cut from a chunk on / by this rule / sorted: distinct rows of 16 floats 186 / 131 / 164, of
// 128 768 / 624 / 638; consecutive ones of 128 757 / 608 / 609; Zipf 1.05 and 1.3, of 128, 277 / 278 / 324 and
// 187 / 185 / 236 (277-287 and 191 with whole buckets of up to two chunks).
uint32_t whole_for(int64_t n, int bucket_bits) {
  return std::max(chunk_for(n), (uint32_t)((n >> bucket_bits) * 5 / 4));
}
static_assert((kRunsMax >> 10) * 5 / 4 <= kListMax, "a whole bucket is one workgroup's");

// Places of keys below `keys`.
RunHash make_hash(int bucket_bits, uint64_t keys) {
  RunHash h;
  h.bucket_bits = bucket_bits;
  h.bits = bucket_bits + 1;
  while (h.bits < 32 && ((uint64_t)1 << h.bits) < keys) ++h.bits;
  h.mask = h.bits >= 32 ? 0xFFFFFFFFu : (1u << h.bits) - 1u;
  h.mult = 0x9E3779B1u;
  h.inverse = h.mult;                                  // Newton's iteration: right to 3, 6, 12, 24, 48 bits
  for (int i = 0; i < 4; ++i) h.inverse *= 2u - h.mult * h.inverse;
  return h;
}

// Buckets and chunks of a request, and what its plan takes.
struct RunShape {
  int bucket_bits;
  RunCut cut;
  size_t buckets, cuts, chunks;
  RunShape(int64_t n) {
    bucket_bits = bucket_bits_for(n);
    cut = RunCut{whole_for(n, bucket_bits), chunk_for(n)};
    buckets = (size_t)1 << bucket_bits;
    cuts = (size_t)(n / cut.chunk);      // a cut bucket holds more than that, in at most twice as many chunks
    chunks = 2 * cuts;
  }
  size_t plan_words() const { return 4 * cuts + 4 + (buckets + 1) + cuts + chunks; }
};
// The longest requests of a form that takes more work space than the next one does: small tiles of the
// partition, short chunks.
constexpr int64_t kShapeEdges[] = {(int64_t)1 << 16, (int64_t)1 << 18};

}  // namespace

int32_t reserve_runs(const ReduceShape& sh, DeviceBuffer* scratch, int64_t n) {
  const RunShape r(n);
  size_t partition = partition_work_bytes(n, r.bucket_bits), plan = r.plan_words();
  for (const int64_t edge : kShapeEdges) {
    if (edge >= n) break;
    // so that a shorter request that follows finds its room there: freeing waits for the device
    const RunShape shorter(edge);
    partition = std::max(partition, partition_work_bytes(edge, shorter.bucket_bits));
    plan = std::max(plan, shorter.plan_words());
  }
  KRK_TRY(scratch[0].reserve(4 * (size_t)n * sizeof(uint32_t)));   // keys, payload, and as much again
  KRK_TRY(scratch[1].reserve(partition));
  KRK_TRY(scratch[2].reserve(plan * sizeof(uint32_t)));
  // The sum of a run of kCutSum entries lies where the run's first pair does, divided by kCutSum: which
  // buckets are cut is known on the device only, so there is room for all (134 MB for 2^20 pairs of 128 floats,
  // a quarter of their gradient rows).
  return scratch[3].reserve(r.cuts ? (size_t)(n / kCutSum + 1) * (size_t)sh.dim * sizeof(float) : 0);
}

int32_t reduce_runs(const ReduceShape& sh, hipStream_t stream, DeviceBuffer* scratch, const TableView& tv, int opt,
                    int64_t n, uint32_t miss_key, const NotedRows& noted, const float* vals, const ApplyArgs& args,
                    const PooledSrc& ps, const GroupSrc* gs, const GroupPooledSrc* gps) {
  const RunShape shape(n);
  RunArgs a{};
  a.hash = make_hash(shape.bucket_bits, miss_key);
  a.cut = shape.cut;
  a.max_chunks = (uint32_t)shape.chunks;
  a.dim = (int)sh.dim;
  a.elems = sh.elems;
  a.group = sh.group;
  uint32_t* word = scratch[2].as<uint32_t>();
  a.plan.cut = reinterpret_cast<CutBucket*>(word);
  word += 4 * shape.cuts;
  a.plan.head = word;
  word += 4;
  a.plan.begin = word;
  word += shape.buckets + 1;
  a.plan.done = word;
  word += shape.cuts;
  a.plan.count = word;
  a.sums = scratch[3].as<float>();
  uint32_t* pairs = scratch[0].as<uint32_t>();
  uint32_t* h = pairs + 2 * n;
  KRK_TRY(partition_pairs(pairs, pairs + n, noted, tv, n, miss_key, a.hash, h, h + n, a.cut, a.plan, scratch[1].ptr,
                          stream));
  a.h = h;
  a.refs = h + n;
  a.list_h = pairs;                                    // the partition's input has been read
  a.list_refs = pairs + n;
  if (sh.vec == 4) return launch_opt<4>(opt, a, nullptr, tv, args, vals, ps, gs, gps, stream);
  return launch_opt<1>(opt, a, nullptr, tv, args, vals, ps, gs, gps, stream);
}

int32_t pick_runs(const ReduceShape& sh, hipStream_t stream, const TableView& tv, int opt, const uint32_t* keys,
                  uint32_t miss_key, int row_bits, uint32_t row_mask, const uint64_t* noted_ids, bool noted, int64_t n,
                  int64_t longest, const float* vals, const ApplyArgs& args, const PooledSrc& ps, const GroupSrc* gs,
                  const GroupPooledSrc* gps) {
  const int members = gps ? gps->call.n_tables : 1;
  // sixteen pairs a bucket, as long as that is two workgroups a compute unit at most (8 and 32 pairs, and
  // twice the workgroups, are within 5 % of it)
  int bits = 3;
  while (bits < 8 && ((int64_t)16 << bits) < longest && (members << (bits + 1)) <= 512) ++bits;
  RunArgs a{};
  a.hash = make_hash(bits, (uint64_t)1 << row_bits);
  a.dim = (int)sh.dim;
  a.elems = sh.elems;
  a.group = sh.group;
  const PickArgs pick{keys, miss_key, row_mask, noted, noted_ids, (int)n};
  if (sh.vec == 4) return launch_opt<4>(opt, a, &pick, tv, args, vals, ps, gs, gps, stream);
  return launch_opt<1>(opt, a, &pick, tv, args, vals, ps, gs, gps, stream);
}

}  // namespace krk
