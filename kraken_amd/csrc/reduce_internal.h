// What the kernels that add gradients up and update rows have in common: vector accesses, a lane's
// slice of a record and its update, and where the gradient rows of a request lie.
#pragma once

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "sparse_internal.h"

namespace krk {

constexpr int kBlock = 256;
constexpr uint32_t kNoRow = 0xFFFFFFFFu;

template <int VEC>
__device__ __forceinline__ void vload(const float* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  } else {
    v[0] = *p;
  }
}
template <int VEC>
__device__ __forceinline__ void vstore_once(float* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const vfloat4_t x = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(x, reinterpret_cast<vfloat4_t*>(p));
  } else {
    __builtin_nontemporal_store(v[0], p);
  }
}
// A row that is read exactly once (the gradient rows a reduction gathers): non-temporal, so the
// half gigabyte that passes through does not push the table's records out of the caches.
template <int VEC>
__device__ __forceinline__ void gload_once(const KRK_GLOBAL float* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const vfloat4_t x = __builtin_nontemporal_load((const KRK_GLOBAL vfloat4_t*)p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  } else {
    v[0] = __builtin_nontemporal_load(p);
  }
}
template <int VEC>
__device__ __forceinline__ void gstore_once(float* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const vfloat4_t x = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(x, (KRK_GLOBAL vfloat4_t*)p);
  } else {
    __builtin_nontemporal_store(v[0], (KRK_GLOBAL float*)p);
  }
}
template <int VEC>
__device__ __forceinline__ void vstore(float* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    *p = v[0];
  }
}

static inline unsigned grid_for(int64_t items, int per_block) {
  return (unsigned)((items + per_block - 1) / per_block);
}

// A payload or bag word that stands for "outside every bag".
constexpr uint32_t kNoBag = 0xFFFFFFFFu;

// What a pooled push carries for a position instead of a bag number alone: the bag in the low
// bag_bits bits and above them the bag's length, as far as it fits (all ones: look it up). A mean bag
// hands on grads * ratio, ratio = (float)(1.0 / float(len)) (pytorch/py/jagged_ops.cc:303-334), and
// the length is what the reduction needs for that: a scaled copy of the gradients takes a pass of
// its own (852k bags of 32 floats: 85 us), and an array of ratios costs the reduction one more
// random read per entry (8.5 million entries: 585 us instead of 461).
struct BagWord {
  int bag_bits;                          // bags < 2^bag_bits, so that no word is kNoBag
  __host__ __device__ uint32_t bag(uint32_t w) const { return w & ((1u << bag_bits) - 1u); }
  __host__ __device__ uint32_t longest() const { return (1u << (32 - bag_bits)) - 1u; }
  __device__ uint32_t pack(uint32_t b, long long len) const {
    const uint32_t most = longest();
    return b | ((len < (long long)most ? (uint32_t)(len < 0 ? 0 : len) : most) << bag_bits);
  }
};
inline BagWord bag_word(int64_t bags) {
  BagWord w{1};
  while (((int64_t)1 << w.bag_bits) <= bags) ++w.bag_bits;
  return w;
}
// 1.0f / x in fp32 is (float)(1.0 / (double)x) for every fp32 x that is a whole number: the quotient
// of two 24-bit significands is never close enough to the middle of two floats for the
// intermediate rounding to matter.
__device__ __forceinline__ float mean_ratio(long long len) { return len > 0 ? 1.0f / (float)len : 0.0f; }
__device__ __forceinline__ float mean_ratio(const BagWord& words, uint32_t word, const long long* offsets) {
  const uint32_t len = word >> words.bag_bits, b = words.bag(word);
  return mean_ratio(len == words.longest() ? offsets[b + 1] - offsets[b] : (long long)len);
}

struct ApplyArgs {
  float lr;
  RowOptimK k;
  int c0, c1, c2, meta_off;
};

// What a closed run does with its sum: one of the four optimizers, or (stand-alone dedup + sum)
// just store it as row `row` of the output.
constexpr int kOptStore = 4;

// A lane's slice of a record: weight and the optimizer's state columns.
template <int VEC>
struct RowRegs {
  float w[VEC], s0[VEC], s1[VEC], s2[VEC];
};

// Requests the lane's slice of row `row`. Kept apart from the update so that a caller can have
// the record on its way while it is still adding up the row's gradient.
template <int OPT, int VEC>
__device__ __forceinline__ void load_row(const TableView& tv, uint32_t row, int e, bool lane_on, const ApplyArgs& a,
                                         RowRegs<VEC>& r) {
  if constexpr (OPT == kOptStore) return;
  const float* rec = tv.recs + (int64_t)row * tv.stride;
  if (lane_on) {
    gload<VEC>(rec + e * VEC, r.w);
    if (a.c0 >= 0) gload<VEC>(rec + a.c0 + e * VEC, r.s0);
    if (a.c1 >= 0) gload<VEC>(rec + a.c1 + e * VEC, r.s1);
    if (a.c2 >= 0) gload<VEC>(rec + a.c2 + e * VEC, r.s2);
  }
}

// The update of row `row` with the summed gradient, on the slice load_row requested.
template <int OPT, int VEC>
__device__ __forceinline__ void finish_row(const TableView& tv, uint32_t row, const float (&gsum)[VEC], int e,
                                           bool lane_on, int gl, bool last_chunk, int dim, const ApplyArgs& a,
                                           RowRegs<VEC>& r) {
  float* rec = tv.recs + (int64_t)row * tv.stride;
  if constexpr (OPT == kOptStore) {
    if (lane_on) vstore<VEC>(rec + e * VEC, gsum);
    return;
  }
  bool first = false;
  float bc1 = 1.0f, bc2 = 1.0f;
  uint64_t steps = 0;
  if (a.meta_off >= 0) {
    const KRK_GLOBAL uint32_t* meta = (const KRK_GLOBAL uint32_t*)(rec + a.meta_off);
    steps = (uint64_t)meta[0] | ((uint64_t)meta[1] << 32);
    if (OPT == KRK_ADAM) {
      steps += 1;                           // the flag bit rides along untouched
    } else {
      first = (steps & kHasMomentumBit) == 0;
      steps |= kHasMomentumBit;
    }
    if (OPT == KRK_ADAM) {
      bc1 = one_minus_power(a.k.log2_beta1, a.k.beta1, steps & ~kHasMomentumBit);
      bc2 = one_minus_power(a.k.log2_beta2, a.k.beta2, steps & ~kHasMomentumBit);
    }
  }
  if (lane_on) {
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      if (a.c0 < 0) r.s0[c] = 0.0f;
      if (a.c1 < 0) r.s1[c] = 0.0f;
      if (a.c2 < 0) r.s2[c] = 0.0f;
      optim_element<OPT>(a.k, a.lr, gsum[c], r.w[c], r.s0[c], r.s1[c], r.s2[c], first, bc1, bc2);
    }
    // a record is written once per request: past the caches, so the kernel ends with no dirty
    // lines to write back
    gstore_once<VEC>(rec + e * VEC, r.w);
    if (a.c0 >= 0) gstore_once<VEC>(rec + a.c0 + e * VEC, r.s0);
    if (a.c1 >= 0) gstore_once<VEC>(rec + a.c1 + e * VEC, r.s1);
    if (a.c2 >= 0) gstore_once<VEC>(rec + a.c2 + e * VEC, r.s2);
  }
  // The counter is read by every chunk of the row before the last chunk advances it.
  if (a.meta_off >= 0 && last_chunk) store_row_word<VEC>(rec + a.meta_off, steps, gl, dim, (int)tv.stride - a.meta_off);
}

// The lane's slice of the record is requested before the 64-bit word is looked at: the bias
// corrections then overlap with the loads instead of preceding them.
template <int OPT, int VEC>
__device__ __forceinline__ void apply_row(const TableView& tv, uint32_t row, const float (&gsum)[VEC],
                                          int e, bool lane_on, int gl, bool last_chunk, int dim,
                                          const ApplyArgs& a) {
  RowRegs<VEC> r;
  load_row<OPT, VEC>(tv, row, e, lane_on, a, r);
  finish_row<OPT, VEC>(tv, row, gsum, e, lane_on, gl, last_chunk, dim, a, r);
}

// ---- a request's (key, payload) pairs ----------------------------------------------------------
// Pooled pushes . Weighted bags: the payload is a position p, its gradient row
// is that of bag bag_of[p], times weight[p]; otherwise weight is null and the payload itself names
// the bag. pooled false: the payload names the gradient row.
struct PooledSrc {
  bool pooled, mean;
  BagWord words;
  const uint32_t* bag_of;
  const float* weight;
  const long long* offsets;
};
// The same for a combined push: the gradient rows lie where the members have them, and payloads
// and bags count from the member's first.
struct GroupPooledSrc {
  PooledCall call;
  BagWord words;
  const uint32_t* bag_of;
  bool pooled, weighted;          // weighted: some member is
};
// Combined pushes (GROUPED): a key is (member number << row_bits) | row, and a closed run takes
// its member's record layout from descs. st0..st2 are the state types of the optimizer's three
// slots (-1 = unused); the column each lives in differs from member to member.
struct GroupSrc {
  const TableDesc* descs;
  int row_bits;
  int st0, st1, st2;
  int use_meta;
};

// Row width and lane mapping of a reduction: a table's, or those of a stand-alone call.
struct ReduceShape {
  int64_t dim;
  int vec, elems, group;
};

// A barrier for phases that exchange data through LDS only: waits for the wavefront's LDS operations, not
// for its global loads and stores as __syncthreads() does.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Stable sort of a short list in LDS by the bits `mask` of the key: every lane counts the entries that
// come before its own. All lanes of the workgroup call it, a barrier behind the list's writes; key
// lies on 16 bytes, and up to the next multiple of four entries it holds 0xFFFFFFFF behind the list.
// A radix sort takes 1.7 us a pass whatever the length, each pass a chain of LDS round trips and
// barriers; this one reads four keys at a time, the same ones in all lanes, and has two barriers.
constexpr int kRankMax = 256;
template <typename Ref>
__device__ __forceinline__ void rank_list(uint32_t* key, Ref* ref, int len, uint32_t mask) {
  const int t = threadIdx.x;
  const int base = __builtin_amdgcn_readfirstlane(t / kWave * kWave);
  uint32_t whole = 0u, rank = 0u;
  Ref r = 0;
  if (base < len) {
    if (t < len) {
      whole = key[t];
      r = ref[t];
    }
    const uint32_t k = whole & mask;
    const uint4* four = reinterpret_cast<const uint4*>(key);
    for (int j = 0; j < base; j += 4) {
      const uint4 x = four[j / 4];
      rank += ((x.x & mask) <= k) + ((x.y & mask) <= k) + ((x.z & mask) <= k) + ((x.w & mask) <= k);
    }
    const int past = len < base + kWave ? len : base + kWave;
    for (int j = base; j < past; j += 4) {
      const uint4 x = four[j / 4];
      rank += ((x.x & mask) < k + (j < t)) + ((x.y & mask) < k + (j + 1 < t)) + ((x.z & mask) < k + (j + 2 < t)) +
              ((x.w & mask) < k + (j + 3 < t));
    }
    for (int j = base + kWave; j < len; j += 4) {
      const uint4 x = four[j / 4];
      rank += ((x.x & mask) < k) + ((x.y & mask) < k) + ((x.z & mask) < k) + ((x.w & mask) < k);
    }
  }
  lds_barrier();                                       // everyone has read the list
  if (t < len) {
    key[rank] = whole;
    ref[rank] = r;
  }
  lds_barrier();
}

// Rows of a single table's positions as the pull of these ids noted them (KRK_IDS_AS_PULLED), in place of
// keys and payloads. A note of kEmptyRow was taken while the row's creator, another wavefront of
// that pull, had not published its number yet: those ids are looked up.
struct NotedRows {
  const uint32_t* rows;
  const uint64_t* ids;
};

// The key of a position whose row was noted.
__device__ __forceinline__ uint32_t noted_key(const TableView& tv, uint32_t row, const uint64_t* __restrict__ id,
                                              uint32_t member_key, uint32_t miss_key) {
  if (row == kEmptyRow) {
    row = probe_find_alone(tv, *id);
    if (row == kEmptyRow) {
      atomicOr(&tv.counters[1], kErrMissingId);
      return miss_key;
    }
  }
  return member_key | row;
}

// The positions of a single table's pooled push whose rows the pull noted, in place of keys and payloads.
struct NotedBags {
  const uint32_t* rows;
  const uint64_t* ids;
  const long long* offsets;      // null: the pairs come from somewhere else
  int64_t bags;
  BagWord words;
  uint32_t* bag_of;              // null: a payload is a bag's word. Otherwise it is the position, and the word goes here
};

// radix_sort_pairs (krk_internal.h) of the pairs that these positions are; its first pass puts them together
// (radix_sort.hip). The first two arrays may be written as the others are.
int32_t radix_sort_noted_bags(const NotedBags& bags, const TableView& tv, uint32_t miss_key, uint32_t* keys,
                              uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n, int bits, void* work,
                              hipStream_t stream, uint32_t** keys_sorted, uint32_t** vals_sorted);

// ---- partition.hip -----------------------------------------------------------------------------
// Which workgroup of the reduction takes what: the pairs of a bucket lie side by side, and a bucket
// of more than `whole` pairs is cut into chunks of `chunk`.
struct RunCut {
  uint32_t whole, chunk;
  __host__ __device__ uint32_t pieces(uint32_t len) const { return (len + chunk - 1u) / chunk; }
};
struct CutBucket {
  uint32_t bucket;
  uint32_t base;       // chunks of the cut buckets before this one
  uint32_t begin, len; // its pairs
};
struct RunPlan {
  uint32_t* begin;     // [buckets + 1] where a bucket's pairs start
  uint32_t* head;      // [0] cut buckets, [1] their chunks
  CutBucket* cut;      // in ascending order of bucket and base
  uint32_t* done;      // chunks of each cut bucket that are through
  uint32_t* count;     // entries that each chunk of a cut bucket leaves for the merge
};
// A key's place: h = key * mult mod 2^bits, an odd multiplier, so that no two keys share it; the
// upper bucket_bits of h are the bucket.
struct RunHash {
  uint32_t mult, inverse, mask;
  int bits, bucket_bits;
};
// Requests of more pairs are sorted (radix_sort.hip). Up to here 1024 buckets of 1024 pairs on average, which a
// workgroup's LDS holds twice over, and the scatter's 32-bit counts of that many buckets for sixteen
// wavefronts fill 104 of the 160 KB. Pushes just below the line, us, buckets / sort: 2^20 ids of 16
// floats, distinct / consecutive / Zipf 1.05 / 1.3, 124 / 121 / 98 / 86 against 163 / 150 / 133 / 132; of 128 floats
// 617 / 602 / 268 / 185 against 640 / 590 / 297 / 217 (rows of 256 and 512 floats, distinct, 1145 and 2236 against
// 1043 and 2126, Zipf 1.3 310 and 570 against 355 and 648: the sort leaves the rows in the order they lie in).
// Above it, with 2048 buckets of 16-bit counts, which cost 3 to 9 % below it: 1.5 million ids of 128
// floats 882 / 868 / 382 / 242 against 886 / 842 / 435 / 301, 2^21 1208 / 1198 / 508 / 313 against 1200 / 1141 / 562 / 382,
// i.e. skewed requests gain a tenth to a fifth and consecutive rows lose a twentieth. (The sort's side of all this is
// from before spans of one row had a way of their own; with that, forward, backward and forward by buckets / by the
// sort: 2^20 ids of 128 floats, Zipf 1.3, 360 / 401, a million of 16, Zipf 1.05, 139 / 180, 950,000 pooled of 32,
// Zipf 1.1, 158 / 193.)
constexpr int64_t kRunsMax = (int64_t)1 << 20;
// Bytes of the partition's work space.
size_t partition_work_bytes(int64_t n, int bucket_bits);
// Groups n (key, payload) pairs by bucket, in their order inside one; pairs whose key is miss_key or
// above are left out, and keys become their h. noted: the rows of the pairs' positions in place of
// keys and payloads.
int32_t partition_pairs(const uint32_t* keys, const uint32_t* refs, const NotedRows& noted, const TableView& tv,
                        int64_t n, uint32_t miss_key, const RunHash& hash, uint32_t* out_h, uint32_t* out_refs,
                        const RunCut& cut, const RunPlan& plan, void* work, hipStream_t stream);

// ---- run_reduce.hip ----------------------------------------------------------------------------
// Work space for n pairs: scratch[0] holds the n keys, then the n payloads, and as much again;
// scratch[1..3] what the steps need.
int32_t reserve_runs(const ReduceShape& sh, DeviceBuffer* scratch, int64_t n);
// Adds the value rows of equal keys up in payload order and hands every sum to optimizer `opt` (or
// stores it, kOptStore) once. The pairs lie in scratch[0]; keys at or above miss_key are skipped. vals
// holds one row per payload (combined requests: gps says where they lie).
int32_t reduce_runs(const ReduceShape& sh, hipStream_t stream, DeviceBuffer* scratch, const TableView& tv, int opt,
                    int64_t n, uint32_t miss_key, const NotedRows& noted, const float* vals, const ApplyArgs& args,
                    const PooledSrc& ps, const GroupSrc* gs, const GroupPooledSrc* gps);

// Requests of at most this many ids a table need no partition: every bucket's workgroup picks its pairs out
// of the member's keys.
constexpr int64_t kPickMax = 2048;
// keys: n rows (combined requests: members' numbers above their row_bits bits, or noted rows); payloads are
// positions, or bags where bag_of says so (PooledSrc). noted: the keys are row notes (NotedRows, with
// the ids of a single table; combined requests have theirs in gps). longest: ids of the longest member.
int32_t pick_runs(const ReduceShape& sh, hipStream_t stream, const TableView& tv, int opt, const uint32_t* keys,
                  uint32_t miss_key, int row_bits, uint32_t row_mask, const uint64_t* noted_ids, bool noted, int64_t n,
                  int64_t longest, const float* vals, const ApplyArgs& args, const PooledSrc& ps, const GroupSrc* gs,
                  const GroupPooledSrc* gps);

}  // namespace krk
