// Block bucketization of a feature-major KJT into up to 64 buckets.
//
// Bucket p of the output holds, feature by feature and bag by bag, the ids with
// id / block_size == p in their input order: it is a stable partition of the
// ids by bucket.  Four launches:
//   tile_totals   ids per tile of consecutive bags of one feature
//   bucket_counts ids per (bucket, bag) = the new lengths, and per (bucket, tile)
//   bucket_scan   where each tile's ids of each bucket go; bucket totals to the host
//   bucket_move   the ids to their place
// Calls of few lengths leave the first out (every block of bucket_counts adds up
// the lengths in front of its tile), calls of few tiles the third (every block
// of bucket_move adds up the counts): two launches where the launches themselves
// are most of the call.
// Lengths that are no partition of the ids (a negative one, or more in a tile
// than there are ids) are found by the first launch; no id is moved then, and
// every total that reaches the host is -1.
// Bound by memory: ids are read twice, everything else moves once (7.9 M int64
// ids with weights in 64 x 4096 bags, 8 buckets: 270 MB).
#include <algorithm>
#include <type_traits>

#include "tra_common.h"

namespace tra {

typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kBktThreads = 256;
constexpr int kBktWaves = kBktThreads / kWaveSize;
constexpr int kBktRounds = 8;                            // ids per lane and step of bucket_move
constexpr int kBktStep = kBktThreads * kBktRounds;       // ids per step
constexpr int kBktMax = 64;                              // buckets: one per lane of a wave
constexpr int kBktMaxBags = 512;                         // bags per tile
constexpr int kBktMaxCounts = 8192;                      // (bag, bucket) counters of a tile
constexpr int kBktCountStep = 4096;                      // ids per step of bucket_counts
constexpr int kBktCountWords = kBktCountStep / kWaveSize;
static_assert(kBktCountWords == kWaveSize, "a lane holds one word of the step's bitmap");
constexpr int kBktRowPad = 4;                            // (a wave's ids belong to few bags: their buckets lie in different banks)

struct BucketArgs {
  const void* lengths;
  const void* indices;
  const float* weights;
  const int64_t* block_sizes;
  int32_t* tile_total;    // [tiles] -1: bad lengths
  int64_t* tile_first;    // [tiles] first id of the tile
  int32_t* counts;        // [W][tiles] ids of a bucket in a tile, -1: bad lengths
  int64_t* place;         // [W][tiles] the bucket's ids in front of the tile
  int64_t* bucket_total;  // [W] -1: bad lengths somewhere
  int64_t* host_totals;   // [W] pinned
  void* new_lengths;      // [W][n]
  void* new_indices;
  float* new_weights;
  int64_t* order;         // [ids] where each id went, -1: dropped
  void* bucket_of;        // [ids] floor(id / block size)
  int64_t num_indices;
  int64_t n;              // bags
  int32_t B;
  int32_t W;
  int32_t bags;           // per tile
  int32_t per_feature;    // tiles per feature
  int32_t tiles;
  int32_t bits;           // W <= 1 << bits
  int32_t keep;
};
constexpr int kBktOwnLengths = 16384;  // lengths up to which bucket_counts sums them itself
constexpr size_t kBktSpareLds = 6000;  // beside the 30 KB of bucket_move's weighted 64-bit instances: four blocks a compute unit
constexpr int kBktOwnCounts = 4096;    // tiles * buckets up to which bucket_move adds the counts itself

// q = id / bs, r = id % bs of unsigned ids for one block size.  Below 2^32:
// id * floor(2^32 / bs) / 2^32 is the quotient or one less.  (The floor by a
// division of doubles: 2^32 / bs is a whole number or 1 / bs and more away from
// one, the rounding at most 2^-21 of that.)
struct Divider {
  uint64_t bs;
  uint32_t magic;
  bool small;
  __device__ __forceinline__ explicit Divider(uint64_t b) : bs(b), small((b >> 32) == 0 && b != 0) {
    magic = small && b > 1 ? (uint32_t)(4294967296.0 / (double)(uint32_t)b) : 0xffffffffu;
  }
  // Whether all ids of the wave's lanes are below 2^32, and the block size as well: asked once for several ids, so that
  // the step of an id has no branch.
  template <typename T, int N>
  __device__ __forceinline__ bool short_ids(const T (&id)[N]) const {
    uint32_t high = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) high |= sizeof(T) == 8 ? (uint32_t)((uint64_t)id[k] >> 32) : (uint32_t)id[k] & 0x80000000u;
    return small && __builtin_amdgcn_ballot_w64(high != 0) == 0;
  }
  // SHORT: short_ids() of the id.
  template <bool SHORT>
  __device__ __forceinline__ void split(uint64_t id, uint64_t& q, uint64_t& r) const {
    if constexpr (SHORT) {
      const uint32_t a = (uint32_t)id, b = (uint32_t)bs;
      const uint32_t qq = __umulhi(a, magic), rr = a - qq * b;
      q = rr >= b ? qq + 1 : qq;
      r = rr >= b ? rr - b : rr;
    } else {
      q = id / bs;
      r = id - q * bs;
    }
  }
};

// Lane moves of the vector ALU (shifts inside rows of sixteen lanes, then lanes 15 and 31 into the rows behind them),
// as the scans need them: CTRL and the rows that receive.  Lanes without a source receive 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ int from_lanes(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, ROWS == 0xf);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ int64_t from_lanes(int64_t v) {
  const uint32_t lo = (uint32_t)from_lanes<CTRL, ROWS>((int)v), hi = (uint32_t)from_lanes<CTRL, ROWS>((int)(v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
// Inclusive scan over the lanes of a wave, all of them active.
template <typename S>
__device__ __forceinline__ S wave_scan(S v) {
  v += from_lanes<0x111, 0xf>(v);
  v += from_lanes<0x112, 0xf>(v);
  v += from_lanes<0x114, 0xf>(v);
  v += from_lanes<0x118, 0xf>(v);
  v += from_lanes<0x142, 0xa>(v);
  v += from_lanes<0x143, 0xc>(v);
  return v;
}
__device__ __forceinline__ int last_lane(int v) { return __builtin_amdgcn_readlane(v, kWaveSize - 1); }
__device__ __forceinline__ int64_t last_lane(int64_t v) {
  return (int64_t)(((uint64_t)(uint32_t)last_lane((int)(v >> 32)) << 32) | (uint32_t)last_lane((int)v));
}
template <typename S>
__device__ __forceinline__ S wave_sum(S v) {
  return last_lane(wave_scan(v));
}
// Bits of a mask below the lane's own.
__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The tile's bags: first bag and how many.
__device__ __forceinline__ int64_t tile_bags(int tile, int f, int per_feature, int bags, int B, int& cnt) {
  const int b0 = (tile - f * per_feature) * bags;
  cnt = min(bags, B - b0);
  return (int64_t)f * B + b0;
}

// One wave per tile.
template <typename T>
__global__ __launch_bounds__(kBktThreads) void tile_totals_kernel(const BucketArgs a) {
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int tile = blockIdx.x * kBktWaves + threadIdx.x / kWaveSize;
  if (tile >= a.tiles) return;
  int cnt;
  const int64_t bag = tile_bags(tile, tile / a.per_feature, a.per_feature, a.bags, a.B, cnt);
  int64_t sum = 0;
  bool bad = false;
  constexpr int U = 4;
  for (int i0 = 0; i0 < cnt; i0 += U * kWaveSize) {
    T x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = reinterpret_cast<const T*>(a.lengths)[bag + min(i0 + u * kWaveSize + lane, cnt - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t v = i0 + u * kWaveSize + lane < cnt ? (int64_t)x[u] : 0;
      bad |= v < 0 || v > a.num_indices;
      sum += v;
    }
  }
  bad = __builtin_amdgcn_ballot_w64(bad) != 0;
  sum = wave_sum(sum);
  if (lane == 0) a.tile_total[tile] = bad || sum > a.num_indices ? -1 : (int32_t)sum;
}

// One block per tile.  A tile's (bag, bucket) counters are in LDS.  The ids are
// walked in order, 64 to a wave: a bitmap in LDS marks the last id of every bag,
// so an id's bag is the number of marks in front of it (a count of the bits below
// the lane), looked up among the bags that hold ids.
//
// Bound by memory once a block's ids are under way, by the trip to its bounds in
// front of that: 7.9 M int64 ids in 64 x 4096 bags of about 30, 8 buckets, 16.4 us
// (82 MB at 5.0 TB/s).  A bag's ids walked by four lanes of their own, block sizes
// and tile totals fetched one behind the other and 64-bit sums by cross-lane reads
// took 19.7 us; of the 16.4 about 8 pass in front of the first ids.  (Counters of a
// bag's buckets in one LDS bank: 37 us.  The tiles' counts added up for bucket_move
// by atomics, 64 tiles to a sum, instead of a scan of them: 34 us, the adds to one
// line follow one another 28 ns apart.)
template <typename T, bool OWN_PREFIX>
__global__ __launch_bounds__(kBktThreads) void bucket_counts_kernel(
    const void* p_lengths, const int32_t* p_tile_total, const int64_t* p_block_sizes, int32_t p_bags,
    int32_t p_per_feature, int32_t p_B, const BucketArgs a) {
  // (sized by the launch: with room for the largest tile only four blocks fit a compute unit)
  extern __shared__ int bkt_smem[];
  const int row = p_bags + kBktRowPad;
  int* s_cnt = bkt_smem;                    // [W + 1][row], the last one for ids without a bucket
  int* s_bag = bkt_smem + (a.W + 1) * row;  // [bags + 1] the bags that hold ids
  __shared__ uint64_t s_last[kBktCountWords];  // bit j of word w: place 64 * w + j of the step is a bag's last id
  __shared__ int64_t s_sum[kBktWaves], s_own[OWN_PREFIX ? kBktWaves : 1];
  __shared__ int s_wave[kBktWaves], s_held[kBktWaves], s_bad[OWN_PREFIX ? kBktWaves : 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int tile = blockIdx.x;
  int cnt;
  const int f = tile / p_per_feature;
  const int64_t bag = tile_bags(tile, f, p_per_feature, p_bags, p_B, cnt);
  // All that the block needs before its ids is requested at once (the leading parameters come with the wave): one trip
  // to memory instead of several is what a block with nothing else to do waits for.
  const uint64_t block_size = (uint64_t)p_block_sizes[f];
  // the bags' ends: two bags per thread
  const T* lengths = reinterpret_cast<const T*>(p_lengths) + bag;
  const int i0 = 2 * threadIdx.x;
  T g0 = lengths[min(i0, cnt - 1)], g1 = lengths[min(i0 + 1, cnt - 1)];
  // ids in front of the tile: 16 bytes per load
  int64_t before = 0;
  int given_total = 0;
  if constexpr (OWN_PREFIX) {
    constexpr int V = 16 / (int)sizeof(T);
    struct __align__(16) Vec { T v[V]; };
    const Vec* v = reinterpret_cast<const Vec*>(p_lengths);
    const int nv = (int)(bag / V);
    for (int u0 = threadIdx.x; u0 < nv; u0 += 4 * kBktThreads) {
      Vec x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = v[min(u0 + k * kBktThreads, nv - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        int64_t sum = 0;
#pragma unroll
        for (int i = 0; i < V; ++i) sum += (int64_t)x[k].v[i];
        before += u0 + k * kBktThreads < nv ? sum : 0;
      }
    }
    if (V * nv + (int64_t)threadIdx.x < bag) before += (int64_t) reinterpret_cast<const T*>(p_lengths)[V * nv + threadIdx.x];
  } else {
    given_total = p_tile_total[tile];
    const i32x4_t* v = reinterpret_cast<const i32x4_t*>(p_tile_total);
    const int nv = tile / 4;
    const int rest = p_tile_total[min(4 * nv + (int)threadIdx.x, tile)];
    const auto add = [&](auto loads, int u0) {
      constexpr int N = decltype(loads)::value;
      i32x4_t x[N];
#pragma unroll
      for (int k = 0; k < N; ++k) x[k] = v[min(u0 + k * kBktThreads, max(nv - 1, 0))];
#pragma unroll
      for (int k = 0; k < N; ++k)
        before += u0 + k * kBktThreads < nv ? (int64_t)x[k].x + x[k].y + x[k].z + x[k].w : 0;
    };
    if (nv <= 2 * kBktThreads)
      add(std::integral_constant<int, 2>(), (int)threadIdx.x);
    else
      for (int u0 = 0; u0 < nv; u0 += 4 * kBktThreads) add(std::integral_constant<int, 4>(), u0 + (int)threadIdx.x);
    before += 4 * nv + (int)threadIdx.x < tile ? rest : 0;
  }
  g0 = i0 < cnt ? g0 : (T)0;
  g1 = i0 + 1 < cnt ? g1 : (T)0;
  const int l0 = (int)g0, l1 = (int)g1;
  asm volatile("" ::"s"(block_size), "s"(given_total), "s"(a.indices), "s"(a.num_indices), "s"(a.W));
  for (int x = threadIdx.x; x < row * a.W; x += kBktThreads) s_cnt[x] = 0;
  for (int x = threadIdx.x; x < kBktCountWords; x += kBktThreads) s_last[x] = 0;
  const int incl = wave_scan(l0 + l1);
  const uint64_t held0 = __builtin_amdgcn_ballot_w64(l0 > 0), held1 = __builtin_amdgcn_ballot_w64(l1 > 0);
  before = wave_sum(before);
  if constexpr (OWN_PREFIX) {
    const bool odd = g0 < 0 || (int64_t)g0 > a.num_indices || g1 < 0 || (int64_t)g1 > a.num_indices;
    const int64_t own = wave_sum((int64_t)g0 + (int64_t)g1);
    const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
    if (lane == 0) {
      s_own[wave] = own;
      s_bad[wave] = any;
    }
  }
  if (lane == kWaveSize - 1) s_wave[wave] = incl;
  if (lane == 0) {
    s_sum[wave] = before;
    s_held[wave] = __builtin_popcountll(held0) + __builtin_popcountll(held1);
  }
  lds_barrier();
  int front = 0, total = 0, held_front = 0, held = 0;
  int64_t own = 0;
  bool odd = false;
  before = 0;
#pragma unroll
  for (int w = 0; w < kBktWaves; ++w) {
    front += w < wave ? s_wave[w] : 0;
    total += s_wave[w];
    held_front += w < wave ? s_held[w] : 0;
    held += s_held[w];
    before += s_sum[w];
    if constexpr (OWN_PREFIX) {
      own += s_own[w];
      odd = odd || s_bad[w] != 0;
    }
  }
  const int tile_total = OWN_PREFIX && (odd || own > a.num_indices) ? -1 : (int)own;
  const int end1 = front + incl, end0 = end1 - l1;
  {
    int at = held_front + lanes_below(held0) + lanes_below(held1);
    if (l0 > 0) s_bag[at++] = i0;
    if (l1 > 0) s_bag[at] = i0 + 1;
  }
  if (threadIdx.x == 0) {
    s_bag[held] = 0;  // (what places behind the last id look up)
    a.tile_first[tile] = before;
    if constexpr (OWN_PREFIX) a.tile_total[tile] = tile_total;
  }
  // (never outside the ids array, whatever the lengths say; the bags' ends are no places where the lengths are bad)
  const bool bad = (OWN_PREFIX ? tile_total : given_total) < 0;
  const int ids = __builtin_amdgcn_readfirstlane(
      bad || before < 0 ? 0 : (int)max(min((int64_t)total, a.num_indices - before), (int64_t)0));
  const T* in = reinterpret_cast<const T*>(a.indices) + before;
  const Divider div(block_size);
  int held_before = 0;  // bags whose last id lies in front of the step
  constexpr int U = 8;
  T id[U];
  const auto load = [&](int at) {
#pragma unroll
    for (int u = 0; u < U; ++u) id[u] = in[min(at + u * kBktThreads + lane, ids - 1)];
  };
  for (int j0 = 0; j0 < ids; j0 += kBktCountStep) {
    const int words = (min(ids - j0, kBktCountStep) + kWaveSize - 1) / kWaveSize;
    load(j0 + wave * kWaveSize);  // (words are dealt to the waves, so that a short tile keeps all busy)
    const auto mark = [&](int len, int end) {
      const uint32_t at = (uint32_t)(end - 1 - j0);
      if (len > 0 && at < (uint32_t)kBktCountStep)
        atomicOr(reinterpret_cast<uint32_t*>(s_last) + at / 32, 1u << (at % 32));
    };
    mark(l0, end0);
    mark(l1, end1);
    lds_barrier();
    // Lane w holds word w, and how many bags end in front of it.
    const uint64_t last = s_last[lane];
    const int ends = __builtin_popcountll(last);
    const int ends_incl = wave_scan(ends);
    const int ends_front = held_before + ends_incl - ends;
    held_before += last_lane(ends_incl);
    for (int w0 = wave; w0 < words; w0 += U * kBktWaves) {
      const auto count = [&](auto is_short) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int w = w0 + u * kBktWaves;
          if (w >= words) break;
          uint64_t q, r;
          div.split<decltype(is_short)::value>((uint64_t)(int64_t)id[u], q, r);
          const bool counts = j0 + w * kWaveSize + lane < ids && q < (uint64_t)a.W;
          const int bag_at = __builtin_amdgcn_mbcnt_hi(
              (uint32_t)__builtin_amdgcn_readlane((int)(last >> 32), w),
              __builtin_amdgcn_mbcnt_lo((uint32_t)__builtin_amdgcn_readlane((int)last, w),
                                        (uint32_t)__builtin_amdgcn_readlane(ends_front, w)));
          atomicAdd(&s_cnt[__umul24(counts ? (int)q : a.W, row) + s_bag[bag_at]], 1);
        }
      };
      if (div.short_ids(id)) count(std::true_type()); else count(std::false_type());
      if (w0 + U * kBktWaves < words) load(j0 + (w0 + U * kBktWaves) * kWaveSize);
    }
    lds_barrier();
    if (j0 + kBktCountStep < ids) {
      for (int x = threadIdx.x; x < kBktCountWords; x += kBktThreads) s_last[x] = 0;
      lds_barrier();
    }
  }
  // new lengths, and the tile's total per bucket: a wave takes every fourth bucket
  T* out = reinterpret_cast<T*>(a.new_lengths);
  for (int p = wave; p < a.W; p += kBktWaves) {
    int sum = 0;
    for (int i = lane; i < cnt; i += kWaveSize) {
      const int c = s_cnt[p * row + i];
      out[(int64_t)p * a.n + bag + i] = (T)c;
      sum += c;
    }
    sum = wave_sum(sum);
    if (lane == 0) a.counts[(int64_t)p * a.tiles + tile] = bad ? -1 : sum;
  }
}

// One block per bucket: exclusive scan over the tiles.
constexpr int kBktScanThreads = 1024;
__global__ __launch_bounds__(kBktScanThreads) void bucket_scan_kernel(const BucketArgs a) {
  __shared__ int64_t s_wave[kBktScanThreads / kWaveSize];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int32_t* in = a.counts + (int64_t)blockIdx.x * a.tiles;
  int64_t* out = a.place + (int64_t)blockIdx.x * a.tiles;
  int64_t carry = 0;
  int bad = 0;
  constexpr int U = 4;  // consecutive tiles per thread
  for (int t0 = 0; t0 < a.tiles; t0 += U * kBktScanThreads) {
    const int t = t0 + U * (int)threadIdx.x;
    int64_t x[U], mine = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = t + u < a.tiles ? in[t + u] : 0;
      bad |= x[u] < 0;
      mine += x[u];
    }
    const int64_t incl = wave_scan(mine);
    if (lane == kWaveSize - 1) s_wave[wave] = incl;
    __syncthreads();
    int64_t front = carry, all = 0;
    for (int w = 0; w < kBktScanThreads / kWaveSize; ++w) {
      front += w < wave ? s_wave[w] : 0;
      all += s_wave[w];
    }
    int64_t run = front + incl - mine;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (t + u < a.tiles) out[t + u] = run;
      run += x[u];
    }
    carry += all;
    __syncthreads();
  }
  if (__syncthreads_or(bad)) carry = -1;
  if (threadIdx.x == 0) {
    a.bucket_total[blockIdx.x] = carry;
    // (left to the move, this launch ends 0.7 us sooner, but the host waits longer: 2 x 16384 bags of 3 ids 53.6 us a call
    // instead of 49.6)
    publish_total(carry, a.host_totals + blockIdx.x);
  }
}

// One block per tile.  A step takes kBktStep ids; wave w holds a run of
// consecutive ones, kBktRounds per lane.  An id's rank among the wave's ids of
// its bucket comes from the lanes that hold the same bucket (one ballot per bit
// of the bucket number); with the counts of the waves in front that is its
// place in the step, where the ids are brought together in LDS, so that they
// leave in runs of a bucket instead of one by one: 34.4 us for the ids and weights
// above, 188 MB at the rate of a copy (38.4 us with the block's bounds fetched one
// behind the other and five full barriers a step; 84 us when every wave stored its
// ids one by one behind cursors per bucket and bag).  Measured and left out: the
// next step's ids requested a step ahead (104 registers, four waves per SIMD
// instead of five: 36.8 us), steps of 1024 ids 36.8 us, loads or stores with the
// non-temporal hint 41 us.
template <typename T, bool WEIGHTED, bool OWN_SCAN>
__global__ __launch_bounds__(kBktThreads) void bucket_move_kernel(
    const int64_t* p_tile_first, const int32_t* p_tile_total, const int64_t* p_block_sizes, const int64_t* p_place,
    const int64_t* p_bucket_total, int32_t p_per_feature, int32_t p_tiles, const BucketArgs a) {
  __shared__ T s_val[kBktStep];
  __shared__ float s_w[WEIGHTED ? kBktStep : 1];
  __shared__ uint8_t s_bucket[kBktStep];
  __shared__ int s_cnt[kBktWaves][kBktMax];   // ids of a bucket in the wave's run
  __shared__ int s_from[kBktWaves][kBktMax];  // place in the step of the wave's first id of a bucket
  __shared__ int64_t s_to[kBktMax];           // what a bucket's places in the step lack to output positions
  __shared__ int s_moved;
  __shared__ int64_t s_all[OWN_SCAN ? kBktMax : 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int tile = blockIdx.x;
  // All that the block needs before its ids, requested at once (the leading parameters come with the wave).
  const int64_t first = p_tile_first[tile];
  const int tile_total = p_tile_total[tile];
  const uint64_t block_size = (uint64_t)p_block_sizes[tile / p_per_feature];
  int64_t place = 0, bucket_total = 0;
  if constexpr (!OWN_SCAN) {
    const int p = min(lane, a.W - 1);
    place = p_place[(int64_t)p * p_tiles + tile];
    bucket_total = p_bucket_total[p];  // (bad lengths: all are -1 or none, the last lane's too)
  }
  asm volatile("" ::"s"(first), "s"(tile_total), "s"(block_size), "v"(place), "v"(bucket_total));
  if constexpr (OWN_SCAN) {
    // The buckets' totals, and their ids in the tiles in front of this one: a wave takes every fourth bucket.
    int bad = 0;
    for (int p = wave; p < a.W; p += kBktWaves) {
      int64_t in_front = 0, all = 0;
      for (int t = lane; t < a.tiles; t += kWaveSize) {
        const int c = a.counts[(int64_t)p * a.tiles + t];
        bad |= c < 0;
        all += c;
        in_front += t < tile ? c : 0;
      }
      all = wave_sum(all);
      in_front = wave_sum(in_front);
      if (lane == 0) {
        s_all[p] = all;
        s_to[p] = in_front;
      }
    }
    bad = __syncthreads_or(bad);
    bucket_total = bad ? -1 : s_all[min(lane, a.W - 1)];
    if (tile == 0 && (int)threadIdx.x < a.W) publish_total(bucket_total, a.host_totals + threadIdx.x);
  }
  if (last_lane(bucket_total) < 0) return;  // (bad lengths)
  const int ids = first < 0 ? 0 : (int)max(min((int64_t)tile_total, a.num_indices - first), (int64_t)0);
  if (ids == 0) return;
  const Divider div(block_size);
  int64_t next = 0;  // the first wave's lane p: output position of bucket p's next id
  if (wave == 0) {
    // buckets in front of this one, and its ids in the tiles in front
    const int64_t total = lane >= a.W ? 0 : bucket_total;
    next = wave_scan(total) - total + (lane >= a.W ? 0 : OWN_SCAN ? s_to[lane] : place);
  }
  const T* in = reinterpret_cast<const T*>(a.indices) + first;
  const float* win = a.weights + first;
  for (int j00 = 0; j00 < ids; j00 += kBktStep) {
    const int j0 = j00 + wave * (kBktRounds * kWaveSize) + lane;
    T id[kBktRounds];
    float w[kBktRounds];
#pragma unroll
    for (int k = 0; k < kBktRounds; ++k) id[k] = in[min(j0 + k * kWaveSize, ids - 1)];
    if constexpr (WEIGHTED) {
#pragma unroll
      for (int k = 0; k < kBktRounds; ++k) w[k] = win[min(j0 + k * kWaveSize, ids - 1)];
    }
    s_cnt[wave][lane] = 0;
    int bucket[kBktRounds], rank[kBktRounds];
    T val[kBktRounds];
    const auto place = [&](auto is_short) {
#pragma unroll
      for (int k = 0; k < kBktRounds; ++k) {
        const int j = j0 + k * kWaveSize;
        uint64_t q, r;
        div.split<decltype(is_short)::value>((uint64_t)(int64_t)id[k], q, r);
        const bool in_bucket = j < ids && q < (uint64_t)a.W;
        const int p = in_bucket ? (int)q : 0;
        val[k] = a.keep ? id[k] : (T)r;
        if (a.bucket_of != nullptr && j < ids) {
          const int64_t s = (int64_t)id[k];  // (a negative id lies below bucket 0)
          reinterpret_cast<T*>(a.bucket_of)[first + j] =
              decltype(is_short)::value || s >= 0 ? (T)q : (T)(-(int64_t)((uint64_t)(-(s + 1)) / div.bs) - 1);
        }
        uint64_t same = __builtin_amdgcn_ballot_w64(in_bucket);
        for (int bit = 0; bit < a.bits; ++bit) {
          const uint64_t set = __builtin_amdgcn_ballot_w64((p >> bit) & 1);
          same &= ((p >> bit) & 1) ? set : ~set;
        }
        const int in_front = lanes_below(same);
        const int count = __builtin_popcountll(same);
        const int base = s_cnt[wave][p];
        bucket[k] = in_bucket ? p : -1;
        rank[k] = base + in_front;
        // (program order inside the wave: every lane has read the count)
        __builtin_amdgcn_wave_barrier();
        if (in_bucket && in_front == count - 1) s_cnt[wave][p] = base + count;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
      }
    };
    if (div.short_ids(id)) place(std::true_type()); else place(std::false_type());
    lds_barrier();
    if (wave == 0) {
      int per[kBktWaves], sum = 0;
#pragma unroll
      for (int v = 0; v < kBktWaves; ++v) {
        per[v] = s_cnt[v][lane];
        sum += per[v];
      }
      const int incl = wave_scan(sum);
      int run = incl - sum;
      s_to[lane] = next - run;
      next += sum;
      if (lane == kWaveSize - 1) s_moved = incl;
#pragma unroll
      for (int v = 0; v < kBktWaves; ++v) {
        s_from[v][lane] = run;
        run += per[v];
      }
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < kBktRounds; ++k) {
      const int j = j0 + k * kWaveSize;
      int64_t to = -1;
      if (bucket[k] >= 0) {
        const int at = s_from[wave][bucket[k]] + rank[k];
        s_val[at] = val[k];
        if constexpr (WEIGHTED) s_w[at] = w[k];
        s_bucket[at] = (uint8_t)bucket[k];
        to = s_to[bucket[k]] + at;
      }
      if (a.order != nullptr && j < ids) a.order[first + j] = to;
    }
    lds_barrier();
    const int moved = s_moved;  // ids of the step that have a bucket
    for (int i = threadIdx.x; i < moved; i += kBktThreads) {
      const int64_t to = s_to[s_bucket[i]] + i;
      reinterpret_cast<T*>(a.new_indices)[to] = s_val[i];
      if constexpr (WEIGHTED) a.new_weights[to] = s_w[i];
    }
    // (the next step writes what has been read here only behind its first barrier)
  }
}

// Bags per tile: an average of 4096 ids (two steps of bucket_move) where that
// leaves 1536 tiles, six for each of an MI355X's 256 compute units (7.9 M ids in
// 64 x 4096 bags, the four kernels together, best passes, when they took 64 us
// with 4096 ids a tile: 2048 74 us, 1024 99 us, 8192 71 us; a fixed figure, so that the workspace
// does not depend on the device that asks for its size), down to 256
// ids; more where that makes over 8192 tiles (every block of bucket_counts adds
// up the totals of the tiles in front of its own); no more than the counters hold.
static int bags_per_tile(int64_t n, int64_t num_indices, int32_t B, int32_t W) {
  const int64_t ids = std::max<int64_t>(256, std::min<int64_t>(2 * kBktStep, num_indices / 1536));
  int bags = 1;
  while (bags < kBktMaxBags && bags < B && 2 * bags * W <= kBktMaxCounts &&
         (2 * (int64_t)bags * num_indices <= ids * n || n / bags > 8192))
    bags *= 2;
  return bags;
}

struct BucketSizes {
  int bags, per_feature;
  int64_t tiles, first, counts, place, total, bytes;  // byte offsets in the workspace
};
static BucketSizes bucket_sizes(int32_t F, int32_t B, int32_t W, int64_t num_indices) {
  BucketSizes z;
  const int64_t n = (int64_t)F * B;
  z.bags = bags_per_tile(n, num_indices, B, W);
  z.per_feature = (B + z.bags - 1) / z.bags;
  z.tiles = (int64_t)F * z.per_feature;
  const auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  z.first = up(z.tiles * 4);
  z.counts = z.first + up(z.tiles * 8);
  z.place = z.counts + up(z.tiles * W * 4);
  z.total = z.place + up(z.tiles * W * 8);
  z.bytes = z.total + W * 8;
  return z;
}

}  // namespace tra

using namespace tra;

extern "C" {

int64_t tra_bucketize_ids_workspace_bytes(int32_t num_features, int32_t batch_size, int32_t num_buckets,
                                          int64_t num_indices) {
  if (num_features < 1 || batch_size < 1 || num_buckets < 1 || num_buckets > kBktMax || num_indices < 0) return 0;
  return bucket_sizes(num_features, batch_size, num_buckets, num_indices).bytes;
}

int tra_bucketize_ids(const void* lengths, const void* indices, int32_t is_i64, const float* weights,
                      const int64_t* block_sizes, int32_t num_features, int32_t batch_size, int32_t num_buckets,
                      int64_t num_indices, int32_t keep_orig_idx, void* workspace, void* new_lengths,
                      void* new_indices, float* new_weights, int64_t* unbucketize_permute, void* bucket_of,
                      int32_t* ticket, void* stream) {
  if (num_features < 1 || batch_size < 1 || num_buckets < 1 || num_indices < 0 || !lengths || !block_sizes ||
      !workspace || !new_lengths || !ticket || (num_indices > 0 && (!indices || !new_indices)) ||
      (weights && !new_weights && num_indices > 0)) {
    set_error("tra_bucketize_ids: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const BucketSizes z = bucket_sizes(num_features, batch_size, std::min(num_buckets, (int32_t)kBktMax), num_indices);
  // (the kernels count a tile's ids in 32 bits and look up to a step behind its last one)
  if (num_buckets > kBktMax || z.tiles > 0x7fffffff || num_indices > 0x7fffffff - 2 * kBktStep) {
    set_error("tra_bucketize_ids: %d buckets (at most %d), %lld ids", num_buckets, kBktMax, (long long)num_indices);
    return TRA_ERR_TOO_LARGE;
  }
  hipStream_t s = (hipStream_t)stream;
  BucketArgs a = BucketArgs();
  a.lengths = lengths;
  a.indices = indices;
  a.weights = weights;
  a.block_sizes = block_sizes;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  a.tile_total = reinterpret_cast<int32_t*>(ws);
  a.tile_first = reinterpret_cast<int64_t*>(ws + z.first);
  a.counts = reinterpret_cast<int32_t*>(ws + z.counts);
  a.place = reinterpret_cast<int64_t*>(ws + z.place);
  a.bucket_total = reinterpret_cast<int64_t*>(ws + z.total);
  a.new_lengths = new_lengths;
  a.new_indices = new_indices;
  a.new_weights = new_weights;
  a.order = unbucketize_permute;
  a.bucket_of = bucket_of;
  a.num_indices = num_indices;
  a.n = (int64_t)num_features * batch_size;
  a.B = batch_size;
  a.W = num_buckets;
  a.bags = z.bags;
  a.per_feature = z.per_feature;
  a.tiles = (int32_t)z.tiles;
  a.keep = keep_orig_idx;
  while ((1 << a.bits) < num_buckets) ++a.bits;
  // (calls, us, four launches / two: 5 keys x 133 bags, 1.3 K ids, 2 buckets 46 / 38; 52 x 29, 44 K ids, 3 buckets 61 / 52)
  // (instances of their own: the branches alone cost the large calls 3 %)
  const bool own_prefix = a.n <= kBktOwnLengths && (uintptr_t)lengths % 16 == 0;
  const bool own_scan = num_indices > 0 && z.tiles * num_buckets <= kBktOwnCounts;
  const int rc = mail_open(s, num_buckets, ticket, &a.host_totals);
  if (rc != TRA_OK) return rc;
  const dim3 block(kBktThreads), tiles((unsigned)z.tiles), waves((unsigned)((z.tiles + kBktWaves - 1) / kBktWaves));
  const size_t counters = ((size_t)(z.bags + kBktRowPad) * (num_buckets + 1) + z.bags + 1) * sizeof(int);
  const auto counts = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, tiles, block, counters, s, a.lengths, a.tile_total, a.block_sizes, a.bags, a.per_feature,
                       a.B, a);
  };
  // Weighted 64-bit ids whose places are wanted too, more bytes than the 256 MB of the memory-side cache: four blocks on a
  // compute unit instead of the five that registers allow (us a call, five / four: 7.9 M ids, 2 buckets 104.5 / 101.0, 8
  // buckets 91.1 / 88.4; but 5.2 M ids, 210 MB 73.5 / 75.3, and without places 74.3 / 75.6).
  const int64_t moved = num_indices * (2 * (8 + 4) + 8 + (bucket_of != nullptr ? 8 : 0));
  const size_t spare = is_i64 && weights && unbucketize_permute && moved > (int64_t(1) << 28) ? kBktSpareLds : 0;
  const auto move = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, tiles, block, spare, s, a.tile_first, a.tile_total, a.block_sizes, a.place, a.bucket_total,
                       a.per_feature, a.tiles, a);
  };
  const auto launch = [&](auto id) {
    using T = decltype(id);
    if (own_prefix) {
      counts(bucket_counts_kernel<T, true>);
    } else {
      hipLaunchKernelGGL(tile_totals_kernel<T>, waves, block, 0, s, a);
      counts(bucket_counts_kernel<T, false>);
    }
    if (!own_scan) hipLaunchKernelGGL(bucket_scan_kernel, dim3(num_buckets), dim3(kBktScanThreads), 0, s, a);
    if (num_indices == 0) return;
    if (weights && own_scan)
      move(bucket_move_kernel<T, true, true>);
    else if (weights)
      move(bucket_move_kernel<T, true, false>);
    else if (own_scan)
      move(bucket_move_kernel<T, false, true>);
    else
      move(bucket_move_kernel<T, false, false>);
  };
  if (is_i64) launch(int64_t()); else launch(int32_t());
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    // (the scan may have been queued: its slot is not given back)
    *ticket = -1;
    return hip_fail(e, "tra_bucketize_ids");
  }
  return TRA_OK;
}

}  // extern "C"
