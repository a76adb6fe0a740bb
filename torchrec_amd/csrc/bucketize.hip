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
  int32_t lanes;          // bucket_counts: lanes per bag (a power of two)
  int32_t keep;
};
constexpr int kBktOwnLengths = 16384;  // lengths up to which bucket_counts sums them itself
constexpr int kBktOwnCounts = 4096;    // tiles * buckets up to which bucket_move adds the counts itself

// q = id / bs, r = id % bs of unsigned ids for one block size.  Below 2^32:
// id * floor(2^32 / bs) / 2^32 is the quotient or one less.
struct Divider {
  uint64_t bs;
  uint32_t magic;
  bool small;
  __device__ __forceinline__ explicit Divider(uint64_t b) : bs(b), small((b >> 32) == 0 && b != 0) {
    magic = small && b > 1 ? (uint32_t)((1ull << 32) / b) : 0xffffffffu;
  }
  __device__ __forceinline__ void operator()(uint64_t id, uint64_t& q, uint64_t& r) const {
    if (small && (id >> 32) == 0) {
      const uint32_t a = (uint32_t)id, b = (uint32_t)bs;
      uint32_t qq = __umulhi(a, magic);
      uint32_t rr = a - qq * b;
      if (rr >= b) {
        ++qq;
        rr -= b;
      }
      q = qq;
      r = rr;
    } else {
      q = id / bs;
      r = id - q * bs;
    }
  }
};

__device__ __forceinline__ int wave_scan32(int v, int lane) {
#pragma unroll
  for (int off = 1; off < kWaveSize; off <<= 1) {
    const int o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
}
__device__ __forceinline__ int64_t wave_sum64(int64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The tile's bags: first bag and how many.
__device__ __forceinline__ int64_t tile_bags(const BucketArgs& a, int tile, int& cnt) {
  const int f = tile / a.per_feature;
  const int b0 = (tile - f * a.per_feature) * a.bags;
  cnt = min(a.bags, a.B - b0);
  return (int64_t)f * a.B + b0;
}

// One wave per tile.
template <typename T>
__global__ __launch_bounds__(kBktThreads) void tile_totals_kernel(const BucketArgs a) {
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int tile = blockIdx.x * kBktWaves + threadIdx.x / kWaveSize;
  if (tile >= a.tiles) return;
  int cnt;
  const int64_t bag = tile_bags(a, tile, cnt);
  int64_t sum = 0;
  bool bad = false;
  for (int i = lane; i < cnt; i += kWaveSize) {
    const int64_t x = (int64_t) reinterpret_cast<const T*>(a.lengths)[bag + i];
    bad |= x < 0 || x > a.num_indices;
    sum += x;
  }
  bad = __builtin_amdgcn_ballot_w64(bad) != 0;
  sum = wave_sum64(sum);
  if (lane == 0) a.tile_total[tile] = bad || sum > a.num_indices ? -1 : (int32_t)sum;
}

// One block per tile.  A tile's (bag, bucket) counters are in LDS; a bag's ids are
// walked by a.lanes lanes, four ids per lane in flight.  (Walking the tile's ids
// in order and looking each id's bag up in LDS took 48 us where this takes
// 19 us: 7.9 M ids in 64 x 4096 bags.)
template <typename T, bool OWN_PREFIX>
__global__ __launch_bounds__(kBktThreads) void bucket_counts_kernel(const BucketArgs a) {
  // (sized by the launch: with room for the largest tile only four blocks fit a compute unit)
  extern __shared__ int bkt_smem[];
  int* s_end = bkt_smem;           // [bags] ids up to and including the bag
  int* s_cnt = bkt_smem + a.bags;  // [W][bags]
  __shared__ int64_t s_sum[kBktWaves], s_own[OWN_PREFIX ? kBktWaves : 1];
  __shared__ int s_wave[kBktWaves], s_bad[OWN_PREFIX ? kBktWaves : 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int tile = blockIdx.x;
  int cnt;
  const int64_t bag = tile_bags(a, tile, cnt);
  // the bags' ends: two bags per thread
  const T* lengths = reinterpret_cast<const T*>(a.lengths) + bag;
  const int i0 = 2 * threadIdx.x;
  const T g0 = i0 < cnt ? lengths[i0] : (T)0, g1 = i0 + 1 < cnt ? lengths[i0 + 1] : (T)0;
  const int l0 = (int)g0, l1 = (int)g1;
  // ids in front of the tile: 16 bytes per load, four loads in flight
  int64_t before = 0;
  if constexpr (OWN_PREFIX) {
    constexpr int V = 16 / (int)sizeof(T);
    struct __align__(16) Vec { T v[V]; };
    const Vec* v = reinterpret_cast<const Vec*>(a.lengths);
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
    if (V * nv + (int64_t)threadIdx.x < bag) before += (int64_t) reinterpret_cast<const T*>(a.lengths)[V * nv + threadIdx.x];
  } else {
    const i32x4_t* v = reinterpret_cast<const i32x4_t*>(a.tile_total);
    const int nv = tile / 4;
    for (int u0 = threadIdx.x; u0 < nv; u0 += 4 * kBktThreads) {
      i32x4_t x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = v[min(u0 + k * kBktThreads, nv - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        before += u0 + k * kBktThreads < nv ? (int64_t)x[k].x + x[k].y + x[k].z + x[k].w : 0;
    }
    if (4 * nv + (int)threadIdx.x < tile) before += a.tile_total[4 * nv + threadIdx.x];
  }
  for (int x = threadIdx.x; x < a.bags * a.W; x += kBktThreads) s_cnt[x] = 0;
  const int incl = wave_scan32(l0 + l1, lane);
  before = wave_sum64(before);
  if constexpr (OWN_PREFIX) {
    const bool odd = g0 < 0 || (int64_t)g0 > a.num_indices || g1 < 0 || (int64_t)g1 > a.num_indices;
    const int64_t own = wave_sum64((int64_t)g0 + (int64_t)g1);
    const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
    if (lane == 0) {
      s_own[wave] = own;
      s_bad[wave] = any;
    }
  }
  if (lane == kWaveSize - 1) s_wave[wave] = incl;
  if (lane == 0) s_sum[wave] = before;
  __syncthreads();
  int front = 0, total = 0;
  int64_t own = 0;
  bool odd = false;
  before = 0;
#pragma unroll
  for (int w = 0; w < kBktWaves; ++w) {
    front += w < wave ? s_wave[w] : 0;
    total += s_wave[w];
    before += s_sum[w];
    if constexpr (OWN_PREFIX) {
      own += s_own[w];
      odd = odd || s_bad[w] != 0;
    }
  }
  const int tile_total = OWN_PREFIX && (odd || own > a.num_indices) ? -1 : (int)own;
  if (i0 < cnt) s_end[i0] = front + incl - l1;
  if (i0 + 1 < cnt) s_end[i0 + 1] = front + incl;
  if (threadIdx.x == 0) {
    a.tile_first[tile] = before;
    if constexpr (OWN_PREFIX) a.tile_total[tile] = tile_total;
  }
  __syncthreads();
  // (never outside the ids array, whatever the lengths say; the bags' ends are no places where the lengths are bad)
  const bool bad = (OWN_PREFIX ? tile_total : a.tile_total[tile]) < 0;
  const int ids = before < 0 ? 0 : (int)max(min((int64_t)total, a.num_indices - before), (int64_t)0);
  const T* in = reinterpret_cast<const T*>(a.indices) + before;
  const Divider div((uint64_t)a.block_sizes[tile / a.per_feature]);
  const int sub = threadIdx.x & (a.lanes - 1);
  constexpr int U = 4;
  for (int b = threadIdx.x / a.lanes; !bad && b < cnt; b += kBktThreads / a.lanes) {
    const int end = min(s_end[b], ids);
    for (int j0 = max(b > 0 ? s_end[b - 1] : 0, 0) + sub; j0 < end; j0 += U * a.lanes) {
      T id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) id[u] = in[min(j0 + u * a.lanes, end - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint64_t q, r;
        div((uint64_t)(int64_t)id[u], q, r);
        if (j0 + u * a.lanes < end && q < (uint64_t)a.W) atomicAdd(&s_cnt[(int)q * a.bags + b], 1);
      }
    }
  }
  __syncthreads();
  // new lengths, and the tile's total per bucket: a wave takes every fourth bucket
  T* out = reinterpret_cast<T*>(a.new_lengths);
  for (int p = wave; p < a.W; p += kBktWaves) {
    int sum = 0;
    for (int i = lane; i < cnt; i += kWaveSize) {
      const int c = s_cnt[p * a.bags + i];
      out[(int64_t)p * a.n + bag + i] = (T)c;
      sum += c;
    }
    sum = (int)wave_sum64(sum);
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
    int64_t incl = mine;
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
      const int64_t o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
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
    publish_total(carry, a.host_totals + blockIdx.x);
  }
}

// One block per tile.  A step takes kBktStep ids; wave w holds a run of
// consecutive ones, kBktRounds per lane.  An id's rank among the wave's ids of
// its bucket comes from the lanes that hold the same bucket (one ballot per bit
// of the bucket number); with the counts of the waves in front that is its
// place in the step, where the ids are brought together in LDS, so that they
// leave in runs of a bucket instead of one by one: 38 us for the ids and weights
// above, 188 MB at the rate of a copy (84 us when every wave stored its ids one
// by one behind cursors per bucket and bag).
template <typename T, bool WEIGHTED, bool OWN_SCAN>
__global__ __launch_bounds__(kBktThreads) void bucket_move_kernel(const BucketArgs a) {
  __shared__ T s_val[kBktStep];
  __shared__ float s_w[WEIGHTED ? kBktStep : 1];
  __shared__ uint8_t s_bucket[kBktStep];
  __shared__ int s_cnt[kBktWaves][kBktMax];   // ids of a bucket in the wave's run
  __shared__ int s_from[kBktWaves][kBktMax];  // place in the step of the wave's first id of a bucket
  __shared__ int s_start[kBktMax];            // place in the step of a bucket's first id
  __shared__ int64_t s_to[kBktMax];           // output position of the bucket's next id
  __shared__ int64_t s_all[OWN_SCAN ? kBktMax : 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int tile = blockIdx.x;
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
      all = wave_sum64(all);
      in_front = wave_sum64(in_front);
      if (lane == 0) {
        s_all[p] = all;
        s_to[p] = in_front;
      }
    }
    bad = __syncthreads_or(bad);
    if (tile == 0 && (int)threadIdx.x < a.W) publish_total(bad ? -1 : s_all[threadIdx.x], a.host_totals + threadIdx.x);
    if (bad) return;  // (bad lengths)
  } else {
    if (a.bucket_total[0] < 0) return;  // (bad lengths)
  }
  const int64_t first = a.tile_first[tile];
  const int ids = first < 0 ? 0 : (int)max(min((int64_t)a.tile_total[tile], a.num_indices - first), (int64_t)0);
  if (ids == 0) return;
  const Divider div((uint64_t)a.block_sizes[tile / a.per_feature]);
  if (wave == 0) {
    // buckets in front of this one, and its ids in the tiles in front
    const int64_t total = lane >= a.W ? 0 : OWN_SCAN ? s_all[lane] : a.bucket_total[lane];
    int64_t incl = total;
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
      const int64_t o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    if (lane < a.W) s_to[lane] = incl - total + (OWN_SCAN ? s_to[lane] : a.place[(int64_t)lane * a.tiles + tile]);
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
    if (lane < a.W) s_cnt[wave][lane] = 0;
    int bucket[kBktRounds], rank[kBktRounds];
    T val[kBktRounds];
#pragma unroll
    for (int k = 0; k < kBktRounds; ++k) {
      const int j = j0 + k * kWaveSize;
      uint64_t q, r;
      div((uint64_t)(int64_t)id[k], q, r);
      const bool in_bucket = j < ids && q < (uint64_t)a.W;
      const int p = in_bucket ? (int)q : 0;
      val[k] = a.keep ? id[k] : (T)r;
      if (a.bucket_of != nullptr && j < ids) {
        const int64_t s = (int64_t)id[k];  // (a negative id lies below bucket 0)
        reinterpret_cast<T*>(a.bucket_of)[first + j] =
            s >= 0 ? (T)q : (T)(-(int64_t)((uint64_t)(-(s + 1)) / div.bs) - 1);
      }
      uint64_t same = __builtin_amdgcn_ballot_w64(in_bucket);
      for (int bit = 0; bit < a.bits; ++bit) {
        const uint64_t set = __builtin_amdgcn_ballot_w64((p >> bit) & 1);
        same &= ((p >> bit) & 1) ? set : ~set;
      }
      const int in_front = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
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
    __syncthreads();
    if (wave == 0) {
      int per[kBktWaves], sum = 0;
#pragma unroll
      for (int v = 0; v < kBktWaves; ++v) {
        per[v] = lane < a.W ? s_cnt[v][lane] : 0;
        sum += per[v];
      }
      int run = wave_scan32(sum, lane) - sum;
      s_start[lane] = run;
#pragma unroll
      for (int v = 0; v < kBktWaves; ++v) {
        s_from[v][lane] = run;
        run += per[v];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kBktRounds; ++k) {
      const int j = j0 + k * kWaveSize;
      int64_t to = -1;
      if (bucket[k] >= 0) {
        const int at = s_from[wave][bucket[k]] + rank[k];
        s_val[at] = val[k];
        if constexpr (WEIGHTED) s_w[at] = w[k];
        s_bucket[at] = (uint8_t)bucket[k];
        to = s_to[bucket[k]] + (at - s_start[bucket[k]]);
      }
      if (a.order != nullptr && j < ids) a.order[first + j] = to;
    }
    __syncthreads();
    const int last = a.W - 1;
    int moved = s_start[last];  // ids of the step that have a bucket
#pragma unroll
    for (int v = 0; v < kBktWaves; ++v) moved += s_cnt[v][last];
    for (int i = threadIdx.x; i < moved; i += kBktThreads) {
      const int p = s_bucket[i];
      const int64_t to = s_to[p] + (i - s_start[p]);
      reinterpret_cast<T*>(a.new_indices)[to] = s_val[i];
      if constexpr (WEIGHTED) a.new_weights[to] = s_w[i];
    }
    __syncthreads();
    if (wave == 0 && lane < a.W) {
      int sum = 0;
#pragma unroll
      for (int v = 0; v < kBktWaves; ++v) sum += s_cnt[v][lane];
      s_to[lane] += sum;
    }
    __syncthreads();
  }
}

// Bags per tile: an average of 4096 ids (two steps of bucket_move) where that
// leaves 1536 tiles, six for each of an MI355X's 256 compute units (7.9 M ids in
// 64 x 4096 bags, the four kernels together, best passes: 4096 ids a tile 64 us,
// 2048 74 us, 1024 99 us, 8192 71 us; a fixed figure, so that the workspace
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
  a.lanes = 1;
  while (a.lanes < kWaveSize && 8 * a.lanes * a.n < num_indices) a.lanes *= 2;  // an average bag in two steps of four
  // (calls, us, four launches / two: 5 keys x 133 bags, 1.3 K ids, 2 buckets 46 / 38; 52 x 29, 44 K ids, 3 buckets 61 / 52)
  // (instances of their own: the branches alone cost the large calls 3 %)
  const bool own_prefix = a.n <= kBktOwnLengths && (uintptr_t)lengths % 16 == 0;
  const bool own_scan = num_indices > 0 && z.tiles * num_buckets <= kBktOwnCounts;
  const int rc = mail_open(s, num_buckets, ticket, &a.host_totals);
  if (rc != TRA_OK) return rc;
  const dim3 block(kBktThreads), tiles((unsigned)z.tiles), waves((unsigned)((z.tiles + kBktWaves - 1) / kBktWaves));
  const auto go = [&](auto kernel, dim3 grid, dim3 threads, size_t lds = 0) {
    hipLaunchKernelGGL(kernel, grid, threads, lds, s, a);
  };
  const size_t counters = (size_t)z.bags * (num_buckets + 1) * sizeof(int);
  const auto launch = [&](auto id) {
    using T = decltype(id);
    if (own_prefix) {
      go(bucket_counts_kernel<T, true>, tiles, block, counters);
    } else {
      go(tile_totals_kernel<T>, waves, block);
      go(bucket_counts_kernel<T, false>, tiles, block, counters);
    }
    if (!own_scan) go(bucket_scan_kernel, dim3(num_buckets), dim3(kBktScanThreads));
    if (num_indices == 0) return;
    if (weights && own_scan)
      go(bucket_move_kernel<T, true, true>, tiles, block);
    else if (weights)
      go(bucket_move_kernel<T, true, false>, tiles, block);
    else if (own_scan)
      go(bucket_move_kernel<T, false, true>, tiles, block);
    else
      go(bucket_move_kernel<T, false, false>, tiles, block);
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
