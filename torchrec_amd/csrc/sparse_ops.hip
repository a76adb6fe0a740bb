// Index math around the lookup (offsets, per-key totals, feature permutation,
// block bucketization) and the row-wise quantizer.  Integer results are
// bit-exact by construction; these are bandwidth-trivial next to the gather.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstring>

#include "tra_common.h"

namespace tra {

// (native vectors: an array of HIP's uint4 objects is kept in scratch memory, which doubled the regroup kernel's time)
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef int64_t i64x2_t __attribute__((ext_vector_type(2), aligned(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kScanThreads = 256;

template <typename T>
__device__ __forceinline__ int64_t ld(const void* p, int64_t i) {
  return (int64_t) reinterpret_cast<const T*>(p)[i];
}
template <typename T>
__device__ __forceinline__ void st(void* p, int64_t i, int64_t v) {
  reinterpret_cast<T*>(p)[i] = (T)v;
}

__device__ __forceinline__ int64_t wave_sum(int64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Inclusive scan over a wave.
__device__ __forceinline__ int64_t wave_scan(int64_t v, int lane) {
#pragma unroll
  for (int off = 1; off < kWaveSize; off <<= 1) {
    const int64_t o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
}

// Block-wide sum; result valid in every thread.  `smem` holds >= 4 int64.
__device__ __forceinline__ int64_t block_sum(int64_t v, int64_t* smem) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWaveSize;
  __syncthreads();
  if ((threadIdx.x & (kWaveSize - 1)) == 0) smem[wave] = v;
  __syncthreads();
  int64_t t = 0;
  for (int w = 0; w < (int)(blockDim.x / kWaveSize); ++w) t += smem[w];
  return t;
}

// ---- complete cumsum --------------------------------------------------------
// Two launches for inputs beyond the one-launch scan below: sums of tiles of
// kScanTile lengths, then every tile scanned behind the sum of the sums in front
// of it.  At 262144 lengths both are bound by the latency of their few dependent
// steps on 64 blocks, so a thread holds four consecutive lengths that come with
// one 16-byte load (two for int64), the scan's own loads are under way while the
// sums are added, and the offsets leave as 16-byte vectors.  One length per load
// (sixteen consecutive ones per thread in the second kernel) took 10.1 us for
// 262144 int32 lengths and 20.1 us for 2 M; now 6.6 us, of which two empty
// launches are about 5, and 10.0 us.
constexpr int kTileThreads = 1024;
constexpr int kTileItems = 4;
constexpr int kScanTile = kTileThreads * kTileItems;

// This thread's lengths of the tile (zeros past the end).  VEC: `in` lies on a 16-byte boundary.
template <typename T, bool VEC>
__device__ __forceinline__ void load_tile_items(const T* __restrict__ in, int64_t base, int64_t n,
                                                int64_t (&x)[kTileItems]) {
  struct __align__(16) Vec { T v[kTileItems]; };
  if (VEC && base + kTileItems <= n) {
    const Vec q = *reinterpret_cast<const Vec*>(in + base);
#pragma unroll
    for (int i = 0; i < kTileItems; ++i) x[i] = (int64_t)q.v[i];
  } else {
#pragma unroll
    for (int i = 0; i < kTileItems; ++i) x[i] = base + i < n ? (int64_t)in[base + i] : 0;
  }
}

template <typename T, bool VEC>
__global__ __launch_bounds__(kTileThreads) void tile_sums_kernel(const T* __restrict__ in, int64_t n,
                                                                 int64_t* __restrict__ sums) {
  __shared__ int64_t smem[kTileThreads / kWaveSize];
  int64_t x[kTileItems];
  load_tile_items<T, VEC>(in, (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kTileItems, n, x);
  int64_t v = 0;
#pragma unroll
  for (int i = 0; i < kTileItems; ++i) v += x[i];
  v = block_sum(v, smem);
  if (threadIdx.x == 0) sums[blockIdx.x] = v;
}

// One-launch variant for short inputs: every block first sums everything in
// front of its tile (redundant reads, a few hundred KB from L2 at most), then
// scans the tile.  Tiles are kSmallThreads * (16 / sizeof(T)) elements.
constexpr int kSmallThreads = 1024;
constexpr int kSmallMaxTiles = 64;

template <typename T, bool VEC>
__global__ __launch_bounds__(kSmallThreads) void scan_small_kernel(const T* __restrict__ in,
                                                                    int64_t n, T* __restrict__ out) {
  constexpr int V = 16 / (int)sizeof(T);
  struct __align__(16) Vec { T v[V]; };
  __shared__ int64_t smem[kSmallThreads / kWaveSize];
  __shared__ int64_t wave_tot[kSmallThreads / kWaveSize];
  const int t = threadIdx.x;
  int64_t pre = 0;
  if (VEC) {
    // The tiles in front of this block's: sixteen loads in flight per thread (the last block of
    // a 64-tile input reads 63 tiles; one load at a time would be 63 round trips).
    const Vec* vin = reinterpret_cast<const Vec*>(in);
    const int nk = (int)blockIdx.x;
    int k = 0;
    for (; k + 16 <= nk; k += 16) {
      Vec x[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = vin[(int64_t)(k + j) * kSmallThreads + t];
#pragma unroll
      for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int i = 0; i < V; ++i) pre += (int64_t)x[j].v[i];
    }
    for (; k + 4 <= nk; k += 4) {
      Vec x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = vin[(int64_t)(k + j) * kSmallThreads + t];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < V; ++i) pre += (int64_t)x[j].v[i];
    }
    for (; k < nk; ++k) {
      const Vec x = vin[(int64_t)k * kSmallThreads + t];
#pragma unroll
      for (int i = 0; i < V; ++i) pre += (int64_t)x.v[i];
    }
  } else {
#pragma unroll 4
    for (int k = 0; k < (int)blockIdx.x * V; ++k) pre += (int64_t)in[(int64_t)k * kSmallThreads + t];
  }
  pre = block_sum(pre, smem);
  const int64_t base = ((int64_t)blockIdx.x * kSmallThreads + t) * V;
  int64_t x[V];
  if (VEC && base + V <= n) {
    const Vec q = reinterpret_cast<const Vec*>(in)[base / V];
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = (int64_t)q.v[i];
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) x[i] = base + i < n ? (int64_t)in[base + i] : 0;
  }
  int64_t tsum = 0;
#pragma unroll
  for (int i = 0; i < V; ++i) tsum += x[i];
  const int lane = t & (kWaveSize - 1);
  const int wave = t / kWaveSize;
  int64_t inc = tsum;
#pragma unroll
  for (int off = 1; off < kWaveSize; off <<= 1) {
    const int64_t o = __shfl_up(inc, off, 64);
    if (lane >= off) inc += o;
  }
  if (lane == kWaveSize - 1) wave_tot[wave] = inc;
  __syncthreads();
  int64_t wprefix = 0;
  for (int w = 0; w < wave; ++w) wprefix += wave_tot[w];
  int64_t run = pre + wprefix + inc - tsum;
  if (blockIdx.x == 0 && t == 0) out[0] = 0;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    run += x[i];
    if (base + i < n) out[base + i + 1] = (T)run;
  }
}

// VEC: `in` and `out` lie on 16-byte boundaries.
template <typename T, bool VEC>
__global__ __launch_bounds__(kTileThreads) void scan_tiles_kernel(const T* __restrict__ in, int64_t n,
                                                                  const int64_t* __restrict__ sums,
                                                                  T* __restrict__ out) {
  struct __align__(16) Vec { T v[kTileItems]; };
  __shared__ int64_t smem[kTileThreads / kWaveSize];
  __shared__ int64_t wave_tot[kTileThreads / kWaveSize];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kTileItems;
  int64_t x[kTileItems];
  load_tile_items<T, VEC>(in, base, n, x);
  // Sum of all earlier tiles.
  int64_t prefix = 0;
  for (int i = threadIdx.x; i < (int)blockIdx.x; i += kTileThreads) prefix += sums[i];
  prefix = block_sum(prefix, smem);
  // Exclusive scan of the per-thread sums: wave scan, then wave totals.
  int64_t tsum = 0;
#pragma unroll
  for (int i = 0; i < kTileItems; ++i) tsum += x[i];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int64_t inc = wave_scan(tsum, lane);
  if (lane == kWaveSize - 1) wave_tot[wave] = inc;
  __syncthreads();
  int64_t run = prefix + inc - tsum;
  for (int w = 0; w < wave; ++w) run += wave_tot[w];
  // out[i] is what lies in front of length i: the vectors stay aligned.
  Vec q;
#pragma unroll
  for (int i = 0; i < kTileItems; ++i) {
    q.v[i] = (T)run;
    run += x[i];
  }
  if (VEC && base + kTileItems <= n) {
    *reinterpret_cast<Vec*>(out + base) = q;
  } else {
#pragma unroll
    for (int i = 0; i < kTileItems; ++i)
      if (base + i < n) out[base + i] = q.v[i];
  }
  if (base < n && base + kTileItems >= n) out[n] = (T)run;
}

template <typename T, bool VEC>
static void launch_scan_tiles(const void* lengths, int64_t n, int64_t* sums, void* offsets, unsigned tiles,
                              hipStream_t s) {
  hipLaunchKernelGGL((tile_sums_kernel<T, VEC>), dim3(tiles), dim3(kTileThreads), 0, s, (const T*)lengths, n, sums);
  hipLaunchKernelGGL((scan_tiles_kernel<T, VEC>), dim3(tiles), dim3(kTileThreads), 0, s, (const T*)lengths, n, sums,
                     (T*)offsets);
}

// ---- per-key totals ---------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kScanThreads) void length_per_key_kernel(const void* lengths,
                                                                       int32_t B, int64_t* out) {
  __shared__ int64_t smem[kScanThreads / kWaveSize];
  const int64_t base = (int64_t)blockIdx.x * B;
  int64_t v = 0;
  for (int i = threadIdx.x; i < B; i += kScanThreads) v += ld<T>(lengths, base + i);
  v = block_sum(v, smem);
  if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// ---- feature permutation ----------------------------------------------------
template <typename T>
__global__ void permute_lengths_kernel(const int32_t* permute, int64_t total, int32_t B,
                                       const void* lengths, void* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t tp = i / B;
  const int64_t b = i - tp * B;
  st<T>(out, i, ld<T>(lengths, (int64_t)permute[tp] * B + b));
}

// All values of one feature are contiguous on both sides, so each output
// feature is one straight copy.  grid = (blocks per feature, T').
template <typename OffT, typename ValT>
__global__ void permute_data_kernel(const int32_t* permute, int32_t B, const void* in_off,
                                    const void* out_off, const ValT* values, const float* weights,
                                    ValT* out_values, float* out_weights) {
  const int tp = blockIdx.y;
  const int64_t src = ld<OffT>(in_off, (int64_t)permute[tp] * B);
  const int64_t dst = ld<OffT>(out_off, (int64_t)tp * B);
  const int64_t n = ld<OffT>(out_off, (int64_t)(tp + 1) * B) - dst;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    out_values[dst + i] = values[src + i];
    if (weights) out_weights[dst + i] = weights[src + i];
  }
}

// ---- block bucketization ----------------------------------------------------
// One thread per bag (f, b); a bag's ids are visited in order, so the order
// inside one (bucket, f, b) is the input order.
template <typename T>
__global__ void bucketize_lengths_kernel(const void* offsets, const void* indices,
                                         const int64_t* block_sizes, int32_t B, int64_t n,
                                         int32_t W, void* new_lengths) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T* nl = reinterpret_cast<T*>(new_lengths);
  for (int p = 0; p < W; ++p) nl[(int64_t)p * n + i] = 0;
  const int64_t bs = block_sizes[i / B];
  const int64_t s = ld<T>(offsets, i), e = ld<T>(offsets, i + 1);
  for (int64_t j = s; j < e; ++j) {
    const int64_t id = ld<T>(indices, j);
    const uint64_t p = (uint64_t)id / (uint64_t)bs;
    if (p < (uint64_t)W) nl[(int64_t)p * n + i] += 1;
  }
}

template <typename T>
__global__ void bucketize_scatter_kernel(const void* offsets, const void* indices,
                                         const float* weights, const int64_t* block_sizes,
                                         int32_t B, int64_t n, int32_t W, int keep_orig,
                                         const void* new_offsets, int64_t* cursor,
                                         void* new_indices, float* new_weights,
                                         int64_t* unbucketize_permute) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int p = 0; p < W; ++p) cursor[(int64_t)p * n + i] = ld<T>(new_offsets, (int64_t)p * n + i);
  const int64_t bs = block_sizes[i / B];
  const int64_t s = ld<T>(offsets, i), e = ld<T>(offsets, i + 1);
  for (int64_t j = s; j < e; ++j) {
    const int64_t id = ld<T>(indices, j);
    const uint64_t p = (uint64_t)id / (uint64_t)bs;
    if (p >= (uint64_t)W) {
      if (unbucketize_permute) unbucketize_permute[j] = -1;
      continue;
    }
    const int64_t pos = cursor[(int64_t)p * n + i]++;
    st<T>(new_indices, pos, keep_orig ? id : (int64_t)((uint64_t)id % (uint64_t)bs));
    if (weights) new_weights[pos] = weights[j];
    if (unbucketize_permute) unbucketize_permute[j] = pos;
  }
}

// ---- a wave walking the ids of its own run of bags ---------------------------
// The id-parallel kernels below (bucketization, positions in bags, position
// weights) share one mapping: a wave owns `bpw` consecutive bags (a power of
// two, at most 64), keeps their bounds in LDS and visits their ids in order,
// 64 at a time, so every load and store of ids is coalesced; the bag of an id
// is found by a branch-free search over the wave's bounds.  Waves never share
// LDS, so the only synchronization is program order inside the wave.
constexpr int kWalkThreads = 256;
constexpr int kWalkWaves = kWalkThreads / kWaveSize;
constexpr int kWalkMaxBuckets = 1024;  // wider bucketizations take the thread-per-bag kernels

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// Largest b in [0, cnt) with off[b] <= j; off[0] <= j holds.  top_step = bpw / 2.
__device__ __forceinline__ int find_bag(const int64_t* off, int cnt, int top_step, int64_t j) {
  int lo = 0;
  for (int step = top_step; step >= 1; step >>= 1) {
    const int c = lo + step;
    if (c < cnt && off[c] <= j) lo = c;
  }
  return lo;
}

// id / bs and id % bs; 32-bit arithmetic where both fit.
__device__ __forceinline__ void div_mod(uint64_t id, uint64_t bs, uint64_t& q, uint64_t& r) {
  if (((id | bs) >> 32) == 0) {
    const uint32_t a = (uint32_t)id, b = (uint32_t)bs;
    const uint32_t qq = a / b;
    q = qq;
    r = a - qq * b;
  } else {
    q = id / bs;
    r = id - q * bs;
  }
}

// Bags per wave for n bags.  The kernels are bound by the latency of a wave's
// chain (bounds, search, ids, stores), so many short waves beat few long ones:
// 64 bags, halved down to 8 while that leaves fewer than 16384 waves (measured
// on 131072 and 262144 bags: 1.5x faster than 4096 waves), further only while
// fewer than 4096 (a wave should still find about a wave's worth of ids), and
// never more than `cap`.
static int bags_per_wave(int64_t n, int cap) {
  int bpw = 64;
  while (bpw > 8 && (n + bpw - 1) / bpw < 16384) bpw >>= 1;
  while (bpw > 1 && (n + bpw - 1) / bpw < 4096) bpw >>= 1;
  while (bpw > cap) bpw >>= 1;
  return bpw;
}

template <typename T>
__global__ __launch_bounds__(kWalkThreads) void bucketize_lengths_wave_kernel(
    const T* __restrict__ offsets, const T* __restrict__ indices, const int64_t* __restrict__ block_sizes,
    int32_t B, int64_t n, int32_t W, int bpw, T* __restrict__ new_lengths) {
  extern __shared__ int64_t walk_smem[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int per_wave = (bpw + 1) + bpw + (W * bpw + 1) / 2;  // int64 units
  int64_t* s_off = walk_smem + (size_t)wave * per_wave;
  int64_t* s_bs = s_off + bpw + 1;
  int32_t* s_cnt = reinterpret_cast<int32_t*>(s_bs + bpw);
  const int64_t i0 = ((int64_t)blockIdx.x * kWalkWaves + wave) * bpw;
  if (i0 >= n) return;
  const int cnt = (int)(n - i0 < bpw ? n - i0 : bpw);
  for (int k = lane; k <= cnt; k += kWaveSize) s_off[k] = (int64_t)offsets[i0 + k];
  for (int k = lane; k < cnt; k += kWaveSize) s_bs[k] = block_sizes[(i0 + k) / B];
  for (int k = lane; k < W * bpw; k += kWaveSize) s_cnt[k] = 0;
  wave_lds_sync();
  const int64_t first = s_off[0], last = s_off[cnt];
  for (int64_t j0 = first; j0 < last; j0 += kWaveSize) {
    const int64_t j = j0 + lane;
    if (j < last) {
      const int64_t id = (int64_t)indices[j];
      const int b = find_bag(s_off, cnt, bpw >> 1, j);
      uint64_t q, r;
      div_mod((uint64_t)id, (uint64_t)s_bs[b], q, r);
      if (q < (uint64_t)W) atomicAdd(&s_cnt[(int)q * bpw + b], 1);
    }
  }
  wave_lds_sync();
  for (int x = lane; x < W * cnt; x += kWaveSize) {
    const int p = x / cnt, k = x - p * cnt;
    new_lengths[(int64_t)p * n + i0 + k] = (T)s_cnt[p * bpw + k];
  }
}

template <typename T>
__global__ __launch_bounds__(kWalkThreads) void bucketize_scatter_wave_kernel(
    const T* __restrict__ offsets, const T* __restrict__ indices, const float* __restrict__ weights,
    const int64_t* __restrict__ block_sizes, int32_t B, int64_t n, int32_t W, int bpw, int keep_orig,
    const T* __restrict__ new_offsets, T* __restrict__ new_indices, float* __restrict__ new_weights,
    int64_t* __restrict__ unbucketize_permute) {
  extern __shared__ int64_t walk_smem[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int per_wave = (bpw + 1) + bpw + W * bpw;
  int64_t* s_off = walk_smem + (size_t)wave * per_wave;
  int64_t* s_bs = s_off + bpw + 1;
  int64_t* s_cur = s_bs + bpw;  // next output position of (bucket p, bag b) at [p * bpw + b]
  const int64_t i0 = ((int64_t)blockIdx.x * kWalkWaves + wave) * bpw;
  if (i0 >= n) return;
  const int cnt = (int)(n - i0 < bpw ? n - i0 : bpw);
  for (int k = lane; k <= cnt; k += kWaveSize) s_off[k] = (int64_t)offsets[i0 + k];
  for (int k = lane; k < cnt; k += kWaveSize) s_bs[k] = block_sizes[(i0 + k) / B];
  for (int x = lane; x < W * cnt; x += kWaveSize) {
    const int p = x / cnt, k = x - p * cnt;
    s_cur[p * bpw + k] = (int64_t)new_offsets[(int64_t)p * n + i0 + k];
  }
  wave_lds_sync();
  const int64_t first = s_off[0], last = s_off[cnt];
  const uint64_t below_me = lane == 0 ? 0ull : (~0ull >> (kWaveSize - lane));
  for (int64_t j0 = first; j0 < last; j0 += kWaveSize) {
    const int64_t j = j0 + lane;
    const bool valid = j < last;
    const int64_t id = valid ? (int64_t)indices[j] : 0;
    const int b = find_bag(s_off, cnt, bpw >> 1, valid ? j : first);
    uint64_t q = 0, r = 0;
    div_mod((uint64_t)id, (uint64_t)s_bs[b], q, r);
    const bool in = valid && q < (uint64_t)W;
    const int p = in ? (int)q : -1;
    // The lanes of this chunk that hold ids of my bag: [lo_lane, hi_lane).
    const int64_t lo64 = s_off[b] - j0, hi64 = s_off[b + 1] - j0;
    const int lo_lane = lo64 < 0 ? 0 : (lo64 > kWaveSize - 1 ? kWaveSize - 1 : (int)lo64);
    const int hi_lane = hi64 > kWaveSize ? kWaveSize : (hi64 < 0 ? 0 : (int)hi64);
    const uint64_t my_bag = (hi_lane >= kWaveSize ? ~0ull : ((1ull << hi_lane) - 1)) & ~((1ull << lo_lane) - 1);
    // Rank of my id among the ids of the same bag and bucket in this chunk
    // (input order), one pass per bucket value present in the wave.
    int rank = 0, same_count = 0;
    uint64_t rem = __builtin_amdgcn_ballot_w64(in);
    while (rem != 0) {
      const int leader = __builtin_amdgcn_readfirstlane(__builtin_ctzll(rem));
      const int pl = __builtin_amdgcn_readlane(p, leader);
      const uint64_t m = __builtin_amdgcn_ballot_w64(in && p == pl);
      if (in && p == pl) {
        const uint64_t same = m & my_bag;
        rank = __builtin_popcountll(same & below_me);
        same_count = __builtin_popcountll(same);
      }
      rem &= ~m;
    }
    int64_t pos = -1;
    if (in) {
      pos = s_cur[p * bpw + b] + rank;
      new_indices[pos] = keep_orig ? (T)id : (T)r;
      if (weights) new_weights[pos] = weights[j];
    }
    if (valid && unbucketize_permute) unbucketize_permute[j] = pos;
    wave_lds_sync();  // every lane has read its cursor
    if (in && rank == same_count - 1) s_cur[p * bpw + b] = pos + 1;
    wave_lds_sync();
  }
}

// ---- row-wise N-bit quantization -------------------------------------------
// One wave per row.  Same operation order as fbgemm's
// FloatOrHalfToFusedNBitRowwiseQuantizedSBHalf: min/max, bias = fp16(min),
// scale = fp16((max - bias) / (2^bits - 1)), q = clamp(rint((x - bias) * (1/scale))).
// header_first: TBE row [scale][bias][payload]; otherwise fbgemm's trailer row.
// A row's header dword (fp16 scale, fp16 bias) from its extremes, with the bias
// and the reciprocal scale its elements are quantized by.
template <int BITS>
__device__ __forceinline__ uint32_t row_header(float mn, float mx, float& bias, float& inv) {
  constexpr int kQMax = (1 << BITS) - 1;
  const __half bias_h = __float2half_rn(mn);
  bias = __half2float(bias_h);
  const float range = mx - bias;
  float scale = range == 0.0f ? 1.0f : range / (float)kQMax;
  scale = __half2float(__float2half_rn(scale));
  if (scale == 0.0f) scale = 1.0f;
  inv = 1.0f / scale;
  if (__builtin_isinf(inv)) {
    scale = 1.0f;
    inv = 1.0f;
  }
  return (uint32_t)__half_as_ushort(__float2half_rn(scale)) | ((uint32_t)__half_as_ushort(bias_h) << 16);
}

// DPL output dwords from their elements.
template <int BITS, int DPL>
__device__ __forceinline__ void pack_elements(const float* v, float bias, float inv, uint32_t* packed) {
  constexpr int EPD = 32 / BITS;
  constexpr int kQMax = (1 << BITS) - 1;
#pragma unroll
  for (int d = 0; d < DPL; ++d) packed[d] = 0;
#pragma unroll
  for (int e = 0; e < DPL * EPD; ++e) {
    const float t = (v[e] - bias) * inv;
    float q = __builtin_rintf(t);
    q = q < 0.0f ? 0.0f : q;
    q = q > (float)kQMax ? (float)kQMax : q;
    packed[e / EPD] |= (uint32_t)(int)q << ((e % EPD) * BITS);
  }
}

template <int BITS>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const float* in, int64_t rows,
                                                            int32_t dim, uint8_t* out,
                                                            int64_t row_bytes, int header_first) {
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int64_t r = (int64_t)blockIdx.x * (blockDim.x / kWaveSize) + threadIdx.x / kWaveSize;
  if (r >= rows) return;
  const float* x = in + r * dim;
  float mn = x[0], mx = x[0];
  for (int c = lane; c < dim; c += kWaveSize) {
    const float v = x[c];
    mn = v < mn ? v : mn;
    mx = v > mx ? v : mx;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float a = __shfl_xor(mn, off, 64), b = __shfl_xor(mx, off, 64);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  constexpr int kQMax = (1 << BITS) - 1;
  constexpr int kEpb = 8 / BITS;
  float bias, inv;
  const uint32_t header = row_header<BITS>(mn, mx, bias, inv);
  const int payload = dim / kEpb;
  uint8_t* o = out + r * row_bytes;
  uint8_t* pay = header_first ? o + 4 : o;
  uint8_t* hdr = header_first ? o : o + payload;
  for (int byte = lane; byte < payload; byte += kWaveSize) {
    uint32_t packed = 0;
#pragma unroll
    for (int e = 0; e < kEpb; ++e) {
      const float t = (x[byte * kEpb + e] - bias) * inv;
      float q = __builtin_rintf(t);
      q = q < 0.0f ? 0.0f : q;
      q = q > (float)kQMax ? (float)kQMax : q;
      packed |= (uint32_t)(int)q << (e * BITS);
    }
    pay[byte] = (uint8_t)packed;
  }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) hdr[i] = (uint8_t)(header >> (8 * i));
  }
}

// The same quantizer for rows whose elements and output rows are 4-byte
// aligned (dim a multiple of 32 / BITS): a lane owns the 32 / BITS consecutive
// elements of one output dword, loads them 16 bytes at a time and stores the
// dword whole; `lpr` lanes (a power of two) share a row, 64 / lpr rows a wave.
// Per element the arithmetic is that of quantize_rows_kernel.
// DPL: output dwords a lane owns per step.  More than one means fewer lanes per
// row, fewer steps of the min / max exchange and fewer memory instructions per
// byte; 8-bit rows use two.
template <int BITS, int DPL = 1>
__global__ __launch_bounds__(256) void quantize_rows_vec_kernel(const float* __restrict__ in, int64_t rows,
                                                                int32_t dim, uint8_t* __restrict__ out,
                                                                int64_t row_bytes, int header_first,
                                                                int lpr, int pad_dwords) {
  constexpr int EPD = 32 / BITS;    // elements per output dword
  constexpr int EPL = DPL * EPD;    // elements per lane and step
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int g = lane / lpr, c = lane - g * lpr;
  const int rows_per_wave = kWaveSize / lpr;
  const int64_t r_raw = ((int64_t)blockIdx.x * (blockDim.x / kWaveSize) + threadIdx.x / kWaveSize) * rows_per_wave + g;
  const bool active = r_raw < rows;
  const int64_t r = active ? r_raw : rows - 1;  // every lane takes part in the reductions
  const float* x = in + r * dim;
  const int chunks = dim / EPL;
  float mn = x[0], mx = mn;
  float keep[EPL];  // the lane's first chunk stays in registers for the second pass
#pragma unroll
  for (int e = 0; e < EPL; ++e) keep[e] = mn;
  for (int ch = c; ch < chunks; ch += lpr) {
    float v[EPL];
#pragma unroll
    for (int k = 0; k < EPL / 4; ++k) {
      const float4 q = *reinterpret_cast<const float4*>(x + ch * EPL + 4 * k);
      v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      mn = v[e] < mn ? v[e] : mn;
      mx = v[e] > mx ? v[e] : mx;
      if (ch == c) keep[e] = v[e];
    }
  }
  for (int off = lpr >> 1; off > 0; off >>= 1) {
    const float a = __shfl_xor(mn, off, 64), b = __shfl_xor(mx, off, 64);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  float bias, inv;
  const uint32_t header = row_header<BITS>(mn, mx, bias, inv);
  if (!active) return;
  uint8_t* o = out + r * row_bytes;
  uint32_t* pay = reinterpret_cast<uint32_t*>(header_first ? o + 4 : o);
  uint32_t* hdr = reinterpret_cast<uint32_t*>(header_first ? o : o + (int64_t)chunks * (4 * DPL));
  for (int ch = c; ch < chunks; ch += lpr) {
    float v[EPL];
    if (ch == c) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) v[e] = keep[e];
    } else {
#pragma unroll
      for (int k = 0; k < EPL / 4; ++k) {
        const float4 q = *reinterpret_cast<const float4*>(x + ch * EPL + 4 * k);
        v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
      }
    }
    uint32_t packed[DPL];
    pack_elements<BITS, DPL>(v, bias, inv, packed);
    // one store of DPL dwords (the payload is 4-byte aligned, not more)
    __builtin_memcpy(__builtin_assume_aligned(pay + ch * DPL, 4), packed, sizeof(packed));
  }
  if (c == 0) *hdr = header;
  for (int w = c; w < pad_dwords; w += lpr) pay[chunks * DPL + w] = 0;  // (header_first rows only)
}

// The same for the padded rows of a lookup operator's store: header, payload,
// zeros up to the row stride, and `tail_dwords` zeros behind the last row, so
// that the store needs no clearing first and nothing is copied into it
// afterwards.  A wave builds its rows in LDS and writes them out as one
// contiguous run of 16-byte vectors: with a 4-byte store per lane a 68-byte
// row leaves in pieces (int4 rows of dim 128 at a 128-byte stride, 1 M rows,
// steady state of one table quantized again and again: 122 us written directly,
// 111 us built in LDS; four tables in turn take 133 us each; 8-bit rows are even, 2-bit
// rows 4 % slower, so those take the kernel above).  Rows of at most 64 lanes.
template <int BITS, int DPL>
__global__ __launch_bounds__(256) void quantize_rows_padded_kernel(const float* __restrict__ in, int64_t rows,
                                                                   int32_t dim, uint32_t* __restrict__ out,
                                                                   int32_t stride_dwords, int lpr, int tail_dwords) {
  extern __shared__ __align__(16) uint32_t qrow_smem[];
  constexpr int EPD = 32 / BITS;
  constexpr int EPL = DPL * EPD;
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int g = lane / lpr, c = lane - g * lpr;
  const int rows_per_wave = kWaveSize / lpr;
  if (blockIdx.x == 0)
    for (int w = threadIdx.x; w < tail_dwords; w += blockDim.x) out[rows * stride_dwords + w] = 0;
  const int64_t base = ((int64_t)blockIdx.x * (blockDim.x / kWaveSize) + wave) * rows_per_wave;
  if (base >= rows) return;
  const int64_t r = base + g < rows ? base + g : rows - 1;  // every lane takes part in the reductions
  const int chunks = dim / EPL;
  const float* x = in + r * dim + (c < chunks ? c : 0) * EPL;
  float v[EPL];
#pragma unroll
  for (int k = 0; k < EPL / 4; ++k) {
    const f32x4_t q = *reinterpret_cast<const f32x4_t*>(x + 4 * k);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[4 * k + i] = q[i];
  }
  float mn = __shfl(v[0], lane - c, 64), mx = mn;  // (the row's first element, as in the kernels above)
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    mn = v[e] < mn ? v[e] : mn;
    mx = v[e] > mx ? v[e] : mx;
  }
  for (int off = lpr >> 1; off > 0; off >>= 1) {
    const float a = __shfl_xor(mn, off, 64), b = __shfl_xor(mx, off, 64);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  float bias, inv;
  const uint32_t header = row_header<BITS>(mn, mx, bias, inv);
  uint32_t* row = qrow_smem + (size_t)(wave * rows_per_wave + g) * stride_dwords;
  if (c < chunks) {
    uint32_t packed[DPL];
    pack_elements<BITS, DPL>(v, bias, inv, packed);
#pragma unroll
    for (int d = 0; d < DPL; ++d) row[1 + c * DPL + d] = packed[d];
  }
  if (c == 0) row[0] = header;
  for (int w = 1 + chunks * DPL + c; w < stride_dwords; w += lpr) row[w] = 0;
  wave_lds_sync();
  // the wave's rows are neighbours in LDS and in the store
  const uint32_t* src = qrow_smem + (size_t)wave * rows_per_wave * stride_dwords;
  const int n = (int)(rows - base < rows_per_wave ? rows - base : rows_per_wave) * stride_dwords;
  uint32_t* dst = out + base * stride_dwords;
  if (stride_dwords % 4 == 0 && (uintptr_t)out % 16 == 0) {
    for (int i = lane * 4; i < n; i += 4 * kWaveSize)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4_t*>(src + i), reinterpret_cast<u32x4_t*>(dst + i));
  } else {
    for (int i = lane; i < n; i += kWaveSize) dst[i] = src[i];
  }
}

__global__ __launch_bounds__(256) void zero_dwords_kernel(uint32_t* out, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = 0;
}

// ---- positions inside bags ---------------------------------------------------
// range[j] = j - start(bag of j), for j < range_size; `offsets` has n entries
// and the last bag ends at range_size.
template <typename T>
__global__ __launch_bounds__(kWalkThreads) void offsets_range_kernel(const T* __restrict__ offsets, int64_t n,
                                                                      int64_t range_size, int bpw,
                                                                      T* __restrict__ out) {
  extern __shared__ int64_t walk_smem[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  int64_t* s_off = walk_smem + (size_t)wave * (bpw + 1);
  const int64_t i0 = ((int64_t)blockIdx.x * kWalkWaves + wave) * bpw;
  if (i0 >= n) return;
  const int cnt = (int)(n - i0 < bpw ? n - i0 : bpw);
  for (int k = lane; k <= cnt; k += kWaveSize) {
    int64_t v = i0 + k < n ? (int64_t)offsets[i0 + k] : range_size;
    v = v < 0 ? 0 : v;
    s_off[k] = v < range_size ? v : range_size;
  }
  wave_lds_sync();
  const int64_t first = s_off[0], last = s_off[cnt];
  for (int64_t j = first + lane; j < last; j += kWaveSize) {
    const int b = find_bag(s_off, cnt, bpw >> 1, j);
    out[j] = (T)(j - s_off[b]);
  }
}

// weight[j] = table[key_start[k] + (j - start of j's bag)] for an id of key k,
// 1.0 for keys without a table.  Positions at or beyond the key's table length
// take the last entry.
template <typename T>
__global__ __launch_bounds__(kWalkThreads) void position_weights_kernel(
    const T* __restrict__ offsets, int32_t B, int64_t n, const int32_t* __restrict__ key_start,
    const int32_t* __restrict__ key_len, const float* __restrict__ table, int bpw, float* __restrict__ out) {
  extern __shared__ int64_t walk_smem[];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  int64_t* s_off = walk_smem + (size_t)wave * (2 * bpw + 1);
  int32_t* s_start = reinterpret_cast<int32_t*>(s_off + bpw + 1);
  int32_t* s_len = s_start + bpw;
  const int64_t i0 = ((int64_t)blockIdx.x * kWalkWaves + wave) * bpw;
  if (i0 >= n) return;
  const int cnt = (int)(n - i0 < bpw ? n - i0 : bpw);
  for (int k = lane; k <= cnt; k += kWaveSize) s_off[k] = (int64_t)offsets[i0 + k];
  for (int k = lane; k < cnt; k += kWaveSize) {
    const int key = (int)((i0 + k) / B);
    s_start[k] = key_start[key];
    s_len[k] = key_len[key];
  }
  wave_lds_sync();
  const int64_t first = s_off[0], last = s_off[cnt];
  for (int64_t j = first + lane; j < last; j += kWaveSize) {
    const int b = find_bag(s_off, cnt, bpw >> 1, j);
    const int len = s_len[b];
    const int64_t pos = j - s_off[b];
    float w = 1.0f;
    if (len > 0) w = table[s_start[b] + (int)(pos < len ? pos : len - 1)];
    out[j] = w;
  }
}

// ---- ids moved key by key, with or without a remap -------------------------------
// Output key j of a launch is input key perm[j]: its ids (and weights, and
// lengths) are one contiguous run on both sides.  With REMAP every id goes
// through its key's sorted table on the way:
//   out = mapping[i] when sorted_ids[i] == id, with i the first index in
//   [0, size-1] whose entry is >= id (searched over the first size-1 entries;
//   the last one is the table's delimiter), else miss_id.
constexpr int kMoveThreads = 512;
constexpr int kMoveKeys = 256;   // input keys, and output keys, of a call
constexpr int kRemapKeys = 64;   // keys with a table per launch
constexpr int kPivots = 512;     // entries of a table that a block keeps in LDS

// Where the input keys' ids lie.
constexpr int kKeysTotals = 0;   // int64 totals[num_in] on the device
constexpr int kKeysOffsets = 1;  // offsets[k * B]; output positions are the input's
constexpr int kKeysOne = 2;      // one key, all num_values ids

struct RemapTables {
  const int64_t* sorted_ids[kRemapKeys];
  const int64_t* mapping[kRemapKeys];
  int64_t size[kRemapKeys];
  int64_t miss_id[kRemapKeys];
};
struct MoveArgs {
  const void* bounds;
  const void* values;
  void* out_values;
  const float* weights;
  float* out_weights;
  const void* lengths;
  void* out_lengths;
  int64_t num_values;
  int64_t out_values_end;  // ids the output holds
  int32_t kind;
  int32_t bounds_i64;
  int32_t lengths_i64;
  int32_t num_in;
  int32_t num_out;     // output keys of the call
  int32_t first_key;   // output keys of this launch: first_key .. first_key + launch_keys
  int32_t launch_keys;
  int32_t B;
  int32_t tile;          // ids per tile
  int32_t tile_blocks;   // blocks that move ids (they stride over the tiles); the ones behind them move lengths
  int16_t perm[kMoveKeys];
};

// First index in [0, n] whose entry is >= v, and that entry; n < 1 or no such
// index below n: n.  `pivots`: entry min((i + 1) * seg, n) - 1 for i < kPivots.
//
// Bound by the reads of the table, one behind the other and each lane in a line
// of its own: a bisection over half a million entries takes nineteen (8 tables
// x 500,000, 410 K ids: 37 us).  Here the first nine steps are taken in LDS;
// inside the segment the place is guessed from the values at its ends (raw ids
// are usually spread evenly: hashes) and four neighbouring entries are read in
// two loads, which mostly ends the search in three or four reads; every second
// later step bisects, so that any distribution ends.  20 us on warm tables, of
// it 7 outside the segments; four single loads 29 us, two entries a read 24 us,
// eight 21 us (24 us behind other work, which takes the tables out of the caches).
__device__ __forceinline__ int64_t remap_lower_bound(const int64_t* __restrict__ sorted, int64_t n, int64_t seg,
                                                     const int64_t* pivots, int64_t v, int64_t& entry) {
  int p = 0;
#pragma unroll
  for (int step = kPivots / 2; step >= 1; step >>= 1)
    if (pivots[p + step - 1] < v) p += step;
  if (pivots[p] < v) {  // (only the last pivot: every entry below n is smaller)
    entry = sorted[n];
    return n;
  }
  int64_t lo = p * seg;
  int64_t hi = min(lo + seg, n) - 1;
  int64_t vh = pivots[p];                   // sorted[hi] >= v
  int64_t vl = p > 0 ? pivots[p - 1] : vh;  // sorted[lo - 1] < v where vl_known
  bool vl_known = p > 0;
  for (int it = 0; lo < hi; ++it) {
    int64_t mid = lo + ((hi - lo) >> 1);
    if (vl_known && (it < 3 || (it & 1) == 0)) {
      const float f = (float)((uint64_t)v - (uint64_t)vl) / (float)((uint64_t)vh - (uint64_t)vl);
      mid = lo + (int64_t)(f * (float)(hi - lo + 1)) - 1;
    }
    // Entries base .. base + 3: inside [lo, hi] where that holds four, else reaching into what is
    // known already, but never behind the table (n + 1 entries; a segment of two means n > 512).
    int64_t base = max(min(mid - 1, hi - 3), lo);
    base = max(min(base, n - 3), (int64_t)0);
    int64_t x[4];
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const i64x2_t q = *reinterpret_cast<const i64x2_t*>(sorted + base + e);
      x[e] = q.x;
      x[e + 1] = q.y;
    }
    int below = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) below += x[e] < v && (e < 3 || base + 3 < n) ? 1 : 0;  // (entry n need not be in order)
    if (below == 4) {
      lo = base + 4;
      vl = x[3];
      vl_known = true;
    } else {
      hi = base + below;
      vh = below == 0 ? x[0] : below == 1 ? x[1] : below == 2 ? x[2] : x[3];
      if (below != 0) lo = hi;
    }
  }
  entry = vh;
  return lo;
}

template <typename T, bool REMAP>
__global__ __launch_bounds__(kMoveThreads) void move_keys_kernel(const MoveArgs m, const RemapTables t) {
  __shared__ int64_t s_first[kMoveKeys + 1];
  __shared__ int64_t s_found[4];
  __shared__ int64_t s_pivot[REMAP ? kPivots : 1];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  if ((int)blockIdx.x >= m.tile_blocks) {  // lengths: no bounds needed
    const int64_t stride = (int64_t)(gridDim.x - m.tile_blocks) * kMoveThreads;
    const int64_t total = (int64_t)m.launch_keys * m.B;
    for (int64_t i = (int64_t)(blockIdx.x - m.tile_blocks) * kMoveThreads + threadIdx.x; i < total; i += stride) {
      const int64_t j = i / m.B;
      const int64_t src = (int64_t)m.perm[m.first_key + j] * m.B + (i - j * m.B), dst = (int64_t)m.first_key * m.B + i;
      if (m.lengths_i64)
        st<int64_t>(m.out_lengths, dst, ld<int64_t>(m.lengths, src));
      else
        st<int32_t>(m.out_lengths, dst, ld<int32_t>(m.lengths, src));
    }
    return;
  }
  if (wave == 0) {
    if (m.kind == kKeysTotals) {
      int64_t before = 0;
      for (int k0 = 0; k0 < m.num_in; k0 += kWaveSize) {
        int64_t incl = k0 + lane < m.num_in ? ld<int64_t>(m.bounds, k0 + lane) : 0;
        incl = wave_scan(incl, lane);
        if (k0 + lane < m.num_in) s_first[k0 + lane + 1] = before + incl;
        before += __shfl(incl, kWaveSize - 1, kWaveSize);
      }
      if (lane == 0) s_first[0] = 0;
    } else {
      for (int k = lane; k <= m.num_in; k += kWaveSize)
        s_first[k] = m.kind == kKeysOne ? (k == 0 ? 0 : m.num_values)
                     : m.bounds_i64     ? ld<int64_t>(m.bounds, (int64_t)k * m.B)
                                        : ld<int32_t>(m.bounds, (int64_t)k * m.B);
    }
  }
  __syncthreads();
  for (int64_t tile = blockIdx.x;; tile += m.tile_blocks) {
    // The tile's output key, and where its ids come from and go to.
    if (wave == 0) {
      int64_t to = 0, tiles_before = 0;
      int key = -1;
      for (int j0 = 0; key < 0 && j0 < m.num_out; j0 += kWaveSize) {
        const int j = j0 + lane;
        int64_t first = 0, n = 0;
        if (j < m.num_out) {
          const int k = m.perm[j];
          first = s_first[k] < 0 ? 0 : s_first[k];
          n = (s_first[k + 1] > m.num_values ? m.num_values : s_first[k + 1]) - first;
          n = n < 0 ? 0 : n;
        }
        const bool mine = j >= m.first_key && j < m.first_key + m.launch_keys;
        const int64_t tiles = mine ? (n + m.tile - 1) / m.tile : 0;
        const int64_t to_incl = wave_scan(n, lane), tiles_incl = wave_scan(tiles, lane);
        const uint64_t past = __builtin_amdgcn_ballot_w64(tiles_before + tiles_incl > tile);
        if (past != 0) {
          const int hit = __builtin_ctzll(past);
          key = j0 + hit;
          if (lane == hit) {
            const int64_t in_key = (tile - (tiles_before + tiles_incl - tiles)) * m.tile;
            s_found[0] = key;
            s_found[1] = first + in_key;
            s_found[2] = (m.kind == kKeysTotals ? to + to_incl - n : first) + in_key;
            s_found[3] = n - in_key < m.tile ? n - in_key : m.tile;
          }
        }
        to += __shfl(to_incl, kWaveSize - 1, kWaveSize);
        tiles_before += __shfl(tiles_incl, kWaveSize - 1, kWaveSize);
      }
      if (key < 0 && lane == 0) s_found[0] = -1;
    }
    __syncthreads();
    const int key = (int)s_found[0];
    const int64_t src = s_found[1], dst = s_found[2];
    int64_t n = s_found[3];
    if (key < 0) return;
    n = dst + n > m.out_values_end ? m.out_values_end - dst : n;
    const T* __restrict__ in = reinterpret_cast<const T*>(m.values) + src;
    T* __restrict__ out = reinterpret_cast<T*>(m.out_values) + dst;
    if constexpr (REMAP) {
      const int tk = key - m.first_key;
      const int64_t* __restrict__ sorted = t.sorted_ids[tk];
      const int64_t* __restrict__ mapping = t.mapping[tk];
      const int64_t last = t.size[tk] - 1, miss = t.miss_id[tk];
      const int64_t seg = (last + kPivots - 1) / kPivots;
      if ((int)threadIdx.x < kPivots && last > 0) {
        const int64_t end = (threadIdx.x + 1) * seg;
        s_pivot[threadIdx.x] = sorted[(end < last ? end : last) - 1];
      }
      __syncthreads();
      for (int64_t i = threadIdx.x; i < n; i += kMoveThreads) {
        const int64_t v = (int64_t)in[i];
        int64_t entry;
        int64_t at = 0;
        if (last > 0)
          at = remap_lower_bound(sorted, last, seg, s_pivot, v, entry);
        else
          entry = sorted[0];
        out[i] = (T)(entry == v ? mapping[at] : miss);
      }
    } else {
#pragma unroll 4
      for (int64_t i = threadIdx.x; i < n; i += kMoveThreads) out[i] = in[i];
    }
    if (m.weights)
#pragma unroll 4
      for (int64_t i = threadIdx.x; i < n; i += kMoveThreads) m.out_weights[dst + i] = m.weights[src + i];
    __syncthreads();  // s_found and s_pivot have been read by everyone
  }
}

// Column blocks of row-major matrices copied into other matrices: block k is
// `width` elements of every row, from src[k] (row stride src_stride[k]) to
// dst[k] (row stride dst_stride[k]); both pointers already include the
// block's first column.
//
// A pure copy, bound by memory.  The columns of all blocks are laid side by
// side and cut into vectors of V bytes (the largest of 16, 8, 4, 2 that
// divides every address, row stride and width of the launch); a thread owns one
// vector column, looks its block up once and walks R rows with all R loads in
// flight, so there is no division and no table access per element and a
// workgroup reads and writes long pieces of few rows.
constexpr int kRegroupBlocks = 96;
struct RegroupBlocks {
  const uint8_t* src[kRegroupBlocks];
  uint8_t* dst[kRegroupBlocks];
  int64_t src_stride[kRegroupBlocks];  // bytes
  int64_t dst_stride[kRegroupBlocks];  // bytes
  int32_t first[kRegroupBlocks];       // first vector column of the block
};

// blockIdx.x: tile of rp * R rows; blockIdx.y: tile of `cw` vector columns.
// Thread t of the workgroup holds column t % cw and rows t / cw + k * rp.
template <typename V, int R>
__global__ __launch_bounds__(256) void regroup_kernel(const RegroupBlocks b, int n_blocks, int columns, int cw,
                                                      int rp, int64_t rows) {
  __shared__ int32_t s_first[kRegroupBlocks];
  for (int k = threadIdx.x; k < n_blocks; k += blockDim.x) s_first[k] = b.first[k];
  __syncthreads();
  const int rt = threadIdx.x / cw;
  const int col = blockIdx.y * cw + (threadIdx.x - rt * cw);
  const int64_t r0 = (int64_t)blockIdx.x * (rp * R) + rt;
  if (rt >= rp || col >= columns || r0 >= rows) return;
  int lo = 0, hi = n_blocks - 1;  // the last block whose first column is <= col
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_first[mid] <= col) lo = mid; else hi = mid - 1;
  }
  const int64_t off = (int64_t)(col - s_first[lo]) * (int)sizeof(V);
  const int64_t ss = b.src_stride[lo], ds = b.dst_stride[lo];
  const uint8_t* src = b.src[lo] + off + r0 * ss;
  uint8_t* dst = b.dst[lo] + off + r0 * ds;
  V v[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int64_t step = r0 + k * rp < rows ? (int64_t)k * rp : 0;  // past the end: the first row again
    v[k] = *reinterpret_cast<const V*>(src + step * ss);
  }
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (r0 + k * rp < rows) *reinterpret_cast<V*>(dst + (int64_t)k * rp * ds) = v[k];
}

template <typename V>
static void launch_regroup(const RegroupBlocks& b, int n_blocks, int columns, int64_t rows, hipStream_t s) {
  // Column tiles of at most 256 threads and nearly equal width; rows side by side where the tile is narrow.
  const int tiles = (columns + 255) / 256;
  const int cw = (columns + tiles - 1) / tiles;
  const int rp = (int)std::max<int64_t>(1, std::min<int64_t>(256 / cw, rows));
  const unsigned threads = (unsigned)((cw * rp + kWaveSize - 1) / kWaveSize * kWaveSize);
  // Rows per thread: as many as leave 512 workgroups, two for each of an MI355X's 256 compute units
  // (best passes: 16 loads in flight 12.9 us for 4096 rows of 4480 fp16 columns in 60 blocks, 8 13.9 us,
  // 4 14.1 us; 13.4 us on average; the copy rate is 14.5 us.
  // One thread per element and a grid row per block took 42 us).
  const auto row_tiles = [&](int r) { return (rows + (int64_t)rp * r - 1) / ((int64_t)rp * r); };
  const auto go = [&](auto kernel, int r) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)row_tiles(r), tiles), dim3(threads), 0, s, b, n_blocks, columns, cw, rp,
                       rows);
  };
  if (row_tiles(16) * tiles >= 512)
    go(regroup_kernel<V, 16>, 16);
  else if (row_tiles(4) * tiles >= 512)
    go(regroup_kernel<V, 4>, 4);
  else
    go(regroup_kernel<V, 1>, 1);
}

// Plain streaming copy, 16 bytes per lane per step.
__global__ __launch_bounds__(256) void tra_copy_kernel(const uint4* __restrict__ src,
                                                        uint4* __restrict__ dst, int64_t n16) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
    dst[i] = src[i];
}

static int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, what);
  return TRA_OK;
}

struct RemapSpec {
  const int64_t* const* sorted_ids;
  const int64_t* const* mapping;
  const int64_t* table_size;
  const int64_t* miss_id;
};

// Launches move_keys_kernel over all output keys: in one go, or kRemapKeys keys with a table at a time.
static int move_keys(MoveArgs& m, int value_bytes, const RemapSpec* spec, hipStream_t s) {
  const int group = spec ? kRemapKeys : kMoveKeys;
  for (int k0 = 0; k0 < m.num_out; k0 += group) {
    m.first_key = k0;
    m.launch_keys = std::min(group, m.num_out - k0);
    // Ids per tile: a block's worth, up to eight of them where that leaves 256 tiles, one for each
    // of an MI355X's compute units (a block with a table reads its pivots once per tile: 410 K ids in
    // tiles of 512 24 us, of 1024 20 us, of 1536 24 us, warm tables).
    const int64_t ids = std::min(m.num_values, m.out_values_end);
    m.tile = kMoveThreads;
    while (m.tile < 8 * kMoveThreads && ids / (2 * m.tile) >= 256) m.tile *= 2;
    // (all ids may belong to this launch's keys, some several times; every key may leave a partial tile)
    const int64_t tiles = m.out_values_end > 0 ? m.out_values_end / m.tile + m.launch_keys : 0;
    m.tile_blocks = (int)std::min<int64_t>(tiles, 1 << 20);
    const int64_t moved = m.out_lengths ? (int64_t)m.launch_keys * m.B : 0;
    const int64_t blocks = m.tile_blocks + std::min<int64_t>((moved + kMoveThreads - 1) / kMoveThreads, 4096);
    if (blocks == 0) continue;
    RemapTables t;
    if (spec) {
      for (int k = 0; k < m.launch_keys; ++k) {
        if (!spec->sorted_ids[k0 + k] || !spec->mapping[k0 + k] || spec->table_size[k0 + k] < 1) {
          set_error("managed-collision remap: key %d has no table", k0 + k);
          return TRA_ERR_INVALID_ARGUMENT;
        }
        t.sorted_ids[k] = spec->sorted_ids[k0 + k];
        t.mapping[k] = spec->mapping[k0 + k];
        t.size[k] = spec->table_size[k0 + k];
        t.miss_id[k] = spec->miss_id[k0 + k];
      }
    }
    const auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kMoveThreads), 0, s, m, t);
    };
    if (spec && value_bytes == 8)
      go(move_keys_kernel<int64_t, true>);
    else if (spec)
      go(move_keys_kernel<int32_t, true>);
    else if (value_bytes == 8)
      go(move_keys_kernel<int64_t, false>);
    else
      go(move_keys_kernel<int32_t, false>);
    const int rc = check_launch("move_keys");
    if (rc != TRA_OK) return rc;
  }
  return TRA_OK;
}

struct RegroupBlock {
  const uint8_t* src;
  uint8_t* dst;
  int64_t src_stride;
  int64_t dst_stride;
  int32_t width;
};

// Both regroup entry points: `block(k)` yields block k's pointers (first column included), row strides in elements and
// width in elements.
template <typename F>
static int regroup_impl(F&& block, int32_t num_blocks, int64_t rows, int32_t elem_bytes, hipStream_t s) {
  if (rows > 0x7fffffff) {  // (blockIdx.x counts row tiles)
    set_error("tra_regroup: %lld rows", (long long)rows);
    return TRA_ERR_TOO_LARGE;
  }
  for (int k0 = 0; k0 < num_blocks;) {
    RegroupBlocks b;
    uint64_t bits = 16;  // its lowest set bit: the widest vector every block of the launch can use
    int nk = 0;
    for (; k0 < num_blocks && nk < kRegroupBlocks; ++k0) {
      const RegroupBlock x = block(k0);
      if (!x.src || !x.dst || x.width < 0 || x.src_stride < x.width || x.dst_stride < x.width) {
        set_error("tra_regroup: block %d is null or wider than its row stride", k0);
        return TRA_ERR_INVALID_ARGUMENT;
      }
      if (x.width == 0) continue;
      b.src[nk] = x.src;
      b.dst[nk] = x.dst;
      b.src_stride[nk] = x.src_stride * elem_bytes;
      b.dst_stride[nk] = x.dst_stride * elem_bytes;
      b.first[nk] = x.width * elem_bytes;  // bytes for now
      bits |= (uint64_t)(uintptr_t)x.src | (uint64_t)(uintptr_t)x.dst | (uint64_t)b.src_stride[nk] |
              (uint64_t)b.dst_stride[nk] | (uint64_t)b.first[nk];
      ++nk;
    }
    if (nk == 0) break;
    const int vec = (int)(bits & (~bits + 1));
    int64_t wide = 0;
    for (int k = 0; k < nk; ++k) {
      const int n = b.first[k] / vec;
      b.first[k] = (int32_t)wide;
      wide += n;
      if (wide > (int64_t)65535 * 256) {  // (blockIdx.y counts column tiles)
        set_error("tra_regroup: %lld column vectors", (long long)wide);
        return TRA_ERR_TOO_LARGE;
      }
    }
    const int columns = (int)wide;
    if (vec == 16)
      launch_regroup<u32x4_t>(b, nk, columns, rows, s);
    else if (vec == 8)
      launch_regroup<u32x2_t>(b, nk, columns, rows, s);
    else if (vec == 4)
      launch_regroup<uint32_t>(b, nk, columns, rows, s);
    else
      launch_regroup<uint16_t>(b, nk, columns, rows, s);
    const int rc = check_launch("tra_regroup");
    if (rc != TRA_OK) return rc;
  }
  return TRA_OK;
}

// pad: the bytes between a row's payload and the next row, and tail_bytes behind the last row, are zeroed
// (header-first rows only).
static int quantize_impl(const float* in, int64_t rows, int32_t dim, int32_t bits, uint8_t* out, int64_t row_bytes,
                         int header_first, hipStream_t s, bool pad = false, int64_t tail_bytes = 0) {
  if (bits != 8 && bits != 4 && bits != 2) {
    set_error("quantize: bits must be 8, 4 or 2 (got %d)", bits);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (dim <= 0 || dim % (8 / bits) != 0 || rows < 0 || row_bytes < dim * bits / 8 + 4) {
    set_error("quantize: bad dim %d / row_bytes %lld for %d bits", dim, (long long)row_bytes, bits);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (rows == 0) return TRA_OK;
  if (!in || !out) {
    set_error("quantize: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  int epl = 32 / bits;
  const bool vec = dim % epl == 0 && row_bytes % 4 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 4 == 0;
  if (pad && (!vec || tail_bytes < 0 || tail_bytes % 4 != 0 || tail_bytes > (1 << 20))) {
    set_error("quantize: padded rows need whole dwords, a 16-byte aligned input and a tail of at most 1 MiB");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (vec) {
    // 8-bit rows: two output dwords (8 elements, two 16-byte loads) per lane and step where the
    // dim allows.  Measured on 1 M rows x 128: 204 us with one dword per lane, 158 us with two,
    // 170 us with four; 4-bit rows are fastest with one (127 us against 133 us with two).
    const bool wide = bits == 8 && dim % 8 == 0;
    if (wide) epl = 8;
    const int chunks = dim / epl;
    int lpr = 1;
    while (lpr < chunks && lpr < kWaveSize) lpr <<= 1;
    const int64_t rows_per_block = 4 * (kWaveSize / lpr);
    const int64_t vblocks = (rows + rows_per_block - 1) / rows_per_block;
    if (vblocks > 0x7fffffff) {
      set_error("quantize: too many rows in one call");
      return TRA_ERR_TOO_LARGE;
    }
    dim3 vg((unsigned)vblocks), vb(256);
    const int64_t lds = rows_per_block * row_bytes;
    if (pad && bits != 2 && chunks <= kWaveSize && lds <= 32 * 1024) {
      const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, vg, vb, (size_t)lds, s, in, rows, dim, (uint32_t*)out, (int32_t)(row_bytes / 4), lpr,
                           (int)(tail_bytes / 4));
      };
      if (wide)
        go(quantize_rows_padded_kernel<8, 2>);
      else if (bits == 8)
        go(quantize_rows_padded_kernel<8, 1>);
      else
        go(quantize_rows_padded_kernel<4, 1>);
      return check_launch("quantize_rows");
    }
    const int pad_dwords = pad ? (int)((row_bytes - 4 - (int64_t)dim * bits / 8) / 4) : 0;
    const auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, vg, vb, 0, s, in, rows, dim, out, row_bytes, header_first, lpr, pad_dwords);
    };
    if (wide)
      go(quantize_rows_vec_kernel<8, 2>);
    else if (bits == 8)
      go(quantize_rows_vec_kernel<8>);
    else if (bits == 4)
      go(quantize_rows_vec_kernel<4>);
    else
      go(quantize_rows_vec_kernel<2>);
    if (pad && tail_bytes > 0)
      hipLaunchKernelGGL(zero_dwords_kernel, dim3(1), dim3(256), 0, s, (uint32_t*)(out + rows * row_bytes),
                         (int)(tail_bytes / 4));
    return check_launch("quantize_rows");
  }
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffff) {
    set_error("quantize: too many rows in one call");
    return TRA_ERR_TOO_LARGE;
  }
  dim3 g((unsigned)blocks), b(256);
  if (bits == 8)
    hipLaunchKernelGGL(quantize_rows_kernel<8>, g, b, 0, s, in, rows, dim, out, row_bytes, header_first);
  else if (bits == 4)
    hipLaunchKernelGGL(quantize_rows_kernel<4>, g, b, 0, s, in, rows, dim, out, row_bytes, header_first);
  else
    hipLaunchKernelGGL(quantize_rows_kernel<2>, g, b, 0, s, in, rows, dim, out, row_bytes, header_first);
  return check_launch("quantize_rows");
}

}  // namespace tra

using namespace tra;

extern "C" {

// The one-launch scan takes up to 131072 lengths: every block sums what lies in front of its tile
// itself, so the last block reads the whole input through one compute unit (512 KB of int32 in
// about 4 us): 7.8 us for 131072 int32 lengths.
constexpr int64_t kSmallScanMax = (int64_t)kSmallMaxTiles * kSmallThreads * 2;
int64_t tra_cumsum_workspace_bytes(int64_t n) {
  if (n <= kSmallScanMax) return 0;
  return (n + kScanTile - 1) / kScanTile * (int64_t)sizeof(int64_t);
}

int tra_cumsum(const void* lengths, int64_t n, int32_t is_i64, void* offsets, void* workspace,
               void* stream) {
  if (n < 0 || !offsets || (n > 0 && !lengths)) {
    set_error("tra_cumsum: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (n > 0x7fffffffLL) {
    set_error("tra_cumsum: n too large");
    return TRA_ERR_TOO_LARGE;
  }
  hipStream_t s = (hipStream_t)stream;
  if (n <= kSmallScanMax) {
    const int per_tile = kSmallThreads * (is_i64 ? 2 : 4);
    const unsigned g = (unsigned)std::max<int64_t>(1, (n + per_tile - 1) / per_tile);
    const bool vec = (uintptr_t)lengths % 16 == 0;
    if (is_i64) {
      if (vec)
        hipLaunchKernelGGL((scan_small_kernel<int64_t, true>), dim3(g), dim3(kSmallThreads), 0, s,
                           (const int64_t*)lengths, n, (int64_t*)offsets);
      else
        hipLaunchKernelGGL((scan_small_kernel<int64_t, false>), dim3(g), dim3(kSmallThreads), 0, s,
                           (const int64_t*)lengths, n, (int64_t*)offsets);
    } else {
      if (vec)
        hipLaunchKernelGGL((scan_small_kernel<int32_t, true>), dim3(g), dim3(kSmallThreads), 0, s,
                           (const int32_t*)lengths, n, (int32_t*)offsets);
      else
        hipLaunchKernelGGL((scan_small_kernel<int32_t, false>), dim3(g), dim3(kSmallThreads), 0, s,
                           (const int32_t*)lengths, n, (int32_t*)offsets);
    }
    return check_launch("tra_cumsum");
  }
  const unsigned tiles = (unsigned)((n + kScanTile - 1) / kScanTile);
  if (!workspace) {
    set_error("tra_cumsum: workspace of %lld bytes required", (long long)tra_cumsum_workspace_bytes(n));
    return TRA_ERR_INVALID_ARGUMENT;
  }
  int64_t* sums = (int64_t*)workspace;
  const bool vec = (uintptr_t)lengths % 16 == 0 && (uintptr_t)offsets % 16 == 0;
  if (is_i64)
    vec ? launch_scan_tiles<int64_t, true>(lengths, n, sums, offsets, tiles, s)
        : launch_scan_tiles<int64_t, false>(lengths, n, sums, offsets, tiles, s);
  else
    vec ? launch_scan_tiles<int32_t, true>(lengths, n, sums, offsets, tiles, s)
        : launch_scan_tiles<int32_t, false>(lengths, n, sums, offsets, tiles, s);
  return check_launch("tra_cumsum");
}

int tra_length_per_key(const void* lengths, int32_t num_features, int32_t batch_size,
                       int32_t is_i64, int64_t* out, void* stream) {
  if (num_features < 0 || batch_size < 0 || (num_features > 0 && (!out || (!lengths && batch_size)))) {
    set_error("tra_length_per_key: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (num_features == 0) return TRA_OK;
  hipStream_t s = (hipStream_t)stream;
  if (is_i64)
    hipLaunchKernelGGL(length_per_key_kernel<int64_t>, dim3(num_features), dim3(kScanThreads), 0, s,
                       lengths, batch_size, out);
  else
    hipLaunchKernelGGL(length_per_key_kernel<int32_t>, dim3(num_features), dim3(kScanThreads), 0, s,
                       lengths, batch_size, out);
  return check_launch("tra_length_per_key");
}

int tra_permute_2d_lengths(const int32_t* permute, int32_t num_out_features, int32_t num_features,
                           int32_t batch_size, const void* lengths, int32_t is_i64,
                           void* out_lengths, void* stream) {
  (void)num_features;
  const int64_t total = (int64_t)num_out_features * batch_size;
  if (num_out_features < 0 || batch_size < 0) {
    set_error("tra_permute_2d_lengths: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (total == 0) return TRA_OK;
  if (!permute || !lengths || !out_lengths) {
    set_error("tra_permute_2d_lengths: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  hipStream_t s = (hipStream_t)stream;
  dim3 g((unsigned)((total + 255) / 256)), b(256);
  if (is_i64)
    hipLaunchKernelGGL(permute_lengths_kernel<int64_t>, g, b, 0, s, permute, total, batch_size,
                       lengths, out_lengths);
  else
    hipLaunchKernelGGL(permute_lengths_kernel<int32_t>, g, b, 0, s, permute, total, batch_size,
                       lengths, out_lengths);
  return check_launch("tra_permute_2d_lengths");
}

int tra_permute_2d_data(const int32_t* permute, int32_t num_out_features, int32_t batch_size,
                        const void* in_offsets, const void* out_offsets, int32_t is_i64,
                        const void* values, int32_t value_bytes, const float* weights,
                        void* out_values, float* out_weights, void* stream) {
  if (num_out_features < 0 || batch_size < 0 || (value_bytes != 4 && value_bytes != 8)) {
    set_error("tra_permute_2d_data: bad argument (value_bytes must be 4 or 8)");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (num_out_features == 0 || batch_size == 0) return TRA_OK;
  if (!permute || !in_offsets || !out_offsets || (weights && !out_weights)) {
    set_error("tra_permute_2d_data: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  hipStream_t s = (hipStream_t)stream;
  dim3 g(64, (unsigned)num_out_features), b(256);
#define GO(OFF, VAL)                                                                          \
  hipLaunchKernelGGL((permute_data_kernel<OFF, VAL>), g, b, 0, s, permute, batch_size,        \
                     in_offsets, out_offsets, (const VAL*)values, weights, (VAL*)out_values,  \
                     out_weights)
  if (is_i64) {
    if (value_bytes == 8) GO(int64_t, int64_t); else GO(int64_t, int32_t);
  } else {
    if (value_bytes == 8) GO(int32_t, int64_t); else GO(int32_t, int32_t);
  }
#undef GO
  return check_launch("tra_permute_2d_data");
}

int tra_bucketize_lengths(const void* offsets, const void* indices, int32_t is_i64,
                          const int64_t* block_sizes, int32_t num_features, int32_t batch_size,
                          int32_t num_buckets, void* new_lengths, void* stream) {
  const int64_t n = (int64_t)num_features * batch_size;
  if (num_features < 0 || batch_size < 0 || num_buckets <= 0) {
    set_error("tra_bucketize_lengths: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (n == 0) return TRA_OK;
  if (!offsets || !block_sizes || !new_lengths) {
    set_error("tra_bucketize_lengths: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  hipStream_t s = (hipStream_t)stream;
  if (num_buckets <= kWalkMaxBuckets) {
    const int bpw = bags_per_wave(n, std::max(1, kWalkMaxBuckets / num_buckets));
    const int64_t waves = (n + bpw - 1) / bpw;
    dim3 g((unsigned)((waves + kWalkWaves - 1) / kWalkWaves)), b(kWalkThreads);
    const size_t lds = (size_t)kWalkWaves * ((bpw + 1) + bpw + ((size_t)num_buckets * bpw + 1) / 2) * sizeof(int64_t);
    if (is_i64)
      hipLaunchKernelGGL(bucketize_lengths_wave_kernel<int64_t>, g, b, lds, s, (const int64_t*)offsets,
                         (const int64_t*)indices, block_sizes, batch_size, n, num_buckets, bpw,
                         (int64_t*)new_lengths);
    else
      hipLaunchKernelGGL(bucketize_lengths_wave_kernel<int32_t>, g, b, lds, s, (const int32_t*)offsets,
                         (const int32_t*)indices, block_sizes, batch_size, n, num_buckets, bpw,
                         (int32_t*)new_lengths);
    return check_launch("tra_bucketize_lengths");
  }
  dim3 g((unsigned)((n + 127) / 128)), b(128);
  if (is_i64)
    hipLaunchKernelGGL(bucketize_lengths_kernel<int64_t>, g, b, 0, s, offsets, indices, block_sizes,
                       batch_size, n, num_buckets, new_lengths);
  else
    hipLaunchKernelGGL(bucketize_lengths_kernel<int32_t>, g, b, 0, s, offsets, indices, block_sizes,
                       batch_size, n, num_buckets, new_lengths);
  return check_launch("tra_bucketize_lengths");
}

int64_t tra_bucketize_workspace_bytes(int32_t num_features, int32_t batch_size, int32_t num_buckets) {
  if (num_features <= 0 || batch_size <= 0 || num_buckets <= kWalkMaxBuckets) return 0;
  return (int64_t)num_features * batch_size * num_buckets * (int64_t)sizeof(int64_t);
}

int tra_bucketize_scatter(const void* offsets, const void* indices, int32_t is_i64,
                          const float* weights, const int64_t* block_sizes, int32_t num_features,
                          int32_t batch_size, int32_t num_buckets, int32_t keep_orig_idx,
                          const void* new_offsets, int64_t* cursor_workspace, void* new_indices,
                          float* new_weights, int64_t* unbucketize_permute, void* stream) {
  const int64_t n = (int64_t)num_features * batch_size;
  if (num_features < 0 || batch_size < 0 || num_buckets <= 0) {
    set_error("tra_bucketize_scatter: bad argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (n == 0) return TRA_OK;
  if (!offsets || !block_sizes || !new_offsets || (weights && !new_weights)) {
    set_error("tra_bucketize_scatter: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  hipStream_t s = (hipStream_t)stream;
  if (num_buckets <= kWalkMaxBuckets) {
    const int bpw = bags_per_wave(n, std::max(1, kWalkMaxBuckets / num_buckets));
    const int64_t waves = (n + bpw - 1) / bpw;
    dim3 g((unsigned)((waves + kWalkWaves - 1) / kWalkWaves)), b(kWalkThreads);
    const size_t lds = (size_t)kWalkWaves * ((bpw + 1) + bpw + (size_t)num_buckets * bpw) * sizeof(int64_t);
    if (is_i64)
      hipLaunchKernelGGL(bucketize_scatter_wave_kernel<int64_t>, g, b, lds, s, (const int64_t*)offsets,
                         (const int64_t*)indices, weights, block_sizes, batch_size, n, num_buckets, bpw,
                         keep_orig_idx, (const int64_t*)new_offsets, (int64_t*)new_indices, new_weights,
                         unbucketize_permute);
    else
      hipLaunchKernelGGL(bucketize_scatter_wave_kernel<int32_t>, g, b, lds, s, (const int32_t*)offsets,
                         (const int32_t*)indices, weights, block_sizes, batch_size, n, num_buckets, bpw,
                         keep_orig_idx, (const int32_t*)new_offsets, (int32_t*)new_indices, new_weights,
                         unbucketize_permute);
    return check_launch("tra_bucketize_scatter");
  }
  if (!cursor_workspace) {
    set_error("tra_bucketize_scatter: more than %d buckets need the cursor workspace", kWalkMaxBuckets);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  dim3 g((unsigned)((n + 127) / 128)), b(128);
  if (is_i64)
    hipLaunchKernelGGL(bucketize_scatter_kernel<int64_t>, g, b, 0, s, offsets, indices, weights,
                       block_sizes, batch_size, n, num_buckets, keep_orig_idx, new_offsets,
                       cursor_workspace, new_indices, new_weights, unbucketize_permute);
  else
    hipLaunchKernelGGL(bucketize_scatter_kernel<int32_t>, g, b, 0, s, offsets, indices, weights,
                       block_sizes, batch_size, n, num_buckets, keep_orig_idx, new_offsets,
                       cursor_workspace, new_indices, new_weights, unbucketize_permute);
  return check_launch("tra_bucketize_scatter");
}

int tra_quantize_rows(const float* in, int64_t rows, int32_t dim, int32_t bits, uint8_t* out,
                      int32_t row_bytes, void* stream) {
  return quantize_impl(in, rows, dim, bits, out, row_bytes, 1, (hipStream_t)stream);
}

int tra_quantize_rows_padded(const float* in, int64_t rows, int32_t dim, int32_t bits, uint8_t* out,
                             int32_t row_stride, int64_t tail_bytes, void* stream) {
  return quantize_impl(in, rows, dim, bits, out, row_stride, 1, (hipStream_t)stream, true, tail_bytes);
}

int tra_quantize_rows_sbhalf(const float* in, int64_t rows, int32_t dim, int32_t bits,
                             uint8_t* out, void* stream) {
  const int64_t rb = bits > 0 && bits <= 8 ? (int64_t)dim * bits / 8 + 4 : 0;
  return quantize_impl(in, rows, dim, bits, out, rb, 0, (hipStream_t)stream);
}

int tra_offsets_range(const void* offsets, int64_t num_bags, int32_t is_i64, int64_t range_size,
                      void* out, void* stream) {
  if (num_bags < 0 || range_size < 0) {
    set_error("tra_offsets_range: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (num_bags == 0 || range_size == 0) return TRA_OK;
  if (!offsets || !out) {
    set_error("tra_offsets_range: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int bpw = bags_per_wave(num_bags, 64);
  const int64_t waves = (num_bags + bpw - 1) / bpw;
  dim3 g((unsigned)((waves + kWalkWaves - 1) / kWalkWaves)), b(kWalkThreads);
  const size_t lds = (size_t)kWalkWaves * (bpw + 1) * sizeof(int64_t);
  if (is_i64)
    hipLaunchKernelGGL(offsets_range_kernel<int64_t>, g, b, lds, (hipStream_t)stream, (const int64_t*)offsets,
                       num_bags, range_size, bpw, (int64_t*)out);
  else
    hipLaunchKernelGGL(offsets_range_kernel<int32_t>, g, b, lds, (hipStream_t)stream, (const int32_t*)offsets,
                       num_bags, range_size, bpw, (int32_t*)out);
  return check_launch("tra_offsets_range");
}

int tra_position_weights(const void* offsets, int32_t is_i64, int32_t num_keys, int32_t batch_size,
                         const int32_t* key_start, const int32_t* key_len, const float* table,
                         float* out, void* stream) {
  if (num_keys < 0 || batch_size < 0) {
    set_error("tra_position_weights: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int64_t n = (int64_t)num_keys * batch_size;
  if (n == 0) return TRA_OK;
  if (!offsets || !key_start || !key_len || !out) {
    set_error("tra_position_weights: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int bpw = bags_per_wave(n, 64);
  const int64_t waves = (n + bpw - 1) / bpw;
  dim3 g((unsigned)((waves + kWalkWaves - 1) / kWalkWaves)), b(kWalkThreads);
  const size_t lds = (size_t)kWalkWaves * (2 * bpw + 1) * sizeof(int64_t);
  if (is_i64)
    hipLaunchKernelGGL(position_weights_kernel<int64_t>, g, b, lds, (hipStream_t)stream, (const int64_t*)offsets,
                       batch_size, n, key_start, key_len, table, bpw, out);
  else
    hipLaunchKernelGGL(position_weights_kernel<int32_t>, g, b, lds, (hipStream_t)stream, (const int32_t*)offsets,
                       batch_size, n, key_start, key_len, table, bpw, out);
  return check_launch("tra_position_weights");
}

int tra_mch_remap(const void* values, int64_t n, int32_t is_i64, const int64_t* sorted_ids,
                  const int64_t* mapping, int64_t table_size, int64_t miss_id, void* out,
                  void* stream) {
  if (n < 0 || table_size <= 0) {
    set_error("tra_mch_remap: bad size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (n == 0) return TRA_OK;
  if (!values || !sorted_ids || !mapping || !out) {
    set_error("tra_mch_remap: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  MoveArgs m = MoveArgs();
  m.values = values;
  m.out_values = out;
  m.num_values = m.out_values_end = n;
  m.kind = kKeysOne;
  m.num_in = m.num_out = 1;
  m.B = 1;
  const RemapSpec spec{&sorted_ids, &mapping, &table_size, &miss_id};
  return move_keys(m, is_i64 ? 8 : 4, &spec, (hipStream_t)stream);
}

int tra_mch_remap_keys(const void* values, int64_t n, const void* offsets, int32_t is_i64,
                       int32_t num_keys, int32_t batch_size, const int64_t* const* sorted_ids,
                       const int64_t* const* mapping, const int64_t* table_size,
                       const int64_t* miss_id, void* out, void* stream) {
  if (n < 0 || num_keys < 0 || batch_size < 0) {
    set_error("tra_mch_remap_keys: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (n == 0 || num_keys == 0) return TRA_OK;
  if (!values || !offsets || !out || !sorted_ids || !mapping || !table_size || !miss_id) {
    set_error("tra_mch_remap_keys: null argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  // (kMoveKeys keys at a time; a chunk's offsets start at its first key's)
  for (int k0 = 0; k0 < num_keys; k0 += kMoveKeys) {
    MoveArgs m = MoveArgs();
    m.bounds = static_cast<const uint8_t*>(offsets) + (int64_t)k0 * batch_size * (is_i64 ? 8 : 4);
    m.bounds_i64 = is_i64;
    m.values = values;
    m.out_values = out;
    m.num_values = m.out_values_end = n;
    m.kind = kKeysOffsets;
    m.num_in = m.num_out = std::min(kMoveKeys, num_keys - k0);
    m.B = batch_size;
    for (int k = 0; k < m.num_in; ++k) m.perm[k] = (int16_t)k;
    const RemapSpec spec{sorted_ids + k0, mapping + k0, table_size + k0, miss_id + k0};
    const int rc = move_keys(m, is_i64 ? 8 : 4, &spec, (hipStream_t)stream);
    if (rc != TRA_OK) return rc;
  }
  return TRA_OK;
}

int tra_permute_keys(const int64_t* key_totals, int32_t num_keys, const int32_t* permute, int32_t num_out_keys,
                     int32_t batch_size, const void* lengths, int32_t lengths_i64, void* out_lengths,
                     const void* values, int64_t num_values, int32_t value_bytes, void* out_values,
                     int64_t num_out_values, const float* weights, float* out_weights,
                     const int64_t* const* sorted_ids, const int64_t* const* mapping, const int64_t* table_size,
                     const int64_t* miss_id, void* stream) {
  if (num_keys < 1 || num_out_keys < 0 || batch_size < 0 || num_values < 0 || num_out_values < 0 ||
      (value_bytes != 4 && value_bytes != 8) || !key_totals || !permute) {
    set_error("tra_permute_keys: bad argument (value_bytes must be 4 or 8)");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (num_keys > kMoveKeys || num_out_keys > kMoveKeys) {
    set_error("tra_permute_keys: %d and %d keys, at most %d are supported", num_keys, num_out_keys, kMoveKeys);
    return TRA_ERR_TOO_LARGE;
  }
  if (num_out_keys == 0) return TRA_OK;
  if ((num_values > 0 && !values) || (num_out_values > 0 && (!out_values || (weights && !out_weights))) ||
      (out_lengths && !lengths) || (sorted_ids && (!mapping || !table_size || !miss_id))) {
    set_error("tra_permute_keys: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  MoveArgs m = MoveArgs();
  m.bounds = key_totals;
  m.values = values;
  m.out_values = out_values;
  m.weights = weights;
  m.out_weights = out_weights;
  m.lengths = lengths;
  m.out_lengths = out_lengths;
  m.lengths_i64 = lengths_i64;
  m.num_values = num_values;
  m.out_values_end = num_out_values;
  m.kind = kKeysTotals;
  m.num_in = num_keys;
  m.num_out = num_out_keys;
  m.B = batch_size;
  for (int j = 0; j < num_out_keys; ++j) {
    if (permute[j] < 0 || permute[j] >= num_keys) {
      set_error("tra_permute_keys: key %d of %d", permute[j], num_keys);
      return TRA_ERR_INVALID_ARGUMENT;
    }
    m.perm[j] = (int16_t)permute[j];
  }
  const RemapSpec spec{sorted_ids, mapping, table_size, miss_id};
  return move_keys(m, value_bytes, sorted_ids ? &spec : nullptr, (hipStream_t)stream);
}

int tra_regroup_columns(const void* const* src, const int64_t* src_stride, void* const* dst,
                        const int64_t* dst_stride, const int32_t* width, int32_t num_blocks,
                        int64_t rows, int32_t elem_bytes, void* stream) {
  if (num_blocks < 0 || rows < 0) {
    set_error("tra_regroup_columns: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (elem_bytes != 2 && elem_bytes != 4) {
    set_error("tra_regroup_columns: element size %d (2 or 4 bytes are supported)", elem_bytes);
    return TRA_ERR_UNSUPPORTED;
  }
  if (num_blocks == 0 || rows == 0) return TRA_OK;
  if (!src || !dst || !src_stride || !dst_stride || !width) {
    set_error("tra_regroup_columns: null argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const auto block = [&](int k) {
    return RegroupBlock{static_cast<const uint8_t*>(src[k]), static_cast<uint8_t*>(dst[k]), src_stride[k],
                        dst_stride[k], width[k]};
  };
  return regroup_impl(block, num_blocks, rows, elem_bytes, (hipStream_t)stream);
}

int tra_regroup_tensors(const void* const* src, const int64_t* src_stride, int32_t num_src, void* const* dst,
                        const int64_t* dst_stride, int32_t num_dst, const int32_t* blocks, int32_t num_blocks,
                        int64_t rows, int32_t elem_bytes, void* stream) {
  if (num_blocks < 0 || rows < 0 || num_src < 0 || num_dst < 0) {
    set_error("tra_regroup_tensors: negative size");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (elem_bytes != 2 && elem_bytes != 4) {
    set_error("tra_regroup_tensors: element size %d (2 or 4 bytes are supported)", elem_bytes);
    return TRA_ERR_UNSUPPORTED;
  }
  if (num_blocks == 0 || rows == 0) return TRA_OK;
  if (!src || !dst || !src_stride || !dst_stride || !blocks) {
    set_error("tra_regroup_tensors: null argument");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  for (int k = 0; k < num_blocks; ++k) {
    const int32_t* b = blocks + 5 * k;
    if (b[0] < 0 || b[0] >= num_src || b[2] < 0 || b[2] >= num_dst || b[1] < 0 || b[3] < 0 || b[4] < 0 ||
        (int64_t)b[1] + b[4] > src_stride[b[0]] || (int64_t)b[3] + b[4] > dst_stride[b[2]]) {
      set_error("tra_regroup_tensors: block %d lies outside its tensors", k);
      return TRA_ERR_INVALID_ARGUMENT;
    }
  }
  const auto block = [&](int k) {
    const int32_t* b = blocks + 5 * k;
    const uint8_t* s = static_cast<const uint8_t*>(src[b[0]]);
    uint8_t* d = static_cast<uint8_t*>(dst[b[2]]);
    return RegroupBlock{s ? s + (int64_t)b[1] * elem_bytes : nullptr, d ? d + (int64_t)b[3] * elem_bytes : nullptr,
                        src_stride[b[0]], dst_stride[b[2]], b[4]};
  };
  return regroup_impl(block, num_blocks, rows, elem_bytes, (hipStream_t)stream);
}

int tra_copy_bytes(const void* src, void* dst, int64_t bytes, void* stream) {
  if (bytes < 0 || bytes % 16 != 0 || (uintptr_t)src % 16 != 0 || (uintptr_t)dst % 16 != 0) {
    set_error("tra_copy_bytes: size and pointers must be multiples of 16 bytes");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  if (bytes == 0) return TRA_OK;
  if (!src || !dst) {
    set_error("tra_copy_bytes: null buffer");
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const int64_t n16 = bytes / 16;
  const unsigned grid = (unsigned)std::min<int64_t>((n16 + 255) / 256, 256 * 32);
  hipLaunchKernelGGL(tra_copy_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream,
                     (const uint4*)src, (uint4*)dst, n16);
  return check_launch("tra_copy_bytes");
}

}  // extern "C"
