// Pooled lookup in groups of sixteen lanes: all tables of a call in one launch.
// Included by one .hip file per (id type, weight mode).
#pragma once

#include "tbe_group_run.h"
#include "tbe_lookup_impl.h"

namespace tra {

// (loads through a pointer made from integers are flat ones without the address space, and waited for with the LDS)
typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;

// NE consecutive columns of a row as one lane loads them: the dwords that hold them, and for rows with a header the
// dword in front (in the row's first lane: the header).
template <int DTYPE, int NE>
struct Columns {
  static constexpr int kBits = Traits<DTYPE>::kBits;
  static constexpr int kDwords = NE * kBits < 32 ? 1 : NE * kBits / 32;
  static constexpr int kFront = Traits<DTYPE>::kHeader != 0 ? 1 : 0;
  static constexpr uint32_t kMask = kBits < 32 ? (1u << (kBits & 31)) - 1 : ~0u;
  uint32_t v[kFront + kDwords];

  // The header on its own (a slice of a row that has several).
  __device__ __forceinline__ void load_split(GlobalBytes row, GlobalBytes p) {
    static_assert(kFront == 1, "rows with a header");
    typedef uint32_t Vec __attribute__((ext_vector_type(kDwords == 1 ? 2 : kDwords), aligned(4)));
    v[0] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(row);
    if constexpr (kDwords == 1) {
      v[1] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(p + 4);
    } else {
      const Vec x = *reinterpret_cast<const __attribute__((address_space(1))) Vec*>(p + 4);
#pragma unroll
      for (int i = 0; i < kDwords; ++i) v[i + 1] = x[i];
    }
  }
  __device__ __forceinline__ void load(GlobalBytes p) {
    if constexpr (kDwords == 1 && kFront == 0 && NE * kBits == 16) {
      v[0] = *reinterpret_cast<const __attribute__((address_space(1))) uint16_t*>(p);
    } else if constexpr (kFront + kDwords == 1) {
      v[0] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(p);
    } else if constexpr (kFront + kDwords == 5) {
      typedef uint32_t Vec __attribute__((ext_vector_type(4), aligned(4)));
      v[0] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>(p);
      const Vec x = *reinterpret_cast<const __attribute__((address_space(1))) Vec*>(p + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i + 1] = x[i];
    } else {
      typedef uint32_t Vec __attribute__((ext_vector_type(kFront + kDwords), aligned(4)));
      const Vec x = *reinterpret_cast<const __attribute__((address_space(1))) Vec*>(p);
#pragma unroll
      for (int i = 0; i < kFront + kDwords; ++i) v[i] = x[i];
    }
  }
  // acc = fmaf(s, column, acc + b) of every column (rows without a header: fmaf(s, column, acc)).
  // shift: where the lane's columns start in a dword that holds more than them.
  __device__ __forceinline__ void add_to(float (&acc)[NE], float s, float b, uint32_t shift, const RowWalk& w) const {
    if constexpr (NE * kBits >= 32) {
      constexpr int EPD = 32 / kBits;
#pragma unroll
      for (int i = 0; i < kDwords; ++i)
        accumulate_dword<DTYPE, true, kBits == 4 || kBits == 2>(acc + i * EPD, v[kFront + i], s, b, w.sel0, w.sel1);
    } else if constexpr (kBits == 16) {
      acc[0] = __builtin_fmaf(s, half_bits_to_float(v[0]), acc[0]);
    } else {
      const uint32_t x = v[kFront] >> shift;
#pragma unroll
      for (int e = 0; e < NE; ++e) fma_step(acc[e], s, (float)((x >> (e * kBits)) & kMask), b);
    }
  }
};

// Lane K's value of every row of sixteen lanes.
template <int K>
__device__ __forceinline__ uint32_t row_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + K, 0xf, 0xf, true);
}
template <int K>
__device__ __forceinline__ float row_bcast(float v) {
  return __builtin_bit_cast(float, row_bcast<K>(__builtin_bit_cast(uint32_t, v)));
}

constexpr int kGroup = 16;      // lanes
// Rows per pipeline batch; two batches are in flight.  A block of sixteen ids is two or four of them.
constexpr int group_batch(int dwords, int ne) { return dwords >= 4 || (dwords >= 3 && ne >= 16) ? 4 : 8; }

template <typename F, int... I>
__device__ __forceinline__ void for_each_row(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>()), ...);
}

// The bags [first, first + count) of a window, at most 16, by one group of lanes.  s_start, s_len: where the window's bags' ids
// start and how many there are (none: zero); bag0: the sample of the window's first bag.
//
// A lane owns NE columns (NE = 1, 2, 4, 8 or 16: up to 16, 32, 64, 128, 256
// columns of a row; of wider rows two or four groups walk the same bags, each
// for its columns) and the group walks the rows one after the other, so a bag's
// sum is evaluated in id order as everywhere.  The bags' ids follow one another
// in memory and are walked as one run, sixteen at a time, one per lane; that
// lane also works out the row's offset, and a row step takes it (and the weight,
// and from the row's first lane the header) with the vector ALU's row broadcast,
// mostly as an operand of the instruction that needs it.  Where a bag ends its sum
// is stored; the loads in flight are the next bag's.
//
// Bound by instruction issue and by latency: such a call has a few waves per SIMD at most, and each adds its rows one
// behind the other.  A row step of four rows (one per group) is 16 vector instructions for 4 int8 columns a lane, where
// lane groups of 8-byte chunks that load every id and header themselves take 45 for their 8 columns and a bag's rows
// take 115 ns each; a launch per weight type and lane chunk came on top.  Kernel times, us, that form / this one:
// 8 tables int8 dim 64, 16 samples, ~20 ids of 64 bits 9.1 / 6.2; the same, 512 samples, 20 ids of 32 bits 7.0 / 6.1;
// 39 tables int2 dim 64, 77 samples, ~31 weighted ids 24 / 10.4; 62 tables of four types in five classes, 24 samples
// 34 (all launches) / 7.8.  Tried: a wave per bag, rows read as scalars with v_readlane (5.4 us on the first case, but
// one load instruction per row: 50 us where this takes 33 on 1 M ids); ids dealt evenly to the groups instead of bags
// (+0.8 us for a barrier more, nothing gained); headers gathered with the ids (every row's line then comes twice
// through the L1).
// MODE: kNear, kFar (the table's rows lie beyond the reach of 32-bit offsets) or kSplit (not every group's columns
// begin behind the row's header).
template <int DTYPE, int NE, typename IdxT, int WEIGHTED, int MODE>
__device__ __forceinline__ void pool_group_bags(const GroupArgs& a, const GroupSlice& d, const float* pw,
                                                int pw_len, const int64_t* s_start, const int* s_len, int bag0,
                                                int first, int count, int lane) {
  using Cols = Columns<DTYPE, NE>;
  using UIdxT = typename std::make_unsigned<IdxT>::type;
  constexpr int U = group_batch(Cols::kFront + Cols::kDwords, NE);
  constexpr bool kHasHeader = Traits<DTYPE>::kHeader != 0;
  const int c = lane & (kGroup - 1);
  const int lane0 = lane - c;  // the group's first lane
  const int cl = lane & ((1 << d.lanes_log2) - 1);  // the lane's place among those of its bag
  const bool has_cols = cl * NE < d.cols;
  const int bit0 = has_cols ? cl * NE * Cols::kBits : 0;
  // where what the lane loads of a row starts
  const uint32_t lane_off = (uint32_t)(d.payload + (kHasHeader ? bit0 / 32 * 4 - 4 : bit0 / 8));
  const uint32_t shift = bit0 % 32;
  const uint8_t* table = a.weights + d.table_offset;
  const IdxT last = (IdxT)(a.num_indices - 1);
  const bool bad_to_row0 = a.bad_to_row0 != 0;
  RowWalk w;
  w.sel0 = mfma_byte_selector(lane, 0);
  w.sel1 = mfma_byte_selector(lane, 1);
  const bool pw_on = pw_len > 0;
  const uint32_t pw_last = (uint32_t)(pw_len > 0 ? pw_len - 1 : 0);
  int bad = 0;
  auto group_mask = [&](bool p) -> uint32_t { return (uint32_t)(__builtin_amdgcn_ballot_w64(p) >> lane0) & 0xffffu; };
  auto of_bag = [&](auto v, int j) { return __shfl(v, lane0 + j, kWaveSize); };

  const int elem = a.out_fp16 ? 2 : 4;
  const int64_t out_row = a.out_stride * elem;
  uint8_t* const out =
      reinterpret_cast<uint8_t*>(a.out) + (int64_t)(bag0 + first) * out_row + (int64_t)(d.out_col + cl * NE) * elem;
  const bool pairs = d.even != 0 && a.pairs != 0;
  auto store = [&](int b, const float (&acc)[NE]) {
    if (!has_cols) return;
    uint8_t* o = out + b * out_row;
    if (a.out_fp16) {
      __half* oh = reinterpret_cast<__half*>(o);
      if constexpr (NE == 1) {
        oh[0] = __float2half_rn(acc[0]);
      } else {
        uint32_t h[NE / 2];
#pragma unroll
        for (int e = 0; e < NE; e += 2)
          h[e / 2] = (uint32_t)__half_as_ushort(__float2half_rn(acc[e])) |
                     ((uint32_t)__half_as_ushort(__float2half_rn(acc[e + 1])) << 16);
        if (pairs)
          __builtin_memcpy(__builtin_assume_aligned(oh, 4), h, NE * 2);
        else
#pragma unroll
          for (int e = 0; e < NE; ++e) oh[e] = __ushort_as_half((unsigned short)(h[e / 2] >> (16 * (e & 1))));
      }
    } else {
      __builtin_memcpy(__builtin_assume_aligned(reinterpret_cast<float*>(o), 4), acc, NE * 4);
    }
  };

  // The group's lane j holds bag j.
  const int n_bags = max(count, 0);
  const int64_t bag_start = c < n_bags ? s_start[first + c] : 0;
  const int bag_len = c < n_bags ? s_len[first + c] : 0;
  bool one_run = true;  // (unless the input is malformed)
  if (__builtin_amdgcn_ballot_w64(n_bags > 1) != 0) {
    // the next lane's start, by a row shift
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bag_start, 0x101, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(bag_start >> 32), 0x101, 0xf, 0xf, true);
    const bool joins = bags_join(bag_start, bag_len, (int64_t)(((uint64_t)hi << 32) | lo));
    one_run = __builtin_amdgcn_ballot_w64(c + 1 < n_bags && !joins) == 0;
  }
  const float inv = a.mean && bag_len > 0 ? 1.0f / (float)bag_len : 1.0f;
  const int most = one_run ? 1 : kGroup;  // runs
  for (int seg = 0; seg < most; ++seg) {
    const int seg_end = one_run ? n_bags : min(seg + 1, n_bags);
    const int seg_last = max(seg_end - 1, 0);
    const bool mine = c >= seg && c < seg_end;
    uint32_t bags = group_mask(mine && bag_len > 0);  // still to be summed
    uint32_t empty = group_mask(mine && bag_len == 0);
    const int64_t start = of_bag(bag_start, min(seg, seg_last));
    const int64_t total = bags != 0 ? of_bag(bag_start, seg_last) + of_bag(bag_len, seg_last) - start : 0;
    int64_t longest = 0;
#pragma unroll
    for (int g = 0; g < kWaveSize / kGroup; ++g) {
      const int64_t t = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(total >> 32), g * kGroup) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane((int)total, g * kGroup));
      longest = t > longest ? t : longest;
    }
    float acc[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) acc[e] = 0.0f;
    while (__builtin_amdgcn_ballot_w64(empty != 0) != 0) {
      if (empty != 0) store(__builtin_ctz(empty), acc);
      empty &= empty - 1;
    }
    if (longest == 0) continue;
    int b = bags != 0 ? __builtin_ctz(bags) : 0;      // the bag being summed
    const int len_b = of_bag(bag_len, b);
    int64_t end = bags != 0 ? len_b : INT64_MAX;      // one behind its last id, from the run's first
    bags &= bags - 1;
    int b_next = bags != 0 ? __builtin_ctz(bags) : b;
    int len_next = of_bag(bag_len, b_next);
    auto finish = [&]() {
      if (a.mean) {
        const float f = of_bag(inv, b);
#pragma unroll
        for (int e = 0; e < NE; ++e) acc[e] *= f;
      }
      store(b, acc);
#pragma unroll
      for (int e = 0; e < NE; ++e) acc[e] = 0.0f;
      end = bags != 0 ? end + len_next : INT64_MAX;
      b = b_next;
      // (looked up one bag ahead: nobody waits for it here)
      bags &= bags - 1;
      b_next = bags != 0 ? __builtin_ctz(bags) : b;
      len_next = of_bag(bag_len, b_next);
    };

    // The ids of places [base, base + 16) of the run, a lane each; -1 behind its end.
    IdxT id;
    float wt = 1.0f;
    auto load_ids = [&](int64_t base) {
      const int64_t k = base + c;
      const IdxT j = (IdxT)(start + k);
      const IdxT jc = (UIdxT)j < (UIdxT)last ? j : last;  // (also catches a wrapped position)
      const IdxT x = reinterpret_cast<const IdxT*>(a.indices)[jc];
      id = k < total ? x : (IdxT)-1;
      if constexpr (WEIGHTED == kPerSample) wt = a.psw[jc];
    };
    // What a block's rows need: the lane's row's offset in the table, its weight (0: skipped) and whether it counts.
    struct Block {
      uint64_t off;
      float w;
      uint32_t keep;
    };
    int pos_bag = seg;  // position weights: the bag of the lane's place
    auto prepare = [&](int64_t base) -> Block {
      Block x;
      x.w = wt;
      if constexpr (WEIGHTED == kByPosition) {
        // the last bag that starts at or in front of the place (an empty one shares its start with the next)
        const int64_t k = start + base + c;
        int lo = min(pos_bag, seg_last), hi = seg_last;
        while (__builtin_amdgcn_ballot_w64(lo < hi) != 0) {
          const int mid = (lo + hi + 1) >> 1;
          const int64_t st = of_bag(bag_start, mid);
          if (lo < hi) {
            if (st <= k) lo = mid; else hi = mid - 1;
          }
        }
        pos_bag = lo;
        const int64_t place = max(k - of_bag(bag_start, lo), (int64_t)0);
        const float v = pw[place < (int64_t)pw_last ? (uint32_t)place : pw_last];
        x.w = pw_on ? v : 1.0f;
      }
      bool valid;
      if constexpr (sizeof(IdxT) == 4)
        valid = (uint32_t)id < d.rows32;
      else
        valid = (uint64_t)id < (uint64_t)d.rows;
      const bool is_bad = !valid && id != (IdxT)-1;
      bad += is_bad ? 1 : 0;
      const UIdxT idc = valid ? (UIdxT)id : (UIdxT)0;
      valid = valid || (is_bad && bad_to_row0);  // (row 0 is what the offset says then)
      x.off = (uint64_t)idc * (uint64_t)(uint32_t)d.row_bytes;
      x.w = valid ? x.w : 0.0f;
      x.keep = valid ? ~0u : 0u;
      return x;
    };
    Cols xa[U], xb[U];
    constexpr std::make_integer_sequence<int, U> rows_of_batch;
    // Requests rows first .. first + U - 1 of a block.
    auto issue = [&](Cols (&x)[U], const Block& blk, auto first) {
      GlobalBytes t = (GlobalBytes)(uintptr_t)table;
      uint32_t lo = lane_off;
      asm volatile("" : "+v"(lo));  // (widened where it is used: the table's address stays a scalar)
      const uint32_t off_lo = (uint32_t)blk.off, off_hi = (uint32_t)(blk.off >> 32);
      for_each_row(rows_of_batch, [&](auto u) {
        constexpr int k = first() + u();
        if constexpr (MODE == kNear) {
          x[u()].load(t + (row_bcast<k>(off_lo) + lo));
        } else {
          GlobalBytes row = t + (((uint64_t)row_bcast<k>(off_hi) << 32) | row_bcast<k>(off_lo));
          if constexpr (MODE == kSplit) x[u()].load_split(row, row + lo); else x[u()].load(row + lo);
        }
      });
    };
    load_ids(0);
    Block cur = prepare(0);
    load_ids(kGroup);
    issue(xa, cur, std::integral_constant<int, 0>());
    for (int64_t base = 0;; base += kGroup) {
      int bag_end = (int)min(end - base, (int64_t)(1 << 30));
      // Adds rows first .. first + U - 1.
      auto consume = [&](Cols (&xs)[U], auto first) {
        for_each_row(rows_of_batch, [&](auto u) {
          constexpr int k = first() + u();
          Cols x = xs[u()];
          // (a skipped row is row 0: its header, or what it holds, inf / nan perhaps, counts as zeros)
          const uint32_t keep = row_bcast<k>(cur.keep);
          float s, b = 0.0f;
          if constexpr (kHasHeader) {
            const uint32_t hdr = row_bcast<0>(x.v[0]) & keep;
            s = half_bits_to_float(hdr & 0xffffu);
            b = half_bits_to_float(hdr >> 16);
            if constexpr (WEIGHTED != 0) {
              s = row_bcast<k>(cur.w) * s;
              b = row_bcast<k>(cur.w) * b;
            }
          } else {
            s = row_bcast<k>(cur.w);
#pragma unroll
            for (int i = 0; i < Cols::kDwords; ++i) x.v[i] &= keep;
          }
          x.add_to(acc, s, b, shift, w);
          if (bag_end == k + 1) {
            finish();
            bag_end = (int)min(end - base, (int64_t)(1 << 30));
          }
        });
      };
      // (rows behind the run's end, up to the end of a batch, are row 0 times zero)
      constexpr std::integral_constant<int, U> second;
      issue(xb, cur, second);
      consume(xa, std::integral_constant<int, 0>());
      if (base + U >= longest) break;
      if constexpr (U == 4) {
        issue(xa, cur, std::integral_constant<int, 8>());
        consume(xb, second);
        if (base + 8 >= longest) break;
        issue(xb, cur, std::integral_constant<int, 12>());
        consume(xa, std::integral_constant<int, 8>());
        if (base + 12 >= longest) break;
      }
      const Block nxt = prepare(base + kGroup);
      load_ids(base + 2 * kGroup);
      issue(xa, nxt, std::integral_constant<int, 0>());
      consume(xb, std::integral_constant<int, kGroup - U>());
      if (base + kGroup >= longest) break;
      cur = nxt;
    }
  }
  // Bad ids are counted by the lanes that hold column 0 and their fifteen neighbours.
  if (d.first_slice != 0 && cl < kGroup && bad != 0) atomicAdd(a.err_count, (unsigned long long)bad);
}

// A block owns a window of consecutive bags of one feature (column slice), each
// of its sixteen lane groups p_per_group (at most 16) consecutive ones of them.
// FROM_LENGTHS: p_bags points at the KJT's lengths; the block sums what lies in
// front of its window and scans the window in LDS.
template <typename IdxT, int WEIGHTED, bool FROM_LENGTHS>
__global__ __launch_bounds__(kBlockThreads, 4) void tbe_pooled_kernel(
    const void* p_bags, const GroupSlice* p_slices, int32_t p_B, int32_t p_per_group, int32_t p_tiles, int32_t p_key0,
    const GroupArgs a, const std::conditional_t<WEIGHTED == kByPosition, GroupPositions, NoPositions> positions) {
  constexpr int kGroups = kBlockThreads / kGroup;
  __shared__ int64_t s_start[kBlockThreads];
  __shared__ int s_len[kBlockThreads];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int ci = blockIdx.x / p_tiles;
  const int b0 = (blockIdx.x - ci * p_tiles) * p_per_group * kGroups;
  const int nb = min(p_per_group * kGroups, p_B - b0);
  const int wave = threadIdx.x / kWaveSize;
  const GroupSlice d = p_slices[ci];
  // (consecutive keys: from the preloaded parameters, so that the bags' bounds are requested at once)
  const int64_t first_bag = (int64_t)(p_key0 >= 0 ? p_key0 + ci : d.key) * p_B + b0;
  const IdxT* bags = reinterpret_cast<const IdxT*>(p_bags) + first_bag;
  const int t = min((int)threadIdx.x, nb - 1);
  if constexpr (FROM_LENGTHS) {
    using Sum = typename SumOf<IdxT>::type;
    __shared__ Sum s_front[kWavesPerBlock], s_tot[kWavesPerBlock];
    const IdxT own = bags[t];
    PrefixSumAtOnce<IdxT> front_sum;
    const Sum part = front_sum.run(reinterpret_cast<const IdxT*>(p_bags), first_bag, (int)threadIdx.x, kBlockThreads);
    // Kept as given: bag starts are the running sum of the lengths as they are.
    const Sum raw = (int)threadIdx.x < nb ? (Sum)own : (Sum)0;
    const Sum incl = wave_scan_incl(raw);
    const Sum front_w = wave_last(wave_scan_incl(part));
    if (lane == kWaveSize - 1) {
      s_tot[wave] = incl;
      s_front[wave] = front_w;
    }
    __syncthreads();
    Sum at = 0;
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w) at += s_front[w] + (w < wave ? s_tot[w] : (Sum)0);
    if ((int)threadIdx.x < nb) {
      s_start[threadIdx.x] = (int64_t)(at + incl - raw);
      s_len[threadIdx.x] = bag_ids((int64_t)raw);
    }
  } else {
    const int64_t start = (int64_t)bags[t], end = (int64_t)bags[t + 1];
    if ((int)threadIdx.x < nb) {
      s_start[threadIdx.x] = start;
      s_len[threadIdx.x] = bag_ids((int64_t)((uint64_t)end - (uint64_t)start));
    }
  }
  __syncthreads();
  const int first = (((int)threadIdx.x >> d.lanes_log2) + d.part * (kBlockThreads >> d.lanes_log2)) * p_per_group;
  const int count = min(p_per_group, nb - first);  // (negative: none)
  if (__builtin_amdgcn_ballot_w64(count > 0) == 0) return;
  const float* pw = nullptr;
  int pw_len = 0;
  if constexpr (WEIGHTED == kByPosition) {
    pw_len = positions.len[ci];
    pw = a.posw + (pw_len > 0 ? positions.off[ci] : 0);
  }

#define TRA_GROUP(D, NE, MODE)                                                                                       \
  case group_kind(D, NE, MODE):                                                                                      \
    pool_group_bags<D, NE, IdxT, WEIGHTED, MODE>(a, d, pw, pw_len, s_start, s_len, b0, first, count, lane);          \
    break;
#define TRA_GROUP_WIDTHS(D, MODE)                                                                                    \
  TRA_GROUP(D, 1, MODE) TRA_GROUP(D, 2, MODE) TRA_GROUP(D, 4, MODE) TRA_GROUP(D, 8, MODE) TRA_GROUP(D, 16, MODE)
#define TRA_GROUP_TYPES(MODE)                                                                                        \
  TRA_GROUP_WIDTHS(TRA_INT8, MODE)                                                                                   \
  TRA_GROUP_WIDTHS(TRA_INT4, MODE)                                                                                   \
  TRA_GROUP_WIDTHS(TRA_INT2, MODE)                                                                                   \
  TRA_GROUP(TRA_FP16, 1, MODE) TRA_GROUP(TRA_FP16, 2, MODE) TRA_GROUP(TRA_FP16, 4, MODE) TRA_GROUP(TRA_FP16, 8, MODE) \
  TRA_GROUP(TRA_FP32, 1, MODE) TRA_GROUP(TRA_FP32, 2, MODE) TRA_GROUP(TRA_FP32, 4, MODE)
  switch (d.kind) {
    TRA_GROUP_TYPES(kNear)
    TRA_GROUP_TYPES(kFar)
    TRA_GROUP(TRA_INT8, 4, kSplit) TRA_GROUP(TRA_INT8, 8, kSplit) TRA_GROUP(TRA_INT8, 16, kSplit)
    TRA_GROUP(TRA_INT4, 8, kSplit) TRA_GROUP(TRA_INT4, 16, kSplit)
    TRA_GROUP(TRA_INT2, 16, kSplit)
  }
#undef TRA_GROUP_TYPES
#undef TRA_GROUP_WIDTHS
#undef TRA_GROUP
}

template <int WEIGHTED>
auto positions_of(const GroupPositions* p) {
  if constexpr (WEIGHTED == kByPosition) return *p; else return NoPositions();
}

#define TRA_DEFINE_GROUP(T, W)                                                                                \
  template <>                                                                                                 \
  void launch_group<T, W>(const GroupArgs& a, const GroupPositions* p, const GroupLaunch& l, bool from_lengths, \
                          hipStream_t stream) {                                                               \
    const auto positions = positions_of<W>(p);                                                                \
    const auto go = [&](auto kernel) {                                                                        \
      hipLaunchKernelGGL(kernel, dim3(l.grid), dim3(kBlockThreads), 0, stream, a.offsets, a.slices, a.B,      \
                         l.per_group, l.tiles, l.key0, a, positions);                                         \
    };                                                                                                        \
    if (from_lengths) go(tbe_pooled_kernel<T, W, true>); else go(tbe_pooled_kernel<T, W, false>);             \
  }

}  // namespace tra
