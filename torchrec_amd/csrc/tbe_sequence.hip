// Sequence lookup: one dequantized row per id, no reduction.
#include "tbe_lookup_impl.h"

namespace tra {

// Range of ids of class feature `ci` at key position `pos`.  `starts` (kBoundsTotals) holds the keys' first ids.
template <typename IdxT>
__device__ __forceinline__ void sequence_bounds(const LookupArgs& a, int ci, int pos, const int64_t* starts,
                                                int64_t& first, int64_t& n) {
  int64_t last;
  if (a.bounds_kind == kBoundsOffsets) {
    first = load_index<IdxT>(a.offsets, (int64_t)pos * a.B);
    last = load_index<IdxT>(a.offsets, (int64_t)(pos + 1) * a.B);
  } else if (a.bounds_kind == kBoundsTotals) {
    first = starts[pos];
    last = starts[pos + 1];
  } else {
    first = a.pw_off[ci];
    last = first + a.pw_len[ci];
  }
  // (never outside the ids array, whatever the bounds say)
  first = first < 0 ? 0 : first;
  last = last > a.num_indices ? a.num_indices : last;
  n = last > first ? last - first : 0;
}

__device__ __forceinline__ int64_t from_lane(int64_t v, int lane) {
  return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)v, lane));
}

// How a wave's outputs leave: whole rows as one piece, or a lane's columns for themselves (slices of a row, rows that do
// not begin at multiples of 16 bytes).
constexpr int kColumns = 0;
constexpr int kRowsFp16 = 1;
constexpr int kRowsFp32 = 2;
constexpr int kAny = 3;  // one of them, decided where a row is stored

// The outputs of a wave's consecutive rows as one piece, `rows` of them from `first` on: lane c of group g holds NE
// columns of row g.  A lane with several 16-byte vectors would write a part of every line with each store
// instruction; the wave's vectors change places in LDS first.
template <int NE, bool FP16>
__device__ __forceinline__ void store_rows(const float (&acc)[NE], u32x4_t* stage, unsigned char* first, int lpr,
                                           int lane, int rows) {
  constexpr int V = NE * (FP16 ? 2 : 4) / 16;
  constexpr int kPasses = V > kStageVectors ? V / kStageVectors : 1;  // a part of the lanes each
  constexpr int kLanes = kWaveSize / kPasses;
  const int vectors = rows * lpr * V;
#pragma unroll
  for (int h = 0; h < kPasses; ++h) {
    wave_lds_sync();
    if (lane / kLanes == h)
#pragma unroll
      for (int k = 0; k < V; ++k) stage[stage_slot<V>(lane % kLanes, k)] = out_vector<NE, FP16>(acc, k);
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < V / kPasses; ++k) {
      const int i = k * kWaveSize + lane;
      const u32x4_t x = stage[stage_slot<V>(i / V, i % V)];
      const int at = h * kLanes * V + i;
      if (at < vectors) __builtin_nontemporal_store(x, reinterpret_cast<u32x4_t*>(first) + at);
    }
  }
}

// A feature's ids are cut into tiles of sc.window consecutive ids; the tiles of
// the sub-class's features are numbered through, and block t of the sub-class
// takes tiles t, t + blocks, ...: features of very different sizes still fill
// the chip evenly.  Every wave finds the feature of its tile by a scan over the
// features' tile counts.
//
// A tile is walked in steps of kSequenceUnroll rows per lane group: ids, then all row
// chunks, then the arithmetic and the stores, so a wave has 4 rows per lane
// group in flight.  Every lane runs every step (positions past the tile's end
// are clamped and not stored), which is what the matrix instruction of the
// sub-byte conversions needs.
//
// Bound by memory: a 132-byte row costs two 128-byte lines, so 2.1 M int8 rows
// of 128 columns with fp16 results move 1083 MB.  One row per lane group and
// plain stores took 206 us; four in flight, and results that leave as whole
// lines past the caches, 187 us = 5.8 TB/s, what a gather of random
// lines reaches (rows loaded with the non-temporal hint as well: 208 us).
// Where the rows are in the caches the results are what counts (a fill writes
// 6.9 TB/s), and how they leave: 1.8 M rows, us, lanes' vectors as they lie (two of
// them exchanged by cross-lane reads) / whole rows of a wave through LDS:
//   fp32 results: int8 128 columns 315 / 189, 64 84 / 78, 32 64 / 44, 104 234 / 187;
//                 int4 64 162 / 97, int2 128 297 / 180, fp16 104 244 / 187, 32 73 / 51
//   fp16 results: int4 32 57 / 28, 64 65 / 46, int2 128 159 / 95, int8 96 118 / 79,
//                 128 89 / 84
// (Without the non-temporal hint int8 64 fp16 62 -> 92 us, fp16 128 92 -> 156 us.)
// What describes the tile is scalar, so that more waves fit a SIMD: with eight columns a lane (int8 rows in 8-byte, fp16 in
// 16-byte chunks) 63 to 69 registers instead of 118 to 122, seven waves instead of four; with sixteen of int8 or int4 it is
// five before and after.
// Slower than lanes' vectors as they lie and the tile in vector registers: fp16 rows of 16 and 32 columns to fp16, 32-bit
// ids, 25.1 / 26.5 and 46 / 49 us (64-bit ids 27.5 / 26, 56 / 52); 123 K rows of int8 or int4 128 to fp16 9.5 / 9.8.
template <int DTYPE, int CB, typename IdxT>
__global__ __launch_bounds__(kBlockThreads) void tbe_nobag_kernel(const LookupArgs a) {
  constexpr int NE = CB * 8 / Traits<DTYPE>::kBits;
  constexpr int U = kSequenceUnroll;
  __shared__ int64_t s_starts[kMaxTotalKeys + 1];
  constexpr int kStage = NE <= 4 ? 1 : kWaveSize * (NE < 16 ? NE / 4 : kStageVectors);  // vectors a wave puts by
  __shared__ __align__(16) u32x4_t s_stage[kWavesPerBlock * kStage];
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = uniform((int)(threadIdx.x / kWaveSize));
  u32x4_t* stage = s_stage + wave * kStage;
  if (a.bounds_kind == kBoundsTotals) {
    if (wave == 0) {
      const int64_t* totals = reinterpret_cast<const int64_t*>(a.offsets);
      int64_t before = 0;
      for (int k0 = 0; k0 < a.num_keys; k0 += kWaveSize) {
        const int64_t v = k0 + lane < a.num_keys ? totals[k0 + lane] : 0;
        const int64_t incl = wave_scan_incl(v);
        if (k0 + lane < a.num_keys) s_starts[k0 + lane + 1] = before + incl;
        before += wave_last(incl);
      }
      if (lane == 0) s_starts[0] = 0;
    }
    __syncthreads();
  }
  const int blk = blockIdx.x;
  int s = 0;
#pragma unroll
  for (int i = 1; i < kMaxSub; ++i)
    if (i < a.n_sub && blk >= a.sub[i].tile_start) s = i;
  const SubClass sc = a.sub[s];
  const int tile_ids = sc.window;
  const int lpr = sc.lpr;
  const int gpw = kWaveSize / lpr;
  const int g = lane / lpr;
  const int c = lane - g * lpr;
  for (int64_t t = blk - sc.tile_start;; t += sc.tiles_per_feat) {
    // Tile t of the sub-class: its feature and its place among the feature's tiles.
    int fi = -1;
    int64_t first = 0, n = 0, tile = 0, before = 0;
    for (int i0 = 0; i0 < sc.count; i0 += kWaveSize) {
      const int i = min(i0 + lane, sc.count - 1);
      const int ci = sc.first + i;
      const int pos = sc.key0 >= 0 ? sc.key0 + i : a.cdescs[ci].feature;
      int64_t f1, n1;
      sequence_bounds<IdxT>(a, ci, pos, s_starts, f1, n1);
      // (32-bit arithmetic: tiles of under 128 ids are taken only for calls of a few thousand tiles)
      const int tiles = i0 + lane < sc.count ? (int)((n1 + tile_ids - 1) / tile_ids) : 0;
      const int incl = wave_scan_incl((int32_t)tiles);
      const uint64_t past = __builtin_amdgcn_ballot_w64(before + incl > t);
      if (past != 0) {
        const int hit = __builtin_ctzll(past);
        fi = i0 + hit;
        first = from_lane(f1, hit);
        n = from_lane(n1, hit);
        tile = t - before - __builtin_amdgcn_readlane(incl - tiles, hit);
        break;
      }
      before += wave_last(incl);
    }
    if (fi < 0) return;
    const FeatureDesc d = a.cdescs[__builtin_amdgcn_readfirstlane(sc.first + fi)];
    RowWalk w;
    w.chunk_off = Traits<DTYPE>::kHeader + d.payload_off + c * CB;
    w.lane_base = a.weights + d.table_offset + w.chunk_off;
    w.set_rows(d.rows, d.row_bytes);
    w.count_errors = c == 0 && g < gpw && d.payload_off == 0;
    w.hdr_lane = lane - c;
    w.sel0 = mfma_byte_selector(lane, 0);
    w.sel1 = mfma_byte_selector(lane, 1);
    const int64_t col = (int64_t)d.payload_off * 8 / Traits<DTYPE>::kBits;
    const bool whole_rows = a.vec_store != 0 && lpr * NE == d.dim && (!a.out_fp16 || NE >= 8);
    const int64_t begin = first + tile * tile_ids;
    // Places in a tile, in 32 bits where lanes hold few columns: a 64-bit bound is compared in vector registers, there in
    // those that the last row's load had used, so that every wave waited for its last store to end before it left (1.8 M
    // rows, us, 64 / 32 bits: fp16 32 columns to fp16 52 / 49, 64 62 / 54, int8 64 62 / 56, 123 K rows of 64 7.5 / 7.0).
    // With 16 columns 64 bits are better (int8 128 to fp16 84 / 90).
    using Place = std::conditional_t<(NE <= kNarrowLane), int, int64_t>;
    const Place ids = (Place)(min(begin + tile_ids, first + n) - begin);
    const IdxT* in = reinterpret_cast<const IdxT*>(a.indices) + begin;
    // (a step's rows are dealt to the waves before the unroll, so a short tile still keeps all waves busy)
    const auto walk = [&](auto how) {
      constexpr int HOW = decltype(how)::value;
      for (Place w0 = wave * gpw; w0 < ids; w0 += kWavesPerBlock * gpw * U) {
        IdxT id[U];
        bool active[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const Place j = w0 + u * (kWavesPerBlock * gpw) + g;
          active[u] = g < gpw && j < ids;
          id[u] = in[active[u] ? j : ids - 1];
        }
        // (all ids are asked for before the first is looked at: left to the compiler, the last one's load waited for the
        // first id; 1.8 M rows of 16 fp16 columns 27.5 / 26.5 us)
        if constexpr (NE <= 4) __builtin_amdgcn_sched_barrier(0);
        RowBuf<CB> r[U];
        int bad[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          bad[u] = fetch_row<DTYPE, CB, kUnweighted, IdxT>(r[u], id[u], (IdxT)0, (IdxT)0, a, w);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const Place place = w0 + u * (kWavesPerBlock * gpw);  // of the wave's first group
          // (a short tile fills a part of its only step: rows that it does not have are not exchanged in LDS.  Without / with
          // this, us: 3200 rows of int2 512 columns to fp16 10.0 / 6.5, to fp32 13.7 / 7.8, int4 256 to fp32 7.9 / 6.4; 31 K
          // rows of int8 192 to fp16 11.0 / 8.6, 96 7.7 / 6.5)
          if constexpr (NE >= 16)
            if (place >= ids) break;
          if (bad[u] != 0 && active[u] && w.count_errors) atomicAdd(a.err_count, 1ull);
          if (bad[u] != 0 && a.bad_to_row0 != 0) r[u].valid = 1;  // the row fetched for it is row 0
          float acc[NE];
#pragma unroll
          for (int k = 0; k < NE; ++k) acc[k] = 0.0f;
          if constexpr (NE > 16) __builtin_amdgcn_sched_barrier(0);
          consume_row<DTYPE, CB, false>(acc, r[u], w);
          const int64_t row = begin + place;
          const auto rows_as = [&](auto fp16) {
            constexpr bool FP16 = decltype(fp16)::value;
            unsigned char* at = reinterpret_cast<unsigned char*>(a.out) + row * d.dim * (FP16 ? 2 : 4);
            if constexpr (NE * (FP16 ? 2 : 4) == 16) {
              u32x4_t* mine = reinterpret_cast<u32x4_t*>(at) + lane;
              if (active[u]) __builtin_nontemporal_store(out_vector<NE, FP16>(acc, 0), mine);
            } else {
              store_rows<NE, FP16>(acc, stage, at, lpr, lane, (int)min(max(ids - place, (Place)0), (Place)gpw));
            }
          };
          if (HOW == kRowsFp16 || (HOW == kAny && whole_rows && a.out_fp16)) {
            if constexpr (HOW == kRowsFp16 || HOW == kAny) rows_as(std::true_type());
          } else if (HOW == kRowsFp32 || (HOW == kAny && whole_rows)) {
            if constexpr (HOW == kRowsFp32 || HOW == kAny) rows_as(std::false_type());
          } else if (active[u]) {
            store_outputs<NE>(a, (row + g) * (int64_t)d.dim + col + c * NE, acc, a.vec_store != 0);
          }
        }
      }
    };
    // (Lanes of few columns have a loop for each kind of store: 64 int8 columns, 123 K rows 8.0 -> 7.7 us.  With more,
    // one loop is better, the compiler keeps more rows apart: 128 int8 columns, 1.8 M rows 94 -> 84 us.)
    if constexpr (NE >= 16) {
      walk(std::integral_constant<int, kAny>());
    } else if (NE >= 8 && whole_rows && a.out_fp16) {
      if constexpr (NE >= 8) walk(std::integral_constant<int, kRowsFp16>());
    } else if (NE >= 4 && whole_rows) {
      if constexpr (NE >= 4) walk(std::integral_constant<int, kRowsFp32>());
    } else {
      walk(std::integral_constant<int, kColumns>());
    }
  }
}

// fp32 results of eight columns a lane: LDS that leaves room for five blocks on a compute unit.  Seven, which the registers
// allow, write 1.8 M rows of 64 fp16 columns in 84 us, five in 78, of 64 int8 columns in 84 and 79; fp16 results are better
// with seven (54 and 58, 56 and 60 us).
constexpr int kFiveBlocksLds = 18000;

template <int DTYPE, int CB>
static void launch_sequence_cb(const LookupArgs& a, bool idx64, int grid, hipStream_t stream) {
  const int lds = CB * 8 / Traits<DTYPE>::kBits == 8 && !a.out_fp16 ? kFiveBlocksLds : 0;
  if (idx64)
    hipLaunchKernelGGL((tbe_nobag_kernel<DTYPE, CB, int64_t>), dim3(grid), dim3(kBlockThreads), lds, stream, a);
  else
    hipLaunchKernelGGL((tbe_nobag_kernel<DTYPE, CB, int32_t>), dim3(grid), dim3(kBlockThreads), lds, stream, a);
}

template <int DTYPE>
static bool launch_sequence_type(const LookupArgs& a, int cb, bool idx64, int grid, hipStream_t stream) {
  if (cb == 16) {
    if constexpr (DTYPE < kSplitHeader) launch_sequence_cb<DTYPE, 16>(a, idx64, grid, stream);
    return DTYPE < kSplitHeader;
  }
  if (cb == 8) {
    launch_sequence_cb<DTYPE, 8>(a, idx64, grid, stream);
    return true;
  }
  if (cb == 4) launch_sequence_cb<DTYPE, 4>(a, idx64, grid, stream);
  return cb == 4;
}

int launch_sequence(const LookupArgs& a, int dtype, int cb, bool split, bool idx64, int grid, hipStream_t stream) {
  bool ok = false;
  switch (split ? dtype + kSplitHeader : dtype) {
    case TRA_FP32: ok = launch_sequence_type<TRA_FP32>(a, cb, idx64, grid, stream); break;
    case TRA_FP16: ok = launch_sequence_type<TRA_FP16>(a, cb, idx64, grid, stream); break;
    case TRA_INT8: ok = launch_sequence_type<TRA_INT8>(a, cb, idx64, grid, stream); break;
    case TRA_INT4: ok = launch_sequence_type<TRA_INT4>(a, cb, idx64, grid, stream); break;
    case TRA_INT2: ok = launch_sequence_type<TRA_INT2>(a, cb, idx64, grid, stream); break;
    case TRA_INT8 + kSplitHeader: ok = launch_sequence_type<TRA_INT8 + kSplitHeader>(a, cb, idx64, grid, stream); break;
    case TRA_INT4 + kSplitHeader: ok = launch_sequence_type<TRA_INT4 + kSplitHeader>(a, cb, idx64, grid, stream); break;
    case TRA_INT2 + kSplitHeader: ok = launch_sequence_type<TRA_INT2 + kSplitHeader>(a, cb, idx64, grid, stream); break;
  }
  if (!ok) {
    set_error("bad chunk size %d", cb);
    return TRA_ERR_INVALID_ARGUMENT;
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TRA_OK : hip_fail(e, "sequence lookup launch");
}

}  // namespace tra
